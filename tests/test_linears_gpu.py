"""linears(): the layer's maps of one x as one function, against the modules
themselves: bf16 x with fp32 weights under bf16 autocast and with bf16
weights, odd widths, weights that want no gradient, outputs that go unused;
and the forms that must go through the modules (hooks, fp32 x, a bias, a
subclass, no gradients, few rows). Bounds: outputs are the same products; gradients are sums of bf16
values rounded once instead of once per map."""

import pytest
import torch
import torch.nn as nn

from nested_recurrent_memory_amd.layer_ops import _LinearsFn, linears

pytestmark = pytest.mark.gpu


def _rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-30)).item()


def _mods(d, widths, dtype):
    torch.manual_seed(0)
    return [nn.Linear(d, n, bias=False).cuda().to(dtype) for n in widths]


@pytest.mark.parametrize("rows", [(1, 64), (2, 37), (3, 128)])
@pytest.mark.parametrize("widths", [(128, 24, 3, 64), (128, 24, 8, 64)])   # columns in 16 bytes or not
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
def test_linears_match_the_modules(rows, widths, wdtype):
    d = 64
    mods = _mods(d, widths, wdtype)
    mods[1].weight.requires_grad_(False)
    x = torch.randn(*rows, d, device="cuda").bfloat16().requires_grad_(True)
    dys = [torch.randn(*rows, n, device="cuda").bfloat16() for n in widths]
    used = (0, 1, 3)                       # the third output has no gradient
    with torch.autocast("cuda", dtype=torch.bfloat16, enabled=wdtype == torch.float32):
        ys = linears(x, mods)
        assert type(ys[0].grad_fn).__name__ == "_LinearsFnBackward"
        want = [m(x) for m in mods]
    for y, w in zip(ys, want):
        assert y.shape == w.shape and y.dtype == w.dtype and _rel(y, w) <= 2 ** -8
    torch.autograd.backward([ys[i] for i in used], [dys[i] for i in used])
    got = [x.grad] + [m.weight.grad for m in mods]
    x64 = x.detach().double().requires_grad_(True)
    w64 = [m.weight.detach().bfloat16().double().requires_grad_(True) for m in mods]
    torch.autograd.backward([x64 @ w64[i].t() for i in used], [dys[i].double() for i in used])
    # bf16 results of fp32 sums: half an ulp, 2^-9, of each value
    assert got[0].dtype == torch.bfloat16 and _rel(got[0], x64.grad) <= 2 ** -8
    for i, m in enumerate(mods):
        if i == 1:
            assert m.weight.grad is None
        elif i == 2:
            assert m.weight.grad is None or not m.weight.grad.any()
        else:
            assert m.weight.grad.dtype == wdtype and _rel(m.weight.grad, w64[i].grad) <= 2 ** -8


class _Sub(nn.Linear):
    pass


@pytest.mark.parametrize("case", ["hook", "fp32 x", "bias", "subclass", "no autocast",
                                  "fp16 autocast", "no grad", "few rows"])
def test_other_forms_go_through_the_modules(case, monkeypatch):
    monkeypatch.setattr(_LinearsFn, "apply", lambda *a: pytest.fail("fused"))
    mods = _mods(64, (64, 32), torch.bfloat16 if case == "fp16 autocast" else torch.float32)
    seen = []
    x = torch.randn(63 if case == "few rows" else 64, 64, device="cuda").bfloat16()
    if case == "hook":
        mods[0].register_forward_hook(lambda m, a, y: seen.append(y.shape))
    elif case == "fp32 x":
        x = x.float()
    elif case == "bias":
        mods[1] = nn.Linear(64, 32).cuda()
    elif case == "subclass":
        mods[0] = _Sub(64, 64, bias=False).cuda()
    elif case == "no autocast":
        x = x.float()
    dtype = torch.float16 if case == "fp16 autocast" else torch.bfloat16
    with (torch.set_grad_enabled(case != "no grad"),
          torch.autocast("cuda", dtype=dtype, enabled=case != "no autocast")):
        ys = linears(x, mods)
        want = [m(x) for m in mods]
    assert all(torch.equal(a, b) for a, b in zip(ys, want))
    assert case != "hook" or len(seen) == 2


def test_second_derivatives_are_the_modules():
    mods = _mods(32, (8, 24), torch.bfloat16)
    x = torch.randn(65, 32, device="cuda").bfloat16().requires_grad_(True)
    ws = [m.weight for m in mods]

    def second(ys):
        g, = torch.autograd.grad(sum((y.float() ** 2).sum() for y in ys), x, create_graph=True)
        return torch.autograd.grad((g.float() ** 2).sum(), [x, *ws])

    for a, b in zip(second(linears(x, mods)), second([m(x) for m in mods])):
        assert _rel(a, b) <= 2 ** -6       # three products of bf16-rounded values
