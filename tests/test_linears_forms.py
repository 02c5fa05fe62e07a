"""Which maps the layer may join (linears) and which must run as modules."""

import types

import pytest
import torch
import torch.nn as nn

from nested_recurrent_memory_amd.layer_ops import (_LinearsFn, _PackFn, _plain_linear,
                                                   first_linear, linears)


def _linear():
    return nn.Linear(8, 8, bias=False)


def test_a_patched_forward_runs_as_a_module(monkeypatch):
    """A forward set on an instance, as wrappers that patch modules in place
    set it, or on the class."""
    m, seq = _linear(), nn.Sequential(_linear(), _linear())
    assert _plain_linear(m) and first_linear(seq) is seq[0]
    m.forward = types.MethodType(lambda self, x: x, m)
    assert not _plain_linear(m)
    seq.forward = types.MethodType(lambda self, x: x, seq)
    assert first_linear(seq) is seq
    m, seq = _linear(), nn.Sequential(_linear(), _linear())
    monkeypatch.setattr(nn.Linear, "forward", lambda self, x: x)
    monkeypatch.setattr(nn.Sequential, "forward", lambda self, x: x)
    assert not _plain_linear(m) and first_linear(seq) is seq


@pytest.mark.parametrize("register", ["register_module_forward_hook", "register_module_forward_pre_hook",
                                      "register_module_full_backward_hook"])
def test_a_global_hook_sees_the_sequential(register):
    seq = nn.Sequential(_linear(), _linear())
    handle = getattr(nn.modules.module, register)(lambda *a: None)
    try:
        assert first_linear(seq) is seq
    finally:
        handle.remove()
    assert first_linear(seq) is seq[0]


@pytest.mark.gpu
def test_nothing_to_differentiate_runs_the_modules(monkeypatch):
    """Gradients on, but neither x nor a weight wants one (an evaluation
    without no_grad): no weight is cast into a pack that nothing needs."""
    mods = [nn.Linear(64, n, bias=False).cuda().requires_grad_(False) for n in (64, 32)]
    x = torch.randn(64, 64, device="cuda").bfloat16()
    with monkeypatch.context() as mp, torch.autocast("cuda", dtype=torch.bfloat16):
        mp.setattr(_LinearsFn, "apply", lambda *a: pytest.fail("joined"))
        assert all(torch.equal(y, m(x)) for y, m in zip(linears(x, mods), mods))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        for leaf in (x, mods[1].weight):
            leaf.requires_grad_(True)
            assert type(linears(x, mods)[0].grad_fn).__name__ == "_LinearsFnBackward"
            leaf.requires_grad_(False)


@pytest.mark.parametrize("needs", [(False, True, False, False), (True, False, False, True),
                                   (True, True, True, True), (False, True, True, False)])
def test_only_wanted_weight_gradients_are_formed(needs, monkeypatch):
    """The rows of weights that want no gradient are neither multiplied nor
    handed on; the others are those of one product."""
    ns, d, rows = (8, 24, 3, 16), 16, 64
    gen = torch.Generator().manual_seed(0)
    ws = [torch.randn(n, d, generator=gen).bfloat16().requires_grad_(r) for n, r in zip(ns, needs)]
    x = torch.randn(rows, d, generator=gen).bfloat16().requires_grad_(True)
    dys = [torch.randn(rows, n, generator=gen).bfloat16() for n in ns]
    ys = _LinearsFn.apply(x, _PackFn.apply(*ws), ns, needs)
    formed, mm = [], torch.mm
    monkeypatch.setattr(torch, "mm", lambda a, b, **kw: formed.append(a.shape[0]) or mm(a, b, **kw))
    torch.autograd.backward(ys, dys)
    assert sum(formed) == rows + sum(n for n, r in zip(ns, needs) if r)      # dx, and dw
    for w, dy, r in zip(ws, dys, needs):
        assert (w.grad is not None) == r
        # bf16 results of the same fp32 sums, 2^-9 of each value
        assert not r or (w.grad - dy.t() @ x).float().norm() <= 2 ** -8 * w.grad.float().norm()
