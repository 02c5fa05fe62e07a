"""ngdn_scale: x s in fp32 rounded to the output's type, equal bit for bit to
torch's, over every type pair and the sizes around a thread's eight values
and beyond one grid's first pass (8192 x 256 x 8); and its one caller, the
loss's gradients, where it is and is not taken."""

import pytest
import torch

from nested_recurrent_memory_amd import _lib, model_ops
from nested_recurrent_memory_amd.layer_ops import _code

pytestmark = pytest.mark.gpu

DT = [torch.float32, torch.bfloat16]


@pytest.mark.parametrize("n", [1, 7, 8, 9, 2048 + 3, 8192 * 2048 + 13])
@pytest.mark.parametrize("xd", DT)
@pytest.mark.parametrize("yd", DT)
def test_scale_equals_torch(n, xd, yd):
    g = torch.Generator(device="cuda").manual_seed(n)
    x = torch.randn(n, device="cuda", generator=g).to(xd)
    x[0], x[-1] = float("inf"), -0.0
    s = torch.tensor(1.7, device="cuda")
    y = torch.full((n + 8,), 3.0, device="cuda", dtype=yd)
    _lib.call("ngdn_scale", _code(x), _code(y), n, _lib.ptr(x), _lib.ptr(s), _lib.ptr(y),
              _lib.stream_of(x))
    assert torch.equal(y[:n], (x.float() * 1.7).to(yd)) and bool((y[n:] == 3.0).all())


@pytest.mark.parametrize("wdtype", DT)
def test_loss_gradients_in_blocks_and_differentiated_again(wdtype, monkeypatch):
    torch.manual_seed(0)
    N, d, V = 96, 24, 104
    x = torch.randn(N, d, device="cuda").bfloat16().requires_grad_(True)
    w = torch.randn(V, d, device="cuda").to(wdtype).requires_grad_(True)
    y = torch.randint(0, V, (N,), device="cuda")
    up = torch.tensor(1.7, device="cuda", requires_grad=True)

    def grads(**kw):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss = model_ops.fused_linear_cross_entropy(x, y, w)
        return torch.autograd.grad(loss * up, [x, w], **kw)

    small = grads()                                     # torch's passes
    monkeypatch.setattr(model_ops, "_CARD_BOUND", 0)
    one = grads()
    # bf16 dx: torch rounds the factor and the product to bf16, 2^-9 each, and
    # the kernel the product; dw is fp32 before the product both ways
    assert small[0].dtype == one[0].dtype
    assert (small[0] - one[0]).float().norm() <= 3 * 2 ** -9 * one[0].float().norm()
    assert small[1].dtype == one[1].dtype and torch.equal(small[1], one[1])
    again = grads(create_graph=True)
    for a, b in zip(one, again):
        assert a.dtype == b.dtype and torch.equal(a, b) and b.grad_fn is not None
    monkeypatch.setattr(model_ops, "_BLOCK_BYTES", 32 * V * 2)      # three blocks
    for a, b in zip(one, grads()):
        # each block's gradient rounded to bf16 (2^-9 of a value) before the fp32 sum
        assert a.dtype == b.dtype and (a - b).float().norm() <= 2 ** -8 * a.float().norm()


@pytest.mark.parametrize("wants", [(True, False, False), (True, True, True), (False, True, False)])
def test_loss_of_no_tokens(wants):
    """An empty batch: loss 0, and gradients of zeros in the inputs' shapes
    and types, whichever of them are wanted (a frozen head among them)."""
    x = torch.randn(0, 24, device="cuda").requires_grad_(wants[0])
    w = torch.randn(104, 24, device="cuda").requires_grad_(wants[1])
    b = torch.randn(104, device="cuda").requires_grad_(wants[2])
    with torch.autocast("cuda", dtype=torch.bfloat16):
        loss = model_ops.fused_linear_cross_entropy(x, torch.zeros(0, device="cuda", dtype=torch.long),
                                                    w, b)
    loss.backward()
    assert loss.item() == 0.0
    for t, want in zip((x, w, b), wants):
        assert (t.grad is not None) == want
        assert not want or (t.grad.shape == t.shape and t.grad.dtype == t.dtype and not t.grad.any())
