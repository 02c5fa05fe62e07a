"""Which maps the layer may join (linears) and which must run as modules."""

import types

import pytest
import torch
import torch.nn as nn

from nested_recurrent_memory_amd.layer_ops import _LinearsFn, _plain_linear, first_linear, linears


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
