"""The decoding step at level counts around its specialised kernels (one to
four levels with every load issued ahead, the general form beyond), in place
and out of place, against the float64 oracle at the op's bar."""

import pytest
import torch

import _parity
import ngdn_oracle as ref
from nested_recurrent_memory_amd import step_nested_gdn2
from nested_recurrent_memory_amd.inputs import NAMES, make_inputs

pytestmark = pytest.mark.gpu

TOKEN = ("q", "k", "v", "g", "b", "w", "mix_weights")


@pytest.mark.parametrize("inplace", [False, True])
@pytest.mark.parametrize("L,K", [(1, 64), (2, 128), (3, 64), (4, 64), (4, 128), (5, 64)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_step_levels(dtype, L, K, inplace):
    f = (1, 1, 2, 2, 4)[:L]
    inp = make_inputs(B=3, T=1, H=2, K=K, V=K, L=L, N=16, intervals=f, dtype=dtype, seed=L + K)
    tok = {n: inp[n][:, 0] for n in TOKEN}
    rest = [inp[n] for n in NAMES[7:]]
    state = torch.randn(3, 2, L, K, K, generator=torch.Generator().manual_seed(3)) * 0.3
    pos = torch.tensor([62, 63, 255])          # nothing, levels 1.., every level
    with torch.no_grad():
        s = state.cuda()
        o, s_new = step_nested_gdn2(**{n: x.cuda() for n, x in tok.items()}, state=s,
                                    position=pos.cuda(),
                                    **{n: inp[n].cuda() for n in NAMES[7:]}, L=L, inplace=inplace)
    assert (s_new is s) == inplace and (inplace or torch.equal(s.cpu(), state))
    o_r, s_r = ref.step_forward(*(tok[n].double() for n in TOKEN), state.double(), pos,
                                *(x.double() for x in rest[:5]), *rest[5:], L=L)
    _parity.check_all([("o", o, o_r), ("state", s_new, s_r)], dtype, test=f"step_L{L}")


@pytest.mark.parametrize("name", ["query_banks", "key_projections", "b_projections", "w_projections",
                                  "g_projections"])
@pytest.mark.parametrize("position", [5, 63])      # the level does not fire; it does
def test_step_refuses_parameters_off_the_gpu(name, position):
    inp = make_inputs(B=1, T=1, H=2, K=64, V=64, L=2, N=16, intervals=(1, 1), dtype=torch.bfloat16)
    args = {n: (inp[n][:, 0] if n in TOKEN else inp[n]) for n in NAMES}
    args = {n: x if n == name else x.cuda() for n, x in args.items()}
    with torch.no_grad(), pytest.raises(ValueError, match="GPU"):
        step_nested_gdn2(**args, state=torch.zeros(1, 2, 2, 64, 64, device="cuda"), position=position,
                         L=2)
