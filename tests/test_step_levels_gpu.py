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
