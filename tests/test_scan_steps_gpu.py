"""The scans' loops at the step counts where they can go wrong (they run two
steps per iteration): one step, an odd and an even number, a partial last
chunk; with narrow column slices (few heads) and wide ones; with the
backward's outputs and without. The narrow run is held to the float64 oracle
at the op's bar; a wide run's heads and a run without a backward give the same
bits (a slice only selects columns, an output only adds stores)."""

import pytest
import torch

import _parity
import ngdn_oracle as ref
from nested_recurrent_memory_amd import chunk_nested_gdn2
from nested_recurrent_memory_amd.inputs import LEAVES, NAMES, make_cotangent, make_inputs

pytestmark = pytest.mark.gpu

L = 3
# the axis of the heads in each argument
HEAD = {n: 1 if n.endswith("projections") or n == "query_banks" else 2 for n in LEAVES}


def _heads(inp, do, n):
    return ({m: (inp[m].narrow(HEAD[m], 0, n).contiguous() if m in LEAVES else inp[m])
             for m in NAMES}, do[:, :, :n].contiguous())


def _run(inp, do):
    gpu = {n: (inp[n].cuda().requires_grad_(True) if n in LEAVES else inp[n].cuda())
           for n in NAMES}
    o, s = chunk_nested_gdn2(**gpu, L=L, output_final_state=True)
    o.backward(do.cuda())
    return {"o": o, "state": s, **{"d" + n: gpu[n].grad for n in LEAVES}}


@pytest.mark.parametrize("T", [64, 190, 256])
@pytest.mark.parametrize("K,H", [(64, 33), (128, 17)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_step_counts_and_slice_widths(dtype, K, H, T):
    inp = make_inputs(B=1, T=T, H=H, K=K, V=K, L=L, N=32, intervals=(1, 1, 2), n_queries=(32, 16),
                      dtype=dtype, g_scale=0.3, seed=T + K)
    do = make_cotangent((1, T, H, K), seed=5).to(dtype)
    few, do_few = _heads(inp, do, 2)
    wide, narrow = _run(inp, do), _run(few, do_few)
    for n in narrow:
        axis = 1 if n == "state" else 2 if n == "o" else HEAD[n[1:]]
        assert torch.equal(wide[n].narrow(axis, 0, 2), narrow[n]), n
    with torch.no_grad():
        o, s = chunk_nested_gdn2(**{n: few[n].cuda() for n in NAMES}, L=L, output_final_state=True)
    assert torch.equal(o, narrow["o"]) and torch.equal(s, narrow["state"])

    lv = {n: few[n].double().requires_grad_(True) for n in LEAVES}
    args = [lv[n] for n in LEAVES] + [few["n_queries_per_level"], few["firing_intervals"]]
    o_r, s_r = ref.chunk_forward(*args, L=L, output_final_state=True, out_dtype=torch.float64)
    (o_r * do_few.double()).sum().backward()
    want = {"o": o_r, "state": s_r, **{"d" + n: lv[n].grad if lv[n].grad is not None
                                       else torch.zeros_like(lv[n]) for n in LEAVES}}
    _parity.check_all([(n, narrow[n], want[n]) for n in want], dtype, test=f"steps_{K}_{T}")
