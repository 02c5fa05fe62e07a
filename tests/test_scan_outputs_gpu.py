"""The level-0 forward scan through the C interface with the sets of outputs
that the op itself does not ask for (each store under its own condition):
the same bits as the set that a training forward takes, for odd and even
chunk counts, a partial last chunk, a sequence in one range and in two, and
grids that take narrow column slices and wide ones. The arithmetic is that of
one step in every form, so nothing but equality is allowed."""

import ctypes

import pytest
import torch

from nested_recurrent_memory_amd import _lib
from nested_recurrent_memory_amd.inputs import make_inputs

pytestmark = pytest.mark.gpu

OUTPUTS = [("read0", "vnT"), ("read0", "h"), ("read0", "vn", "hT"), ("read0", "vnT", "h", "vn", "hT"),
           ("vnT",), ("h", "vn")]


@pytest.mark.parametrize("T", [64, 190, 256, 300])
@pytest.mark.parametrize("K,H", [(64, 2), (64, 33), (128, 2), (128, 17)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_every_set_of_outputs_gives_the_same_bits(dtype, K, H, T):
    B, L, NT = 1, 1, -(-T // 64)
    inp = make_inputs(B=B, T=T, H=H, K=K, V=K, L=L, N=16, intervals=(1,), dtype=dtype, g_scale=0.3,
                      seed=T + K)
    q, k, v, b, w = (inp[n].cuda().to(dtype).contiguous() for n in "qkvbw")
    g = inp["g"].cuda().float().contiguous()
    init = torch.randn(B, H, L, K, K, generator=torch.Generator().manual_seed(3)).cuda()
    new = lambda *s: torch.full(s, float("nan"), device="cuda")  # noqa: E731
    W, U, KtT, Qg = new(B, H, NT, 64, K), new(B, H, NT, 64, K), new(B, H, NT, K, 64), new(B, H, NT, 64, K)
    Aqk, gam = new(B, H, NT, 64, 64), new(B, H, NT, K)
    code = _lib.NGDN_BF16 if dtype == torch.bfloat16 else _lib.NGDN_F32
    d, P, st = _lib.dims(B, T, H, L, K, K, code, K ** -0.5), _lib.ptr, _lib.stream_of(q)
    _lib.call("ngdn_l0_intra_fwd", ctypes.byref(d), *(P(x) for x in (
        q, k, v, g, b, w, W, U, KtT, Qg, Aqk, gam)), None, 0, NT, st)

    def scan(names, ranges):
        out = {n: x for n, x in dict(
            hT=new(B, H, NT, K, K), vnT=new(B, H, NT, K, 64), h=new(B, H, NT, K, K),
            vn=new(B, H, NT, 64, K), read0=new(B, T, H, K)).items() if n in names}
        final = new(B, H, L, K, K)
        for c0, n in ranges:
            _lib.call("ngdn_l0_scan_fwd", ctypes.byref(d), *(P(x) for x in (W, U, KtT, gam, Qg, Aqk)),
                      P(final if c0 else init), 1, *(P(out.get(x)) for x in ("hT", "vnT", "h", "vn", "read0")),
                      P(final), c0, n, st)
        return dict(out, final=final)

    want = scan(("read0", "hT", "h", "vn"), [(0, NT)])
    want["vnT"] = want["vn"].transpose(-1, -2)
    assert all(torch.isfinite(x).all() for x in want.values())
    for names in OUTPUTS:
        for ranges in ([(0, NT)], [(0, 1), (1, NT - 1)] if NT > 1 else []):
            if ranges:
                got = scan(names, ranges)
                assert all(torch.equal(got[n], want[n]) for n in got), (names, ranges)
