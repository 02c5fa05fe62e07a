"""The working memory's layouts: sizes that the library refuses reach it, and
a kept buffer read by name has the type that its kernels write."""

import pytest
import torch

from nested_recurrent_memory_amd import _lib, chunk_nested_gdn2
from nested_recurrent_memory_amd import chunk as chunk_mod
from nested_recurrent_memory_amd.inputs import LEAVES, NAMES, make_inputs


def _layout(B, T=130, train=True, es=2):
    return chunk_mod._fwd_layout(B, T, 2, 3, 64, 64, -(-T // 64), (16, 32), (1, 2, 4), False, train,
                                 False, True, 32, es)


@pytest.mark.parametrize("train", [False, True])
def test_layout_of_no_rows(train):
    for lay in _layout(0, train=train)[:2]:
        assert all(row == 0 for _, row, _ in lay.at.values())


@pytest.mark.gpu
@pytest.mark.parametrize("L", [1, 3])
def test_no_rows_is_refused_by_the_library(L):
    inp = make_inputs(B=1, T=130, H=2, K=64, V=64, L=L, N=16, intervals=(1, 2, 4)[:L],
                      dtype=torch.bfloat16)
    rows = ("q", "k", "v", "g", "b", "w", "mix_weights")
    args = {n: (inp[n][:0] if n in rows else inp[n]) for n in NAMES}
    args = {n: (x.cuda() if n in LEAVES else x) for n, x in args.items()}
    with pytest.raises(_lib.NgdnError, match="bad sizes B=0"):
        chunk_nested_gdn2(**args, L=L)


@pytest.mark.parametrize("es,dtype", [(2, torch.bfloat16), (4, torch.float32)])
def test_a_kept_buffer_has_its_own_type(es, dtype):
    """The parameter layouts are of the working type, all else fp32; every
    view lies inside the kept allocation."""
    kept, _, levels = _layout(2, es=es)
    saved = chunk_mod._Saved(kept=torch.zeros(kept.bytes, dtype=torch.uint8), layout=kept,
                             levels=levels)
    for name, (_, _, shape) in kept.at.items():
        params = name in ("bpT", "wpT", "gpT", "kpT", "bankT")
        assert saved[name].shape == shape
        assert saved[name].dtype == (dtype if params else torch.float32), name
    assert saved["bpT"].shape == (2, 2, 64, 64) and saved["states"][0] is None
