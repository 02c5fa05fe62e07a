"""Chunkwise nested Gated DeltaNet on MI355X: the drop-in for the reference's
``nested_gdn2.ops.chunk.chunk_nested_gdn2`` (nested_gdn2/ops/chunk.py:722-766).

Same signature, argument conventions, errors and autograd contract as the
reference op; every arithmetic step runs in the HIP kernels of libngdn.so
(``csrc/``), reached through its C ABI. Python only validates, allocates
outputs and working buffers, and sequences the launches on torch's current
stream. There is no CPU or PyTorch fallback: without the built library or a
GPU the op raises.

Forward, per call (reference composition ops/chunk.py:159-304):
  ngdn_l0_intra_fwd    per-chunk level-0 terms, all chunks in parallel (on
                       small grids range by range, beside the scan)
  ngdn_l0_scan_fwd     level-0 state recurrence: states h per chunk, and
                       the level-0 read (Qg h + Aqk Vn) per row; the states
                       the level above reads (every f_1-th) when L > 1
  for each level l >= 1:
    ngdn_promote_chain_fwd  the level's firings in order per (batch, head):
                            gather, probe and update on chip, one state per
                            group stored (up to 64 pairs per firing), or
    ngdn_probe_fwd          probe the level below at this level's firings,
    ngdn_upper_scan_fwd     then this level's write scan (128 pairs)
  ngdn_output_upper_fwd  every upper read + mix over the scan's level-0
                       read, o written once
"""

from __future__ import annotations

import ctypes
import functools
import math

import torch

from . import _lib
from .schedule import n_firings, n_groups

__all__ = ["chunk_nested_gdn2", "ChunkNestedGDN2Function", "PROMOTIONS"]

PROMOTIONS = ("learned", "merge")
_SUPPORTED_KV = (64, 128)


def _as_ints(x, n):
    vals = [int(v) for v in (x.tolist() if torch.is_tensor(x) else list(x))]
    if len(vals) != n:
        raise ValueError(f"expected {n} entries, got {len(vals)}")
    return vals


def _working_dtype(q):
    if q.dtype == torch.bfloat16:
        return torch.bfloat16, _lib.NGDN_BF16
    # fp32 and fp16 run the fp32 kernels (fp16 -> fp32 is exact)
    return torch.float32, _lib.NGDN_F32


def _validate(q, k, v, L, chunk_size, promotion, n_queries, intervals, query_banks):
    if chunk_size != 64:
        raise ValueError(f"chunk_size must be 64 for GDN-2, got {chunk_size}")
    if promotion not in PROMOTIONS:
        raise ValueError(f"unknown promotion {promotion!r}; expected one of {PROMOTIONS}")
    if q.dim() != 5 or q.shape[3] != L:
        raise ValueError(f"q must be [B, T, H, L={L}, K], got {tuple(q.shape)}")
    B, T, H, _, K = q.shape
    V = v.shape[-1]
    if k.shape != (B, T, H, K) or v.shape[:3] != (B, T, H):
        raise ValueError("k must be [B, T, H, K] and v [B, T, H, V] matching q")
    if K not in _SUPPORTED_KV or V not in _SUPPORTED_KV:
        raise ValueError(f"head dims K={K}, V={V} unsupported; K and V must be 64 or 128")
    if L > 1 and K != V:
        raise ValueError(f"the promotion kernels need K == V, got K={K}, V={V} "
                         "(chunk_nested_gdn2 pads K != V to max(K, V) before this)")
    if L > 8:
        raise ValueError(f"at most 8 levels supported, got L={L}")
    if intervals[0] != 1:
        raise ValueError(f"firing_intervals[0] must be 1, got {intervals[0]}")
    if any(f <= 0 for f in intervals):
        raise ValueError(f"firing intervals must be positive, got {intervals}")
    for lvl in range(1, L):
        n = K if promotion == "merge" else n_queries[lvl - 1]
        if n < 16 or n & (n - 1) or n > 128:
            raise ValueError(f"pairs per firing must be a power of two >= 16, got {n}")
        if promotion == "learned" and n > query_banks.shape[2]:
            raise ValueError(
                f"n_queries={n} exceeds the {query_banks.shape[2]} rows of query_banks")


# Two forms of a level's promotions in the forward. Two launches (the
# default): a probe launch with one workgroup per (batch, head, firing), every
# firing at once, then the level's scan of updates per (batch, head, 32
# columns of V). Fused (True; levels with at most 64 pairs per firing, merge
# at K = 64): one launch per level (ngdn_promote_chain_fwd), one workgroup
# per (batch, head) running its firings in order with the probe and the
# update on chip. The fused form keeps the pairs off HBM but runs B H
# workgroups through a serial chain of firings; at the benchmark shapes the
# two-launch form is faster (c2: 6.67 against 6.91 ms per fwd+bwd step).
FUSED_PROMOTION = False

# The level-0 chunk backward as one launch (ngdn_l0_bwd: the state half per
# chunk in the same workgroup) or two (ngdn_l0_bwd_state, ngdn_l0_bwd_intra);
# read by the forward, which keeps U for the two-launch form only.
FUSED_L0_BWD = True
# dmix_0 (a bandwidth pass over do and the stored read) on the second side
# stream: at the fork, beside the reads' backward (False), or after the
# level-1 probe backward, beside the level-0 reverse scan (True: the reads'
# backward, which the top level's probe backward waits for, then shares the
# GPU with one kernel less; 6.14 -> 6.08 ms at c2)
DMIX0_LATE = True
# The reads' backward of the levels below the top one on the first side
# stream: beside the top level's (False), or after it, beside the top level's
# reverse scan and probe backward (True: the top level's reads backward,
# which starts the chain, then has the GPU to itself; at c2 0.234 -> 0.162
# ms, step 5.32-5.33 -> 5.30-5.31 ms)
READS_AFTER_TOP = True


# Small grids (a long sequence in a small batch: the bf16 level-0 scan then
# runs at most 128 workgroups of 16 columns, half the CUs or fewer): the
# level-0 chunk terms and scan run over L0_PARTS consecutive ranges of
# chunks (at least 64 chunks each), the chunk terms of a range on a side
# stream while the scan works through the range before it; the scan carries
# its state from range to range through the final state, so every chunk's
# arithmetic is that of one launch over all chunks. "Small" is the C
# library's own test for 16-column scan slices (a 32-column grid of at most
# 64 workgroups). Config 3 (T = 65536, B H = 16): 5.47 -> 5.01 ms per forward
# (4 ranges 5.16, 16 ranges 5.08).
L0_PARTS = 8


def _l0_ranges(B, H, V, NT, code):
    """Chunk ranges (c0, n) of the level-0 forward: one for a grid that
    fills the GPU, else up to L0_PARTS of at least 64 chunks."""
    narrow = code == _lib.NGDN_BF16 and B * H * (V // 32) <= 64
    parts = max(1, min(int(L0_PARTS), NT // 64)) if narrow else 1
    bounds = [NT * p // parts for p in range(parts + 1)]
    return [(bounds[p], bounds[p + 1] - bounds[p]) for p in range(parts)]


def _chain_ok(K, N, merge):
    if merge:
        return K == 64 and N == 64
    return K in (64, 128) and N in (16, 32, 64)


# Batch rows are independent all the way through the op, so the kernels run
# per group of batch rows, each group on its own stream: the sequential scans
# of one group (a few workgroups per CU, latency-bound) overlap the chunk
# kernels of another (throughput-bound) instead of leaving most of the GPU idle.
STREAM_GROUPS = 1
_STREAMS = {}


def _side_streams(dev, n):
    key = (dev.index if dev.index is not None else torch.cuda.current_device(), n)
    if key not in _STREAMS:
        _STREAMS[key] = [torch.cuda.Stream(device=dev) for _ in range(n)]   # default priority
    return _STREAMS[key]


def _aux_streams(dev):
    """Two streams (default priority) for independent launches inside one
    backward: the reads' backward next to the top level's scan, and the
    parameter-gradient sums next to the rest of the chain."""
    key = (dev.index if dev.index is not None else torch.cuda.current_device(), "aux")
    if key not in _STREAMS:
        _STREAMS[key] = [torch.cuda.Stream(device=dev) for _ in range(2)]
    return _STREAMS[key]


def _run_groups(B, dev, launch):
    """Calls launch(b0, nb, stream) for each group of batch rows: on the
    current stream when there is one group, else on side streams forked from
    and joined back into the current stream. Returns the number of groups."""
    n = max(1, min(STREAM_GROUPS, B))
    main = torch.cuda.current_stream(dev)
    if n == 1:
        launch(0, B, main)
        return 1
    size = -(-B // n)
    spans = [(b0, min(size, B - b0)) for b0 in range(0, B, size)]
    side = _side_streams(dev, len(spans))
    fork = main.record_event()
    for (b0, nb), st in zip(spans, side):
        st.wait_event(fork)
        with torch.cuda.stream(st):
            launch(b0, nb, st)
    for st in side[:len(spans)]:
        main.wait_stream(st)
    return len(spans)


# ---------------------------------------------------------------- working memory
#
# The working buffers of a pass come from one allocation each (what the
# backward reads again from the forward, and what only the pass itself needs),
# and the kernels take addresses inside it: some forty tensors per pass cost
# more host time than the launches at small shapes (K = 64, B = 2, T = 3000,
# H = 8, four levels: 1.29 -> 0.70 ms per forward + backward, whose kernels take
# 0.64; K = 64, B = 1, T = 333, H = 16, two levels, forward: 145 -> 70 us).
# Where each buffer lies depends on the shapes alone and is worked out once per
# configuration; addresses are formed anew in every call, from the allocation
# as the call (or autograd, for the backward) hands it over.

class _Layout:
    """Buffers in one allocation: name -> (byte offset, bytes per batch row,
    shape), 256-byte aligned; row 0 for buffers without a batch axis.
    ``es``: name -> bytes per value (4: fp32, 2: bf16)."""

    def __init__(self):
        self.at, self.es, self.bytes = {}, {}, 0

    def add(self, name, *shape, es=4, batched=True):
        n = math.prod(shape) * es
        row = n // shape[0] if batched and shape[0] else 0
        self.at[name], self.es[name] = (self.bytes, row, shape), es
        self.bytes += -(-n // 256) * 256

    def ptrs(self, base, b0=0):
        """name -> address of batch row b0 in the allocation at ``base``."""
        return {n: base + o + b0 * r for n, (o, r, _) in self.at.items()}


def _arena(lay, dev):
    return torch.empty(lay.bytes, device=dev, dtype=torch.uint8)


@functools.lru_cache(maxsize=256)
def _fwd_layout(B, T, H, L, K, V, NTF, nq, f, merge, train, fused_promotion, fused_l0, nmax, es):
    """(kept, tmp, levels) of a forward: the buffers the backward reads (an
    empty layout without one), the others, and per level (None for level 0)
    its pairs per firing, firings, groups and form."""
    NT = -(-T // 64)
    kept, tmp = _Layout(), _Layout()
    keep = kept.add if train else tmp.add
    for n, shape in (("W", (64, K)), ("Qg", (64, K)), ("KtT", (K, 64)), ("Aqk", (64, 64)),
                     ("gam", (K,))):
        keep(n, B, H, NT, *shape)
    # U only for the two-launch chunk backward (the fused one forms dA from Vn)
    (tmp.add if fused_l0 else keep)("U", B, H, NT, 64, V)
    # level 0's read of every token, formed by the level-0 scan while each
    # chunk's state is on chip; the output pass adds the upper levels' reads
    # and the mix (and the backward's dmix_0 reads it again)
    keep("read0", B, T, H, V)
    # the state entering each chunk, transposed: read by level 1's probes at
    # every f1-th chunk only, so only those are written
    if L > 1:
        keep("hT", B, H, NT, V, K)
    if train:
        keep("TT", B, H, NT, 64, 64)
        keep("h", B, H, NT, K, V)
        keep("vn", B, H, NT, 64, V)
    levels = [None] * L
    for lvl in range(1, L):
        nf, ng = n_firings(NTF, f[lvl]), n_groups(NT, f[lvl])
        N = K if merge else nq[lvl - 1]
        nf1 = max(nf, 1)
        # one launch: probes and updates on chip; the backward's keys,
        # (keys b e^g)^T and e^g only when training
        chain = fused_promotion and _chain_ok(K, N, merge)
        levels[lvl] = dict(N=N, nf=nf, ng=ng, chain=chain)
        if not chain:
            tmp.add(f"A{lvl}", B, H, nf1, N, K)
            tmp.add(f"KT{lvl}", B, H, nf1, K, N)
            tmp.add(f"U{lvl}", B, H, nf1, N, V)
        if train or not chain:
            keep(f"gam{lvl}", B, H, nf1, K)
        if train:
            keep(f"keys{lvl}", B, H, nf1, N, K)
            keep(f"AT{lvl}", B, H, nf1, K, N)
        # group states as rows and transposed
        keep(f"states{lvl}", B, ng, H, K, V)
        keep(f"statesT{lvl}", B, ng, H, V, K)
    if L > 1:     # the parameters with their last two axes swapped
        for n in ("bpT", "wpT", "gpT") + (("kpT",) if train else ()):
            keep(n, L - 1, H, K, V, es=es, batched=False)
        if train:
            keep("bankT", L - 1, H, K, nmax, es=es, batched=False)
    return kept, tmp, levels


@functools.lru_cache(maxsize=256)
def _bwd_layout(B, T, H, L, K, V, levels, merge, fused_l0, carry):
    """The backward's working buffers; levels: (N, nf) per upper level."""
    NT = -(-T // 64)
    lay = _Layout()
    for lvl in range(1, L):
        N, nf, ng = levels[lvl - 1]
        nfa = max(nf, 1)
        lay.add(f"d_states{lvl}", B, ng, H, K, V)
        lay.add(f"dSp{lvl}", B, H, nfa, K, V)
        lay.add(f"dvn{lvl}", B, H, nfa, N, V)
        for j in range(6):
            lay.add(f"ws{lvl}_{j}", B, H, nfa, N, K)
        if not merge:
            lay.add(f"dbank{lvl}", B, H, nfa, N, K)
        lay.add(f"inj{lvl}", B, H, nfa, K, V)
    # per-slice partials of the parameter-gradient sums, shared by the levels
    # (their sums run one after another on one stream)
    if L > 1:
        lay.add("parts", 4, H, _lib.PARAM_SPLIT, K, V, batched=False)
    lay.add("dSp0", B, H, NT, K, V)
    lay.add("dVnT0", B, H, NT, V, 64)
    # dQg, dKt: the fused chunk backward's workspaces; the rest only for the
    # two-launch form
    lay.add("dQg", B, H, NT, 64, K)
    lay.add("dKt", B, H, NT, 64, K)
    if not fused_l0:
        lay.add("dVn0", B, H, NT, 64, V)
        lay.add("dWT", B, H, NT, K, 64)
        lay.add("dAqk", B, H, NT, 64, 64)
        lay.add("dgam", B, H, NT, K)
    if carry:
        lay.add("carry", B, H, L, K, V)
    return lay


def _row(t, b0):
    """Address of batch row b0 of a contiguous batch-leading tensor (None stays None)."""
    if t is None:
        return None
    return t.data_ptr() + b0 * t.stride(0) * t.element_size() if b0 else t.data_ptr()


class _Saved(dict):
    """What a forward hands to its backward: the tensors (inputs in the
    working dtype, the kept allocation, the final state, the parameters) and
    the configuration. A working buffer's name gives a view of it."""

    def buffer(self, name):
        o, _, shape = self["layout"].at[name]
        es = self["layout"].es[name]
        flat = self["kept"][o:o + math.prod(shape) * es]
        return flat.view(torch.float32 if es == 4 else torch.bfloat16).view(shape)

    def __missing__(self, name):
        if name in ("states", "statesT"):
            return [None] + [self.buffer(f"{name}{lvl}") for lvl in range(1, len(self["levels"]))]
        return self.buffer(name)


def _fire_chunks(T, fire_partial):
    """Chunks whose end can complete an upper level's firing: every chunk,
    or (fire_partial False) the whole ones only, so that a partial last
    chunk fires nothing, as the decoding step treats an incomplete chunk
    (the library's ngdn_dims.hold_partial)."""
    NT = -(-T // 64)
    return NT if fire_partial else T // 64


def _forward(q, k, v, g, b, w, mix, qb, kp, bp, wp, gp, nq, f, L, scale,
             init, promotion, train, fire_partial=True):
    """Runs the forward kernels. Returns (o, final_state [B,H,L,K,V] fp32,
    working tensors kept for the backward when ``train``)."""
    B, T, H, _, K = q.shape
    V = v.shape[-1]
    dev = q.device
    wd, code = _working_dtype(q)
    NT = -(-T // 64)
    NTF = _fire_chunks(T, fire_partial)
    cvt = lambda x: x.to(wd).contiguous()  # noqa: E731
    q_, k_, v_, b_, w_, mix_ = (cvt(x) for x in (q, k, v, b, w, mix))
    g_ = g.to(torch.float32).contiguous()
    init_ = init.to(torch.float32).contiguous() if init is not None else None
    merge = promotion == "merge"
    f, nq = tuple(f), tuple(nq)
    params, nmax = (), 0
    if L > 1:
        params = _working_params(qb, kp, bp, wp, gp, wd)
        nmax = params[0].shape[2]

    # everything is allocated here, on the current stream, before any launch
    kept_lay, tmp_lay, levels = _fwd_layout(B, T, H, L, K, V, NTF, nq, f, merge, train,
                                            FUSED_PROMOTION, FUSED_L0_BWD, nmax,
                                            wd.itemsize)
    kept = _arena(kept_lay, dev) if train else None
    tmp = _arena(tmp_lay, dev)
    final = torch.empty(B, H, L, K, V, device=dev, dtype=torch.float32)
    o = torch.empty(B, T, H, V, device=dev, dtype=wd)
    kept_base, tmp_base = (kept.data_ptr() if train else 0), tmp.data_ptr()
    if L > 1:
        p0 = {**tmp_lay.ptrs(tmp_base), **kept_lay.ptrs(kept_base)}
        bank, kp_, bp_, wp_, gp_ = params
        _transpose_into([bp_, wp_, gp_] + ([kp_, bank] if train else []),
                        [p0[n] for n in ("bpT", "wpT", "gpT")
                         + (("kpT", "bankT") if train else ())])
        bank_p, kp_p = bank.data_ptr(), kp_.data_ptr()

    def launch(b0, nb, st):
        sp = st.cuda_stream
        d = _lib.dims(nb, T, H, L, K, V, code, scale, hold_partial=NTF < NT)
        dp = ctypes.byref(d)
        p = {**tmp_lay.ptrs(tmp_base, b0), **kept_lay.ptrs(kept_base, b0)}
        get = p.get
        xq, xk, xv, xg, xb, xw, xmix = (_row(x, b0) for x in (q_, k_, v_, g_, b_, w_, mix_))
        xinit, xfin = _row(init_, b0), _row(final, b0)
        ranges = _l0_ranges(nb, H, V, NT, code) if nb == B else [(0, NT)]
        ts = _aux_streams(dev)[0] if len(ranges) > 1 else st
        if ts is not st:
            ts.wait_event(st.record_event())
        # every range's chunk terms queued at once on the side stream (holding
        # them to one or two ranges ahead of the scan measured slower)
        ready = []
        for c0, n in ranges:
            _lib.call("ngdn_l0_intra_fwd", dp, xq, xk, xv, xg, xb, xw, p["W"], p["U"], p["KtT"],
                      p["Qg"], p["Aqk"], p["gam"], get("TT"), c0, n, ts.cuda_stream, stream=ts)
            ready.append(ts.record_event() if ts is not st else None)
        # with several ranges and unfused promotions, the upper levels follow
        # on a second side stream, one range behind: after level-0 range p,
        # each level probes and scans the firings whose lower state is stored
        tu = (_aux_streams(dev)[1] if len(ranges) > 1 and L > 1
              and not any(levels[lvl]["chain"] for lvl in range(1, L)) else None)
        done = [0] * L          # firings of each level probed and scanned so far
        for i, (c0, n) in enumerate(ranges):
            if ready[i] is not None:
                st.wait_event(ready[i])
            # a range after the first starts from the state the one before left in final
            _lib.call("ngdn_l0_scan_fwd", dp, p["W"], p["U"], p["KtT"], p["gam"], p["Qg"], p["Aqk"],
                      xinit if i == 0 else xfin, f[1] if L > 1 else 1, get("hT"), None, get("h"),
                      get("vn"), p["read0"], xfin, c0, n, sp)
            if tu is not None:
                tu.wait_event(st.record_event())
                upper_batch(dp, p, xinit, xfin, done, c0 + n, i == len(ranges) - 1, tu)
        if tu is not None:
            st.wait_event(tu.record_event())
        else:
            upper_batch(dp, p, xinit, xfin, done, NT, True, st)
        spT, ngs, fs = _level_arrays([None] + [p[f"statesT{lvl}"] for lvl in range(1, L)], NT, f, L)
        _lib.call("ngdn_output_upper_fwd", dp, p["read0"], xq, xmix, spT, ngs, fs, _row(o, b0), sp)

    def upper_batch(dp, p, xinit, xfin, done, avail, last, su):
        """Probes and scans of every upper level for the firings whose lower
        state is stored: level 0 has stored the states entering chunks
        [0, avail); each level then has stored the groups entering its firings
        so far. A firing i reads the lower level's stored state
        ((i + 1) f_here) / f_below, so the firings with (i + 1) f_here <
        avail f_below are ready; the last batch takes the rest (including
        those that read the lower final state) and stores every level's
        trailing groups. dp, p: the launch's dims and addresses; su: the
        stream."""
        sp = su.cuda_stream
        get = p.get
        for lvl in range(1, L):
            lv = levels[lvl]
            fh, fb = f[lvl], f[lvl - 1]
            nf, N = lv["nf"], lv["N"]
            upto = nf if last else min(nf, max(0, (avail * fb - 1) // fh))
            i0 = done[lvl]
            if lv["chain"]:
                belowT, ngb = (p["hT"], NT) if lvl == 1 else (p[f"statesT{lvl - 1}"], n_groups(NT, fb))
                _lib.call("ngdn_promote_chain_fwd", dp, lvl, int(merge), N, fb, fh, belowT, ngb, xfin,
                          bank_p, nmax, kp_p, p["bpT"], p["wpT"], p["gpT"], xinit,
                          p[f"states{lvl}"], p[f"statesT{lvl}"], get(f"keys{lvl}"), get(f"AT{lvl}"),
                          get(f"gam{lvl}"), sp, tag=f"ngdn_promote_chain_fwd.{lvl}")
                continue
            below, ngb = (p["hT"], NT) if lvl == 1 else (p[f"states{lvl - 1}"], n_groups(NT, fb))
            A, KT, U, gam = p[f"A{lvl}"], p[f"KT{lvl}"], p[f"U{lvl}"], p[f"gam{lvl}"]
            if upto > i0:
                _lib.call("ngdn_probe_fwd", dp, lvl, int(merge), N, fb, fh, below, ngb, xfin, bank_p,
                          nmax, kp_p, p["bpT"], p["wpT"], p["gpT"], A, KT, U, gam, get(f"keys{lvl}"),
                          get(f"AT{lvl}"), None, None, None, None, None, i0, upto - i0, sp,
                          tag=f"ngdn_probe_fwd.{lvl}", stream=su)
            if upto > i0 or (last and nf == 0):
                # a range after the level's first starts from the state in final
                _lib.call("ngdn_upper_scan_fwd", dp, lvl, N, nf, lv["ng"], A, KT, U, gam,
                          xinit if i0 == 0 else xfin, p[f"states{lvl}"], p[f"statesT{lvl}"], xfin, i0,
                          upto - i0, sp, tag=f"ngdn_upper_scan_fwd.{lvl}", stream=su)
            done[lvl] = upto
            # the groups of this level stored so far bound the level above's firings
            avail = upto

    _run_groups(B, dev, launch)
    saved = None
    if train:
        saved = _Saved(q=q_, k=k_, v=v_, b=b_, w=w_, mix=mix_, g=g_, kept=kept, final=final,
                       params=params, layout=kept_lay, levels=levels, fused_l0=FUSED_L0_BWD,
                       NTF=NTF, code=code, wd=wd, nmax=nmax)
    return o, final, saved


def _working_params(qb, kp, bp, wp, gp, wd):
    """The parameters contiguous in the working dtype, the bank padded to a
    multiple of 8 rows so every row start is 16-byte aligned. fp32 parameters
    of a bf16 call (autocast) are cast in one launch."""
    nmax = qb.shape[2]
    if nmax % 8:
        qb = torch.nn.functional.pad(qb, (0, 0, 0, -nmax % 8))
    xs = [qb, kp, bp, wp, gp]
    if wd == torch.bfloat16 and all(x.dtype == torch.float32 and x.is_contiguous() for x in xs):
        return tuple(_cast_bf16(xs))
    return tuple(x.to(wd).contiguous() for x in xs)


def _params(qb, kp, bp, wp, gp, wd):
    """Per-level parameters in the layouts the step's kernels read: the bank
    and key projections as they are, the other projections with their last
    two axes swapped."""
    qb_, kp_, bp_, wp_, gp_ = _working_params(qb, kp, bp, wp, gp, wd)
    tr = _transpose_last2([bp_, wp_, gp_])
    return dict(qb=qb_, nmax=qb_.shape[2], kp=kp_, bpT=tr[0], wpT=tr[1], gpT=tr[2])


def _transpose_last2(xs):
    """Contiguous tensors of one dtype transposed in their last two axes
    (ngdn_transpose: one launch on the current stream)."""
    if any(not x.is_contiguous() or x.dtype != xs[0].dtype or x.dim() < 2 for x in xs):
        raise ValueError("_transpose_last2: contiguous tensors of one dtype, at least 2-D")
    outs = [torch.empty(x.shape[:-2] + (x.shape[-1], x.shape[-2]), device=x.device, dtype=x.dtype)
            for x in xs]
    _transpose_into(xs, [y.data_ptr() for y in outs])
    return outs


def _transpose_into(xs, dsts):
    """xs (contiguous, one dtype) transposed in their last two axes to the
    addresses dsts, in one launch on the current stream."""
    n = len(xs)
    I = ctypes.c_int32 * n  # noqa: E741
    _lib.call("ngdn_transpose", n, (ctypes.c_void_p * n)(*[x.data_ptr() for x in xs]),
              (ctypes.c_void_p * n)(*dsts),
              I(*[x.numel() // max(1, x.shape[-1] * x.shape[-2]) for x in xs]),
              I(*[x.shape[-2] for x in xs]), I(*[x.shape[-1] for x in xs]),
              xs[0].element_size(), _lib.stream_of(xs[0]))


def _cast_bf16(xs):
    """Contiguous fp32 tensors cast to bf16, each into a tensor of its own, in
    one launch on the current stream."""
    outs = [torch.empty(x.shape, device=x.device, dtype=torch.bfloat16) for x in xs]
    n = len(xs)
    _lib.call("ngdn_cast_bf16", n, (ctypes.c_void_p * n)(*[x.data_ptr() for x in xs]),
              (ctypes.c_void_p * n)(*[y.data_ptr() for y in outs]),
              (ctypes.c_int64 * n)(*[x.numel() for x in xs]), _lib.stream_of(xs[0]))
    return outs


def _level_arrays(states, NT, f, L):
    """The per-level argument arrays of the output entry points; states:
    tensors or addresses, the first (level 0) unused."""
    sp = (ctypes.c_void_p * L)(*([None] + [s if isinstance(s, int) else s.data_ptr()
                                           for s in states[1:]]))
    ngs = (ctypes.c_int32 * L)(*([0] + [n_groups(NT, f[l]) for l in range(1, L)]))
    fs = (ctypes.c_int32 * L)(*f)
    return sp, ngs, fs


def _backward(sv, do, dfinal, L, scale, f, nq, has_init, promotion):
    """Runs the backward kernels (ops/chunk.py:374-564, mirrored). Returns the
    gradients in the working dtype (fp32 for g, the states and parameters)."""
    q_, k_, v_, b_, w_, mix_, g_ = (sv[n] for n in ("q", "k", "v", "b", "w", "mix", "g"))
    B, T, H, _, K = q_.shape
    V = v_.shape[-1]
    dev = q_.device
    wd, code, nmax = sv["wd"], sv["code"], sv["nmax"]
    NT = -(-T // 64)
    e = lambda *s, dt=wd: torch.empty(*s, device=dev, dtype=dt)  # noqa: E731
    f32 = lambda *s: e(*s, dt=torch.float32)  # noqa: E731
    do_ = do.to(wd).contiguous()
    merge = promotion == "merge"
    levels, final, params = sv["levels"], sv["final"], sv["params"]
    # the form the forward saved for (U is kept only for the two-launch form)
    fused_l0 = sv["fused_l0"]
    # small grids, one group of rows, the fused chunk backward: the level-0
    # reverse scan runs the chunk ranges of the forward last first, the
    # gradient of the state between ranges carried in a buffer, and each
    # range's chunk backward runs on a side stream beside the scan of the
    # range before it
    l0_ranges = (_l0_ranges(B, H, V, NT, code)
                 if fused_l0 and max(1, min(STREAM_GROUPS, B)) == 1 else [(0, NT)])

    # everything is allocated (and zeroed) here, on the current stream
    lay = _bwd_layout(B, T, H, L, K, V,
                      tuple((lv["N"], lv["nf"], lv["ng"]) for lv in levels[1:]), merge, fused_l0,
                      len(l0_ranges) > 1)
    work = _arena(lay, dev)
    work_base, kept_base, kept_lay = work.data_ptr(), sv["kept"].data_ptr(), sv["layout"]
    dq, dmix = e(B, T, H, L, K), f32(B, T, H, L)
    dk, dv, db, dw = e(B, T, H, K), e(B, T, H, V), e(B, T, H, K), e(B, T, H, V)
    dg = f32(B, T, H, K)
    zeros = []
    if dfinal is not None:
        d_final = dfinal.to(torch.float32).contiguous().clone()
    else:
        d_final = f32(B, H, L, K, V)
        zeros.append(d_final)
    d_init = f32(B, H, L, K, V) if has_init else None
    if has_init:
        zeros.append(d_init)
    dqb = dkp = dbp = dwp = dgp = None
    if L > 1:
        dqb, dkp, dbp, dwp, dgp = (f32(L - 1, H, *s) for s in ((nmax, K), (K, V), (V, K), (V, V),
                                                               (V, K)))
        zeros += [dqb, dkp, dbp, dwp, dgp]
        bank_p, kp_p, bp_p, wp_p, gp_p = (x.data_ptr() for x in params)
        dpar = [x.data_ptr() for x in (dqb, dkp, dbp, dwp, dgp)]
    if zeros:
        torch._foreach_zero_(zeros)

    def param_grads(dp, p, lvl, st):
        lv = levels[lvl]
        _lib.call("ngdn_param_grads", dp, lvl, int(merge), lv["N"], lv["nf"],
                  *[p[f"ws{lvl}_{j}"] for j in range(5)], p.get(f"dbank{lvl}"), nmax, *dpar,
                  p["parts"], st.cuda_stream, tag=f"ngdn_param_grads.{lvl}", stream=st)

    def launch(b0, nb, st):
        sp = st.cuda_stream
        d = _lib.dims(nb, T, H, L, K, V, code, scale, hold_partial=sv["NTF"] < NT)
        dp = ctypes.byref(d)
        p = {**kept_lay.ptrs(kept_base, b0), **lay.ptrs(work_base, b0)}
        get = p.get
        xq, xk, xv, xg, xb, xw, xmix, xdo = (_row(x, b0) for x in (q_, k_, v_, g_, b_, w_, mix_, do_))
        xfin, xdfin, xdinit, xdq, xdmix = (_row(x, b0) for x in (final, d_final, d_init, dq, dmix))
        # With one group of rows, independent launches go to two side streams:
        # (a) the reads' backward of the levels below the top one
        # (each writes its own columns of dmix and dq and its own d_states)
        # beside the top level's reverse scan and probe backward (after the
        # top level's read, or beside it when READS_AFTER_TOP is off; the
        # probe backward's lower-state gradient goes to an injection, not
        # into d_states),
        # joined before the first reverse scan that reads those d_states; (b) each
        # level's parameter-gradient sums (reading only that level's
        # workspaces) and dmix_0 (before level 1's sums, or at the fork when
        # DMIX0_LATE is off) beside the rest of the chain, joined at the end. With
        # several groups of rows the sums run once over all rows after the
        # groups join, so every row group's partials are in place and the
        # result does not depend on the grouping.
        aux = _aux_streams(dev) if (L > 1 and nb == B) else None
        if aux is not None:
            fork = st.record_event()
            for a in aux:
                a.wait_event(fork)
        ta, tb = (aux[0], aux[1]) if aux else (st, st)
        # reads: dmix for every level (level 0 from the stored read, on the
        # second side stream), dq and the group-state gradients for levels >= 1
        dmix0_done = []

        def dmix0():
            _lib.call("ngdn_output_bwd", dp, p["read0"], xdo, xdmix, tb.cuda_stream, stream=tb)
            dmix0_done.append(True)
        if not (DMIX0_LATE and aux is not None):
            dmix0()
        late = READS_AFTER_TOP and aux is not None
        for lvl in ([L - 1] + list(range(1, L - 1)) if late else range(1, L)):
            t = st if lvl == L - 1 else ta
            _lib.call("ngdn_read_state_bwd", dp, lvl, f[lvl], levels[lvl]["ng"], xq, xmix, xdo,
                      p[f"states{lvl}"], p[f"d_states{lvl}"], xdq, xdmix, t.cuda_stream,
                      tag=f"ngdn_read_state_bwd.{lvl}", stream=t)
            if late and lvl == L - 1:
                ta.wait_stream(st)
        joined = aux is None
        inj, nf1 = None, 0
        for lvl in range(L - 1, 0, -1):
            lv = levels[lvl]
            N, nf, ng = lv["N"], lv["nf"], lv["ng"]
            if not joined and lvl < L - 1:
                st.wait_stream(ta)
                joined = True
            # the level above's injection (its probe backward's lower-state
            # gradients), added by this level's reverse scan
            up = lvl + 1 < L and levels[lvl + 1]["nf"] > 0
            dSp, dvn, gam = p[f"dSp{lvl}"], p[f"dvn{lvl}"], get(f"gam{lvl}")
            _lib.call("ngdn_upper_scan_bwd", dp, lvl, N, nf, ng, p[f"keys{lvl}"], p[f"AT{lvl}"], gam,
                      p[f"d_states{lvl}"], p[f"inj{lvl + 1}"] if up else None, f[lvl],
                      f[lvl + 1] if up else 1, levels[lvl + 1]["nf"] if up else 0, xdfin, dSp, dvn,
                      xdinit, sp, tag=f"ngdn_upper_scan_bwd.{lvl}")
            if nf == 0:
                continue
            fh, fb = f[lvl], f[lvl - 1]
            if lvl == 1:
                inj, nf1 = p["inj1"], nf
                b_kv, b_vk, ngb = p["h"], p["hT"], NT
            else:
                b_kv, b_vk = p[f"states{lvl - 1}"], p[f"statesT{lvl - 1}"]
                ngb = n_groups(NT, fb)
            _lib.call("ngdn_probe_bwd", dp, lvl, int(merge), N, fb, fh, b_kv, b_vk, ngb, xfin, bank_p,
                      nmax, kp_p, p["bpT"], p["wpT"], p["gpT"], p["kpT"], p["bankT"], bp_p, wp_p, gp_p,
                      p[f"states{lvl}"], p[f"statesT{lvl}"], ng, dSp, dvn,
                      *[p[f"ws{lvl}_{j}"] for j in range(6)], get(f"dbank{lvl}"), p[f"inj{lvl}"],
                      xdfin, sp, tag=f"ngdn_probe_bwd.{lvl}")
            if nb == B:
                if aux is not None:
                    tb.wait_stream(st)
                if DMIX0_LATE and aux is not None and lvl == 1:
                    dmix0()
                param_grads(dp, p, lvl, tb)
        if not joined:
            st.wait_stream(ta)
        if not dmix0_done:
            # (late placement) after the upper levels' parameter-gradient sums
            dmix0()
        # level 0
        ranges = l0_ranges if nb == B else [(0, NT)]
        tl = _aux_streams(dev)[0] if len(ranges) > 1 else st
        xdk, xdv, xdg, xdb, xdw = (_row(x, b0) for x in (dk, dv, dg, db, dw))
        for i in reversed(range(len(ranges))):
            c0, n = ranges[i]
            last = i == len(ranges) - 1
            _lib.call("ngdn_l0_scan_bwd", dp, p["W"], p["KtT"], p["gam"], p["Qg"], p["Aqk"], xdo, xmix,
                      f[1] if L > 1 else 1, inj, nf1, xdfin if last else p["carry"], p["dSp0"],
                      get("dVn0"), p["dVnT0"], xdinit if i == 0 else p["carry"], c0, n, sp)
            if fused_l0:
                # the chunk backward in one launch: the state half per chunk
                if tl is not st:
                    tl.wait_event(st.record_event())
                _lib.call("ngdn_l0_bwd", dp, xq, xk, xv, xg, xb, xw, p["TT"], p["h"], p["dSp0"], p["vn"],
                          p["dVnT0"], xdo, xmix, p["dQg"], p["dKt"], xdq, xdk, xdv, xdg, xdb, xdw, c0, n,
                          tl.cuda_stream, stream=tl)
        if tl is not st:
            st.wait_stream(tl)
        if not fused_l0:
            _lib.call("ngdn_l0_bwd_state", dp, p["h"], p["dSp0"], p["vn"], p["dVn0"], xdo, xmix,
                      p["dQg"], p["dWT"], p["dKt"], p["dAqk"], p["dgam"], sp)
            _lib.call("ngdn_l0_bwd_intra", dp, xq, xk, xv, xg, xb, xw, p["W"], p["U"], p["TT"], p["dQg"],
                      p["dWT"], p["dKt"], p["dAqk"], p["dgam"], p["dVnT0"], xdq, xdk, xdv, xdg, xdb, xdw,
                      sp)
        if aux is not None:
            st.wait_stream(tb)

    groups = _run_groups(B, dev, launch)
    if groups > 1:
        st = torch.cuda.current_stream(dev)
        d = _lib.dims(B, T, H, L, K, V, code, scale, hold_partial=sv["NTF"] < NT)
        p = lay.ptrs(work_base)
        for lvl in range(L - 1, 0, -1):
            if levels[lvl]["nf"] > 0:
                param_grads(ctypes.byref(d), p, lvl, st)
    return dq, dk, dv, dg, db, dw, dmix, dqb, dkp, dbp, dwp, dgp, d_init


# the entries of _Saved that are tensors (params: five more)
_SAVED_TENSORS = ("q", "k", "v", "b", "w", "mix", "g", "kept", "final")


class ChunkNestedGDN2Function(torch.autograd.Function):
    """Autograd node for the whole op (ops/chunk.py:567-719)."""

    @staticmethod
    def forward(ctx, q, k, v, g, b, w, mix_weights, query_banks, key_projections,
                b_projections, w_projections, g_projections, n_queries_per_level,
                firing_intervals, L, scale, initial_state, output_final_state,
                chunk_size, promotion, fire_partial_chunk=True):
        L = int(L)
        f = _as_ints(firing_intervals, L)
        nq = _as_ints(n_queries_per_level, L - 1) if L > 1 else []
        _validate(q, k, v, L, chunk_size, promotion, nq, f, query_banks)
        if not q.is_cuda:
            raise RuntimeError("chunk_nested_gdn2 runs on the GPU only; got CPU tensors")
        K = q.shape[-1]
        if scale is None:
            scale = K ** -0.5
        # the backward's extra layouts are written only when a gradient is wanted
        train = any(ctx.needs_input_grad)
        o, final, saved = _forward(q, k, v, g, b, w, mix_weights, query_banks,
                                   key_projections, b_projections, w_projections,
                                   g_projections, nq, f, L, scale, initial_state,
                                   promotion, train, fire_partial_chunk)
        o = o.to(q.dtype)
        ctx.meta = (L, scale, f, nq, initial_state is not None, promotion)
        ctx.dtypes = [None if t is None else t.dtype
                      for t in (q, k, v, g, b, w, mix_weights, query_banks, key_projections,
                                b_projections, w_projections, g_projections, initial_state)]
        ctx.nmax = query_banks.shape[2] if L > 1 else 0
        # the working tensors go through save_for_backward, so that activation
        # checkpointing (torch.utils.checkpoint) can drop them after the
        # forward and have them recomputed for the backward
        if saved is not None:
            ctx.save_for_backward(*(saved[n] for n in _SAVED_TENSORS), *saved["params"])
            ctx.saved_config = {n: x for n, x in saved.items()
                                if n not in _SAVED_TENSORS and n != "params"}
        return o, (final if output_final_state else None)

    @staticmethod
    def backward(ctx, do, dfinal):
        L, scale, f, nq, has_init, promotion = ctx.meta
        tensors = ctx.saved_tensors
        n = len(_SAVED_TENSORS)
        sv = {**ctx.saved_config, **dict(zip(_SAVED_TENSORS, tensors)), "params": tensors[n:]}
        grads = _backward(sv, do, dfinal, L, scale, f, nq, has_init, promotion)
        (dq, dk, dv, dg, db, dw, dmix, dqb, dkp, dbp, dwp, dgp, dinit) = grads
        dts = ctx.dtypes
        grads = [dq, dk, dv, dg, db, dw, dmix] + ([dqb, dkp, dbp, dwp, dgp] if L > 1 else [])
        out = _cast_grads(grads, dts[:len(grads)])
        if L > 1:
            if out[7].shape[2] != ctx.nmax:
                out[7] = out[7][:, :, :ctx.nmax]      # drop the alignment padding rows
        else:
            out += [None] * 5
        return (*out, None, None, None, None,
                dinit.to(dts[12]) if dinit is not None else None, None, None, None, None)


def _cast_grads(grads, dtypes):
    """The gradients in their inputs' dtypes. The fp32 -> bf16 casts (dg,
    dmix, the parameter sums for bf16 inputs) run in one launch into
    separately allocated tensors, which autograd takes as the leaves'
    gradients without copying them (views of one shared buffer it copies);
    the rest cast with torch."""
    out = list(grads)
    batch = [i for i, (x, dt) in enumerate(zip(grads, dtypes))
             if x is not None and x.dtype == torch.float32 and dt == torch.bfloat16
             and x.is_contiguous()]
    if len(batch) > 1:
        for i, y in zip(batch, _cast_bf16([grads[i] for i in batch])):
            out[i] = y
    else:
        batch = []
    return [x if x is None or i in batch else x.to(dt)
            for i, (x, dt) in enumerate(zip(out, dtypes))]


def chunk_nested_gdn2(q, k, v, g, b, w, mix_weights, query_banks, key_projections,
                      b_projections, w_projections, g_projections, n_queries_per_level,
                      firing_intervals, L, scale=None, initial_state=None,
                      output_final_state=False, chunk_size=64, promotion="learned",
                      fire_partial_chunk=True):
    """Differentiable chunkwise NestedGDN-2. Signature matches the reference op
    (nested_gdn2/ops/chunk.py:722-743) and its naive twin (ops/naive.py:226-247).

    Returns (o [B, T, H, V] in q's dtype, final_state [B, H, L, K, V] fp32 or None).

    ``fire_partial_chunk`` (an addition; the reference's chunk form always
    fires): with False, a partial last chunk completes no upper level's
    firing, as the reference's decoding step treats an incomplete chunk
    (ops/naive.py:101-113). The op then gives, for any T, what the reference
    layer computes by running whole chunks through the chunk op and stepping
    the rest (layers/nested_gdn2.py:196-224), differentiable throughout.

    K != V with upper levels (the layer's expand_v != 1) runs the K = V
    kernels at D = max(K, V) on zero-padded inputs and parameters: the padded
    channels stay exactly zero through every level and carry no gradient into
    the real ones, so the results are those of the unpadded op (see
    ``pad_kv``).
    """
    K, V = q.shape[-1], v.shape[-1]
    if int(L) > 1 and K != V:
        if promotion == "merge" and K < V:
            raise ValueError(f"merge promotion with K < V (K={K}, V={V}) is not supported: "
                             "its decay is a mean over K pairs")
        (q, k, v, g, b, w, query_banks, key_projections, b_projections, w_projections,
         g_projections, initial_state) = pad_kv(
            K, V, q=q, k=k, v=v, g=g, b=b, w=w, query_banks=query_banks,
            key_projections=key_projections, b_projections=b_projections,
            w_projections=w_projections, g_projections=g_projections,
            initial_state=initial_state)
        o, fin = ChunkNestedGDN2Function.apply(
            q, k, v, g, b, w, mix_weights, query_banks, key_projections, b_projections,
            w_projections, g_projections, n_queries_per_level, firing_intervals, L,
            K ** -0.5 if scale is None else scale, initial_state, output_final_state,
            chunk_size, promotion, fire_partial_chunk)
        return o[..., :V], (fin[..., :K, :V] if fin is not None else None)
    return ChunkNestedGDN2Function.apply(
        q, k, v, g, b, w, mix_weights, query_banks, key_projections, b_projections,
        w_projections, g_projections, n_queries_per_level, firing_intervals, L,
        scale, initial_state, output_final_state, chunk_size, promotion, fire_partial_chunk)


def pad_kv(K, V, *, q=None, k=None, v=None, g=None, b=None, w=None, query_banks=None,
           key_projections=None, b_projections=None, w_projections=None, g_projections=None,
           initial_state=None, state=None):
    """The op's tensors zero-padded to D = max(K, V) in their K and V axes
    (None stays None), in the order of the keywords. With K < V the key axis
    grows: q, k, b, g and the bank get zero channels, so those channels of
    the decay-masked products, of W, Kt, Qg and of every state row stay zero
    (their decay e^0 = 1 keeps a zero row zero), and the write keys
    u = Vals Wk^T get zero columns (the norm is unchanged). With V < K the
    value axis grows: v and w get zero channels, so U, Vn, the states'
    columns and Vals stay zero there, and the zero rows of the b, g, w
    projections keep the gates of the real channels unchanged. Gradients
    reaching the padded channels are zero or are dropped by the padding's
    backward. (Merge with K < V would average its decay over D pairs instead
    of K: refused by the caller.)"""
    D = max(K, V)
    pk, pv = D - K, D - V
    F = torch.nn.functional

    def last(t, p):
        return t if t is None or p == 0 else F.pad(t, (0, p))

    def last2(t, p_row, p_col):
        return t if t is None or (p_row == 0 and p_col == 0) else F.pad(t, (0, p_col, 0, p_row))

    out = [last(q, pk), last(k, pk), last(v, pv), last(g, pk), last(b, pk), last(w, pv),
           last(query_banks, pk), last2(key_projections, pk, pv),
           last2(b_projections, pv, pk), last2(w_projections, pv, pv),
           last2(g_projections, pv, pk), last2(initial_state, pk, pv)]
    if state is not None:
        out.append(last2(state, pk, pv))
    return out


def default_scale(K: int) -> float:
    return 1.0 / math.sqrt(K)
