// The sequential half of every level: a chain of delta-rule steps
//   Vn = U - A S,   S <- diag(gam) S + BT Vn
// run per (batch, head, 32-column slice of V) with the fp32 state held in
// registers across all steps.
//
// Level 0 (the state recurrence of fla's chunk_gdn2_fwd, reached from
// nested_gdn2/ops/chunk.py:236-248; semantics ops/naive.py:367-392): one step
// per chunk with A = W, BT = Kt^T, U = U, gam = e^gc_last.
// Levels >= 1 (ops/update_fwd.py:21-128): one step per firing with
// A = keys * b * e^g, BT = keys^T, U = values * w, gam = e^g, which is
// S' = e^g S - keys^T ((keys*b)(e^g S)) + keys^T (values*w).
//
// Columns of V never interact, so a workgroup owns BV = SCAN_BV of them and
// the grid is B*H*(V/BV), the slices of one (batch, head) placed on one XCD so
// they share its L2. Per step: the state slice is written (transposed, fp32)
// to LDS as the B operand of A S; Vn goes through LDS as the B operand of
// BT Vn. A, BT, U and gam do not depend on the state: each wave reads the
// rows it needs one step ahead into registers, so the loads of step j+1
// overlap step j. Every operand is derived (fp32); for bf16 inputs each
// product is three bf16 MFMAs on split operands.
#include "ngdn_kernels.h"

namespace ngdn {

// OUT (level 0): each step also forms the chunk's level-0 read
//   read0 = Qg S + Aqk Vn
// on the same tiles as Vn, with S^T and Vn^T already in LDS as the B
// operands (the state is on chip, so the output pass needs neither the state
// sequence nor Vn from HBM).
// FRM (bf16): bit 0, BT in fragment order (M % 32 == 0); bit 1, A (and, OUT,
// Qg and Aqk) too.
// SM, the outputs of a step: 1, level 0 without a backward (read0, and the
// transposed state where it is due); 2, level 0 with one (also the state and
// Vn); 3, an upper level (the state, and its transpose when set). These issue
// every store of a step unconditionally (buffer stores, dropped where not
// due) and run two steps per loop iteration on two operand sets, so that a
// step waits for its own operands only: with stores under branches and one
// set copied to the next at the loop's end, every step waited for all of its
// own stores as well. 0, any set of outputs, each store under its condition
// (the entry points' less common calls).
template <typename E, int K, int M, int BV, int NWV, bool OUT, int FRM, int SM>
__global__ __launch_bounds__(NWV * WAVE) void scan_fwd_kernel(ScanArgs a) {
  constexpr int CT = BV / 16;                 // column tiles
  constexpr int RTS = K / 16;                 // state row tiles
  constexpr int TPW = RTS * CT / NWV;         // state tiles per wave
  constexpr int TRT = (TPW + CT - 1) / CT;    // distinct state row tiles per wave
  constexpr int RTV = M / 16;                 // Vn row tiles
  // Vn tiles of a wave, p < NVP: when the waves cover the row tiles a whole
  // number of times (ONE_RT), tile g = wv + NWV p at rt = g % RTV, ct = g / RTV
  // (one row tile per wave); otherwise row tiles wv + NWV q, every column.
  constexpr int NVT = RTV * CT;
  constexpr int NVP = (NVT + NWV - 1) / NWV;
  constexpr bool ONE_RT = (NWV % RTV) == 0;
  constexpr int NAR = ONE_RT ? 1 : RTV / NWV; // A row tiles held per wave
  using ST = SplitTile<E>;
  constexpr int LDS_ST = K + ST::PAD;
  constexpr int LDS_VN = M + ST::PAD;
  constexpr int KS = Mma<E>::KS;
  constexpr int NSK = K / KS;                 // k-steps over K
  constexpr int NSM = (M + KS - 1) / KS;      // k-steps over M
  constexpr bool PADM = (M % KS) != 0;
  constexpr bool FRB = FRM & 1, FRA = FRM & 2;
  static_assert(TPW >= 1 && (TPW % CT == 0 || CT % TPW == 0),
                "state tiles of a wave: whole rows, or a part of one row");
  static_assert(ONE_RT || RTV % NWV == 0, "Vn row tiles spread evenly over the waves");
  // S^T and Vn^T, split once by their writers
  __shared__ __attribute__((aligned(16))) typename ST::T s_st[ST::NPLANE * BV * LDS_ST];
  __shared__ __attribute__((aligned(16))) typename ST::T s_vn[ST::NPLANE * BV * LDS_VN];
  const ST sST{s_st, BV * LDS_ST}, sVn{s_vn, BV * LDS_VN};

  const int V = a.V, S = a.S, H = a.H;
  const int nvt = V / BV;
  int vt, bh;
  xcd_split(blockIdx.x, gridDim.x, nvt, bh, vt);
  const int h = bh % H, b = bh / H;
  const int v0 = vt * BV;
  const int lane = lane_id(), wv = wave_id();
  if (gated_out(a.gate, b)) return;

  // state tiles of this wave: g = wv * TPW + i, rt = g / CT, ct = g % CT
  f4 st[TPW];
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int g = wv * TPW + i, rt = g / CT, ct = g % CT;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = rt * 16 + acc_row(r), v = v0 + ct * 16 + acc_col();
      st[i][r] = a.init ? a.init[b * a.init_sb + h * a.init_sh + (long long)k * V + v] : 0.f;
    }
  }

  const float* Ab = a.A + (size_t)bh * S * M * K;
  const float* Bb = a.BT + (size_t)bh * S * K * M;
  const float* Ub = a.U + (size_t)bh * S * M * V;
  const float* Gb = a.gam + (size_t)bh * S * K;

  // Operands of one step, read a step ahead: they do not depend on the state.
  typedef typename Mma<E>::SFrag SF;
  constexpr int RA = OUT ? NAR : 1, RQ = OUT ? NSK : 1, RP = OUT ? NSM : 1;
  struct Ops {
    SF a[NAR][NSK];             // A rows of this wave's Vn tiles
    float u[NVP][4];            // U at the Vn tiles
    SF bt[TRT][NSM];            // BT rows of this wave's state tiles
    f4 g[TRT];                  // gam at the state rows (one 16-byte load)
    SF qg[RA][RQ];              // OUT: Qg rows of this wave's tiles
    SF aq[RA][RP];              // OUT: Aqk rows
  };
  // p-th Vn tile of this wave: valid, row tile, column tile, A row set
  auto vn_tile = [&](int p, int& rt, int& ct) -> bool {
    if (ONE_RT) {
      const int g = wv + NWV * p;
      rt = g % RTV;
      ct = g / RTV;
      return NVT % NWV == 0 || g < NVT;   // (a test the compiler cannot resolve would branch)
    }
    rt = wv + NWV * (p / CT);
    ct = p % CT;
    return true;
  };
  // The loads of step j's operands in the order in which the step needs them:
  // part 0, A; 1, Qg; 2, U; 3, Aqk; 4, BT and gam.
  auto load = [&](auto part_c, int j, Ops& o) {
    constexpr int PART = decltype(part_c)::value;
    if constexpr (PART < 4) {
      const SplitTile<E> Aj = split_at<E>(Ab + (size_t)j * M * K, M * K);
      const SplitTile<E> Qj = split_at<E>(a.Qg + ((size_t)bh * S + j) * M * K, M * K);
      const SplitTile<E> Pj = split_at<E>(a.Aqk + ((size_t)bh * S + j) * M * M, M * M);
      const float* Uj = Ub + (size_t)j * M * V;
#pragma unroll
      for (int p = 0; p < NVP; ++p) {
        int rt, ct;
        if (!vn_tile(p, rt, ct)) continue;
        const int q = ONE_RT ? 0 : p / CT;
        const int arow = (rt * 16 + (lane & 15)) * K + kofs<E>(lane);
        const int prow = (rt * 16 + (lane & 15)) * M + kofs<E>(lane);
        if (ONE_RT ? p == 0 : p % CT == 0) {
          if constexpr (PART == 0) {
#pragma unroll
            for (int s = 0; s < NSK; ++s) o.a[q][s] = Aj.get(FRA ? frag_at(rt, s, K) : arow + s * KS);
          }
          if constexpr (PART == 1 && OUT) {
#pragma unroll
            for (int s = 0; s < NSK; ++s) o.qg[q][s] = Qj.get(FRA ? frag_at(rt, s, K) : arow + s * KS);
          }
          if constexpr (PART == 3 && OUT) {
#pragma unroll
            for (int s = 0; s < NSM; ++s) o.aq[q][s] = Pj.get(FRA ? frag_at(rt, s, M) : prow + s * KS);
          }
        }
        if constexpr (PART == 2) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            o.u[p][r] = Uj[(size_t)(rt * 16 + acc_row(r)) * V + v0 + ct * 16 + acc_col()];
        }
      }
    } else {
      const SplitTile<E> Bj = split_at<E>(Bb + (size_t)j * K * M, K * M);
      const float* Gj = Gb + (size_t)j * K;
#pragma unroll
      for (int t = 0; t < TRT; ++t) {
        const int rt = (wv * TPW) / CT + t;
        const int brow = (rt * 16 + (lane & 15)) * M + kofs<E>(lane);
#pragma unroll
        for (int s = 0; s < NSM; ++s)
          o.bt[t][s] = FRB ? Bj.get(frag_at(rt, s, M))
                          : (!PADM || s * KS + kofs<E>(lane) < M) ? Bj.get(brow + s * KS)
                                                                  : Mma<E>::szero();
        o.g[t] = *reinterpret_cast<const f4*>(Gj + rt * 16 + acc_row(0));
      }
    }
    __builtin_amdgcn_sched_barrier(0);   // the loads stay where the step places them
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  using P2 = std::integral_constant<int, 2>;
  using P3 = std::integral_constant<int, 3>;
  using P4 = std::integral_constant<int, 4>;
  auto load_all = [&](int j, Ops& o) {
    load(P0{}, j, o);
    load(P1{}, j, o);
    load(P2{}, j, o);
    load(P3{}, j, o);
    load(P4{}, j, o);
  };

  // SM: the next step whose transposed state is due
  const int vk_step = a.vk_every > 1 ? a.vk_every : 1;
  int vk_next = SM ? (a.j0 + vk_step - 1) / vk_step * vk_step : 0;
  auto store_state = [&](int j) {
    // (SM: the mode is known, so no branch stands between a product and the
    // stores of its result)
    const bool by_chunk = SM == 0 ? a.state_mode == 0 : SM < 3;
    const size_t base = (by_chunk ? (size_t)bh * S + j
                                  : ((size_t)b * a.NG + j) * H + h) * K * V;
    if constexpr (SM != 0) {
      const bool due = a.st_vk && j == vk_next;
      if (j == vk_next) vk_next += vk_step;
      const auto rvk = buf(a.st_vk + base, due ? K * V * 4 : 0);
      const auto rkv = buf(a.st_kv + base, K * V * 4);
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const int g = wv * TPW + i, rt = g / CT, ct = g % CT;
        const int k0 = rt * 16 + acc_row(0), v = v0 + ct * 16 + acc_col();
        buf_st(rvk, (v * K + k0) * 4, st[i]);
        if constexpr (SM >= 2) {
#pragma unroll
          for (int r = 0; r < 4; ++r) buf_st(rkv, ((k0 + r) * V + v) * 4, st[i][r]);
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < TPW; ++i) {
      const int g = wv * TPW + i, rt = g / CT, ct = g % CT;
      const int k0 = rt * 16 + acc_row(0), vl = ct * 16 + acc_col(), v = v0 + vl;
      if (a.st_vk && (a.vk_every <= 1 || j % a.vk_every == 0))
        *reinterpret_cast<f4*>(a.st_vk + base + (size_t)v * K + k0) = st[i];
      if (a.st_kv) {
#pragma unroll
        for (int r = 0; r < 4; ++r) a.st_kv[base + (size_t)(k0 + r) * V + v] = st[i][r];
      }
    }
  };

  // A step's stores follow its products, while the next step's operand loads
  // (issued before them) are in flight: the vector memory pipe is in order,
  // so stores ahead of the loads would hold those up, and stores between the
  // products would hold the wave.
  f4 pvn[NVP], prd[OUT ? NVP : 1];
  auto flush = [&](int jj) {
    if constexpr (SM != 0) {
      const auto rvn = buf(a.vn + ((size_t)bh * S + jj) * M * V, M * V * 4);
      // rows of the chunk inside the sequence
      const int rows = min(M, a.T - jj * M);
      const auto rrd = buf(a.read0 + (((size_t)b * a.T + (size_t)jj * M) * H + h) * V,
                           (unsigned)(((rows - 1) * H + 1) * V * 4));
#pragma unroll
      for (int p = 0; p < NVP; ++p) {
        int rt, ct;
        if (!vn_tile(p, rt, ct)) continue;
        const int m0 = rt * 16 + acc_row(0), v = v0 + ct * 16 + acc_col();
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if constexpr (SM == 2) buf_st(rvn, ((m0 + r) * V + v) * 4, pvn[p][r]);
          if constexpr (OUT) buf_st(rrd, ((m0 + r) * H * V + v) * 4, prd[p][r]);
        }
      }
      return;
    }
#pragma unroll
    for (int p = 0; p < NVP; ++p) {
      int rt, ct;
      if (!vn_tile(p, rt, ct)) continue;
      const int m0 = rt * 16 + acc_row(0), vl = ct * 16 + acc_col();
      if (a.vnT)
        *reinterpret_cast<f4*>(a.vnT + (((size_t)bh * S + jj) * V + v0 + vl) * M + m0) = pvn[p];
      if (a.vn) {
        float* vp = a.vn + ((size_t)bh * S + jj) * M * V + (size_t)m0 * V + v0 + vl;
#pragma unroll
        for (int r = 0; r < 4; ++r) vp[(size_t)r * V] = pvn[p][r];
      }
      if constexpr (OUT) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = jj * M + rt * 16 + acc_row(r);
          if (t < a.T) a.read0[(((size_t)b * a.T + t) * H + h) * V + v0 + vl] = prd[p][r];
        }
      }
    }
  };

  // One step with its operands already loaded, placing the loads of step jn's
  // operands between its phases: a wave that issues them all at once (28 KB)
  // stands at the memory pipe, which takes 64 bytes per clock from the four
  // waves, before it starts on the step (B H = 64, T = 8192, K = 128: 606 ->
  // 555 us; B H = 16, T = 16384 without a backward: 629 -> 561 us, where a
  // timing copy without loads takes 200 us and the loads alone 300 us).
  auto step = [&](int j, const Ops& cur, int jn, Ops& nxt) {
      load(P0{}, jn, nxt);
      // ---- the state, transposed, to LDS
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const int g = wv * TPW + i, rt = g / CT, ct = g % CT;
        const int k0 = rt * 16 + acc_row(0), vl = ct * 16 + acc_col();
        sST.put4(vl * LDS_ST + k0, st[i]);
      }
      lds_barrier();

      // ---- Vn = U - A S (and, OUT, the read's Qg S on the same tiles)
      constexpr int CTV = ONE_RT ? NVP : CT;     // column tiles this wave's Vn tiles use
      // (16 pairs, or 32 in 16 columns, leave some waves without a Vn tile: the
      // read, kept unconditional, then takes the last column tile, unused)
      auto vn_ct = [&](int c) {
        if (!ONE_RT) return c;
        const int ct = (wv + NWV * c) / RTV;
        return NVT % NWV == 0 ? ct : min(ct, CT - 1);
      };
      f4 rd[OUT ? NVP : 1];
      {
        SF fb[CTV][NSK];
#pragma unroll
        for (int c = 0; c < CTV; ++c) {
          const int brow = (vn_ct(c) * 16 + (lane & 15)) * LDS_ST + kofs<E>(lane);
#pragma unroll
          for (int s = 0; s < NSK; ++s) fb[c][s] = sST.get(brow + s * KS);
        }
        load(P1{}, jn, nxt);
#pragma unroll
        for (int p = 0; p < NVP; ++p) {
          int rt, ct;
          if (vn_tile(p, rt, ct)) {
            const int c = ONE_RT ? p : p % CT;
            f4 acc = f4_zero();
            if constexpr (OUT) rd[p] = f4_zero();
#pragma unroll
            for (int s = 0; s < NSK; ++s) {
              acc = Mma<E>::mma(acc, cur.a[ONE_RT ? 0 : p / CT][s], fb[c][s]);
              if constexpr (OUT) rd[p] = Mma<E>::mma(rd[p], cur.qg[ONE_RT ? 0 : p / CT][s], fb[c][s]);
            }
            const int m0 = rt * 16 + acc_row(0), vl = ct * 16 + acc_col();
            f4 vn;
#pragma unroll
            for (int r = 0; r < 4; ++r) vn[r] = cur.u[p][r] - acc[r];
            sVn.put4(vl * LDS_VN + m0, vn);
            pvn[p] = vn;
          }
        }
      }
      load(P2{}, jn, nxt);
      lds_barrier();

      // ---- Vn^T of every column tile, once for the read and the state
      SF fv[CT][NSM];
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int brow = (c * 16 + (lane & 15)) * LDS_VN + kofs<E>(lane);
#pragma unroll
        for (int s = 0; s < NSM; ++s) {
          // M = 16 with 32-deep bf16 MFMAs: the upper half of the k range is zero
          const bool live = !PADM || (s * KS + kofs<E>(lane) < M);
          fv[c][s] = Mma<E>::szero();
          if (live) fv[c][s] = sVn.get(brow + s * KS);
        }
      }
      // ---- OUT: read0 = Qg S + Aqk Vn for the chunk's rows in the sequence
      if constexpr (OUT) {
        static_assert(!OUT || (ONE_RT && RTV == NWV), "one row tile per wave, column tile p");
#pragma unroll
        for (int p = 0; p < NVP; ++p) {
#pragma unroll
          for (int s = 0; s < NSM; ++s) rd[p] = Mma<E>::mma(rd[p], cur.aq[0][s], fv[p][s]);
          prd[p] = rd[p];
        }
        if constexpr (SM == 0) mfma_settle();   // its stores stand under branches
      }
      load(P3{}, jn, nxt);
      // ---- this step's stores (the state registers still hold the state
      // entering step j)
      store_state(j);
      flush(j);
      load(P4{}, jn, nxt);

      // ---- S <- diag(gam) S + BT Vn
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        // t and the column tile must be compile-time indices into registers
        constexpr bool WHOLE = TPW % CT == 0;
        const int t = WHOLE ? i / CT : 0;
#pragma unroll
        for (int r = 0; r < 4; ++r) st[i][r] *= cur.g[t][r];
        const int ct = WHOLE ? i % CT : (wv * TPW + i) % CT;
#pragma unroll
        for (int s = 0; s < NSM; ++s) {
          if constexpr (WHOLE) {
            st[i] = Mma<E>::mma(st[i], cur.bt[t][s], fv[i % CT][s]);
          } else {
            SF fb = fv[0][s];
#pragma unroll
            for (int c = 1; c < CT; ++c)
              if (ct == c) fb = fv[c][s];
            st[i] = Mma<E>::mma(st[i], cur.bt[t][s], fb);
          }
        }
      }
    mfma_settle();
    // no barrier needed here: the next writes to s_st do not alias s_vn, and
    // the next writes to s_vn follow the next step's barrier
  };

  // steps [j0, j1): the state registers start from init, the state entering
  // j0. Each step's operand loads are issued a step ahead, unconditionally (the
  // last step reloads its own, so that no branch guards them).
  const int j0 = a.j0, j1 = a.j1 > 0 ? a.j1 : S;
  // (128 pairs at K = 128 in 32 columns keep one set: two would not fit, and
  // with one 8 vector registers in bf16 and 52 in fp32 already go to the
  // accumulation registers; in 16 columns two sets leave 4 over. No scratch.)
  if constexpr (SM != 0 && !(K == 128 && M == 128 && BV == 32)) {
    Ops x, y;
    if (j1 > j0) load_all(j0, x);
    wait_global();
    int j = j0;
    for (; j + 1 < j1; j += 2) {
      step(j, x, j + 1, y);
      step(j + 1, y, j + 2 < j1 ? j + 2 : j + 1, x);
    }
    if (j < j1) step(j, x, j, y);
  } else {
    Ops nxt;
    if (j1 > j0) load_all(j0, nxt);
    for (int j = j0; j < j1; ++j) {
      const Ops cur = nxt;
      step(j, cur, j + 1 < j1 ? j + 1 : j, nxt);
    }
  }
  if (a.state_mode == 1 && j1 == S) {
    for (int j = S; j < a.NG; ++j) store_state(j);
  }
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int g = wv * TPW + i, rt = g / CT, ct = g % CT;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int k = rt * 16 + acc_row(r), v = v0 + ct * 16 + acc_col();
      a.fin[b * a.fin_sb + h * a.fin_sh + (long long)k * V + v] = st[i][r];
    }
  }
}


// Waves per workgroup: four, one per SIMD. Eight (two per SIMD) leave each
// wave half the registers, less than a step's operands read ahead need.
constexpr int SCAN_WAVES = 4;

// The outputs of a call (SM above). The buffer stores of read0 take a chunk's
// rows as byte offsets below 2^31.
static int scan_outputs(const ScanArgs& a) {
  if (a.gate.pos || a.vnT) return 0;
  if (a.read0) {
    if (a.state_mode != 0 || (long long)a.H * a.V * CH * 4 >= (1LL << 31)) return 0;
    return a.st_kv && a.vn ? 2 : !a.st_kv && !a.vn ? 1 : 0;
  }
  return a.state_mode == 1 && a.st_kv && !a.vn ? 3 : 0;
}

template <typename E, int K, int M, int BV, bool OUT, int FRM, int SM>
static hipError_t launch_scan_sm(const ScanArgs& a, hipStream_t st) {
  const unsigned grid = (unsigned)(a.B * a.H * (a.V / BV));
  hipLaunchKernelGGL((scan_fwd_kernel<E, K, M, BV, SCAN_WAVES, OUT, FRM, SM>), dim3(grid),
                     dim3(SCAN_WAVES * WAVE), 0, st, a);
  return hipGetLastError();
}

template <typename E, int K, int M, int BV, int FRM>
static hipError_t launch_scan_frm(const ScanArgs& a, int sm, hipStream_t st) {
  // level 0's read is formed only by the chunk-step (M == CH) kernels whose
  // operand groups share one layout (frag 0 or 3)
  if constexpr (M == CH && FRM != 1) {
    if (sm == 1) return launch_scan_sm<E, K, M, BV, true, FRM, 1>(a, st);
    if (sm == 2) return launch_scan_sm<E, K, M, BV, true, FRM, 2>(a, st);
    if constexpr (BV == SCAN_BV || FRM) {
      if (a.read0) return launch_scan_sm<E, K, M, BV, true, FRM, 0>(a, st);
    }
  }
  if (a.read0) return hipErrorInvalidValue;
  if constexpr (FRM != 3) {
    if (sm == 3) return launch_scan_sm<E, K, M, BV, false, FRM, 3>(a, st);
  }
  if constexpr (BV == SCAN_BV || FRM) return launch_scan_sm<E, K, M, BV, false, FRM, 0>(a, st);
  return hipErrorInvalidValue;
}

template <typename E, int K, int M, int BV>
static hipError_t launch_scan_bv(const ScanArgs& a, int sm, hipStream_t st) {
  constexpr bool BF = std::is_same<E, bf16>::value;
  if constexpr (BF && M == CH) {
    if (a.frag == 3) return launch_scan_frm<E, K, M, BV, 3>(a, sm, st);
  }
  if constexpr (BF && M % 32 == 0) {
    if (a.frag == 1) return launch_scan_frm<E, K, M, BV, 1>(a, sm, st);
  }
  if (a.frag) return hipErrorInvalidValue;
  return launch_scan_frm<E, K, M, BV, 0>(a, sm, st);
}

template <typename E, int K, int M>
static hipError_t launch_scan(const ScanArgs& a, hipStream_t st) {
  // Few (batch, head) pairs (a long sequence in a small batch): 16-column
  // slices, twice the workgroups with half the products per step each; a
  // step's operands are then read by twice as many workgroups, which costs
  // more than it saves once the grid fills the chip. The general outputs have
  // the narrow form where the operands are in fragment order: a decoded token
  // whose level takes 128 pairs, K = 128, one sequence of 16 heads, 47.7 -> 46.3
  // us (merge 34.0 -> 32.5).
  const int sm = scan_outputs(a);
  if ((sm || a.frag) && a.B * a.H * (a.V / SCAN_BV) <= SCAN_NARROW_GRID)
    return launch_scan_bv<E, K, M, 16>(a, sm, st);
  return launch_scan_bv<E, K, M, SCAN_BV>(a, sm, st);
}

hipError_t scan_fwd(const ScanArgs& a, int dtype, int K, hipStream_t st) {
  if (a.V % SCAN_BV != 0) return hipErrorInvalidValue;
#define NGDN_SC(E, KK, MM) \
  if (K == KK && a.M == MM) return launch_scan<E, KK, MM>(a, st);
#define NGDN_SC_K(E, KK) NGDN_SC(E, KK, 16) NGDN_SC(E, KK, 32) NGDN_SC(E, KK, 64) NGDN_SC(E, KK, 128)
  if (dtype == NGDN_BF16) {
    NGDN_SC_K(bf16, 64) NGDN_SC_K(bf16, 128)
  } else {
    NGDN_SC_K(float, 64) NGDN_SC_K(float, 128)
  }
#undef NGDN_SC_K
#undef NGDN_SC
  return hipErrorInvalidValue;
}

}  // namespace ngdn
