// Pair elimination, LU, n <= 64: the getrf + applyT split of the reference
// pair step (buildT BABD_BorderedCR.cc:856, applyT cc:917-982, the border
// update cc:1107-1154), with the right-hand columns on the matrix cores.  The
// augmented panel is the one of bcr_factor_generic.hip: R = 2n + nr rows
// [row jp; row j; border], columns [T = col j | col jp | col jpp | xb].
// Two launches per level, so that the pivot steps of a panel and the products
// each run with the registers and LDS they need.
//
//  A. pair_lu_t: the T panel [E_jp; D_j; C_j] (R x n), one wave per pair, in
//     registers: rows over lanes (row lane + 64 s), columns in 16-wide
//     register vectors; LAPACK partial pivoting among the first 2n rows (first
//     maximum), multiplier a * (1/pivot), fma updates -- the arithmetic of the
//     other LU kernels, so T, the pivots and C_j U^-1 agree with them bit for
//     bit.  The step loop is rolled within each 16-column block (column c
//     read and written through a uniform register index, in groups of four
//     steps that update the block's columns from the group's first on).  In
//     FP64 the trailing blocks take a block's 16 steps at once on the matrix
//     cores (trailing_update); in FP32 each step updates them (a lane read
//     and two FMAs per column: the way through LDS costs as much).  The
//     steps' chain at two waves per SIMD bounds it, VALU issue next (55 %
//     busy): N = 100000, n = 32 FP64, first level 909 -> 750 us with the
//     blocked update, 713 now (loads and stores alone are 0.4 ms).  Rows do
//     not move; each row is stored at its final position (T, C_j U^-1, perm),
//     and the positions themselves go to the unused tail of T (one byte per
//     row).  pair_lu_tw: the same by a wave per block, FP64 beyond n = 48 and
//     small FP32 launches beyond n = 32.
//  B. pair_rhs_mfma: the right-hand part X = [col jp | col jpp | xb], two
//     waves per pair, 16-column tiles, each inside one of the three column
//     blocks.  -L11 below its diagonal blocks, the inverses of those unit
//     lower blocks (forward substitution in LDS, one column per lane) and
//     -[L21; C_j U^-1] are A operands held in registers for all tiles of a
//     wave; a tile is one contiguous run of its source block, loaded one tile
//     ahead and staged in LDS with the rows at their final positions; then
//        U12_kb  = inv(L_kk) (X_kb - sum_{m<kb} L_km U12_m)
//                                           -> pivot rows: D_j', E_j', B_j'
//        X_rest' = X_rest - [L21; C_j U^-1] U12
//                                           -> reduced rows D_jp', E_jp', B_jp'
//     on v_mfma_f32_16x16x4f32 (FP32 factors) or v_mfma_f64_16x16x4f64 (FP64
//     factors), the results leaving through the tile's place in LDS as whole
//     runs.  The sum over k runs as 16-wide blocks, lane group g = lane / 16
//     taking k = 16 kb + kro(g, i) in the i-th MFMA of a block (kro: the row
//     the result layout puts in value i of group g, 4 g + i in FP32, g + 4 i
//     in FP64), so a block of U12 in the accumulator layout is the next
//     products' B operand as it stands.  Memory latency bounds it, so all
//     loads of a tile are issued before the stores of the one before (a wait
//     for loads behind stores waits for those: 1.62 -> 1.27 ms at N = 100000,
//     n = 32 FP64, first level), the operands live in registers instead of
//     LDS (more pairs per CU), and stores are whole runs (1.41 ms with
//     operands in LDS and stores by column; now 0.98 ms, 3.9 TB/s with T).
//     The right-hand part of a QR pair (pair_qr_rhs) is the same kernel with
//     other products: 16 reflectors at a time as I - V T V^T (dlarft), V in
//     LDS, x + V (-T^T (V^T x)) with the tile's rows in registers throughout.
//     The LDS a pair needs sets how many share a CU: N = 20000, n = 32 FP64,
//     first level 401 us.
// The right-hand results differ from the rank-1 kernels in rounding only
// (other summation order, the inverted diagonal blocks).  A pivot whose
// reciprocal overflows (a subnormal pivot) turns the finished T columns into
// NaN here, where the rank-1 kernels leave them; the factorization is
// unusable either way and the refinement reports it.
#include "bcr_launch.hh"
#include "bcr_batch_kernels.hh"
#include "bcr_mfma.hh"
#include "bcr_wave.hh"

namespace bcr {
namespace {

// the most border rows (nr) the matrix-core pair takes
constexpr int kNrB = 8;

// lane `who`'s value of v when K > cc, else 0: a scalar select on the
// v_readlane result (written out: the compiler would move the value to a
// VGPR and select there, two vector instructions instead of none)
template <int K>
__device__ __forceinline__ float rl_after(float v, int who, int cc) {
  int x = __builtin_amdgcn_readlane(__float_as_int(v), who);
  asm("s_cmp_lt_u32 %1, %2\n\ts_cselect_b32 %0, %0, 0" : "+s"(x) : "s"(cc), "n"(K) : "scc");
  return __int_as_float(x);
}
template <int K>
__device__ __forceinline__ double rl_after(double v, int who, int cc) {
  const long long b = __double_as_longlong(v);
  int lo = __builtin_amdgcn_readlane(int(b & 0xffffffff), who);
  int hi = __builtin_amdgcn_readlane(int(b >> 32), who);
  asm("s_cmp_lt_u32 %2, %3\n\ts_cselect_b32 %0, %0, 0\n\ts_cselect_b32 %1, %1, 0"
      : "+s"(lo), "+s"(hi) : "s"(cc), "n"(K) : "scc");
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// columns K.. 15 of one 16-column block of the row sets, those not after
// column cc of the block getting a zero pivot-row entry; the pivot row is in
// row set 0 or 1 (a third row set holds border rows only).  Columns before KM
// may lie at or before cc and are masked; the later ones always lie after it.
template <int K, int KM, int RS, int SP, typename TW>
__device__ __forceinline__ void update_after(V16<TW>& v0, V16<TW>& v1, V16<TW>& v2, bool sp, int who, int cc, TW lv0,
                                             TW lv1, TW lv2) {
  if constexpr (K < 16) {
    const TW x = SP == 2 ? (sp ? v1[K] : v0[K]) : SP ? v1[K] : v0[K];
    const TW u = K < KM ? rl_after<K>(x, who, cc) : wave::rl(x, who);
    v0[K] = fma(-lv0, u, v0[K]);
    v1[K] = fma(-lv1, u, v1[K]);
    if constexpr (RS > 2) v2[K] = fma(-lv2, u, v2[K]);
    update_after<K + 1, KM, RS, SP, TW>(v0, v1, v2, sp, who, cc, lv0, lv1, lv2);
  }
}

// ---- A: the T panel ---------------------------------------------------------------
// One pivot step of a 16-column block held by row (row sets 0 and 1 the 2n
// candidates, a third the border rows): cc the column in the block, c the
// step; v0[cc], v1[cc], v2[cc] become the final column, the block's columns
// from KS on are updated (those before KM masked).  Leaves the pivot lane, its
// row set and the multipliers for columns outside the block.  BRANCH: the
// pivot's row set, which is uniform, chosen by a branch instead of a select per
// entry; two FP64 blocks only (N = 100000, n = 32, first level 750 -> 730 us;
// with three blocks or row sets the compiler spills the two forms).
template <typename TW>
struct PanelRows {
  int pos0, pos1;      // positions of rows lane, lane + 64
  int myperm = 0;      // lane c: ipiv of step c
  bool zero_pivot = false;
};
template <typename TW>
struct PivotStep {
  int who;
  bool sp;
  TW l0, l1, l2;
};
template <int RS, bool ONE, bool BRANCH, int KS, int KM, typename TW>
__device__ __forceinline__ PivotStep<TW> panel_step(V16<TW>& v0, V16<TW>& v1, V16<TW>& v2, PanelRows<TW>& w, int c,
                                                    int cc, int n2, int lane) {
  const TW x0 = v0[cc], x1 = v1[cc];
  const TW x2 = RS > 2 ? v2[cc] : TW(0);   // border rows (row set 2)
  const bool c0 = lane < n2 && w.pos0 >= c;
  const bool c1 = !ONE && lane + 64 < n2 && w.pos1 >= c;
  unsigned h0, l0, h1, l1;
  wave::abs_key(x0, h0, l0);
  wave::abs_key(x1, h1, l1);
  // the better of this lane's two candidates (ties to the smaller position)
  const bool b1 = c1 & (!c0 | (h1 > h0) | ((h1 == h0) & ((l1 > l0) | ((l1 == l0) & (w.pos1 < w.pos0)))));
  bool zero;
  PivotStep<TW> o;
  o.who = wave::argmax_pos<(sizeof(TW) > 4)>(c0 | c1, b1 ? h1 : h0, b1 ? l1 : l0, b1 ? w.pos1 : w.pos0, lane, zero);
  const int P = __builtin_amdgcn_readlane(b1 ? w.pos1 : w.pos0, o.who);
  o.sp = !ONE && __builtin_amdgcn_readlane(int(b1), o.who) != 0;
  w.zero_pivot = w.zero_pivot || zero;
  w.myperm = lane == c ? P + 1 : w.myperm;
  // the pivot row moves to position c, the row at c to the pivot's old place
  w.pos0 = w.pos0 == c ? P : w.pos0 == P ? c : w.pos0;
  if constexpr (!ONE) w.pos1 = w.pos1 == c ? P : w.pos1 == P ? c : w.pos1;
  const TW pv = wave::rl(o.sp ? x1 : x0, o.who);
  const TW rinv = pv != TW(0) ? TW(1) / pv : TW(0);
  // rows below the pivot get the multiplier, the others keep column c
  // (border and padding rows hold positions r >= 2n > c: always below;
  // the padding rows are zero and never stored)
  const bool u0 = w.pos0 > c;
  const bool u1 = w.pos1 > c;
  const TW m0 = x0 * rinv, m1 = x1 * rinv;
  o.l0 = u0 ? m0 : TW(0);
  o.l1 = u1 ? m1 : TW(0);
  v0[cc] = u0 ? m0 : x0;
  v1[cc] = u1 ? m1 : x1;
  o.l2 = TW(0);
  if constexpr (RS > 2) {   // border (and zero padding) rows: never pivots, always updated
    o.l2 = x2 * rinv;
    v2[cc] = o.l2;
  }
  // columns KS .. 15 of the block (those before are never after c)
  if (BRANCH && !ONE) {
    if (o.sp) update_after<KS, KM, RS, 1, TW>(v0, v1, v2, o.sp, o.who, cc, o.l0, o.l1, o.l2);
    else update_after<KS, KM, RS, 0, TW>(v0, v1, v2, o.sp, o.who, cc, o.l0, o.l1, o.l2);
  } else {
    update_after<KS, KM, RS, ONE ? 0 : 2, TW>(v0, v1, v2, o.sp, o.who, cc, o.l0, o.l1, o.l2);
  }
  return o;
}

// Between the 16-column blocks the trailing columns take the block's 16 steps
// at once, on the matrix cores, through LDS (one 16-column buffer):
//   x   the block's multipliers by row (zero for a row from the step on at
//       which it became a pivot row), read as A operands; then each trailing
//       block by row (as the registers hold it) and by tile in turn
//   u   the pivot rows' entries of all trailing columns, solved in place with
//       the block's unit lower triangle lk, a column per lane
// v_mfma_*_16x16x4 forms c + a0 b0 + .. + a3 b3 as the chain of fused
// multiply-adds in that order (measured: equal to it in every bit), and the
// products run over k upwards, so every entry sees the operations of the
// rank-1 steps in their order.
constexpr bool panel_blocked(size_t elem) { return elem == 8; }

template <typename TW, int NB>
struct PanelLds {
  static constexpr int TILES = (2 * 16 * NB + kNrB + 15) / 16;
  // column stride: 16 columns' reads of neighbouring rows on different banks
  static constexpr int RLD = 16 * TILES + 2, ULD = 16 * (NB > 1 ? NB - 1 : 1) + 2;
  alignas(16) TW x[16 * RLD];
  alignas(16) TW u[16 * ULD];
  alignas(16) TW lk[16 * 16];
};

template <int B, int NB, int RS, typename TW>
__device__ __forceinline__ void trailing_update(V16<TW> (&V)[RS][NB], PanelLds<TW, NB>& sm, int pos0, int pos1, int n,
                                                int R, int lane) {
  constexpr int TILES = PanelLds<TW, NB>::TILES, RLD = PanelLds<TW, NB>::RLD, ULD = PanelLds<TW, NB>::ULD;
  const int g = lane >> 4, cl = lane & 15;
  // multipliers by row; the block's pivot rows to u and lk
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const int r = lane + 64 * s;
    const int p = s == 0 ? pos0 - 16 * B : s == 1 ? pos1 - 16 * B : 16;   // (border rows: no pivots)
    if (r < 16 * TILES) {
#pragma unroll
      for (int k = 0; k < 16; ++k) sm.x[k * RLD + r] = keep_if(V[s][B][k], k < p);
    }
    if (s < 2 && p >= 0 && p < 16) {
#pragma unroll
      for (int k = 0; k < 16; ++k) sm.lk[k * 16 + p] = V[s][B][k];
#pragma unroll
      for (int bb = B + 1; bb < NB; ++bb)
#pragma unroll
        for (int k = 0; k < 16; ++k) sm.u[p * ULD + 16 * (bb - B - 1) + k] = V[s][bb][k];
    }
  }
  lds_order();
  if (lane < 16 * (NB - 1 - B)) {
    TW y[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) y[p] = sm.u[p * ULD + lane];
#pragma unroll
    for (int k = 0; k < 15; ++k) {
#pragma unroll
      for (int p = k + 1; p < 16; ++p) y[p] = fma(-sm.lk[k * 16 + p], y[k], y[p]);
      __builtin_amdgcn_sched_barrier(0);   // (the reads of all columns at once would take every register)
    }
#pragma unroll
    for (int p = 1; p < 16; ++p) sm.u[p * ULD + lane] = y[p];
  }
  lds_order();
  // GS row sets at a time (all, or one where the registers hold no more):
  // their multipliers to registers, then their rows of each trailing block
  // through the place they leave
  constexpr int GS = NB >= 3 ? 1 : RS, GT = 4 * GS < TILES ? 4 * GS : TILES;
#pragma unroll
  for (int s0 = 0; s0 < RS; s0 += GS) {
    V4<TW> av[GT];
#pragma unroll
    for (int t = 0; t < GT; ++t)
      if (4 * s0 + t < TILES) {
#pragma unroll
        for (int i = 0; i < 4; ++i) av[t][i] = -sm.x[(g + 4 * i) * RLD + 64 * s0 + 16 * t + cl];
      }
    lds_order();
#pragma unroll
    for (int bb = B + 1; bb < NB; ++bb)
      if (16 * bb < n && 64 * s0 < R) {
#pragma unroll
        for (int s = s0; s < s0 + GS; ++s) {
          const int r = lane + 64 * s;
          if (r < 16 * TILES) {
#pragma unroll
            for (int k = 0; k < 16; ++k) sm.x[k * RLD + r] = V[s][bb][k];
          }
        }
        lds_order();
        V4<TW> u;
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = sm.u[(g + 4 * i) * ULD + 16 * (bb - B - 1) + cl];
#pragma unroll
        for (int t = 0; t < GT; ++t)
          if (4 * s0 + t < TILES && 64 * s0 + 16 * t < R) {
            TW* const blk = sm.x + cl * RLD + 64 * s0 + 16 * t;
            V4<TW> acc;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = blk[kro<TW>(g, i)];
#pragma unroll
            for (int i = 0; i < 4; ++i) acc = mfma1(av[t][i], u[i], acc);
#pragma unroll
            for (int i = 0; i < 4; ++i) blk[kro<TW>(g, i)] = acc[i];
          }
        lds_order();
#pragma unroll
        for (int s = s0; s < s0 + GS; ++s) {
          const int rr = min(lane + 64 * s, 16 * TILES - 1);
#pragma unroll
          for (int k = 0; k < 16; ++k) V[s][bb][k] = sm.x[k * RLD + rr];
        }
        lds_order();
      }
  }
}

template <typename TS, typename TW, int NB, int RS, int NRMAX>
__device__ __forceinline__ void pair_lu_t_body(FactorArgs<TS, TW> const& a, int p) {
  constexpr int NMAX = 16 * NB;
  static_assert(RS == 2 || RS == 3, "two or three row sets");
  static_assert(NMAX <= 64, "the 2n candidate rows lie in row sets 0 and 1");
  constexpr bool BLOCKED = panel_blocked(sizeof(TW));
  // first: border rows C_j and one zero row, NMAX values each
  constexpr int STAGE = (NRMAX + 1) * NMAX * int(sizeof(TW));
  using Lds = std::conditional_t<BLOCKED, PanelLds<TW, NB>, char[STAGE]>;
  static_assert(STAGE <= int(sizeof(Lds)), "the border rows fit the buffer");
  __shared__ __align__(16) Lds sm;
  TW* const stage = reinterpret_cast<TW*>(&sm);
  if (p >= a.npairs) return;
  const int lane = threadIdx.x & 63;
  const int n = a.n, nr = a.nr, n2 = 2 * n;
  const int R = n2 + nr;
  int j, jp, jpp;
  pair_of_uniform(a, p, j, jp, jpp);
  const size_t nn = size_t(n) * n, rn = size_t(nr) * n;
  const TW* pend_cur = a.Cpend + size_t(a.slot_cur) * (a.N + 1) * rn;
  const TW* pend_prv = a.Cpend + size_t(a.slot_cur ^ 1) * (a.N + 1) * rn;

  // the border rows C_j (+ pending C_j) first, coalesced, into LDS rows of
  // NMAX (row nr stays zero for the other lanes)
  for (int e = lane; e < (nr + 1) * NMAX; e += 64) stage[e] = TW(0);
  for (int e = lane; e < nr * n; e += 64) {   // C_j is nr x n, column-major
    const int col = e / nr, ri = e - col * nr;
    TW x = TW(a.sC[j * rn + e]);
    if (!a.first) x += pend_prv[j * rn + e] + pend_cur[j * rn + e];
    stage[ri * NMAX + col] = x;
  }
  V16<TW> V[RS][NB];
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const int r = lane + 64 * s;
    const bool top = r < n, mid = r >= n && r < n2, bord = r >= n2 && r < R;
    // rows of block jp: E_jp; rows of block j: D_j
    const TS* base = top ? a.sE + jp * nn + r : a.sD + j * nn + (mid ? r - n : 0);
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int k = 0; k < 16; ++k) {
        const int col = 16 * b + k, off = (col < n ? col : n - 1) * n;
        V[s][b][k] = keep_if(TW(base[off]), (top || mid) && col < n);
      }
    if (R > 64 * s && n2 < 64 * (s + 1)) {   // this row set holds border rows
      const TW* srow = stage + (bord ? r - n2 : nr) * NMAX;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int k = 0; k < 16; k += 4) {
          const V4<TW> c4 = *reinterpret_cast<const V4<TW>*>(srow + 16 * b + k);
          V[s][b][k] += c4.x;
          V[s][b][k + 1] += c4.y;
          V[s][b][k + 2] += c4.z;
          V[s][b][k + 3] += c4.w;
        }
    }
  }
  PanelRows<TW> rows{lane, lane + 64};
  // 2n <= 64: every pivot candidate sits in row set 0 (row set 1 holds
  // border rows only), and the pivot row's entries come from it unselected
  constexpr bool ONE = 2 * NMAX <= 64;
  // Steps in blocks of 16, each in GR groups of GS steps: step c of block b
  // reads and rewrites column c through a uniform register index
  // (s_set_gpr_idx) and updates the columns of blocks b.. with the pivot
  // row's entries; group g of block b updates its block's columns from
  // GS g + 1 on, those that may not lie after c getting a zero entry.  Each
  // group's loop stays rolled (one copy of a step per group; four groups: a
  // quarter of the masked in-block updates of one).
  constexpr int GR = 4, GS = 16 / GR;
  // step c of block b; the block's columns from KS on are updated, those
  // before KM masked
  auto step = [&](const int b, const int c, auto KS, auto KM) {
    const PivotStep<TW> o = panel_step<RS, ONE, BLOCKED && NB == 2, decltype(KS)::value, decltype(KM)::value, TW>(
        V[0][b], V[1][b], V[RS - 1][b], rows, c, c - 16 * b, n2, lane);
    if constexpr (!BLOCKED) {
#pragma unroll
      for (int bb = b + 1; bb < NB; ++bb)
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const TW u = wave::rl(o.sp ? V[1][bb][k] : V[0][bb][k], o.who);
          V[0][bb][k] = fma(-o.l0, u, V[0][bb][k]);
          V[1][bb][k] = fma(-o.l1, u, V[1][bb][k]);
          if constexpr (RS > 2) V[RS - 1][bb][k] = fma(-o.l2, u, V[RS - 1][bb][k]);
        }
    }
  };
  static_for<0, NB>([&](auto BK) {
    constexpr int b = decltype(BK)::value;
    static_for<0, GR>([&](auto G) {
      constexpr int g = decltype(G)::value;
      const int cend = min(16 * b + GS * g + GS, n);
      for (int c = 16 * b + GS * g; c < cend; ++c)
        step(b, c, std::integral_constant<int, GS * g + 1>{}, std::integral_constant<int, GS * g + GS>{});
    });
    if constexpr (BLOCKED && b + 1 < NB) {
      if (16 * (b + 1) < n) trailing_update<b, NB, RS, TW>(V, sm, rows.pos0, rows.pos1, n, R, lane);
    }
  });
  const int pos0 = rows.pos0, pos1 = rows.pos1;
  if (rows.zero_pivot && lane == 0) atomicOr(a.status, 1);
  // the selector's statistics of this panel (FP32 batches): |U_cc| min and
  // max, |U_rc| max over r <= c, as float bits (non-negative: ordered as
  // unsigned); the row at final position p < n holds U row p
  if (sizeof(TW) == 4 && a.pstat != nullptr) {
    unsigned dmin = 0xffffffffu, dmax = 0u, umax = 0u;
#pragma unroll
    for (int s = 0; s < (ONE ? 1 : 2); ++s) {
      const int q = lane + 64 * s < n2 ? (s == 0 ? pos0 : pos1) : n;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const int c = 16 * b + k;
          const unsigned bits = __float_as_uint(fabsf(float(V[s][b][k])));
          umax = max(umax, q <= c && c < n ? bits : 0u);
          if (q == c && c < n) {
            dmin = min(dmin, bits);
            dmax = max(dmax, bits);
          }
        }
    }
    dmin = wave::min_u32(dmin);
    dmax = wave::max_u32(dmax);
    umax = wave::max_u32(umax);
    if (lane == 0) {
      float* const o = a.pstat + 3 * size_t(j - 1);
      o[0] = __uint_as_float(dmin);
      o[1] = __uint_as_float(dmax);
      o[2] = __uint_as_float(umax);
    }
  }
  // T (2n x n, final row order) and C_j U^-1 to their blocks
  TW* Tj = a.Tm + size_t(j) * tsize(n);
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const int r = lane + 64 * s;
    const int q = r < n2 ? (s == 0 ? pos0 : pos1) : r;
    if (r < R) {
      TW* dst = q < n2 ? Tj + q : a.C + j * rn + (q - n2);
      const int stride = q < n2 ? n2 : nr;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int k = 0; k < 16; ++k)
          if (16 * b + k < n) dst[size_t(16 * b + k) * stride] = V[s][b][k];
    }
  }
  if (lane < n) a.perm[size_t(j) * n + lane] = rows.myperm;
  // the final position of every panel row, one byte each after the panel's
  // 2n^2 entries (the LU pair leaves that tail of T unused): kernel B reads
  // them instead of replaying the swap sequence
  uint8_t* const posb = reinterpret_cast<uint8_t*>(Tj + size_t(2) * n * n);
  if (lane < n2) posb[lane] = uint8_t(pos0);
  if (lane + 64 < n2) posb[lane + 64] = uint8_t(pos1);
}

// The same panel by NB waves, one per 16-column block.  Wave b holds block b as
// tiles in the accumulator layout until its turn; it then factors it by row and
// publishes multipliers, pivot triangle and row positions (two sets, by the
// parity of b), and the waves behind update their blocks from them while wave
// b + 1, done with its own, goes on.  One barrier per block, NB for each wave.
// A wave's tiles are dead before its rows come to life, so 64 FP64 columns
// take 168 registers and three waves share a SIMD; one wave needed 512 and
// spilled.  What is left is the chain of the steps.  Times of one level:
//                         one wave              a wave per block
//   FP64, n = 53          643 / 98 us           442 / 60 us     (4500 / 1 pairs)
//   FP64, n = 40          342 / 43 us           523 / 41 us     (10000 / 1)
//   FP64, n = 32          746 / 25 us           845 / 26 us     (50000 / 1)
//   FP32, n = 60          248, 90, 60 us        302, 65, 48 us  (5000, 625, 1)
//   FP32, n = 40          199, 53, 34 us        253, 47, 29 us  (10000, 1250, 1)
template <typename TW, int NB, int RS>
struct PanelWavesLds {
  static constexpr int TILES = (2 * 16 * NB + kNrB + 15) / 16, RLD = 16 * TILES + 2, ULD = 18;
  alignas(16) TW x[2][16 * RLD];        // multipliers by row (as in PanelLds::x)
  alignas(16) TW u[NB - 1][16 * ULD];   // waves 1 ..: the pivot rows of their blocks
  alignas(16) TW lk[2][16 * 16];
  uint8_t pos[2][128];
};

// BATCH: a launch takes the NB of its largest n, so 16 (NB - 1) < n holds for a
// single system only, and with it the first tile the border rows can lie in
// (every tile tried for a single system too: n = 53, 9001 rows 4255 -> 4284 us).
template <typename TS, typename TW, int NB, int RS, bool BATCH>
__device__ __forceinline__ void pair_lu_tw_body(FactorArgs<TS, TW> const& a, int p) {
  static_assert(NB >= 3, "one wave takes two blocks (times above)");
  using Lds = PanelWavesLds<TW, NB, RS>;
  constexpr int TILES = Lds::TILES, RLD = Lds::RLD, ULD = Lds::ULD;
  __shared__ Lds sm;
  if (p >= a.npairs) return;   // uniform over the workgroup
  const int lane = threadIdx.x & 63, g = lane >> 4, cl = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int n = a.n, nr = a.nr, n2 = 2 * n, R = n2 + nr;   // n <= 16 NB
  int j, jp, jpp;
  pair_of_uniform(a, p, j, jp, jpp);
  const size_t nn = size_t(n) * n, rn = size_t(nr) * n;
  TW* const Tj = a.Tm + size_t(j) * tsize(n);
  V16<TW> V[RS];
  {
    const TW* pend_cur = a.Cpend + size_t(a.slot_cur) * (a.N + 1) * rn + j * rn;
    const TW* pend_prv = a.Cpend + size_t(a.slot_cur ^ 1) * (a.N + 1) * rn + j * rn;
    const TS *const Ejp = a.sE + jp * nn, *const Dj = a.sD + j * nn, *const Cj = a.sC + j * rn;
    // this wave's block as tiles: rows 16 t + g + 4 i, column 16 w + cl
    const int col = 16 * w + cl;
    const unsigned coff = col < n ? unsigned(col) * unsigned(n) : 0;
    V4<TW> T[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = 16 * t + kro<TW>(g, i);
        // rows of block jp: E_jp; rows of block j: D_j; border rows below
        const TS* src = r < n ? Ejp + r : Dj + (r < n2 ? r - n : 0);
        T[t][i] = keep_if(TW(src[coff]), r < n2 && col < n);
      }
#pragma unroll
    for (int t = BATCH ? 0 : 2 * NB - 2; t < TILES; ++t)
      if (16 * t + 16 > n2 && 16 * t < R) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * t + kro<TW>(g, i);
          const bool ok = r >= n2 && r < R && col < n;
          const unsigned off = ok ? unsigned(r - n2) + unsigned(col) * unsigned(nr) : 0;
          TW v = TW(gload(Cj, off));
          if (!a.first) v += gload(pend_prv, off) + gload(pend_cur, off);
          T[t][i] += keep_if(v, ok);
        }
      }

    for (int b = 0; b < w; ++b) {
      __syncthreads();
      TW const* const x = sm.x[b & 1];
      TW const* const lk = sm.lk[b & 1];
      // the block's pivot rows of this wave's columns, solved with its unit
      // lower triangle, a column per lane
      TW* const u = sm.u[w - 1];
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        if (16 * t < n2) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const unsigned q = unsigned(sm.pos[b & 1][(16 * t + kro<TW>(g, i)) & 127]) - 16u * b;
            if (q < 16u && 16 * t + kro<TW>(g, i) < n2) u[q * ULD + cl] = T[t][i];
          }
        }
      lds_order();
      if (lane < 16) {
        TW y[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) y[q] = u[q * ULD + lane];
#pragma unroll
        for (int k = 0; k < 15; ++k) {
#pragma unroll
          for (int q = k + 1; q < 16; ++q) y[q] = fma(-lk[k * 16 + q], y[k], y[q]);
          __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int q = 1; q < 16; ++q) u[q * ULD + lane] = y[q];
      }
      lds_order();
      V4<TW> uv;
#pragma unroll
      for (int i = 0; i < 4; ++i) uv[i] = u[(4 * i + g) * ULD + cl];
#pragma unroll
      for (int t = 0; t < TILES; ++t)
        if (16 * t < R) {
          V4<TW> av;
#pragma unroll
          for (int i = 0; i < 4; ++i) av[i] = -x[(4 * i + g) * RLD + 16 * t + cl];
#pragma unroll
          for (int i = 0; i < 4; ++i) T[t] = mfma1(av[i], uv[i], T[t]);
        }
      lds_order();
    }

    // to the row layout through the place its multipliers will take (its last
    // readers have passed the barrier before)
    TW* const x = sm.x[w & 1];
#pragma unroll
    for (int t = 0; t < TILES; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) x[cl * RLD + 16 * t + kro<TW>(g, i)] = T[t][i];
    lds_order();
#pragma unroll
    for (int s = 0; s < RS; ++s) {
      const int r = lane + 64 * s;
      V[s] = V16<TW>(TW(0));
      if (r < 16 * TILES) {
#pragma unroll
        for (int k = 0; k < 16; ++k) V[s][k] = x[k * RLD + r];
      }
    }
  }
  PanelRows<TW> rows{lane, lane + 64};
  if (w > 0) {
    rows.pos0 = sm.pos[(w & 1) ^ 1][lane];
    rows.pos1 = sm.pos[(w & 1) ^ 1][lane + 64];
  }
  static_for<0, 4>([&](auto G) {
    constexpr int gs = 4 * decltype(G)::value;
    const int cend = min(16 * w + gs + 4, n);
    for (int c = 16 * w + gs; c < cend; ++c)
      panel_step<RS, false, false, gs + 1, gs + 4, TW>(V[0], V[1], V[RS - 1], rows, c, c - 16 * w, n2, lane);
  });
  if (rows.zero_pivot && lane == 0) atomicOr(a.status, 1);
  // columns 16 w .. of the interchanges
  if (lane >= 16 * w && lane < min(16 * w + 16, n)) a.perm[size_t(j) * n + lane] = rows.myperm;
  sm.pos[w & 1][lane] = uint8_t(rows.pos0);
  sm.pos[w & 1][lane + 64] = uint8_t(rows.pos1);
  if (w < NB - 1) {
    TW* const x = sm.x[w & 1];
    lds_order();
#pragma unroll
    for (int s = 0; s < RS; ++s) {
      const int r = lane + 64 * s;
      const int q = s == 0 ? rows.pos0 - 16 * w : s == 1 ? rows.pos1 - 16 * w : 16;   // (border rows: no pivots)
      if (r < 16 * TILES) {
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k * RLD + r] = keep_if(V[s][k], k < q);
      }
      if (s < 2 && q >= 0 && q < 16) {
#pragma unroll
        for (int k = 0; k < 16; ++k) sm.lk[w & 1][k * 16 + q] = V[s][k];
      }
    }
  }
  for (int b = w; b < NB; ++b) __syncthreads();

  // T (2n x n, final row order) and C_j U^-1 to their blocks
  const int pos0 = sm.pos[(NB - 1) & 1][lane], pos1 = sm.pos[(NB - 1) & 1][lane + 64];
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const int r = lane + 64 * s;
    const int q = r < n2 ? (s == 0 ? pos0 : pos1) : r;
    if (r < R) {
      TW* dst = q < n2 ? Tj + q : a.C + j * rn + (q - n2);
      const int stride = q < n2 ? n2 : nr;
#pragma unroll
      for (int k = 0; k < 16; ++k)
        if (16 * w + k < n) dst[size_t(16 * w + k) * stride] = V[s][k];
    }
  }
  uint8_t* const posb = reinterpret_cast<uint8_t*>(Tj + size_t(2) * n * n);
  if (w == 0) {
    if (lane < n2) posb[lane] = uint8_t(pos0);
    if (lane + 64 < n2) posb[lane + 64] = uint8_t(pos1);
  }
}

// ---- B: the right-hand part on the matrix cores ----------------------------------
// LDS of a pair: per wave one staged 16-column tile (rows by final position:
// top slots [0, NT), rest slots [NT, NT + 16 NRT): reduced rows, border rows;
// column stride XLD); the inverses of the unit lower diagonal blocks; the
// final position of every panel row.
template <typename TW, int NB, int NRT, int NW>
struct RhsLds {
  static constexpr int PAD = sizeof(TW) == 8 ? 2 : 4;   // columns' reads on different banks
  static constexpr int NT = 16 * NB, XLD = NT + 16 * NRT + PAD, DLD = 16 + PAD;
  alignas(16) TW x[NW][16 * XLD];
  alignas(16) TW inv[NB][16 * DLD];
  uint8_t pos[2 * NT];
};
// Of a QR pair: inv holds -T^T of each 16-column block (below), v the
// reflectors by column (rows [0, n) in slots [0, NT), rows [n, 2n) from slot
// NT on, zero elsewhere), cb the border rows of C_j R^-1 by column, as rows of
// the two 16-row rest tiles they can lie in.
template <typename TW, int NB, int NRT, int NW>
struct QrRhsLds : RhsLds<TW, NB, NRT, NW> {
  static constexpr int VLD = 2 * 16 * NB + RhsLds<TW, NB, NRT, NW>::PAD, CLD = 32 + RhsLds<TW, NB, NRT, NW>::PAD;
  alignas(16) TW v[16 * NB * VLD];
  alignas(16) TW cb[16 * NB * CLD];
};

template <typename TS, typename TW, int NB, int NRT, int NW, bool QR>
__device__ __forceinline__ void pair_rhs_body(FactorArgs<TS, TW> const& a, int p) {
  using Lds = std::conditional_t<QR, QrRhsLds<TW, NB, NRT, NW>, RhsLds<TW, NB, NRT, NW>>;
  constexpr int NT = Lds::NT, XLD = Lds::XLD, DLD = Lds::DLD, H = 4 * NB;   // H: values per lane of a tile
  __shared__ Lds sm;
  if (p >= a.npairs) return;   // uniform over the workgroup
  const int lane = threadIdx.x & 63, g = lane >> 4, cl = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int n = a.n, nr = a.nr, nx = a.nx, n2 = 2 * n;
  int j, jp, jpp;
  pair_of_uniform(a, p, j, jp, jpp);
  const size_t nn = size_t(n) * n, rn = size_t(nr) * n, bn = size_t(n) * nx;
  TW* pend_cur = a.Cpend + size_t(a.slot_cur) * (a.N + 1) * rn;
  TW* pend_prv = a.Cpend + size_t(a.slot_cur ^ 1) * (a.N + 1) * rn;
  const TW* Tj = a.Tm + size_t(j) * tsize(n);
  // the record's pointers, read once before the first store (a batched
  // kernel's record sits in memory: a field read after a store is fetched
  // again, a dependent memory round trip in front of the load it addresses)
  const TS *const sD = a.sD, *const sE = a.sE, *const sB = a.sB, *const sC = a.sC;
  TW *const Dm = a.D, *const Em = a.E, *const Bm = a.B, *const Cm = a.C, *const Fm = a.Fpart;
  const int first = a.first;
  // the final positions of this lane's two panel rows, stored by kernel A
  // after the panel's 2n^2 entries
  const uint8_t* const posb = reinterpret_cast<const uint8_t*>(Tj + size_t(2) * n * n);
  const uint8_t pb0 = posb[lane < n2 ? lane : 0], pb1 = posb[lane + 64 < n2 ? lane + 64 : 0];

  const int tA = (n + 15) / 16, tC = (nx + 15) / 16;
  const int ntiles = 2 * tA + tC;
  // a tile of D_jp or E_j is one run of 16 n values: element e = lane + 64 h
  // is row e % n of its column e / n (e < 1024: exact through the reciprocal)
  const unsigned rcp = (65536u + unsigned(n) - 1) / unsigned(n);
  const unsigned rcpr = nr > 0 ? (65536u + unsigned(nr) - 1) / unsigned(nr) : 0;

  // the run of tile t's part: D_jp (region 0), E_j (1), B_jp and B_j (2), and
  // with the first part the border rows' terms, nr values per column each:
  // C_jp and its pending slot (region 0), the pending C_jpp the tile adds to
  // (region 1).  Always issued before the stores of the tile before: a wait
  // for loads behind stores waits for those too.
  TS xs[H], cin[2];
  TW pin[2];
  auto load_tile = [&](int t, int part) {
    const int reg = t < tA ? 0 : t < 2 * tA ? 1 : 2;
    const int c0 = 16 * (reg == 0 ? t : reg == 1 ? t - tA : t - 2 * tA);
    const int width = min(16, (reg == 2 ? nx : n) - c0);
    const TS* src = (reg == 0 ? sD + jp * nn : reg == 1 ? sE + j * nn : sB + (part ? j : jp) * bn) + size_t(c0) * n;
#pragma unroll
    for (int h = 0; h < H; ++h) xs[h] = gload(src, unsigned(min(lane + 64 * h, width * n - 1)));
    if (part == 0 && nr > 0) {
      const size_t eb = size_t(c0) * nr;
      const TW* pe = reg == 0 ? pend_prv + jp * rn + eb : pend_cur + jpp * rn + eb;
      const TS* ce = sC + jp * rn + eb;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const unsigned e = reg < 2 ? min(lane + 64 * h, nr * width - 1) : 0;
        cin[h] = gload(reg < 2 ? ce : sC, e);
        pin[h] = gload(reg < 2 ? pe : a.Cpend, e);
      }
    }
  };
  if (w < ntiles) load_tile(w, 0);

  // LU: A operands, in registers for all tiles of the wave: -L below the
  // diagonal blocks, -[L21; C_j U^-1] (rows of T are final positions)
  V4<TW> lb[QR ? 1 : NB][NB], lr[QR ? 1 : NRT][NB];
  // (in flight over the inverses where the registers hold them beside those;
  // where they do not, the inverses stay in LDS too)
  constexpr bool LATE = NB >= 3;
  TW* const x = sm.x[w];
  auto clear_tile = [&] {   // (the padding slots stay zero)
#pragma unroll
    for (int h = 0; h < (16 * XLD + 63) / 64; ++h)
      if (lane + 64 * h < 16 * XLD) x[lane + 64 * h] = TW(0);
  };
  if constexpr (QR) {
    // the reflectors (unit lower trapezoid; R above it left out) by whole
    // columns, and the border rows of C_j R^-1
    clear_tile();
    for (int e = threadIdx.x; e < 16 * NB * Lds::CLD; e += 64 * NW) sm.cb[e] = TW(0);
    constexpr int CH = 4;   // columns in flight
    for (int k0 = w; k0 < 16 * NB; k0 += CH * NW) {
      TW t0[CH], t1[CH];
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const unsigned k = k0 + q * NW, kc = k < unsigned(n) ? k : 0;
        t0[q] = gload(Tj, kc * unsigned(n2) + unsigned(lane < n ? lane : 0));
        t1[q] = gload(Tj, kc * unsigned(n2) + unsigned(n + (lane < n ? lane : 0)));
      }
#pragma unroll
      for (int q = 0; q < CH; ++q) {
        const int k = k0 + q * NW;
        if (k < 16 * NB && lane < NT) {
          TW* const vk = sm.v + k * Lds::VLD;
          vk[lane] = k < n && lane <= k ? (lane == k ? TW(1) : TW(0)) : keep_if(t0[q], k < n && lane < n);
          vk[NT + lane] = keep_if(t1[q], k < n && lane < n);
        }
      }
    }
    __syncthreads();
    const int b0 = n & 15;   // the border rows' first row in their tiles
    for (int k = threadIdx.x; k < n; k += 64 * NW)
      for (int i = 0; i < nr; ++i) sm.cb[k * Lds::CLD + b0 + i] = -Cm[j * rn + size_t(k) * nr + i];
    // T of I - V T V^T = H_0 .. H_15 per 16-column block, from the products
    // V^T V (dlarft's recurrence T(0:c, c) = -tau_c T(0:c, 0:c) (V^T V)(0:c, c)),
    // row lane % 16 of block lane / 16 in a lane's registers; stored negated,
    // so that H^T x = x + V (-T^T (V^T x))
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (b % NW == w) {
        V4<TW> acc{TW(0), TW(0), TW(0), TW(0)};
#pragma unroll
        for (int t = b; t < 2 * NB; ++t) {
          const V4<TW> vt = ld4(sm.v + (16 * b + cl) * Lds::VLD + 16 * t, g);
          acc = mfma4<TW>(vt, vt, acc);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sm.inv[b][cl * DLD + kro<TW>(g, i)] = acc[i];
      }
    lds_order();
    if (lane < 16 * NB && (lane >> 4) % NW == w) {
      TW* const blk = sm.inv[lane >> 4];
      const int ri = lane & 15, c0 = lane & ~15;
      TW y[16];
#pragma unroll
      for (int c = 0; c < 16; ++c) {
        TW t0 = TW(0), t1 = TW(0);
#pragma unroll
        for (int k = 0; k < c; k += 2) {
          const V2<TW> g2 = *reinterpret_cast<const V2<TW>*>(blk + c * DLD + k);
          t0 = fma(g2.x, y[k], t0);
          if (k + 1 < c) t1 = fma(g2.y, y[k + 1], t1);
        }
        const TW tau = keep_if(gload(Tj, unsigned(n2) * unsigned(n) + unsigned(c0 + c < n ? c0 + c : 0)), c0 + c < n);
        y[c] = ri == c ? tau : ri < c ? -tau * (t0 + t1) : TW(0);
        if (c % 4 == 3) __builtin_amdgcn_sched_barrier(0);
      }
      lds_order();
#pragma unroll
      for (int c = 0; c < 16; ++c) blk[c * DLD + ri] = -y[c];
    }
    __syncthreads();   // V, T and the border rows in place
  } else {
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
#pragma unroll
      for (int m = 0; m <= kb; ++m) {
        if (m == kb && kb % NW != w) continue;   // diagonal blocks: this wave's only
        const int r = 16 * kb + cl;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = 16 * m + kro<TW>(g, i);
          const TW v = gload(Tj, (r < n ? r : 0) + unsigned(c < n ? c : 0) * unsigned(n2));
          const bool ok = r < n && c < n && (m < kb || c < r);
          lb[kb][m][i] = keep_if(m < kb ? -v : v, ok);
        }
      }
    auto load_rest = [&] {
#pragma unroll
      for (int rt = 0; rt < NRT; ++rt) {
        const int q = 16 * rt + cl;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int c = 16 * kb + kro<TW>(g, i);
            const TW v = gload(Tj, unsigned(n + (q < n ? q : 0)) + unsigned(c < n ? c : 0) * unsigned(n2));
            lr[rt][kb][i] = keep_if(-v, q < n && c < n);
          }
        if (16 * rt + 16 > n && 16 * rt < n + nr) {   // border rows of C_j U^-1
          const TW* const Cj = Cm + j * rn;
          const bool bord = q >= n && q < n + nr;
#pragma unroll
          for (int kb = 0; kb < NB; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int c = 16 * kb + kro<TW>(g, i);
              const TW v = gload(Cj, unsigned(bord ? q - n : 0) + unsigned(c < n ? c : 0) * unsigned(nr));
              lr[rt][kb][i] += keep_if(-v, bord && c < n);
            }
        }
      }
    };
    if (!LATE) load_rest();
    // this wave's diagonal blocks, row-major, then their inverses in place:
    // column lane % 16 of block lane / 16 by forward substitution; rows beyond
    // n are zero, their inverse rows identity
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
      if (kb % NW == w) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sm.inv[kb][cl * DLD + kro<TW>(g, i)] = lb[kb][kb][i];
      }
    if (w == 0) {
      if (lane < n2) sm.pos[lane] = pb0;
      if (lane + 64 < n2) sm.pos[lane + 64] = pb1;
    }
    clear_tile();
    lds_order();
    if (lane < 16 * NB && (lane >> 4) % NW == w) {
      TW* const blk = sm.inv[lane >> 4];
      const int jj = lane & 15;
      TW y[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) y[i] = TW(0);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const TW* li = blk + i * DLD;
        TW t0 = TW(0), t1 = TW(0);
#pragma unroll
        for (int k = 0; k < i; k += 2) {
          const V2<TW> l2 = *reinterpret_cast<const V2<TW>*>(li + k);
          // (entries 4m, 4m + 2 and 4m + 1, 4m + 3 in two chains)
          t0 = fma(l2.x, y[k], t0);
          t1 = fma(l2.y, y[k + 1], t1);
        }
        y[i] = jj == i ? TW(1) : -(t0 + t1);
        if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);   // (not all rows' reads at once)
      }
      // every lane has read its block's rows (reads precede these writes in this wave)
      lds_order();
#pragma unroll
      for (int i = 0; i < 16; ++i) blk[i * DLD + jj] = y[i];
    }
    __syncthreads();   // the inverses and the row positions in place
    if (LATE) load_rest();
  }
  auto inverse = [&](int kb) { return ld4(&sm.inv[kb][cl * DLD], g); };
  if constexpr (!LATE && !QR) {
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) lb[kb][kb] = inverse(kb);
  }
  // where element h of a run goes: as row of block jp (low half), of block j
  unsigned slot[H];
#pragma unroll
  for (int h = 0; h < H; ++h) {
    const unsigned e = lane + 64 * h, col = (e * rcp) >> 16, row = min(e - col * n, unsigned(n) - 1);
    const unsigned q0 = QR ? row : sm.pos[row], q1 = QR ? n + row : sm.pos[n + row];
    slot[h] = (col * XLD + (q0 < unsigned(n) ? q0 : NT + q0 - n)) | (col * XLD + (q1 < unsigned(n) ? q1 : NT + q1 - n)) << 16;
  }

  for (int t = w; t < ntiles; t += NW) {
    const int reg = t < tA ? 0 : t < 2 * tA ? 1 : 2;
    const int c0 = 16 * (reg == 0 ? t : reg == 1 ? t - tA : t - 2 * tA);
    const int width = min(16, (reg == 2 ? nx : n) - c0);
    const int cnt = width * n;
    const int m = nr * width;
    const size_t eb = size_t(c0) * nr;
    // (at the first level nothing is pending in C_jp's slot, and it is clear)
    TW padd[2] = {TW(0), TW(0)};
    // element h of a run to its slot, the other block's rows zero
    auto stage = [&](bool hi, bool clear) {
#pragma unroll
      for (int h = 0; h < H; ++h)
        if (lane + 64 * h < 16 * n) {
          const unsigned s0 = slot[h] & 0xffffu, s1 = slot[h] >> 16;
          x[hi ? s1 : s0] = TW(xs[h]);
          if (clear) x[hi ? s0 : s1] = TW(0);
        }
    };
    stage(reg == 1, reg < 2);
    if (m > 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const unsigned e = lane + 64 * h, cc = (e * rcpr) >> 16;
        if (e < unsigned(m)) {
          x[cc * XLD + NT + n + (e - cc * nr)] = reg == 0 ? (first ? TW(cin[h]) : TW(cin[h]) + pin[h]) : TW(0);
          padd[h] = pin[h];
          if (reg == 0 && !first) pend_prv[jp * rn + eb + e] = TW(0);   // read once: clear for reuse
        }
      }
    }
    // the next run's loads fly over this tile's work
    if (reg == 2) {   // B_j after B_jp
      load_tile(t, 1);
      stage(true, false);
    }
    if (t + NW < ntiles) load_tile(t + NW, 0);
    lds_order();
    const TW* const xc = x + cl * XLD;
    constexpr bool APART = NB == 4 && sizeof(TW) == 8;
    V4<TW> u[NB];
    if constexpr (QR) {
      // H^T x = x + V (-T^T (V^T x)), a block of 16 reflectors at a time, the
      // tile's rows in registers in the B operand layout throughout
      V4<TW> z[NRT];
#pragma unroll
      for (int t = 0; t < NB; ++t) u[t] = ld4(xc + 16 * t, g);
#pragma unroll
      for (int t = 0; t < NRT; ++t) z[t] = ld4(xc + NT + 16 * t, g);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        // V^T x with a chain per row tile, and V y summed by itself before it
        // meets x: fewer roundings at the size of the result than one
        // reflector at a time has (QR, n = 64 FP64: error of the solution
        // 1.70e-15 in one chain through x, 1.41e-15 so, 1.54e-15 by single reflectors)
        const V4<TW> zero{TW(0), TW(0), TW(0), TW(0)};
        V4<TW> acc[2 * NB];
#pragma unroll
        for (int t = 0; t < 2 * NB; ++t) acc[t] = zero;
#pragma unroll
        for (int t = 0; t < NB; ++t) {
          if (t >= b) acc[t] = mfma4<TW>(ld4(sm.v + (16 * b + cl) * Lds::VLD + 16 * t, g), u[t], acc[t]);
          acc[NB + t] = mfma4<TW>(ld4(sm.v + (16 * b + cl) * Lds::VLD + NT + 16 * t, g), z[t], acc[NB + t]);
        }
#pragma unroll
        for (int t = 0; t < NB; ++t) acc[t] += acc[NB + t];
#pragma unroll
        for (int t = 1; t < NB; ++t) acc[0] += acc[t];
        const V4<TW> y = mfma4<TW>(ld4(&sm.inv[b][cl * DLD], g), acc[0], zero);
#pragma unroll
        for (int t = 0; t < 2 * NB; ++t) acc[t] = zero;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const TW* const vk = sm.v + (16 * b + kro<TW>(g, i)) * Lds::VLD + cl;
#pragma unroll
          for (int t = 0; t < NB; ++t) {
            if (t >= b) acc[t] = mfma1(vk[16 * t], y[i], acc[t]);
            acc[NB + t] = mfma1(vk[NT + 16 * t], y[i], acc[NB + t]);
          }
        }
#pragma unroll
        for (int t = 0; t < NB; ++t) {
          if (t >= b) u[t] += acc[t];
          z[t] += acc[NB + t];
        }
      }
      // the border rows lose the final top rows
#pragma unroll
      for (int t = 0; t < NRT; ++t) {
        const int o = 16 * t + 16 > n && 16 * t < n + nr ? 16 * (t - n / 16) : -1;
        if (o >= 0) {
#pragma unroll
          for (int kb = 0; kb < NB; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) z[t] = mfma1(sm.cb[(16 * kb + kro<TW>(g, i)) * Lds::CLD + o + cl], u[kb][i], z[t]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int q = 16 * t + kro<TW>(g, i);
          x[cl * XLD + NT + q] = q < n + nr ? z[t][i] : TW(0);
        }
      }
    } else {
      // U12 = L11^-1 X_top by 16-row blocks: u_kb = inv(L_kk) (X_kb - sum_{m<kb}
      // L_km u_m).  A block of U12 in the accumulator layout is the B operand
      // layout of the next products as it stands.
#pragma unroll
      for (int kb = 0; kb < NB; ++kb) {
        V4<TW> acc = APART ? V4<TW>{TW(0), TW(0), TW(0), TW(0)} : ld4(xc + 16 * kb, g);
#pragma unroll
        for (int mb = 0; mb < kb; ++mb) acc = mfma4<TW>(lb[kb][mb], u[mb], acc);
        if (APART) acc += ld4(xc + 16 * kb, g);
        u[kb] = mfma4<TW>(LATE ? inverse(kb) : lb[kb][kb], acc, V4<TW>{TW(0), TW(0), TW(0), TW(0)});
      }
      // X_rest' = X_rest - [L21; C_j U^-1] U12, ZT tiles' chains side by side,
      // back to their slots
      // (APART: products of up to 64 terms summed by themselves before they
      // meet x, which outweighs the roundings the inverted blocks add)
      constexpr int ZT = NB == 3 && sizeof(TW) == 8 ? 2 : NRT;
#pragma unroll
      for (int r0 = 0; r0 < NRT; r0 += ZT) {
        V4<TW> z[ZT];
#pragma unroll
        for (int rt = 0; rt < ZT; ++rt)
          if (r0 + rt < NRT) z[rt] = APART ? V4<TW>{TW(0), TW(0), TW(0), TW(0)} : ld4(xc + NT + 16 * (r0 + rt), g);
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int rt = 0; rt < ZT; ++rt)
              if (r0 + rt < NRT) z[rt] = mfma1(lr[r0 + rt < NRT ? r0 + rt : 0][kb][i], u[kb][i], z[rt]);
        if (APART) {
#pragma unroll
          for (int rt = 0; rt < ZT; ++rt)
            if (r0 + rt < NRT) z[rt] += ld4(xc + NT + 16 * (r0 + rt), g);
        }
#pragma unroll
        for (int rt = 0; rt < ZT; ++rt)
          if (r0 + rt < NRT) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int q = 16 * (r0 + rt) + kro<TW>(g, i);
              x[cl * XLD + NT + q] = q < n + nr ? z[rt][i] : TW(0);
            }
          }
        if (ZT < NRT) __builtin_amdgcn_sched_barrier(0);
      }
    }
    // pivot rows -> block j, reduced rows -> block jp, through the tile's
    // place in LDS as whole runs
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = 16 * kb + kro<TW>(g, i);
        x[cl * XLD + q] = q < n ? u[kb][i] : TW(0);
      }
    lds_order();
    TW* const blk = (reg == 0 ? Dm : reg == 1 ? Em : Bm) + size_t(c0) * n;
    const size_t bsz = reg == 2 ? bn : nn;
    TW *const dj = blk + size_t(j) * bsz, *const djp = blk + size_t(jp) * bsz;
#pragma unroll
    for (int h = 0; h < H; ++h) {
      const unsigned e = lane + 64 * h, o = e + ((e * rcp) >> 16) * unsigned(XLD - n);
      if (e < unsigned(cnt)) {
        dj[e] = x[o];
        djp[e] = x[o + NT];
      }
    }
    // border rows: C_jp' (region 0), pending C_jpp += (region 1), F partial (region 2)
    TW* const bdst = reg == 0 ? Cm + jp * rn + eb : reg == 1 ? pend_cur + jpp * rn + eb
                                                              : Fm + size_t(j) * nr * nx + eb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned e = lane + 64 * h, cc = (e * rcpr) >> 16;
      if (e < unsigned(m)) {
        const TW v = x[cc * XLD + NT + n + (e - cc * nr)];
        bdst[e] = reg == 1 ? padd[h] + v : v;
      }
    }
    lds_order();
  }
}

// waves per SIMD the panel's registers have to leave room for
constexpr int panel_waves(int nb, size_t elem) { return elem == 8 && nb == 3 ? 2 : 1; }

template <typename TS, typename TW, int NB, int RS, int NRMAX>
__global__ void __launch_bounds__(64, panel_waves(NB, sizeof(TW))) pair_lu_t_kernel(FactorArgs<TS, TW> a) {
  pair_lu_t_body<TS, TW, NB, RS, NRMAX>(a, blockIdx.x);
}
template <typename TS, typename TW, int NB, int RS, int NRMAX>
__global__ void __launch_bounds__(64, panel_waves(NB, sizeof(TW))) pair_lu_t_batched(BatchTable<FactorArgs<TS, TW>> t) {
  const int e = t.entry[blockIdx.x];
  pair_lu_t_body<TS, TW, NB, RS, NRMAX>(t.args[e], int(blockIdx.x) - t.first[e]);
}
// The panel by waves: in FP64 for n > 48; in FP32 (where one wave's registers
// hold the panel, and fewer instructions fill a large launch better) for n > 32
// and at most kWavesPairs pairs.  Both sides' times stand at pair_lu_tw_body.
constexpr bool panel_by_waves_always(int nb, size_t elem) { return nb >= 4 && elem == 8; }
constexpr bool panel_by_waves_few(int nb, size_t elem) { return nb >= 3 && elem == 4; }
constexpr int kWavesPairs = 1024;

template <typename TS, typename TW, int NB, int RS>
__global__ void __launch_bounds__(64 * NB, 3) pair_lu_tw_kernel(FactorArgs<TS, TW> a) {
  pair_lu_tw_body<TS, TW, NB, RS, false>(a, blockIdx.x);
}
template <typename TS, typename TW, int NB, int RS>
__global__ void __launch_bounds__(64 * NB, 3) pair_lu_tw_batched(BatchTable<FactorArgs<TS, TW>> t) {
  const int e = t.entry[blockIdx.x];
  pair_lu_tw_body<TS, TW, NB, RS, true>(t.args[e], int(blockIdx.x) - t.first[e]);
}
constexpr int rhs_waves(int nb, size_t elem) { return elem == 8 ? (nb <= 3 ? 2 : 1) : nb <= 2 ? 4 : nb == 3 ? 3 : 2; }

template <typename TS, typename TW, int NB, int NRT, int NW>
__global__ void __launch_bounds__(64 * NW, rhs_waves(NB, sizeof(TW))) pair_rhs_mfma_kernel(FactorArgs<TS, TW> a) {
  pair_rhs_body<TS, TW, NB, NRT, NW, false>(a, blockIdx.x);
}
template <typename TS, typename TW, int NB, int NRT, int NW>
__global__ void __launch_bounds__(64 * NW, rhs_waves(NB, sizeof(TW))) pair_rhs_mfma_batched(BatchTable<FactorArgs<TS, TW>> t) {
  const int e = t.entry[blockIdx.x];
  pair_rhs_body<TS, TW, NB, NRT, NW, false>(t.args[e], int(blockIdx.x) - t.first[e]);
}

constexpr int qr_rhs_waves(int nb, size_t elem) { return elem == 8 ? (nb <= 3 ? 2 : 1) : nb <= 2 ? 4 : nb == 3 ? 3 : 2; }
template <typename TS, typename TW, int NB, int NRT, int NW>
__global__ void __launch_bounds__(64 * NW, qr_rhs_waves(NB, sizeof(TW))) pair_qr_rhs_kernel(FactorArgs<TS, TW> a) {
  pair_rhs_body<TS, TW, NB, NRT, NW, true>(a, blockIdx.x);
}
template <typename TS, typename TW, int NB, int NRT, int NW>
__global__ void __launch_bounds__(64 * NW, qr_rhs_waves(NB, sizeof(TW))) pair_qr_rhs_batched(BatchTable<FactorArgs<TS, TW>> t) {
  const int e = t.entry[blockIdx.x];
  pair_rhs_body<TS, TW, NB, NRT, NW, true>(t.args[e], int(blockIdx.x) - t.first[e]);
}

// Waves per pair in the right-hand kernel: two (each holds the operands of L,
// and more waves load them more often: n = 53, 4500 pairs 598 us with two, 874
// with four), four where a launch of at most one pair per CU leaves SIMDs idle
// (one pair, FP64: n = 32 15 -> 12 us, n = 40 28 -> 19, n = 53 53 -> 40).
constexpr int kRhsWaves = 2, kRhsWavesFew = 4;
constexpr int kFewPairs = 256;

// shapes: 1: n <= 32, n + nr <= 48 (two 16-column blocks); 2: n <= 48,
// n + nr <= 64 (three); 3: n <= 64, n + nr <= 80 (four, and a third row set
// for the border rows beyond row 128); all nr <= 8, nx <= 16; 0: not covered
int mfma_variant(int n, int nr, int nx) {
  if (n < 1 || nr > kNrB || nx > 16) return 0;
  if (n <= 32 && n + nr <= 48) return 1;
  if (n <= 48 && n + nr <= 64) return 2;
  if (n <= 64 && n + nr <= 80) return 3;
  return 0;
}

}  // namespace

bool pair_lu_mfma_fits(int n, int nr, int nx) { return mfma_variant(n, nr, nx) != 0; }

namespace {
// the A and B launches of shape variant V
template <int V, typename TS, typename TW>
void launch_pair(FactorArgs<TS, TW> const& a, hipStream_t st) {
  constexpr int NB = V + 1, RS = V == 3 ? 3 : 2, NRT = V + 2;   // NRT: tiles of the n + nr rest rows
  const dim3 pairs(a.npairs);
  bool by_waves = panel_by_waves_always(NB, sizeof(TW));
  if constexpr (panel_by_waves_few(NB, sizeof(TW))) by_waves = a.npairs <= kWavesPairs && a.pstat == nullptr;
  if constexpr (panel_by_waves_always(NB, sizeof(TW)) || panel_by_waves_few(NB, sizeof(TW))) {
    if (by_waves) hipLaunchKernelGGL((pair_lu_tw_kernel<TS, TW, NB, RS>), pairs, dim3(64 * NB), 0, st, a);
  }
  if constexpr (!panel_by_waves_always(NB, sizeof(TW))) {
    if (!by_waves) hipLaunchKernelGGL((pair_lu_t_kernel<TS, TW, NB, RS, kNrB>), pairs, dim3(64), 0, st, a);
  }
  if (a.npairs <= kFewPairs) hipLaunchKernelGGL((pair_rhs_mfma_kernel<TS, TW, NB, NRT, kRhsWavesFew>), pairs, dim3(64 * kRhsWavesFew), 0, st, a);
  else hipLaunchKernelGGL((pair_rhs_mfma_kernel<TS, TW, NB, NRT, kRhsWaves>), pairs, dim3(64 * kRhsWaves), 0, st, a);
}
template <int V, typename TS, typename TW>
void launch_pair_batched(BatchTable<FactorArgs<TS, TW>> const& t, int nblocks, hipStream_t st) {
  constexpr int NB = V + 1, RS = V == 3 ? 3 : 2, NRT = V + 2;   // NRT: tiles of the n + nr rest rows
  const dim3 pairs(nblocks);
  // (FP32 batches: one wave, which also leaves the selector's statistics)
  if constexpr (panel_by_waves_always(NB, sizeof(TW)))
    hipLaunchKernelGGL((pair_lu_tw_batched<TS, TW, NB, RS>), pairs, dim3(64 * NB), 0, st, t);
  else
    hipLaunchKernelGGL((pair_lu_t_batched<TS, TW, NB, RS, kNrB>), pairs, dim3(64), 0, st, t);
  // (four waves may wait here for room behind the other stream's workgroups,
  // but large batches are level with two: 1024 uneven systems FP64 44.0 / 43.8 ms,
  // FP32 32.6 / 32.8, half of them nearly singular 42.5 / 42.5; and one to eight
  // systems of n > 32 take 5-7 % less: 8 of n = 49 .. 64 1.65 / 1.77 ms)
  if (nblocks <= kFewPairs) hipLaunchKernelGGL((pair_rhs_mfma_batched<TS, TW, NB, NRT, kRhsWavesFew>), pairs, dim3(64 * kRhsWavesFew), 0, st, t);
  else hipLaunchKernelGGL((pair_rhs_mfma_batched<TS, TW, NB, NRT, kRhsWaves>), pairs, dim3(64 * kRhsWaves), 0, st, t);
}
}  // namespace

template <typename TS, typename TW>
bool launch_pair_lu_mfma(FactorArgs<TS, TW> const& a, hipStream_t st, hipError_t* err) {
  switch (mfma_variant(a.n, a.nr, a.nx)) {
    case 1: launch_pair<1>(a, st); break;
    case 2: launch_pair<2>(a, st); break;
    case 3: launch_pair<3>(a, st); break;
    default:
      return false;
  }
  *err = hipGetLastError();
  return true;
}

template <typename TS, typename TW>
bool launch_pair_lu_mfma_batched(BatchTable<FactorArgs<TS, TW>> const& t, int nblocks, int n, int nx, int nr,
                                 hipStream_t st, hipError_t* err) {
  switch (mfma_variant(n, nr, nx)) {
    case 1: launch_pair_batched<1>(t, nblocks, st); break;
    case 2: launch_pair_batched<2>(t, nblocks, st); break;
    case 3: launch_pair_batched<3>(t, nblocks, st); break;
    default:
      return false;
  }
  *err = hipGetLastError();
  return true;
}

template <typename TS, typename TW>
void launch_pair_qr_rhs(FactorArgs<TS, TW> const& a, hipStream_t st) {
  const dim3 g(a.npairs);
  // (four waves as in launch_pair: FP64 levels of a few pairs 22 -> 17 us at
  // n = 32, 39 -> 26 at n = 40; beyond n = 48 V leaves the LDS for two tiles)
  const bool few = a.npairs <= kFewPairs;
  switch (mfma_variant(a.n, a.nr, a.nx)) {
    case 1:
      if (few) hipLaunchKernelGGL((pair_qr_rhs_kernel<TS, TW, 2, 3, 4>), g, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((pair_qr_rhs_kernel<TS, TW, 2, 3, 2>), g, dim3(128), 0, st, a);
      break;
    case 2:
      if (few) hipLaunchKernelGGL((pair_qr_rhs_kernel<TS, TW, 3, 4, 4>), g, dim3(256), 0, st, a);
      else hipLaunchKernelGGL((pair_qr_rhs_kernel<TS, TW, 3, 4, 2>), g, dim3(128), 0, st, a);
      break;
    case 3: hipLaunchKernelGGL((pair_qr_rhs_kernel<TS, TW, 4, 5, 2>), g, dim3(128), 0, st, a); break;
  }
}
template <typename TS, typename TW>
void launch_pair_qr_rhs_batched(BatchTable<FactorArgs<TS, TW>> const& t, int nblocks, int n, int nr, int nx, hipStream_t st) {
  const dim3 g(nblocks);
  switch (mfma_variant(n, nr, nx)) {
    case 1: hipLaunchKernelGGL((pair_qr_rhs_batched<TS, TW, 2, 3, 2>), g, dim3(128), 0, st, t); break;
    case 2: hipLaunchKernelGGL((pair_qr_rhs_batched<TS, TW, 3, 4, 2>), g, dim3(128), 0, st, t); break;
    case 3: hipLaunchKernelGGL((pair_qr_rhs_batched<TS, TW, 4, 5, 2>), g, dim3(128), 0, st, t); break;
  }
}
#define BCR_QR_RHS(TS, TW)                                                                                       \
  template void launch_pair_qr_rhs<TS, TW>(FactorArgs<TS, TW> const&, hipStream_t);                              \
  template void launch_pair_qr_rhs_batched<TS, TW>(BatchTable<FactorArgs<TS, TW>> const&, int, int, int, int, hipStream_t);
BCR_QR_RHS(float, float)
BCR_QR_RHS(double, float)
BCR_QR_RHS(double, double)
#undef BCR_QR_RHS

template bool launch_pair_lu_mfma<float, float>(FactorArgs<float, float> const&, hipStream_t, hipError_t*);
template bool launch_pair_lu_mfma<double, float>(FactorArgs<double, float> const&, hipStream_t, hipError_t*);
template bool launch_pair_lu_mfma<double, double>(FactorArgs<double, double> const&, hipStream_t, hipError_t*);
template bool launch_pair_lu_mfma_batched<float, float>(BatchTable<FactorArgs<float, float>> const&, int, int, int, int,
                                                        hipStream_t, hipError_t*);
template bool launch_pair_lu_mfma_batched<double, float>(BatchTable<FactorArgs<double, float>> const&, int, int, int,
                                                         int, hipStream_t, hipError_t*);
template bool launch_pair_lu_mfma_batched<double, double>(BatchTable<FactorArgs<double, double>> const&, int, int,
                                                          int, int, hipStream_t, hipError_t*);

}  // namespace bcr
