// LU solve sweeps for several right-hand sides, n <= 64, on the matrix cores:
// one wavefront per pair and 16 columns.
//
// With m columns a pair's sweep is 2n^2 m (forward) and 3n^2 m (backward)
// flops on factor blocks read once, a contraction: the register and streamed
// sweeps carry four columns at a time through row-per-lane recurrences (one
// lane broadcast and one FMA per factor entry and column) and were bound by
// that VALU work.  Here the blocks go through v_mfma_f64_16x16x4 as 16 x 16
// tiles loaded straight from HBM in the A operand's layout (16 rows of four
// columns: 128-byte runs).  The 16 x 16 diagonal blocks are substituted in
// slabs of four rows: value i of the accumulator holds rows 4i .. 4i + 3 over
// the four lane groups, which is the B operand of the update of the rows
// behind (one product per slab); inside a slab the four rows' values are
// exchanged between the lane groups (v_permlane swaps) and substituted in
// every lane.  HBM bounds it: factors once per 16 columns, the columns once
// in, once out.
//
//   forward  W = P [x_jp; x_j], staged in LDS with rows at their final
//            positions; W1_kb = L_kk^-1 (W1_kb - sum_{m<kb} L_km W1_m) -> x_j,
//            x_jp = W2 - L21 W1, Xpart[j] = -C_j' x_j
//   backward x_j = U^-1 (x_j - D_j x_jp - E_j x_jpp - B_j xb), blocks bottom up
// (cc:1615-1719, cc:1805-1949.)  All arithmetic is FP64, for FP32 objects too
// (the FP32 product's layout does not put four neighbouring rows in one
// value); only the order of the products' sums differs from the other sweeps.
#include "bcr_launch.hh"
#include "bcr_mfma.hh"
#include "bcr_wave.hh"

namespace bcr {
namespace {

using D4 = V4<double>;

// rows r0 + cl, columns c0 + g + 4i of the column-major block M (leading
// dimension ld), zero at and beyond rlim / clim: an A operand.  Addresses are
// clamped, so every load is issued unconditionally.
template <typename TW>
__device__ __forceinline__ D4 tile(const TW* M, unsigned ld, int r0, int c0, int rlim, int clim, int g, int cl) {
  D4 v;
  const int r = r0 + cl;
  const unsigned rr = r < rlim ? r : 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = c0 + g + 4 * i;
    const TW x = gload(M, rr + unsigned(c < clim ? c : 0) * ld);
    v[i] = double(keep_if(x, r < rlim && c < clim));
  }
  return v;
}

__device__ __forceinline__ D4 neg(D4 v) { return D4{-v.x, -v.y, -v.z, -v.w}; }

// v of lane group s (lanes 16 s ..) in all four groups, s = 0 .. 3
__device__ __forceinline__ void group_values(double v, double (&o)[4]) {
  unsigned w[2] = {unsigned(__double2loint(v)), unsigned(__double2hiint(v))};
  unsigned q[4][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    // groups 0,0,2,2 and 1,1,3,3, then each half to both
    const auto p = __builtin_amdgcn_permlane16_swap(w[h], w[h], false, false);
    const auto e = __builtin_amdgcn_permlane32_swap(p[0], p[0], false, false);
    const auto f = __builtin_amdgcn_permlane32_swap(p[1], p[1], false, false);
    q[0][h] = e[0];
    q[2][h] = e[1];
    q[1][h] = f[0];
    q[3][h] = f[1];
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) o[s] = __hiloint2double(int(q[s][1]), int(q[s][0]));
}

// entry (r, c) of the slab's 4 x 4 diagonal block: d holds a diagonal tile
// as an A operand, b is the slab
__device__ __forceinline__ double slab_entry(D4 const& d, int b, int r, int c) {
  return wave::rl(d[b], 4 * b + r + 16 * c);
}

__device__ __forceinline__ double pick(double const (&v)[4], int g) {
  const double lo = g & 1 ? v[1] : v[0], hi = g & 1 ? v[3] : v[2];
  return g & 2 ? hi : lo;
}

// acc <- L^-1 acc for the unit lower 16 x 16 block d
__device__ __forceinline__ void solve_lower(D4& acc, D4 const& d, int g, int cl) {
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    double v[4];
    group_values(acc[b], v);
    v[1] = fma(-slab_entry(d, b, 1, 0), v[0], v[1]);
    v[2] = fma(-slab_entry(d, b, 2, 0), v[0], v[2]);
    v[3] = fma(-slab_entry(d, b, 3, 0), v[0], v[3]);
    v[2] = fma(-slab_entry(d, b, 2, 1), v[1], v[2]);
    v[3] = fma(-slab_entry(d, b, 3, 1), v[1], v[3]);
    v[3] = fma(-slab_entry(d, b, 3, 2), v[2], v[3]);
    acc[b] = pick(v, g);
    if (b < 3) {
      const double y = acc[b];
      acc = mfma1(keep_if(-d[b], cl >= 4 * b + 4), y, acc);
      acc[b] = y;
    }
  }
}

// acc <- U^-1 acc for the upper 16 x 16 block d (rows and columns at and
// beyond lim: identity)
__device__ __forceinline__ void solve_upper(D4& acc, D4 const& d, int lim, int g, int cl) {
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    double v[4], u[4];
    group_values(acc[b], v);
#pragma unroll
    for (int c = 0; c < 4; ++c) u[c] = 1.0 / (4 * b + c < lim ? slab_entry(d, b, c, c) : 1.0);
    v[3] *= u[3];
    v[2] = fma(-slab_entry(d, b, 2, 3), v[3], v[2]) * u[2];
    v[1] = fma(-slab_entry(d, b, 1, 3), v[3], v[1]);
    v[0] = fma(-slab_entry(d, b, 0, 3), v[3], v[0]);
    v[1] = fma(-slab_entry(d, b, 1, 2), v[2], v[1]) * u[1];
    v[0] = fma(-slab_entry(d, b, 0, 2), v[2], v[0]);
    v[0] = fma(-slab_entry(d, b, 0, 1), v[1], v[0]) * u[0];
    acc[b] = pick(v, g);
    if (b > 0) {
      const double y = acc[b];
      acc = mfma1(keep_if(-d[b], cl < 4 * b), y, acc);
      acc[b] = y;
    }
  }
}

// waves per SIMD asked of the compiler (it would otherwise load ahead into
// every register)
constexpr int mfma_waves(int nb) { return nb <= 2 ? 3 : 2; }

template <typename TW, typename TX, int NB>
__global__ void __launch_bounds__(64, mfma_waves(NB)) forward_lu_mfma_kernel(SolveArgs<TW, TX> a) {
  // column stride of X: the lanes of an operand read (16 columns, 4 rows)
  // fall on different banks
  constexpr int NMAX = 16 * NB, RS = (2 * NMAX + 63) / 64, LD = 2 * NMAX + 2;
  __shared__ __align__(16) double X[16 * LD];   // columns: top rows [0, NMAX), rest rows [NMAX, 2 NMAX)
  const int lane = threadIdx.x, g = lane >> 4, cl = lane & 15;
  const int n = a.n, n2 = 2 * n, nr = a.nr, nrhs = a.nrhs;
  const int64_t ldx = a.ldx;
  const int q0 = 16 * int(blockIdx.y), nq = min(16, nrhs - q0);   // this wave's columns
  int j, jp, jpp;
  pair_of_uniform(a, blockIdx.x, j, jp, jpp);
  const TW* Tj = a.Tm + size_t(j) * tsize(n);
  const TW* Cj = a.C + size_t(j) * nr * n;
  // row lane + 64 s of [x_jp; x_j]: where it comes from, where it ends
  const int pvl = lane < n ? a.perm[size_t(j) * n + lane] - 1 : 0;
  size_t in_row[RS], out_row[RS];
  int pos[RS], oslot[RS];
  bool row[RS];
  TX xv[RS][16];
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const int r = lane + 64 * s;
    row[s] = r < n2;
    in_row[s] = r < n ? size_t(jp) * n + r : row[s] ? size_t(j) * n + (r - n) : 0;
    out_row[s] = r < n ? size_t(j) * n + r : size_t(jp) * n + (r - n);
    oslot[s] = r < n ? r : NMAX + (r - n);
    pos[s] = r;
#pragma unroll
    for (int q = 0; q < 16; ++q) xv[s][q] = a.x[in_row[s] + size_t(q0 + min(q, nq - 1)) * ldx];
  }
  // the diagonal tiles of L and those below them, in flight with the columns
  // where the registers hold both (NB <= 2)
  D4 lt[NB][NB];
  auto load_l = [&] {
#pragma unroll
    for (int kb = 0; kb < NB; ++kb)
#pragma unroll
      for (int m = 0; m <= kb; ++m) lt[kb][m] = tile(Tj, n2, 16 * kb, 16 * m, n, n, g, cl);
  };
  D4 w[NB], rt[NB];   // W1; a row of tiles of L21
  auto load_r = [&](int b) {
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) rt[kb] = tile(Tj + n, n2, 16 * b, 16 * kb, n, n, g, cl);
  };
  if (NB <= 2) load_l();
  // the row interchanges (1-based ipiv): the row at c and the row at ipiv[c] swap
  for (int c = 0; c < n; ++c) {
    const int pv = __builtin_amdgcn_readlane(pvl, c);
#pragma unroll
    for (int s = 0; s < RS; ++s) pos[s] = pos[s] == c ? pv : pos[s] == pv ? c : pos[s];
  }
#pragma unroll
  for (int s = 0; s < RS; ++s) {
    const int r = lane + 64 * s, i = r - n2;   // the lanes beyond 2n zero the padding slots
    const int slot = row[s] ? (pos[s] < n ? pos[s] : NMAX + pos[s] - n) : i < NMAX - n ? n + i : 2 * n + i;
    if (slot < 2 * NMAX) {
#pragma unroll
      for (int q = 0; q < 16; ++q) X[q * LD + slot] = double(keep_if(xv[s][q], row[s] && q < nq));
    }
  }
  lds_order();
  double* const xc = X + cl * LD;   // this lane's column
  if (NB <= 2) load_r(0);
  else load_l();
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) {
    D4 acc = ld4(xc + 16 * kb, g);
#pragma unroll
    for (int m = 0; m < kb; ++m) acc = mfma4<double>(neg(lt[kb][m]), w[m], acc);
    solve_lower(acc, lt[kb][kb], g, cl);
    w[kb] = acc;
  }
  lds_order();
  if (NB > 2) load_r(0);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    D4 cur[NB];
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) cur[kb] = rt[kb];
    if (b + 1 < NB) load_r(b + 1);
    D4 acc = ld4(xc + NMAX + 16 * b, g);
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) acc = mfma4<double>(neg(cur[kb]), w[kb], acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      xc[NMAX + 16 * b + g + 4 * i] = acc[i];
      xc[16 * b + g + 4 * i] = w[b][i];
    }
  }
  lds_order();
#pragma unroll
  for (int s = 0; s < RS; ++s)
    if (row[s]) {
#pragma unroll
      for (int q = 0; q < 16; ++q)
        if (q < nq) a.x[out_row[s] + size_t(q0 + q) * ldx] = TX(X[q * LD + oslot[s]]);
    }
  if (nr > 0) {   // the border partial
    D4 acc{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kb = 0; kb < NB; ++kb) acc = mfma4<double>(tile(Cj, nr, 0, 16 * kb, nr, n, g, cl), w[kb], acc);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = g + 4 * i;
      if (r < nr && cl < nq) a.Xpart[size_t(j) * nr * nrhs + r + size_t(q0 + cl) * nr] = TX(-acc[i]);
    }
  }
}

template <typename TW, typename TX, int NB>
__global__ void __launch_bounds__(64, mfma_waves(NB)) backward_lu_mfma_kernel(SolveArgs<TW, TX> a) {
  const int lane = threadIdx.x, g = lane >> 4, cl = lane & 15;
  const int n = a.n, n2 = 2 * n, nx = a.nx, nrhs = a.nrhs;
  const int q0 = 16 * int(blockIdx.y), nq = min(16, nrhs - q0);   // this wave's columns
  int j, jp, jpp;
  pair_of_uniform(a, blockIdx.x, j, jp, jpp);
  const size_t nn = size_t(n) * n;
  const TW* Tj = a.Tm + size_t(j) * tsize(n);
  const TW *Dj = a.D + size_t(j) * nn, *Ej = a.E + size_t(j) * nn, *Bj = a.B + size_t(j) * n * nx;
  const bool live = cl < nq;
  TX* const xc = a.x + size_t(q0 + min(cl, nq - 1)) * size_t(a.ldx);   // this lane's column
  TX *const xj = xc + size_t(j) * n, *const xb = xc + size_t(a.N + 1) * n + a.qx;
  const TX *const xp = xc + size_t(jp) * n, *const xpp = xc + size_t(jpp) * n;
  // rows r0 + g + 4i of a column block of this lane's column: a B operand
  auto rows = [&](const TX* v, int r0, int lim) {
    D4 o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + g + 4 * i;
      const TX x = v[r < lim ? r : 0];
      o[i] = double(keep_if(x, r < lim && live));
    }
    return o;
  };
  D4 acc[NB], x0[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    x0[b] = rows(xj, 16 * b, n);
    acc[b] = D4{0.0, 0.0, 0.0, 0.0};
  }
  // D_j x_jp + E_j x_jpp, one 16-column block of both at a time
#pragma unroll
  for (int kb = 0; kb < NB; ++kb) {
    const D4 b0 = rows(xp, 16 * kb, n), b1 = rows(xpp, 16 * kb, n);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      acc[b] = mfma4<double>(tile(Dj, n, 16 * b, 16 * kb, n, n, g, cl), b0, acc[b]);
      acc[b] = mfma4<double>(tile(Ej, n, 16 * b, 16 * kb, n, n, g, cl), b1, acc[b]);
    }
  }
  for (int c0 = 0; c0 < nx; c0 += 16) {   // + B_j xb
    const D4 bx = rows(xb, c0, nx);
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = mfma4<double>(tile(Bj, n, 16 * b, c0, n, nx, g, cl), bx, acc[b]);
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = x0[b] - acc[b];
  // U^-1, blocks bottom up; the tiles of column block kb of U
  D4 ut[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) ut[b] = tile(Tj, n2, 16 * b, 16 * (NB - 1), n, n, g, cl);
#pragma unroll
  for (int kb = NB - 1; kb >= 0; --kb) {
    D4 cur[NB];
#pragma unroll
    for (int b = 0; b <= kb; ++b) {
      cur[b] = ut[b];
      if (b < kb) ut[b] = tile(Tj, n2, 16 * b, 16 * (kb - 1), n, n, g, cl);
    }
    solve_upper(acc[kb], cur[kb], n - 16 * kb, g, cl);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 16 * kb + g + 4 * i;
      if (r < n && live) xj[r] = TX(acc[kb][i]);
    }
#pragma unroll
    for (int b = 0; b < kb; ++b) acc[b] = mfma4<double>(neg(cur[b]), acc[kb], acc[b]);
  }
}

}  // namespace

template <typename TW, typename TX>
bool launch_sweep_lu_mfma(bool forward, SolveArgs<TW, TX> const& a, hipStream_t st, hipError_t* err) {
  if (a.n < 1 || a.n > 64 || a.nr > 16 || a.npairs < 1) return false;
  const int chunks = (a.nrhs + 15) / 16;
  if (chunks < 1 || chunks > 65535) return false;
  auto go = [&](auto kf, auto kb) {
    hipLaunchKernelGGL(forward ? kf : kb, dim3(a.npairs, chunks), dim3(64), 0, st, a);
    *err = hipGetLastError();
    return true;
  };
  if (a.n <= 16) return go(forward_lu_mfma_kernel<TW, TX, 1>, backward_lu_mfma_kernel<TW, TX, 1>);
  if (a.n <= 32) return go(forward_lu_mfma_kernel<TW, TX, 2>, backward_lu_mfma_kernel<TW, TX, 2>);
  if (a.n <= 48) return go(forward_lu_mfma_kernel<TW, TX, 3>, backward_lu_mfma_kernel<TW, TX, 3>);
  return go(forward_lu_mfma_kernel<TW, TX, 4>, backward_lu_mfma_kernel<TW, TX, 4>);
}

template bool launch_sweep_lu_mfma<double, double>(bool, SolveArgs<double, double> const&, hipStream_t, hipError_t*);
template bool launch_sweep_lu_mfma<float, float>(bool, SolveArgs<float, float> const&, hipStream_t, hipError_t*);
template bool launch_sweep_lu_mfma<float, double>(bool, SolveArgs<float, double> const&, hipStream_t, hipError_t*);

}  // namespace bcr
