// One system with n <= 16: the reduction levels that no longer fill the chip,
// and the last block, in one launch of one workgroup each way.
//
// From the level on where a level's pairs fit a few rounds of one workgroup,
// separate launches cost more than the work: a level of a few pairs is bound
// by its launch, the first fetch of its instructions on every CU and its own
// chain.  Here the levels follow each other behind a workgroup barrier with
// the code already in the instruction cache; the boundary sums, the last
// block's assembly and LU (or its solve) run in the same launch.
//   small_factor: [clear + copies] levels L0, 2 L0, .. [F sum, assembly, LU]
//   small_solve : forward L0 .., xb sum, last solve, backward .. L0
// The pair and sweep bodies are those of the wide launches, so the results
// are the same bits; the two boundary sums run in FP64 and another order.
#include "bcr_small.hh"

#include "bcr_factor_fast.inc"
#include "bcr_last_body.hh"
#include "bcr_sweep_body.hh"

namespace bcr {
namespace {

template <typename TA, typename TW>
__device__ __forceinline__ void prep_body(SingleArgs<TA, TW> const& a, int64_t tid, int64_t nth) {
  const int N = a.f.N, n = a.f.n, nr = a.f.nr, nx = a.f.nx;
  const int64_t nn = int64_t(n) * n, bn = int64_t(n) * nx, rn = int64_t(nr) * n;
  if (tid < 4) a.f.status[tid] = 0;
  for (int64_t i = tid; i < a.npend; i += nth) a.f.Cpend[i] = TW(0);
  if (N % 2 == 1) {
    const int64_t k = N - 1;
    for (int64_t i = tid; i < nn; i += nth) {
      a.f.D[k * nn + i] = TW(a.pD[k * nn + i]);
      a.f.E[k * nn + i] = TW(a.pE[k * nn + i]);
    }
    for (int64_t i = tid; i < bn; i += nth) a.f.B[k * bn + i] = TW(a.pB[k * bn + i]);
    for (int64_t i = tid; i < rn; i += nth) a.f.C[k * rn + i] = TW(a.pC[k * rn + i]);
  }
  for (int64_t i = tid; i < rn; i += nth) a.f.C[N * rn + i] = TW(a.pC[N * rn + i]);
}

template <typename TA, typename TW>
__global__ void __launch_bounds__(256) prep_single_kernel(SingleArgs<TA, TW> a) {
  prep_body(a, int64_t(blockIdx.x) * 256 + threadIdx.x, int64_t(gridDim.x) * 256);
}

// sum over j = 1 .. N-1 of part[j m + i] for i < m (m <= nth), returned by
// thread i; red: nth doubles of LDS.  Ends with a barrier behind it.
template <typename T>
__device__ __forceinline__ double column_sum(const T* part, int N, int m, double* red, int tid, int nth) {
  const int per = nth / m * m;
  const int64_t end = int64_t(N) * m;
  double s = 0;
  if (tid < per) {
    int64_t e = m + tid;
    for (; e + 3 * int64_t(per) < end; e += 4 * int64_t(per)) {
      const T v0 = part[e], v1 = part[e + per], v2 = part[e + 2 * per], v3 = part[e + 3 * per];
      s += (double(v0) + double(v1)) + (double(v2) + double(v3));
    }
    for (; e < end; e += per) s += double(part[e]);
  }
  red[tid] = s;
  __syncthreads();
  for (int g = per / m; g > 1;) {
    const int h = (g + 1) / 2;
    if (tid < (g - h) * m) red[tid] += red[tid + h * m];
    __syncthreads();
    g = h;
  }
  return tid < m ? red[tid] : 0.0;
}

// wavefronts of the factor workgroup: as many as the pair body's registers let
// one CU hold
constexpr int factor_waves(int nmax, size_t elem) { return nmax <= 4 ? 16 : nmax <= 8 || elem == 4 ? 8 : 4; }
constexpr int solve_waves(int nmax) { return nmax <= 8 ? 16 : 8; }

template <typename TA, typename TW, int NMAX, int NXMAX, int NRMAX>
__global__ void __launch_bounds__(64 * factor_waves(NMAX, sizeof(TW))) small_factor_kernel(SingleArgs<TA, TW> a) {
  constexpr int NW = factor_waves(NMAX, sizeof(TW)), G = kWave / (2 * NMAX), NT = 64 * NW;
  __shared__ FastLds<TW, NMAX, NXMAX, NRMAX, true> sm[NW];
  __shared__ LastLuLds<1> lu;
  __shared__ double red[NT];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  const int N = a.f.N;
  if (a.prep) {
    prep_body(a, tid, NT);
    __syncthreads();
  }
  FactorArgs<TW, TW> f = a.f;
  for (int64_t L = a.L0; L < N; L *= 2) {
    f.L = int(L);
    f.npairs = int((N + L - 1) / (2 * L));
    f.slot_cur = (31 - __clz(int(L))) & 1;
    f.first = L == 1 ? 1 : 0;
    if constexpr (sizeof(TA) == sizeof(TW)) {   // level 1 reads the operator
      f.sD = L == 1 ? reinterpret_cast<const TW*>(a.pD) : f.D;
      f.sE = L == 1 ? reinterpret_cast<const TW*>(a.pE) : f.E;
      f.sB = L == 1 ? reinterpret_cast<const TW*>(a.pB) : f.B;
      f.sC = L == 1 ? reinterpret_cast<const TW*>(a.pC) : f.C;
    }
    for (int b = w; b * G < f.npairs; b += NW)
      pair_lu_fast_body<true, TW, TW, NMAX, NXMAX, NRMAX>(f, b, sm[w]);
    __syncthreads();
  }
  if (!(a.last & kSmallAssemble)) return;
  const int m = f.nr * f.nx;
  if (m > 0) {
    const double s = column_sum(f.Fpart, N, m, red, tid, NT);
    if (tid < m) a.Feff[tid] = double(a.pF[tid]) + s;
    __syncthreads();
  }
  assemble_last_body<TW, TA>(a.as, tid, NT);
  if (!(a.last & kSmallFactor)) return;
  __syncthreads();
  lu_last_regs_body<1, 4, false>(a.as.Hm, a.as.Nc, a.ipiv, f.status, w, tid & 63, lu);
}

template <typename TW, typename TX, int NMAX, int QB>
__global__ void __launch_bounds__(64 * solve_waves(NMAX)) small_solve_kernel(SmallSolveArgs<TW, TX> a) {
  constexpr int NW = solve_waves(NMAX), NT = 64 * NW, PG = 64 / (2 * NMAX);
  __shared__ double red[NT];
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  SolveArgs<TW, TX> s = a.s;
  const int N = s.N;
  if (a.phases & kSmallFwd)
    for (int64_t L = a.L0; L < N; L *= 2) {
      s.L = int(L);
      s.npairs = int((N + L - 1) / (2 * L));
      for (int b = w; b * PG < s.npairs; b += NW) forward_lu_fast_body<TW, TX, NMAX, QB>(s, b);
      __syncthreads();
    }
  const int m = s.nr * s.nrhs;
  if ((a.phases & kSmallXb) && m > 0 && N > 1) {
    const double v = column_sum(s.Xpart, N, m, red, tid, NT);
    if (tid < m) {
      TX* const d = s.x + size_t(N + 1) * s.n + s.qr + tid % s.nr + size_t(tid / s.nr) * s.ldx;
      *d = TX(double(*d) + v);
    }
    __syncthreads();
  }
  if (a.phases & kSmallLast) {
    for (int q = w; q < s.nrhs; q += NW) last_solve_lu_wave_body<TX, 1>(a.last, s.x + size_t(q) * s.ldx, tid & 63);
    __syncthreads();
  }
  if (a.phases & kSmallBwd) {
    int64_t L = a.L0;
    while (2 * L < N) L *= 2;
    for (; L >= a.L0; L /= 2) {
      if (L >= N) continue;
      s.L = int(L);
      s.npairs = int((N + L - 1) / (2 * L));
      for (int b = w; b * PG < s.npairs; b += NW) backward_lu_fast_body<TW, TX, NMAX, QB>(s, b);
      __syncthreads();
    }
  }
}

// the first level (stride, from Lmin on) with at most cap pairs, else N
int first_level(int N, int cap, int Lmin) {
  int64_t L = Lmin;
  while (L < N && (N + L - 1) / (2 * L) > cap) L *= 2;
  return int(L < N ? L : N);
}

int nmax_of(int n) { return n <= 4 ? 4 : n <= 8 ? 8 : 16; }

}  // namespace

// Rounds of one workgroup that a level of the factorization may take: a further
// round of pairs costs about what a launch of its own does.
constexpr int kRounds = 2;

// The round is that of the configuration the launch takes, which grows with the
// border too (counted by n alone, n = 4 with nx = nr = 8 took eight rounds:
// N = 1000 factor and solve 379 us, so 253).
int small_factor_level(int N, int n, int nx, int nr, size_t elem, bool first_ok) {
  int nm = 16;
  pair_lu_fast_pick(n, nx, nr, [&](auto NM, auto, auto) { nm = decltype(NM)::value; });
  return first_level(N, kRounds * factor_waves(nm, elem) * (kWave / (2 * nm)), first_ok ? 1 : 2);
}

// A level of the sweeps: one round, its waves already fill the CU; half of one
// where the border sums of a pair are many, two where a pair has little work in
// FP32.  FP64, N = 1000, against two rounds and against a launch per level: n = 8,
// 1 column 90, 97, 126 us; nr = 16, 4 columns 256, 333, 284; n = 16, 1 column 133,
// 142, 164; n = 2, nr = 16, 4 columns 199, 257, 218.  FP32, n = 2, nr = 2, 1 column,
// N = 1000, factor and solve: two rounds 117, one 122.
int small_solve_level(int N, int n, int nr, int nrhs, size_t elem) {
  const int nm = nmax_of(n), round = solve_waves(nm) * (kWave / (2 * nm)), sums = nr * nrhs;
  return first_level(N, sums >= 32 ? round / 2 : nm == 4 && elem == 4 && sums <= 4 ? 2 * round : round, 1);
}

template <typename TA, typename TW>
hipError_t launch_prep_single(SingleArgs<TA, TW> const& a, hipStream_t st) {
  const int64_t blocks = (a.npend + 1023) / 1024;
  hipLaunchKernelGGL((prep_single_kernel<TA, TW>), dim3(unsigned(blocks < 1 ? 1 : blocks > 4096 ? 4096 : blocks)),
                     dim3(256), 0, st, a);
  return hipGetLastError();
}

template <typename TA, typename TW>
bool launch_small_factor(SingleArgs<TA, TW> const& a, hipStream_t st, hipError_t* err) {
  return pair_lu_fast_pick(a.f.n, a.f.nx, a.f.nr, [&](auto NM, auto NX, auto NR) {
    constexpr int nm = decltype(NM)::value, nxm = decltype(NX)::value, nrm = decltype(NR)::value;
    hipLaunchKernelGGL((small_factor_kernel<TA, TW, nm, nxm, nrm>), dim3(1), dim3(64 * factor_waves(nm, sizeof(TW))), 0, st, a);
    *err = hipGetLastError();
  });
}

template <typename TW, typename TX>
bool launch_small_solve(SmallSolveArgs<TW, TX> const& a, hipStream_t st, hipError_t* err) {
  const int n = a.s.n;
  if (n < 1 || n > 16) return false;
  auto go = [&](auto k1, auto k4) {
    const dim3 block(64 * solve_waves(nmax_of(n)));
    if (a.s.nrhs == 1) hipLaunchKernelGGL(k1, dim3(1), block, 0, st, a);
    else hipLaunchKernelGGL(k4, dim3(1), block, 0, st, a);
    *err = hipGetLastError();
    return true;
  };
  if (n <= 4) return go(small_solve_kernel<TW, TX, 4, 1>, small_solve_kernel<TW, TX, 4, 4>);
  if (n <= 8) return go(small_solve_kernel<TW, TX, 8, 1>, small_solve_kernel<TW, TX, 8, 4>);
  return go(small_solve_kernel<TW, TX, 16, 1>, small_solve_kernel<TW, TX, 16, 4>);
}

template hipError_t launch_prep_single<double, double>(SingleArgs<double, double> const&, hipStream_t);
template hipError_t launch_prep_single<float, float>(SingleArgs<float, float> const&, hipStream_t);
template hipError_t launch_prep_single<double, float>(SingleArgs<double, float> const&, hipStream_t);
template bool launch_small_factor<double, double>(SingleArgs<double, double> const&, hipStream_t, hipError_t*);
template bool launch_small_factor<float, float>(SingleArgs<float, float> const&, hipStream_t, hipError_t*);
template bool launch_small_factor<double, float>(SingleArgs<double, float> const&, hipStream_t, hipError_t*);
template bool launch_small_solve<double, double>(SmallSolveArgs<double, double> const&, hipStream_t, hipError_t*);
template bool launch_small_solve<float, float>(SmallSolveArgs<float, float> const&, hipStream_t, hipError_t*);
template bool launch_small_solve<float, double>(SmallSolveArgs<float, double> const&, hipStream_t, hipError_t*);

}  // namespace bcr
