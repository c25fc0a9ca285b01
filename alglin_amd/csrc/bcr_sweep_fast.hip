// Wave-synchronous solve sweeps for LU-eliminated pairs, n <= 32: the launches
// of the bodies in bcr_sweep_body.hh, four wavefronts per workgroup.
#include "bcr_sweep_body.hh"

namespace bcr {
namespace {

// this wavefront's index in the launch, workgroup bid of it
__device__ __forceinline__ int sweep_wave(int bid) {
  return bid * 4 + __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
}

template <typename TW, typename TX, int NMAX, int QB>
__global__ void __launch_bounds__(256) forward_lu_fast_kernel(SolveArgs<TW, TX> a) {
  forward_lu_fast_body<TW, TX, NMAX, QB>(a, sweep_wave(blockIdx.x));
}


template <typename TW, typename TX, int NMAX, int QB>
__global__ void __launch_bounds__(256) backward_lu_fast_kernel(SolveArgs<TW, TX> a) {
  backward_lu_fast_body<TW, TX, NMAX, QB>(a, sweep_wave(blockIdx.x));
}


template <typename TW, typename TX, int NMAX, int QB, bool FWD>
__global__ void __launch_bounds__(256) sweep_lu_fast_batched(BatchTable<SolveArgs<TW, TX>> t) {
  const int e = t.entry[blockIdx.x];
  if (skipped(t.args[e].skip)) return;
  if (FWD) forward_lu_fast_body<TW, TX, NMAX, QB>(t.args[e], sweep_wave(int(blockIdx.x) - t.first[e]));
  else backward_lu_fast_body<TW, TX, NMAX, QB>(t.args[e], sweep_wave(int(blockIdx.x) - t.first[e]));
}

// four columns at a time only for n <= 8: beyond, several columns go through
// the matrix cores (all but some 10^6 of them, which its grid does not hold)
template <typename TW, typename TX, int NMAX>
hipError_t launch_sweep_nmax(bool forward, SolveArgs<TW, TX> const& a, hipStream_t st) {
  constexpr int PG = 64 / (2 * NMAX), QB = NMAX <= 8 ? 4 : 1;
  const int blocks = (a.npairs + 4 * PG - 1) / (4 * PG);
  if (forward) {
    if (a.nrhs == 1) hipLaunchKernelGGL((forward_lu_fast_kernel<TW, TX, NMAX, 1>), dim3(blocks), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((forward_lu_fast_kernel<TW, TX, NMAX, QB>), dim3(blocks), dim3(256), 0, st, a);
  } else {
    if (a.nrhs == 1) hipLaunchKernelGGL((backward_lu_fast_kernel<TW, TX, NMAX, 1>), dim3(blocks), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((backward_lu_fast_kernel<TW, TX, NMAX, QB>), dim3(blocks), dim3(256), 0, st, a);
  }
  return hipGetLastError();
}

}  // namespace

template <typename TW, typename TX>
bool launch_sweep_lu_fast(bool forward, SolveArgs<TW, TX> const& a, hipStream_t st, hipError_t* err) {
  if (a.n < 1 || a.n > 32 || a.npairs < 1) return false;
  if (a.n <= 4) *err = launch_sweep_nmax<TW, TX, 4>(forward, a, st);
  else if (a.n <= 8) *err = launch_sweep_nmax<TW, TX, 8>(forward, a, st);
  else if (a.n <= 16) *err = launch_sweep_nmax<TW, TX, 16>(forward, a, st);
  else *err = launch_sweep_nmax<TW, TX, 32>(forward, a, st);
  return true;
}

// pairs per workgroup of the sweep kernels for block size bound n (<= 32)
int sweep_lu_fast_pairs_per_block(int n) {
  const int nmax = n <= 4 ? 4 : n <= 8 ? 8 : n <= 16 ? 16 : 32;
  return 4 * (64 / (2 * nmax));
}

template <typename TW, typename TX>
bool launch_sweep_lu_fast_batched(bool forward, BatchTable<SolveArgs<TW, TX>> const& t, int nblocks, int n, int nrhs,
                                  hipStream_t st, hipError_t* err) {
  if (n < 1 || n > 32) return false;
  auto go = [&](auto k1, auto k4) {
    if (nrhs == 1) hipLaunchKernelGGL(k1, dim3(nblocks), dim3(256), 0, st, t);
    else hipLaunchKernelGGL(k4, dim3(nblocks), dim3(256), 0, st, t);
    *err = hipGetLastError();
    return true;
  };
#define BCR_SW(NM)                                                                                                \
  return forward ? go(sweep_lu_fast_batched<TW, TX, NM, 1, true>, sweep_lu_fast_batched<TW, TX, NM, 4, true>)     \
                 : go(sweep_lu_fast_batched<TW, TX, NM, 1, false>, sweep_lu_fast_batched<TW, TX, NM, 4, false>);
  if (n <= 4) { BCR_SW(4) }
  if (n <= 8) { BCR_SW(8) }
  if (n <= 16) { BCR_SW(16) }
  BCR_SW(32)
#undef BCR_SW
}

template bool launch_sweep_lu_fast_batched<double, double>(bool, BatchTable<SolveArgs<double, double>> const&, int, int,
                                                           int, hipStream_t, hipError_t*);
template bool launch_sweep_lu_fast_batched<float, float>(bool, BatchTable<SolveArgs<float, float>> const&, int, int,
                                                         int, hipStream_t, hipError_t*);
template bool launch_sweep_lu_fast_batched<float, double>(bool, BatchTable<SolveArgs<float, double>> const&, int, int,
                                                          int, hipStream_t, hipError_t*);
template bool launch_sweep_lu_fast<double, double>(bool, SolveArgs<double, double> const&, hipStream_t, hipError_t*);
template bool launch_sweep_lu_fast<float, float>(bool, SolveArgs<float, float> const&, hipStream_t, hipError_t*);
template bool launch_sweep_lu_fast<float, double>(bool, SolveArgs<float, double> const&, hipStream_t, hipError_t*);

}  // namespace bcr
