// Host interface of the fused kernels for small block sizes (bcr_small.hip).
#pragma once
#include "bcr_launch.hh"

namespace bcr {

// the last block in small_factor: F summed and the block assembled; its LU too
enum SmallLast : int { kSmallAssemble = 1, kSmallFactor = 2 };

// One factorization's start: status word and pending slots cleared, the rows
// and border blocks the first level does not read (row N-1 and C_{N-1} when N
// is odd, C_N) copied from the operator.
template <typename TA, typename TW>
struct SingleArgs {
  FactorArgs<TW, TW> f;             // sources: the working blocks
  const TA *pD, *pE, *pB, *pC, *pF; // pristine operator
  int64_t npend;                    // elements of f.Cpend
  // small_factor only
  int prep;                         // this launch starts the factorization
  int L0;                           // first level it takes (>= N: none)
  int last;                         // SmallLast bits
  AssembleArgs<TW, TA> as;
  double* Feff;
  int32_t* ipiv;
};

template <typename TA, typename TW>
hipError_t launch_prep_single(SingleArgs<TA, TW> const& a, hipStream_t st);

// first level (stride) that one workgroup takes over; N when none is worth it
int small_factor_level(int N, int n, int nx, int nr, size_t elem, bool first_ok);
int small_solve_level(int N, int n, int nr, int nrhs, size_t elem);
constexpr int kSmallSum = 1 << 16;   // values one workgroup sums

// levels a.L0 .. of an LU factorization in one workgroup: n <= 16, nx, nr <= 8;
// with a.last also the last block: its assembly ((N - 1) nr nx <= kSmallSum)
// and its LU (square, Nc <= 64);
// false when the shape is not covered
template <typename TA, typename TW>
bool launch_small_factor(SingleArgs<TA, TW> const& a, hipStream_t st, hipError_t* err);

enum SmallPhase : int { kSmallFwd = 1, kSmallXb = 2, kSmallLast = 4, kSmallBwd = 8 };
template <typename TW, typename TX>
struct SmallSolveArgs {
  SolveArgs<TW, TX> s;
  int L0;       // first level of the launch's sweeps
  int phases;   // SmallPhase bits, run in this order
  LastSolveArgs<TX> last;
};
// sweeps of the levels from L0 on (n <= 16, LU), the sum of the xb partials
// ((N - 1) nr nrhs <= kSmallSum, nr nrhs <= 512) and the last solve (LU,
// square, Nc <= 64) in one workgroup
template <typename TW, typename TX>
bool launch_small_solve(SmallSolveArgs<TW, TX> const& a, hipStream_t st, hipError_t* err);

}  // namespace bcr
