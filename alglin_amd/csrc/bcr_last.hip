// The bordered last block (BABD_BorderedCR.cc:1281-1479), FP64.
//
// After the cyclic reduction only block row 0 (coupling x_0 and x_N) is left;
// with the boundary rows H and the border rows it forms the Nr x Nc matrix
//
//      n   n  qx  nx
//   [ D0 | E0 | 0 | B0 ]  n        (reduced row 0)
//   [ H0 | HN | Hq| Hp ]  n+qr     (pristine boundary rows)
//   [ C0 | CN | Cq| F  ]  nr       (reduced border rows)
//
// assemble_last_kernel builds it (folding the pending C_N contributions and
// the summed F partials), lu_last_kernel factors it with partial pivoting in
// one workgroup (lu_last_regs in registers up to 192 columns, else in place),
// last_solve_kernel gathers the last-block right-hand side straight from the
// solution vector, solves, and scatters (x_0, x_N, q, xb) back (the
// reference's swap of x[0:n] with x[(N-1)n:Nn], cc:1392-1423, is the same
// gather/scatter written in place).
#include "bcr_last_body.hh"

namespace bcr {


template <typename TW, typename TA>
__global__ void __launch_bounds__(256) assemble_last_kernel(AssembleArgs<TW, TA> a) {
  assemble_last_body<TW, TA>(a, blockIdx.x * 256 + threadIdx.x, gridDim.x * 256);
}

// LU with partial pivoting (dgetf2 order: first max, whole-row swaps,
// reciprocal scaling) of the square Nc x Nc last block.
// Past 192 columns (up to there lu_last_regs), in place: too large for LDS.
__device__ __forceinline__ void lu_last_body(double* __restrict__ Hm, int Nc, int32_t* __restrict__ ipiv,
                                             int32_t* __restrict__ status) {
  __shared__ int s_piv;
  const int tid = threadIdx.x, nth = blockDim.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int ld = Nc;
  double* A = Hm;
  for (int c = 0; c < Nc; ++c) {
    if (wid == 0) {
      double best = -1;
      int bi = c;   // a NaN column keeps the diagonal: the index stays valid
      for (int r = c + lane; r < Nc; r += 64) {
        const double v = fabs(A[r + c * ld]);
        if (v > best) { best = v; bi = r; }
      }
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) {
        const double ov = __shfl_xor(best, off);
        const int oi = __shfl_xor(bi, off);
        if (ov > best || (ov == best && oi < bi)) { best = ov; bi = oi; }
      }
      if (lane == 0) {
        s_piv = bi;
        ipiv[c] = bi + 1;
        if (best == 0.0) atomicOr(status, 2);
      }
    }
    __syncthreads();
    const int pv = s_piv;
    if (pv != c)
      for (int s = tid; s < Nc; s += nth) {
        const double t = A[c + s * ld];
        A[c + s * ld] = A[pv + s * ld];
        A[pv + s * ld] = t;
      }
    __syncthreads();
    const double piv = A[c + c * ld];
    const double rinv = piv != 0.0 ? 1.0 / piv : 0.0;
    for (int r = c + 1 + tid; r < Nc; r += nth) A[r + c * ld] *= rinv;
    __syncthreads();
    const int m = Nc - c - 1;
    for (int i = tid; i < m * m; i += nth) {
      const int r = c + 1 + i % m, s = c + 1 + i / m;
      A[r + s * ld] -= A[r + c * ld] * A[c + s * ld];
    }
    __syncthreads();
  }
}

// A_LDS: the factored last block is staged in LDS; otherwise (Nr*Nc*8 bytes
// above the LDS limit, e.g. 152 x 152) it is read from global memory, where
// it stays L2-resident, and only the right-hand-side chunk lives in LDS.
// The Nr right-hand-side rows are gathered from x, the Nc solution rows are
// scattered back.  Methods (kLastLU .. kLastQRP):
//   LU   ipiv (1-based, row swaps), L then U            (getrs)
//   LUPQ row swaps P, L, U, column swaps Q in reverse
//   QR   y = Q^T b (reflectors in order), R^{-1} y      (ormqr + trsv)
//   QRP  as QR, then x[jpvt[i]] = y[i]
__global__ void __launch_bounds__(1024) lu_last_kernel(double* __restrict__ Hm, int Nc, int32_t* __restrict__ ipiv,
                                                        int32_t* __restrict__ status) {
  lu_last_body(Hm, Nc, ipiv, status);
}

template <typename TX, bool A_LDS>
__device__ __forceinline__ void last_solve_body(LastSolveArgs<TX> const& a) {
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n = a.n, Nr = a.Nr, Nc = a.Nc, N = a.N, nrhs = a.nrhs;
  const int method = (a.method >= kLastSVD || (a.status && (*a.status & 8))) ? int(kLastSVD) : a.method;
  const int tid = threadIdx.x, nth = blockDim.x, lane = tid & 63, wid = tid >> 6;
  const int ld = Nr;   // column-major Nr x Nc
  const int R = Nr > Nc ? Nr : Nc;
  double* sm = reinterpret_cast<double*>(smem_raw);
  const double* A = A_LDS ? sm : a.Hm;
  double* X = A_LDS ? sm + size_t(Nr) * Nc : sm;   // R x 16
  double* Z = X + size_t(R) * 16;                   // Nc x 16 (QRP permutation)
  double* s_w = Z + size_t(Nc) * 16;                // 16 (a reflector's products)
  constexpr int QC = 16;
  if (A_LDS)
    for (int i = tid; i < Nr * Nc; i += nth) sm[i] = a.Hm[i];
  const size_t xN = size_t(N) * n;
  const size_t xC = size_t(N + 1) * n + a.qr;
  const int64_t ldx = a.ldx;
  for (int q0 = 0; q0 < nrhs; q0 += QC) {
    const int nq = min(QC, nrhs - q0);
    for (int i = tid; i < R * nq; i += nth) {
      const int r = i % R, q = i / R;
      double v = 0;
      if (r < Nr) {
        size_t row;
        if (r < n) row = r;
        else if (r < 2 * n + a.qr) row = xN + (r - n);
        else row = xC + (r - 2 * n - a.qr);
        v = double(a.x[row + size_t(q0 + q) * ldx]);
      }
      X[r + q * R] = v;
    }
    __syncthreads();
    if (method == kLastSVD) {
      // x = V S^+ U^T b over the rank retained singular triplets
      const int k = Nr < Nc ? Nr : Nc, rank = *a.rank;
      for (int i = tid; i < k * nq; i += nth) {
        const int l = i % k, q = i / k;
        double c = 0;
        if (l < rank) {
          for (int r = 0; r < Nr; ++r) c += a.U[r + size_t(l) * Nr] * X[r + q * R];
          c /= a.S[l];
        }
        Z[l + q * Nc] = c;
      }
      __syncthreads();
      for (int i = tid; i < Nc * nq; i += nth) {
        const int r = i % Nc, q = i / Nc;
        double y = 0;
        for (int l = 0; l < rank; ++l) y += a.V[r + size_t(l) * Nc] * Z[l + q * Nc];
        X[r + q * R] = y;
      }
      __syncthreads();
    } else if (method == kLastLU || method == kLastLUPQ) {
      for (int q = tid; q < nq; q += nth)
        for (int c = 0; c < Nc; ++c) {
          const int pv = method == kLastLU ? a.P[c] - 1 : a.P[c];
          if (pv != c) { const double t = X[c + q * R]; X[c + q * R] = X[pv + q * R]; X[pv + q * R] = t; }
        }
      __syncthreads();
      for (int c = 0; c < Nc; ++c) {
        const int m = Nc - c - 1;
        for (int i = tid; i < m * nq; i += nth) {
          const int r = c + 1 + i % m, q = i / m;
          X[r + q * R] -= A[r + c * ld] * X[c + q * R];
        }
        __syncthreads();
      }
    } else {
      // y = Q^T b: H_0 first; wave q forms v' y for column q
      for (int k = 0; k < Nc; ++k) {
        const double tk = a.tau[k];
        if (tk != 0.0) {
          if (wid < nq) {
            double s = 0;
            for (int r = k + lane; r < Nr; r += 64) s += (r == k ? 1.0 : A[r + k * ld]) * X[r + wid * R];
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off);
            if (lane == 0) s_w[wid] = s * tk;
          }
          __syncthreads();
          const int m = Nr - k;
          for (int i = tid; i < m * nq; i += nth) {
            const int r = k + i % m, q = i / m;
            X[r + q * R] -= (r == k ? 1.0 : A[r + k * ld]) * s_w[q];
          }
          __syncthreads();
        }
      }
    }
    // R^{-1} (or U^{-1}), bottom up
    for (int c = method == kLastSVD ? -1 : Nc - 1; c >= 0; --c) {
      const double uinv = 1.0 / A[c + c * ld];
      for (int i = tid; i < c * nq; i += nth) {
        const int r = i % c, q = i / c;
        X[r + q * R] -= A[r + c * ld] * (X[c + q * R] * uinv);
      }
      __syncthreads();
      for (int q = tid; q < nq; q += nth) X[c + q * R] *= uinv;
      __syncthreads();
    }
    const double* Y = X;
    int ldy = R;
    if (method == kLastLUPQ) {
      for (int q = tid; q < nq; q += nth)
        for (int c = Nc - 1; c >= 0; --c) {
          const int pv = a.Q[c];
          if (pv != c) { const double t = X[c + q * R]; X[c + q * R] = X[pv + q * R]; X[pv + q * R] = t; }
        }
      __syncthreads();
    } else if (method == kLastQRP) {
      for (int i = tid; i < Nc * nq; i += nth) {
        const int r = i % Nc, q = i / Nc;
        Z[a.P[r] + q * Nc] = X[r + q * R];
      }
      __syncthreads();
      Y = Z;
      ldy = Nc;
    }
    for (int i = tid; i < Nc * nq; i += nth) {
      const int r = i % Nc, q = i / Nc;
      size_t row;
      if (r < n) row = r;
      else if (r < 2 * n) row = xN + (r - n);
      else row = size_t(N + 1) * n + (r - 2 * n);
      a.x[row + size_t(q0 + q) * ldx] = TX(Y[r + q * ldy]);
    }
    __syncthreads();
  }
}

template <typename TX, bool A_LDS>
__global__ void __launch_bounds__(1024) last_solve_kernel(LastSolveArgs<TX> a) {
  last_solve_body<TX, A_LDS>(a);
}

// ---- batched: one workgroup per system ------------------------------------
template <typename TW, typename TA>
__global__ void __launch_bounds__(256) assemble_last_batched(const AssembleArgs<TW, TA>* args) {
  assemble_last_body<TW, TA>(args[blockIdx.x], threadIdx.x, blockDim.x);
}

__global__ void __launch_bounds__(1024) lu_last_batched(const LastSolveArgs<double>* args, int32_t* const* status) {
  const LastSolveArgs<double>& a = args[blockIdx.x];
  lu_last_body(const_cast<double*>(a.Hm), a.Nc, const_cast<int32_t*>(a.P), status[blockIdx.x]);
}

template <typename TX, bool A_LDS>
__global__ void __launch_bounds__(1024) last_solve_batched(const LastSolveArgs<TX>* args) {
  if (skipped(args[blockIdx.x].skip)) return;
  last_solve_body<TX, A_LDS>(args[blockIdx.x]);
}

// one wavefront per system (see last_solve_lu_wave_body)
template <typename TX, int RPL>
__global__ void __launch_bounds__(64) last_solve_lu_wave_batched(const LastSolveArgs<TX>* args) {
  const LastSolveArgs<TX>& a = args[blockIdx.x];
  if (skipped(a.skip)) return;
  last_solve_lu_wave_body<TX, RPL>(a, a.x, threadIdx.x);
}

// one system, one wavefront per right-hand side
template <typename TX, int RPL>
__global__ void __launch_bounds__(64) last_solve_lu_wave(LastSolveArgs<TX> a) {
  last_solve_lu_wave_body<TX, RPL>(a, a.x + size_t(blockIdx.x) * a.ldx, threadIdx.x);
}

template <typename TW, typename TA>
hipError_t launch_assemble_last_batched(const AssembleArgs<TW, TA>* args, int nsys, hipStream_t st) {
  hipLaunchKernelGGL((assemble_last_batched<TW, TA>), dim3(nsys), dim3(256), 0, st, args);
  return hipGetLastError();
}

template <int RPL, int NWV>
__global__ void __launch_bounds__(64 * NWV) lu_last_regs_batched(const LastSolveArgs<double>* args,
                                                                 int32_t* const* status) {
  __shared__ LastLuLds<RPL> sm;
  const LastSolveArgs<double>& a = args[blockIdx.x];
  const int w = NWV == 1 ? 0 : __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6));
  lu_last_regs_body<RPL, NWV, (RPL < 3)>(const_cast<double*>(a.Hm), a.Nc, const_cast<int32_t*>(a.P), status[blockIdx.x], w,
                              threadIdx.x & 63, sm);
}

template <int RPL, int NWV>
__global__ void __launch_bounds__(64 * NWV) lu_last_regs(double* Hm, int Nc, int32_t* ipiv, int32_t* status) {
  __shared__ LastLuLds<RPL> sm;
  lu_last_regs_body<RPL, NWV, false>(Hm, Nc, ipiv, status, __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)),
                              threadIdx.x & 63, sm);
}

// args[s].Hm / .P (ipiv) / .Nc describe the square last block of system s;
// Ncmax is the largest of the launch
hipError_t launch_lu_last_batched(const LastSolveArgs<double>* args, int32_t* const* status, int nsys, int Ncmax,
                                  hipStream_t st) {
  if (Ncmax <= 64) {
    hipLaunchKernelGGL((lu_last_regs_batched<1, 1>), dim3(nsys), dim3(64), 0, st, args, status);
    return hipGetLastError();
  }
  if (Ncmax > 128 && Ncmax <= 192) {
    hipLaunchKernelGGL((lu_last_regs_batched<3, 12>), dim3(nsys), dim3(768), 0, st, args, status);
    return hipGetLastError();
  }
  if (Ncmax <= 128) {
    hipLaunchKernelGGL((lu_last_regs_batched<2, 4>), dim3(nsys), dim3(256), 0, st, args, status);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(lu_last_batched, dim3(nsys), dim3(1024), 0, st, args, status);
  return hipGetLastError();
}

// LDS of the last solve beside the factored block: the columns X and Z, and
// the products of a reflector
static size_t last_solve_bytes(int Nr, int Nc) {
  return (size_t(Nr > Nc ? Nr : Nc) + Nc + 1) * 16 * sizeof(double);
}

template <typename TX>
hipError_t launch_last_solve_batched(const LastSolveArgs<TX>* args, int nsys, int Nrmax, int Ncmax, size_t lds_limit,
                                     hipStream_t st) {
  const size_t xbytes = last_solve_bytes(Nrmax, Ncmax);
  const size_t bytes = size_t(Nrmax) * Ncmax * sizeof(double) + xbytes;
  if (xbytes > lds_limit) return hipErrorInvalidConfiguration;
  if (bytes <= lds_limit)
    hipLaunchKernelGGL((last_solve_batched<TX, true>), dim3(nsys), dim3(1024), bytes, st, args);
  else
    hipLaunchKernelGGL((last_solve_batched<TX, false>), dim3(nsys), dim3(1024), xbytes, st, args);
  return hipGetLastError();
}

template hipError_t launch_assemble_last_batched<float, double>(const AssembleArgs<float, double>*, int, hipStream_t);
template hipError_t launch_assemble_last_batched<double, double>(const AssembleArgs<double, double>*, int, hipStream_t);
template hipError_t launch_last_solve_batched<double>(const LastSolveArgs<double>*, int, int, int, size_t, hipStream_t);
// the wavefront LU solve above, for square last blocks with Nc <= 256 solved
// by LU for one right-hand side; false when it does not apply
template <typename TX>
bool launch_last_solve_lu_wave_batched(const LastSolveArgs<TX>* args, int nsys, int Ncmax, hipStream_t st,
                                       hipError_t* err) {
  if (Ncmax < 1 || Ncmax > 256) return false;
  if (Ncmax <= 64) hipLaunchKernelGGL((last_solve_lu_wave_batched<TX, 1>), dim3(nsys), dim3(64), 0, st, args);
  else if (Ncmax <= 128) hipLaunchKernelGGL((last_solve_lu_wave_batched<TX, 2>), dim3(nsys), dim3(64), 0, st, args);
  else hipLaunchKernelGGL((last_solve_lu_wave_batched<TX, 4>), dim3(nsys), dim3(64), 0, st, args);
  *err = hipGetLastError();
  return true;
}
template bool launch_last_solve_lu_wave_batched<double>(const LastSolveArgs<double>*, int, int, hipStream_t,
                                                        hipError_t*);


template <typename TW, typename TA>
hipError_t launch_assemble_last(AssembleArgs<TW, TA> const& a, hipStream_t st) {
  const int blocks = (a.Nr * a.Nc + 255) / 256;   // one element per thread
  hipLaunchKernelGGL((assemble_last_kernel<TW, TA>), dim3(blocks < 1 ? 1 : blocks), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_lu_last(double* Hm, int Nc, int32_t* ipiv, int32_t* status, hipStream_t st) {
  if (Nc <= 192) {   // in registers, 16 columns per wavefront
    if (Nc <= 64) hipLaunchKernelGGL((lu_last_regs<1, 4>), dim3(1), dim3(256), 0, st, Hm, Nc, ipiv, status);
    else if (Nc <= 128) hipLaunchKernelGGL((lu_last_regs<2, 8>), dim3(1), dim3(512), 0, st, Hm, Nc, ipiv, status);
    else hipLaunchKernelGGL((lu_last_regs<3, 12>), dim3(1), dim3(768), 0, st, Hm, Nc, ipiv, status);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(lu_last_kernel, dim3(1), dim3(1024), 0, st, Hm, Nc, ipiv, status);
  return hipGetLastError();
}

template <typename TX>
hipError_t launch_last_solve(LastSolveArgs<TX> const& a, size_t lds_limit, hipStream_t st) {
  // LU, square, no second solver behind it: one wavefront per right-hand side
  if (a.method == kLastLU && a.status == nullptr && a.Nr == a.Nc && a.Nc <= 256) {
    if (a.Nc <= 64) hipLaunchKernelGGL((last_solve_lu_wave<TX, 1>), dim3(a.nrhs), dim3(64), 0, st, a);
    else if (a.Nc <= 128) hipLaunchKernelGGL((last_solve_lu_wave<TX, 2>), dim3(a.nrhs), dim3(64), 0, st, a);
    else hipLaunchKernelGGL((last_solve_lu_wave<TX, 4>), dim3(a.nrhs), dim3(64), 0, st, a);
    return hipGetLastError();
  }
  const size_t xbytes = last_solve_bytes(a.Nr, a.Nc);
  const size_t bytes = size_t(a.Nr) * a.Nc * sizeof(double) + xbytes;
  if (xbytes > lds_limit) return hipErrorInvalidConfiguration;
  if (bytes <= lds_limit)
    hipLaunchKernelGGL((last_solve_kernel<TX, true>), dim3(1), dim3(1024), bytes, st, a);
  else
    hipLaunchKernelGGL((last_solve_kernel<TX, false>), dim3(1), dim3(1024), xbytes, st, a);
  return hipGetLastError();
}

template hipError_t launch_assemble_last<double, double>(AssembleArgs<double, double> const&, hipStream_t);
template hipError_t launch_assemble_last<float, float>(AssembleArgs<float, float> const&, hipStream_t);
template hipError_t launch_assemble_last<float, double>(AssembleArgs<float, double> const&, hipStream_t);
template hipError_t launch_last_solve<double>(LastSolveArgs<double> const&, size_t, hipStream_t);
template hipError_t launch_last_solve<float>(LastSolveArgs<float> const&, size_t, hipStream_t);

}  // namespace bcr
