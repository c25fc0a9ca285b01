// Device bodies of the bordered last block shared by the single-system, the
// batched and the fused small-system kernels (see bcr_last.hip).
#pragma once
#include "bcr_launch.hh"
#include "bcr_wave.hh"

namespace bcr {

template <typename TW, typename TA>
__device__ __forceinline__ void assemble_last_body(AssembleArgs<TW, TA> const& a, int tid, int nth) {
  const int n = a.n, Nr = a.Nr, Nc = a.Nc, qr = a.qr, qx = a.qx, nr = a.nr, nx = a.nx;
  const size_t rn = size_t(nr) * n;
  for (int i = tid; i < Nr * Nc; i += nth) {
    const int r = i % Nr, c = i / Nr;
    double v = 0;
    if (r < n) {
      if (c < n) v = double(a.D0[r + c * n]);
      else if (c < 2 * n) v = double(a.E0[r + (c - n) * n]);
      else if (c >= 2 * n + qx) v = double(a.B0[r + (c - 2 * n - qx) * n]);
    } else if (r < 2 * n + qr) {
      v = double(a.H[(r - n) + size_t(c) * (n + qr)]);
    } else {
      const int rr = r - 2 * n - qr;
      if (c < n) {
        v = double(a.C[rr + c * nr]);
      } else if (c < 2 * n) {
        const size_t off = size_t(a.N) * rn + rr + (c - n) * nr;
        v = double(a.C[off]) + double(a.Cpend[off]) + double(a.Cpend[size_t(a.N + 1) * rn + off]);
      } else if (c < 2 * n + qx) {
        v = double(a.Cq[rr + (c - 2 * n) * nr]);
      } else {
        v = a.Feff[rr + (c - 2 * n - qx) * nr];
      }
    }
    a.Hm[i] = v;
  }
}

// The LU factorization of a square last block (Nc <= 64 RPL) by NWV
// wavefronts of one workgroup with the block in registers: wavefront w holds
// columns [CW w, CW w + CW) of every row (lane l: rows l + 64 k).  Rows stay
// in their lanes with their current positions tracked (the pivot row takes
// position c, the row there the pivot's old place); the wavefront owning
// column c searches it (largest |a|, ties to the smaller position, as
// lu_last_body's scan) and publishes the multipliers through LDS, and every
// wavefront applies the rank-1 update to its columns after c.  The rows are
// stored back in their final positions with the 1-based ipiv, so the result
// and its arithmetic per element are lu_last_body's.
//
// The chain of a step bounds it: search, reciprocal, LDS, barrier, update of
// the wave's columns.  Every lane forms the reciprocal of its own candidate
// beside the search; for one system alone (few workgroups) a wave holds 16
// columns only (NWV = 4 RPL), which shortens the update and lets the column
// blocks share one copy of the step's code.  Wavefronts beyond NWV of a
// larger workgroup take part in the barriers only.
template <int RPL>
struct LastLuLds {
  double l[2][64 * RPL];
  int piv[2][2];
};

// A NaN is not a candidate (a column of NaN and zeros has a zero pivot); with
// nothing but NaNs left the row at c stays and no zero pivot is reported.
// NANZERO: a NaN ranks as a zero, and a column of NaNs counts as a zero pivot
// (the batched LU's answer).
template <int RPL, int NWV, bool NANZERO>
__device__ __forceinline__ void lu_last_regs_body(double* Hm, int Nc, int32_t* ipiv, int32_t* st, int w, int lane,
                                                  LastLuLds<RPL>& sm) {
  using V16d = double __attribute__((ext_vector_type(16)));
  constexpr int CW = 64 * RPL / NWV, CB = CW / 16;   // columns and 16-column blocks per wavefront
  static_assert(CW * NWV == 64 * RPL && CW % 16 == 0, "the waves cover the columns in 16-column blocks");
  if (NWV > 1 && w >= NWV) {
    for (int c = 0; c < Nc; ++c) __syncthreads();
    return;
  }
  V16d V[RPL][CB];
  int pos[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    pos[k] = r;
#pragma unroll
    for (int jj = 0; jj < CW; ++jj) {
      const int gj = CW * w + jj;
      const double v = Hm[(r < Nc ? r : 0) + size_t(gj < Nc ? gj : 0) * Nc];
      V[k][jj / 16][jj % 16] = keep_if(v, r < Nc && gj < Nc);
    }
  }
  // steps of column block gb (owner wave o, its block lb): rolled, the column
  // read through a uniform register index
  auto block = [&](const int gb, const int o, const int lb) {
    const int cend = min(16 * gb + 16, Nc);
    for (int c = 16 * gb; c < cend; ++c) {
      const int cc = c - 16 * gb;
      double lk[RPL];
      int who = 0, ps = 0, P = 0;
      if (w == o) {
        double x[RPL];
        bool cb = false;
        unsigned hb = 0, lbits = 0;
        int pb = 0, kb = 0;
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          x[k] = V[k][lb][cc];
          unsigned h, l;
          wave::abs_key(x[k], h, l);
          if (x[k] != x[k]) h = l = 0;   // a NaN is never preferred
          const bool cand = pos[k] >= c && lane + 64 * k < Nc && (NANZERO || x[k] == x[k]);
          const bool better = cand && (!cb || h > hb || (h == hb && (l > lbits || (l == lbits && pos[k] < pb))));
          if (better) {
            cb = true;
            hb = h;
            lbits = l;
            pb = pos[k];
            kb = k;
          }
        }
        if (!NANZERO && __ballot(cb) == 0) {   // only NaNs
#pragma unroll
          for (int k = 0; k < RPL; ++k)
            if (pos[k] == c) {
              cb = true;
              pb = c;
              kb = k;
            }
        }
        double xs = x[0];
#pragma unroll
        for (int k = 1; k < RPL; ++k) xs = kb == k ? x[k] : xs;
        const double rown = xs != 0.0 ? 1.0 / xs : 0.0;   // beside the search
        bool zero;
        who = wave::argmax_pos<true>(cb, hb, lbits, pb, lane, zero);
        P = __builtin_amdgcn_readlane(pb, who);
        ps = __builtin_amdgcn_readlane(kb, who);
        const double rinv = wave::rl(rown, who);
        const bool pz = wave::rl(xs, who) == 0.0;
        if (lane == 0) {
          if (zero && (NANZERO || pz)) atomicOr(st, 2);
          ipiv[c] = P + 1;
        }
#pragma unroll
        for (int k = 0; k < RPL; ++k) {
          const int np = pos[k] == c ? P : pos[k] == P ? c : pos[k];
          const bool below = np > c && lane + 64 * k < Nc;
          const double m = x[k] * rinv;
          lk[k] = below ? m : 0.0;
          V[k][lb][cc] = below ? m : x[k];
          if constexpr (NWV > 1) sm.l[c & 1][lane + 64 * k] = lk[k];
        }
        if (NWV > 1 && lane == 0) {
          sm.piv[c & 1][0] = who | (ps << 8);
          sm.piv[c & 1][1] = P;
        }
      }
      if constexpr (NWV > 1) {
        __syncthreads();
        if (w != o) {
          const int q = __builtin_amdgcn_readfirstlane(sm.piv[c & 1][0]);
          who = q & 255;
          ps = q >> 8;
          P = __builtin_amdgcn_readfirstlane(sm.piv[c & 1][1]);
#pragma unroll
          for (int k = 0; k < RPL; ++k) lk[k] = sm.l[c & 1][lane + 64 * k];
        }
      }
#pragma unroll
      for (int k = 0; k < RPL; ++k) pos[k] = pos[k] == c ? P : pos[k] == P ? c : pos[k];
      // this wavefront's columns after c: A[r][j] -= l_r * A[c][j]
      if (CW * w + CW - 1 > c) {
#pragma unroll
        for (int jj = 0; jj < CW; ++jj) {
          if (CW * w + jj > c) {
            double v = V[0][jj / 16][jj % 16];
#pragma unroll
            for (int k = 1; k < RPL; ++k) v = ps == k ? V[k][jj / 16][jj % 16] : v;
            const double u = wave::rl(v, who);
#pragma unroll
            for (int k = 0; k < RPL; ++k) V[k][jj / 16][jj % 16] -= lk[k] * u;
          }
        }
      }
    }
  };
  if constexpr (CB == 1) {
#pragma unroll 1
    for (int gb = 0; gb < 4 * RPL; ++gb) block(gb, gb, 0);
  } else {   // the owning wavefront's block is compile-time per block
#pragma unroll
    for (int gb = 0; gb < 4 * RPL; ++gb) block(gb, 16 * gb / CW, (16 * gb % CW) / 16);
  }
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    if (lane + 64 * k < Nc) {
#pragma unroll
      for (int jj = 0; jj < CW; ++jj) {
        const int gj = CW * w + jj;
        if (gj < Nc) Hm[pos[k] + size_t(gj) * Nc] = V[k][jj / 16][jj % 16];
      }
    }
  }
}

// The LU solve of a square last block (Nc <= 64 RPL) for one right-hand side
// by one wavefront: lane l holds rows l + 64 k (k < RPL) of y, the row
// interchanges are composed into a source row per lane (no serial swaps),
// and the two substitutions walk the columns of the factors from HBM/L2
// eight at a time (the next eight in flight) with y[c] broadcast by
// v_readlane, without a workgroup barrier.  Same arithmetic per element as
// last_solve_body's LU path.
template <typename TX, int RPL>
__device__ __forceinline__ void last_solve_lu_wave_body(LastSolveArgs<TX> const& a, TX* const x, int lane) {
  constexpr int CH = 8;
  const int n = a.n, Nc = a.Nc, ld = a.Nr;
  const double* A = a.Hm;
  const size_t xN = size_t(a.N) * n, xC = size_t(a.N + 1) * n + a.qr;
  // the source row of each row after the interchanges c = 0 .. Nc-1
  // (1-based ipiv), found by undoing them from the last
  int pos[RPL], pv[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    pos[k] = lane + 64 * k;
    pv[k] = a.P[min(lane + 64 * k, Nc - 1)] - 1;
  }
#pragma unroll
  for (int kc = RPL - 1; kc >= 0; --kc)
    for (int c = min(64 * kc + 63, Nc - 1); c >= 64 * kc; --c) {
      const int q = __builtin_amdgcn_readlane(pv[kc], c - 64 * kc);
#pragma unroll
      for (int k = 0; k < RPL; ++k) pos[k] = pos[k] == c ? q : pos[k] == q ? c : pos[k];
    }
  double y[RPL], dinv[RPL];
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k, s = r < Nc ? pos[k] : 0;
    const size_t row = s < n ? size_t(s) : s < 2 * n + a.qr ? xN + (s - n) : xC + (s - 2 * n - a.qr);
    y[k] = keep_if(double(x[row]), r < Nc);
    dinv[k] = 1.0 / (r < Nc ? A[r + size_t(r) * ld] : 1.0);
  }
  // y <- L^{-1} y (unit lower), column c of L below the diagonal
  auto load = [&](double (&l)[CH][RPL], int c0, int dir) {
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
      for (int k = 0; k < RPL; ++k) {
        const int c = max(min(c0 + dir * i, Nc - 1), 0), r = lane + 64 * k;
        l[i][k] = A[(r < Nc ? r : 0) + size_t(c) * ld];
      }
  };
  double nxt[CH][RPL];
  load(nxt, 0, 1);
#pragma unroll
  for (int kc = 0; kc < RPL; ++kc) {
    const int cend = min(64 * kc + 64, Nc);
    for (int c0 = 64 * kc; c0 < cend; c0 += CH) {
      double l[CH][RPL];
#pragma unroll
      for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int k = 0; k < RPL; ++k) l[i][k] = nxt[i][k];
      load(nxt, c0 + CH, 1);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int c = c0 + i;
        if (c < cend) {
          const double yc = wave::rl(y[kc], c - 64 * kc);
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const int r = lane + 64 * k;
            if (r > c && r < Nc) y[k] -= l[i][k] * yc;
          }
        }
      }
    }
  }
  // y <- U^{-1} y, bottom up: y_c = y_c / u_cc, then the rows above
  load(nxt, Nc - 1, -1);
#pragma unroll
  for (int kc = RPL - 1; kc >= 0; --kc) {
    const int cbeg = 64 * kc;
    for (int c1 = min(64 * kc + 63, Nc - 1); c1 >= cbeg; c1 -= CH) {
      double u[CH][RPL];
#pragma unroll
      for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int k = 0; k < RPL; ++k) u[i][k] = nxt[i][k];
      // the chunk after this one (the next 64-column part starts at its top)
      load(nxt, max(c1 - CH, cbeg - 1), -1);
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        const int c = c1 - i;
        if (c >= cbeg) {
          const double xc = wave::rl(y[kc] * dinv[kc], c - 64 * kc);
#pragma unroll
          for (int k = 0; k < RPL; ++k) {
            const int r = lane + 64 * k;
            y[k] = r < c ? y[k] - u[i][k] * xc : r == c ? xc : y[k];
          }
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < RPL; ++k) {
    const int r = lane + 64 * k;
    if (r < Nc) {
      const size_t row = r < n ? size_t(r) : r < 2 * n ? xN + (r - n) : size_t(a.N + 1) * n + (r - 2 * n);
      x[row] = TX(y[k]);
    }
  }
}

}  // namespace bcr
