// Dense local solve in registers: the micro matrix of a local linear system
// of at most 64 unknowns (96 with eight waves) is assembled straight into
// registers and solved by LU with partial pivoting, one workgroup.
//
// What bounds it: N dependent elimination steps.  Lane = matrix row (two rows
// past 64), each wave a block of CB columns in registers, so a step is one
// LDS exchange of the pivot column and one barrier; every wave then finds the
// pivot itself and takes its row's entries by lane reads.  Rows are not
// swapped: a row that has been a pivot keeps its place and its step number.
// The operations on every entry are those of the global-memory LU
// (wg_lu_solve), which read and wrote the matrix in L2 with four barriers a
// step: a sweep of local solves of 64 unknowns (rank 4, n = 4) spent 225 us on
// each position there, 73 us here, everything else in the position included.
#pragma once
#include "ttals_dev.hpp"

namespace ttals {

constexpr int LU_MAX = 96;
// the register form's largest system: with four waves 96 unknowns would take
// 24 columns of two rows per lane (280 registers, 116 KB of unrolled code:
// one workgroup per CU instead of two)
constexpr int LU_REG_MAX = NWAVE == 8 ? LU_MAX : 64;
constexpr int LU_SCRATCH = 4 * 64 + LU_MAX + 2 * 64;  // pivot columns (two steps in turn), solution, rhs hand-over

// Does the local system take the register form: size, and its operator pieces
// and scratch in `cap` doubles of LDS
__host__ __device__ __forceinline__ bool lu_reg_fits(int a, int P, int n, int Q, int b, long cap) {
  return a * n * b <= LU_REG_MAX &&
         (long)a * P * a + (long)P * n * n * Q + (long)b * Q * b + LU_SCRATCH <= cap;
}

// M v = f with M as micro_dense builds it (rows (a', m, b'), cols (a, n, b)),
// N = a n b <= RH * 64 and <= NWAVE * CB.  L, A, R, f, v global; lds as
// lu_reg_fits counts it.  Returns false (v untouched) on an exactly zero pivot.
template <int CB, int RH>
__device__ __attribute__((noinline)) bool lu_reg_run(int a_, int P_, int n_, int Q_, int b_, const double* L,
                                                     const double* A, const double* R, const double* f, double* v,
                                                     double* lds_) {
  const int a = __builtin_amdgcn_readfirstlane(a_), P = __builtin_amdgcn_readfirstlane(P_);
  const int n = __builtin_amdgcn_readfirstlane(n_), Q = __builtin_amdgcn_readfirstlane(Q_);
  const int b = __builtin_amdgcn_readfirstlane(b_);
  const int N = a * n * b, nb = n * b;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  TT_LDS double* cols = (TT_LDS double*)lds_;
  TT_LDS double* xs = cols + 4 * 64;
  TT_LDS double* yb = xs + LU_MAX;
  TT_LDS double* Ls = yb + 2 * 64;
  TT_LDS double* As = Ls + a * P * a;
  TT_LDS double* Rs = As + P * n * n * Q;
  __syncthreads();
  for (int e = threadIdx.x; e < a * P * a; e += NT) Ls[e] = L[e];
  for (int e = threadIdx.x; e < P * n * n * Q; e += NT) As[e] = A[e];
  for (int e = threadIdx.x; e < b * Q * b; e += NT) Rs[e] = R[e];
  double M[RH][CB], y[RH];
  int a2[RH], m2[RH], b2[RH];
#pragma unroll
  for (int h = 0; h < RH; ++h) {
    const int r = min(lane + 64 * h, N - 1);
    a2[h] = r / nb;
    m2[h] = (r - a2[h] * nb) / b;
    b2[h] = r - a2[h] * nb - m2[h] * b;
    y[h] = f[r];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < CB; ++q) {
    const int j = w * CB + q;
#pragma unroll
    for (int h = 0; h < RH; ++h) M[h][q] = 0.0;
    if (j < N) {
      const int a1 = j / nb, nn = (j - a1 * nb) / b, b1 = j - a1 * nb - nn * b;
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int h = 0; h < RH; ++h) {
          const double l = Ls[(a1 * P + p) * a + a2[h]];
          if (l == 0.0) continue;
          const TT_LDS double* ap = As + ((p * n + m2[h]) * n + nn) * Q;
          const TT_LDS double* rp = Rs + b1 * Q * b + b2[h];
          for (int qq = 0; qq < Q; ++qq) M[h][q] += l * ap[qq] * rp[qq * b];
        }
    }
  }
  bool used[RH];
  int ord[RH];  // the step a row was pivot of
#pragma unroll
  for (int h = 0; h < RH; ++h) {
    used[h] = lane + 64 * h >= N;
    ord[h] = 1 << 30;
  }
  bool ok = true;
  for (int wo = 0; wo < NWAVE && ok; ++wo) {
    static_for<0, CB>([&](auto Qc) {
      constexpr int q = decltype(Qc)::value;
      const int k = wo * CB + q;
      if (k >= N || !ok) return;
      TT_LDS double* col = cols + (k & 1) * 128;
      if (w == wo) {
#pragma unroll
        for (int h = 0; h < RH; ++h) col[64 * h + lane] = M[h][q];
      }
      __syncthreads();
      double c[RH], mx = -1.0;
#pragma unroll
      for (int h = 0; h < RH; ++h) {
        c[h] = col[64 * h + lane];
        if (!used[h]) mx = fmax(mx, fabs(c[h]));
      }
      mx = wave_max(mx);
      if (mx == 0.0) {
        ok = false;
        return;
      }
      // the pivot: the first row of the largest magnitude (a column of NaN: the first free row)
      int p = -1;
#pragma unroll
      for (int h = 0; h < RH; ++h) {
        const unsigned long long hit = __ballot(!used[h] && fabs(c[h]) == mx);
        if (p < 0 && hit) p = 64 * h + (int)__builtin_ctzll(hit);
      }
#pragma unroll
      for (int h = 0; h < RH; ++h) {
        const unsigned long long hit = __ballot(!used[h]);
        if (p < 0 && hit) p = 64 * h + (int)__builtin_ctzll(hit);
      }
      p = __builtin_amdgcn_readfirstlane(p);
      const bool top = RH == 2 && p >= 64;
      const int pl = p & 63;
      auto row = [&](double lo, double hi) { return rdlane(top ? hi : lo, pl); };
      const double inv = 1.0 / row(c[0], c[RH - 1]);
      double l[RH];
#pragma unroll
      for (int h = 0; h < RH; ++h) {
        const bool piv = lane + 64 * h == p;
        l[h] = (used[h] || piv) ? 0.0 : c[h] * inv;
        if (piv) {
          used[h] = true;
          ord[h] = k;
        }
      }
      const double yp = row(y[0], y[RH - 1]);
#pragma unroll
      for (int h = 0; h < RH; ++h) y[h] -= l[h] * yp;
      if (w > wo) {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          const double rp = row(M[0][j], M[RH - 1][j]);
#pragma unroll
          for (int h = 0; h < RH; ++h) M[h][j] -= l[h] * rp;
        }
      } else if (w == wo) {
#pragma unroll
        for (int j = q + 1; j < CB; ++j) {
          const double rp = row(M[0][j], M[RH - 1][j]);
#pragma unroll
          for (int h = 0; h < RH; ++h) M[h][j] -= l[h] * rp;
        }
      }
    });
  }
  if (!ok) return false;
  // back substitution: the columns from the last, the right-hand side handed
  // from wave to wave
  for (int wo = NWAVE - 1; wo >= 0; --wo) {
    if (w == wo && wo * CB < N) {
      if (wo < NWAVE - 1 && (wo + 1) * CB < N) {
#pragma unroll
        for (int h = 0; h < RH; ++h) y[h] = yb[64 * h + lane];
      }
      static_for<0, CB>([&](auto Qc) {
        constexpr int q = CB - 1 - decltype(Qc)::value;
        const int k = wo * CB + q;
        if (k >= N) return;
        int p = 0;
#pragma unroll
        for (int h = 0; h < RH; ++h) {
          const unsigned long long hit = __ballot(ord[h] == k);
          if (hit) p = 64 * h + (int)__builtin_ctzll(hit);
        }
        p = __builtin_amdgcn_readfirstlane(p);
        const bool top = RH == 2 && p >= 64;
        const int pl = p & 63;
        const double x = rdlane(top ? y[RH - 1] : y[0], pl) / rdlane(top ? M[RH - 1][q] : M[0][q], pl);
        if (lane == 0) xs[k] = x;
#pragma unroll
        for (int h = 0; h < RH; ++h)
          if (ord[h] < k) y[h] -= M[h][q] * x;
      });
#pragma unroll
      for (int h = 0; h < RH; ++h) yb[64 * h + lane] = y[h];
    }
    __syncthreads();
  }
  for (int k = threadIdx.x; k < N; k += NT) v[k] = xs[k];
  __syncthreads();
  return true;
}

__device__ __forceinline__ bool lu_reg_solve(int a, int P, int n, int Q, int b, const double* L, const double* A,
                                             const double* R, const double* f, double* v, double* lds) {
  const int N = a * n * b;
  if (N <= 32) return lu_reg_run<32 / NWAVE, 1>(a, P, n, Q, b, L, A, R, f, v, lds);
  if constexpr (LU_REG_MAX > 64) {
    if (N > 64) return lu_reg_run<LU_REG_MAX / NWAVE, 2>(a, P, n, Q, b, L, A, R, f, v, lds);
  }
  return lu_reg_run<64 / NWAVE, 1>(a, P, n, Q, b, L, A, R, f, v, lds);
}

}  // namespace ttals
