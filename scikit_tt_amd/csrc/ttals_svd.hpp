// One-sided (Hestenes) Jacobi SVD of a small matrix held in LDS.
//
// The method of wg_jacobi_svd (same pairing, the same rotations up to rounding,
// the same convergence test, here safe from underflow), reorganised: B and the
// accumulated rotations V sit in LDS by columns (odd stride), a pair of columns
// takes L lanes (8 to 64) with its entries in registers between the dot
// products and the rotation, and all pairs of a round run at once.  A round is
// then bound by the LDS traffic of B and V and one barrier instead of by global
// memory latency per column element, and the final sort counts ranks in
// parallel instead of selecting on one thread.
// An 80 x 80 triangular factor of a rounding sweep: 5.5 ms in global memory
// with one wave per pair, 0.8 ms here; one root and one division a rotation
// then took a 64 x 64 one from 1.00 to 0.73 ms.
#pragma once
#include "ttals_dev.hpp"
#include "ttals_qr.hpp"

namespace ttals {

constexpr int JS_ROWS = 12;  // entries of a column per lane

__host__ __device__ __forceinline__ long js_doubles(int c, int k) { return (long)k * (c | 1) + (long)k * (k | 1) + k; }
// fits `cap` doubles of LDS, and a column fits 64 lanes
__device__ __forceinline__ bool js_fits(int c, int k, long cap) {
  return js_doubles(c, k) <= cap && c <= 64 * JS_ROWS && k <= 64 * JS_ROWS;
}

// sum over groups of L neighbouring lanes, in every lane of the group
__device__ __forceinline__ double lanes_sum(double v, int L) {
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0x141>(v);
  if (L >= 16) v += dpp_mov<0x140>(v);
  if (L >= 32) v += __shfl_xor(v, 16, 64);
  if (L >= 64) v += __shfl_xor(v, 32, 64);
  return v;
}

// Factors of up to JS_ONE columns and rows are one wave's work: the barriers of
// eight waves cost more than the rotations (truncated_svd of an 8 x 8 matrix:
// 108 us with eight waves, 80 us with one, the same bits).
constexpr int JS_ONE = 16;
// a barrier of the working threads: the workgroup, or (ONE) the first wave alone
template <bool ONE>
__device__ __forceinline__ void js_sync() {
  if constexpr (ONE) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// Sweeps of rotations over all column pairs of Bl (k columns, c rows, ld lb)
// and Vl (k rows, ld lv) until a sweep rotates nothing (at most 60): RM entries
// of a column per lane, L lanes per pair (RM * L >= c, k).
template <int RM, bool ONE>
__device__ __forceinline__ void js_sweeps(TT_LDS double* Bl, TT_LDS double* Vl, int c, int k, int lb, int lv, int L,
                                          int* s_rot) {
  const int kk = (k & 1) ? k + 1 : k, pairs = kk / 2, mod = kk - 1;
  const int l = threadIdx.x & (L - 1), g = threadIdx.x / L, ng = (ONE ? 64 : NT) / L;
  for (int sweep = 0; sweep < 60; ++sweep) {
    const int flag = sweep & 1;
    for (int round = 0; round < mod; ++round) {
      for (int pr = g; pr < pairs; pr += ng) {
        // round-robin: position 0 fixed, the others rotate
        int p0 = pr - 1 + round, p1 = kk - 2 - pr + round;
        if (p0 >= mod) p0 -= mod;
        if (p1 >= mod) p1 -= mod;
        p0 = pr == 0 ? 0 : 1 + p0;
        p1 = 1 + p1;
        const int i = p0 < p1 ? p0 : p1, j = p0 < p1 ? p1 : p0;
        if (j >= k) continue;  // dummy partner
        TT_LDS double *ci = Bl + i * lb, *cj = Bl + j * lb, *wi = Vl + i * lv, *wj = Vl + j * lv;
        // the entries of V travel with those of B: their latency is off the chain
        double bi[RM], bj[RM], vi[RM], vj[RM];
#pragma unroll
        for (int u = 0; u < RM; ++u) {
          const int r = l + u * L;
          bi[u] = r < c ? ci[r] : 0.0;
          bj[u] = r < c ? cj[r] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < RM; ++u) {
          const int r = l + u * L;
          vi[u] = r < k ? wi[r] : 0.0;
          vj[u] = r < k ? wj[r] : 0.0;
        }
        double aii = 0.0, ajj = 0.0, aij = 0.0;
#pragma unroll
        for (int u = 0; u < RM; ++u) {
          aii = fma(bi[u], bi[u], aii);
          ajj = fma(bj[u], bj[u], ajj);
          aij = fma(bi[u], bj[u], aij);
        }
        aii = lanes_sum(aii, L);
        ajj = lanes_sum(ajj, L);
        aij = lanes_sum(aij, L);
        // the rotation depends on the ratios of the three sums alone: where a product of them could leave the range
        // of a double (columns some 1e-70 below the largest), an exact power of two takes them near 1
        double prod = aii * ajj;
        if (__builtin_expect(__any(prod < 0x1p-900), 0)) {
          const int e = -__builtin_amdgcn_frexp_exp(fmax(aii, ajj));
          aii = ldexp(aii, e);
          ajj = ldexp(ajj, e);
          aij = ldexp(aij, e);
          prod = aii * ajj;
        }
        if (fabs(aij) <= 1e-15 * sqrt(prod) || aij == 0.0) continue;
        // t = sign(zeta) / (|zeta| + sqrt(1 + zeta^2)) for zeta = d / h: one root and one division
        const double d = ajj - aii, h = 2.0 * aij;
        const double t = (d >= 0.0 ? h : -h) / (fabs(d) + sqrt(fma(d, d, h * h)));
        const double cs = 1.0 / sqrt(fma(t, t, 1.0)), sn = cs * t;
#pragma unroll
        for (int u = 0; u < RM; ++u) {
          const int r = l + u * L;
          if (r < c) {
            ci[r] = cs * bi[u] - sn * bj[u];
            cj[r] = sn * bi[u] + cs * bj[u];
          }
          if (r < k) {
            wi[r] = cs * vi[u] - sn * vj[u];
            wj[r] = sn * vi[u] + cs * vj[u];
          }
        }
        if (l == 0) s_rot[flag] = 1;
      }
      js_sync<ONE>();
    }
    const int rot = s_rot[flag];
    if (threadIdx.x == 0) s_rot[flag ^ 1] = 0;
    js_sync<ONE>();
    if (rot == 0) break;
  }
}

// B (c x k, row-major, global) <- B V = U diag(sig) (orthogonal columns), V (k
// x k, row-major, global) the rotations; sig the column norms, perm the
// columns by decreasing norm.  lds: js_doubles(c, k).  B is scaled by a power
// of two (exactly) while it is worked on, so that the squares of its norms
// neither overflow nor vanish.  The work of wg_jacobi_lds between its barriers,
// by the whole workgroup or (ONE) by its first wave.
template <bool ONE>
__device__ __attribute__((noinline)) void js_run(double* B, int c_, int k_, double* V, double* sig, int* perm,
                                                 double* lds_) {
  constexpr int TH = ONE ? 64 : NT;
  __shared__ int s_rot[2];
  __shared__ double s_mx[NWAVE];
  const int c = uni(c_), k = uni(k_);
  TT_LDS double* Bl = (TT_LDS double*)lds_;
  const int lb = c | 1, lv = k | 1;
  TT_LDS double* Vl = Bl + k * lb;
  TT_LDS double* sg = Vl + k * lv;
  // the first TH entries stay in registers for the scaled copy below (all of a small factor)
  const int n = c * k;
  const double first = threadIdx.x < n ? B[threadIdx.x] : 0.0;
  double mx = fabs(first);
  for (int e = threadIdx.x + TH; e < n; e += TH) mx = fmax(mx, fabs(B[e]));
  mx = wave_max(mx);
  if ((threadIdx.x & 63) == 0) s_mx[threadIdx.x >> 6] = mx;
  if (threadIdx.x < 2) s_rot[threadIdx.x] = 0;
  for (int e = threadIdx.x; e < k * lv; e += TH) {
    const int j = e / lv, i = e - j * lv;
    Vl[e] = i == j ? 1.0 : 0.0;
  }
  js_sync<ONE>();
#pragma unroll
  for (int q = 0; q < (ONE ? 1 : NWAVE); ++q) mx = fmax(mx, s_mx[q]);
  const int ex = (mx > 0.0 && isfinite(mx)) ? -ilogb(mx) : 0;  // applied in two halves: 2^ex itself may overflow
  const double up0 = ldexp(1.0, ex / 2), up1 = ldexp(1.0, ex - ex / 2);
  const double dn0 = ldexp(1.0, -(ex / 2)), dn1 = ldexp(1.0, ex / 2 - ex);
  for (int e = threadIdx.x; e < n; e += TH) {
    const int i = e / k, j = e - i * k;
    Bl[j * lb + i] = (e < TH ? first : B[e]) * up0 * up1;
  }
  const int rows = c > k ? c : k, pairs = (k + 1) / 2;
  int L = 8;
  while (rows > L * JS_ROWS) L <<= 1;
  while (L < 64 && 2 * L * pairs <= TH) L <<= 1;
  L = ONE ? JS_ONE : __builtin_amdgcn_readfirstlane(L);  // ONE: an entry per lane, the sums of the other form
  js_sync<ONE>();
  if constexpr (ONE) {
    js_sweeps<1, true>(Bl, Vl, c, k, lb, lv, L, s_rot);
  } else {
    if (rows <= 2 * L) js_sweeps<2, false>(Bl, Vl, c, k, lb, lv, L, s_rot);
    else if (rows <= 4 * L) js_sweeps<4, false>(Bl, Vl, c, k, lb, lv, L, s_rot);
    else if (rows <= 8 * L) js_sweeps<8, false>(Bl, Vl, c, k, lb, lv, L, s_rot);
    else js_sweeps<JS_ROWS, false>(Bl, Vl, c, k, lb, lv, L, s_rot);
  }
  // column norms (a non-finite one sorts first) and ranks by decreasing norm
  for (int j = threadIdx.x; j < k; j += TH) {
    double s0 = 0.0, s1 = 0.0;
    for (int r = 0; r + 1 < c; r += 2) {
      s0 = fma(Bl[j * lb + r], Bl[j * lb + r], s0);
      s1 = fma(Bl[j * lb + r + 1], Bl[j * lb + r + 1], s1);
    }
    if (c & 1) s0 = fma(Bl[j * lb + c - 1], Bl[j * lb + c - 1], s0);
    const double s = sqrt(s0 + s1);
    sig[j] = s * dn0 * dn1;
    sg[j] = s == s ? s : INFINITY;
  }
  js_sync<ONE>();
  for (int j = threadIdx.x; j < k; j += TH) {
    const double s = sg[j];
    int rank = 0;
    for (int q = 0; q < k; ++q) rank += (sg[q] > s || (sg[q] == s && q < j)) ? 1 : 0;
    perm[rank] = j;
  }
  for (int e = threadIdx.x; e < c * k; e += TH) {
    const int i = e / k, j = e - i * k;
    B[e] = Bl[j * lb + i] * dn0 * dn1;
  }
  for (int e = threadIdx.x; e < k * k; e += TH) {
    const int i = e / k, j = e - i * k;
    V[e] = Vl[j * lv + i];
  }
}

// Starts and ends with a barrier.
__device__ void wg_jacobi_lds(double* B, int c, int k, double* V, double* sig, int* perm, double* lds) {
  __syncthreads();
  if (c > JS_ONE || k > JS_ONE) js_run<false>(B, c, k, V, sig, perm, lds);
  else if (threadIdx.x < 64) js_run<true>(B, c, k, V, sig, perm, lds);
  __syncthreads();
}

}  // namespace ttals
