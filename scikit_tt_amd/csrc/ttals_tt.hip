// TT-algebra kernels that run one workgroup of eight waves per train: norm,
// orthonormalisation / rounding, truncated SVD, residual norms.
//
// A translation unit of its own: each of these kernels has a CU to itself
// (its panels are bound by FP64 arithmetic and by the serial column chain of
// the QR, and the QR's block lives in the registers of all eight waves), so
// the building blocks are compiled for 512 threads here.
#define TTALS_NT 512
#define TTALS_QR_IEEE
#include "ttals_tt.hpp"

#include "ttals_dev.hpp"
#include "ttals_qr.hpp"
#include "ttals_svd.hpp"

namespace ttals {

// The workgroup's LDS: the QR's block, or the GEMM's staging tiles.
struct TtLDS {
  HqL qr;
  double* gemm;
};
constexpr size_t TT_LDS_BYTES = sizeof(HqLDS) > 8 * GEMM_LDS_DOUBLES ? sizeof(HqLDS) : 8 * GEMM_LDS_DOUBLES;
// kernels with an SVD: factors of up to 96 x 96 in LDS (one workgroup per CU either way)
constexpr size_t SVD_LDS_BYTES = 152 * 1024;
static_assert(SVD_LDS_BYTES >= TT_LDS_BYTES, "the QR's block and the GEMM tiles fit too");

// SVD of the factor B (c x k, row-major) as B V = U diag(sig): in LDS where B
// and V fit it, else in global memory, a wave per column pair.
__device__ void jacobi_svd(double* B, int c, int k, double* V, double* sig, int* perm, const TtLDS& S, double* red) {
  if (js_fits(c, k, SVD_LDS_BYTES / 8)) wg_jacobi_lds(B, c, k, V, sig, perm, S.gemm);
  else wg_jacobi_svd(B, c, k, V, sig, perm, red);
}

// How many of the k singular values (sorted by perm) pass: s/s0 > thr (rel) or
// s > thr, all of them when thr is 0.
__device__ int count_kept(const double* sig, const int* perm, int k, double thr, bool rel, double* red) {
  const double s0 = sig[perm[0]];
  double n = 0.0;
  for (int j = threadIdx.x; j < k; j += NT)
    if (thr == 0.0 || (rel ? sig[j] / s0 > thr : sig[j] > thr)) n += 1.0;
  return (int)wg_sum(n, red);
}

// Panels that the register QR (wg_qr_small) takes, copied to LDS, instead of the
// blocks: there a block of 16 columns costs more than the panel (rounding of a
// train of order 4, n = 2, ranks 2: 105 us with blocks, 93 us so; its residual
// norm 181 and 160 us).
__device__ __forceinline__ bool qr_in_lds(int m, int c) { return (m <= 32 && c <= 32) || (m <= 64 && c <= 16); }
static_assert(8 * (4 * 1024 + 64) <= TT_LDS_BYTES, "panel, Q, R and tau of the register QR");
// R on and above W's diagonal, the reflectors below it; Q into Qm.
template <bool WITH_Q>
__device__ void qr_small(double* W, int m, int c, double* Qm, const TtLDS& S) {
  const int k = m < c ? m : c;
  double *w = S.gemm, *q = w + 1024, *r = q + 1024, *t = r + 1024;
  __syncthreads();
  for (int e = threadIdx.x; e < m * c; e += NT) w[e] = W[e];
  __syncthreads();
  if constexpr (WITH_Q) {
    wg_qr_small(w, m, c, t, q, r);
  } else {  // m <= 32, c <= 16
    if (m <= 16) wg_qr_small_t<1, 1, false>(w, m, c, t, q, r);
    else wg_qr_small_t<2, 1, false>(w, m, c, t, q, r);
  }
  for (int e = threadIdx.x; e < m * c; e += NT) W[e] = w[e];
  if constexpr (WITH_Q)
    for (int e = threadIdx.x; e < m * k; e += NT) Qm[e] = q[e];
  __syncthreads();
}
// A column, or two of some hundred rows: the column sweep (100 x 1: 50 us a
// truncated sweep, 55 us with a block).
__device__ __forceinline__ bool qr_by_columns(int m, int c) { return m <= 256 && (c == 1 || (c == 2 && m > 64)); }

// R of the QR of the panel W (m x c, row-major, overwritten): in the top rows
// of the returned matrix (row stride c).  Panels of more columns than half
// the rows a block holds take the column sweep.  SMALL: the register QR up to
// 32 x 16 (alone, it gains nothing on R: the norm of a train of order 4,
// n = 4, ranks 4 takes 53 us either way).
template <bool SMALL>
__device__ const double* qr_r(double* W, int m, int c, double* tau, const TtLDS& S, double* red) {
  const bool by_columns = qr_by_columns(m, c);
  if constexpr (SMALL) {
    if (!by_columns && m <= 32 && c <= 16) {
      qr_small<false>(W, m, c, nullptr, S);
      return W;
    }
  }
  if (!by_columns && (m <= HQ_ROWS_MAX || 2 * c <= HQ_ROWS_MAX) && hq_fits(m, c))
    return wg_hqr_r(W, m, c, c, S.qr);
  wg_householder(W, m, c, tau, red);
  return W;
}

// The same with the reflectors left in W and the explicit Q (m x min(m, c))
// in Qm; the column sweep for panels taller than a block holds.
__device__ void qr_rq_blocks(double* W, int m, int c, double* tau, double* Tg, double* Qm, const TtLDS& S,
                             double* red) {
  if (m <= HQ_ROWS_MAX && hq_fits(m, c)) {
    wg_hqr(W, m, c, c, Tg, S.qr);
    wg_hqr_form_q(W, m, c, c, Tg, Qm, S.qr);
  } else {
    wg_householder(W, m, c, tau, red);
    wg_form_q(W, m, c, tau, Qm);
  }
}

// ... with the forms for small panels.
__device__ void qr_rq(double* W, int m, int c, double* tau, double* Tg, double* Qm, const TtLDS& S, double* red) {
  if (qr_by_columns(m, c)) {
    wg_householder(W, m, c, tau, red);
    wg_form_q(W, m, c, tau, Qm);
  } else if (qr_in_lds(m, c)) {
    qr_small<true>(W, m, c, Qm, S);
  } else {
    qr_rq_blocks(W, m, c, tau, Tg, Qm, S, red);
  }
}

// ---------------------------------------------------------------------------
// Batched residual norms ||A x - b|| and ||b|| of TT systems, one workgroup
// per system, without forming A x - b: the cores of the residual train
//   Z_0 = [ (A x)_0  -b_0 ],  Z_i = [[ (A x)_i, 0 ], [ 0, b_i ]],
//   Z_{d-1} = [[ (A x)_{d-1} ], [ b_{d-1} ]]
// (the rank layout of scikit_tt/tensor_train.py:313-333 for x - y with the
// product ranks of tensor_train.py:471-479) are generated block by block,
// already multiplied by the R factor coming from the right, straight into the
// panel of a right-to-left Householder QR sweep.  Only R factors are kept:
// the norm is invariant under the orthogonal factors, and the last core's
// Frobenius norm is the residual norm (the orthogonalisation form of
// scikit_tt/tensor_train.py:1334-1430, here without ever storing Z).
// One right-to-left sweep.  with_ax: the residual train; else b alone.
__device__ double resid_sweep(const ResidDesc& D, bool with_ax, const TtLDS& S, double* red) {
  double* lds = S.gemm;
  const int d = D.d;
  int k = 1;         // columns of the current right factor (k_{i+1})
  int ldr = 1;       // its leading dimension (rho_{i+1})
  if (threadIdx.x == 0) D.Rf[0] = 1.0;
  __syncthreads();
  for (int i = d - 1; i >= 0; --i) {
    const int n = D.n[i];
    const int P = with_ax ? D.ra[i] : 0, Q = D.ra[i + 1];
    const int a = D.rx[i], b = D.rx[i + 1];
    const int p = D.rb[i], q = D.rb[i + 1];
    // row block sizes of Z_i: (A x) block P a rows (one row on core 0), then the b rows
    const int top = (i == 0) ? (with_ax ? 1 : 0) : P * a;
    const int rho = (i == 0) ? 1 : top + p;
    const int boff_row = (i == 0) ? 0 : top;          // core 0: both blocks share row 0
    // column offset of the b block in Z_i (the last core stacks rows only)
    const int boff_col = (i == d - 1 || !with_ax) ? 0 : Q * b;
    const int mk = n * k;
    // W (mk x rho) = C_i^T, C_i[row, m, c] = sum_col Z_i[row, m, col] Rf[c, col]
    if (with_ax) {
      // U[a, n, Q, c] = sum_b x[a, n, b] Rf[c, Q b + b]
      wg_gemm<double, double>(a * n, Q * k, b, crm<double>(D.xc[i], b),
                              cview<double>(D.Rf, plain(1), split(k, b, ldr)), mrm<double>(D.U, Q * k), lds);
      // C_top[(P, a), m, c] = sum_{n', Q} A[P, m, n', Q] U[a, n', Q, c]; rows (P, m), cols (a, c)
      wg_gemm<double, double>(P * n, a * k, n * Q, crm<double>(D.ac[i], n * Q),
                              cview<double>(D.U, plain(k), split(k, n * Q * k, 1)),
                              mview<double>(D.W, split(n, a, k * rho), split(k, 1, rho)), lds);
    }
    // C_bot[j, m, c] = sum_j' b[j, m, j'] Rf[c, boff_col + j']; on core 0 it is subtracted
    // from the (A x) row, so it goes to U first
    double* dst = (i == 0 && with_ax) ? D.U : D.W;
    const int drho = (i == 0 && with_ax) ? 1 : rho;
    wg_gemm<double, double>(p * n, k, q, crm<double>(D.bc[i], q), cview<double>(D.Rf + boff_col, plain(1), plain(ldr)),
                            mview<double>(dst + (dst == D.W ? boff_row : 0), split(n, 1, k * drho), plain(drho)),
                            lds);
    if (i == 0) {
      // the last panel is one column: its norm is the residual norm
      double* v = D.W;
      if (with_ax)
        for (int e = threadIdx.x; e < mk; e += NT) v[e] -= D.U[e];
      __syncthreads();
      return wg_nrm2(v, mk, red);
    }
    const double* R = qr_r<true>(D.W, mk, rho, D.tau, S, red);
    const int kk = mk < rho ? mk : rho;
    for (int e = threadIdx.x; e < kk * rho; e += NT) {
      const int r = e / rho, c = e - r * rho;
      D.Rf[e] = (c >= r) ? R[(long)r * rho + c] : 0.0;
    }
    __syncthreads();
    k = kk;
    ldr = rho;
  }
  return 0.0;
}

__global__ __launch_bounds__(NT) void k_residual_norm(const ResidDesc* descs) {
  extern __shared__ double dyn_lds[];
  const TtLDS S{(HqL)dyn_lds, dyn_lds};
  __shared__ double red[4 * NWAVE];
  const ResidDesc& D = descs[blockIdx.x];
  const double rn = resid_sweep(D, true, S, red);
  const double bn = resid_sweep(D, false, S, red);
  if (threadIdx.x == 0) {
    D.out[0] = rn;
    D.out[1] = bn;
  }
}

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(NT) void k_tt_norm(NormArgs A) {
  extern __shared__ double dyn_lds[];
  const TtLDS S{(HqL)dyn_lds, dyn_lds};
  __shared__ double red[4 * NWAVE];
  int right = A.r[A.d];
  for (int i = A.d - 1; i >= 1; --i) {
    const int a = A.r[i], q = A.mn[i], b = right;
    const int m = q * b, c = a;
    // W (m x c) = core_i^T, core_i is (a x q*b); the last core is still the caller's
    const double* ci = (i == A.d - 1) ? A.src[i] : A.c[i];
    for (long e = threadIdx.x; e < (long)m * c; e += NT) {
      const int ii = (int)(e / c), jj = (int)(e % c);
      A.W[e] = ci[(long)jj * m + ii];
    }
    __syncthreads();
    const double* R = qr_r<false>(A.W, m, c, A.tau, S, red);
    const int k = m < c ? m : c;
    for (long e = threadIdx.x; e < (long)k * c; e += NT) {
      const int ii = (int)(e / c), jj = (int)(e % c);
      A.Rc[e] = (jj >= ii) ? R[(long)ii * c + jj] : 0.0;
    }
    __syncthreads();
    // core_{i-1} (rows x a) <- core_{i-1} * R^T  (rows x k)
    const int rows = A.r[i - 1] * A.mn[i - 1];
    wg_gemm<double, double>(rows, k, a, crm<double>(A.src[i - 1], a), ctr<double>(A.Rc, c), mrm<double>(A.T, k),
                            S.gemm);
    wg_copy(A.T, A.c[i - 1], rows * k);
    __syncthreads();
    right = k;
  }
  const long n0 = (long)A.r[0] * A.mn[0] * right;
  const double nrm = wg_nrm2(A.d == 1 ? A.src[0] : A.c[0], (int)n0, red);
  if (threadIdx.x == 0) A.out[0] = nrm;
}


// T (mt x ct) tall unfolding in A.W; on return the kept left factor
// (mt x kk, row-major) is in A.Qm and the pushed factor in A.Bm:
// B[:, perm] (ct x kk, row-major, ld kk).  Returns kk.
__device__ int ortho_factor(const OrthoArgs& A, int mt, int ct, int cap, const TtLDS& S, double* red) {
  qr_rq(A.W, mt, ct, A.tau, A.Tg, A.T, S, red);  // Q (mt x k) in T
  const int k = mt < ct ? mt : ct;
  if (!A.trunc) {
    wg_copy(A.T, A.Qm, mt * k);
    // pushed factor R^T (ct x k)
    for (long e = threadIdx.x; e < (long)ct * k; e += NT) {
      const int ii = (int)(e / k), jj = (int)(e % k);
      A.Bm[e] = (ii >= jj) ? A.W[(long)jj * ct + ii] : 0.0;
    }
    __syncthreads();
    return k;
  }
  // B = R^T (ct x k); Jacobi: B = U_B S, V
  for (long e = threadIdx.x; e < (long)ct * k; e += NT) {
    const int ii = (int)(e / k), jj = (int)(e % k);
    A.Rc[e] = (ii >= jj) ? A.W[(long)jj * ct + ii] : 0.0;
  }
  __syncthreads();
  jacobi_svd(A.Rc, ct, k, A.Vm, A.sig, A.perm, S, red);
  // number kept: s/s0 > thr, then the cap
  int kk = count_kept(A.sig, A.perm, k, A.thr, true, red);
  if (cap > 0 && kk > cap) kk = cap;
  if (kk < 1) kk = 1;
  // left factor (Q V)[:, perm[:kk]] -> Qm (mt x kk)
  wg_gemm<double, double>(mt, k, k, crm<double>(A.T, k), crm<double>(A.Vm, k), mrm<double>(A.W, k), S.gemm);
  for (long e = threadIdx.x; e < (long)mt * kk; e += NT) {
    const int ii = (int)(e / kk), jj = (int)(e % kk);
    A.Qm[e] = A.W[(long)ii * k + A.perm[jj]];
  }
  // pushed factor B[:, perm[:kk]] (ct x kk)
  for (long e = threadIdx.x; e < (long)ct * kk; e += NT) {
    const int ii = (int)(e / kk), jj = (int)(e % kk);
    A.Bm[e] = A.Rc[(long)ii * k + A.perm[jj]];
  }
  __syncthreads();
  return kk;
}

__global__ __launch_bounds__(NT) void k_tt_ortho(OrthoArgs A) {
  extern __shared__ double dyn_lds[];
  const TtLDS S{(HqL)dyn_lds, dyn_lds};
  __shared__ double red[4 * NWAVE];
  if (A.dir == 0) {
    for (int i = A.start; i <= A.end; ++i) {
      const int a = A.r[i], q = A.mn[i], b = A.r[i + 1];
      const int m = a * q, c = b;
      wg_copy(A.c[i], A.W, m * c);
      __syncthreads();
      const int k = ortho_factor(A, m, c, A.maxr[i + 1], S, red);
      wg_copy(A.Qm, A.c[i], m * k);
      __syncthreads();
      // core_{i+1} (b x rest) <- Bm^T (k x b) * core_{i+1}
      const int rest = A.mn[i + 1] * A.r[i + 2];
      wg_gemm<double, double>(k, rest, b, ctr<double>(A.Bm, k), crm<double>(A.c[i + 1], rest),
                              mrm<double>(A.T, rest), S.gemm);
      wg_copy(A.T, A.c[i + 1], k * rest);
      if (threadIdx.x == 0) A.r[i + 1] = k;
      __syncthreads();
    }
  } else {
    for (int i = A.start; i >= A.end; --i) {
      const int a = A.r[i], q = A.mn[i], b = A.r[i + 1];
      const int m = q * b, c = a;
      for (long e = threadIdx.x; e < (long)m * c; e += NT) {
        const int ii = (int)(e / c), jj = (int)(e % c);
        A.W[e] = A.c[i][(long)jj * m + ii];
      }
      __syncthreads();
      const int k = ortho_factor(A, m, c, A.maxr[i], S, red);
      // core_i (k x m) = Qm^T
      for (long e = threadIdx.x; e < (long)k * m; e += NT) {
        const int rr = (int)(e / m), cc = (int)(e % m);
        A.c[i][e] = A.Qm[(long)cc * k + rr];
      }
      __syncthreads();
      const int rows = A.r[i - 1] * A.mn[i - 1];
      wg_gemm<double, double>(rows, k, a, crm<double>(A.c[i - 1], a), crm<double>(A.Bm, k), mrm<double>(A.T, k),
                              S.gemm);
      wg_copy(A.T, A.c[i - 1], rows * k);
      if (threadIdx.x == 0) A.r[i] = k;
      __syncthreads();
    }
  }
}

__global__ __launch_bounds__(NT) void k_svd_trunc(SvdArgs A) {
  extern __shared__ double dyn_lds[];
  const TtLDS S{(HqL)dyn_lds, dyn_lds};
  __shared__ double red[4 * NWAVE];
  const bool tall = A.m >= A.c;
  const int mt = tall ? A.m : A.c, ct = tall ? A.c : A.m;
  for (long e = threadIdx.x; e < (long)mt * ct; e += NT) {
    const int i = (int)(e / ct), j = (int)(e % ct);
    A.W[e] = tall ? A.Y[e] : A.Y[(long)j * A.c + i];
  }
  __syncthreads();
  // the small panels' forms from two columns on would save some 4 us a call, but a threshold near rounding then cuts
  // elsewhere (the two-site solver's ranks at 1e-14)
  if (ct == 1) qr_rq(A.W, mt, ct, A.tau, A.Tg, A.Qm, S, red);
  else qr_rq_blocks(A.W, mt, ct, A.tau, A.Tg, A.Qm, S, red);
  // B = R^T (ct x ct)
  for (long e = threadIdx.x; e < (long)ct * ct; e += NT) {
    const int i = (int)(e / ct), j = (int)(e % ct);
    A.B[e] = (i >= j) ? A.W[(long)j * ct + i] : 0.0;
  }
  __syncthreads();
  jacobi_svd(A.B, ct, ct, A.Vm, A.sig, A.perm, S, red);
  int kk = count_kept(A.sig, A.perm, ct, A.thr, A.rel != 0, red);
  if (A.maxr > 0 && kk > A.maxr) kk = A.maxr;
  // left factor of the tall orientation: (Q V)[:, perm[:kk]] (mt x kk)
  wg_gemm<double, double>(mt, ct, ct, crm<double>(A.Qm, ct), crm<double>(A.Vm, ct), mrm<double>(A.L, ct), S.gemm);
  for (long e = threadIdx.x; e < (long)mt * kk; e += NT) {
    const int i = (int)(e / kk), j = (int)(e % kk);
    const double v = A.L[(long)i * ct + A.perm[j]];
    if (tall) A.U[(long)i * kk + j] = v;       // U = left factor
    else A.Vt[(long)j * mt + i] = v;            // Vt = (left factor)^T
  }
  // right factor: B[:, perm[j]] / s (ct x kk)
  for (long e = threadIdx.x; e < (long)ct * kk; e += NT) {
    const int i = (int)(e / kk), j = (int)(e % kk);
    const double sj = A.sig[A.perm[j]];
    const double v = sj > 0.0 ? A.B[(long)i * ct + A.perm[j]] / sj : 0.0;
    if (tall) A.Vt[(long)j * ct + i] = v;       // Vt = (right factor)^T
    else A.U[(long)i * kk + j] = v;             // U = right factor
  }
  for (int j = threadIdx.x; j < kk; j += NT) A.s[j] = A.sig[A.perm[j]];
  if (threadIdx.x == 0) *A.kout = kk;
}

hipError_t residual_norm_launch(int count, hipStream_t stream, const ResidDesc* descs) {
  hipLaunchKernelGGL(k_residual_norm, dim3(count), dim3(NT), TT_LDS_BYTES, stream, descs);
  return hipGetLastError();
}
hipError_t tt_norm_launch(hipStream_t stream, const NormArgs& a) {
  hipLaunchKernelGGL(k_tt_norm, dim3(1), dim3(NT), TT_LDS_BYTES, stream, a);
  return hipGetLastError();
}
hipError_t tt_ortho_launch(hipStream_t stream, const OrthoArgs& a) {
  hipLaunchKernelGGL(k_tt_ortho, dim3(1), dim3(NT), SVD_LDS_BYTES, stream, a);
  return hipGetLastError();
}
hipError_t svd_trunc_launch(hipStream_t stream, const SvdArgs& a) {
  hipLaunchKernelGGL(k_svd_trunc, dim3(1), dim3(NT), SVD_LDS_BYTES, stream, a);
  return hipGetLastError();
}

}  // namespace ttals
