// Argument records and launch helpers of the TT-algebra kernels that run one
// workgroup of eight waves per train (ttals_tt.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ttals {

// ||t||_2 by a right-to-left QR sweep: only the R factors are needed
// (the norm is invariant under the orthogonal factors).  Cores are working
// copies with dims (r, mn, r'); they are overwritten.
struct NormArgs {
  int d;
  const int* mn;
  const int* r;
  const double* const* src;  // the caller's cores (read only)
  double* const* c;   // working cores: c[i-1] is written when core i is absorbed
  double* W;          // >= max_i mn_i * r_{i+1} * r_i
  double* Rc;         // >= r_i^2
  double* T;          // >= max_i r_{i-1} * mn_{i-1} * r_i
  double* tau;        // >= max rank
  double* out;
};

// Left/right orthonormalisation sweep of a TT (one workgroup).  Cores are
// updated in place (capacity of the input ranks); ranks (device int[d+1]) are
// updated.  dims: mn[i] = m_i * n_i.
//   no truncation: Householder QR of the tall unfolding, Q kept, R pushed on;
//   truncation (threshold > 0 or a finite max rank): the same QR, then a
//   one-sided Jacobi SVD of R, singular triplets with s/s0 > threshold (then
//   at most max_rank[bond]) kept, S V^T (or U S) pushed on
//   (scikit_tt/tensor_train.py:1162-1189, 1268-1299).
struct OrthoArgs {
  int d, dir, start, end;  // dir 0: left (i = start..end), 1: right (i = start..end descending)
  int trunc;
  double thr;
  const int* maxr;  // [d+1], <= 0 = unbounded
  const int* mn;
  int* r;
  double* const* c;
  double* W;   // >= max core size
  double* Qm;  // >= max core size
  double* Rc;  // >= rmax^2
  double* T;   // >= max core size
  double* tau; // >= rmax
  double* Bm;  // >= rmax^2
  double* Vm;  // >= rmax^2
  double* sig; // >= rmax
  int* perm;   // >= rmax
  double* Tg;  // qr_tg_doubles(rmax)
};

// Truncated SVD of a row-major m x c matrix Y (one workgroup): Householder
// QR of the tall orientation (Y, or Y^T when m < c), one-sided Jacobi SVD of
// R^T, singular triplets kept by s/s0 > thr (rel) or s > thr (absolute) when
// thr != 0, then at most maxr (the rule of scikit_tt/utils.py:145-156).
// U (m x k), s (k), Vt (k x c) row-major; k written to *kout.
struct SvdArgs {
  int m, c, maxr, rel;
  double thr;
  const double* Y;
  double* U;
  double* s;
  double* Vt;
  double* W;    // mt x ct
  double* Qm;   // mt x ct
  double* B;    // ct x ct
  double* Vm;   // ct x ct
  double* L;    // mt x ct
  double* sig;  // ct
  double* tau;  // ct
  int* perm;    // ct
  double* Tg;   // qr_tg_doubles(ct)
  int* kout;
};

// One system of k_residual_norm.
struct ResidDesc {
  int d;
  int pad;
  const int* n;              // [d] mode sizes
  const int* ra;             // [d+1] operator ranks
  const int* rx;             // [d+1] x ranks
  const int* rb;             // [d+1] rhs ranks
  const double* const* ac;   // operator cores (P, n, n, Q)
  const double* const* xc;   // x cores (r, n, 1, r')
  const double* const* bc;   // rhs cores (p, n, 1, q)
  double* W;                 // panel: max_i n_i k_{i+1} rho_i doubles
  double* U;                 // max_i r_i n_i R_{i+1} k_{i+1} doubles
  double* Rf;                // rho_max^2 doubles (R factor carried to the left)
  double* tau;               // rho_max doubles
  double* out;               // [2]: ||A x - b||, ||b||
};

// doubles of block-reflector storage a (. x c) panel needs
inline long qr_tg_doubles(long c) { return (c + 16) * 16; }

hipError_t residual_norm_launch(int count, hipStream_t stream, const ResidDesc* descs);
hipError_t tt_norm_launch(hipStream_t stream, const NormArgs& a);
hipError_t tt_ortho_launch(hipStream_t stream, const OrthoArgs& a);
hipError_t svd_trunc_launch(hipStream_t stream, const SvdArgs& a);

}  // namespace ttals
