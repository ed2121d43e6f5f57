// Pieces of one local problem, a workgroup each: interface updates, matvec,
// local right-hand side, local solve and eigensolve, panel QR.
#pragma once
#include <hip/hip_runtime.h>

#include "ttals_engine.hpp"

namespace ttals {

struct PieceArgs {
  int op, a, P, n, Q, b;
  const double* L;
  const double* A;
  const double* R;   // or Lb/Rb/x depending on op
  const double* x;
  const double* f;
  double* out;
  double* v;
  double* t1;
  double* t2;
  double* V;
  double* res;       // [4] scalars out
  int method, sym, maxit, mode;
  double tol, sigma;
  long arena;        // dynamic LDS of the launch in doubles (on-chip path when the problem fits)
  int mvar;          // on-chip matvec form (SysDesc::mvar)
};

enum PieceOp { P_LEFT_OP, P_RIGHT_OP, P_LEFT_RHS, P_RIGHT_RHS, P_MICRO_DENSE, P_MATVEC, P_MICRO_RHS, P_SOLVE,
               P_EIG, P_QR };

// Static LDS bytes of k_piece_wide (ttals_piece.hip).
hipError_t piece_wide_static_lds(size_t* bytes);

// Launches one piece on k_piece_wide with `dyn_lds` bytes of dynamic LDS
// (a.arena doubles).
hipError_t piece_wide_launch(size_t dyn_lds, hipStream_t stream, const PieceArgs& a);

// One workgroup.  The matvec, local solve and local eigensolve take the
// engine's on-chip path (operator and working vectors in the dynamic LDS
// arena) whenever the problem fits `A.arena`, else the global path.
__device__ __forceinline__ void piece_block(const PieceArgs& A, double* dyn_lds, double* lds, SolveLDS& S) {
  const long N = (long)A.a * A.n * A.b;
  switch (A.op) {
    case P_LEFT_OP:
    case P_RIGHT_OP: {
      // on-chip matrix-core update (the engine's) when it fits the arena; a
      // right stack is the left-form update of the mirrored problem
      const bool left = A.op == P_LEFT_OP;
      const int al = left ? A.a : A.b, Pl = left ? A.P : A.Q, Ql = left ? A.Q : A.P, bl = left ? A.b : A.a;
      const long need = (long)al * Pl * al + N + (long)A.P * A.n * A.n * A.Q + ds_t1_size(al, Pl, A.n, bl) +
                        ds_t2_size(al, A.n, Ql, bl) + (long)bl * Ql * bl;
      if (need <= A.arena) {
        double* Lc = dyn_lds;
        double* xc = Lc + (long)al * Pl * al;
        double* Ac = xc + N;
        double* t1 = Ac + (long)A.P * A.n * A.n * A.Q;
        double* t2 = t1 + ds_t1_size(al, Pl, A.n, bl);
        double* out = t2 + ds_t2_size(al, A.n, Ql, bl);
        if (left) {
          wg_copy(A.L, Lc, al * Pl * al);
          wg_copy(A.x, xc, (int)N);
          wg_copy_opcore_pnmq(A.A, Ac, A.P, A.n, A.Q);
        } else {
          wg_copy(A.R, Lc, al * Pl * al);
          wg_copy_core_t(A.x, xc, A.a, A.n, A.b);
          wg_copy_opcore_qnmp(A.A, Ac, A.P, A.n, A.Q);
        }
        __syncthreads();
        stack_left_mf(al, Pl, A.n, Ql, bl, Lc, Ac, xc, out, t1, t2);
        wg_copy(out, A.out, bl * Ql * bl);
      } else if (left) {
        stack_left_op<double, double>(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.x, A.out, A.t1, A.t2, lds);
      } else {
        stack_right_op<double, double>(A.a, A.P, A.n, A.Q, A.b, A.R, A.A, A.x, A.out, A.t1, A.t2, lds);
      }
      break;
    }
    case P_LEFT_RHS:
      stack_left_rhs<double, double>(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.x, A.out, A.t1, lds);
      break;
    case P_RIGHT_RHS:
      stack_right_rhs<double, double>(A.a, A.P, A.n, A.Q, A.b, A.R, A.A, A.x, A.out, A.t1, lds);
      break;
    case P_MICRO_DENSE:
      micro_dense<double>(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.out, A.a * A.n * A.b);
      break;
    case P_MATVEC:
      if (arena_need_onchip(A.a, A.P, A.n, A.Q, A.b, 2, A.mvar) <= A.arena) {
        LocalOp<double> op{A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.t1, A.t2, false};
        double* vec = onchip_operator(op, dyn_lds, A.arena, 2, A.mvar);
        wg_copy(A.x, vec, (int)N);
        __syncthreads();
        apply_op<double, double>(op, vec, vec + N, lds);
        wg_copy(vec + N, A.out, (int)N);
      } else {
        local_matvec<double, double>(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.x, A.out, A.t1, A.t2, lds);
      }
      break;
    case P_MICRO_RHS:
      micro_rhs<double, double>(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.out, A.t1, lds);
      break;
    case P_SOLVE: {
      LocalOp<double> op{A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.t1, A.t2, false};
      int its = 0, r = 0;
      int method = A.method;
      if (method == 0) method = (N <= NDENSE) ? 1 : (A.sym ? 2 : 3);
      if (method == 1 && lu_reg_fits(A.a, A.P, A.n, A.Q, A.b, A.arena)) {
        r = lu_reg_solve(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.f, A.v, dyn_lds) ? 0 : 1;
      } else if (method == 1) {
        micro_dense<double>(A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.V, N);
        wg_copy(A.f, A.v, N);
        __syncthreads();
        r = wg_lu_solve(A.V, N, A.v, reinterpret_cast<int*>(A.V + (long)N * N), S.red) ? 0 : 1;
      } else if (arena_need_onchip(A.a, A.P, A.n, A.Q, A.b, 5, A.mvar) <= A.arena) {
        Work W;
        W.V = A.V;
        onchip_work(W, onchip_operator(op, dyn_lds, A.arena, 5, A.mvar), (int)N, true);
        wg_copy(A.f, W.f, (int)N);
        wg_copy(A.v, W.x, (int)N);
        __syncthreads();
        if (method == 2) r = wg_cg<double, true>(op, W, A.tol, A.maxit, lds, S, &its);
        if (method == 3 || r == 1) r = wg_gmres<double>(op, W, A.tol, A.maxit, KMAX, lds, S, &its);
        wg_copy(W.x, A.v, (int)N);
      } else {
        Work W;
        W.V = A.V;
        W.f = const_cast<double*>(A.f);
        W.x = A.v;
        W.r = A.V;
        W.p = A.V + N;
        W.q = A.V + 2 * (long)N;
        W.cur = A.V + (long)(KMAX + 1) * N;
        W.w = A.V + (long)(KMAX + 2) * N;
        if (method == 2) r = wg_cg<double, false>(op, W, A.tol, A.maxit, lds, S, &its);
        if (method == 3 || r == 1) r = wg_gmres<double>(op, W, A.tol, A.maxit, KMAX, lds, S, &its);
      }
      if (threadIdx.x == 0) {
        A.res[0] = r;
        A.res[1] = its;
      }
      break;
    }
    case P_EIG: {
      LocalOp<double> op{A.a, A.P, A.n, A.Q, A.b, A.L, A.A, A.R, A.t1, A.t2, false};
      Work W;
      W.V = A.V;
      int its = 0, r;
      double lam = 0.0;
      if (arena_need_onchip(A.a, A.P, A.n, A.Q, A.b, 3, A.mvar) <= A.arena) {
        onchip_work(W, onchip_operator(op, dyn_lds, A.arena, 3, A.mvar), (int)N, false);
        __syncthreads();
        r = wg_lanczos<double, true>(op, A.v, W, A.mode, A.sigma, A.tol, A.maxit, LKMAX, lds, S, &lam, &its);
      } else {
        W.cur = A.V + (long)(LKMAX + 1) * N;
        W.w = A.V + (long)(LKMAX + 2) * N;
        W.r = A.V + (long)(LKMAX + 3) * N;
        r = wg_lanczos<double, false>(op, A.v, W, A.mode, A.sigma, A.tol, A.maxit, LKMAX, lds, S, &lam, &its);
      }
      if (threadIdx.x == 0) {
        A.res[0] = r;
        A.res[1] = its;
        A.res[2] = lam;
      }
      break;
    }
    case P_QR: {
      // m = a, c = b; input x (m x c); out = Q (m x k); v = R (k x c); t1 = work
      // (W, then tau, then (c + 16) * 16 for the blocked QR's T).  The forms the
      // engine keeps for panels of up to 64 x 64 and for those of more rows than
      // wg_hqr holds; its register-blocked QR would be a second caller of wg_hqr
      // in k_als's translation unit, which costs k_als 28 more spilled registers.
      const int m = A.a, c = A.b;
      double* W = A.t1;
      for (long e = threadIdx.x; e < (long)m * c; e += NT) W[e] = A.x[e];
      __syncthreads();
      if (m <= 64 && c <= 64) {  // the engine's small-panel path
        wg_qr_small(W, m, c, A.t2, A.out, A.v);
        break;
      }
      if (wg_hhqr_blocked(W, m, c, A.out, A.v, A.t2 + (m > c ? m : c), A.t2, dyn_lds, A.arena, S.red)) break;
      wg_householder(W, m, c, A.t2, S.red);
      wg_form_q(W, m, c, A.t2, A.out);
      const int k = m < c ? m : c;
      for (long e = threadIdx.x; e < (long)k * c; e += NT) {
        const int i = (int)(e / c), j = (int)(e % c);
        A.v[e] = (j >= i) ? W[(long)i * c + j] : 0.0;
      }
      break;
    }
  }
}

}  // namespace ttals
