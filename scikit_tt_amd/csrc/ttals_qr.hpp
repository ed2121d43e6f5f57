// Blocked Householder QR of a tall row-major panel in global memory by one
// workgroup (LAPACK dgeqrf / dlarft / dlarfb in structure and in signs: the
// same reflectors, R and Q as the column sweep wg_householder, up to
// rounding).
//
// What bounds it: the FP64 arithmetic of the trailing update (2 m c^2 flops;
// a CU does 128 FP64 flops a clock on the matrix or the vector units alike)
// and, per column, one chain of a reduction over the panel's rows, a square
// root and two reciprocals.  So:
//  * a block of 16 columns is held in registers for its factorisation, rows
//    split over the waves (wave w: rows [w RW, (w+1) RW) below the pivot row
//    of the block), in the matrix-core accumulator layout: lane (lk, li) =
//    (lane / 16, lane % 16) holds rows 4 s + lk of column li.  A column's dot
//    products with the other 15 are 16 lanes' work at once; one workgroup
//    barrier per column (the sweep over global memory paid two and three
//    passes over the trailing matrix per column);
//  * that layout is also the operand layout of the 16x16x4 FP64 matrix
//    instruction for V^T (A operand) and for the trailing columns (B operand)
//    and of its result: Y = V^T X, Z = T' Y and X -= V Z run from loads and
//    registers without any rearrangement;
//  * the trailing matrix makes two passes through L2 per 16 columns instead
//    of per column.
// A (2112 x 132) panel (the largest of a rank-32 residual train, n = 16) in
// L2 on one workgroup: 1.09 ms here -- 0.36 ms in the block factorisations
// (1 us a column at 256 rows, 2.4 us at 2112), 0.73 ms in the trailing updates
// (0.25 ms of it arithmetic) -- against about 15 ms by the column sweep.
#pragma once
#include "ttals_dev.hpp"

namespace ttals {

constexpr int HQ_NB = 16;        // columns per block
constexpr int HQ_GROUP = 4;      // column tiles of one sweep of a trailing update (in registers)
// rows one call handles: HQ_RP_MAX doubles of panel per lane
constexpr int HQ_RP_MAX = 72;
constexpr int HQ_ROWS_MAX = NWAVE * 4 * HQ_RP_MAX;

struct HqLDS {
  double part[NWAVE][HQ_GROUP][4][64];  // per-wave partial Y tiles, then Z in [0]
  double red[2][NWAVE][HQ_NB];          // per-wave dots of a column step (two columns in turn)
  double prow[2][HQ_NB];                // its pivot row
  double T[HQ_NB][HQ_NB + 1];
};
typedef TT_LDS HqLDS* HqL;

// lane J of each 16-lane row to all lanes of the row
template <int J>
__device__ __forceinline__ double row_bcast(double v) {
  const long r = __builtin_amdgcn_mov_dpp(__builtin_bit_cast(long, v), 0x150 + J, 0xF, 0xF, true);
  return __builtin_bit_cast(double, r);
}
// Two dot products' partial sums over four entries of a column tile,
// a0/a1 += row_bcast<J>(b) * b, and the tile's update b += row_bcast<J>(b) * c:
// one instruction per entry (the broadcast is the multiply-add's own operand
// move; the two wait states a DPP read of a fresh VALU result needs come
// first).
template <int J>
__device__ __forceinline__ void dpp_dot4(double& a0, double& a1, double b0, double b1, double b2, double b3) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %2, %2 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %3, %3 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %0, %4, %4 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %5, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf"
      : "+&v"(a0), "+&v"(a1)
      : "v"(b0), "v"(b1), "v"(b2), "v"(b3), "n"(J));
}
template <int J>
__device__ __forceinline__ void dpp_axpy4(double& b0, double& b1, double& b2, double& b3, double c) {
  asm("s_nop 1\n\t"
      "v_fmac_f64_dpp %0, %0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %1, %1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %2, %2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f64_dpp %3, %3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
      : "+v"(b0), "+v"(b1), "+v"(b2), "+v"(b3)
      : "v"(c), "n"(J));
}
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));
// sum over the four 16-lane rows, in every lane (rows 0+1 and 2+3 first)
__device__ __forceinline__ double rows4_sum(double v) {
  {
    const u32x2_t a = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
    const u32x2_t b = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
    v = __hiloint2double(b.x, a.x) + __hiloint2double(b.y, a.y);
  }
  const u32x2_t a = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
  const u32x2_t b = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
  return __hiloint2double(b.x, a.x) + __hiloint2double(b.y, a.y);
}

// A block's columns in registers: rows [w RW, (w+1) RW) of the `rows` below
// (and with) the block's first pivot row; b[s] = row w RW + 4 s + lk, column li.
template <int RP>
struct HqTile {
  double b[RP];
};

template <int RP>
__device__ __forceinline__ void hq_load(HqTile<RP>& P, const double* Wp, int ld, int rows, int kb, int RW) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int r0 = w * RW + lk, rend = min(rows, (w + 1) * RW);
  const bool on = li < kb;
#pragma unroll
  for (int s = 0; s < RP; ++s) {
    const int r = r0 + 4 * s;
    P.b[s] = (on && r < rend) ? Wp[(unsigned)(r * ld + li)] : 0.0;
  }
}

// Factors the block: on return P holds R on and above the diagonal and the
// reflectors below it, S->T the block's T (dlarft, forward, columnwise).  One
// barrier per column.  At column j the lanes of the columns li > j apply H_j,
// lanes li < j contribute the dots of their reflectors with it (the Gram
// entries of T).  A finished column stays unscaled (x, with v = scl x) until
// the end, so that the update is the same instruction in every lane.  The
// rows of the first 16 (wave 0), which hold the diagonal, are masked.
template <int RP>
__device__ __forceinline__ void hq_factor(HqTile<RP>& P, int kb, HqL S) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  double scl = 0.0;
  static_for<0, HQ_NB>([&](auto Jc) {
    constexpr int j = decltype(Jc)::value, sp = j >> 2, kp = j & 3, buf = j & 1;
    if (j >= kb) return;
    // column j's entries below the pivot (zero elsewhere) in the first 16 rows
    auto below = [&](int s) -> double {
      double x = row_bcast<j>(P.b[s]);
      if (s < sp) x = (w == 0) ? 0.0 : x;
      if (s == sp) x = (w == 0 && lk <= kp) ? 0.0 : x;
      return x;
    };
    double a0 = 0.0, a1 = 0.0;
#pragma unroll
    for (int s = 4; s < RP; s += 4) dpp_dot4<j>(a0, a1, P.b[s], P.b[s + 1], P.b[s + 2], P.b[s + 3]);
#pragma unroll
    for (int s = 0; s < 4; ++s) a0 = fma(below(s), P.b[s], a0);
    const double part = rows4_sum(a0 + a1);
    if (lk == 0) S->red[buf][w][li] = part;
    if (w == 0 && lk == kp) S->prow[buf][li] = P.b[sp];
    __syncthreads();
    double dot = 0.0;
#pragma unroll
    for (int q = 0; q < NWAVE; ++q) dot += S->red[buf][q][li];
    const double pr = S->prow[buf][li];
    const double s2 = row_bcast<j>(dot), alpha = row_bcast<j>(pr);
    double t = 0.0, beta = alpha, sc = 0.0;
    if (s2 != 0.0) {  // else H_j = I (LAPACK convention for an already-reduced column)
      const double nrm = sqrt(alpha * alpha + s2);
      beta = alpha >= 0.0 ? -nrm : nrm;
      t = (beta - alpha) / beta;
      sc = 1.0 / (alpha - beta);
    }
    const double wq = fma(sc, dot, pr);  // H_j: the update's w_q (li > j) ...
    if (s2 != 0.0) {
      const double cx = li > j ? -(t * wq) * sc : 0.0;
#pragma unroll
      for (int s = 0; s < 4; ++s) P.b[s] = fma(cx, below(s), P.b[s]);
#pragma unroll
      for (int s = 4; s < RP; s += 4) dpp_axpy4<j>(P.b[s], P.b[s + 1], P.b[s + 2], P.b[s + 3], cx);
      if (w == 0 && lk == kp) P.b[sp] = li == j ? beta : (li > j ? pr - t * wq : P.b[sp]);
    }
    if (w == NWAVE - 1) {  // T[l][j] = -tau_j sum_{p=l}^{j-1} T[l][p] G[p][j], T[j][j] = tau_j
      const double gl = wq * scl;  // the Gram entry G[li][j] (li < j)
      double sm = 0.0;
      static_for<0, j>([&](auto Pc) {
        sm = fma(S->T[li][decltype(Pc)::value], row_bcast<decltype(Pc)::value>(gl), sm);
      });
      if (lk == 0) S->T[li][j] = li < j ? -t * sm : (li == j ? t : 0.0);
    }
    scl = li == j ? sc : scl;
  });
  if (w == NWAVE - 1 && lk == 0)
    for (int q = kb; q < HQ_NB; ++q) S->T[li][q] = 0.0;
#pragma unroll
  for (int s = 0; s < RP; ++s)
    if (s >= 4 || w != 0 || 4 * s + lk > li) P.b[s] *= scl;
}

template <int RP>
__device__ __forceinline__ void hq_store(const HqTile<RP>& P, double* Wp, int ld, int rows, int kb, int RW) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, li = lane & 15, lk = lane >> 4;
  const int r0 = w * RW + lk, rend = min(rows, (w + 1) * RW);
  if (li < kb) {
#pragma unroll
    for (int s = 0; s < RP; ++s) {
      const int r = r0 + 4 * s;
      if (r < rend) Wp[(unsigned)(r * ld + li)] = P.b[s];
    }
  }
}

// X (rows x nc, global, ld ldx) <- (I - V T' V^T) X with the block's
// reflectors V (rows x kb, stored below the diagonal of Wp, ld ld) and S->T;
// T' = T^T (trans: H^T X, the factorisation's trailing update) or T (forming
// Q).  Wave w takes the 16-row blocks w, w + NWAVE, ...; a group of up to
// HQ_GROUP column tiles is swept twice, Y = V^T X accumulating in registers
// and then X -= V Z with Z in registers, the next row block's operands loading
// during one's matrix instructions.  Four tiles a group and uniform (scalar)
// bounds keep all of it in registers.  Eight 16-column tiles of a 2112-row
// panel: 407 us with eight tiles a group and vector bounds (spilled), 162 us
// with four, 132 us with the operands one block ahead; 56 us is arithmetic.
// Ends with a barrier.
__device__ __attribute__((noinline)) void hq_apply(const double* Wp_, int ld_, int kb_, double* X_, int ldx_, int rows_,
                                                   int nc_, bool trans_, HqL S) {
  const double* Wp = uni(Wp_);
  double* X = uni(X_);
  const int ld = uni(ld_), kb = uni(kb_), ldx = uni(ldx_), rows = uni(rows_), nc = uni(nc_);
  const bool trans = uni((int)trans_) != 0;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15, lk = lane >> 4;
  const int nblk = (rows + 15) >> 4;
  // entry (r, c) of V: 1 on the diagonal, 0 above it, past the rows and past kb
  auto v_at = [&](int r, int c) -> double {
    const double x = Wp[(unsigned)(min(r, rows - 1) * ld + min(c, kb - 1))];
    return (r < rows && c < kb && r >= c) ? (r == c ? 1.0 : x) : 0.0;
  };
  for (int g0 = 0; g0 < nc; g0 += HQ_GROUP * 16) {
    const int tiles = min(HQ_GROUP, (nc - g0 + 15) >> 4);
    const double* xc = X + g0;
    auto col = [&](int t) { return min(16 * t + li, nc - 1 - g0); };
    dx4_t acc[HQ_GROUP];
#pragma unroll
    for (int t = 0; t < HQ_GROUP; ++t) acc[t] = dx4_t{0.0, 0.0, 0.0, 0.0};
    double vn[4];
    dx4_t xn[HQ_GROUP];
    auto load_x = [&](int blk) {
#pragma unroll
      for (int t = 0; t < HQ_GROUP; ++t)
        if (t < tiles) {
#pragma unroll
          for (int e = 0; e < 4; ++e) xn[t][e] = xc[(unsigned)(min(16 * blk + 4 * e + lk, rows - 1) * ldx + col(t))];
        }
    };
    auto load_v = [&](int blk) {
#pragma unroll
      for (int e = 0; e < 4; ++e) vn[e] = v_at(16 * blk + 4 * e + lk, li);
    };
    if (w < nblk) {
      load_v(w);
      load_x(w);
    }
#pragma unroll 1
    for (int blk = w; blk < nblk; blk += NWAVE) {
      double v[4];
      dx4_t x[HQ_GROUP];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = vn[e];
#pragma unroll
      for (int t = 0; t < HQ_GROUP; ++t) x[t] = xn[t];
      if (blk + NWAVE < nblk) {
        load_v(blk + NWAVE);
        load_x(blk + NWAVE);
      }
#pragma unroll
      for (int t = 0; t < HQ_GROUP; ++t)
        if (t < tiles) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[t] = mfma16x16x4(v[e], x[t][e], acc[t]);
        }
    }
#pragma unroll
    for (int t = 0; t < HQ_GROUP; ++t)
      if (t < tiles) {
#pragma unroll
        for (int e = 0; e < 4; ++e) S->part[w][t][e][lane] = acc[t][e];
      }
    __syncthreads();
    // wave t: Y of tile t over the waves, Z = -T' Y into part[0][t]
    if (w < tiles) {
      double y[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        y[e] = S->part[0][w][e][lane];
#pragma unroll
        for (int q = 1; q < NWAVE; ++q) y[e] += S->part[q][w][e][lane];
      }
      dx4_t z = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int s = 0; s < 4; ++s) z = mfma16x16x4(trans ? S->T[4 * s + lk][li] : S->T[li][4 * s + lk], y[s], z);
#pragma unroll
      for (int e = 0; e < 4; ++e) S->part[0][w][e][lane] = -z[e];
    }
    __syncthreads();
    double z[HQ_GROUP][4];
#pragma unroll
    for (int t = 0; t < HQ_GROUP; ++t)
      if (t < tiles) {
#pragma unroll
        for (int e = 0; e < 4; ++e) z[t][e] = S->part[0][t][e][lane];
      }
    double* xs = X + g0;
    auto load_vt = [&](int blk) {
#pragma unroll
      for (int s = 0; s < 4; ++s) vn[s] = v_at(16 * blk + li, 4 * s + lk);
    };
    if (w < nblk) {
      load_vt(w);
      load_x(w);
    }
#pragma unroll 1
    for (int blk = w; blk < nblk; blk += NWAVE) {
      double v[4];
      dx4_t x[HQ_GROUP];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = vn[e];
#pragma unroll
      for (int t = 0; t < HQ_GROUP; ++t) x[t] = xn[t];
      if (blk + NWAVE < nblk) {
        load_vt(blk + NWAVE);
        load_x(blk + NWAVE);
      }
#pragma unroll
      for (int t = 0; t < HQ_GROUP; ++t)
        if (t < tiles) {
#pragma unroll
          for (int s = 0; s < 4; ++s) x[t] = mfma16x16x4(v[s], z[t][s], x[t]);
          if (g0 + 16 * t + li < nc) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int r = 16 * blk + 4 * e + lk;
              if (r < rows) xs[(unsigned)(r * ldx + 16 * t + li)] = x[t][e];
            }
          }
        }
    }
    __syncthreads();
  }
}

// Factors one block of columns with RP doubles of panel per lane; T to S->T
// and, when wanted, to Tg.  Ends with a barrier.
template <int RP>
__device__ __attribute__((noinline)) void hq_block(double* Wp_, int ld_, int rows_, int kb_, double* Tg, HqL S) {
  double* Wp = uni(Wp_);
  const int ld = uni(ld_), rows = uni(rows_), kb = uni(kb_);
  const int RW = ((rows + 16 * NWAVE - 1) / (16 * NWAVE)) * 16;
  HqTile<RP> P;
  hq_load<RP>(P, Wp, ld, rows, kb, RW);
  hq_factor<RP>(P, kb, S);
  hq_store<RP>(P, Wp, ld, rows, kb, RW);
  __syncthreads();
  if (Tg)
    for (int e = threadIdx.x; e < HQ_NB * HQ_NB; e += NT) Tg[e] = S->T[e >> 4][e & 15];
}

// byte offsets into the panel stay below 2^31
__device__ __forceinline__ bool hq_fits(int m, int c) { return (long)m * c < (1L << 28); }

// the smallest panel form that holds `rows` rows
template <class F>
__device__ __forceinline__ void hq_dispatch(int rows, F&& f) {
  const int rp = ((rows + 16 * NWAVE - 1) / (16 * NWAVE)) * 4;
  if (rp <= 8) f(std::integral_constant<int, 8>{});
  else if (rp <= 16) f(std::integral_constant<int, 16>{});
  else if (rp <= 32) f(std::integral_constant<int, 32>{});
  else if (rp <= 48) f(std::integral_constant<int, 48>{});
  else f(std::integral_constant<int, HQ_RP_MAX>{});
}

// W (m x c, ld ld, global) <- its Householder QR: R on and above the
// diagonal, the reflectors below it; Tg (optional): 256 doubles per block of
// 16 columns for wg_hqr_form_q.  m <= HQ_ROWS_MAX.  Starts and ends with a
// barrier.
__device__ void wg_hqr(double* W, int m, int c, int ld, double* Tg, HqL S) {
  const int k = m < c ? m : c;
  __syncthreads();
  for (int jb = 0; jb < k; jb += HQ_NB) {
    const int kb = min(HQ_NB, k - jb);
    double* Wp = W + (long)jb * ld + jb;
    double* T = Tg ? Tg + (long)jb * HQ_NB : nullptr;
    hq_dispatch(m - jb, [&](auto RPc) { hq_block<decltype(RPc)::value>(Wp, ld, m - jb, kb, T, S); });
    if (c > jb + kb) hq_apply(Wp, ld, kb, Wp + kb, ld, m - jb, c - jb - kb, true, S);
  }
  __syncthreads();
}

// Explicit Q (m x k, row-major, ld k) from wg_hqr's W and Tg.
__device__ void wg_hqr_form_q(const double* W, int m, int c, int ld, const double* Tg, double* Qm, HqL S) {
  const int k = m < c ? m : c;
  for (long e = threadIdx.x; e < (long)m * k; e += NT) {
    const int i = (int)(e / k), j = (int)(e - (long)i * k);
    Qm[e] = i == j ? 1.0 : 0.0;
  }
  __syncthreads();
  for (int jb = ((k - 1) / HQ_NB) * HQ_NB; jb >= 0; jb -= HQ_NB) {
    for (int e = threadIdx.x; e < HQ_NB * HQ_NB; e += NT) S->T[e >> 4][e & 15] = Tg[(long)jb * HQ_NB + e];
    __syncthreads();
    hq_apply(W + (long)jb * ld + jb, ld, min(HQ_NB, k - jb), Qm + (long)jb * k + jb, k, m - jb, k - jb, false, S);
  }
}

// R of a panel of any height, R only: rows in chunks of at most HQ_ROWS_MAX,
// each later chunk under the R of the ones before it, which is copied into
// the rows above the chunk (already factored).  R ends in the top k rows of
// the matrix at the returned pointer (ld ld).  c < HQ_ROWS_MAX.
__device__ double* wg_hqr_r(double* W, int m, int c, int ld, HqL S) {
  int end = min(m, HQ_ROWS_MAX);
  wg_hqr(W, end, c, ld, nullptr, S);
  double* top = W;
  while (end < m) {  // here end >= HQ_ROWS_MAX > c: R has c rows
    const int next = min(m, end + HQ_ROWS_MAX - c);
    double* at = W + (long)(end - c) * ld;
    // R into the c rows above `end` (bottom up: the two may overlap), a thread
    // per column
    for (int j = threadIdx.x; j < c; j += NT)
      for (int i = c - 1; i >= 0; --i) at[(long)i * ld + j] = j >= i ? top[(long)i * ld + j] : 0.0;
    __syncthreads();
    wg_hqr(at, next - end + c, c, ld, nullptr, S);
    top = at;
    end = next;
  }
  return top;
}

}  // namespace ttals
