// k_piece_wide: pieces of local problems that do not fit k_als's arena, the
// local solves of the two-site scheme among them.
//
// A translation unit of its own: a launch is a single workgroup with a CU to
// itself, so it runs eight waves and takes the CU's LDS, where k_als leaves
// room for a second system.  What still does not fit streams its contractions
// through L2 and is bound by that latency, which eight waves hide better than
// four.  Two-site sweep of order 6, n = 8, ranks up to 8 (4096 unknowns, off
// both arenas): 15.6 ms with k_piece, 11.7 ms here.
#define TTALS_NT 512
#include "ttals_piece.hpp"

namespace ttals {

__global__ __launch_bounds__(NT) void k_piece_wide(PieceArgs A) {
  extern __shared__ double dyn_lds[];
  __shared__ double lds[GEMM_LDS_DOUBLES];
  __shared__ SolveLDS S;
  piece_block(A, dyn_lds, lds, S);
}

hipError_t piece_wide_static_lds(size_t* bytes) {
  hipFuncAttributes fa;
  const hipError_t e = hipFuncGetAttributes(&fa, reinterpret_cast<const void*>(k_piece_wide));
  if (e == hipSuccess) *bytes = fa.sharedSizeBytes;
  return e;
}

hipError_t piece_wide_launch(size_t dyn_lds, hipStream_t stream, const PieceArgs& a) {
  hipLaunchKernelGGL(k_piece_wide, dim3(1), dim3(NT), dyn_lds, stream, a);
  return hipGetLastError();
}

}  // namespace ttals
