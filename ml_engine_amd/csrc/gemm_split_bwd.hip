// Split-bf16 GEMM kernels of transposed A: TN (weight gradients, with the bias
// gradient's column sums) and TT, and the Linear backward's pair.
#include "gemm_split.hpp"

namespace gemm {

void launch_split_a(hipStream_t s, bool trans_b, const GemmArgs& g, int tile, bool tail, int epi, int gx, int gy,
                    int items);

void launch_split(hipStream_t s, int trans, const GemmArgs& g, int tile, bool tail, bool colsum, int epi, int gx, int gy,
                  int items) {
  if (trans < 2) return launch_split_a(s, trans == 1, g, tile, tail, epi, gx, gy, items);
  if (trans == 3) {
    if (tail) return launch_split_tile<1, 1, true, false, kEpiPlain>(s, g, tile, gx, gy, items);
    return launch_split_tile<1, 1, false, false, kEpiPlain>(s, g, tile, gx, gy, items);
  }
  // neither operand is k-contiguous: no tail
  if (colsum) return launch_split_tile<1, 0, false, true, kEpiPlain>(s, g, tile, gx, gy, items);
  return launch_split_tile<1, 0, false, false, kEpiPlain>(s, g, tile, gx, gy, items);
}

// Two independent products in one launch, one tile per workgroup, each
// computed exactly as gemm_split_kernel computes it.  A Linear layer's dX and
// dW products (Engine/engine.cu:3553-3560) often fill half the chip each.
// The weight gradient's tiles, the deeper ones, start first; problem 0 starts
// at a multiple of 8 workgroups (those between do nothing), so that its item
// L runs on XCD L % 8 as item_tile assumes.
template <class S, bool COLSUM>
__global__ __launch_bounds__(S::NTH, 2) void gemm_split_pair_kernel(GemmArgs g0, GemmArgs g1, PairGrid pg) {
  __shared__ __attribute__((aligned(16))) char lds[S::LDS];
  const int b = blockIdx.x;
  int tm, tn, z;
  if (b < pg.items1) {
    item_tile(b, pg.items1, pg.gx1, pg.gy1, tm, tn, z);
    split_tile<S, 1, 0, false, COLSUM, kEpiPlain>(g1, tm, tn, z, lds);
  } else if (b >= pg.start0) {
    item_tile(b - pg.start0, pg.items0, pg.gx0, pg.gy0, tm, tn, z);
    split_tile<S, 0, 1, false, false, kEpiPlain>(g0, tm, tn, z, lds);
  }
}

template <class S>
static void launch_pair(hipStream_t s, const GemmArgs& g0, const GemmArgs& g1, bool colsum, const PairGrid& pg) {
  const dim3 grid((unsigned)(pg.start0 + pg.items0));
  if (colsum) mle::launch(gemm_split_pair_kernel<S, true>, grid, S::NTH, 0, s, g0, g1, pg);
  else mle::launch(gemm_split_pair_kernel<S, false>, grid, S::NTH, 0, s, g0, g1, pg);
}

void launch_split_pair(hipStream_t s, const GemmArgs& g0, const GemmArgs& g1, int tile, bool colsum, const PairGrid& pg) {
  if (tile == kSplitLarge) launch_pair<LargeTile>(s, g0, g1, colsum, pg);
  else launch_pair<MediumTile>(s, g0, g1, colsum, pg);
}

}  // namespace gemm
