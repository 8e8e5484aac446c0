// Split-bf16 GEMM kernels of untransposed A: NN (forward products, with their
// epilogues) and NT (input gradients).
#include "gemm_split.hpp"

namespace gemm {

void launch_split_a(hipStream_t s, bool trans_b, const GemmArgs& g, int tile, bool tail, int epi, int gx, int gy,
                    int items) {
  if (!trans_b) {
    if (epi == kEpiRowstats) return launch_split_tile<0, 0, false, false, kEpiRowstats>(s, g, tile, gx, gy, items);
    if (epi == kEpiActFwd) return launch_split_tile<0, 0, false, false, kEpiActFwd>(s, g, tile, gx, gy, items);
    if (tail) return launch_split_tile<0, 0, true, false, kEpiPlain>(s, g, tile, gx, gy, items);
    return launch_split_tile<0, 0, false, false, kEpiPlain>(s, g, tile, gx, gy, items);
  }
  if (epi == kEpiActBwd) return launch_split_tile<0, 1, false, false, kEpiActBwd>(s, g, tile, gx, gy, items);
  if (tail) return launch_split_tile<0, 1, true, false, kEpiPlain>(s, g, tile, gx, gy, items);
  return launch_split_tile<0, 1, false, false, kEpiPlain>(s, g, tile, gx, gy, items);
}

}  // namespace gemm
