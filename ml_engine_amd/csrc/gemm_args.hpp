// Arguments and tile order of the GEMM kernels (gemm.hip, gemm_split*.hip).
#pragma once
#include "common.hpp"

#include <algorithm>

namespace gemm {

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  float* colsum;
  int64_t lda, ldb, ldc, sa, sb, sc;
  int M, N, K;
  float alpha, beta;
  // split-K: blockIdx.z = batch item * splits + split; each split covers
  // kchunk of K and writes its raw tile to part (and its column sums to
  // part_cs); split_reduce_kernel combines them in split order.
  int splits, kchunk;
  float* part;
  float* part_cs;
  const float* bias;  // nullable: C[r, c] += bias[c] after alpha/beta
  // Two-level batch: item z = zo * inner + zi sits at zo * s + zi * s2 of
  // each operand (inner == 1: one stride).  Lets per-head products address
  // the heads of a [batch, seq, heads * dim] tensor in place.
  int inner;
  int64_t sa2, sb2, sc2;
  // Per batch item bias and column-sum strides (0: shared).
  int64_t sbias, scs;
  // Sum of products: when grouped, split s multiplies A + s*gsa by B + s*gsb
  // over the whole K (the splits are the terms), and the reduce adds them in
  // term order.
  int grouped;
  int64_t gsa, gsb;
  // Sum of products folded into K (split kernel, one K split): the K loop
  // walks term t of A + t*gsa and B + t*gsb for t = 0 .. kterms - 1.
  int kterms;
  // Row statistics of C (split kernel): for row r and 64-column block b,
  // rowpart[r * rp_ld + 2 b] = max over the block, [.. + 1] = sum of
  // exp(C - max).  nullptr: none.
  float* rowpart;
  int64_t rp_ld;
  // Activation epilogues (split kernel, C's layout): forward writes
  // act_y = act(C); backward writes act_dx (+)= C * act'(act_x).
  float* act_y;
  const float* act_x;
  float* act_dx;
  int act_acc;
  // 1 + an activation kind: the split reduce also writes act_y = act(C) in
  // C's layout (0: not).
  int act_red;
  // Column sums: 0 adds them into colsum (the default), 1 assigns (colsum is
  // logically zero).
  int cs_assign;
  // 1 + an activation kind: the small-product kernels (simple, K-split) also
  // write act_dx (+)= act'(act_x) * C in C's layout, act_acc choosing add or
  // assign (0: not).
  int act_bwd;
  // Split kernel: the activation of an activation epilogue, and whether C's
  // rows (and the bias) can be written (read) 16 bytes at a time.
  int act_kind;
  int c_vec;
};

// Tile shapes of the split kernel (split_core.hpp), and a launch of it.
enum SplitTile { kSplitLarge = 0, kSplitMedium = 1, kSplitSmall = 2 };
constexpr int kSplitTm[3] = {256, 128, 64}, kSplitTn[3] = {128, 128, 64};
// Time model of a grid of them.
// Measured on MI355X over 33 products of 100 .. 8192 rows, columns and depth, us
// per stage and per tile for a round of at most 256 workgroups: large 2.3 + 8
// (+ 13 where a round follows another: every workgroup writes its 128 KB of C
// at once), medium 1.4 + 5.5, small 0.53 + 4.5 (one workgroup per CU, two K
// groups; 0.67 with one, where the terms of a sum follow each other: 3 terms of
// 512 x 512 x 1024 in 70 us); 0.53 + 1.7 for each small tile of a CU that several
// share, and 3.0 more (2.2 for one or two stages; 2500 x 512 x 64: small 9.0, medium 9.9).
constexpr double kStageUs[3] = {2.3, 1.4, 0.53}, kTileUs[3] = {8.0, 5.5, 4.5};
constexpr double kFullTileUs = 13.0, kSharedTileUs = 1.7, kSharedUs = 3.0, kSharedShortUs = 2.2, kOneGroupStageUs = 0.67;
constexpr int kChipCus = 256;

inline long long tiles_of(int tile, int M, int N) {
  return (long long)((M + kSplitTm[tile] - 1) / kSplitTm[tile]) * ((N + kSplitTn[tile] - 1) / kSplitTn[tile]);
}

// Time of n workgroups of `stages` stages each on tile shape `tile`; k_groups:
// small tiles may share their K between two groups.
inline double split_grid_us(int tile, long long n, int stages, bool k_groups = true) {
  const long long per = (n + kChipCus - 1) / kChipCus;  // workgroups per CU
  if (per == 1) return stages * (tile == kSplitSmall && !k_groups ? kOneGroupStageUs : kStageUs[tile]) + kTileUs[tile];
  const double t = tile == kSplitLarge ? kFullTileUs : tile == kSplitMedium ? kTileUs[tile] : kSharedTileUs;
  return (double)per * (stages * kStageUs[tile] + t) + (tile != kSplitSmall ? 0.0 : stages <= 2 ? kSharedShortUs : kSharedUs);
}

// trans: 2 * trans_a + trans_b.  tail: K % 4 != 0 beside a k-contiguous operand
// (kEpiPlain only).  epi: kEpi*.
void launch_split(hipStream_t s, int trans, const GemmArgs& g, int tile, bool tail, bool colsum, int epi, int gx, int gy,
                  int items);
// A Linear's dX (NT, problem 0) and dW (+ db; TN, problem 1) in one grid;
// workgroups [0, items1) take problem 1, those from `start0` on problem 0.
struct PairGrid {
  int items0, gx0, gy0, start0;
  int items1, gx1, gy1;
};
void launch_split_pair(hipStream_t s, const GemmArgs& g0, const GemmArgs& g1, int tile, bool colsum, const PairGrid& pg);

// colsum[i] (+)= v as GemmArgs::cs_assign says.
__device__ __forceinline__ void put_colsum(const GemmArgs& g, int64_t i, float v) {
  g.colsum[i] = g.cs_assign ? v : g.colsum[i] + v;
}

// Epilogue modes of the split kernel.
constexpr int kEpiPlain = 0, kEpiRowstats = 1, kEpiActFwd = 2, kEpiActBwd = 3;

__device__ __forceinline__ int64_t batch_off(int64_t z, const GemmArgs& g, int64_t s, int64_t s2) {
  if (g.inner == 1) return z * s;
  return (z / g.inner) * s + (z % g.inner) * s2;
}

// Tile order.  Workgroups are handed to the 8 XCDs round-robin (linear id
// L on XCD L % 8), and each XCD has its own L2.  XCD x therefore gets the
// contiguous logical range [x*T/8, (x+1)*T/8) of the T tiles, walked in
// groups of 8 tile-rows with the columns inside a group, so the workgroups
// resident on one XCD share a few A row-panels and B column-panels.  A
// bijection on [0, T): every tile is still computed by exactly one workgroup.
constexpr int kXcds = 8, kGroupRows = 8;

// Tile (tm, tn) and batch item z of work item L of a launch over `items` =
// gx * gy * batch tiles.  The order above: item L runs on
// XCD L % 8 (workgroups are dispatched round-robin), XCD x owns a contiguous
// logical range, walked in groups of 8 tile-rows per batch item.  A bijection
// on [0, items).
__device__ __forceinline__ void item_tile(int L, int items, int gx, int gy, int& tm, int& tn, int& z) {
  const int q = items / kXcds, r = items % kXcds, x = L % kXcds;
  const int logical = x * q + min(x, r) + L / kXcds;
  const int T = gx * gy;
  z = logical / T;
  const int t = logical - z * T;
  const int per_group = kGroupRows * gx;
  const int grp = t / per_group;
  const int first_m = grp * kGroupRows;
  const int rows = min(gy - first_m, kGroupRows);
  const int in_group = t - grp * per_group;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
}

}  // namespace gemm
