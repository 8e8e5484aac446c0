// The split-bf16 GEMM (split_core.hpp): C = alpha op(A) op(B) + beta C with the
// epilogues of gemm_args.hpp.  Included by gemm_split_*.hip, which
// instantiate the layouts.
#pragma once
#include "activation.hpp"
#include "gemm_tiles.hpp"

#include <float.h>

namespace gemm {

// One tile (tm, tn) of batch item / K split bz.
template <class S, int TA, int TB, bool TAIL, bool COLSUM, int EPI>
__device__ __forceinline__ void split_tile(const GemmArgs& g, int tm, int tn, int bz, char* lds) {
  constexpr int BI = S::BI, BN = S::BN;
  constexpr bool A_MC = TA != 0, B_MC = TB == 0;
  using LA = split::MatLoad<A_MC, S::TM, S::NTH, TAIL>;
  using LB = split::MatLoad<B_MC, S::TN, S::NTH, TAIL, COLSUM>;
  const int m0 = tm * S::TM, n0 = tn * S::TN;
  const int64_t z = bz / g.splits;
  const int part = bz % g.splits;
  const float* A = g.A + batch_off(z, g, g.sa, g.sa2) + (g.grouped ? part * g.gsa : 0);
  const float* B = g.B + batch_off(z, g, g.sb, g.sb2) + (g.grouped ? part * g.gsb : 0);
  float* C = g.C + batch_off(z, g, g.sc, g.sc2);
  const int kbeg = g.grouped ? 0 : part * g.kchunk;
  const int klen = (g.grouped ? g.K : min(g.K, kbeg + g.kchunk)) - kbeg;
  const int tid = threadIdx.x, group = split::k_group<S>(), t = tid % S::NTH;
  f32x4 v[BI][BN], lo[BI][BN];
  {
    LA la;
    LB lb;
    // With two K groups (kterms == 1) each takes half of the stages.
    const int nk = ((klen + split::KS - 1) / split::KS + S::KG - 1) / S::KG;
    const int k0 = group * nk * split::KS, kl = S::KG == 1 ? klen : min(klen - k0, nk * split::KS);
    la.init(A, g.lda, g.M, g.K, m0, kbeg + k0, kl, g.kterms, g.gsa, t);
    lb.init(B, g.ldb, g.N, g.K, n0, kbeg + k0, kl, g.kterms, g.gsb, t);
    split::mma_loop<S>(lds + group * S::LDS, la, lb, g.kterms * nk, v, lo);
    if (COLSUM && tm == 0) {
      // the lane groups' sums of each column, added in order
      double* red = reinterpret_cast<double*>(lds);
      static_assert(4 * S::KG * S::TN * 8 <= S::LDS * S::KG, "column sums");
      __syncthreads();
#pragma unroll
      for (int c = 0; c < LB::NC; ++c) {
        int r, q;
        LB::unit(t, c, r, q);
        red[(4 * group + q) * S::TN + r] = lb.sum[c];
      }
      __syncthreads();
      if (tid < S::TN && n0 + tid < g.N) {
        double cs = red[tid];
#pragma unroll
        for (int q = 1; q < 4 * S::KG; ++q) cs += red[q * S::TN + tid];
        if (g.splits > 1) g.part_cs[(int64_t)bz * g.N + n0 + tid] = (float)cs;
        else put_colsum(g, z * g.scs + n0 + tid, (float)cs);
      }
    }
  }
  const bool redo = __syncthreads_or(split::needs_fp32<S>(v, lo));
  split::join_groups<S>(lds, v, lo);
  if (group != 0) return;  // (no barrier follows)
  if (redo) {
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int n = 0; n < BN; ++n) v[i][n] = lo[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int t = 0; t < g.kterms; ++t) {
      const float* At = A + t * g.gsa;
      const float* Bt = B + t * g.gsb;
      split::fp32_tile<S>(
          [&](int r, int k) {
            const int64_t row = m0 + r, kk = kbeg + k;
            return row < g.M ? At[A_MC ? kk * g.lda + row : row * g.lda + kk] : 0.f;
          },
          [&](int c, int k) {
            const int64_t col = n0 + c, kk = kbeg + k;
            return col < g.N ? Bt[B_MC ? kk * g.ldb + col : col * g.ldb + kk] : 0.f;
          },
          klen, v);
    }
  }

  // Epilogue.  Lane (lr, q) holds rows row(i, 4 q + r), columns col .. col + BN - 1.
  const split::WaveMap<S> w;
  const int col = n0 + w.col0();
  const bool split_mode = g.splits > 1;
  const float alpha = split_mode ? 1.f : g.alpha, beta = split_mode ? 0.f : g.beta;
  float* out = split_mode ? g.part + (int64_t)bz * g.M * g.N : C;
  const int64_t ldo = split_mode ? g.N : g.ldc;
  const int64_t zc = batch_off(z, g, g.sc, g.sc2);
  typedef float vec_t __attribute__((ext_vector_type(BN)));
  const bool vec = g.c_vec && (!split_mode || g.N % 4 == 0);  // N % 4 == 0 where c_vec is set
  float bias[BN];
#pragma unroll
  for (int n = 0; n < BN; ++n) bias[n] = !split_mode && g.bias && col + n < g.N ? g.bias[z * g.sbias + col + n] : 0.f;
#pragma unroll
  for (int i = 0; i < BI; ++i) {
#pragma unroll
    for (int n = 0; n < BN; ++n) v[i][n] = alpha * (v[i][n] + lo[i][n]);
  }
  if (beta != 0.f) {
    // every previous value is loaded before the first store: one memory
    // counter covers both, in order
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + w.row(i, 4 * w.q + r);
        const float* p = out + (int64_t)row * ldo + col;
#pragma unroll
        for (int n = 0; n < BN; ++n) lo[i][n][r] = 0.f;
        if (row < g.M && vec && col < g.N) {
          const vec_t o = *reinterpret_cast<const vec_t*>(p);
#pragma unroll
          for (int n = 0; n < BN; ++n) lo[i][n][r] = o[n];
        } else if (row < g.M) {
#pragma unroll
          for (int n = 0; n < BN; ++n)
            if (col + n < g.N) lo[i][n][r] = p[n];
        }
      }
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int n = 0; n < BN; ++n) v[i][n] += beta * lo[i][n];
  }
  constexpr int kRsLd = 64 + 4;  // row statistics: staging row stride (floats)
  float* stage = reinterpret_cast<float*>(lds) + (threadIdx.x >> 6) * (16 * BI * kRsLd);
  static_assert(EPI != kEpiRowstats || (BN == 4 && S::NTH / 64 * 16 * BI * kRsLd * 4 <= S::LDS), "row statistics staging");
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + w.row(i, 4 * w.q + r);
      const int64_t o = (int64_t)row * ldo + col;
      float y[BN];
#pragma unroll
      for (int n = 0; n < BN; ++n) y[n] = v[i][n][r] + bias[n];
      if (row < g.M) {
        if (vec && col < g.N) {
          vec_t t;
#pragma unroll
          for (int n = 0; n < BN; ++n) t[n] = y[n];
          *reinterpret_cast<vec_t*>(out + o) = t;
        } else {
#pragma unroll
          for (int n = 0; n < BN; ++n)
            if (col + n < g.N) out[o + n] = y[n];
        }
        // (an activation epilogue runs with 16-byte rows only)
        if (EPI == kEpiActFwd && col < g.N) {
          vec_t t;
#pragma unroll
          for (int n = 0; n < BN; ++n) t[n] = mle::act_rt(g.act_kind, y[n]);
          *reinterpret_cast<vec_t*>(g.act_y + zc + o) = t;
        }
        if (EPI == kEpiActBwd && col < g.N) {
          const vec_t xh = *reinterpret_cast<const vec_t*>(g.act_x + zc + o);
          vec_t* d = reinterpret_cast<vec_t*>(g.act_dx + zc + o);
          vec_t t = vec_t(0.f);
          if (g.act_acc) t = *d;
#pragma unroll
          for (int n = 0; n < BN; ++n)  // the elementwise backward's bits: the product rounded before the add
            t[n] = mle::act_bwd_rt(g.act_kind, xh[n], y[n], t[n], g.act_acc);
          *d = t;
        }
      }
      if (EPI == kEpiRowstats) {
        f32x4 t;
#pragma unroll
        for (int n = 0; n < BN; ++n) t[n] = col + n < g.N ? y[n] : -FLT_MAX;
        *reinterpret_cast<f32x4*>(stage + (16 * i + 4 * w.q + r) * kRsLd + 4 * w.lr) = t;
      }
    }
  if (EPI == kEpiRowstats) {
    // Lane l < 16 BI reduces row slot l's 64 columns to (max, sum of exp(x - max)).
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    const int slot_row = w.lane % (16 * BI);
    const float* rp = stage + slot_row * kRsLd;
    f32x4 x[16];
#pragma unroll
    for (int c = 0; c < 16; ++c) x[c] = *reinterpret_cast<const f32x4*>(rp + 4 * c);
    float m = -FLT_MAX;
#pragma unroll
    for (int c = 0; c < 16; ++c) m = fmaxf(fmaxf(m, fmaxf(x[c][0], x[c][1])), fmaxf(x[c][2], x[c][3]));
    float e = 0.f;
#pragma unroll
    for (int c = 0; c < 16; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) e += __expf(x[c][j] - m);
    const int row = m0 + w.row(slot_row >> 4, slot_row & 15);
    const int c0 = n0 + w.wn * 64;  // this wave's 64-column block
    if (w.lane < 16 * BI && row < g.M && c0 < g.N)
      *reinterpret_cast<float2*>(g.rowpart + (int64_t)row * g.rp_ld + 2 * (c0 >> 6)) = make_float2(m, e);
  }
}

template <class S, int TA, int TB, bool TAIL, bool COLSUM, int EPI>
__global__ __launch_bounds__(S::NTH * S::KG, 2) void gemm_split_kernel(GemmArgs g, int gx, int gy, int items) {
  __shared__ __attribute__((aligned(16))) char lds[S::LDS * S::KG];
  int tm, tn, z;
  item_tile(blockIdx.x, items, gx, gy, tm, tn, z);
  split_tile<S, TA, TB, TAIL, COLSUM, EPI>(g, tm, tn, z, lds);
}

template <int TA, int TB, bool TAIL, bool COLSUM, int EPI>
void launch_split_tile(hipStream_t s, const GemmArgs& g, int tile, int gx, int gy, int items) {
  if (tile == kSplitLarge)
    mle::launch(gemm_split_kernel<LargeTile, TA, TB, TAIL, COLSUM, EPI>, dim3((unsigned)items), LargeTile::NTH, 0, s, g, gx, gy, items);
  else if (tile == kSplitMedium)
    mle::launch(gemm_split_kernel<MediumTile, TA, TB, TAIL, COLSUM, EPI>, dim3((unsigned)items), MediumTile::NTH, 0, s, g, gx, gy, items);
  else if constexpr (EPI == kEpiPlain) {
    if (items <= kChipCus && g.kterms == 1)
      mle::launch(gemm_split_kernel<PairedTile, TA, TB, TAIL, COLSUM, EPI>, dim3((unsigned)items), PairedTile::NTH * PairedTile::KG, 0, s, g, gx, gy, items);
    else
      mle::launch(gemm_split_kernel<SmallTile, TA, TB, TAIL, COLSUM, EPI>, dim3((unsigned)items), SmallTile::NTH, 0, s, g, gx, gy, items);
  }
}

}  // namespace gemm
