// mle_gemm: batched / broadcast fp32 GEMM on MFMA with an optional fused
// column sum of op(B) (the Linear bias gradient).  Replaces the 32 x 32
// scalar-FMA tiles and atomicAdd epilogues of bcmm / bcmmABT / bcmmATB / bcmmT
// (Engine/kernels.cu:387-539): every C element is written by exactly one lane,
// so results are deterministic.
#include "activation.hpp"
#include "gemm_args.hpp"
#include "gemm_core.hpp"

#include <float.h>

#include <algorithm>

using namespace mle;
using namespace gemm;

namespace {

// Load 4 consecutive elements base[r*ld + c .. c+3] with bounds (R rows, Cc cols).
template <bool VEC>
__device__ __forceinline__ f32x4 ld_guard(const float* __restrict__ base, int64_t ld, int r, int c, int R, int Cc) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (r < R) {
    const float* p = base + (int64_t)r * ld + c;
    if (VEC && c + 3 < Cc) {
      v = *reinterpret_cast<const f32x4*>(p);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c + j < Cc) v[j] = p[j];
    }
  }
  return v;
}

// Global -> registers for one stage.  A tile is TM x KD (TM*KD/1024 float4
// per thread), a B tile KD x TN.  A_MC == trans_a (A stored K x M); B_KC ==
// trans_b.  `kend` bounds K for this workgroup's split.  k-contiguous tiles
// give each row KD/4 float4; m/n-contiguous ones T/4 per k row.
template <bool MC, int T, int KD>
__device__ __forceinline__ void tile_coord(int f, int& r, int& c) {
  if (!MC) {  // [T][KD]: r = row along M/N, c = k
    r = f / (KD / 4);
    c = (f % (KD / 4)) * 4;
  } else {  // [KD][T]: r = k, c = along M/N
    r = f / (T / 4);
    c = (f % (T / 4)) * 4;
  }
}

template <bool A_MC, bool VEC, int TM, int KD>
__device__ __forceinline__ void load_a(const GemmArgs& g, const float* A, int m0, int k0, int kend, int tid,
                                       f32x4 (&r)[TM * KD / 1024]) {
#pragma unroll
  for (int i = 0; i < TM * KD / 1024; ++i) {
    int a, b;
    tile_coord<A_MC, TM, KD>(tid + NT * i, a, b);
    r[i] = A_MC ? ld_guard<VEC>(A, g.lda, k0 + a, m0 + b, kend, g.M) : ld_guard<VEC>(A, g.lda, m0 + a, k0 + b, g.M, kend);
  }
}
template <bool B_KC, bool VEC, int TN, int KD>
__device__ __forceinline__ void load_b(const GemmArgs& g, const float* B, int n0, int k0, int kend, int tid,
                                       f32x4 (&r)[TN * KD / 1024]) {
#pragma unroll
  for (int i = 0; i < TN * KD / 1024; ++i) {
    int a, b;
    tile_coord<!B_KC, TN, KD>(tid + NT * i, a, b);
    r[i] = B_KC ? ld_guard<VEC>(B, g.ldb, n0 + a, k0 + b, g.N, kend) : ld_guard<VEC>(B, g.ldb, k0 + a, n0 + b, kend, g.N);
  }
}

// Registers -> LDS (same element mapping as the loads).  KC: k-contiguous.
template <bool KC, int T, int KD>
__device__ __forceinline__ void store_tile(float* S, int tid, const f32x4 (&r)[T * KD / 1024]) {
#pragma unroll
  for (int i = 0; i < T * KD / 1024; ++i) {
    int a, b;
    tile_coord<!KC, T, KD>(tid + NT * i, a, b);
    *reinterpret_cast<f32x4*>(S + a * (KC ? KD + PAD : T + PAD) + b) = r[i];
  }
}

__device__ __forceinline__ void tile_of(int gx, int gy, int& tm, int& tn) {
  const int T = gx * gy;
  const int L = blockIdx.x + gx * blockIdx.y;
  const int q = T / kXcds, r = T % kXcds, x = L % kXcds;
  const int logical = x * q + min(x, r) + L / kXcds;
  const int per_group = kGroupRows * gx;
  const int first_m = (logical / per_group) * kGroupRows;
  const int rows = min(gy - first_m, kGroupRows);
  const int in_group = logical % per_group;
  tm = first_m + in_group % rows;
  tn = in_group / rows;
}

// The general fp32 MFMA kernel, 64-bit addresses and guarded loads: products
// that the split-bf16 kernel (gemm_split.hpp) does not take, i.e. an operand of
// 2 GiB or more, a column sum beside an untransposed A or a transposed B, an
// empty K.  VEC: 16-byte loads.
template <int TA, int TB, bool VEC, bool COLSUM>
__global__ __launch_bounds__(NT, 3) void gemm_kernel(GemmArgs g) {
  constexpr int WM = 4, WN = 4, KD = 16;
  constexpr bool A_MC = TA != 0;
  constexpr bool B_KC = TB != 0;
  constexpr int TM = 32 * WM, TN = 32 * WN;
  constexpr int ASZ = a_tile_floats<A_MC, TM, KD>();
  constexpr int BSZ = b_tile_floats<B_KC, TN, KD>();
  __shared__ __attribute__((aligned(16))) float smem[2 * (ASZ + BSZ)];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, q = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  int tm, tn;
  tile_of(gridDim.x, gridDim.y, tm, tn);
  const int m0 = tm * TM, n0 = tn * TN;
  const int64_t z = blockIdx.z / g.splits;
  const int split = blockIdx.z % g.splits;
  const float* A = g.A + batch_off(z, g, g.sa, g.sa2) + (g.grouped ? split * g.gsa : 0);
  const float* B = g.B + batch_off(z, g, g.sb, g.sb2) + (g.grouped ? split * g.gsb : 0);
  float* C = g.C + batch_off(z, g, g.sc, g.sc2);
  const int kbeg = g.grouped ? 0 : split * g.kchunk;
  const int kend = g.grouped ? g.K : min(g.K, kbeg + g.kchunk);
  f32x4 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int n = 0; n < WN; ++n) acc[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};

  const bool do_cs = COLSUM && tm == 0;
  constexpr int CS_T = NT / TN;  // threads per column of the column sum
  float csum = 0.f;
  const int nk = kend > kbeg ? (kend - kbeg + KD - 1) / KD : 0;
  f32x4 ra[TM * KD / 1024], rb[TN * KD / 1024];
  if (nk > 0) {
    load_a<A_MC, VEC, TM, KD>(g, A, m0, kbeg, kend, tid, ra);
    load_b<B_KC, VEC, TN, KD>(g, B, n0, kbeg, kend, tid, rb);
    store_tile<!A_MC, TM, KD>(smem, tid, ra);
    store_tile<B_KC, TN, KD>(smem + 2 * ASZ, tid, rb);
  }
  __syncthreads();

  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    const float* As = smem + cur * ASZ;
    const float* Bs = smem + 2 * ASZ + cur * BSZ;
    const bool more = kt + 1 < nk;
    if (more) {
      load_a<A_MC, VEC, TM, KD>(g, A, m0, kbeg + (kt + 1) * KD, kend, tid, ra);
      load_b<B_KC, VEC, TN, KD>(g, B, n0, kbeg + (kt + 1) * KD, kend, tid, rb);
    }
    mma_stage<A_MC, B_KC, WM, WN, KD>(As, Bs, acc, wm, wn, lr, q);
    if (do_cs) {
      const int c = tid % TN, h = tid / TN;
#pragma unroll
      for (int k = 0; k < KD / CS_T; ++k) {
        const int kk = h * (KD / CS_T) + k;
        csum += B_KC ? Bs[c * (KD + PAD) + kk] : Bs[kk * (TN + PAD) + c];
      }
    }
    if (more) {
      store_tile<!A_MC, TM, KD>(smem + (cur ^ 1) * ASZ, tid, ra);
      store_tile<B_KC, TN, KD>(smem + 2 * ASZ + (cur ^ 1) * BSZ, tid, rb);
    }
    __syncthreads();
  }

  const float alpha = g.alpha, beta = g.beta;
  const bool split_mode = g.splits > 1;
  float* P = split_mode ? g.part + (int64_t)blockIdx.z * g.M * g.N : nullptr;
  {
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
      for (int n = 0; n < WN; ++n) {
        const int col = n0 + acc_col<WN>(wn, n, lr);
        if (col >= g.N) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = m0 + acc_row<WM>(wm, i, q, r);
          if (row < g.M) {
            if (split_mode) {
              P[(int64_t)row * g.N + col] = acc[i][n][r];
            } else {
              float* p = C + (int64_t)row * g.ldc + col;
              float v = alpha * acc[i][n][r];
              if (beta != 0.f) v += beta * *p;
              if (g.bias) v += g.bias[z * g.sbias + col];
              *p = v;
            }
          }
        }
      }
  }

  if (do_cs) {
    // smem is free after the final barrier of the K loop.
    smem[tid] = csum;
    __syncthreads();
    if (tid < TN && n0 + tid < g.N) {
      float cs = 0.f;
#pragma unroll
      for (int h = 0; h < CS_T; ++h) cs += smem[tid + h * TN];
      if (split_mode) g.part_cs[(int64_t)blockIdx.z * g.N + n0 + tid] = cs;
      else put_colsum(g, z * g.scs + n0 + tid, cs);
    }
  }
}

// Row statistics of a finished C when the GEMM did not produce them in its
// epilogue: one wave per (row, 64-column block): max and sum of exp(C - max).
__global__ __launch_bounds__(256) void rowstats_kernel(const float* __restrict__ C, int64_t ldc, int M, int N,
                                                       float* __restrict__ part, int64_t ld) {
  const int nblk = (N + 63) / 64;
  const int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= (int64_t)M * nblk) return;
  const int row = (int)(w / nblk), blk = (int)(w % nblk);
  const int lane = threadIdx.x & 63, c = blk * 64 + lane;
  const float x = c < N ? C[(int64_t)row * ldc + c] : -FLT_MAX;
  float m = x;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  float e = c < N ? expf(x - m) : 0.f;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
  if (lane == 0) *reinterpret_cast<float2*>(part + (int64_t)row * ld + 2 * blk) = make_float2(m, e);
}

// C = alpha * sum_s part[s] + beta * C (+ bias) and colsum (+)= sum_s
// part_cs[s], in a fixed order.  A workgroup covers 64 units -- a unit is W
// (4 with VEC, else 1) columns of one row of one batch item, numbered over
// (batch, row, column group) so every thread has one -- with four split
// groups: thread (unit, g) adds splits g, g + 4, g + 8, ... in order (four
// loads in flight), and the group sums are added in group order through LDS.
// Workgroups from `nmain` on take the column sums: one thread per (batch,
// column), splits added in order.
template <bool VEC>
__global__ __launch_bounds__(256) void split_reduce_kernel(GemmArgs g, int64_t units, unsigned nmain) {
  constexpr int W = VEC ? 4 : 1;
  __shared__ f32x4 grp[4][64];
  const int64_t mn = (int64_t)g.M * g.N;
  if (blockIdx.x >= nmain) {
    const int64_t j = (int64_t)(blockIdx.x - nmain) * 256 + threadIdx.x;
    const int batch = (int)(units / ((int64_t)g.M * (g.N / W)));
    if (j >= (int64_t)batch * g.N) return;
    const int64_t b = j / g.N, col = j - b * g.N;
    const float* p = g.part_cs + b * g.splits * (int64_t)g.N + col;
    float acc = 0.f;
    int sp = 0;
    for (; sp + 4 <= g.splits; sp += 4) {
      float v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = p[(int64_t)(sp + u) * g.N];
#pragma unroll
      for (int u = 0; u < 4; ++u) acc += v[u];
    }
    for (; sp < g.splits; ++sp) acc += p[(int64_t)sp * g.N];
    put_colsum(g, b * g.scs + col, acc);
    return;
  }
  const int lane = threadIdx.x & 63, sg = threadIdx.x >> 6;
  const int64_t u = (int64_t)blockIdx.x * 64 + lane;
  const bool live = u < units;
  int64_t b = 0, row = 0, col = 0;
  if (live) {
    const int64_t nw = g.N / W, per = (int64_t)g.M * nw;
    b = u / per;
    const int64_t r = u - b * per;
    row = r / nw;
    col = (r - row * nw) * W;
  }
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  if (live) {
    const float* p = g.part + b * g.splits * mn + row * g.N + col;
    int sp = sg;
    for (; sp + 12 < g.splits; sp += 16) {
      f32x4 v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (VEC) v[k] = *reinterpret_cast<const f32x4*>(p + (int64_t)(sp + 4 * k) * mn);
        else v[k] = f32x4{p[(int64_t)(sp + 4 * k) * mn], 0.f, 0.f, 0.f};
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) acc += v[k];
    }
    for (; sp < g.splits; sp += 4) {
      if (VEC) acc += *reinterpret_cast<const f32x4*>(p + (int64_t)sp * mn);
      else acc[0] += p[(int64_t)sp * mn];
    }
  }
  grp[sg][lane] = acc;
  __syncthreads();
  if (sg != 0 || !live) return;
  const f32x4 r = ((grp[0][lane] + grp[1][lane]) + grp[2][lane]) + grp[3][lane];
  float* c = g.C + batch_off(b, g, g.sc, g.sc2) + row * g.ldc + col;
  const int64_t co = batch_off(b, g, g.sc, g.sc2) + row * g.ldc + col;
  if (VEC) {
    f32x4 v = g.alpha * r;
    if (g.beta != 0.f) v += g.beta * *reinterpret_cast<const f32x4*>(c);
    if (g.bias) v += *reinterpret_cast<const f32x4*>(g.bias + b * g.sbias + col);
    *reinterpret_cast<f32x4*>(c) = v;
    if (g.act_red) {
      f32x4 y;
#pragma unroll
      for (int k = 0; k < 4; ++k) y[k] = act_rt(g.act_red - 1, v[k]);
      *reinterpret_cast<f32x4*>(g.act_y + co) = y;
    }
  } else {
    float v = g.alpha * r[0];
    if (g.beta != 0.f) v += g.beta * *c;
    if (g.bias) v += g.bias[b * g.sbias + col];
    *c = v;
    if (g.act_red) g.act_y[co] = act_rt(g.act_red - 1, v);
  }
}

// 64 C elements per workgroup, one per lane, the four waves taking a quarter
// of K each and adding their partial sums in wave order: products with a tiny
// M or K (a Linear layer applied to one row, or the weight gradient of one),
// where the tile kernels would spend split-K and reduce launches on little
// work.
template <int TA, int TB>
__device__ __forceinline__ void simple_body(const GemmArgs& g, int bx, int64_t z, float (&red)[2][4][64]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t idx = (int64_t)bx * 64 + lane;
  const bool live = idx < (int64_t)g.M * g.N;
  const int m = live ? (int)(idx / g.N) : 0, n = live ? (int)(idx % g.N) : 0;
  const int kq = (g.K + 3) / 4, k0 = w * kq, k1 = min(g.K, k0 + kq);
  const float* A = g.A + z * g.sa;
  const float* B = g.B + z * g.sb;
  float acc = 0.f, cs = 0.f;
  if (live) {
#pragma unroll 8
    for (int k = k0; k < k1; ++k) {
      const float a = TA ? A[(int64_t)k * g.lda + m] : A[(int64_t)m * g.lda + k];
      const float b = TB ? B[(int64_t)n * g.ldb + k] : B[(int64_t)k * g.ldb + n];
      acc += a * b;
      cs += b;
    }
  }
  red[0][w][lane] = acc;
  red[1][w][lane] = cs;
  __syncthreads();
  if (w != 0 || !live) return;
  acc = ((red[0][0][lane] + red[0][1][lane]) + red[0][2][lane]) + red[0][3][lane];
  float* c = g.C + z * g.sc + (int64_t)m * g.ldc + n;
  float v = g.alpha * acc;
  if (g.beta != 0.f) v += g.beta * *c;
  if (g.bias) v += g.bias[z * g.sbias + n];
  *c = v;
  if (g.act_bwd) {
    const int64_t co = z * g.sc + (int64_t)m * g.ldc + n;
    g.act_dx[co] = act_bwd_rt(g.act_bwd - 1, g.act_x[co], v, g.act_acc ? g.act_dx[co] : 0.f, g.act_acc);
  }
  if (g.colsum && m == 0)
    put_colsum(g, z * g.scs + n, ((red[1][0][lane] + red[1][1][lane]) + red[1][2][lane]) + red[1][3][lane]);
}

template <int TA, int TB>
__global__ __launch_bounds__(256) void gemm_simple_kernel(GemmArgs g) {
  __shared__ float red[2][4][64];
  simple_body<TA, TB>(g, blockIdx.x, blockIdx.y, red);
}

// A Linear layer's two small products (dX = dY W^T and dW = X^T dY with db)
// in one launch: workgroups [0, nb0) compute problem 0, the rest problem 1,
// each exactly as gemm_simple_kernel does.  One launch less per small layer
// (a C1 step is bound by the host's launch rate).
__global__ __launch_bounds__(256) void gemm_simple_pair_kernel(GemmArgs g0, GemmArgs g1, int nb0) {
  __shared__ float red[2][4][64];
  if ((int)blockIdx.x < nb0) simple_body<0, 1>(g0, blockIdx.x, blockIdx.y, red);
  else simple_body<1, 0>(g1, blockIdx.x - nb0, blockIdx.y, red);
}

// Small products with a long K (an MLP's 784-wide input layer: 64 x 256 x
// 784 and its gradients): one C tile of TT x TT per workgroup of NW waves.
// Wave w multiplies the tile's operands over its K range [w kc, (w + 1) kc)
// (whole 16-deep slabs) on MFMA, the workgroup adds the NW partial tiles in
// wave order through LDS and applies the epilogue: one launch where split K
// needs two (partials, then the reduce), and more workgroups than the
// 64-wide tiles give the same shape.  Within a 16-deep slab lane group q =
// l / 16 feeds k = 4q + e to MFMA step e (the k permutation of the tile
// kernels), so an operand stored k-contiguous is read with one 16-byte load
// per lane and slab (scattered 4-byte loads of it took twice the kernel's
// time), and one stored m- or n-contiguous with four 4-byte loads, 64
// contiguous bytes per k row.  Column sums of B (the bias gradient) come
// from the workgroups of the first tile row, in (wave, lane group) order.
template <int TT, int NW>
constexpr int ks_lds_floats() {
  return NW * TT * TT + NW * 4 * TT;
}

// Four k-consecutive elements p[0..3] of a k-contiguous operand row, zero at
// k >= k1 (k = kq + e).
__device__ __forceinline__ f32x4 ks_row4(const float* p, int kq, int k1, bool vec) {
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
  if (vec && kq + 3 < k1) {
    v = *reinterpret_cast<const f32x4*>(p);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (kq + e < k1) v[e] = p[e];
  }
  return v;
}

template <int TA, int TB, int TT, int NW>
__device__ __forceinline__ void ksplit_body(const GemmArgs& g, int tx, int ty, int64_t z, int kc, float* lds) {
  constexpr int S = TT / 16;
  const int lane = threadIdx.x & 63, li = lane & 15, lq = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int m0 = ty * TT, n0 = tx * TT;
  const float* __restrict__ A = g.A + batch_off(z, g, g.sa, g.sa2);
  const float* __restrict__ B = g.B + batch_off(z, g, g.sb, g.sb2);
  // 16-byte loads along k need 16-byte aligned rows
  const bool a_vec = !TA && g.lda % 4 == 0 && (reinterpret_cast<uintptr_t>(A) & 15) == 0;
  const bool b_vec = TB && g.ldb % 4 == 0 && (reinterpret_cast<uintptr_t>(B) & 15) == 0;
  const bool cs_on = g.colsum != nullptr && ty == 0;
  const int k0 = w * kc, k1 = min(g.K, k0 + kc);
  int am[S], bn[S];
  bool aok[S], bok[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    am[i] = m0 + 16 * i + li;
    aok[i] = am[i] < g.M;
    bn[i] = n0 + 16 * i + li;
    bok[i] = bn[i] < g.N;
  }
  f32x4 acc[S][S];
  float cs[S];
#pragma unroll
  for (int i = 0; i < S; ++i) {
    cs[i] = 0.f;
#pragma unroll
    for (int j = 0; j < S; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // Chunks of SL slabs: every load of a chunk is issued before its products
  // (one memory latency per chunk); slabs past the wave's range are skipped
  // on a wave-uniform branch.
  constexpr int SL = 4 / S;
  for (int kb = k0; kb < k1; kb += 16 * SL) {
    f32x4 a[SL][S], b[SL][S];  // element e: MFMA step e of the slab
#pragma unroll
    for (int t = 0; t < SL; ++t)
#pragma unroll
      for (int i = 0; i < S; ++i) {
        a[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        b[t][i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
#pragma unroll
    for (int t = 0; t < SL; ++t) {
      const int kq = kb + 16 * t + 4 * lq;  // this lane's four k of the slab
      if (kb + 16 * t < k1) {
#pragma unroll
        for (int i = 0; i < S; ++i) {
          if (aok[i]) {
            if (TA) {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (kq + e < k1) a[t][i][e] = A[(int64_t)(kq + e) * g.lda + am[i]];
            } else {
              a[t][i] = ks_row4(A + (int64_t)am[i] * g.lda + kq, kq, k1, a_vec);
            }
          }
          if (bok[i]) {
            if (TB) {
              b[t][i] = ks_row4(B + (int64_t)bn[i] * g.ldb + kq, kq, k1, b_vec);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (kq + e < k1) b[t][i][e] = B[(int64_t)(kq + e) * g.ldb + bn[i]];
            }
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < SL; ++t) {
      if (kb + 16 * t >= k1) break;
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < S; ++i)
#pragma unroll
          for (int j = 0; j < S; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][i][e], b[t][j][e], acc[i][j], 0, 0, 0);
      if (cs_on)
#pragma unroll
        for (int j = 0; j < S; ++j) cs[j] += ((b[t][j][0] + b[t][j][1]) + b[t][j][2]) + b[t][j][3];
    }
  }
  // Partial tiles: result lane l holds rows 4 (l / 16) + r of column l % 16.
  float* part = lds + w * (TT * TT);
#pragma unroll
  for (int i = 0; i < S; ++i)
#pragma unroll
    for (int j = 0; j < S; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) part[(16 * i + 4 * lq + r) * TT + 16 * j + li] = acc[i][j][r];
  float* cpart = lds + NW * TT * TT;  // [wave][lane group][column]
  if (cs_on)
#pragma unroll
    for (int j = 0; j < S; ++j) cpart[(w * 4 + lq) * TT + 16 * j + li] = cs[j];
  __syncthreads();
  const int64_t cz = batch_off(z, g, g.sc, g.sc2);
  for (int o = threadIdx.x; o < TT * TT; o += 64 * NW) {
    const int m = m0 + o / TT, n = n0 + o % TT;
    if (m >= g.M || n >= g.N) continue;
    float v = lds[o];
#pragma unroll
    for (int q = 1; q < NW; ++q) v += lds[q * (TT * TT) + o];
    const int64_t co = cz + (int64_t)m * g.ldc + n;
    float y = g.alpha * v;
    if (g.beta != 0.f) y += g.beta * g.C[co];
    if (g.bias) y += g.bias[z * g.sbias + n];
    g.C[co] = y;
    if (g.act_red) g.act_y[co] = act_rt(g.act_red - 1, y);
    if (g.act_bwd)
      g.act_dx[co] = act_bwd_rt(g.act_bwd - 1, g.act_x[co], y, g.act_acc ? g.act_dx[co] : 0.f, g.act_acc);
  }
  if (cs_on && (int)threadIdx.x < TT && n0 + (int)threadIdx.x < g.N) {
    const int c = threadIdx.x;
    float t = 0.f;
    for (int q = 0; q < 4 * NW; ++q) t += cpart[q * TT + c];
    put_colsum(g, z * g.scs + n0 + c, t);
  }
}

template <int TA, int TB, int TT, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_ksplit_kernel(GemmArgs g, int kc) {
  __shared__ __attribute__((aligned(16))) float lds[ks_lds_floats<TT, NW>()];
  ksplit_body<TA, TB, TT, NW>(g, blockIdx.x, blockIdx.y, blockIdx.z, kc, lds);
}

// A Linear's two backward products on the K-split kernel in one launch:
// workgroups [0, nb0) take dX = dY W^T (NT, tiles of T0, gx0 per tile row),
// the rest dW = X^T dY with db (TN, tiles of T1).
template <int T0, int T1, int NW>
__global__ __launch_bounds__(64 * NW) void gemm_ksplit_pair_kernel(GemmArgs g0, GemmArgs g1, int nb0, int gx0,
                                                                   int gx1, int kc0, int kc1) {
  constexpr int F0 = ks_lds_floats<T0, NW>(), F1 = ks_lds_floats<T1, NW>();
  __shared__ __attribute__((aligned(16))) float lds[F0 > F1 ? F0 : F1];
  const int b = blockIdx.x;
  if (b < nb0) {
    ksplit_body<0, 1, T0, NW>(g0, b % gx0, b / gx0, 0, kc0, lds);
  } else {
    const int c = b - nb0;
    ksplit_body<1, 0, T1, NW>(g1, c % gx1, c / gx1, 0, kc1, lds);
  }
}

// Tile and K splits of a product on the split kernel: the cheapest by a model
// of its time in us -- rounds of workgroups times (stages x time of a stage +
// prologue and epilogue), plus the reduce of the partial products.  A function
// of the shape only, as mle_gemm_ws_bytes needs.  sum: K is the terms of a sum.
struct SplitChoice {
  int tile = kSplitLarge, splits = 1, kchunk = 0;
  double us = 0;
};

SplitChoice choose_split(int M, int N, int K, int batch, bool may_split, bool sum = false) {
  SplitChoice best;
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return best;  // nothing to multiply, nothing to divide
  best.us = 1e30;
  const int st = (K + 31) / 32;
  for (int tile = 0; tile < 3; ++tile) {
    const long long tiles = tiles_of(tile, M, N) * batch;
    // splits that fill one, two or three rounds, none deeper than 4 stages
    long long last = 0;
    for (int target = 0; target <= 6; ++target) {
      long long sp = target == 0 ? 1 : (long long)target * (kChipCus / 2) / tiles;
      if (sp < 1) sp = 1;
      if (sp > st / 4) sp = st / 4 > 1 ? st / 4 : 1;
      if (sp * batch > 65535) sp = 1;
      if (!may_split) sp = 1;
      if (sp == last) continue;
      last = sp;
      int depth = (int)((st + sp - 1) / sp);
      sp = (st + depth - 1) / depth;
      double us = split_grid_us(tile, tiles * sp, depth, !sum);
      // the reduce: 5 us and its bytes, element by element where rows are no multiple of 4
      if (sp > 1) us += 5.0 + (double)(sp + 1) * M * N * batch * 4.0 / (N % 4 == 0 ? 4.0e6 : 1.5e6);
      if (us < best.us) best = {tile, (int)sp, sp > 1 ? depth * 32 : K, us};
    }
  }
  return best;
}

// Split count, and the K range of a split.
int choose_splits(int M, int N, int K, int batch, int& kchunk) {
  const SplitChoice c = choose_split(M, N, K, batch, true);
  kchunk = c.kchunk;
  return c.splits;
}

template <int TA, int TB>
void launch_lds(hipStream_t s, const GemmArgs& g, dim3 grid, bool vec, bool cs) {
  if (vec) {
    if (cs) mle::launch(gemm_kernel<TA, TB, true, true>, grid, NT, 0, s, g);
    else mle::launch(gemm_kernel<TA, TB, true, false>, grid, NT, 0, s, g);
  } else {
    if (cs) mle::launch(gemm_kernel<TA, TB, false, true>, grid, NT, 0, s, g);
    else mle::launch(gemm_kernel<TA, TB, false, false>, grid, NT, 0, s, g);
  }
}

// Bytes spanned by one batch item of an operand stored rows x cols with leading dimension ld.
double extent_bytes(int rows, int cols, int64_t ld) { return ((double)(rows - 1) * (double)ld + cols) * 4.0; }

}  // namespace

// A GEMM call resolved to its arguments, tile shape, grid and kernel family.
struct GemmPlan {
  GemmArgs g;
  int tile = kSplitLarge;
  dim3 grid;
  bool vec = false;     // 16-byte operand loads (gemm_kernel)
  bool tail = false;    // K % 4 != 0 beside a k-contiguous operand (split kernel)
  int which = 0;
  bool cs = false, empty = false;
  bool split = false;   // the split-bf16 kernel; else (not simple, not ksplit) gemm_kernel
  bool simple = false;  // gemm_simple_kernel: one thread per C element, no split
  bool ksplit = false;  // gemm_ksplit_kernel: K split over a workgroup's waves
  int ks_nw = 16;       // its waves per workgroup
  int ks_kc = 0;        // and K range per wave
  double flop = 0, bytes = 0;
};

// Products small enough for gemm_simple_kernel: M of at most 4, K of at most
// 16 or at most 4096 outputs, and at most 4 Mi multiply-adds (one batch
// level, no sum of terms).
// Measured on MI355X with the C1 MLP's products (one launch each, launch
// included): 64 x 10 x 256 4.2 us against 7.6 for split K + reduce; 64 x 256
// x 10 3.9 against 7.2; 256 x 10 x 64 4.1 against 8.4; but 784 x 256 x 64
// 8.1 against 7.0 and 64 x 784 x 256 11.4 against 8.5 on the tile kernels.
static bool simple_shape(int M, int N, int K, int batch, int inner, int terms) {
  return (M <= 4 || K <= 16 || (double)M * N * batch <= 4096.0) &&
         (double)M * N * (double)(K > 0 ? K : 1) * batch <= 4194304.0 && inner == 1 && terms <= 1 &&
         (double)M * N <= 64.0 * 2147483647.0 && batch <= 65535;
}

// Products for gemm_ksplit_kernel: at most 256 Ki outputs and no sum of
// terms, with a K long enough to share over 16 waves but short enough that
// one workgroup's products stay a few microseconds of its CU's matrix cores
// (2 K cycles per SIMD for 16-wide tiles, 8 K for 32-wide).  Tiles of 32 when
// that still gives 128 workgroups, else 16.
static int ksplit_tile(int M, int N, int batch) {
  const long long t32 = (long long)((M + 31) / 32) * ((N + 31) / 32) * batch;
  return t32 >= 128 ? 32 : 16;
}
static bool ksplit_shape(int M, int N, int K, int batch, int terms) {
  if (terms > 1 || K < 32 || (double)M * N * batch > 262144.0) return false;
  const int tt = ksplit_tile(M, N, batch);
  return K <= (tt == 16 ? 4096 : 1024) && (M + tt - 1) / tt <= 65535 && batch <= 65535;
}
// Waves per workgroup: 16 for a long K (one memory latency per 64-deep chunk
// of each wave), 4 when K <= 256 (each wave's share still fits one chunk, and
// the partial tiles to add are fewer).
static int ksplit_nw(int K) { return K <= 256 ? 4 : 16; }
// K range of one wave: whole 16-deep slabs.
static int ksplit_kc(int K, int nw) { return ((K + nw - 1) / nw + 15) / 16 * 16; }

const char* const kFamily[4] = {"gemm_nn", "gemm_nt", "gemm_tn", "gemm_tt"};

static int gemm_plan(GemmPlan& P, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                     int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta, float* C,
                     int64_t ldc, int64_t stride_c, int batch, float* colsum, const float* bias, void* ws,
                     size_t ws_bytes, int inner = 1, int64_t sa2 = 0, int64_t sb2 = 0, int64_t sc2 = 0,
                     int64_t sbias = 0, int64_t scs = 0, int terms = 0, int64_t gsa = 0, int64_t gsb = 0) {
  MLE_CHECK_ARG(M >= 0 && N >= 0 && K >= 0 && batch >= 0, "mle_gemm: negative size");
  P.empty = M == 0 || N == 0 || batch == 0;
  if (P.empty) return MLE_OK;
  MLE_CHECK_ARG(C != nullptr && (K == 0 || (A != nullptr && B != nullptr)), "mle_gemm: null operand");
  MLE_CHECK_ARG(ldc >= N, "mle_gemm: ldc %lld < N %d", (long long)ldc, N);
  MLE_CHECK_ARG(lda >= (trans_a ? M : K) && ldb >= (trans_b ? K : N), "mle_gemm: leading dimension too small");
  MLE_CHECK_ARG(colsum == nullptr || batch == 1 || scs != 0, "mle_gemm: fused colsum over a batch needs a stride");
  MLE_CHECK_ARG((M + 127) / 128 <= 65535 && batch <= 65535, "mle_gemm: grid too large (M %d, batch %d)", M, batch);
  MLE_CHECK_ARG(inner >= 1 && batch % inner == 0, "mle_gemm: batch %d not a multiple of inner %d", batch, inner);
  GemmArgs g{A,    B,    C,       colsum,  lda,  ldb,    ldc,  stride_a, stride_b, stride_c, M,    N,   K,
             alpha, beta, 1,       K,       nullptr, nullptr, bias, inner,    sa2,      sb2,      sc2,      sbias, scs,
             0,     gsa,  gsb,     1,       nullptr, 0,       nullptr, nullptr, nullptr, 0};
  const bool v4 = (lda % 4 == 0) && (ldb % 4 == 0) && (stride_a % 4 == 0) && (stride_b % 4 == 0) &&
                  (sa2 % 4 == 0) && (sb2 % 4 == 0) && (gsa % 4 == 0) && (gsb % 4 == 0) && aligned16(A) &&
                  aligned16(B);
  // The split kernel reads its operands through 31-bit buffer offsets (all
  // terms of a sum, and for a row-contiguous operand the rows that the last
  // stage and the prefetch compute offsets of).
  const int a_rows = trans_a ? K : M, a_cols = trans_a ? M : K;
  const int b_rows = trans_b ? N : K, b_cols = trans_b ? K : N;
  const double t_extra = terms > 1 ? (double)(terms - 1) : 0.0;
  const bool cs = colsum != nullptr;
  bool split = K > 0 && (!cs || (trans_a && !trans_b)) && gsa >= 0 && gsb >= 0 &&
               extent_bytes(a_rows + (trans_a ? 64 : 0), a_cols, lda) + t_extra * 4.0 * (double)gsa < 2147483648.0 - 64 &&
               extent_bytes(b_rows + (trans_b ? 0 : 64), b_cols, ldb) + t_extra * 4.0 * (double)gsb < 2147483648.0 - 64;
  // Folded terms end on whole stages unless both operands are k-contiguous
  // (whose last stage is masked).
  const bool fold = K % 32 == 0 || (!trans_a && trans_b);
  const bool simple = simple_shape(M, N, K, batch, inner, terms);
  const bool ksplit = !simple && ksplit_shape(M, N, K, batch, terms);
  SplitChoice ch;
  if (!simple && !ksplit && terms <= 1) ch = choose_split(M, N, K, batch, ws != nullptr);
  if (terms > 1) ch = choose_split(M, N, (int)std::min(2147483000.0, (double)K * terms), batch, false, true);
  const double items = (double)tiles_of(ch.tile, M, N) * batch * std::max(ch.splits, std::max(terms, 1));
  split = split && items < 1073741824.0;
  if (terms > 1) {
    // Sum of `terms` products.  The workspace is part of the contract either
    // way.  On the split kernel the terms extend its K loop (one
    // accumulator, terms in order, no partials); otherwise one split per
    // term, reduced in term order.
    const size_t need = ((size_t)terms * batch * M * N + (size_t)terms * batch * N) * sizeof(float);
    MLE_CHECK_ARG(ws && ws_bytes >= need, "mle_gemm_sum: workspace of %zu bytes needed", need);
    MLE_CHECK_ARG(terms * batch <= 65535, "mle_gemm_sum: too many terms");
    if (split && fold && (long long)terms * (K / 32 + 1) < (1LL << 24)) {
      g.kterms = terms;
    } else {
      g.grouped = 1;
      g.splits = terms;
      g.part = static_cast<float*>(ws);
      g.part_cs = g.part + (size_t)terms * batch * M * N;
    }
  } else {
    if (ch.splits > 1 && ws_bytes < mle_gemm_ws_bytes(M, N, K, batch)) ch = choose_split(M, N, K, batch, false);
    if (ch.splits > 1) {
      g.splits = ch.splits;
      g.kchunk = ch.kchunk;
      g.part = static_cast<float*>(ws);
      g.part_cs = g.part + (size_t)ch.splits * batch * M * N;
    }
  }
  if (simple) {
    g.splits = 1;
    g.kchunk = K;
    g.part = g.part_cs = nullptr;
    P.simple = true;
  } else if (ksplit) {
    g.splits = 1;
    g.kchunk = K;
    g.part = g.part_cs = nullptr;
    P.ksplit = true;
    P.ks_nw = ksplit_nw(K);
    P.ks_kc = ksplit_kc(K, P.ks_nw);
  }
  // 16-byte stores of C's rows (and reads of the bias and of C)
  g.c_vec = N % 4 == 0 && ldc % 4 == 0 && stride_c % 4 == 0 && sc2 % 4 == 0 && aligned16(C) &&
            (bias == nullptr || (aligned16(bias) && sbias % 4 == 0)) && (g.splits == 1 || aligned16(g.part));
  P.g = g;
  P.tile = ch.tile;
  P.split = split && !P.simple && !P.ksplit;
  P.vec = v4;
  P.tail = K % 4 != 0 && (!trans_a || trans_b);
  P.cs = cs;
  const int tm = P.split ? kSplitTm[ch.tile] : 128, tn = P.split ? kSplitTn[ch.tile] : 128;
  P.grid = dim3((N + tn - 1) / tn, (M + tm - 1) / tm, batch * g.splits);
  if (P.ksplit) {
    const int tt = ksplit_tile(M, N, batch);
    P.grid = dim3((N + tt - 1) / tt, (M + tt - 1) / tt, batch);
  }
  P.which = (trans_a ? 2 : 0) + (trans_b ? 1 : 0);
  P.flop = 2.0 * M * (double)N * K * batch * (terms > 1 ? terms : 1);
  P.bytes = 4.0 * batch * ((double)M * K + (double)K * N + (double)M * N * (beta != 0.f ? 2 : 1));
  return MLE_OK;
}

static int split_items(const GemmPlan& P) { return (int)((long long)P.grid.x * P.grid.y * P.grid.z); }

static void gemm_launch_main(hipStream_t s, const GemmPlan& P, int epi = kEpiPlain) {
  if (P.split) {
    launch_split(s, P.which, P.g, P.tile, P.tail, P.cs, epi, (int)P.grid.x, (int)P.grid.y, split_items(P));
    return;
  }
  if (P.simple) {
    const dim3 grid((unsigned)(((int64_t)P.g.M * P.g.N + 63) / 64), P.grid.z);
    switch (P.which) {
      case 0: mle::launch(gemm_simple_kernel<0, 0>, grid, 256, 0, s, P.g); break;
      case 1: mle::launch(gemm_simple_kernel<0, 1>, grid, 256, 0, s, P.g); break;
      case 2: mle::launch(gemm_simple_kernel<1, 0>, grid, 256, 0, s, P.g); break;
      default: mle::launch(gemm_simple_kernel<1, 1>, grid, 256, 0, s, P.g); break;
    }
    return;
  }
  if (P.ksplit) {
    const bool t32 = ksplit_tile(P.g.M, P.g.N, (int)P.grid.z) == 32;
    const int kc = P.ks_kc;
    if (P.ks_nw == 4) {
      switch (P.which * 2 + (t32 ? 1 : 0)) {
        case 0: mle::launch(gemm_ksplit_kernel<0, 0, 16, 4>, P.grid, 256, 0, s, P.g, kc); break;
        case 1: mle::launch(gemm_ksplit_kernel<0, 0, 32, 4>, P.grid, 256, 0, s, P.g, kc); break;
        case 2: mle::launch(gemm_ksplit_kernel<0, 1, 16, 4>, P.grid, 256, 0, s, P.g, kc); break;
        case 3: mle::launch(gemm_ksplit_kernel<0, 1, 32, 4>, P.grid, 256, 0, s, P.g, kc); break;
        case 4: mle::launch(gemm_ksplit_kernel<1, 0, 16, 4>, P.grid, 256, 0, s, P.g, kc); break;
        case 5: mle::launch(gemm_ksplit_kernel<1, 0, 32, 4>, P.grid, 256, 0, s, P.g, kc); break;
        case 6: mle::launch(gemm_ksplit_kernel<1, 1, 16, 4>, P.grid, 256, 0, s, P.g, kc); break;
        default: mle::launch(gemm_ksplit_kernel<1, 1, 32, 4>, P.grid, 256, 0, s, P.g, kc); break;
      }
    } else {
      switch (P.which * 2 + (t32 ? 1 : 0)) {
        case 0: mle::launch(gemm_ksplit_kernel<0, 0, 16, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        case 1: mle::launch(gemm_ksplit_kernel<0, 0, 32, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        case 2: mle::launch(gemm_ksplit_kernel<0, 1, 16, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        case 3: mle::launch(gemm_ksplit_kernel<0, 1, 32, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        case 4: mle::launch(gemm_ksplit_kernel<1, 0, 16, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        case 5: mle::launch(gemm_ksplit_kernel<1, 0, 32, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        case 6: mle::launch(gemm_ksplit_kernel<1, 1, 16, 16>, P.grid, 1024, 0, s, P.g, kc); break;
        default: mle::launch(gemm_ksplit_kernel<1, 1, 32, 16>, P.grid, 1024, 0, s, P.g, kc); break;
      }
    }
    return;
  }
  switch (P.which) {
    case 0: launch_lds<0, 0>(s, P.g, P.grid, P.vec, P.cs); break;
    case 1: launch_lds<0, 1>(s, P.g, P.grid, P.vec, P.cs); break;
    case 2: launch_lds<1, 0>(s, P.g, P.grid, P.vec, P.cs); break;
    default: launch_lds<1, 1>(s, P.g, P.grid, P.vec, P.cs); break;
  }
}

static void gemm_launch_reduce(hipStream_t s, const GemmPlan& P) {
  const GemmArgs& g = P.g;
  if (g.splits <= 1) return;
  const bool rv = g.N % 4 == 0 && g.ldc % 4 == 0 && g.sc % 4 == 0 && g.sc2 % 4 == 0 && aligned16(g.C) &&
                  aligned16(g.part) && (!g.bias || (aligned16(g.bias) && g.sbias % 4 == 0));
  const int w = rv ? 4 : 1;
  const int batch = (int)P.grid.z / g.splits;
  const int64_t units = (int64_t)batch * g.M * (g.N / w);
  const unsigned nmain = (unsigned)((units + 63) / 64);
  const unsigned ncs = g.colsum ? (unsigned)(((int64_t)batch * g.N + 255) / 256) : 0u;
  if (rv) mle::launch(split_reduce_kernel<true>, nmain + ncs, 256, 0, s, g, units, nmain);
  else mle::launch(split_reduce_kernel<false>, nmain + ncs, 256, 0, s, g, units, nmain);
}

// True when the split kernel's epilogue can take an extra output of C's shape
// (row statistics, an activation): whole 64-column blocks per wave, one split.
static bool epilogue_ok(const GemmPlan& P) {
  return !P.empty && P.split && !P.tail && P.g.c_vec && P.g.splits == 1 && P.tile != kSplitSmall;
}

static int gemm_impl(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                     int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta, float* C,
                     int64_t ldc, int64_t stride_c, int batch, float* colsum, const float* bias, void* ws,
                     size_t ws_bytes, int inner = 1, int64_t sa2 = 0, int64_t sb2 = 0, int64_t sc2 = 0,
                     int64_t sbias = 0, int64_t scs = 0, int terms = 0, int64_t gsa = 0, int64_t gsb = 0) {
  GemmPlan P;
  const int rc = gemm_plan(P, trans_a, trans_b, M, N, K, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C, ldc,
                           stride_c, batch, colsum, bias, ws, ws_bytes, inner, sa2, sb2, sc2, sbias, scs, terms, gsa,
                           gsb);
  if (rc != MLE_OK || P.empty) return rc;
  hipStream_t s = as_stream(stream);
  {
    // The probe times the whole product: the GEMM kernel and, with split K,
    // the reduce that completes C.
    ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
    gemm_launch_main(s, P);
    gemm_launch_reduce(s, P);
  }
  return check_launch(kFamily[P.which]);
}

extern "C" {

size_t mle_gemm_ws_bytes(int M, int N, int K, int batch) {
  int kchunk;
  int splits = choose_splits(M, N, K, batch, kchunk);
  // A product of at most 4096 outputs and 4 Mi multiply-adds runs on the simple
  // kernel, which leaves the workspace unused; its size stays that of one split
  // per 32 deep stage, at most 768.
  const double outs = (double)M * N * batch;
  if (outs > 0.0 && outs <= 4096.0 && simple_shape(M, N, K, batch, 1, 0)) splits = std::max(splits, std::min(768, (K + 31) / 32));
  if (splits <= 1) return 0;
  return ((size_t)splits * batch * M * N + (size_t)splits * batch * N) * sizeof(float);
}

size_t mle_gemm_sum_ws_bytes(int M, int N, int terms) {
  if (terms <= 1) return 0;
  return ((size_t)terms * M * N + (size_t)terms * N) * sizeof(float);
}

int mle_gemm_batched_ex(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                        int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta,
                        float* C, int64_t ldc, int64_t stride_c, int batch, float* colsum, int64_t stride_colsum,
                        const float* bias, int64_t stride_bias, void* ws, size_t ws_bytes) {
  return gemm_impl(stream, trans_a, trans_b, M, N, K, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C, ldc,
                   stride_c, batch, colsum, bias, ws, ws_bytes, 1, 0, 0, 0, stride_bias, stride_colsum);
}

int mle_gemm_sum(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                 int64_t lda, int64_t stride_a_term, const float* B, int64_t ldb, int64_t stride_b_term, float beta,
                 float* C, int64_t ldc, int terms, void* ws, size_t ws_bytes) {
  MLE_CHECK_ARG(terms >= 1, "mle_gemm_sum: terms %d", terms);
  return gemm_impl(stream, trans_a, trans_b, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, nullptr,
                   nullptr, ws, ws_bytes, 1, 0, 0, 0, 0, 0, terms, stride_a_term, stride_b_term);
}

int mle_gemm_rowstats(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                      int64_t lda, const float* B, int64_t ldb, float beta, float* C, int64_t ldc, const float* bias,
                      float* rowpart, int64_t ldp, void* ws, size_t ws_bytes) {
  MLE_CHECK_ARG(rowpart != nullptr && ldp >= 2 * (int64_t)((N + 63) / 64) && (ldp % 2) == 0 &&
                    (reinterpret_cast<uintptr_t>(rowpart) & 7) == 0,
                "mle_gemm_rowstats: rowpart needs %d float pairs per row (8-byte aligned)", (N + 63) / 64);
  GemmPlan P;
  const int rc = gemm_plan(P, trans_a, trans_b, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, nullptr,
                           bias, ws, ws_bytes);
  if (rc != MLE_OK || P.empty) return rc;
  hipStream_t s = as_stream(stream);
  const bool fused = epilogue_ok(P) && P.which == 0;
  if (fused) P.g.rowpart = rowpart, P.g.rp_ld = ldp;
  {
    ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
    gemm_launch_main(s, P, fused ? kEpiRowstats : kEpiPlain);
  }
  gemm_launch_reduce(s, P);
  if (!fused) {
    const int64_t waves = (int64_t)M * ((N + 63) / 64);
    MLE_CHECK_ARG((waves + 3) / 4 <= 2147483647LL, "mle_gemm_rowstats: too many rows");
    mle::launch(rowstats_kernel, (unsigned)((waves + 3) / 4), 256, 0, s, C, ldc, M, N, rowpart, ldp);
  }
  return check_launch("mle_gemm_rowstats");
}

int mle_gemm_act_fwd(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                     int64_t lda, const float* B, int64_t ldb, float beta, float* C, const float* bias, int kind,
                     float* Y, void* ws, size_t ws_bytes) {
  MLE_CHECK_ARG(Y != nullptr && kind >= MLE_RELU && kind <= MLE_LEAKY_RELU, "mle_gemm_act_fwd: bad argument");
  GemmPlan P;
  int rc = gemm_plan(P, trans_a, trans_b, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, N, 0, 1, nullptr, bias, ws,
                     ws_bytes);
  if (rc != MLE_OK || P.empty) return rc;
  hipStream_t s = as_stream(stream);
  if (epilogue_ok(P) && P.which == 0 && aligned16(Y)) {
    P.g.act_y = Y;
    P.g.act_kind = kind;
    {
      ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
      gemm_launch_main(s, P, kEpiActFwd);
    }
    return check_launch("mle_gemm_act_fwd");
  }
  // Split K: the reduce that completes C writes Y too; on the K-split kernel
  // its epilogue does.
  if ((P.g.splits > 1 && aligned16(Y)) || P.ksplit) {
    P.g.act_y = Y;
    P.g.act_red = 1 + kind;
    ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
    gemm_launch_main(s, P);
    gemm_launch_reduce(s, P);
    return check_launch("mle_gemm_act_fwd");
  }
  {
    ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
    gemm_launch_main(s, P);
  }
  gemm_launch_reduce(s, P);
  rc = check_launch("mle_gemm_act_fwd");
  if (rc != MLE_OK) return rc;
  return mle_act_fwd(stream, kind, C, Y, (size_t)M * N);
}

int mle_gemm_act_bwd(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                     int64_t lda, const float* B, int64_t ldb, float beta, float* C, int kind, const float* X,
                     float* dX, int accumulate_dx, void* ws, size_t ws_bytes) {
  MLE_CHECK_ARG(X != nullptr && dX != nullptr && kind >= MLE_RELU && kind <= MLE_LEAKY_RELU,
                "mle_gemm_act_bwd: bad argument");
  GemmPlan P;
  int rc = gemm_plan(P, trans_a, trans_b, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, N, 0, 1, nullptr, nullptr,
                     ws, ws_bytes);
  if (rc != MLE_OK || P.empty) return rc;
  hipStream_t s = as_stream(stream);
  if (P.simple || P.ksplit) {  // the small-product kernels' epilogue
    P.g.act_x = X;
    P.g.act_dx = dX;
    P.g.act_acc = accumulate_dx ? 1 : 0;
    P.g.act_bwd = 1 + kind;
    {
      ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
      gemm_launch_main(s, P);
    }
    return check_launch("mle_gemm_act_bwd");
  }
  if (epilogue_ok(P) && P.which == 1 && aligned16(X) && aligned16(dX)) {
    P.g.act_x = X;
    P.g.act_dx = dX;
    P.g.act_acc = accumulate_dx ? 1 : 0;
    P.g.act_kind = kind;
    {
      ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
      gemm_launch_main(s, P, kEpiActBwd);
    }
    return check_launch("mle_gemm_act_bwd");
  }
  {
    ProbeScope probe(kFamily[P.which], s, P.flop, P.bytes);
    gemm_launch_main(s, P);
  }
  gemm_launch_reduce(s, P);
  rc = check_launch("mle_gemm_act_bwd");
  if (rc != MLE_OK) return rc;
  return mle_act_bwd(stream, kind, X, C, dX, (size_t)M * N, accumulate_dx);
}

}  // extern "C"

// The Linear backward's two products in one grid (gemm_split_pair_kernel): the
// tile and the weight gradient's K splits.  Its depth is cut to about the
// chip's share of the whole work, so that no CU is left with one deep tile
// while the others are done; the input gradient is not split.  `us` is the
// model's time of the pair, the reduce included.  A function of the shape only.
struct PairChoice {
  int tile = kSplitLarge, splits = 1, kchunk = 0;
  double us = 1e30;
};
static PairChoice choose_pair(int rows, int in, int out, int layers) {
  PairChoice best;
  if (rows <= 0 || in <= 0 || out <= 0) return best;
  for (int tile = 0; tile < 2; ++tile) {
    const long long n0 = tiles_of(tile, rows, in), t1 = tiles_of(tile, in, out) * layers;
    const long long d0 = (long long)layers * ((out + 31) / 32), st1 = (rows + 31) / 32;
    if (n0 > (1 << 24) || t1 > (1 << 24)) continue;
    const long long share = (n0 * d0 + t1 * st1 + kChipCus - 1) / kChipCus;
    const long long want = share > 0 ? st1 / share : 1;
    for (long long sp : {1LL, want, want + 1, 2 * want + 1}) {
      sp = std::max(1LL, std::min({sp, st1 / 4, 65535LL / layers}));
      const long long d1 = (st1 + sp - 1) / sp;
      sp = (st1 + d1 - 1) / d1;
      const long long n1 = t1 * sp;
      // dW's n1 items first, then dX's n0: `full` rounds of the former on
      // every CU, a last one on `busy` CUs, and the earliest end of the n0.
      const double u0 = d0 * kStageUs[tile] + kTileUs[tile], u1 = d1 * kStageUs[tile] + kTileUs[tile];
      const long long full = n1 / kChipCus, busy = n1 % kChipCus, idle = kChipCus - busy;
      double us = busy ? u1 : 0.0;
      for (long long k = 0, done = 0; done < n0 && k < 4096; ++k) {  // k dX rounds on the idle CUs
        const long long late = k * u0 > u1 ? (long long)((k * u0 - u1) / u0) : 0;
        done = idle * k + busy * late;
        us = std::max(us, k * u0);
        if (done < n0 && idle * k + busy * (late + 1) >= n0) {
          us = std::max(us, u1 + (late + 1) * u0);
          break;
        }
      }
      us += (double)full * u1;
      if (sp > 1) us += 5.0 + (double)(sp + 1) * in * out * layers * 4.0 / 4.0e6;
      if (us < best.us) best = {tile, (int)sp, (int)(sp > 1 ? d1 * 32 : rows), us};
    }
  }
  return best;
}

extern "C" {

size_t mle_linear_bwd_ws_bytes(int rows, int in, int out, int layers) {
  const size_t dx = layers > 1 ? mle_gemm_sum_ws_bytes(rows, in, layers) : mle_gemm_ws_bytes(rows, in, out, 1);
  size_t dw = mle_gemm_ws_bytes(in, out, rows, layers);
  // (a product on a small-product kernel never shares a launch with a split one)
  const bool small = simple_shape(rows, in, out, 1, 1, layers > 1 ? layers : 0) || ksplit_shape(rows, in, out, 1, layers > 1 ? layers : 0) ||
                     simple_shape(in, out, rows, layers, 1, 0) || ksplit_shape(in, out, rows, layers, 0);
  PairChoice pc;
  if (!small) pc = choose_pair(rows, in, out, layers);
  if (pc.splits > 1) dw = std::max(dw, (size_t)pc.splits * layers * ((size_t)in * out + out) * sizeof(float));
  return std::max(dx, dw);
}

int mle_linear_bwd(mle_stream stream, int rows, int in, int out, int layers, const float* X, const float* dY,
                   int64_t stride_dy, const float* W, int64_t stride_w, float* dX, int accumulate_dx, float* dW,
                   float* db, int64_t stride_db, void* ws, size_t ws_bytes) {
  return mle_linear_bwd_ex(stream, rows, in, out, layers, X, dY, stride_dy, W, stride_w, dX, accumulate_dx, dW, db,
                           stride_db, 1, ws, ws_bytes);
}

}  // extern "C"

// Linear backward, optionally with the backward of the activation whose
// output is X' = this layer's input: act_dx (+)= act'(act_x) * dX (act_kind
// < 0: none).  On the small-product kernels the activation gradient is their
// epilogue; otherwise it is a pass after the products.
static int linear_bwd_impl(mle_stream stream, int rows, int in, int out, int layers, const float* X, const float* dY,
                           int64_t stride_dy, const float* W, int64_t stride_w, float* dX, int accumulate_dx,
                           float* dW, float* db, int64_t stride_db, int accumulate_dw, int act_kind,
                           const float* act_x, float* act_dx, int act_acc, void* ws, size_t ws_bytes) {
  MLE_CHECK_ARG(rows >= 0 && in >= 0 && out >= 0 && layers >= 1, "mle_linear_bwd: bad sizes");
  MLE_CHECK_ARG(layers == 1 || (stride_dy != 0 && stride_w != 0 && (db == nullptr || stride_db != 0)),
                "mle_linear_bwd: %d layers need strides", layers);
  MLE_CHECK_ARG(ws_bytes >= mle_linear_bwd_ws_bytes(rows, in, out, layers) && (ws || ws_bytes == 0),
                "mle_linear_bwd: workspace of %zu bytes needed", mle_linear_bwd_ws_bytes(rows, in, out, layers));
  // dX (+)= sum_l dY_l W_l^T: NT, rows x in, depth out (terms over layers).
  GemmPlan P0, P1;
  int rc = gemm_plan(P0, 0, 1, rows, in, out, 1.0f, dY, out, 0, W, out, 0, accumulate_dx ? 1.0f : 0.0f, dX, in, 0, 1,
                     nullptr, nullptr, ws, ws_bytes, 1, 0, 0, 0, 0, 0, layers > 1 ? layers : 0, stride_dy, stride_w);
  if (rc != MLE_OK) return rc;
  // dW_l (+)= X^T dY_l and db_l (+)= colsum dY_l: TN, in x out, depth rows.
  rc = gemm_plan(P1, 1, 0, in, out, rows, 1.0f, X, in, 0, dY, out, stride_dy, accumulate_dw ? 1.0f : 0.0f, dW, out,
                 stride_w, layers, db, nullptr, ws, ws_bytes, 1, 0, 0, 0, 0, stride_db);
  if (rc != MLE_OK) return rc;
  P1.g.cs_assign = accumulate_dw ? 0 : 1;
  hipStream_t s = as_stream(stream);
  bool act_done = act_kind < 0 || P0.empty;
  if (!act_done && (P0.simple || P0.ksplit)) {
    P0.g.act_bwd = 1 + act_kind;
    P0.g.act_x = act_x;
    P0.g.act_dx = act_dx;
    P0.g.act_acc = act_acc ? 1 : 0;
    act_done = true;
  }
  // The activation pass when no epilogue took it.
  auto finish = [&](int code) {
    if (code != MLE_OK || act_done) return code;
    return mle_act_bwd(stream, act_kind, act_x, dX, act_dx, (size_t)rows * in, act_acc);
  };
  // Both small (gemm_simple_kernel, one batch item): one launch.
  if (!P0.empty && !P1.empty && P0.simple && P1.simple && P0.grid.z == 1 && P1.grid.z == 1) {
    const unsigned nb0 = (unsigned)(((int64_t)P0.g.M * P0.g.N + 63) / 64);
    const unsigned nb1 = (unsigned)(((int64_t)P1.g.M * P1.g.N + 63) / 64);
    {
      ProbeScope probe("gemm_pair", s, P0.flop + P1.flop, P0.bytes + P1.bytes);
      mle::launch(gemm_simple_pair_kernel, dim3(nb0 + nb1, 1), 256, 0, s, P0.g, P1.g, (int)nb0);
    }
    return finish(check_launch("gemm_pair"));
  }
  // Both on the K-split kernel (one batch item): one launch.
  if (!P0.empty && !P1.empty && P0.ksplit && P1.ksplit && P0.grid.z == 1 && P1.grid.z == 1) {
    const int gx0 = (int)P0.grid.x, gx1 = (int)P1.grid.x;
    const int nb0 = gx0 * (int)P0.grid.y, nb1 = gx1 * (int)P1.grid.y;
    const bool w0 = ksplit_tile(P0.g.M, P0.g.N, 1) == 32, w1 = ksplit_tile(P1.g.M, P1.g.N, 1) == 32;
    // one workgroup size for both: the larger wave count, K ranges re-cut for it
    const int nw = std::max(P0.ks_nw, P1.ks_nw);
    const int kc0 = ksplit_kc(P0.g.K, nw), kc1 = ksplit_kc(P1.g.K, nw);
    auto k = nw == 4 ? (w0 ? (w1 ? gemm_ksplit_pair_kernel<32, 32, 4> : gemm_ksplit_pair_kernel<32, 16, 4>)
                           : (w1 ? gemm_ksplit_pair_kernel<16, 32, 4> : gemm_ksplit_pair_kernel<16, 16, 4>))
                     : (w0 ? (w1 ? gemm_ksplit_pair_kernel<32, 32, 16> : gemm_ksplit_pair_kernel<32, 16, 16>)
                           : (w1 ? gemm_ksplit_pair_kernel<16, 32, 16> : gemm_ksplit_pair_kernel<16, 16, 16>));
    {
      ProbeScope probe("gemm_pair", s, P0.flop + P1.flop, P0.bytes + P1.bytes);
      mle::launch(k, dim3((unsigned)(nb0 + nb1)), 64 * nw, 0, s, P0.g, P1.g, nb0, gx0, gx1, kc0, kc1);
    }
    return finish(check_launch("gemm_pair"));
  }
  // One launch when both run on the split kernel without a K tail, and the
  // model says that sharing the chip beats one product after the other.
  if (!P0.empty && !P1.empty && P0.split && P1.split && !P0.tail && !P1.tail && !P0.g.grouped && !P1.g.grouped) {
    const SplitChoice c0 = choose_split(rows, in, out * layers, 1, layers <= 1, layers > 1);
    const SplitChoice c1 = choose_split(in, out, rows, layers, true);
    const PairChoice pc = choose_pair(rows, in, out, layers);
    const double parts = (double)pc.splits * layers * ((double)in * out + out) * sizeof(float);
    if (pc.us < c0.us + c1.us + 3.0 && (pc.splits == 1 || (ws && (double)ws_bytes >= parts))) {
      GemmArgs g0 = P0.g, g1 = P1.g;
      g0.splits = 1;
      g0.kchunk = out;
      g1.splits = pc.splits;
      g1.kchunk = pc.kchunk;
      g1.part = static_cast<float*>(ws);
      g1.part_cs = g1.part + (size_t)pc.splits * layers * in * out;
      if (pc.splits > 1 && !aligned16(ws)) g1.c_vec = 0;
      const int tm = kSplitTm[pc.tile], tn = kSplitTn[pc.tile];
      PairGrid pg;
      pg.gx0 = (in + tn - 1) / tn, pg.gy0 = (rows + tm - 1) / tm, pg.items0 = pg.gx0 * pg.gy0;
      pg.gx1 = (out + tn - 1) / tn, pg.gy1 = (in + tm - 1) / tm, pg.items1 = pg.gx1 * pg.gy1 * layers * pc.splits;
      pg.start0 = (pg.items1 + 7) / 8 * 8;
      {
        ProbeScope probe("gemm_pair", s, P0.flop + P1.flop, P0.bytes + P1.bytes);
        launch_split_pair(s, g0, g1, pc.tile, P1.cs, pg);
        GemmPlan R = P1;
        R.g = g1;
        R.grid.z = layers * pc.splits;
        gemm_launch_reduce(s, R);
      }
      return finish(check_launch("gemm_pair"));
    }
  }
  // Otherwise one launch each, in order (they may share the workspace).
  if (!P0.empty) {
    ProbeScope probe(kFamily[P0.which], s, P0.flop, P0.bytes);
    gemm_launch_main(s, P0);
    gemm_launch_reduce(s, P0);
  }
  rc = check_launch(kFamily[P0.which]);
  if (rc != MLE_OK || P1.empty) return finish(rc);
  {
    ProbeScope probe(kFamily[P1.which], s, P1.flop, P1.bytes);
    gemm_launch_main(s, P1);
    gemm_launch_reduce(s, P1);
  }
  return finish(check_launch(kFamily[P1.which]));
}


extern "C" {

int mle_linear_bwd_ex(mle_stream stream, int rows, int in, int out, int layers, const float* X, const float* dY,
                      int64_t stride_dy, const float* W, int64_t stride_w, float* dX, int accumulate_dx, float* dW,
                      float* db, int64_t stride_db, int accumulate_dw, void* ws, size_t ws_bytes) {
  return linear_bwd_impl(stream, rows, in, out, layers, X, dY, stride_dy, W, stride_w, dX, accumulate_dx, dW, db,
                         stride_db, accumulate_dw, -1, nullptr, nullptr, 0, ws, ws_bytes);
}

int mle_linear_bwd_act(mle_stream stream, int rows, int in, int out, const float* X, const float* dY,
                       const float* W, float* dX, int accumulate_dx, float* dW, float* db, int accumulate_dw,
                       int act_kind, const float* act_x, float* act_dx, int act_accumulate, void* ws,
                       size_t ws_bytes) {
  MLE_CHECK_ARG(act_kind >= MLE_RELU && act_kind <= MLE_LEAKY_RELU && act_x != nullptr && act_dx != nullptr,
                "mle_linear_bwd_act: bad activation argument");
  MLE_CHECK_ARG(act_dx != dX && act_dx != dY && act_dx != X && act_dx != W,
                "mle_linear_bwd_act: act_dx must not alias X, dY, W or dX");
  return linear_bwd_impl(stream, rows, in, out, 1, X, dY, 0, W, 0, dX, accumulate_dx, dW, db, 0, accumulate_dw,
                         act_kind, act_x, act_dx, act_accumulate, ws, ws_bytes);
}

int mle_gemm(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
             int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta, float* C,
             int64_t ldc, int64_t stride_c, int batch, float* colsum) {
  return gemm_impl(stream, trans_a, trans_b, M, N, K, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C, ldc,
                   stride_c, batch, colsum, nullptr, nullptr, 0);
}

int mle_gemm_ex(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                int64_t lda, int64_t stride_a, const float* B, int64_t ldb, int64_t stride_b, float beta, float* C,
                int64_t ldc, int64_t stride_c, int batch, float* colsum, const float* bias, void* ws,
                size_t ws_bytes) {
  return gemm_impl(stream, trans_a, trans_b, M, N, K, alpha, A, lda, stride_a, B, ldb, stride_b, beta, C, ldc,
                   stride_c, batch, colsum, bias, ws, ws_bytes);
}

int mle_gemm_grid(mle_stream stream, int trans_a, int trans_b, int M, int N, int K, float alpha, const float* A,
                  int64_t lda, int64_t sa_outer, int64_t sa_inner, const float* B, int64_t ldb, int64_t sb_outer,
                  int64_t sb_inner, float beta, float* C, int64_t ldc, int64_t sc_outer, int64_t sc_inner, int outer,
                  int inner, void* ws, size_t ws_bytes) {
  MLE_CHECK_ARG(outer >= 0 && inner >= 1, "mle_gemm_grid: bad batch grid %d x %d", outer, inner);
  return gemm_impl(stream, trans_a, trans_b, M, N, K, alpha, A, lda, sa_outer, B, ldb, sb_outer, beta, C, ldc,
                   sc_outer, outer * inner, nullptr, nullptr, ws, ws_bytes, inner, sa_inner, sb_inner, sc_inner);
}

}  // extern "C"
