// Convolution as implicit GEMM on the split-bf16 tile engine (split_core.hpp):
//
//   forward : C[co][(b,oh,ow)]  = W[co][(ci,kh,kw)] * im2col(X)[(ci,kh,kw)][(b,oh,ow)]
//   dgrad   : C[ci][(b,ih,iw)]  = W^T[ci][(co,kh,kw)] * gather(dY)[(co,kh,kw)][(b,ih,iw)]
//   wgrad   : C[co][(ci,kh,kw)] = dY[co][(b,oh,ow)] * im2col(X)^T[(b,oh,ow)][(ci,kh,kw)]
//
// (CV2D, CV2D_GradInput, GV2D: Engine/kernels.cu:985-1089.)  What the gathers
// cost bounds the small maps, the matrix cores (and their power) the large
// ones.  Forward and dgrad: the workgroup tabulates its k in LDS before the K
// loop (source offset of the tap, tap bit, and for dgrad the weight's offset);
// a pixel keeps its base offset and one bit per tap that says whether the tap
// falls on the image, and an element costs an add, a bit test and a select.
// (Channel and tap of each k by scalar multiplications in the loop: 61 against
// 48 us for the forward of 32 x 128 -> 192 channels on 14 x 14.)
// wgrad: the same table over the workgroup's pixels (source offset, tap bits,
// dY offset), CHUNK of them at a time.
#include "conv_args.hpp"
#include "gemm_tiles.hpp"
#include "split_core.hpp"

using namespace split;

namespace conv {
namespace {

using LargeTile = gemm::LargeTile;
using MediumTile = gemm::MediumTile;
using SmallTile = gemm::SmallTile;
using PairedTile = gemm::PairedTile;
using WideTile = Shape<4, 4, 2, 4>;     // 128 channels x 256 pixels
using SlimTile = Shape<2, 4, 2, 2, 2>;  // 64 channels x 128 pixels

constexpr int kMaxTaps = 32;

struct GatherArgs {
  const float* src;   // x (forward) or dy (dgrad)
  const float* wt;
  const float* bias;  // forward only (nullable)
  float* out;
  uint32_t src_bytes, wt_bytes;
  int M, N, K;
  ConvGeom g;
  int acc, c_vec;
};

// The k table: one period of 32 khw k (whole stages, whole channels); 32
// channels further on, every offset is larger by a constant.
struct TapTable {
  uint2* tap;     // byte offset of the tap from the pixel's base, tap bit
  uint32_t* wt;   // dgrad: byte offset of the weight from its row's
};
template <bool DG>
__device__ __forceinline__ void fill_table(const GatherArgs& a, const TapTable& t, int tid, int nth) {
  const ConvGeom& g = a.g;
  const int khw = g.kh * g.kw;
  for (int k = tid; k < KS * khw; k += nth) {
    const int ch = k / khw, tap = k - ch * khw, kh = tap / g.kw, kw = tap - kh * g.kw;
    // dgrad: a tap that is valid for the pixel has its remainder, so whole strides remain
    const int o = DG ? ch * g.oh * g.ow - (kh / g.stride) * g.ow - kw / g.stride : ch * g.h * g.w + kh * g.w + kw;
    t.tap[k] = make_uint2((uint32_t)o * 4u, 1u << tap);
    if (DG) t.wt[k] = (uint32_t)(ch * a.M * khw + tap) * 4u;
  }
}
// A loader's place in it: the first k, within the period, of this lane
// group's next stage; next() says when a period is passed.  k past K stand for
// channels past the last: the weights read there are 0 (masked, or past their
// buffer), so whatever the other operand reads adds nothing.
struct TapCursor {
  int at, period;
  uint32_t per_period;
  __device__ __forceinline__ uint32_t init(int k0, int lane_group, int khw, uint32_t bytes) {
    period = KS * khw;
    per_period = bytes;
    at = k0 % period + 4 * lane_group;
    return (uint32_t)(k0 / period) * bytes;  // of the periods before k0
  }
  __device__ __forceinline__ bool next() {
    at += KS;
    if (at < period) return false;
    at -= period;
    return true;
  }
};

// Gathered operand: R pixels of the output grid as rows, k = (channel, tap).
template <bool DG, int R, int NTH>
struct PixLoad : Chunks<R * 4 / NTH, false> {
  using Base = Chunks<R * 4 / NTH, false>;
  using Base::NC;
  __amdgpu_buffer_rsrc_t rs;
  const uint2* tab;
  uint32_t base[NC];
  unsigned bits[NC];  // bit t: tap t reads inside the source
  uint2 e[8];
  TapCursor cur;      // the same for a wave
  __device__ __forceinline__ void init(const GatherArgs& a, const uint2* table, int k0, int n0, int t) {
    const ConvGeom& g = a.g;
    rs = rsrc(a.src, a.src_bytes);
    tab = table;
    const uint32_t run = cur.init(k0, __builtin_amdgcn_readfirstlane(t >> 6) & 3, g.kh * g.kw,
                                  (uint32_t)(DG ? g.oh * g.ow : g.h * g.w) * (4u * KS));
    const int ph = DG ? g.h : g.oh, pw = DG ? g.w : g.ow, phw = ph * pw;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      int r, q;
      chunk_at<true, NTH>(t, c, r, q);
      this->place(c, r, q);
      const int n = n0 + r;
      const int b = n / phw, pix = n - b * phw, py = pix / pw, px = pix - py * pw;
      unsigned ybits = 0, xbits = 0;  // valid kh, kw
      int o;
      if (DG) {
        const int Y = py + g.pad, X = px + g.pad;
        for (int i = 0; i < g.kh; ++i)
          ybits |= (unsigned)(Y - i >= 0 && (Y - i) % g.stride == 0 && (Y - i) / g.stride < g.oh) << i;
        for (int i = 0; i < g.kw; ++i)
          xbits |= (unsigned)(X - i >= 0 && (X - i) % g.stride == 0 && (X - i) / g.stride < g.ow) << i;
        o = b * g.cout * g.oh * g.ow + (Y / g.stride) * g.ow + X / g.stride;
      } else {
        const int Y = py * g.stride - g.pad, X = px * g.stride - g.pad;
        for (int i = 0; i < g.kh; ++i) ybits |= (unsigned)((unsigned)(Y + i) < (unsigned)g.h) << i;
        for (int i = 0; i < g.kw; ++i) xbits |= (unsigned)((unsigned)(X + i) < (unsigned)g.w) << i;
        o = b * g.cin * g.h * g.w + Y * g.w + X;
      }
      unsigned m = 0;
      for (int i = 0; i < g.kh; ++i)
        if (ybits >> i & 1u) m |= xbits << (i * g.kw);
      bits[c] = n < a.N ? m : 0u;
      base[c] = (uint32_t)o * 4u + run;
    }
  }
  __device__ __forceinline__ void pre() {
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = tab[cur.at + chunk_k(j)];
  }
  __device__ __forceinline__ void load(float (&x)[NC][8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) x[c][j] = ld1(rs, bits[c] & e[j].y ? base[c] + e[j].x : kOOB);
    const uint32_t step = cur.next() ? cur.per_period : 0u;
#pragma unroll
    for (int c = 0; c < NC; ++c) base[c] += step;
  }
};

// The weights of the dgrad: rows ci, k = (co, tap) at (co * cin + ci) * khw + tap.
template <int R, int NTH>
struct WeightLoad : Chunks<R * 4 / NTH, false> {
  using Base = Chunks<R * 4 / NTH, false>;
  using Base::NC;
  __amdgpu_buffer_rsrc_t rs;
  const uint32_t* tab;
  uint32_t off[NC], e[8];
  TapCursor cur;
  __device__ __forceinline__ void init(const GatherArgs& a, const uint32_t* table, int k0, int m0, int t) {
    rs = rsrc(a.wt, a.wt_bytes);
    tab = table;
    const int khw = a.g.kh * a.g.kw;
    const uint32_t run = cur.init(k0, __builtin_amdgcn_readfirstlane(t >> 6) & 3, khw, (uint32_t)(a.M * khw) * (4u * KS));
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      int r, q;
      chunk_at<true, NTH>(t, c, r, q);
      this->place(c, r, q);
      off[c] = m0 + r < a.M ? (uint32_t)((m0 + r) * khw) * 4u + run : kOOB;
    }
  }
  __device__ __forceinline__ void pre() {
#pragma unroll
    for (int j = 0; j < 8; ++j) e[j] = tab[cur.at + chunk_k(j)];
  }
  __device__ __forceinline__ void load(float (&x)[NC][8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int c = 0; c < NC; ++c) x[c][j] = ld1(rs, off[c] + e[j]);
    const uint32_t step = cur.next() ? cur.per_period : 0u;
#pragma unroll
    for (int c = 0; c < NC; ++c) off[c] += step;
  }
};

// True on every thread when some thread of the workgroup saw a value the split
// cannot represent; then v (+ lo) is cleared for fp32_tile.
template <class S>
__device__ __forceinline__ bool redo(f32x4 (&v)[S::BI][S::BN], f32x4 (&lo)[S::BI][S::BN]) {
  if (!__syncthreads_or(needs_fp32<S>(v, lo))) return false;
#pragma unroll
  for (int i = 0; i < S::BI; ++i)
#pragma unroll
    for (int n = 0; n < S::BN; ++n) v[i][n] = lo[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  return true;
}

template <class S, bool DG, bool TAIL>
__global__ __launch_bounds__(S::NTH * S::KG, 2) void conv_split_kernel(GatherArgs a, int gx, int gy, int items) {
  constexpr int BI = S::BI, BN = S::BN;
  __shared__ __attribute__((aligned(16))) char lds[S::LDS * S::KG];
  int tm, tn, z;
  gemm::item_tile(blockIdx.x, items, gx, gy, tm, tn, z);
  const int m0 = tm * S::TM, n0 = tn * S::TN, tid = threadIdx.x;
  extern __shared__ __attribute__((aligned(16))) char table[];
  const TapTable tab{reinterpret_cast<uint2*>(table),
                     reinterpret_cast<uint32_t*>(table + (size_t)KS * a.g.kh * a.g.kw * sizeof(uint2))};
  fill_table<DG>(a, tab, tid, S::NTH * S::KG);
  __syncthreads();
  f32x4 v[BI][BN], lo[BI][BN];
  {
    // With two K groups each takes half of the stages.
    const int group = k_group<S>(), t = tid % S::NTH;
    const int nk = ((a.K + KS - 1) / KS + S::KG - 1) / S::KG, k0 = group * nk * KS;
    char* buf = lds + group * S::LDS;
    PixLoad<DG, S::TN, S::NTH> lb;
    lb.init(a, tab.tap, k0, n0, t);
    if constexpr (DG) {
      WeightLoad<S::TM, S::NTH> la;
      la.init(a, tab.wt, k0, m0, t);
      mma_loop<S>(buf, la, lb, nk, v, lo);
    } else {
      MatLoad<false, S::TM, S::NTH, TAIL> la;
      la.init(a.wt, a.K, a.M, a.K, m0, k0, S::KG == 1 ? a.K : min(a.K - k0, nk * KS), 1, 0, t);
      mma_loop<S>(buf, la, lb, nk, v, lo);
    }
  }
  const bool again = redo<S>(v, lo);
  join_groups<S>(lds, v, lo);
  if (k_group<S>() != 0) return;  // (no barrier follows)
  if (again) {
    if constexpr (DG) {
      const DgradOps op{a.src, a.wt, a.out, a.g, a.M, a.N, a.K, a.acc};
      fp32_tile<S>([&](int r, int k) { return op.a(m0 + r, k); }, [&](int c, int k) { return op.b(k, n0 + c); }, a.K, v);
    } else {
      const FwdOps op{a.src, a.wt, a.bias, a.out, a.g, a.M, a.N, a.K};
      fp32_tile<S>([&](int r, int k) { return op.a(m0 + r, k); }, [&](int c, int k) { return op.b(k, n0 + c); }, a.K, v);
    }
  }
  // Lane (lr, q) holds channels row(i, 4 q + r) of pixels col .. col + BN - 1.
  const WaveMap<S> w;
  const int col = n0 + w.col0();
  const int phw = DG ? a.g.h * a.g.w : a.g.oh * a.g.ow;
  typedef float vec_t __attribute__((ext_vector_type(BN)));
  const bool vec = a.c_vec;
  size_t po[BN];  // channel 0 of each pixel
#pragma unroll
  for (int n = 0; n < BN; ++n) {
    const int b = (col + n) / phw;
    po[n] = (size_t)b * a.M * phw + (col + n - b * phw);
  }
  if (DG && a.acc) {
    // every previous value is loaded before the first store
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int n = 0; n < BN; ++n) v[i][n] += lo[i][n];
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = m0 + w.row(i, 4 * w.q + r);
        const size_t ro = (size_t)row * phw;
        if (row < a.M && vec && col < a.N) {
          const vec_t o = *reinterpret_cast<const vec_t*>(a.out + po[0] + ro);
#pragma unroll
          for (int n = 0; n < BN; ++n) lo[i][n][r] = o[n];
        } else {
#pragma unroll
          for (int n = 0; n < BN; ++n) lo[i][n][r] = row < a.M && col + n < a.N ? a.out[po[n] + ro] : 0.f;
        }
      }
  }
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + w.row(i, 4 * w.q + r);
      if (row >= a.M) continue;
      const float bias = !DG && a.bias ? a.bias[row] : 0.f;
      const size_t ro = (size_t)row * phw;
      float y[BN];
#pragma unroll
      for (int n = 0; n < BN; ++n) y[n] = (v[i][n][r] + lo[i][n][r]) + bias;
      if (vec) {
        if (col < a.N) {
          vec_t t;
#pragma unroll
          for (int n = 0; n < BN; ++n) t[n] = y[n];
          *reinterpret_cast<vec_t*>(a.out + po[0] + ro) = t;
        }
      } else {
#pragma unroll
        for (int n = 0; n < BN; ++n)
          if (col + n < a.N) a.out[po[n] + ro] = y[n];
      }
    }
}

// ------------------------------------------------------------ weight gradient
struct WgradArgs {
  const float* x;
  const float* dy;
  float* out;    // dW, or splits x dW
  float* db;     // nullable
  float* part_b; // splits x db (splits > 1)
  uint32_t x_bytes, dy_bytes;
  int M, N, K, chunk, splits;
  int db_assign, c_vec;
  ConvGeom g;
};

// Up to CHUNK of the workgroup's pixels: source offset (bytes) of the pixel's
// corner, tap bits, and dY offset (bytes, channel 0).  PAD more entries read as
// outside.
template <int CHUNK>
struct PixTable {
  static constexpr int kPad = 5 * KS, kN = CHUNK + kPad;
  static_assert(CHUNK % KS == 0, "whole stages");
  uint32_t src[kN], dy[kN], bits[kN];
  __device__ __forceinline__ void fill(const WgradArgs& a, int kbeg, int klen, int t, int nth) {
    const ConvGeom& g = a.g;
    const int ohw = g.oh * g.ow, n = (klen + KS - 1) / KS * KS + 4 * KS;
    for (int e = t; e < n; e += nth) {
      uint32_t s = 0, d = kOOB;
      unsigned m = 0;
      if (e < klen) {
        const int p = kbeg + e, b = p / ohw, pix = p - b * ohw, oh = pix / g.ow, ow = pix - oh * g.ow;
        const int Y = oh * g.stride - g.pad, X = ow * g.stride - g.pad;
        unsigned xb = 0;
        for (int i = 0; i < g.kw; ++i) xb |= (unsigned)((unsigned)(X + i) < (unsigned)g.w) << i;
        for (int i = 0; i < g.kh; ++i)
          if ((unsigned)(Y + i) < (unsigned)g.h) m |= xb << (i * g.kw);
        s = (uint32_t)(b * g.cin * g.h * g.w + Y * g.w + X) * 4u;
        d = (uint32_t)(b * g.cout * ohw + pix) * 4u;
      }
      src[e] = s;
      dy[e] = d;
      bits[e] = m;
    }
  }
};

// Rows of whole maps (channels), k = pixels at the table's offsets: dY, or the
// x of a 1 x 1 filter.  V4: images of a multiple of 4 pixels, so 4 consecutive
// ones are 16 contiguous bytes.
template <int R, int NTH, bool V4, bool SUM>
struct RowLoad : Chunks<R * 4 / NTH, SUM> {
  using Base = Chunks<R * 4 / NTH, SUM>;
  using Base::NC;
  __amdgpu_buffer_rsrc_t rs;
  const uint32_t* tab;
  uint32_t off[NC], e[8];
  int k, left;  // the stages left are this K group's: past them the rows read as 0 (the sums count every stage put)
  __device__ __forceinline__ void init(const float* src, uint32_t bytes, int rows, int hw, const uint32_t* table, int r0,
                                       int t) {
    rs = rsrc(src, bytes);
    tab = table;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      int r, q;
      chunk_at<false, NTH>(t, c, r, q);
      this->place(c, r, q);
      off[c] = r0 + r < rows ? (uint32_t)((r0 + r) * hw) * 4u : kOOB;
    }
  }
  // Start at pixel k0 of the table.
  __device__ __forceinline__ void seek(int k0, int stages, int t) {
    k = k0 + 4 * (t & 3);
    left = stages;
  }
  __device__ __forceinline__ void pre() {
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (!V4 || (j & 3) == 0) e[j] = left > 0 ? tab[k + chunk_k(j)] : kOOB;
    k += KS;
    --left;
  }
  __device__ __forceinline__ void load(float (&x)[NC][8]) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      if (V4) {
        const f32x4 v0 = ld4(rs, off[c] + e[0]), v1 = ld4(rs, off[c] + e[4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          x[c][j] = v0[j];
          x[c][4 + j] = v1[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) x[c][j] = ld1(rs, off[c] + e[j]);
      }
    }
  }
};

// x gathered: rows (ci, tap), k = pixels.
template <int R, int NTH, class T>
struct XLoad : Chunks<R * 4 / NTH, false> {
  using Base = Chunks<R * 4 / NTH, false>;
  using Base::NC;
  __amdgpu_buffer_rsrc_t rs;
  const T* tab;
  uint32_t off[NC], e[8];
  uint32_t bit[NC], m[8];
  int k;
  __device__ __forceinline__ void init(const WgradArgs& a, const T* table, int n0, int t) {
    const ConvGeom& g = a.g;
    rs = rsrc(a.x, a.x_bytes);
    tab = table;
    const int khw = g.kh * g.kw;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      int r, q;
      chunk_at<false, NTH>(t, c, r, q);
      this->place(c, r, q);
      const int n = n0 + r, ci = n / khw, tap = n - ci * khw, kh = tap / g.kw, kw = tap - kh * g.kw;
      off[c] = (uint32_t)(ci * g.h * g.w + kh * g.w + kw) * 4u;
      bit[c] = n < a.N ? 1u << tap : 0u;
    }
  }
  __device__ __forceinline__ void seek(int k0, int, int t) { k = k0 + 4 * (t & 3); }
  __device__ __forceinline__ void pre() {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      e[j] = tab->src[k + chunk_k(j)];
      m[j] = tab->bits[k + chunk_k(j)];
    }
    k += KS;
  }
  __device__ __forceinline__ void load(float (&x)[NC][8]) {
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[c][j] = ld1(rs, m[j] & bit[c] ? off[c] + e[j] : kOOB);
  }
};

// ONE: a 1 x 1 filter, no padding, stride 1, on maps of a multiple of 4 pixels.
template <class S, bool V4, bool ONE, int CHUNK>
__global__ __launch_bounds__(S::NTH * S::KG, 2) void wgrad_split_kernel(WgradArgs a, int gx, int gy, int items) {
  constexpr int BI = S::BI, BN = S::BN;
  // Stages summed before they join the total: 1536 pixels of the medium tile, 768
  // of the small ones.  Error against 64 bits, one sum per split / so: 22 x 188 ->
  // 16 on 56 x 56 (9 splits of two K groups) 3.8e-7 / 1.4e-7, 30 x 250 -> 250 on
  // 28 x 28 (7 splits) 3.3e-7 / 2.3e-7.
  constexpr int kRun = S::TM == 128 ? 48 : 24 / S::KG;
  using T = PixTable<CHUNK>;
  __shared__ __attribute__((aligned(16))) char lds[S::LDS * S::KG];
  __shared__ __attribute__((aligned(16))) T tab;
  int tm, tn, z;
  gemm::item_tile(blockIdx.x, items, gx, gy, tm, tn, z);
  const int m0 = tm * S::TM, n0 = tn * S::TN, tid = threadIdx.x;
  const int kbeg = z * a.chunk, klen = min(a.K - kbeg, a.chunk);
  f32x4 v[BI][BN], lo[BI][BN];
  {
    using LA = RowLoad<S::TM, S::NTH, V4, true>;
    LA la;
    const int group = k_group<S>(), t = tid % S::NTH;
    la.init(a.dy, a.dy_bytes, a.M, a.g.oh * a.g.ow, tab.dy, m0, t);
    Sums<S> total;
    clear_sums<S>(v, lo);
    clear_sums<S>(total.v, lo);
    auto chunks = [&](auto& lb) {
#pragma unroll 1
      for (int c0 = 0; c0 < klen; c0 += CHUNK) {
        const int n = min(klen - c0, CHUNK);
        if (c0 > 0) __syncthreads();  // the table and the stage buffers have been read
        tab.fill(a, kbeg + c0, n, tid, S::NTH * S::KG);
        __syncthreads();
        // With two K groups each takes half of the stages.
        const int nk = ((n + KS - 1) / KS + S::KG - 1) / S::KG, k0 = group * nk * KS;
        la.seek(k0, nk, t);
        lb.seek(k0, nk, t);
        mma_stages<S, kRun>(lds + group * S::LDS, la, lb, nk, v, lo, &total);
      }
    };
    if constexpr (ONE) {
      RowLoad<S::TN, S::NTH, V4, false> lb;
      lb.init(a.x, a.x_bytes, a.N, a.g.h * a.g.w, tab.src, n0, t);
      chunks(lb);
    } else {
      XLoad<S::TN, S::NTH, T> lb;
      lb.init(a, &tab, n0, t);
      chunks(lb);
    }
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int n = 0; n < BN; ++n) v[i][n] = total.v[i][n];
    unscale_sums<S>(v, lo);
    if (a.db && tn == 0) {  // the lane groups' sums of each dY row, added in order
      double* red = reinterpret_cast<double*>(lds);
      static_assert(4 * S::KG * S::TM * 8 <= S::LDS * S::KG, "row sums");
      __syncthreads();
#pragma unroll
      for (int c = 0; c < LA::NC; ++c) {
        int r, q;
        chunk_at<false, S::NTH>(t, c, r, q);
        red[(4 * group + q) * S::TM + r] = la.sum[c];
      }
      __syncthreads();
      if (tid < S::TM && m0 + tid < a.M) {
        double s = red[tid];
#pragma unroll
        for (int q = 1; q < 4 * S::KG; ++q) s += red[q * S::TM + tid];
        const float b = (float)s;
        if (a.splits > 1) a.part_b[(size_t)z * a.M + m0 + tid] = b;
        else a.db[m0 + tid] = a.db_assign ? b : a.db[m0 + tid] + b;
      }
    }
  }
  const bool again = redo<S>(v, lo);
  join_groups<S>(lds, v, lo);
  if (k_group<S>() != 0) return;  // (no barrier follows)
  if (again) {
    const WgradOps op{a.x, a.dy, a.out, a.g, a.M, a.N, a.K};
    fp32_tile<S>([&](int r, int k) { return op.a(m0 + r, kbeg + k); }, [&](int c, int k) { return op.b(kbeg + k, n0 + c); },
                 klen, v);
  }
  const WaveMap<S> w;
  const int col = n0 + w.col0();
  float* out = a.out + (size_t)z * a.M * a.N;
  typedef float vec_t __attribute__((ext_vector_type(BN)));
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = m0 + w.row(i, 4 * w.q + r);
      if (row >= a.M) continue;
      float* p = out + (size_t)row * a.N + col;
      if (a.c_vec) {
        if (col < a.N) {
          vec_t t;
#pragma unroll
          for (int n = 0; n < BN; ++n) t[n] = v[i][n][r] + lo[i][n][r];
          *reinterpret_cast<vec_t*>(p) = t;
        }
      } else {
#pragma unroll
        for (int n = 0; n < BN; ++n)
          if (col + n < a.N) p[n] = v[i][n][r] + lo[i][n][r];
      }
    }
}

// ------------------------------------------------------------------ host side
bool below_2g(double elems) { return elems * 4.0 < 2147483647.0 - 4096.0; }

// The cheapest tile by the model of gemm_args.hpp (no K split: these calls
// have no workspace).
constexpr int kWide = 3, kSlim = 4;
int pick_tile(int M, int N, int K) {
  int best = 0;
  double us = 1e30;
  for (int t = 0; t < 5; ++t) {
    if (t == kSlim) {  // two share a CU
      const long long n = (long long)((M + 63) / 64) * ((N + 127) / 128), per = (n + gemm::kChipCus - 1) / gemm::kChipCus;
      const int st = (K + KS - 1) / KS;
      const double u = per == 1 ? 1.1 * st + 6.0 : (double)per * (0.9 * st + 4.0);
      if (u < us) us = u, best = t;
      continue;
    }
    const int like = t == kWide ? gemm::kSplitLarge : t;  // wide: the large tile's cost, sides swapped
    const long long n = t == kWide ? gemm::tiles_of(like, N, M) : gemm::tiles_of(like, M, N);
    const double u = gemm::split_grid_us(like, n, (K + KS - 1) / KS);
    if (u < us) us = u, best = t;
  }
  return best;
}

template <class S, bool DG>
void launch_gather(hipStream_t s, const GatherArgs& a) {
  const int gx = (a.N + S::TN - 1) / S::TN, gy = (a.M + S::TM - 1) / S::TM, items = gx * gy;
  const uint32_t tab = (uint32_t)(KS * a.g.kh * a.g.kw * (DG ? 12 : 8));  // the k table
  if constexpr (!DG) {
    if (a.K % 4 != 0) {
      mle::launch(conv_split_kernel<S, DG, true>, dim3((unsigned)items), S::NTH * S::KG, tab, s, a, gx, gy, items);
      return;
    }
  }
  mle::launch(conv_split_kernel<S, DG, false>, dim3((unsigned)items), S::NTH * S::KG, tab, s, a, gx, gy, items);
}

template <bool DG>
void launch_gather_tile(hipStream_t s, const GatherArgs& a) {
  switch (pick_tile(a.M, a.N, a.K)) {
    case gemm::kSplitLarge: launch_gather<LargeTile, DG>(s, a); break;
    case gemm::kSplitMedium: launch_gather<MediumTile, DG>(s, a); break;
    case kWide: launch_gather<WideTile, DG>(s, a); break;
    case kSlim: launch_gather<SlimTile, DG>(s, a); break;
    default:
      if (gemm::tiles_of(gemm::kSplitSmall, a.M, a.N) <= gemm::kChipCus) launch_gather<PairedTile, DG>(s, a);
      else launch_gather<SmallTile, DG>(s, a);
      break;
  }
}

// Pixels of the table: what fits beside the tile's buffers in 160 KB (medium, one
// workgroup per CU, and the paired small tile) or in half of it (small, two per CU).
constexpr int kWgradChunk[2] = {3072, 2304};

struct WgradPlan {
  int tile = 0, splits = 1, chunk = 0;
};

// Tile (medium or small) and pixel splits: the cheapest by the model, the
// reduce of the partial gradients and three stages per fill of the table included.
// A stage with x gathered takes 1.6 / 0.64 us where the GEMM's takes 1.4 / 0.53
// (16 x 128 -> 128 and 128 -> 32 on 64 x 64, one round), 0.66 with two K groups (28 x
// 144 -> 16 on 32 x 32: 58 us, 54.6 with two small tiles on a CU instead).  The table does not bound
// the splits, so the workspace does not grow with the pixels: four copies of dW
// or what fills the chip (1024 -> 1024 on 32 x 32, batch 32: 151 MB for 3.7 ms,
// where one split takes 4.8; 256 -> 256 on 128 x 128, batch 16: 17 MB).
WgradPlan wgrad_plan(const ConvGeom& g) {
  const int M = g.cout, N = g.cin * g.kh * g.kw, K = g.n * g.oh * g.ow;
  const int st = (K + KS - 1) / KS;
  WgradPlan best;
  double best_us = 1e30;
  for (int i = 0; i < 2; ++i) {
    const int tile = i == 0 ? gemm::kSplitMedium : gemm::kSplitSmall, per_fill = kWgradChunk[i] / KS;
    const long long tiles = gemm::tiles_of(tile, M, N);
    for (int c = 1; c <= 12; ++c) {  // 1 .. 4 splits, and grids of half a chip's workgroups and more
      long long sp = c <= 4 ? c : (c - 4) * (long long)(gemm::kChipCus / 2) / tiles;
      sp = std::max(1LL, std::min<long long>(sp, st / 4));
      const int depth = (int)((st + sp - 1) / sp);
      sp = (st + depth - 1) / depth;
      // (two small tiles fit a CU beside their tables: full rounds are of 512)
      const long long n = i == 1 && tiles * sp > gemm::kChipCus ? (tiles * sp + 511) / 512 * 512 : tiles * sp;
      double us = (i == 0 ? 1.14 : n <= gemm::kChipCus ? 1.25 : 1.2) *
                  gemm::split_grid_us(tile, n, depth + 3 * ((depth + per_fill - 1) / per_fill) - 1);
      if (sp > 1) us += 5.0 + (double)(sp + 1) * M * N * 4.0 / 4.0e6;
      if (us < best_us) best_us = us, best = {tile, (int)sp, depth * KS};
    }
  }
  return best;
}

template <class S, int CHUNK>
void launch_wgrad(hipStream_t s, const WgradArgs& a) {
  const int gx = (a.N + S::TN - 1) / S::TN, gy = (a.M + S::TM - 1) / S::TM, items = gx * gy * a.splits;
  const bool v4 = a.g.oh * a.g.ow % 4 == 0;
  auto k = v4 && a.g.kh == 1 && a.g.kw == 1 && a.g.pad == 0 && a.g.stride == 1
               ? wgrad_split_kernel<S, true, true, CHUNK>
               : v4 ? wgrad_split_kernel<S, true, false, CHUNK> : wgrad_split_kernel<S, false, false, CHUNK>;
  mle::launch(k, dim3((unsigned)items), S::NTH * S::KG, 0, s, a, gx, gy, items);
}

}  // namespace

bool split_ok(const ConvGeom& g) {
  const double khw = (double)g.kh * g.kw;
  // extents with the rows that the last stage computes offsets of
  return khw <= kMaxTaps && below_2g((double)g.n * g.cin * g.h * g.w) && below_2g((double)g.n * g.cout * g.oh * g.ow) &&
         below_2g(((double)g.cout + KS) * g.cin * khw) && (double)std::max(g.cin, g.cout) * khw < 67108864.0 &&
         (double)g.n * g.oh * g.ow < 1073741824.0 && (double)g.n * g.h * g.w < 1073741824.0;
}

bool few_tiles(const ConvGeom& g) {
  return gemm::tiles_of(gemm::kSplitSmall, g.cout, g.n * g.oh * g.ow) <= gemm::kChipCus;
}

bool split_fwd(hipStream_t s, const ConvGeom& g, const float* x, const float* w, const float* bias, float* y) {
  if (!split_ok(g)) return false;
  GatherArgs a{x, w, bias, y, (uint32_t)((size_t)g.n * g.cin * g.h * g.w * 4),
               (uint32_t)((size_t)g.cout * g.cin * g.kh * g.kw * 4), g.cout, g.n * g.oh * g.ow, g.cin * g.kh * g.kw, g,
               0, g.oh * g.ow % 4 == 0 && mle::aligned16(y)};
  launch_gather_tile<false>(s, a);
  return true;
}

bool split_dgrad(hipStream_t s, const ConvGeom& g, const float* dy, const float* w, float* dx, int accumulate) {
  if (!split_ok(g)) return false;
  GatherArgs a{dy, w, nullptr, dx, (uint32_t)((size_t)g.n * g.cout * g.oh * g.ow * 4),
               (uint32_t)((size_t)g.cout * g.cin * g.kh * g.kw * 4), g.cin, g.n * g.h * g.w, g.cout * g.kh * g.kw, g,
               accumulate, g.h * g.w % 4 == 0 && mle::aligned16(dx)};
  launch_gather_tile<true>(s, a);
  return true;
}

int split_wgrad_splits(const ConvGeom& g) { return split_ok(g) ? wgrad_plan(g).splits : 0; }

void split_wgrad(hipStream_t s, const ConvGeom& g, const float* x, const float* dy, float* dw, float* db,
                 int accumulate_db, float* part, int splits) {
  const WgradPlan p = wgrad_plan(g);
  const int M = g.cout, N = g.cin * g.kh * g.kw;
  float* out = splits > 1 ? part : dw;
  WgradArgs a{x, dy, out, db, splits > 1 ? part + (size_t)splits * M * N : nullptr,
              (uint32_t)((size_t)g.n * g.cin * g.h * g.w * 4), (uint32_t)((size_t)g.n * g.cout * g.oh * g.ow * 4), M, N,
              g.n * g.oh * g.ow, p.chunk, splits, accumulate_db ? 0 : 1, N % 4 == 0 && mle::aligned16(out), g};
  if (p.tile == gemm::kSplitMedium) launch_wgrad<MediumTile, kWgradChunk[0]>(s, a);
  else if (gemm::tiles_of(gemm::kSplitSmall, M, N) * splits <= gemm::kChipCus) launch_wgrad<PairedTile, kWgradChunk[1]>(s, a);
  else launch_wgrad<SmallTile, kWgradChunk[1]>(s, a);
}

}  // namespace conv
