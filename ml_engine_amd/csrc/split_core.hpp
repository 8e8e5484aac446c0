// fp32 products on the bf16 matrix cores, with fp32 accuracy.
//
// An fp32 value is the exact sum of three bf16 values, x = x0 + x1 + x2
// (round to nearest, then the two remainders: 8 + 8 + 8 bits), and a product
// of two bf16 values is exact in fp32.  x y is therefore
//   x0 y0 + (x0 y1 + x1 y0) + (x0 y2 + x1 y1 + x2 y0) + terms below 2^-26 |x y|,
// six bf16 MFMAs in place of one fp32 MFMA at 1/16 of their rate each: on
// gfx950 v_mfma_f32_16x16x32_bf16 multiplies 16 times as many pairs per cycle
// as v_mfma_f32_16x16x4_f32.  x0 y0 goes to one fp32 accumulator (`hi`) and
// the five corrections to another (`lo`): the corrections are then not
// truncated against the large sums, and `hi` takes one rounding per 32
// products instead of one per 4.  Error against 64 bits (2-norm, relative),
// measured on 128 x 128 products:
//   normal x normal, K 64 / 1024 / 8192:    5.0e-8 / 1.8e-7 / 5.7e-7
//   fp32 MFMA, the same:                    1.4e-7 / 5.8e-7 / 1.6e-6
//   ReLU(normal) x normal, K 1024:          1.5e-7 against 4.2e-7
// (all six in one accumulator is biased by the MFMA's truncation and loses to
// the fp32 MFMA on one-sided operands: 9.2e-7 against 8.0e-7 at K 4096.)
//
// What is split is 2^24 x: the last bit of any fp32 value is then at least
// 2^-125, so every part of every value, the smallest included, is exact and
// normal; the sums are scaled back by 2^-48.  (Without the scale values
// under 2^-110 lose bits.  They are ordinary: after some 60 steps a transformer
// block's gradients hold them in many tiles, and sending those to fp32_tile
// took its step from 2.3 to 6.5 ms.)
//
// What the split cannot represent goes to the fp32 MFMA instead, tile by
// tile: an infinity or NaN, a value of 2^104 or more, or a sum of 2^80 or more
// makes its accumulators infinite or NaN.  Such a tile is multiplied again by
// fp32_tile (fp32 products).
//
// Tile engine: a workgroup of CM x CN waves, each (16 BI) x (16 BN) of C.
// 32-deep K stages, double-buffered in LDS as three bf16 planes per operand.
// While the MFMAs of stage t run, every thread splits its share of stage
// t + 1 (raw fp32 in registers, loaded DEPTH stages earlier) and writes it to
// the other buffer, then issues the loads of stage t + 1 + DEPTH.  The barrier sits
// before the last row block's MFMAs, so the first fragments of the next
// stage arrive under them.
//
// LDS layout of a plane: 64-row groups of 4 KB, each four 16-row blocks of
// 1 KB, each 4 lane groups (q) of 256 B, each 16 rows of 16 B (8 k values).
// Row r of a group is row r / 4 of block r % 4, so a lane ends with 4
// consecutive columns of C.  The 16-byte slot of row p in (block b, group q)
// is p ^ (q + 4 b): ds_read_b128 of a block and ds_write_b128 from either
// load order are free of bank conflicts.  Lane group q's 8 k values are
// 4q .. 4q + 3 and 16 + 4q .. 16 + 4q + 3 of the stage, so four lanes read 64
// contiguous bytes of a k-contiguous row.
#pragma once
#include "common.hpp"

namespace split {

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

constexpr int KS = 32;                      // K depth of a stage
constexpr uint32_t kOOB = 0x80000000u;      // byte offset past every buffer: reads 0
constexpr int kWord3 = 0x00020000;          // raw buffer descriptor word 3

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const float* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)bytes, kWord3);
}
// (The whole offset goes through the vector offset: the range check subtracts
// a scalar offset from the extent, which must not go below zero.)
__device__ __forceinline__ f32x4 ld4(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}
__device__ __forceinline__ float ld1(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)off, 0, 0));
}

__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  const bf16x2 v = {(__bf16)a, (__bf16)b};
  return __builtin_bit_cast(unsigned, v);
}
__device__ __forceinline__ float low_f(unsigned h) { return __builtin_bit_cast(float, h << 16); }
__device__ __forceinline__ float high_f(unsigned h) { return __builtin_bit_cast(float, h & 0xffff0000u); }

constexpr float kScale = 0x1p24f, kUnscale = 0x1p-48f;  // of an operand, of a sum of products

// Eight fp32 values to their three bf16 parts.
__device__ __forceinline__ void split8(const float (&x)[8], u32x4& p0, u32x4& p1, u32x4& p2) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float a = x[2 * j], b = x[2 * j + 1];
    const unsigned h = pack_bf16(a, b);
    const float ra = a - low_f(h), rb = b - high_f(h);
    const unsigned m = pack_bf16(ra, rb);
    p0[j] = h;
    p1[j] = m;
    p2[j] = pack_bf16(ra - low_f(m), rb - high_f(m));
  }
}
__device__ __forceinline__ f32x4 mma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Byte offset, inside a plane, of the 16-byte slot of row r (of the tile), lane group q.
__device__ __forceinline__ uint32_t slot(int r, int q) {
  const int b = r & 3, p = (r & 63) >> 2;
  return (uint32_t)((r >> 6) * 4096 + b * 1024 + q * 256 + ((p ^ (q + 4 * b)) * 16));
}

// DEPTH: raw register sets, i.e. how many stages ahead of the splitting the
// loads run.  KG: groups of CM x CN waves that share the tile's K, each with
// its own buffers (NTH and LDS are a group's); join_groups adds their sums.
template <int BI_, int BN_, int CM_, int CN_, int DEPTH_ = 1, int KG_ = 1>
struct Shape {
  static constexpr int BI = BI_, BN = BN_, CM = CM_, CN = CN_, DEPTH = DEPTH_, KG = KG_;
  static constexpr int TM = 16 * BI * CM, TN = 16 * BN * CN, NTH = 64 * CM * CN;
  static constexpr int PA = TM * 64, PB = TN * 64;  // bytes of one plane
  static constexpr int STAGE = 3 * (PA + PB), LDS = 2 * STAGE;
  static_assert(TM % 64 == 0 && TN % 64 == 0, "64-row groups");
};

// Where a wave's accumulators lie in the tile: hi[i][n][r] of lane (lr, q) is
// row(i, 4 q + r) and column col(n, lr).  With BN == 4 the n are consecutive
// columns.
template <class S>
struct WaveMap {
  int lane, lr, q, wm, wn;
  __device__ __forceinline__ WaveMap() {
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) % (S::CM * S::CN);
    lane = tid & 63;
    lr = lane & 15;
    q = lane >> 4;
    wm = wave % S::CM;
    wn = wave / S::CM;
  }
  __device__ __forceinline__ int row(int i, int d) const {
    const int blk = wm * S::BI + i;
    return (blk >> 2) * 64 + 4 * d + (blk & 3);
  }
  __device__ __forceinline__ int col0() const {  // column of n == 0
    const int blk = wn * S::BN;
    return (blk >> 2) * 64 + 4 * lr + (blk & 3);
  }
};

// Sums before the first stage, and after the last: mma_stages adds products of
// scaled operands.
template <class S>
struct Sums {  // of finished runs of stages
  f32x4 v[S::BI][S::BN];
};
template <class S>
__device__ __forceinline__ void clear_sums(f32x4 (&hi)[S::BI][S::BN], f32x4 (&lo)[S::BI][S::BN]) {
#pragma unroll
  for (int i = 0; i < S::BI; ++i)
#pragma unroll
    for (int n = 0; n < S::BN; ++n) hi[i][n] = lo[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
}
template <class S>
__device__ __forceinline__ void unscale_sums(f32x4 (&hi)[S::BI][S::BN], f32x4 (&lo)[S::BI][S::BN]) {
#pragma unroll
  for (int i = 0; i < S::BI; ++i)
#pragma unroll
    for (int n = 0; n < S::BN; ++n) {
      hi[i][n] *= kUnscale;
      lo[i][n] *= kUnscale;
    }
}

// hi + lo += 2^48 A B^T over nk stages.  RUN > 0 (a multiple of DEPTH): after every
// RUN stages and at the end the sums move to `total`, so that a long K rounds
// like the sum of short ones.  The loaders la / lb give CA / CB chunks of
// 8 k values per thread and stage: load(x) fetches the next stage's raw values
// (zeros outside the operand) into a register set, put(lds, x[c], c)
// splits chunk c into the planes.  nk >= 0; stages past nk are loaded but
// never multiplied.
template <class S, int RUN = 0, class LA, class LB>
__device__ __forceinline__ void mma_stages(char* lds, LA& la, LB& lb, int nk, f32x4 (&hi)[S::BI][S::BN],
                                           f32x4 (&lo)[S::BI][S::BN], Sums<S>* total = nullptr) {
  constexpr int BI = S::BI, BN = S::BN, PA = S::PA, PB = S::PB, STG = S::STAGE;
  constexpr int CA = LA::NC, CB = LB::NC, CT = CA + CB;
  const WaveMap<S> w;
  int ao[BI], bo[BN];  // this lane's fragment slots in plane 0
#pragma unroll
  for (int i = 0; i < BI; ++i) ao[i] = (int)slot(w.row(i, w.lr), w.q);
#pragma unroll
  for (int n = 0; n < BN; ++n) {
    const int blk = w.wn * BN + n;
    bo[n] = 3 * PA + (int)slot((blk >> 2) * 64 + 4 * w.lr + (blk & 3), w.q);
  }
  auto frag = [&](const char* p) { return *reinterpret_cast<const u32x4*>(p); };
  constexpr int D = S::DEPTH;
  float xa[D][CA][8], xb[D][CB][8];  // stage kt + 1 + u waits in set (kt + u) % D
  la.pre();
  lb.pre();
  la.load(xa[0]);
  lb.load(xb[0]);
#pragma unroll
  for (int c = 0; c < CA; ++c) la.template put<PA>(lds, xa[0][c], c);
#pragma unroll
  for (int c = 0; c < CB; ++c) lb.template put<PB>(lds + 3 * PA, xb[0][c], c);
#pragma unroll
  for (int u = 0; u < D; ++u) {
    la.pre();
    lb.pre();
    la.load(xa[u]);
    lb.load(xb[u]);
  }
  __syncthreads();
  u32x4 b[BN][3], a0[2], a1, a2;
#pragma unroll
  for (int n = 0; n < BN; ++n)
#pragma unroll
    for (int p = 0; p < 3; ++p) b[n][p] = frag(lds + bo[n] + p * PB);
  a0[0] = frag(lds + ao[0]);
  a1 = frag(lds + ao[0] + PA);
  a2 = frag(lds + ao[0] + 2 * PA);
  auto stage = [&](int kt, float(&sa)[CA][8], float(&sb)[CB][8]) {
    char* cur = lds + (kt & 1) * STG;
    char* nxt = lds + ((kt & 1) ^ 1) * STG;
#pragma unroll
    for (int i = 0; i < BI; ++i) {
      const bool last = i + 1 == BI;
      const char* src = last ? nxt : cur;
      const int in = last ? 0 : i + 1;
      if (last) __syncthreads();  // stage kt fully read, stage kt + 1 fully written
      a0[(i + 1) & 1] = frag(src + ao[in]);
      if (i + 2 == BI) {
        la.pre();
        lb.pre();
      }
      const u32x4 x0 = a0[i & 1];
      // x0 y2, x1 y1, x0 y1, x2 y0, x1 y0 into lo, x0 y0 into hi; a plane's
      // registers take the next fragments after its last use
#pragma unroll
      for (int n = 0; n < BN; ++n) lo[i][n] = mma(x0, b[n][2], lo[i][n]);
      if (last)
#pragma unroll
        for (int n = 0; n < BN; ++n) b[n][2] = frag(nxt + bo[n] + 2 * PB);
#pragma unroll
      for (int n = 0; n < BN; ++n) lo[i][n] = mma(a1, b[n][1], lo[i][n]);
#pragma unroll
      for (int n = 0; n < BN; ++n) lo[i][n] = mma(x0, b[n][1], lo[i][n]);
      if (last)
#pragma unroll
        for (int n = 0; n < BN; ++n) b[n][1] = frag(nxt + bo[n] + PB);
#pragma unroll
      for (int n = 0; n < BN; ++n) lo[i][n] = mma(a2, b[n][0], lo[i][n]);
      a2 = frag(src + ao[in] + 2 * PA);
#pragma unroll
      for (int n = 0; n < BN; ++n) lo[i][n] = mma(a1, b[n][0], lo[i][n]);
      a1 = frag(src + ao[in] + PA);
#pragma unroll
      for (int n = 0; n < BN; ++n) hi[i][n] = mma(x0, b[n][0], hi[i][n]);
      if (last)
#pragma unroll
        for (int n = 0; n < BN; ++n) b[n][0] = frag(nxt + bo[n]);
      if (!last) {
#pragma unroll
        for (int c = 0; c < CT; ++c)
          if (c * (BI - 1) / CT == i) {
            if (c < CA) la.template put<PA>(nxt, sa[c], c);
            else lb.template put<PB>(nxt + 3 * PA, sb[c < CA ? 0 : c - CA], c - CA);
          }
        if (i + 2 == BI && !LA::kBranch && !LB::kBranch) {
          la.load(sa);
          lb.load(sb);
        }
      }
      // the splitting's vector instructions and the LDS traffic between the MFMAs
#pragma unroll
      for (int j = 0; j < 6 * BN; ++j) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
        if ((j & 3) == 3) {
          if (last) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
          else __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if (!last && j >= 4 * BN) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (i + 2 == BI && (LA::kBranch || LB::kBranch)) {
        la.load(sa);
        lb.load(sb);
      }
    }
  };
  static_assert(RUN % D == 0, "whole rounds of the register sets");
  for (int k0 = 0; k0 < nk; k0 += RUN) {
    const int end = RUN > 0 ? min(nk, k0 + RUN) : nk;
    for (int kt = k0; kt < end; kt += D) {
#pragma unroll
      for (int u = 0; u < D; ++u)
        if (kt + u < end) stage(kt + u, xa[u], xb[u]);
    }
    if (RUN == 0) break;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int n = 0; n < BN; ++n) total->v[i][n] += hi[i][n] + lo[i][n];
    clear_sums<S>(hi, lo);
  }
}
// hi + lo = A B^T over nk stages.
template <class S, class LA, class LB>
__device__ __forceinline__ void mma_loop(char* lds, LA& la, LB& lb, int nk, f32x4 (&hi)[S::BI][S::BN],
                                         f32x4 (&lo)[S::BI][S::BN]) {
  clear_sums<S>(hi, lo);
  mma_stages<S>(lds, la, lb, nk, hi, lo);
  unscale_sums<S>(hi, lo);
}

// This thread's K group.
template <class S>
__device__ __forceinline__ int k_group() {
  return S::KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) / (S::CM * S::CN);
}

// Group 0's hi += lo + the other groups' sums, in group order; lo = 0.
template <class S>
__device__ __forceinline__ void join_groups(char* lds, f32x4 (&hi)[S::BI][S::BN], f32x4 (&lo)[S::BI][S::BN]) {
  if (S::KG == 1) return;
  static_assert(S::KG <= 2 && S::NTH * S::BI * S::BN * 16 <= S::LDS * S::KG, "exchange buffer");
  f32x4* x = reinterpret_cast<f32x4*>(lds) + threadIdx.x % S::NTH;
  __syncthreads();
  if (k_group<S>() == 1) {
#pragma unroll
    for (int i = 0; i < S::BI; ++i)
#pragma unroll
      for (int n = 0; n < S::BN; ++n) x[(i * S::BN + n) * S::NTH] = hi[i][n] + lo[i][n];
  }
  __syncthreads();
  if (k_group<S>() == 0) {
#pragma unroll
    for (int i = 0; i < S::BI; ++i)
#pragma unroll
      for (int n = 0; n < S::BN; ++n) {
        hi[i][n] = (hi[i][n] + lo[i][n]) + x[(i * S::BN + n) * S::NTH];
        lo[i][n] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
}

// Whether this thread's sums show something the split cannot represent.
template <class S>
__device__ __forceinline__ bool needs_fp32(const f32x4 (&hi)[S::BI][S::BN], const f32x4 (&lo)[S::BI][S::BN]) {
  float t = 0.f;  // 0 * finite is 0, 0 * infinity and 0 * NaN are NaN
#pragma unroll
  for (int i = 0; i < S::BI; ++i)
#pragma unroll
    for (int n = 0; n < S::BN; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) t = fmaf(0.f, hi[i][n][r] + lo[i][n][r], t);
  return !(t == 0.f);
}

// The tile on the fp32 MFMA: a(row, k) and b(col, k) read the operands (0
// outside them), k < klen.  16-deep steps, lane group q feeding k = 4 q + j to
// step j.  Off the fast path (see above), so plain loads and no staging.
template <class S, class FA, class FB>
__device__ __forceinline__ void fp32_tile(FA a, FB b, int klen, f32x4 (&acc)[S::BI][S::BN]) {
  const WaveMap<S> w;
#pragma unroll 1
  for (int k0 = 0; k0 < klen; k0 += 16) {
    float fa[S::BI][4], fb[S::BN][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = k0 + 4 * w.q + j;
#pragma unroll
      for (int i = 0; i < S::BI; ++i) fa[i][j] = k < klen ? a(w.row(i, w.lr), k) : 0.f;
#pragma unroll
      for (int n = 0; n < S::BN; ++n) fb[n][j] = k < klen ? b(w.col0() + n, k) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < S::BI; ++i)
#pragma unroll
        for (int n = 0; n < S::BN; ++n)
          acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[i][j], fb[n][j], acc[i][n], 0, 0, 0);
  }
}

// The slots of a thread's chunks: the part every loader shares.
// kBranch: load() has a branch, and is kept out of the interleaved schedule;
// pre() may read ahead what load() needs.
template <int NC_, bool SUM>
struct Chunks {
  static constexpr int NC = NC_;
  static constexpr bool kBranch = false;
  uint32_t dst[NC];
  double sum[SUM ? NC : 1];  // SUM: each chunk's sum over k (one add per stage and chunk)
  __device__ __forceinline__ void place(int c, int r, int q) {
    dst[c] = slot(r, q);
    if (SUM) sum[c] = 0.0;
  }
  __device__ __forceinline__ void pre() {}
  template <int PL>
  __device__ __forceinline__ void put(char* lds, const float (&x)[8], int c) {
    u32x4 p0, p1, p2;
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = x[j] * kScale;
    split8(s, p0, p1, p2);
    if (SUM)
      sum[c] += ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
    char* d = lds + dst[c];
    *reinterpret_cast<u32x4*>(d) = p0;
    *reinterpret_cast<u32x4*>(d + PL) = p1;
    *reinterpret_cast<u32x4*>(d + 2 * PL) = p2;
  }
};
// Tile row and lane group of chunk c of thread t: rows along a wave (a lane
// group per wave), or four lane groups of a row beside each other.
template <bool ROWS, int NTH>
__device__ __forceinline__ void chunk_at(int t, int c, int& r, int& q) {
  const int e = t + c * NTH;
  q = ROWS ? (e >> 6) & 3 : e & 3;
  r = ROWS ? (e & 63) + 64 * (e >> 8) : e >> 2;
}
// k (within a stage) of element j of a chunk of lane group 0.
__device__ __forceinline__ constexpr int chunk_k(int j) { return (j & 3) + 16 * (j >> 2); }

// ------------------------------------------------------------- matrix operand
// A tile of R rows of a strided matrix, by NTH threads; a thread's chunks are
// 8 k values of one row each.  MC: row-contiguous (element (row, k) at
// k * ld + row), read 4 bytes at a time, a wave along 64 rows (256 contiguous
// bytes; 16-byte loads of 4 rows, whose chunks land in two LDS blocks at
// once, measured 14 % slower on the large tile).  Else k-contiguous
// (row * ld + k), read 16 bytes at a time, at any 4-byte alignment.  TAIL:
// K % 4 != 0, so the last stage of a k-contiguous operand is read element by
// element.  SUM: also keeps each chunk's sum over k (the bias gradient).
template <bool MC, int R, int NTH, bool TAIL, bool SUM = false>
struct MatLoad : Chunks<R * 4 / NTH, SUM> {
  using Base = Chunks<R * 4 / NTH, SUM>;
  using Base::NC;
  static constexpr bool kBranch = !MC && TAIL;
  static_assert(NC * NTH == R * 4, "chunks per thread");
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[NC];
  uint32_t ld4b, step, so, jump;  // bytes: one row of ld, one stage, the cursor, the extra step past a term's end
  int left, stages, terms;        // stages left of this term, stages per term, terms left
  int kq, kfull;                  // k of this lane group in the stage; K % 32 bound of the last stage (32: full)

  // Rows [r0, r0 + R) of `rows`, k in [k0, k0 + klen); `nterms` copies
  // term_stride elements apart, one after another.  base's extent, 64 more rows
  // of a row-contiguous one included, is below 2 GiB.
  __device__ __forceinline__ void init(const float* base, int64_t ld, int rows, int K, int r0, int k0, int klen,
                                       int nterms, int64_t term_stride, int t) {
    terms = nterms;
    const int64_t extent = (int64_t)((MC ? K : rows) - 1) * ld + (MC ? rows : K) + (int64_t)(nterms - 1) * term_stride;
    rs = rsrc(base, (uint32_t)(extent * 4));
    ld4b = (uint32_t)ld * 4u;
    step = MC ? KS * ld4b : KS * 4u;
    so = MC ? (uint32_t)k0 * ld4b : (uint32_t)k0 * 4u;
    stages = left = (klen + KS - 1) / KS;
    jump = (uint32_t)(term_stride * 4) - (uint32_t)stages * step;
    kfull = klen - (stages - 1) * KS;
    if (klen <= 0) so = kOOB, step = jump = 0, left = stages = 1 << 30;  // nothing: every load gives zeros
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      int r, q;
      unit(t, c, r, q);
      kq = 4 * q;  // the same for every chunk
      const int64_t o = MC ? (int64_t)kq * ld + r0 + r : (int64_t)(r0 + r) * ld + kq;
      off[c] = r0 + r < rows ? (uint32_t)(o * 4) : kOOB;
      this->place(c, r, q);
    }
  }
  __device__ __forceinline__ static void unit(int t, int c, int& r, int& q) { chunk_at<MC, NTH>(t, c, r, q); }
  // A row-contiguous operand ends at its extent (reads past it give zeros; a
  // term or split that ends before it ends on a whole stage, see the host's
  // rule); along k of a k-contiguous one the last stage masks what lies past
  // it.  Past the last term every load gives zeros.
  __device__ __forceinline__ void load(float (&x)[NC][8]) {
    const int kmax = left == 1 ? kfull : KS;
    if (!MC && TAIL && kmax < KS) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int k = chunk_k(j);
          x[c][j] = ld1(rs, kq + k < kmax ? off[c] + so + 4u * k : kOOB);
        }
    } else {
      const uint32_t t0 = !MC && kq >= kmax ? kOOB : so, t1 = !MC && kq + 16 >= kmax ? kOOB : so + 64u;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        if (!MC) {
          // kOOB + an offset inside the extent stays outside it; two kOOBs
          // cancel, but a row outside the matrix only feeds unstored outputs
          const f32x4 v0 = ld4(rs, off[c] + t0), v1 = ld4(rs, off[c] + t1);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            x[c][j] = v0[j];
            x[c][4 + j] = v1[j];
          }
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j)
            x[c][j] = ld1(rs, off[c] + (so + (uint32_t)chunk_k(j) * ld4b));
        }
      }
    }
    so += step;
    if (--left == 0) {
      left = stages;
      so += jump;
      if (--terms == 0) so = kOOB, step = jump = 0;
    }
  }
};

}  // namespace split
