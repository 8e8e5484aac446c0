// Convolution geometry and the element functors of its three products, shared
// by the general kernel (conv.hip) and the split-bf16 one (conv_split.hip):
// a(m, k) and b(k, n) return the GEMM element, or 0 outside the problem.
#pragma once
#include "common.hpp"

namespace conv {

struct ConvGeom {
  int n, cin, h, w, cout, kh, kw, pad, stride, oh, ow;
};

struct FwdOps {
  const float* x;
  const float* wt;
  const float* bias;
  float* y;
  ConvGeom g;
  int M, N, K;
  __device__ float a(int m, int k) const { return (m < M && k < K) ? wt[(size_t)m * K + k] : 0.f; }
  __device__ float b(int k, int n) const {
    if (k >= K || n >= N) return 0.f;
    const int khw = g.kh * g.kw;
    const int ci = k / khw, r = k - ci * khw, kh = r / g.kw, kw = r - kh * g.kw;
    const int ohw = g.oh * g.ow;
    const int bb = n / ohw, pix = n - bb * ohw, oh = pix / g.ow, ow = pix - oh * g.ow;
    const int ih = oh * g.stride - g.pad + kh, iw = ow * g.stride - g.pad + kw;
    if (ih < 0 || ih >= g.h || iw < 0 || iw >= g.w) return 0.f;
    return x[(((size_t)bb * g.cin + ci) * g.h + ih) * g.w + iw];
  }
  __device__ void store(int m, int n, float v, int) const {
    const int ohw = g.oh * g.ow;
    const int bb = n / ohw, pix = n - bb * ohw;
    y[((size_t)bb * g.cout + m) * ohw + pix] = bias ? v + bias[m] : v;
  }
};

struct DgradOps {
  const float* dy;
  const float* wt;
  float* dx;
  ConvGeom g;
  int M, N, K;
  int acc;
  __device__ float a(int m, int k) const {
    if (m >= M || k >= K) return 0.f;
    const int khw = g.kh * g.kw;
    const int co = k / khw, r = k - co * khw;
    return wt[((size_t)co * g.cin + m) * khw + r];
  }
  __device__ float b(int k, int n) const {
    if (k >= K || n >= N) return 0.f;
    const int khw = g.kh * g.kw;
    const int co = k / khw, r = k - co * khw, kh = r / g.kw, kw = r - kh * g.kw;
    const int hw = g.h * g.w;
    const int bb = n / hw, pix = n - bb * hw, ih = pix / g.w, iw = pix - ih * g.w;
    const int nr = ih + g.pad - kh, nc = iw + g.pad - kw;
    if (nr < 0 || nc < 0 || nr % g.stride != 0 || nc % g.stride != 0) return 0.f;
    const int oy = nr / g.stride, ox = nc / g.stride;
    if (oy >= g.oh || ox >= g.ow) return 0.f;
    return dy[(((size_t)bb * g.cout + co) * g.oh + oy) * g.ow + ox];
  }
  __device__ void store(int m, int n, float v, int) const {
    const int hw = g.h * g.w;
    const int bb = n / hw, pix = n - bb * hw;
    float* d = dx + ((size_t)bb * g.cin + m) * hw + pix;
    *d = acc ? *d + v : v;
  }
};

struct WgradOps {
  const float* x;
  const float* dy;
  float* part;  // [splits][M*N]
  ConvGeom g;
  int M, N, K;
  __device__ float a(int m, int k) const {
    if (m >= M || k >= K) return 0.f;
    const int ohw = g.oh * g.ow;
    const int bb = k / ohw, pix = k - bb * ohw;
    return dy[((size_t)bb * g.cout + m) * ohw + pix];
  }
  __device__ float b(int k, int n) const {
    if (k >= K || n >= N) return 0.f;
    const int khw = g.kh * g.kw;
    const int ci = n / khw, r = n - ci * khw, kh = r / g.kw, kw = r - kh * g.kw;
    const int ohw = g.oh * g.ow;
    const int bb = k / ohw, pix = k - bb * ohw, oh = pix / g.ow, ow = pix - oh * g.ow;
    const int ih = oh * g.stride - g.pad + kh, iw = ow * g.stride - g.pad + kw;
    if (ih < 0 || ih >= g.h || iw < 0 || iw >= g.w) return 0.f;
    return x[(((size_t)bb * g.cin + ci) * g.h + ih) * g.w + iw];
  }
  __device__ void store(int m, int n, float v, int split) const { part[(size_t)split * M * N + (size_t)m * N + n] = v; }
};

// The split-bf16 kernels (conv_split.hip).  Filters of at most 32 taps,
// tensors below 2 GiB; false where they do not take the geometry.
bool split_ok(const ConvGeom& g);
bool few_tiles(const ConvGeom& g);  // the forward has at most one 64 x 64 tile per CU
bool split_fwd(hipStream_t s, const ConvGeom& g, const float* x, const float* w, const float* bias, float* y);
bool split_dgrad(hipStream_t s, const ConvGeom& g, const float* dy, const float* w, float* dx, int accumulate);
// K splits of the weight gradient; `part` (splits > 1) receives splits x dW
// then splits x db partials, else dW and db are written.
int split_wgrad_splits(const ConvGeom& g);
void split_wgrad(hipStream_t s, const ConvGeom& g, const float* x, const float* dy, float* dw, float* db,
                 int accumulate_db, float* part, int splits);

}  // namespace conv
