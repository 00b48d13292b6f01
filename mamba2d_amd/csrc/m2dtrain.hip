// m2dtrain.hip -- the operators of an M2D residual block in training that the stock libraries serve badly on gfx950
// (models/mamba2d.py:191-254, models/utils.py:58-118): the weight gradients of its linear layers (64 to 512 outputs
// summed over all positions), the backward of the depthwise 3x3 convolution, the LayerNorms with the residual update
// next to them.  bf16-mixed: the residual stream, its gradient and the parameters are fp32, everything between the
// norms and the residual updates is bf16 (rounded where autocast rounds), arithmetic and sums are fp32.
//
// Sums over positions (parameter gradients) are made in two steps: every workgroup leaves its sums in a slice of a
// workspace, m2d_train_reduce adds the slices in order.  No atomics: results are bit-reproducible.
#include <hip/hip_runtime.h>

#include <atomic>
#include <stdint.h>

#include "../../include/m2dscan.h"
#include "m2dcommon.h"

namespace {

__device__ __forceinline__ void ld4bf(const void* p, float (&v)[4]) {      // 4 bf16
  const uint2 q = *reinterpret_cast<const uint2*>(p);
  v[0] = bf_lo(q.x); v[1] = bf_hi(q.x); v[2] = bf_lo(q.y); v[3] = bf_hi(q.y);
}
__device__ __forceinline__ void st4bf(void* p, const float (&v)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
}
__device__ __forceinline__ void ld4(const float* p, float (&v)[4]) {
  const float4 q = *reinterpret_cast<const float4*>(p);
  v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
}
__device__ __forceinline__ void st4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }

enum { kActNone = 0, kActGelu = 1, kActStarRelu = 2 };
__device__ __forceinline__ float act(int kind, float v, float s, float b) {
  if (kind == kActGelu) return gelu_exact(v);
  if (kind == kActStarRelu) return star_relu(v, s, b);
  return v;
}

template <int G>
__device__ __forceinline__ float row_sum(float v) {      // over the G lanes of a row, left in all of them
#pragma unroll
  for (int off = G >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// ------------------------------------------------------------- residual update and LayerNorms, forward
// xo = x * s[c] + keep[sample] * (r + r2)   (the update; left out where r is null: xo is x)
// y1 = LayerNorm1(xo), y2 = LayerNorm2(y1 before its rounding): norm1 of a block and the local path's own norm, which
// reads norm1's output.  One pass over the fp32 rows; every output is optional.
struct NormArgs {
  const float* x;
  const uint16_t *r, *r2;
  const float *s, *keep;
  float* xo;
  const float *w1, *b1, *w2, *b2;
  uint16_t *y1, *y2;
  int64_t rows;
  int C, rps;              // rps: rows per sample
  float eps1, eps2;
};

template <int G, int NC>
__global__ __launch_bounds__(256) void m2d_train_norm_kernel(const NormArgs a) {
  const int g = threadIdx.x & (G - 1);
  constexpr int kRows = 256 / G;
  const int nchunks = a.C / 4;
  const float inv_c = 1.f / (float)a.C;
  float sv[NC][4], w1[NC][4], b1[NC][4], w2[NC][4], b2[NC][4];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = g + k * G;
#pragma unroll
    for (int j = 0; j < 4; ++j) { sv[k][j] = 1.f; w1[k][j] = b1[k][j] = w2[k][j] = b2[k][j] = 0.f; }
    if (c < nchunks) {
      if (a.s) ld4(a.s + 4 * c, sv[k]);
      if (a.y1 || a.y2) { ld4(a.w1 + 4 * c, w1[k]); ld4(a.b1 + 4 * c, b1[k]); }
      if (a.y2) { ld4(a.w2 + 4 * c, w2[k]); ld4(a.b2 + 4 * c, b2[k]); }
    }
  }
  for (int64_t row = (int64_t)blockIdx.x * kRows + threadIdx.x / G; row < a.rows; row += (int64_t)gridDim.x * kRows) {
    float v[NC][4];
    float sum = 0.f;
    const float keep = a.keep ? a.keep[row / a.rps] : 1.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = g + k * G;
#pragma unroll
      for (int j = 0; j < 4; ++j) v[k][j] = 0.f;
      if (c < nchunks) {
        const int64_t at = row * a.C + 4 * c;
        ld4(a.x + at, v[k]);
        if (a.r) {
          float r[4];
          ld4bf(a.r + at, r);
          if (a.r2) {
            float q[4];
            ld4bf(a.r2 + at, q);
#pragma unroll
            for (int j = 0; j < 4; ++j) r[j] += q[j];
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) v[k][j] = __builtin_fmaf(v[k][j], sv[k][j], r[j] * keep);
          st4(a.xo + at, v[k]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) sum += v[k][j];
      }
    }
    if (!a.y1 && !a.y2) continue;      // (uniform)
    const float mean = row_sum<G>(sum) * inv_c;
    float q = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { v[k][j] -= mean; q = __builtin_fmaf(v[k][j], v[k][j], q); }
      }
    const float rstd = rsqrtf(row_sum<G>(q) * inv_c + a.eps1);
    sum = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { v[k][j] = __builtin_fmaf(v[k][j] * rstd, w1[k][j], b1[k][j]); sum += v[k][j]; }
        if (a.y1) st4bf(a.y1 + row * a.C + 4 * (g + k * G), v[k]);
      }
    if (!a.y2) continue;
    const float mean2 = row_sum<G>(sum) * inv_c;
    q = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { v[k][j] -= mean2; q = __builtin_fmaf(v[k][j], v[k][j], q); }
      }
    const float rstd2 = rsqrtf(row_sum<G>(q) * inv_c + a.eps2);
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = __builtin_fmaf(v[k][j] * rstd2, w2[k][j], b2[k][j]);
        st4bf(a.y2 + row * a.C + 4 * (g + k * G), o);
      }
  }
}

// ------------------------------------------------------------ residual update and LayerNorms, backward
// For y1 = LN1(x), y2 = LN2(y1) and an update xo = x * s + ...: with the gradients d1 of y1, d2 of y2 (or null) and
// dxo of xo, dx = LN1'(d1 + LN2'(d2)) + dxo * s, and the sums over rows of the five parameter gradients (w1, b1, w2,
// b2, s) per workgroup.  Also leaves bf16(dx * keep[sample]), the gradient that the branches of the update before
// x take.  Statistics are computed again from x: the row is read anyway.
struct NormBwdArgs {
  const float *x, *dxo;
  const uint16_t *d1, *d2;
  const float *s, *keep;
  const float *w1, *b1, *w2;
  float* dx;
  uint16_t* branch;
  float* part;             // (gridDim.x, 5, C)
  int64_t rows;
  int C, rps;
  float eps1, eps2;
};

template <int G, int NC, bool TWO>
__global__ __launch_bounds__(256) void m2d_train_norm_bwd_kernel(const NormBwdArgs a) {
  constexpr int NS = TWO ? 5 : 3;      // sums: w1, b1, s (, w2, b2)
  __shared__ float red[4][NS][NC * G * 4];
  const int g = threadIdx.x & (G - 1);
  constexpr int kRows = 256 / G;
  const int nchunks = a.C / 4;
  const float inv_c = 1.f / (float)a.C;
  float sv[NC][4], w1[NC][4], b1[NC][4], w2[NC][4], acc[NS][NC][4];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = g + k * G;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      sv[k][j] = 1.f; w1[k][j] = b1[k][j] = w2[k][j] = 0.f;
#pragma unroll
      for (int n = 0; n < NS; ++n) acc[n][k][j] = 0.f;
    }
    if (c < nchunks) {
      if (a.s) ld4(a.s + 4 * c, sv[k]);
      ld4(a.w1 + 4 * c, w1[k]);
      if (TWO) { ld4(a.b1 + 4 * c, b1[k]); ld4(a.w2 + 4 * c, w2[k]); }
    }
  }
  for (int64_t row = (int64_t)blockIdx.x * kRows + threadIdx.x / G; row < a.rows; row += (int64_t)gridDim.x * kRows) {
    float x[NC][4], xh[NC][4], dn[NC][4], gx[NC][4], d2[NC][4];
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int c = g + k * G;
#pragma unroll
      for (int j = 0; j < 4; ++j) { x[k][j] = xh[k][j] = dn[k][j] = gx[k][j] = d2[k][j] = 0.f; }
      if (c < nchunks) {
        const int64_t at = row * a.C + 4 * c;
        ld4(a.x + at, x[k]);
        ld4bf(a.d1 + at, dn[k]);
        ld4(a.dxo + at, gx[k]);
        if (TWO) ld4bf(a.d2 + at, d2[k]);
#pragma unroll
        for (int j = 0; j < 4; ++j) sum += x[k][j];
      }
    }
    const float keep = a.keep ? a.keep[row / a.rps] : 1.f;
    const float mean = row_sum<G>(sum) * inv_c;
    float q = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) { xh[k][j] = x[k][j] - mean; q = __builtin_fmaf(xh[k][j], xh[k][j], q); }
      }
    const float rstd = rsqrtf(row_sum<G>(q) * inv_c + a.eps1);
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) xh[k][j] *= rstd;
    if constexpr (TWO) {
      float nh[NC][4];
      float s2 = 0.f, q2 = 0.f, t0 = 0.f, t1 = 0.f;
#pragma unroll
      for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) { nh[k][j] = __builtin_fmaf(xh[k][j], w1[k][j], b1[k][j]); s2 += nh[k][j]; }
      const float mean2 = row_sum<G>(s2) * inv_c;
#pragma unroll
      for (int k = 0; k < NC; ++k)
        if (g + k * G < nchunks) {
#pragma unroll
          for (int j = 0; j < 4; ++j) { nh[k][j] -= mean2; q2 = __builtin_fmaf(nh[k][j], nh[k][j], q2); }
        }
      const float rstd2 = rsqrtf(row_sum<G>(q2) * inv_c + a.eps2);
#pragma unroll
      for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          nh[k][j] *= rstd2;
          acc[3][k][j] = __builtin_fmaf(d2[k][j], nh[k][j], acc[3][k][j]);
          acc[4][k][j] += d2[k][j];
          d2[k][j] *= w2[k][j];
          t0 += d2[k][j];
          t1 = __builtin_fmaf(d2[k][j], nh[k][j], t1);
        }
      t0 = row_sum<G>(t0) * inv_c;
      t1 = row_sum<G>(t1) * inv_c;
#pragma unroll
      for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int j = 0; j < 4; ++j) dn[k][j] = __builtin_fmaf(rstd2, d2[k][j] - t0 - nh[k][j] * t1, dn[k][j]);
    }
    float t0 = 0.f, t1 = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          acc[0][k][j] = __builtin_fmaf(dn[k][j], xh[k][j], acc[0][k][j]);
          acc[1][k][j] += dn[k][j];
          acc[2][k][j] = __builtin_fmaf(gx[k][j], x[k][j], acc[2][k][j]);
          dn[k][j] *= w1[k][j];
          t0 += dn[k][j];
          t1 = __builtin_fmaf(dn[k][j], xh[k][j], t1);
        }
      }
    t0 = row_sum<G>(t0) * inv_c;
    t1 = row_sum<G>(t1) * inv_c;
#pragma unroll
    for (int k = 0; k < NC; ++k)
      if (g + k * G < nchunks) {
        const int64_t at = row * a.C + 4 * (g + k * G);
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] = __builtin_fmaf(rstd, dn[k][j] - t0 - xh[k][j] * t1, gx[k][j] * sv[k][j]);
        st4(a.dx + at, o);
        if (a.branch) {
#pragma unroll
          for (int j = 0; j < 4; ++j) o[j] *= keep;
          st4bf(a.branch + at, o);
        }
      }
  }
  // the rows of a wave by lane exchanges, the waves through LDS, in order
#pragma unroll
  for (int n = 0; n < NS; ++n)
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float v = acc[n][k][j];
#pragma unroll
        for (int off = G; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
        if ((threadIdx.x & 63) < G) red[threadIdx.x >> 6][n][4 * (g + k * G) + j] = v;
      }
  __syncthreads();
  constexpr int kMap[5] = {0, 1, 4, 2, 3};      // slots of the part: w1, b1, w2, b2, s
  for (int i = threadIdx.x; i < NS * a.C; i += 256) {
    const int n = i / a.C, c = i - n * a.C;
    int slot = 0;
#pragma unroll
    for (int m = 0; m < NS; ++m) slot = n == m ? kMap[m] : slot;
    a.part[((int64_t)blockIdx.x * 5 + slot) * a.C + c] = ((red[0][n][c] + red[1][n][c]) + red[2][n][c]) + red[3][n][c];
  }
}

// fp32 -> bf16 with the sample's factor: the gradient that the last branch of a block takes from the block's output
__global__ __launch_bounds__(256) void m2d_train_branch_kernel(const float* x, const float* keep, uint16_t* y, int64_t chunks, int64_t cps) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < chunks; i += (int64_t)gridDim.x * 256) {
    float v[8];
    float lo[4], hi[4];
    ld4(x + 8 * i, lo);
    ld4(x + 8 * i + 4, hi);
    const float k = keep ? keep[i / cps] : 1.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] = lo[j] * k; v[4 + j] = hi[j] * k; }
    *reinterpret_cast<uint4*>(y + 8 * i) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
  }
}

// --------------------------------------------------------- backward of the depthwise 3x3, channel-last
// Input p (before the StarReLU in front of the convolution), g the gradient of the convolution's output:
//   ds[h,w] = sum_ij wt[i][j] g[h-i+1, w-j+1],  dp = ds * slope(p),  dwt[i][j] = sum_hw star(p)[h,w] g[h-i+1, w-j+1]
// and the sums for the StarReLU's scale and bias.  Both products slide the same 3x3 window of g along a strip of a row:
// a thread owns 4 channels and a strip at a time, so an output costs three loads of g and one of p for 72
// multiply-adds, and the 36 weight sums stay in registers over all the thread's strips.
constexpr int kDwStrip = 14;
struct DwBwdArgs {
  const uint16_t *p, *g;
  const float* w;            // (C, 1, 3, 3)
  const float *star_s, *star_b;
  uint16_t* dp;
  float* part;               // (gridDim.x, C * 9 + 2): dwt, then the sums for the StarReLU's scale and bias
  int B, H, W, C, strips, lanes;      // lanes: threads of a workgroup that have work, a multiple of C / 4
};

__global__ __launch_bounds__(256) void m2d_train_dwconv_bwd_kernel(const DwBwdArgs a) {
  extern __shared__ float smem[];
  const int nchunks = a.C / 4;
  const int c = threadIdx.x % nchunks, slot = threadIdx.x / nchunks, slots = a.lanes / nchunks;
  const float sc = a.star_s[0], bi = a.star_b[0];
  float wt[9][4], acc[11][4];
#pragma unroll
  for (int t = 0; t < 11; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[t][j] = 0.f;
  if (threadIdx.x < a.lanes) {
    float flat[9][4];
#pragma unroll
    for (int t = 0; t < 9; ++t) ld4(a.w + (int64_t)c * 36 + 4 * t, flat[t]);
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) wt[t][j] = flat[(j * 9 + t) / 4][(j * 9 + t) % 4];
    const int tasks = a.B * a.H * a.strips;
    for (int task = blockIdx.x * slots + slot; task < tasks; task += gridDim.x * slots) {
      const int sidx = task % a.strips, bh = task / a.strips, h = bh % a.H, b = bh / a.H;
      const int w0 = sidx * kDwStrip;
      const int64_t img = (int64_t)b * a.H * a.W * a.C + 4 * c;
      const uint16_t* G = a.g + img;
      // window: rows h-1..h+1 of g, columns w-1, w, w+1 unpacked, column w+2 on its way
      float win[3][3][4];
      uint2 next[3];
      uint2 pn;
      auto fetch = [&](int col) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          const int hh = h + i - 1;
          next[i] = make_uint2(0u, 0u);
          if (hh >= 0 && hh < a.H && col >= 0 && col < a.W)
            next[i] = *reinterpret_cast<const uint2*>(G + ((int64_t)hh * a.W + col) * a.C);
        }
      };
      auto unpack = [&](int at) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          win[i][at][0] = bf_lo(next[i].x); win[i][at][1] = bf_hi(next[i].x);
          win[i][at][2] = bf_lo(next[i].y); win[i][at][3] = bf_hi(next[i].y);
        }
      };
      auto fetch_p = [&](int col) {
        pn = make_uint2(0u, 0u);
        if (col < a.W) pn = *reinterpret_cast<const uint2*>(a.p + img + ((int64_t)h * a.W + col) * a.C);
      };
      fetch(w0 - 1);
      unpack(0);
      fetch(w0);
      unpack(1);
      fetch(w0 + 1);
      fetch_p(w0);
#pragma unroll
      for (int s = 0; s < kDwStrip; ++s) {
        const int w = w0 + s;
        if (w >= a.W) break;
        const int l = s % 3, m = (s + 1) % 3, r = (s + 2) % 3;
        unpack(r);
        const float p[4] = {bf_lo(pn.x), bf_hi(pn.x), bf_lo(pn.y), bf_hi(pn.y)};
        if (s + 1 < kDwStrip) { fetch(w + 2); fetch_p(w + 1); }
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float t = relu(p[j]);
          // (the forward's convolution read this rounded to bf16)
          const float st = __builtin_fmaf(sc * t, t, bi);
          float d = 0.f;
#pragma unroll
          for (int i = 0; i < 3; ++i) {      // tap (i, k) of the convolution meets g at (h - i + 1, w - k + 1)
            d = __builtin_fmaf(wt[3 * i][j], win[2 - i][r][j], d);
            d = __builtin_fmaf(wt[3 * i + 1][j], win[2 - i][m][j], d);
            d = __builtin_fmaf(wt[3 * i + 2][j], win[2 - i][l][j], d);
            acc[3 * i][j] = __builtin_fmaf(st, win[2 - i][r][j], acc[3 * i][j]);
            acc[3 * i + 1][j] = __builtin_fmaf(st, win[2 - i][m][j], acc[3 * i + 1][j]);
            acc[3 * i + 2][j] = __builtin_fmaf(st, win[2 - i][l][j], acc[3 * i + 2][j]);
          }
          acc[9][j] = __builtin_fmaf(d, t * t, acc[9][j]);
          acc[10][j] += d;
          o[j] = star_relu_back(d, t, sc);
        }
        st4bf(a.dp + img + ((int64_t)h * a.W + w) * a.C, o);
      }
    }
#pragma unroll
    for (int t = 0; t < 11; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) smem[(slot * 11 + t) * a.C + 4 * c + j] = acc[t][j];
  }
  __syncthreads();
  float* out = a.part + (int64_t)blockIdx.x * (a.C * 9 + 2);
  for (int i = threadIdx.x; i < 9 * a.C; i += 256) {
    const int t = i / a.C, ch = i - t * a.C;
    float v = 0.f;
    for (int s = 0; s < slots; ++s) v += smem[(s * 11 + t) * a.C + ch];
    out[ch * 9 + t] = v;
  }
  if (threadIdx.x < 128) {      // a wave each for the two scalar sums
    const int t = 9 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    float v = 0.f;
    for (int s = 0; s < slots; ++s)
      for (int ch = lane; ch < a.C; ch += 64) v += smem[(s * 11 + t) * a.C + ch];
    v = row_sum<64>(v);
    if (lane == 0) out[a.C * 9 + t - 9] = v;
  }
}

// -------------------------------------------------- gradient of a linear layer's input, bf16
// dx = (dy * slope_post(z)) W, times slope_pre(x), for y = post(pre(x) W^T + b), z the layer's output before post:
// the forward kernel of the narrow linear layers with the weight turned while it is put into LDS, the slope of the
// activation behind the layer applied to the rows as they come in, that of the one in front as they leave (with the
// per-workgroup sums for a StarReLU's scale and bias).
constexpr int kLinThreads = 256;
constexpr int kLinWaves = 4;
constexpr int kLinStage = 72;

struct LinBwdArgs {
  const uint16_t* dy;      // (P, N)
  const uint16_t* z;       // (P, N), read where post is an activation
  const float* w;          // (N, K)
  const uint16_t* x;       // (P, K), read where pre is an activation
  uint16_t* dx;            // (P, K)
  const float* pre_s;      // StarReLU scale
  float* part;             // (gridDim.x, 2) sums for the StarReLU's scale and bias, where pre is one
  int64_t P;
  int K, N, pre, post, ntiles, nsplit, Ks;      // the workgroups share out the K inputs in nsplit slices of Ks
};

template <int NCMAX>      // steps of 32 along N
__global__ __launch_bounds__(kLinThreads) void m2d_train_linear_bwd_kernel(const LinBwdArgs a) {
  extern __shared__ float smem[];
  const int tid = threadIdx.x, l = tid & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ws = a.N + 8;
  uint16_t* wl = reinterpret_cast<uint16_t*>(smem);      // W^T slice: (Ks, N + 8)
  float* stage = smem + (a.Ks * ws / 2 + 3) / 4 * 4 + wave * 16 * kLinStage;
  const int kbase = (blockIdx.x % a.nsplit) * a.Ks;
  const int first_tile = blockIdx.x / a.nsplit, tile_step = gridDim.x / a.nsplit;
  // Two rows of W at a time, consecutive lanes take consecutive inputs; kAhead pairs are on their way at once (64 images of 56x56, a pair
  // at a time: 39.5, 24.5 and 43.6 us for up to 64, 128 and 256 outputs; now 38.0, 21.1 and 37.4.  The rows' loads taken out of their
  // branches as well cost more in registers than they gave: 36.7, 26.8 and 44.8).
  constexpr int kAhead = 8;
  const int pairs = (a.N / 2) * a.Ks;
  for (int i0 = tid; i0 < pairs; i0 += kAhead * kLinThreads) {
    float lo[kAhead], hi[kAhead];
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int i = i0 + j * kLinThreads < pairs ? i0 + j * kLinThreads : i0;
      const float* src = a.w + (int64_t)(2 * (i / a.Ks)) * a.K + kbase + i % a.Ks;
      lo[j] = src[0];
      hi[j] = src[a.K];
    }
#pragma unroll
    for (int j = 0; j < kAhead; ++j) {
      const int i = i0 + j * kLinThreads;
      if (i < pairs) *reinterpret_cast<uint32_t*>(wl + i % a.Ks * ws + 2 * (i / a.Ks)) = pack_bf16(lo[j], hi[j]);
    }
  }
  __syncthreads();
  const float pre_s = a.pre == kActStarRelu ? a.pre_s[0] : 0.f;
  const int NC = a.N / 32;
  float sum_s = 0.f, sum_b = 0.f;
  uint4 Anext[NCMAX];
  auto fetch = [&](int tile) {
    const int64_t q0 = (int64_t)tile * 64 + wave * 16;
#pragma unroll
    for (int kc = 0; kc < NCMAX; ++kc) {
      Anext[kc] = make_uint4(0u, 0u, 0u, 0u);
      if (kc < NC && tile < a.ntiles && q0 + mn < a.P) Anext[kc] = ld16(a.dy + (q0 + mn) * a.N + 32 * kc + 8 * kb);
    }
  };
  fetch(first_tile);
  for (int tile = first_tile; tile < a.ntiles; tile += tile_step) {
    const int64_t p0 = (int64_t)tile * 64 + wave * 16;
    const int rows = (int)(a.P - p0 < 16 ? a.P - p0 : 16);
    uint4 A[NCMAX];
#pragma unroll
    for (int kc = 0; kc < NCMAX; ++kc) A[kc] = Anext[kc];
    fetch(tile + tile_step);
    if (a.post != kActNone) {
#pragma unroll
      for (int kc = 0; kc < NCMAX; ++kc)
        if (kc < NC && mn < rows) {
          const uint4 zq = ld16(a.z + (p0 + mn) * a.N + 32 * kc + 8 * kb);
          const uint32_t z4[4] = {zq.x, zq.y, zq.z, zq.w};
          uint32_t w4[4] = {A[kc].x, A[kc].y, A[kc].z, A[kc].w};
#pragma unroll
          for (int j = 0; j < 4; ++j)
            w4[j] = pack_bf16(bf_lo(w4[j]) * gelu_slope(bf_lo(z4[j])), bf_hi(w4[j]) * gelu_slope(bf_hi(z4[j])));
          A[kc] = make_uint4(w4[0], w4[1], w4[2], w4[3]);
        }
    }
    for (int n0 = 0; n0 < a.Ks; n0 += 64) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
        if (n0 + 16 * nt < a.Ks) {
          const uint16_t* wrow = wl + (n0 + 16 * nt + mn) * ws + 8 * kb;
#pragma unroll
          for (int kc = 0; kc < NCMAX; ++kc)
            if (kc < NC) acc = mfma_bf16(A[kc], ld16(wrow + 32 * kc), acc);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) stage[(4 * kb + i) * kLinStage + 16 * nt + mn] = acc[i];
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int piece = l + 64 * k, c = piece >> 3, c8 = 8 * (piece & 7);
        if (c < rows && n0 + c8 < a.Ks) {
          const int64_t at = (p0 + c) * a.K + kbase + n0 + c8;
          float v[8];
          const float4 lo = *reinterpret_cast<const float4*>(stage + c * kLinStage + c8);
          const float4 hi = *reinterpret_cast<const float4*>(stage + c * kLinStage + c8 + 4);
          v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
          if (a.pre != kActNone) {
            float xv[8];
            Chunk<bf16_t>::load(reinterpret_cast<const bf16_t*>(a.x + at), xv);
            if (a.pre == kActStarRelu) {
#pragma unroll
              for (int j = 0; j < 8; ++j) {
                const float t = relu(xv[j]);
                sum_s = __builtin_fmaf(v[j], t * t, sum_s);
                sum_b += v[j];
                v[j] = star_relu_back(v[j], t, pre_s);
              }
            } else {
#pragma unroll
              for (int j = 0; j < 8; ++j) v[j] *= gelu_slope(xv[j]);
            }
          }
          *reinterpret_cast<uint4*>(a.dx + at) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
        }
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  if (a.pre == kActStarRelu) {      // (uniform)
    __shared__ float red[kLinWaves][2];
    sum_s = row_sum<64>(sum_s);
    sum_b = row_sum<64>(sum_b);
    if (l == 0) { red[wave][0] = sum_s; red[wave][1] = sum_b; }
    __syncthreads();
    if (tid < 2) a.part[(int64_t)blockIdx.x * 2 + tid] = ((red[0][tid] + red[1][tid]) + red[2][tid]) + red[3][tid];
  }
}

// ------------------------------------------------------- gradient of a linear layer's weight, bf16
// dW[n][k] = sum_p g[p][n] zx[p][k] with g = dy * slope_post(z) and zx = pre(x), db[n] = sum_p g[p][n]: a product with
// a long contraction (P positions) and a small result.  A workgroup owns 64 x 64 results and a share of the positions
// (gridDim.x shares); its waves take 32 positions at a time, each on its own: 16-byte pieces of rows from memory to LDS
// (activations applied on the way), from there the matrix operands by ds_read_b64_tr_b16, which hands a lane four
// positions of one column, exactly what a contraction over positions wants.  The library's kernels for this
// shape take 531 us each for 200704 x 64 x 64 to 256; memory would take 12 to 32 us.
constexpr int kWgRow = 72;      // bf16 per row of a tile in LDS
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4_t lds_s16x4_t;

struct WgradArgs {
  const uint16_t *dy, *z, *x;      // (P, N), (P, N) where post is an activation, (P, K)
  const float *pre_s, *pre_b;
  float* part;                     // (shares, N * K + N)
  int64_t P;
  int N, K, pre, post, shares, bias;
};

// the 8 positions {8 kb + j} of column c0 + (l & 15) of a tile of 32 rows
__device__ __forceinline__ uint4 column_operand(const uint16_t* tile, int c0, int l) {
  const uint16_t* p = tile + (8 * (l >> 4) + ((l & 15) >> 2)) * kWgRow + c0 + 4 * (l & 3);
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 4 * kWgRow));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return make_uint4(a.x, a.y, b.x, b.y);
}

__global__ __launch_bounds__(256, 2) void m2d_train_wgrad_kernel(const WgradArgs a) {
  __shared__ __attribute__((aligned(16))) char raw[3 * 64 * 64 * 4];      // tiles of the four waves (36.9 KB), then three waves' results (48 KB)
  const int tid = threadIdx.x, l = tid & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint16_t* Gt = reinterpret_cast<uint16_t*>(raw) + wave * 2 * 32 * kWgRow;
  uint16_t* Xt = Gt + 32 * kWgRow;
  const int kblocks = (a.K + 63) / 64;
  const int n0 = (blockIdx.y / kblocks) * 64, k0 = (blockIdx.y % kblocks) * 64;
  const float pre_s = a.pre == kActStarRelu ? a.pre_s[0] : 0.f, pre_b = a.pre == kActStarRelu ? a.pre_b[0] : 0.f;
  const int64_t tiles = (a.P + 31) / 32;
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[4][4], accb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    accb[i] = zero;
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero;
  }
  const bool with_bias = a.bias && k0 == 0;
  const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
  const int c8 = 8 * (l & 7);
  const bool gcol = n0 + c8 < a.N, xcol = k0 + c8 < a.K;
  uint4 gq[4], zq[4], xq[4];
  auto fetch = [&](int64_t t) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t p = t * 32 + (l >> 3) + 8 * k;
      gq[k] = zq[k] = xq[k] = make_uint4(0u, 0u, 0u, 0u);
      if (t < tiles && p < a.P) {
        if (gcol) {
          gq[k] = ld16(a.dy + p * a.N + n0 + c8);
          if (a.post != kActNone) zq[k] = ld16(a.z + p * a.N + n0 + c8);
        }
        if (xcol) xq[k] = ld16(a.x + p * a.K + k0 + c8);
      }
    }
  };
  int64_t t = (int64_t)blockIdx.x * 4 + wave;
  fetch(t);
  for (; t < tiles; t += (int64_t)a.shares * 4) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t g4[4] = {gq[k].x, gq[k].y, gq[k].z, gq[k].w}, x4[4] = {xq[k].x, xq[k].y, xq[k].z, xq[k].w};
      if (a.post != kActNone) {
        const uint32_t z4[4] = {zq[k].x, zq[k].y, zq[k].z, zq[k].w};
#pragma unroll
        for (int j = 0; j < 4; ++j)
          g4[j] = pack_bf16(bf_lo(g4[j]) * gelu_slope(bf_lo(z4[j])), bf_hi(g4[j]) * gelu_slope(bf_hi(z4[j])));
      }
      if (a.pre != kActNone) {      // (rows past the end meet zero rows of g)
#pragma unroll
        for (int j = 0; j < 4; ++j) x4[j] = pack_bf16(act(a.pre, bf_lo(x4[j]), pre_s, pre_b), act(a.pre, bf_hi(x4[j]), pre_s, pre_b));
      }
      const int row = (l >> 3) + 8 * k;
      *reinterpret_cast<uint4*>(Gt + row * kWgRow + c8) = make_uint4(g4[0], g4[1], g4[2], g4[3]);
      *reinterpret_cast<uint4*>(Xt + row * kWgRow + c8) = make_uint4(x4[0], x4[1], x4[2], x4[3]);
    }
    fetch(t + (int64_t)a.shares * 4);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    uint4 bx[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bx[j] = column_operand(Xt, 16 * j, l);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 ag = column_operand(Gt, 16 * i, l);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mfma_bf16(ag, bx[j], acc[i][j]);
      if (with_bias) accb[i] = mfma_bf16(ag, ones, accb[i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  // the four waves' results in order; a lane holds, of tile (i, j), rows n = 16 i + 4 kb + r and column k = 16 j + mn
  float* dump = reinterpret_cast<float*>(raw);
  __syncthreads();
  if (wave > 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) dump[((wave - 1) * 64 + (i * 4 + j) * 4 + r) * 64 + l] = acc[i][j][r];
  }
  __syncthreads();
  float* out = a.part + (int64_t)blockIdx.x * ((int64_t)a.N * a.K + a.N);
  if (wave == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int at = ((i * 4 + j) * 4 + r) * 64 + l;
          const int n = n0 + 16 * i + 4 * kb + r, k = k0 + 16 * j + mn;
          const float v = ((acc[i][j][r] + dump[at]) + dump[4096 + at]) + dump[8192 + at];
          if (n < a.N && k < a.K) out[(int64_t)n * a.K + k] = v;
        }
  }
  if (!with_bias) return;      // (uniform)
  __syncthreads();
  if (mn == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) dump[wave * 64 + 16 * i + 4 * kb + r] = accb[i][r];
  }
  __syncthreads();
  if (tid < 64 && n0 + tid < a.N) out[(int64_t)a.N * a.K + n0 + tid] = ((dump[tid] + dump[64 + tid]) + dump[128 + tid]) + dump[192 + tid];
}

// ------------------------------------- both gradients of a linear layer in one pass over its activations, bf16
// dx = (g W) * slope_pre(x) and dW = g^T pre(x), db = sum g, with g = dy * slope_post(z), for layers of up to 256 inputs and outputs
// whose tiles eight waves share evenly.  The two kernels above read dy (and x, z) once each and are bound by that; here a
// tile of T positions is read once: g and pre(x) go to LDS as bf16, where the input's gradient takes g by rows and the weight's gradient takes both by
// columns (ds_read_b64_tr_b16).  A wave owns 32 inputs (K / 32 waves) and a share of the rest: of the positions for the input's gradient, of the outputs
// for the weight's, whose sums stay in its registers over all tiles of the workgroup, so that nothing is added up across
// waves.  W's rows are listed so that a lane ends with the 8 neighbouring inputs of a position that it fetched itself: the slope is
// taken from registers and 16 bytes are stored, 64 of a row.  One barrier a tile (two buffers); the next tile's loads are under way meanwhile.
// One workgroup to a unit: each leaves N K sums.  200704 positions, both kernels above -> this one: 64 -> 64 with the GELU
// before it 42 -> 28 us, 256 -> 64 with it 124 -> 87 (the GELU and its slope at 51 million values: 42 at the rate of the vector ALUs), 64 -> 256 59 -> 36, 128 -> 64 with a StarReLU 52 -> 41.
constexpr int kGrThreads = 512, kGrMost = 256;      // workgroups at most: the compute units of an MI355X
template <int N, int K, int PT>
struct GradsPlan {
  static constexpr int WK = K / 32, WN = 8 / WK, T = 16 * WN * PT;      // waves along the inputs, and beside each other; positions of a tile
  static constexpr int NTW = N / 16 / WN;                               // tiles of 16 outputs of a wave
  static constexpr int GS = N + 8, XS = K + 8;                          // bf16 per row in LDS
  static constexpr int kBuf = T * (GS + XS);                            // bf16 of a buffer
  static constexpr size_t kLds = 2 * (size_t)kBuf * 2;
  static constexpr int GP = T * N / 8 / kGrThreads;                     // 16-byte pieces of g of a thread
  static_assert(WK * WN == 8 && NTW * WN * 16 == N && GP >= 1 && T % 32 == 0, "eight waves share the tiles evenly");
};
struct GradsArgs {
  const uint16_t *dy, *z, *x;      // (P, N), (P, N) where post is an activation, (P, K)
  const float* w;                  // (N, K)
  const float *pre_s, *pre_b;
  uint16_t* dx;                    // (P, K)
  float *part, *star;              // (gridDim.x, N K + N), (gridDim.x, 2) where pre is a StarReLU
  int64_t P;
  int post, bias;
};

// 8 positions of a column, as column_operand, of rows RS apart
template <int RS>
__device__ __forceinline__ uint4 column_of(const uint16_t* tile, int c0, int l) {
  const uint16_t* p = tile + (8 * (l >> 4) + ((l & 15) >> 2)) * RS + c0 + 4 * (l & 3);
  const s16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p));
  const s16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(p + 4 * RS));
  const uint2 a = __builtin_bit_cast(uint2, lo), b = __builtin_bit_cast(uint2, hi);
  return make_uint4(a.x, a.y, b.x, b.y);
}

template <int N, int K, int PT, int PRE>
__global__ __launch_bounds__(kGrThreads) void m2d_train_linear_grads_kernel(const GradsArgs a) {
  using L = GradsPlan<N, K, PT>;
  constexpr int T = L::T, NS = N / 32;
  extern __shared__ float smem[];
  uint16_t* lds = reinterpret_cast<uint16_t*>(smem);
  const int tid = threadIdx.x, l = tid & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % L::WK, wn = wave / L::WK;
  const float pre_s = PRE == kActStarRelu ? a.pre_s[0] : 0.f, pre_b = PRE == kActStarRelu ? a.pre_b[0] : 0.f;
  const int64_t tiles = (a.P + T - 1) / T;
  const uint4 z4 = make_uint4(0u, 0u, 0u, 0u);
  const int xcol = 32 * wk + 8 * kb;                    // the lane's 8 inputs
  uint4 gq[L::GP], zq[L::GP], xq[PT];
  auto fetch = [&](int64_t t) {
#pragma unroll
    for (int u = 0; u < L::GP; ++u) {
      const int i = tid + u * kGrThreads, c = 8 * (i % (N / 8));
      const int64_t pos = t * T + i / (N / 8);
      gq[u] = zq[u] = z4;
      if (pos < a.P) {
        gq[u] = ld16(a.dy + pos * N + c);
        if (a.post != kActNone) zq[u] = ld16(a.z + pos * N + c);
      }
    }
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int64_t pos = t * T + 16 * (wn * PT + j) + mn;
      xq[j] = pos < a.P ? ld16(a.x + pos * K + xcol) : z4;
    }
  };
  fetch(blockIdx.x);
  // W as the first operand of the input's gradient: lane (m, kb) of step s and tile t holds the outputs 32 s + 8 kb + j of input 32 wk + 8 (m >> 2) + 4 t + (m & 3)
  uint4 W[2][NS];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const float* src = a.w + (int64_t)(32 * s + 8 * kb) * K + 32 * wk + 8 * (mn >> 2) + 4 * t + (mn & 3);
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = src[j * K];
      W[t][s] = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
    }
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const uint4 ones = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
  const bool with_bias = a.bias && wk == 0;             // (uniform)
  f32x4_t acc[L::NTW][2], accb[L::NTW];
#pragma unroll
  for (int i = 0; i < L::NTW; ++i) acc[i][0] = acc[i][1] = accb[i] = zero;
  float sum_s = 0.f, sum_b = 0.f;
  int buf = 0;
  for (int64_t t = blockIdx.x; t < tiles; t += gridDim.x) {
    uint16_t* Gt = lds + buf * L::kBuf;
    uint16_t* Xt = Gt + T * L::GS;
    buf ^= 1;
#pragma unroll
    for (int u = 0; u < L::GP; ++u) {
      const int i = tid + u * kGrThreads, c = 8 * (i % (N / 8));
      uint32_t g4[4] = {gq[u].x, gq[u].y, gq[u].z, gq[u].w};
      if (a.post != kActNone) {      // (uniform)
        const uint32_t q4[4] = {zq[u].x, zq[u].y, zq[u].z, zq[u].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) g4[j] = pack_bf16(bf_lo(g4[j]) * gelu_slope(bf_lo(q4[j])), bf_hi(g4[j]) * gelu_slope(bf_hi(q4[j])));
      }
      *reinterpret_cast<uint4*>(Gt + i / (N / 8) * L::GS + c) = make_uint4(g4[0], g4[1], g4[2], g4[3]);
    }
    float slope[PT][8];      // of GELU; relu(x) for StarReLU
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      uint4 q = xq[j];
      if constexpr (PRE != kActNone) {
        float v[8], o[8];
        Chunk<bf16_t>::unpack(q, v);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          if constexpr (PRE == kActGelu) gelu_and_slope(v[i], o[i], slope[j][i]);
          else { slope[j][i] = relu(v[i]); o[i] = act(kActStarRelu, v[i], pre_s, pre_b); }
        }
        q = make_uint4(pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]), pack_bf16(o[4], o[5]), pack_bf16(o[6], o[7]));
      }
      *reinterpret_cast<uint4*>(Xt + (16 * (wn * PT + j) + mn) * L::XS + xcol) = q;
    }
    if (t + gridDim.x < tiles) fetch(t + gridDim.x);
    __syncthreads();
    // the weight's gradient: contraction over the tile's positions
#pragma unroll
    for (int s = 0; s < T / 32; ++s) {
      uint4 bx[2];
#pragma unroll
      for (int j = 0; j < 2; ++j) bx[j] = column_of<L::XS>(Xt + 32 * s * L::XS, 32 * wk + 16 * j, l);
#pragma unroll
      for (int i = 0; i < L::NTW; ++i) {
        const uint4 ag = column_of<L::GS>(Gt + 32 * s * L::GS, 16 * (wn * L::NTW + i), l);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = mfma_bf16(ag, bx[j], acc[i][j]);
        if (with_bias) accb[i] = mfma_bf16(ag, ones, accb[i]);
      }
    }
    // the input's gradient at the lane's positions
#pragma unroll
    for (int j = 0; j < PT; ++j) {
      const int row = 16 * (wn * PT + j) + mn;
      f32x4_t d[2] = {zero, zero};
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const uint4 g = ld16(Gt + row * L::GS + 32 * s + 8 * kb);
        d[0] = mfma_bf16(W[0][s], g, d[0]);
        d[1] = mfma_bf16(W[1][s], g, d[1]);
      }
      float v[8] = {d[0][0], d[0][1], d[0][2], d[0][3], d[1][0], d[1][1], d[1][2], d[1][3]};
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        if constexpr (PRE == kActGelu) v[i] *= slope[j][i];
        if constexpr (PRE == kActStarRelu) {      // (rows past the end: g and so v are 0)
          const float r = slope[j][i];
          sum_s = __builtin_fmaf(v[i], r * r, sum_s);
          sum_b += v[i];
          v[i] = star_relu_back(v[i], r, pre_s);
        }
      }
      const int64_t pos = t * T + row;
      if (pos < a.P) *reinterpret_cast<uint4*>(a.dx + pos * K + xcol) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
    }
  }
  // a lane holds, of tile (i, j), the outputs 4 kb + r and the input mn
  float* out = a.part + (int64_t)blockIdx.x * (N * K + N);
#pragma unroll
  for (int i = 0; i < L::NTW; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * (wn * L::NTW + i) + 4 * kb + r;
#pragma unroll
      for (int j = 0; j < 2; ++j) out[n * K + 32 * wk + 16 * j + mn] = acc[i][j][r];
      if (with_bias && mn == 0) out[N * K + n] = accb[i][r];
    }
  if constexpr (PRE == kActStarRelu) {
    __syncthreads();      // (the buffers are free)
    sum_s = row_sum<64>(sum_s);
    sum_b = row_sum<64>(sum_b);
    if (l == 0) { smem[2 * wave] = sum_s; smem[2 * wave + 1] = sum_b; }
    __syncthreads();
    if (tid < 2) {
      float v = smem[tid];
#pragma unroll
      for (int w = 1; w < 8; ++w) v += smem[2 * w + tid];
      a.star[(int64_t)blockIdx.x * 2 + tid] = v;
    }
  }
}

// ------------------------------------------------------------- sums of the workgroups' parts
// out[i] = sum_s part[s * stride + i], in a fixed order; up to kMaxSegs sums in one launch.  Bound by memory (58 MB of parts
// for a block of 64 channels, most of them still in the last-level cache) as long as enough loads are under way: a
// workgroup takes 16 shares of the parts for 64 results, four to a thread where the parts are whole 16-byte pieces
// (the weights), else for 16 results (the StarReLU's and the depthwise filters' sums, a few thousand), and a thread has
// four loads under way (37 -> 17 us for the block of 64x56x56x64).  The shares are added in order through LDS, so the sums
// do not depend on the form.
constexpr int kMaxSegs = 24;
struct Seg { const float* part; float* out; int64_t stride; int n, parts, first, wide; };
struct ReduceArgs { Seg s[kMaxSegs]; int nsegs; };

template <typename V> __device__ __forceinline__ V zero_of();
template <> __device__ __forceinline__ float zero_of<float>() { return 0.f; }
template <> __device__ __forceinline__ f32x4_t zero_of<f32x4_t>() { return f32x4_t{0.f, 0.f, 0.f, 0.f}; }

template <typename V>
__device__ __forceinline__ void reduce_parts(const Seg& s, int block, V (*red)[17]) {
  constexpr int kV = sizeof(V) / 4;
  const int col = threadIdx.x & 15, share = threadIdx.x >> 4;
  const int i = (block * 16 + col) * kV;
  V v = zero_of<V>();
  if (i < s.n) {
    const float* src = s.part + i;
    int p = share;
    for (; p + 48 < s.parts; p += 64) {
      V o[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = *reinterpret_cast<const V*>(src + (p + 16 * u) * s.stride);
#pragma unroll
      for (int u = 0; u < 4; ++u) v += o[u];
    }
    for (; p < s.parts; p += 16) v += *reinterpret_cast<const V*>(src + p * s.stride);
  }
  red[share][col] = v;
  __syncthreads();
  if (share == 0 && i < s.n) {
    V t = zero_of<V>();
#pragma unroll
    for (int k = 0; k < 16; ++k) t += red[k][col];
    *reinterpret_cast<V*>(s.out + i) = t;
  }
}

__global__ __launch_bounds__(256) void m2d_train_reduce_kernel(const ReduceArgs a) {
  __shared__ f32x4_t red[16][17];
  int si = 0;
  while (si + 1 < a.nsegs && (int)blockIdx.x >= a.s[si + 1].first) ++si;
  const Seg s = a.s[si];
  const int block = (int)blockIdx.x - s.first;
  if (s.wide) reduce_parts<f32x4_t>(s, block, red);
  else reduce_parts<float>(s, block, reinterpret_cast<float (*)[17]>(red));
}

inline int launched() { return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP; }

template <int G, int NC>
void launch_norm(const NormArgs& a, hipStream_t st) {
  int64_t blocks = (a.rows + 256 / G - 1) / (256 / G);
  if (blocks > 2048) blocks = 2048;
  hipLaunchKernelGGL((m2d_train_norm_kernel<G, NC>), dim3((unsigned)blocks), dim3(256), 0, st, a);
}
template <int G, int NC>
void launch_norm_bwd(const NormBwdArgs& a, unsigned blocks, hipStream_t st) {
  if (a.d2) hipLaunchKernelGGL((m2d_train_norm_bwd_kernel<G, NC, true>), dim3(blocks), dim3(256), 0, st, a);
  else hipLaunchKernelGGL((m2d_train_norm_bwd_kernel<G, NC, false>), dim3(blocks), dim3(256), 0, st, a);
}

constexpr int kMaxC = 256;      // channels of the norm kernels: 64 lanes of 4, or 16 lanes x 4
inline int norm_group(int C) { return C <= 16 ? 4 : C <= 32 ? 8 : 16; }

inline size_t lin_lds(int N, int Ks) { return ((size_t)Ks * (N + 8) / 2 + 3) / 4 * 4 * 4 + (size_t)kLinWaves * 16 * kLinStage * 4; }

constexpr size_t kLinMaxLds = 152 * 1024;      // dynamic part of the 160 KB of a compute unit

inline bool allow_big_lds() {
  static std::atomic<uint64_t> seen{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  const uint64_t bit = 1ull << (dev & 63);
  if (seen.load(std::memory_order_acquire) & bit) return true;
  const void* kernels[] = {reinterpret_cast<const void*>(&m2d_train_linear_bwd_kernel<2>), reinterpret_cast<const void*>(&m2d_train_linear_bwd_kernel<4>),
                           reinterpret_cast<const void*>(&m2d_train_linear_bwd_kernel<8>), reinterpret_cast<const void*>(&m2d_train_linear_bwd_kernel<16>)};
  for (const void* k : kernels)
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLinMaxLds) != hipSuccess) return false;
  seen.fetch_or(bit, std::memory_order_release);
  return true;
}

struct LinPlan { int nsplit, Ks, grid, ntiles; size_t lds; };
inline bool plan_linear_bwd(int64_t P, int K, int N, LinPlan& p) {
  if (K % 16 != 0 || N % 32 != 0 || N > 512 || K > 512 || (P + 63) / 64 >= ((int64_t)1 << 31)) return false;
  p.nsplit = 1;
  while (lin_lds(N, K / p.nsplit) > 40 * 1024 && (K / p.nsplit) % 32 == 0 && K / p.nsplit > 64) p.nsplit *= 2;
  p.Ks = K / p.nsplit;
  p.lds = lin_lds(N, p.Ks);
  if (p.lds > kLinMaxLds) return false;
  p.ntiles = (int)((P + 63) / 64);
  int per_cu = (int)(160 * 1024 / p.lds);
  if (per_cu > 8) per_cu = 8;
  p.grid = 256 * per_cu / p.nsplit;
  if (p.grid > p.ntiles) p.grid = p.ntiles;
  if (p.grid < 1) p.grid = 1;
  p.grid *= p.nsplit;
  return true;
}

struct DwPlan { int lanes, slots, grid, strips; size_t lds; };
inline bool plan_dw_bwd(int B, int H, int W, int C, DwPlan& p) {
  const int nchunks = C / 4;
  if (C % 4 != 0 || nchunks > 256 || (int64_t)B * H * ((W + kDwStrip - 1) / kDwStrip) >= ((int64_t)1 << 30)) return false;
  p.slots = 256 / nchunks;
  p.lanes = p.slots * nchunks;
  p.strips = (W + kDwStrip - 1) / kDwStrip;
  const int tasks = B * H * p.strips;
  p.grid = (tasks + p.slots - 1) / p.slots;
  if (p.grid > 768) p.grid = 768;      // three workgroups to a compute unit
  p.lds = (size_t)p.slots * 11 * C * 4;
  return true;
}

inline int wgrad_shares(int64_t P, int N, int K) {
  const int blocks = ((N + 63) / 64) * ((K + 63) / 64);
  int64_t shares = 512 / blocks;
  const int64_t most = (P + 127) / 128;      // every wave has a tile
  if (shares > most) shares = most;
  return (int)(shares < 1 ? 1 : shares);
}

// The layers whose two gradients come from one kernel: those of a block of 64 channels, and of 128 but for its MLP.  (Outputs, inputs, tiles of 16 positions of
// a wave: as many as two buffers of them fit the LDS, up to 128 positions in all.)  At any number of positions: with the adding up of what each leaves, all eight
// at 196 to 200704 positions take 0.49 to 0.98 of the two kernels' time, but for 128 -> 256 at 6272, where it is 25.2 us either way (14x14 cells: 8.8 us
// against 16.9 for 64 -> 64, 11.1 against 17.8 for 256 -> 128).  What grows is the memory of the sums: 256 sets beside 64 at 256 x 128, 34 MB.
#define M2D_GRADS_SHAPES(X) X(64, 64, 2) X(64, 256, 4) X(256, 64, 1) X(64, 128, 4) X(128, 64, 2) X(128, 128, 2) X(128, 256, 2) X(256, 128, 1)
template <int N, int K, int PT>
int grads_parts(int64_t P) {
  const int64_t tiles = (P + GradsPlan<N, K, PT>::T - 1) / GradsPlan<N, K, PT>::T;
  return (int)(tiles < kGrMost ? tiles : kGrMost);
}
template <int N, int K, int PT, int PRE>
int launch_grads(const GradsArgs& a, hipStream_t st) {
  using L = GradsPlan<N, K, PT>;
  static_assert(L::kLds <= kLinMaxLds, "two buffers fit the LDS");
  static std::atomic<uint64_t> seen{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return M2D_ERR_HIP;
  const uint64_t bit = 1ull << (dev & 63);
  const auto kernel = &m2d_train_linear_grads_kernel<N, K, PT, PRE>;
  if (L::kLds > 64 * 1024 && !(seen.load(std::memory_order_acquire) & bit)) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::kLds) != hipSuccess) return M2D_ERR_HIP;
    seen.fetch_or(bit, std::memory_order_release);
  }
  hipLaunchKernelGGL(kernel, dim3((unsigned)grads_parts<N, K, PT>(a.P)), dim3(kGrThreads), L::kLds, st, a);
  return launched();
}
template <int N, int K, int PT>
int launch_grads_act(const GradsArgs& a, int pre, hipStream_t st) {
  if (pre == kActGelu) return launch_grads<N, K, PT, kActGelu>(a, st);
  if (pre == kActStarRelu) return launch_grads<N, K, PT, kActStarRelu>(a, st);
  return launch_grads<N, K, PT, kActNone>(a, st);
}

}  // namespace

extern "C" {

int m2d_train_linear_grads_parts(int64_t P, int N, int K) {
  if (P < 1) return 0;
#define X(n, k, pt) if (N == n && K == k) return grads_parts<n, k, pt>(P);
  M2D_GRADS_SHAPES(X)
#undef X
  return 0;
}

int m2d_train_linear_grads(int64_t P, int N, int K, const void* dy, const void* z, int post_act, const float* weight, const void* x, int pre_act,
                           const float* pre_scale, const float* pre_bias, int bias, void* dx, float* part, float* star_part, void* stream) {
  if (!dy || !weight || !x || !dx || !part || (post_act != kActNone && !z)) return M2D_ERR_NULL_POINTER;
  if (pre_act == kActStarRelu && (!pre_scale || !pre_bias || !star_part)) return M2D_ERR_NULL_POINTER;
  if (P < 1 || K < 1 || N < 1) return M2D_ERR_BAD_SHAPE;
  if ((post_act != kActNone && post_act != kActGelu) || pre_act < kActNone || pre_act > kActStarRelu) return M2D_ERR_UNSUPPORTED;
  if (misaligned(dy, 16) || misaligned(z, 16) || misaligned(x, 16) || misaligned(dx, 16) || misaligned(weight, 4)) return M2D_ERR_MISALIGNED;
  GradsArgs a = {static_cast<const uint16_t*>(dy), static_cast<const uint16_t*>(z), static_cast<const uint16_t*>(x), weight, pre_scale, pre_bias,
                 static_cast<uint16_t*>(dx), part, star_part, P, post_act, bias};
  hipStream_t st = static_cast<hipStream_t>(stream);
#define X(n, k, pt) if (N == n && K == k) return launch_grads_act<n, k, pt>(a, pre_act, st);
  M2D_GRADS_SHAPES(X)
#undef X
  return M2D_ERR_UNSUPPORTED;
}

int m2d_train_norm_fwd(int64_t rows, int C, int rows_per_sample, const float* x, const float* scale, const void* r, const void* r2,
                       const float* keep, float* x_out, const float* w1, const float* b1, float eps1, void* y1, const float* w2,
                       const float* b2, float eps2, void* y2, void* stream) {
  if (!x || (r && !x_out) || ((y1 || y2) && (!w1 || !b1)) || (y2 && (!w2 || !b2))) return M2D_ERR_NULL_POINTER;
  if (rows < 1 || C < 4 || rows_per_sample < 1) return M2D_ERR_BAD_SHAPE;
  if (C % 4 != 0 || C > kMaxC) return M2D_ERR_UNSUPPORTED;
  const void* all[] = {x, scale, r, r2, x_out, w1, b1, y1, w2, b2, y2};
  for (const void* p : all) if (misaligned(p, 16)) return M2D_ERR_MISALIGNED;
  NormArgs a = {};
  a.x = x; a.s = scale; a.r = static_cast<const uint16_t*>(r); a.r2 = static_cast<const uint16_t*>(r2); a.keep = keep; a.xo = x_out;
  a.w1 = w1; a.b1 = b1; a.w2 = w2; a.b2 = b2; a.y1 = static_cast<uint16_t*>(y1); a.y2 = static_cast<uint16_t*>(y2);
  a.rows = rows; a.C = C; a.rps = rows_per_sample; a.eps1 = eps1; a.eps2 = eps2;
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (norm_group(C)) {
    case 4: launch_norm<4, 1>(a, st); break;
    case 8: launch_norm<8, 1>(a, st); break;
    default:
      if (C <= 64) launch_norm<16, 1>(a, st);
      else if (C <= 128) launch_norm<16, 2>(a, st);
      else launch_norm<16, 4>(a, st);
  }
  return launched();
}

int m2d_train_norm_parts(int64_t rows, int C) {
  const int64_t blocks = (rows + 256 / norm_group(C) - 1) / (256 / norm_group(C));
  return (int)(blocks > 1024 ? 1024 : blocks);
}

int m2d_train_norm_bwd(int64_t rows, int C, int rows_per_sample, const float* x, const void* d1, const void* d2, const float* dx_out,
                       const float* scale, const float* keep, const float* w1, const float* b1, float eps1, const float* w2, float eps2,
                       float* dx, void* branch, float* part, void* stream) {
  if (!x || !d1 || !dx_out || !w1 || !dx || !part || (d2 && (!b1 || !w2))) return M2D_ERR_NULL_POINTER;
  if (rows < 1 || C < 4 || rows_per_sample < 1) return M2D_ERR_BAD_SHAPE;
  if (C % 4 != 0 || C > kMaxC) return M2D_ERR_UNSUPPORTED;
  const void* all[] = {x, d1, d2, dx_out, scale, w1, b1, w2, dx, branch};
  for (const void* p : all) if (misaligned(p, 16)) return M2D_ERR_MISALIGNED;
  NormBwdArgs a = {};
  a.x = x; a.d1 = static_cast<const uint16_t*>(d1); a.d2 = static_cast<const uint16_t*>(d2); a.dxo = dx_out; a.s = scale; a.keep = keep;
  a.w1 = w1; a.b1 = b1; a.w2 = w2; a.dx = dx; a.branch = static_cast<uint16_t*>(branch); a.part = part;
  a.rows = rows; a.C = C; a.rps = rows_per_sample; a.eps1 = eps1; a.eps2 = eps2;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)m2d_train_norm_parts(rows, C);
  switch (norm_group(C)) {
    case 4: launch_norm_bwd<4, 1>(a, blocks, st); break;
    case 8: launch_norm_bwd<8, 1>(a, blocks, st); break;
    default:
      if (C <= 64) launch_norm_bwd<16, 1>(a, blocks, st);
      else if (C <= 128) launch_norm_bwd<16, 2>(a, blocks, st);
      else launch_norm_bwd<16, 4>(a, blocks, st);
  }
  return launched();
}

int m2d_train_branch(int64_t n, int64_t per_sample, const float* x, const float* keep, void* y, void* stream) {
  if (!x || !y) return M2D_ERR_NULL_POINTER;
  if (n < 1 || per_sample < 1) return M2D_ERR_BAD_SHAPE;
  if (n % 8 != 0 || per_sample % 8 != 0) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(y, 16)) return M2D_ERR_MISALIGNED;
  int64_t blocks = (n / 8 + 255) / 256;
  if (blocks > 8192) blocks = 8192;
  hipLaunchKernelGGL(m2d_train_branch_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), x, keep,
                     static_cast<uint16_t*>(y), n / 8, per_sample / 8);
  return launched();
}

int m2d_train_dwconv_parts(int B, int H, int W, int C) {
  DwPlan p;
  return plan_dw_bwd(B, H, W, C, p) ? p.grid : 0;
}

int m2d_train_dwconv_bwd(int B, int H, int W, int C, const void* p, const void* g, const float* weight, const float* star_scale,
                         const float* star_bias, void* dp, float* part, void* stream) {
  if (!p || !g || !weight || !star_scale || !star_bias || !dp || !part) return M2D_ERR_NULL_POINTER;
  if (B < 1 || H < 1 || W < 1 || C < 1) return M2D_ERR_BAD_SHAPE;
  DwPlan pl;
  if (!plan_dw_bwd(B, H, W, C, pl)) return M2D_ERR_UNSUPPORTED;
  if (misaligned(p, 16) || misaligned(g, 16) || misaligned(dp, 16) || misaligned(weight, 16)) return M2D_ERR_MISALIGNED;
  DwBwdArgs a = {};
  a.p = static_cast<const uint16_t*>(p); a.g = static_cast<const uint16_t*>(g); a.w = weight; a.star_s = star_scale; a.star_b = star_bias;
  a.dp = static_cast<uint16_t*>(dp); a.part = part; a.B = B; a.H = H; a.W = W; a.C = C; a.strips = pl.strips; a.lanes = pl.lanes;
  hipLaunchKernelGGL(m2d_train_dwconv_bwd_kernel, dim3((unsigned)pl.grid), dim3(256), pl.lds, static_cast<hipStream_t>(stream), a);
  return launched();
}

int m2d_train_linear_parts(int64_t P, int K, int N) {
  LinPlan p;
  return plan_linear_bwd(P, K, N, p) ? p.grid : 0;
}

int m2d_train_linear_bwd(int64_t P, int K, int N, const void* dy, const void* z, int post_act, const float* weight, const void* x,
                         int pre_act, const float* pre_scale, void* dx, float* part, void* stream) {
  if (!dy || !weight || !dx || (post_act != kActNone && !z) || (pre_act != kActNone && !x)) return M2D_ERR_NULL_POINTER;
  if (pre_act == kActStarRelu && (!pre_scale || !part)) return M2D_ERR_NULL_POINTER;
  if (P < 1 || K < 1 || N < 1) return M2D_ERR_BAD_SHAPE;
  LinPlan p;
  if ((post_act != kActNone && post_act != kActGelu) || pre_act < kActNone || pre_act > kActStarRelu || !plan_linear_bwd(P, K, N, p))
    return M2D_ERR_UNSUPPORTED;
  if (misaligned(dy, 16) || misaligned(z, 16) || misaligned(x, 16) || misaligned(dx, 16) || misaligned(weight, 16)) return M2D_ERR_MISALIGNED;
  if (p.lds > 64 * 1024 && !allow_big_lds()) return M2D_ERR_HIP;
  LinBwdArgs a = {};
  a.dy = static_cast<const uint16_t*>(dy); a.z = static_cast<const uint16_t*>(z); a.w = weight; a.x = static_cast<const uint16_t*>(x);
  a.dx = static_cast<uint16_t*>(dx); a.pre_s = pre_scale; a.part = part; a.P = P; a.K = K; a.N = N; a.pre = pre_act; a.post = post_act;
  a.ntiles = p.ntiles; a.nsplit = p.nsplit; a.Ks = p.Ks;
  const dim3 g((unsigned)p.grid), t(kLinThreads);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (N <= 64) hipLaunchKernelGGL(m2d_train_linear_bwd_kernel<2>, g, t, p.lds, st, a);
  else if (N <= 128) hipLaunchKernelGGL(m2d_train_linear_bwd_kernel<4>, g, t, p.lds, st, a);
  else if (N <= 256) hipLaunchKernelGGL(m2d_train_linear_bwd_kernel<8>, g, t, p.lds, st, a);
  else hipLaunchKernelGGL(m2d_train_linear_bwd_kernel<16>, g, t, p.lds, st, a);
  return launched();
}

int m2d_train_wgrad_parts(int64_t P, int N, int K) { return wgrad_shares(P, N, K); }

int m2d_train_wgrad(int64_t P, int N, int K, const void* dy, const void* z, int post_act, const void* x, int pre_act,
                    const float* pre_scale, const float* pre_bias, int bias, float* part, void* stream) {
  if (!dy || !x || !part || (post_act != kActNone && !z)) return M2D_ERR_NULL_POINTER;
  if (pre_act == kActStarRelu && (!pre_scale || !pre_bias)) return M2D_ERR_NULL_POINTER;
  if (P < 1 || K < 1 || N < 1) return M2D_ERR_BAD_SHAPE;
  if ((post_act != kActNone && post_act != kActGelu) || pre_act < kActNone || pre_act > kActStarRelu || K % 8 != 0 || N % 8 != 0 ||
      K > 4096 || N > 4096)
    return M2D_ERR_UNSUPPORTED;
  if (misaligned(dy, 16) || misaligned(z, 16) || misaligned(x, 16)) return M2D_ERR_MISALIGNED;
  WgradArgs a = {};
  a.dy = static_cast<const uint16_t*>(dy); a.z = static_cast<const uint16_t*>(z); a.x = static_cast<const uint16_t*>(x);
  a.pre_s = pre_scale; a.pre_b = pre_bias; a.part = part; a.P = P; a.N = N; a.K = K; a.pre = pre_act; a.post = post_act; a.bias = bias;
  a.shares = wgrad_shares(P, N, K);
  const dim3 g((unsigned)a.shares, (unsigned)(((N + 63) / 64) * ((K + 63) / 64)));
  hipLaunchKernelGGL(m2d_train_wgrad_kernel, g, dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return launched();
}

int m2d_train_reduce(int nsegs, const m2d_reduce_seg* segs, void* stream) {
  if (!segs) return M2D_ERR_NULL_POINTER;
  if (nsegs < 1) return M2D_ERR_BAD_SHAPE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  for (int at = 0; at < nsegs;) {
    ReduceArgs a = {};
    int64_t blocks = 0;
    for (; at < nsegs && a.nsegs < kMaxSegs; ++at) {
      const m2d_reduce_seg& s = segs[at];
      if (!s.part || !s.out) return M2D_ERR_NULL_POINTER;
      if (s.n < 1 || s.parts < 1) return M2D_ERR_BAD_SHAPE;
      const int wide = s.n % 4 == 0 && s.stride % 4 == 0 && !misaligned(s.part, 16) && !misaligned(s.out, 16) ? 1 : 0;
      a.s[a.nsegs++] = {s.part, s.out, s.stride, s.n, s.parts, (int)blocks, wide};
      blocks += wide ? (s.n + 63) / 64 : (s.n + 15) / 16;
      if (blocks >= ((int64_t)1 << 30)) return M2D_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(m2d_train_reduce_kernel, dim3((unsigned)blocks), dim3(256), 0, st, a);
  }
  return launched();
}

}  // extern "C"
