// m2dblock.hip -- memory-bound operators of an M2D residual block that the stock libraries serve
// badly on gfx950 at this model's shapes, or in several passes where one will do: LayerNorm over
// a short channel axis (64 to 512 channels: models/mamba2d.py:57,220,248,363, models/utils.py:13,
// 232-233), the depthwise 3x3 convolution of the local path on channel-last tensors
// (models/utils.py:101-114), StarReLU (models/utils.py:26-44), the scaled residual sum
// (models/mamba2d.py:258-259), the rotary embedding + LayerNorm of q and k in the attention stages,
// and that attention as a whole where a head is 32 wide and the grid has up to 256 cells.  Inference
// forward only; each reads every input byte once and writes every output byte once.
//
// Layout: activations are row-major (rows, C) / (B, H, W, C), element type float or bf16; weights
// are float or bf16, independently of the activations (a bf16 model holds bf16 weights, a fp32
// model under autocast hands fp32 weights to bf16 activations).  Arithmetic is fp32.
#include <hip/hip_runtime.h>

#include <atomic>
#include <stdint.h>
#include <type_traits>

#include "../../include/m2dscan.h"
#include "m2dcommon.h"

namespace {

// ------------------------------------------------------------------------------------ LayerNorm
// G lanes share a row (G a power of two, 4..64), lane g holds the chunks g, g + G, ... of it: at
// most kMaxChunks of them, all in registers, so the row is read once.  Mean first, then the sum of
// squared deviations (the data is at hand, and E[x^2] - mean^2 would cancel for rows far from zero).
constexpr int kLnThreads = 256;
constexpr int kMaxChunks = 8;

struct LnArgs {
  const void* x;
  const void* w;
  const void* b;
  void* y;
  int64_t rows;
  int C, wbf16;
  float eps;
  // with the residual update in front (RES): the rows normalised are xo = x * s[c] + r (+ r2), also written out
  const void *s, *r, *r2;
  void* xo;
};

// WB: the weights are bf16.  A template, not a branch at every load: with the branch the loads of a lane's weights waited
// for each other, 7 us for the 196 rows of one image where the whole kernel now takes 4.
template <typename T, int G, int NC, bool RES, bool WB>
__global__ __launch_bounds__(kLnThreads) void m2d_layernorm_kernel(const LnArgs a) {
  constexpr int V = Chunk<T>::kV;
  const int lane_in_row = threadIdx.x & (G - 1);
  const int row_in_block = threadIdx.x / G;
  constexpr int kRows = kLnThreads / G;
  const int nchunks = a.C / V;
  const float inv_c = 1.f / (float)a.C;
  // A lane without a k-th chunk loads the row's last one again and drops it: a load in a branch is waited for at the
  // branch's end, and with one branch per chunk the few workgroups of a small image waited for memory once per chunk and
  // tensor (196 rows of 40 chunks with the residual update: 6.4 -> 4.1 us; the calls of a batch of 128, 25088 rows of 40
  // chunks and 6272 of 64, 16.3 -> 12.4 us on average).
  int at[NC];
  bool own[NC];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    const int c = lane_in_row + k * G;
    own[k] = c < nchunks;
    at[k] = (own[k] ? c : nchunks - 1) * V;
  }
  // this lane's share of weight and bias, kept for all its rows
  float wv[NC][V], bv[NC][V], sv[RES ? NC : 1][V];
#pragma unroll
  for (int k = 0; k < NC; ++k) {
    ldwv<V>(a.w, WB, at[k], wv[k]);
    ldwv<V>(a.b, WB, at[k], bv[k]);
    if constexpr (RES) ldwv<V>(a.s, WB, at[k], sv[k]);
  }
  const T* X = static_cast<const T*>(a.x);
  const T* R = static_cast<const T*>(a.r);
  const T* R2 = static_cast<const T*>(a.r2);
  T* XO = static_cast<T*>(a.xo);
  T* Y = static_cast<T*>(a.y);
  for (int64_t row = (int64_t)blockIdx.x * kRows + row_in_block; row < a.rows; row += (int64_t)gridDim.x * kRows) {
    // (all of the row's loads before its first store: the compiler does not know that the stores leave the rest of the row alone)
    float v[NC][V], r[RES ? NC : 1][V];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      Chunk<T>::load(X + row * a.C + at[k], v[k]);
      if constexpr (RES) Chunk<T>::load(R + row * a.C + at[k], r[k]);
    }
    if constexpr (RES) {   // the residual update, as m2d_scale_residual_kernel computes it; the norm sees what was stored
      if (R2) {
        float r2[NC][V];
#pragma unroll
        for (int k = 0; k < NC; ++k) Chunk<T>::load(R2 + row * a.C + at[k], r2[k]);
#pragma unroll
        for (int k = 0; k < NC; ++k)
#pragma unroll
          for (int j = 0; j < V; ++j) r[k][j] += r2[k][j];
      }
#pragma unroll
      for (int k = 0; k < NC; ++k) {
#pragma unroll
        for (int j = 0; j < V; ++j) v[k][j] = __builtin_fmaf(v[k][j], sv[k][j], r[k][j]);
        if (own[k]) Chunk<T>::store_rounded(XO + row * a.C + at[k], v[k]);
      }
    }
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
#pragma unroll
      for (int j = 0; j < V; ++j) s += own[k] ? v[k][j] : 0.f;
    }
#pragma unroll
    for (int off = G >> 1; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
    const float mean = s * inv_c;
    float q = 0.f;
#pragma unroll
    for (int k = 0; k < NC; ++k) {
#pragma unroll
      for (int j = 0; j < V; ++j) { const float d = own[k] ? v[k][j] - mean : 0.f; q = __builtin_fmaf(d, d, q); }
    }
#pragma unroll
    for (int off = G >> 1; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
    const float rstd = rsqrtf(q * inv_c + a.eps);
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      float o[V];
#pragma unroll
      for (int j = 0; j < V; ++j) o[j] = __builtin_fmaf((v[k][j] - mean) * rstd, wv[k][j], bv[k][j]);
      if (own[k]) Chunk<T>::store(Y + row * a.C + at[k], o);
    }
  }
}

template <typename T, int G, int NC, bool RES>
int launch_ln(const LnArgs& a, hipStream_t st) {
  constexpr int kRows = kLnThreads / G;
  int64_t blocks = (a.rows + kRows - 1) / kRows;
  if (blocks > 256 * 8) blocks = 256 * 8;   // grid-stride beyond that: the lane's weights are loaded once and serve several rows
  if (a.wbf16) hipLaunchKernelGGL((m2d_layernorm_kernel<T, G, NC, RES, true>), dim3((unsigned)blocks), dim3(kLnThreads), 0, st, a);
  else hipLaunchKernelGGL((m2d_layernorm_kernel<T, G, NC, RES, false>), dim3((unsigned)blocks), dim3(kLnThreads), 0, st, a);
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

template <typename T, bool RES>
int run_ln(const LnArgs& a, hipStream_t st) {
  const int nchunks = a.C / Chunk<T>::kV;
  // the fewest lanes per row that keep a lane's share within kMaxChunks, but at least 4 chunks in
  // flight per row where the row is long enough
  if (nchunks <= 4) return launch_ln<T, 4, 1, RES>(a, st);
  if (nchunks <= 8) return launch_ln<T, 8, 1, RES>(a, st);
  if (nchunks <= 16) return launch_ln<T, 16, 1, RES>(a, st);
  if (nchunks <= 32) return launch_ln<T, 16, 2, RES>(a, st);
  if (nchunks <= 48) return launch_ln<T, 16, 3, RES>(a, st);
  if (nchunks <= 64) return launch_ln<T, 16, 4, RES>(a, st);
  if (nchunks <= 128) return launch_ln<T, 32, 4, RES>(a, st);
  if (nchunks <= 256) return launch_ln<T, 64, 4, RES>(a, st);
  return launch_ln<T, 64, kMaxChunks, RES>(a, st);
}

// ------------------------------------------------------------------ depthwise 3x3, channel-last
// y[b,h,w,c] = sum_{i,j} wt[c][i][j] x[b,h+i-1,w+j-1,c], zero padding (STAR: of StarReLU(x)).  A thread owns one chunk of
// channels and a strip of STRIP cells along W; the 3x3 window slides along the strip, so every
// output costs three 16-byte loads plus the strip's two extra columns, and the 9 x kV weights of
// the chunk stay in registers.  The kernel is bound by the number of loads: strips of 14 (which
// divide the model's widths 56, 28, 14) run 7 % faster than strips of 8, strips of 4 45 % slower.
constexpr int kDwThreads = 256;
constexpr int kDwAhead = 4;        // columns between a fetch and its first use (2: 52 us, 3: 50 us, 4: 48 us at 56x56x128, B=128)

struct DwArgs {
  const void* x;
  const void* w;    // (C, 1, 3, 3)
  void* y;
  int B, H, W, C, wbf16;
  int strips;       // strips per image row
  const void *star_s, *star_b;   // STAR: scale and bias (one element each, type of w) of a StarReLU in front of the convolution
};

template <typename T, int STRIP, bool STAR = false>
__global__ __launch_bounds__(kDwThreads) void m2d_dwconv3x3_kernel(const DwArgs a) {
  constexpr int V = Chunk<T>::kV;
  const int nchunks = a.C / V;
  const int64_t total = (int64_t)a.B * a.H * a.strips * nchunks;
  const int64_t gid = (int64_t)blockIdx.x * kDwThreads + threadIdx.x;
  if (gid >= total) return;
  const int c = (int)(gid % nchunks);
  int64_t rest = gid / nchunks;
  const int sidx = (int)(rest % a.strips);
  rest /= a.strips;
  const int h = (int)(rest % a.H);
  const int b = (int)(rest / a.H);
  // the 9 taps of the chunk's V channels are 9 V consecutive weights: fetched as 9 groups of V
  float wt[9][V];
  {
    float flat[9][V];   // flat[g][i] = weight number g V + i of the chunk = channel (g V + i) / 9, tap (g V + i) % 9
#pragma unroll
    for (int g = 0; g < 9; ++g) ldwv<V>(a.w, a.wbf16, (c * 9 + g) * V, flat[g]);
#pragma unroll
    for (int t = 0; t < 9; ++t)
#pragma unroll
      for (int j = 0; j < V; ++j) wt[t][j] = flat[(j * 9 + t) / V][(j * 9 + t) % V];
  }
  const T* X = static_cast<const T*>(a.x) + ((int64_t)b * a.H * a.W) * a.C + c * V;
  T* Y = static_cast<T*>(a.y) + ((int64_t)b * a.H * a.W) * a.C + c * V;
  const int w0 = sidx * STRIP;
  // Window: the 16-byte chunks of the cells (h+i-1, w-1 .. w+kDwAhead) as they come from memory, columns that
  // rotate with the step; column w+kDwAhead is fetched kDwAhead steps before its first use, so that a thread has
  // 3 kDwAhead loads in flight (with one column ahead and three waves per SIMD the kernel waited for memory half of
  // the time).  Unpacked at every use: the conversions are cheap next to the registers a float window costs.
  constexpr int NS = kDwAhead + 2;      // columns held
  uint4 win[3][NS];
  // STAR: a column passes through StarReLU when it becomes the window's right one, and is rounded as an activation
  // kernel in front would have stored it; the padding around the image stays zero
  float star_s = 0.f, star_b = 0.f;
  if constexpr (STAR) { star_s = ldw(a.star_s, a.wbf16, 0); star_b = ldw(a.star_b, a.wbf16, 0); }
  auto activate = [&](int col, int slot) {
    if constexpr (STAR) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int hh = h + i - 1;
        if (hh >= 0 && hh < a.H && col >= 0 && col < a.W) {
          float v[V];
          Chunk<T>::unpack(win[i][slot], v);
#pragma unroll
          for (int j = 0; j < V; ++j) v[j] = star_relu(v[j], star_s, star_b);
          Chunk<T>::store(reinterpret_cast<T*>(&win[i][slot]), v);
        }
      }
    }
  };
  auto load_col = [&](int col, int slot) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int hh = h + i - 1;
      win[i][slot] = make_uint4(0u, 0u, 0u, 0u);
      if (hh >= 0 && hh < a.H && col >= 0 && col < a.W)
        win[i][slot] = *reinterpret_cast<const uint4*>(X + ((int64_t)hh * a.W + col) * a.C);
    }
  };
#pragma unroll
  for (int k = 0; k <= kDwAhead; ++k) load_col(w0 - 1 + k, k);
  activate(w0 - 1, 0);
  activate(w0, 1);
#pragma unroll
  for (int s = 0; s < STRIP; ++s) {
    const int w = w0 + s;
    if (w >= a.W) break;
    const int sl = s % NS, sm = (s + 1) % NS, sr = (s + 2) % NS;      // slots of columns w-1, w, w+1
    if (s + kDwAhead <= STRIP) load_col(w + kDwAhead, (s + kDwAhead + 1) % NS);
    activate(w + 1, sr);
    float o[V];
#pragma unroll
    for (int j = 0; j < V; ++j) o[j] = 0.f;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      float xl[V], xm[V], xr[V];
      Chunk<T>::unpack(win[i][sl], xl);
      Chunk<T>::unpack(win[i][sm], xm);
      Chunk<T>::unpack(win[i][sr], xr);
#pragma unroll
      for (int j = 0; j < V; ++j) {
        o[j] = __builtin_fmaf(wt[3 * i][j], xl[j], o[j]);
        o[j] = __builtin_fmaf(wt[3 * i + 1][j], xm[j], o[j]);
        o[j] = __builtin_fmaf(wt[3 * i + 2][j], xr[j], o[j]);
      }
    }
    Chunk<T>::store(Y + ((int64_t)h * a.W + w) * a.C, o);
  }
}

// ------------------------------------------------------------------------ fused elementwise
// StarReLU, y = scale * relu(x)^2 + bias with scalar scale and bias (models/utils.py:22-37), and the
// residual update of a block, y = x * scale[c] + r (models/mamba2d.py:258-259), with a second branch
// r2 where the token mixer's answer is itself a sum (models/mamba2d.py:176): one pass each where stock
// operators take three and two or three.
constexpr int kEwThreads = 256;

struct EwArgs {
  const void* x;
  const void* r;      // residual branch (scale-residual only)
  const void* r2;     // second branch, or null (scale-residual only)
  const void* s;      // one scale (StarReLU) or C of them
  const void* b;      // one bias (StarReLU)
  void* y;
  int64_t chunks;     // 16-byte chunks in all
  int cpr;            // chunks per row (scale-residual)
  int wbf16;
};

template <typename T>
__global__ __launch_bounds__(kEwThreads) void m2d_starrelu_kernel(const EwArgs a) {
  constexpr int V = Chunk<T>::kV;
  const float sc = ldw(a.s, a.wbf16, 0), bi = ldw(a.b, a.wbf16, 0);
  const T* X = static_cast<const T*>(a.x);
  T* Y = static_cast<T*>(a.y);
  for (int64_t i = (int64_t)blockIdx.x * kEwThreads + threadIdx.x; i < a.chunks; i += (int64_t)gridDim.x * kEwThreads) {
    float v[V];
    Chunk<T>::load(X + i * V, v);
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = star_relu(v[j], sc, bi);
    Chunk<T>::store(Y + i * V, v);
  }
}

template <typename T>
__global__ __launch_bounds__(kEwThreads) void m2d_scale_residual_kernel(const EwArgs a) {
  constexpr int V = Chunk<T>::kV;
  const T* X = static_cast<const T*>(a.x);
  const T* R = static_cast<const T*>(a.r);
  const T* R2 = static_cast<const T*>(a.r2);
  T* Y = static_cast<T*>(a.y);
  for (int64_t i = (int64_t)blockIdx.x * kEwThreads + threadIdx.x; i < a.chunks; i += (int64_t)gridDim.x * kEwThreads) {
    const int c = (int)(i % a.cpr);
    float v[V], r[V];
    Chunk<T>::load(X + i * V, v);
    Chunk<T>::load(R + i * V, r);
    if (R2) {
      float r2[V];
      Chunk<T>::load(R2 + i * V, r2);
#pragma unroll
      for (int j = 0; j < V; ++j) r[j] += r2[j];
    }
    float sc[V];
    ldwv<V>(a.s, a.wbf16, c * V, sc);
#pragma unroll
    for (int j = 0; j < V; ++j) v[j] = __builtin_fmaf(v[j], sc[j], r[j]);
    Chunk<T>::store(Y + i * V, v);
  }
}

inline unsigned ew_blocks(int64_t chunks) {
  int64_t blocks = (chunks + kEwThreads - 1) / kEwThreads;
  return (unsigned)(blocks > 256 * 64 ? 256 * 64 : blocks);
}

// ------------------------------------------------------- rotary embedding + LayerNorm of q and k
// The attention stages rotate q and k by position (pairs of neighbouring features share an angle,
// models/utils.py:253-297) and then LayerNorm each head (:299-301).  Input is the output of the
// qkv projection, (B, L, 3, heads, hd); q and k leave as (B, heads, L, hd), the layout the attention
// kernel wants.  A head's hd features are G = hd / kV chunks on G neighbouring lanes; the pairs of
// the rotation never straddle a chunk.  One pass where stock operators take sixteen.
struct RopeArgs {
  const void* qkv;
  const void *cos, *sin;          // (L, hd), element type of qkv
  const void *qw, *qb, *kw, *kb;  // LayerNorm weights of q and k, (hd)
  void *q, *k;
  int64_t total;                  // B * L * 2 * heads * G chunks
  int L, heads, hd, wbf16;
  int token_major;                // q and k as (B, L, heads, hd) instead of (B, heads, L, hd)
  float eps;
};

template <typename T, int G>
__global__ __launch_bounds__(kEwThreads) void m2d_rope_qknorm_kernel(const RopeArgs a) {
  constexpr int V = Chunk<T>::kV;
  const int64_t gid = (int64_t)blockIdx.x * kEwThreads + threadIdx.x;
  if (gid >= a.total) return;          // whole groups of G lanes leave together (total is a multiple of G)
  const int c = (int)(gid % G);
  int64_t rest = gid / G;
  const int head = (int)(rest % a.heads);
  rest /= a.heads;
  const int which = (int)(rest % 2);   // 0: q, 1: k
  rest /= 2;
  const int l = (int)(rest % a.L);
  const int64_t b = rest / a.L;
  const T* src = static_cast<const T*>(a.qkv) + (((b * a.L + l) * 3 + which) * a.heads + head) * (int64_t)a.hd + c * V;
  float x[V], cs[V], sn[V];
  Chunk<T>::load(src, x);
  Chunk<T>::load(static_cast<const T*>(a.cos) + (int64_t)l * a.hd + c * V, cs);
  Chunk<T>::load(static_cast<const T*>(a.sin) + (int64_t)l * a.hd + c * V, sn);
  float v[V];
#pragma unroll
  for (int j = 0; j < V; j += 2) {
    v[j] = __builtin_fmaf(x[j], cs[j], -x[j + 1] * sn[j]);
    v[j + 1] = __builtin_fmaf(x[j + 1], cs[j + 1], x[j] * sn[j + 1]);
  }
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < V; ++j) s += v[j];
#pragma unroll
  for (int off = G >> 1; off > 0; off >>= 1) s += __shfl_xor(s, off, 64);
  const float inv = 1.f / (float)a.hd;
  const float mean = s * inv;
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < V; ++j) { const float d = v[j] - mean; q = __builtin_fmaf(d, d, q); }
#pragma unroll
  for (int off = G >> 1; off > 0; off >>= 1) q += __shfl_xor(q, off, 64);
  const float rstd = rsqrtf(q * inv + a.eps);
  const void* w = which ? a.kw : a.qw;
  const void* bi = which ? a.kb : a.qb;
  float o[V], wv[V], bv[V];
  ldwv<V>(w, a.wbf16, c * V, wv);
  ldwv<V>(bi, a.wbf16, c * V, bv);
#pragma unroll
  for (int j = 0; j < V; ++j) o[j] = __builtin_fmaf((v[j] - mean) * rstd, wv[j], bv[j]);
  T* dst = static_cast<T*>(which ? a.k : a.q) +
           (a.token_major ? ((b * a.L + l) * a.heads + head) : ((b * a.heads + head) * a.L + l)) * (int64_t)a.hd + c * V;
  Chunk<T>::store(dst, o);
}

template <typename T>
int run_rope(const RopeArgs& a, int G, hipStream_t st) {
  const int64_t blocks = (a.total + kEwThreads - 1) / kEwThreads;
  if (blocks >= ((int64_t)1 << 31)) return M2D_ERR_UNSUPPORTED;
  const dim3 grid((unsigned)blocks), block(kEwThreads);
  switch (G) {
    case 1: hipLaunchKernelGGL((m2d_rope_qknorm_kernel<T, 1>), grid, block, 0, st, a); break;
    case 2: hipLaunchKernelGGL((m2d_rope_qknorm_kernel<T, 2>), grid, block, 0, st, a); break;
    case 4: hipLaunchKernelGGL((m2d_rope_qknorm_kernel<T, 4>), grid, block, 0, st, a); break;
    case 8: hipLaunchKernelGGL((m2d_rope_qknorm_kernel<T, 8>), grid, block, 0, st, a); break;
    case 16: hipLaunchKernelGGL((m2d_rope_qknorm_kernel<T, 16>), grid, block, 0, st, a); break;
    case 32: hipLaunchKernelGGL((m2d_rope_qknorm_kernel<T, 32>), grid, block, 0, st, a); break;
    default: return M2D_ERR_UNSUPPORTED;
  }
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

// ---------------------------------------------------------------- small linear layers, bf16
// y = post(pre(x) W^T + bias) for the narrow layers of a block (K and N up to 512): in_proj, out_proj,
// the pointwise convolutions of the local path and the MLP at 64 or 128 channels
// (models/mamba2d.py:166-176, models/utils.py:58-81, 87-118).  These products are bandwidth-bound: a row
// of x is 128 to 512 bytes and is used once.  The weight matrix lives in LDS as bf16 for the whole
// (persistent) workgroup; a wave owns 16 rows, whose 16-byte pieces are the second operands of
// v_mfma_f32_16x16x32_bf16 as they come from memory (lane l: row l & 15, columns 8 (l >> 4) + j of a step
// of 32), W's rows are the first operands (lane l: output l & 15, the same columns), so that a lane ends with
// four neighbouring outputs of a row and, after an exchange with a neighbour, stores 16 bytes.  pre and post are
// nothing, GELU (exact form) or StarReLU: the activation that the block applies before or after the layer.
// A workgroup sees few tiles, so the waits count: per launch (batch of 128, 64 to 256 inputs), with a load in a branch
// for every step of 32, a read of the bias per tile and the results through a block in LDS, 43, 38 and 44 us for up to
// 64, 128 and 256 inputs; with loads and bias ahead of the tiles 33, 36 and 40; with the results stored from registers, and as
// many workgroups as registers allow, 32, 35 and 34 (x and y at the rate of a copy: 10 to 20).
constexpr int kLinThreads = 256;
constexpr int kLinMargin = 18 * 1024;   // bytes of LDS that the choice of slices leaves free
constexpr int kLinMaxKC = 16;      // steps of 32 along K: K <= 512
enum { kActNone = 0, kActGelu = 1, kActStarRelu = 2, kActLayerNorm = 3 };   // the last one only before the layer, and only inside this file

__device__ __forceinline__ float act(int kind, float v, float s, float b) {
  if (kind == kActGelu) return gelu_exact(v);
  if (kind == kActStarRelu) return star_relu(v, s, b);
  return v;
}

// LayerNorm of the 16 rows a wave holds as MFMA operands (lane (mn, kb): the 8 values at 32 kc + 8 kb + j of row
// mn, for kc < KC), in place, rounded to bf16 as a LayerNorm kernel in front of the layer would store them.
// lnp: weight then bias, K floats each, in LDS.  Two-pass mean / variance; the four lanes of a row meet through
// two lane exchanges.
template <int KCMAX>
__device__ __forceinline__ void norm_rows(uint4 (&A)[KCMAX], int KC, int K, const float* lnp, float eps, int kb) {
  float v[KCMAX][8];
  float s = 0.f;
#pragma unroll
  for (int kc = 0; kc < KCMAX; ++kc) {
    Chunk<bf16_t>::unpack(A[kc], v[kc]);
    if (kc < KC) {
#pragma unroll
      for (int j = 0; j < 8; ++j) s += v[kc][j];
    }
  }
  s += __shfl_xor(s, 16, 64);
  s += __shfl_xor(s, 32, 64);
  const float inv = 1.f / (float)K, mean = s * inv;
  float q = 0.f;
#pragma unroll
  for (int kc = 0; kc < KCMAX; ++kc)
    if (kc < KC) {
#pragma unroll
      for (int j = 0; j < 8; ++j) { const float d = v[kc][j] - mean; q = __builtin_fmaf(d, d, q); }
    }
  q += __shfl_xor(q, 16, 64);
  q += __shfl_xor(q, 32, 64);
  const float rstd = rsqrtf(q * inv + eps);
#pragma unroll
  for (int kc = 0; kc < KCMAX; ++kc)
    if (kc < KC) {
      const float* w = lnp + 32 * kc + 8 * kb;
      const float4 w0 = *reinterpret_cast<const float4*>(w), w1 = *reinterpret_cast<const float4*>(w + 4);
      const float4 b0 = *reinterpret_cast<const float4*>(w + K), b1 = *reinterpret_cast<const float4*>(w + K + 4);
      const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w}, bv[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
      float o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = __builtin_fmaf((v[kc][j] - mean) * rstd, wv[j], bv[j]);
      A[kc] = make_uint4(pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]), pack_bf16(o[4], o[5]), pack_bf16(o[6], o[7]));
    }
}

// Pieces 0 .. pieces-1 of 8 weights from element `first` on, as bf16, to put(piece, value): kStageAhead loads of a thread in
// flight (one at a time, staging was most of the 8 us that such a layer took on one image's rows).
constexpr int kStageAhead = 4;
// COLS of a row's STRIDE elements are taken (0: the pieces follow each other).
template <int TH = kLinThreads, int COLS = 0, int STRIDE = 0, typename PUT>
__device__ __forceinline__ void stage_rows(const void* w, int wbf16, int64_t first, int pieces, int tid, PUT&& put) {
  auto element = [](int i) { return COLS ? (int64_t)(i / (COLS / 8 + !COLS)) * STRIDE + 8 * (i % (COLS / 8 + !COLS)) : (int64_t)8 * i; };
  if (wbf16) {
    const uint16_t* src = static_cast<const uint16_t*>(w) + first;
    for (int i0 = tid; i0 < pieces; i0 += kStageAhead * TH) {
      uint4 q[kStageAhead];
#pragma unroll
      for (int k = 0; k < kStageAhead; ++k) {
        const int i = i0 + k * TH;
        q[k] = ld16(src + element(i < pieces ? i : i0));
      }
#pragma unroll
      for (int k = 0; k < kStageAhead; ++k)
        if (i0 + k * TH < pieces) put(i0 + k * TH, q[k]);
    }
  } else {
    const float* src = static_cast<const float*>(w) + first;
    for (int i0 = tid; i0 < pieces; i0 += kStageAhead * TH) {
      float4 lo[kStageAhead], hi[kStageAhead];
#pragma unroll
      for (int k = 0; k < kStageAhead; ++k) {
        const int i = i0 + k * TH;
        const float* p = src + element(i < pieces ? i : i0);
        lo[k] = *reinterpret_cast<const float4*>(p);
        hi[k] = *reinterpret_cast<const float4*>(p + 4);
      }
#pragma unroll
      for (int k = 0; k < kStageAhead; ++k)
        if (i0 + k * TH < pieces)
          put(i0 + k * TH, make_uint4(pack_bf16(lo[k].x, lo[k].y), pack_bf16(lo[k].z, lo[k].w), pack_bf16(hi[k].x, hi[k].y), pack_bf16(hi[k].z, hi[k].w)));
    }
  }
}

struct LinArgs {
  const void* x;        // (P, K) bf16
  const void* w;        // (N, K)
  const void* bias;     // (N) or null
  void* y;              // (P, N) bf16
  int64_t P;
  int K, N, wbf16, pre, post, ntiles;
  int nsplit, Ns;       // the workgroups share out the N outputs in nsplit slices of Ns
  const void *pre_s, *pre_b, *post_s, *post_b;   // StarReLU scale and bias (one element each, type of w) where pre / post is StarReLU
  const void *ln_w, *ln_b;                       // LayerNorm over the K inputs in front of the layer (pre == kActLayerNorm): weight and bias, (K), type of w
  float ln_eps;
  void* z;              // (P, N) bf16 or null: the layer's output before post, for a caller whose backward wants its slope
  const void *res_x, *res_r, *res_s;   // RES: the residual stream (P, N) bf16, a second branch (P, N) bf16 or null, and the scale of the stream (N), type of w
};

// a and b hold 4 values each of two tiles of 16 in lane row kb (the lane's number / 16).  Rows 0 and 2 end with a's values of
// rows kb and kb + 1, rows 1 and 3 with b's of rows kb - 1 and kb.
__device__ __forceinline__ uint4 halves_exchanged(const uint2 a, const uint2 b) {
  const auto x = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false), y = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
  return make_uint4(x[0], y[0], x[1], y[1]);
}

constexpr int lin_per_cu(int kcmax, bool res = false) { return res ? (kcmax <= 2 ? 4 : 3) : kcmax <= 2 ? 6 : kcmax <= 8 ? 4 : 2; }   // workgroups whose registers fit a compute unit

// KCMAX: steps of 32 along K that the kernel is built for: 2, 4, 8 or 16.
// RES: y = res_x * res_s + (layer + res_r), the residual update of the block around the layer, in the bits that the layer's kernel and
// m2d_scale_residual_kernel gave one after the other (the layer's output is rounded to bf16 before it is added).  Both kernels ran at the rate of
// memory: without the layer's output going out and back 128x56x56x64 takes 49, 128x28x28x128 37 us where they took 27 + 35 and 25 + 18.
// The stream's pieces are fetched a tile ahead into the registers that the last tile's pieces have just left: a wait for one leaves the
// stores behind it under way.
template <int KCMAX, bool RES = false>
__global__ __launch_bounds__(kLinThreads, lin_per_cu(KCMAX, RES)) void m2d_linear_kernel(const LinArgs a) {
  extern __shared__ float smem[];
  const int tid = threadIdx.x, l = tid & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ws = a.K + 8;                                // bf16 per row of W in LDS: rows stay 16-byte aligned and spread over the banks
  uint16_t* wl = reinterpret_cast<uint16_t*>(smem);
  float* bias = smem + (a.Ns * ws / 2 + 3) / 4 * 4;
  float* lnp = bias + a.Ns;
  // Workgroups go to the 8 XCDs in turn: the slices of a tile follow each other on one XCD, so that its L2 fetches the rows
  // of x once for all of them.
  const int j = blockIdx.x / 8;
  const int slice = j % a.nsplit, nbase = slice * a.Ns;   // this workgroup's outputs: nbase .. nbase + Ns
  const int first_tile = j / a.nsplit * 8 + blockIdx.x % 8, tile_step = gridDim.x / a.nsplit;
  if (first_tile >= a.ntiles) return;      // (the whole workgroup: the grid is rounded up to whole eights)
  const int kp = a.K / 8, pieces = a.Ns * kp;
  const int KC = a.K / 32;
  const uint16_t* X = static_cast<const uint16_t*>(a.x);
  uint16_t* Y = static_cast<uint16_t*>(a.y);
  // The rows of the next tile are fetched while the current one is worked on: with the weights in LDS
  // few waves fit a compute unit, too few to cover the latency of memory by themselves.  Rows past the end repeat the last
  // one and are not stored, steps past K repeat the last one and are not used: a load in a branch is waited for at the
  // branch's end, which made one wait per step of a tile's rows instead of none.
  uint4 Anext[KCMAX];
  auto fetch = [&](int tile) {
    const int64_t q = (int64_t)tile * 64 + wave * 16 + mn;
    const uint16_t* row = X + (q < a.P ? q : a.P - 1) * a.K + 8 * kb;
#pragma unroll
    for (int kc = 0; kc < KCMAX; ++kc) Anext[kc] = ld16(row + 32 * (kc < KC ? kc : KC - 1));
  };
  // a lane's 8 neighbouring outputs of the step of 32 that starts at n0 (see the stores below)
  auto piece_at = [&](int n0) { return n0 + (kb & 1 && n0 + 16 < a.Ns ? 16 : 0) + 4 * (kb & 2); };
  constexpr int NR = RES ? KCMAX : 1;                    // (the host sees to Ns <= 32 KCMAX)
  uint4 RX[NR], RR[NR];
  auto fetch_res = [&](int tile, int c) {
    const int64_t q = (int64_t)tile * 64 + wave * 16 + mn, at = (q < a.P ? q : a.P - 1) * a.N + nbase + piece_at(32 * c < a.Ns ? 32 * c : 0);
    RX[c] = ld16(static_cast<const uint16_t*>(a.res_x) + at);
    if (a.res_r) RR[c] = ld16(static_cast<const uint16_t*>(a.res_r) + at);      // (uniform)
  };
  // Everything a workgroup reads once is on its way before the first of it is waited for.
  fetch(first_tile);
  if constexpr (RES) {
#pragma unroll
    for (int c = 0; c < NR; ++c) fetch_res(first_tile, c);
  }
  const int tn = tid < a.Ns ? tid : a.Ns - 1, tk = tid < a.K ? tid : a.K - 1;
  const float bias0 = a.bias ? ldw(a.bias, a.wbf16, nbase + tn) : 0.f;
  const float lnw0 = a.pre == kActLayerNorm ? ldw(a.ln_w, a.wbf16, tk) : 0.f, lnb0 = a.pre == kActLayerNorm ? ldw(a.ln_b, a.wbf16, tk) : 0.f;
  const float pre_s = a.pre == kActStarRelu ? ldw(a.pre_s, a.wbf16, 0) : 0.f, pre_b = a.pre == kActStarRelu ? ldw(a.pre_b, a.wbf16, 0) : 0.f;
  const float post_s = a.post == kActStarRelu ? ldw(a.post_s, a.wbf16, 0) : 0.f, post_b = a.post == kActStarRelu ? ldw(a.post_b, a.wbf16, 0) : 0.f;
  stage_rows(a.w, a.wbf16, (int64_t)nbase * a.K, pieces, tid, [&](int i, const uint4& q) {
    const int n = i / kp;
    *reinterpret_cast<uint4*>(wl + n * ws + 8 * (i - n * kp)) = q;
  });
  // (read from memory at every tile, the bias's wait was one for the next tile's rows too: they are counted in order)
  if (tid < a.Ns) bias[tid] = bias0;
  for (int i = tid + kLinThreads; i < a.Ns; i += kLinThreads) bias[i] = a.bias ? ldw(a.bias, a.wbf16, nbase + i) : 0.f;
  if (a.pre == kActLayerNorm && tid < a.K) { lnp[tid] = lnw0; lnp[a.K + tid] = lnb0; }      // (K <= 128)
  if constexpr (RES)                                     // (no normalisation here: the scale lies in its place)
    for (int i = tid; i < a.Ns; i += kLinThreads) lnp[i] = ldw(a.res_s, a.wbf16, nbase + i);
  __syncthreads();
  // A wave's tiles end at the last row.  Its lanes past that row hold and store the row's own values once more, so no store
  // sits in a branch and the wait for the next tile's rows leaves the stores behind them under way.
  for (int tile = first_tile; (int64_t)tile * 64 + wave * 16 < a.P; tile += tile_step) {
    const int64_t p = (int64_t)tile * 64 + wave * 16 + mn;
    const int64_t out = (p < a.P ? p : a.P - 1) * a.N + nbase;
    uint4 A[KCMAX];
#pragma unroll
    for (int kc = 0; kc < KCMAX; ++kc) A[kc] = Anext[kc];
    fetch(tile + tile_step);
    if (a.pre == kActLayerNorm) {   // (uniform; the host only asks for it where K <= 128)
      if constexpr (KCMAX <= 4) norm_rows<KCMAX>(A, KC, a.K, lnp, a.ln_eps, kb);
    } else if (a.pre != kActNone) {   // (uniform)
#pragma unroll
      for (int kc = 0; kc < KCMAX; ++kc)
        if (kc < KC) {
          uint32_t w4[4] = {A[kc].x, A[kc].y, A[kc].z, A[kc].w};
#pragma unroll
          for (int j = 0; j < 4; ++j)
            w4[j] = pack_bf16(act(a.pre, bf_lo(w4[j]), pre_s, pre_b), act(a.pre, bf_hi(w4[j]), pre_s, pre_b));
          A[kc] = make_uint4(w4[0], w4[1], w4[2], w4[3]);
        }
    }
    // W's rows are the first operand: lane (mn, kb) ends with outputs 4 kb + i of position mn.  Two tiles of 16 outputs at a time;
    // lanes of neighbouring kb exchange halves and store 8 neighbouring outputs each.  An odd last tile is taken twice.
    auto outputs = [&](int n0, auto&& leave) {
      const int second = n0 + 16 < a.Ns ? 16 : 0;
      uint2 zq[2], yq[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int nt = n0 + (t ? second : 0);
        const uint16_t* wrow = wl + (nt + mn) * ws + 8 * kb;
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kc = 0; kc < KCMAX; ++kc)
          if (kc < KC) acc = mfma_bf16(ld16(wrow + 32 * kc), A[kc], acc);
        const float4 bn = *reinterpret_cast<const float4*>(bias + nt + 4 * kb);
        acc[0] += bn.x; acc[1] += bn.y; acc[2] += bn.z; acc[3] += bn.w;
        if (a.z) {   // (uniform) both values leave; the activation reads what is stored, as the backward will
          zq[t] = make_uint2(pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]));
          acc[0] = bf_lo(zq[t].x); acc[1] = bf_hi(zq[t].x); acc[2] = bf_lo(zq[t].y); acc[3] = bf_hi(zq[t].y);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] = act(a.post, acc[i], post_s, post_b);
        yq[t] = make_uint2(pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]));
      }
      const int64_t at = out + piece_at(n0);
      if (a.z) *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.z) + at) = halves_exchanged(zq[0], zq[1]);
      leave(at, halves_exchanged(yq[0], yq[1]));
    };
    if constexpr (RES) {
#pragma unroll
      for (int c = 0; c < NR; ++c)
        if (32 * c < a.Ns)                               // (uniform)
          outputs(32 * c, [&](int64_t at, const uint4& layer) {
            const float4* sp = reinterpret_cast<const float4*>(lnp + piece_at(32 * c));
            const float4 s0 = sp[0], s1 = sp[1];
            const float sc[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
            const uint32_t xw[4] = {RX[c].x, RX[c].y, RX[c].z, RX[c].w}, lw[4] = {layer.x, layer.y, layer.z, layer.w};
            float r[8];
#pragma unroll
            for (int j = 0; j < 4; ++j) { r[2 * j] = bf_lo(lw[j]); r[2 * j + 1] = bf_hi(lw[j]); }
            if (a.res_r) {
              const uint32_t rw[4] = {RR[c].x, RR[c].y, RR[c].z, RR[c].w};
#pragma unroll
              for (int j = 0; j < 4; ++j) { r[2 * j] += bf_lo(rw[j]); r[2 * j + 1] += bf_hi(rw[j]); }
            }
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = pack_bf16(__builtin_fmaf(bf_lo(xw[j]), sc[2 * j], r[2 * j]), __builtin_fmaf(bf_hi(xw[j]), sc[2 * j + 1], r[2 * j + 1]));
            fetch_res(tile + tile_step, c);
            *reinterpret_cast<uint4*>(Y + at) = make_uint4(o[0], o[1], o[2], o[3]);
          });
    } else {
      for (int n0 = 0; n0 < a.Ns; n0 += 32) outputs(n0, [&](int64_t at, const uint4& q) { *reinterpret_cast<uint4*>(Y + at) = q; });
    }
  }
}

// ------------------------------------------------ wide linear layers of a few positions, bf16
// y = post(x W^T + bias) for the wide layers of the attention stages when a batch has few positions (one image: 196 and
// 49 rows).  The stock product takes the host 19 us to issue and the device 6 to 9 us; here the weights are the
// traffic and latency is the cost, so nothing is staged: a workgroup owns 32 positions x 16 NT outputs, its four
// waves share out the contraction in steps of 32 (neighbouring waves read neighbouring 64-byte pieces of a row), every
// operand is a 16-byte piece of a row straight from memory with the loads of kWideAhead steps in flight, and the
// waves' sums meet in LDS.  W's rows are the first operand: a lane ends with four neighbouring outputs of a position.
constexpr int kWideAhead = 4;
constexpr int kWideWaves = 4;
struct WideArgs {
  const uint16_t* x;      // (P, K)
  const void* w;          // (N, K)
  const void* bias;       // (N) or null
  uint16_t* y;            // (P, N)
  int P, K, N, post;
};

template <int NT, bool WBF16>
__global__ __launch_bounds__(256) void m2d_wide_linear_kernel(const WideArgs a) {
  __shared__ f32x4_t sums[kWideWaves][2 * NT][64];
  const int l = threadIdx.x & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 32;
  const uint16_t* xr[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int m = m0 + 16 * j + mn;
    xr[j] = a.x + (int64_t)(m < a.P ? m : a.P - 1) * a.K + 8 * kb;      // rows past the end repeat the last one and are not stored
  }
  const int64_t wrow = (int64_t)(n0 + mn) * a.K + 8 * kb;
  auto load_w = [&](int i, int step) {
    const int64_t at = wrow + (int64_t)16 * i * a.K + 32 * step;
    if constexpr (WBF16) {
      return ld16(static_cast<const uint16_t*>(a.w) + at);
    } else {
      const float4 lo = *reinterpret_cast<const float4*>(static_cast<const float*>(a.w) + at), hi = *reinterpret_cast<const float4*>(static_cast<const float*>(a.w) + at + 4);
      return make_uint4(pack_bf16(lo.x, lo.y), pack_bf16(lo.z, lo.w), pack_bf16(hi.x, hi.y), pack_bf16(hi.z, hi.w));
    }
  };
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[NT][2];
#pragma unroll
  for (int i = 0; i < NT; ++i) acc[i][0] = acc[i][1] = zero;
  const int steps = a.K / 32;
  for (int s0 = wave; s0 < steps; s0 += kWideWaves * kWideAhead) {
    uint4 wf[kWideAhead][NT], xf[kWideAhead][2];
#pragma unroll
    for (int k = 0; k < kWideAhead; ++k) {
      const int s = s0 + kWideWaves * k < steps ? s0 + kWideWaves * k : s0;
#pragma unroll
      for (int i = 0; i < NT; ++i) wf[k][i] = load_w(i, s);
#pragma unroll
      for (int j = 0; j < 2; ++j) xf[k][j] = ld16(xr[j] + 32 * s);
    }
#pragma unroll
    for (int k = 0; k < kWideAhead; ++k)
      if (s0 + kWideWaves * k < steps) {      // (uniform)
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = mfma_bf16(wf[k][i], xf[k][j], acc[i][j]);
      }
  }
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) sums[wave][2 * i + j][l] = acc[i][j];
  __syncthreads();
  for (int t = wave; t < 2 * NT; t += kWideWaves) {
    f32x4_t v = sums[0][t][l];
#pragma unroll
    for (int w = 1; w < kWideWaves; ++w) v += sums[w][t][l];
    const int n = n0 + 16 * (t >> 1) + 4 * kb, m = m0 + 16 * (t & 1) + mn;
    if (a.bias) {
      float b[4];
      ldwv<4>(a.bias, WBF16, n, b);
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] += b[r];
    }
    if (a.post == kActGelu) {
      // the stock layer stores its output before the activation reads it: the same rounding here
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        const uint32_t q = pack_bf16(v[r], v[r + 1]);
        v[r] = gelu_exact(bf_lo(q));
        v[r + 1] = gelu_exact(bf_hi(q));
      }
    }
    if (m < a.P) *reinterpret_cast<uint2*>(a.y + (int64_t)m * a.N + n) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
  }
}

// ------------------------------------------------------ wide linear layers with a GELU behind them, bf16
// y = GELU(x W^T + bias) for more positions than the kernel above is made for and up to 320 inputs (the first layer of the
// MLP in the third stage).  The stock product and the activation after it write the widest tensor of a block twice and
// read it once; here it is written once, and the kernel is bound by the exact GELU of every output (about 16 vector
// slots a value, half of the time) and the products.  A wave keeps 32 positions' rows in registers as they come from
// memory and walks over the outputs 32 at a time; the 32 rows of W lie in LDS, read by all waves, while the next 32 are
// on their way; three workgroups fit a compute unit, which is why 320 inputs are the most (with workgroups of 8 waves, two
// waves to a SIMD, 320 -> 1280 took 68 us at 25088 positions).  W's rows are the first operand of the product, so a lane
// ends with four neighbouring outputs of a position at a time, which leave through LDS as 64-byte pieces.
// 320 -> 1280, the fewest equal slices of a tile's outputs that make 768 workgroups, and the slices chosen below: 50176 positions 93 and 77 us,
// 25088 52 and 46, 19600 43 and 40, 12544 31 and 27, 6272 22 and 18, 1568 11.5 both; the stock pair 61 us at 25088, 28 at 6272.
// Equal ranges of the whole work for 768 workgroups, a range going on into the next tile, took 77, 46, 38, 29, 21 and 11.5, but lost 2 to 20 %
// to slices where outputs are few or inputs many (40000 positions, 320 -> 256: 28.4 us against 23.2), as a tile's rows of x are then
// waited for in the middle of a workgroup.
// 512 -> 2048 at 6272 positions, with 16 positions to a wave so that it fits: 44 us against 34, so those stay stock.
typedef float f32x16_t __attribute__((ext_vector_type(16)));
constexpr int64_t kGlFewest = 512;      // positions up to which the kernel above is the faster one
constexpr int kGlInputs = 320;          // most inputs with which three workgroups fit a compute unit's LDS
constexpr int64_t kGlMost = 8192;       // workgroups beyond which more slices are not looked at
constexpr int kGlWaves = 4, kGlThreads = 64 * kGlWaves, kGlRows = 32 * kGlWaves;
constexpr int kGlStage = 32 + 8;        // bf16 per staged position
struct GeluLinArgs {
  const uint16_t *x, *w, *bias;
  uint16_t* y;
  int64_t P;
  int K, N;
  int nsplit, steps, over;       // slices of the outputs; steps of 64 of them in a slice, `over` slices have one more
  uint32_t per_slice;            // 2^32 / nsplit, rounded up: exact as a quotient while (workgroups) x nsplit < 2^32
};

// KS: steps of 16 inputs the kernel is built for (the operands past K are zero)
template <int KS>
__global__ __launch_bounds__(kGlThreads, 3) void m2d_gelu_linear_kernel(const GeluLinArgs a) {
  constexpr int kRow = 16 * KS + 8;      // bf16 per row of W in LDS: 16-byte aligned, 16 rows cover all banks
  constexpr int kPer = kGlThreads / 32;  // threads that bring a row of W, 16 bytes each at a time
  constexpr int kPieces = (2 * KS + kPer - 1) / kPer;
  __shared__ __attribute__((aligned(16))) uint16_t wl[2][32 * kRow];
  __shared__ __attribute__((aligned(16))) uint16_t staged[kGlWaves][32 * kGlStage];
  __shared__ __attribute__((aligned(16))) float bl[2][32];      // bias of the 32 outputs
  const int tid = threadIdx.x, l = tid & 63, r = l & 31, h = l >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // the slices of the same positions go to the same XCD (workgroups are dealt out round-robin over 8), whose L2 then holds their
  // rows of x for all of them: an eighth of all slices each, which may part those of one tile, so that no XCD has a tile more than another.
  // (Every division here was 0.1 us of each workgroup's start: 4000 positions, 256 -> 1024 10.7 us, 11.2 with four of them.)
  const uint32_t mine = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const uint32_t tile = a.nsplit == 1 ? mine : __umulhi(mine, a.per_slice);
  const int slice = (int)(mine - tile * (uint32_t)a.nsplit);
  const int n0 = 64 * (slice * a.steps + (slice < a.over ? slice : a.over)), chunks = 2 * (a.steps + (slice < a.over ? 1 : 0));
  const int64_t p0 = (int64_t)tile * kGlRows + wave * 32;
  if ((int64_t)tile * kGlRows >= a.P) return;      // (the whole workgroup)
  const int64_t first = p0 < a.P ? p0 : a.P - 1;      // rows past the end repeat the last one and are not stored
  const int left = a.P - first < 32 ? (int)(a.P - first) : 32, stored = p0 < a.P ? left : 0;
  const int row = r < left ? r : left - 1;
  uint16_t* y = a.y + first * a.N + n0;
  const int wr = tid / kPer, wc = 8 * (tid % kPer);
  uint4 next[kPieces];
  float nb = 0.f;
  const uint4 z4 = make_uint4(0u, 0u, 0u, 0u);
  auto fetch = [&](int chunk) {
    const uint16_t* src = a.w + (int64_t)(n0 + 32 * chunk) * a.K;
#pragma unroll
    for (int u = 0; u < kPieces; ++u)
      if (wc + 8 * kPer * u < a.K) next[u] = ld16(src + (uint32_t)(wr * a.K + wc + 8 * kPer * u));
    if (tid < 32) nb = a.bias ? __uint_as_float((uint32_t)a.bias[n0 + 32 * chunk + tid] << 16) : 0.f;
  };
  auto put = [&](int b) {
#pragma unroll
    for (int u = 0; u < kPieces; ++u)
      if (wc + 8 * kPer * u < a.K) *reinterpret_cast<uint4*>(&wl[b][wr * kRow + wc + 8 * kPer * u]) = next[u];
    if (tid < 32) bl[b][tid] = nb;
  };
  if (a.K < 16 * KS) {      // (uniform) inputs past K
#pragma unroll
    for (int u = 0; u < kPieces; ++u) {
      const int at = wc + 8 * kPer * u;
      if (at >= a.K && at < 16 * KS) *reinterpret_cast<uint4*>(&wl[0][wr * kRow + at]) = *reinterpret_cast<uint4*>(&wl[1][wr * kRow + at]) = z4;
    }
  }
  fetch(0);
  uint4 X[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) X[s] = 16 * s < a.K ? ld16(a.x + first * a.K + (uint32_t)(row * a.K + 16 * s + 8 * h)) : z4;
  put(0);
  __syncthreads();
  uint16_t* st = staged[wave];
  for (int c = 0; c < chunks; ++c) {
    const bool more = c + 1 < chunks;
    if (more) fetch(c + 1);
    f32x16_t acc;
    const uint16_t* wrow = &wl[c & 1][r * kRow + 8 * h];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x4_t b4 = *reinterpret_cast<const f32x4_t*>(&bl[c & 1][8 * g + 4 * h]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[4 * g + i] = b4[i];
    }
#pragma unroll
    for (int s = 0; s < KS; ++s)
      acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, ld16(wrow + 16 * s)), __builtin_bit_cast(bf16x8_t, X[s]), acc, 0, 0, 0);
#pragma unroll
    for (int g = 0; g < 4; ++g) {      // the lane's outputs 8 g + 4 h .. + 3
      // the stock layer stores its output before the activation reads it: the same rounding here
      const uint32_t q0 = pack_bf16(acc[4 * g], acc[4 * g + 1]), q1 = pack_bf16(acc[4 * g + 2], acc[4 * g + 3]);
      *reinterpret_cast<uint2*>(st + r * kGlStage + 8 * g + 4 * h) =
          make_uint2(pack_bf16(gelu_exact(bf_lo(q0)), gelu_exact(bf_hi(q0))), pack_bf16(gelu_exact(bf_lo(q1)), gelu_exact(bf_hi(q1))));
    }
    if (more) put((c + 1) & 1);      // (its readers passed the barrier at the end of the last chunk)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int m = (l >> 2) + 16 * k, c8 = 8 * (l & 3);
      if (m < stored) *reinterpret_cast<uint4*>(y + (int64_t)16 * k * a.N + 32 * c + (uint32_t)((l >> 2) * a.N + c8)) = ld16(st + m * kGlStage + c8);
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------ the MLP of a narrow stage, bf16
// y = fc2(GELU(fc1 x)) (models/utils.py:58-81) where both weight matrices fit LDS together (C = 32 or 64
// channels, 4 C hidden units): the hidden activations, four times the size of x and y and the reason why
// the two layers run at the speed of memory writes when they are separate kernels, never leave the
// registers.  A wave owns 16 rows.  H^T = W1 X^T puts, in lane (mn, kb), the hidden units 16 nt + 4 kb + i of
// row mn; Y^T = W2 H^T contracts 32 hidden units per instruction and, as its operands may list them in any
// order as long as both agree, takes for the lane's eight slots exactly the units the lane holds (4 kb + i of
// two neighbouring tiles), with W2's rows read to match: no exchange of H between lanes.  Y^T leaves lane
// (mn, kb) with outputs 16 no + 4 kb + i of row mn: 8-byte stores.
struct MlpArgs {
  const void* x;          // (P, C) bf16
  const void *w1, *b1;    // (H, C), (H) or null
  const void *w2, *b2;    // (C, H), (C) or null
  void* y;                // (P, C) bf16
  int64_t P;
  int wbf16, ntiles;
  const void *ln_w, *ln_b;   // LayerNorm over C in front of fc1: weight and bias, (C), or null
  float ln_eps;
  const void *res_s, *nx_w, *nx_b;   // RES: scale of the residual stream, weight and bias of the norm behind the update, (C)
  float nx_eps;
  void* xo;               // RES: (P, C) the updated stream; y is its norm
  void* z;                // KEEP: (P, 4 C) bf16, the first layer's output before the GELU
};

// KC: C = 32 KC channels, 128 KC hidden units.
// RES: xo = x * res_s + MLP(x), y = LayerNorm(xo), the residual update and the next block's norm in the bits that m2d_layernorm_kernel gives behind
// this one: after an exchange of halves a lane holds whole 8-channel pieces of its row (piece 4 c + {0, 2, 1, 3}[kb]), and the row's sums are
// folded in that kernel's order: pieces 8, 4, 2 and 1 apart.  The products and the GELU are what takes this kernel's time, so what
// it moves beside them costs little: 128x56x56x64 83 us where the two kernels took 110 + 33.
// 32 hidden units at a time go from the first product into the second, one such step a turn of the loop: a wave then needs 113 registers where all 256
// units of a row at once took 256, and four waves to a SIMD in place of two cover each other's waits for LDS, products and exponentials
// (401408 rows of 64 channels, RES: 119 -> 83 us; two rows' tiles a wave on the same weights, with three waves a SIMD, 107).
// 128 channels: a quarter of the hidden units has its weights in LDS at a time, fetched for every tile of 128 rows; of the two workgroups of a unit
// one computes while the other fetches.  100352 rows 78 us, where layer, library product and update with norm took 110 (hidden activations of 103 MB out
// and back); 50176 40 and 62.
constexpr int mlp_slices(int kc) { return kc <= 2 ? 1 : 4; }
// KEEP: fc1's output leaves too, and the GELU reads what is stored, as the backward will: without reading it back the two layers of
// a training forward take 48 us for 200704 rows of 64 channels where two kernels took 76 (12544: 9.7 and 18).
template <int KC, bool RES, int TH, bool KEEP = false>
__global__ __launch_bounds__(TH, TH / 128) void m2d_mlp_kernel(const MlpArgs a) {
  constexpr int C = 32 * KC, HD = 4 * C, SL = mlp_slices(KC), HS = HD / SL, NO = C / 16, NP = HS / 32;
  constexpr int W1S = C + 8;      // bf16 per row of W1 in LDS (a row per hidden unit)
  constexpr int W2S = HS + 4;     // bf16 per row of W2 (a row per output): rows stay 8-byte aligned and spread over the banks
  extern __shared__ float smem[];
  uint16_t* w1l = reinterpret_cast<uint16_t*>(smem);
  uint16_t* w2l = w1l + HS * W1S;
  float* b1l = reinterpret_cast<float*>(w2l + C * W2S);
  const int tid = threadIdx.x, l = tid & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto put = [&](uint16_t* row, int k8, const uint4& q) {
    uint2* d = reinterpret_cast<uint2*>(row + 8 * k8);      // rows of W2 are 8-byte aligned only
    d[0] = make_uint2(q.x, q.y);
    d[1] = make_uint2(q.z, q.w);
  };
  auto stage_weights = [&](int slice) {                       // hidden units slice * HS ..., 8 elements at a time
    int tid = threadIdx.x;
    if constexpr (SL > 1) asm volatile("" : "+v"(tid));      // (addresses are worked out here: held across the products they cost 40 registers)
    stage_rows<TH>(a.w1, a.wbf16, (int64_t)slice * HS * C, HS * (C / 8), tid, [&](int i, const uint4& q) { put(w1l + i / (C / 8) * W1S, i % (C / 8), q); });
    stage_rows<TH, HS, HD>(a.w2, a.wbf16, slice * HS, C * (HS / 8), tid, [&](int i, const uint4& q) { put(w2l + i / (HS / 8) * W2S, i % (HS / 8), q); });
  };
  const uint16_t* X = static_cast<const uint16_t*>(a.x);
  uint16_t* Y = static_cast<uint16_t*>(a.y);
  uint4 Xnext[KC];
  auto fetch = [&](int tile) {      // (rows past the end repeat the last one, see m2d_linear_kernel)
    const int64_t q = ((int64_t)tile * (TH / 64) + wave) * 16 + mn;
    const uint16_t* row = X + (q < a.P ? q : a.P - 1) * C + 8 * kb;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) Xnext[kc] = ld16(row + 32 * kc);
  };
  static_assert(HD <= TH && C <= TH, "one hidden unit's bias a thread");
  if constexpr (SL == 1) fetch(blockIdx.x);
  const int th = tid < HD ? tid : HD - 1, tc = tid < C ? tid : C - 1;
  const float b10 = a.b1 ? ldw(a.b1, a.wbf16, th) : 0.f;
  const float lnw0 = a.ln_w ? ldw(a.ln_w, a.wbf16, tc) : 0.f, lnb0 = a.ln_w ? ldw(a.ln_b, a.wbf16, tc) : 0.f;
  const float b20 = a.b2 ? ldw(a.b2, a.wbf16, tc) : 0.f;
  if constexpr (SL == 1) stage_weights(0);
  if (tid < HD) b1l[tid] = b10;
  float* lnp = b1l + HD;
  float* b2l = lnp + 2 * C;
  if (tid < C) b2l[tid] = b20;
  if (a.ln_w && tid < C) { lnp[tid] = lnw0; lnp[C + tid] = lnb0; }
  const float* nxp = b2l + C;      // RES: scale, weight, bias
  if constexpr (RES) {
    if (tid < C) {
      float* d = b2l + C + tid;
      d[0] = ldw(a.res_s, a.wbf16, tid); d[C] = ldw(a.nx_w, a.wbf16, tid); d[2 * C] = ldw(a.nx_b, a.wbf16, tid);
    }
  }
  __syncthreads();
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  const int piece = (kb & 1 ? 16 : 0) + 4 * (kb & 2);
  for (int tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    const int64_t p = ((int64_t)tile * (TH / 64) + wave) * 16 + mn;      // the lane's row
    uint4 Xf[KC];
    if constexpr (SL > 1) {      // (the weights are waited for at every tile anyhow)
      fetch(tile);
      __syncthreads();
      stage_weights(0);
    }
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) Xf[kc] = Xnext[kc];
    if constexpr (SL == 1) fetch(tile + gridDim.x);
    if (a.ln_w) norm_rows<KC>(Xf, KC, C, lnp, a.ln_eps, kb);      // (uniform)
    f32x4_t out[NO];
#pragma unroll
    for (int no = 0; no < NO; ++no) out[no] = zero;
#pragma unroll 1
    for (int slice = 0; slice < SL; ++slice) {
      if constexpr (SL > 1) {      // (a workgroup's waves have the same tiles)
        if (slice) {
          __syncthreads();
          stage_weights(slice);
        }
        __syncthreads();
      }
#pragma unroll 1
      for (int ks = 0; ks < NP; ++ks) {
        uint2 hq[2], zq[2];      // the hidden activations as bf16, as fc2 of the stock path would read them
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          const uint16_t* w = w1l + (32 * ks + 16 * half + mn) * W1S + 8 * kb;
          f32x4_t acc = zero;
#pragma unroll
          for (int kc = 0; kc < KC; ++kc) acc = mfma_bf16(ld16(w + 32 * kc), Xf[kc], acc);
          const float4 b1 = *reinterpret_cast<const float4*>(b1l + slice * HS + 32 * ks + 16 * half + 4 * kb);
          acc[0] += b1.x; acc[1] += b1.y; acc[2] += b1.z; acc[3] += b1.w;
          if constexpr (KEEP) {
            zq[half] = make_uint2(pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]));
            acc[0] = bf_lo(zq[half].x); acc[1] = bf_hi(zq[half].x); acc[2] = bf_lo(zq[half].y); acc[3] = bf_hi(zq[half].y);
          }
          hq[half] = make_uint2(pack_bf16(gelu_exact(acc[0]), gelu_exact(acc[1])), pack_bf16(gelu_exact(acc[2]), gelu_exact(acc[3])));
        }
        if constexpr (KEEP) {
          const uint4 q = halves_exchanged(zq[0], zq[1]);
          if (p < a.P) *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.z) + p * HD + slice * HS + 32 * ks + piece) = q;
        }
#pragma unroll
        for (int no = 0; no < NO; ++no) {
          const uint16_t* w = w2l + (16 * no + mn) * W2S + 32 * ks + 4 * kb;      // output 16 no + mn, units 32 ks + 4 kb + {0..3, 16..19}
          const uint2 lo = *reinterpret_cast<const uint2*>(w), hi = *reinterpret_cast<const uint2*>(w + 16);
          out[no] = mfma_bf16(make_uint4(lo.x, lo.y, hi.x, hi.y), make_uint4(hq[0].x, hq[0].y, hq[1].x, hq[1].y), out[no]);
        }
      }
    }
    uint2 yq[NO];
#pragma unroll
    for (int no = 0; no < NO; ++no) {
      const float4 b2 = *reinterpret_cast<const float4*>(b2l + 16 * no + 4 * kb);
      yq[no] = make_uint2(pack_bf16(out[no][0] + b2.x, out[no][1] + b2.y), pack_bf16(out[no][2] + b2.z, out[no][3] + b2.w));
    }
    if constexpr (!RES) {
#pragma unroll
      for (int no = 0; no < NO; ++no)
        if (p < a.P) *reinterpret_cast<uint2*>(Y + p * C + 16 * no + 4 * kb) = yq[no];
    } else {
      uint4 xr[KC], xo[KC];             // the stream again, as the results lie
#pragma unroll
      for (int c = 0; c < KC; ++c) xr[c] = ld16(X + (p < a.P ? p : a.P - 1) * C + 32 * c + piece);
      float part[KC];
      // the sum of a row's pieces: piece ^ 8 and ^ 4 are the lane's own, ^ 2 and ^ 1 are in the lanes 16 and 32 further
      auto row_sum = [&](const float (&v)[KC]) {
        float s = KC == 4 ? (v[0] + v[KC / 2]) + (v[KC / 4] + v[KC - 1]) : KC == 2 ? v[0] + v[KC - 1] : v[0];
        s += __shfl_xor(s, 16, 64);
        s += __shfl_xor(s, 32, 64);
        return s;
      };
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const uint4 m = halves_exchanged(yq[2 * c], yq[2 * c + 1]);
        const uint32_t mw[4] = {m.x, m.y, m.z, m.w}, xw[4] = {xr[c].x, xr[c].y, xr[c].z, xr[c].w};
        const float* sc = nxp + 32 * c + piece;
        uint32_t o[4];
        part[c] = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          o[j] = pack_bf16(__builtin_fmaf(bf_lo(xw[j]), sc[2 * j], bf_lo(mw[j])), __builtin_fmaf(bf_hi(xw[j]), sc[2 * j + 1], bf_hi(mw[j])));
          part[c] += bf_lo(o[j]); part[c] += bf_hi(o[j]);      // (the norm sees what is stored)
        }
        xo[c] = make_uint4(o[0], o[1], o[2], o[3]);
      }
      const float mean = row_sum(part) * (1.f / C);
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const uint32_t xw[4] = {xo[c].x, xo[c].y, xo[c].z, xo[c].w};
        part[c] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; ++j) { const float d = (j & 1 ? bf_hi(xw[j / 2]) : bf_lo(xw[j / 2])) - mean; part[c] = __builtin_fmaf(d, d, part[c]); }
      }
      const float rstd = rsqrtf(row_sum(part) * (1.f / C) + a.nx_eps);
#pragma unroll
      for (int c = 0; c < KC; ++c) {
        const float *w = nxp + C + 32 * c + piece, *b = w + C;
        const uint32_t xw[4] = {xo[c].x, xo[c].y, xo[c].z, xo[c].w};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
          o[j] = pack_bf16(__builtin_fmaf((bf_lo(xw[j]) - mean) * rstd, w[2 * j], b[2 * j]), __builtin_fmaf((bf_hi(xw[j]) - mean) * rstd, w[2 * j + 1], b[2 * j + 1]));
        if (p < a.P) {
          const int64_t at = p * C + 32 * c + piece;
          *reinterpret_cast<uint4*>(static_cast<uint16_t*>(a.xo) + at) = xo[c];
          *reinterpret_cast<uint4*>(Y + at) = make_uint4(o[0], o[1], o[2], o[3]);
        }
      }
    }
  }
}

template <int KC>
constexpr size_t mlp_lds_bytes() {
  constexpr size_t C = 32 * KC, HS = 4 * C / mlp_slices(KC);
  return HS * (C + 8) * 2 + C * (HS + 4) * 2 + 4 * C * 4 + 3 * C * 4;
}

constexpr size_t kLinMaxLds = 160 * 1024;   // LDS of a compute unit

constexpr int kMlpThreads = 512;      // of the kernel for many positions
// More than 64 KB of dynamic LDS has to be allowed per kernel and device, once.
inline bool allow_big_lds() {
  static std::atomic<uint64_t> seen{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  const uint64_t bit = 1ull << (dev & 63);
  if (seen.load(std::memory_order_acquire) & bit) return true;
  const void* kernels[] = {reinterpret_cast<const void*>(&m2d_linear_kernel<2>), reinterpret_cast<const void*>(&m2d_linear_kernel<4>),
                           reinterpret_cast<const void*>(&m2d_linear_kernel<8>), reinterpret_cast<const void*>(&m2d_linear_kernel<16>),
                           reinterpret_cast<const void*>(&m2d_mlp_kernel<2, false, kMlpThreads>), reinterpret_cast<const void*>(&m2d_mlp_kernel<2, false, kLinThreads>),
                           reinterpret_cast<const void*>(&m2d_mlp_kernel<2, true, kMlpThreads>), reinterpret_cast<const void*>(&m2d_mlp_kernel<2, true, kLinThreads>),
                           reinterpret_cast<const void*>(&m2d_mlp_kernel<4, true, kMlpThreads>),
                           reinterpret_cast<const void*>(&m2d_mlp_kernel<2, false, kMlpThreads, true>), reinterpret_cast<const void*>(&m2d_mlp_kernel<2, false, kLinThreads, true>)};
  for (const void* k : kernels)
    if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLinMaxLds) != hipSuccess) return false;
  seen.fetch_or(bit, std::memory_order_release);
  return true;
}

// LDS of the kernel: the slice of W, its bias, the normalisation's weight and bias.
inline size_t linear_lds_bytes(int K, int N, bool ln) {
  return ((size_t)N * (K + 8) / 2 + 3) / 4 * 4 * 4 + (size_t)N * 4 + (ln ? (size_t)2 * K * 4 : 0);
}
// What the choice of slices and the limit of what is taken count with.
inline size_t linear_slice_bytes(int K, int N, bool ln) {
  return ((size_t)N * (K + 8) / 2 + 3) / 4 * 4 * 4 + kLinMargin + (ln ? (size_t)2 * K * 4 : 0);
}

// ------------------------------------------ attention of the rotary stages, one head per workgroup
// softmax(q k^T / sqrt(hd)) v with q and k rotated by position and LayerNormed per head first
// (models/utils.py:253-316), for heads of 32 features and up to 256 tokens (the 14x14 and 7x7 grids of
// the attention stages), straight from the output of the qkv projection, (B, L, 3, heads, 32), to
// (B, L, heads, 32), the input of the output projection: one pass in place of the rotation, the two
// LayerNorms, the attention kernel and the copies between them.
//   staging: a quad of lanes rotates and normalises q and k of a token (8 features per lane) and leaves
//     them in LDS as bf16 rows, and v transposed (feature-major), rows and columns past L zero;
//   a wave takes 16 queries at a time.  S^T = K Q^T, one v_mfma_f32_16x16x32_bf16 per 16 keys (the
//     contraction is the 32 features): lane (mn, kb) holds the scores of query mn for keys 16 kt + 4 kb + i.
//     Row maximum and sum are in-lane plus two lane exchanges (kb).  O^T = V^T P^T contracts 32 keys per
//     instruction; its operands may list the keys in any order as long as both agree, so the lane's
//     eight slots take the probabilities it already holds (keys 4 kb + i of two neighbouring tiles) and
//     V^T supplies the same keys: no exchange of the probabilities between lanes.
constexpr int kAttHd = 32;
constexpr int kAttRow = kAttHd + 8;     // bf16 per row of q and k in LDS
constexpr int kAttMaxL = 256;

struct AttnArgs {
  const void* qkv;                 // (B, L, 3, heads, 32) bf16
  const void *cos, *sin;           // (L, 32) bf16
  const void *qw, *qb, *kw, *kb;   // LayerNorm weights of q and k, (32)
  void* out;                       // (B, L, heads, 32) bf16
  int L, heads, wbf16;
  float eps, scale_log2e;          // softmax scale times log2(e)
};

// sum over the four lanes of a quad (lanes 4 g .. 4 g + 3), left in all of them
__device__ __forceinline__ float quad_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, true));   // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, true));   // quad_perm [2,3,0,1]
  return v;
}

// A quarter (8 features, one lane of a quad) of one token's q or k: rotation, LayerNorm over the quad, bf16 to dst.
__device__ __forceinline__ void rope_norm_quarter(const uint16_t* src, const float (&cs)[8], const float (&sn)[8], const float (&wv)[8],
                                                  const float (&bv)[8], float eps, uint16_t* dst) {
  float x[8], v[8];
  Chunk<bf16_t>::load(reinterpret_cast<const bf16_t*>(src), x);
#pragma unroll
  for (int j = 0; j < 8; j += 2) {
    v[j] = __builtin_fmaf(x[j], cs[j], -x[j + 1] * sn[j]);
    v[j + 1] = __builtin_fmaf(x[j + 1], cs[j + 1], x[j] * sn[j + 1]);
  }
  const float mean = quad_sum(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]))) * (1.f / kAttHd);
  float d[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) d[j] = v[j] - mean;
  const float sq = quad_sum(((d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3])) + ((d[4] * d[4] + d[5] * d[5]) + (d[6] * d[6] + d[7] * d[7])));
  const float rstd = rsqrtf(sq * (1.f / kAttHd) + eps);
  float o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = __builtin_fmaf(d[j] * rstd, wv[j], bv[j]);
  *reinterpret_cast<uint4*>(dst) = make_uint4(pack_bf16(o[0], o[1]), pack_bf16(o[2], o[3]), pack_bf16(o[4], o[5]), pack_bf16(o[6], o[7]));
}

constexpr int att_waves(int nt) { return nt <= 4 ? nt : (nt + 1) / 2; }   // one or two tiles of 16 queries per wave

template <int NT>   // tiles of 16 tokens: 16 (NT - 1) < L <= 16 NT
__global__ __launch_bounds__(64 * att_waves(NT)) __attribute__((amdgpu_waves_per_eu(4, 8)))
void m2d_rope_attention_kernel(const AttnArgs a) {
  constexpr int NP = (NT + 1) / 2;      // steps of 32 keys in the second product
  constexpr int LQ = 16 * NT;           // rows of q and k
  constexpr int LP = 32 * NP;           // columns of V^T
  constexpr int VS = LP + 4;            // bf16 per row of V^T: rows stay 8-byte aligned and spread over the banks
  constexpr int kThreads = 64 * att_waves(NT);
  __shared__ __attribute__((aligned(16))) uint16_t Qs[LQ * kAttRow];
  __shared__ __attribute__((aligned(16))) uint16_t Ks[LQ * kAttRow];
  __shared__ __attribute__((aligned(16))) uint16_t Vt[kAttHd * VS];
  const int tid = threadIdx.x, l = tid & 63, mn = l & 15, kb = l >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = blockIdx.x % a.heads;
  const int64_t b = blockIdx.x / a.heads;
  const int part = a.heads * kAttHd;                     // elements from q to k to v of a token
  const uint16_t* base = static_cast<const uint16_t*>(a.qkv) + (b * a.L * 3 * a.heads + head) * (int64_t)kAttHd;
  {   // staging: a quad of lanes per token, 8 features each, so that a token's 64 bytes are one piece of a load
    const int c8 = 8 * (tid & 3);
    float wq[8], bq[8], wk[8], bk[8];
    ldwv<8>(a.qw, a.wbf16, c8, wq);
    ldwv<8>(a.qb, a.wbf16, c8, bq);
    ldwv<8>(a.kw, a.wbf16, c8, wk);
    ldwv<8>(a.kb, a.wbf16, c8, bk);
    for (int t = tid >> 2; t < LP; t += kThreads / 4) {
      uint16_t* qd = Qs + t * kAttRow + c8;
      uint16_t* kd = Ks + t * kAttRow + c8;
      if (t < a.L) {     // (whole quads take the same side)
        const uint16_t* row = base + (int64_t)t * 3 * part + c8;
        float cs[8], sn[8];
        Chunk<bf16_t>::load(static_cast<const bf16_t*>(a.cos) + t * kAttHd + c8, cs);
        Chunk<bf16_t>::load(static_cast<const bf16_t*>(a.sin) + t * kAttHd + c8, sn);
        const uint4 vq = ld16(row + 2 * part);
        rope_norm_quarter(row, cs, sn, wq, bq, a.eps, qd);
        rope_norm_quarter(row + part, cs, sn, wk, bk, a.eps, kd);
        const uint32_t w4[4] = {vq.x, vq.y, vq.z, vq.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          Vt[(c8 + 2 * j) * VS + t] = (uint16_t)(w4[j] & 0xffffu);
          Vt[(c8 + 2 * j + 1) * VS + t] = (uint16_t)(w4[j] >> 16);
        }
      } else {
        if (t < LQ) {
          *reinterpret_cast<uint4*>(qd) = make_uint4(0u, 0u, 0u, 0u);
          *reinterpret_cast<uint4*>(kd) = make_uint4(0u, 0u, 0u, 0u);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) Vt[(c8 + j) * VS + t] = 0;
      }
    }
  }
  __syncthreads();
  const float ninf = -__builtin_huge_valf();
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
  uint16_t* out = static_cast<uint16_t*>(a.out);
  for (int qt = wave; qt < NT; qt += att_waves(NT)) {
    // The operands from k and v are the same for both tiles of a wave; read again, they cost LDS cycles that are
    // free here, kept in registers they would cost a quarter of the waves.  An offset the compiler cannot see
    // through keeps the loads inside the loop.
    int again = 0;
    asm volatile("" : "+v"(again));
    const uint16_t* Kl = Ks + again;
    const uint16_t* Vl = Vt + again;
    const uint4 qf = ld16(Qs + (16 * qt + mn) * kAttRow + 8 * kb);
    f32x4_t s[NT];
#pragma unroll
    for (int kt = 0; kt < NT; ++kt) s[kt] = mfma_bf16(ld16(Kl + (16 * kt + mn) * kAttRow + 8 * kb), qf, zero);
#pragma unroll
    for (int i = 0; i < 4; ++i)      // only the last tile can hold keys past the end: they take no part
      if (16 * (NT - 1) + 4 * kb + i >= a.L) s[NT - 1][i] = ninf;
    // maximum and sum run as four chains (one per i) and meet at the end
    float mx[4] = {ninf, ninf, ninf, ninf};
#pragma unroll
    for (int kt = 0; kt < NT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx[i] = fmaxf(mx[i], s[kt][i]);
    float m = fmaxf(fmaxf(mx[0], mx[1]), fmaxf(mx[2], mx[3]));
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    const float mc = m * a.scale_log2e;
    float sm[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kt = 0; kt < NT; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][i], a.scale_log2e, -mc));
        s[kt][i] = pr;
        sm[i] += pr;
      }
    float sum = (sm[0] + sm[1]) + (sm[2] + sm[3]);
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    f32x4_t o0 = zero, o1 = zero;
#pragma unroll
    for (int ks = 0; ks < NP; ++ks) {
      uint4 pf;
      pf.x = pack_bf16(s[2 * ks][0], s[2 * ks][1]);
      pf.y = pack_bf16(s[2 * ks][2], s[2 * ks][3]);
      if (2 * ks + 1 < NT) {
        pf.z = pack_bf16(s[2 * ks + 1][0], s[2 * ks + 1][1]);
        pf.w = pack_bf16(s[2 * ks + 1][2], s[2 * ks + 1][3]);
      } else {      // an odd number of tiles: the last step holds 16 keys
        pf.z = 0u; pf.w = 0u;
      }
      const uint16_t* v0 = Vl + mn * VS + 32 * ks + 4 * kb;      // features mn and 16 + mn, keys 32 ks + 4 kb + {0..3, 16..19}
      const uint2 a0 = *reinterpret_cast<const uint2*>(v0), a1 = *reinterpret_cast<const uint2*>(v0 + 16);
      const uint2 c0 = *reinterpret_cast<const uint2*>(v0 + 16 * VS), c1 = *reinterpret_cast<const uint2*>(v0 + 16 * VS + 16);
      o0 = mfma_bf16(make_uint4(a0.x, a0.y, a1.x, a1.y), pf, o0);
      o1 = mfma_bf16(make_uint4(c0.x, c0.y, c1.x, c1.y), pf, o1);
    }
    const float inv = 1.f / sum;
    const int q = 16 * qt + mn;
    if (q < a.L) {      // lane (mn, kb): features 4 kb + i and 16 + 4 kb + i of query mn
      uint16_t* dst = out + ((b * a.L + q) * a.heads + head) * (int64_t)kAttHd + 4 * kb;
      *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16(o0[0] * inv, o0[1] * inv), pack_bf16(o0[2] * inv, o0[3] * inv));
      *reinterpret_cast<uint2*>(dst + 16) = make_uint2(pack_bf16(o1[0] * inv, o1[1] * inv), pack_bf16(o1[2] * inv, o1[3] * inv));
    }
  }
}

// ------------------------------------------------------------------ parameters held in bf16
// One launch for all the small parameters that the scans of a stage want in fp32 (48 casts of 4.4 us each in a batch of
// the backbone otherwise).
constexpr int kWidenSegs = 64;
struct WidenArgs {
  struct { const uint16_t* in; float* out; int n, first; } s[kWidenSegs];
  int nsegs;
};
__global__ __launch_bounds__(256) void m2d_widen_kernel(const WidenArgs a) {
  int k = 0;
  while (k + 1 < a.nsegs && (int)blockIdx.x >= a.s[k + 1].first) ++k;
  const int i = ((int)blockIdx.x - a.s[k].first) * 256 + threadIdx.x;
  if (i < a.s[k].n) a.s[k].out[i] = __uint_as_float((uint32_t)a.s[k].in[i] << 16);
}

template <int NT>
void launch_attention(const AttnArgs& a, unsigned blocks, hipStream_t st) {
  hipLaunchKernelGGL(m2d_rope_attention_kernel<NT>, dim3(blocks), dim3(64 * att_waves(NT)), 0, st, a);
}

}  // namespace

extern "C" {

int m2d_widen(int nsegs, const m2d_widen_seg* segs, void* stream) {
  if (!segs) return M2D_ERR_NULL_POINTER;
  if (nsegs < 1) return M2D_ERR_BAD_SHAPE;
  for (int at = 0; at < nsegs;) {
    WidenArgs a = {};
    int64_t blocks = 0;
    for (; at < nsegs && a.nsegs < kWidenSegs; ++at) {
      if (!segs[at].in || !segs[at].out) return M2D_ERR_NULL_POINTER;
      if (segs[at].n < 1 || segs[at].n >= ((int64_t)1 << 31)) return M2D_ERR_BAD_SHAPE;
      auto& s = a.s[a.nsegs++];
      s.in = static_cast<const uint16_t*>(segs[at].in); s.out = segs[at].out; s.n = (int)segs[at].n; s.first = (int)blocks;
      blocks += (segs[at].n + 255) / 256;
      if (blocks >= ((int64_t)1 << 31)) return M2D_ERR_UNSUPPORTED;
    }
    hipLaunchKernelGGL(m2d_widen_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  }
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_layernorm_fwd(int64_t rows, int C, int dtype, int weight_dtype, const void* x, const void* weight,
                      const void* bias, float eps, void* y, void* stream) {
  if (!x || !weight || !bias || !y) return M2D_ERR_NULL_POINTER;
  if (rows < 1 || C < 1) return M2D_ERR_BAD_SHAPE;
  if ((dtype != M2D_F32 && dtype != M2D_BF16) || (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;
  const int V = dtype == M2D_BF16 ? 8 : 4;
  if (C % V != 0 || C / V > 64 * kMaxChunks) return M2D_ERR_UNSUPPORTED;   // rows of whole 16-byte chunks, at most 4096 (bf16) / 2048 (fp32) channels
  if (misaligned(x, 16) || misaligned(y, 16) || misaligned(weight, 16) || misaligned(bias, 16)) return M2D_ERR_MISALIGNED;
  LnArgs a = {};
  a.x = x; a.w = weight; a.b = bias; a.y = y; a.rows = rows; a.C = C; a.wbf16 = weight_dtype == M2D_BF16; a.eps = eps;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == M2D_F32 ? run_ln<float, false>(a, st) : run_ln<bf16_t, false>(a, st);
}

int m2d_scale_residual_layernorm_fwd(int64_t rows, int C, int dtype, int weight_dtype, const void* x, const void* scale,
                                     const void* residual, const void* residual2, const void* weight, const void* bias,
                                     float eps, void* x_out, void* y, void* stream) {
  if (!x || !scale || !residual || !weight || !bias || !x_out || !y) return M2D_ERR_NULL_POINTER;
  if (rows < 1 || C < 1) return M2D_ERR_BAD_SHAPE;
  if ((dtype != M2D_F32 && dtype != M2D_BF16) || (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;
  const int V = dtype == M2D_BF16 ? 8 : 4;
  if (C % V != 0 || C / V > 64 * kMaxChunks) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(residual, 16) || misaligned(residual2, 16) || misaligned(x_out, 16) || misaligned(y, 16) ||
      misaligned(scale, 16) || misaligned(weight, 16) || misaligned(bias, 16))
    return M2D_ERR_MISALIGNED;
  LnArgs a = {};
  a.x = x; a.w = weight; a.b = bias; a.y = y; a.rows = rows; a.C = C; a.wbf16 = weight_dtype == M2D_BF16; a.eps = eps;
  a.s = scale; a.r = residual; a.r2 = residual2; a.xo = x_out;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == M2D_F32 ? run_ln<float, true>(a, st) : run_ln<bf16_t, true>(a, st);
}

static int run_dwconv(int B, int H, int W, int C, int dtype, int weight_dtype, const void* x, const void* weight, void* y,
                      const void* star_scale, const void* star_bias, void* stream) {
  if (!x || !weight || !y) return M2D_ERR_NULL_POINTER;
  if (B < 1 || H < 1 || W < 1 || C < 1) return M2D_ERR_BAD_SHAPE;
  if ((dtype != M2D_F32 && dtype != M2D_BF16) || (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;
  const int V = dtype == M2D_BF16 ? 8 : 4;
  if (C % V != 0) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(y, 16) || misaligned(weight, 16)) return M2D_ERR_MISALIGNED;
  DwArgs a = {};
  a.x = x; a.w = weight; a.y = y; a.B = B; a.H = H; a.W = W; a.C = C; a.wbf16 = weight_dtype == M2D_BF16;
  a.star_s = star_scale; a.star_b = star_bias;
  const int strip = W % 14 == 0 ? 14 : 8;
  a.strips = (W + strip - 1) / strip;
  const int64_t total = (int64_t)B * H * a.strips * (C / V);
  const int64_t blocks = (total + kDwThreads - 1) / kDwThreads;
  if (blocks >= ((int64_t)1 << 31)) return M2D_ERR_UNSUPPORTED;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)blocks), block(kDwThreads);
  if (star_scale) {
    if (strip == 14) hipLaunchKernelGGL((m2d_dwconv3x3_kernel<bf16_t, 14, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((m2d_dwconv3x3_kernel<bf16_t, 8, true>), grid, block, 0, st, a);
  } else if (dtype == M2D_F32) {
    if (strip == 14) hipLaunchKernelGGL((m2d_dwconv3x3_kernel<float, 14>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((m2d_dwconv3x3_kernel<float, 8>), grid, block, 0, st, a);
  } else {
    if (strip == 14) hipLaunchKernelGGL((m2d_dwconv3x3_kernel<bf16_t, 14>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((m2d_dwconv3x3_kernel<bf16_t, 8>), grid, block, 0, st, a);
  }
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_dwconv3x3_fwd(int B, int H, int W, int C, int dtype, int weight_dtype, const void* x, const void* weight,
                      void* y, void* stream) {
  return run_dwconv(B, H, W, C, dtype, weight_dtype, x, weight, y, nullptr, nullptr, stream);
}

int m2d_starrelu_dwconv3x3_fwd(int B, int H, int W, int C, int weight_dtype, const void* x, const void* star_scale,
                               const void* star_bias, const void* weight, void* y, void* stream) {
  if (!star_scale || !star_bias) return M2D_ERR_NULL_POINTER;
  return run_dwconv(B, H, W, C, M2D_BF16, weight_dtype, x, weight, y, star_scale, star_bias, stream);
}

int m2d_starrelu_fwd(int64_t n, int dtype, int weight_dtype, const void* x, const void* scale, const void* bias, void* y,
                     void* stream) {
  if (!x || !scale || !bias || !y) return M2D_ERR_NULL_POINTER;
  if (n < 1) return M2D_ERR_BAD_SHAPE;
  if ((dtype != M2D_F32 && dtype != M2D_BF16) || (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;
  const int V = dtype == M2D_BF16 ? 8 : 4;
  if (n % V != 0) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(y, 16)) return M2D_ERR_MISALIGNED;
  EwArgs a = {};
  a.x = x; a.s = scale; a.b = bias; a.y = y; a.chunks = n / V; a.wbf16 = weight_dtype == M2D_BF16;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == M2D_F32) hipLaunchKernelGGL(m2d_starrelu_kernel<float>, dim3(ew_blocks(a.chunks)), dim3(kEwThreads), 0, st, a);
  else hipLaunchKernelGGL(m2d_starrelu_kernel<bf16_t>, dim3(ew_blocks(a.chunks)), dim3(kEwThreads), 0, st, a);
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_scale_residual_fwd(int64_t rows, int C, int dtype, int weight_dtype, const void* x, const void* scale,
                           const void* residual, const void* residual2, void* y, void* stream) {
  if (!x || !scale || !residual || !y) return M2D_ERR_NULL_POINTER;
  if (rows < 1 || C < 1) return M2D_ERR_BAD_SHAPE;
  if ((dtype != M2D_F32 && dtype != M2D_BF16) || (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;
  const int V = dtype == M2D_BF16 ? 8 : 4;
  if (C % V != 0) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(residual, 16) || misaligned(residual2, 16) || misaligned(y, 16) || misaligned(scale, 16))
    return M2D_ERR_MISALIGNED;
  EwArgs a = {};
  a.x = x; a.r = residual; a.r2 = residual2; a.s = scale; a.y = y; a.cpr = C / V; a.chunks = rows * a.cpr; a.wbf16 = weight_dtype == M2D_BF16;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dtype == M2D_F32) hipLaunchKernelGGL(m2d_scale_residual_kernel<float>, dim3(ew_blocks(a.chunks)), dim3(kEwThreads), 0, st, a);
  else hipLaunchKernelGGL(m2d_scale_residual_kernel<bf16_t>, dim3(ew_blocks(a.chunks)), dim3(kEwThreads), 0, st, a);
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_rope_qknorm_fwd(int B, int L, int heads, int head_dim, int dtype, int weight_dtype, const void* qkv,
                        const void* cos, const void* sin, const void* q_weight, const void* q_bias, const void* k_weight,
                        const void* k_bias, float eps, int token_major, void* q, void* k, void* stream) {
  const void* req[] = {qkv, cos, sin, q_weight, q_bias, k_weight, k_bias, q, k};
  for (const void* p : req) if (!p) return M2D_ERR_NULL_POINTER;
  if (B < 1 || L < 1 || heads < 1 || head_dim < 1) return M2D_ERR_BAD_SHAPE;
  if ((dtype != M2D_F32 && dtype != M2D_BF16) || (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;
  const int V = dtype == M2D_BF16 ? 8 : 4;
  const int G = head_dim / V;
  if (head_dim % V != 0 || (G & (G - 1)) != 0 || G > 32) return M2D_ERR_UNSUPPORTED;   // a head is 1, 2, 4 ... 32 chunks
  for (const void* p : req) if (misaligned(p, 16)) return M2D_ERR_MISALIGNED;
  RopeArgs a = {};
  a.qkv = qkv; a.cos = cos; a.sin = sin; a.qw = q_weight; a.qb = q_bias; a.kw = k_weight; a.kb = k_bias; a.q = q; a.k = k;
  a.L = L; a.heads = heads; a.hd = head_dim; a.wbf16 = weight_dtype == M2D_BF16; a.eps = eps; a.token_major = token_major != 0;
  a.total = (int64_t)B * L * 2 * heads * G;
  hipStream_t st = static_cast<hipStream_t>(stream);
  return dtype == M2D_F32 ? run_rope<float>(a, G, st) : run_rope<bf16_t>(a, G, st);
}

static int run_mlp(int64_t P, int C, int hidden, int weight_dtype, const void* x, const void* ln_weight, const void* ln_bias, float eps,
                   const void* w1, const void* b1, const void* w2, const void* b2, void* y, void* stream, const MlpArgs* res, void* z = nullptr) {
  if (!x || !w1 || !w2 || !y || (ln_weight != nullptr) != (ln_bias != nullptr)) return M2D_ERR_NULL_POINTER;
  if (P < 1 || C < 1 || hidden < 1) return M2D_ERR_BAD_SHAPE;
  if (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16) return M2D_ERR_UNSUPPORTED;
  if ((C != 32 && C != 64 && !(res && C == 128)) || hidden != 4 * C) return M2D_ERR_UNSUPPORTED;
  if ((P + 63) / 64 >= ((int64_t)1 << 31)) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(y, 16) || misaligned(w1, 16) || misaligned(w2, 16) || (b1 && misaligned(b1, 4)) || (b2 && misaligned(b2, 4)) ||
      (ln_weight && (misaligned(ln_weight, 4) || misaligned(ln_bias, 4))))
    return M2D_ERR_MISALIGNED;
  MlpArgs a = {};
  a.ln_w = ln_weight; a.ln_b = ln_bias; a.ln_eps = eps;
  a.x = x; a.w1 = w1; a.b1 = b1; a.w2 = w2; a.b2 = b2; a.y = y; a.P = P; a.wbf16 = weight_dtype == M2D_BF16;
  if (res) { a.res_s = res->res_s; a.nx_w = res->nx_w; a.nx_b = res->nx_b; a.nx_eps = res->nx_eps; a.xo = res->xo; }
  a.z = z;
  const size_t lds = (C == 128 ? mlp_lds_bytes<4>() : C == 64 ? mlp_lds_bytes<2>() : mlp_lds_bytes<1>()) + (res ? (size_t)3 * C * 4 : 0);
  if (lds > 64 * 1024 && !allow_big_lds()) return M2D_ERR_HIP;
  // persistent: the weights go to LDS once per workgroup
  const int fit = (int)(160 * 1024 / lds);
  // 64 channels: workgroups of 8 waves where they fill the device: twice the waves that share a copy of the weights (RES: 50176 positions 17.0 us, 401408
  // 82.8; of 6 waves 21.9 and 106); of 4 below, where more of them share out the rows.  32 channels: of 4 at any size, up to 8 on a unit, whose tiles of 64 rows leave
  // less of a round empty (m2d_mlp_fwd, fp32 weights, 2 workgroups of 8 waves on a unit, 4 and 8 of 4 waves: 33000 positions 7.8, 7.1 and 7.1 us, 100352 13.3,
  // 11.6 and 12.5, 300000 29.7, 28.1 and 27.9, 401408 36.5, 35.7 and 34.6; 65536 8.3, 8.6 and 8.7; RES 100352 16.0, 14.0 and 15.0, 300000 33.5, 31.5 and 31.0).
  const bool many = C == 128 || (C == 64 && P > 256 * 128);
  const int rows = many ? kMlpThreads / 4 : 64, most = many ? 2 : C == 32 ? 8 : 4, per_cu = fit < most ? fit : most;
  a.ntiles = (int)((P + rows - 1) / rows);
  int grid = 256 * per_cu;
  if (grid > a.ntiles) grid = a.ntiles;
  hipStream_t st = static_cast<hipStream_t>(stream);
  auto go = [&](auto kc, auto with, auto keep, auto threads) {
    constexpr int KC = decltype(kc)::value, TH = decltype(threads)::value;
    constexpr bool RES = decltype(with)::value, KEEP = decltype(keep)::value;
    hipLaunchKernelGGL((m2d_mlp_kernel<KC, RES, TH, KEEP>), dim3((unsigned)grid), dim3(TH), lds, st, a);
  };
  auto with = [&](auto kc, auto threads) {
    if (z) go(kc, std::false_type{}, std::true_type{}, threads);
    else if (res) go(kc, std::true_type{}, std::false_type{}, threads);
    else go(kc, std::false_type{}, std::false_type{}, threads);
  };
  constexpr std::integral_constant<int, kLinThreads> four{};
  constexpr std::integral_constant<int, kMlpThreads> eight{};
  if (C == 128) hipLaunchKernelGGL((m2d_mlp_kernel<4, true, kMlpThreads>), dim3((unsigned)grid), dim3(kMlpThreads), lds, st, a);
  else if (C == 64 && many) with(std::integral_constant<int, 2>{}, eight);
  else if (C == 64) with(std::integral_constant<int, 2>{}, four);
  else with(std::integral_constant<int, 1>{}, four);
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_mlp_fwd(int64_t P, int C, int hidden, int weight_dtype, const void* x, const void* ln_weight, const void* ln_bias, float eps,
                const void* w1, const void* b1, const void* w2, const void* b2, void* y, void* stream) {
  return run_mlp(P, C, hidden, weight_dtype, x, ln_weight, ln_bias, eps, w1, b1, w2, b2, y, stream, nullptr);
}

int m2d_mlp_keep_fwd(int64_t P, int C, int hidden, int weight_dtype, const void* x, const void* w1, const void* b1, const void* w2, const void* b2,
                     void* z, void* y, void* stream) {
  if (!z) return M2D_ERR_NULL_POINTER;
  if (misaligned(z, 16)) return M2D_ERR_MISALIGNED;
  return run_mlp(P, C, hidden, weight_dtype, x, nullptr, nullptr, 0.f, w1, b1, w2, b2, y, stream, nullptr, z);
}

int m2d_mlp_residual_layernorm_fwd(int64_t P, int C, int hidden, int weight_dtype, const void* x, const void* ln_weight, const void* ln_bias,
                                   float eps, const void* w1, const void* b1, const void* w2, const void* b2, const void* scale,
                                   const void* next_weight, const void* next_bias, float next_eps, void* x_out, void* y, void* stream) {
  if (!scale || !next_weight || !next_bias || !x_out) return M2D_ERR_NULL_POINTER;
  if (misaligned(x_out, 16) || misaligned(scale, 4) || misaligned(next_weight, 4) || misaligned(next_bias, 4)) return M2D_ERR_MISALIGNED;
  MlpArgs res = {};
  res.res_s = scale; res.nx_w = next_weight; res.nx_b = next_bias; res.nx_eps = next_eps; res.xo = x_out;
  return run_mlp(P, C, hidden, weight_dtype, x, ln_weight, ln_bias, eps, w1, b1, w2, b2, y, stream, &res);
}

int m2d_rope_attention_fwd(int B, int L, int heads, int head_dim, int weight_dtype, const void* qkv, const void* cos,
                           const void* sin, const void* q_weight, const void* q_bias, const void* k_weight,
                           const void* k_bias, float eps, float scale, void* out, void* stream) {
  if (!qkv || !cos || !sin || !q_weight || !q_bias || !k_weight || !k_bias || !out) return M2D_ERR_NULL_POINTER;
  if (B < 1 || L < 1 || heads < 1) return M2D_ERR_BAD_SHAPE;
  if (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16) return M2D_ERR_UNSUPPORTED;
  if (head_dim != kAttHd || L > kAttMaxL) return M2D_ERR_UNSUPPORTED;
  if ((int64_t)B * heads >= ((int64_t)1 << 31)) return M2D_ERR_UNSUPPORTED;
  if (misaligned(qkv, 16) || misaligned(cos, 16) || misaligned(sin, 16) || misaligned(out, 16) || misaligned(q_weight, 16) ||
      misaligned(q_bias, 16) || misaligned(k_weight, 16) || misaligned(k_bias, 16))
    return M2D_ERR_MISALIGNED;
  AttnArgs a = {};
  a.qkv = qkv; a.cos = cos; a.sin = sin; a.qw = q_weight; a.qb = q_bias; a.kw = k_weight; a.kb = k_bias; a.out = out;
  a.L = L; a.heads = heads; a.wbf16 = weight_dtype == M2D_BF16; a.eps = eps; a.scale_log2e = scale * 1.44269504088896341f;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const unsigned blocks = (unsigned)((int64_t)B * heads);
  switch ((L + 15) / 16) {
    case 1: launch_attention<1>(a, blocks, st); break;
    case 2: launch_attention<2>(a, blocks, st); break;
    case 3: launch_attention<3>(a, blocks, st); break;
    case 4: launch_attention<4>(a, blocks, st); break;
    case 5: launch_attention<5>(a, blocks, st); break;
    case 6: launch_attention<6>(a, blocks, st); break;
    case 7: launch_attention<7>(a, blocks, st); break;
    case 8: launch_attention<8>(a, blocks, st); break;
    case 9: launch_attention<9>(a, blocks, st); break;
    case 10: launch_attention<10>(a, blocks, st); break;
    case 11: launch_attention<11>(a, blocks, st); break;
    case 12: launch_attention<12>(a, blocks, st); break;
    case 13: launch_attention<13>(a, blocks, st); break;
    case 14: launch_attention<14>(a, blocks, st); break;
    case 15: launch_attention<15>(a, blocks, st); break;
    default: launch_attention<16>(a, blocks, st); break;
  }
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

static int run_linear(int64_t P, int K, int N, int weight_dtype, const void* x, const void* weight, const void* bias,
                      int pre_act, const void* pre_scale, const void* pre_bias, int post_act, const void* post_scale,
                      const void* post_bias, void* y, void* stream, const void* ln_w, const void* ln_b, float ln_eps,
                      void* z = nullptr, const LinArgs* res = nullptr) {
  if (!x || !weight || !y) return M2D_ERR_NULL_POINTER;
  const bool ln = pre_act == kActLayerNorm;
  if (ln && (!ln_w || !ln_b)) return M2D_ERR_NULL_POINTER;
  if ((pre_act == kActStarRelu && (!pre_scale || !pre_bias)) || (post_act == kActStarRelu && (!post_scale || !post_bias)))
    return M2D_ERR_NULL_POINTER;
  if (P < 1 || K < 1 || N < 1) return M2D_ERR_BAD_SHAPE;
  if (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16) return M2D_ERR_UNSUPPORTED;
  if (pre_act < kActNone || pre_act > kActLayerNorm || post_act < kActNone || post_act > kActStarRelu) return M2D_ERR_UNSUPPORTED;
  if (K % 32 != 0 || K > 32 * kLinMaxKC || N % 16 != 0) return M2D_ERR_UNSUPPORTED;
  if (ln && K > 128) return M2D_ERR_UNSUPPORTED;      // the normalised rows live in registers next to the operands
  // Slices of the outputs, so that a workgroup's share of the weights leaves room for four workgroups on a
  // compute unit (each slice reads the rows of x again; they are the smaller side where N is large).
  int nsplit = 1;
  while (linear_slice_bytes(K, N / nsplit, ln) > 40 * 1024 && (N / nsplit) % 32 == 0 && N / nsplit > 64) nsplit *= 2;
  const int Ns = N / nsplit;
  if (linear_slice_bytes(K, Ns, ln) > kLinMaxLds) return M2D_ERR_UNSUPPORTED;
  if ((P + 63) / 64 >= ((int64_t)1 << 31)) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(y, 16) || misaligned(weight, 16) || (bias && misaligned(bias, 4))) return M2D_ERR_MISALIGNED;
  if (ln && (misaligned(ln_w, 4) || misaligned(ln_b, 4))) return M2D_ERR_MISALIGNED;
  LinArgs a = {};
  a.ln_w = ln_w; a.ln_b = ln_b; a.ln_eps = ln_eps;
  a.x = x; a.w = weight; a.bias = bias; a.y = y; a.P = P; a.K = K; a.N = N; a.wbf16 = weight_dtype == M2D_BF16;
  a.pre = pre_act; a.post = post_act; a.pre_s = pre_scale; a.pre_b = pre_bias; a.post_s = post_scale; a.post_b = post_bias;
  a.ntiles = (int)((P + 63) / 64);
  a.nsplit = nsplit; a.Ns = Ns; a.z = z;
  if (res) { a.res_x = res->res_x; a.res_r = res->res_r; a.res_s = res->res_s; }
  const size_t lds = linear_lds_bytes(K, Ns, ln) + (res ? (size_t)Ns * 4 : 0);
  if (lds > 64 * 1024 && !allow_big_lds()) return M2D_ERR_HIP;
  // persistent: the weights are loaded into LDS once per workgroup; as many workgroups as fit the device at once
  int per_cu = (int)(160 * 1024 / lds);
  const int most = lin_per_cu(K <= 64 ? 2 : K <= 128 ? 4 : K <= 256 ? 8 : 16, res != nullptr);
  if (per_cu > most) per_cu = most;
  int grid = 256 * per_cu / nsplit;     // workgroups per slice
  grid = grid / 8 * 8;
  if (grid > a.ntiles) grid = (a.ntiles + 7) / 8 * 8;
  if (grid < 8) grid = 8;
  grid *= nsplit;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 g((unsigned)grid), t(kLinThreads);
  if (res && K <= 64) hipLaunchKernelGGL((m2d_linear_kernel<2, true>), g, t, lds, st, a);
  else if (res) hipLaunchKernelGGL((m2d_linear_kernel<4, true>), g, t, lds, st, a);
  else if (K <= 64) hipLaunchKernelGGL(m2d_linear_kernel<2>, g, t, lds, st, a);
  else if (K <= 128) hipLaunchKernelGGL(m2d_linear_kernel<4>, g, t, lds, st, a);
  else if (K <= 256) hipLaunchKernelGGL(m2d_linear_kernel<8>, g, t, lds, st, a);
  else hipLaunchKernelGGL(m2d_linear_kernel<16>, g, t, lds, st, a);
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_linear_fwd(int64_t P, int K, int N, int weight_dtype, const void* x, const void* weight, const void* bias,
                   int pre_act, const void* pre_scale, const void* pre_bias, int post_act, const void* post_scale,
                   const void* post_bias, void* y, void* stream) {
  if (pre_act == kActLayerNorm) return M2D_ERR_UNSUPPORTED;      // that one has an entry point of its own
  return run_linear(P, K, N, weight_dtype, x, weight, bias, pre_act, pre_scale, pre_bias, post_act, post_scale, post_bias, y, stream,
                    nullptr, nullptr, 0.f);
}

int m2d_linear_residual_fwd(int64_t P, int K, int N, int weight_dtype, const void* x, const void* weight, const void* bias, int pre_act,
                            const void* residual, const void* scale, const void* residual2, void* y, void* stream) {
  if (!residual || !scale) return M2D_ERR_NULL_POINTER;
  if (pre_act != kActNone && pre_act != kActGelu) return M2D_ERR_UNSUPPORTED;
  if (K > 128 || N > (K <= 64 ? 64 : 128)) return M2D_ERR_UNSUPPORTED;      // the stream's pieces of a row are held in registers
  if (misaligned(residual, 16) || misaligned(residual2, 16) || misaligned(scale, 4)) return M2D_ERR_MISALIGNED;
  LinArgs res = {};
  res.res_x = residual; res.res_r = residual2; res.res_s = scale;
  return run_linear(P, K, N, weight_dtype, x, weight, bias, pre_act, nullptr, nullptr, kActNone, nullptr, nullptr, y, stream, nullptr, nullptr,
                    0.f, nullptr, &res);
}

int m2d_wide_linear_fwd(int64_t P, int K, int N, int weight_dtype, const void* x, const void* weight, const void* bias, int post_act,
                        void* y, void* stream) {
  if (!x || !weight || !y) return M2D_ERR_NULL_POINTER;
  if (P < 1 || K < 1 || N < 1) return M2D_ERR_BAD_SHAPE;
  if (weight_dtype != M2D_F32 && weight_dtype != M2D_BF16) return M2D_ERR_UNSUPPORTED;
  if (K % 32 != 0 || N % 32 != 0 || P > ((int64_t)1 << 20) || (post_act != kActNone && post_act != kActGelu)) return M2D_ERR_UNSUPPORTED;
  if (misaligned(x, 16) || misaligned(weight, 16) || misaligned(y, 16) || misaligned(bias, 16)) return M2D_ERR_MISALIGNED;
  if (post_act == kActGelu && weight_dtype == M2D_BF16 && P > kGlFewest && K <= kGlInputs && N % 64 == 0) {
    GeluLinArgs a = {static_cast<const uint16_t*>(x), static_cast<const uint16_t*>(weight), static_cast<const uint16_t*>(bias),
                     static_cast<uint16_t*>(y), P, K, N, 1, 0, 0, 0};
    hipStream_t st = static_cast<hipStream_t>(stream);
    const int64_t tiles = (P + kGlRows - 1) / kGlRows;
    // Slices of whole 64-output steps.  A compute unit is done when the one with the most workgroups is: an eighth of them goes to
    // each XCD, to its 32 units evenly, and one workgroup on a unit takes as long as two (chains of loads and products).  A workgroup's
    // start is worth half a unit of 32 outputs.  More slices have to save a twenty-fifth: where they come out about even, fewer are faster, as outputs
    // beyond the last-level cache then leave in longer rows (150000 positions, 320 -> 1024: 1 slice 181 us, 4 slices 212, which cost 1 in 160
    // less by this rule).  Of all numbers of slices, measured for 392 sizes (600 to 250000 positions, 64 to 1280 outputs, 64 to 320 inputs),
    // the one chosen takes 1.005 of the fastest's time, 1.16 at most (100000 positions, 320 -> 448); the fewest with 768 workgroups 1.04 of the chosen one's.
    int64_t least = 0;
    for (int d = 1; d <= N / 64 && (d == 1 || tiles * d <= kGlMost); ++d) {
      const int64_t on_unit = ((tiles * d + 7) / 8 + 31) / 32, cost = (on_unit < 2 ? 2 : on_unit) * (4 * ((N / 64 + d - 1) / d) + 1);
      if (d == 1 || 25 * cost < 24 * least) { least = cost; a.nsplit = d; }
    }
    a.steps = N / 64 / a.nsplit;
    a.over = N / 64 % a.nsplit;
    a.per_slice = a.nsplit == 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + a.nsplit - 1) / a.nsplit);
    const dim3 g((unsigned)((tiles * a.nsplit + 7) / 8 * 8)), t(kGlThreads);
    if (K <= 256) hipLaunchKernelGGL(m2d_gelu_linear_kernel<16>, g, t, 0, st, a);
    else hipLaunchKernelGGL(m2d_gelu_linear_kernel<20>, g, t, 0, st, a);
    return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
  }
  WideArgs a = {static_cast<const uint16_t*>(x), weight, bias, static_cast<uint16_t*>(y), (int)P, K, N, post_act};
  const unsigned mt = (unsigned)((P + 31) / 32);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const bool narrow = (int64_t)mt * (N / 32) < 128;      // few workgroups: 16 outputs each instead of 32
  const dim3 g((unsigned)(narrow ? N / 16 : N / 32), mt), t(64 * kWideWaves);
  auto go = [&](auto wb) {
    constexpr bool WB = decltype(wb)::value;
    if (narrow) hipLaunchKernelGGL((m2d_wide_linear_kernel<1, WB>), g, t, 0, st, a);
    else hipLaunchKernelGGL((m2d_wide_linear_kernel<2, WB>), g, t, 0, st, a);
  };
  if (weight_dtype == M2D_BF16) go(std::true_type{});
  else go(std::false_type{});
  return hipGetLastError() == hipSuccess ? M2D_OK : M2D_ERR_HIP;
}

int m2d_linear_keep_fwd(int64_t P, int K, int N, int weight_dtype, const void* x, const void* weight, const void* bias,
                        int post_act, const void* post_scale, const void* post_bias, void* z, void* y, void* stream) {
  if (!z) return M2D_ERR_NULL_POINTER;
  if (misaligned(z, 16)) return M2D_ERR_MISALIGNED;
  return run_linear(P, K, N, weight_dtype, x, weight, bias, kActNone, nullptr, nullptr, post_act, post_scale, post_bias, y, stream,
                    nullptr, nullptr, 0.f, z);
}

int m2d_layernorm_linear_fwd(int64_t P, int K, int N, int weight_dtype, const void* x, const void* ln_weight, const void* ln_bias,
                             float eps, const void* weight, const void* bias, int post_act, const void* post_scale,
                             const void* post_bias, void* y, void* stream) {
  return run_linear(P, K, N, weight_dtype, x, weight, bias, kActLayerNorm, nullptr, nullptr, post_act, post_scale, post_bias, y, stream,
                    ln_weight, ln_bias, eps);
}

}  // extern "C"
