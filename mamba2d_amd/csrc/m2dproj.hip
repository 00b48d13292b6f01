// Projections either side of the 2-D selective scan, for gfx950.
//
// The reference derives the scan's parameters from x with three library GEMMs and a softplus
// (proj_params, models/kernels/wavefront_cuda.py:63-95) and leaves their backward to autograd
// (wavefront_cuda.py:262-296).  The products are skinny -- the inner dimensions are d_model,
// dt_rank and 2*dt_rank + 3*d_state -- and the weight gradients reduce over every position of
// the batch, which general GEMM libraries handle poorly.  Here each pass is a few kernels that
// walk the (position, channel) arrays once, a tile of 64 positions at a time:
//
//   forward   z = x Wx^T ;  [rT | rL | B_T | B_L | C] = z ;  delta = softplus(r w^T + b)
//   backward  dpre = d_delta * (1 - exp(-delta))            (softplus'(pre) = 1 - exp(-softplus(pre)))
//             dz = [dpreT wT | dpreL wL | dB_T | dB_L | dC] ;  dx += dz Wx
//             dWx = dz^T x ;  dw = dpre^T r ;  db = sum dpre      (sums over all positions)
//
// The products run on the matrix cores: bf16 tensors whose rows are whole 16-byte chunks through bf16 operands, all
// others through fp32 ones; sums are fp32 in both.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "m2dscan.h"

namespace {

constexpr int kN = 16;        // d_state the scan is built for
constexpr int kTP = 64;       // positions per tile (one per lane)
constexpr int kKC = 64;       // channels per chunk of the inner dimension
constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxR = 32;     // largest dt_rank

struct bf16_t { uint16_t v; };

__device__ __forceinline__ float ld(const float* p) { return *p; }
__device__ __forceinline__ float ld(const bf16_t* p) { return __uint_as_float((uint32_t)p->v << 16); }
// round to nearest even; the conversion is one instruction on gfx950 (v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16_pair(float lo, float hi) {   // one v_cvt_pk_bf16_f32
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ void st(float* p, float v) { *p = v; }
__device__ __forceinline__ void st(bf16_t* p, float v) { p->v = f32_to_bf16_bits(v); }
// the value a tensor of type T would hold
__device__ __forceinline__ float as_stored(float v, const float*) { return v; }
__device__ __forceinline__ float as_stored(float v, const bf16_t*) { return __uint_as_float((uint32_t)f32_to_bf16_bits(v) << 16); }

// exp and log as the bare hardware instructions: the arguments below stay in ranges that
// need none of the library's scaling (results that underflow may flush to zero).
__device__ __forceinline__ float exp_neg(float v) { return __builtin_amdgcn_exp2f(v * 1.44269504088896341f); }   // v <= 0

// softplus with torch's defaults (beta 1; above the threshold of 20 the two agree in fp32):
// max(v,0) + log1p(t), t = exp(-|v|), with log1p(t) = log(u) + (t - (u-1)) for u = fl(1+t): the
// second term makes up for the rounding of 1+t when t is small.  (Exactly it would be divided by u;
// it is at most half an ulp of u, 6e-8, and u lies in [1, 2], so leaving the division out changes
// the result by less than 6e-8 t.)
__device__ __forceinline__ float softplus(float v) {
  const float t = exp_neg(-fabsf(v));
  const float u = 1.f + t;
  return fmaxf(v, 0.f) + __builtin_fmaf(__builtin_amdgcn_logf(u), 0.693147180559945309f, t - (u - 1.f));
}
// d softplus / d pre, from the softplus value: sigmoid(pre) = 1 - exp(-softplus(pre)).  Small
// arguments take the series, where 1 - exp(-d) would cancel.
__device__ __forceinline__ float softplus_slope(float d) {
  const float series = d * __builtin_fmaf(d, __builtin_fmaf(d, __builtin_fmaf(d, -1.f / 24.f, 1.f / 6.f), -0.5f), 1.f);
  return d < 0.0625f ? series : 1.f - exp_neg(-d);
}

// Where the scan kernels expect value n (0..47: B_T, B_L, C, 16 states each) inside a position's
// record of 48 floats: the four states n = 4q + m, q = 0..3, that the scan's backward folds together
// share a float4, in the order q = 0, 2, 1, 3 (the scan source calls this the fold order).
__device__ __forceinline__ int record_slot(int n48) {
  const int n = n48 & 15, q = n >> 2, m = n & 3;
  return (n48 & ~15) + 4 * m + (q == 1 ? 2 : (q == 2 ? 1 : q));
}

struct ProjArgs {
  // activations, (P, .) row-major, element type T
  const void *x, *r, *dT, *dL;           // x (P,E); r (P,2R) = low-rank inputs of the two dt projections; delta (P,E)
  const void *ddT, *ddL, *dBT, *dBL, *dC;
  int dpre_given;                        // ddT, ddL hold the gradients before the softplus already (dT, dL are not read)
  int sum_parts;                         // > 0: dBT points to that many fp32 records [P][dC | dBT | dBL][16] to add up (the scan's per-workgroup sums)
  void *r_out, *dT_out, *dL_out, *BT_out, *BL_out, *C_out, *dx;
  float* bc_packed;                      // (P,48) fp32 records for the scan kernels instead of BT_out, BL_out, C_out (or null)
  const float *Wx, *wT, *bT, *wL, *bL;   // the weights as the caller holds them (for the fp32 products)
  int round;                             // ... to be rounded to bf16 by the kernels that read them
  const float *bTp, *bLp;                // [Epad] packed biases, fp32, zero where padded
  // packed weights for the bf16 products, zero where padded
  const uint16_t *Wb;                    // [Opad][Epad]   Wx
  const uint16_t *wTb, *wLb;             // [Epad][32]     dt weights
  const uint16_t *wTtb, *wLtb;           // [Rpad][Epad]   dt weights transposed
  const uint16_t *WxTb;                  // [Epad][Opad32] Wx transposed
  float* dz;                             // (P,Opad) fp32, padding behind the low-rank part (o' order)
  // the same for the bf16 products
  uint16_t* dzt;                         // (P16, Opad)    dz, P16 = positions rounded up to 16
  uint16_t* dpt;                         // [2](P16, E)    dpreT, dpreL
  float* part;                           // per-workgroup sums of the weight gradients
  float *dWx, *dwT, *dbT, *dwL, *dbL;    // outputs of the reduction
  int64_t P;
  int E, R, O, Epad, Opad, Opad32, Rpad;
  int ntiles, G, ne;
};

__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// ------------------------------------------------------------------------------- weights
struct PackArgs {
  const float *Wx, *wT, *bT, *wL, *bL;
  float *bTp, *bLp;                      // forward set (or null)
  uint16_t *Wb, *wTb, *wLb;
  uint16_t *wTtb, *wLtb, *WxTb;          // backward set (or null)
  int E, R, O, Epad, Opad, Opad32, Rpad;
  int round;                             // round the biases to bf16 first (the bf16 copies are rounded anyway)
};

// Padded copies of the weights for the bf16 products.  One thread per element of the largest copy.
__global__ void m2d_proj_pack_kernel(const PackArgs k) {
  // a bias as the kernels are to see it
  auto w = [&](const float* p, int i) { return k.round ? as_stored(p[i], static_cast<const bf16_t*>(nullptr)) : p[i]; };
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (k.bTp && i < k.Epad) {
    k.bTp[i] = i < k.E ? w(k.bT, i) : 0.f;
    k.bLp[i] = i < k.E ? w(k.bL, i) : 0.f;
  }
  if (k.Wb) {
    if (i < k.Opad * k.Epad) {
      const int o = i / k.Epad, e = i - o * k.Epad;
      k.Wb[i] = (o < k.O && e < k.E) ? f32_to_bf16_bits(k.Wx[o * k.E + e]) : 0;
    }
    if (i < k.Epad * 32) {
      const int e = i >> 5, q = i & 31;
      const bool ok = e < k.E && q < k.R;
      k.wTb[i] = ok ? f32_to_bf16_bits(k.wT[e * k.R + q]) : 0;
      k.wLb[i] = ok ? f32_to_bf16_bits(k.wL[e * k.R + q]) : 0;
    }
  }
  if (k.WxTb) {
    if (i < k.Epad * k.Opad32) {
      const int e = i / k.Opad32, o = i - e * k.Opad32;
      k.WxTb[i] = (o < k.O && e < k.E) ? f32_to_bf16_bits(k.Wx[o * k.E + e]) : 0;
    }
    if (i < k.Rpad * k.Epad) {
      const int q = i / k.Epad, e = i - q * k.Epad;
      const bool ok = e < k.E && q < k.R;
      k.wTtb[i] = ok ? f32_to_bf16_bits(k.wT[e * k.R + q]) : 0;
      k.wLtb[i] = ok ? f32_to_bf16_bits(k.wL[e * k.R + q]) : 0;
    }
  }
}

// ------------------------------------------------------------------------------- matrix cores
// bf16 tensors whose rows start on 16-byte boundaries take the products through
// v_mfma_f32_16x16x32_bf16.  A wave owns 16 positions and needs nothing from the other waves of
// its workgroup.  Operand layout of the instruction (lane l, m = n = l & 15, kb = l >> 4):
//   A[m][8 kb + j], B[8 kb + j][n] (j < 8, one 16-byte register set each);  D[4 kb + i][n], i < 4.
// With positions as rows of A, the 8 values a lane needs are 8 consecutive channels of one
// position: one 16-byte load straight from the (P,E) array.  The weights are packed so that the
// same holds for B.
#ifndef M2D_PROJ_OCC
#define M2D_PROJ_OCC 5
#endif
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int kMaxNT = (2 * kMaxR + 3 * kN + 15) / 16;   // 16-wide tiles of the 2R+48 outputs
constexpr int kLowStride = 40;   // bf16 per row of the low-rank scratch: 32 + 8, rows 16-byte aligned and spread over the banks

__device__ __forceinline__ f32x4 mfma16(uint4 a, uint4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// written out at every use: as a named constant the register allocator has kept it in scratch memory
__device__ __forceinline__ uint4 zero16() { return make_uint4(0u, 0u, 0u, 0u); }
__device__ __forceinline__ uint4 load16(const void* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}

// Results leave the accumulators (4 positions x 1 channel per lane and tile) through a per-wave
// LDS block of 16 positions x 64 channels, so that memory sees 16-byte pieces of rows.
constexpr int kStageStride = 72;   // floats per row: 64 + 8, rows 16-byte aligned (also holds 2 x [16][72] bf16)
__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ __forceinline__ void stage_put(float* stage, int nt, int mn, int kb, f32x4 v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) stage[(4 * kb + i) * kStageStride + 16 * nt + mn] = v[i];
}
// f(position, first channel, 8 values) for the lane's two pieces of the block
template <typename F>
__device__ __forceinline__ void stage_rows(const float* stage, int l, F f) {
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int piece = l + 64 * k, c = piece >> 3, c8 = 8 * (piece & 7);
    const float4 lo = *reinterpret_cast<const float4*>(stage + c * kStageStride + c8);
    const float4 hi = *reinterpret_cast<const float4*>(stage + c * kStageStride + c8 + 4);
    const float v[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    f(c, c8, v);
  }
}
__device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
  return make_uint4(pack2(v[0], v[1]), pack2(v[2], v[3]), pack2(v[4], v[5]), pack2(v[6], v[7]));
}

// Forward.  LDS: per wave two [16][40] bf16 blocks (low-rank inputs of the T and L projection)
// and the [16][68] fp32 block the delta tiles leave through.
__global__ __launch_bounds__(kThreads, M2D_PROJ_OCC) void m2d_proj_fwd_mfma_kernel(const ProjArgs a) {
  extern __shared__ float smem[];
  const int wave = wave_id(), l = threadIdx.x & 63, mn = l & 15, kb = l >> 4;
  float* stage = smem + wave * (16 * kStageStride + 16 * kLowStride);   // [16][68] floats, then 2 x [16][40] bf16
  uint16_t* lowT = reinterpret_cast<uint16_t*>(stage + 16 * kStageStride);
  uint16_t* lowL = lowT + 16 * kLowStride;
  // columns past the rank meet zero weights; they only have to be finite
  for (int i = l; i < 16 * kLowStride; i += 64) reinterpret_cast<uint32_t*>(lowT)[i] = 0u;
  const int64_t p0 = (int64_t)blockIdx.x * kTP + wave * 16;
  const bf16_t* x = static_cast<const bf16_t*>(a.x);
  const int64_t pm = p0 + mn;
  const int NT = a.Opad / 16, R = a.R, R2 = 2 * a.R;

  f32x4 acc[kMaxNT];
#pragma unroll
  for (int nt = 0; nt < kMaxNT; ++nt) acc[nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int e = 8 * kb; e < a.Epad; e += 32) {
    const uint4 A = (pm < a.P && e < a.E) ? load16(x + pm * a.E + e) : make_uint4(0, 0, 0, 0);
#pragma unroll
    for (int nt = 0; nt < kMaxNT; ++nt)
      if (nt < NT) acc[nt] = mfma16(A, load16(a.Wb + (16 * nt + mn) * a.Epad + e), acc[nt]);
  }

  // z[position 4 kb + i][output 16 nt + mn]: low-rank inputs, B_T, B_L, C.  Addresses are a
  // wave-uniform base (the wave's first position) plus a 32-bit element offset.
  const int rows = (int)(a.P - p0 < 16 ? a.P - p0 : 16);   // positions of the wave inside the array (may be <= 0)
  bf16_t* r_out = static_cast<bf16_t*>(a.r_out) + p0 * R2;
  bf16_t* bt_out = static_cast<bf16_t*>(a.BT_out) + p0 * kN;
  bf16_t* bl_out = static_cast<bf16_t*>(a.BL_out) + p0 * kN;
  bf16_t* c_out = static_cast<bf16_t*>(a.C_out) + p0 * kN;
#pragma unroll
  for (int nt = 0; nt < kMaxNT; ++nt) {
    if (nt >= NT) break;
    const int o = 16 * nt + mn;
    const int oo = o - R2;
    bf16_t* bc = (oo < kN ? bt_out : (oo < 2 * kN ? bl_out : c_out)) + (oo & (kN - 1));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = 4 * kb + i;
      const uint16_t h = f32_to_bf16_bits(acc[nt][i]);
      if (o < R) lowT[c * kLowStride + o] = h;
      else if (o < R2) lowL[c * kLowStride + o - R] = h;
      if (c < rows) {
        if (o < R2) r_out[(uint32_t)(c * R2 + o)].v = h;
        else if (o < a.O) {
          if (a.bc_packed) a.bc_packed[(p0 + c) * (3 * kN) + record_slot(oo)] = bf16_lo(h);
          else bc[(uint32_t)(c * kN)].v = h;
        }
      }
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  // delta = softplus(low w^T + b): the rank is the inner dimension (one step of 32)
  const uint4 AT = load16(lowT + mn * kLowStride + 8 * kb), AL = load16(lowL + mn * kLowStride + 8 * kb);
  bf16_t* dT_out = static_cast<bf16_t*>(a.dT_out) + p0 * a.E;
  bf16_t* dL_out = static_cast<bf16_t*>(a.dL_out) + p0 * a.E;
  for (int e0 = 0; e0 < a.Epad; e0 += kKC) {
    f32x4 sT[4], sL[4];
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int e = e0 + 16 * nt + mn;
      const float bT = a.bTp[e], bL = a.bLp[e];
      sT[nt] = mfma16(AT, load16(a.wTb + e * 32 + 8 * kb), (f32x4){bT, bT, bT, bT});
      sL[nt] = mfma16(AL, load16(a.wLb + e * 32 + 8 * kb), (f32x4){bL, bL, bL, bL});
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const f32x4 v = h ? sL[nt] : sT[nt];
        stage_put(stage, nt, mn, kb, (f32x4){softplus(v[0]), softplus(v[1]), softplus(v[2]), softplus(v[3])});
      }
      wave_sync_lds();
      bf16_t* out = h ? dL_out : dT_out;
      stage_rows(stage, l, [&](int c, int c8, const float (&v)[8]) {
        if (c < rows && e0 + c8 < a.E) *reinterpret_cast<uint4*>(out + (uint32_t)(c * a.E + e0 + c8)) = pack8(v);
      });
      wave_sync_lds();
    }
  }
}

// Forward for up to 256 channels and a rank of up to 16.  The kernel above, left with the wider ones (whose weights fill the LDS, and whose low-rank
// inputs don't fit one step of 32), is bound by its weight tiles: every wave of 16 positions fetches all of them, 14 KB for 2 KB of x at 64 channels,
// from the caches.  Here a workgroup stays for many tiles and holds the weights in LDS, rounded to bf16 as it
// reads them from the caller's tensors (no packing launch), and the weights' rows are the first operands, so that a lane (position mn, group kb) ends with
// neighbouring outputs of its position and stores them from registers: 4 of a record of B_T, B_L, C, whose rows are listed in the records' order, and 8
// step sizes, for which a pair of tiles lists its rows as 8 (m >> 2) + 4 t + (m & 3).  The low-rank inputs of the step sizes stay in the registers
// that they were made in: the second product lists its contraction in their order, and those of the other step size are masked out, so that
// an infinite value of one does not meet the other's zero weights.  With a rank above 4 a step size's fp32 sum is thereby formed in another order than in
// the kernel above, of the same operands: it may round to the neighbouring bf16 value.  Against the kernel above
// and its packing launch, ten calls in a row: 64x56x56x64 43.1 -> 24.7 us (104 MB, 4.2 TB/s), 4x128x128x64 19.6 -> 11.8, 64x28x28x128 28.2 -> 18.4,
// 64x14x14x256 27.0 -> 18.6, 200000 positions of 32 channels 39.2 -> 16.6, 4096 of 64 11.1 -> 5.2; no size measured was slower.  A thread's share of the
// weights is asked for at once: with loops that waited for each load they were 28.8, 13.4, 22.7, 24.4, 18.3 and 7.2.  What is left at 64 channels is
// the copying in of the weights and the softplus.
constexpr int kFlD = 40;      // bf16 per row of the step sizes' weights in LDS: 32 + 8
constexpr int kFlMaxE = 256, kFlMaxR = 16;
constexpr int kUnits = 256;   // compute units of an MI355X
constexpr size_t fl_lds_bytes(int Epad, int NL) { return ((size_t)(16 * NL + 3 * kN) * (Epad + 8) + 2 * (size_t)Epad * kFlD) * 2 + 2 * (size_t)Epad * 4; }
__device__ __forceinline__ f32x4 load_f4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }

template <int KS, int NL, bool PACKED>   // steps of 32 channels at most; tiles of 16 low-rank inputs
__global__ __launch_bounds__(kThreads) void m2d_proj_fwd_lds_kernel(const ProjArgs a) {
  extern __shared__ float smem[];
  const int tid = threadIdx.x, wave = wave_id(), l = tid & 63, mn = l & 15, kb = l >> 4;
  constexpr int NZ = 16 * NL + 3 * kN;
  const int E = a.E, Epad = (E + 31) / 32 * 32, ks = Epad / 32, R = a.R, R2 = 2 * a.R, LW = Epad + 8;
  uint16_t* wz = reinterpret_cast<uint16_t*>(smem);
  uint16_t* wT = wz + NZ * LW;
  uint16_t* wL = wT + Epad * kFlD;
  float* bT = reinterpret_cast<float*>(wL + Epad * kFlD);
  float* bL = bT + Epad;
  const bf16_t* x = static_cast<const bf16_t*>(a.x);
  const int ntiles = (int)((a.P + kTP - 1) / kTP);
  uint4 next[KS];
  auto fetch = [&](int tile) {
    const int64_t pm = (int64_t)tile * kTP + wave * 16 + mn;
    const bf16_t* row = x + (pm < a.P ? pm : a.P - 1) * E;      // rows past the end repeat the last one and are not stored
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const int e = 32 * s + 8 * kb;
      next[s] = load16(row + (e < E ? e : 0));                  // (channels past E meet zero weights, but must be finite: masked below)
    }
  };
  // All of the workgroup's loads go out before the first wait: the weights, a thread's share unrolled, then its first rows of x.
  constexpr int kPieces = (NZ * 8 * KS + kThreads - 1) / kThreads, kDt = 2 * KS;
  const int nz = NZ * (Epad / 4), ndt = E * R;
  f32x4 hz[kPieces];
  float hT[kDt], hL[kDt];
#pragma unroll
  for (int u = 0; u < kPieces; ++u) {
    const int i = tid + u * kThreads, row = i / (Epad / 4), c = 4 * (i - row * (Epad / 4)), t = row >> 4, m = row & 15;
    const int q = m & 3, state = PACKED ? 4 * (q == 1 ? 2 : (q == 2 ? 1 : q)) + (m >> 2) : m;
    const int o = t < NL ? row : R2 + 16 * (t - NL) + state;
    const bool ok = i < nz && c < E && (t >= NL || o < R2);
    hz[u] = load_f4(a.Wx + (ok ? o * E + c : 0));
    if (!ok) hz[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int u = 0; u < kDt; ++u) {
    const int i = tid + u * kThreads;
    hT[u] = a.wT[i < ndt ? i : 0];
    hL[u] = a.wL[i < ndt ? i : 0];
  }
  const float hbT = a.bT[tid < E ? tid : 0], hbL = a.bL[tid < E ? tid : 0];   // (E <= the threads of a workgroup)
  fetch(blockIdx.x);
  for (int i = tid; i < 2 * Epad * kFlD / 8; i += kThreads) reinterpret_cast<uint4*>(wT)[i] = zero16();   // (wL follows)
  if (tid < Epad) {
    bT[tid] = tid >= E ? 0.f : (a.round ? as_stored(hbT, static_cast<const bf16_t*>(nullptr)) : hbT);
    bL[tid] = tid >= E ? 0.f : (a.round ? as_stored(hbL, static_cast<const bf16_t*>(nullptr)) : hbL);
  }
#pragma unroll
  for (int u = 0; u < kPieces; ++u) {
    const int i = tid + u * kThreads, row = i / (Epad / 4), c = 4 * (i - row * (Epad / 4));
    if (i < nz) *reinterpret_cast<uint2*>(wz + row * LW + c) = make_uint2(pack2(hz[u][0], hz[u][1]), pack2(hz[u][2], hz[u][3]));
  }
  __syncthreads();
  auto slot_of = [](int o) { return 8 * ((o & 15) >> 2) + (o & 3) + (o < 16 ? 0 : 4); };   // of low-rank input o in the second product
#pragma unroll
  for (int u = 0; u < kDt; ++u) {
    const int i = tid + u * kThreads, e = i / R, q = i - e * R;
    if (i < ndt) {
      wT[e * kFlD + slot_of(q)] = f32_to_bf16_bits(hT[u]);
      wL[e * kFlD + slot_of(q + R)] = f32_to_bf16_bits(hL[u]);
    }
  }
  // which of the lane's low-rank inputs are the T step size's, which the L one's
  uint32_t mT[2 * NL], mL[2 * NL];
#pragma unroll
  for (int w = 0; w < 2 * NL; ++w) {
    const int o = 16 * (w >> 1) + 4 * kb + 2 * (w & 1);
    mT[w] = (o < R ? 0xffffu : 0u) | (o + 1 < R ? 0xffff0000u : 0u);
    mL[w] = (o >= R && o < R2 ? 0xffffu : 0u) | (o + 1 >= R && o + 1 < R2 ? 0xffff0000u : 0u);
  }
  __syncthreads();
  for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t pm = (int64_t)tile * kTP + wave * 16 + mn;
    const bool in = pm < a.P;
    uint4 X[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) X[s] = 32 * s + 8 * kb < E ? next[s] : zero16();
    if (tile + (int)gridDim.x < ntiles) fetch(tile + gridDim.x);
    uint2 z[NL + 3];
#pragma unroll
    for (int t = 0; t < NL + 3; ++t) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
        if (s < ks) acc = mfma16(load16(wz + (16 * t + mn) * LW + 32 * s + 8 * kb), X[s], acc);
      z[t] = make_uint2(pack2(acc[0], acc[1]), pack2(acc[2], acc[3]));
    }
    if (in) {
      bf16_t* r = static_cast<bf16_t*>(a.r_out) + pm * R2;
#pragma unroll
      for (int t = 0; t < NL; ++t) {
        const int o = 16 * t + 4 * kb;
        if ((R2 & 3) == 0) {      // (uniform)
          if (o < R2) *reinterpret_cast<uint2*>(r + o) = z[t];
        } else {
          const uint32_t w[2] = {z[t].x, z[t].y};
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (o + i < R2) r[o + i].v = (uint16_t)(w[i >> 1] >> (16 * (i & 1)));
        }
      }
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        const uint2 q = z[NL + w];
        if constexpr (PACKED) {
          *reinterpret_cast<float4*>(a.bc_packed + pm * (3 * kN) + w * kN + 4 * kb) = make_float4(bf16_lo(q.x), bf16_hi(q.x), bf16_lo(q.y), bf16_hi(q.y));
        } else {
          *reinterpret_cast<uint2*>(static_cast<bf16_t*>(w == 0 ? a.BT_out : (w == 1 ? a.BL_out : a.C_out)) + pm * kN + 4 * kb) = q;
        }
      }
    }
    const uint4 lowT = make_uint4(z[0].x & mT[0], z[0].y & mT[1], NL > 1 ? z[NL - 1].x & mT[2 * NL - 2] : 0u, NL > 1 ? z[NL - 1].y & mT[2 * NL - 1] : 0u);
    const uint4 lowL = make_uint4(z[0].x & mL[0], z[0].y & mL[1], NL > 1 ? z[NL - 1].x & mL[2 * NL - 2] : 0u, NL > 1 ? z[NL - 1].y & mL[2 * NL - 1] : 0u);
    for (int e0 = 0; e0 < E; e0 += 32) {
      const int e = e0 + 8 * kb, row = e0 + 8 * (mn >> 2) + (mn & 3);
      uint4 out[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float v[8];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x4 d = mfma16(load16((h ? wL : wT) + (row + 4 * t) * kFlD + 8 * kb), h ? lowL : lowT, load_f4((h ? bL : bT) + e + 4 * t));
#pragma unroll
          for (int i = 0; i < 4; ++i) v[4 * t + i] = softplus(d[i]);
        }
        out[h] = pack8(v);
      }
      if (in && e < E) {
        *reinterpret_cast<uint4*>(static_cast<bf16_t*>(a.dT_out) + pm * E + e) = out[0];
        *reinterpret_cast<uint4*>(static_cast<bf16_t*>(a.dL_out) + pm * E + e) = out[1];
      }
    }
  }
}

// The gradients of B_T, B_L, C of a wave's positions, four values of position p0 + cb from n0 on: the caller's arrays, or
// (sum_parts > 0) the scan's per-workgroup channel sums, added up here in their order and rounded once.
__device__ __forceinline__ void sum_channels(const ProjArgs& a, int64_t p0, int rows, int cb, int n0, uint2 (&bc)[3]) {
  if (a.sum_parts > 0) {   // (uniform)
    // Twelve loads are under way at a time: with one (a loop over the parts for each of the three sums) a wave of 16
    // positions waited for memory 3 x parts times in a row: 70 -> 43 us for 4x128x128x64 (8 parts), 79 -> 60 for
    // 64x56x56x64 (4 parts; 283 MB, 4.7 TB/s).
    const float* rec = static_cast<const float*>(a.dBT) + (p0 + (cb < rows ? cb : 0)) * (3 * kN) + n0;
    const int64_t step = a.P * (3 * kN);
    float4 sum[3];
    const bool in = cb < rows;
#pragma unroll
    for (int v = 0; v < 3; ++v) sum[v] = in ? *reinterpret_cast<const float4*>(rec + v * kN) : make_float4(0.f, 0.f, 0.f, 0.f);
    auto add = [](float4& t, const float4& o) { t.x += o.x; t.y += o.y; t.z += o.z; t.w += o.w; };
    if (in) {
      int g = 1;
      for (; g + 4 <= a.sum_parts; g += 4) {
        float4 o[4][3];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < 3; ++v) o[u][v] = *reinterpret_cast<const float4*>(rec + (g + u) * step + v * kN);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int v = 0; v < 3; ++v) add(sum[v], o[u][v]);
      }
      // (the last one to three: their loads go out together too)
      float4 o[3][3];
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (g + u < a.sum_parts)
#pragma unroll
          for (int v = 0; v < 3; ++v) o[u][v] = *reinterpret_cast<const float4*>(rec + (g + u) * step + v * kN);
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (g + u < a.sum_parts)
#pragma unroll
          for (int v = 0; v < 3; ++v) add(sum[v], o[u][v]);
    }
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      const float4 t = sum[w == 0 ? 1 : (w == 1 ? 2 : 0)];   // the records hold dC, dBT, dBL in this order
      bc[w] = make_uint2(pack2(t.x, t.y), pack2(t.z, t.w));
    }
  } else {
#pragma unroll
    for (int w = 0; w < 3; ++w) {
      const bf16_t* src = static_cast<const bf16_t*>(w == 0 ? a.dBT : (w == 1 ? a.dBL : a.dC)) + p0 * kN;
      bc[w] = cb < rows ? *reinterpret_cast<const uint2*>(src + (uint32_t)(cb * kN + n0)) : make_uint2(0, 0);
    }
  }
}

// Backward, data.  LDS: per wave one [16][Opad32 + 8] bf16 block (the rows of dz) and the [16][68]
// fp32 block the dx tiles leave through.  dz and dpre are also written out as bf16 arrays for the
// weight-gradient kernel.
__global__ __launch_bounds__(kThreads, M2D_PROJ_OCC) void m2d_proj_bwd_data_mfma_kernel(const ProjArgs a) {
  extern __shared__ float smem[];
  const int wave = wave_id(), l = threadIdx.x & 63, mn = l & 15, kb = l >> 4;
  const int zst = a.Opad32 + 8;
  float* stage = smem + wave * (16 * kStageStride + 16 * zst / 2);   // [16][68] floats, then [16][zst] bf16
  uint16_t* zs = reinterpret_cast<uint16_t*>(stage + 16 * kStageStride);
  for (int i = l; i < 16 * zst / 2; i += 64) reinterpret_cast<uint32_t*>(zs)[i] = 0u;   // padding columns: zero
  const int64_t p0 = (int64_t)blockIdx.x * kTP + wave * 16;
  const int rows = (int)(a.P - p0 < 16 ? a.P - p0 : 16);   // positions of the wave inside the array (may be <= 0)
  const int R = a.R, R2 = 2 * a.R, NQ = a.Rpad / 16;
  // wave-uniform bases (the wave's first position); lanes add 32-bit element offsets
  const bf16_t* dT = static_cast<const bf16_t*>(a.dT) + p0 * a.E;
  const bf16_t* dL = static_cast<const bf16_t*>(a.dL) + p0 * a.E;
  const bf16_t* ddT = static_cast<const bf16_t*>(a.ddT) + p0 * a.E;
  const bf16_t* ddL = static_cast<const bf16_t*>(a.ddL) + p0 * a.E;
  bf16_t* dx = static_cast<bf16_t*>(a.dx) + p0 * a.E;
  // rows past the end of the arrays (up to the next multiple of 16) are written too, as zeros
  uint16_t* dzt = a.dzt + p0 * a.Opad;
  uint16_t* dptT = a.dpt + p0 * a.E;
  uint16_t* dptL = dptT + (int64_t)a.ntiles * kTP * a.E;
  const uint4 z4 = make_uint4(0, 0, 0, 0);
  const bool given = a.dpre_given != 0;   // (uniform) ddT, ddL are dpre already: nothing to derive or to write out

  // Memory latency is covered by the other waves of the compute unit (registers are kept low
  // for that), not by fetching ahead.
  // dB_T, dB_L, dC: lane l holds 4 values of position l >> 2
  const int cb = l >> 2, n0 = 4 * (l & 3);
  uint2 bc[3];
  sum_channels(a, p0, rows, cb, n0, bc);

  // dz[., rank] = dpre w, channels as the inner dimension
  f32x4 accT[2], accL[2];
#pragma unroll
  for (int nq = 0; nq < 2; ++nq) { accT[nq] = (f32x4){0.f, 0.f, 0.f, 0.f}; accL[nq] = accT[nq]; }
  auto dpre = [](uint4 g, uint4 v) {
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, vw[4] = {v.x, v.y, v.z, v.w};
    uint32_t r[4];
#pragma unroll
    for (int h = 0; h < 4; ++h)
      r[h] = pack2(bf16_lo(gw[h]) * softplus_slope(bf16_lo(vw[h])), bf16_hi(gw[h]) * softplus_slope(bf16_hi(vw[h])));
    return make_uint4(r[0], r[1], r[2], r[3]);
  };
  for (int e = 8 * kb; e < a.Epad; e += 32) {
    const bool ok = mn < rows && e < a.E;
    const uint32_t off = (uint32_t)(mn * a.E + e);
    uint4 AT = ok ? load16(ddT + off) : z4, AL = ok ? load16(ddL + off) : z4;
    if (!given) {
      AT = dpre(AT, ok ? load16(dT + off) : z4);
      AL = dpre(AL, ok ? load16(dL + off) : z4);
    }
#pragma unroll
    for (int nq = 0; nq < 2; ++nq)
      if (nq < NQ) {
        accT[nq] = mfma16(AT, load16(a.wTtb + (16 * nq + mn) * a.Epad + e), accT[nq]);
        accL[nq] = mfma16(AL, load16(a.wLtb + (16 * nq + mn) * a.Epad + e), accL[nq]);
      }
    if (given) continue;   // the weight-gradient kernel reads the caller's arrays
    // dpre leaves through LDS, 64 channels at a time, so that memory sees whole 128-byte rows
    uint16_t* pst = reinterpret_cast<uint16_t*>(stage);
    *reinterpret_cast<uint4*>(pst + mn * kStageStride + (e & 63)) = AT;
    *reinterpret_cast<uint4*>(pst + (16 + mn) * kStageStride + (e & 63)) = AL;
    if ((e & 32) != 0) {   // uniform: second half of a group of 64
      const int e0 = e & ~63;
      wave_sync_lds();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int piece = l + 64 * k, c = piece >> 3, c8 = 8 * (piece & 7);
        if (e0 + c8 < a.E) {
          *reinterpret_cast<uint4*>(dptT + (uint32_t)(c * a.E + e0 + c8)) = load16(pst + c * kStageStride + c8);
          *reinterpret_cast<uint4*>(dptL + (uint32_t)(c * a.E + e0 + c8)) = load16(pst + (16 + c) * kStageStride + c8);
        }
      }
      wave_sync_lds();
    }
  }
  // rows of dz to LDS as bf16: operand of the next product, and source of the copy in memory
#pragma unroll
  for (int nq = 0; nq < 2; ++nq) {
    const int q = 16 * nq + mn;
    if (nq < NQ && q < R) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = 4 * kb + i;
        zs[c * zst + q] = f32_to_bf16_bits(accT[nq][i]);
        zs[c * zst + R + q] = f32_to_bf16_bits(accL[nq][i]);
      }
    }
  }
#pragma unroll
  for (int w = 0; w < 3; ++w) {
    uint32_t* dst = reinterpret_cast<uint32_t*>(zs + cb * zst + R2 + w * kN + n0);   // even offsets: 4-byte aligned
    dst[0] = bc[w].x;
    dst[1] = bc[w].y;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  {
    const int per_row = a.Opad / 8;   // 16-byte pieces of a row
    for (int i = l; i < 16 * per_row; i += 64) {
      const int c = i / per_row, o8 = i - c * per_row;
      *reinterpret_cast<uint4*>(dzt + (uint32_t)(c * a.Opad + 8 * o8)) = load16(zs + c * zst + 8 * o8);
    }
  }

  // dx += dz Wx, outputs as the inner dimension
  constexpr int kMaxKS = (2 * kMaxR + 3 * kN + 31) / 32;
  uint4 A2[kMaxKS];
#pragma unroll
  for (int ks = 0; ks < kMaxKS; ++ks)
    A2[ks] = 32 * ks < a.Opad32 ? load16(zs + mn * zst + 32 * ks + 8 * kb) : z4;
  for (int e0 = 0; e0 < a.Epad; e0 += kKC) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int e = e0 + 16 * nt + mn;
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < kMaxKS; ++ks)
        if (32 * ks < a.Opad32) s = mfma16(A2[ks], load16(a.WxTb + e * a.Opad32 + 32 * ks + 8 * kb), s);
      stage_put(stage, nt, mn, kb, s);
    }
    wave_sync_lds();
    stage_rows(stage, l, [&](int c, int c8, const float (&v)[8]) {
      if (c < rows && e0 + c8 < a.E) {
        bf16_t* at = dx + (uint32_t)(c * a.E + e0 + c8);
        const uint4 was = load16(at);
        const uint32_t w[4] = {was.x, was.y, was.z, was.w};
        float sum[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) { sum[2 * j] = bf16_lo(w[j]) + v[2 * j]; sum[2 * j + 1] = bf16_hi(w[j]) + v[2 * j + 1]; }
        *reinterpret_cast<uint4*>(at) = pack8(sum);
      }
    });
    wave_sync_lds();
  }
}

// Backward, data, for up to 256 channels and a rank of up to 16; the kernel above has the wider ones, whose weights fill the LDS, and many positions of the
// widest of these (proj_bwd_in_lds).  It moves what it must (64x56x56x64 with
// 4 parts of channel sums: 283 MB), and what it lost were waits: for the packing launch before it, for weight tiles that each wave fetched from the caches,
// and for dx, asked for at the end.  Here a workgroup rounds the weights into LDS from the caller's tensors, and most of what it reads is asked for before the
// first wait: the step sizes' weights, their gradients, three pieces of x_proj a thread (two outputs of four channels
// each: all of it up to 64 channels; of the 4 pieces at 128 channels and the 12 at 256 with a rank of 16 the rest are fetched one by one), and dx where registers allow four workgroups a compute unit (up to 64 channels; with 128
// three fitted, and 784 tiles of 64x28x28x128 took a second generation for the last 16: whole backward 56.5 us against 50.3 without).  The channel sums
// follow when the weights are in place, and without dpre the step sizes are fetched where they are used.  The weights' rows are the first operands, so dx leaves from registers, 16 bytes a lane.
// Backward of the projections in all, ten calls in a row: 64x56x56x64, 4 parts 91.5 -> 77.6 us, 64x28x28x128, 8 parts 57.7 -> 48.0, 4x128x128x64, 8 parts 47.2 ->
// 40.8, 64x14x14x256, 16 parts 46.7 -> 39.8, 200000 positions of 32 channels 68.8 -> 51.9, 1568 of 64 17.4 -> 13.9 (with the step sizes' weights in a loop that
// waited for each load 81.9, 50.3, 42.3, 43.1, 53.7 and 14.9); bit for bit the same results.
template <int KS>   // steps of 32 channels at most
__global__ __launch_bounds__(kThreads, KS <= 4 ? 4 : 2) void m2d_proj_bwd_data_lds_kernel(const ProjArgs a) {
  extern __shared__ float smem[];
  const int tid = threadIdx.x, wave = wave_id(), l = tid & 63, mn = l & 15, kb = l >> 4;
  const int E = a.E, Epad = (E + 31) / 32 * 32, R = a.R, R2 = 2 * a.R, O = a.O, LQ = Epad + 8, zst = a.Opad32 + 8;
  uint16_t* wq = reinterpret_cast<uint16_t*>(smem);   // [2][16 ranks][LQ]: weights of the step sizes
  uint16_t* wx = wq + 32 * LQ;                         // [Epad][zst]: x_proj transposed
  uint16_t* zs = wx + Epad * zst + wave * 16 * zst;    // the wave's rows of dz
  const int64_t p0 = (int64_t)blockIdx.x * kTP + wave * 16;
  const int rows = (int)(a.P - p0 < 16 ? a.P - p0 : 16);   // positions of the wave inside the array (may be <= 0)
  const bool given = a.dpre_given != 0;   // (uniform) ddT, ddL are dpre already: nothing to derive or to write out
  const bool in = mn < rows;
  const int64_t off = (p0 + mn < a.P ? p0 + mn : a.P - 1) * E;   // rows past the end repeat the last one: masked, not stored
  const uint4 z4 = make_uint4(0, 0, 0, 0);

  // the weights first, then the gradients and dx, all under way before the first wait
  constexpr int kHold = 3;   // pairs of outputs x 4 channels of a thread
  f32x4 hw0[kHold], hw1[kHold];
  const int nwx = (a.Opad32 / 2) * (Epad / 4);
  auto wx_at = [&](int i, int& o, int& c) {
    o = 2 * (i / (Epad / 4));
    c = 4 * (i - (o / 2) * (Epad / 4));
    return i < nwx;
  };
  auto get_wx = [&](int i, int k) -> f32x4 {      // output 2 pair + k, padding: zeros
    int o, c;
    const bool ok = wx_at(i, o, c) && o < O && c < E;   // (O is even)
    const f32x4 v = load_f4(a.Wx + (ok ? (o + k) * E + c : 0));
    return ok ? v : (f32x4){0.f, 0.f, 0.f, 0.f};
  };
  auto put_wx = [&](int i, f32x4 u, f32x4 v) {
    int o, c;
    if (!wx_at(i, o, c)) return;
    uint32_t* dst = reinterpret_cast<uint32_t*>(wx + c * zst + o);
    dst[0] = pack2(u[0], v[0]);
    dst[zst / 2] = pack2(u[1], v[1]);
    dst[zst] = pack2(u[2], v[2]);
    dst[3 * (zst / 2)] = pack2(u[3], v[3]);
  };
#pragma unroll
  for (int u = 0; u < kHold; ++u) { hw0[u] = get_wx(tid + u * kThreads, 0); hw1[u] = get_wx(tid + u * kThreads, 1); }
  constexpr int kDt = 2 * KS;
  const int ndt = E * R;
  float hT[kDt], hL[kDt];
#pragma unroll
  for (int u = 0; u < kDt; ++u) {
    const int i = tid + u * kThreads;
    hT[u] = a.wT[i < ndt ? i : 0];
    hL[u] = a.wL[i < ndt ? i : 0];
  }
  uint4 X[2][KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int e = 32 * s + 8 * kb, at = e < E ? e : 0;
    X[0][s] = load16(static_cast<const bf16_t*>(a.ddT) + off + at);
    X[1][s] = load16(static_cast<const bf16_t*>(a.ddL) + off + at);
  }
  constexpr bool kAhead = KS <= 2;   // (registers) dx is asked for ahead too
  uint4 was[kAhead ? KS : 1];
  if constexpr (kAhead) {
#pragma unroll
    for (int s = 0; s < KS; ++s) was[s] = load16(static_cast<const bf16_t*>(a.dx) + off + (32 * s + 8 * kb < E ? 32 * s + 8 * kb : 0));
  }
  for (int i = tid; i < 32 * LQ / 8; i += kThreads) reinterpret_cast<uint4*>(wq)[i] = z4;
  for (int i = l; i < 16 * zst / 2; i += 64) reinterpret_cast<uint32_t*>(zs)[i] = 0u;   // padding columns: zero
  __syncthreads();
#pragma unroll
  for (int u = 0; u < kDt; ++u) {
    const int i = tid + u * kThreads, e = i / R, q = i - e * R;
    if (i < ndt) {
      wq[q * LQ + e] = f32_to_bf16_bits(hT[u]);
      wq[(16 + q) * LQ + e] = f32_to_bf16_bits(hL[u]);
    }
  }
#pragma unroll
  for (int u = 0; u < kHold; ++u) put_wx(tid + u * kThreads, hw0[u], hw1[u]);
  for (int i = tid + kHold * kThreads; i < nwx; i += kThreads) put_wx(i, get_wx(i, 0), get_wx(i, 1));

  const int cb = l >> 2, n0 = 4 * (l & 3);   // dB_T, dB_L, dC: lane l holds 4 values of position l >> 2
  uint2 bc[3];
  sum_channels(a, p0, rows, cb, n0, bc);
  __syncthreads();

  // dz[., rank] = dpre w, channels as the inner dimension
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int e = 32 * s + 8 * kb;
    if (32 * s >= E) break;      // (uniform)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      uint4 v = in && e < E ? X[h][s] : z4;
      if (!given) {
        const uint4 d = in && e < E ? load16(static_cast<const bf16_t*>(h ? a.dL : a.dT) + off + e) : z4;
        const uint32_t gw[4] = {v.x, v.y, v.z, v.w}, dw[4] = {d.x, d.y, d.z, d.w};
        uint32_t r[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = pack2(bf16_lo(gw[k]) * softplus_slope(bf16_lo(dw[k])), bf16_hi(gw[k]) * softplus_slope(bf16_hi(dw[k])));
        v = make_uint4(r[0], r[1], r[2], r[3]);
        // for the weight-gradient kernel; rows past the end too, as zeros
        if (e < E) *reinterpret_cast<uint4*>(a.dpt + (h ? (int64_t)a.ntiles * kTP * E : 0) + (p0 + mn) * E + e) = v;
      }
      acc[h] = mfma16(load16(wq + (16 * h + mn) * LQ + e), v, acc[h]);
    }
  }
  // rows of dz to LDS as bf16: operand of the next product, and source of the copy in memory
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int q = 4 * kb + i;
    if (q < R) {
      zs[mn * zst + q] = f32_to_bf16_bits(acc[0][i]);
      zs[mn * zst + R + q] = f32_to_bf16_bits(acc[1][i]);
    }
  }
#pragma unroll
  for (int w = 0; w < 3; ++w) {
    uint32_t* dst = reinterpret_cast<uint32_t*>(zs + cb * zst + R2 + w * kN + n0);   // even offsets: 4-byte aligned
    dst[0] = bc[w].x;
    dst[1] = bc[w].y;
  }
  wave_sync_lds();
  {
    uint16_t* dzt = a.dzt + p0 * a.Opad;   // rows past the end of the arrays (up to the next tile) are written too, as zeros
    const int per_row = a.Opad / 8;        // 16-byte pieces of a row
    for (int i = l; i < 16 * per_row; i += 64) {
      const int c = i / per_row, o8 = i - c * per_row;
      *reinterpret_cast<uint4*>(dzt + (uint32_t)(c * a.Opad + 8 * o8)) = load16(zs + c * zst + 8 * o8);
    }
  }
  // dx += dz Wx, outputs as the inner dimension; a pair of tiles lists its rows so that a lane ends with 8 neighbouring channels
  uint4 A2[3];
#pragma unroll
  for (int ks = 0; ks < 3; ++ks) A2[ks] = 32 * ks < a.Opad32 ? load16(zs + mn * zst + 32 * ks + 8 * kb) : z4;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int e = 32 * s + 8 * kb, row = 32 * s + 8 * (mn >> 2) + (mn & 3);
    if (32 * s >= E) break;      // (uniform)
    bf16_t* at = static_cast<bf16_t*>(a.dx) + off + (e < E ? e : 0);
    const uint4 old = kAhead ? was[kAhead ? s : 0] : load16(at);
    float v[8];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      f32x4 d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 3; ++ks)
        if (32 * ks < a.Opad32) d = mfma16(load16(wx + (row + 4 * t) * zst + 32 * ks + 8 * kb), A2[ks], d);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[4 * t + i] = d[i];
    }
    const uint32_t w[4] = {old.x, old.y, old.z, old.w};
    float sum[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) { sum[2 * k] = bf16_lo(w[k]) + v[2 * k]; sum[2 * k + 1] = bf16_hi(w[k]) + v[2 * k + 1]; }
    if (in && e < E) *reinterpret_cast<uint4*>(at) = pack8(sum);
  }
}

// Backward, weights, on the matrix cores.  Positions are the inner dimension of all three sums,
//   dWx[o][e] = sum_p dz[p][o] x[p][e],  dw[e][q] = sum_p dpre[p][e] r[p][q],  db[e] = sum_p dpre[p][e] * 1,
// so every operand is wanted position-last while the arrays are position-first.  A tile of 64
// positions is turned in LDS: a lane loads 16 bytes of one position's row and writes its 8 values
// into 8 rows of the position-last block (lanes = consecutive positions: no bank conflicts).
// LDS: xT[64][72], pT[2][64][72], zT[Opad][72], rT[2][16 NQ1][72] with a row of ones after the
// R rows of r (its column of the product is db).  Grid, parts and the prefetch of the next tile
// are those of the vector-ALU kernel.
constexpr int kPosStride = 72;   // bf16 per row of a position-last block: 64 + 8, rows 16-byte aligned
constexpr int kMaxNQ1 = (kMaxR + 1 + 15) / 16;
constexpr int kMaxZP = (kMaxNT * 2 + kWaves - 1) / kWaves;   // 16-byte pieces of a dz row per wave

__global__ __launch_bounds__(kThreads) void m2d_proj_bwd_weights_mfma_kernel(const ProjArgs a) {
  extern __shared__ float smem[];
  const int wave = wave_id(), l = threadIdx.x & 63, mn = l & 15, kb = l >> 4, tid = threadIdx.x;
  const int ey = blockIdx.y;
  const int R = a.R, R2 = 2 * a.R;
  const int NQ1 = (R + 1 + 15) / 16, MT = a.Opad / 16, ZP = a.Opad / 8;
  uint16_t* xT = reinterpret_cast<uint16_t*>(smem);
  uint16_t* pT = xT + kKC * kPosStride;
  uint16_t* zT = pT + 2 * kKC * kPosStride;
  uint16_t* rT = zT + a.Opad * kPosStride;
  const int rblk = 16 * NQ1 * kPosStride;   // one tensor's block of rT
  for (int i = tid; i < rblk; i += kThreads) reinterpret_cast<uint32_t*>(rT)[i] = 0u;   // both blocks (2 * rblk / 2 words)
  __syncthreads();
  if (tid < 2 * kTP) rT[(tid >> 6) * rblk + R * kPosStride + (tid & 63)] = 0x3F80;   // 1.0
  const bf16_t* x = static_cast<const bf16_t*>(a.x);
  const bf16_t* rr = static_cast<const bf16_t*>(a.r);
  // dpre: the copy the data kernel wrote for whole tiles, or the caller's arrays (P rows)
  const bool given = a.dpre_given != 0;
  const uint16_t* dptT = given ? static_cast<const uint16_t*>(a.ddT) : a.dpt;
  const uint16_t* dptL = given ? static_cast<const uint16_t*>(a.ddL) : a.dpt + (int64_t)a.ntiles * kTP * a.E;

  // this thread's part of the r tile (64 x 2R values, contiguous): up to two 16-byte pieces
  int rp[2], rq[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int first = 8 * (k * kThreads + tid);
    rp[k] = first / R2;
    rq[k] = first - rp[k] * R2;
  }
  const int nr = kTP * R2;   // values in the r tile

  f32x4 aw[2][4], ar[2][kMaxNQ1];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) aw[h][nt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nq = 0; nq < kMaxNQ1; ++nq) ar[h][nq] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }

  uint4 xr[2], pr[2][2], zr[kMaxZP], rv[2];
  auto fetch = [&](int tile) {
    const int64_t p0 = (int64_t)tile * kTP;
    const int64_t left = a.P - p0;   // positions of the tile inside the array, if fewer than 64
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int e = ey * kKC + 8 * (2 * wave + k);
      const bool ok = e < a.E;
      xr[k] = (l < left && ok) ? load16(x + (p0 + l) * a.E + e) : zero16();
      // dz and the data kernel's dpre are written for whole tiles (zeros past the end of the arrays)
      const bool pok = ok && (!given || l < left);
      pr[0][k] = pok ? load16(dptT + (p0 + l) * a.E + e) : zero16();
      pr[1][k] = pok ? load16(dptL + (p0 + l) * a.E + e) : zero16();
      const int first = 8 * (k * kThreads + tid);
      // a piece of r may straddle the end of the array, by whole values
      rv[k] = zero16();
      if (first < nr) {
        if ((int64_t)(first + 8) <= left * R2) rv[k] = load16(rr + p0 * R2 + first);
        else if ((int64_t)first < left * R2) {
          uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
          for (int j = 0; j < 8; ++j)   // (unrolled: w stays in registers)
            if ((int64_t)(first + j) < left * R2) w[j >> 1] |= (uint32_t)rr[p0 * R2 + first + j].v << (16 * (j & 1));
          rv[k] = make_uint4(w[0], w[1], w[2], w[3]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kMaxZP; ++k) {
      const int o8 = wave + kWaves * k;
      zr[k] = o8 < ZP ? load16(a.dzt + (p0 + l) * a.Opad + 8 * o8) : zero16();
    }
  };
  // lane = position: the 8 values of a 16-byte piece go to 8 consecutive rows of a position-last block
  auto turn = [&](uint16_t* blk, uint4 v) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int j = 0; j < 8; ++j) blk[j * kPosStride + l] = (uint16_t)(w[j >> 1] >> (16 * (j & 1)));
  };

  if ((int)blockIdx.x < a.ntiles) fetch(blockIdx.x);
  for (int tile = blockIdx.x; tile < a.ntiles; tile += a.G) {
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int row0 = 8 * (2 * wave + k);
      turn(xT + row0 * kPosStride, xr[k]);
      turn(pT + row0 * kPosStride, pr[0][k]);
      turn(pT + (kKC + row0) * kPosStride, pr[1][k]);
      const int first = 8 * (k * kThreads + tid);
      if (first < nr) {
        const uint32_t v[4] = {rv[k].x, rv[k].y, rv[k].z, rv[k].w};
        int p = rp[k], q = rq[k];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          if (p < kTP) rT[(q >= R ? rblk + (q - R) * kPosStride : q * kPosStride) + p] = (uint16_t)(v[j >> 1] >> (16 * (j & 1)));
          if (++q == R2) { q = 0; ++p; }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kMaxZP; ++k) {
      const int o8 = wave + kWaves * k;
      if (o8 < ZP) turn(zT + 8 * o8 * kPosStride, zr[k]);
    }
    __syncthreads();
    if (tile + a.G < a.ntiles) fetch(tile + a.G);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int koff = 32 * ks + 8 * kb;
      const uint4 A0 = load16(zT + (16 * wave + mn) * kPosStride + koff);
      const uint4 A1 = wave + kWaves < MT ? load16(zT + (16 * (wave + kWaves) + mn) * kPosStride + koff) : zero16();
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        const uint4 B = load16(xT + (16 * nt + mn) * kPosStride + koff);
        aw[0][nt] = mfma16(A0, B, aw[0][nt]);
        if (wave + kWaves < MT) aw[1][nt] = mfma16(A1, B, aw[1][nt]);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint4 Ap = load16(pT + (h * kKC + 16 * wave + mn) * kPosStride + koff);
#pragma unroll
        for (int nq = 0; nq < kMaxNQ1; ++nq)
          if (nq < NQ1) ar[h][nq] = mfma16(Ap, load16(rT + h * rblk + (16 * nq + mn) * kPosStride + koff), ar[h][nq]);
      }
    }
    __syncthreads();
  }

  // parts: D[4 kb + i][mn] of each accumulator
  float* out = a.part + ((int64_t)blockIdx.x * a.ne + ey) * (int64_t)(a.O + R2 + 2) * kKC;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int mt = wave + kWaves * h;
#pragma unroll
    for (int nt = 0; nt < 4; ++nt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int o = 16 * mt + 4 * kb + i;
        if (mt < MT && o < a.O) out[o * kKC + 16 * nt + mn] = aw[h][nt][i];
      }
#pragma unroll
    for (int nq = 0; nq < kMaxNQ1; ++nq) {
      const int q = 16 * nq + mn;
      const int row = q < R ? a.O + h * R + q : a.O + R2 + h;   // column R of the product is the bias gradient
      if (nq < NQ1 && q <= R) {
#pragma unroll
        for (int i = 0; i < 4; ++i) out[row * kKC + 16 * wave + 4 * kb + i] = ar[h][nq][i];
      }
    }
  }
}

// ------------------------------------------------------------------------------- fp32 products
// fp32 tensors, and bf16 ones whose rows are no whole 16-byte chunks, take the products through
// v_mfma_f32_16x16x4f32: fp32 operands and sums, half again the rate of the vector ALUs measured here, and a weight is
// one register of a lane in place of a scalar load the whole wave waits for.  Operands (lane l, n = l & 15, kb = l >> 4):
//   A[n][kb], B[kb][n], one register each;  D[4 kb + i][n], i < 4.
// The inner index may run in any order, the same one for A and B: at step j of 16 a lane holds index 4 kb + j, so both
// operands are float4 loads along a row, and a D tile (4 consecutive rows of a column per lane) is at once the B operand
// of the next product over its rows.  Positions are columns everywhere: z feeds the step sizes' products, and dz those
// of dx, without leaving the registers, and a lane stores 4 consecutive channels.
// A wave owns NT x 16 positions and needs no other wave: no LDS, no barrier, no packed copies of the weights.
// What bounds them is the traffic of the (P,E) arrays and, on few positions, the chain load - product - product - store.
// The outputs of Wx come in NL = ceil(2R/16) tiles of low-rank inputs and one tile each of B_T, B_L, C; "o'" below counts
// them with the padding behind 2R.
template <typename T, bool V4>
__device__ __forceinline__ f32x4 row4(const T* row, int c, int n) {   // elements c..c+3 of a row of n; past the end any element of the row
  f32x4 v;
  if constexpr (V4) {
    const int cc = c < n ? c : n - 4;
    if constexpr (sizeof(T) == 4) v = *reinterpret_cast<const f32x4*>(row + cc);
    else {
      const uint2 q = *reinterpret_cast<const uint2*>(row + cc);
      v[0] = __uint_as_float(q.x << 16); v[1] = __uint_as_float(q.x & 0xffff0000u);
      v[2] = __uint_as_float(q.y << 16); v[3] = __uint_as_float(q.y & 0xffff0000u);
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = ld(row + (c + j < n ? c + j : n - 1));
  }
  return v;
}
__device__ __forceinline__ f32x4 none_past(f32x4 v, int c, int n) {   // element j zero where c + j >= n
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = c + j < n ? v[j] : 0.f;
  return v;
}
template <typename T, bool V4>
__device__ __forceinline__ void put4(T* row, int c, int n, f32x4 v) {
  if constexpr (V4) {
    if (c >= n) return;
    if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4*>(row + c) = v;
    else *reinterpret_cast<uint2*>(row + c) = make_uint2(pack_bf16_pair(v[0], v[1]), pack_bf16_pair(v[2], v[3]));
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (c + j < n) st(row + c + j, v[j]);
  }
}
// a weight as the kernels are to see it (bf16 tensors: rounded if the caller asks for it)
template <typename T>
__device__ __forceinline__ f32x4 weights_of(const ProjArgs& a, f32x4 v) {
  if constexpr (sizeof(T) == 2) {
    if (a.round) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = as_stored(v[j], static_cast<const bf16_t*>(nullptr));
    }
  }
  return v;
}
__device__ __forceinline__ f32x4 mfma4(float x, float y, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0); }
// The four ranks o' = c .. c+3 of the stacked dt weights as they are for one of the two (first: its first o'): the
// element index inside a row of R, and whether the rank is one of its own.
struct Ranks { int at[4]; bool own[4]; };
__device__ __forceinline__ Ranks ranks_of(int c, int first, int R) {
  Ranks r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int q = c + j - first;
    r.own[j] = q >= 0 && q < R;
    r.at[j] = r.own[j] ? q : 0;
  }
  return r;
}

// Of the NL = ceil(2R / 16) tiles of ranks, those before this one hold ranks of T only, those behind it ranks of L and
// padding; this one may hold both.  Its products are made for each half on its own, with zeros (forward) or rows that are
// dropped (backward) in the place of the other's: an infinite value must not meet a zero weight.
template <int NL> constexpr int kMixed = (NL - 1) / 2;

template <typename T, bool V4, int NL, int NT>
__global__ __launch_bounds__(kThreads) void m2d_proj_fwd_f32_kernel(const ProjArgs a) {
  constexpr int NO = NL + 3;
  const int lane = threadIdx.x & 63, n = lane & 15, kb = lane >> 4;
  const int64_t p0 = ((int64_t)blockIdx.x * kWaves + wave_id()) * (16 * NT);
  if (p0 >= a.P) return;
  const int E = a.E, R = a.R, R2 = 2 * a.R;
  const int left = (int)(a.P - p0 < 16 * NT ? a.P - p0 : 16 * NT);
  const T* x = static_cast<const T*>(a.x) + p0 * E;
  int pl[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) pl[t] = 16 * t + n < left ? 16 * t + n : left - 1;
  // the rows of Wx behind row n of every tile: B_T, B_L, C in the order of the scan's records (see record_slot) if packed
  int wrow[NO];
#pragma unroll
  for (int ot = 0; ot < NO; ++ot) {
    const int i = n & 3, state = 4 * (i == 1 ? 2 : (i == 2 ? 1 : i)) + (n >> 2);
    const int o = ot < NL ? 16 * ot + n : R2 + 16 * (ot - NL) + (a.bc_packed ? state : n);
    wrow[ot] = (ot < NL && o >= R2 ? R2 - 1 : o) * E;    // (rows of padding repeat one: their products are dropped)
  }
  f32x4 z[NT][NO];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) z[t][ot] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 xv[NT], wv[NO];
  auto fetch = [&](int c) {
    const int e = c + 4 * kb;
#pragma unroll
    for (int t = 0; t < NT; ++t) xv[t] = row4<T, V4>(x + (int64_t)pl[t] * E, e, E);
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) wv[ot] = row4<float, V4>(a.Wx + wrow[ot], e, E);
  };
  fetch(0);
  for (int c = 0; c < E; c += 16) {
    f32x4 xc[NT], wc[NO];
#pragma unroll
    for (int t = 0; t < NT; ++t) xc[t] = xv[t];
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) wc[ot] = weights_of<T>(a, wv[ot]);
    if (c + 16 < E) fetch(c + 16);
    if (c + 16 > E) {
#pragma unroll
      for (int t = 0; t < NT; ++t) xc[t] = none_past(xc[t], c + 4 * kb, E);
#pragma unroll
      for (int ot = 0; ot < NO; ++ot) wc[ot] = none_past(wc[ot], c + 4 * kb, E);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int ot = 0; ot < NO; ++ot)
#pragma unroll
        for (int t = 0; t < NT; ++t) z[t][ot] = mfma4(wc[ot][j], xc[t][j], z[t][ot]);
  }

  // low-rank inputs (the step sizes' products see them as the tensor holds them) and B_T, B_L, C
  const T* as = nullptr;
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const bool live = 16 * t + n < left;
    const int64_t p = p0 + 16 * t + n;
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) {
#pragma unroll
      for (int j = 0; j < 4; ++j) z[t][ot][j] = as_stored(z[t][ot][j], as);
      const int o = 16 * ot + 4 * kb;
      if (!live) continue;
      if (ot < NL) {
        T* dst = static_cast<T*>(a.r_out) + p * R2;
        if (R2 % 4 == 0) put4<T, true>(dst, o, R2, z[t][ot]);
        else put4<T, false>(dst, o, R2, z[t][ot]);
      } else if (a.bc_packed) {
        put4<float, true>(a.bc_packed + p * (3 * kN) + (ot - NL) * kN, 4 * kb, kN, z[t][ot]);
      } else {
        put4<T, true>(static_cast<T*>(ot == NL ? a.BT_out : (ot == NL + 1 ? a.BL_out : a.C_out)) + p * kN, 4 * kb, kN, z[t][ot]);
      }
    }
  }

  // delta = softplus(r w^T + b), 16 channels at a time
  Ranks rk[2][NL];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int lt = 0; lt < NL; ++lt) rk[h][lt] = ranks_of(16 * lt + 4 * kb, h * R, R);
  f32x4 zl[NT];      // the mixed tile as L has it
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int lt = kMixed<NL>; lt < NL; ++lt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float v = z[t][lt][j];
        if (lt == kMixed<NL>) zl[t][j] = rk[1][lt].own[j] ? v : 0.f;
        z[t][lt][j] = rk[lt > kMixed<NL>][lt].own[j] ? v : 0.f;
      }
  f32x4 dw[2][NL], bias[2];
  auto fetch_dt = [&](int e0) {
    const int e = e0 + n < E ? e0 + n : E - 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float* w = (h ? a.wL : a.wT) + e * R;
#pragma unroll
      for (int lt = 0; lt < NL; ++lt)
#pragma unroll
        for (int j = 0; j < 4; ++j) dw[h][lt][j] = w[rk[h][lt].at[j]];
      bias[h] = row4<float, V4>(h ? a.bL : a.bT, e0 + 4 * kb, E);
    }
  };
  fetch_dt(0);
  for (int e0 = 0; e0 < E; e0 += 16) {
    f32x4 s[NT][2], w[2][NL];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const f32x4 b = weights_of<T>(a, bias[h]);
#pragma unroll
      for (int t = 0; t < NT; ++t) s[t][h] = b;
#pragma unroll
      for (int lt = 0; lt < NL; ++lt) {
        w[h][lt] = weights_of<T>(a, dw[h][lt]);
#pragma unroll
        for (int j = 0; j < 4; ++j) w[h][lt][j] = rk[h][lt].own[j] ? w[h][lt][j] : 0.f;
      }
    }
    if (e0 + 16 < E) fetch_dt(e0 + 16);
#pragma unroll
    for (int lt = 0; lt < NL; ++lt)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if ((h ? lt < kMixed<NL> : lt > kMixed<NL>) || (h && 16 * lt + 16 <= R)) continue;   // (uniform) no rank of this half
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < NT; ++t) s[t][h] = mfma4(w[h][lt][j], h && lt == kMixed<NL> ? zl[t][j] : z[t][lt][j], s[t][h]);
      }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (16 * t + n >= left) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int j = 0; j < 4; ++j) s[t][h][j] = softplus(s[t][h][j]);
        put4<T, V4>(static_cast<T*>(h ? a.dL_out : a.dT_out) + (p0 + 16 * t + n) * E, e0 + 4 * kb, E, s[t][h]);
      }
    }
  }
}

// Writes dz (fp32, rows of 16 (NL + 3), o' order) for the weights' gradients and adds dz Wx to dx.
template <typename T, bool V4, int NL, int NT>
__global__ __launch_bounds__(kThreads) void m2d_proj_bwd_data_f32_kernel(const ProjArgs a) {
  constexpr int NO = NL + 3;
  const int lane = threadIdx.x & 63, n = lane & 15, kb = lane >> 4;
  const int64_t p0 = ((int64_t)blockIdx.x * kWaves + wave_id()) * (16 * NT);
  if (p0 >= a.P) return;
  const int E = a.E, R = a.R, R2 = 2 * a.R;
  const int left = (int)(a.P - p0 < 16 * NT ? a.P - p0 : 16 * NT);
  const bool given = a.dpre_given != 0;   // (uniform) ddT, ddL are dpre already
  int64_t at[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) at[t] = p0 + (16 * t + n < left ? 16 * t + n : left - 1);

  f32x4 z[NT][NO];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
#pragma unroll
    for (int ot = 0; ot < NL; ++ot) z[t][ot] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 3; ++w)
      z[t][NL + w] = row4<T, true>(static_cast<const T*>(w == 0 ? a.dBT : (w == 1 ? a.dBL : a.dC)) + at[t] * kN, 4 * kb, kN);
  }
  // dz of the low-rank inputs: row n of tile lt is rank 16 lt + n of the two stacked (rows of the other half, and of
  // padding, repeat one: they are dropped)
  int q[2][NL];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int lt = 0; lt < NL; ++lt) {
      const int k = 16 * lt + n - h * R;
      q[h][lt] = k >= 0 && k < R ? k : 0;
    }
  f32x4 zl[NT];      // L's product with the mixed tile
#pragma unroll
  for (int t = 0; t < NT; ++t) zl[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 gv[2][NT], dv[2][NT], wv[2][NL];
  auto fetch = [&](int c) {
    const int e = c + 4 * kb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        gv[h][t] = row4<T, V4>(static_cast<const T*>(h ? a.ddL : a.ddT) + at[t] * E, e, E);
        if (!given) dv[h][t] = row4<T, V4>(static_cast<const T*>(h ? a.dL : a.dT) + at[t] * E, e, E);
      }
#pragma unroll
      for (int lt = 0; lt < NL; ++lt)
#pragma unroll
        for (int j = 0; j < 4; ++j) wv[h][lt][j] = (h ? a.wL : a.wT)[(e + j < E ? e + j : E - 1) * R + q[h][lt]];
    }
  };
  fetch(0);
  for (int c = 0; c < E; c += 16) {
    f32x4 g[2][NT], w[2][NL];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        g[h][t] = gv[h][t];
        if (!given) {
#pragma unroll
          for (int j = 0; j < 4; ++j) g[h][t][j] *= softplus_slope(dv[h][t][j]);
        }
      }
#pragma unroll
      for (int lt = 0; lt < NL; ++lt) w[h][lt] = weights_of<T>(a, wv[h][lt]);
    }
    if (c + 16 < E) fetch(c + 16);
    if (c + 16 > E) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t) g[h][t] = none_past(g[h][t], c + 4 * kb, E);
    }
#pragma unroll
    for (int lt = 0; lt < NL; ++lt)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if ((h ? lt < kMixed<NL> : lt > kMixed<NL>) || (h && 16 * lt + 16 <= R)) continue;   // (uniform) no rank of this half
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            f32x4& to = h && lt == kMixed<NL> ? zl[t] : z[t][lt];
            to = mfma4(w[h][lt][j], g[h][t][j], to);
          }
      }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int lt = kMixed<NL>; lt < NL; ++lt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int o = 16 * lt + 4 * kb + j;
        if (lt == kMixed<NL>) z[t][lt][j] = o < R ? z[t][lt][j] : zl[t][j];
        z[t][lt][j] = o < R2 ? z[t][lt][j] : 0.f;
      }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    if (16 * t + n >= left) continue;
#pragma unroll
    for (int ot = 0; ot < NO; ++ot) *reinterpret_cast<f32x4*>(a.dz + at[t] * (16 * NO) + 16 * ot + 4 * kb) = z[t][ot];
  }

  // dx += dz Wx, 64 channels at a time: a float4 of a row of Wx is row n of four tiles, channel 4n + c of the 64 in tile c,
  // so the four tiles of a lane hold the channels 16 kb + 4i + c
  for (int e0 = 0; e0 < E; e0 += 64) {
    f32x4 s[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x4 old = row4<T, V4>(static_cast<const T*>(a.dx) + at[t] * E, e0 + 16 * kb + 4 * i, E);
#pragma unroll
        for (int c = 0; c < 4; ++c) s[t][c][i] = old[c];
      }
#pragma unroll
    for (int ot = 0; ot < NO; ++ot)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int oo = 16 * ot + 4 * kb + j;
        const int o = ot < NL ? (oo < R2 ? oo : R2 - 1) : oo - 16 * NL + R2;   // (rows of padding: dz is zero)
        f32x4 w = weights_of<T>(a, row4<float, V4>(a.Wx + o * E, e0 + 4 * n, E));
        if (ot == NL - 1) {
#pragma unroll
          for (int c = 0; c < 4; ++c) w[c] = oo < R2 ? w[c] : 0.f;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
          for (int t = 0; t < NT; ++t) s[t][c] = mfma4(w[c], z[t][ot][j], s[t][c]);
      }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if (16 * t + n >= left) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        put4<T, V4>(static_cast<T*>(a.dx) + at[t] * E, e0 + 16 * kb + 4 * i, E, f32x4{s[t][0][i], s[t][1][i], s[t][2][i], s[t][3][i]});
    }
  }
}

// Grid (G, ne): workgroup (g, ey) adds up, over the tiles of 64 positions g, g+G, ..., the gradients of the weights that
// touch channels [64 ey, 64 ey + 64) and leaves them in part[g][ey][row][64]:
//   rows 0..O-1      dWx[o][.]      = sum_p dz[p][o] x[p][.]
//   rows O..O+R-1    dwT[.][q]      = sum_p dpreT[p][.] rT[p][q]      rows O+R..O+2R-1 the same for L
//   rows O+2R, +1    dbT[.], dbL[.] = sum_p dpre[p][.]
// Positions are the inner index here, 4 to a step, one per lane group kb: a lane's float4 along the channels (or along
// the first 64 outputs) is row or column n of four tiles, so a step is four float4 loads and 24 to 44 products.  A wave
// takes 16 positions of a tile; the four waves add up in LDS at the end.
template <typename T, bool V4, int NL>
__global__ __launch_bounds__(kThreads) void m2d_proj_bwd_weights_f32_kernel(const ProjArgs a) {
  constexpr int NO = NL + 3, RT = NL > 2 ? 2 : 1;
  extern __shared__ float sum[];
  const int lane = threadIdx.x & 63, n = lane & 15, kb = lane >> 4, wave = wave_id();
  const int E = a.E, R = a.R, R2 = 2 * a.R, e0 = blockIdx.y * kKC;
  const bool given = a.dpre_given != 0;   // (uniform) ddT, ddL are dpre already
  f32x4 aw[4][4], ax[NL > 1 ? NL - 1 : 1][4], ad[2][RT][4], ab[2];
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int c = 0; c < 4; ++c) {
#pragma unroll
    for (int o = 0; o < 4; ++o) aw[o][c] = zero;
#pragma unroll
    for (int o = 0; o + 1 < NL; ++o) ax[o][c] = zero;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int r = 0; r < RT; ++r) ad[h][r][c] = zero;
  }
  ab[0] = ab[1] = zero;

  f32x4 zv, xv, gv[2], dv[2];
  float zx[NL > 1 ? NL - 1 : 1], rv[2][RT];
  auto fetch = [&](int64_t p_raw) {
    const bool ok = p_raw < a.P;
    const int64_t p = ok ? p_raw : a.P - 1;
    const float* z = a.dz + p * (16 * NO);
    zv = *reinterpret_cast<const f32x4*>(z + 4 * n);
    xv = row4<T, V4>(static_cast<const T*>(a.x) + p * E, e0 + 4 * n, E);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      gv[h] = row4<T, V4>(static_cast<const T*>(h ? a.ddL : a.ddT) + p * E, e0 + 4 * n, E);
      if (!given) dv[h] = row4<T, V4>(static_cast<const T*>(h ? a.dL : a.dT) + p * E, e0 + 4 * n, E);
#pragma unroll
      for (int r = 0; r < RT; ++r) rv[h][r] = ld(static_cast<const T*>(a.r) + p * R2 + h * R + (16 * r + n < R ? 16 * r + n : R - 1));
    }
#pragma unroll
    for (int o = 0; o + 1 < NL; ++o) zx[o] = z[64 + 16 * o + n];
  };
  const int steps = ((a.ntiles - (int)blockIdx.x + a.G - 1) / a.G) * 4;    // (G <= ntiles: at least 4)
  auto position = [&](int s) { return ((int64_t)blockIdx.x + (int64_t)(s >> 2) * a.G) * kTP + wave * 16 + (s & 3) * 4 + kb; };
  fetch(position(0));
  for (int s = 0; s < steps; ++s) {
    const bool ok = position(s) < a.P;
    f32x4 zc = zv, xc = xv, g[2];
    float zxc[NL > 1 ? NL - 1 : 1], rc[2][RT];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      g[h] = gv[h];
      if (!given) {
#pragma unroll
        for (int j = 0; j < 4; ++j) g[h][j] *= softplus_slope(dv[h][j]);
      }
#pragma unroll
      for (int r = 0; r < RT; ++r) rc[h][r] = rv[h][r];
    }
#pragma unroll
    for (int o = 0; o + 1 < NL; ++o) zxc[o] = zx[o];
    if (s + 1 < steps) fetch(position(s + 1));
#pragma unroll
    for (int j = 0; j < 4; ++j) { zc[j] = ok ? zc[j] : 0.f; g[0][j] = ok ? g[0][j] : 0.f; g[1][j] = ok ? g[1][j] : 0.f; }
    ab[0] += g[0]; ab[1] += g[1];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
      for (int o = 0; o < 4; ++o) aw[o][c] = mfma4(zc[o], xc[c], aw[o][c]);
#pragma unroll
      for (int o = 0; o + 1 < NL; ++o) ax[o][c] = mfma4(ok ? zxc[o] : 0.f, xc[c], ax[o][c]);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < RT; ++r) ad[h][r][c] = mfma4(g[h][c], rc[h][r], ad[h][r][c]);
    }
  }

  // the four waves in turn, in the layout of the parts
  const int rows = a.O + R2 + 2;
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      ab[h][j] += __shfl_xor(ab[h][j], 16, 64);
      ab[h][j] += __shfl_xor(ab[h][j], 32, 64);
    }
  for (int w = 0; w < kWaves; ++w) {
    if (w == wave) {
      auto add4 = [&](int row, int col, f32x4 v) {
        f32x4* d = reinterpret_cast<f32x4*>(sum + row * kKC + col);
        *d = w ? *d + v : v;
      };
      auto row_of = [&](int oo) { return oo < 16 * NL ? (oo < R2 ? oo : -1) : oo - 16 * NL + R2; };   // o' -> row, -1: padding
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int o = 0; o < 4; ++o) {
          const int row = row_of(4 * (4 * kb + i) + o);
          if (row >= 0) add4(row, 4 * n, f32x4{aw[o][0][i], aw[o][1][i], aw[o][2][i], aw[o][3][i]});
        }
#pragma unroll
        for (int o = 0; o + 1 < NL; ++o) {
          const int row = row_of(64 + 16 * o + 4 * kb + i);
          if (row >= 0) add4(row, 4 * n, f32x4{ax[o][0][i], ax[o][1][i], ax[o][2][i], ax[o][3][i]});
        }
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int r = 0; r < RT; ++r)
            if (16 * r + n < R)
              add4(a.O + h * R + 16 * r + n, 4 * (4 * kb + i), f32x4{ad[h][r][0][i], ad[h][r][1][i], ad[h][r][2][i], ad[h][r][3][i]});
      }
      if (kb < 2) add4(a.O + R2 + kb, 4 * n, kb ? ab[1] : ab[0]);
    }
    __syncthreads();
  }
  float* out = a.part + ((int64_t)blockIdx.x * a.ne + blockIdx.y) * (int64_t)rows * kKC;
  for (int i = threadIdx.x; i < rows * (kKC / 4); i += kThreads) reinterpret_cast<f32x4*>(out)[i] = reinterpret_cast<const f32x4*>(sum)[i];
}

// Sums the per-workgroup parts in a fixed order and scatters them to the five weight gradients.
// Grid (rows, ne), 1024 threads: 64 channels x 16 slices of the workgroup index.
constexpr int kRedSlices = 16;
__global__ __launch_bounds__(64 * kRedSlices) void m2d_proj_reduce_kernel(const ProjArgs a) {
  __shared__ float sums[kRedSlices][64];
  const int rows = a.O + 2 * a.R + 2;
  const int row = blockIdx.x, ey = blockIdx.y;
  const int el = threadIdx.x & 63, gs = threadIdx.x >> 6;
  const float* src = a.part + ((int64_t)ey * rows + row) * kKC + el;
  const int64_t gstride = (int64_t)a.ne * rows * kKC;
  float s = 0.f;
#pragma unroll 8
  for (int g = gs; g < a.G; g += kRedSlices) s += src[g * gstride];
  sums[gs][el] = s;
  __syncthreads();
  if (gs != 0) return;
#pragma unroll
  for (int k = 1; k < kRedSlices; ++k) s += sums[k][el];
  const int e = ey * kKC + el;
  if (e >= a.E) return;
  if (row < a.O) a.dWx[row * a.E + e] = s;
  else if (row < a.O + a.R) a.dwT[e * a.R + (row - a.O)] = s;
  else if (row < a.O + 2 * a.R) a.dwL[e * a.R + (row - a.O - a.R)] = s;
  else if (row == a.O + 2 * a.R) a.dbT[e] = s;
  else a.dbL[e] = s;
}

// ------------------------------------------------------------------------------- host
inline size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
inline bool misaligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) & (a - 1)) != 0; }

struct ProjGeometry {
  int64_t P;
  int E, R, O, Epad, Opad, Opad32, Rpad, ntiles, G, ne;
  bool mfma;   // bf16, and rows of the (P,E) arrays start on 16-byte boundaries: products with bf16 operands
  // forward workspace
  size_t off_bTp, off_bLp, off_Wb, off_wTb, off_wLb, bytes_fwd;
  // backward workspace
  size_t off_wTtb, off_wLtb, off_WxTb, off_dz, off_dpt, off_part, bytes_bwd;
};

int check_proj(const m2d_desc* d, int R) {
  if (!d) return M2D_ERR_NULL_POINTER;
  if (d->B < 1 || d->H < 1 || d->W < 1 || d->E < 1 || d->N < 1 || R < 1) return M2D_ERR_BAD_SHAPE;
  if (d->N != kN || (d->dtype != M2D_F32 && d->dtype != M2D_BF16)) return M2D_ERR_UNSUPPORTED;   // (ckpt_interval is the scan's)
  if (d->flags & ~(M2D_FLAG_FLIP | M2D_FLAG_ROUND_WEIGHTS | M2D_FLAG_RAW_PARAMS | M2D_FLAG_PACKED_BC | M2D_FLAG_DPRE | M2D_FLAG_SPLIT_STATES | M2D_FLAG_WHOLE_STATES)) return M2D_ERR_UNSUPPORTED;
  if (R > kMaxR || d->E > 4096) return M2D_ERR_UNSUPPORTED;
  if ((int64_t)d->B * d->H * d->W >= ((int64_t)1 << 31) * kTP) return M2D_ERR_UNSUPPORTED;   // tiles counted in 32 bits
  return M2D_OK;
}

ProjGeometry proj_geometry(const m2d_desc* d, int R) {
  ProjGeometry g;
  g.P = (int64_t)d->B * d->H * d->W;
  g.E = d->E; g.R = R; g.O = 2 * R + 3 * kN;
  g.Epad = (g.E + kKC - 1) / kKC * kKC;
  g.Opad = (g.O + 15) / 16 * 16;
  g.Opad32 = (g.O + 31) / 32 * 32;
  g.Rpad = (R + 15) / 16 * 16;
  g.ntiles = (int)((g.P + kTP - 1) / kTP);
  g.ne = g.Epad / kKC;
  g.mfma = d->dtype == M2D_BF16 && d->E % 8 == 0;
  const int want = 512 / g.ne > 0 ? 512 / g.ne : 1;   // about two workgroups per compute unit in all
  g.G = g.ntiles < want ? g.ntiles : want;
  size_t o = 0;
  g.off_bTp = o; o += align256((size_t)g.Epad * 4);
  g.off_bLp = o; o += align256((size_t)g.Epad * 4);
  g.off_Wb = o; o += align256((size_t)g.Opad * g.Epad * 2);
  g.off_wTb = o; o += align256((size_t)g.Epad * 32 * 2);
  g.off_wLb = o; o += align256((size_t)g.Epad * 32 * 2);
  g.bytes_fwd = o;
  o = 0;
  g.off_wTtb = o; o += align256((size_t)g.Rpad * g.Epad * 2);
  g.off_wLtb = o; o += align256((size_t)g.Rpad * g.Epad * 2);
  g.off_WxTb = o; o += align256((size_t)g.Epad * g.Opad32 * 2);
  if (g.mfma) {   // dz and dpre as bf16 blocks per tile
    g.off_dz = o; o += align256((size_t)g.ntiles * kTP * g.Opad * 2);
    g.off_dpt = o; o += align256((size_t)2 * g.ntiles * kTP * g.E * 2);
  } else {
    g.off_dz = o; o += align256((size_t)g.P * g.Opad * 4);
    g.off_dpt = o;
  }
  g.off_part = o; o += align256((size_t)g.G * g.ne * (g.O + 2 * R + 2) * kKC * 4);
  g.bytes_bwd = o;
  return g;
}

void fill(ProjArgs& a, const ProjGeometry& g) {
  a.P = g.P; a.E = g.E; a.R = g.R; a.O = g.O; a.Epad = g.Epad; a.Opad = g.Opad; a.Opad32 = g.Opad32; a.Rpad = g.Rpad;
  a.ntiles = g.ntiles; a.G = g.G; a.ne = g.ne;
}

inline bool launched() { return hipGetLastError() == hipSuccess; }

int run_proj_fwd_mfma(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  const size_t lds = (size_t)kWaves * (16 * kStageStride * 4 + 2 * 16 * kLowStride * 2);
  hipLaunchKernelGGL(m2d_proj_fwd_mfma_kernel, dim3(g.ntiles), dim3(kThreads), lds, st, a);
  return launched() ? M2D_OK : M2D_ERR_HIP;
}

// The weights in LDS, straight from the caller's tensors: see the kernels.
bool proj_in_lds(const ProjGeometry& g) { return g.mfma && g.E <= kFlMaxE && g.R <= kFlMaxR; }
// In the backward a workgroup of 64 positions fills the LDS for itself, so two have to share a compute unit, one filling while the other
// multiplies, unless one round of workgroups does it.  More than 224 channels with a rank above 8 (84 KB) are alone: projections' backward at
// 16384 positions of 256 channels, packed weights against LDS, 47.6 and 41.9 us, but at 16500 53.6 and 59.4, at 50176 101 and 117; 240 channels,
// rank 13, 400000 positions 753 and 810.  With a rank of 8 (63 KB) the LDS stays ahead: 400000 of 256 channels 679 and 623 us.
size_t bwd_lds_bytes(int Epad, int Opad32) { return ((size_t)32 * (Epad + 8) + (size_t)(Epad + 16 * kWaves) * (Opad32 + 8)) * 2; }
bool proj_bwd_in_lds(const ProjGeometry& g) {
  return proj_in_lds(g) && (2 * bwd_lds_bytes((g.E + 31) / 32 * 32, g.Opad32) <= 160 * 1024 || g.ntiles <= kUnits);
}
// More dynamic LDS than 64 KB has to be allowed, once per kernel and device.
template <auto Kernel>
bool allow_lds(size_t bytes) {
  static std::atomic<uint64_t> seen{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  const uint64_t bit = 1ull << (dev & 63);
  if (seen.load(std::memory_order_acquire) & bit) return true;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return false;
  seen.fetch_or(bit, std::memory_order_release);
  return true;
}
template <int KS, int NL, bool PACKED>
int launch_proj_fwd_lds(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  const size_t lds = fl_lds_bytes((g.E + 31) / 32 * 32, NL);
  if (lds > 64 * 1024 && !allow_lds<&m2d_proj_fwd_lds_kernel<KS, NL, PACKED>>(fl_lds_bytes(kFlMaxE, NL))) return M2D_ERR_HIP;
  const int64_t tiles = (g.P + kTP - 1) / kTP;
  constexpr size_t most = KS == 2 ? 6 : (KS == 4 ? 4 : 2);   // workgroups whose registers fit a compute unit
  int64_t grid = kUnits * (int64_t)((160 * 1024) / lds < most ? (160 * 1024) / lds : most);   // as many as the device holds
  if (grid > tiles) grid = tiles;
  hipLaunchKernelGGL((m2d_proj_fwd_lds_kernel<KS, NL, PACKED>), dim3((unsigned)grid), dim3(kThreads), lds, st, a);
  return launched() ? M2D_OK : M2D_ERR_HIP;
}
int run_proj_fwd_lds(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  auto ranks = [&](auto ks) -> int {
    constexpr int KS = decltype(ks)::value;
    if (g.R <= 8) return a.bc_packed ? launch_proj_fwd_lds<KS, 1, true>(g, a, st) : launch_proj_fwd_lds<KS, 1, false>(g, a, st);
    return a.bc_packed ? launch_proj_fwd_lds<KS, 2, true>(g, a, st) : launch_proj_fwd_lds<KS, 2, false>(g, a, st);
  };
  if (g.E <= 64) return ranks(std::integral_constant<int, 2>{});
  return g.E <= 128 ? ranks(std::integral_constant<int, 4>{}) : ranks(std::integral_constant<int, 8>{});
}

// The fp32 products' kernels: V4 where the rows of the (P,E) arrays and of Wx are whole runs of 4 elements, NL tiles of
// low-rank inputs, NT tiles of 16 positions per wave.
template <typename F>
int with_tiles(int R, F f) {
  switch ((2 * R + 15) / 16) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    default: return f(std::integral_constant<int, 4>{});
  }
}

template <typename T, bool V4, int NT>
int run_proj_fwd_f32(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  return with_tiles(g.R, [&](auto nl) -> int {
    const unsigned grid = (unsigned)((g.P + 16 * NT * kWaves - 1) / (16 * NT * kWaves));
    hipLaunchKernelGGL((m2d_proj_fwd_f32_kernel<T, V4, nl(), NT>), dim3(grid), dim3(kThreads), 0, st, a);
    return launched() ? M2D_OK : M2D_ERR_HIP;
  });
}

int run_reduce(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  hipLaunchKernelGGL(m2d_proj_reduce_kernel, dim3(g.O + 2 * g.R + 2, g.ne), dim3(64 * kRedSlices), 0, st, a);
  return launched() ? M2D_OK : M2D_ERR_HIP;
}

template <int KS>
int launch_proj_bwd_lds(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  const size_t lds = bwd_lds_bytes((g.E + 31) / 32 * 32, g.Opad32), most = bwd_lds_bytes(32 * KS, 96);
  if (most > 64 * 1024 && !allow_lds<&m2d_proj_bwd_data_lds_kernel<KS>>(most)) return M2D_ERR_HIP;
  hipLaunchKernelGGL(m2d_proj_bwd_data_lds_kernel<KS>, dim3(g.ntiles), dim3(kThreads), lds, st, a);
  return launched() ? M2D_OK : M2D_ERR_HIP;
}
int run_proj_bwd_mfma(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  int rc;
  if (proj_bwd_in_lds(g)) {
    rc = g.E <= 64 ? launch_proj_bwd_lds<2>(g, a, st) : (g.E <= 128 ? launch_proj_bwd_lds<4>(g, a, st) : launch_proj_bwd_lds<8>(g, a, st));
  } else {
    const size_t lds_data = (size_t)kWaves * (16 * kStageStride * 4 + 16 * (g.Opad32 + 8) * 2);
    hipLaunchKernelGGL(m2d_proj_bwd_data_mfma_kernel, dim3(g.ntiles), dim3(kThreads), lds_data, st, a);
    rc = launched() ? M2D_OK : M2D_ERR_HIP;
  }
  if (rc) return rc;
  const size_t lds_w = (size_t)(3 * kKC + g.Opad + 2 * 16 * ((g.R + 1 + 15) / 16)) * kPosStride * 2;
  hipLaunchKernelGGL(m2d_proj_bwd_weights_mfma_kernel, dim3(g.G, g.ne), dim3(kThreads), lds_w, st, a);
  if (!launched()) return M2D_ERR_HIP;
  return run_reduce(g, a, st);
}

template <typename T, bool V4, int NT>
int run_proj_bwd_f32(const ProjGeometry& g, const ProjArgs& a, hipStream_t st) {
  return with_tiles(g.R, [&](auto nl) -> int {
    const unsigned grid = (unsigned)((g.P + 16 * NT * kWaves - 1) / (16 * NT * kWaves));
    hipLaunchKernelGGL((m2d_proj_bwd_data_f32_kernel<T, V4, nl(), NT>), dim3(grid), dim3(kThreads), 0, st, a);
    if (!launched()) return M2D_ERR_HIP;
    const size_t lds_w = (size_t)(g.O + 2 * g.R + 2) * kKC * 4;   // (at most 45 KB)
    hipLaunchKernelGGL((m2d_proj_bwd_weights_f32_kernel<T, V4, nl()>), dim3(g.G, g.ne), dim3(kThreads), lds_w, st, a);
    if (!launched()) return M2D_ERR_HIP;
    return run_reduce(g, a, st);
  });
}

// Two tiles of positions per wave share the loads of the weights, where that still leaves every SIMD two waves.
template <typename F>
int with_layout(bool f32, const ProjGeometry& g, F f) {
  using std::integral_constant;
  auto tiles = [&](auto t, auto v4) -> int { return g.P >= 65536 ? f(t, v4, integral_constant<int, 2>{}) : f(t, v4, integral_constant<int, 1>{}); };
  auto rows = [&](auto t) -> int { return g.E % 4 == 0 ? tiles(t, std::true_type{}) : tiles(t, std::false_type{}); };
  return f32 ? rows(float{}) : rows(bf16_t{});
}

}  // namespace

extern "C" {

size_t m2d_proj_workspace_bytes(const m2d_desc* desc, int dt_rank, int pass) {
  if (check_proj(desc, dt_rank) != M2D_OK || (pass != M2D_PASS_FWD && pass != M2D_PASS_BWD)) return 0;
  const ProjGeometry g = proj_geometry(desc, dt_rank);
  return pass == M2D_PASS_FWD ? g.bytes_fwd : g.bytes_bwd;
}

int m2d_proj_fwd(const m2d_desc* desc, int dt_rank, const void* x, const float* x_proj_w, const float* dt_projT_w,
                 const float* dt_projT_b, const float* dt_projL_w, const float* dt_projL_b, void* lowrank,
                 void* deltaT, void* deltaL, void* BT, void* BL, void* C, void* workspace, size_t workspace_bytes,
                 void* stream) {
  int rc = check_proj(desc, dt_rank);
  if (rc) return rc;
  const bool packed = (desc->flags & M2D_FLAG_PACKED_BC) != 0;   // B_T takes the records, B_L and C are not written
  const void* req[] = {x, x_proj_w, dt_projT_w, dt_projT_b, dt_projL_w, dt_projL_b, lowrank, deltaT, deltaL, BT,
                       packed ? BT : BL, packed ? BT : C, workspace};
  for (const void* q : req) if (!q) return M2D_ERR_NULL_POINTER;
  for (const void* q : req) if (misaligned(q, 16)) return M2D_ERR_MISALIGNED;
  if (misaligned(workspace, 256)) return M2D_ERR_MISALIGNED;
  const ProjGeometry g = proj_geometry(desc, dt_rank);
  if (workspace_bytes < g.bytes_fwd) return M2D_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  PackArgs k = {};
  k.Wx = x_proj_w; k.wT = dt_projT_w; k.bT = dt_projT_b; k.wL = dt_projL_w; k.bL = dt_projL_b;
  if (g.mfma && !proj_in_lds(g)) {
    k.bTp = reinterpret_cast<float*>(ws + g.off_bTp);
    k.bLp = reinterpret_cast<float*>(ws + g.off_bLp);
    k.Wb = reinterpret_cast<uint16_t*>(ws + g.off_Wb);
    k.wTb = reinterpret_cast<uint16_t*>(ws + g.off_wTb);
    k.wLb = reinterpret_cast<uint16_t*>(ws + g.off_wLb);
    k.E = g.E; k.R = g.R; k.O = g.O; k.Epad = g.Epad; k.Opad = g.Opad; k.Opad32 = g.Opad32; k.Rpad = g.Rpad;
    k.round = (desc->flags & M2D_FLAG_ROUND_WEIGHTS) != 0;
    const int n = g.Epad * (g.Opad > 32 ? g.Opad : 32);   // the largest forward copy
    hipLaunchKernelGGL(m2d_proj_pack_kernel, dim3((n + 255) / 256), dim3(256), 0, st, k);
    if (!launched()) return M2D_ERR_HIP;
  }
  ProjArgs a = {};
  fill(a, g);
  a.x = x; a.bTp = k.bTp; a.bLp = k.bLp;
  a.Wx = x_proj_w; a.wT = dt_projT_w; a.bT = dt_projT_b; a.wL = dt_projL_w; a.bL = dt_projL_b;
  a.round = (desc->flags & M2D_FLAG_ROUND_WEIGHTS) && desc->dtype == M2D_BF16;
  a.Wb = k.Wb; a.wTb = k.wTb; a.wLb = k.wLb;
  a.r_out = lowrank; a.dT_out = deltaT; a.dL_out = deltaL; a.BT_out = BT; a.BL_out = BL; a.C_out = C;
  a.bc_packed = packed ? static_cast<float*>(BT) : nullptr;
  if (proj_in_lds(g)) return run_proj_fwd_lds(g, a, st);
  return g.mfma ? run_proj_fwd_mfma(g, a, st) : with_layout(desc->dtype == M2D_F32, g, [&](auto t, auto v4, auto nt) -> int {
    return run_proj_fwd_f32<decltype(t), v4(), nt()>(g, a, st);
  });
}

int m2d_proj_bwd(const m2d_desc* desc, int dt_rank, const void* x, const void* lowrank, const void* deltaT,
                 const void* deltaL, const float* x_proj_w, const float* dt_projT_w, const float* dt_projL_w,
                 const void* d_deltaT, const void* d_deltaL, const void* d_BT, const void* d_BL, const void* d_C,
                 void* dx, float* d_x_proj_w, float* d_dt_projT_w, float* d_dt_projT_b, float* d_dt_projL_w,
                 float* d_dt_projL_b, void* workspace, size_t workspace_bytes, void* stream) {
  return m2d_proj_bwd_parts(desc, dt_rank, 0, x, lowrank, deltaT, deltaL, x_proj_w, dt_projT_w, dt_projL_w, d_deltaT, d_deltaL, d_BT, d_BL,
                            d_C, dx, d_x_proj_w, d_dt_projT_w, d_dt_projT_b, d_dt_projL_w, d_dt_projL_b, workspace, workspace_bytes, stream);
}

int m2d_proj_bwd_parts(const m2d_desc* desc, int dt_rank, int sum_parts, const void* x, const void* lowrank, const void* deltaT,
                       const void* deltaL, const float* x_proj_w, const float* dt_projT_w, const float* dt_projL_w,
                       const void* d_deltaT, const void* d_deltaL, const void* d_BT, const void* d_BL, const void* d_C,
                       void* dx, float* d_x_proj_w, float* d_dt_projT_w, float* d_dt_projT_b, float* d_dt_projL_w,
                       float* d_dt_projL_b, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check_proj(desc, dt_rank);
  if (rc) return rc;
  if (sum_parts < 0) return M2D_ERR_BAD_SHAPE;
  if (sum_parts > 0 && !proj_geometry(desc, dt_rank).mfma) return M2D_ERR_UNSUPPORTED;
  const bool given = (desc->flags & M2D_FLAG_DPRE) != 0;   // d_deltaT, d_deltaL are dpre: deltaT, deltaL are not read
  const void* req[] = {x, lowrank, x_proj_w, dt_projT_w, dt_projL_w, d_deltaT, d_deltaL, d_BT, sum_parts ? d_BT : d_BL, sum_parts ? d_BT : d_C,
                       dx, d_x_proj_w, d_dt_projT_w, d_dt_projT_b, d_dt_projL_w, d_dt_projL_b, workspace};
  for (const void* q : req) if (!q) return M2D_ERR_NULL_POINTER;
  if (!given && (!deltaT || !deltaL)) return M2D_ERR_NULL_POINTER;
  for (const void* q : req) if (misaligned(q, 16)) return M2D_ERR_MISALIGNED;
  if (!given && (misaligned(deltaT, 16) || misaligned(deltaL, 16))) return M2D_ERR_MISALIGNED;
  if (misaligned(workspace, 256)) return M2D_ERR_MISALIGNED;
  const ProjGeometry g = proj_geometry(desc, dt_rank);
  if (workspace_bytes < g.bytes_bwd) return M2D_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  char* ws = static_cast<char*>(workspace);
  PackArgs k = {};
  k.Wx = x_proj_w; k.wT = dt_projT_w; k.wL = dt_projL_w;
  if (g.mfma && !proj_bwd_in_lds(g)) {   // for the data kernel; the weight-gradient kernel needs no weights
    k.wTtb = reinterpret_cast<uint16_t*>(ws + g.off_wTtb);
    k.wLtb = reinterpret_cast<uint16_t*>(ws + g.off_wLtb);
    k.WxTb = reinterpret_cast<uint16_t*>(ws + g.off_WxTb);
    k.E = g.E; k.R = g.R; k.O = g.O; k.Epad = g.Epad; k.Opad = g.Opad; k.Opad32 = g.Opad32; k.Rpad = g.Rpad;
    int n = g.Opad32 * g.Epad;
    if (g.Epad * g.Rpad > n) n = g.Epad * g.Rpad;
    hipLaunchKernelGGL(m2d_proj_pack_kernel, dim3((n + 255) / 256), dim3(256), 0, st, k);
    if (!launched()) return M2D_ERR_HIP;
  }
  ProjArgs a = {};
  fill(a, g);
  a.x = x; a.r = lowrank; a.dT = deltaT; a.dL = deltaL; a.dpre_given = given ? 1 : 0; a.sum_parts = sum_parts;
  a.ddT = d_deltaT; a.ddL = d_deltaL; a.dBT = d_BT; a.dBL = d_BL; a.dC = d_C; a.dx = dx;
  a.Wx = x_proj_w; a.wT = dt_projT_w; a.wL = dt_projL_w;
  a.round = (desc->flags & M2D_FLAG_ROUND_WEIGHTS) && desc->dtype == M2D_BF16;
  a.wTtb = k.wTtb; a.wLtb = k.wLtb; a.WxTb = k.WxTb;
  a.dz = reinterpret_cast<float*>(ws + g.off_dz);
  a.dzt = reinterpret_cast<uint16_t*>(ws + g.off_dz);
  a.dpt = reinterpret_cast<uint16_t*>(ws + g.off_dpt);
  a.part = reinterpret_cast<float*>(ws + g.off_part);
  a.dWx = d_x_proj_w; a.dwT = d_dt_projT_w; a.dbT = d_dt_projT_b; a.dwL = d_dt_projL_w; a.dbL = d_dt_projL_b;
  return g.mfma ? run_proj_bwd_mfma(g, a, st) : with_layout(desc->dtype == M2D_F32, g, [&](auto t, auto v4, auto nt) -> int {
    return run_proj_bwd_f32<decltype(t), v4(), nt()>(g, a, st);
  });
}

}  // extern "C"
