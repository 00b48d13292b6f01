// Forward scan without snapshots for batches that fill the device: the rows of a band one after the other in a lane (m2d_fwd_rows_kernel).
//
// The kernels of m2dscan.hip put 14 rows of a band on 14 of 16 lanes and sweep anti-diagonals; two lanes in 16 replay the neighbouring
// bands' rows, a sweep has 15 steps of fill, and every lane has positions, constants and predicates of its own.  Here a lane walks its
// band's cells itself, column by column and down each column: lane = (channel, quarter of the states), 16 channels and 4 states of each per lane, so that a
// wave's 64 lanes are at one cell.  h[i-1,j] is the value of the cell before, h[i,j-1] is in a register of its own per row; what a cell's
// place means (first row, first column, past the end) is the same for the whole wave and lies in scalar registers.
//
// A workgroup is 8 sweeping waves, `NB` bands side by side of 8 / NB groups of 16 channels, and 4 waves that stage, one to a SIMD beside two
// sweeping ones.  Band slot s works on the block of 2 columns behind the one of slot s - 1; the last row of a band goes to the next
// slot through LDS, from the last slot to the first of the next round through memory.  One barrier a block.
// The staging waves fetch x, deltaT, deltaL and B_T, B_L, C two blocks ahead and put the coefficients c*x*deltaT, c*x*deltaL and the step
// sizes into LDS 2 cells ahead of the block that the sweeping waves are at, whose loads thus run on across the barrier; y
// comes back as sums over a lane's states and quarters (lane swaps), gets x*D and leaves in rows of 16 channels.
//
// Bound by the issue of vector instructions: a unit (cell, channel, state) is 9 of arithmetic, 2 of them exponentials at half rate; with the sums of y and what the
// staging waves do it is 11.6 to 11.8 as counted (SQ_INSTS_VALU), against 17.8 in m2d_fwd_split_kernel.  The two sweeping waves and the
// staging one of a SIMD keep it issuing 86 % of the time where a sweep has 56 blocks (128x56x56x64) and 71 % where it has 14 (64x28x28x128: start and end of the
// only round); without the staging waves, each wave bringing its own operands, it was 60 % (128x56x56x64: 0.245 ms).
// Products on the matrix cores do not help: an fp32 16x16x4 takes the vector ALU's time (32 clocks, measured), as much as the 8 multiply-adds it replaces.
// Forward without snapshots, bf16, a whole call, against the kernels that it takes over from: 128x56x56x64 0.247 -> 0.187 ms, 128x28x28x128 0.128 -> 0.089,
// 64x28x28x128 0.075 -> 0.052; rows of 4 channels past a whole chunk of 8, which those fetch value by value: 43x21x39x108 0.109 -> 0.059,
// 28x51x10x180 0.116 -> 0.046, 34x109x25x52 0.112 -> 0.091.  Images of one band (14x14, 7x7) are stacked in m2d_fwd_kernel: the rule does not price this kernel for them.
#include "m2drows.h"

#include <type_traits>

namespace m2drows {
namespace {

constexpr int kN = 16;
constexpr int kJC = 2;              // columns of a block
constexpr int kSweepers = 8, kStagers = 4;
constexpr int kAhead = 2;           // cells by which staging runs ahead of the blocks
constexpr float kLog2e = 1.4426950408889634f;

struct bf16_t { uint16_t v; };
typedef float f2v __attribute__((ext_vector_type(2)));
typedef __bf16 b2v __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float fexp2(float v) { return __builtin_amdgcn_exp2f(v); }
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f2v){lo, hi}, b2v)); }

// Four neighbouring channels (or states) of a tensor
template <typename T> struct Quad;
template <> struct Quad<float> {
  typedef float4 raw;
  static __device__ __forceinline__ void widen(const raw& q, float (&v)[4]) { v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w; }
  static __device__ __forceinline__ raw narrow(const float (&v)[4]) { return make_float4(v[0], v[1], v[2], v[3]); }
  static __device__ __forceinline__ float one(const void* p, int i) { return static_cast<const float*>(p)[i]; }
  static __device__ __forceinline__ float as_stored(float v) { return v; }
};
template <> struct Quad<bf16_t> {
  typedef uint2 raw;
  static __device__ __forceinline__ void widen(const raw& q, float (&v)[4]) { v[0] = bf_lo(q.x); v[1] = bf_hi(q.x); v[2] = bf_lo(q.y); v[3] = bf_hi(q.y); }
  static __device__ __forceinline__ raw narrow(const float (&v)[4]) { return make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3])); }
  static __device__ __forceinline__ float one(const void* p, int i) { return __uint_as_float((uint32_t)static_cast<const uint16_t*>(p)[i] << 16); }
  static __device__ __forceinline__ float as_stored(float v) { return __uint_as_float((uint32_t)__builtin_bit_cast(uint16_t, (__bf16)v) << 16); }
};
// A * log2 e and D from the caller's tensors, or from the parameters as a module holds them (A = -exp(A_log); both rounded to T, which
// is what the reference's casts to x.dtype do, wavefront_cuda.py:72-73, 90-91, 332)
template <typename T> __device__ __forceinline__ float gate_rate(const Args& p, const void* A, int i) {
  return (p.raw ? Quad<T>::as_stored(-expf(static_cast<const float*>(A)[i])) : Quad<T>::one(A, i)) * kLog2e;
}
template <typename T> __device__ __forceinline__ float skip_gain(const Args& p, int e) {
  return p.raw ? Quad<T>::as_stored(static_cast<const float*>(p.D)[e]) : Quad<T>::one(p.D, e);
}

// lanes 0..31 hold the sum of both halves of a, lanes 32..63 that of b
__device__ __forceinline__ float fold32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// rows of 16 lanes: even rows hold the (row, row + 1) sum of a, odd rows that of b
__device__ __forceinline__ float fold16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// The order of the states in a record, in LDS and in lanes is that of the packed records: place 4*m + f(q) holds state 4*q + m
__device__ __forceinline__ constexpr int swap12(int q) { return q == 1 ? 2 : (q == 2 ? 1 : q); }
__device__ __forceinline__ constexpr int state_at(int place) { return swap12(place & 3) * 4 + (place >> 2); }

// Everything this wave has asked of LDS is done, and that of the others is too.  (Stores to memory are not waited for.)
__device__ __forceinline__ void block_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// LDS, in floats
template <int R, int NB>
struct Lds {
  static constexpr int NG = kSweepers / NB, NC = R * kJC;
  static constexpr int kRec = NC * 3 * kN;          // B_T, B_L, C of a block
  static constexpr int kChan = NC * 64;             // [cell][channel] c*x*deltaT, c*x*deltaL, deltaT, deltaL
  static constexpr int kY = NC * 16;
  static constexpr int kRow = kJC * 256;            // boundary rows of a block: [column][lane] float4
  static constexpr int kRecAt = 0, kChanAt = kRecAt + NB * 2 * kRec, kYAt = kChanAt + kSweepers * 2 * kChan, kRowAt = kYAt + kSweepers * 2 * kY;
  static constexpr size_t kBytes = 4 * (size_t)(kRowAt + kSweepers * 2 * kRow);
};

// Where the blocks of a band slot are: item = (image of the workgroup, round of bands), b = block of the row of `stride` blocks
struct Turn {
  int item, b;
  __device__ __forceinline__ void next(int stride) { if (++b == stride) { b = 0; ++item; } }
};

template <typename T, int R, int NB, bool PACKED>
__global__ __launch_bounds__((kSweepers + kStagers) * 64, 3) void m2d_fwd_rows_kernel(const Args p) {
  using L = Lds<R, NB>;
  using Q = Quad<T>;
  using raw = typename Q::raw;
  using rec_raw = std::conditional_t<PACKED, float4, raw>;
  constexpr int NG = L::NG, NC = L::NC, JC = kJC;
  static_assert(NC % 2 == 0 && NC * 4 <= 64, "a lane stages one quad of one cell of a block");
  extern __shared__ float4 smem4[];
  float* smem = reinterpret_cast<float*>(smem4);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (p.link_err && blockIdx.x == 0 && threadIdx.x == 0) *p.link_err = 0;
  // consecutive workgroups are dealt round-robin to 8 XCDs: the channel groups of an image, which read the same records and lines, go to one
  int id = blockIdx.x;
  const int per = gridDim.x >> 3;
  if (per && id < per * 8) id = (id & 7) * per + (id >> 3);
  const int set = id / p.groups, wg = id - set * p.groups;      // images set * p.images ..., channels wg * NG * 16 ...
  const int img0 = set * p.images, nimg = p.B - img0 < p.images ? p.B - img0 : p.images;
  const int items = nimg * p.rounds;
  const int HW = p.H * p.W, groups16 = (p.E + 15) / 16;
  auto cell_at = [&](int row, int col) { const int c = row * p.W + col; return p.flip ? HW - 1 - c : c; };
  const int steps = items * p.stride + NB;                      // (the last one only stores y)
  const float ninf = -__builtin_huge_valf();

  if (wave >= kSweepers) {   // ------------------------------------------------------------------ stages
    // two sweeping waves' operands and results: of one band slot, or (8 slots) of two
    constexpr int NSL = NB == 8 ? 2 : 1, U = 2 / NSL;
    const int s = wave - kSweepers;
    const bool brings_rec = NB == 8 || s / NB == 0;
    const int pc = lane < NC * 4 ? lane >> 2 : NC - 1, pq = lane & 3, pj = pc / R, pi = pc - pj * R;   // the lane's cell of a block, for y; its quad
    const int sc = (pc + kAhead) % NC, sj = sc / R, si = sc - sj * R;                                 // ... and the one it stages,
    const bool ahead = pc + kAhead >= NC, lane_on = lane < NC * 4;                                    // of the block after
    struct Slot {
      Turn f, y, w;            // fetched next; swept now; wrapped rows
      int q;                   // blocks swept so far
      raw gx[U], gt[U], gl[U], xo[U];
      rec_raw gb[3];
      float4 tn[U][JC];
      float cT, cL;
      int64_t yo;
      bool on, yon;
    } st[NSL];
    float D4[NSL][U][4];
    int quad_ch[NSL][U];       // first channel of the lane's quad
    bool unit_on[NSL][U], quad_on[NSL][U];
    const int rounds = p.rounds;
    auto slot_of = [&](int k) { return NB == 8 ? s + 4 * k : s % NB; };
    auto grp_of = [&](int u) { return NB == 8 ? 0 : (s / NB) * 2 + u; };
    auto sweeper_of = [&](int k, int u) { return grp_of(u) * NB + slot_of(k); };
#pragma unroll
    for (int k = 0; k < NSL; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e0 = (wg * NG + grp_of(u)) * 16, e = e0 + pq * 4;
        unit_on[k][u] = e0 < p.E;
        quad_on[k][u] = e < p.E;                               // (whole quads: E is a multiple of 4)
        quad_ch[k][u] = e < p.E ? e : p.E - 4;
#pragma unroll
        for (int m = 0; m < 4; ++m) D4[k][u][m] = skip_gain<T>(p, quad_ch[k][u] + m);
      }
    // the operands of block t (and of the first cells of the one after it) into registers
    auto fetch = [&](Slot& z, int k, Turn t) {
      Turn t1 = t;
      t1.next(p.stride);
      const int item = ahead ? t1.item : t.item, b = ahead ? t1.b : t.b;
      const int im = rounds == 1 ? item : item / rounds, band = (item - im * rounds) * NB + slot_of(k);
      z.on = lane_on && b >= 0 && b < p.nblk && band < p.nbands && im < nimg;
      int row = band * R + si, col = b * JC + sj;
      const bool r0 = row == 0, c0 = col == 0;
      z.cT = r0 ? 0.f : c0 ? 1.f : 0.5f;
      z.cL = r0 ? 1.f : c0 ? 0.f : 0.5f;
      row = row < p.H ? row : p.H - 1;                         // (rows and columns off the grid: nothing that is on it depends on them)
      col = col < p.W ? (col < 0 ? 0 : col) : p.W - 1;
      const int64_t cell = (int64_t)(img0 + (im < nimg ? im : nimg - 1)) * HW + cell_at(row, col);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t o = cell * p.E + quad_ch[k][u];
        z.gx[u] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.x) + o);
        z.gt[u] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.dT) + o);
        z.gl[u] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.dL) + o);
      }
      if (brings_rec) {
        if constexpr (PACKED) {
          const float4* r = reinterpret_cast<const float4*>(p.rec + cell * (3 * kN)) + pq;
          z.gb[0] = r[0]; z.gb[1] = r[4]; z.gb[2] = r[8];
        } else {
          const int64_t o = cell * kN + pq * 4;
          z.gb[0] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.BT) + o);
          z.gb[1] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.BL) + o);
          z.gb[2] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.C) + o);
        }
      }
    };
    auto place = [&](const Slot& z, int k, int par) {          // par: of the block (that the lanes which run ahead are ahead of)
      const int at = ahead ? par ^ 1 : par;
      if (!z.on) return;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float x[4], t[4], l[4];
        Q::widen(z.gx[u], x); Q::widen(z.gt[u], t); Q::widen(z.gl[u], l);
        float4* c = reinterpret_cast<float4*>(smem + L::kChanAt + (sweeper_of(k, u) * 2 + at) * L::kChan + sc * 64) + pq * 4;
#pragma unroll
        for (int m = 0; m < 4; ++m) c[m] = make_float4(x[m] * z.cT * t[m], x[m] * z.cL * l[m], t[m], l[m]);
      }
      if (brings_rec) {
        float* d = smem + L::kRecAt + (slot_of(k) * 2 + at) * L::kRec + sc * (3 * kN);
        if constexpr (PACKED) {
          float4* d4 = reinterpret_cast<float4*>(d) + pq;
          d4[0] = z.gb[0]; d4[4] = z.gb[1]; d4[8] = z.gb[2];
        } else {
          float* to = d + swap12(pq);                          // states 4*pq + m
#pragma unroll
          for (int w = 0; w < 3; ++w) {
            float v[4];
            Q::widen(z.gb[w], v);
#pragma unroll
            for (int m = 0; m < 4; ++m) to[w * kN + 4 * m] = v[m];
          }
        }
      }
    };
    // slot 0: the rows that the last slot left in the round before (the first round: nothing above)
    auto wrap_at = [&](int item, int u, int col) {
      const int im = item / rounds, round = item - im * rounds;
      return reinterpret_cast<float4*>(p.wrap) + ((((int64_t)(round - 1) * p.B + img0 + im) * groups16 + wg * NG + grp_of(u)) * p.W + col) * 64 + lane;
    };
    auto has_wrap = [&](const Turn& t) { return t.item < items && t.b < p.nblk && rounds > 1 && t.item % rounds > 0; };
    auto wraps = [&](Slot& z, int k) {
      if (slot_of(k) != 0 || !has_wrap(z.w)) return;
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (unit_on[k][u])
#pragma unroll
          for (int j = 0; j < JC; ++j) z.tn[u][j] = *wrap_at(z.w.item, u, z.w.b * JC + j < p.W ? z.w.b * JC + j : p.W - 1);
    };
    auto put_wraps = [&](const Slot& z, int k, int par) {
      if (slot_of(k) != 0) return;
      const bool some = has_wrap(z.w);
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int j = 0; j < JC; ++j)
          reinterpret_cast<float4*>(smem + L::kRowAt + (sweeper_of(k, u) * 2 + par) * L::kRow)[j * 64 + lane] = some ? z.tn[u][j] : make_float4(0.f, 0.f, 0.f, 0.f);
    };
#pragma unroll
    for (int k = 0; k < NSL; ++k) {
      Slot& z = st[k];
      fetch(z, k, Turn{0, -1}); place(z, k, 1);
      fetch(z, k, Turn{0, 0}); place(z, k, 0);
      z.w = Turn{0, 0};
      put_wraps(z, k, 0);
      z.w.next(p.stride);
      z.f = Turn{0, 0};
      z.f.next(p.stride);
      fetch(z, k, z.f);
      z.y = Turn{0, 0};
      z.q = -slot_of(k);
      z.yon = false;
    }
    block_barrier();
    block_barrier();           // the first cells are in the sweeping waves' registers: from here on their place is that of block 2's
    for (int t = 0; t < steps; ++t) {
#pragma unroll
      for (int k = 0; k < NSL; ++k) {
        Slot& z = st[k];
        if (z.q >= 0) {
          if (z.yon) {   // y of the block before
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const float4 v = *reinterpret_cast<const float4*>(smem + L::kYAt + (sweeper_of(k, u) * 2 + ((z.q + 1) & 1)) * L::kY + pc * 16 + pq * 4);
              float x[4];
              Q::widen(z.xo[u], x);
              const float y[4] = {__builtin_fmaf(D4[k][u][0], x[0], v.x), __builtin_fmaf(D4[k][u][1], x[1], v.y), __builtin_fmaf(D4[k][u][2], x[2], v.z), __builtin_fmaf(D4[k][u][3], x[3], v.w)};
              if (quad_on[k][u]) *reinterpret_cast<raw*>(static_cast<T*>(p.y) + z.yo + quad_ch[k][u]) = Q::narrow(y);
            }
          }
          place(z, k, (z.q + 1) & 1);
          put_wraps(z, k, (z.q + 1) & 1);
          // what is swept now leaves in the next step
          const int im = rounds == 1 ? z.y.item : z.y.item / rounds, row = ((z.y.item - im * rounds) * NB + slot_of(k)) * R + pi, col = z.y.b * JC + pj;
          z.yon = lane_on && z.y.b < p.nblk && row < p.H && col < p.W && im < nimg;
          if (z.yon) {
            z.yo = ((int64_t)(img0 + im) * HW + cell_at(row, col)) * p.E;
#pragma unroll
            for (int u = 0; u < U; ++u) z.xo[u] = *reinterpret_cast<const raw*>(static_cast<const T*>(p.x) + z.yo + quad_ch[k][u]);
          }
          z.f.next(p.stride);
          fetch(z, k, z.f);
          z.w.next(p.stride);
          wraps(z, k);
          z.y.next(p.stride);
        }
        ++z.q;
      }
      block_barrier();
    }
    return;
  }
  // ------------------------------------------------------------------------------------------- sweeps
  const int slot = wave % NB, grp = wave / NB;
  const int ch = lane & 15, g = lane >> 4;
  const int e_raw = (wg * NG + grp) * 16 + ch, e = e_raw < p.E ? e_raw : p.E - 1;
  const bool group_on = (wg * NG + grp) * 16 < p.E;            // (uniform)
  float a2t[4], a2l[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = swap12(r) * 4 + g;                           // state_at(4 * g + r)
    a2t[r] = gate_rate<T>(p, p.AT, e * kN + n);
    a2l[r] = gate_rate<T>(p, p.AL, e * kN + n);
  }
  float hl[R][4];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) hl[i][r] = 0.f;
  struct Op { float4 v, bt, bl, c; } op[NC + kAhead];
  struct Gates { float aL[4], aT[4], u[4]; } ga[NC];
  const float* rec0 = smem + L::kRecAt + slot * 2 * L::kRec + g * 4;
  const float* chan0 = smem + L::kChanAt + wave * 2 * L::kChan + ch * 4;
  float* y0 = smem + L::kYAt + wave * 2 * L::kY + ch;
  const float4* above = reinterpret_cast<const float4*>(smem + L::kRowAt + wave * 2 * L::kRow) + lane;
  float4* below = reinterpret_cast<float4*>(smem + L::kRowAt + (wave + 1) * 2 * L::kRow) + lane;   // (of the next slot; the last slot has none)
  auto read = [&](int par, int c, Op& o) {
    const float4* lv = reinterpret_cast<const float4*>(chan0 + par * L::kChan);
    const float4* ls = reinterpret_cast<const float4*>(rec0 + par * L::kRec);
    o.v = lv[c * 16]; o.bt = ls[c * 12]; o.bl = ls[c * 12 + 4]; o.c = ls[c * 12 + 8];
  };
  block_barrier();
#pragma unroll
  for (int c = 0; c < kAhead; ++c) read(0, c, op[c]);
  block_barrier();
  Turn at{0, 0};
  int q = -slot;
  for (int t = 0; t < steps; ++t, ++q) {
    if (q >= 0) {
      const int par = q & 1;
      const int im = p.rounds == 1 ? at.item : at.item / p.rounds, round = at.item - im * p.rounds, b = at.b;
      const int band = round * NB + slot;
      if (b < p.nblk && band < p.nbands && im < nimg && group_on) {
        float4 tp[JC];
#pragma unroll
        for (int j = 0; j < JC; ++j) tp[j] = above[par * (L::kRow / 4) + j * 64];
        if (b == 0) {
#pragma unroll
          for (int i = 0; i < R; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) hl[i][r] = 0.f;
        }
        // gate offsets: log2 of the coefficient, and closed gates at the edges
        float kL[JC], kT[JC], kL0[JC], kT0[JC];
#pragma unroll
        for (int j = 0; j < JC; ++j) {
          const bool c0 = b == 0 && j == 0;
          kL[j] = c0 ? ninf : -1.f;
          kT[j] = c0 ? 0.f : -1.f;
          kL0[j] = band == 0 ? 0.f : kL[j];
          kT0[j] = band == 0 ? ninf : kT[j];
        }
        auto gates = [&](int c) {
          const int j = c / R, i = c % R;
          const float oL = i == 0 ? kL0[j] : kL[j], oT = i == 0 ? kT0[j] : kT[j];
          const float bt[4] = {op[c].bt.x, op[c].bt.y, op[c].bt.z, op[c].bt.w}, bl[4] = {op[c].bl.x, op[c].bl.y, op[c].bl.z, op[c].bl.w};
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            ga[c].aL[r] = fexp2(__builtin_fmaf(op[c].v.w, a2l[r], oL));
            ga[c].aT[r] = fexp2(__builtin_fmaf(op[c].v.z, a2t[r], oT));
            ga[c].u[r] = __builtin_fmaf(bl[r], op[c].v.y, bt[r] * op[c].v.x);
          }
        };
        gates(0);
        float hT[4], pr[4];
        float* yb = y0 + par * L::kY;
        // A cell's operands are read from LDS two cells ahead, its gates worked out one cell ahead
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          const int j = c / R, i = c % R;
          __builtin_amdgcn_sched_barrier(0);
          read(c + kAhead < NC ? par : par ^ 1, c + kAhead < NC ? c + kAhead : c + kAhead - NC, op[c + kAhead]);
          if (c + 1 < NC) gates(c + 1);
          if (i == 0) { hT[0] = tp[j].x; hT[1] = tp[j].y; hT[2] = tp[j].z; hT[3] = tp[j].w; }
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float h = __builtin_fmaf(ga[c].aL[r], hl[i][r], __builtin_fmaf(ga[c].aT[r], hT[r], ga[c].u[r]));
            hl[i][r] = h;
            hT[r] = h;
          }
          const float4 C = op[c].c;
          pr[c & 3] = __builtin_fmaf(C.w, hT[3], __builtin_fmaf(C.z, hT[2], __builtin_fmaf(C.y, hT[1], C.x * hT[0])));
          if ((c & 3) == 3) yb[(c - 3 + (g & 1) * 2 + (g >> 1)) * 16] = fold16(fold32(pr[0], pr[1]), fold32(pr[2], pr[3]));
          else if (c == NC - 1) { const float f = fold32(pr[0], pr[1]); yb[(c - 1 + (g >> 1)) * 16] = fold16(f, f); }   // (two cells are left)
          // the rows of the step before are in memory when this step ends
          if (c == R - 1 && slot == NB - 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          if (i == R - 1) {
            const float4 last = make_float4(hT[0], hT[1], hT[2], hT[3]);
            if (slot == NB - 1) {
              const int col = b * JC + j;
              if (col < p.W && band + 1 < p.nbands)
                reinterpret_cast<float4*>(p.wrap)[((((int64_t)round * p.B + img0 + im) * groups16 + wg * NG + grp) * p.W + col) * 64 + lane] = last;
            } else {
              below[par * (L::kRow / 4) + j * 64] = last;
            }
          }
        }
#pragma unroll
        for (int c = 0; c < kAhead; ++c) op[c] = op[NC + c];
      } else {   // nothing to sweep here, but perhaps in the next block
#pragma unroll
        for (int c = 0; c < kAhead; ++c) read(par ^ 1, c, op[c]);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      at.next(p.stride);
    }
    block_barrier();
  }
}

template <typename T, int R, int NB, bool PACKED>
int launch_packed(const Plan& plan, const Args& a, hipStream_t st) {
  constexpr size_t lds = Lds<R, NB>::kBytes;
  static_assert(lds <= 160 * 1024, "a compute unit has 160 KB");
  static std::atomic<uint64_t> seen{0};
  if (!allow_dynamic_lds(reinterpret_cast<const void*>(&m2d_fwd_rows_kernel<T, R, NB, PACKED>), lds, seen)) return (int)hipErrorInvalidValue;
  hipLaunchKernelGGL((m2d_fwd_rows_kernel<T, R, NB, PACKED>), dim3((unsigned)plan.workgroups), dim3((kSweepers + kStagers) * 64), lds, st, a);
  return (int)hipGetLastError();
}
template <typename T, int R, int NB>
int launch_as(const Plan& plan, const Args& a, hipStream_t st) {
  return a.rec ? launch_packed<T, R, NB, true>(plan, a, st) : launch_packed<T, R, NB, false>(plan, a, st);
}
template <typename T, int R>
int launch_rows(const Plan& plan, const Args& a, hipStream_t st) {
  switch (plan.slots) {
    case 1: return launch_as<T, R, 1>(plan, a, st);
    case 2: return launch_as<T, R, 2>(plan, a, st);
    case 4: return launch_as<T, R, 4>(plan, a, st);
    default: return launch_as<T, R, 8>(plan, a, st);
  }
}
template <typename T>
int launch(const Plan& plan, const Args& a, hipStream_t st) {
  switch (plan.rows) {
    case 6: return launch_rows<T, 6>(plan, a, st);
    case 7: return launch_rows<T, 7>(plan, a, st);
    default: return launch_rows<T, 8>(plan, a, st);
  }
}

}  // namespace

Plan make_plan(int B, int H, int W, int E, int compute_units) {
  Plan best;
  if (E % 4) return best;
  const int groups16 = (E + 15) / 16;
  for (int rows = 6; rows <= 8; ++rows)
    for (int slots = 1; slots <= 8; slots *= 2) {
      Plan c;
      c.rows = rows;
      c.slots = slots;
      c.nbands = (H + rows - 1) / rows;
      c.nblk = (W + kJC - 1) / kJC;
      c.rounds = (c.nbands + slots - 1) / slots;
      // a row that the last slot stores is read two steps before the first slot of the next round comes to it, and one step behind the store's wait
      c.stride = c.rounds > 1 && c.nblk < slots + 4 ? slots + 4 : c.nblk;
      const int ng = kSweepers / slots;
      c.groups = (groups16 + ng - 1) / ng;
      // images that a workgroup sweeps one after the other: one start for all of them, and one round of workgroups
      const int64_t sets = (int64_t)B * c.groups;
      c.images = (int)((sets + compute_units - 1) / compute_units);
      if (c.images > B) c.images = B;
      c.workgroups = (B + c.images - 1) / c.images * c.groups;
      c.wrap_bytes = (size_t)(c.rounds - 1) * B * groups16 * W * 64 * sizeof(float) * 4;
      const int64_t turns = ((int64_t)c.workgroups + compute_units - 1) / compute_units;
      c.cells = turns * ((int64_t)c.images * c.rounds * c.stride + slots + 1) * rows * kJC;
      if (best.rows == 0 || c.cells < best.cells) best = c;
    }
  return best;
}

int launch_fwd(const Plan& plan, Args a, bool bf16, hipStream_t stream) {
  a.nbands = plan.nbands; a.nblk = plan.nblk; a.rounds = plan.rounds; a.stride = plan.stride; a.groups = plan.groups; a.images = plan.images;
  return bf16 ? launch<bf16_t>(plan, a, stream) : launch<float>(plan, a, stream);
}

}  // namespace m2drows
