// Scan kernels for few images: the 16 states of a channel split over the 4 lane groups of a wave (included by
// m2dscan.hip, inside its namespace; m2d_fwd_split_kernel and m2d_bwd_split_kernel).
//
// A sweep of few images takes as long as ONE wave needs for its chain of steps: there are fewer waves than the device
// could hold.  So a wave does as little as possible per step: lane = (state group g, row r), 4 states of one channel per
// lane, and the first NW waves of a workgroup (one channel each) only sweep: they read operands from LDS one step
// ahead of their use and drop every result in LDS, without positions, addresses, predicates, global stores or waits for memory
// (one snapshot access per block of 4 steps aside).  Four more waves (one to a SIMD beside the sweeping ones) do the rest, each its own part:
//   waves 0..2  B_T, B_L, C of the blocks to come (SplitBC); in the forward also x, deltaT, deltaL, a tensor each, wave 0 the band's last rows
//               out and the progress count, waves 1 and 2 y (the 4 groups' shares of a cell added up); in the backward a tensor's sums over the
//               channels of the workgroup each, and one each of d_deltaT, d_deltaL, d_x
//   wave 3      the rows' constants, the link's wait and the neighbouring band's rows in; in the backward also x, deltaT,
//               deltaL, dy, the upper boundary rows, and the band's own rows out
// What bounds a block is the longer of two chains of instructions, a sweeping wave's (184 vector and 32 LDS instructions for 4 forward
// steps, about 1500 clocks alone on its SIMD) and a staging wave's, so the work above is shared out to be even and a staging wave works out as few
// places as it can.  A store takes several times as long to be acknowledged as a block takes, and the counter that a wave waits on
// retires in order: every block issues the same operations whatever lanes they are for, so that a wave knows how many of them may still be under way
// (split_landed), and rows of a neighbour, which are fetched at the last moment, come in through a wave that stores nothing before them.
// Against sweeping waves that also stage, forward keeping snapshots / backward: 1x256x256x64 fp32 0.298 / 0.683 -> 0.196 / 0.480 ms (0.183 / 0.382 with the wider stores),
// 1x256x256x62 (rows of no whole chunks) 0.476 / 1.157 -> 0.226 / 0.572, 4x128x128x64 bf16 0.183 / 0.442 -> 0.111 / 0.315.
// Memory formats and schedules are those of the whole-state kernels, so either pass may use either layout.
constexpr int kSplitWaves = 8;       // sweeping waves (channels) per workgroup
constexpr int kSplitHalfWaves = 4;   // ... where workgroups of 8 would leave compute units idle
constexpr int kSplitStagers = 4;

// the value a tensor of type T would hold
__device__ __forceinline__ float as_stored(float v, const float*) { return v; }
__device__ __forceinline__ float as_stored(float v, const bf16_t*) { return bf16_bits_to_f32(f32_to_bf16_bits(v)); }

// A * log2 e and D from the caller's tensors: of type T, or the parameters as the module holds them (fp32 A_log and D:
// A = -exp(A_log), and both are rounded to T, which is what the reference's casts to x.dtype do, wavefront_cuda.py:72-73,
// 90-91, 332).
template <typename T>
__device__ __forceinline__ float gate_rate(const ScanParams& p, const void* A, int i) {
  return (p.raw ? as_stored(-expf(static_cast<const float*>(A)[i]), static_cast<const T*>(nullptr)) : IO<T>::ld(static_cast<const T*>(A) + i)) * kLog2e;
}
template <typename T>
__device__ __forceinline__ float skip_gain(const ScanParams& p, int e) {
  return p.raw ? as_stored(static_cast<const float*>(p.D)[e], static_cast<const T*>(nullptr)) : IO<T>::ld(static_cast<const T*>(p.D) + e);
}
// The set-up launch (m2d_prep_kernel) is for kernels whose lanes hold all states of a channel, and for progress counts.  A lane
// here holds 4 states of a channel or two, so a forward of one stream per image works its own out and saves the launch and the gap
// behind it (4.7 us); where it keeps snapshots, the workgroups of the first image leave the area as a backward will want it.
template <int MODE>
constexpr bool split_owns_setup() { return MODE != kModeSliced; }
__device__ float m2d_zero_page[kZeroFloats];     // the page of zeros of such a forward: never written

// ------------------------------------------------------------------------------ operands in LDS
// A block of kCK = 4 steps:
//   B_T, B_L, C  [tensor][step] sets of 1 KB (and 16 bytes), 64 bytes (4 state groups) for each of the 16 lane rows.  Four consecutive lanes of a wave-wide
//                copy fetch the 64 bytes of one cell; group g of row r is at place g ^ (r >> 2), so that the 16 rows that a
//                sweeping wave reads together are in different banks
//   constants    [step][lane row] 16 bytes: offT, offL, cT, cL
//   TOP          the last row of the band above, [4 channels][step][channel][state group] 16 bytes
//   BOT          (backward) the muT of the first row of the band below, likewise
//   x, deltaT, deltaL[, dy]: rows of whole 16-byte chunks (SX) as chunks of the tensors' type, [tensor][chunk][step][lane row];
//                otherwise single values widened to fp32, [tensor][channel][step][lane row]
// Rows and cells off the grid are copied from a page of zeros.
template <typename T, int NT, int CW, bool BWD, bool SX>
struct SplitStage {
  static constexpr int kElem = 16 / (int)sizeof(T);
  static constexpr int kChunks = CW > kElem ? CW / kElem : 1;
  static constexpr int kSet = kCK * kHB * 16;        // 1 KB: what a wave-wide copy fills
  static constexpr int kStep = kHB * 16;             // constants, boundary rows and chunks: bytes per step
  static constexpr int kG4 = CW / 4;
  static constexpr int kBCStep = kSet + 16, kBCTensor = kCK * kBCStep;   // (16 bytes more: split_raw_widen writes four steps at once)
  static constexpr int kConst = 3 * kBCTensor;
  static constexpr int kTop = kConst + kSet;
  static constexpr int kBot = kTop + kG4 * kSet;
  static constexpr int kX = kBot + (BWD ? kG4 * kSet : 0);
  static constexpr int kXTensor = SX ? kChunks * kSet : CW * kCK * kHB * 4;   // bytes per tensor
  static constexpr int kXStep = SX ? kStep : kHB * 4;
  static constexpr int kBytes = kX + NT * kXTensor;                           // one buffer
  static_assert(kCK == 4 && kHB == 16 && CW % 4 == 0, "a set is one wave-wide copy");
  static __device__ __forceinline__ uint32_t bc_off(int tensor, int g, int r) { return (uint32_t)(tensor * kBCTensor + r * 64 + (g ^ (r >> 2)) * 16); }
  static __device__ __forceinline__ uint32_t row_off(int base, int ch, int g) { return (uint32_t)(base + (ch / 4) * kSet + (ch % 4) * 64 + g * 16); }
  // channel ch of the workgroup; e_wg0: its first channel (SX: 4 channels of a 16-bit tensor are a half of their chunk)
  static __device__ __forceinline__ uint32_t x_off(int ch, int r, int e_wg0) {
    if constexpr (SX) {
      const int c = ch + (CW < kElem ? e_wg0 & (kElem - 1) : 0);
      return (uint32_t)(kX + (c / kElem) * kSet + r * 16 + (c % kElem) * (int)sizeof(T));
    } else {
      return (uint32_t)(kX + (ch * kCK * kHB + r) * 4);
    }
  }
};
template <typename T, bool SX>
__device__ __forceinline__ float split_x(const char* at) {   // one value of x, deltaT, deltaL or dy
  if constexpr (SX) return IO<T>::ld(reinterpret_cast<const T*>(at)); else return *reinterpret_cast<const float*>(at);
}

// A wave-wide copy of 16 bytes a lane to a place in LDS that the whole wave computed alike (bytes from the start of the kernel's one array,
// which is where its LDS starts)
template <bool DEVICE_SCOPE>
__device__ __forceinline__ void split_fill16(const void* src, uint32_t at) { lds_fill16_at<DEVICE_SCOPE>(src, __builtin_amdgcn_readfirstlane(at)); }

// EC values of neighbouring channels (two: they are in one chunk)
template <typename T, bool SX, int EC>
__device__ __forceinline__ void split_xs(const char* at, float (&v)[EC]) {
  if constexpr (EC == 1) v[0] = split_x<T, SX>(at);
  else if constexpr (sizeof(T) == 4) { const float2 q = *reinterpret_cast<const float2*>(at); v[0] = q.x; v[1] = q.y; }
  else { const uint32_t q = *reinterpret_cast<const uint32_t*>(at); v[0] = __uint_as_float(q << 16); v[1] = __uint_as_float(q & 0xffff0000u); }
}

// Where a lane's (step, row) of a block is.  The linked sweep stays inside one band, and its columns count from the start of the
// band's window (below 0 and from W on: off the grid); otherwise the stream wraps from band to band.
template <bool SLICED>
struct Track {
  int bnd, col;
  int cell;      // of its image; means something on the grid only
  int limit;     // linked sweep: columns of the lane's row (0: not a row of this band); else the bands that have the row
  // at: steps from the start of the window to the lane's step, in lane row `row`
  __device__ __forceinline__ void start(const ScanParams& p, int band, int at, int row) {
    const int rbands = row_bands(p, row);
    if constexpr (SLICED) {
      bnd = band;
      col = at - row;
      limit = band < rbands ? p.W : 0;
    } else {
      const Pos q = pos_of(p, at - row);
      bnd = q.bnd;
      col = q.col;
      limit = rbands;
    }
    cell = cell_of(p, bnd, row, col);
  }
  __device__ __forceinline__ bool on(const ScanParams& p) const {
    if constexpr (SLICED) return (unsigned)col < (unsigned)limit; else return (unsigned)bnd < (unsigned)limit && col < p.W;
  }
  // `steps` further on (|steps| at most a block)
  __device__ __forceinline__ Track moved(const ScanParams& p, int steps) const {
    Track t = *this;
    t.col += steps;
    t.cell += p.flip ? -steps : steps;
    if constexpr (!SLICED) {
      const int wrap = p.rb * p.W - p.S;
      if (t.col >= p.S) { t.col -= p.S; t.bnd += 1; t.cell += p.flip ? -wrap : wrap; }
      else if (t.col < 0) { t.col += p.S; t.bnd -= 1; t.cell -= p.flip ? -wrap : wrap; }
    }
    return t;
  }
};
// Boundary row record of column t.col in row buffer `at` (of the band the lane is in, moved by `bands`); base: the record of channel and state group at band 0, column 0
template <bool SLICED>
__device__ __forceinline__ char* row_record(const ScanParams& p, char* base, const Track<SLICED>& t, int bands, int64_t band_bytes) {
  const uint32_t rec = (uint32_t)p.E * (uint32_t)(kN * sizeof(float));
  if constexpr (SLICED) return base + (uint64_t)(uint32_t)t.col * rec;   // (the band is in the base)
  else return base + (int64_t)(t.bnd + bands) * band_bytes + (uint64_t)(uint32_t)t.col * rec;
}
// All but the N youngest vector-memory operations of the wave have completed (see staging_landed_behind; N up to 63)
template <int N>
__device__ __forceinline__ void split_landed() {
  static_assert(N >= 0 && N < 64, "six bits of the counter");
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
  asm volatile("" ::: "memory");
}
// Stores by the lanes for which `live` holds, always issued, so that the number of operations under way is known without looking: the
// compiler would branch around a store that no lane makes.
__device__ __forceinline__ void split_store4(void* dst, float v, bool live) {
  uint64_t saved;
  asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dword %1, %2, off\n\ts_mov_b64 exec, %0" : "=&s"(saved) : "v"(dst), "v"(v), "s"(__ballot(live)) : "memory", "scc");
}
__device__ __forceinline__ void split_store(float* dst, float v, bool live) { split_store4(dst, v, live); }
__device__ __forceinline__ void split_store(bf16_t* dst, float v, bool live) {
  uint64_t saved;
  const uint32_t bits = f32_to_bf16_bits(v);
  asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_short %1, %2, off\n\ts_mov_b64 exec, %0" : "=&s"(saved) : "v"(dst), "v"(bits), "s"(__ballot(live)) : "memory", "scc");
}
// two neighbouring values
__device__ __forceinline__ void split_store_pair(float* dst, float a, float b, bool live) {
  uint64_t saved;
  typedef float v2f_t __attribute__((ext_vector_type(2)));
  const v2f_t w = {a, b};
  asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx2 %1, %2, off\n\ts_mov_b64 exec, %0" : "=&s"(saved) : "v"(dst), "v"(w), "s"(__ballot(live)) : "memory", "scc");
}
__device__ __forceinline__ void split_store_pair(bf16_t* dst, float a, float b, bool live) { split_store4(dst, __uint_as_float(pack_bf16(a, b)), live); }
// four neighbouring values
__device__ __forceinline__ void split_store_quad(float* dst, float4 v, bool live) {
  uint64_t saved;
  const v4f_t w = {v.x, v.y, v.z, v.w};
  asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, off\n\ts_mov_b64 exec, %0\n\ts_nop 0" : "=&s"(saved) : "v"(dst), "v"(w), "s"(__ballot(live)) : "memory", "scc");
}
__device__ __forceinline__ void split_store_quad(bf16_t* dst, float4 v, bool live) {
  uint64_t saved;
  const uint64_t w = (uint64_t)f32_to_bf16_bits(v.x) | (uint64_t)f32_to_bf16_bits(v.y) << 16 | (uint64_t)f32_to_bf16_bits(v.z) << 32 | (uint64_t)f32_to_bf16_bits(v.w) << 48;
  asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx2 %1, %2, off\n\ts_mov_b64 exec, %0" : "=&s"(saved) : "v"(dst), "v"(w), "s"(__ballot(live)) : "memory", "scc");
}
// 16 bytes of a boundary row (device scope: see store_row_device_scope, also for the wait states behind it)
template <bool DEVICE_SCOPE>
__device__ __forceinline__ void split_store_row(void* dst, float4 row, bool live) {
  uint64_t saved;
  const v4f_t w = {row.x, row.y, row.z, row.w};
  if constexpr (DEVICE_SCOPE)
    asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, off sc1\n\ts_mov_b64 exec, %0\n\ts_nop 0" : "=&s"(saved) : "v"(dst), "v"(w), "s"(__ballot(live)) : "memory", "scc");
  else
    asm volatile("s_and_saveexec_b64 %0, %3\n\tglobal_store_dwordx4 %1, %2, off\n\ts_mov_b64 exec, %0\n\ts_nop 0" : "=&s"(saved) : "v"(dst), "v"(w), "s"(__ballot(live)) : "memory", "scc");
}
// (both below 2^24: the full-rate multiplier)
__device__ __forceinline__ uint32_t cell_bytes_off(int cell, uint32_t bytes) { return __umul24((uint32_t)cell, bytes); }

// B_T, B_L, C of a block, as fp32 in fold order from the packed records (192 bytes a cell), or in natural order from the caller's
// fp32 tensors (64 bytes a cell): 12 copies, 4 by each of the waves 0, 1, 2 -- the tensors at step sw, and tensor sw at step 3, so that a wave works
// out two places and not four.  A lane copies a state group (SplitStage) of lane row lane >> 2.
template <bool SLICED>
struct SplitBC {
  Track<SLICED> own, last;         // steps sw and 3 of the block to be fetched next
  const char *at0, *at1, *at2, *mine;   // (uniform) image b's first cell of each tensor, and of tensor sw
  uint32_t cell, group;            // bytes per cell; byte offset of the lane's state group
  __device__ __forceinline__ void start(const ScanParams& p, int band, int step, int sw, int lane, bool direct, int64_t first_cell) {
    const int64_t skip = first_cell * cell;
    at0 = (direct ? static_cast<const char*>(p.bcd[0]) : reinterpret_cast<const char*>(p.bt)) + skip;
    at1 = (direct ? static_cast<const char*>(p.bcd[1]) : reinterpret_cast<const char*>(p.bt) + kN * 4) + skip;
    at2 = (direct ? static_cast<const char*>(p.bcd[2]) : reinterpret_cast<const char*>(p.bt) + 2 * kN * 4) + skip;
    mine = sw == 0 ? at0 : (sw == 1 ? at1 : at2);
    own.start(p, band, step + (sw < 3 ? sw : 0), lane >> 2);
    last.start(p, band, step + 3, lane >> 2);
    group = ((lane & 3) ^ (lane >> 4)) * 16;
  }
  template <typename SG>
  __device__ __forceinline__ void copy(const ScanParams& p, uint32_t buf, int sw, int steps) {
    const char* zeros = reinterpret_cast<const char*>(p.zeros);
    const bool on = own.on(p), on3 = last.on(p);
    const uint32_t off = cell_bytes_off(own.cell, cell) + group, off3 = cell_bytes_off(last.cell, cell) + group;
    split_fill16<false>(on ? at0 + off : zeros, buf + sw * SG::kBCStep);
    split_fill16<false>(on ? at1 + off : zeros, buf + SG::kBCTensor + sw * SG::kBCStep);
    split_fill16<false>(on ? at2 + off : zeros, buf + 2 * SG::kBCTensor + sw * SG::kBCStep);
    split_fill16<false>(on3 ? mine + off3 : zeros, buf + sw * SG::kBCTensor + 3 * SG::kBCStep);
    own = own.moved(p, steps);
    last = last.moved(p, steps);
  }
};
// ... or from the caller's bf16 tensor: copied as it is (32 bytes a cell, the lane's (row, step) = (lane >> 2, lane & 3)) into the
// sets of the steps 0 and 1, and spread over the tensor's sets as fp32 when it has landed, by the same wave.
template <typename SG>
__device__ __forceinline__ void split_raw_copy(const char* src, uint32_t sets) {
  split_fill16<false>(src, sets);
  split_fill16<false>(src + 16, sets + SG::kBCStep);
}
template <typename SG>
__device__ __forceinline__ void split_raw_widen(char* sets, int lane) {
  const uint4 lo = *reinterpret_cast<const uint4*>(sets + lane * 16), hi = *reinterpret_cast<const uint4*>(sets + SG::kBCStep + lane * 16);
  uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};   // word i: states 2i, 2i + 1
  // every lane's words are in registers before any lane's values take their place
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3]), "+v"(w[4]), "+v"(w[5]), "+v"(w[6]), "+v"(w[7]) : : "memory");
  const int r = lane >> 2, k = lane & 3;
  char* dst = sets + k * SG::kBCStep;
#pragma unroll
  for (int g = 0; g < 4; ++g) {   // the states g, 8 + g, 4 + g, 12 + g (sinv)
    float v[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = sinv<true>(4 * g + i);
      v[i] = __uint_as_float((n & 1) ? w[n >> 1] & 0xffff0000u : w[n >> 1] << 16);
    }
    *reinterpret_cast<float4*>(dst + SG::bc_off(0, g, r)) = make_float4(v[0], v[1], v[2], v[3]);
  }
}
// The constants of the lane's (step, row)
template <typename SG>
__device__ __forceinline__ void split_consts(const LaneK& K, int col, char* buf, int lane) {
  const bool col0 = col == 0;
  *reinterpret_cast<float4*>(buf + SG::kConst + lane * 16) =
      make_float4(col0 ? K.oT0 : K.oT, col0 ? -__builtin_huge_valf() : K.oL, col0 ? K.cT0 : K.cT, col0 ? K.cL0 : K.cL);
}
// One of x, deltaT, deltaL, dy of a block where rows are whole chunks
template <typename T, typename SG>
__device__ __forceinline__ void split_x_copy(const ScanParams& p, const char* img, uint32_t cell, bool ok, int e_wg0, uint32_t tensor) {
  const int e_chunk = e_wg0 & ~(SG::kElem - 1);   // (a workgroup of fewer channels than a chunk copies the chunk they are in)
#pragma unroll
  for (int c = 0; c < SG::kChunks; ++c) {
    const int ch = e_chunk + c * SG::kElem;
    const uint32_t off = cell_bytes_off((int)cell, (uint32_t)p.E * (uint32_t)sizeof(T)) + (uint32_t)ch * (uint32_t)sizeof(T);
    split_fill16<false>(ok && ch < p.E ? img + off : reinterpret_cast<const char*>(p.zeros), tensor + c * SG::kSet);
  }
}
// ... and where they are not: value by value, through registers, by wave sw for its channels sw, sw + 4 of the workgroup.  The registers take the values as
// they are in memory, and 16-bit ones are widened when they are put in place, a block later: widened where they are fetched, a wave waited there for its loads
// and for every store before them (bf16, forward keeping snapshots / backward: 3x64x90x292 156 / 420 -> 125 / 363 us, 2x100x26x100 72 / 167 -> 61 / 144).
template <typename T, int NT, int CW>
struct SplitVals { T v[CW / kSplitStagers][NT]; };
template <typename T, int NT, int CW>
__device__ __forceinline__ void split_vals_fetch(const ScanParams& p, const char* const (&img)[4], uint32_t cell, bool ok, int e_wg0, int sw, SplitVals<T, NT, CW>& o) {
#pragma unroll
  for (int j = 0; j < CW / kSplitStagers; ++j) {
    const int e = e_wg0 + sw + kSplitStagers * j;
    const uint32_t off = (cell * (uint32_t)p.E + (uint32_t)e) * (uint32_t)sizeof(T);
    const bool live = ok && e < p.E;
#pragma unroll
    for (int t = 0; t < NT; ++t) o.v[j][t] = live ? *reinterpret_cast<const T*>(img[t] + off) : T{};
  }
}
template <typename T, int NT, int CW, typename SG>
__device__ __forceinline__ void split_vals_put(const SplitVals<T, NT, CW>& o, char* buf, int sw, int lane) {
#pragma unroll
  for (int j = 0; j < CW / kSplitStagers; ++j)
#pragma unroll
    for (int t = 0; t < NT; ++t)
      *reinterpret_cast<float*>(buf + SG::kX + t * SG::kXTensor + ((sw + kSplitStagers * j) * kCK * kHB + lane) * 4) = IO<T>::ld(&o.v[j][t]);
}

// ---------------------------------------------------------------------------------------- forward
// One barrier per block, before the block's last step (its operands are in registers by then, so the block's buffer can be
// handed over): between two barriers the sweeping waves run the last step of a block and the first three of the next,
// whose results make a window: window q holds those of the steps 4q - 1 .. 4q + 2.  While window q is filled, the staging
// waves send window q - 1 to memory and fetch the operands of block q + 3 (boundary rows: of block q + 1): a block takes
// less time than a fetch from memory.
template <typename T, int NW, bool SX, int EC = 1>
struct SplitFwdLds {
  static constexpr int CW = NW * EC;
  using SG = SplitStage<T, 3, CW, false, SX>;
  static constexpr int kBufs = 4;
  // the shares of y of one channel at one step: [row][state group] floats (a few bytes more: lanes that read together meet different banks)
  static constexpr int kYCh = kHB * 16 + (EC == 1 ? 32 : 16);
  static constexpr int kYStep = CW * kYCh;
  static constexpr int kYBytes = kCK * kYStep;             // one window
  static constexpr int kRStep = CW * 64;                   // the band's last row at one step: [channel][state group] float4s
  static constexpr int kRBytes = kCK * kRStep;
  static constexpr int kY = kBufs * SG::kBytes, kR = kY + 2 * kYBytes, kFlag = kR + 2 * kRBytes, kBytes = kFlag + 16;   // flag: the wave that waits has given up
};
template <typename T, bool CKPT, bool WRITE_Y, bool SX, int MODE, int NW = kSplitWaves, int EC = 1, bool HALF = false>
__global__ __launch_bounds__((NW + kSplitStagers) * 64) void m2d_fwd_split_kernel(const ScanParams pin) {
  static_assert(MODE != kModeStacked, "stacked images are many: they never need the split");
  constexpr bool SLICED = MODE == kModeSliced;
  constexpr bool OWN_SETUP = split_owns_setup<MODE>();
  constexpr bool WIDEN = sizeof(T) == 2;
  constexpr int CW = NW * EC;
  static_assert(EC == 1 || (EC == 2 && SX && NW == kSplitWaves && !SLICED), "two channels a wave: rows of whole chunks, one stream per image");
  static_assert(!HALF || (CKPT && !SLICED), "snapshots every 2 steps: kept by a forward of one stream per image");
  const ScanParams& p = pin;
  __builtin_assume(p.stacked == 0);
  __builtin_assume(p.rb == kRB);
  __builtin_assume(p.S >= kHB + kCK - 1);
  using L = SplitFwdLds<T, NW, SX, EC>;
  using SG = typename L::SG;
  extern __shared__ float4 smem[];
  char* lds = reinterpret_cast<char*>(smem);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lb = 0, turn = 0;
  if constexpr (SLICED) { if (!linked_place(p, turn, lb)) return; } else lb = logical_block(p.nwg);
  int m_lo = 0, m_hi = p.nblk;
  int my_band = 0;
  LinkT<(NW + 3) * 64> link;
  if constexpr (SLICED) {
    const int per = p.B * p.bpb;
    my_band = turn;
    m_lo = my_band * p.sl_nbb;
    m_hi = m_lo + p.sl_nbb;
    link.mine = p.prog + ((int64_t)my_band * per + lb) * kLinkStride;
    link.dep = my_band > 0 ? link.mine - per * kLinkStride : nullptr;
    link.err = p.link_err;
    link.rig(p, my_band);
  }
  const int b = lb / p.bpb;
  const int e_wg0 = (lb % p.bpb) * CW;
  // fp32 records straight from the caller's tensors hold the states in natural order
  const bool direct = (WIDEN || !CKPT) && p.bc_direct != 0;   // (uniform)

  if (wave < NW) {
    // ------------------------------------------------------------------------------ sweeps
    const int g = lane >> kHBShift, r = lane & (kHB - 1);   // state group, lane row
    const int ch = wave * EC;                               // the wave's (first) channel
    const bool ch_ok = e_wg0 + ch < p.E;                    // (uniform) idle waves still take part in the barriers (EC = 2: E is even)
    const int e0 = ch_ok ? e_wg0 + ch : p.E - EC;
    float a2t[EC][4], a2l[EC][4], dskg[EC];
#pragma unroll
    for (int c = 0; c < EC; ++c) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int n = (!WIDEN && direct) ? 4 * g + w : (w == 1 ? 2 : (w == 2 ? 1 : w)) * 4 + g;   // the state that register w meets: 4g + w, or sinv(4g + w)
        a2t[c][w] = OWN_SETUP ? gate_rate<T>(p, p.AT, (e0 + c) * kN + n) : p.A2T[(e0 + c) * kN + n];
        a2l[c][w] = OWN_SETUP ? gate_rate<T>(p, p.AL, (e0 + c) * kN + n) : p.A2L[(e0 + c) * kN + n];
      }
      dskg[c] = g == 0 ? (OWN_SETUP ? skip_gain<T>(p, e0 + c) : p.Df[e0 + c]) : 0.f;   // (x * D is in the share of group 0)
    }
    static_assert(sinv<true>(1) == 8 && sinv<true>(6) == 5 && sinv<true>(15) == 15, "fold order");
    if constexpr (OWN_SETUP && CKPT) {   // the area that m2d_prep_kernel fills for others: [zeros][A2T][A2L][D]
      if (b == 0 && ch_ok && r == 0) {
        float* A2T = const_cast<float*>(p.A2T);
        float* A2L = const_cast<float*>(p.A2L);
#pragma unroll
        for (int c = 0; c < EC; ++c) {
#pragma unroll
          for (int w = 0; w < 4; ++w) {   // (a forward that keeps snapshots has the states in fold order)
            const int n = (e0 + c) * kN + (w == 1 ? 2 : (w == 2 ? 1 : w)) * 4 + g;
            A2T[n] = a2t[c][w];
            A2L[n] = a2l[c][w];
          }
          if (g == 0) const_cast<float*>(p.Df)[e0 + c] = dskg[c];
        }
      }
      static_assert(kZeroFloats == 64, "a lane each");
      if (b == 0 && e_wg0 == 0 && wave == 0) const_cast<float*>(p.A2T)[lane - kZeroFloats] = 0.f;
    }
    const float g1 = r == 0 ? 1.f : 0.f;                    // the ghost's T input coefficient
    // a grid row reads its own B_T; the ghost (lane 0) the row above as its B_T, and zeros as its B_L and C
    const uint32_t bt_off = r == 0 ? SG::row_off(SG::kTop, ch, g) : SG::bc_off(0, g, r);
    const uint32_t bt_ch = r == 0 ? 64 : 0;                 // (EC = 2) ... of the second channel
    const uint32_t bt_step = r == 0 ? SG::kStep : SG::kBCStep;
    const uint32_t bl_off = SG::bc_off(1, g, r);
    const uint32_t k_off = SG::kConst + r * 16;
    const uint32_t x_off = SG::x_off(ch, r, e_wg0);
    char* yw = lds + L::kY + ch * L::kYCh + r * 16 + g * 4;
    char* rw = lds + L::kR + ch * 64 + g * 16;
    const bool last_row = r == kRB && p.nbands > 1;         // the band's last row: the next band's ghost will replay it
    typename Snap<T>::quad* ckp = nullptr;
    if constexpr (CKPT) ckp = snapshot_at<T>(p, b, HALF ? 2 * m_lo : m_lo, e0, p.ck_nblk) + snap_lane(r) + snap_quad(g);
    const int64_t ck_step = (int64_t)p.E * (kN / 4 * kHB);  // (from one snapshot to the next)
    settle_loads();

    struct Ops { float4 kk, bt[EC], bl, cc; float x[EC], dt[EC], dl[EC]; };
    auto fetch = [&](uint32_t buf, int k, Ops& o) {
      const char* at = lds + buf;
      o.kk = *reinterpret_cast<const float4*>(at + k_off + k * SG::kStep);
      split_xs<T, SX, EC>(at + x_off + SG::kXTensor + k * SG::kXStep, o.dt);
      split_xs<T, SX, EC>(at + x_off + 2 * SG::kXTensor + k * SG::kXStep, o.dl);
      split_xs<T, SX, EC>(at + x_off + k * SG::kXStep, o.x);
      o.bl = *reinterpret_cast<const float4*>(at + bl_off + k * SG::kBCStep);
#pragma unroll
      for (int c = 0; c < EC; ++c) o.bt[c] = *reinterpret_cast<const float4*>(at + bt_off + c * bt_ch + k * bt_step);
      if constexpr (WRITE_Y) o.cc = *reinterpret_cast<const float4*>(at + bl_off + SG::kBCTensor + k * SG::kBCStep);
    };
    float h[EC][4];
#pragma unroll
    for (int c = 0; c < EC; ++c)
#pragma unroll
      for (int w = 0; w < 4; ++w) h[c][w] = 0.f;
    auto step = [&](const Ops& o, int k, int par) {   // par: the window that takes the results
#pragma unroll
      for (int c = 0; c < EC; ++c) {
        const float sT = __builtin_fmaf(o.kk.z * o.dt[c], o.x[c], g1);
        const float sL = o.kk.w * o.dl[c] * o.x[c];
        // gates before chains (see m2d_fwd_kernel: no DPP multiply-add right behind the v_exp that makes its gate)
        float aT[4], aL[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) aT[w] = fexp2(__builtin_fmaf(o.dt[c], a2t[c][w], o.kk.x));
#pragma unroll
        for (int w = 0; w < 4; ++w) aL[w] = fexp2(__builtin_fmaf(o.dl[c], a2l[c][w], o.kk.y));
        pin4(aT); pin4(aL);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (CKPT) {   // the lane's states as they are before this step
          if ((k == 0 || (HALF && k == 2)) && ch_ok) Snap<T>::store(ckp + (HALF && k == 2 ? ck_step : 0) + c * (kN / 4 * kHB), h[c][0], h[c][1], h[c][2], h[c][3]);
        }
        const float bq[4] = {o.bt[c].x, o.bt[c].y, o.bt[c].z, o.bt[c].w}, lq[4] = {o.bl.x, o.bl.y, o.bl.z, o.bl.w};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          float u = sL * lq[w];
          u = __builtin_fmaf(sT, bq[w], u);
          u = fma_row_below(aT[w], h[c][w], u);
          h[c][w] = __builtin_fmaf(aL[w], h[c][w], u);
        }
        const int slot = (k + 1) & (kCK - 1);
        if (last_row) *reinterpret_cast<float4*>(rw + c * 64 + par * L::kRBytes + slot * L::kRStep) = make_float4(h[c][0], h[c][1], h[c][2], h[c][3]);
        if constexpr (WRITE_Y) {
          const float y0 = __builtin_fmaf(h[c][2], o.cc.z, __builtin_fmaf(h[c][0], o.cc.x, o.x[c] * dskg[c]));
          const float y1 = __builtin_fmaf(h[c][3], o.cc.w, h[c][1] * o.cc.y);
          *reinterpret_cast<float*>(yw + c * L::kYCh + par * L::kYBytes + slot * L::kYStep) = y0 + y1;
        }
      }
    };
    __syncthreads();   // the first block is in place
    Ops opsA, opsB;
    uint32_t buf = 0;
    int par = 0;
    fetch(buf, 0, opsA);
    for (int m = m_lo; m < m_hi; ++m) {
      const uint32_t next = buf == (L::kBufs - 1) * SG::kBytes ? 0 : buf + SG::kBytes;
      fetch(buf, 1, opsB);
      step(opsA, 0, par);
      fetch(buf, 2, opsA);
      step(opsB, 1, par);
      if constexpr (EC == 2) lead_if_younger<NW>(wave, false);
      fetch(buf, 3, opsB);
      step(opsA, 2, par);
      __syncthreads();
      if constexpr (EC == 2) lead_if_younger<NW>(wave, true);   // (64 images of 56x56x64 bf16: 0.132 -> 0.127 ms; with one channel a wave it changes nothing)
      fetch(next, 0, opsA);          // (behind the last block: what an earlier one left there, never used)
      step(opsB, 3, par ^ 1);
      if constexpr (CKPT) ckp += HALF ? 2 * ck_step : ck_step;
      par ^= 1;
      buf = next;
    }
    if constexpr (CKPT && HALF) {   // the state behind the last block: what the sweep's last step left is among it
#pragma unroll
      for (int c = 0; c < EC; ++c)
        if (ch_ok) Snap<T>::store(ckp + c * (kN / 4 * kHB), h[c][0], h[c][1], h[c][2], h[c][3]);
    }
    __syncthreads();   // the last window
  } else {
    // ------------------------------------------------------------------------------ stages
    const int sw = wave - NW;
    if (sw == 3) __builtin_amdgcn_s_setprio(3);   // (its few instructions are what the neighbouring bands wait for)
    const int k = lane >> kHBShift, r = lane & (kHB - 1);   // the lane's (step, row) of a block
    const int rbands = row_bands(p, r);
    const int64_t img_cell0 = (int64_t)b * p.Hs * p.W;
    const char* zeros = reinterpret_cast<const char*>(p.zeros);
    const char* const img[4] = {static_cast<const char*>(p.x) + img_cell0 * p.E * (int64_t)sizeof(T), static_cast<const char*>(p.dT) + img_cell0 * p.E * (int64_t)sizeof(T),
                          static_cast<const char*>(p.dL) + img_cell0 * p.E * (int64_t)sizeof(T), nullptr};
    const char* x_img = img[sw < 3 ? sw : 0];
    char* Yimg = static_cast<char*>(p.y) + img_cell0 * p.E * (int64_t)sizeof(T);
    // B_T, B_L, C: bytes per cell and where image b starts
    const uint32_t bc_cell = direct ? (uint32_t)(kN * (WIDEN ? 2 : 4)) : (uint32_t)(3 * kN * 4);
    const bool raw = WIDEN && direct;                       // (uniform)
    SplitBC<SLICED> bc;
    bc.cell = bc_cell;
    bc.start(p, my_band, 0, sw, lane, direct, img_cell0);
    SplitVals<T, 3, CW> vals;
    typedef Track<SLICED> Tr;
    Tr sq, bq;                                              // the block to be fetched next: the lane's (step, row); raw B_T, B_L, C: (lane & 3, lane >> 2)
    sq.start(p, my_band, k, r);
    bq.start(p, my_band, lane & 3, lane >> 2);
    LaneK consts = lane_consts<false>(p, clamp_band(p, sq.bnd), r, true);
    auto buf_of = [&](int j) { return (uint32_t)(j & (L::kBufs - 1)) * (uint32_t)SG::kBytes; };   // j: block of the window
    // Every block issues the same operations, also those behind the window (which fetch zeros): the waits below count on it.
    constexpr int kX = SX ? SG::kChunks : 0, kCopies = 4 + kX, kRawCopies = 2 + kX;   // a wave's copies per block
    auto stage = [&](uint32_t buf) {                            // (waves 0..2)
      if (raw) {
        split_raw_copy<SG>(bq.on(p) ? bc.mine + cell_bytes_off(bq.cell, bc_cell) : zeros, buf + sw * SG::kBCTensor);
        bq = bq.moved(p, kCK);
      } else {
        bc.template copy<SG>(p, buf, sw, kCK);
      }
      if constexpr (SX) {
        split_x_copy<T, SG>(p, x_img, (uint32_t)sq.cell, sq.on(p), e_wg0, buf + SG::kX + sw * SG::kXTensor);
        sq = sq.moved(p, kCK);
      }
    };
    auto put_consts = [&](uint32_t buf) {                       // (wave 3)
      if constexpr (!SLICED) consts = lane_consts<false>(p, clamp_band(p, sq.bnd), r, true);
      split_consts<SG>(consts, sq.col, lds + buf, lane);
      sq = sq.moved(p, kCK);
    };
    auto widen = [&](uint32_t buf) { if (raw) split_raw_widen<SG>(lds + buf + sw * SG::kBCTensor, lane); };
    Tr vq = sq;                                              // (values, all four waves: the block to be fetched next)
    auto fetch_vals = [&] {
      split_vals_fetch<T, 3, CW>(p, img, (uint32_t)vq.cell, vq.on(p), e_wg0, sw, vals);
      vq = vq.moved(p, kCK);
    };
    // boundary rows: lane (step k, channel of four, state group)
    const int row_ch = (lane >> 2) & 3, row_g = lane & 3;
    const int64_t band_bytes = (int64_t)p.B * p.W * p.E * (int64_t)(kN * sizeof(float));
    char* rows = reinterpret_cast<char*>(p.top) + (((int64_t)b * p.W * p.E + e_wg0 + row_ch) * kN + row_g * 4) * (int64_t)sizeof(float) + (SLICED ? my_band * band_bytes : 0);
    char* rows_above = SLICED ? rows - band_bytes : rows;
    Tr tq;                                                   // the upper ghost (lane row 0) of the block whose TOP comes next
    tq.start(p, my_band, k, 0);
    auto copy_top = [&](uint32_t buf) {
      const bool ok = tq.bnd >= 1 && tq.bnd < p.nbands && (unsigned)tq.col < (unsigned)p.W;
#pragma unroll
      for (int j = 0; j < SG::kG4; ++j)
        split_fill16<true>(ok && e_wg0 + 4 * j + row_ch < p.E ? row_record<SLICED>(p, rows_above, tq, -1, band_bytes) + j * (4 * kN * (int)sizeof(float)) : zeros, buf + SG::kTop + j * SG::kSet);
      tq = tq.moved(p, kCK);
    };
    Tr rq;                                                   // the band's last row (lane row 14) in the window to be sent next
    rq.start(p, my_band, k - 1, kRB);
    auto send_rows = [&](int par) {                          // kG4 stores
      const bool ok = rq.bnd >= 0 && rq.bnd + 1 < p.nbands && (unsigned)rq.col < (unsigned)p.W;
      char* dst = row_record<SLICED>(p, rows, rq, 0, band_bytes);
#pragma unroll
      for (int j = 0; j < SG::kG4; ++j) {
        const float4 row = *reinterpret_cast<const float4*>(lds + L::kR + par * L::kRBytes + k * L::kRStep + (4 * j + row_ch) * 64 + row_g * 16);
        split_store_row<SLICED>(dst + j * (4 * kN * (int)sizeof(float)), row, ok && e_wg0 + 4 * j + row_ch < p.E);
      }
      rq = rq.moved(p, kCK);
    };
    // y: wave 1 the steps 0 and 1 of a window, wave 2 the steps 2 and 3; lane (row, channel of four), or (16 channels) (row, four channels)
    const int y_row = lane >> 2, y_ch = (lane & 3) * (EC == 2 ? 4 : 1);
    Tr yq;                                                   // the lane's row at the first of the wave's steps in the window to be sent next
    yq.start(p, my_band, 2 * (sw - 1) - 1, y_row);
    constexpr int kYStores = !WRITE_Y ? 0 : (EC == 2 ? 2 : 2 * (CW / 4));
    auto send_y = [&](int par, int steps) {                  // kYStores
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const Tr t = yq.moved(p, i);
        const int kw = 2 * (sw - 1) + i;                     // (uniform) step of the window
        const bool ok = t.on(p) && kw < steps;
        const uint32_t off = cell_bytes_off(t.cell, (uint32_t)p.E * (uint32_t)sizeof(T)) + (uint32_t)(e_wg0 + y_ch) * (uint32_t)sizeof(T);
        auto share = [&](int c) {
          const float4 s = *reinterpret_cast<const float4*>(lds + L::kY + par * L::kYBytes + kw * L::kYStep + c * L::kYCh + y_row * 16);
          return (s.x + s.y) + (s.z + s.w);
        };
        if constexpr (EC == 2) {
          split_store_quad(reinterpret_cast<T*>(Yimg + off), make_float4(share(y_ch), share(y_ch + 1), share(y_ch + 2), share(y_ch + 3)), ok && e_wg0 + y_ch < p.E);
        } else {
#pragma unroll
          for (int j = 0; j < CW / 4; ++j) split_store(reinterpret_cast<T*>(Yimg + off) + 4 * j, share(4 * j + y_ch), ok && e_wg0 + 4 * j + y_ch < p.E);
        }
      }
      yq = yq.moved(p, kCK);
    };

    const int n = m_hi - m_lo;                               // blocks of the window
    // Rows of this workgroup's own previous band are sent and acknowledged two blocks before they are read back, if the stream's
    // stride leaves the time; the shortest strides (26 .. 30) have wave 0 send, wait and fetch.
    const int top_wave = !SLICED && p.S < kRB + 17 ? 0 : 3;
    if (sw < 3) {
#pragma unroll 1
      for (int j = 0; j < 3; ++j) stage(buf_of(j));
      if (raw) split_landed<2 * kRawCopies>(); else split_landed<2 * kCopies>();
      widen(buf_of(0));
    } else {
#pragma unroll 1
      for (int j = 0; j < 3; ++j) put_consts(buf_of(j));
    }
    // wave 3 waits for the neighbour above, wave 0 tells the one below
    auto wait_above = [&](int j) {
      if constexpr (SLICED) {
        link.wait_for(link_need_fwd(j, p.sl_nbb));
        if (lane == 0) *reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(smem) + L::kFlag) = link.broken() ? 1u : 0u;
      }
    };
    auto tell_below = [&](uint32_t done) {
      if constexpr (SLICED) { if (lane == 0) link_publish(link.mine, *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(smem) + L::kFlag) != 0u ? kLinkAbort : done); }
    };
    if (sw == 3) wait_above(0);
    if (sw == top_wave) {
      copy_top(buf_of(0));
      staging_landed();
    }
    if constexpr (!SX) {
      fetch_vals();
      split_vals_put<T, 3, CW, SG>(vals, lds + buf_of(0), sw, lane);
      fetch_vals();
    }
    __syncthreads();
    for (int j = 0; j < n; ++j) {                            // window j - 1 is complete, block j is being swept
      const int par = (j + 1) & 1;
      if constexpr (!SX) {
        if (j + 1 < n) split_vals_put<T, 3, CW, SG>(vals, lds + buf_of(j + 1), sw, lane);
        if (j + 2 < n) fetch_vals();
      }
      if (sw < 3) {
        const bool rows_out = sw == 0 && p.nbands > 1 && j > 0;
        if (rows_out) send_rows(par);
        if (WRITE_Y && sw > 0 && j > 0) send_y(par, kCK);
        const bool top_late = sw == top_wave;
        if (top_late) {
          staging_landed();
          copy_top(buf_of(j + 1));
        }
        stage(buf_of(j + 3));
        // Block j + 1 has landed -- the two blocks fetched behind it, and what was stored since, may be under way -- and so have
        // the rows that were sent in the block before.
        auto landed = [&](auto copies) {
          constexpr int c = decltype(copies)::value;
          if (top_late) split_landed<c>();
          else if (j == 0 || (sw == 0 && p.nbands == 1)) split_landed<2 * c>();
          else if (sw == 0) { if (SLICED && j > 2) split_landed<2 * c + SG::kG4 + 1>(); else split_landed<2 * c + SG::kG4>(); }
          else if (j == 1) split_landed<2 * c + kYStores>();
          else split_landed<2 * c + 2 * kYStores>();
        };
        if (raw) landed(std::integral_constant<int, kRawCopies>{}); else landed(std::integral_constant<int, kCopies>{});
        if (SLICED && rows_out && j > 1) tell_below((uint32_t)(j - 1));
        widen(buf_of(j + 1));
      } else {
        put_consts(buf_of(j + 3));
        if (sw == top_wave && j + 1 < n) {
          wait_above(j + 1);
          copy_top(buf_of(j + 1));
          staging_landed();
        }
      }
      __syncthreads();
    }
    const int par = (n + 1) & 1;                             // window n - 1
    if (sw == 0) {
      if (p.nbands > 1) send_rows(par);
      if constexpr (SLICED) { staging_landed(); tell_below((uint32_t)p.sl_nbb); }
    }
    if (WRITE_Y && (sw == 1 || sw == 2)) send_y(par, kCK);
    __syncthreads();
    if (WRITE_Y && (sw == 1 || sw == 2)) send_y(par ^ 1, 1); // the last step of the sweep
    staging_landed();                                        // (copies of the blocks behind the window: the LDS is still this workgroup's)
  }
  if constexpr (SLICED) {   // only the wave that waits knows of a wait given up: it tells the others (the staging buffers are free now)
    if ((int)threadIdx.x == link.pub) *reinterpret_cast<volatile uint32_t*>(lds) = link.broken() ? 1u : 0u;
    staging_landed();
    __syncthreads();
    if (WRITE_Y && *reinterpret_cast<volatile uint32_t*>(lds) != 0u) poison_band<T>(p, my_band, b, e_wg0, CW, p.y, nullptr, nullptr);
  }
}

// --------------------------------------------------------------------------------------- backward
// The counterpart: a block is swept in one pass (4 states a lane leave room for the gates and operands of all four
// steps, kept from the recomputation to the adjoint).  Results go to LDS by phases of XS steps, two sets used in turn
// and a barrier at the end of a phase: per step a float4 of the lane's 4 states of d_C, d_BT and d_BL (added up over the
// channels by the staging waves) and the lane's shares of d_deltaT, d_deltaL and d_x (added up over the state groups),
// the fourth place carrying what the sums need beside them.
// Phases of the band below that must be done (counted from the end of its window, PH to a block) before the BOT of block j is
// copied: through the steps 3 and 2 of its block j - 4 (see link_need_bwd).
__device__ __forceinline__ uint32_t link_need_bwd_phases(int j, int nbb, int PH) { return (uint32_t)(j >= 4 ? PH * (nbb - j + 3) + PH / 2 : PH * nbb); }
template <typename T, int NW, bool SX>
struct SplitBwdLds {
  using SG = SplitStage<T, 4, NW, true, SX>;
  static constexpr int kPhaseSteps = NW == kSplitHalfWaves ? 2 : 1;   // (8 channels: two sets of one step are what fits)
  static constexpr int kKind = NW * 1024;                  // one step of d_C, d_BT, d_BL or the shares: [channel][lane] float4s
  static constexpr int kXStep = 4 * kKind;
  static constexpr int kXBytes = kPhaseSteps * kXStep;     // one set
  static constexpr int kRStep = NW * 64;                   // muT of the band's first row at one step: [channel][state group] float4s
  static constexpr int kRBytes = kPhaseSteps * kRStep;
  static constexpr int kBufs = 3;
  static constexpr int kX = kBufs * SG::kBytes, kR = kX + 2 * kXBytes, kBytes = kR + 2 * kRBytes;
};
template <typename T, bool SX, int MODE, int NW = kSplitWaves>
__global__ __launch_bounds__((NW + kSplitStagers) * 64) void m2d_bwd_split_kernel(const ScanParams pin) {
  static_assert(MODE != kModeStacked, "stacked images are many: they never need the split");
  constexpr bool SLICED = MODE == kModeSliced;
  constexpr bool WIDEN = sizeof(T) == 2;
  constexpr int CW = NW;
  const ScanParams& p = pin;
  __builtin_assume(p.stacked == 0);
  __builtin_assume(p.rb == kRB);
  __builtin_assume(p.S >= kHB + kCK - 1);
  using L = SplitBwdLds<T, NW, SX>;
  using SG = typename L::SG;
  constexpr int XS = L::kPhaseSteps, PH = kCK / XS;        // steps per phase, phases per block
  constexpr bool KEEP = NW == kSplitHalfWaves;             // B_T, B_L and coefficients of a block stay in registers (workgroups of 8 have too few)
  extern __shared__ float4 smem[];
  char* lds = reinterpret_cast<char*>(smem);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lb = 0, turn = 0;
  if constexpr (SLICED) { if (!linked_place(p, turn, lb)) return; } else lb = logical_block(p.nwg);
  int m_lo = 0, m_hi = p.nblk;
  int my_band = 0;
  LinkT<(NW + 3) * 64> link;
  if constexpr (SLICED) {   // the window of one band; the bands are launched from the last to the first
    const int per = p.B * p.bpb;
    my_band = p.nbands - 1 - turn;
    m_lo = my_band * p.sl_nbb;
    m_hi = m_lo + p.sl_nbb;
    link.mine = p.prog + ((int64_t)my_band * per + lb) * kLinkStride;
    link.dep = my_band + 1 < p.nbands ? link.mine + per * kLinkStride : nullptr;
    link.err = p.link_err;
    link.rig(p, my_band);
  }
  const int b = lb / p.bpb;
  const int eg = lb % p.bpb;
  const int e_wg0 = eg * CW;
  const bool direct = WIDEN && p.bc_direct != 0;   // (uniform)
  const int g = lane >> kHBShift, r = lane & (kHB - 1);   // sweeps: state group, lane row
  const bool ch_ok = wave < NW && e_wg0 + wave < p.E;     // (uniform)
  const int e = ch_ok ? e_wg0 + wave : p.E - 1;
  // register w of the lane meets position 4g + w of a record: state perm(w) * 4 + g (fold order)
  int state_of[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) state_of[w] = (w == 1 ? 2 : (w == 2 ? 1 : w)) * 4 + g;
  float accAT[4], accAL[4], accD = 0.f;
#pragma unroll
  for (int w = 0; w < 4; ++w) { accAT[w] = 0.f; accAL[w] = 0.f; }

  if (wave < NW) {
    // ------------------------------------------------------------------------------ sweeps
    const int ch = wave;
    float a2t[4], a2l[4], muT[4], muL[4];
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      a2t[w] = p.A2T[e * kN + state_of[w]];
      a2l[w] = p.A2L[e * kN + state_of[w]];
      muT[w] = 0.f; muL[w] = 0.f;
    }
    const float dsk = p.Df[e];
    const float g1 = r == 0 ? 1.f : 0.f;
    const float gb1 = r == kHB - 1 ? 1.f : 0.f;            // 1 on the lower ghost: lambda = 1 * (row of mu_T below)
    // a grid row reads B_T, B_L, C of its cell; the upper ghost (lane 0) the row above as its B_T; the lower ghost
    // (lane 15) the row of mu_T below as its C; zeros in the other places
    const uint32_t bt_off = r == 0 ? SG::row_off(SG::kTop, ch, g) : SG::bc_off(0, g, r);
    const uint32_t bl_off = SG::bc_off(1, g, r);
    const uint32_t cc_off = r == kHB - 1 ? SG::row_off(SG::kBot, ch, g) : SG::bc_off(2, g, r);
    const uint32_t bt_step = r == 0 ? SG::kStep : SG::kBCStep, cc_step = r == kHB - 1 ? SG::kStep : SG::kBCStep;
    const uint32_t k_off = SG::kConst + r * 16;
    const uint32_t x_off = SG::x_off(ch, r, e_wg0);
    char* xw = lds + L::kX + ch * 1024 + lane * 16;
    // the shares of a row are at place row ^ 4 (pair of channels) ^ 8 (step of the phase): 16 lanes of the wave that adds them up read four
    // rows of four (pair, step), which are in different banks then
    char* xw_share = lds + L::kX + 3 * L::kKind + ch * 1024 + (SX ? (lane ^ ((ch >> 1) * 4)) : lane) * 16;
    char* xw_share_odd = lds + L::kX + 3 * L::kKind + ch * 1024 + (lane ^ ((ch >> 1) * 4) ^ 8) * 16;
    char* rw = lds + L::kR + ch * 64 + g * 16;
    const bool first_row = r == 1 && p.nbands > 1;         // the band's first row: the lower ghost of the band above will replay its muT
    Pos at = pos_of(p, (m_hi - 1) * kCK - r);              // the row at the first step of the block
    typename Snap<T>::quad cknext = Snap<T>::zero();
    const typename Snap<T>::quad* ckp = snapshot_at<T>(p, b, m_hi - 1, e, p.nblk) + snap_lane(r) + snap_quad(g);
    const int64_t ck_step = (int64_t)p.E * (kN / 4 * kHB);
    auto load_ckpt = [&](int mm) {   // (the forward kept the lane's state where snapshot_lane says so)
      cknext = Snap<T>::zero();
      if (mm != 0 && snapshot_lane(p, at, r, ch_ok)) cknext = *ckp;
    };
    load_ckpt(m_hi - 1);

    struct Fwd { float4 kk, bt, bl; float x, dt, dl; };
    auto fetch = [&](uint32_t buf, int k, Fwd& o) {
      const char* s = lds + buf;
      o.kk = *reinterpret_cast<const float4*>(s + k_off + k * SG::kStep);
      o.dt = split_x<T, SX>(s + x_off + SG::kXTensor + k * SG::kXStep);
      o.dl = split_x<T, SX>(s + x_off + 2 * SG::kXTensor + k * SG::kXStep);
      o.x = split_x<T, SX>(s + x_off + k * SG::kXStep);
      o.bl = *reinterpret_cast<const float4*>(s + bl_off + k * SG::kBCStep);
      o.bt = *reinterpret_cast<const float4*>(s + bt_off + k * bt_step);
    };
    __syncthreads();   // the first block is in place
    uint32_t buf = 0;
    int par = 0;
    Fwd ops[kCK];
    fetch(buf, 0, ops[0]);
    for (int m = m_hi - 1; m >= m_lo; --m) {
      float hb[kCK + 1][4], gT[kCK][4], gL[kCK][4], qT[kCK], qL[kCK];
      { const float4 v = Snap<T>::widen(cknext); hb[0][0] = v.x; hb[0][1] = v.y; hb[0][2] = v.z; hb[0][3] = v.w; }
      // ---- recompute the states of the block, keeping the gates
#pragma unroll
      for (int k = 0; k < kCK; ++k) {
        if (k + 1 < kCK) fetch(buf, k + 1, ops[k + 1]);
        const Fwd& o = ops[k];
        const float sT = __builtin_fmaf(o.kk.z * o.dt, o.x, g1);
        const float sL = o.kk.w * o.dl * o.x;
        qT[k] = sT - g1; qL[k] = sL;      // zero on lanes that are not grid cells
#pragma unroll
        for (int w = 0; w < 4; ++w) gT[k][w] = fexp2(__builtin_fmaf(o.dt, a2t[w], o.kk.x));
#pragma unroll
        for (int w = 0; w < 4; ++w) gL[k][w] = fexp2(__builtin_fmaf(o.dl, a2l[w], o.kk.y));
        pin4(gT[k]); pin4(gL[k]);
        __builtin_amdgcn_sched_barrier(0);
        const float bq[4] = {o.bt.x, o.bt.y, o.bt.z, o.bt.w}, lq[4] = {o.bl.x, o.bl.y, o.bl.z, o.bl.w};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          float u = sL * lq[w];
          u = __builtin_fmaf(sT, bq[w], u);
          u = fma_row_below(gT[k][w], hb[k][w], u);
          hb[k + 1][w] = __builtin_fmaf(gL[k][w], hb[k][w], u);
        }
      }
      at.col -= kCK;
      if (at.col < 0) { at.col += p.S; at.bnd -= 1; }
      ckp -= ck_step;
      if (m > m_lo) load_ckpt(m - 1);
      // ---- adjoint over the block, last step first
      float4 c4 = *reinterpret_cast<const float4*>(lds + buf + cc_off + (kCK - 1) * cc_step);
      float dyv = split_x<T, SX>(lds + buf + x_off + 3 * SG::kXTensor + (kCK - 1) * SG::kXStep);
      const uint32_t next = buf == (L::kBufs - 1) * SG::kBytes ? 0 : buf + SG::kBytes;
#pragma unroll
      for (int k = kCK - 1; k >= 0; --k) {
        float4 c4n = c4;
        float dyn = dyv;
        if (k > 0) {
          c4n = *reinterpret_cast<const float4*>(lds + buf + cc_off + (k - 1) * cc_step);
          dyn = split_x<T, SX>(lds + buf + x_off + 3 * SG::kXTensor + (k - 1) * SG::kXStep);
        }
        Fwd& o = ops[k];
        if constexpr (!KEEP) {
          o.bt = *reinterpret_cast<const float4*>(lds + buf + bt_off + k * bt_step);
          o.bl = *reinterpret_cast<const float4*>(lds + buf + bl_off + k * SG::kBCStep);
          const float2 c = *reinterpret_cast<const float2*>(lds + buf + k_off + k * SG::kStep + 8);
          o.kk.z = c.x;
          o.kk.w = c.y;
        }
        const float cT = o.kk.z, cL = o.kk.w, xv = o.x, dtv = o.dt, dlv = o.dl;
        const float bq[4] = {o.bt.x, o.bt.y, o.bt.z, o.bt.w}, lq[4] = {o.bl.x, o.bl.y, o.bl.z, o.bl.w}, cq[4] = {c4.x, c4.y, c4.z, c4.w};
        const float dyl = dyv + gb1;
        float sT = 0.f, sL = 0.f, zT = 0.f, zL = 0.f;
        float vC[4], vBT[4], vBL[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float lam = __builtin_fmaf(dyl, cq[w], add_row_above(muL[w], muT[w]));
          const float mT = gT[k][w] * lam, mL = gL[k][w] * lam;
          muT[w] = mT;
          muL[w] = mL;
          const float ZT = mul_row_below(mT, hb[k][w]), ZL = mL * hb[k][w];
          accAT[w] = __builtin_fmaf(ZT, dtv, accAT[w]);
          accAL[w] = __builtin_fmaf(ZL, dlv, accAL[w]);
          zT = __builtin_fmaf(ZT, a2t[w], zT);
          zL = __builtin_fmaf(ZL, a2l[w], zL);
          sT = __builtin_fmaf(lam, bq[w], sT);
          sL = __builtin_fmaf(lam, lq[w], sL);
          vBT[w] = qT[k] * lam;
          vBL[w] = qL[k] * lam;
          vC[w] = dyv * hb[k + 1][w];
        }
        accD = __builtin_fmaf(dyv, xv, accD);
        char* xs = xw + par * L::kXBytes + (XS == 1 ? 0 : k % XS) * L::kXStep;
        *reinterpret_cast<float4*>(xs) = make_float4(vC[0], vC[1], vC[2], vC[3]);
        *reinterpret_cast<float4*>(xs + L::kKind) = make_float4(vBT[0], vBT[1], vBT[2], vBT[3]);
        *reinterpret_cast<float4*>(xs + 2 * L::kKind) = make_float4(vBL[0], vBL[1], vBL[2], vBL[3]);
        // the lane's share (its 4 states) of d_deltaT, d_deltaL and d_x of the cell, and beside them the two step sizes
        // (groups 0, 1) and dy * D (group 2)
        const float pT = __builtin_fmaf(cT * xv, sT, kLn2 * zT);
        const float pL = __builtin_fmaf(cL * xv, sL, kLn2 * zL);
        const float pX = __builtin_fmaf(cT * dtv, sT, cL * dlv * sL);
        char* xsh = xw_share + par * L::kXBytes + (XS == 1 ? 0 : k % XS) * L::kXStep;
        if (SX && XS > 1 && k % XS == 1) xsh = xw_share_odd + par * L::kXBytes + L::kXStep;
        *reinterpret_cast<float4*>(xsh) = make_float4(pT, pL, pX, g == 0 ? dtv : (g == 1 ? dlv : dyv * dsk));
        if (first_row) *reinterpret_cast<float4*>(rw + par * L::kRBytes + (XS == 1 ? 0 : k % XS) * L::kRStep) = make_float4(muT[0], muT[1], muT[2], muT[3]);
        if (k == 0) fetch(next, 0, ops[0]);   // (the operands of the block before are in place since the phase before; behind the last block: never used)
        if (k % XS == 0) { __syncthreads(); par ^= 1; }
        c4 = c4n;
        dyv = dyn;
      }
      buf = next;
    }
  } else {
    // ------------------------------------------------------------------------------ stages and adds up
    const int sw = wave - NW;
    if (sw == 3) __builtin_amdgcn_s_setprio(3);   // (its few instructions are what the neighbouring bands wait for)
    const int k = lane >> kHBShift;                         // the lane's (step, row) of a block
    const int64_t img_cell0 = (int64_t)b * p.Hs * p.W;
    const int64_t img_bytes = img_cell0 * p.E * (int64_t)sizeof(T);
    const char* zeros = reinterpret_cast<const char*>(p.zeros);
    const char* const img[4] = {static_cast<const char*>(p.x) + img_bytes, static_cast<const char*>(p.dT) + img_bytes,
                                static_cast<const char*>(p.dL) + img_bytes, static_cast<const char*>(p.dy) + img_bytes};
    char* PARTimg = reinterpret_cast<char*>(p.part + ((int64_t)eg * p.Ptot + img_cell0) * (3 * kN));   // channel sums: [cell][C, B_T, B_L][16]
    const uint32_t bc_cell = direct ? (uint32_t)(kN * 2) : (uint32_t)(3 * kN * 4);
    const bool raw = direct;                                // (uniform)
    SplitBC<SLICED> bc;
    bc.cell = bc_cell;
    SplitVals<T, 4, CW> vals;
    typedef Track<SLICED> Tr;
    const int at0 = (m_hi - 1 - m_lo) * kCK;                // the last block of the window comes first
    // boundary rows: lane (step k, channel of four, state group)
    const int row_ch = (lane >> 2) & 3, row_g = lane & 3;
    const int64_t rec_bytes = kN * (int64_t)sizeof(float), band_bytes = (int64_t)p.B * p.W * p.E * rec_bytes, bot_bytes = p.bot_stride * (int64_t)sizeof(float);
    char* rows_above = reinterpret_cast<char*>(p.top) + ((int64_t)b * p.W * p.E + e_wg0 + row_ch) * rec_bytes + row_g * 16 + (SLICED ? (my_band - 1) * band_bytes : 0);
    char* rows_below = reinterpret_cast<char*>(p.bot) + ((int64_t)b * p.W * p.E + e_wg0 + row_ch) * rec_bytes + row_g * 16 + (SLICED ? (my_band + 1) * bot_bytes : 0);
    Tr tq;                                                  // the upper ghost (lane row 0) of the block whose TOP comes next
    tq.start(p, my_band, at0 + k, 0);
    auto copy_top = [&](uint32_t buf) {
      const bool ok = tq.bnd >= 1 && tq.bnd < p.nbands && (unsigned)tq.col < (unsigned)p.W;
#pragma unroll
      for (int j = 0; j < SG::kG4; ++j)
        split_fill16<true>(ok && e_wg0 + 4 * j + row_ch < p.E ? row_record<SLICED>(p, rows_above, tq, -1, band_bytes) + j * 4 * rec_bytes : zeros, buf + SG::kTop + j * SG::kSet);
      tq = tq.moved(p, -kCK);
    };
    Tr lq;                                                  // the lower ghost (lane row 15) of the block whose BOT comes next
    lq.start(p, my_band, at0 + k, kHB - 1);
    auto copy_bot = [&](uint32_t buf) {
      const bool ok = lq.bnd >= 0 && lq.bnd + 1 < p.nbands && (unsigned)lq.col < (unsigned)p.W;
#pragma unroll
      for (int j = 0; j < SG::kG4; ++j)
        split_fill16<true>(ok && e_wg0 + 4 * j + row_ch < p.E ? row_record<SLICED>(p, rows_below, lq, 1, bot_bytes) + j * 4 * rec_bytes : zeros, buf + SG::kBot + j * SG::kSet);
      lq = lq.moved(p, -kCK);
    };
    Tr sq, bq;                                              // the block to be fetched next (see the forward)
    sq.start(p, my_band, at0 + k, r);
    bq.start(p, my_band, at0 + (lane & 3), lane >> 2);
    bc.start(p, my_band, at0, sw, lane, direct, img_cell0);
    LaneK consts = lane_consts<true>(p, clamp_band(p, sq.bnd), r, true);
    auto buf_of = [&](int j) { return (uint32_t)(j % L::kBufs) * (uint32_t)SG::kBytes; };   // j: block of the window, from its end
    // Every block issues the same operations, also those behind the window (which fetch zeros): the waits below count on it.
    constexpr int kCopies = 4, kRawCopies = 2, kXCopies = (SX ? 4 * SG::kChunks : 0) + SG::kG4;   // per block: of a wave of 0..2; of wave 3
    // a wave's stores per phase: sums and results (SX: wave 2 all results)
    constexpr int kStores = SX ? XS : XS + XS * (CW / 4), kStores2 = SX ? XS + 3 : kStores;
    auto stage_bc = [&](uint32_t buf) {                        // (waves 0..2)
      if (raw) {
        split_raw_copy<SG>(bq.on(p) ? bc.mine + cell_bytes_off(bq.cell, bc_cell) : zeros, buf + sw * SG::kBCTensor);
        bq = bq.moved(p, -kCK);
      } else {
        bc.template copy<SG>(p, buf, sw, -kCK);
      }
    };
    auto stage_x = [&](uint32_t buf) {                         // (wave 3; the constants and the upper boundary rows too)
      const bool ok = sq.on(p);
      if constexpr (SX) {
#pragma unroll
        for (int t = 0; t < 4; ++t) split_x_copy<T, SG>(p, img[t], (uint32_t)sq.cell, ok, e_wg0, buf + SG::kX + t * SG::kXTensor);
      }
      copy_top(buf);
      if constexpr (!SLICED) consts = lane_consts<true>(p, clamp_band(p, sq.bnd), r, true);
      split_consts<SG>(consts, sq.col, lds + buf, lane);
      sq = sq.moved(p, -kCK);
    };
    auto widen = [&](uint32_t buf) { if (raw) split_raw_widen<SG>(lds + buf + sw * SG::kBCTensor, lane); };
    Tr vq = sq;                                              // (values, all four waves: the block to be fetched next)
    auto fetch_vals = [&] {
      split_vals_fetch<T, 4, CW>(p, img, (uint32_t)vq.cell, vq.on(p), e_wg0, sw, vals);
      vq = vq.moved(p, -kCK);
    };
    // What the sweeping waves left in set `par` in a phase whose steps are k0 .. k0 + XS - 1 of their block.  The tracks are those of the
    // block being swept; behind: the phase is the last one of the block before.
    Tr rq, cq, oq;                                          // first row of the band (lane row 1); the sums' lane row; the results'
    rq.start(p, my_band, at0, 1);
    cq.start(p, my_band, at0, r);
    oq.start(p, my_band, at0, lane >> 2);
    auto send_rows = [&](const Tr& t0, int k0, int par) {   // (wave 3) lane (step, channel, state group)
      const int i = lane >> 2, ks = XS == 1 ? 0 : i / CW, c = i % CW;
      const Tr t = t0.moved(p, k0 + ks);
      const float4 row = *reinterpret_cast<const float4*>(lds + L::kR + par * L::kRBytes + ks % XS * L::kRStep + c * 64 + row_g * 16);
      const bool live = i < XS * CW && t.bnd >= 1 && t.bnd < p.nbands && (unsigned)t.col < (unsigned)p.W && e_wg0 + c < p.E;
      char* base = reinterpret_cast<char*>(p.bot) + ((int64_t)b * p.W * p.E + e_wg0 + c) * rec_bytes + row_g * 16 + (SLICED ? my_band * bot_bytes : 0);
      split_store_row<SLICED>(row_record<SLICED>(p, base, t, 0, bot_bytes), row, live);
    };
    // A lane holds the states perm(j) * 4 + g of its cell (perm = 0, 2, 1, 3); turned over the four state groups, group g holds the neighbours
    // perm(g) * 4 .. + 3, and a row's 64 bytes leave in one store: as four stores of 4 bytes a lane, 16 bytes of a row each,
    // the sums kept the memory pipeline from the copies and snapshots beside them (1x256x256x64 fp32 0.483 -> 0.396 ms, 1x28x4096x64 2.64 -> 1.94).
    const uint32_t sum_off = (uint32_t)((sw * kN + ((g & 1) * 2 + (g >> 1)) * 4) * 4);
    auto send_sums = [&](const Tr& t0, int k0, int par) {   // tensor sw (C, B_T, B_L), lane (state group, row)
      float4 sum[XS];
#pragma unroll
      for (int ks = 0; ks < XS; ++ks) {
        const float4* sl = reinterpret_cast<const float4*>(lds + L::kX + par * L::kXBytes + ks * L::kXStep + sw * L::kKind) + lane;
        sum[ks] = sl[0];
#pragma unroll
        for (int w = 1; w < NW; ++w) { const float4 o = sl[w * 64]; sum[ks].x += o.x; sum[ks].y += o.y; sum[ks].z += o.z; sum[ks].w += o.w; }
      }
#pragma unroll
      for (int ks = 0; ks < XS; ++ks) {
        const Tr t = t0.moved(p, k0 + ks);
        split_store_quad(reinterpret_cast<float*>(PARTimg + cell_bytes_off(t.cell, 3 * kN * sizeof(float)) + sum_off), slots_turned(sum[ks]), t.on(p));
      }
    };
    // d_deltaT, d_deltaL, d_x.  SX: by wave 2, which has all four shares of a channel's results from four reads: lane (row, two neighbouring channels[, step of the phase]).
    // Otherwise a tensor each by the waves 0, 1, 2; lane (row, channel of four).
    auto send_results = [&](const Tr& t0, int k0, int par) {
      if constexpr (SX) {
        if (sw != 2) return;
        constexpr int kPairs = CW / 2;
        static_assert(kPairs * XS == 4, "a wave has the results of a phase");
        const int row = lane >> 2, pair = lane % kPairs, ks = XS == 1 ? 0 : (lane / kPairs) & 1;
        const Tr t = t0.moved(p, k0 + ks);
        const bool ok = t.on(p) && e_wg0 + 2 * pair < p.E;
        const float4* sh = reinterpret_cast<const float4*>(lds + L::kX + par * L::kXBytes + ks * L::kXStep + 3 * L::kKind + pair * 2048) + (row ^ (pair * 4) ^ (ks * 8));
        float vT[2], vL[2], vX[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float4 q0 = sh[c * 64], q1 = sh[c * 64 + 16], q2 = sh[c * 64 + 32], q3 = sh[c * 64 + 48];
          vT[c] = (q0.x + q1.x) + (q2.x + q3.x);
          vL[c] = (q0.y + q1.y) + (q2.y + q3.y);
          vX[c] = (q0.z + q1.z) + (q2.z + q3.z) + q2.w;
          if (p.dpre) {   // (uniform) gradients with respect to what the softplus was applied to
            vT[c] *= softplus_slope<T>(q0.w);
            vL[c] *= softplus_slope<T>(q1.w);
          }
        }
        const uint32_t off = cell_bytes_off(t.cell, (uint32_t)p.E * (uint32_t)sizeof(T)) + (uint32_t)(e_wg0 + 2 * pair) * (uint32_t)sizeof(T);
        split_store_pair(reinterpret_cast<T*>(static_cast<char*>(p.ddT) + img_bytes + off), vT[0], vT[1], ok);
        split_store_pair(reinterpret_cast<T*>(static_cast<char*>(p.ddL) + img_bytes + off), vL[0], vL[1], ok);
        split_store_pair(reinterpret_cast<T*>(static_cast<char*>(p.dx) + img_bytes + off), vX[0], vX[1], ok);
        return;
      }
      char* const out_img = static_cast<char*>(sw == 0 ? p.ddT : (sw == 1 ? p.ddL : p.dx)) + img_bytes;
      const int row = lane >> 2, c4 = lane & 3;
#pragma unroll
      for (int ks = 0; ks < XS; ++ks) {
        const Tr t = t0.moved(p, k0 + ks);
#pragma unroll
        for (int j = 0; j < CW / 4; ++j) {
          const int c = 4 * j + c4;
          const bool ok = t.on(p) && e_wg0 + c < p.E;
          const float* sh = reinterpret_cast<const float*>(lds + L::kX + par * L::kXBytes + ks * L::kXStep + 3 * L::kKind + c * 1024) + row * 4;
          float v = (sh[sw] + sh[64 + sw]) + (sh[128 + sw] + sh[192 + sw]);
          const float with = sh[sw * 64 + 3];
          if (sw == 2) v += with;
          else if (p.dpre) v *= softplus_slope<T>(with);   // (uniform) gradients with respect to what the softplus was applied to
          split_store(reinterpret_cast<T*>(out_img + cell_bytes_off(t.cell, (uint32_t)p.E * (uint32_t)sizeof(T)) + (uint32_t)(e_wg0 + c) * (uint32_t)sizeof(T)), v, ok);
        }
      }
    };

    const int n = m_hi - m_lo;                              // blocks of the window
    if (sw < 3) {
      stage_bc(buf_of(0));
      stage_bc(buf_of(1));
      if (raw) split_landed<kRawCopies>(); else split_landed<kCopies>();
      widen(buf_of(0));
    } else {
      stage_x(buf_of(0));
      if constexpr (SLICED) link.wait_for(link_need_bwd_phases(p.sl_nbb - 1, p.sl_nbb, PH));
      copy_bot(buf_of(0));
      stage_x(buf_of(1));
      split_landed<kXCopies>();
    }
    if constexpr (!SX) {
      fetch_vals();
      split_vals_put<T, 4, CW, SG>(vals, lds + buf_of(0), sw, lane);
      fetch_vals();
    }
    __syncthreads();
    uint32_t done = 0;                                      // phases of the window whose rows are in memory, as the neighbour was told
    bool pending = false;                                   // (uniform) rows are on their way to memory, and the neighbour has not been told
    int par = 0;
    for (int j = 0; j < n; ++j) {                           // block n - 1 - j of the window is being swept
#pragma unroll
      for (int ph = 0; ph < PH; ++ph) {
        const bool first = ph == 0 && j == 0;
        const int kp = ph == 0 ? kCK : kCK - XS * ph;       // first step of the phase that ended at the last barrier (kCK: of the block swept before, 4 steps on)
        if constexpr (!SX) {                                // (in place a phase before their block, like all operands)
          if (ph == 0 && j + 1 < n) {
            split_vals_put<T, 4, CW, SG>(vals, lds + buf_of(j + 1), sw, lane);
            if (j + 2 < n) fetch_vals();
          }
        }
        if (sw < 3) {
          if (!first) {
            send_sums(cq, kp, par ^ 1);
            send_results(oq, kp, par ^ 1);
          }
          if (ph == 0) {                                    // block j + 1 has landed; the block fetched behind it, and what was stored since, may be under way
            stage_bc(buf_of(j + 2));
            if (raw) { if (j == 0) split_landed<kRawCopies>(); else { if (sw == 2) split_landed<PH * kStores2 + kRawCopies>(); else split_landed<PH * kStores + kRawCopies>(); } }
            else { if (j == 0) split_landed<kCopies>(); else { if (sw == 2) split_landed<PH * kStores2 + kCopies>(); else split_landed<PH * kStores + kCopies>(); } }
            widen(buf_of(j + 1));
          }
        } else {
          const bool told = pending;
          if (told) {                                       // rows sent in the phase before have arrived by now, or soon will: the neighbour is told
            if (ph == 2 % PH) split_landed<kXCopies>(); else staging_landed();   // (x and its like were fetched behind them in phase 1)
            if constexpr (SLICED) link.publish(++done);
            pending = false;
          }
          const bool rows_out = p.nbands > 1 && !first, bot_in = ph == PH - 1 && j + 1 < n;
          // Boundary rows in before rows out, so that the wait for the former leaves the latter under way -- unless the
          // neighbour is not there yet
          bool late = false;
          if constexpr (SLICED) late = bot_in && !link.ready(link_need_bwd_phases(n - 2 - j, n, PH));
          if (late && rows_out) {
            send_rows(rq, kp, par ^ 1);
            staging_landed();
            if constexpr (SLICED) link.publish(++done);
          }
          if (bot_in) {
            if constexpr (SLICED) link.wait_for(link_need_bwd_phases(n - 2 - j, n, PH));
            copy_bot(buf_of(j + 1));
          }
          if (!late && rows_out) {
            send_rows(rq, kp, par ^ 1);
            pending = true;
          }
          if (ph == 1) stage_x(buf_of(j + 2));
          // x and its like of block j + 1 have landed (workgroups of 8: with the lower boundary rows, in the phase before), and so have those rows
          if (PH == 2 && ph == 0) { if (SLICED && told && pending) split_landed<2>(); else if (pending) split_landed<1>(); else staging_landed(); }
          if (bot_in) {
            constexpr int behind = PH == 2 ? kXCopies : 0;
            if (pending) split_landed<behind + 1>(); else split_landed<behind>();
          }
        }
        __syncthreads();
        par ^= 1;
      }
      rq = rq.moved(p, -kCK);
      cq = cq.moved(p, -kCK);
      oq = oq.moved(p, -kCK);
    }
    if (sw < 3) {
      send_sums(cq, kCK, par ^ 1);
      send_results(oq, kCK, par ^ 1);
    } else {
      if (p.nbands > 1) send_rows(rq, kCK, par ^ 1);
      if constexpr (SLICED) { staging_landed(); link.publish((uint32_t)(PH * n)); }
    }
    staging_landed();                                       // (see the forward)
  }
  bool broken = false;
  if constexpr (SLICED) {   // only the wave that waits knows of a wait given up: it tells the others (the staging buffers are free now)
    if ((int)threadIdx.x == link.pub) *reinterpret_cast<volatile uint32_t*>(lds) = link.broken() || link_poll(p.link_err) != 0u ? 1u : 0u;   // (also a workgroup of the forward sweep that rebuilt the snapshots for this launch)
    staging_landed();
    __syncthreads();
    broken = *reinterpret_cast<volatile uint32_t*>(lds) != 0u;
    if (broken) poison_band<T>(p, my_band, b, e_wg0, CW, p.dx, p.ddT, p.ddL);
  }

  // ---- sums over positions: reduce over the rows of the band (the 16 lanes of a group)
  float red[9];
#pragma unroll
  for (int w = 0; w < 4; ++w) { red[w] = accAT[w]; red[4 + w] = accAL[w]; }
  red[8] = broken ? __builtin_nanf("") : accD;
  if (broken) { red[0] = __builtin_nanf(""); red[4] = __builtin_nanf(""); }   // (d_AT, d_AL, d_D of the channel say so too)
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    float v = red[k];
#pragma unroll
    for (int off = kHB >> 1; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    red[k] = v;
  }
  if (ch_ok && r == 0) {
    const int64_t slot_e = ((int64_t)b * p.pa_slots + (SLICED ? my_band : 0)) * p.E + e;
    float* pa = p.pA + slot_e * (2 * kN);
#pragma unroll
    for (int w = 0; w < 4; ++w) { pa[state_of[w]] = red[w]; pa[kN + state_of[w]] = red[4 + w]; }
    if (g == 0) p.pD[slot_e] = red[8];
  }
}
