// Host side of m2drows.hip, for the launch logic of m2dscan.hip.
#ifndef M2D_ROWS_H
#define M2D_ROWS_H
#include <hip/hip_runtime.h>
#include <atomic>
#include <stddef.h>
#include <stdint.h>

// A kernel that needs more than 64 KB of dynamic LDS has to be told so once per device (each
// device loads its own copy of the code object).  `seen` holds one bit per device ordinal.
inline bool allow_dynamic_lds(const void* kernel, size_t bytes, std::atomic<uint64_t>& seen) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  const uint64_t bit = 1ull << (dev & 63);
  if (seen.load(std::memory_order_relaxed) & bit) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return false;
  seen.fetch_or(bit, std::memory_order_relaxed);
  return true;
}

namespace m2drows {

// A problem as m2d_fwd_rows_kernel sees it.
struct Args {
  const void *x, *dT, *dL;          // (B,H,W,E)
  const void *AT, *AL, *D;          // the caller's; raw: fp32 A_log and D as a module holds them
  const float* rec;                 // packed fp32 records of B_T, B_L, C, or null:
  const void *BT, *BL, *C;          // ... (B,H,W,16) in the tensors' type
  void* y;
  float* wrap;                      // [rounds - 1][B][groups of 16 channels][W][64] float4: last rows of the last bands of a round
  uint32_t* link_err;               // error word of a linked sweep's workspace, which this kernel leaves at 0: nothing waits here; null where the plan has none
  int B, H, W, E, flip, raw;
  // the plan (make_plan)
  int nbands, nblk, rounds, stride, groups, images;
};
// Rows of a band, bands side by side in a workgroup (of 8 sweeping waves: the rest is channel groups); rows = 0: not for these kernels
struct Plan {
  int rows = 0, slots = 0;
  int nbands, nblk, rounds, stride, groups, images, workgroups;
  size_t wrap_bytes;
  int64_t cells;                    // cells that a sweeping wave works through one after the other
};
Plan make_plan(int B, int H, int W, int E, int compute_units);
// 0, or the HIP error of the launch
int launch_fwd(const Plan& plan, Args args, bool bf16, hipStream_t stream);

}  // namespace m2drows
#endif
