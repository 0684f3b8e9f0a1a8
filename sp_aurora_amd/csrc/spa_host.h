// Host-side helpers shared by the launchers: per-device facts read once, the
// dynamic-LDS attribute of a kernel set once per device, and the kernel-variant
// overrides of spa_tune().  Nothing here allocates device memory.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

constexpr int SPA_MAX_DEVICES = 64;

// Variant overrides for experiments and tests (set through spa_tune, never read from the
// environment); 0 = the library's own choice.
enum {
  SPA_KNOB_FWD_GROUPS = 0,    // 1 | 2 | 4 wave groups per forward workgroup (4: block calls)
  SPA_KNOB_FWD_SHARE = 1,     // 1: private K/V buffers per group, 2: 256-row workgroups sharing them
  SPA_KNOB_BWD_DQ_WAVES = 2,  // the backward's dq kernel: 4 | 8 waves, 32 rows each; 20 | 24: 4 | 8 waves, pairs share 32 rows
  SPA_KNOB_BWD_DKDV_FORM = 3, // dk/dv kernel: 1 compiler-scheduled MFMAs at D = 128 (test twin), 2 | 3: 64 | 128 keys a workgroup, 4 | 5: their twins
  SPA_KNOB_FWD32_SPLIT = 4,   // 1: never the fp32 kernels of 32 rows whose waves share the tiles, 2: always
  SPA_KNOB_FEW_ROWS = 5,     // 1: a forward of up to 16 unmasked query rows stays on the kernels for long rows
  SPA_KNOB_COUNT = 6
};
extern std::atomic<int> g_spa_knob[SPA_KNOB_COUNT];
static inline int spa_knob(int k) { return g_spa_knob[k].load(std::memory_order_relaxed); }

// The current device, or -1.
static inline int spa_current_device() {
  int dev = -1;
  return hipGetDevice(&dev) == hipSuccess ? dev : -1;
}

// Compute units of the current device (256 when the query fails), cached per device.
static inline int spa_device_cus() {
  static std::atomic<int> cache[SPA_MAX_DEVICES];
  const int dev = spa_current_device();
  if (dev >= 0 && dev < SPA_MAX_DEVICES) {
    const int c = cache[dev].load(std::memory_order_relaxed);
    if (c > 0) return c;
  }
  int n = 0;
  if (dev < 0 || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
  if (dev >= 0 && dev < SPA_MAX_DEVICES) cache[dev].store(n, std::memory_order_relaxed);
  return n;
}

// hipFuncAttributeMaxDynamicSharedMemorySize of `kernel`, set the first time the kernel is
// launched on a device instead of at every launch.  One instantiation (and one flag word)
// per kernel: the kernel is a template VALUE parameter.
template <auto kernel>
hipError_t spa_allow_dynamic_lds(int smem) {
  static std::atomic<unsigned long long> ready{0};  // bit d: done on device d
  const int dev = spa_current_device();
  if (dev >= 0 && dev < SPA_MAX_DEVICES && ((ready.load(std::memory_order_acquire) >> dev) & 1ull)) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (e == hipSuccess && dev >= 0 && dev < SPA_MAX_DEVICES) ready.fetch_or(1ull << dev, std::memory_order_release);
  return e;
}

// Grid of an attention launch with `tiles` workgroups per (batch, head) pair: x = the pairs of one group, y = tiles, z =
// groups, dispatched in that order, so that a group's tiles run side by side and then the next group's.  A head's tiles
// share its streamed tensors in the L2 of the XCD they run on (round-robin placement: x % 8 while x has a multiple of 8 pairs), but
// only while they run at the same time: with more pairs than CUs and no groups, every tile of a head reads them from memory
// again.  A group holds as many pairs per XCD as fill its CUs with their tiles, at least 4 (fewer were not measured to help
// long rows, whose tiles walk the keys in step).
static inline dim3 spa_head_groups(int64_t pairs, int tiles) {
  const int64_t per_xcd = (spa_device_cus() / 8 + tiles - 1) / tiles;
  const int64_t group = 8 * (per_xcd > 4 ? per_xcd : 4);
  if (pairs <= group) return dim3((unsigned)pairs, (unsigned)tiles, 1);
  const int64_t n = (pairs + group - 1) / group;
  if (n < 4 || n > 65535) return dim3((unsigned)pairs, (unsigned)tiles, 1);
  return dim3((unsigned)group, (unsigned)tiles, (unsigned)n);
}

// Grid of a launch over a packed variable-length batch: sequences x tiles of the longest sequence, as for fixed lengths
// (numbered = 0), or one workgroup per head and tile number, heads first (sequence_tile).  A workgroup of the first that finds no
// rows costs 0.5 us of a CU; one of the second searches for 0.4 us (24 sequences) to 3 us (2000), but the tiles of a long sequence
// run side by side and the heavy ones first.  So numbers where the mean sequence is long and the other grid has more workgroups (us, forward /
// backward, H = 16, D = 128, causal: 24 sequences of 500 to 2000 rows 264 / 919, by sequences 278 / 1005; 64 of 200 to 2000 570 / 1977 and
// 574 / 2129), by sequences for short ones (2000 of 32 to 256 rows 1083 / 4276, numbered 1918 / 7779; 200 of 100 to 1000, H = 8,
// D = 64, 193 / 616 and 229 / 698) until a bound far above the lengths that are there makes that grid eight times the other (512 of
// 32 to 256 rows with a bound of 2048 378 / 1463 and 407 / 1705, of 4096 506 / 1880).
static inline bool spa_varlen_grid(int H, int nseq, int64_t total_rows, int64_t longest, int rows, unsigned z, dim3& grid, int& numbered) {
  const int64_t tiles = (longest + rows - 1) / rows, numbers = total_rows / rows + nseq, pairs = (int64_t)nseq * H;
  const bool short_rows = total_rows < (int64_t)nseq * 640;
  numbered = tiles * nseq > (short_rows ? 8 : 1) * numbers || tiles > 65535 || pairs > 0x7fffffffLL;
  if (!numbered) {
    grid = z == 1 ? spa_head_groups(pairs, (int)tiles) : dim3((unsigned)pairs, (unsigned)tiles, z);
    return true;
  }
  const int64_t n = numbers * H;
  if (n <= 0 || n > 0x7fffffffLL) return false;
  grid = dim3((unsigned)n, 1, z);
  return true;
}
