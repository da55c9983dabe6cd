// Shared host-side pieces of libmrg8_amd: per-device context, error helpers,
// single-stream fill.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <mutex>
#include <vector>

#include "../../include/mrg8.h"
#include "mrg8_device.hpp"

namespace mrg8 {

struct TunedShape {
  bool valid = false;
  int block_threads = 0;
  int per_lane = 0;
  uint64_t tile = 0;
};

struct DeviceContext {
  int device = 0;
  int num_cu = 0;
  int num_xcc = 1;  // XCDs the dispatcher deals blocks to in turn
  DeviceTables tables;
  TunedShape tuned[3][64];  // [format][floor(log2 n)], set by mrg8_tune_fill
  std::mutex tuned_mu;      // guards `tuned` (fills on other handles read it)
  std::mutex wide_mu;       // guards the first-use build of tables.wide
  uint8_t* noalloc_scratch = nullptr;  // this device's copy of the fixed scratch area
};

// Blocks per XCD run for kernels that map blocks through xcd_block: runs of
// 32768 threads (64 blocks of 512) on a device with more than one XCD.
inline uint32_t xcd_run_blocks(const DeviceContext& ctx, int block_threads) {
  uint32_t run = ctx.num_xcc > 1 && block_threads > 0 ? (uint32_t)std::max(1, 32768 / block_threads) : 1;
  while (run & (run - 1)) run &= run - 1;  // xcd_block's counts are powers of two
  return run;
}

// Threads per block of a one-tile-per-wave grid with these configured ones.
inline int tile_block_threads(int block_threads) { return std::min(block_threads, kTileBlockThreads); }

// A new batch's launch configuration.
constexpr mrg8_batch_config kDefaultBatchConfig{kTileBlockThreads, 0, 2048};

// What mrg8_batch_autotune times: threads per block x waves per CU x tile size.
std::vector<mrg8_batch_config> batch_candidates();

// Builds the table of byte positions kJumpPositions..kWidePositions-1 on the
// context's device if it is not there yet.
int ensure_wide_table(DeviceContext& ctx);

// Records `fmt` as this thread's last error message and returns `code`.
int fail(int code, const char* fmt, ...);
int hip_fail(hipError_t e, const char* what);
void clear_error();

const JumpTable& host_jump_table();
const DigitTable& host_digit_table();
int device_context(int device, DeviceContext** out);
// The device's context if mrg8_init_device (or any call that needs it) has
// created it, else null; creates nothing.
DeviceContext* existing_device_context(int device);
bool state_valid(const uint32_t st[8]);
int format_size(int format);

// Fills dptr[0..n) with stream positions offset..offset+n-1 of the stream
// whose state is `state`; stream-ordered.  block_threads/tile/per_lane 0 =
// default.
int fill_device(DeviceContext& ctx, const uint32_t state[8], uint64_t offset, void* dptr, uint64_t n, int format,
                hipStream_t stream, int block_threads, uint64_t tile, int per_lane);

// The same without a look at the tuned shapes; n >= 1.
int fill_shaped(DeviceContext& ctx, const uint32_t state[8], uint64_t offset, void* dptr, uint64_t n, int format,
                hipStream_t stream, int block_threads, uint64_t tile, int per_lane);

// What mrg8_tune_fill times: the automatic shape (not valid, all 0) first.
std::vector<TunedShape> fill_candidates(int format);

// A grid's work-items are a 32-bit quantity.
constexpr uint64_t kMaxGridWaves = 0xffffffffull / 64;

// Automatic shapes: threads per block and outputs per wave of the vector
// kernel (where they are 0), and tiles (of `tile` outputs) per wave of the
// matrix-core fill.
void default_shape(const DeviceContext& ctx, uint64_t n, int format, int per_lane, int* block, uint64_t* tile);
uint64_t mfma_tiles_per_wave(const DeviceContext& ctx, int format, uint64_t tile, uint64_t tiles);
// Blocks per XCD run of a vector-kernel fill (1: blocks in dispatch order).
uint32_t fill_xcd_group(const DeviceContext& ctx, int format, uint64_t waves, int block_threads, uint64_t tile);
// Whether the waves of a block of such a fill start their outputs together.
bool fill_in_step(uint32_t xcd_group, int block_threads, uint64_t tile);

// Batch descriptors (include/mrg8.h): checks a launch configuration; checks
// `count` descriptors and sums their tiles (of `tile` outputs) and outputs;
// converts them to the device segment layout (inline states).
int validate_batch_config(const mrg8_batch_config& c);
int check_descriptors(const mrg8_stream_desc* descs, uint32_t count, uint64_t tile, uint64_t* tiles,
                      uint64_t* total);
void write_segments(BatchSegment* segs, const mrg8_stream_desc* descs, uint32_t count);

// Device address of the library's fixed scratch area on the current device
// (taken once per device when its context is created).
int noalloc_scratch_address(uint8_t** ptr);

// RAII device switch.
class DeviceGuard {
 public:
  explicit DeviceGuard(int dev) : dev_(dev) {
    (void)hipGetDevice(&prev_);
    if (prev_ != dev_) (void)hipSetDevice(dev_);
  }
  ~DeviceGuard() {
    if (prev_ != dev_) (void)hipSetDevice(prev_);
  }

 private:
  int prev_ = 0, dev_ = 0;
};

// Host wall clock in seconds (steady).
double now_seconds();

}  // namespace mrg8
