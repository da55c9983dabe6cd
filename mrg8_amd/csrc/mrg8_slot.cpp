#include "mrg8_slot.hpp"

#include <algorithm>
#include <cstring>

#include "../../include/mrg8.h"

namespace mrg8 {

namespace {
size_t align_up(size_t x, size_t a) { return (x + a - 1) / a * a; }

// Byte offsets of the tables behind `n` segments (see mrg8_device.hpp).
size_t tile_begin_offset(uint32_t n) { return sizeof(BatchHeader) + sizeof(BatchSegment) * (size_t)n; }
size_t tile_seg_offset(uint32_t n) { return tile_begin_offset(n) + sizeof(uint64_t) * ((size_t)n + 1); }
}  // namespace

int BatchSlot::init(DeviceContext* ctx, uint32_t cap, uint64_t max_tiles, const uint32_t* states) {
  release();
  ctx_ = ctx;
  cap_ = cap;
  max_tiles_ = max_tiles;
  states_ = states;
  const size_t total = align_up(tile_seg_offset(cap) + sizeof(uint32_t) * (size_t)max_tiles, 256);
  DeviceGuard dg(ctx->device);
  hipError_t e = hipMalloc((void**)&dmem_, total);
  // coherent: the staging kernel reads it over the bus every run, never a
  // copy the GPU cached from an earlier run of this slot
  if (e == hipSuccess) e = hipHostMalloc((void**)&hmem_, total, hipHostMallocCoherent);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&staged_, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&run_done_, hipEventDisableTiming);
  if (e != hipSuccess) {
    int rc = hip_fail(e, "batch slot allocation");
    release();
    return rc;
  }
  std::memset(hmem_, 0, total);
  h_segs_ = reinterpret_cast<BatchSegment*>(hmem_ + sizeof(BatchHeader));
  return MRG8_OK;
}

void BatchSlot::release() {
  if (!ctx_) return;
  DeviceGuard dg(ctx_->device);
  if (copy_pending_ && staged_) (void)hipEventSynchronize(staged_);
  if (run_pending_ && run_done_) (void)wait_done();
  for (Captured& c : captured_) c.release();
  if (staged_) (void)hipEventDestroy(staged_);
  if (run_done_) (void)hipEventDestroy(run_done_);
  if (hmem_) (void)hipHostFree(hmem_);
  if (dmem_) (void)hipFree(dmem_);
  staged_ = run_done_ = nullptr;
  hmem_ = dmem_ = nullptr;
  copy_pending_ = run_pending_ = false;
  last_stream_ = nullptr;
  last_marked_ = true;
  last_queue_ = false;
  ctx_ = nullptr;
}

int BatchSlot::wait_staging() {
  if (!copy_pending_) return MRG8_OK;
  DeviceGuard dg(ctx_->device);
  hipError_t e = hipEventSynchronize(staged_);
  if (e != hipSuccess) return hip_fail(e, "hipEventSynchronize(staging)");
  copy_pending_ = false;
  return MRG8_OK;
}

size_t batch_block_bytes(uint32_t count, uint64_t ntiles) {
  return tile_seg_offset(count) + sizeof(uint32_t) * (size_t)ntiles;
}

size_t layout_batch_block(uint8_t* mem, uint32_t count, uint64_t tile, uint64_t max_tiles, BatchWork* work) {
  const size_t tb_off = tile_begin_offset(count), ts_off = tile_seg_offset(count);
  BatchHeader* hdr = reinterpret_cast<BatchHeader*>(mem);
  const BatchSegment* segs = reinterpret_cast<const BatchSegment*>(mem + sizeof(BatchHeader));
  uint64_t* tiles = reinterpret_cast<uint64_t*>(mem + tb_off);
  uint32_t* tile_seg = reinterpret_cast<uint32_t*>(mem + ts_off);
  uint64_t t = 0;
  BatchWork w;
  auto add = [&](uint64_t outputs, uint64_t times) {
    const uint64_t runs = outputs / kShortRunOutputs + (outputs % kShortRunOutputs != 0);
    w.runs += runs * times;
    w.longest = std::max(w.longest, runs);
  };
  for (uint32_t i = 0; i < count; ++i) {
    tiles[i] = t;
    const uint64_t c = segs[i].count, head = segment_head(segs[i].out, segs[i].format, c, tile);
    const uint64_t n = head_tiles(head, c, tile);
    w.weight += c * (segs[i].format == 2 ? 1 : kShortDouble);
    if (n == 1) {
      add(c, 1);
    } else if (n) {  // the first tile with the head, whole ones, the last
      add(head + tile, 1);
      if (n > 2) add(tile, n - 2);
      add(c - head - (n - 1) * tile, 1);
    }
    const uint64_t end = std::min<uint64_t>(t + n, max_tiles);
    if (t < end) std::fill(tile_seg + t, tile_seg + end, i);
    t += n;
  }
  tiles[count] = t;
  hdr->nsegs = count;
  hdr->ntiles = t;
  hdr->tile_begin_off = tb_off;
  hdr->tile_seg_off = ts_off;
  hdr->queue_next = 0;  // k_batch_queue's counter starts at zero
  w.tiles = t;
  *work = w;
  return batch_block_bytes(count, std::min<uint64_t>(t, max_tiles));
}

uint64_t BatchSlot::finalise(uint32_t count, uint64_t tile) {
  used_bytes_ = layout_batch_block(hmem_, count, tile, max_tiles_, &work_);
  count_ = count;
  dirty_ = true;
  return work_.tiles;
}

BatchArgs batch_args(const DeviceContext& ctx, const uint8_t* block, const LaunchConfig& cfg, const uint32_t* states) {
  BatchArgs a{};
  a.block = block;
  a.tile = cfg.tile;
  a.states = states;
  a.lane = ctx.tables.lane;
  a.digits = ctx.tables.digits;
  a.xcds = (uint32_t)ctx.num_xcc;
  a.xcd_group = xcd_run_blocks(ctx, cfg.blocks_per_cu ? cfg.block_threads : tile_block_threads(cfg.block_threads));
  a.mfma_a = ctx.tables.mfma_a;
  a.mfma_c = ctx.tables.mfma_c;
  a.mfma_skip_a = ctx.tables.mfma_skip_a;
  a.mfma_skip_k = ctx.tables.mfma_skip_k;
  a.min_waves = (uint32_t)ctx.num_cu * 4;  // one per SIMD
  return a;
}

// A striding grid of at least eight tiles for each SIMD takes the short-tile
// kernel while its tiles average up to 1024 words or 128 doubles.  MI355X, us
// per run, 63-bit offsets, striding (256 x 8 | 256 x 4) against short:
//   tiles, outputs        striding       short
//   65536 x  256 words    30.6 | 28.7    20.9
//   65536 x   16 words    20.6 | 19.9    16.2
//   65536 x 1024 words    72.8 | 70.5    61.5
//   51205 x  128 words    19.8 | 19.1    17.2
//    8192 x  256 words    12.1 |  8.8     7.1
//    8192 x 1024 words    17.2 | 14.2    13.2
//    4096 x  512 words     8.7 |  8.5     8.4   (1024: 10.5 | 10.3, 12.0)
//   65536 x  128 doubles  23.5 | 22.5    21.2   (256: 34.1 | 30.8, 31.4)
//   32768 x  128 doubles  17.0 | 13.8    13.7   (256: 20.5 | 17.6, 18.3)
// Doubles are bound by their stores from there on, and the vector kernel, with
// more waves per SIMD, has more of them in flight (32768 x 512: 29 against 34).
// A wave works on eight tiles until the longest of them is done, so the longest may
// take 2.8 times the mean's runs of 256 outputs (or two of them, which cost
// little more than one).  us, 256 x 8, striding against short:
//   longest / mean   tiles                               striding  short
//   2.0              16384: 512 words, 15872: 16           12.4     10.3
//   2.6              65536, log-uniform in 8 to 1023       46.4     42.3
//   2.9              65536: 8192 of 1024, the rest 16      34.6     40.1
//   3.7              65536: 2048 of 1024, the rest 16      26.8     33.8
//   3.9              65536, log-uniform in 8 to 2047       58.5     69.1
//   6.8              32768: 128 of 2048, the rest 128      19.6     32.8
//   43               32768: 128 of 16384, the rest 128     46.4    192
BatchKernel batch_kernel(const DeviceContext& ctx, const LaunchConfig& cfg, const BatchWork& work) {
  if (cfg.blocks_per_cu == 0) return BatchKernel::Tiles;
  if (cfg.blocks_per_cu < 0) return BatchKernel::Queue;
  const bool many = work.tiles >= 8ull * 4 * ctx.num_cu, is_short = work.weight <= 1024 * work.tiles;
  const bool even = work.longest <= 2 || 5 * work.longest * work.tiles <= 14 * work.runs;
  return ctx.tables.mfma_a && many && is_short && even ? BatchKernel::Short : BatchKernel::Striding;
}

hipError_t launch_batch_kernel(const DeviceContext& ctx, const BatchArgs& a, const LaunchConfig& cfg, BatchKernel kernel,
                               uint64_t ntiles, hipStream_t stream) {
  switch (kernel) {
    case BatchKernel::Tiles: return launch_batch_tiles(a, ntiles, tile_block_threads(cfg.block_threads), stream);
    case BatchKernel::Queue: return launch_batch_queue(a, ctx.num_cu * -cfg.blocks_per_cu, cfg.block_threads, stream);
    case BatchKernel::Striding: return launch_batch(a, ctx.num_cu * cfg.blocks_per_cu, cfg.block_threads, stream);
    case BatchKernel::Short:
      // at most the three waves per SIMD that its registers allow: what a
      // larger grid costs to start is not hidden (65536 x 256 words, 12 waves
      // per CU 20.9 us, 8 22.5, 16 24.6)
      return launch_batch_short(a, (uint32_t)(ctx.num_cu * std::min(12, cfg.blocks_per_cu * (cfg.block_threads / 64))), stream);
  }
  return hipErrorInvalidValue;
}

hipError_t BatchSlot::launch(const LaunchConfig& cfg, hipStream_t stream) const {
  return launch_batch_kernel(*ctx_, batch_args(*ctx_, dmem_, cfg, states_), cfg,
                             batch_kernel(*ctx_, cfg, work_), work_.tiles, stream);
}

void BatchSlot::Captured::release() {
  if (exec) (void)hipGraphExecDestroy(exec);
  if (graph) (void)hipGraphDestroy(graph);
  *this = Captured{};
}

// A one-tile-per-wave grid depends on the tile count, a persistent one does
// not (its kernel reads the count from the device block).  The striding
// grid's kernel depends on how short the staged tiles are: it has a graph for
// each, so that restaging from one kind to the other neither waits for the
// runs before it nor captures anew (165 us of host time a run, 52 us without).
int BatchSlot::capture(const LaunchConfig& cfg, hipGraphExec_t* exec) {
  Captured& c = captured_[batch_kernel(*ctx_, cfg, work_) == BatchKernel::Short ? 0 : 1];
  if (c.exec && cfg.block_threads == c.cfg.block_threads && cfg.blocks_per_cu == c.cfg.blocks_per_cu &&
      cfg.tile == c.cfg.tile && (cfg.blocks_per_cu != 0 || c.ntiles == work_.tiles)) {
    *exec = c.exec;
    return MRG8_OK;
  }
  if (int rc = wait_done()) return rc;  // the old graph may still be running
  c.release();
  hipStream_t cs = nullptr;
  hipError_t e = hipStreamCreateWithFlags(&cs, hipStreamNonBlocking);
  if (e != hipSuccess) return hip_fail(e, "hipStreamCreate(capture)");
  e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
  if (e == hipSuccess) {
    hipError_t e1 = launch(cfg, cs);
    hipError_t e2 = hipStreamEndCapture(cs, &c.graph);
    e = e1 != hipSuccess ? e1 : e2;
  }
  if (e == hipSuccess) e = hipGraphInstantiate(&c.exec, c.graph, nullptr, nullptr, 0);
  (void)hipStreamDestroy(cs);
  if (e != hipSuccess) {
    c.release();
    return hip_fail(e, "graph capture");
  }
  c.cfg = cfg;
  c.ntiles = work_.tiles;
  *exec = c.exec;
  return MRG8_OK;
}

hipError_t BatchSlot::mark_last_run() {
  if (!run_pending_ || last_marked_) return hipSuccess;
  hipError_t e = hipEventRecord(run_done_, last_stream_);
  if (e == hipSuccess) last_marked_ = true;
  return e;
}

int BatchSlot::run(const LaunchConfig& cfg, hipStream_t stream, bool graph, bool track) {
  if (count_ == 0 || work_.tiles == 0) return MRG8_OK;
  if (work_.tiles > max_tiles_) return fail(MRG8_ERR_CAPACITY, "staged work needs more than max_tiles tiles");
  const uint64_t wpb = (uint64_t)cfg.block_threads / 64;
  if (cfg.blocks_per_cu == 0) {  // one wave per tile: the grid (work-items in total) is a 32-bit quantity
    if ((work_.tiles + wpb - 1) / wpb * (uint64_t)cfg.block_threads > 0xffffffffull)
      return fail(MRG8_ERR_CAPACITY, "%llu tiles need more than 2^32 - 1 work-items at one tile per wave; use larger "
                  "tiles or a persistent grid", (unsigned long long)work_.tiles);
  } else if (cfg.blocks_per_cu < 0) {  // a group's number, the grid's blocks plus the work counter, is 32 bits
    if ((work_.tiles + wpb - 1) / wpb + (uint64_t)ctx_->num_cu * (uint64_t)-cfg.blocks_per_cu > 0xffffffffull)
      return fail(MRG8_ERR_CAPACITY, "%llu tiles are more groups than the address-order grid counts; use larger tiles",
                  (unsigned long long)work_.tiles);
  }
  DeviceGuard dg(ctx_->device);
  hipGraphExec_t exec = nullptr;
  int rc = graph ? capture(cfg, &exec) : MRG8_OK;
  if (rc) return rc;
  hipError_t e = hipSuccess;
  // The device block may be overwritten once this slot's previous launch has
  // finished, and an address-order grid (blocks_per_cu < 0) may start only
  // after the previous one has reset the work counter in it: on the same
  // stream both are ordered after the previous launch; on another stream
  // they wait for it.  Runs next to an address-order run wait as well, so
  // that two such runs are never apart by one unordered run in between.
  if (run_pending_ && stream != last_stream_ && (dirty_ || cfg.blocks_per_cu < 0 || last_queue_)) {
    if (mark_last_run() == hipSuccess) e = hipStreamWaitEvent(stream, run_done_, 0);
    else if ((rc = wait_done()) != MRG8_OK) return rc;  // the last stream no longer accepts work
    if (e != hipSuccess) return hip_fail(e, "hipStreamWaitEvent(previous run)");
  }
  if (dirty_) {  // runs of an unchanged batch copy nothing
    e = launch_stage(hmem_, dmem_, used_bytes_, stream);
    if (e == hipSuccess) e = hipEventRecord(staged_, stream);
    if (e != hipSuccess) return hip_fail(e, "batch staging copy");
    copy_pending_ = true;
    dirty_ = false;
  }
  e = graph ? hipGraphLaunch(exec, stream) : launch(cfg, stream);
  if (e != hipSuccess) return hip_fail(e, graph ? "hipGraphLaunch" : "batch launch");
  run_pending_ = true;
  last_stream_ = stream;
  last_marked_ = false;
  last_queue_ = cfg.blocks_per_cu < 0;
  if (track && (e = mark_last_run()) != hipSuccess) return hip_fail(e, "hipEventRecord(run)");
  return MRG8_OK;
}

bool BatchSlot::done() {
  if (!run_pending_) return true;
  DeviceGuard dg(ctx_->device);
  if (mark_last_run() != hipSuccess) return false;
  if (hipEventQuery(run_done_) == hipSuccess) {
    run_pending_ = false;
    copy_pending_ = false;
    return true;
  }
  return false;
}

int BatchSlot::wait_done() {
  if (!run_pending_) return MRG8_OK;
  DeviceGuard dg(ctx_->device);
  hipError_t e = mark_last_run();
  e = e == hipSuccess ? hipEventSynchronize(run_done_) : hipDeviceSynchronize();
  if (e != hipSuccess) return hip_fail(e, "waiting for the last batch run");
  run_pending_ = false;
  copy_pending_ = false;
  return MRG8_OK;
}

}  // namespace mrg8
