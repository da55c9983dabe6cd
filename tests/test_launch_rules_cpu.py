"""The host's launch rules, called in the library with a device context made up here (256 CUs, 8 XCDs, no device)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "mrg8_amd", "libmrg8_amd.so")
ROCM = "/opt/rocm"

pytestmark = pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(ROCM + "/include/hip/hip_runtime.h"),
                                reason="needs g++ and the HIP headers")

HEAD = r"""
#include <cstdio>
#include <cstring>
#include <vector>
#include "mrg8_slot.hpp"
using namespace mrg8;
static int bad = 0;
#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); bad = 1; } } while (0)
"""

MAIN = r"""
int main() {
  static DeviceContext ctx;
  ctx.num_cu = 256;
  ctx.num_xcc = 8;
  static uint32_t table;
  ctx.tables.mfma_a = &table;
  run(ctx);
  if (!bad) std::printf("ok\n");
  return bad;
}
"""


def check(tmp_path, body):
    src, exe = tmp_path / "rules.cpp", tmp_path / "rules"
    src.write_text(HEAD + "#line 1\n" + body + MAIN)
    r = subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{ROCM}/include",
                        "-I" + os.path.join(ROOT, "mrg8_amd", "csrc"), str(src), LIB, f"-L{ROCM}/lib", "-lamdhip64",
                        "-Wl,-rpath," + os.path.dirname(LIB), f"-Wl,-rpath,{ROCM}/lib", "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr


def test_short_tile_kernel_takes_even_batches_only(tmp_path):
    """Batches of 10240 segments on a striding grid: the short-tile kernel works
    on eight tiles until the longest is done, so one long tile among many short
    ones goes to the other striding kernel, whatever the average."""
    check(tmp_path, r"""
static BatchKernel kernel_of(const DeviceContext& ctx, uint64_t usual, uint64_t other, uint32_t every, int format, uint64_t tile,
                             uint32_t count = 10240, uint64_t misalign = 0) {
  std::vector<uint8_t> mem(batch_block_bytes(count, 1 << 20));
  BatchSegment* segs = reinterpret_cast<BatchSegment*>(mem.data() + sizeof(BatchHeader));
  for (uint32_t i = 0; i < count; ++i) {
    segs[i].count = every && i % every == 0 ? other : usual;
    segs[i].out = reinterpret_cast<void*>((uintptr_t(1) << 40) + (uintptr_t(i) << 24) + misalign);
    segs[i].format = format;
  }
  BatchWork work;
  layout_batch_block(mem.data(), count, tile, 1 << 20, &work);
  LaunchConfig cfg;
  cfg.block_threads = 256;
  cfg.blocks_per_cu = 8;
  cfg.tile = tile;
  return batch_kernel(ctx, cfg, work);
}
static void run(const DeviceContext& ctx) {
  for (uint64_t n : {1, 16, 256, 257, 512, 1024}) CHECK(kernel_of(ctx, n, 0, 0, 2, 2048) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 1025, 0, 0, 2, 2048) == BatchKernel::Striding);
  CHECK(kernel_of(ctx, 128, 0, 0, 0, 2048) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 129, 0, 0, 0, 2048) == BatchKernel::Striding);
  CHECK(kernel_of(ctx, 16, 0, 0, 2, 2048, 8191) == BatchKernel::Striding);
  // two runs of 256 are always close enough; from three on, 2.8 times the average
  CHECK(kernel_of(ctx, 16, 512, 10240, 2, 2048) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 16, 513, 10240, 2, 2048) == BatchKernel::Striding);
  CHECK(kernel_of(ctx, 16, 1024, 2, 2, 2048) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 16, 1024, 8, 2, 2048) == BatchKernel::Striding);
  CHECK(kernel_of(ctx, 64, 16384, 17, 2, 16384) == BatchKernel::Striding);
  CHECK(kernel_of(ctx, 64, 16384, 10240, 2, 16384) == BatchKernel::Striding);
  // long segments cut into equal tiles, and one whose first tile has a long head
  CHECK(kernel_of(ctx, 1024 * 20, 0, 0, 2, 1024) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 1024 * 20, 0, 0, 2, 1024, 512) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 1024 * 20, 0, 0, 2, 1024, 10240, 8) == BatchKernel::Short);
  CHECK(kernel_of(ctx, 64, 1024 + 700, 10240, 2, 1024, 10240, 4 * 324) == BatchKernel::Striding);
}
""")


def test_xcd_runs_of_fills(tmp_path):
    """Only one-wave blocks of up to 2048 doubles run on the XCDs in runs below
    64 waves per CU; blocks of several waves in such runs start in step."""
    check(tmp_path, r"""
static void run(const DeviceContext& ctx) {
  CHECK(fill_xcd_group(ctx, MRG8_F64, 4096, 64, 1024) == 64);
  CHECK(fill_xcd_group(ctx, MRG8_F64, 4095, 64, 1024) == 1);
  CHECK(fill_xcd_group(ctx, MRG8_F64, 4096, 64, 2048) == 64 && fill_xcd_group(ctx, MRG8_F64, 16383, 64, 4096) == 1);
  CHECK(fill_xcd_group(ctx, MRG8_F64_01, 4096, 64, 65536) == 1);
  CHECK(fill_xcd_group(ctx, MRG8_F64, 4096, 256, 1024) == 1);
  CHECK(fill_xcd_group(ctx, MRG8_F64, 16383, 512, 2048) == 1);
  CHECK(fill_xcd_group(ctx, MRG8_F64, 16384, 512, 2048) == 64);
  CHECK(fill_xcd_group(ctx, MRG8_F64, 16384, 1024, 2048) == 32);
  CHECK(fill_xcd_group(ctx, MRG8_U32, 1 << 20, 256, 2048) == 1);
  CHECK(fill_in_step(64, 512, 2048) && fill_in_step(32, 1024, 8192));
  CHECK(!fill_in_step(1, 512, 2048) && !fill_in_step(64, 64, 2048));
  CHECK(!fill_in_step(64, 512, 1024) && !fill_in_step(64, 512, 16384));
}
""")


def test_fill_tuner_times_the_automatic_shape(tmp_path):
    """The automatic shape is a candidate, and so are the shapes that large fills of either kernel do best with."""
    check(tmp_path, r"""
static void run(const DeviceContext&) {
  for (int format : {MRG8_F64, MRG8_F64_01, MRG8_U32}) {
    const std::vector<TunedShape> all = fill_candidates(format);
    CHECK(!all[0].valid && !all[0].block_threads && !all[0].per_lane && !all[0].tile);
    bool short_waves = false, small_mfma = false;
    for (size_t i = 1; i < all.size(); ++i) {
      const TunedShape& c = all[i];
      CHECK(c.valid && c.block_threads >= 256 && c.tile);
      short_waves |= c.block_threads == 256 && c.per_lane == 4 && c.tile == 1024;
      small_mfma |= c.block_threads == 256 && c.per_lane == 32 && c.tile == 4096;
    }
    CHECK(short_waves && small_mfma);
  }
}
""")


def test_batch_tuner_times_no_launch_twice(tmp_path):
    """Candidates are valid and their launches differ; a one-tile-per-wave grid says the block size that it runs in,
    and so does the configuration of a new batch."""
    check(tmp_path, r"""
static void run(const DeviceContext&) {
  const std::vector<mrg8_batch_config> all = batch_candidates();
  bool kinds[3] = {};
  for (size_t i = 0; i < all.size(); ++i) {
    const mrg8_batch_config& c = all[i];
    CHECK(validate_batch_config(c) == MRG8_OK);
    CHECK(c.blocks_per_cu || tile_block_threads(c.block_threads) == c.block_threads);
    for (size_t j = 0; j < i; ++j) CHECK(std::memcmp(&all[j], &c, sizeof c) != 0);
    kinds[(c.blocks_per_cu > 0) - (c.blocks_per_cu < 0) + 1] = true;
  }
  CHECK(kinds[0] && kinds[1] && kinds[2]);
  CHECK(tile_block_threads(kDefaultBatchConfig.block_threads) == kDefaultBatchConfig.block_threads);
}
""")


def test_largest_fills_fit_the_grid(tmp_path):
    """Fills of up to 2^37 doubles and 2^39 words (into mapped host memory, say) stay within a grid's 2^32 - 1
    work-items; the shapes up to there are the measured ones."""
    check(tmp_path, r"""
static void run(const DeviceContext& ctx) {
  for (uint64_t n : {1ull << 28, (1ull << 36) - 4096, 1ull << 36, (1ull << 37) - (1ull << 20)})
    for (int format : {MRG8_F64, MRG8_F64_01}) {
      int block = 0;
      uint64_t tile = 0;
      default_shape(ctx, n, format, 4, &block, &tile);
      CHECK(block == 64 && fill_waves(n, 127, tile) * 64 <= 0xffffffffull);
      CHECK(tile == (n < 1ull << 36 ? 1024u : 2048u));
    }
  for (uint64_t n : {1ull << 28, 1ull << 37, (1ull << 38) + 4096, (1ull << 39) - (1ull << 20)}) {
    const uint64_t tiles = n / 2048, per = mfma_tiles_per_wave(ctx, MRG8_U32, 2048, tiles);
    CHECK(((tiles + per - 1) / per + 2 + 3) / 4 * 256 <= 0xffffffffull);
    CHECK(per == (n <= 1ull << 37 ? 2u : 4u));
  }
  CHECK(mfma_tiles_per_wave(ctx, MRG8_U32, 2048, 12 * 256) == 1 && mfma_tiles_per_wave(ctx, MRG8_U32, 2048, 12 * 256 + 1) == 2);
  CHECK(mfma_tiles_per_wave(ctx, MRG8_U32, 2048, 24 * 256 + 1) == 4 && mfma_tiles_per_wave(ctx, MRG8_U32, 2048, 64 * 256) == 2);
  CHECK(mfma_tiles_per_wave(ctx, MRG8_U32, 1024, 64 * 256) == 8 && mfma_tiles_per_wave(ctx, MRG8_U32, 1024, 128 * 256) == 4);
  CHECK(mfma_tiles_per_wave(ctx, MRG8_U32, 1024, 24 * 256) == 2 && mfma_tiles_per_wave(ctx, MRG8_F64, 1024, 1 << 18) == 4);
}
""")


def test_half_given_fill_shapes(tmp_path):
    """A caller's threads per block get fitting outputs per wave, and outputs per wave fitting blocks."""
    check(tmp_path, r"""
static bool is(const DeviceContext& ctx, uint64_t n, int format, int per_lane, int block, uint64_t tile, int want_block,
               uint64_t want_tile) {
  default_shape(ctx, n, format, per_lane, &block, &tile);
  return block == want_block && tile == want_tile;
}
static void run(const DeviceContext& ctx) {
  const uint64_t large = 1 << 28, small = 1 << 20;
  CHECK(is(ctx, large, MRG8_F64, 4, 0, 0, 64, 1024) && is(ctx, small, MRG8_F64, 4, 0, 0, 64, 512));
  CHECK(is(ctx, large, MRG8_F64, 4, 256, 0, 256, 1024) && is(ctx, large, MRG8_F64_01, 4, 512, 0, 512, 1024));
  CHECK(is(ctx, large, MRG8_F64, 4, 1024, 0, 1024, 2048) && is(ctx, small, MRG8_F64, 4, 1024, 0, 1024, 512));
  CHECK(is(ctx, 1 << 22, MRG8_F64, 1, 1024, 0, 1024, 1024) && is(ctx, 1 << 23, MRG8_F64, 1, 1024, 0, 1024, 2048));
  CHECK(is(ctx, large, MRG8_F64, 4, 0, 2048, 64, 2048) && is(ctx, large, MRG8_F64, 4, 0, 16384, 64, 16384));
  CHECK(is(ctx, large, MRG8_F64, 4, 0, 8192, 512, 8192) && is(ctx, large, MRG8_F64, 4, 0, 4096, 512, 4096));
  CHECK(is(ctx, small, MRG8_F64, 4, 0, 4096, 256, 4096) && is(ctx, large, MRG8_F64, 4, 100, 7, 100, 7));
  CHECK(is(ctx, large, MRG8_U32, 4, 0, 0, 256, 8192) && is(ctx, small, MRG8_U32, 4, 512, 0, 512, 1024));
  CHECK(is(ctx, large, MRG8_U32, 4, 0, 2048, 256, 2048));
}
""")
