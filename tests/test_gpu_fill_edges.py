"""GPU parity of the fills and batches at the edges of their launch rules.

Fills: the sizes where the outputs per wave and the XCD runs change (4, 16
waves of 1024 per CU on 256 CUs), a partial last wave, and unaligned
destinations.  Jumps: offsets whose digits sit in the low half, the high half
or both, next to states with zero words and the all-zero state, on each kind of
batch grid.  All outputs against the oracle, bit for bit.
"""
import numpy as np
import pytest

from test_gpu_parity import SEED, run_device, say

pytestmark = pytest.mark.gpu

P = 2**31 - 1


@pytest.mark.parametrize("fmt", [0, 1, 2])
@pytest.mark.parametrize("n,pad", [(511, 0), (512, 1), (513, 127), (1024 * 1024, 0), (1024 * 1024 + 1, 1),
                                   (1024 * 4095 + 1, 0), (1024 * 4096 + 129, 3), (1024 * 4096 + 8 * 64 * 1024 - 1, 0)])
def test_fill_rule_edges(gpu, oracle_mod, fmt, n, pad):
    say("fill edges", fmt, n, pad)
    g = gpu.mrg8_cuda(SEED + n)
    got = run_device(gpu, g, n, fmt, pad_elems=pad)
    want, st = oracle_mod.generate(oracle_mod.seed_state(SEED + n), n, fmt)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    assert np.array_equal(g.get_state(), st)


@pytest.mark.parametrize("grid", [(1024, 0, 256), (256, 4, 256), (512, -2, 256)],
                         ids=["tile-per-wave", "persistent", "address-order"])
def test_jump_digits_and_zero_words(gpu, oracle_mod, grid):
    from mrg8_amd.hip import DeviceBuffer

    rng = np.random.default_rng(5)
    offsets = [0, 1, 255, 256, 0xff00, 1 << 24, (1 << 32) - 1, 1 << 32, 255 << 56, (1 << 63) + 1, (1 << 63) + (1 << 31)]
    offsets += [int(x) for x in rng.integers(0, 2**63, size=6)]
    states = [rng.integers(1, P + 1, size=8) for _ in range(3)]
    states += [np.array([0, 0, 0, 0, 0, 0, 0, 5]), np.array([0, P, 0, 0, 7, 0, 0, 0]), np.zeros(8, int), np.full(8, P)]
    segs = [(st, off, 300 + 7 * i, (i + j) % 3) for i, off in enumerate(offsets) for j, st in enumerate(states)]
    at, place = 0, []
    for _, _, cnt, fmt in segs:
        place.append(at)
        at += (cnt * (4 if fmt == 2 else 8) + 7) // 8 * 8
    buf = DeviceBuffer(at + 8)
    b = gpu.Batch(len(segs), 4096)
    b.set_config(*grid)
    b.set((st, off, cnt, buf.ptr + p, fmt) for (st, off, cnt, fmt), p in zip(segs, place))
    say("jump digits", grid, len(segs))
    b.run()
    gpu.hip.synchronize()
    got = buf.copy_to_host(np.uint8, at)
    b.close()
    buf.free()
    for (st, off, cnt, fmt), p in zip(segs, place):
        want, _ = oracle_mod.generate(oracle_mod.jump(np.asarray(st, np.uint32), off), cnt, fmt)
        have = got[p:p + cnt * want.itemsize]
        assert np.array_equal(have, want.view(np.uint8)), (list(st), off, fmt)


SHORT_LENGTHS = [1, 2, 3, 15, 16, 17, 63, 127, 128, 129, 130, 255, 256, 257, 258, 300, 511, 512, 513, 0, 769]


@pytest.mark.parametrize("grid,fmts,more", [((256, 8, 2048), (2,), 0), ((256, 4, 256), (2,), 5), ((64, 1, 2048), (2, 2, 2, 0), 1),
                                            ((128, 2, 256), (0,), 8), ((256, 8, 512), (1, 2, 2, 0, 2), 16399)])
def test_many_short_tiles(gpu, oracle_mod, grid, fmts, more):
    """Batches of at least 32 tiles per CU on a striding grid: tiles of less,
    exactly and more than a run of 256 outputs, groups of one and of several
    formats, zero words and the all-zero state, alignments of one element; the
    graph across a restaging with too few tiles, and the no-alloc entry point."""
    import ctypes

    import torch
    from mrg8_amd import capi

    rng = np.random.default_rng(7)
    few = fmts == (0,)
    lengths = [n for n in SHORT_LENGTHS if not few or n <= 256]
    states = [rng.integers(1, P + 1, size=8) for _ in range(3)]
    states += [np.array([0, 0, 0, 0, 0, 0, 0, 5]), np.zeros(8, int)]
    kinds = []
    for i in range(5 * len(lengths)):  # 5 states x 21 (or 14) lengths, every pair
        off = [0, 1, 255, 1 << 32, int(rng.integers(0, 2**63))][(i // 3) % 5]
        kinds.append((states[i % 5], off, lengths[i % len(lengths)], fmts[i % len(fmts)]))
    want = [np.frombuffer(oracle_mod.generate(oracle_mod.jump(np.asarray(st, np.uint32), off), n, f)[0].tobytes(), np.uint8)
            for st, off, n, f in kinds]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n = (32 * cus + more) * len(lengths) // (len(lengths) - (0 in lengths)) + 1  # empty segments have no tile
    place, at = [], 0
    for i in range(n):
        place.append(at := at + (-at) % (4 if kinds[i % len(kinds)][3] == 2 else 8))
        at += want[i % len(kinds)].size
    weight = sum((1 if f == 2 else 8) * c for _, _, c, f in kinds) / sum(c > 0 for _, _, c, f in kinds)
    assert weight <= 1024
    expected = np.full(at + 64, 0xA5, np.uint8)
    for i in range(n):
        expected[place[i]:place[i] + want[i % len(kinds)].size] = want[i % len(kinds)]

    buf = gpu.hip.DeviceBuffer(at + 64)
    b = gpu.Batch(n, 8 * n)
    b.set_config(*grid)
    b.use_graph(True)
    for count in (n, 300, n):
        buf.fill_byte(0xA5)
        b.set((*kinds[i % len(kinds)][:3], buf.ptr + place[i], kinds[i % len(kinds)][3]) for i in range(count))
        say("short tiles", grid, fmts, count)
        b.run()
        b.run()
        gpu.hip.synchronize()
        got = buf.copy_to_host(np.uint8, at + 64)
        end = place[count] if count < n else at
        assert np.array_equal(got[:end], expected[:end]), np.flatnonzero(got[:end] != expected[:end])[:8]
        assert (got[end:] == 0xA5).all()
    b.close()
    if more == 5:
        arr = (capi.StreamDesc * n)()
        for i in range(n):
            st, off, cnt, f = kinds[i % len(kinds)]
            arr[i].state = (ctypes.c_uint32 * 8)(*[int(x) for x in st])
            arr[i].offset, arr[i].count, arr[i].out, arr[i].format = off, cnt, buf.ptr + place[i], f
        buf.fill_byte(0xA5)
        say("short tiles", "noalloc", grid, n)
        capi.call("mrg8_batch_generate_noalloc", 0, arr, ctypes.c_uint32(n), ctypes.byref(capi.BatchConfig(*grid)), None)
        gpu.hip.synchronize()
        assert np.array_equal(buf.copy_to_host(np.uint8, at + 64), expected)
    buf.free()


@pytest.mark.parametrize("tiles,more,pad", [(12, 2047, 0), (12, 2048, 1), (24, 0, 0), (24, 2049, 3), (64, -1, 0), (64, 1, 2)])
def test_word_fill_tiles_per_wave(gpu, oracle_mod, tiles, more, pad):
    """The matrix-core fill where its tiles per wave and its XCD runs change
    (12, 24 and 64 tiles of 2048 words per CU)."""
    import torch

    n = tiles * torch.cuda.get_device_properties(0).multi_processor_count * 2048 + more + (-pad) % 256
    say("word fill", n, pad)
    g = gpu.mrg8_cuda(SEED + tiles)
    got = run_device(gpu, g, n, 2, pad_elems=pad)
    want, st = oracle_mod.generate(oracle_mod.seed_state(SEED + tiles), n, 2)
    assert np.array_equal(got, want)
    assert np.array_equal(g.get_state(), st)


@pytest.mark.parametrize("threads", [64, 512])
@pytest.mark.parametrize("groups", [-1, 0, 1, 777])
@pytest.mark.parametrize("graph", [False, True])
def test_address_order_counter(gpu, oracle_mod, threads, groups, graph):
    """An address-order grid of one block per CU around the group count from
    which its blocks take further groups from the counter, run after run."""
    import torch

    tiles = (torch.cuda.get_device_properties(0).multi_processor_count + groups) * (threads // 64)
    n = tiles * 256 - 5
    buf = gpu.hip.DeviceBuffer(n * 4)
    b = gpu.Batch(1, tiles + 1)
    b.set_config(threads, -1, 256)
    b.use_graph(graph)
    want, _ = oracle_mod.generate(oracle_mod.jump(oracle_mod.seed_state(SEED), 1 << 33), n, 2)
    b.set([(oracle_mod.seed_state(SEED), 1 << 33, n, buf.ptr, 2)])
    for run in range(3):
        say("address order", threads, groups, graph, run)
        buf.fill_byte(0xA5)
        b.run()
        gpu.hip.synchronize()
        assert np.array_equal(buf.copy_to_host(np.uint32, n), want)
    b.close()
    buf.free()


def test_striding_grid_with_uneven_tiles(gpu, oracle_mod):
    """More than 32 tiles per CU on a striding grid, one of 16384 outputs among
    sixteen tiny ones (which the short-tile kernel leaves alone), against the
    oracle."""
    from mrg8_amd.hip import DeviceBuffer

    import torch

    rng = np.random.default_rng(17)
    tiny = 34 * torch.cuda.get_device_properties(0).multi_processor_count
    state = rng.integers(1, P + 1, size=8)
    words, _ = oracle_mod.generate(oracle_mod.jump(np.asarray(state, np.uint32), 1 << 40), 20000, 2)
    lengths = [16384 if i % 17 == 0 else 1 + i % 90 for i in range(tiny)]
    skip = [i % 1000 for i in range(tiny)]  # segment i starts this far into `words`
    place = np.concatenate([[0], np.cumsum(lengths)])
    buf = DeviceBuffer(int(place[-1]) * 4)
    b = gpu.Batch(tiny, 2 * tiny)
    b.set_config(256, 8, 16384)
    b.set((state, (1 << 40) + k, n, buf.ptr + 4 * int(at), 2) for k, n, at in zip(skip, lengths, place))
    say("uneven tiles", tiny)
    b.run()
    gpu.hip.synchronize()
    got = buf.copy_to_host(np.uint32, int(place[-1]))
    b.close()
    buf.free()
    for k, n, at in zip(skip, lengths, place):
        assert np.array_equal(got[at:at + n], words[k:k + n]), (k, n)


def test_graph_of_each_striding_kernel_is_kept(gpu, oracle_mod):
    """A striding grid's runs as graph replays, restaged from long tiles to many
    short ones and back: once both graphs are there, a run returns while the
    runs before it still execute."""
    import ctypes

    import torch
    from mrg8_amd import capi

    cus = torch.cuda.get_device_properties(0).multi_processor_count
    state = oracle_mod.seed_state(SEED)
    long, short = (64, 1 << 20), (40 * cus, 20)  # segments, words each
    bufs = [gpu.hip.DeviceBuffer(4 * k * n) for k, n in (long, short)]
    descs = []
    for (k, n), buf in zip((long, short), bufs):
        arr = (capi.StreamDesc * k)()
        for i in range(k):
            arr[i].state = (ctypes.c_uint32 * 8)(*state.tolist())
            arr[i].offset, arr[i].count, arr[i].out, arr[i].format = i * n, n, buf.ptr + 4 * i * n, 2
        descs.append((arr, ctypes.c_uint32(k)))
    b = gpu.Batch(40 * cus, 1 << 17)
    b.set_config(256, 8, 2048)
    b.use_graph(True)
    stream, issued = torch.cuda.Stream(), torch.cuda.Event()
    for which in (0, 1, 0, 1, 0):
        capi.call("mrg8_batch_set", b._h, *descs[which])
        b.run(stream)
    stream.synchronize()
    for repeat in range(3):
        for buf in bufs:
            buf.fill_byte(0xA5)
        capi.call("mrg8_batch_set", b._h, *descs[0])
        say("graph of each kernel", repeat)
        for _ in range(600):  # some 30 ms
            b.run(stream)
        issued.record(stream)
        capi.call("mrg8_batch_set", b._h, *descs[1])
        b.run(stream)
        assert not issued.query(), "the run waited for those before it"
        stream.synchronize()
        for (k, n), buf in zip((long, short), bufs):
            want, _ = oracle_mod.generate(state, k * n, 2)
            assert np.array_equal(buf.copy_to_host(np.uint32, k * n), want)
    b.close()
    for buf in bufs:
        buf.free()


@pytest.mark.parametrize("threads,tile,more,pad", [(128, 2048, -1, 0), (512, 2048, 5 * 2048 + 3, 1), (1024, 2048, 1, 127),
                                                   (256, 8192, 3 * 8192 - 1, 3)])
def test_fill_blocks_in_step(gpu, oracle_mod, threads, tile, more, pad):
    """Blocks whose waves wait for one another (64 or more waves of 2048 to 8192
    doubles per CU), the last block with waves that have no outputs."""
    import torch

    n = 64 * torch.cuda.get_device_properties(0).multi_processor_count * tile + more
    say("in step", threads, tile, n, pad)
    buf = gpu.hip.DeviceBuffer((n + pad) * 8)
    g = gpu.mrg8_cuda(SEED + threads)
    g.generate(buf.ptr + 8 * pad, n, 0, block_threads=threads, tile=tile, per_lane=4)
    gpu.hip.synchronize()
    state = oracle_mod.seed_state(SEED + threads)
    for first in (0, tile * (threads // 64) - 200, n // 2, n - 3 * tile - 7):  # windows across waves and blocks
        count = min(400 if first < n // 2 else 3 * tile + 7, n - first)
        want, _ = oracle_mod.generate(oracle_mod.jump(state, first), count, 0)
        got = buf.copy_to_host(np.float64, count, 8 * (pad + first))
        assert np.array_equal(got.view(np.uint64), want.view(np.uint64)), first
    got = buf.copy_to_host(np.float64, n, 8 * pad)
    buf.free()
    assert oracle_mod.wsum(got) == int(oracle_mod.stream_wsums(state[None], np.zeros(1, np.uint64), np.array([n], np.uint64),
                                                               np.zeros(1, np.int32))[0])
    assert np.array_equal(g.get_state(), oracle_mod.jump(state, n))


def test_fill_tuner_cache_entries(gpu, oracle_mod, tmp_path):
    """Cache entries of a tuned and of the automatic shape are used; those of the
    sweep that did not time the automatic shape are not."""
    say("tuner cache")
    n, cache = 1 << 21, tmp_path / "shapes.txt"
    gpu.tune_fill(0, n, cache_path=str(cache))
    key = cache.read_text().split()[0].removesuffix(":auto")
    old = tmp_path / "old.txt"
    old.write_text(key.replace(":shape:", ":fill:") + " 1024 1 16384 0.000001\n")
    assert list(gpu.tune_fill(0, n, cache_path=str(old)).values()) != [1024, 1, 16384]
    assert len(old.read_text().splitlines()) == 2
    want, _ = oracle_mod.generate(oracle_mod.seed_state(SEED), n, 0)
    for suffix in ("", ":auto"):
        kept = tmp_path / ("kept" + suffix[1:])
        kept.write_text(f"{key}{suffix} 512 2 4096 0.1\n")
        assert list(gpu.tune_fill(0, n, cache_path=str(kept)).values()) == [512, 2, 4096]
        got = run_device(gpu, gpu.mrg8_cuda(SEED), n, 0)
        assert np.array_equal(got.view(np.uint64), want.view(np.uint64))
    assert len(kept.read_text().splitlines()) == 1


@pytest.mark.parametrize("threads", [None, 64, 128, 192, 256, 320, 1024])
def test_tile_per_wave_block_sizes(gpu, oracle_mod, threads):
    """One tile per wave in every size of block, a last block with idle waves;
    a new batch says the block size that it runs in."""
    tiles = 4 * 7 + 1
    n = tiles * 256 - 9
    buf = gpu.hip.DeviceBuffer(n * 8)
    b = gpu.Batch(1, tiles + 1)
    assert b.config == {"block_threads": 256, "blocks_per_cu": 0, "tile_outputs": 2048}
    if threads:
        b.set_config(threads, 0, 256)
        assert b.config["block_threads"] == threads
    b.set([(oracle_mod.seed_state(SEED), 1 << 20, n, buf.ptr, 0)])
    say("tile per wave", threads)
    buf.fill_byte(0xA5)
    b.run()
    gpu.hip.synchronize()
    want, _ = oracle_mod.generate(oracle_mod.jump(oracle_mod.seed_state(SEED), 1 << 20), n, 0)
    assert np.array_equal(buf.copy_to_host(np.uint64, n), want.view(np.uint64))
    b.close()
    buf.free()
