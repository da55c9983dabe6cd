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
