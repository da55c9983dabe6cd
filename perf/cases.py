"""Performance cases: the calls that programs make of this library, over the sizes they make them at.

Every case goes through the package's public entry points (`mrg8_amd`,
`mrg8_amd.torch_ops`).  Fills start from `seed_init` on each pass, as the
reference's drivers do, so that a pass can be repeated with the same outputs.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mrg8_amd
from mrg8_amd import F64, F64_01, U32, torch_ops

P = 2**31 - 1
COEFF = (1089656042, 1906537547, 1764115693, 1304127872, 189748160, 1984088114, 626062218, 1927846343)
FORMATS = {"f64": F64, "f64_01": F64_01, "u32": U32}
BYTES = {"f64": 8, "f64_01": 8, "u32": 4}


def listed():
    return [
        # the smallest call: one training step's or one particle's thousand
        # draws; launch and host time are all there is
        {"name": "fill_f64_1000", "kind": "fill", "via": "generate", "fmt": "f64", "n": 1000, "shift": 0},
        # a Monte Carlo kernel's million draws into a slice of a larger buffer
        # (8 bytes off every vector and line boundary, not a power of two)
        {"name": "fill_f64_1m_ragged", "kind": "fill", "via": "generate", "fmt": "f64", "n": 1_000_003, "shift": 1},
        # the reference's full-compare size through its own blocking launcher
        {"name": "outer_32_2p24", "kind": "fill", "via": "outer_32", "fmt": "f64_01", "n": 1 << 24, "shift": 0},
        # the headline: one stream, 2^28 doubles
        {"name": "fill_f64_2p28", "kind": "fill", "via": "generate", "fmt": "f64", "n": 1 << 28, "shift": 0},
        # a torch program that addresses one stream by position (no hidden
        # state): raw words into an int32 tensor, an odd size
        {"name": "torch_fill_u32_3m", "kind": "torch_fill", "fmt": "u32", "n": 3_000_017, "offset_bits": 50},
        # raw words at the headline's size
        {"name": "fill_u32_2p28", "kind": "fill", "via": "generate", "fmt": "u32", "n": 1 << 28, "shift": 0},
        # thousands of independent streams of uneven length, one launch, packed
        # back to back, the batch's own default configuration
        {"name": "batch_4096_streams", "kind": "batch", "streams": 4096, "lo_exp": 10, "hi_exp": 22, "sizes": 42,
         "offset_bits": 0, "fmt": "f64", "grid": "default"},
        # many short substreams, each reached by a long jump (the
        # configuration documented for such batches)
        {"name": "batch_65536_jumps", "kind": "batch", "streams": 65536, "lo_exp": 8, "hi_exp": 8, "sizes": 43,
         "offset_bits": 63, "fmt": "u32", "grid": "persistent"},
        # substreams for a large ensemble: a million states 200-bit distances apart
        {"name": "advance_200bit_2p20", "kind": "advance", "n": 1 << 20, "bits": 200},
        # re-positioning a working set of states by 64-bit distances
        {"name": "advance_64bit_20k", "kind": "advance", "n": 20_011, "bits": 64},
        # a burst of requests to the server, sizes of its benchmark's mix
        {"name": "server_burst_48", "kind": "server", "requests": 48, "lo_exp": 8, "hi_exp": 26, "sizes": 44},
        # host-memory form of class mrg8: doubles into a numpy array
        {"name": "host_rand_4m", "kind": "host", "fmt": "f64", "n": (1 << 22) + 7},
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["fill", "fill", "fill", "fill", "torch_fill", "batch", "jumps", "advance", "advance", "server",
                       "host"])
    if kind == "fill":
        via = rng.choice(["generate", "generate", "generate", "outer_32"])
        fmt = "f64_01" if via == "outer_32" else rng.choice(["f64", "u32", "f64_01", "f64", "u32"])
        return {"kind": "fill", "via": via, "fmt": fmt, "n": _log_int(rng, 256, 1 << 28),
                "shift": rng.choice([0, rng.randrange(512)])}
    if kind == "torch_fill":
        return {"kind": "torch_fill", "fmt": rng.choice(["u32", "f64"]), "n": _log_int(rng, 256, 1 << 26),
                "offset_bits": rng.randrange(1, 63)}
    if kind == "batch":
        return {"kind": "batch", "streams": _log_int(rng, 16, 4096), "lo_exp": rng.randrange(6, 11),
                "hi_exp": rng.randrange(14, 22), "sizes": rng.randrange(1 << 30), "offset_bits": rng.choice([0, 20, 40]),
                "fmt": rng.choice(["f64", "f64_01", "u32", "mixed"]), "grid": rng.choice(["default", "queue", "persistent"])}
    if kind == "jumps":
        exp = rng.randrange(4, 11)
        return {"kind": "batch", "streams": _log_int(rng, 512, 65536), "lo_exp": exp, "hi_exp": exp + rng.randrange(2),
                "sizes": rng.randrange(1 << 30), "offset_bits": rng.randrange(20, 64), "fmt": rng.choice(["f64", "u32"]),
                "grid": "persistent"}
    if kind == "advance":
        return {"kind": "advance", "n": _log_int(rng, 64, 1 << 20), "bits": rng.choice([32, 64, 100, 128, 200, 256])}
    if kind == "server":
        return {"kind": "server", "requests": rng.randrange(8, 49), "lo_exp": 8, "hi_exp": rng.randrange(18, 27),
                "sizes": rng.randrange(1 << 30)}
    return {"kind": "host", "fmt": rng.choice(["f64", "u32"]), "n": _log_int(rng, 256, 1 << 24)}


# ---- inputs ----------------------------------------------------------------------


def _lengths(case, count):
    """The segment or request sizes of a case: floor(2^(lo + (hi - lo) u)), the same for every seed."""
    rng = np.random.default_rng(case["sizes"])
    lo, hi = case["lo_exp"], case["hi_exp"]
    return np.floor(2.0 ** (lo + (hi - lo) * rng.random(count))).astype(np.int64)


def _batch_plan(case):
    """Per segment: format, length, byte offset in the one output buffer (packed, each at its own element size)."""
    count = case["streams"]
    lengths = _lengths(case, count)
    if case["fmt"] == "mixed":
        fmts = [("f64", "u32", "f64_01")[i % 3] for i in range(count)]
    else:
        fmts = [case["fmt"]] * count
    at, starts = 0, []
    for fmt, n in zip(fmts, lengths.tolist()):
        at = (at + BYTES[fmt] - 1) // BYTES[fmt] * BYTES[fmt]
        starts.append(at)
        at += n * BYTES[fmt]
    return fmts, lengths, starts, (at + 7) // 8 * 8


def _random_states(rng, count):
    return rng.integers(1, P, size=(count, 8), dtype=np.int64).astype(np.uint32)


def _advance_words(case):
    return (case["bits"] + 63) // 64


# (threads per block, blocks per CU, outputs per tile) of the documented grid kinds
GRIDS = {"persistent": (256, 8, 2048), "queue": (512, 3, 2048)}


class _DeviceArray:
    """A server's output buffer as an array that torch can wrap without a copy."""

    def __init__(self, ptr, count):
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": "<f8", "data": (int(ptr), False), "version": 2}


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "fill":
        s["seed"] = int(rng.integers(1, 2**32))
        s["gen"] = mrg8_amd.mrg8_cuda(s["seed"])
        dtype = torch.int32 if case["fmt"] == "u32" else torch.float64
        s["out"] = torch.empty(case["n"] + case["shift"], dtype=dtype, device="cuda")[case["shift"]:]
    elif kind == "torch_fill":
        s["state"] = [int(x) for x in _random_states(rng, 1)[0]]
        s["offset"] = int(rng.integers(0, 1 << case["offset_bits"]))
        s["out"] = torch.empty(case["n"], dtype=torch.int32 if case["fmt"] == "u32" else torch.float64, device="cuda")
    elif kind == "batch":
        fmts, lengths, starts, nbytes = _batch_plan(case)
        states = _random_states(rng, case["streams"])
        top = 1 << case["offset_bits"]
        offsets = rng.integers(0, top, size=case["streams"], dtype=np.uint64)
        words = case["fmt"] in ("u32", "mixed")
        # zeros: a mixed batch leaves alignment gaps between its segments
        s["out"] = torch.zeros(nbytes // (4 if words else 8), dtype=torch.int32 if words else torch.float64, device="cuda")
        base = s["out"].data_ptr()
        s["batch"] = mrg8_amd.Batch(case["streams"], int(sum(n // 2048 + 2 for n in lengths.tolist())))
        if case["grid"] != "default":
            threads, blocks, tile = GRIDS[case["grid"]]
            s["batch"].set_config(threads, -blocks if case["grid"] == "queue" else blocks, tile)
        s["batch"].set((states[i], offsets[i], lengths[i], base + starts[i], FORMATS[fmts[i]])
                       for i in range(case["streams"]))
    elif kind == "advance":
        n, words = case["n"], _advance_words(case)
        offsets = rng.integers(0, 2**64, size=(n, words), dtype=np.uint64)
        if case["bits"] % 64:
            offsets[:, -1] &= np.uint64((1 << (case["bits"] % 64)) - 1)
        s["states"] = torch.from_numpy(_random_states(rng, n).view(np.int32)).cuda()
        s["offsets"] = torch.from_numpy(offsets.view(np.int64)).cuda()
        s["out"] = torch.empty_like(s["states"])
    elif kind == "server":
        sizes = _lengths(case, case["requests"])
        s["sizes"] = [int(x) for x in sizes]
        s["server"] = mrg8_amd.Server(16384, int(sum((n * 8 + 255) // 256 * 256 for n in s["sizes"])))
        s["server"].set_streams(_random_states(rng, 16384))
        s["streams"] = [int(x) for x in rng.integers(0, 16384, size=case["requests"])]
        s["held"] = []
    else:
        s["seed"] = int(rng.integers(1, 2**32))
        s["gen"] = mrg8_amd.mrg8(s["seed"])
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fill":
        gen, out = state["gen"], state["out"]
        gen.seed_init(state["seed"])
        if case["via"] == "outer_32":
            gen.mrg8_outer_32(out, case["n"])
        else:
            gen.generate(out, case["n"], FORMATS[case["fmt"]], stream=torch.cuda.current_stream())
        return out
    if kind == "torch_fill":
        torch.ops.mrg8.fill_(state["out"], state["state"], state["offset"], FORMATS[case["fmt"]])
        return state["out"]
    if kind == "batch":
        state["batch"].run(stream=torch.cuda.current_stream())
        return state["out"]
    if kind == "advance":
        mrg8_amd.advance_states(state["states"], state["offsets"], _advance_words(case), state["out"], case["n"],
                                stream=torch.cuda.current_stream())
        return state["out"]
    if kind == "server":
        server = state["server"]
        for rid in state["held"]:  # the outputs of the burst before
            server.release(rid)
        ids = [server.submit(st, n) for st, n in zip(state["streams"], state["sizes"])]
        done = {}
        while len(done) < len(ids):
            for c in server.progress(max_done=64, wait_ms=100):
                done[c["request_id"]] = c
        state["held"] = ids
        outs = [torch.as_tensor(_DeviceArray(done[i]["out"], done[i]["count"]), device="cuda") for i in ids]
        for t in outs:
            t.server = server  # the buffers are the server's: it lives as long as they are looked at
        return outs
    gen = state["gen"]
    gen.seed_init(state["seed"])
    return gen.randint(case["n"]) if case["fmt"] == "u32" else gen.rand(case["n"])


def work(case):
    kind = case["kind"]
    if kind == "batch":
        fmts, lengths, _, _ = _batch_plan(case)
        out = sum(int(n) * BYTES[f] for f, n in zip(fmts, lengths.tolist()))
        # a segment's descriptor: state, offset, length, address
        return {"bytes": out + 64 * case["streams"], "flops": 16 * int(lengths.sum())}
    if kind == "server":
        total = int(_lengths(case, case["requests"]).sum())
        return {"bytes": 8 * total, "flops": 16 * total}
    if kind == "advance":
        n = case["n"]
        return {"bytes": n * (64 + 8 * _advance_words(case)), "flops": n * 128 * ((case["bits"] + 7) // 8)}
    # eight multiply-adds an output
    return {"bytes": case["n"] * BYTES[case["fmt"]], "flops": 16 * case["n"]}


# ---- expected outputs -------------------------------------------------------------


def _seeded(seed):
    x, st = seed or 97531, []
    for _ in range(8):
        x = x * 6364136223846793005 % 2**64
        st.append(x >> 33)
    return st


def _mat_mul(a, b):
    return [[sum(a[i][k] * b[k][j] for k in range(8)) % P for j in range(8)] for i in range(8)]


def _power(e):
    a = [list(COEFF)] + [[int(j == i) for j in range(8)] for i in range(7)]
    r = [[int(i == j) for j in range(8)] for i in range(8)]
    while e:
        if e & 1:
            r = _mat_mul(a, r)
        a = _mat_mul(a, a)
        e >>= 1
    return r


def _words(state, offset, n):
    """Outputs offset .. offset+n-1 of a stream (residues, a residue of 0 as P): columns of a power of two stepped together."""
    length = 1 << max(4, (n.bit_length() + 1) // 2)
    cols = (n + length - 1) // length
    v = [sum(a * b for a, b in zip(row, state)) % P for row in _power(offset)]
    step = _power(length)
    starts = np.empty((cols, 8), dtype=np.uint64)
    for c in range(cols):
        starts[c] = v
        v = [sum(a * b for a, b in zip(row, v)) % P for row in step]
    hist = [starts[:, q].copy() for q in range(8)]  # newest first
    out = np.empty((length, cols), dtype=np.uint32)
    for i in range(length):
        x = np.zeros(cols, dtype=np.uint64)
        for a, h in zip(COEFF, hist):
            x += np.uint64(a) * h % np.uint64(P)
        x %= np.uint64(P)
        out[i] = np.where(x == 0, P, x)
        hist = [x] + hist[:7]
    return out.T.reshape(-1)[:n]


def exact(case, seed):
    """Fills of up to 2^24 outputs; the others take too long in numpy, or are whole numbers."""
    if case["kind"] not in ("fill", "torch_fill", "host") or case["n"] > 1 << 24:
        return None
    rng = np.random.default_rng(seed)
    if case["kind"] == "torch_fill":
        state = [int(x) for x in _random_states(rng, 1)[0]]
        words = _words(state, int(rng.integers(0, 1 << case["offset_bits"])), case["n"])
    else:
        words = _words(_seeded(int(rng.integers(1, 2**32))), 0, case["n"])
    if case["fmt"] == "u32":
        return words.astype(np.int32) if case["kind"] != "host" else words
    return (words if case["fmt"] == "f64" else words - 1).astype(np.float64) * (1.0 / P)
