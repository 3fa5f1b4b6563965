"""Performance cases: what a program does with this library, call by call.

Every case goes through public entry points (mtgp_amd, mtgp_amd.torch_ext)
and writes whole outputs.  Operations ("op"):

  fill        Generator32 / Generator64.fill into host memory, the drop-in
              bulk call of a host generator (init, then numbers on demand)
  rand        torch_ext.Generator.uniform_ / random_ into a torch tensor on
              the GPU: one stream, continued call by call
  sets        TensorGenSet.generate_: many small generators, a few thousand
              numbers each (the shape of a simulation's per-block streams)
  batch       a plan over many long streams, rebased, launched and committed
              in a loop: the continuous bulk producer
  substreams  start states at multiples of a jump, then numbers from each
  jump        fast_jump of a host generator by a given polynomial
  serve       a burst of mixed requests through the request server, results
              copied into the caller's tensors
"""
import math
import random

import numpy as np
import torch

import mtgp_amd as M
import mtgp_amd.torch_ext as mt

_MASK64 = (1 << 64) - 1
_MEXPS = {32: (11213, 23209, 44497), 64: (23209, 44497, 110503)}


# -------------------------------------------------------------------- cases
def listed():
    return [
        # a thousand floats into a numpy array: the smallest call a host
        # program makes, all latency
        {"name": "fill-host-1k", "op": "fill", "bits": 32, "mexp": 11213, "index": 0, "kind": "close_open", "n": 1000},
        # a jump by 3^162 (the reference's substream distance) of a host
        # generator, state in and state out
        {"name": "jump32", "op": "jump", "bits": 32, "mexp": 11213, "index": 0, "log3": 162},
        # a tensor of ordinary size, ragged: a weight initialisation, a mask
        {"name": "rand32-1m", "op": "rand", "bits": 32, "mexp": 11213, "index": 0, "kind": "close_open", "n": 1000003},
        # one long stream of raw words (the single-generator configuration)
        {"name": "rand32-16m", "op": "rand", "bits": 32, "mexp": 11213, "index": 0, "kind": "uint", "n": 1 << 24},
        # doubles in (0, 1) for a logarithm, one MTGP64 stream, ragged
        {"name": "rand64-5m", "op": "rand", "bits": 64, "mexp": 23209, "index": 3, "kind": "open_open", "n": 5000011},
        # 200 dynamic-creator generators, one short stream each, in [1, 2)
        # (the shape of the reference's device samples)
        {"name": "sets-dc200", "op": "sets", "bits": 32, "mexp": 0, "gens": 200, "kind": "close1_open2", "n": 24000},
        # a burst of the serving mix over device-resident generators
        {"name": "serve-128", "op": "serve", "requests": 128, "gens": 64, "mix": 1},
        # 64 larger-state MTGP32 streams of moderate length
        {"name": "batch32-44497", "op": "batch", "bits": 32, "mexp": 44497, "gens": 64, "log2_min": 22.0, "log2_max": 22.0,
         "mix": 1},
        # the batched MTGP64 configurations: 64 sets, 2^24 uint64 and 2^24
        # doubles in [0, 1) each
        {"name": "batch64-23209", "op": "batch", "bits": 64, "mexp": 23209, "gens": 64, "log2_min": 24.0, "log2_max": 24.0,
         "mix": 1},
        {"name": "batch64-44497", "op": "batch", "bits": 64, "mexp": 44497, "gens": 64, "log2_min": 24.0, "log2_max": 24.0,
         "mix": 1},
        # 4096 substreams of one generator, 2^20 words each
        {"name": "substreams-4096", "op": "substreams", "mexp": 11213, "gens": 4096, "log3": 162, "n": 1 << 20},
        # the headline batch: all 128 sets of MTGP32-11213, uneven lengths
        # 2^20..2^26 words and as many floats in [0, 1) each
        {"name": "batch32-11213", "op": "batch", "bits": 32, "mexp": 11213, "gens": 128, "log2_min": 20.0, "log2_max": 26.0,
         "mix": 7},
    ]


def draw(rng):
    def logint(lo, hi):
        return int(2.0 ** rng.uniform(math.log2(lo), math.log2(hi)))

    def table():
        bits = rng.choice((32, 32, 64))
        return bits, rng.choice((11213, 11213, 23209, 44497) if bits == 32 else (23209, 44497))

    op = rng.choice(("fill", "rand", "rand", "sets", "batch", "batch", "substreams", "jump", "serve"))
    bits, mexp = table()
    kind = rng.choice(("uint", "close1_open2", "close_open", "open_close", "open_open"))
    if op == "fill":
        return {"op": op, "bits": bits, "mexp": mexp, "index": rng.randrange(128), "kind": kind, "n": logint(100, 1 << 21)}
    if op == "rand":
        return {"op": op, "bits": bits, "mexp": mexp, "index": rng.randrange(128), "kind": kind, "n": logint(1000, 1 << 26)}
    if op == "sets":
        if rng.random() < 0.4:
            mexp = 0
        return {"op": op, "bits": bits, "mexp": mexp, "gens": rng.randint(16, 200), "kind": kind, "n": logint(1000, 1 << 17)}
    if op == "batch":
        gens = rng.randint(16, 128)
        # at most as many bytes as the headline batch
        top = min(26.0, math.log2(18.0e9 / (2 * gens * bits / 8)))
        hi = rng.uniform(18.0, top)
        lo = max(16.0, hi - rng.choice((0.0, 1.0, 4.0)))
        return {"op": op, "bits": bits, "mexp": mexp, "gens": gens, "log2_min": lo, "log2_max": hi,
                "mix": rng.randrange(1 << 30)}
    if op == "substreams":
        return {"op": op, "mexp": rng.choice((11213, 11213, 23209)), "gens": logint(64, 4096),
                "log3": rng.randint(60, 162), "n": logint(1 << 10, 1 << 19)}
    if op == "jump":
        return {"op": op, "bits": bits, "mexp": mexp, "index": rng.randrange(128), "log3": rng.randint(20, 200)}
    return {"op": op, "requests": rng.randint(16, 192), "gens": rng.choice((16, 64, 128)), "mix": rng.randrange(1 << 30)}


# ------------------------------------------------------------------- inputs
def _splitmix(state, count):
    out = []
    for _ in range(count):
        state = (state + 0x9E3779B97F4A7C15) & _MASK64
        z = state
        z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & _MASK64
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & _MASK64
        out.append(z ^ (z >> 31))
    return out


def _record(case, index):
    return M.params(case["bits"], case["mexp"], index) if case["mexp"] else M.dc_params(case["bits"], index)


def _specs(case):
    if case["mexp"]:
        return [(case["bits"], case["mexp"], g % 128) for g in range(case["gens"])]
    return [M.dc_params(case["bits"], g % 200) for g in range(case["gens"])]


def _dtype(bits, kind):
    if kind == "uint":
        return torch.int32 if bits == 32 else torch.int64
    return torch.float32 if bits == 32 else torch.float64


def _lengths(case):
    """Numbers per request of a batch, uneven between 2^log2_min and 2^log2_max."""
    u = [(v >> 11) * 2.0**-53 for v in _splitmix(case["mix"], case["gens"])]
    return [int(2.0 ** (case["log2_min"] + (case["log2_max"] - case["log2_min"]) * x)) for x in u]


def _serving_mix(case):
    """Generators and requests of a burst: half MTGP32-11213, a quarter each
    MTGP32-23209 and MTGP64-23209; log-normal sizes, a tenth of the requests
    with a skip of up to 2^30 numbers first."""
    n = case["gens"]
    a, b = n // 2, n // 4
    specs = ([(32, 11213, i) for i in range(a)] + [(32, 23209, i) for i in range(b)]
             + [(64, 23209, i) for i in range(n - a - b)])
    rng = random.Random(case["mix"])
    reqs = []
    for _ in range(case["requests"]):
        kind = rng.choice(("uint", "close1_open2", "close_open"))
        gen = rng.randrange(a + b) if kind != "close_open" else a + b + rng.randrange(n - a - b)
        x = min(21.0, max(10.0, rng.gauss(16.0, 2.5)))
        count = int(2.0**x) & ~3
        skip = int(2.0 ** rng.uniform(10, 30)) if rng.random() < 0.1 else 0
        reqs.append((gen, kind, count, skip))
    return specs, reqs


def prepare(case, seed):
    op, s = case["op"], {"case": case}
    seeds = _splitmix(seed * 2654435761 + 12345, max(1, case.get("gens", 1)))
    if op in ("fill", "jump"):
        cls = M.Generator32 if case["bits"] == 32 else M.Generator64
        s["gen"] = cls(case["mexp"], case["index"], seed=seeds[0] & (0xFFFFFFFF if case["bits"] == 32 else _MASK64))
        if op == "fill":
            s["out"] = np.empty(case["n"], M.out_dtype(case["bits"], M.KINDS[case["kind"]]))
        else:
            s["hex"] = M.jump_hex(case["bits"], case["mexp"], case["index"], 3 ** case["log3"])
    elif op == "rand":
        s["gen"] = mt.Generator(case["bits"], case["mexp"], case["index"], seed=seeds[0])
        s["out"] = torch.empty(case["n"], dtype=_dtype(case["bits"], case["kind"]), device="cuda")
    elif op == "sets":
        s["set"] = mt.TensorGenSet(_specs(case))
        s["set"].init_seed(seeds)
        s["out"] = torch.empty(case["gens"], case["n"], dtype=_dtype(case["bits"], case["kind"]), device="cuda")
        s["reqs"] = [(g, M.KINDS[case["kind"]], s["out"][g]) for g in range(case["gens"])]
    elif op == "batch":
        s["set"] = M.GenSet(_specs(case))
        if case["bits"] == 32:
            s["set"].init_seed(seeds)
        else:
            s["set"].init_array([_splitmix(v, 4) for v in seeds])
        lens = _lengths(case)
        s["ints"] = torch.empty(sum(lens), dtype=_dtype(case["bits"], "uint"), device="cuda")
        s["floats"] = torch.empty(sum(lens), dtype=_dtype(case["bits"], "close_open"), device="cuda")
        reqs, off = [], 0
        for g, n in enumerate(lens):
            reqs.append((g, "uint", n, 0, s["ints"].data_ptr() + off))
            reqs.append((g, "close_open", n, 0, s["floats"].data_ptr() + off))
            off += n * case["bits"] // 8
        s["plan"] = s["set"].plan(reqs)
    elif op == "substreams":
        base = M.GenSet([(32, case["mexp"], 0)])
        base.init_seed([seeds[0]])
        s["base"] = base.state(0)
        s["hex"] = M.jump_hex(32, case["mexp"], 0, 3 ** case["log3"])
        s["set"] = M.GenSet([(32, case["mexp"], 0)] * case["gens"])
        s["set"].substreams(s["base"], s["hex"])
        s["out"] = torch.empty(case["gens"], case["n"], dtype=torch.int32, device="cuda")
        s["plan"] = s["set"].plan([(g, "uint", case["n"], 0, s["out"][g].data_ptr()) for g in range(case["gens"])])
    elif op == "serve":
        specs, reqs = _serving_mix(case)
        s["set"] = M.GenSet(specs)
        s["set"].init_seed(seeds)
        s["reqs"] = reqs
        kinds = {"uint": torch.int32, "close1_open2": torch.float32, "close_open": torch.float64}
        s["outs"] = {k: torch.zeros(max(4, sum(c for _, q, c, _ in reqs if q == k)), dtype=d, device="cuda")
                     for k, d in kinds.items()}
        s["dst"], at = [], dict.fromkeys(kinds, 0)
        for _, kind, count, _ in reqs:
            t = s["outs"][kind]
            nbytes = count * t.element_size()
            s["dst"].append((t.data_ptr() + at[kind], nbytes))
            at[kind] += nbytes
        s["server"] = M.Server(s["set"], arena_bytes=1 << 30)
    else:
        raise ValueError(op)
    return s


# ----------------------------------------------------------------- one pass
def run(s):
    case = s["case"]
    op = case["op"]
    if op == "fill":
        return s["gen"].fill(case["kind"], case["n"], s["out"])
    if op == "jump":
        s["gen"].fast_jump(s["hex"])
        return s["gen"].window().view(np.int32 if case["bits"] == 32 else np.int64)
    if op == "rand":
        if case["kind"] == "uint":
            return s["gen"].random_(s["out"])
        return s["gen"].uniform_(s["out"], M.KINDS[case["kind"]])
    if op == "sets":
        s["set"].generate_(s["reqs"])
        return s["out"]
    if op == "batch":
        s["plan"].rebase()
        s["plan"].launch()
        s["plan"].commit()
        return s["ints"], s["floats"]
    if op == "substreams":
        s["set"].substreams(s["base"], s["hex"])
        s["plan"].rebase()
        s["plan"].launch()
        s["plan"].commit()
        return s["out"]
    # serve: everything is submitted at once; results are copied into the
    # caller's tensors as they complete, then given back to the server
    srv, place = s["server"], {}
    for (gen, kind, count, skip), dst in zip(s["reqs"], s["dst"]):
        place[srv.submit(gen, kind, count, skip)] = dst
    done = []
    while len(done) < len(place):
        for c in srv.poll(wait_ms=100):
            dst, nbytes = place[c["ticket"]]
            M.device_copy(dst, c["out"], nbytes)
            done.append(c["ticket"])
    M.synchronize()
    for t in done:
        srv.release(t)
    return s["outs"]


# --------------------------------------------------------- what it must move
def work(case):
    op = case["op"]
    width = case.get("bits", 32) // 8
    window = 4 * (case.get("mexp") or 11213) // 32  # bytes of one state, about
    if op in ("fill", "rand"):
        return {"bytes": float(case["n"] * width + 2 * window), "flops": 0.0}
    if op == "sets":
        return {"bytes": float(case["gens"] * (case["n"] * width + 2 * window)), "flops": 0.0}
    if op == "batch":
        return {"bytes": float(2 * sum(_lengths(case)) * width + 2 * window * case["gens"]), "flops": 0.0}
    if op == "substreams":
        return {"bytes": float(case["gens"] * (4 * case["n"] + 2 * window)), "flops": 0.0}
    if op == "jump":
        return {"bytes": float(3 * window), "flops": 0.0}  # window in, polynomial, window out
    reqs = _serving_mix(case)[1]
    # written by the generators, then read and written by the copy
    return {"bytes": float(3 * sum(c * (8 if k == "close_open" else 4) for _, k, c, _ in reqs)), "flops": 0.0}


# ------------------------------------------ the same numbers in plain numpy
def _window(bits, p, seed):
    W = np.uint32 if bits == 32 else np.uint64
    mask, mul, sh = ((1 << 32) - 1, 1812433253, 30) if bits == 32 else (_MASK64, 6364136223846793005, 62)
    n = p.mexp // bits + 1
    hidden = (int(p.tbl[4]) ^ (int(p.tbl[8]) << 16)) & mask
    v = hidden & 0xFFFFFFFF if bits == 32 else hidden >> 32
    v = (v + (v >> 16)) & 0xFFFFFFFF
    v = (v + (v >> 8)) & 0xFF
    fill = int.from_bytes(bytes([v]) * (bits // 8), "little")
    a = [fill] * n
    a[0], a[1] = seed & mask, hidden
    for i in range(1, n):
        a[i] ^= (mul * (a[i - 1] ^ (a[i - 1] >> sh)) + i) & mask
    return np.array(a, W)


def _numbers(bits, p, seed, kind, count):
    """The first `count` numbers of the stream, as float64."""
    n, pos, step = p.mexp // bits + 1, p.pos, p.mexp // bits + 1 - p.pos
    W = np.uint32 if bits == 32 else np.uint64
    w = np.empty(n + count + step, W)
    w[:n] = _window(bits, p, seed)
    tbl = np.array(list(p.tbl), W)
    tmp = np.array(list(p.tmp_tbl), W)
    mask, s1, s2 = W(p.mask), np.uint32(p.sh1), np.uint32(p.sh2)
    for k in range(0, count, step):
        x = (w[k:k + step] & mask) ^ w[k + 1:k + 1 + step]
        y = w[k + pos:k + pos + step]
        if bits == 32:
            r = x ^ (x << s1) ^ (y >> s2)
        else:
            xh, xl = (x >> W(32)).astype(np.uint32), x.astype(np.uint32)
            nh = xl ^ (xl << s1) ^ ((y >> W(32)).astype(np.uint32) >> s2)
            nl = xh ^ (xh << s1) ^ (y.astype(np.uint32) >> s2)
            r = (nh.astype(W) << W(32)) | nl.astype(W)
        w[n + k:n + k + step] = r ^ tbl[r & W(15)]
    r = w[n:n + count]
    t = w[pos - 1:pos - 1 + count].astype(np.uint32)
    t ^= t >> np.uint32(16)
    t ^= t >> np.uint32(8)
    u = r ^ tmp[t & np.uint32(15)]
    # the leading 23 (52) bits of the tempered word as a fraction
    frac, scale = (u >> W(9), 2.0**-23) if bits == 32 else (u >> W(12), 2.0**-52)
    if kind == "open_open":
        frac = frac | W(1)
    f = frac.astype(np.float64) * scale
    return {"close1_open2": 1.0 + f, "close_open": f, "open_open": f, "open_close": 1.0 - f}[kind]


def exact(case, seed):
    """Floating outputs of the shorter cases; whole numbers, polynomials'
    windows and batches too long for numpy have none."""
    op = case["op"]
    if op not in ("fill", "rand", "sets") or case["kind"] == "uint":
        return None
    gens = case.get("gens", 1)
    if gens * case["n"] > 1 << 25:
        return None
    seeds = _splitmix(seed * 2654435761 + 12345, gens)
    if op == "sets":
        return np.stack([_numbers(case["bits"], _record(case, g % (128 if case["mexp"] else 200)), seeds[g], case["kind"],
                                  case["n"]) for g in range(gens)])
    return _numbers(case["bits"], _record(case, case["index"]), seeds[0], case["kind"], case["n"])
