"""Timed cases of the candidate-verification library, through its public entry points.

A case is a batch of reads with their candidate windows and the way a caller
hands it over: `api` "device" (the batch sits in HBM, verify_device and a wait
for the buffer's stream, as in bench.py), "host" (the reference's buffer API:
fill the pinned buffers, send, receive) or "serve" (the batch cut into
requests, all submitted to the continuous-batching server at once).

The data are the repository's synthetic workloads (seeded reference with N
runs; reads sampled from it with substitutions and indels; one candidate at
the true locus, the others at random loci) over a 256 Mbase reference, the
size of a large human chromosome.  The library handle, with the reference in
HBM and its buffers, and the server are made once per process, as a mapper
does; every batch is made from its seed.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "myers-gpu_amd", "python"))
import myers_amd as M  # noqa: E402

REF_SEED, REF_SIZE = 7, 256_000_000
DISTANCE = 0.1
BUFFER_BYTES = 768 << 20        # per buffer: the largest case's candidates and Peq entries fit
SERVE_BUFFER_BYTES = 128 << 20
MIXED = "100,200,400,600,800,1000"      # bench.py's mixed-length workload

_kept = {}


def _reference():
    if "ref" not in _kept:
        _kept["ref"] = M.synth_reference(REF_SEED, REF_SIZE)
    return _kept["ref"]


def _library():
    if "lib" not in _kept:
        _kept["lib"] = M.Myers(_reference(), REF_SIZE, num_buffers=1, avg_query=1000, cands_per_query=8,
                               buffer_bytes=BUFFER_BYTES)
    return _kept["lib"]


def _server():
    if "server" not in _kept:
        _kept["serve_lib"] = M.Myers(_reference(), REF_SIZE, num_buffers=3, avg_query=1000, cands_per_query=8,
                                     buffer_bytes=SERVE_BUFFER_BYTES)
        _kept["server"] = M.Server(_kept["serve_lib"], distance=DISTANCE)
    return _kept["server"]


def _case(name, api, reads, lengths, cands, err, exact=False, threshold=-1.0, long_share=0.0, requests=0):
    """lengths: "L" (one length), "a,b,c" (uniform over these) or "lo:hi"
    (log-uniform); cands: candidates per read, Poisson with that mean when negative; err: error
    rates of the reads "lo:hi"; long_share: that part of the reads is 2-20 kb long
    with 12% errors and four candidates."""
    return {"name": name, "api": api, "reads": reads, "lengths": lengths, "cands": cands, "err": err,
            "exact_windows": exact, "threshold": threshold, "long_share": long_share, "requests": requests}


def listed():
    return [
        # one read's candidates, sent and waited for: the smallest call, all latency
        _case("one_read_host", "host", 1, "150", 11, "0.02:0.02"),
        # 10K reads of 100 bases resident in HBM: bench.py's smallest workload
        _case("short_device", "device", 10_000, "100", 11, "0.025:0.025"),
        # a mapper's batch of short reads through the reference's buffer API
        _case("short_host", "host", 20_000, "150", 11, "0.01:0.05"),
        # quality-trimmed short reads: every length, odd ones, exact-start windows
        _case("trimmed_exact_device", "device", 150_000, "36:400", -11, "0.01:0.05", exact=True),
        # 100K reads of 1000 bases: bench.py's one-length workload
        _case("kilobase_device", "device", 100_000, "1000", 11, "0.04:0.04"),
        # mixed lengths: bench.py's headline workload at 300K reads
        _case("mixed_device", "device", 300_000, MIXED, -11, "0.01:0.05"),
        # the same mix when only hits within 20% error are wanted (threshold mode)
        _case("mixed_threshold_device", "device", 200_000, MIXED, -11, "0.01:0.05", threshold=0.2),
        # reads between the short and the long workloads
        _case("medium_device", "device", 40_000, "1000:4000", 4, "0.05:0.12"),
        # long noisy reads, throughput: bench.py's long-read workload at 20K reads
        _case("long_device", "device", 20_000, "2000:20000", 4, "0.12:0.12"),
        # a few long reads, waited for: bound by each candidate's own chain
        _case("long_few_host", "host", 100, "2000:20000", 4, "0.12:0.12"),
        # one serving request's mix of short and long reads as a batch of its own
        _case("request_host", "host", 500, MIXED, -11, "0.01:0.05", long_share=0.1),
        # a burst of such requests at the batching server
        _case("serve_burst", "serve", 6_000, MIXED, -11, "0.01:0.05", long_share=0.1, requests=24),
    ]


def draw(rng):
    """One more case of the same ranges: any interface, 1 to 150K reads, 36 to
    20,000 bases, one length or many, both window kinds, with or without a
    threshold; at most 4e12 cells."""
    api = rng.choice(["device", "device", "device", "host", "host", "serve"])
    kind = rng.choice(["one", "few", "spread", "long"])
    long_share = 0.0
    if kind == "one":
        top = int(math.exp(rng.uniform(math.log(36), math.log(2000))))
        lengths, cands, err = str(top), rng.choice([4, 8, 11, -11]), "0.01:0.05"
    elif kind == "few":
        picks = sorted({int(math.exp(rng.uniform(math.log(60), math.log(1500)))) for _ in range(rng.randint(2, 6))})
        top = picks[-1]
        lengths, cands, err = ",".join(map(str, picks)), rng.choice([8, 11, -11]), "0.01:0.05"
        long_share = rng.choice([0.0, 0.0, 0.1])
    elif kind == "spread":
        lo = int(math.exp(rng.uniform(math.log(36), math.log(500))))
        top = int(lo * rng.uniform(1.5, 6.0))
        lengths, cands, err = "%d:%d" % (lo, top), rng.choice([8, -11]), "0.01:0.08"
    else:
        lo = int(math.exp(rng.uniform(math.log(1000), math.log(6000))))
        top = min(20_000, int(lo * rng.uniform(1.3, 8.0)))
        lengths, cands, err = "%d:%d" % (lo, top), 4, "0.05:0.12"
    most = 4e12 / (max(float(top), 4000.0 if long_share else 0.0) ** 2 * 1.2 * abs(cands))
    if long_share:
        most = min(most, 40_000.0)
    most = max(2.0, min(150_000.0, most))
    reads = max(1, int(math.exp(rng.uniform(0.0, math.log(most)))))
    requests = min(reads, rng.randint(2, 32)) if api == "serve" else 0
    threshold = rng.choice([-1.0, -1.0, 0.1, 0.2]) if api != "serve" else -1.0
    return {k: v for k, v in _case("", api, reads, lengths, cands, err, exact=api != "serve" and rng.random() < 0.35,
                                   threshold=threshold, long_share=long_share, requests=requests).items() if k != "name"}


# ------------------------------------------------------------------ batches

def _spec(seed, reads, lengths, cands, err):
    kw = {"err_range": tuple(float(x) for x in err.split(":")), "distance": DISTANCE}
    if cands < 0:
        kw.update(poisson=float(-cands), cap=64)
    else:
        kw["candidates"] = cands
    if ":" in lengths:
        kw["log_uniform"] = tuple(int(x) for x in lengths.split(":"))
    elif "," in lengths:
        kw["choices"] = [int(x) for x in lengths.split(",")]
    else:
        kw["length"] = int(lengths)
    return M.make_spec(seed, reads, **kw)


def _merge(a, b):
    qi, ca = b["qinfo"].copy(), b["cands"].copy()
    qi[:, 0] += np.uint32(len(a["peq"]))
    ca["query"] += np.uint32(len(a["qinfo"]))
    return {"peq": np.concatenate([a["peq"], b["peq"]]), "qinfo": np.concatenate([a["qinfo"], qi]),
            "cands": np.concatenate([a["cands"], ca])}


def _short_batch(case, seed, reads):
    """`reads` reads; with Poisson candidate counts as many reads as it takes to
    make mean * reads candidates, so that every seed's results have one shape."""
    if case["cands"] >= 0:
        return M.synth_batch(_spec(seed, reads, case["lengths"], case["cands"], case["err"]), _reference(), REF_SIZE)
    total = -case["cands"] * reads
    more = reads + 8 + int(8 * math.sqrt(reads / -case["cands"]))
    b = M.synth_batch(_spec(seed, more, case["lengths"], case["cands"], case["err"]), _reference(), REF_SIZE)
    cands = b["cands"][:total]
    used = int(cands["query"].max()) + 1
    last = b["qinfo"][used - 1].astype(np.int64)
    return {"peq": b["peq"][:last[0] + (last[1] + 127) // 128], "qinfo": b["qinfo"][:used], "cands": cands}


def _batch(case, seed, reads):
    n_long = int(round(reads * case["long_share"]))
    b = _short_batch(case, 2 * seed + 1, reads - n_long)
    if n_long:
        b = _merge(b, M.synth_batch(_spec(2 * seed + 2, n_long, "2000:20000", 4, "0.12:0.12"), _reference(), REF_SIZE))
    return b


def _batches(case, seed):
    """The case's requests (one for a batch of its own), sizes as even as they come."""
    parts = max(1, case["requests"])
    each = [case["reads"] // parts + (1 if i < case["reads"] % parts else 0) for i in range(parts)]
    return [_batch(case, seed * 64 + i, n) for i, n in enumerate(each)]


class _Device:
    """A batch array in HBM, as verify_device takes it."""

    def __init__(self, a):
        self.tensor = torch.from_numpy(np.ascontiguousarray(a).view(np.int32).reshape(-1)).cuda()
        self.ptr = ctypes.c_void_p(self.tensor.data_ptr())


def prepare(case, seed):
    batches = _batches(case, seed)
    state = {"api": case["api"], "flags": M.WINDOW_EXACT if case["exact_windows"] else M.WINDOW_ALIGNED,
             "threshold": case["threshold"]}
    if case["api"] == "serve":
        state["server"] = _server()
        state["requests"] = [M.Server.request(b["peq"], b["qinfo"], b["cands"]) for b in batches]
        return state
    state["lib"] = _library()
    b = batches[0]
    if case["api"] == "host":
        state["batch"] = b
        return state
    state.update(entries=len(b["peq"]), queries=len(b["qinfo"]), count=len(b["cands"]), qinfo=b["qinfo"],
                 d_peq=_Device(b["peq"]), d_qinfo=_Device(b["qinfo"]), d_cands=_Device(b["cands"].view(np.uint8)),
                 d_results=_Device(np.zeros((len(b["cands"]), 2), np.uint32)))
    torch.cuda.synchronize()
    return state


def run(state):
    if state["api"] == "serve":
        server = state["server"]
        for ticket in [server.submit(req) for req, _ in state["requests"]]:
            server.wait(ticket)
        return [keep[3] for _, keep in state["requests"]]
    lib = state["lib"]
    lib.set_threshold(state["threshold"], 0)
    if state["api"] == "host":
        b = state["batch"]
        return lib.verify(b["peq"], b["qinfo"], b["cands"], DISTANCE, flags=state["flags"])
    M.verify_device(lib, state["d_peq"], state["entries"], state["d_qinfo"], state["queries"], state["d_cands"],
                    state["count"], DISTANCE, state["d_results"], flags=state["flags"], h_qinfo=state["qinfo"])
    M.synchronize(lib)
    return state["d_results"].tensor.view(-1, 2)


# ------------------------------------------------------------- work, values

def _window(m):
    f = np.float32(1.0) + np.float32(2.0) * np.float32(DISTANCE)
    return np.floor(np.asarray(m).astype(np.float32) * f).astype(np.int64)


def work(case):
    """Bytes: each window's packed text, candidate and result once, each read's
    Peq and qinfo once.  Operations: ten 32-bit logic operations per 32 cells of
    the DP (m rows by n window columns), bench.py's unit."""
    def part(reads, lengths, cands):
        if ":" in lengths:
            lo, hi = (int(x) for x in lengths.split(":"))
            m = np.exp(np.linspace(math.log(lo), math.log(hi), 2001)).round()
        else:
            m = np.array([int(x) for x in lengths.split(",")])
        m, c = m.astype(np.int64), abs(cands)
        n = _window(m)
        return (reads * float((c * ((n + 1) // 2 + 24) + 80 * ((m + 127) // 128) + 8).mean()),
                reads * c * float((m * n).mean()))
    n_long = int(round(case["reads"] * case["long_share"]))
    b1, c1 = part(case["reads"] - n_long, case["lengths"], case["cands"])
    b2, c2 = part(n_long, "2000:20000", 4)
    return {"bytes": b1 + b2, "flops": (c1 + c2) * 10 / 32}


def exact(case, seed):
    """{column, score} of every candidate from the plain DP over its window
    (64-bit integers), for batches where that takes seconds."""
    if work(case)["flops"] * 3.2 > 2.5e9 or case["requests"]:
        return None
    b = _batch(case, seed * 64, case["reads"])
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    m_of, entry_of = b["qinfo"][:, 1].astype(np.int64), b["qinfo"][:, 0].astype(np.int64)
    query, pos = b["cands"]["query"].astype(np.int64), b["cands"]["position"].astype(np.int64)
    if len(np.unique(m_of)) > 64:
        return None
    words = torch.from_numpy(_reference().view(np.int32)).to(dev)
    peq = torch.from_numpy(b["peq"].view(np.int32)).to(dev)
    out = np.zeros((len(query), 2), np.int64)
    for m in np.unique(m_of):
        pick = np.nonzero(m_of[query] == m)[0]
        n = int(_window(m))
        skip = REF_SIZE - pos[pick] <= n
        start = pos[pick] if case["exact_windows"] else pos[pick] // 8 * 8
        cols = n if case["exact_windows"] else 8 * (n // 8 + (2 if n % 8 else 1))
        at = torch.from_numpy(start).to(dev)
        q = torch.from_numpy(entry_of[query[pick]]).to(dev)
        row = torch.arange(int(m), device=dev)
        # match[c][candidate][row]: the read's base at this row matches code c
        match = torch.stack([(peq[q[:, None] + row // 128, 4 * c + row % 128 // 32] >> (row % 32)) & 1 for c in range(5)])
        d = torch.arange(1, int(m) + 1, device=dev).repeat(len(pick), 1)
        best, where = d[:, -1].clone(), torch.zeros(len(pick), dtype=torch.int64, device=dev)
        who = torch.arange(len(pick), device=dev)
        for j in range(cols):
            p = at + j
            word = p // 8
            code = torch.where(word < len(words), (words[word.clamp(max=len(words) - 1)] >> (4 * (p % 8)).int()) & 7, 4)
            same = match[torch.where(code > 4, 0, code).long(), who].long()
            diag = torch.cat([torch.zeros_like(d[:, :1]), d[:, :-1]], 1)
            d = torch.minimum(diag + 1 - same, d + 1)
            d = torch.cummin(torch.cat([torch.zeros_like(d[:, :1]), d - row - 1], 1), 1).values[:, 1:] + row + 1
            better = d[:, -1] < best
            best, where = torch.where(better, d[:, -1], best), torch.where(better, j, where)
        best, where = best.cpu().numpy(), where.cpu().numpy()
        none = np.int64(0xFFFFFFFF)
        if case["threshold"] >= 0:
            over = best > int(np.float32(m) * np.float32(case["threshold"]))
            best, where = np.where(over, none, best), np.where(over, none, where)
        out[pick, 0], out[pick, 1] = np.where(skip, 0, where), np.where(skip, none, best)
    # the device path's results are int32 tensors, the buffer API's unsigned numbers
    return out.astype(np.uint32).view(np.int32) if case["api"] == "device" else out.astype(np.uint32)
