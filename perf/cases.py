"""The work that performance is measured on: searches, writes and builds as a user's program makes them.

``listed`` holds the named cases, ``draw`` gives further ones of the same ranges, ``prepare`` makes what a program has
in hand before the call (a trained and filled index, the queries), and ``run`` is one pass through the public entry
points: the Python classes for data in host memory, the C ABI's ``*_device`` calls for data in GPU memory.

Four kinds of work:

* ``search``  -- ``AscendIndexIVFPQ.search`` of a batch of queries on a filled index;
* ``ingest``  -- a sliding window: a batch of vectors is added, queries are served, the batch leaves again;
* ``build``   -- a new index: training, bulk add, a first search;
* ``flat_f32`` / ``flat_i8`` -- brute-force search (ground truth, small collections, int8 descriptors).
"""
import ctypes
import math

import numpy as np
import torch

import indexsdk_amd as ix
from indexsdk_amd import _capi


def listed():
    return [
        # One query of an interactive service, at the shape of the reference's latency targets
        # (10M x 128, 1024 lists, 4 sub-quantizers, top 300), through host pointers: launches and latency count.
        {"name": "search_1", "kind": "search", "n": 10_000_000, "d": 128, "comp": 1024, "sigma": 0.25, "zipf": 0.0,
         "nlist": 1024, "m": 4, "metric": "L2", "lut_fp16": False, "nq": 1, "nprobe": 64, "k": 300, "io": "host"},
        # The largest batch of those targets, 64 queries at 128 probes, resident in GPU memory.
        {"name": "search_64", "kind": "search", "n": 10_000_000, "d": 128, "comp": 1024, "sigma": 0.25, "zipf": 0.0,
         "nlist": 1024, "m": 4, "metric": "L2", "lut_fp16": False, "nq": 64, "nprobe": 128, "k": 300, "io": "device"},
        # A small collection: 100k x 128, the first benchmark configuration.
        {"name": "search_100k", "kind": "search", "n": 100_000, "d": 128, "comp": 64, "sigma": 0.3, "zipf": 0.0,
         "nlist": 256, "m": 16, "metric": "L2", "lut_fp16": False, "nq": 1000, "nprobe": 16, "k": 10, "io": "device"},
        # Sizes nobody tuned for: dimension, list count, batch and k off every tile, through host pointers.
        {"name": "search_ragged", "kind": "search", "n": 1_234_567, "d": 200, "comp": 500, "sigma": 0.3, "zipf": 0.0,
         "nlist": 1500, "m": 40, "metric": "L2", "lut_fp16": False, "nq": 999, "nprobe": 33, "k": 150, "io": "host"},
        # The headline configuration: 10M x 128, 16384 lists, a batch of 10k queries.
        {"name": "search_10m", "kind": "search", "n": 10_000_000, "d": 128, "comp": 1024, "sigma": 0.25, "zipf": 0.0,
         "nlist": 16384, "m": 32, "metric": "L2", "lut_fp16": False, "nq": 10_000, "nprobe": 64, "k": 100,
         "io": "device"},
        # Inner product over unit-norm embeddings of 768 dimensions with the half-precision table.
        {"name": "search_ip_768", "kind": "search", "n": 4_000_000, "d": 768, "comp": 4096, "sigma": 0.05, "zipf": 0.0,
         "nlist": 8192, "m": 96, "metric": "IP", "lut_fp16": True, "nq": 4096, "nprobe": 128, "k": 100,
         "io": "device"},
        # Large k over lists of very uneven lengths (Zipf-sized clusters).
        {"name": "search_k1024", "kind": "search", "n": 20_000_000, "d": 96, "comp": 256, "sigma": 0.25, "zipf": 1.1,
         "nlist": 16384, "m": 48, "metric": "L2", "lut_fp16": False, "nq": 1024, "nprobe": 256, "k": 1024,
         "io": "device"},
        # A live index: 20k vectors come in, 32 queries are served, the same 20k leave.
        {"name": "ingest_20k", "kind": "ingest", "n": 2_000_000, "d": 128, "comp": 1024, "sigma": 0.25, "zipf": 0.0,
         "nlist": 4096, "m": 32, "metric": "L2", "lut_fp16": False, "nq": 32, "nprobe": 32, "k": 100, "nadd": 20_000,
         "io": "host"},
        # A new index from a million vectors in GPU memory.
        {"name": "build_1m", "kind": "build", "n": 1_000_000, "d": 128, "comp": 1024, "sigma": 0.25, "zipf": 0.0,
         "nlist": 1024, "m": 32, "metric": "L2", "lut_fp16": False, "nq": 64, "nprobe": 32, "k": 10,
         "ntrain": 131_072, "niter": 10, "io": "device"},
        # Exact neighbours in a million float vectors: ground truth for recall, and collections that need no lists.
        {"name": "flat_f32_1m", "kind": "flat_f32", "n": 1_000_000, "d": 128, "comp": 1024, "sigma": 0.25,
         "metric": "L2", "nq": 1000, "k": 100, "io": "host"},
        # A few queries against int8 descriptors (250k x 384, top 128), the small batches of the reference's own test.
        {"name": "flat_i8_8", "kind": "flat_i8", "n": 250_000, "d": 384, "nq": 8, "k": 128, "io": "host"},
        # The int8 benchmark configuration: 10M x 512, 2048 queries.
        {"name": "flat_i8_10m", "kind": "flat_i8", "n": 10_000_000, "d": 512, "nq": 2048, "k": 100, "io": "device"},
    ]


def _log_int(rng, lo, hi):
    """An integer between lo and hi, uniform over the logarithm; every second one is rounded to a multiple of 8 where it
    is large enough, the others stay as odd as they come."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if v >= 64 and rng.random() < 0.5:
        v = v // 8 * 8
    return max(lo, min(hi, v))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "search", "flat_f32", "flat_i8", "ingest", "build"])
    io = rng.choice(["host", "device"])
    if kind == "flat_i8":
        d = rng.choice([64, 96, 128, 256, 384, 512, 768, 1024])
        n = _log_int(rng, 20_000, 5_000_000_000 // d if d > 512 else 10_000_000)
        nq = min(_log_int(rng, 1, 2048), max(1, int(1.0e13 / (float(n) * d))))
        return {"kind": kind, "n": n, "d": d, "nq": nq, "k": _log_int(rng, 1, 300), "io": io}
    if kind == "flat_f32":
        d = rng.choice([64, 96, 100, 128, 200, 256, 384, 512, 768])
        n = _log_int(rng, 10_000, min(4_000_000, 600_000_000 // d))
        nq = min(_log_int(rng, 1, 4096), max(1, int(4.0e11 / (float(n) * d))))
        return {"kind": kind, "n": n, "d": d, "comp": _log_int(rng, 16, 1024), "sigma": round(rng.uniform(0.2, 1.0), 2),
                "metric": rng.choice(["L2", "L2", "IP"]), "nq": nq, "k": _log_int(rng, 1, 300), "io": io}
    d, m = rng.choice([(64, 16), (64, 8), (96, 48), (96, 24), (100, 20), (128, 4), (128, 8), (128, 16), (128, 32),
                       (128, 64), (160, 40), (200, 40), (256, 32), (256, 64), (384, 48), (384, 96), (512, 64),
                       (768, 96)])
    metric = rng.choice(["L2", "L2", "L2", "IP"])
    case = {"kind": kind, "d": d, "m": m, "metric": metric, "lut_fp16": rng.random() < 0.25,
            "comp": _log_int(rng, 64, 4096), "sigma": 0.05 if metric == "IP" else round(rng.uniform(0.2, 1.0), 2),
            "zipf": rng.choice([0.0, 0.0, 0.0, 1.1]), "io": io}
    if kind == "search":
        n = _log_int(rng, 50_000, min(10_000_000, 2_500_000_000 // d))
        nlist = _log_int(rng, max(64, n // 10_000), min(16384, n // 150))
        nprobe = _log_int(rng, 1, min(256, nlist))
        codes = nprobe * (n / nlist) * m * (3.0 if case["zipf"] else 1.0)   # bytes a query scans, uneven lists counted
        nq = min(_log_int(rng, 1, 10_000), max(1, int(1.3e10 / codes)))
        case.update(n=n, nlist=nlist, nq=nq, nprobe=nprobe, k=_log_int(rng, 1, 1024))
    elif kind == "ingest":
        n = _log_int(rng, 100_000, min(4_000_000, 600_000_000 // d))
        nlist = _log_int(rng, 64, min(8192, n // 150))
        case.update(n=n, nlist=nlist, nq=_log_int(rng, 1, 256), nprobe=_log_int(rng, 1, min(64, nlist)),
                    k=_log_int(rng, 1, 300), nadd=_log_int(rng, 100, 50_000))
    else:
        ntrain = _log_int(rng, 20_000, 150_000_000 // (8 * d))
        case.update(n=_log_int(rng, ntrain, 150_000_000 // d), nlist=_log_int(rng, 64, min(2048, ntrain // 50)),
                    nq=_log_int(rng, 1, 256), nprobe=16, k=_log_int(rng, 1, 100), ntrain=ntrain, niter=10)
    return case


# ---- data ---------------------------------------------------------------------------------------------------------

_CHUNK = 1 << 28   # floats generated and added at a time


def _metric(case):
    return ix.METRIC_INNER_PRODUCT if case["metric"] == "IP" else ix.METRIC_L2


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


class _Mixture:
    """Vectors of a Gaussian mixture made on the GPU: centres ~ N(0, 1) with noise of deviation sigma; for inner product
    both are normalised (unit-norm embeddings); zipf skews the cluster sizes."""

    def __init__(self, case, seed):
        self.d, self.sigma, self.unit = case["d"], case["sigma"], case["metric"] == "IP"
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)
        self.centres = torch.randn(case["comp"], self.d, generator=self.gen, device="cuda")
        if self.unit:
            self.centres /= self.centres.norm(dim=1, keepdim=True)
        self.bounds = None
        if case.get("zipf"):
            w = 1.0 / torch.arange(1, case["comp"] + 1, device="cuda", dtype=torch.float64) ** case["zipf"]
            self.bounds = torch.cumsum(w / w.sum(), 0)

    def rows(self, n):
        if self.bounds is None:
            which = torch.randint(0, self.centres.shape[0], (n,), generator=self.gen, device="cuda")
        else:
            at = torch.rand(n, generator=self.gen, device="cuda", dtype=torch.float64)
            which = torch.searchsorted(self.bounds, at).clamp_(max=self.centres.shape[0] - 1)
        x = torch.randn(n, self.d, generator=self.gen, device="cuda").mul_(self.sigma).add_(self.centres[which])
        if self.unit:
            x /= x.norm(dim=1, keepdim=True)
        return x


def _new_index(case, niter):
    cfg = ix.AscendIndexIVFPQConfig(niter=niter, lut_fp16=int(case["lut_fp16"]))
    return ix.AscendIndexIVFPQ(case["d"], _metric(case), case["nlist"], case["m"], 8, cfg)


def _filled_index(case, mix):
    """An index trained on a sample of the mixture (a few iterations: enough for lists as uneven as real ones) and
    filled with case["n"] of its vectors."""
    index = _new_index(case, 3)
    train = mix.rows(min(case["n"], max(20_000, 32 * case["nlist"])))
    torch.cuda.synchronize()
    _capi.check(_capi.load().ivfpq_train_device(index._h, train.shape[0], _ptr(train)))
    del train
    for s in range(0, case["n"], _CHUNK // case["d"]):
        x = mix.rows(min(_CHUNK // case["d"], case["n"] - s))
        torch.cuda.synchronize()
        _capi.check(_capi.load().ivfpq_add_with_ids_device(index._h, x.shape[0], _ptr(x), None))
    index.setNumProbes(case["nprobe"])
    return index


def _io(case, state, queries):
    """The queries, and for a device call its result arrays, where the case's program keeps them."""
    if case["io"] == "host":
        state["q"] = queries.cpu().numpy()
        return
    state["q"] = queries
    state["D"] = torch.empty(case["nq"], case["k"], device="cuda",
                             dtype=torch.int32 if case["kind"] == "flat_i8" else torch.float32)
    state["I"] = torch.empty(case["nq"], case["k"], device="cuda", dtype=torch.int64)


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "flat_i8":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        index = ix.AscendIndexInt8Flat(case["d"], ix.METRIC_L2)
        for s in range(0, case["n"], 4 * _CHUNK // case["d"]):
            rows = min(4 * _CHUNK // case["d"], case["n"] - s)
            x = torch.randint(-127, 128, (rows, case["d"]), generator=gen, device="cuda", dtype=torch.int8)
            torch.cuda.synchronize()
            _capi.check(_capi.load().flat_i8_add_with_ids_device(index._h, rows, _ptr(x), None))
        state["index"] = index
        _io(case, state, torch.randint(-127, 128, (case["nq"], case["d"]), generator=gen, device="cuda",
                                       dtype=torch.int8))
    elif case["kind"] == "flat_f32":
        mix = _Mixture(case, seed)
        index = ix.AscendIndexFlat(case["d"], _metric(case))
        x = mix.rows(case["n"])
        torch.cuda.synchronize()
        _capi.check(_capi.load().flat_add_with_ids_device(index._h, case["n"], _ptr(x), None))
        state["index"] = index
        _io(case, state, mix.rows(case["nq"]))
    elif case["kind"] == "build":
        mix = _Mixture(case, seed)
        x = mix.rows(case["n"])
        state["x"] = x.cpu().numpy() if case["io"] == "host" else x
        _io(case, state, mix.rows(case["nq"]))
    else:
        mix = _Mixture(case, seed)
        state["index"] = _filled_index(case, mix)
        if case["kind"] == "ingest":
            x = mix.rows(case["nadd"])
            ids = torch.arange(case["nadd"], dtype=torch.int64, device="cuda") + case["n"]
            state["x"], state["ids"] = (x.cpu().numpy(), ids.cpu().numpy()) if case["io"] == "host" else (x, ids)
        _io(case, state, mix.rows(case["nq"]))
    torch.cuda.synchronize()
    return state


# ---- one pass -----------------------------------------------------------------------------------------------------

def _search(state, index, call):
    """The batch's (distances, labels): through the Python class from host arrays, through the C ABI on the GPU."""
    case = state["case"]
    if case["io"] == "host":
        return index.search_int32(state["q"], case["k"]) if case["kind"] == "flat_i8" else index.search(state["q"], case["k"])
    _capi.check(call(index._h, case["nq"], _ptr(state["q"]), case["k"], _ptr(state["D"]), _ptr(state["I"])))
    return state["D"], state["I"]


def run(state):
    case, lib = state["case"], _capi.load()
    if case["kind"] == "flat_i8":
        return _search(state, state["index"], lib.flat_i8_search_device)
    if case["kind"] == "flat_f32":
        return _search(state, state["index"], lib.flat_search_device)
    if case["kind"] == "search":
        return _search(state, state["index"], lib.ivfpq_search_device)
    if case["kind"] == "ingest":
        index = state["index"]
        if case["io"] == "host":
            index.add_with_ids(state["x"], state["ids"])
        else:
            _capi.check(lib.ivfpq_add_with_ids_device(index._h, case["nadd"], _ptr(state["x"]), _ptr(state["ids"])))
        found = _search(state, index, lib.ivfpq_search_device)
        return found, index.remove_range(case["n"], case["n"] + case["nadd"])
    index = _new_index(case, case["niter"])
    if case["io"] == "host":
        index.train(state["x"][: case["ntrain"]])
        index.add(state["x"])
    else:
        _capi.check(lib.ivfpq_train_device(index._h, case["ntrain"], _ptr(state["x"])))
        _capi.check(lib.ivfpq_add_with_ids_device(index._h, case["n"], _ptr(state["x"]), None))
    index.setNumProbes(case["nprobe"])
    return index.get_trained(), _search(state, index, lib.ivfpq_search_device)


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def _search_work(case, nq):
    """Codes of the probed lists (a list that several queries probe is read once), centroids, codebooks, queries, results;
    coarse products, table products, one addition per code byte and query."""
    d, m, nlist = case["d"], case["m"], case["nlist"]
    codes = case["n"] * min(case["nprobe"], nlist) / nlist * m      # bytes one query looks up
    read = min(nq * codes, float(case["n"]) * m)
    return (read + 4.0 * (nlist + 256 + nq) * d + 12.0 * nq * case["k"],
            2.0 * nq * nlist * d + 512.0 * nq * d + nq * codes)


def work(case):
    n, d, nq, k = float(case["n"]), case["d"], case["nq"], case["k"]
    if case["kind"] == "flat_i8":
        return {"bytes": n * d + nq * d + 12.0 * nq * k, "flops": 2.0 * nq * n * d}
    if case["kind"] == "flat_f32":
        return {"bytes": 4.0 * (n + nq) * d + 12.0 * nq * k, "flops": 2.0 * nq * n * d}
    moved, flops = _search_work(case, nq)
    if case["kind"] == "ingest":   # vectors in; codes and ids written, and met again when they leave
        fresh = case["nadd"]
        moved += fresh * (4.0 * d + 2.0 * (case["m"] + 8))
        flops += 2.0 * fresh * (case["nlist"] + 256) * d
    elif case["kind"] == "build":   # the sample assigned to lists and codewords in every iteration, then every vector
        assigned = case["ntrain"] * case["niter"] + n
        moved += n * (4.0 * d + case["m"] + 8)
        flops += 2.0 * assigned * (case["nlist"] + 256) * d
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    if case["kind"] == "flat_i8":   # integers
        return "exact"
    if case["kind"] == "build":
        # k-means follows single roundings into other clusters, so training is defined bit for bit: sums in float64 in
        # sample order, assignments and codes by exact scores
        return "exact"
    if case["kind"] == "flat_f32":
        # expanded-form distances against float64: rel 4e-6, max 2.5e-5, 0.4 % of the ids trade places with a near tie
        return {"rel": 2e-5, "max": 1e-4, "differ": 0.01}
    # the same codes summed in another order (plain against rotated code layout): rel 1.3e-7, max 7e-7, 0.1 % of the ids
    return {"rel": 1e-6, "max": 5e-6, "differ": 0.004}
