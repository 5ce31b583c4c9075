"""What is timed when the speed of this library is looked at: its work, through its public entry points.

Two layers are used the way programs use them.  The index layer (vsag_amd.pyvsag: build / add / knn_search /
knn_search_batch) takes and returns host arrays, as the reference's python binding does.  The kernel layer
(vsag_amd.capi, the C ABI of include/vsag_amd.h) works on device memory: a serving or training program that keeps its
vectors on the GPU hands over torch tensors, and the stores, workspaces and result arrays that it keeps between calls.

  knn     one query per call, micro-batches and batches on an index of either type
  build   an index from host rows, and more rows added to it
  scan    flat scan of a device-resident store, with a filter or a rerank where the case says so
  ivf     route -> scan of the posting lists -> rerank
  kmeans  one Lloyd iteration (assignment and update)
  encode  training of a quantizer and encoding of the rows

The sizes are those of bench.py and of the tests, or generic ones between them.
"""
import ctypes as C
import json
import math

import numpy as np
import torch

from vsag_amd import capi, pyvsag

DEVICE = "cuda"


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # The reference's own calling pattern: one query per KnnSearch call, every code of a large flat index.
        {"name": "knn one flat sq8 1M", "path": "knn", "index": "brute_force", "quant": "sq8", "metric": "l2",
         "n": 1000000, "dim": 128, "nq": 1, "k": 10},
        # The same on the ivf index with its default codec (fp32 lists): interactive search.
        {"name": "knn one ivf fp32 300k", "path": "knn", "index": "ivf", "quant": "fp32", "metric": "l2", "n": 300000,
         "dim": 128, "nq": 1, "k": 10, "nlist": 1024, "nprobe": 32, "reorder": False},
        # A server that gathers a few dozen requests before it calls: text embeddings under cosine, raw vectors.
        {"name": "knn 32 flat fp32 768d", "path": "knn", "index": "brute_force", "quant": "fp32", "metric": "cosine",
         "n": 100003, "dim": 768, "nq": 32, "k": 10},
        # A batch job against an ivf index that reranks, inner product, a dimension that fills no tile.
        {"name": "knn 1000 ivf sq8 200d", "path": "knn", "index": "ivf", "quant": "sq8", "metric": "ip", "n": 200000,
         "dim": 200, "nq": 1000, "k": 20, "nlist": 512, "nprobe": 24, "reorder": True},
        # Ingestion: train, build and a later add, all from host rows.
        {"name": "build ivf sq8 120k", "path": "build", "index": "ivf", "quant": "sq8", "metric": "l2", "n": 120000,
         "dim": 96, "nlist": 256},
        # Exact search, the smallest of the benchmark's configurations.
        {"name": "scan fp32 100k 1000q", "path": "scan", "quant": "fp32", "metric": "l2", "n": 100000, "dim": 128,
         "nq": 1000, "k": 10, "keep": 1.0, "kcand": 0, "data": "uniform"},
        # The headline: every code of 1M against 10 000 queries.
        {"name": "scan sq8 1M 10000q", "path": "scan", "quant": "sq8", "metric": "l2", "n": 1000000, "dim": 128,
         "nq": 10000, "k": 10, "keep": 1.0, "kcand": 0, "data": "mixture"},
        # Search under a pre-filter (an attribute or permission mask that keeps a third of the vectors).
        {"name": "scan sq8 filtered 200q", "path": "scan", "quant": "sq8", "metric": "ip", "n": 500000, "dim": 100,
         "nq": 200, "k": 100, "keep": 0.3, "kcand": 0, "data": "mixture"},
        # Binary codes with an exact rerank of the candidates, the largest flat configuration.
        {"name": "scan rabitq 5M 10000q", "path": "scan", "quant": "rabitq", "metric": "ip", "n": 5000000, "dim": 768,
         "nq": 10000, "k": 10, "keep": 1.0, "kcand": 200, "data": "sphere"},
        # The largest index: 10M vectors in 4-bit posting lists.
        {"name": "ivf sq4u 10M 10000q", "path": "ivf", "quant": "sq4_uniform", "metric": "l2", "n": 10000000, "dim": 128,
         "nq": 10000, "k": 10, "kcand": 100, "nlist": 4096, "nprobe": 64},
        # One iteration of k-means training at the benchmark's size.
        {"name": "kmeans 1M 960d k4096", "path": "kmeans", "n": 1000000, "dim": 960, "k": 4096},
        # Re-encoding a collection: bounds from a sample, then the codes.
        {"name": "encode sq8 1M", "path": "encode", "quant": "sq8", "metric": "l2", "n": 1000000, "dim": 128},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dim(rng, most=960):
    d = rng.choice([32, 64, 96, 100, 128, 128, 128, 200, 256, 384, 512, 768, 960, 0])
    return min(most, d if d else rng.randint(17, 960))


def draw(rng):
    path = rng.choice(["knn"] * 6 + ["scan"] * 5 + ["ivf"] * 3 + ["kmeans", "kmeans", "encode", "build"])
    metric = rng.choice(["l2", "l2", "ip", "cosine"])
    if path == "knn":
        index = rng.choice(["brute_force", "ivf"])
        quant = rng.choice(["fp32", "fp32", "sq8", "sq8", "sq4_uniform", "sq8_uniform"])
        dim = _dim(rng)
        n = min(_log(rng, 20000, 1000000 if index == "brute_force" else 300000), 128000000 // dim)
        nq = 1 if rng.random() < 0.4 else _log(rng, 2, 10000)
        c = {"path": path, "index": index, "quant": quant, "metric": metric, "n": n, "dim": dim,
             "k": rng.choice([1, 10, 10, 10, 20, 50, 100])}
        share = 1.0
        if index == "ivf":
            c["nlist"] = _log(rng, 0.5 * math.sqrt(n), 2 * math.sqrt(n))
            c["nprobe"] = _log(rng, 4, max(5, c["nlist"] // 8))
            c["reorder"] = quant != "fp32" and rng.random() < 0.7
            share = c["nprobe"] / c["nlist"]
        c["nq"] = max(1, min(nq, int(1.28e12 / (share * n * dim))))
        return c
    if path == "scan":
        quant = rng.choice(["fp32", "fp32", "sq8", "sq8", "sq8", "sq4", "sq4_uniform", "sq8_uniform", "rabitq", "rabitq"])
        dim = _dim(rng)
        keep = rng.uniform(0.05, 0.9) if rng.random() < 0.3 else 1.0
        rabitq = quant == "rabitq"
        n = min(_log(rng, 50000, 5000000 if rabitq else 2000000), (3840000000 if rabitq else 640000000) // dim)
        c = {"path": path, "quant": quant, "metric": rng.choice(["l2", "ip"]) if rabitq else metric, "n": n, "dim": dim,
             "k": 10 if rabitq else rng.choice([1, 10, 10, 20, 50, 100]), "keep": keep,
             "kcand": 200 if rabitq else 0, "data": "sphere" if rabitq else rng.choice(["mixture", "mixture", "uniform"])}
        most = 6.4e11 if keep < 1.0 else 3.84e13 if rabitq else 1.28e12
        c["nq"] = max(1, min(_log(rng, 16, 10000), int(most / (n * dim))))
        return c
    if path == "ivf":
        quant = rng.choice(["fp32", "sq8", "sq8", "sq4_uniform", "sq4_uniform", "sq8_uniform", "rabitq", "pqfs"])
        dim = _dim(rng, 768)
        if quant == "pqfs":
            dim = min(256, dim + dim % 2)
        n = min(_log(rng, 200000, 10000000), 1280000000 // dim)
        nlist = min(4096, _log(rng, 0.5 * math.sqrt(n), 2 * math.sqrt(n)))
        nprobe = _log(rng, 4, max(8, nlist // 16))
        k = rng.choice([1, 10, 10, 20])
        return {"path": path, "quant": quant, "metric": rng.choice(["l2", "ip"]), "n": n, "dim": dim,
                "nq": max(1, min(_log(rng, 16, 10000), int(2e11 * nlist / (nprobe * n * dim)))), "k": k,
                "kcand": 0 if quant == "fp32" else 10 * k, "nlist": nlist, "nprobe": nprobe}
    if path == "kmeans":
        dim = _dim(rng)
        n = min(_log(rng, 20000, 1000000), 960000000 // dim)
        return {"path": path, "n": n, "dim": dim, "k": min(_log(rng, 64, 4096), n // 16)}
    if path == "encode":
        quant = rng.choice(["sq8", "sq8", "sq4", "sq4_uniform", "sq8_uniform", "rabitq"])
        dim = _dim(rng)
        n = min(_log(rng, 50000, 2000000), 256000000 // dim)
        return {"path": path, "quant": quant, "metric": rng.choice(["l2", "ip"]) if quant == "rabitq" else metric, "n": n,
                "dim": dim}
    dim = _dim(rng, 128)
    n = _log(rng, 10000, 110000)
    return {"path": "build", "index": rng.choice(["ivf", "ivf", "brute_force"]), "quant": rng.choice(["fp32", "sq8", "sq4_uniform"]),
            "metric": metric, "n": n, "dim": dim, "nlist": min(256, _log(rng, 0.5 * math.sqrt(n), 2 * math.sqrt(n)))}


# ------------------------------------------------------------------------------------------------ inputs
def _rows(gen, n, dim, data, means=None):
    """n rows on the GPU: clustered vectors (a Gaussian mixture), uniform ones, or unit vectors in random directions."""
    if data == "uniform":
        return torch.rand(n, dim, device=DEVICE, generator=gen)
    x = torch.randn(n, dim, device=DEVICE, generator=gen)
    for s in range(0, n, 1 << 20):
        block = x[s:s + (1 << 20)]
        if data == "sphere":
            block /= block.norm(dim=1, keepdim=True)
        else:
            which = torch.randint(0, means.shape[0], (block.shape[0],), device=DEVICE, generator=gen)
            block.mul_(0.05).add_(means[which])
    return x


def _inputs(case, seed, nq):
    """Base rows and queries of one distribution."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    data = case.get("data", "mixture")
    means = torch.rand(max(100, case["n"] // 1000), case["dim"], device=DEVICE, generator=gen)
    x = _rows(gen, case["n"], case["dim"], data, means)
    q = _rows(gen, nq, case["dim"], data, means) if nq else None
    return gen, x, q


def _device_bytes(nbytes):
    return torch.empty(int(nbytes) + 256, dtype=torch.uint8, device=DEVICE)


def _check(rc):
    capi.check(rc)


class Store:
    """A store of codes on the device with the buffers that belong to it."""

    def __init__(self, quantizer, kind, metric, dim):
        self.lib, self.keep = capi.load_library(), quantizer
        p = capi.StoreParams()
        p.kind, p.metric, p.dim = kind, metric, dim
        for field, name in (("lower_bound_dev", "lb"), ("diff_dev", "diff"), ("rotation_dev", "rotation"),
                            ("centroid_dev", "centroid"), ("codebooks_dev", "codebooks")):
            if name in quantizer:
                setattr(p, field, quantizer[name].data_ptr())
        p.rabitq_query_bits = 4
        p.pq_dim = quantizer.get("pq_dim", 0)
        self.handle = C.c_void_p()
        _check(self.lib.vsag_amd_store_create(C.byref(p), C.byref(self.handle)))

    def __del__(self):
        if self.handle:
            torch.cuda.synchronize()
            self.lib.vsag_amd_store_destroy(self.handle)
            self.handle = None


def _quantizer_buffers(quant, dim, seed):
    f = lambda *shape: torch.empty(*shape, dtype=torch.float32, device=DEVICE)  # noqa: E731
    if quant in ("sq8", "sq4"):
        return {"lb": f(dim), "diff": f(dim)}
    if quant in ("sq8_uniform", "sq4_uniform"):
        return {"lb": f(2)}
    if quant == "rabitq":
        rotation, r = np.linalg.qr(np.random.default_rng(seed).standard_normal((dim, dim)))
        rotation = np.ascontiguousarray(rotation * np.sign(np.diag(r)), dtype=np.float32)
        return {"rotation": torch.from_numpy(rotation).to(DEVICE), "centroid": f(dim)}
    if quant == "pqfs":
        return {"codebooks": f(dim * 16), "pq_dim": dim // 2}
    return {}


def _train_workspace(lib, quant, n, dim, quantizer):
    if quant == "pqfs":
        return _device_bytes(lib.vsag_amd_pq_train_workspace_bytes(n, dim, quantizer["pq_dim"]))
    return _device_bytes(lib.vsag_amd_sq_train_workspace_bytes(n, dim, 0))


def _train(lib, quant, metric, x, n, dim, quantizer, ws):
    p, wp, wn = x.data_ptr(), ws.data_ptr(), ws.numel()
    bits = 8 if quant.startswith("sq8") else 4
    if quant in ("sq8", "sq4"):
        _check(lib.vsag_amd_sq_train(p, n, dim, bits, metric, capi.SQ_TRAIN_TRUNC_BOUND, 0.05, 0,
                                     quantizer["lb"].data_ptr(), quantizer["diff"].data_ptr(), wp, wn, None))
    elif quant in ("sq8_uniform", "sq4_uniform"):
        mode = capi.SQ_TRAIN_CLASSIC if bits == 8 else capi.SQ_TRAIN_TRUNC_BOUND
        _check(lib.vsag_amd_sq_train_uniform(p, n, dim, bits, metric, mode, 0.05, 0, quantizer["lb"].data_ptr(), wp, wn,
                                             None))
    elif quant == "rabitq":
        _check(lib.vsag_amd_rabitq_train(p, n, dim, quantizer["rotation"].data_ptr(), quantizer["centroid"].data_ptr(),
                                         None))
    elif quant == "pqfs":
        _check(lib.vsag_amd_pq_train(p, n, dim, quantizer["pq_dim"], metric, 11, quantizer["codebooks"].data_ptr(), wp,
                                     wn, None))


def _code_size(lib, quant, metric, dim, quantizer):
    bits = 4 if quant == "rabitq" else 0
    return int(lib.vsag_amd_code_size(capi.KINDS[quant], metric, quantizer.get("pq_dim", dim), bits))


def _encode(lib, quant, metric, x, n, dim, quantizer, codes):
    bits = 8 if quant.startswith("sq8") else 4
    if quant in ("sq8", "sq4"):
        _check(lib.vsag_amd_sq_encode(x.data_ptr(), n, dim, bits, metric, quantizer["lb"].data_ptr(),
                                      quantizer["diff"].data_ptr(), codes.data_ptr(), None))
    elif quant in ("sq8_uniform", "sq4_uniform"):
        _check(lib.vsag_amd_squ_encode(x.data_ptr(), n, dim, bits, metric, quantizer["lb"].data_ptr(), codes.data_ptr(),
                                       None))
    elif quant == "rabitq":
        _check(lib.vsag_amd_rabitq_encode(x.data_ptr(), n, dim, quantizer["rotation"].data_ptr(),
                                          quantizer["centroid"].data_ptr(), metric, 4, codes.data_ptr(), None))
    elif quant == "pqfs":
        _check(lib.vsag_amd_pq_encode(x.data_ptr(), n, dim, quantizer["pq_dim"], quantizer["codebooks"].data_ptr(),
                                      metric, codes.data_ptr(), None, None))


def _encoded(lib, case, metric, x, seed):
    """A quantizer trained on the first rows, and the codes of all rows (fp32: the rows themselves)."""
    quant, n, dim = case["quant"], case["n"], case["dim"]
    if quant == "fp32":
        return {}, x
    quantizer = _quantizer_buffers(quant, dim, seed)
    sample = min(n, 262144)
    _train(lib, quant, metric, x, sample, dim, quantizer, _train_workspace(lib, quant, sample, dim, quantizer))
    codes = torch.empty(n * _code_size(lib, quant, metric, dim, quantizer), dtype=torch.uint8, device=DEVICE)
    _encode(lib, quant, metric, x, n, dim, quantizer, codes)
    return quantizer, codes


def _index(case, host_rows, count):
    params = {"base_quantization_type": case["quant"]}
    if case["index"] == "ivf":
        params["buckets_count"] = case["nlist"]
        if case.get("reorder"):
            params.update(use_reorder=True, precise_quantization_type="fp32")
    index = pyvsag.Index(case["index"], json.dumps({"dtype": "float32", "metric_type": case["metric"], "dim": case["dim"],
                                                    "index_param": params}))
    index.build(host_rows[:count], np.arange(count, dtype=np.int64) * 3 + 7, count, case["dim"])
    return index


def _search_parameters(case, nprobe):
    if case["index"] == "ivf":
        return json.dumps({"ivf": {"scan_buckets_count": nprobe, "factor": 4.0}})
    return "{}"


def _results(nq, k):
    return (torch.empty(nq, k, dtype=torch.int32, device=DEVICE), torch.empty(nq, k, dtype=torch.float32, device=DEVICE))


def prepare(case, seed):
    capi.init(0)
    path, dim = case["path"], case["dim"]
    lib = capi.load_library()
    s = {"case": case, "lib": lib}
    if path in ("knn", "build"):
        _, x, q = _inputs(case, seed, case["nq"] if path == "knn" else 100)
        rows, s["queries"] = x.cpu().numpy(), q.cpu().numpy()
        if path == "knn":
            s["index"] = _index(case, rows, case["n"])
            s["parameters"] = _search_parameters(case, case.get("nprobe", 0))
        else:
            s["rows"] = rows
        return s
    metric = s["metric"] = capi.METRICS[case.get("metric", "l2")]
    gen, x, q = _inputs(case, seed, case.get("nq", 0))
    s["x"], s["q"] = x, q
    if path == "scan":
        nq, kc = case["nq"], case["kcand"] or case["k"]
        quantizer, codes = _encoded(lib, case, metric, x, seed)
        s["store"] = Store(quantizer, capi.KINDS[case["quant"]], metric, dim)
        _check(lib.vsag_amd_store_append(s["store"].handle, codes.data_ptr(), case["n"], None))
        s["options"] = None
        if case["keep"] < 1.0:
            words = (case["n"] + 31) // 32
            denied = torch.rand(words, 32, device=DEVICE, generator=gen) >= case["keep"]
            weights = 1 << torch.arange(32, dtype=torch.int64, device=DEVICE)
            s["deny"] = (denied * weights).sum(1).to(torch.int32)
            s["options"] = capi.SearchOptions()
            s["options"].deny_bits_dev = s["deny"].data_ptr()
        s["ids"], s["dists"] = _results(nq, kc)
        if case["kcand"]:
            s["out_ids"], s["out_dists"] = _results(nq, case["k"])
        else:
            s["x"] = None
        s["ws"] = _device_bytes(lib.vsag_amd_flat_scan_workspace_bytes(s["store"].handle, nq, kc))
    elif path == "ivf":
        n, nq, nlist, nprobe = case["n"], case["nq"], case["nlist"], case["nprobe"]
        kc = case["kcand"] or case["k"]
        centroids = x[torch.randint(0, n, (nlist,), device=DEVICE, generator=gen)].contiguous()
        sample = min(n, 64 * nlist)
        labels = torch.empty(n, dtype=torch.int32, device=DEVICE)
        ws = _device_bytes(lib.vsag_amd_kmeans_run_workspace_bytes(sample, dim, nlist))
        _check(lib.vsag_amd_kmeans_run(x.data_ptr(), sample, dim, centroids.data_ptr(), nlist, 5, 7, labels.data_ptr(), None,
                                       ws.data_ptr(), ws.numel(), None))
        ws = _device_bytes(lib.vsag_amd_kmeans_assign_workspace_bytes(n, dim, nlist))
        _check(lib.vsag_amd_kmeans_assign(x.data_ptr(), n, dim, centroids.data_ptr(), nlist, labels.data_ptr(), None, None,
                                          ws.data_ptr(), ws.numel(), None))
        quantizer, codes = _encoded(lib, case, metric, x, seed)
        s["lists"] = Store(quantizer, capi.KINDS[case["quant"]], metric, dim)
        _check(lib.vsag_amd_store_set_lists(s["lists"].handle, codes.data_ptr(), labels.data_ptr(), n, nlist, None))
        s["router"] = Store({}, capi.KIND_FP32, metric, dim)
        _check(lib.vsag_amd_store_append(s["router"].handle, centroids.data_ptr(), nlist, None))
        s["buckets"], s["bucket_dists"] = _results(nq, nprobe)
        s["ids"], s["dists"] = _results(nq, kc)
        s["out_ids"], s["out_dists"] = _results(nq, case["k"])
        s["route_ws"] = _device_bytes(lib.vsag_amd_ivf_route_workspace_bytes(s["router"].handle, nq, nprobe))
        s["ws"] = _device_bytes(lib.vsag_amd_ivf_scan_workspace_bytes(s["lists"].handle, nq, nprobe, kc))
    elif path == "kmeans":
        n, k = case["n"], case["k"]
        s["start"] = x[torch.randperm(n, device=DEVICE, generator=gen)[:k]].contiguous()
        s["centroids"] = torch.empty_like(s["start"])
        s["labels"] = torch.empty(n, dtype=torch.int32, device=DEVICE)
        s["min_dist"] = torch.empty(n, dtype=torch.float32, device=DEVICE)
        s["loss"] = torch.empty(1, dtype=torch.float64, device=DEVICE)
        s["counts"] = torch.empty(k, dtype=torch.int32, device=DEVICE)
        s["ws"] = _device_bytes(max(lib.vsag_amd_kmeans_assign_workspace_bytes(n, dim, k),
                                    lib.vsag_amd_kmeans_update_workspace_bytes(n, dim, k)))
    else:
        quantizer = s["quantizer"] = _quantizer_buffers(case["quant"], dim, seed)
        s["codes"] = torch.empty(case["n"], _code_size(lib, case["quant"], metric, dim, quantizer), dtype=torch.uint8,
                                 device=DEVICE)
        s["ws"] = _train_workspace(lib, case["quant"], case["n"], dim, quantizer)
    return s


# ------------------------------------------------------------------------------------------------ one pass
def run(s):
    case, lib = s["case"], s["lib"]
    path, dim = case["path"], case["dim"]
    if path == "knn":
        if case["nq"] == 1:
            return s["index"].knn_search(s["queries"][0], case["k"], s["parameters"])
        return s["index"].knn_search_batch(s["queries"], case["k"], s["parameters"])
    if path == "build":
        # nine tenths of the rows at once, the rest added to the filled index; a first search shows what was built
        first = case["n"] * 9 // 10
        more = case["n"] - first
        index = _index(case, s["rows"], first)
        index.add(s["rows"][first:], np.arange(first, case["n"], dtype=np.int64) * 3 + 7, more, dim)
        found = index.knn_search_batch(s["queries"], 10, _search_parameters(case, 16))
        count = index.get_num_elements()
        index.close()
        return found + (count,)
    if path == "scan":
        nq, k, kc = case["nq"], case["k"], case["kcand"] or case["k"]
        options = C.byref(s["options"]) if s["options"] is not None else None
        _check(lib.vsag_amd_flat_scan_topk_ex(s["store"].handle, s["q"].data_ptr(), nq, kc, options, s["ids"].data_ptr(),
                                              s["dists"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), None))
        if not case["kcand"]:
            return s["ids"], s["dists"]
        _check(lib.vsag_amd_rerank_fp32(s["x"].data_ptr(), case["n"], dim, s["metric"], s["q"].data_ptr(), nq,
                                        s["ids"].data_ptr(), kc, k, s["out_ids"].data_ptr(), s["out_dists"].data_ptr(), None))
        return s["ids"], s["dists"], s["out_ids"], s["out_dists"]
    if path == "ivf":
        nq, k, kc, nprobe = case["nq"], case["k"], case["kcand"] or case["k"], case["nprobe"]
        q = s["q"].data_ptr()
        _check(lib.vsag_amd_ivf_route(s["router"].handle, q, nq, nprobe, s["buckets"].data_ptr(), s["bucket_dists"].data_ptr(),
                                      s["route_ws"].data_ptr(), s["route_ws"].numel(), None))
        _check(lib.vsag_amd_ivf_scan_topk(s["lists"].handle, q, nq, s["buckets"].data_ptr(), nprobe, kc, s["ids"].data_ptr(),
                                          s["dists"].data_ptr(), s["ws"].data_ptr(), s["ws"].numel(), None))
        if not case["kcand"]:
            return s["buckets"], s["ids"], s["dists"]
        _check(lib.vsag_amd_rerank_fp32(s["x"].data_ptr(), case["n"], dim, s["metric"], q, nq, s["ids"].data_ptr(), kc, k,
                                        s["out_ids"].data_ptr(), s["out_dists"].data_ptr(), None))
        return s["buckets"], s["ids"], s["dists"], s["out_ids"], s["out_dists"]
    if path == "kmeans":
        n, k, x, ws = case["n"], case["k"], s["x"].data_ptr(), s["ws"]
        s["centroids"].copy_(s["start"])
        _check(lib.vsag_amd_kmeans_assign(x, n, dim, s["centroids"].data_ptr(), k, s["labels"].data_ptr(),
                                          s["min_dist"].data_ptr(), s["loss"].data_ptr(), ws.data_ptr(), ws.numel(), None))
        _check(lib.vsag_amd_kmeans_update(x, s["labels"].data_ptr(), n, dim, k, s["centroids"].data_ptr(),
                                          s["counts"].data_ptr(), ws.data_ptr(), ws.numel(), None))
        return s["labels"], s["min_dist"], s["loss"], s["centroids"], s["counts"]
    _train(lib, case["quant"], s["metric"], s["x"], case["n"], dim, s["quantizer"], s["ws"])
    _encode(lib, case["quant"], s["metric"], s["x"], case["n"], dim, s["quantizer"], s["codes"])
    quantizer = s["quantizer"]
    return tuple(quantizer[name] for name in ("lb", "diff", "centroid") if name in quantizer) + (s["codes"],)


# ------------------------------------------------------------------------------------------------ what it takes
_BITS = {"fp32": 32, "sq8": 8, "sq4": 4, "sq8_uniform": 8, "sq4_uniform": 4, "rabitq": 1, "pqfs": 2}


def work(case):
    path, n, dim = case["path"], case["n"], case["dim"]
    if path in ("knn", "scan", "ivf"):
        nq, k = case["nq"], case["k"]
        code = dim * _BITS[case["quant"]] / 8.0
        pairs, codes, flops = float(nq) * n, float(n), 0.0
        read = 4.0 * nq * dim + 12.0 * nq * k
        if "nlist" in case:
            pairs *= case["nprobe"] / case["nlist"]
            codes = min(codes, pairs)
            flops += 2.0 * nq * case["nlist"] * dim
            read += 4.0 * case["nlist"] * dim
        if case.get("keep", 1.0) < 1.0:
            pairs, codes = pairs * case["keep"], codes * case["keep"]
            read += n / 8.0
        reranked = case.get("kcand", 0) or (4 * k if case.get("reorder") else 0)
        read += min(float(n), float(nq) * reranked) * dim * 4.0
        return {"bytes": read + codes * code, "flops": flops + 2.0 * (pairs + float(nq) * reranked) * dim}
    if path == "kmeans":
        k = case["k"]
        return {"bytes": 4.0 * n * dim + 8.0 * n + 8.0 * k * dim, "flops": 2.0 * n * k * dim + float(n) * dim}
    if path == "encode":
        code = dim * _BITS[case["quant"]] / 8.0
        rotation = 2.0 * n * dim * dim if case["quant"] == "rabitq" else 4.0 * n * dim
        return {"bytes": 4.0 * n * dim + n * code, "flops": rotation}
    # build: the rows, their codes, k-means on the sample of the ivf index (25 iterations), routing of every row
    code = dim * _BITS[case["quant"]] / 8.0
    flops = 2.0 * case["nlist"] * dim * (25.0 * min(n, 65536) + n) if case["index"] == "ivf" else 4.0 * n * dim
    return {"bytes": 4.0 * n * dim + n * code + 8.0 * n, "flops": flops}


def tolerance(case):
    if case["path"] == "encode":
        return "exact"  # codes are bytes, and the bounds that they are formed from are order statistics of the input
    if case["path"] == "build":
        # k-means in 32-bit sums: a row between two centroids may change its list, and with it what 16 lists return
        return {"rel": 1e-3, "max": 0.1, "differ": 0.01}
    if case["path"] == "kmeans":
        # 32-bit products; a row at the same distance of two centroids may change its label and move both means a little
        return {"rel": 1e-5, "max": 5e-3, "differ": 1e-3}
    # 32-bit sums; neighbours at equal distances may change places
    return {"rel": 1e-5, "max": 1e-4, "differ": 1e-3}
