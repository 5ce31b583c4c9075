"""Large batches on flat fp32 / sq8 stores: the matrix-core contraction pre-selects, the streaming arithmetic
decides.  Its results must equal the streaming scan's bit for bit (and therefore the checker's within the usual
tolerance), including when candidates overflow and the streaming kernel takes over."""
import time

import numpy as np
import pytest

import oracle as orc
from gpu_helpers import Store, assert_topk_close, dev, gaussian_mixture
from vsag_amd import capi

pytestmark = pytest.mark.gpu


@pytest.fixture()
def modes(lib):
    L = capi.load_library()

    def both(store, q, k, mode=1, deny=None):
        capi.check(L.vsag_amd_set_scan_contraction(-1))
        plain = store.flat_scan(q, k, deny)
        capi.check(L.vsag_amd_set_scan_contraction(mode))
        fast = store.flat_scan(q, k, deny)
        tile = capi.C.c_int()
        L.vsag_amd_last_scan_info(capi.C.byref(tile), None, None)
        capi.check(L.vsag_amd_set_scan_contraction(0))
        return plain, fast, tile.value
    yield both
    capi.check(L.vsag_amd_set_scan_contraction(0))


def same(a, b):
    return np.array_equal(a[0], b[0]) and np.array_equal(a[1].view(np.uint32), b[1].view(np.uint32))


@pytest.mark.parametrize("metric", [orc.L2, orc.IP])
@pytest.mark.parametrize("n,d,nq,k", [(40000, 128, 300, 10), (20001, 100, 129, 100), (9000, 960, 64, 10),
                                      (5000, 33, 1000, 7)])
def test_sq8_contraction_equals_streaming(lib, modes, metric, n, d, nq, k):
    rng = np.random.default_rng(n + d + k)
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    lb, diff = orc.sq_train(x, 8, metric)
    codes = orc.sq_encode(x, 8, lb, diff, metric)
    st = Store(capi.KIND_SQ8, metric, d, lb=lb, diff=diff)
    st.append(codes[:n // 3])
    st.append(codes[n // 3:])  # the per-code terms follow appends
    # mode 1: the int8 matrix cores up to 128 dimensions (256 queries per pass); mode 2: always the fp32 ones
    for mode, tile_expected in ((1, 256 if d <= 128 else 128), (2, 128)):
        plain, fast, tile = modes(st, q, k, mode)
        assert tile == tile_expected, "the contraction path did not run"
        assert same(plain, fast)
    ri, rd = orc.flat_scan_topk(orc.SQ8, metric, d, codes, q[:16], k, lb=lb, diff=diff)
    assert_topk_close(fast[0][:16], fast[1][:16], ri, rd, label="sq8 contraction")
    st.destroy()


@pytest.mark.parametrize("kind,d,nq,k,pre", [("fp32", 100, 16, 10, False), ("fp32", 100, 64, 10, False),
                                             ("fp32", 100, 127, 10, True), ("fp32", 131, 511, 1, True),
                                             ("sq8", 100, 33, 10, False), ("sq8", 100, 450, 10, True),
                                             ("sq8", 260, 17, 10, False), ("sq8", 260, 190, 10, True),
                                             ("sq8", 260, 511, 100, False)])
def test_small_batches_equal_streaming(lib, modes, kind, d, nq, k, pre):
    """Batches on both sides of the line from which fewer than 512 queries are pre-selected; a workspace without room for
    the candidate lists serves them by streaming."""
    rng = np.random.default_rng(d + nq)
    n = 70001
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    if kind == "fp32":
        st = Store(capi.KIND_FP32, orc.L2, d)
        st.append(x.view(np.uint8).reshape(n, -1))
    else:
        lb, diff = orc.sq_train(x, 8, orc.L2)
        st = Store(capi.KIND_SQ8, orc.L2, d, lb=lb, diff=diff)
        st.append(orc.sq_encode(x, 8, lb, diff, orc.L2))
    L, ws = st.lib, st.lib.vsag_amd_flat_scan_workspace_bytes
    need = ws(st.handle, nq, k)
    plain, auto, tile = modes(st, q, k, 0)
    assert same(plain, auto) and (tile >= 128) == pre
    capi.check(L.vsag_amd_store_set_scan_contraction(st.handle, -1))
    streaming = ws(st.handle, nq, k)
    capi.check(L.vsag_amd_store_set_scan_contraction(st.handle, -2))
    assert (need > streaming) == pre
    qb, ids, ds, room = dev(q), capi.DeviceBuffer(nq * k * 4), capi.DeviceBuffer(nq * k * 4), capi.DeviceBuffer(streaming)
    capi.check(L.vsag_amd_flat_scan_topk(st.handle, qb.ptr, nq, k, ids.ptr, ds.ptr, room.ptr, streaming, None))
    assert np.array_equal(ids.to_numpy(np.uint32, (nq, k)), plain[0].view(np.uint32))
    assert np.array_equal(ds.to_numpy(np.uint32, (nq, k)), plain[1].view(np.uint32))
    st.destroy()


@pytest.mark.parametrize("nq", [40, 600])
def test_workspace_between_the_routes(lib, modes, nq):
    """A workspace that has room for a streaming scan and for some, not all, of the bf16 route's records: the level-by-level
    pre-selection where that fits (600 queries), streaming otherwise, the same results."""
    rng = np.random.default_rng(nq)
    n, d, k = 82000, 40, 10
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    st = Store(capi.KIND_FP32, orc.L2, d)
    st.append(x.view(np.uint8).reshape(n, -1))
    L = st.lib
    plain, auto, tile = modes(st, q, k, 0)
    assert same(plain, auto) and tile == (64 if nq == 40 else 128)
    need = L.vsag_amd_flat_scan_workspace_bytes(st.handle, nq, k)
    capi.check(L.vsag_amd_store_set_scan_contraction(st.handle, -1))
    streaming = L.vsag_amd_flat_scan_workspace_bytes(st.handle, nq, k)
    capi.check(L.vsag_amd_store_set_scan_contraction(st.handle, -2))
    assert need > streaming
    qb, ids, ds, room = dev(q), capi.DeviceBuffer(nq * k * 4), capi.DeviceBuffer(nq * k * 4), capi.DeviceBuffer(need)
    used = capi.C.c_int()
    for size, tile_expected in ((need, tile), (need - 4096, None), (streaming + 4096, None), (streaming, 8)):
        capi.check(L.vsag_amd_flat_scan_topk(st.handle, qb.ptr, nq, k, ids.ptr, ds.ptr, room.ptr, size, None))
        L.vsag_amd_last_scan_info(capi.C.byref(used), None, None)
        if tile_expected is None:
            tile_expected = 128 if nq == 600 and size > streaming + 4096 else 8
        assert used.value == tile_expected, (size, used.value)
        assert np.array_equal(ids.to_numpy(np.uint32, (nq, k)), plain[0].view(np.uint32))
        assert np.array_equal(ds.to_numpy(np.uint32, (nq, k)), plain[1].view(np.uint32))
    st.destroy()


def _store_of(kind, metric, x, rng, train=None):
    """A store of the rows' codes, quantizer trained on the first of them, or on others."""
    d = x.shape[1]
    train = x[:20000] if train is None else train
    if kind == "fp32":
        st, codes = Store(capi.KIND_FP32, metric, d), x.view(np.uint8).reshape(len(x), -1)
    elif kind == "rabitq":
        rot, _ = np.linalg.qr(rng.standard_normal((d, d)))
        rot = rot.astype(np.float32)
        cen = orc.rabitq_train(train, rot)
        st, codes = Store(capi.KIND_RABITQ, metric, d, rot=rot, centroid=cen), orc.rabitq_encode(x, rot, cen, metric)
    elif kind.endswith("uniform"):
        bits = int(kind[2])
        lb, diff = orc.sq_train_uniform(train, bits, metric, mode=3 if bits == 4 else 1)
        st, codes = Store(capi.KINDS[kind], metric, d, bounds=[lb, diff]), orc.squ_encode(x, bits, lb, diff, metric)
    else:
        bits = int(kind[2])
        lb, diff = orc.sq_train(train, bits, metric)
        st, codes = Store(capi.KINDS[kind], metric, d, lb=lb, diff=diff), orc.sq_encode(x, bits, lb, diff, metric)
    st.append(codes)
    return st


@pytest.mark.parametrize("kind,metric,n,d,k,last_streamed", [
    ("fp32", orc.IP, 70001, 100, 10, 175), ("fp32", orc.COSINE, 70001, 64, 1, 274), ("fp32", orc.L2, 150001, 131, 100, 402),
    ("sq8", orc.IP, 150001, 100, 10, 289), ("sq8", orc.L2, 1000001, 100, 10, 31), ("sq4", orc.L2, 70001, 128, 10, 323),
    ("sq4", orc.COSINE, 150001, 128, 7, 226), ("sq4", orc.IP, 150001, 300, 10, 108), ("sq8", orc.COSINE, 100001, 200, 10, 243),
    ("sq8", orc.IP, 320001, 960, 10, 16), ("sq4", orc.COSINE, 320001, 960, 7, 15),
    ("sq8_uniform", orc.L2, 300001, 128, 10, 307), ("sq8_uniform", orc.IP, 300001, 128, 10, 460),
    ("sq4_uniform", orc.COSINE, 500001, 96, 10, 368), ("sq4_uniform", orc.L2, 300001, 128, 10, 307),
    ("rabitq", orc.L2, 2000001, 96, 200, 402), ("rabitq", orc.IP, 2500001, 96, 10, 483)])
def test_small_batches_of_every_kind_and_metric(lib, modes, kind, metric, n, d, k, last_streamed):
    """The largest batch that streams and the smallest that is pre-selected, of every kind and metric: the line lies between
    them, and both return what streaming returns."""
    rng = np.random.default_rng(n + d)
    x, means = gaussian_mixture(rng, n, d, 100, 0.05)
    q, _ = gaussian_mixture(rng, 511, d, 100, 0.05, means=means)
    st = _store_of(kind, metric, x, rng)
    for nq, pre in ((last_streamed, False), (last_streamed + 1, True)):
        plain, auto, tile = modes(st, q[:nq], k, 0)
        assert same(plain, auto), nq
        assert (tile >= 128) == pre, (nq, tile)
    st.destroy()


@pytest.mark.parametrize("kind,metric,n,d,k,streamed", [
    ("fp32", orc.L2, 81857, 64, 10, 4), ("fp32", orc.COSINE, 82000, 30, 21, 7), ("sq8", orc.L2, 81857, 100, 20, 3),
    ("sq8", orc.IP, 90001, 17, 128, 8), ("sq4", orc.COSINE, 81900, 129, 1, 3), ("sq8", orc.L2, 81857, 300, 21, 5),
    ("sq8_uniform", orc.IP, 81857, 130, 21, 8), ("sq4_uniform", orc.L2, 82001, 64, 20, 4)])
def test_smallest_batches_on_the_bf16_matrix_cores(lib, modes, kind, metric, n, d, k, streamed):
    """A handful of queries against 1280 tiles of codes: the largest batch that streams, and from the next one on the bf16
    matrix cores with 32, 64 and 128 queries per workgroup, with the streaming kernel's ids and distance bits."""
    rng = np.random.default_rng(n + d)
    x, means = gaussian_mixture(rng, n, d, 60, 0.05)
    q, _ = gaussian_mixture(rng, 129, d, 60, 0.05, means=means)
    q[1] = x[5]
    st = _store_of(kind, metric, x, rng)
    for nq in (streamed, streamed + 1, 32, 33, 64, 65, 129):
        plain, auto, tile = modes(st, q[:nq], k, 0)
        assert same(plain, auto), nq
        assert (tile >= 64) == (nq > streamed), (nq, tile)
    st.destroy()
    # one tile fewer: as before
    if n == 81857:
        st = _store_of(kind, metric, x[:n - 1], rng)
        plain, auto, tile = modes(st, q[:16], k, 0)
        assert same(plain, auto) and tile < 64
        st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("kind,n,d,nq,k", [("sq8_uniform", 30001, 130, 40, 10), ("sq8_uniform", 9000, 960, 129, 100),
                                           ("sq4_uniform", 20011, 161, 65, 1), ("sq4_uniform", 7000, 300, 5, 20),
                                           ("sq8_uniform", 82001, 33, 64, 10), ("sq4_uniform", 90000, 128, 33, 50)])
def test_uniform_codes_on_the_bf16_matrix_cores(lib, modes, kind, metric, n, d, nq, k):
    """Byte and nibble rows as one bf16 part: beyond 128 dimensions, in small batches, and under a deny mask, with the
    streaming kernel's ids and distance bits."""
    rng = np.random.default_rng(n + d)
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    q[0] = x[3]
    q[1] = -1e3
    st = _store_of(kind, metric, x, rng)
    plain, fast, tile = modes(st, q, k, 1 if d > 128 else 0)
    assert tile in (64, 128), "the bf16 pass did not run"
    assert same(plain, fast)
    deny = rng.random(n) < 0.6
    res = []
    for mode in (-1, 1):
        capi.check(st.lib.vsag_amd_store_set_scan_contraction(st.handle, mode))
        res.append(st.flat_scan(q, k, deny=deny))
    assert same(*res)
    st.destroy()


@pytest.mark.parametrize("bounds", [[0.0, 0.0], [3.0, 1e-30], [0.0, 1e-20], [-1e18, 1e19], [0.0, -2.0]])
def test_uniform_bounds_at_the_ends_of_fp32(lib, modes, bounds):
    """A rate of zero (every distance the same: the first ids), one that makes the distances denormal numbers, of which many
    are the same, one whose distances leave fp32, a negative width: what streaming returns.  Fewer codes than a query has
    room for records, so none of them streams only because its records overflow."""
    rng = np.random.default_rng(3)
    n, d, nq, k = 1500, 160, 20, 10
    x = rng.random((n, d), dtype=np.float32)
    q = rng.random((nq, d), dtype=np.float32)
    for metric in (orc.L2, orc.IP):
        codes = orc.squ_encode(x, 8, 0.0, 1.0, metric)
        st = Store(capi.KIND_SQ8_UNIFORM, metric, d, bounds=bounds)
        st.append(codes)
        plain, fast, tile = modes(st, q, k, 1)
        assert tile == 128, "the contraction path did not run"
        if metric == orc.L2 and bounds[1] == 0.0:
            assert np.all(plain[0] == np.arange(k))
        assert same(plain, fast)
        st.destroy()


@pytest.mark.parametrize("kind,bits", [("sq8", 8), ("sq4", 4)])
def test_fp16_preselection_keeps_few_candidates_under_cosine(lib, modes, kind, bits):
    """The thresholds of a cosine batch are as narrow as its distances: no query overflows its candidates (every query did,
    and the batch then took twenty times as long as streaming it; three times is the line here)."""
    rng = np.random.default_rng(12)
    n, d, nq, k = 70001, 200, 512, 10
    x, means = gaussian_mixture(rng, n, d, 70, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 70, 0.05, means=means)
    lb, diff = orc.sq_train(x, bits, orc.COSINE)
    st = Store(capi.KIND_SQ8 if bits == 8 else capi.KIND_SQ4, orc.COSINE, d, lb=lb, diff=diff)
    st.append(orc.sq_encode(x, bits, lb, diff, orc.COSINE))
    plain, auto, tile = modes(st, q, k, 0)
    assert same(plain, auto) and tile == 128
    qb, ids, ds = dev(q), capi.DeviceBuffer(nq * k * 4), capi.DeviceBuffer(nq * k * 4)
    best = {-1: 1e9, 0: 1e9}
    for _ in range(8):
        for mode in best:
            capi.check(st.lib.vsag_amd_store_set_scan_contraction(st.handle, mode))
            wsb = st.lib.vsag_amd_flat_scan_workspace_bytes(st.handle, nq, k)
            ws = capi.DeviceBuffer(wsb)
            capi.synchronize()
            t0 = time.perf_counter()
            capi.check(st.lib.vsag_amd_flat_scan_topk(st.handle, qb.ptr, nq, k, ids.ptr, ds.ptr, ws.ptr, wsb, None))
            capi.synchronize()
            best[mode] = min(best[mode], time.perf_counter() - t0)
            ws.free()
    assert best[0] < 3.0 * best[-1], best
    st.destroy()


def _times(st, q, k, rounds=8):
    """The best time of a call that streams and of one on the route the library takes, in turn."""
    nq = len(q)
    qb, ids, ds = dev(q), capi.DeviceBuffer(nq * k * 4), capi.DeviceBuffer(nq * k * 4)
    best = {-1: 1e9, 0: 1e9}
    for _ in range(rounds):
        for mode in best:
            capi.check(st.lib.vsag_amd_store_set_scan_contraction(st.handle, mode))
            wsb = st.lib.vsag_amd_flat_scan_workspace_bytes(st.handle, nq, k)
            ws = capi.DeviceBuffer(wsb)
            capi.synchronize()
            t0 = time.perf_counter()
            capi.check(st.lib.vsag_amd_flat_scan_topk(st.handle, qb.ptr, nq, k, ids.ptr, ds.ptr, ws.ptr, wsb, None))
            capi.synchronize()
            best[mode] = min(best[mode], time.perf_counter() - t0)
            ws.free()
    capi.check(st.lib.vsag_amd_store_set_scan_contraction(st.handle, -2))
    return best


@pytest.mark.parametrize("size", [1e30, 1e37])
def test_queries_that_stream_leave_no_records(lib, modes, size):
    """Queries whose distances, or products, leave fp32 stream; every code of the store was a record of theirs first (seven
    times the streaming kernel's time; three times is the line here)."""
    rng = np.random.default_rng(6)
    n, d, nq, k = 100000, 128, 8, 10
    x = rng.random((n, d), dtype=np.float32)
    q = (1 + rng.random((nq, d), dtype=np.float32)) * np.float32(size)
    st = Store(capi.KIND_FP32, orc.L2, d)
    st.append(x.view(np.uint8).reshape(n, -1))
    plain, fast, tile = modes(st, q, k, 0)
    assert tile == 64 and same(plain, fast)
    best = _times(st, q, k)
    assert best[0] < 3.0 * best[-1], best
    st.destroy()


def _in_cluster_order(rng, n, d, nq, clusters):
    """Rows stored cluster by cluster, and queries near a few of the clusters."""
    means = rng.random((clusters, d), dtype=np.float32)
    x = means[np.sort(rng.integers(0, clusters, n))] + 0.05 * rng.standard_normal((n, d)).astype(np.float32)
    q = means[rng.integers(0, clusters, nq)] + 0.05 * rng.standard_normal((nq, d)).astype(np.float32)
    return x.astype(np.float32), q.astype(np.float32)


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("kind,n,d,nq,k", [("fp32", 100001, 33, 40, 10), ("fp32", 90000, 20, 130, 100), ("sq8", 120000, 100, 9, 100),
                                           ("sq4", 100003, 140, 70, 10), ("sq8_uniform", 90001, 160, 33, 10),
                                           ("sq4_uniform", 100000, 64, 20, 20)])
def test_rows_in_the_order_of_their_clusters(lib, modes, kind, metric, n, d, nq, k):
    """The sample misses most queries' clusters, and more codes pass their thresholds than there is room for: a second pass
    with thresholds from the records, and the streaming kernel's ids and distance bits; so under masks over one run of the
    rows, and over all but a run."""
    rng = np.random.default_rng(n + d)
    x, q = _in_cluster_order(rng, n, d, nq, 70)
    st = _store_of(kind, metric, x, rng)
    plain, fast, tile = modes(st, q, k, 0)
    assert tile in (64, 128), "the bf16 pass did not run"
    assert same(plain, fast)
    run = np.zeros(n, bool)
    run[n // 3:n // 3 + n // 15] = True
    for deny in (run, ~run):
        res = []
        for mode in (-1, 0):
            capi.check(st.lib.vsag_amd_store_set_scan_contraction(st.handle, mode))
            res.append(st.flat_scan(q, k, deny=deny))
        assert same(*res)
    st.destroy()


@pytest.mark.parametrize("kind,n,d,nq,k", [("fp32", 100000, 128, 32, 10), ("sq8", 500000, 100, 32, 100),
                                           ("sq8_uniform", 200000, 256, 64, 10)])
def test_rows_in_the_order_of_their_clusters_do_not_stream(lib, modes, kind, n, d, nq, k):
    """A second pass costs less than streaming the batch (1.4 to 1.9 times as long as streaming, with both passes in front of
    it, when it streamed all the same)."""
    rng = np.random.default_rng(n + d)
    x, q = _in_cluster_order(rng, n, d, nq, 256)
    st = _store_of(kind, orc.L2, x, rng, train=x[::15])
    plain, fast, tile = modes(st, q, k, 0)
    assert tile == 64 and same(plain, fast)
    best = _times(st, q, k)
    assert best[0] < 1.1 * best[-1], best
    st.destroy()


@pytest.mark.parametrize("kind,d", [("fp32", 24), ("sq8", 32), ("sq4", 40), ("sq8_uniform", 160), ("sq4_uniform", 200)])
def test_records_that_overflow_twice_stream(lib, modes, kind, d):
    """Thousands of equal distances at the k-th: no threshold keeps the records within their room, with a mask and without."""
    rng = np.random.default_rng(d)
    n, nq, k = 90000, 20, 10
    x = rng.random((12, d), dtype=np.float32)[rng.integers(0, 12, n)]
    q = rng.random((nq, d), dtype=np.float32)
    st = _store_of(kind, orc.L2, x, rng)
    plain, fast, tile = modes(st, q, k, 0)
    assert tile == 64 and same(plain, fast)
    deny = rng.random(n) < 0.5
    res = []
    for mode in (-1, 0):
        capi.check(st.lib.vsag_amd_store_set_scan_contraction(st.handle, mode))
        res.append(st.flat_scan(q, k, deny=deny))
    assert same(*res)
    st.destroy()


@pytest.mark.parametrize("tile,chunks", [(2, -1), (8, 0), (-1, 7), (0, 7)])
def test_tuning_knobs_ask_for_the_streaming_kernel(lib, modes, tile, chunks):
    """A query tile or a number of chunks set by hand: a batch of fewer than 512 queries that would be pre-selected streams
    with them; from 512 on they do not change the route."""
    rng = np.random.default_rng(5)
    n, d, k = 70001, 100, 10
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, 512, d, 30, 0.05, means=means)
    lb, diff = orc.sq_train(x, 8, orc.L2)
    st = Store(capi.KIND_SQ8, orc.L2, d, lb=lb, diff=diff)
    st.append(orc.sq_encode(x, 8, lb, diff, orc.L2))
    plain, auto, route = modes(st, q[:450], k, 0)
    assert same(plain, auto) and route == 256
    capi.check(st.lib.vsag_amd_store_set_scan_tuning(st.handle, tile, chunks))
    plain2, tuned, route = modes(st, q[:450], k, 0)
    assert same(plain, plain2) and same(plain, tuned) and route == (tile if tile > 0 else 4)
    assert modes(st, q, k, 0)[2] == 256
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(30000, 129, 600, 10), (20000, 200, 520, 100), (12000, 960, 512, 10),
                                      (9000, 1000, 130, 7)])
def test_sq8_beyond_128_dimensions_on_the_fp16_matrix_cores(lib, modes, metric, n, d, nq, k):
    """sq8 stores of more than 128 dimensions: the code bytes and the two fp16 parts of the scaled query on
    v_mfma_f32_32x32x16_f16 (prefilter_h16.hip), rescored exactly.  Awkward queries as for the int8 planes: zeros,
    tiny and huge magnitudes, one dominant dimension, copies of stored vectors, far outside the trained range, NaN."""
    rng = np.random.default_rng(n + d + k + metric)
    x, means = gaussian_mixture(rng, n, d, 20, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 20, 0.05, means=means)
    if metric != orc.COSINE:  # no direction to normalise
        q[0] = 0.0
        q[1] = 1e-20
        q[6] = np.nan
        q[7, 3] = np.inf
    q[2] *= 1e6
    q[3] *= 1e-6
    q[4] = 0.0
    q[4, d // 2] = 1e4
    q[5] = 1e-30
    q[5, 1] = 3e37 if metric != orc.COSINE else 3.0
    q[8:40] = x[8:40]
    q[40:60] = -q[40:60]
    q[60:80] += 100.0
    lb, diff = orc.sq_train(x, 8, metric)
    codes = orc.sq_encode(x, 8, lb, diff, metric)
    st = Store(capi.KIND_SQ8, metric, d, lb=lb, diff=diff)
    st.append(codes[:n // 2])
    st.append(codes[n // 2:])
    plain, fast, tile = modes(st, q, k, 1)
    assert tile == 128, "the contraction path did not run"
    assert same(plain, fast)
    plain, fp32, tile = modes(st, q, k, 2)  # the fp32 matrix cores: the same again
    assert tile == 128 and same(plain, fp32)
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(30000, 160, 600, 10), (12000, 960, 512, 10), (9000, 1000, 130, 100)])
def test_sq4_beyond_128_dimensions_on_the_fp16_matrix_cores(lib, modes, metric, n, d, nq, k):
    """sq4 stores of more than 128 dimensions take the fp16 pass as well (the nibbles are exact in fp16), in mode 2 too:
    sq4 has no route on the fp32 matrix cores."""
    rng = np.random.default_rng(n + d + k + metric)
    x, means = gaussian_mixture(rng, n, d, 20, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 20, 0.05, means=means)
    if metric != orc.COSINE:
        q[0] = 0.0
        q[1] = 1e-20
        q[6] = np.nan
    q[2] *= 1e6
    q[3] *= 1e-6
    q[4] = 0.0
    q[4, d // 2] = 1e4
    q[8:40] = x[8:40]
    q[60:80] += 100.0
    lb, diff = orc.sq_train(x, 4, metric)
    codes = orc.sq_encode(x, 4, lb, diff, metric)
    st = Store(capi.KIND_SQ4, metric, d, lb=lb, diff=diff)
    st.append(codes[:n // 2])
    st.append(codes[n // 2:])
    for mode in (1, 2):
        plain, fast, tile = modes(st, q, k, mode)
        assert tile == 128, "the contraction path did not run"
        assert same(plain, fast)
    qs, om = q[8:24], metric
    if metric == orc.COSINE:  # inner product of the unit query with the codes of the unit rows
        qs, om = (qs / np.linalg.norm(qs, axis=1, keepdims=True)).astype(np.float32), orc.IP
    ri, rd = orc.flat_scan_topk(orc.SQ4, om, d, codes, qs, k, lb=lb, diff=diff)
    assert_topk_close(fast[0][8:24], fast[1][8:24], ri, rd, label="sq4 beyond 128 dimensions")
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("d", [16, 100, 128])
def test_sq8_int8_planes_hold_for_awkward_queries(lib, modes, metric, d):
    """Queries the two int8 planes represent badly or trivially: one dominant dimension, tiny and huge magnitudes,
    all zeros, copies of stored vectors, far outside the trained range."""
    rng = np.random.default_rng(1000 + d + metric)
    n, nq, k = 30000, 320, 10
    x, means = gaussian_mixture(rng, n, d, 20, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 20, 0.05, means=means)
    if metric != orc.COSINE:  # no direction to normalise
        q[0] = 0.0
        q[1] = 1e-20
    q[2] *= 1e6
    q[3] *= 1e-6
    q[4] = 0.0
    q[4, d // 2] = 1e4
    q[5:40] = x[5:40]          # duplicates of stored vectors
    q[40:60] = -q[40:60]
    q[60:80] += 100.0          # far outside [lb, lb + diff]
    q[80, :] = np.where(np.arange(d) % 2 == 0, 1e-3, 1e3)
    lb, diff = orc.sq_train(x, 8, metric)
    codes = orc.sq_encode(x, 8, lb, diff, metric)
    st = Store(capi.KIND_SQ8, metric, d, lb=lb, diff=diff)
    st.append(codes)
    plain, fast, tile = modes(st, q, k)
    assert tile == 256
    assert same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(40000, 128, 300, 10), (20001, 100, 129, 100), (9000, 31, 640, 7),
                                      (30000, 16, 320, 10)])
def test_sq4_contraction_equals_streaming(lib, modes, metric, n, d, nq, k):
    """sq4 (a range per dimension, two 4-bit values per byte): the two int8 planes of a query against the nibbles as
    they are; awkward queries among the ordinary ones."""
    rng = np.random.default_rng(n + d + k + metric)
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    if metric != orc.COSINE:
        q[0] = 0.0
        q[1] = 1e-20
    q[2] *= 1e6
    q[3] *= 1e-6
    q[5:40] = x[5:40]
    q[60:80] += 100.0
    lb, diff = orc.sq_train(x, 4, metric)
    codes = orc.sq_encode(x, 4, lb, diff, metric)
    st = Store(capi.KIND_SQ4, metric, d, lb=lb, diff=diff)
    st.append(codes[:n // 3])
    st.append(codes[n // 3:])  # the per-code terms follow appends
    plain, fast, tile = modes(st, q, k)
    assert tile == 256, "the contraction path did not run"
    assert same(plain, fast)
    # asking for the fp32 matrix cores finds no route for this kind and the int8 one serves
    plain, fast, tile = modes(st, q, k, 2)
    assert tile == 256 and same(plain, fast)
    om, oq = (orc.IP, (q[100:116] / np.linalg.norm(q[100:116], axis=1, keepdims=True)).astype(np.float32)) \
        if metric == orc.COSINE else (metric, q[100:116])
    ri, rd = orc.flat_scan_topk(orc.SQ4, om, d, codes, oq, k, lb=lb, diff=diff)
    assert_topk_close(fast[0][100:116], fast[1][100:116], ri, rd, atol=4e-6, label="sq4 contraction")
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(30000, 128, 200, 10), (7000, 65, 77, 32)])
def test_fp32_contraction_equals_streaming(lib, modes, metric, n, d, nq, k):
    rng = np.random.default_rng(n + d + k + metric)
    x = rng.random((n, d), dtype=np.float32)
    q = rng.random((nq, d), dtype=np.float32)
    x[5] = q[3]  # an exact duplicate of a query: distance 0 must come out as 0
    st = Store(capi.KIND_FP32, metric, d)
    st.append(x.view(np.uint8).reshape(n, 4 * d))
    plain, fast, tile = modes(st, q, k)
    assert tile == 128
    assert same(plain, fast)
    if metric == orc.L2:
        assert fast[0][3, 0] == 5 and fast[1][3, 0] == 0.0
    st.destroy()


@pytest.mark.parametrize("kind,d", [("sq8_uniform", 8192), ("sq8_uniform", 8193), ("sq4_uniform", 8192), ("sq4_uniform", 8200)])
def test_longest_uniform_codes(lib, modes, kind, d):
    """Up to 8192 dimensions on the bf16 matrix cores, beyond by streaming."""
    rng = np.random.default_rng(d)
    n, nq, k = 700, 9, 5
    x = rng.random((n, d), dtype=np.float32)
    st = _store_of(kind, orc.L2, x, rng)
    plain, fast, tile = modes(st, x[:nq] + np.float32(0.1), k, 1)
    assert (tile == 128) == (d <= 8192) and same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(1500, 17, 1, 1), (2049, 32, 31, 5), (4097, 36, 33, 10), (5003, 130, 64, 10),
                                      (3001, 64, 65, 20), (6000, 260, 129, 3)])
def test_fp32_on_the_bf16_matrix_cores(lib, modes, metric, n, d, nq, k):
    """Two bf16 values per operand select, the streaming arithmetic decides: 32, 64 and 128 queries per workgroup, code
    tiles and stages with a remainder, rows of very different lengths and copies of stored rows among the queries."""
    rng = np.random.default_rng(n + d)
    x, means = gaussian_mixture(rng, n, d, 20, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 20, 0.05, means=means)
    x[::7] *= np.float32(1e3)
    x[1::7] *= np.float32(1e-6)
    x[2::70] = 0
    q[::3] = x[rng.integers(0, n, len(q[::3]))]
    for scale in (1.0, 1e-18, 1e12):
        st = Store(capi.KIND_FP32, metric, d)
        st.append((x * np.float32(scale)).view(np.uint8).reshape(n, -1))
        plain, fast, tile = modes(st, q * np.float32(scale), k)
        assert tile == 128, "the contraction path did not run"
        assert same(plain, fast)
        st.destroy()


def _near_one(units):
    return np.float32(1 + units * 2.0 ** -16)


@pytest.mark.parametrize("metric", [orc.L2, orc.IP])
@pytest.mark.parametrize("d", [16, 20, 48, 64, 128])
def test_rows_that_two_bf16_values_miss_by_as_much_as_they_can(lib, modes, metric, d):
    """1 + 254.5 units of 2^-16 loses nearly 2^-17 of itself and has a low part of nearly 2^-8, and so, with the other sign,
    has what lies as far below 1 + 2^-7.  The best row's products come out too small in every dimension, the others' too
    large: the best must still be among the records."""
    n, nq = 1500, 40
    x = np.full((n, d), _near_one(512 - 254.5), np.float32)
    q = np.full((nq, d), _near_one(254), np.float32)
    x[700] = _near_one(254.5)
    if metric == orc.IP:
        q[:, -1] = 1
        x[:, -1] = 0
        lead = (x[0, :-1].astype(np.float64) - x[700, :-1]) @ q[0, :-1].astype(np.float64)
        x[700, -1] = np.float16(1.05 * lead)  # (no more bits than a bf16 value's two parts hold)
    st = Store(capi.KIND_FP32, metric, d)
    st.append(x.view(np.uint8).reshape(n, -1))
    plain, fast, tile = modes(st, q, 1)
    assert tile == 128, "the contraction path did not run"
    assert np.all(plain[0] == 700) and same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("kind", ["fp32", "sq8"])
def test_many_short_tiles_per_workgroup(lib, modes, kind):
    """100000 x 128 against 1000 queries: every workgroup walks many code tiles with a short contraction each, so
    the epilogue of one tile runs next to the start of the following one."""
    rng = np.random.default_rng(77)
    n, d, nq, k = 100000, 128, 1000, 10
    x = rng.standard_normal((n, d)).astype(np.float32)
    q = rng.standard_normal((nq, d)).astype(np.float32)
    if kind == "fp32":
        st = Store(capi.KIND_FP32, orc.L2, d)
        st.append(x.view(np.uint8).reshape(n, 4 * d))
    else:
        lb, diff = orc.sq_train(x, 8, orc.L2)
        st = Store(capi.KIND_SQ8, orc.L2, d, lb=lb, diff=diff)
        st.append(orc.sq_encode(x, 8, lb, diff, orc.L2))
    for _ in range(3):
        plain, fast, tile = modes(st, q, k)
        assert tile == (128 if kind == "fp32" else 256)
        assert same(plain, fast)
    st.destroy()


def test_contraction_overflow_falls_back_to_streaming(lib, modes):
    """Thousands of equal distances per query: the candidate buffers overflow, the streaming kernel serves the query."""
    rng = np.random.default_rng(8)
    n, d, nq, k = 30000, 32, 150, 10
    base = rng.integers(0, 256, (40, d), dtype=np.uint8)
    codes = base[rng.integers(0, 40, n)]  # 40 distinct codes, 750 copies each
    lb, diff = np.zeros(d, np.float32), np.ones(d, np.float32)
    q = rng.random((nq, d), dtype=np.float32)
    st = Store(capi.KIND_SQ8, orc.L2, d, lb=lb, diff=diff)
    st.append(codes)
    for mode, tile_expected in ((1, 256), (2, 128)):
        plain, fast, tile = modes(st, q, k, mode)
        assert tile == tile_expected
        assert same(plain, fast)
    ri, rd = orc.flat_scan_topk(orc.SQ8, orc.L2, d, codes, q[:8], k, lb=lb, diff=diff)
    # which of the equal distances the checker keeps is its heap's business; the distances must agree
    np.testing.assert_allclose(fast[1][:8], rd, rtol=1e-5)
    assert np.all(np.diff(fast[0], axis=1)[np.diff(fast[1], axis=1) == 0] > 0), "ties are ordered by id"
    st.destroy()


def _rabitq_store(rng, n, d, metric, centered=True):
    x = rng.standard_normal((n, d)).astype(np.float32)
    if centered:
        x /= np.linalg.norm(x, axis=1, keepdims=True)
    else:
        x = x * 0.1 + 1.0  # far from the origin: large raw norms, small residuals
    g = rng.standard_normal((d, d))
    rot, r = np.linalg.qr(g)
    rot = (rot * np.sign(np.diag(r))).astype(np.float32)
    cen = orc.rabitq_train(x, rot)
    st = Store(capi.KIND_RABITQ, metric, d, rot=rot, centroid=cen)
    st.append(orc.rabitq_encode(x, rot, cen, metric))
    return x, st


@pytest.mark.parametrize("metric", [orc.L2, orc.IP])
@pytest.mark.parametrize("n,d,nq,k,centered", [(30000, 128, 300, 10, True), (20000, 768, 260, 200, True),
                                               (9000, 100, 129, 50, False), (70000, 256, 700, 100, True),
                                               (12000, 1024, 150, 20, True)])
def test_rabitq_contraction_equals_streaming(lib, modes, metric, n, d, nq, k, centered):
    """1-bit codes against 4-bit queries on the int8 matrix cores: the estimator is affine in the integer inner
    product, so the pre-selection is a threshold on it; the rescored result must equal the streaming scan's bits."""
    rng = np.random.default_rng(n + d + k + metric)
    x, st = _rabitq_store(rng, n, d, metric, centered)
    q = rng.standard_normal((nq, d)).astype(np.float32)
    if centered:
        q /= np.linalg.norm(q, axis=1, keepdims=True)
    else:
        q = q * 0.1 + 1.0
    q[3] = x[17]                 # a stored vector
    q[4] = 0.0                   # no direction at all
    q[5] = 1.0                   # constant coordinates before the rotation
    plain, fast, tile = modes(st, q, k)
    assert tile == 128, "the contraction path did not run"
    assert same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP])
def test_rabitq_store_of_many_appends_and_codes_outside_the_pass(lib, modes, metric):
    """The store keeps its code bits and per-code constants once more for the matrix cores, renewed by every append
    (also of the tile an earlier append left part full).  Codes the pre-selection's derivation does not cover -- a zero
    norm, a non-positive error factor, a sum field that is not the number of set bits -- must still come out as the
    streaming scan has them."""
    n, d, nq, k = 21000, 200, 200, 30
    rng = np.random.default_rng(77 + metric)
    x = rng.standard_normal((n, d)).astype(np.float32)
    x /= np.linalg.norm(x, axis=1, keepdims=True)
    g = rng.standard_normal((d, d))
    rot, r = np.linalg.qr(g)
    rot = (rot * np.sign(np.diag(r))).astype(np.float32)
    cen = orc.rabitq_train(x, rot)
    x[5] = cen @ rot                    # the centroid itself (rotated back): a zero norm after centring
    codes = orc.rabitq_encode(x, rot, cen, metric)
    tail = codes[:, -(12 if metric == orc.L2 else 16):].view(np.float32)  # norm, error factor, sum[, raw norm]
    tail[70, 1] = -0.5                  # a negative error factor
    tail[131, 2] += 3.0                 # a sum field that is not the set bits
    tail[4000, 0] = 0.0                 # a zero norm
    tail[20999, 2] = 0.0
    st = Store(capi.KIND_RABITQ, metric, d, rot=rot, centroid=cen)
    at = 0
    for step in (1, 63, 64, 65, 1000, 37, 12000, 3, n):   # ragged: tiles left part full and filled later
        end = min(n, at + step)
        if end > at:
            st.append(codes[at:end])
        at = end
    assert at == n
    q = rng.standard_normal((nq, d)).astype(np.float32)
    q /= np.linalg.norm(q, axis=1, keepdims=True)
    plain, fast, tile = modes(st, q, k)
    assert tile == 128, "the contraction path did not run"
    assert same(plain, fast)
    whole = Store(capi.KIND_RABITQ, metric, d, rot=rot, centroid=cen)
    whole.append(codes)
    assert same(plain, whole.flat_scan(q, k))
    whole.destroy()
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(40000, 128, 300, 10), (20001, 100, 129, 100), (5000, 33, 1000, 7),
                                      (70000, 64, 600, 1)])
def test_sq8_uniform_contraction_equals_streaming(lib, modes, metric, n, d, nq, k):
    """sq8_uniform: code and query are both rows of bytes, the product is an integer the int8 matrix cores deliver
    exactly; distances are integers scaled once, so ties abound and must come out in id order on both routes."""
    rng = np.random.default_rng(n + d + k + 3 * metric)
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    q[3] = x[17]          # a stored vector
    q[4] = 0.0            # clamps to the lower bound everywhere
    q[5] = 10.0           # clamps to the upper bound everywhere
    lb, diff = orc.sq_train_uniform(x, 8, metric, mode=1)
    codes = orc.squ_encode(x, 8, lb, diff, metric)
    st = Store(capi.KIND_SQ8_UNIFORM, metric, d, bounds=[lb, diff])
    st.append(codes[:n // 3])
    st.append(codes[n // 3:])
    plain, fast, tile = modes(st, q, k)
    assert tile == 256, "the int8 route did not run"
    assert same(plain, fast)
    plain, fast, tile = modes(st, q, k, mode=2)  # no fp32 route for this kind: still the int8 matrix cores
    assert tile == 256 and same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("metric", [orc.L2, orc.IP, orc.COSINE])
@pytest.mark.parametrize("n,d,nq,k", [(40000, 128, 300, 10), (20001, 100, 129, 100), (5000, 33, 1000, 7),
                                      (70000, 64, 600, 1)])
def test_sq4_uniform_contraction_equals_streaming(lib, modes, metric, n, d, nq, k):
    """sq4_uniform: two 4-bit values per byte, split into low- and high-nibble granules when staged."""
    rng = np.random.default_rng(n + d + k + 5 * metric)
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    q[3] = x[17]
    q[4] = 0.0
    q[5] = 10.0
    lb, diff = orc.sq_train_uniform(x, 4, metric, mode=3)
    codes = orc.squ_encode(x, 4, lb, diff, metric)
    st = Store(capi.KIND_SQ4_UNIFORM, metric, d, bounds=[lb, diff])
    st.append(codes[:n // 3])
    st.append(codes[n // 3:])
    plain, fast, tile = modes(st, q, k)
    assert tile == 256, "the int8 route did not run"
    assert same(plain, fast)
    st.destroy()


def test_settings_of_one_store_leave_the_others_alone(lib):
    """vsag_amd_store_set_scan_contraction / _set_scan_tuning: a store's own settings go before the process-wide ones
    and do not touch searches on another store."""
    L = capi.load_library()
    n, d, nq, k = 70000, 64, 600, 10
    rng = np.random.default_rng(21)
    x, means = gaussian_mixture(rng, n, d, 30, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 30, 0.05, means=means)
    lb, diff = orc.sq_train(x, 8, orc.L2)
    codes = orc.sq_encode(x, 8, lb, diff, orc.L2)
    a = Store(capi.KIND_SQ8, orc.L2, d, lb=lb, diff=diff)
    b = Store(capi.KIND_SQ8, orc.L2, d, lb=lb, diff=diff)
    a.append(codes)
    b.append(codes)
    tile = capi.C.c_int()

    def last_tile():
        L.vsag_amd_last_scan_info(capi.C.byref(tile), None, None)
        return tile.value
    capi.check(L.vsag_amd_store_set_scan_contraction(a.handle, -1))
    ws_a, ws_b = (int(L.vsag_amd_flat_scan_workspace_bytes(s.handle, nq, k)) for s in (a, b))
    assert ws_a < ws_b, "the streaming scan needs no candidate buffers"
    ra = a.flat_scan(q, k)
    assert last_tile() == 4, "store a was told to stream"
    rb = b.flat_scan(q, k)
    assert last_tile() == 256, "store b follows the process-wide default"
    assert same(ra, rb)
    capi.check(L.vsag_amd_store_set_scan_tuning(a.handle, 2, -1))
    ra2 = a.flat_scan(q, k)
    assert last_tile() == 2
    assert same(ra, ra2)
    b.flat_scan(q[:8], k)
    assert last_tile() == 4, "store b keeps the default tile"
    # back to the process-wide settings; a bad mode is refused
    capi.check(L.vsag_amd_store_set_scan_contraction(a.handle, -2))
    capi.check(L.vsag_amd_store_set_scan_tuning(a.handle, -1, -1))
    a.flat_scan(q, k)
    assert last_tile() == 256
    assert L.vsag_amd_store_set_scan_contraction(a.handle, 3) == capi.INVALID_ARGUMENT
    assert L.vsag_amd_store_set_scan_tuning(a.handle, 3, 0) == capi.INVALID_ARGUMENT
    a.destroy()
    b.destroy()


@pytest.mark.parametrize("kind,metric,d", [("fp32", orc.L2, 127), ("fp32", orc.COSINE, 129), ("fp32", orc.IP, 261),
                                           ("sq8", orc.L2, 513), ("sq8", orc.IP, 1030), ("sq4", orc.L2, 1030),
                                           ("sq8_uniform", orc.L2, 513), ("sq4_uniform", orc.IP, 1030)])
@pytest.mark.parametrize("k", [1, 31, 33, 128])
def test_rescoring_at_the_edges_of_its_pieces(lib, modes, kind, metric, d, k):
    """Candidates on both sides of 32 and 64, rows a granule short of and beyond the 32 or 64 that are in LDS at a time; rows
    that are copies of each other, so that more candidates than k are equal to the last bit.  (Mode 1 sends sq8 and sq4 stores
    through this pass under a mask.)"""
    rng = np.random.default_rng(d + k)
    n, nq = 2100, 17
    x, means = gaussian_mixture(rng, n, d, 12, 0.05)
    x[100:260] = x[99]
    q, _ = gaussian_mixture(rng, nq, d, 12, 0.05, means=means)
    q[0] = x[99]
    st = _store_of(kind, metric, x, rng)
    if kind in ("sq8", "sq4"):
        plain, fast, _ = modes(st, q, k, 1)
        assert same(plain, fast)
    deny = rng.random(n) < 0.03 if kind in ("sq8", "sq4") else None
    plain, fast, tile = modes(st, q, k, 1, deny)
    assert tile in (64, 128), "the bf16 pass did not run"
    assert same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("kind,metric", [("fp32", orc.L2), ("fp32", orc.IP), ("sq8_uniform", orc.L2), ("sq4_uniform", orc.IP)])
def test_either_form_of_rescoring(lib, modes, kind, metric):
    """512 queries have a workgroup each, 513 a wave."""
    rng = np.random.default_rng(11)
    n, d, k = 3000, 200, 33
    x, means = gaussian_mixture(rng, n, d, 15, 0.05)
    x[500:620] = x[499]
    q, _ = gaussian_mixture(rng, 513, d, 15, 0.05, means=means)
    q[7] = x[499]
    st = _store_of(kind, metric, x, rng)
    for nq in (512, 513):
        plain, fast, tile = modes(st, q[:nq], k, 1)
        assert tile in (64, 128), "the bf16 pass did not run"
        assert same(plain, fast)
    st.destroy()


@pytest.mark.parametrize("kind,metric,d", [("fp32", orc.L2, 100), ("fp32", orc.IP, 37), ("sq8", orc.L2, 100),
                                           ("sq4", orc.IP, 132), ("sq8_uniform", orc.L2, 200), ("sq4_uniform", orc.IP, 200)])
@pytest.mark.parametrize("nq", [33, 513])
def test_many_neighbours_behind_the_bf16_pass(lib, modes, kind, metric, d, nq):
    """Beyond 128 neighbours a query has room for more records than a workgroup of the rescoring holds in registers; mode 1 asks
    for the bf16 pass all the same (of sq8 and sq4 stores under a mask)."""
    rng = np.random.default_rng(d + nq)
    n = 9000
    x, means = gaussian_mixture(rng, n, d, 12, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 12, 0.05, means=means)
    st = _store_of(kind, metric, x, rng)
    deny = rng.random(n) < 0.1 if kind in ("sq8", "sq4") else None
    for k in (129, 256, 1024):
        plain, fast, tile = modes(st, q, k, 1, deny)
        assert tile in (64, 128), "the bf16 pass did not run"
        assert same(plain, fast), k
    st.destroy()


@pytest.mark.parametrize("kind,metric,d,mode,tiles", [("fp32", orc.L2, 100, 1, (64, 128)), ("fp32", orc.IP, 60, 2, (128,)),
                                                      ("sq8", orc.L2, 100, 1, (256,)), ("sq4_uniform", orc.IP, 64, 1, (256,))])
def test_odd_numbers_of_neighbours(lib, modes, kind, metric, d, mode, tiles):
    """The keys that the rescoring ranks stand behind the k kept ones, with an odd k on 8 bytes only (up to 32 and from 129 to 160
    neighbours): each route that ranks them, with a wave per query."""
    rng = np.random.default_rng(d)
    n, nq = 6000, 513
    x, means = gaussian_mixture(rng, n, d, 60, 0.05)
    q, _ = gaussian_mixture(rng, nq, d, 60, 0.05, means=means)
    st = _store_of(kind, metric, x, rng)
    for k in (1, 2, 5, 21, 31, 32, 33, 129, 131, 160):
        plain, fast, tile = modes(st, q, k, mode)
        assert tile in tiles, "the matrix cores did not run"
        assert same(plain, fast), k
    st.destroy()
