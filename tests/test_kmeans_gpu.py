"""k-means on the device against the CPU checker and against an fp64 brute force."""
import ctypes as C
import time

import numpy as np
import pytest

import oracle as orc
from gpu_helpers import dev, gaussian_mixture
from vsag_amd import capi

pytestmark = pytest.mark.gpu


def gpu_assign(x, cent):
    L = capi.load_library()
    n, d = x.shape
    k = cent.shape[0]
    xb, cb = dev(x), dev(cent)
    labels, mind, loss = capi.DeviceBuffer(n * 4), capi.DeviceBuffer(n * 4), capi.DeviceBuffer(8)
    wsb = L.vsag_amd_kmeans_assign_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(wsb)
    capi.check(L.vsag_amd_kmeans_assign(xb.ptr, n, d, cb.ptr, k, labels.ptr, mind.ptr, loss.ptr, ws.ptr, wsb, None))
    return labels.to_numpy(np.int32, (n,)), mind.to_numpy(np.float32, (n,)), float(loss.to_numpy(np.float64, (1,))[0])


def check_assignment(x, cent, labels, mind, rel=1e-5):
    """labels must be the exact argmin except where the runner-up is within rel of the winner."""
    x64, c64 = x.astype(np.float64), cent.astype(np.float64)
    d2 = (c64 ** 2).sum(1)[None, :] - 2.0 * x64 @ c64.T
    best = d2.argmin(1)
    scale = (x64 ** 2).sum(1) + np.abs(d2.min(1))
    chosen = d2[np.arange(len(x)), labels]
    wrong = labels != best
    gap = chosen - d2.min(1)
    assert np.all(gap[wrong] <= rel * scale[wrong]), "assignment differs outside the near-tie band: %d rows" % int(
        (gap > rel * scale).sum())
    assert np.allclose(mind, d2.min(1), rtol=1e-4, atol=1e-4 * scale.max())
    return int(wrong.sum())


@pytest.mark.parametrize("n,d,k", [(3000, 128, 100), (1000, 960, 257), (129, 7, 3), (5000, 33, 1000), (64, 16, 64),
                                   (3000, 100, 100), (2000, 104, 500), (1500, 12, 40)])
def test_assign_matches_bruteforce_and_oracle(lib, n, d, k):
    rng = np.random.default_rng(n + d + k)
    x, _ = gaussian_mixture(rng, n, d, max(2, k // 4), 0.2, uniform_means=False)
    cent = x[rng.choice(n, k, replace=False)].copy()
    labels, mind, loss = gpu_assign(x, cent)
    assert labels.min() >= 0 and labels.max() < k
    check_assignment(x, cent, labels, mind)
    olabels, omind, oloss = orc.kmeans_assign(x, cent)
    agree = (labels == olabels).mean()
    assert agree > 0.999, agree
    assert abs(loss - oloss) <= 1e-4 * abs(oloss) + 1e-6


@pytest.mark.parametrize("d,k", [(4, 1), (20, 100), (36, 128), (12, 129), (60, 384)])
def test_assign_on_both_sides_of_two_workgroups_a_compute_unit(lib, d, k):
    """As many workgroups as the chip holds at once and one row of tiles more: labels and distances of a few thousand rows at a
    time, bit for bit."""
    rng = np.random.default_rng(d + k)
    tiles = -(-k // 128)
    cus = 256
    n = 2 * cus // tiles * 256
    x = rng.standard_normal((n + 1, d)).astype(np.float32)
    cent = rng.standard_normal((k, d)).astype(np.float32)
    for rows in (n, n + 1):
        labels, dist, _ = gpu_assign(x[:rows], cent)
        for a in list(range(0, rows, 40000)) + [rows - 1]:
            part, pdist, _ = gpu_assign(x[a:min(a + 3000, rows)], cent)
            assert np.array_equal(labels[a:a + 3000], part)
            assert np.array_equal(dist[a:a + 3000].view(np.uint32), pdist.view(np.uint32))


def test_first_minimum_wins_ties(lib):
    # duplicated centroids: std::min_element keeps the first of equal minima
    rng = np.random.default_rng(3)
    x = rng.standard_normal((500, 32)).astype(np.float32)
    base = rng.standard_normal((40, 32)).astype(np.float32)
    cent = np.concatenate([base, base, base]).astype(np.float32)
    labels, _, _ = gpu_assign(x, cent)
    assert labels.max() < 40


@pytest.mark.parametrize("n,d,k", [(4000, 64, 50), (700, 960, 9)])
def test_update_matches_oracle(lib, n, d, k):
    L = lib.load_library()
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((n, d)).astype(np.float32)
    labels = rng.integers(0, k, n).astype(np.int32)
    labels[labels == 3] = 4  # cluster 3 is empty
    cent0 = rng.standard_normal((k, d)).astype(np.float32)
    xb, lb, cb = dev(x), dev(labels), dev(cent0)
    counts = capi.DeviceBuffer(k * 4)
    wsb = L.vsag_amd_kmeans_update_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(wsb)
    capi.check(L.vsag_amd_kmeans_update(xb.ptr, lb.ptr, n, d, k, cb.ptr, counts.ptr, ws.ptr, wsb, None))
    cent = cb.to_numpy(np.float32, (k, d))
    cnt = counts.to_numpy(np.int32, (k,))
    rcent, rcnt = orc.kmeans_update(x, labels, cent0)
    assert np.array_equal(cnt, rcnt) and cnt[3] == 0
    assert np.array_equal(cent[3], cent0[3])  # empty cluster untouched
    assert np.allclose(cent, rcent, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("d", [1, 3, 5, 20, 64, 65, 68, 128, 131])
def test_update_sums_in_row_order(lib, d):
    """Clusters around the kernel's stages of 64 rows (and empty ones): the means are the sequential fp32 sums, bit for bit."""
    L = lib.load_library()
    rng = np.random.default_rng(d)
    sizes = np.concatenate([[0, 1, 2, 15, 17, 63, 64, 65, 127, 128, 129, 191, 192, 193, 1000, 0, 16],
                            rng.integers(1, 40, 600)])
    k, n = len(sizes), int(sizes.sum())
    labels = rng.permutation(np.repeat(np.arange(k), sizes)).astype(np.int32)
    x = rng.standard_normal((n, d)).astype(np.float32)
    cent0 = rng.standard_normal((k, d)).astype(np.float32)
    xb, lb, cb, counts = dev(x), dev(labels), dev(cent0), capi.DeviceBuffer(k * 4)
    wsb = L.vsag_amd_kmeans_update_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(wsb)
    capi.check(L.vsag_amd_kmeans_update(xb.ptr, lb.ptr, n, d, k, cb.ptr, counts.ptr, ws.ptr, wsb, None))
    want = cent0.copy()
    for j in range(k):
        if sizes[j]:
            sums = np.cumsum(x[labels == j], axis=0, dtype=np.float32)[-1]
            want[j] = sums * (np.float32(1) / np.float32(sizes[j]))
    assert np.array_equal(counts.to_numpy(np.int32, (k,)), sizes)
    assert np.array_equal(cb.to_numpy(np.float32, (k, d)), want)


def test_run_matches_oracle_and_reduces_loss(lib):
    L = lib.load_library()
    rng = np.random.default_rng(11)
    n, d, k, iters = 6000, 48, 64, 6
    x, _ = gaussian_mixture(rng, n, d, 64, 0.2, uniform_means=False)
    cent0 = x[rng.choice(n, k, replace=False)].copy()
    xb, cb = dev(x), dev(cent0)
    labels = capi.DeviceBuffer(n * 4)
    loss = C.c_double()
    wsb = L.vsag_amd_kmeans_run_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(wsb)
    capi.check(L.vsag_amd_kmeans_run(xb.ptr, n, d, cb.ptr, k, iters, 7, labels.ptr, C.byref(loss), ws.ptr, wsb, None))
    cent = cb.to_numpy(np.float32, (k, d))
    rcent, rlabels, rloss = orc.kmeans_run(x, cent0, iters, 7)
    _, _, loss0 = orc.kmeans_assign(x, cent0)
    assert loss.value < loss0
    assert abs(loss.value - rloss) <= 1e-3 * abs(rloss)
    assert (labels.to_numpy(np.int32, (n,)) == rlabels).mean() > 0.99
    assert np.allclose(cent, rcent, rtol=1e-3, atol=1e-3)


def test_kmeans_argument_errors(lib):
    L = lib.load_library()
    x = dev(np.zeros((4, 4), np.float32))
    rc = L.vsag_amd_kmeans_run(x.ptr, 4, 4, x.ptr, 8, 1, 0, x.ptr, None, None, 0, None)
    assert rc == capi.INVALID_ARGUMENT and b"k cannot be larger than count" in L.vsag_amd_last_error()
    rc = L.vsag_amd_kmeans_assign(x.ptr, 4, 4, x.ptr, 0, x.ptr, None, None, None, 0, None)
    assert rc == capi.INVALID_ARGUMENT and b"k must be positive" in L.vsag_amd_last_error()


def gpu_init_pp(x, k, first, draws):
    L = capi.load_library()
    n, d = x.shape
    xb = dev(x)
    cent, picks = capi.DeviceBuffer(k * d * 4), capi.DeviceBuffer(k * 8)
    wsb = L.vsag_amd_kmeans_init_plus_plus_workspace_bytes(n)
    ws = capi.DeviceBuffer(wsb)
    draws = np.ascontiguousarray(draws, np.float64)
    capi.check(L.vsag_amd_kmeans_init_plus_plus(xb.ptr, n, d, k, first, draws.ctypes.data, cent.ptr, picks.ptr, ws.ptr,
                                                wsb, None))
    capi.synchronize()
    out = cent.to_numpy(np.float32, (k, d)), picks.to_numpy(np.uint64, (k,))
    for b in (xb, cent, picks, ws):
        b.free()
    return out


@pytest.mark.parametrize("n,d,k", [(5000, 128, 64), (777, 7, 100), (20000, 65, 33), (64, 960, 64), (130, 16, 130)])
def test_plus_plus_seeding_matches_oracle(lib, n, d, k):
    """k-means++ seeding (kmeans_cluster.cpp:383-435) with the same draws as the checker: the same rows, except where a
    threshold falls within the rounding of the (differently associated) double sums of a boundary."""
    rng = np.random.default_rng(n + d + k)
    x, _ = gaussian_mixture(rng, n, d, max(2, k // 4), 0.2, uniform_means=False)
    draws = rng.random(k - 1)
    first = int(rng.integers(n))
    cent, picks = gpu_init_pp(x, k, first, draws)
    rcent, rpicks = orc.kmeans_init_pp(x, k, first, draws)
    assert np.array_equal(picks, rpicks), np.nonzero(picks != rpicks)[0][:5]
    assert np.array_equal(cent, rcent)
    assert len(set(picks.tolist())) == k


def test_plus_plus_seeding_on_coincident_rows(lib):
    rng = np.random.default_rng(4)
    y = np.repeat(rng.standard_normal((3, 20)).astype(np.float32), 50, axis=0)
    draws = np.array([0.5, 0.99, 0.0, 0.5, 0.999])
    cent, picks = gpu_init_pp(y, 6, 0, draws)
    _, rpicks = orc.kmeans_init_pp(y, 6, 0, draws)
    assert np.array_equal(picks, rpicks) and list(picks[3:]) == [0, 75, 149]
    L = capi.load_library()
    assert L.vsag_amd_kmeans_init_plus_plus(1, 10, 4, 3, 10, draws.ctypes.data, 1, None, None, 0, None) == capi.INVALID_ARGUMENT


def _routed_data(kind, n, d, k):
    rng = np.random.default_rng(n + 3 * d + k)
    x = rng.standard_normal((n, d)).astype(np.float32)
    cent = x[rng.choice(n, k, replace=False)].copy()
    if kind == "offset":  # far from the origin: the centre takes the common part away
        x += 30.0
        cent += 30.0
    elif kind == "scaled":  # lengths over twelve octaves
        x *= np.exp2(rng.integers(-6, 7, (n, 1))).astype(np.float32)
    elif kind == "copies":  # every centroid five times: ties, and here and there a whole group that stays possible
        cent = np.tile(cent[: k // 5], (5, 1))[rng.permutation(k // 5 * 5)]
        cent = np.concatenate([cent, cent[: k - len(cent)]])
    elif kind == "same":  # one point: every distance ties
        x[:] = x[0]
        cent[:] = x[0]
    elif kind == "crowd":  # every centroid forty times, more than a row's list holds: every row goes to the fp32 kernels
        cent = cent[np.arange(k) % (k // 40)][rng.permutation(k)]
    elif kind == "holes":  # a row in 64 too long for fp16: every tile of the fp32 kernels has something to do
        x[::64] *= np.float32(1e16)
    elif kind == "long start":
        x[:65536] *= np.float32(1e16)
    elif kind == "exact":  # whole numbers of eleven bits around a centre of zero: fp16 holds them, only sums are rounded
        x = rng.integers(-2047, 2048, (n, d)).astype(np.float32)
        cent = rng.integers(-2047, 2048, (k, d)).astype(np.float32)
        cent[k // 2:k // 2 * 2] = cent[:k // 2]  # near ties: copies with one entry off by one
        cent[np.arange(k // 2), rng.integers(0, d, k // 2)] += 1.0
        step = k // 256  # the centre is made of sums of the rows (w + 16 i) * step: opposites in pairs
        for w in range(16):
            for i in range(0, 16, 2):
                cent[(w + 16 * (i + 1)) * step] = -cent[(w + 16 * i) * step]
    elif kind == "outliers":  # centroids far out, one of them with rows next to it, and centroids that are not finite
        cent[3] *= np.float32(100.0)
        cent[k - 1] *= np.float32(1e12)
        cent[64] *= np.float32(1e20)
        cent[70, 1] = np.nan
        cent[130, 0] = np.inf
        x[5], x[n - 1] = cent[3], cent[k - 1]
        x[700] = cent[3] * np.float32(0.5)  # halfway
    return x, cent


# At the edges of the pre-selection's tiles (256 x 256 x 64), with 4e9 products and more each.
@pytest.mark.parametrize("kind,n,d,k", [("plain", 20011, 130, 1601), ("plain", 65537, 64, 1024), ("plain", 4096, 1030, 1025),
                                        ("plain", 62001, 257, 257), ("offset", 20011, 101, 2049), ("scaled", 16385, 128, 2048),
                                        ("copies", 16385, 128, 2050), ("same", 16384, 128, 2048), ("plain", 33000, 64, 2111),
                                        ("outliers", 16385, 128, 2048), ("outliers", 20011, 101, 2049),
                                        ("outliers", 62001, 260, 256), ("plain", 20011, 100, 2049), ("plain", 20011, 132, 1601),
                                        ("plain", 62001, 196, 400), ("exact", 20011, 132, 1601), ("crowd", 20011, 101, 2049),
                                        ("crowd", 70001, 192, 320), ("holes", 20011, 101, 2049), ("holes", 70001, 192, 320),
                                        # one, two and three stages of 64 dimensions
                                        ("plain", 81921, 33, 1601), ("plain", 65537, 65, 1024), ("plain", 65537, 129, 512),
                                        # more rows than are rounded at a time (65536)
                                        ("holes", 70001, 1000, 260), ("outliers", 70001, 1000, 260),
                                        # the rows behind a slab of open ones are not pre-selected
                                        ("crowd", 70001, 1000, 260), ("long start", 70001, 1000, 260),
                                        ("long start", 70001, 1001, 260)])
def test_assign_after_the_fp16_preselection(lib, kind, n, d, k):
    x, cent = _routed_data(kind, n, d, k)
    labels, mind, loss = gpu_assign(x, cent)
    assert labels.min() >= 0 and labels.max() < k
    if kind not in ("outliers", "holes", "long start"):
        check_assignment(x, cent, labels, mind)
    # bit for bit what the fp32 kernels return: pieces too small for the pre-selection take those
    rows = min(n, int(3.9e9 / (k * d)))
    for r0 in range(0, n, rows):
        few, few_mind, _ = gpu_assign(x[r0:r0 + rows], cent)
        assert np.array_equal(labels[r0:r0 + rows], few)
        assert np.array_equal(mind[r0:r0 + rows].view(np.int32), few_mind.view(np.int32))
    x64, c64 = x.astype(np.float64), cent.astype(np.float64)
    assert abs(loss - (mind.astype(np.float64) + (x64 ** 2).sum(1)).mean()) <= 1e-5 * (x64 ** 2).sum(1).mean()
    if kind in ("copies", "same"):  # of equal centroids the first
        first = {}
        for j in range(k):
            first.setdefault(c64[j].tobytes(), j)
        assert all(first[c64[j].tobytes()] == j for j in np.unique(labels))


def test_centroids_far_out_do_not_open_every_row(lib):
    """The rows that are not near them stay with the pre-selection: all of them went to the fp32 kernels behind it, which took
    four times as long; twice is the line here."""
    L = lib.load_library()
    n, d, k = 200000, 256, 2048
    x, cent = _routed_data("plain", n, d, k)
    bad = cent.copy()
    bad[77] *= np.float32(1000.0)
    bad[1500, 3] = np.nan
    xb, lab = dev(x), capi.DeviceBuffer(n * 4)
    wsb = L.vsag_amd_kmeans_assign_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(wsb)
    cents, best = (dev(cent), dev(bad)), [1e9, 1e9]
    for _ in range(8):
        for i in range(2):
            capi.synchronize()
            t0 = time.perf_counter()
            capi.check(L.vsag_amd_kmeans_assign(xb.ptr, n, d, cents[i].ptr, k, lab.ptr, None, None, ws.ptr, wsb, None))
            capi.synchronize()
            best[i] = min(best[i], time.perf_counter() - t0)
    assert best[1] < 2.0 * best[0], best


def test_rows_that_stay_open_are_not_preselected_over_and_over(lib):
    """Where rows all over the place go to the fp32 kernels (the distances of clusters far from the origin are rounded to a
    good part of their spread), only every fourth slab is tried first: all were, which took 1.46 times as long as the fp32
    kernels alone, and 1.11 now; 1.3 is the line here."""
    L = lib.load_library()
    n, d, k = 480000, 960, 256
    rng = np.random.default_rng(3)
    x = gaussian_mixture(rng, n // 10, d, 1000, 0.05)[0] + np.float32(10.0)
    cent = x[rng.choice(len(x), k, replace=False)]
    xb, cb, lab = dev(np.tile(x, (10, 1))), dev(cent), capi.DeviceBuffer(n * 4)
    sizes = (_fp32_assign_bytes(n, k), L.vsag_amd_kmeans_assign_workspace_bytes(n, d, k))
    ws, best, out = capi.DeviceBuffer(sizes[1]), [1e9, 1e9], [None, None]
    for _ in range(8):
        for i in range(2):
            capi.synchronize()
            t0 = time.perf_counter()
            capi.check(L.vsag_amd_kmeans_assign(xb.ptr, n, d, cb.ptr, k, lab.ptr, None, None, ws.ptr, sizes[i], None))
            capi.synchronize()
            best[i] = min(best[i], time.perf_counter() - t0)
            out[i] = lab.to_numpy(np.int32, (n,))
    assert np.array_equal(out[0], out[1])
    assert best[1] < 1.3 * best[0], best


@pytest.mark.parametrize("n,d,k,iters", [(16400, 128, 2048, 6), (70001, 1000, 260, 3)])
def test_run_from_crowded_centroids(lib, n, d, k, iters):
    """Every row is open in the first iteration, few are in the later ones, some of which are not pre-selected: the centroids
    are those of the fp32 kernels alone."""
    L = lib.load_library()
    x, cent = _routed_data("crowd", n, d, k)
    xb, lab, out = dev(x), capi.DeviceBuffer(n * 4), []
    whole = L.vsag_amd_kmeans_run_workspace_bytes(n, d, k)
    rest = whole - L.vsag_amd_kmeans_assign_workspace_bytes(n, d, k)
    for wsb in (whole, _fp32_assign_bytes(n, k) + rest):
        cc, ws = dev(cent), capi.DeviceBuffer(wsb)
        capi.check(L.vsag_amd_kmeans_run(xb.ptr, n, d, cc.ptr, k, iters, 7, lab.ptr, None, ws.ptr, wsb, None))
        out.append((cc.to_numpy(np.int32, (k, d)), lab.to_numpy(np.int32, (n,))))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("scale", [1e-16, 1e-19, 1e-21, 1e-23, 1e-30])
def test_assign_after_the_fp16_preselection_of_tiny_values(lib, scale):
    """Distances down among the denormal numbers (and below): what the fp32 kernels return, bit for bit."""
    n, d, k = 16385, 128, 2048
    x, cent = _routed_data("plain", n, d, k)
    x *= np.float32(scale)
    cent *= np.float32(scale)
    labels, mind, _ = gpu_assign(x, cent)
    half = n // 2 + 1  # too few rows for the pre-selection
    few = [gpu_assign(part, cent) for part in (x[:half], x[half:])]
    assert np.array_equal(labels, np.concatenate([f[0] for f in few]))
    assert np.array_equal(mind.view(np.int32), np.concatenate([f[1] for f in few]).view(np.int32))


def _fp32_assign_bytes(n, k):
    """What the fp32 kernels need: |c|^2, |x|^2, a key a row, the partial sums of the loss."""
    return sum((b + 255) // 256 * 256 for b in (4 * k, 4 * n, 8 * n, 8 * ((n + 255) // 256), 8))


def test_a_workspace_without_room_for_the_preselection_is_served_by_the_fp32_kernels(lib):
    L = lib.load_library()
    n, d, k = 20011, 128, 2048
    x, cent = _routed_data("plain", n, d, k)
    labels, mind, _ = gpu_assign(x, cent)
    xb, cb, lab, dist = dev(x), dev(cent), capi.DeviceBuffer(n * 4), capi.DeviceBuffer(n * 4)
    room = _fp32_assign_bytes(n, k)
    assert room < L.vsag_amd_kmeans_assign_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(room)
    args = (xb.ptr, n, d, cb.ptr, k, lab.ptr, dist.ptr, None, ws.ptr)
    capi.check(L.vsag_amd_kmeans_assign(*args, room, None))
    assert np.array_equal(lab.to_numpy(np.int32, (n,)), labels)
    assert np.array_equal(dist.to_numpy(np.int32, (n,)), mind.view(np.int32))
    assert L.vsag_amd_kmeans_assign(*args, room - 256, None) == capi.INVALID_ARGUMENT
    assert b"workspace too small" in L.vsag_amd_last_error()
    # Lloyd iterations: the same centroids with either workspace
    out = []
    rest = L.vsag_amd_kmeans_run_workspace_bytes(n, d, k) - L.vsag_amd_kmeans_assign_workspace_bytes(n, d, k)
    for wsb in (L.vsag_amd_kmeans_run_workspace_bytes(n, d, k), room + rest):
        cc, ws, loss = dev(cent), capi.DeviceBuffer(wsb), C.c_double()
        capi.check(L.vsag_amd_kmeans_run(xb.ptr, n, d, cc.ptr, k, 3, 7, lab.ptr, C.byref(loss), ws.ptr, wsb, None))
        out.append((cc.to_numpy(np.int32, (k, d)), lab.to_numpy(np.int32, (n,)), loss.value))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    # (the two routes add |x|^2 up in different orders, each a wave's sum of d / 64 terms a lane)
    assert abs(out[0][2] - out[1][2]) <= 2 * (d / 64 + 12) * 2.0 ** -24 * (x.astype(np.float64) ** 2).sum(1).mean()


def test_assign_after_the_fp16_preselection_with_values_out_of_range(lib):
    # rows that fp16 or the error bound cannot cover go to the fp32 kernels; what they return is what those return alone
    n, d, k = 16500, 128, 2048
    x, cent = _routed_data("plain", n, d, k)
    odd = [3, 64, 700, 4097, n - 1]
    x[3, 5] = np.nan
    x[64] *= np.float32(1e18)
    x[700] = 0.0
    x[4097, 0] = np.inf
    x[n - 1] *= np.float32(1e-25)
    labels, mind, _ = gpu_assign(x, cent)
    few, few_mind, _ = gpu_assign(x[odd].copy(), cent)  # too few rows for the pre-selection
    assert np.array_equal(labels[odd], few)
    assert np.array_equal(mind[odd].view(np.int32), few_mind.view(np.int32))
    keep = np.setdiff1d(np.arange(n), odd)
    check_assignment(x[keep], cent, labels[keep], mind[keep])
    cent[7, 3] = np.inf  # one centroid out of range: nobody chooses it
    labels2, _, _ = gpu_assign(x[keep], cent)
    assert not (labels2 == 7).any() and (labels2 == labels[keep]).mean() > 0.999


@pytest.mark.parametrize("n,d,k,iters", [(16400, 128, 2048, 4), (70001, 1000, 260, 3)])
def test_run_with_the_fp16_preselection_keeps_its_rows(lib, n, d, k, iters):
    # the rows are rounded once per run where one slab holds them, and the centre is that of the first iteration; more rows
    # are rounded again in every iteration, and only their lengths are kept
    L = lib.load_library()
    rng = np.random.default_rng(5)
    x, means = gaussian_mixture(rng, n, d, 300, 0.2, uniform_means=False)
    # (no cluster may run empty: the steps below do not re-seed)
    cent0 = np.ascontiguousarray(means[:k]) if k <= len(means) else x[rng.choice(n, k, replace=False)].copy()
    xb, cb = dev(x), dev(cent0)
    labels = capi.DeviceBuffer(n * 4)
    loss = C.c_double()
    wsb = L.vsag_amd_kmeans_run_workspace_bytes(n, d, k)
    ws = capi.DeviceBuffer(wsb)
    capi.check(L.vsag_amd_kmeans_run(xb.ptr, n, d, cb.ptr, k, iters, 7, labels.ptr, C.byref(loss), ws.ptr, wsb, None))
    lab = labels.to_numpy(np.int32, (n,))
    # the same steps one by one
    cc, last = dev(cent0), None
    counts = capi.DeviceBuffer(k * 4)
    for _ in range(iters):
        last = gpu_assign(x, cc.to_numpy(np.float32, (k, d)))
        lb = dev(last[0])
        wsu = capi.DeviceBuffer(L.vsag_amd_kmeans_update_workspace_bytes(n, d, k))
        capi.check(L.vsag_amd_kmeans_update(xb.ptr, lb.ptr, n, d, k, cc.ptr, counts.ptr, wsu.ptr,
                                            L.vsag_amd_kmeans_update_workspace_bytes(n, d, k), None))
        assert (counts.to_numpy(np.int32, (k,)) > 0).all()
    assert np.array_equal(lab, last[0]) and loss.value == last[2]


@pytest.mark.parametrize("n,k,kind", [(1, 1, "even"), (63, 2, "even"), (1023, 3, "even"), (1024, 64, "even"), (1025, 65, "even"),
                                      (5000, 98, "skewed"), (5000, 98, "runs"), (40000, 4097, "even"),
                                      # the most labels of the counting sort (five units of 8256 rows, their table fits in 2 n
                                      # words), a table too large, and more labels: the general sort
                                      (41280, 16384, "even"), (41280, 16384, "skewed"), (40000, 16384, "even"),
                                      (40000, 16385, "even"), (41280, 16385, "even"), (70000, 1000, "one")])
def test_update_groups_the_rows_of_every_label(lib, n, k, kind):
    """Rows grouped by label around the edges of the counting sort's units and label bits: every mean is the sequential fp32 sum
    of the rows in row order, bit for bit, which holds only if the grouping is stable and complete."""
    L = lib.load_library()
    rng = np.random.default_rng(n * 7 + k)
    labels = rng.integers(0, k, n).astype(np.int32)
    if kind == "skewed":
        labels = (k * rng.random(n) ** 6).astype(np.int32)
    elif kind == "runs":
        labels = np.sort(labels)
    elif kind == "one":
        labels[:] = k - 1
    x = rng.standard_normal((n, 4)).astype(np.float32)
    cent0 = rng.standard_normal((k, 4)).astype(np.float32)
    xb, lb, cb, counts = dev(x), dev(labels), dev(cent0), capi.DeviceBuffer(k * 4)
    wsb = L.vsag_amd_kmeans_update_workspace_bytes(n, 4, k)
    ws = capi.DeviceBuffer(wsb)
    capi.check(L.vsag_amd_kmeans_update(xb.ptr, lb.ptr, n, 4, k, cb.ptr, counts.ptr, ws.ptr, wsb, None))
    sizes = np.bincount(labels, minlength=k)
    want, order = cent0.copy(), np.argsort(labels, kind="stable")
    begin = np.concatenate([[0], np.cumsum(sizes)])
    for j in np.nonzero(sizes)[0]:
        sums = np.cumsum(x[order[begin[j]:begin[j + 1]]], axis=0, dtype=np.float32)[-1]
        want[j] = sums * (np.float32(1) / np.float32(sizes[j]))
    assert np.array_equal(counts.to_numpy(np.int32, (k,)), sizes)
    # below 65 centroids of 8 dimensions and fewer in all the sums are added block by block of 1024 rows
    if k <= 64 and k * 4 <= 512 and n > 1024:
        assert np.allclose(cb.to_numpy(np.float32, (k, 4)), want, rtol=1e-5, atol=1e-6)
    else:
        assert np.array_equal(cb.to_numpy(np.float32, (k, 4)), want)
