"""GPU parity tests of the k-means assignment (hmlKmeansAssign) against the
oracle's restatement of the reference assign kernels
(include/hml_kmeans_kernel_template.h:18-88, 90-316, 323-367) and CPU path
(src/hml_kmeans_cpu.cu:55-95).  Indices are compared bit-exactly, including
near-ties (rows halfway between two centroids), duplicate centroids, NaN and
overflowing rows, dims that are not multiples of 4, centroid counts that
need several LDS chunks, and both distance arithmetics."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


KERNELS = [None, "screened", "direct"]


def kernels(D):
    """Kernel choices to check for D dims (the direct one takes <= 32)."""
    return KERNELS if D <= 32 else KERNELS[:2]


def run(hml, rows, ctrds, separate=False, offset=0, kernel=None):
    n, D = rows.shape
    K = ctrds.shape[0]
    flat = np.concatenate([np.full(offset, 7, np.float32), rows.ravel()]).astype(np.float32)
    dr = hml.DeviceBuffer.from_numpy(flat)
    dc = hml.DeviceBuffer.from_numpy(np.ascontiguousarray(ctrds, np.float32))
    da = hml.DeviceBuffer(4 * max(n, 1))
    hml.kmeans_assign(dr.ptr + 4 * offset, dc, da, n, D, K, separate_rounding=separate,
                      kernel=kernel)
    hml.synchronize()
    return da.to_numpy((n,), np.uint32)


def clustered(rng, n, D, K, spread=0.5):
    ctrds = rng.standard_normal((K, D)).astype(np.float32)
    rows = ctrds[rng.integers(0, K, n)] + spread * rng.standard_normal((n, D)).astype(np.float32)
    return rows.astype(np.float32), ctrds


def near_ties(rng, n, D, K, eps=1e-5):
    ctrds = rng.standard_normal((K, D)).astype(np.float32)
    a, b = ctrds[rng.integers(0, K, n)], ctrds[rng.integers(0, K, n)]
    rows = (a + b) / 2 + eps * rng.standard_normal((n, D))
    return rows.astype(np.float32), ctrds


@pytest.mark.parametrize("D", [1, 3, 4, 7, 16, 17, 31, 32, 48, 50, 63, 64])
@pytest.mark.parametrize("K", [1, 5, 16, 33, 64, 100])
def test_matches_oracle(hml, D, K):
    rng = np.random.default_rng(D * 1000 + K)
    n = 3001
    print("case D=%d K=%d" % (D, K), flush=True)
    for make in (clustered, near_ties):
        rows, ctrds = make(rng, n, D, K)
        for sep in (False, True):
            want = oracle.kmeans_assign(rows, ctrds, fused=not sep)
            for kern in kernels(D):
                got = run(hml, rows, ctrds, sep, kernel=kern)
                np.testing.assert_array_equal(got, want, err_msg="%s sep=%s kernel=%s" % (
                    make.__name__, sep, kern))


@pytest.mark.parametrize("D,K", [(64, 129), (64, 300), (16, 1000), (8, 4097), (2, 70), (64, 1000), (3, 9000)])
def test_many_centroids(hml, D, K):
    """More centroids than one LDS chunk holds (several chunks per row step:
    above 256 x 64 dims for the direct kernel, 128 x 64 for the screened
    one) and several screening passes."""
    rng = np.random.default_rng(K)
    print("case D=%d K=%d" % (D, K), flush=True)
    for make in (clustered, near_ties):
        rows, ctrds = make(rng, 2000, D, K)
        want = oracle.kmeans_assign(rows, ctrds)
        for kern in kernels(D):
            got = run(hml, rows, ctrds, kernel=kern)
            np.testing.assert_array_equal(got, want, err_msg="%s kernel=%s" % (make.__name__, kern))


def test_fused_vs_separate_flip(hml):
    """The constructed input on which the two arithmetics disagree: the
    kernel follows the requested one."""
    from test_oracle import fused_flip_case
    rows, ctrds = fused_flip_case()
    rows = np.repeat(rows, 37, 0)
    for kern in KERNELS:
        assert (run(hml, rows, ctrds, separate=False, kernel=kern) == 1).all()
        assert (run(hml, rows, ctrds, separate=True, kernel=kern) == 0).all()


def test_edge_rows(hml):
    """Duplicate centroids (the first wins), rows equal to centroids,
    NaN / overflowing rows (numClusts), zero rows, an odd row offset."""
    rng = np.random.default_rng(3)
    D, K = 21, 40
    ctrds = rng.standard_normal((K, D)).astype(np.float32)
    ctrds[30] = ctrds[4]
    ctrds[31] = ctrds[4]
    rows = ctrds[rng.integers(0, K, 500)].copy()
    rows[7] = np.nan
    rows[8] = 3e38
    rows[9, 3] = np.inf
    rows[10] = 0
    want = oracle.kmeans_assign(rows, ctrds)
    assert want[7] == K and want[8] == K and want[9] == K
    assert not np.isin(want, [30, 31]).any()
    for off in (0, 1):
        for kern in KERNELS:
            np.testing.assert_array_equal(run(hml, rows, ctrds, offset=off, kernel=kern), want)


def test_sizes(hml):
    """Row counts around the 16-row tile and the 4-tile workgroup step, one
    cluster, and a large problem checked through a sample of rows."""
    rng = np.random.default_rng(5)
    for n in (1, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1000):
        rows, ctrds = clustered(rng, n, 10, 7)
        for kern in KERNELS:
            np.testing.assert_array_equal(run(hml, rows, ctrds, kernel=kern),
                                          oracle.kmeans_assign(rows, ctrds))
    rows, ctrds = clustered(rng, 100, 5, 1)
    assert (run(hml, rows, ctrds) == 0).all()
    n, D, K = 1 << 22, 32, 64
    rows, ctrds = clustered(rng, n, D, K)
    got = run(hml, rows, ctrds)
    idx = rng.choice(n, 20000, replace=False)
    np.testing.assert_array_equal(got[idx], oracle.kmeans_assign(rows[idx], ctrds))
    # every index in range, and each cluster's rows are nearer to it than
    # to a random other centroid (size-independent property)
    assert got.max() < K
    other = rng.integers(0, K, n)
    d_own = ((rows - ctrds[got]) ** 2).sum(1)
    d_oth = ((rows - ctrds[other]) ** 2).sum(1)
    assert (d_own <= d_oth * (1 + 1e-5) + 1e-30).all()


def test_direct_kernel_dim_limit(hml):
    """Forcing the direct kernel above 32 dims is rejected, not rerouted."""
    rows = np.zeros((10, 33), np.float32)
    ctrds = np.zeros((3, 33), np.float32)
    with pytest.raises(hml.HmlError):
        run(hml, rows, ctrds, kernel="direct")


def test_centroid_scales(hml):
    """Centroids of very different norms (the screen's margin is bounded
    with each chunk's largest norm), and an infinite and a NaN centroid
    (never chosen; the infinite norm widens the screen to every centroid),
    over several screening passes and LDS chunks."""
    rng = np.random.default_rng(11)
    for D, K in ((16, 200), (64, 300), (5, 40)):
        print("case D=%d K=%d" % (D, K), flush=True)
        for make in (clustered, near_ties):
            rows, ctrds = make(rng, 2000, D, K)
            ctrds = ctrds.copy()
            ctrds[3] *= 1e4
            ctrds[K // 2] *= 1e-3
            want = oracle.kmeans_assign(rows, ctrds)
            for kern in kernels(D):
                np.testing.assert_array_equal(run(hml, rows, ctrds, kernel=kern), want,
                                              err_msg="%s kernel=%s" % (make.__name__, kern))
            ctrds[7, 0] = np.inf
            ctrds[9] = np.nan
            want = oracle.kmeans_assign(rows, ctrds)
            assert not np.isin(want, [7, 9]).any()
            for kern in kernels(D):
                np.testing.assert_array_equal(run(hml, rows, ctrds, kernel=kern), want,
                                              err_msg="inf/nan %s kernel=%s" % (make.__name__, kern))


def integer_grid(rng, n, D, K):
    """Small whole numbers: many rows equidistant from several centroids."""
    ctrds = rng.integers(-2, 3, (K, D)).astype(np.float32)
    return rng.integers(-2, 3, (n, D)).astype(np.float32), ctrds


@pytest.mark.parametrize("D", [2, 15, 16, 18, 33, 47, 60, 64])
@pytest.mark.parametrize("K", [1, 31, 32, 33, 64, 65, 97])
def test_screen_edges(hml, D, K):
    """The screened kernel at the edges of its 32-row and 32-centroid tiles
    and 16-dim steps, where the screen decides alone (clustered rows), where
    trackers or a second screening decide (near ties, whole-number grids),
    and at scales where squares overflow, underflow or leave the screen's
    range, with centroids padded by FLT_MAX / 2."""
    rng = np.random.default_rng(100 * D + K)
    for n in (1, 31, 32, 33, 8 * 32 + 5):
        for make in (clustered, near_ties, integer_grid):
            rows, ctrds = make(rng, n, D, K)
            want = oracle.kmeans_assign(rows, ctrds)
            got = run(hml, rows, ctrds, kernel="screened", offset=n % 3)
            np.testing.assert_array_equal(got, want, err_msg="%s n=%d" % (make.__name__, n))
    rows, ctrds = clustered(rng, 70, D, K)
    pad = np.full((5, D), 3.4028235e38 / 2, np.float32)
    for scale in (1e-30, 1e-19, 1e15, 3e17, 2e18, 1e19, 1e30):
        r, c = (rows * np.float32(scale)), (ctrds * np.float32(scale))
        for cc in (c, np.concatenate([c, pad])):
            want = oracle.kmeans_assign(r, cc)
            got = run(hml, r, cc, kernel="screened")
            np.testing.assert_array_equal(got, want, err_msg="scale %g" % scale)


@pytest.mark.parametrize("D,K", [(4, 70), (17, 33), (32, 64), (50, 100), (64, 300)])
def test_off_centre(hml, D, K):
    """Rows and centroids far from the origin, with a far centroid, with most
    of the sampled centroids equal or not finite: the point that the screen
    moves them by, and its scale, change no index."""
    rng = np.random.default_rng(D + K)
    for make in (clustered, near_ties):
        rows, ctrds = make(rng, 1500, D, K)
        for off in (3.0, 300.0, 3e4, np.float32(1e4) * rng.standard_normal(D).astype(np.float32)):
            for change in (None, "far", "equal", "nan"):
                r, c = (rows + off).astype(np.float32), (ctrds + off).astype(np.float32)
                if change == "far":
                    c[K // 2] += 1e3
                elif change == "equal":
                    c[: K - 3] = c[0]
                elif change == "nan":
                    c[:: max(1, K // 8)] = np.nan
                want = oracle.kmeans_assign(r, c)
                got = run(hml, r, c, kernel="screened")
                np.testing.assert_array_equal(got, want, err_msg="%s %s %s" % (make.__name__, off, change))


def seconds(hml, rows, ctrds, reps=20):
    """Best of three timings of `reps` assignments."""
    n, D = rows.shape
    dr, dc = hml.DeviceBuffer.from_numpy(rows), hml.DeviceBuffer.from_numpy(ctrds)
    da = hml.DeviceBuffer(4 * n)
    best = float("inf")
    for _ in range(4):
        e0, e1 = hml.Event(), hml.Event()
        e0.record()
        for _ in range(reps):
            hml.kmeans_assign(dr, dc, da, n, D, ctrds.shape[0], kernel="screened")
        e1.record()
        e1.synchronize()
        best = min(best, e0.elapsed_ms(e1) / reps)
    return best


@pytest.mark.parametrize("D,K", [(32, 64), (64, 256)])
def test_off_centre_is_not_slower(hml, D, K):
    """Moving the data away from the origin, or one centroid away from the
    others, does not send every row to the exact comparison (30 times slower
    when it does): within 3 times the centred time."""
    rng = np.random.default_rng(1)
    ctrds = rng.uniform(-1, 1, (K, D)).astype(np.float32)
    rows = rng.uniform(-1, 1, (1 << 17, D)).astype(np.float32)
    centred = seconds(hml, rows, ctrds)
    far = ctrds.copy()
    far[K // 2] = 1000.0
    for r, c in ((rows + np.float32(100), ctrds + np.float32(100)), (rows, far)):
        assert seconds(hml, r, c) < 3 * centred


@pytest.mark.parametrize("D,K", [(5, 60), (16, 100), (33, 64), (64, 130), (64, 500)])
def test_equidistant(hml, D, K):
    """Rows with many candidates: 0/1 features with centroids among the rows,
    all centroids equal (every pair is compared), all but one equal, and such
    rows beside rows with none, in whole and partial tiles."""
    rng = np.random.default_rng(D * K)
    for n in (1, 31, 33, 700):
        rows = rng.integers(0, 2, (n, D)).astype(np.float32)
        ctrds = rng.integers(0, 2, (K, D)).astype(np.float32)
        ctrds[: min(n, K // 2)] = rows[: min(n, K // 2)]
        same = np.repeat(ctrds[:1], K, 0)
        one = same.copy()
        one[K - 2] += 0.25
        some, spread = clustered(rng, n, D, K)
        some[::3] = rows[::3]
        some[1::7] = np.nan
        for r, c in ((rows, ctrds), (rows, same), (rows, one), (some, spread), (some, one)):
            for sep in (False, True):
                np.testing.assert_array_equal(run(hml, r, c, sep, kernel="screened"),
                                              oracle.kmeans_assign(r, c, fused=not sep))


def test_ties_are_compared_together(hml):
    """0/1 features, as in a first iteration from sampled rows: most rows have
    a tie to decide.  Within 3 times the time of clustered rows (4.2 when every
    lane compares its own candidates in turn)."""
    rng = np.random.default_rng(2)
    D, K, n = 32, 64, 1 << 20
    rows, ctrds = clustered(rng, n, D, K, 0.1)
    free = seconds(hml, rows, ctrds)
    rows = rng.integers(0, 2, (n, D)).astype(np.float32)
    assert seconds(hml, rows, rows[rng.choice(n, K, replace=False)]) < 3 * free


def test_ragged_dims_cost_what_whole_ones_do(hml):
    """62 dims, read float by float, against 64 at 55 clusters: within 1.4
    times the time (1.7 when the kernel spills its registers)."""
    rng = np.random.default_rng(3)
    t = {}
    for D in (62, 64):
        rows, ctrds = clustered(rng, 1 << 20, D, 55, 0.1)
        t[D] = seconds(hml, rows, ctrds)
    assert t[62] < 1.4 * t[64], t
