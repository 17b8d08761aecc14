"""The half-precision ranking sweep and its exact pass (csrc/rank16.hip) against the serial oracle, bit for bit: every number of
blocks of 16 dimensions, resident and streamed centroids, one to four groups of listed points per unit, lists that overflow,
SoA points in one part and in several (-m gpu)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def flat(rows, layout):
    return np.ascontiguousarray(rows if layout == 0 else rows.T).ravel()


@pytest.mark.parametrize("kind", ["clustered", "grid", "same"])
@pytest.mark.parametrize("dim,k,n", [
    (5, 33, 1), (16, 1, 64), (17, 40, 65), (32, 1024, 3001), (33, 31, 500), (48, 700, 2049), (49, 65, 4100),
    (64, 1300, 1025), (65, 64, 600), (96, 300, 515), (97, 33, 513), (128, 700, 1030), (129, 250, 1000),
    (192, 32, 700), (193, 900, 600), (256, 330, 1025), (20, 5000, 1500), (40, 16, 70001),
])
def test_half_precision_sweep_matches_the_oracle(km, orc, gpu, dim, k, n, kind):
    rng = np.random.default_rng(dim * 37 + k)
    centres = rng.uniform(-3, 3, size=(k, dim)).astype(np.float32)
    rows = (centres[rng.integers(0, k, n)] + rng.normal(size=(n, dim))).astype(np.float32)
    means = (centres + rng.normal(size=(k, dim)) * 0.3).astype(np.float32)
    if kind == "grid":       # many exact ties: duplicated centroids, points on bisectors
        rows, means = np.round(rows * 0.5).astype(np.float32), np.round(means * 0.5).astype(np.float32)
        means[k // 2:] = means[:k - k // 2]
    elif kind == "same":     # every centroid within every threshold: the lists of pairs overflow
        means[:] = means[0]
    if n > 20:
        rows[7, 3] = np.nan
        rows[11, dim - 1] = np.inf
        rows[13] *= np.float32(1e-30)
        rows[17, 0] = 1e30
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    a = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for layout, layout_means, pad, limit in [(0, 0, 0, 1 << 30), (0, 1, 5, 1 << 30), (1, 0, 0, 1 << 30), (1, 1, 0, 1)]:
            stride = dim + pad if layout == 0 else n
            padded = rows
            if pad:
                padded = np.full((n, stride), np.float32(np.nan)); padded[:, :dim] = rows
            d = km.DeviceBuffer(padded.nbytes); d.write(flat(padded, layout))
            m = km.DeviceBuffer(4 * k * dim); m.write(flat(means, layout_means))
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            km.set_queued_rows_limit(limit)  # (1 byte: parts of 1024 points)
            km.assign(km.ASSIGN_MFMA_BF16X3, d, layout, stride, m, layout_means, km.layout_stride(layout_means, k, dim), a, dim, k, n)
            km.sync()
            got = a.read(np.uint32, n)
            d.free(); m.free()
            assert np.array_equal(got, want), "layouts %d/%d: %d mismatches" % (layout, layout_means, int((got != want).sum()))
    finally:
        km.set_two_level_sweep(1)
        km.set_queued_rows_limit(1 << 30)
    a.free()


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -18, 2.0 ** 10])
def test_half_precision_products_accumulate_as_the_certificate_assumes(km, gpu, scale):
    """At most one 2^-23 of the running magnitude per accumulated product; operands down to the smallest subnormal (2^-24) count."""
    rng = np.random.default_rng(5)
    depth = 256
    a = (rng.normal(size=(32, depth)) * scale * np.exp2(rng.integers(-8, 3, (32, depth)))).astype(np.float16).astype(np.float32)
    b = (rng.normal(size=(32, depth)) * scale * np.exp2(rng.integers(-8, 3, (32, depth)))).astype(np.float16).astype(np.float32)
    a[:, 1::2] = -a[:, 0::2]; b[:, 1::2] = b[:, 0::2]          # cancelling pairs ...
    a[:, 5] = 2.0 ** -24; b[:, 5] = 2.0 ** -24                 # ... next to the smallest numbers there are
    c = (rng.normal(size=(32, 32)) * scale * scale).astype(np.float32)
    d = km.probe_matrix_chain(3, a, b, c).astype(np.float64)
    exact = c.astype(np.float64) + a.astype(np.float64) @ b.astype(np.float64).T
    magnitude = np.abs(c).astype(np.float64) + np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64).T
    assert (np.abs(d - exact) <= (depth + 1) * 2.0 ** -23 * magnitude).all()
    only = np.zeros((32, 16), np.float32); only[:, 3] = 2.0 ** -24
    alone = km.probe_matrix_chain(3, only, np.full((32, 16), 1024.0, np.float32), np.zeros((32, 32), np.float32))
    assert (alone == np.float32(2.0 ** -14)).all()             # subnormal operands are not flushed


@pytest.mark.parametrize("dim,k,n,mode", [(8, 130, 40001, 1), (50, 300, 70007, 1), (50, 60, 40003, 1), (9, 40, 33000, 1), (256, 129, 33001, 1), (300, 20, 33003, 1), (50, 300, 40000, 0), (390, 70, 33001, 0)])
def test_iterations_on_soa_points_match_the_oracle(km, orc, gpu, dim, k, n, mode):
    """The assignment's copy of the rows, or the one made ahead of it, is what the update adds up."""
    rng = np.random.default_rng(dim + k)
    rows = rng.normal(size=(n, dim)).astype(np.float32)
    means = np.ascontiguousarray(rows[rng.choice(n, k, replace=False)])
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, 1))
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 1))
    o = km.DeviceBuffer(means.nbytes); a = km.DeviceBuffer(4 * n); s = km.DeviceBuffer(4 * k)
    km.set_two_level_sweep(mode)
    try:
        km.iteration(d, 1, n, m, o, 1, k, a, s, dim, k, n)
        km.sync()
    finally:
        km.set_two_level_sweep(1)
    assert np.array_equal(a.read(np.uint32, n), want)
    counts = np.bincount(want, minlength=k)
    assert np.array_equal(s.read(np.uint32, k), counts)
    sums = np.zeros((k, dim)); np.add.at(sums, want, rows.astype(np.float64))
    got = o.read(np.float32, k * dim).reshape(dim, k).T
    assert np.allclose(got, sums / counts[:, None], rtol=1e-5, atol=1e-6)
    for b in (d, m, o, a, s):
        b.free()


@pytest.mark.parametrize("dim,k,n,budget", [
    (100, 700, 263003, 0), (60, 1250, 263003, 0), (20, 2300, 140001, 0),   # two chunks as large as fit, several units per work-group
    (250, 330, 263003, 0), (177, 290, 140001, 0),                           # slots of a tile, two work-groups per compute unit
    (16, 3000, 700, 56 * 1024), (96, 90, 700, 56 * 1024), (256, 65, 700, 78 * 1024),  # as little LDS as the exact pass runs in
])
def test_centroids_that_stream_by(km, orc, gpu, dim, k, n, budget):
    rng = np.random.default_rng(dim + n)
    means = rng.normal(size=(k, dim)).astype(np.float32)
    rows = (means[rng.integers(0, k, n)] + rng.normal(size=(n, dim)) * 0.5).astype(np.float32)
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 0))
    a = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for layout in (0, 1):
            d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, layout))
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            ex = km.ExecParams(shared_mem_bytes=budget)
            km.assign(km.ASSIGN_MFMA_BF16X3, d, layout, km.layout_stride(layout, n, dim), m, 0, dim, a, dim, k, n, ex)
            km.sync()
            got = a.read(np.uint32, n)
            d.free()
            assert ex.block_count <= 2 * gpu.compute_units
            assert np.array_equal(got, want), "layout %d: %d mismatches" % (layout, int((got != want).sum()))
    finally:
        km.set_two_level_sweep(1)
    m.free(); a.free()


@pytest.mark.parametrize("dim,k,budget", [
    (16, 1184, 56 * 1024), (16, 1344, 56 * 1024), (16, 1345, 56 * 1024),   # the longest lists, shorter ones, centroids that stream by instead
    (32, 640, 56 * 1024), (30, 704, 56 * 1024), (48, 470, 56 * 1024), (61, 350, 56 * 1024), (96, 230, 56 * 1024), (128, 160, 56 * 1024),
    (200, 60, 78 * 1024), (16, 64, 0),
])
def test_lists_that_share_lds_with_the_centroids(km, orc, gpu, dim, k, budget):
    """Every centroid twice: all points are listed, more of them per wavefront than its list holds, whatever the centroids leave for it."""
    n = 263003
    rng = np.random.default_rng(dim + k)
    means = np.repeat(rng.normal(size=((k + 1) // 2, dim)), 2, axis=0)[:k].astype(np.float32)
    rows = (means[rng.integers(0, k, n)] + rng.normal(size=(n, dim)) * 0.5).astype(np.float32)
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 0))
    a = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for layout in (0, 1):
            d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, layout))
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            km.assign(km.ASSIGN_MFMA_BF16X3, d, layout, km.layout_stride(layout, n, dim), m, 0, dim, a, dim, k, n, km.ExecParams(shared_mem_bytes=budget))
            km.sync()
            got = a.read(np.uint32, n)
            d.free()
            assert np.array_equal(got, want), "layout %d: %d mismatches" % (layout, int((got != want).sum()))
    finally:
        km.set_two_level_sweep(1)
    m.free(); a.free()


@pytest.mark.parametrize("dim,k,more,bound", [(12, 3600, 4000, 1.3), (64, 1050, 1150, 1.19)])
def test_soa_points_around_as_many_centroids_as_fit(km, gpu, dim, k, more, bound):
    """The room in which SoA rows are exchanged does not push the centroids out of LDS: a tenth more of them takes 1.08 and 1.05 to 1.11 times
    as long (1.53 and 1.27 where they streamed by instead)."""
    n = 1 << 20
    rng = np.random.default_rng(dim)
    rows = rng.standard_normal((n, dim), dtype=np.float32)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, 1))
    a = km.DeviceBuffer(4 * n)
    start, stop = km.Event(), km.Event()
    ms = []
    for count in (k, more):
        m = km.DeviceBuffer(4 * count * dim); m.write(flat(rows[:count], 1))
        times = []
        for call in range(30):
            start.record()
            km.assign(km.ASSIGN_BEST, d, 1, n, m, 1, count, a, dim, count, n)
            stop.record()
            km.sync()
            if call > 9:
                times.append(start.elapsed_ms(stop))
        ms.append(float(np.median(times)))
        m.free()
    d.free(); a.free()
    print("%d: %.3f ms, %d: %.3f ms" % (k, ms[0], more, ms[1]))
    assert ms[1] <= bound * ms[0]


def group_of(row):
    """Of a centroid's row in its tile: the half-wave that holds its result, and the group of that lane's 16 results (rank16_impl.h)."""
    result, half = row // 8 * 4 + row % 4, row // 4 % 2
    return half * 6 + (5 if result == 15 else 4 if result % 4 == 3 else result // 4)


@pytest.mark.parametrize("dim,k", [(5, 32), (16, 70), (16, 96), (20, 64), (32, 129)])
def test_every_place_of_the_runner_up(km, orc, gpu, dim, k):
    """Points on the line between every two centroids, next to the middle: the nearest two lie in one group of a tile's results, in two
    groups, in the two half-waves and in two tiles, in every combination, with margins from nothing to what the sweep settles by itself."""
    rng = np.random.default_rng(dim + k)
    means = rng.normal(size=(k, dim)).astype(np.float32)
    a, b = (i.ravel() for i in np.meshgrid(np.arange(k), np.arange(k), indexing="ij"))
    a, b = a[a != b], b[a != b]
    shift = np.array([0, 1e-7, 1e-6, 1e-5, 1e-4, 1e-3, 1e-2, 0.1])
    at = (0.5 - shift)[:, None, None]  # (b, a as well as a, b: to either side of the middle)
    rows = (means[a] * (1 - at) + means[b] * at).astype(np.float32).reshape(-1, dim)
    n = len(rows)
    if 16 <= dim <= 20:  # the tile's groups as winner and runner-up, each with each
        far = ((rows[:, None, :].astype(np.float64) - means[None]) ** 2).sum(2)
        first, second = np.argsort(far, axis=1)[:, :2].T
        same = first // 32 == second // 32
        met = {(group_of(i % 32), group_of(j % 32)) for i, j in zip(first[same], second[same])}
        alone = {5, 11}  # (groups of one result)
        assert met >= {(i, j) for i in range(12) for j in range(12) if i != j or i not in alone}
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0)
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 0))
    out = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for layout in (0, 1):
            d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, layout))
            out.write(np.full(n, 0xFFFFFFF1, np.uint32))
            km.assign(km.ASSIGN_MFMA_BF16X3, d, layout, km.layout_stride(layout, n, dim), m, 0, dim, out, dim, k, n)
            km.sync()
            got = out.read(np.uint32, n)
            d.free()
            assert np.array_equal(got, want), "layout %d: %d mismatches" % (layout, int((got != want).sum()))
    finally:
        km.set_two_level_sweep(1)
    m.free(); out.free()


@pytest.mark.parametrize("share", [0.01, 0.12, 0.3, 0.5, 1.0])
@pytest.mark.parametrize("dim,k,n", [(5, 40, 4099), (17, 40, 4099), (40, 64, 3001), (63, 40, 70003), (90, 64, 3001), (128, 600, 5001), (180, 64, 3001), (250, 200, 5001)])
def test_listed_rows_of_soa_points_are_copied_behind_the_sweep(km, orc, gpu, dim, k, n, share):
    """Points halfway between two centroids, which no ranking settles: none, up to eight, more than eight and nearly all of a wavefront's 64."""
    rng = np.random.default_rng(dim + n + int(100 * share))
    means = rng.integers(-8, 9, size=(k, dim)).astype(np.float32)
    near = means[rng.integers(0, k, n)]
    halfway = rng.random(n) < share
    rows = np.where(halfway[:, None], (near + means[rng.integers(0, k, n)]) / 2, near + rng.normal(size=(n, dim)).astype(np.float32) * np.float32(0.1)).astype(np.float32)
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, 1))
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 0))
    a = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for limit in (1 << 30, 1):
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            km.set_queued_rows_limit(limit)
            km.assign(km.ASSIGN_MFMA_BF16X3, d, 1, n, m, 0, dim, a, dim, k, n)
            km.sync()
            got = a.read(np.uint32, n)
            assert np.array_equal(got, want), "%d mismatches" % int((got != want).sum())
    finally:
        km.set_two_level_sweep(1)
        km.set_queued_rows_limit(1 << 30)
    for b in (d, m, a):
        b.free()


@pytest.mark.parametrize("dim,k,n", [(5, 100, 300001), (7, 500, 40003), (100, 2, 70001), (250, 20, 33001), (60, 20, 40003), (40, 33, 70001), (24, 96, 131072), (64, 20, 530001), (300, 33, 60000)])
def test_iterations_on_soa_points_with_few_centroids(km, orc, gpu, dim, k, n):
    """Both sides of the line between the sweeps, and the update of columns behind each of them."""
    test_iterations_on_soa_points_match_the_oracle(km, orc, gpu, dim, k, n, 1)


@pytest.mark.parametrize("dim,k", [(97, 40), (128, 600), (200, 40), (250, 600)])
@pytest.mark.parametrize("n", [65, 192, 520, 577, 5001, 33281])
def test_columns_read_by_wavefronts_without_points(km, orc, gpu, dim, k, n):
    """Numbers of points that leave one to seven wavefronts of the last unit without any, centroids in LDS and streamed: those read the last point again."""
    test_listed_rows_of_soa_points_are_copied_behind_the_sweep(km, orc, gpu, dim, k, n, 0.12)


# rows of 12 and 16 blocks: as many centroids as are kept in LDS, one more, and as many as would just fit without room to exchange rows
@pytest.mark.parametrize("dim,k,streamed", [(150, 352, False), (150, 353, True), (185, 384, True), (250, 256, False), (250, 257, True), (200, 288, True)])
def test_wide_soa_rows_around_as_many_centroids_as_fit(km, orc, gpu, dim, k, streamed):
    n = 4099
    rng = np.random.default_rng(dim + k)
    means = rng.normal(size=(k, dim)).astype(np.float32) * np.float32(3)
    rows = (means[rng.integers(0, k, n)] + rng.normal(size=(n, dim)) * 0.5).astype(np.float32)
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, 1))
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 0))
    a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
    ex = km.ExecParams()
    km.set_two_level_sweep(2)
    try:
        km.assign(km.ASSIGN_MFMA_BF16X3, d, 1, n, m, 0, dim, a, dim, k, n, ex)
        km.sync()
    finally:
        km.set_two_level_sweep(1)
    assert np.array_equal(a.read(np.uint32, n), want)
    assert ex.block_count == -(-n // (256 if streamed else 512))        # units of four or of eight wavefronts
    for b in (d, m, a):
        b.free()


# the rows of all points from the sweep: every number of blocks, with more centroids than a column's sums fit the budget
@pytest.mark.parametrize("dim", [12, 30, 45, 64, 90, 120, 180, 250])
@pytest.mark.parametrize("n", [12011, 8191])
def test_iterations_around_more_centroids_than_sums_fit(km, orc, gpu, dim, n):
    k = 6850
    rng = np.random.default_rng(dim + k)
    rows = rng.normal(size=(n, dim)).astype(np.float32)
    means = np.ascontiguousarray(rows[rng.choice(n, k, replace=False)])
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, 1))
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 1))
    o = km.DeviceBuffer(means.nbytes); a = km.DeviceBuffer(4 * n); s = km.DeviceBuffer(4 * k)
    km.set_two_level_sweep(2)
    try:
        km.iteration(d, 1, n, m, o, 1, k, a, s, dim, k, n, km.ExecParams(shared_mem_bytes=80 * 1024))
        km.sync()
    finally:
        km.set_two_level_sweep(1)
    assert np.array_equal(a.read(np.uint32, n), want)
    counts = np.bincount(want, minlength=k)
    assert np.array_equal(s.read(np.uint32, k), counts)
    sums = np.zeros((k, dim)); np.add.at(sums, want, rows.astype(np.float64))
    got = o.read(np.float32, k * dim).reshape(dim, k).T
    assert np.allclose(got, sums / np.maximum(counts, 1)[:, None], rtol=1e-5, atol=1e-6)
    for b in (d, m, o, a, s):
        b.free()
