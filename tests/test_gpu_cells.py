"""Rows of 2 to 4 dimensions through the grid of cells (csrc/assign_cells.hip) against the serial oracle, bit for bit: points inside and
outside the grid, on its edges, exact ties, degenerate boxes, lists that do not fit, values that are not finite (-m gpu)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def flat(rows, layout):
    return np.ascontiguousarray(rows if layout == 0 else rows.T).ravel()


@pytest.mark.parametrize("kind", ["uniform", "clustered", "lattice", "offset", "line", "same", "dense", "nan", "huge", "tiny"])
@pytest.mark.parametrize("dim,k,n", [(2, 2, 1), (2, 129, 2049), (2, 6000, 20000), (3, 7, 1025), (3, 1000, 9000), (3, 4097, 12000), (4, 33, 1000), (4, 512, 5000), (4, 4096, 20001)])
def test_cells_match_the_oracle(km, orc, gpu, dim, k, n, kind):
    rng = np.random.default_rng(dim * 41 + k)
    means = rng.uniform(0, 1, size=(k, dim)).astype(np.float32)
    rows = rng.uniform(-0.05, 1.05, size=(n, dim)).astype(np.float32)
    if kind == "clustered":
        centres = rng.uniform(-10, 10, size=(20, dim))
        means = (centres[rng.integers(0, 20, k)] + rng.normal(size=(k, dim))).astype(np.float32)
        rows = (centres[rng.integers(0, 20, n)] + rng.normal(size=(n, dim))).astype(np.float32)
    elif kind == "lattice":   # ties everywhere, points on the edges of cells
        means = np.round(means * 8).astype(np.float32); rows = (np.round(rows * 32) / 4).astype(np.float32)
    elif kind == "offset":
        means += np.float32(1000); rows += np.float32(1000)
    elif kind == "line":      # no extent in one dimension
        means[:, dim - 1] = 0.5; rows[::2, dim - 1] = 0.5
    elif kind == "same":
        means[:] = means[0]
    elif kind == "dense":     # almost all centroids and points in one cell
        means[1:] = (0.5 + means[1:] * 1e-3).astype(np.float32); rows[1:] = (0.5 + rows[1:] * 1e-3).astype(np.float32)
        means[0] = 30
    elif kind == "nan":
        means[k // 2] = np.nan
    elif kind == "huge":
        means *= np.float32(1e19); rows *= np.float32(1e19)
    elif kind == "tiny":
        means *= np.float32(1e-22); rows *= np.float32(1e-22)
    if n > 20:
        rows[3] = means[min(3, k - 1)]
        rows[7, 0] = np.nan; rows[11, dim - 1] = np.inf; rows[13] = -1e30; rows[17] = 1e6
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    a = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for layout, layout_means, pad in [(0, 0, 0), (0, 1, 3), (1, 1, 0)]:
            stride = dim + pad if layout == 0 else n
            padded = rows
            if pad:
                padded = np.full((n, stride), np.float32(np.nan)); padded[:, :dim] = rows
            d = km.DeviceBuffer(padded.nbytes); d.write(flat(padded, layout))
            m = km.DeviceBuffer(4 * k * dim); m.write(flat(means, layout_means))
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            km.assign(km.ASSIGN_MFMA_BF16X3, d, layout, stride, m, layout_means, km.layout_stride(layout_means, k, dim), a, dim, k, n)
            km.sync()
            got = a.read(np.uint32, n)
            d.free(); m.free()
            assert np.array_equal(got, want), "layouts %d/%d: %d mismatches" % (layout, layout_means, int((got != want).sum()))
    finally:
        km.set_two_level_sweep(1)
    a.free()


@pytest.mark.parametrize("dim,k", [(2, 2), (2, 130), (2, 4094), (3, 130), (3, 2000), (4, 64), (4, 4096)])
def test_near_ties_are_told_apart_as_the_serial_scan_does(km, orc, gpu, dim, k):
    """Pairs of centroids, and points whose squared distances to both differ by 0 to some 1e-5 of themselves: on either side of what the
    fused sums decide by themselves."""
    rng = np.random.default_rng(dim * 7 + k)
    first = rng.uniform(0, 1, size=(k // 2, dim))
    apart = rng.normal(size=(k // 2, dim))
    apart *= 0.3 / k ** (1 / dim) / np.linalg.norm(apart, axis=1, keepdims=True)
    means = np.concatenate([first, first + apart]).astype(np.float32)
    n = 20001
    pair = rng.integers(0, k // 2, n)
    a, b = means[pair].astype(np.float64), means[pair + k // 2].astype(np.float64)
    off = rng.choice([0, 1e-7, 2e-7, 5e-7, 1e-6, 2e-6], n) * rng.uniform(-1, 1, n)
    rows = ((a + b) / 2 + (b - a) * off[:, None]).astype(np.float32)
    want = orc.assign(rows.ravel(), means.ravel(), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    m = km.DeviceBuffer(means.nbytes); m.write(means.ravel())
    out = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        km.assign(km.ASSIGN_MFMA_BF16X3, d, km.AOS, dim, m, km.AOS, dim, out, dim, k, n)
        km.sync()
    finally:
        km.set_two_level_sweep(1)
    got = out.read(np.uint32, n)
    d.free(); m.free(); out.free()
    assert np.array_equal(got, want), "%d mismatches" % int((got != want).sum())


@pytest.mark.parametrize("kind", ["planar", "outside", "lattice", "tiny", "huge", "nan"])
@pytest.mark.parametrize("dim,k", [(2, 600), (3, 6100), (4, 601), (4, 700)])   # (6100: streamed centroids; 600 and more: tracked per tile)
@pytest.mark.parametrize("layout,pad", [(0, 0), (0, 3), (1, 0)])
def test_points_the_cells_are_no_good_for_match_the_oracle(km, orc, gpu, dim, k, kind, layout, pad):
    """In the default mode such points are left to the packed sweep, whose queue goes to the exact pass of the cells."""
    n = (1 << 18) + 17
    rng = np.random.default_rng(dim * 41 + k)
    means = rng.normal(size=(k, dim)).astype(np.float32)
    rows = rng.normal(size=(n, dim)).astype(np.float32)
    if kind == "planar":      # no extent in one dimension: no grid
        means[:, dim - 1] = 0; rows[:, dim - 1] = 0
    else:                     # all points outside the grid
        rows[:, 0] += np.float32(20)
    if kind == "lattice":     # ties
        means, rows = (np.round(means * 4) / 4).astype(np.float32), (np.round(rows * 8) / 8).astype(np.float32)
    elif kind in ("tiny", "huge"):
        factor = np.float32(1e-17 if kind == "tiny" else 3e16)
        means *= factor; rows *= factor
    elif kind == "nan":
        means[k // 2, 0] = np.nan
    rows[3] = means[3]; rows[7, 0] = np.nan; rows[11, dim - 1] = np.inf; rows[13] = -1e30; rows[17] = 1e6; rows[19] = 1e-30
    sample = np.concatenate([np.arange(40), rng.choice(n, 30000, replace=False)])
    stride = dim + pad if layout == 0 else n
    padded = rows
    if pad:
        padded = np.full((n, stride), np.float32(np.nan)); padded[:, :dim] = rows
    d = km.DeviceBuffer(padded.nbytes); d.write(flat(padded, layout))
    m = km.DeviceBuffer(4 * k * dim); m.write(flat(means, 0))
    a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
    km.assign(km.ASSIGN_BEST, d, layout, stride, m, 0, dim, a, dim, k, n)
    km.sync()
    got = a.read(np.uint32, n)
    for b in (d, m, a):
        b.free()
    want = orc.assign(np.ascontiguousarray(rows[sample]).ravel(), means.ravel(), dim, k, len(sample), threads=0, fast=True)
    assert got.max() < k
    assert np.array_equal(got[sample], want), "%d of %d differ" % (int((got[sample] != want).sum()), len(sample))


@pytest.mark.parametrize("budget,limit", [(0, 1 << 20), (46 * 1024, 0), (64 * 1024, 1 << 20), (100 * 1024, 0)])
@pytest.mark.parametrize("layout", [0, 1])
def test_the_way_back_keeps_to_the_limits_of_the_caller(km, orc, gpu, budget, limit, layout):
    """Little LDS (centroids streamed behind the cells, or no cells at all) and a small block for copied rows."""
    dim, k, n = 4, 1500, (1 << 18) + 5
    rng = np.random.default_rng(budget + layout)
    means, rows = rng.normal(size=(k, dim)).astype(np.float32), rng.normal(size=(n, dim)).astype(np.float32)
    means[:, 3] = 0; rows[:, 3] = 0
    d, m, a = km.DeviceBuffer(rows.nbytes), km.DeviceBuffer(means.nbytes), km.DeviceBuffer(4 * n)
    d.write(flat(rows, layout)); m.write(flat(means, 0)); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
    if limit:
        km.set_queued_rows_limit(limit)
    try:
        km.assign(km.ASSIGN_BEST, d, layout, dim if layout == 0 else n, m, 0, dim, a, dim, k, n, km.ExecParams(shared_mem_bytes=budget))
        km.sync()
    finally:
        km.set_queued_rows_limit(1 << 30)
    got = a.read(np.uint32, n)
    for b in (d, m, a):
        b.free()
    sample = rng.choice(n, 30000, replace=False)
    want = orc.assign(np.ascontiguousarray(rows[sample]).ravel(), means.ravel(), dim, k, len(sample), threads=0, fast=True)
    assert np.array_equal(got[sample], want), "%d of %d differ" % (int((got[sample] != want).sum()), len(sample))


@pytest.mark.parametrize("kind", ["inside", "outside"])
def test_recorded_cells_replay(km, orc, gpu, kind):
    """Recorded right after a reservation, replayed with eager calls of another shape in between: the choice between cells and sweep is
    made anew in every replay, and no counter is left over."""
    dim, k, n = 4, 700, (1 << 18) + 5
    rng = np.random.default_rng(7)
    means = rng.random((k, dim), dtype=np.float32)
    rows = rng.random((n, dim), dtype=np.float32)
    far = (rows + np.float32(3)).astype(np.float32)
    d = km.DeviceBuffer(rows.nbytes); m = km.DeviceBuffer(means.nbytes); m.write(means.ravel())
    a = km.DeviceBuffer(4 * n)
    km.sync()
    km.check(km.hip_lib().kmx_shutdown())
    km.reserve(km.ASSIGN_BEST, km.UPDATE_ATOMIC_SHM, 0, 0, dim, k, n)
    with km.Graph() as g:
        km.assign(km.ASSIGN_BEST, d, 0, dim, m, 0, dim, a, dim, k, n)
    sample = rng.choice(n, 20000, replace=False)
    for turn in range(4):
        points = rows if (turn + (kind == "outside")) % 2 == 0 else far
        d.write(points.ravel())
        a.write(np.full(n, 0xFFFFFFF1, np.uint32))
        g.launch()
        km.sync()
        got = a.read(np.uint32, n)
        want = orc.assign(np.ascontiguousarray(points[sample]).ravel(), means.ravel(), dim, k, len(sample), threads=0, fast=True)
        assert got.max() < k and np.array_equal(got[sample], want), turn
        km.assign(km.ASSIGN_BEST, d, 0, 3, m, 0, 3, a, 3, 600, n)     # eager, another grid in the same buffers
        km.sync()
    g.destroy()
    for b in (d, m, a):
        b.free()


@pytest.mark.parametrize("dim", [2, 3, 4])
@pytest.mark.parametrize("k", [3, 64, 65, 66, 129, 1023, 1024, 1025, 1026, 2049, 6144])
def test_lists_of_every_length(km, orc, gpu, dim, k):
    """All centroids but one in one cell, whose list they all are on: 1 to 16 full turns of 64, one less and one more, the longest that is kept
    (1024 centroids) and the first that is not; and as many centroids as a thread of the building kernel has at most, and at the steps between. The rest of
    the cells have short lists, which no longer share a counter. The result is the serial scan's, bit for bit."""
    rng = np.random.default_rng(dim * 101 + k)
    means = (0.37 + rng.uniform(0, 1e-3, size=(k, dim))).astype(np.float32)
    means[rng.integers(0, k)] = 1.0
    n = 4099
    rows = np.where(rng.random((n, 1)) < 0.5, 0.37 + rng.uniform(-1e-3, 2e-3, size=(n, dim)), rng.uniform(0.2, 1.2, size=(n, dim))).astype(np.float32)
    want = orc.assign(rows.ravel(), means.ravel(), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    m = km.DeviceBuffer(means.nbytes)
    a = km.DeviceBuffer(4 * n)
    km.set_two_level_sweep(2)
    try:
        for layout in (0, 1):
            m.write(flat(means, layout))
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            km.assign(km.ASSIGN_MFMA_BF16X3, d, 0, dim, m, layout, km.layout_stride(layout, k, dim), a, dim, k, n)
            km.sync()
            assert np.array_equal(a.read(np.uint32, n), want)
    finally:
        km.set_two_level_sweep(1)
    for b in (d, m, a): b.free()
