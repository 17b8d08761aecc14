"""Small inputs (csrc/small.hip): assignment, iteration and update in one launch each, at the edges of their tiles and ranges, floats
and doubles, both layouts, against the serial oracle (-m gpu)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def flat(rows, layout):
    return np.ascontiguousarray(rows if layout == 0 else rows.T).ravel()


def unflat(values, layout, count, dim):
    return values.reshape(count, dim) if layout == 0 else values.reshape(dim, count).T


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k,n", [(1, 1, 1), (1, 12, 63), (4, 13, 64), (5, 33, 65), (17, 64, 129), (20, 128, 1000), (64, 64, 640),
                                     (65, 63, 333), (256, 5, 200), (255, 40, 130), (3, 1365, 5461), (2, 300, 32769)])
@pytest.mark.parametrize("layout,layout_means", [(0, 0), (1, 1), (0, 1), (1, 0)])
def test_small_assignment_and_iteration(km, orc, gpu, dtype, dim, k, n, layout, layout_means):
    rng = np.random.default_rng(dim * 7 + k)
    rows = np.round(rng.normal(size=(n, dim)) * 4).astype(dtype) / dtype(4)      # a coarse grid: exact ties
    rows[::3] += rng.normal(size=rows[::3].shape).astype(dtype)
    means = rows[rng.integers(0, n, k)].copy()
    if n > 40 and dtype == np.float32:
        rows[17, 0], rows[33, dim - 1] = np.inf, np.nan
    fn = orc.assign if dtype == np.float32 else orc.assign_f64
    want = fn(flat(rows, 0), flat(means, 0), dim, k, n, threads=0) if dtype == np.float64 else fn(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    item = np.dtype(dtype).itemsize
    d = km.DeviceBuffer(item * n * dim); d.write(flat(rows, layout))
    m = km.DeviceBuffer(item * k * dim); m.write(flat(means, layout_means))
    a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
    s, sm = km.layout_stride(layout, n, dim), km.layout_stride(layout_means, k, dim)
    km.assign(km.ASSIGN_BEST, d, layout, s, m, layout_means, sm, a, dim, k, n, None, dtype)
    km.sync()
    assert np.array_equal(a.read(np.uint32, n), want)
    if dtype == np.float32:
        out = km.DeviceBuffer(4 * k * dim); out.write(np.full(k * dim, 0x7FC54321, np.uint32))
        sizes = km.DeviceBuffer(4 * k); sizes.write(np.full(k, 7, np.uint32))
        a.write(np.full(n, 0xFFFFFFF1, np.uint32))
        km.iteration(d, layout, s, m, out, layout_means, sm, a, sizes, dim, k, n)
        km.sync()
        assert np.array_equal(a.read(np.uint32, n), want)
        counts = np.bincount(want, minlength=k)
        assert np.array_equal(sizes.read(np.uint32, k), counts)
        got = unflat(out.read(np.float32, k * dim), layout_means, k, dim)
        sums = np.zeros((k, dim)); np.add.at(sums, want, rows.astype(np.float64))
        truth = np.where(counts[:, None] > 0, sums / np.maximum(counts, 1)[:, None], 0.0)
        clean = np.isfinite(truth)                       # what an infinity or a NaN among the points must not reach
        assert np.array_equal(np.isfinite(got), clean)
        assert np.abs(got[clean] - truth[clean]).max() < 1e-4 * max(1.0, np.abs(truth[clean]).max())
        out.free(); sizes.free()
    for b in (d, m, a):
        b.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k,n", [(128, 64, 64), (132, 62, 65), (64, 128, 100), (64, 129, 100),   # 2048 pieces of four coordinates travel together, then more
                                     (31, 66, 70), (32, 64, 64), (33, 65, 70), (127, 17, 64)])       # 2048 coordinates, or 32 columns of 64 rows
@pytest.mark.parametrize("layout,layout_means", [(0, 0), (1, 1), (0, 1)])
def test_small_staging_at_the_edges_of_its_batches(km, orc, gpu, dtype, dim, k, n, layout, layout_means):
    test_small_assignment_and_iteration(km, orc, gpu, dtype, dim, k, n, layout, layout_means)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k,n", [(1, 1, 1), (3, 2, 4095), (4, 256, 4096), (5, 257, 4097), (20, 128, 12288), (9, 600, 12289), (2, 4096, 32768), (300, 40, 700)])
@pytest.mark.parametrize("layout,layout_means", [(0, 0), (1, 1)])
@pytest.mark.parametrize("kind", ["uniform", "hot"])
def test_small_update(km, gpu, dtype, dim, k, n, layout, layout_means, kind):
    rng = np.random.default_rng(dim + k)
    rows = rng.normal(size=(n, dim)).astype(dtype)
    asg = rng.integers(0, k, n).astype(np.uint32)
    if kind == "hot":
        asg[rng.random(n) < 0.9] = k - 1
    outside = rng.random(n) < 0.01
    asg[outside] = k + 5                                 # belongs to no cluster
    item = np.dtype(dtype).itemsize
    d = km.DeviceBuffer(item * n * dim); d.write(flat(rows, layout))
    a = km.DeviceBuffer(4 * n); a.write(asg)
    m = km.DeviceBuffer(item * k * dim); m.zero()
    sizes = km.DeviceBuffer(4 * k); sizes.zero()
    km.update(km.UPDATE_ATOMIC_SHM, d, layout, km.layout_stride(layout, n, dim), a, m, layout_means, km.layout_stride(layout_means, k, dim), sizes,
              dim, k, n, None, dtype)
    km.sync()
    counts = np.bincount(asg[~outside], minlength=k)
    assert np.array_equal(sizes.read(np.uint32, k), counts)
    sums = np.zeros((k, dim)); np.add.at(sums, asg[~outside], rows[~outside].astype(np.float64))
    truth = np.where(counts[:, None] > 0, sums / np.maximum(counts, 1)[:, None], 0.0)
    got = unflat(m.read(dtype, k * dim), layout_means, k, dim)
    assert np.abs(got - truth).max() < (1e-5 if dtype == np.float32 else 1e-13) * max(1.0, np.abs(truth).max())
    for b in (d, a, m, sizes):
        b.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k,n", [(1, 600, 700), (3, 130, 140), (7, 200, 210), (8, 129, 140), (9, 128, 140), (15, 193, 200), (16, 193, 200), (17, 65, 70),   # blocks of 64 rows
                                     (49, 130, 140), (50, 63, 70)])   # six single coordinates a lane at a time, eight columns a wavefront
@pytest.mark.parametrize("layout,layout_means", [(0, 0), (1, 1), (1, 0)])
def test_small_staging_of_columns_and_single_coordinates(km, orc, gpu, dtype, dim, k, n, layout, layout_means):
    test_small_assignment_and_iteration(km, orc, gpu, dtype, dim, k, n, layout, layout_means)


@pytest.mark.parametrize("dim,k,n", [(252, 2, 3895), (100, 5, 3750)])
def test_columns_cost_little_more_than_rows(km, gpu, dim, k, n):
    """Points and centroids in columns beside the same in rows: staging them costs the same number of trips to memory (1.1 to 1.2
    times the rows' call; it was 1.5 to 1.9 times while columns went in batches of four with branches between the loads)."""
    rng = np.random.default_rng(dim)
    rows, means = rng.normal(size=(n, dim)).astype(np.float32), rng.normal(size=(k, dim)).astype(np.float32)
    a = km.DeviceBuffer(4 * n)
    start, stop = km.Event(), km.Event()
    took = []
    for layout in (0, 1):
        d = km.DeviceBuffer(rows.nbytes); d.write(np.ascontiguousarray(rows if layout == 0 else rows.T).ravel())
        m = km.DeviceBuffer(means.nbytes); m.write(np.ascontiguousarray(means if layout == 0 else means.T).ravel())
        times = []
        for series in range(9):
            start.record()
            for _ in range(100):
                km.assign(km.ASSIGN_BEST, d, layout, km.layout_stride(layout, n, dim), m, layout, km.layout_stride(layout, k, dim), a, dim, k, n)
            stop.record()
            km.sync()
            times.append(start.elapsed_ms(stop) * 10)
        took.append(float(np.median(times[1:])))
        d.free(); m.free()
    a.free()
    print("rows %.2f us, columns %.2f us" % tuple(took))
    assert took[1] <= 1.4 * took[0], "rows %.2f us, columns %.2f us" % tuple(took)
