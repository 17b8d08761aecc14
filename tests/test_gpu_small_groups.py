"""Small inputs (csrc/small.hip): work-groups of 32 points, of 16 wavefronts, and the sums in doubles, on both sides of every line between them, against the
serial oracle. The centroids' bound: per work-group one rounding of a sum in doubles, then at most 1024 partial sums added and one division."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,k", [(1, 2), (3, 12), (20, 13), (30, 128), (64, 64), (7, 585)])
@pytest.mark.parametrize("n", [31, 33, 8191, 8192, 8193, 12289, 20000, 20001])
@pytest.mark.parametrize("layout", [0, 1])
def test_both_sides_of_the_lines(km, orc, gpu, dim, k, n, layout):
    if n < k:
        pytest.skip("fewer points than centroids")
    rng = np.random.default_rng(dim + n)
    rows = np.round(rng.normal(size=(n, dim)) * 4).astype(np.float32) / np.float32(4)      # a coarse grid: ties
    rows[::3] += rng.normal(size=rows[::3].shape).astype(np.float32)
    means = rows[rng.permutation(n)[:k]].copy()
    flat = lambda v: np.ascontiguousarray(v if layout == 0 else v.T).ravel()
    s, sm = km.layout_stride(layout, n, dim), km.layout_stride(layout, k, dim)
    for dtype in (np.float32, np.float64):
        item = np.dtype(dtype).itemsize
        fn = orc.assign if dtype == np.float32 else orc.assign_f64
        want = fn(rows.astype(dtype).ravel(), means.astype(dtype).ravel(), dim, k, n, threads=0)
        d = km.DeviceBuffer(item * n * dim); d.write(flat(rows.astype(dtype)))
        m = km.DeviceBuffer(item * k * dim); m.write(flat(means.astype(dtype)))
        a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
        km.assign(km.ASSIGN_BEST, d, layout, s, m, layout, sm, a, dim, k, n, None, dtype)
        km.sync()
        assert np.array_equal(a.read(np.uint32, n), want)
        if dtype == np.float32:
            a.write(np.full(n, 0xFFFFFFF1, np.uint32))
            out = km.DeviceBuffer(4 * k * dim); out.write(np.full(k * dim, 0x7FC54321, np.uint32))
            sizes = km.DeviceBuffer(4 * k); sizes.write(np.full(k, 7, np.uint32))
            km.iteration(d, layout, s, m, out, layout, sm, a, sizes, dim, k, n)
            km.sync()
            assert np.array_equal(a.read(np.uint32, n), want)
            counts = np.bincount(want, minlength=k)
            assert np.array_equal(sizes.read(np.uint32, k), counts)
            total, size = np.zeros((k, dim)), np.zeros((k, dim))
            np.add.at(total, want, rows.astype(np.float64))
            np.add.at(size, want, np.abs(rows).astype(np.float64))
            got = out.read(np.float32, k * dim)
            got = got.reshape(k, dim) if layout == 0 else got.reshape(dim, k).T
            div = np.maximum(counts, 1)[:, None]
            assert np.all(np.abs(got - total / div) <= 1026 * 2.0 ** -24 * size / div)
            out.free(); sizes.free()
        for b in (d, m, a):
            b.free()


@pytest.mark.parametrize("dim,k", [(196, 128), (197, 132), (200, 64), (204, 100), (204, 32), (205, 28), (237, 16), (250, 14), (252, 12), (256, 14)])
@pytest.mark.parametrize("n", [8192, 8193, 10000, 16384, 16385])
def test_wide_rows_beside_what_lds_holds(km, orc, gpu, dim, k, n):
    """Rows of around 200 doubles, where 16 wavefronts' candidates do not fit beside them."""
    for layout in (0, 1):
        test_both_sides_of_the_lines(km, orc, gpu, dim, k, n, layout)


@pytest.mark.parametrize("budget", [48 * 1024, 72 * 1024, 100 * 1024])
@pytest.mark.parametrize("dim,k", [(20, 13), (48, 64), (64, 64), (100, 40)])
def test_small_inputs_under_a_callers_budget(km, orc, gpu, dim, k, budget):
    n = 10000
    rng = np.random.default_rng(dim + budget)
    rows = np.round(rng.normal(size=(n, dim)) * 4) / 4
    means = rows[rng.permutation(n)[:k]].copy()
    execution = km.ExecParams()
    execution.shared_mem_bytes = budget
    for dtype, fn in ((np.float32, orc.assign), (np.float64, orc.assign_f64)):
        item = np.dtype(dtype).itemsize
        want = fn(rows.astype(dtype).ravel(), means.astype(dtype).ravel(), dim, k, n, threads=0)
        d = km.DeviceBuffer(item * n * dim); d.write(rows.astype(dtype).ravel())
        m = km.DeviceBuffer(item * k * dim); m.write(means.astype(dtype).ravel())
        a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
        km.assign(km.ASSIGN_BEST, d, 0, dim, m, 0, dim, a, dim, k, n, execution, dtype)
        km.sync()
        assert np.array_equal(a.read(np.uint32, n), want)
        for b in (d, m, a):
            b.free()


@pytest.mark.parametrize("dim,k,n", [(220, 15, 24497), (221, 15, 16385), (208, 16, 38139), (252, 12, 25494), (187, 3, 48841), (164, 12, 34223), (255, 14, 32700), (136, 4, 60177)])
def test_sums_in_parts_of_the_coordinates(km, orc, gpu, dim, k, n):
    """Whole sums would take a round of work-groups more (small_shape)."""
    for layout in (0, 1):
        test_both_sides_of_the_lines(km, orc, gpu, dim, k, n, layout)
