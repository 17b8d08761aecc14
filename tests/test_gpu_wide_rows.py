"""Rows of more than 256 dimensions (csrc/assign_wide.hip) against the serial oracle, bit for bit: one half-precision product and
three bf16 products, both unit sizes, one and several groups of centroids, rows kept in LDS and rows staged again, ragged ends
everywhere (-m gpu)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def flat(rows, layout):
    return np.ascontiguousarray(rows if layout == 0 else rows.T).ravel()


@pytest.mark.parametrize("kind", ["clustered", "grid", "offset"])
@pytest.mark.parametrize("dim,k,n", [
    (257, 1, 1), (300, 5, 31), (320, 33, 130), (511, 400, 700), (257, 290, 1500),   # units of 32 points
    (384, 520, 16500), (512, 545, 16384), (515, 100, 16421),                         # units of 128; groups of 512; resident rows
    (1030, 600, 16400), (2560, 40, 300),                                             # rows staged again per group; the widest
    (300, 40, 33000),                                                                # units of 128 points, two tiles
])
def test_wide_rows_match_the_oracle(km, orc, gpu, dim, k, n, kind):
    rng = np.random.default_rng(dim * 31 + k)
    centres = rng.uniform(-3, 3, size=(k, dim)).astype(np.float32)
    rows = (centres[rng.integers(0, k, n)] + rng.normal(size=(n, dim))).astype(np.float32)
    means = (centres + rng.normal(size=(k, dim)) * 0.3).astype(np.float32)
    if kind == "grid":       # many exact ties: duplicated centroids, points on bisectors
        rows, means = np.round(rows * 0.5).astype(np.float32), np.round(means * 0.5).astype(np.float32)
        means[k // 2:] = means[:k - k // 2]
    elif kind == "offset":
        rows, means = (rows + np.float32(1000)).astype(np.float32), (means + np.float32(1000)).astype(np.float32)
    if n > 20:
        rows[7, 3] = np.nan
        rows[11, dim - 1] = np.inf
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    a = km.DeviceBuffer(4 * n)
    for layout, layout_means, pad in [(0, 0, 0), (0, 1, 5), (1, 0, 0)]:
        stride = dim + pad if layout == 0 else n
        if pad:
            padded = np.full((n, stride), np.float32(np.nan)); padded[:, :dim] = rows
        else:
            padded = rows
        d = km.DeviceBuffer(padded.nbytes); d.write(flat(padded, layout))
        m = km.DeviceBuffer(4 * k * dim); m.write(flat(means, layout_means))
        for mode in (0, 1, 2):  # three bf16 products; one half-precision product (rows of up to 2304 dimensions), the same
            km.set_two_level_sweep(mode)
            try:
                a.write(np.full(n, 0xFFFFFFF1, np.uint32))
                km.assign(km.ASSIGN_BEST, d, layout, stride, m, layout_means, km.layout_stride(layout_means, k, dim), a, dim, k, n)
                km.sync()
            finally:
                km.set_two_level_sweep(1)
            got = a.read(np.uint32, n)
            assert km.last_assign_variant() == km.ASSIGN_MFMA_BF16X3
            assert np.array_equal(got, want), "layouts %d/%d, mode %d: %d mismatches" % (layout, layout_means, mode, int((got != want).sum()))
        d.free(); m.free()
    a.free()


@pytest.mark.parametrize("dim,k,n", [(300, 40, 9000), (257, 300, 8225),    # units of 32 points, one and several groups
                                     (320, 520, 33000), (1030, 600, 32800), (300, 3, 66000)])   # of 128: resident, staged again, one tile
@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("layout", [0, 1])
def test_units_that_follow_one_another_match_the_oracle(km, orc, gpu, dim, k, n, mode, layout):
    """More units than work-groups: the first chunk of a work-group's next unit is staged during the last step of the one before."""
    rng = np.random.default_rng(dim + k)
    centres = rng.uniform(-3, 3, size=(k, dim)).astype(np.float32)
    rows = (centres[rng.integers(0, k, n)] + rng.normal(size=(n, dim))).astype(np.float32)
    want = orc.assign(flat(rows, 0), flat(centres, 0), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, layout))
    m = km.DeviceBuffer(centres.nbytes); m.write(flat(centres, layout))
    a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
    km.set_two_level_sweep(mode)
    try:
        km.assign(km.ASSIGN_BEST, d, layout, km.layout_stride(layout, n, dim), m, layout, km.layout_stride(layout, k, dim), a, dim, k, n)
        km.sync()
    finally:
        km.set_two_level_sweep(1)
    got = a.read(np.uint32, n)
    d.free(); m.free(); a.free()
    assert np.array_equal(got, want), "%d mismatches" % int((got != want).sum())


@pytest.mark.parametrize("budget,variant,blocks", [
    (0, "MFMA_BF16X3", 129),           # 129 units of 128 points
    (54 * 1024, "MFMA_BF16X3", 256),   # too little for those: units of 32
    (31 * 1024, "MFMA_BF16X3", 256),   # too little for the half-precision exact pass: three products
    (16 * 1024, "BASE", None),         # no sweep fits
])
def test_wide_rows_keep_to_the_lds_budget(km, orc, gpu, budget, variant, blocks):
    dim, k, n = 512, 40, 16400
    rng = np.random.default_rng(budget)
    rows = rng.normal(size=(n, dim)).astype(np.float32)
    means = np.ascontiguousarray(rows[rng.choice(n, k, replace=False)])
    want = orc.assign(flat(rows, 0), flat(means, 0), dim, k, n, threads=0, fast=True)
    d = km.DeviceBuffer(rows.nbytes); d.write(flat(rows, 0))
    m = km.DeviceBuffer(means.nbytes); m.write(flat(means, 0))
    a = km.DeviceBuffer(4 * n); a.write(np.full(n, 0xFFFFFFF1, np.uint32))
    ex = km.ExecParams(shared_mem_bytes=budget)
    km.assign(km.ASSIGN_BEST, d, 0, dim, m, 0, dim, a, dim, k, n, ex)
    km.sync()
    assert km.last_assign_variant() == getattr(km, "ASSIGN_" + variant)
    assert blocks is None or ex.block_count == min(blocks, gpu.compute_units)
    assert np.array_equal(a.read(np.uint32, n), want)
    if variant == "BASE":
        with pytest.raises(km.KmxError, match="LDS budget"):
            km.assign(km.ASSIGN_MFMA_BF16X3, d, 0, dim, m, 0, dim, a, dim, k, n, km.ExecParams(shared_mem_bytes=budget))
    for b in (d, m, a):
        b.free()
