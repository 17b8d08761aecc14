"""The serial-order update for clusters of many members (ordered_staged_sum_kernel, csrc/update_ordered.hip): the bits of one
addition after the other, at the edges of its blocks of coordinates, pieces and fetches (-m gpu)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k", [(1, 3), (2, 40), (3, 20), (4, 9), (5, 33), (16, 2), (17, 12), (31, 5), (33, 7), (35, 6), (64, 4), (65, 3), (130, 2)])
def test_staged_sums_have_the_bits_of_the_serial_loop(km, gpu, dim, k, dtype):
    rng = np.random.default_rng(dim + 100 * k)
    sizes = [0, 1, 3, 4, 15, 16, 17, 255, 256, 257, 1024, 4097, 9000][:k] + [90] * max(0, k - 13)
    sizes[-1] += max(0, 600 * k - sum(sizes))  # well over 512 members on average, most of them in one cluster
    which = rng.permutation(np.repeat(np.arange(k), sizes)).astype(np.uint32)
    n = len(which)
    which[5:n:97] = k  # not a cluster: left out
    rows = (rng.normal(size=(n, dim)) * np.exp(rng.normal(size=(n, 1)) * 4)).astype(dtype)
    want = np.zeros((k, dim), dtype)
    counts = np.zeros(k, np.uint32)
    for c in range(k):
        members = rows[which == c]
        counts[c] = len(members)
        if len(members):  # cumsum adds one after the other (numpy's sum does not)
            want[c] = np.cumsum(np.concatenate([np.zeros((1, dim), dtype), members]), axis=0, dtype=dtype)[-1] / dtype(len(members))
    size = np.dtype(dtype).itemsize
    a = km.DeviceBuffer(4 * n); a.write(which)
    m = km.DeviceBuffer(size * k * dim); s = km.DeviceBuffer(4 * k)
    for layout, pad in [(0, 0), (0, 3), (1, 0)]:
        stride = dim + pad if layout == 0 else n
        data = np.full((n, stride), np.nan, dtype) if layout == 0 else rows.T
        if layout == 0:
            data[:, :dim] = rows
        data = np.ascontiguousarray(data).ravel()
        d = km.DeviceBuffer(data.nbytes); d.write(data)
        for layout_means in (0, 1):
            km.update(km.UPDATE_SERIAL_ORDER, d, layout, stride, a, m, layout_means, km.layout_stride(layout_means, k, dim), s, dim, k, n, dtype=dtype)
            km.sync()
            got = m.read(dtype, k * dim)
            got = got.reshape(k, dim) if layout_means == 0 else got.reshape(dim, k).T
            assert np.array_equal(s.read(np.uint32, k), counts)
            assert np.array_equal(got, want), "layouts %d/%d: %d differ" % (layout, layout_means, int((got != want).sum()))
        d.free()
    a.free(); m.free(); s.free()


@pytest.mark.parametrize("dtype,dim", [(np.float32, d) for d in (4, 8, 12, 16, 20, 24, 28, 32, 36, 64, 100)] + [(np.float64, d) for d in (2, 6, 10, 14, 16, 18, 50)])
@pytest.mark.parametrize("k", [5, 600])
def test_streamed_sums_have_the_bits_of_the_serial_loop(km, gpu, dim, k, dtype):
    """Rows of whole 16-byte pieces (ordered_stream_sum_kernel): clusters at the edges of requests, of batches and of what is requested
    at once, few chains (more of them ahead) and many."""
    rng = np.random.default_rng(dim + k)
    rows_of = 64 // min(8, dim * np.dtype(dtype).itemsize // 16)  # of a request; a batch is eight, three to six batches travel ahead
    edges = [0, 1, rows_of - 1, rows_of, rows_of + 1] + [8 * rows_of * b + o for b in (1, 3, 4, 6, 7) for o in (-1, 0, 1)]
    sizes = (edges if k > 5 else [0, 3 * rows_of + 1, 24 * rows_of, 48 * rows_of + 1, 130 * rows_of + 7])
    sizes = sizes + [140] * (k - len(sizes))
    which = rng.permutation(np.repeat(np.arange(k), sizes)).astype(np.uint32)
    n = len(which)
    which[5:n:97] = k  # not a cluster: left out
    rows = (rng.normal(size=(n, dim)) * np.exp(rng.normal(size=(n, 1)) * 4)).astype(dtype)
    want = np.zeros((k, dim), dtype)
    order = np.argsort(which, kind="stable")
    ends = np.cumsum(np.bincount(which, minlength=k + 1))
    for c in range(k):
        members = rows[order[ends[c - 1] if c else 0:ends[c]]]
        if len(members):
            want[c] = np.cumsum(np.concatenate([np.zeros((1, dim), dtype), members]), axis=0, dtype=dtype)[-1] / dtype(len(members))
    size = np.dtype(dtype).itemsize
    a = km.DeviceBuffer(4 * n); a.write(which)
    m = km.DeviceBuffer(size * k * dim); s = km.DeviceBuffer(4 * k)
    for pad, layout_means in [(0, 0), (16 // size, 1)]:
        data = np.full((n, dim + pad), np.nan, dtype)
        data[:, :dim] = rows
        d = km.DeviceBuffer(data.nbytes); d.write(data.ravel())
        km.update(km.UPDATE_SERIAL_ORDER, d, 0, dim + pad, a, m, layout_means, km.layout_stride(layout_means, k, dim), s, dim, k, n, dtype=dtype)
        km.sync()
        got = m.read(dtype, k * dim)
        got = got.reshape(k, dim) if layout_means == 0 else got.reshape(dim, k).T
        d.free()
        assert np.array_equal(s.read(np.uint32, k), np.bincount(which[which < k], minlength=k))
        assert np.array_equal(got, want), "pad %d: %d differ" % (pad, int((got != want).sum()))
    a.free(); m.free(); s.free()


@pytest.mark.parametrize("k,n", [(1, 1), (1, 5000), (2, 63), (7, 513), (2048, 9001), (2049, 9001), (4096, 20003), (4097, 20003), (16384, 40001), (16385, 40001), (1000, 300007)])
def test_members_are_added_in_point_order(km, gpu, k, n):
    """The stable sort by work-groups of eight, four and one wavefronts, counters in LDS and in memory."""
    rng = np.random.default_rng(k + n)
    which = np.minimum(rng.integers(0, k + 1, n), rng.integers(0, k + 1, n)).astype(np.uint32)  # (k: not a cluster)
    rows = (rng.normal(size=(n, 4)) * np.exp(rng.normal(size=(n, 1)) * 4)).astype(np.float32)
    want = np.zeros((k, 4), np.float32)
    for i in np.flatnonzero(which < k) if n < 50000 else []:
        want[which[i]] += rows[i]
    if n >= 50000:
        for c in range(k):
            want[c] = np.cumsum(np.concatenate([np.zeros((1, 4), np.float32), rows[which == c]]), axis=0, dtype=np.float32)[-1]
    counts = np.bincount(which[which < k], minlength=k)
    want = np.where(counts[:, None] > 0, want / np.maximum(counts, 1)[:, None].astype(np.float32), np.float32(0))
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    a = km.DeviceBuffer(4 * n); a.write(which)
    m = km.DeviceBuffer(16 * k); s = km.DeviceBuffer(4 * k)
    km.update(km.UPDATE_SERIAL_ORDER, d, 0, 4, a, m, 0, 4, s, 4, k, n)
    km.sync()
    assert np.array_equal(s.read(np.uint32, k), counts)
    assert np.array_equal(m.read(np.float32, 4 * k).reshape(k, 4), want)
    for b in (d, a, m, s):
        b.free()


@pytest.mark.parametrize("dtype,dim,k,members", [(np.float32, 100, 1600, 33), (np.float32, 260, 700, 33), (np.float32, 8, 6200, 130), (np.float32, 64, 3100, 60),
                                                (np.float64, 50, 1600, 40), (np.float64, 16, 6200, 33)])
@pytest.mark.parametrize("large", [(), (255, 256, 257, 0, 5000)])
def test_small_clusters_beside_large_ones_have_the_bits_of_the_serial_loop(km, gpu, dtype, dim, k, members, large):
    """Small clusters in many blocks: a lane per chain, and the clusters of 256 members and more streamed (ORDERED_SPLIT)."""
    rng = np.random.default_rng(dim + k)
    sizes = np.full(k, members)
    sizes[rng.choice(k, len(large), replace=False)] = large
    sizes[-1] = max(1, sizes[-1] - max(0, int(sizes.sum()) - (256 * k - 1)))   # fewer than 256 on average
    which = rng.permutation(np.repeat(np.arange(k), sizes)).astype(np.uint32)
    n = len(which)
    which[5:n:197] = k  # not a cluster: left out
    rows = (rng.normal(size=(n, dim)) * np.exp(rng.normal(size=(n, 1)) * 4)).astype(dtype)
    want = np.zeros((k, dim), dtype)
    order = np.argsort(which, kind="stable")
    ends = np.cumsum(np.bincount(which, minlength=k + 1))
    for c in range(k):
        mine = rows[order[ends[c - 1] if c else 0:ends[c]]]
        if len(mine):
            want[c] = np.cumsum(np.concatenate([np.zeros((1, dim), dtype), mine]), axis=0, dtype=dtype)[-1] / dtype(len(mine))
    size = np.dtype(dtype).itemsize
    a = km.DeviceBuffer(4 * n); a.write(which)
    m = km.DeviceBuffer(size * k * dim); s = km.DeviceBuffer(4 * k)
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    for layout_means in (0, 1):
        m.write(np.full(size * k * dim // 4, 0x7FC54321, np.uint32))
        km.update(km.UPDATE_SERIAL_ORDER, d, 0, dim, a, m, layout_means, km.layout_stride(layout_means, k, dim), s, dim, k, n, dtype=dtype)
        km.sync()
        got = m.read(dtype, k * dim)
        got = got.reshape(k, dim) if layout_means == 0 else got.reshape(dim, k).T
        assert np.array_equal(s.read(np.uint32, k), np.bincount(which[which < k], minlength=k))
        assert np.array_equal(got, want), "means %d: %d differ" % (layout_means, int((got != want).sum()))
    for b in (d, a, m, s):
        b.free()


@pytest.mark.parametrize("dim,k,n", [(512, 3000, 100000), (128, 8000, 300000)])
def test_small_clusters_of_wide_rows_take_no_work_group_each(km, gpu, dim, k, n):
    """Beside the same rows a word off the 16-byte pieces, which the lane-per-chain kernel adds up whatever their number: rows of whole pieces
    take no longer (0.9 to 1 times; it was 1.4 to 1.8 times while every cluster and block of a row had a work-group)."""
    rng = np.random.default_rng(dim)
    a = km.DeviceBuffer(4 * n); a.write(rng.integers(0, k, n).astype(np.uint32))
    m = km.DeviceBuffer(4 * k * dim); s = km.DeviceBuffer(4 * k)
    start, stop = km.Event(), km.Event()
    took = []
    for stride in (dim, dim + 1):
        d = km.DeviceBuffer(4 * n * stride); d.write(rng.random(n * stride, dtype=np.float32))
        times = []
        for series in range(7):
            start.record()
            for _ in range(10):
                km.update(km.UPDATE_SERIAL_ORDER, d, 0, stride, a, m, 0, dim, s, dim, k, n)
            stop.record()
            km.sync()
            times.append(start.elapsed_ms(stop) * 100)
        took.append(float(np.median(times[1:])))
        d.free()
    for b in (a, m, s):
        b.free()
    print("whole pieces %.1f us, others %.1f us" % tuple(took))
    assert took[0] <= 1.15 * took[1], "whole pieces %.1f us, others %.1f us" % tuple(took)
