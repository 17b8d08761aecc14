"""The update whose sums lie in LDS as doubles (csrc/update_sums64.hip): every number of lanes per row, whole and partly filled slices, ends of chunks and
steps, copies of the sums, members of no cluster, against sums in 64 bits.

The bound: a chunk's sums are exact to a double's rounding and rounded to the result's type once, then at most 256 chunks are added one after the other and the
sum is divided: 258 roundings of at most the sum of the magnitudes (doubles: one more per member)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
AOS, SOA = 0, 1


def check(km, dim, k, n, dtype, stride=None, layout_means=AOS, outside=False, one=False, seed=0, layout=AOS, by_cluster=False):
    rng = np.random.default_rng(seed + 1000 * dim + k)
    stride = stride or dim
    rows = np.full((n, stride), np.nan, dtype)
    rows[:, :dim] = rng.normal(size=(n, dim)) * np.exp2(rng.integers(-20, 20, size=dim))
    member = rng.integers(0, k + (2 if outside else 0), size=n).astype(np.uint32)
    if one:
        member[:] = k - 1
    member[-1] = k - 1
    if by_cluster:
        member.sort()
    stored = rows if layout == AOS else np.ascontiguousarray(rows[:, :dim].T)
    d = km.DeviceBuffer(stored.nbytes); d.write(stored.ravel())
    a = km.DeviceBuffer(4 * n); a.write(member)
    stride_means = dim if layout_means == AOS else k
    m = km.DeviceBuffer(rows.itemsize * k * dim); s = km.DeviceBuffer(4 * k)
    m.zero(); s.zero()
    km.update(km.UPDATE_ATOMIC_SHM, d, layout, stride if layout == AOS else n, a, m, layout_means, stride_means, s, dim, k, n, None, dtype)
    got = m.read(dtype, k * dim)
    got = got.reshape(k, dim) if layout_means == AOS else got.reshape(dim, k).T
    sizes = s.read(np.uint32, k)
    for b in (d, a, m, s):
        b.free()
    inside = member < k
    want_sizes = np.bincount(member[inside], minlength=k)
    assert np.array_equal(sizes, want_sizes)
    x = rows[inside, :dim].astype(np.longdouble)
    total, size = np.zeros((k, dim), np.longdouble), np.zeros((k, dim), np.longdouble)
    np.add.at(total, member[inside], x)
    np.add.at(size, member[inside], np.abs(x))
    count = np.maximum(want_sizes, 1)[:, None]
    unit = np.finfo(dtype).eps / 2
    roundings = 258 + (count if dtype is np.float64 else 0)
    assert np.all(np.abs(got - total / count) <= roundings * unit * size / count)


# rows of every number of lanes, full and not; 300 clusters of up to 64 coordinates as a whole, 1024 in slices; a chunk is 512 or k points and more
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k", [(1, 70), (2, 70), (3, 70), (4, 70), (5, 70), (8, 70), (9, 70), (16, 70), (17, 70), (32, 70), (33, 70), (63, 70), (64, 70), (65, 70), (100, 70), (128, 70), (300, 20), (640, 20), (641, 20),
                                   (16, 1200), (24, 1200), (32, 1024), (36, 1200), (48, 1024), (56, 1200), (80, 900), (100, 1000), (36, 2500), (4, 4500), (12, 4200), (13, 13000)])
def test_sums_of_every_width(km, gpu, dim, k, dtype):
    for n in (20011, 70003):
        check(km, dim, k, n, dtype, outside=n == 20011)


@pytest.mark.parametrize("dim,k", [(1, 2), (2, 2), (4, 3), (7, 2), (16, 4), (30, 5), (64, 2)])
@pytest.mark.parametrize("n", [16384, 40961, 262144 + 65])
def test_few_clusters(km, gpu, dim, k, n):
    check(km, dim, k, n, np.float32)
    check(km, dim, k, n, np.float32, one=True, seed=1)
    check(km, dim, k, n, np.float64, one=True, seed=2)


@pytest.mark.parametrize("dim,stride", [(5, 9), (16, 19), (33, 40), (50, 56), (96, 101)])
def test_padded_rows_and_centroids_by_columns(km, gpu, dim, stride):
    check(km, dim, 200, 50021, np.float32, stride=stride, layout_means=SOA)
    check(km, dim, 200, 50021, np.float64, stride=stride, layout_means=SOA)


def test_infinities_stay_in_their_cluster(km, gpu):
    dim, k, n = 20, 300, 60000
    rng = np.random.default_rng(1)
    rows = rng.normal(size=(n, dim)).astype(np.float32)
    member = (np.arange(n) % k).astype(np.uint32)
    rows[7, 3], rows[8, 19], rows[9, 0], rows[9 + k, 0] = np.inf, np.nan, np.inf, -np.inf
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    a = km.DeviceBuffer(4 * n); a.write(member)
    m = km.DeviceBuffer(4 * k * dim); s = km.DeviceBuffer(4 * k)
    km.update(km.UPDATE_ATOMIC_SHM, d, AOS, dim, a, m, AOS, dim, s, dim, k, n)
    got = m.read(np.float32, k * dim).reshape(k, dim)
    assert np.isinf(got[7, 3]) and np.isnan(got[8, 19]) and np.isnan(got[9, 0])
    odd = np.zeros((k, dim), bool)
    odd[7, 3] = odd[8, 19] = odd[9, 0] = True
    assert np.all(np.isfinite(got[~odd]))
    for b in (d, a, m, s):
        b.free()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_recorded_without_room_for_partial_sums(km, gpu, dtype):
    """Nothing is allocated while a graph is recorded: kernels without partial sums take the call, and every replay gives their result."""
    dim, k, n = 16, 16, 1 << 16
    rng = np.random.default_rng(2)
    rows = rng.normal(size=(n, dim)).astype(dtype)
    member = rng.integers(0, k, size=n).astype(np.uint32)
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    a = km.DeviceBuffer(4 * n); a.write(member)
    m = km.DeviceBuffer(rows.itemsize * k * dim); s = km.DeviceBuffer(4 * k)
    update = lambda n: km.update(km.UPDATE_ATOMIC_SHM, d, AOS, dim, a, m, AOS, dim, s, dim, k, n, None, dtype)
    km.sync()
    km.check(km.hip_lib().kmx_shutdown())
    if dtype == np.float32:
        update(64)   # the work space as such, without partial sums
    with km.Graph() as g:
        m.zero(); s.zero()
        update(n)
    want = np.stack([rows[member == c].astype(np.float64).mean(0) for c in range(k)])
    for _ in range(3):
        m.write(np.full(k * dim, np.nan, dtype)); s.write(np.full(k, 7, np.uint32))
        g.launch()
        km.sync()
        assert np.array_equal(s.read(np.uint32, k), np.bincount(member, minlength=k))
        assert np.abs(m.read(dtype, k * dim).reshape(k, dim) - want).max() < 1e-5
    g.destroy()
    for b in (d, a, m, s):
        b.free()


# columns: one to sixteen at a time, last slices of fewer, sums in up to 32 places, more slices than compute units; points sorted by cluster
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("dim,k", [(1, 2), (2, 3), (3, 9), (4, 300), (5, 70), (6, 70), (7, 70), (8, 500), (9, 70), (10, 70), (11, 70), (12, 70), (13, 70), (14, 70), (15, 70), (16, 900),
                                   (17, 70), (33, 1024), (50, 300), (100, 2500), (4, 4500), (3, 13000), (260, 20), (4200, 3)])
def test_points_by_columns(km, gpu, dim, k, dtype):
    for n in (5003, 9001) if dim > 1000 else (20011, 150001):
        check(km, dim, k, n, dtype, layout=SOA, outside=n == 20011)
        check(km, dim, k, n, dtype, layout=SOA, layout_means=SOA, by_cluster=True)


# ranges of clusters: two to 32 of them, one and more slices of up to 256 coordinates, ranges without points or with nearly all
@pytest.mark.parametrize("dim,k,n", [(260, 700, 20011), (300, 600, 9001), (512, 2000, 20011), (1024, 601, 5003), (516, 640, 1501), (768, 1500, 16385), (200, 610, 126001)])
def test_ranges_of_clusters(km, gpu, dim, k, n):
    check(km, dim, k, n, np.float32, outside=True, stride=dim + 3)
    check(km, dim, k, n, np.float32, one=True, layout_means=SOA)
    if dim > 256:
        check(km, dim, k, n, np.float32, by_cluster=True)


@pytest.mark.parametrize("dim,k,n,layout,pad", [(300, 600, 60032, SOA, 5), (50, 300, 40000, SOA, 5), (260, 600, 20000, AOS, 0)])
def test_recorded_iterations_in_reserved_room(km, orc, gpu, dim, k, n, layout, pad):
    """The room is sized for columns without a stride of their own; padded columns, which copy rows first otherwise, have to do with it."""
    rng = np.random.default_rng(dim + n)
    rows = rng.normal(size=(n, dim)).astype(np.float32)
    cents = rows[rng.choice(n, k, replace=False)].copy()
    stride = dim if layout == AOS else n + pad
    stored = rows
    if layout == SOA:
        stored = np.full((dim, stride), np.nan, np.float32)
        stored[:, :n] = rows.T
    d = km.DeviceBuffer(stored.nbytes); d.write(stored.ravel())
    m = km.DeviceBuffer(4 * k * dim); m.write(cents.ravel())
    a = km.DeviceBuffer(4 * n); out = km.DeviceBuffer(4 * k * dim); sizes = km.DeviceBuffer(4 * k)
    want = orc.assign(rows.ravel(), cents.ravel(), dim, k, n, threads=0, fast=True)
    counts = np.bincount(want, minlength=k)
    sums = np.zeros((k, dim)); np.add.at(sums, want, rows.astype(np.float64))
    km.sync()
    km.check(km.hip_lib().kmx_shutdown())
    km.reserve(km.ASSIGN_BEST, km.UPDATE_ATOMIC_SHM, layout, AOS, dim, k, n)
    with km.Graph() as g:
        km.iteration(d, layout, stride, m, out, AOS, dim, a, sizes, dim, k, n)
    for _ in range(3):
        a.write(np.full(n, 0xFFFFFFF1, np.uint32)); out.write(np.full(k * dim, np.nan, np.float32)); sizes.write(np.full(k, 7, np.uint32))
        g.launch()
        km.sync()
        assert np.array_equal(a.read(np.uint32, n), want)
        assert np.array_equal(sizes.read(np.uint32, k), counts)
        assert np.allclose(out.read(np.float32, k * dim).reshape(k, dim), sums / counts[:, None], rtol=1e-5, atol=1e-6)
    g.destroy()
    for b in (d, m, a, out, sizes):
        b.free()


# shapes whose update used no work space until its sums lay in LDS as doubles: few clusters, columns of fewer than eight dimensions, doubles
NO_WORK_SPACE = [(16, 16, 1 << 16, AOS, np.float32), (4, 300, 70001, SOA, np.float32), (32, 200, 70001, AOS, np.float64), (20, 300, 70001, SOA, np.float64)]


def runtime():
    """The HIP runtime this process has loaded."""
    return ctypes.CDLL("libamdhip64.so")


def own_stream():
    stream = ctypes.c_void_p()
    assert runtime().hipStreamCreateWithFlags(ctypes.byref(stream), 1) == 0   # (non-blocking)
    return stream


class Prepared:
    def __init__(self, km, dim, k, n, layout, dtype, seed):
        rng = np.random.default_rng(seed)
        rows = rng.normal(size=(n, dim)).astype(dtype)
        self.member = rng.integers(0, k, size=n).astype(np.uint32)
        self.member[:k] = np.arange(k)
        self.want = np.zeros((k, dim)); np.add.at(self.want, self.member, rows.astype(np.float64))
        self.want /= np.bincount(self.member, minlength=k)[:, None]
        self.args = (dim, k, n); self.dtype = dtype; self.layout = layout
        self.d = km.DeviceBuffer(rows.nbytes); self.d.write(rows.ravel() if layout == AOS else rows.T.copy().ravel())
        self.a = km.DeviceBuffer(4 * n); self.a.write(self.member)
        self.m = km.DeviceBuffer(rows.itemsize * k * dim); self.s = km.DeviceBuffer(4 * k)

    def update(self, km):
        dim, k, n = self.args
        km.update(km.UPDATE_ATOMIC_SHM, self.d, self.layout, dim if self.layout == AOS else n, self.a, self.m, AOS, dim, self.s, dim, k, n, None, self.dtype)

    def spoil(self):
        dim, k, n = self.args
        self.m.write(np.full(k * dim, np.nan, self.dtype)); self.s.write(np.full(k, 7, np.uint32))

    def check(self):
        dim, k, n = self.args
        assert np.array_equal(self.s.read(np.uint32, k), np.bincount(self.member, minlength=k))
        assert np.abs(self.m.read(self.dtype, k * dim).reshape(k, dim) - self.want).max() < 1e-5   # (|x| < 6: sums of a thousandth of that per rounding)

    def free(self):
        for b in (self.d, self.a, self.m, self.s):
            b.free()


@pytest.mark.parametrize("dim,k,n,layout,dtype", NO_WORK_SPACE)
def test_recorded_updates_outlive_the_work_space(km, gpu, dim, k, n, layout, dtype):
    """Recorded with room for the partial sums in the work space, which then moves (a larger call) and goes (kmx_shutdown)."""
    p = Prepared(km, dim, k, n, layout, dtype, 5)
    large = Prepared(km, 24, 500, 1 << 18, AOS, np.float64, 6)
    p.update(km)
    km.sync()
    with km.Graph() as g:
        p.m.zero(); p.s.zero()
        p.update(km)
    for _ in range(2):
        large.update(km)
        large.check()
        for _ in range(2):
            p.spoil()
            g.launch()
            km.sync()
            p.check()
        km.check(km.hip_lib().kmx_shutdown())
    g.destroy()
    p.free(); large.free()


@pytest.mark.parametrize("dim,k,n,layout,dtype", NO_WORK_SPACE)
def test_updates_on_two_streams(km, gpu, dim, k, n, layout, dtype):
    """The calls of two streams share the partial sums' array: the second waits for the first, eager or recorded."""
    pair = [Prepared(km, dim, k, n, layout, dtype, seed) for seed in (7, 8)]
    streams = [own_stream() for _ in pair]
    graphs = []
    for p in pair:
        p.update(km)
        with km.Graph() as g:
            p.m.zero(); p.s.zero()
            p.update(km)
        graphs.append(g)
    lib = km.hip_lib()
    try:
        for recorded in (False, True):
            for p in pair:
                p.spoil()
            km.sync()
            for _ in range(20):
                for p, stream, g in zip(pair, streams, graphs):
                    km.check(lib.kmx_set_stream(stream))
                    g.launch() if recorded else p.update(km)
            km.sync()
            for p in pair:
                p.check()
    finally:
        km.check(lib.kmx_set_stream(None))
    km.sync()
    for g in graphs:
        g.destroy()
    for stream in streams:
        assert runtime().hipStreamDestroy(stream) == 0
    for p in pair:
        p.update(km)                                      # (the stream that used the array last is gone)
        p.check()
        p.free()


def test_doubles_on_a_stream_that_the_caller_records(km, gpu):
    """Without a work space: nothing is allocated, and nothing is left in the recording that would not run."""
    hip, lib = runtime(), km.hip_lib()
    for dim, k, n, layout in ((32, 200, 70001, AOS), (20, 300, 70001, SOA)):
        p = Prepared(km, dim, k, n, layout, np.float64, 9)
        p.update(km)                                      # (kernels are loaded)
        km.sync()
        km.check(lib.kmx_shutdown())
        stream, graph, launched = own_stream(), ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(stream, 0) == 0  # (the strictest mode)
        try:
            km.check(lib.kmx_set_stream(stream))
            p.m.zero(); p.s.zero()
            p.update(km)
        finally:
            km.check(lib.kmx_set_stream(None))
            assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(launched), graph, None, None, ctypes.c_size_t(0)) == 0
        for _ in range(3):
            p.spoil()
            km.sync()
            assert hip.hipGraphLaunch(launched, stream) == 0
            km.sync()
            p.check()
        assert hip.hipGraphExecDestroy(launched) == 0 and hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
        p.free()


@pytest.mark.parametrize("dim,k", [(17, 70), (37, 300), (48, 400), (37, 900)])
def test_whole_rows_of_many_points(km, gpu, dim, k):
    """Both sides of the line from which rows of 17 to 48 floats go as a whole (37 x 900 sums do not fit so). Small whole numbers: every sum is exact."""
    line = -(-60000000 // dim)
    rng = np.random.default_rng(dim + k)
    rows = rng.integers(-8, 9, size=(line, dim), dtype=np.int8).astype(np.float32)
    member = rng.integers(0, k, size=line).astype(np.uint32)
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    a = km.DeviceBuffer(4 * line); a.write(member)
    m = km.DeviceBuffer(4 * k * dim); s = km.DeviceBuffer(4 * k)
    for n in (line, line - 1):
        m.write(np.full(k * dim, np.nan, np.float32)); s.write(np.full(k, 7, np.uint32))
        km.update(km.UPDATE_ATOMIC_SHM, d, AOS, dim, a, m, AOS, dim, s, dim, k, n)
        counts = np.bincount(member[:n], minlength=k)
        want = np.stack([np.bincount(member[:n], weights=rows[:n, q], minlength=k) for q in range(dim)], axis=1)
        assert np.array_equal(s.read(np.uint32, k), counts)
        assert np.array_equal(m.read(np.float32, k * dim).reshape(k, dim), want.astype(np.float32) / counts.astype(np.float32)[:, None])
    for b in (d, a, m, s):
        b.free()


@pytest.mark.parametrize("dim,k,n", [(160, 100, 150001), (176, 60, 150001), (144, 30, 100003), (192, 200, 200001), (128, 400, 300001), (112, 100, 100003), (160, 100, 20011)])
def test_slices_of_whole_lines(km, gpu, dim, k, n):
    """Rows of whole 64 bytes in three slices and more, the last one narrower; the last two: equal slices, and slices of 32."""
    check(km, dim, k, n, np.float32, outside=True)
    check(km, dim, k, n, np.float32, layout_means=SOA, stride=dim + 3)


def test_many_clusters_of_many_points_without_allocation(km, gpu):
    """Slices of four coordinates, where the sorted chunks are faster but their partial sums would not fit the scratch array: taken there and while recorded, as slices."""
    dim, k, n = 32, 4000, (1 << 21) + 5
    rng = np.random.default_rng(11)
    rows = rng.integers(-8, 9, size=(n, dim), dtype=np.int8).astype(np.float32)
    member = rng.integers(0, k, size=n).astype(np.uint32)
    counts = np.bincount(member, minlength=k)
    want = np.stack([np.bincount(member, weights=rows[:, q], minlength=k) for q in range(dim)], axis=1).astype(np.float32) / counts.astype(np.float32)[:, None]
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    a = km.DeviceBuffer(4 * n); a.write(member)
    m = km.DeviceBuffer(4 * k * dim); s = km.DeviceBuffer(4 * k)

    def check_result():
        assert np.array_equal(s.read(np.uint32, k), counts)
        assert np.array_equal(m.read(np.float32, k * dim).reshape(k, dim), want)       # (whole numbers: every sum is exact)
        m.write(np.full(k * dim, np.nan, np.float32)); s.write(np.full(k, 7, np.uint32))
    for fn in (km.update, km.update_noalloc):
        fn(km.UPDATE_ATOMIC_SHM, d, AOS, dim, a, m, AOS, dim, s, dim, k, n)
        check_result()
    km.sync()
    km.check(km.hip_lib().kmx_shutdown())
    km.update(km.UPDATE_ATOMIC_SHM, d, AOS, dim, a, m, AOS, dim, s, dim, k, 64)
    with km.Graph() as g:
        km.update(km.UPDATE_ATOMIC_SHM, d, AOS, dim, a, m, AOS, dim, s, dim, k, n)
    for _ in range(3):
        g.launch()
        km.sync()
        check_result()
    g.destroy()
    for b in (d, a, m, s):
        b.free()


# both sides of the lines between slices of doubles and the kernels without partial sums
@pytest.mark.parametrize("dim,k,n", [(100, 300, 399999), (100, 300, 400001), (105, 600, 380001), (105, 600, 381001), (97, 1000, 300001), (4, 2000, 300001), (8, 2000, 500001), (11, 1105, 331499), (11, 1105, 331500), (6, 2000, 400001)])
def test_doubles_beside_the_lines(km, gpu, dim, k, n):
    check(km, dim, k, n, np.float64, outside=True)


def work_groups(km, dim, k, n, dtype=np.float32, stride=None):
    """Of an update of AoS points (all in cluster 0)."""
    stride = stride or dim
    item = np.dtype(dtype).itemsize
    bufs = [km.DeviceBuffer(b) for b in (item * n * stride, 4 * n, item * k * dim, 4 * k)]
    for b in bufs:
        b.zero()
    ex = km.ExecParams()
    km.update(km.UPDATE_ATOMIC_SHM, bufs[0], AOS, stride, bufs[1], bufs[2], AOS, dim, bufs[3], dim, k, n, ex, dtype)
    km.sync()
    for b in bufs:
        b.free()
    return ex.block_count


# both sides of the lines between ranges of clusters and the sorted chunks (us, ranges / sorted chunks: 22.6 / 18.1, 23.3 / 19.9; 21.2 / 27.9)
@pytest.mark.parametrize("dim,k,n,ranges", [(372, 606, 8830, False), (304, 717, 16343, False), (304, 717, 16448, True), (400, 1585, 6706, True), (400, 700, 6706, True), (400, 699, 6706, False)])
def test_wide_rows_of_few_points(km, gpu, dim, k, n, ranges):
    check(km, dim, k, n, np.float32, outside=True)
    slices = -(-dim // 32)
    chunk = -(-(-(-n // (gpu.compute_units // slices))) // 1024) * 1024
    assert (work_groups(km, dim, k, n) != -(-n // chunk) * slices) == ranges


# rows with a gap behind them, on both sides of the lines from which they go as a whole: a work-group per compute unit, not a third or half of it per slice
@pytest.mark.parametrize("dim,k,stride,whole", [(17, 52, 49, True), (20, 41, 36, True), (20, 41, 35, False), (34, 66, 50, True), (42, 30, 74, True), (26, 40, 46, False)])
def test_rows_with_gaps_behind_them(km, gpu, dim, k, stride, whole):
    line = -(-(45000000 if (dim - 1) % 16 < 8 else 75000000) // stride)
    n = line if whole or stride < dim + 16 else line - 1
    rng = np.random.default_rng(dim + k)
    member = rng.integers(0, k, size=n).astype(np.uint32)
    rows = np.full((n, stride), np.nan, np.float32)
    rows[:, :dim] = rng.integers(-8, 9, size=(n, dim), dtype=np.int8)
    d = km.DeviceBuffer(rows.nbytes); d.write(rows.ravel())
    a = km.DeviceBuffer(4 * n); a.write(member)
    m = km.DeviceBuffer(4 * k * dim); s = km.DeviceBuffer(4 * k)
    ex = km.ExecParams()
    km.update(km.UPDATE_ATOMIC_SHM, d, AOS, stride, a, m, AOS, dim, s, dim, k, n, ex)
    counts = np.bincount(member, minlength=k)
    want = np.stack([np.bincount(member, weights=rows[:, q], minlength=k) for q in range(dim)], axis=1)   # (whole numbers: every sum is exact)
    assert np.array_equal(s.read(np.uint32, k), counts)
    assert np.array_equal(m.read(np.float32, k * dim).reshape(k, dim), want.astype(np.float32) / counts.astype(np.float32)[:, None])
    slices = 1 if whole else -(-dim // 16)
    chunk = -(-n // (gpu.compute_units // 8 // slices * 8) // 64) * 64                 # whole wavefronts of points
    assert ex.block_count == -(-n // chunk) * slices
    for b in (d, a, m, s):
        b.free()
