"""Which kernel adds the members up in the serial-order update (csrc/update_ordered_route.h), at sizes that no test could allocate: a
launch has fewer than 2^32 work-items, and what does not fit one goes to the kernel with a work-item per chain (no GPU needed)."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STREAM, STAGED, LANES, SPLIT = 0, 1, 2, 3
THREADS = {STREAM: 128, STAGED: 512}
LARGE = 256


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    folder = tmp_path_factory.mktemp("route")
    src, lib = folder / "route.cpp", folder / "libroute.so"
    src.write_text('#include "update_ordered_route.h"\n'
                   'extern "C" uint64_t route(uint32_t bytes, int whole, uint32_t dim, uint32_t k, uint32_t n)\n'
                   "{ const kmx::OrderedSumRoute r = kmx::ordered_sum_route(bytes, whole != 0, dim, k, n); return (uint64_t)r.kernel << 32 | r.blocks; }\n")
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "cuda-kmeans_amd", "csrc"), str(src), "-o", str(lib)])
    fn = ctypes.CDLL(str(lib)).route
    fn.restype, fn.argtypes = ctypes.c_uint64, [ctypes.c_uint32, ctypes.c_int] + [ctypes.c_uint32] * 3

    def call(value_bytes, whole, dim, k, n):
        r = fn(value_bytes, int(whole), dim, k, n)
        return r >> 32, r & 0xFFFFFFFF
    return call


def work_items(kernel, blocks, k, n):
    """of the launch that has a work-group per cluster (of SPLIT: per cluster that can be large) and block"""
    return 0 if kernel == LANES else (n // LARGE * blocks * THREADS[STREAM]) if kernel == SPLIT else k * blocks * THREADS[kernel]


@pytest.mark.parametrize("value_bytes,whole,dim,k,n,want", [
    (4, True, 128, (1 << 23) - 1, 256 * ((1 << 23) - 1), STREAM), (4, True, 128, 1 << 23, 1 << 31, LANES),       # 2^32 - 512 and 2^32 work-items
    (8, True, 66, (1 << 22), 1 << 30, STREAM), (8, True, 130, 1 << 22, 1 << 30, LANES),                         # five and nine blocks a row
    (4, True, 12, 1 << 25, 1 << 30, SPLIT), (4, True, 256, 1 << 25, 1 << 30, LANES),                            # 2^22 clusters that can be large, one and eight blocks
    (4, True, 4, 1 << 25, (1 << 32) - (1 << 21), LANES), (4, True, 120000, 2, 70, LANES),                       # none can be large
    (4, False, 5, (1 << 23) - 1, 256 * ((1 << 23) - 1), STAGED), (4, False, 5, 1 << 23, 1 << 31, LANES), (4, False, 33, 1 << 22, 1 << 30, LANES),
    (4, True, 32, 1024, 1 << 21, STREAM), (4, False, 31, 1024, 1 << 21, STAGED), (4, True, 8, 4096, 4096 * 127, LANES), (4, True, 12, 4096, 4096 * 31, LANES),
    (4, True, 192, 1024, 1024 * 255, STREAM), (4, True, 196, 1024, 1024 * 255, SPLIT), (4, True, 196, 1024, 1024 * 256, STREAM),
])
def test_launches_hold_their_work_items(route, value_bytes, whole, dim, k, n, want):
    kernel, blocks = route(value_bytes, whole, dim, k, n)
    assert kernel == want
    assert work_items(kernel, blocks, k, n) < 1 << 32


@pytest.mark.parametrize("value_bytes", [4, 8])
@pytest.mark.parametrize("whole", [False, True])
def test_no_size_asks_for_more_than_there_is(route, value_bytes, whole):
    """Work-items of a launch; at least one work-group; the list of large clusters in the words of the histograms (k of them at least)."""
    for dim in (1, 2, 4, 8, 16, 32, 36, 64, 100, 1024, 1 << 20):
        for k in {max(1, (1 << e) + o) for e in range(0, 30) for o in (-1, 0, 1)}:
            for members in (1, 31, 32, 127, 128, 255, 256, 511, 512):
                for n in (k * members, k * members + k - 1):
                    if n >= (1 << 32) - (1 << 20):
                        continue
                    kernel, blocks = route(value_bytes, whole, dim, k, n)
                    assert work_items(kernel, blocks, k, n) < 1 << 32, (dim, k, members)
                    if kernel == SPLIT:
                        assert n // LARGE >= 1 and 1 + n // LARGE <= k, (dim, k, members)
