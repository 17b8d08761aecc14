"""Which kernel adds the members up in the serial-order update (csrc/update_ordered_route.h), at sizes that no test could allocate: a
launch has fewer than 2^32 work-items, and what does not fit one goes to the kernel with a work-item per chain (no GPU needed)."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STREAM, STAGED, LANES = 0, 1, 2
THREADS = {STREAM: 128, STAGED: 512}


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


@pytest.mark.parametrize("value_bytes,whole,dim,k,n,want", [
    (4, True, 12, (1 << 25) - 1, 32 * ((1 << 25) - 1), STREAM), (4, True, 12, 1 << 25, 1 << 30, LANES),          # 2^32 - 128 and 2^32 work-items
    (8, True, 18, (1 << 24) - 1, 32 * ((1 << 24) - 1), STREAM), (8, True, 18, 1 << 24, 1 << 29, LANES),          # two blocks a row
    (4, True, 4, 1 << 25, (1 << 32) - (1 << 21), LANES),
    (4, False, 5, (1 << 23) - 1, 256 * ((1 << 23) - 1), STAGED), (4, False, 5, 1 << 23, 1 << 31, LANES), (4, False, 33, 1 << 22, 1 << 30, LANES),
    (4, True, 32, 1024, 1 << 21, STREAM), (4, False, 31, 1024, 1 << 21, STAGED), (4, True, 8, 4096, 4096 * 127, LANES), (4, True, 12, 4096, 4096 * 31, LANES),
])
def test_launches_hold_their_work_items(route, value_bytes, whole, dim, k, n, want):
    kernel, blocks = route(value_bytes, whole, dim, k, n)
    assert kernel == want
    if kernel != LANES:
        assert k * blocks * THREADS[kernel] < 1 << 32


@pytest.mark.parametrize("value_bytes", [4, 8])
@pytest.mark.parametrize("whole", [False, True])
def test_no_size_asks_for_more_work_items_than_a_launch_has(route, value_bytes, whole):
    for dim in (1, 2, 4, 8, 16, 32, 36, 64, 100, 1024, 1 << 20):
        for k in {max(1, (1 << e) + o) for e in range(0, 30) for o in (-1, 0, 1)}:
            for members in (1, 31, 32, 127, 128, 255, 256, 511, 512):
                if k * members < (1 << 32) - (1 << 20):
                    kernel, blocks = route(value_bytes, whole, dim, k, k * members)
                    assert kernel == LANES or k * blocks * THREADS[kernel] < 1 << 32, (dim, k, members)
