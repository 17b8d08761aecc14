"""The reads of the half-precision sweep that takes 64 points of a column per request (csrc/rank16_columns.h): every lane of every wavefront of a
launch reads inside the points, those of wavefronts without points too (no GPU needed: the address arithmetic is enumerated)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def points_read(tmp_path_factory):
    folder = tmp_path_factory.mktemp("columns")
    src, lib = folder / "columns.cpp", folder / "libcolumns.so"
    src.write_text('#include "rank16_columns.h"\n'
                   'extern "C" void points_read(uint32_t first, uint32_t n, uint64_t* base, uint64_t* point)\n'
                   "{ *base = kmx::rank16_column_base(first, n); for (uint32_t lane = 0; lane < 64; ++lane) point[lane] = *base + kmx::rank16_column_inside((uint32_t)*base, lane, n); }\n")
    subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "cuda-kmeans_amd", "csrc"), str(src), "-o", str(lib)])
    fn = ctypes.CDLL(str(lib)).points_read
    fn.restype, fn.argtypes = None, [ctypes.c_uint32, ctypes.c_uint32, ctypes.c_void_p, ctypes.c_void_p]

    def call(first, n):
        base, point = np.zeros(1, np.uint64), np.zeros(64, np.uint64)
        fn(first, n, base.ctypes.data, point.ctypes.data)
        return int(base[0]), point.astype(np.int64)
    return call


def outside(points_read, n, waves, dim, stride):
    """Reads behind the last element of n points, over all wavefronts of a launch: (first point, lane) of the worst, or None."""
    units = -(-n // (waves * 64))
    for wave in range(max(0, (units - 2) * waves), units * waves):      # (the units before the last two are full)
        first = wave * 64
        base, point = points_read(first, n)
        held = point < n
        assert np.all(point[: max(0, min(64, n - first))] == np.arange(first, min(first + 64, n)))
        if base >= n or not held.all() or ((dim - 1) * stride + point).max() >= (dim - 1) * stride + n:
            return first, int(np.argmax(point))
    return None


@pytest.mark.parametrize("waves,dim", [(8, 97), (8, 128), (4, 193), (4, 256), (8, 256)])
@pytest.mark.parametrize("n", [1, 8, 63, 64, 65, 191, 192, 393, 448, 449, 511, 512, 513, 520, 575, 576, 5001, 100000, 262143, (1 << 32) - 1 - 4096])
def test_no_wavefront_reads_behind_the_points(points_read, waves, dim, n):
    assert outside(points_read, n, waves, dim, n) is None


def test_a_base_that_is_not_held_would_be_noticed():
    """The same with the first point as it is: 1 to 7 wavefronts of the last unit read behind the points."""
    def as_it_is(first, n):
        return first, first + np.minimum(np.arange(64), n - 1 - min(first, n - 1))
    for n in (8, 64, 65, 393, 448, 520, 5001):
        assert outside(as_it_is, n, 8, 128, n) is not None
    for n in (449, 512, 961, 1024):                                       # every wavefront of the last unit has a point
        assert outside(as_it_is, n, 8, 128, n) is None
