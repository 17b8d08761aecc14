"""Small inputs (csrc/small_plan.h): every shape that the rule accepts is launched with work-groups whose LDS fits the budget, static arrays included, and
with as many partial sums as there is room for (no GPU needed: all shapes are enumerated)."""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "small_plan.h"
using namespace kmx;
/* number of accepted shapes, and of those whose launch asks for more than the budget; always_wide: as if 16 wavefronts were taken whatever they need */
extern "C" int accepts(uint32_t value_bytes, int columns, uint32_t dim, uint32_t k, uint32_t n) { return small_assign_accepts(value_bytes, columns != 0, dim, k, n, 160 * 1024); }
extern "C" uint32_t threads(uint32_t value_bytes, uint32_t dim, uint32_t k, uint32_t n) { return small_shape(value_bytes, dim, k, n, false, 160 * 1024).threads; }
extern "C" void count(uint32_t value_bytes, int columns, int sums, uint32_t budget, int always_wide, uint64_t* accepted, uint64_t* beyond, uint64_t* wide)
{
	*accepted = *beyond = *wide = 0;
	const uint32_t points[] = { 1, 31, 32, 33, 64, 1000, 8191, 8192, 8193, 10000, 16383, 16384, 16385, 30000, 65535, 65536, 65537 };
	for (uint32_t n : points)
		for (uint32_t dim = 1; dim <= 257; ++dim)
			for (uint32_t k = 1; k <= 1200; k += k < 300 ? 1 : 37) {
				if (!(sums ? value_bytes == 4 && small_iteration_accepts(columns != 0, dim, k, n, budget) : small_assign_accepts(value_bytes, columns != 0, dim, k, n, budget))) continue;
				++*accepted;
				const SmallShape s = small_shape(value_bytes, dim, k, n, sums != 0, budget);
				const uint32_t threads = always_wide && n > SMALL_HALF_POINTS && n <= SMALL_WIDE_POINTS ? SMALL_WIDE_THREADS : s.threads;
				*beyond += s.lds_bytes + small_static_bytes(value_bytes, s.tile, s.points, threads) > budget || (n + s.points - 1) / s.points > assign_small_max_blocks(n);
				*wide += threads == SMALL_WIDE_THREADS;
			}
}
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    folder = tmp_path_factory.mktemp("small")
    src, lib = folder / "small.cpp", folder / "libsmall.so"
    src.write_text(SOURCE)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "cuda-kmeans_amd", "csrc"), str(src), "-o", str(lib)])
    return ctypes.CDLL(str(lib))


@pytest.fixture(scope="module")
def count(library):
    fn = library.count
    fn.restype = None

    def call(value_bytes, columns, sums, budget, always_wide=False):
        out = [ctypes.c_uint64() for _ in range(3)]
        fn(value_bytes, int(columns), int(sums), budget, int(always_wide), *[ctypes.byref(v) for v in out])
        return [v.value for v in out]
    return call


@pytest.mark.parametrize("columns", [False, True])
@pytest.mark.parametrize("value_bytes,sums", [(4, False), (4, True), (8, False)])
@pytest.mark.parametrize("budget", [160 * 1024, 128 * 1024, 64 * 1024 + 8, 48 * 1024, 16 * 1024])
def test_what_is_accepted_fits(count, value_bytes, columns, sums, budget):
    accepted, beyond, wide = count(value_bytes, columns, sums, budget)
    assert accepted > 0 and beyond == 0
    assert wide > 0                                                     # the rule is not kept by never taking 16 wavefronts


def test_candidates_that_are_not_counted_would_be_noticed(count):
    """16 wavefronts whatever they need: more than there is, for rows of around 200 doubles."""
    assert count(8, False, False, 160 * 1024, always_wide=True)[1] > 0


# measured slower here than in the general path (us, these kernels / that): 34.6 / 24.2, 36.9 / 26.2, 38.4 / 21.9, 35.3 / 21.2
@pytest.mark.parametrize("dim,k,n", [(14, 420, 17391), (6, 614, 16611), (42, 261, 19340), (41, 252, 17741)])
def test_work_groups_a_little_more_than_compute_units_go_to_the_general_path(library, dim, k, n):
    assert not library.accepts(4, 0, dim, k, n) and not library.accepts(4, 1, dim, k, n)


# and faster: 28.7 / 40.3 per iteration; columns of 129 to 192 dimensions 0.6 of the time
@pytest.mark.parametrize("columns,dim,k,n", [(0, 32, 100, 40000), (0, 4, 190, 65536), (1, 150, 24, 65536)])
def test_shapes_beyond_the_lower_line_that_stay(library, columns, dim, k, n):
    assert library.accepts(4, columns, dim, k, n)


# doubles, us of 16 wavefronts / eight: 10.2 / 8.3, 6.3 / 5.1; 30.8 / 32.0 and more with many centroids
@pytest.mark.parametrize("dim,k,n,threads", [(34, 46, 15066, 512), (60, 8, 12485, 512), (36, 46, 11715, 512), (20, 387, 14211, 1024), (4, 8, 15075, 1024)])
def test_doubles_take_16_wavefronts_for_many_centroids(library, dim, k, n, threads):
    assert library.threads(8, dim, k, n) == threads


# one work-group per compute unit: half of the general path's time and less
@pytest.mark.parametrize("columns", [0, 1])
@pytest.mark.parametrize("dim,k,n", [(2, 840, 3000), (4, 740, 8192), (20, 330, 16384), (90, 157, 5458), (254, 61, 8307)])
def test_few_work_groups_stay(library, columns, dim, k, n):
    assert library.accepts(4, columns, dim, k, n)


ROUNDS = """
#include "small_plan.h"
using namespace kmx;
/* iterations whose sums, were they all in LDS at once, would take a round of work-groups more than the assignment, and of those the ones that still do; width: the least of all */
extern "C" void rounds(int columns, uint64_t* whole, uint64_t* still, uint32_t* width)
{
	*whole = *still = 0;
	*width = 1u << 30;
	for (uint32_t n = 16385; n <= 65536; n += 997)
		for (uint32_t dim = 1; dim <= 256; ++dim)
			for (uint32_t k = 1; k * dim <= SMALL_SUMS; ++k) {
				if (!small_iteration_accepts(columns != 0, dim, k, n, 160 * 1024)) continue;
				const SmallShape s = small_shape(4, dim, k, n, true, 160 * 1024);
				const uint32_t groups = (n + s.points - 1) / s.points, held = small_static_bytes(4, s.tile, s.points, s.threads);
				const uint32_t least = small_rounds(groups, assign_small_lds(4, dim, k, s.points, 0) + held);
				*whole += small_rounds(groups, assign_small_lds(4, dim, k, s.points, dim) + held) > least;
				*still += small_rounds(groups, s.lds_bytes + held) > least;
				if (s.sums_width < dim) *width = std::min(*width, s.sums_width);
			}
}
extern "C" uint32_t width(uint32_t dim, uint32_t k, uint32_t n) { return small_shape(4, dim, k, n, true, 160 * 1024).sums_width; }
"""


@pytest.fixture(scope="module")
def plan_of_sums(tmp_path_factory):
    folder = tmp_path_factory.mktemp("rounds")
    src, lib = folder / "rounds.cpp", folder / "librounds.so"
    src.write_text(ROUNDS)
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", os.path.join(ROOT, "cuda-kmeans_amd", "csrc"), str(src), "-o", str(lib)])
    return ctypes.CDLL(str(lib))


@pytest.mark.parametrize("columns", [0, 1])
def test_sums_take_no_round_of_work_groups_more(plan_of_sums, columns):
    whole, still, width = ctypes.c_uint64(), ctypes.c_uint64(), ctypes.c_uint32()
    plan_of_sums.rounds(columns, ctypes.byref(whole), ctypes.byref(still), ctypes.byref(width))
    assert whole.value > 0 and still.value == 0
    assert width.value >= 2                                             # the kernel's division by the width


# in parts where whole sums were slower, whole where they cost nothing
@pytest.mark.parametrize("dim,k,n,parts", [(220, 15, 24497, 2), (208, 16, 38139, 2), (187, 3, 48841, 2), (20, 128, 10240, 1), (8, 64, 65536, 1), (100, 30, 20000, 1)])
def test_sums_in_parts(plan_of_sums, dim, k, n, parts):
    assert plan_of_sums.width(dim, k, n) == (dim if parts == 1 else (dim - 1) // parts + 1)
