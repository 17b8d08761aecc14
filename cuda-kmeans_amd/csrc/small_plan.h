/*
 * Which small inputs assign_small_kernel (small.hip) takes and with which work-groups, and the LDS they need. Plain host code without a HIP
 * header: the tests look at every shape that is accepted. value_bytes: 4 for floats, 8 for doubles.
 */
#ifndef KMX_SMALL_PLAN_H
#define KMX_SMALL_PLAN_H

#include <algorithm>
#include <cstdint>

namespace kmx {

constexpr uint32_t SMALL_WAVE = 64, SMALL_POINTS = SMALL_WAVE;
constexpr uint32_t SMALL_THREADS = 512, SMALL_WIDE_THREADS = 1024;
constexpr uint32_t SMALL_SUMS = 4096; /* elements of the sums: beyond, reading the memberships again (update_small_kernel) is cheaper than as many partial sums */
constexpr uint32_t SMALL_FEW_CENTROIDS = 12; /* up to here a tile of one point times one centroid per lane */

/* a candidate: a root and its centroid's number, floats as 64 bits (SmallKey) */
constexpr uint32_t small_key_bytes(uint32_t value_bytes) { return value_bytes == 4 ? 8 : 16; }
/* shares of the centroids: a wavefront has 16 * tile of the points */
constexpr uint32_t small_shares(uint32_t tile, uint32_t points, uint32_t threads) { return threads / SMALL_WAVE / (points / 16 / tile); }
/* the kernel's static arrays: a candidate per share and point, a membership per point */
constexpr uint32_t small_static_bytes(uint32_t value_bytes, uint32_t tile, uint32_t points, uint32_t threads)
{
	return small_shares(tile, points, threads) * points * small_key_bytes(value_bytes) + points * 4;
}

constexpr uint32_t small_row_stride(uint32_t dim) { return (((dim + 3) / 4) | 1u) * 4; }
/* LDS next to the static arrays: the rows of the points and as many centroids as 32 KB hold (at least 32: one step of all wavefronts) */
inline uint32_t assign_small_chunk(uint32_t value_bytes, uint32_t dim, uint32_t k)
{
	const uint32_t fit = 32 * 1024 / (small_row_stride(dim) * value_bytes) / 32 * 32;
	return std::min(k, std::max(32u, fit));
}
/* sums_width: coordinates whose sums lie in LDS at a time, where the centroids were; 0: no sums */
inline uint32_t assign_small_lds(uint32_t value_bytes, uint32_t dim, uint32_t k, uint32_t points, uint32_t sums_width)
{
	const uint32_t centroids = assign_small_chunk(value_bytes, dim, k) * small_row_stride(dim) * value_bytes;
	return points * small_row_stride(dim) * value_bytes + (sums_width ? std::max(centroids, k * sums_width * 8 + k * 4) : centroids);
}

/*
 * Every pair costs 3 dim operations and about 30 to compare and keep, four cycles each on a SIMD; a work-group of 64 points keeps one
 * compute unit, so fewer than 256 of them leave units idle. The line is 450 million, 530 million where small_more says so, and three halves of either for more than 32 dimensions.
 * Between the two, 3236 shapes, these kernels in shares of the general path's time: up to 256 work-groups 0.43 to 1.13, 0.69 in the mean; a little more of them, whose second
 * round is nearly empty, 1.0 to 1.75 (N = 17391, d = 14, k = 420 34.6 / 24.2 us; N = 19340, d = 42, k = 261 38.4 / 21.9); else rows of 5 to 16 floats 0.85 to 1.32, 1.08 in the mean; of up to
 * 4 0.76 to 1.0, of 17 to 32 0.59 to 1.05 (N = 40000, d = 32, k = 100 28.7 / 40.3 us per iteration), wider 0.82 to 1.56, 1.1 in the mean; columns, 5 to 8 of them 0.89 to 1.11, 9 to 16
 * 0.76 to 1.01, 129 to 192 0.58 to 0.96, others beyond 32 0.86 to 1.58. Doubles: twice 450 million.
 * From 65536 points on the work-groups run in rounds and the general path's larger ones are ahead.
 */
constexpr uint32_t SMALL_MAX_POINTS = 1u << 16;
constexpr uint64_t SMALL_EFFORT = 450000000, SMALL_EFFORT_MORE = 530000000; /* (doubles, N = 56478, d = 56, k = 128, 475: 87 us per iteration, general path 54) */
/* `columns`: SoA points */
constexpr bool small_more(bool columns, uint32_t dim, uint32_t n)
{
	if (n <= 256 * SMALL_POINTS) return true;
	if (dim > 32) return columns && dim > 128 && dim <= 192;
	return columns ? (dim > 16 && n > 20480) || (n > 24576 && (dim <= 4 || dim > 8)) : n > 24576 && (dim <= 4 || dim > 16);
}
/* what the rule leaves for the static arrays: those of every work-group of eight wavefronts fit; one of 16 is taken only where its own do (small_shape) */
constexpr uint32_t small_static_room(uint32_t value_bytes) { return SMALL_THREADS / SMALL_WAVE * SMALL_POINTS * (value_bytes + 4) + SMALL_POINTS * 4 + 64; }
constexpr bool small_static_fits(uint32_t value_bytes, uint32_t tile, uint32_t points) { return small_static_bytes(value_bytes, tile, points, SMALL_THREADS) <= small_static_room(value_bytes); }
static_assert(small_static_fits(4, 1, 64) && small_static_fits(4, 2, 64) && small_static_fits(4, 1, 32) && small_static_fits(4, 2, 32) &&
              small_static_fits(8, 1, 64) && small_static_fits(8, 2, 64) && small_static_fits(8, 1, 32) && small_static_fits(8, 2, 32), "eight wavefronts");

inline bool small_assign_accepts(uint32_t value_bytes, bool columns, uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget)
{
	if (n == 0 || n > SMALL_MAX_POINTS || dim > 256 || k > (1u << 20)) return false;
	const uint64_t effort = std::max<uint64_t>(n, 256 * SMALL_POINTS) * k * (3 * (uint64_t)dim + 30);
	const uint64_t limit = (value_bytes == 8 ? 2 * SMALL_EFFORT : small_more(columns, dim, n) ? SMALL_EFFORT_MORE : SMALL_EFFORT) * (dim > 32 ? 3 : 2) / 2;
	return effort <= limit && assign_small_lds(value_bytes, dim, k, SMALL_POINTS, 0) + small_static_room(value_bytes) <= lds_budget;
}
/* floats, points added up too (the partial sums of all work-groups are written and read once) */
inline bool small_iteration_accepts(bool columns, uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget)
{
	return (uint64_t)k * dim <= SMALL_SUMS && (uint64_t)k * dim * ((n + SMALL_POINTS - 1) / SMALL_POINTS) <= (2u << 20) && small_assign_accepts(4, columns, dim, k, n, lds_budget) &&
	       assign_small_lds(4, dim, k, SMALL_POINTS, dim) + small_static_room(4) <= lds_budget;
}

/*
 * Up to 128 work-groups of 64 points leave half of the compute units idle: 32 points each (us per iteration, 64 / 32 points: N = 1000, d = 20, k = 128 14.4 / 12.0;
 * N = 5000, d = 32, k = 100 16.5 / 14.5; N = 10240, d = 20, k = 128 16.4 / 16.6: twice the partial sums). One work-group per compute unit at most: 16
 * wavefronts each, whose waits for the LDS others cover (eight / 16: N = 10240, d = 20, k = 128 16.4 / 15.2; N = 16384 15.9 / 15.0); with two, the waits
 * are covered already (N = 20000, d = 100, k = 30, SoA 23.3 / 26.7; d = 8, k = 30 12.7 / 15.1; AoS d = 20, k = 100 20.0 / 19.8; N = 32768, d = 8, k = 64 13.6 / 14.6).
 * 16 wavefronts have twice as many candidates in LDS, which rows of around 200 doubles leave no room for: eight there. Candidates of doubles have 16 bytes, and merging twice as
 * many costs more than the waits unless there are many centroids (1368 shapes of 8193 to 16384 points, 16 wavefronts in shares of the time of eight: 13 to 200 centroids 0.95 to 1.24, 1.07
 * in the mean, more than that in up to 64 dimensions 0.92 to 1.10, 0.97 in the mean, beyond 0.99 to 1.06; up to 12 centroids 0.94 to 1.04 in up to 16 dimensions, beyond 0.96 to 1.24).
 */
constexpr uint32_t SMALL_HALF_POINTS = 128 * SMALL_POINTS, SMALL_WIDE_POINTS = 256 * SMALL_POINTS;

/* How many times all compute units are filled: work-groups of 512 lanes whose LDS, static arrays included, is given out in pieces of 1280 bytes, four a compute unit at most. */
constexpr uint32_t small_rounds(uint32_t groups, uint32_t lds_bytes)
{
	const uint32_t each = 160 * 1024 / ((lds_bytes + 1279) / 1280 * 1280), resident = 256 * (each < 4 ? each : 4);
	return resident ? (groups + resident - 1) / resident : groups;
}

struct SmallShape { uint32_t tile, points, threads, lds_bytes /* without the static arrays */, sums_width; };

inline SmallShape small_shape(uint32_t value_bytes, uint32_t dim, uint32_t k, uint32_t n, bool sums, uint32_t lds_budget)
{
	const uint32_t tile = k > SMALL_FEW_CENTROIDS ? 2 : 1, points = n <= SMALL_HALF_POINTS ? SMALL_POINTS / 2 : SMALL_POINTS;
	/*
	 * Sums of doubles need more LDS than the centroids they replace. Where that takes a round of work-groups more, they are added up and written in parts of the coordinates, as few as make
	 * up for it (us per iteration, whole / in parts / whole in floats, before: N = 24497, d = 220, k = 15 39.4 / 27.3 / 26.6; N = 38139, d = 208, k = 16 51.0 / 40.1 / 38.3;
	 * N = 48841, d = 187, k = 3, SoA 32.1 / 26.2 / 25.7; assignment and update by themselves 26.5, 37.9, 30.6).
	 */
	uint32_t width = sums ? dim : 0;
	const uint32_t groups = (n + points - 1) / points, held = small_static_bytes(value_bytes, tile, points, SMALL_THREADS);
	const uint32_t least = small_rounds(groups, assign_small_lds(value_bytes, dim, k, points, 0) + held);
	for (uint32_t parts = 2; sums && parts <= 4 && parts < dim && small_rounds(groups, assign_small_lds(value_bytes, dim, k, points, width) + held) > least; ++parts) width = (dim - 1) / parts + 1;
	const uint32_t lds = assign_small_lds(value_bytes, dim, k, points, width);
	const bool many = value_bytes == 4 || (k > 200 && dim <= 64) || (k <= SMALL_FEW_CENTROIDS && dim <= 16);
	const bool wide = many && n > SMALL_HALF_POINTS && n <= SMALL_WIDE_POINTS && lds + small_static_bytes(value_bytes, tile, points, SMALL_WIDE_THREADS) <= lds_budget;
	return SmallShape{ tile, points, wide ? SMALL_WIDE_THREADS : SMALL_THREADS, lds, width };
}
inline uint32_t assign_small_max_blocks(uint32_t n) { return n <= SMALL_HALF_POINTS ? (n + SMALL_POINTS / 2 - 1) / (SMALL_POINTS / 2) : (n + SMALL_POINTS - 1) / SMALL_POINTS; }

} // namespace kmx

#endif
