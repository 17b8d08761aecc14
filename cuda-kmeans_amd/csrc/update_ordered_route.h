/*
 * Which kernel of update_ordered.hip adds the members up. Plain host code without a HIP header: the tests look at sizes that no device
 * memory holds.
 */
#ifndef KMX_UPDATE_ORDERED_ROUTE_H
#define KMX_UPDATE_ORDERED_ROUTE_H

#include <cstdint>

namespace kmx {

enum OrderedSumKernel { ORDERED_STREAM, ORDERED_STAGED, ORDERED_LANES, ORDERED_SPLIT /* LANES, and STREAM for the clusters of ORDERED_LARGE members and more */ };

constexpr uint32_t STREAM_BLOCK_BYTES = 128, STREAM_THREADS = 128, STAGED_THREADS = 512;
constexpr uint32_t ORDERED_LARGE = 256;
constexpr uint32_t STREAM_GROUPS = 6144;

struct OrderedSumRoute {
	OrderedSumKernel kernel;
	uint32_t block_dims, blocks; /* all but ORDERED_LANES: coordinates and number of the blocks of a row; a work-group per cluster and block */
};

/* clusters of ORDERED_LARGE members among n points (fewer than there are clusters wherever ORDERED_SPLIT is taken) */
inline uint32_t ordered_most_large(uint32_t n) { return n / ORDERED_LARGE; }

/* A launch has fewer than 2^32 work-items. (Beyond: ORDERED_LANES, a work-item per coordinate or 16-byte piece) */
inline bool ordered_launch_holds(uint64_t groups, uint32_t threads) { return groups * threads <= 0xFFFFFFFFull; }

/*
 * whole_pieces: AoS rows of whole, aligned 16-byte pieces whose stride in bytes fits 32 bits.
 *
 * ORDERED_STREAM (all of an iteration, us, the kernels below -> this: N = 2M, d = 32, k = 1024 421 -> 332; N = 30k, d = 512, k = 512 167 -> 109; N = 40k,
 * d = 32, k = 1024 57 -> 51; N = 10240, d = 20, k = 128 29.8 -> 29.4; N = 20k, d = 100, k = 1000 75 -> 79; rows of a piece or two: N = 1M, d = 4,
 * k = 4096 194 -> 191, N = 270k 127 -> 131).
 *
 * ORDERED_SPLIT: a work-group costs 2.5 us however few its members, which 1024 of them at a time have to hide behind the memory; small clusters in more than
 * STREAM_GROUPS blocks leave that to the lane-per-chain kernel, whose chains are all under way at once (all of the update, us, every cluster streamed and this:
 * 32 members, k = 3000, d = 128 47, 36; d = 512 119, 58; d = 1000 251, 107; k = 8000, d = 32 80, 74; 128 members, k = 1024, d = 512 78, 64; doubles, d = 256
 * 83, 68; k = 8000, d = 16 134, 128). One large cluster among them would hold that kernel up, at 69 ns a member instead of 5 (N = 1M, d = 64, k = 5000, half of the
 * points in one cluster: 36 ms, this 2.6), so those are listed and streamed first, which takes 5 us when there are none. In fewer blocks, or with 256 members
 * and more, that does not pay (128 members, k = 1024, doubles, d = 64 35, 48; k = 3000, d = 16 41, 50; 256 members, k = 1024, d = 512 128, 215).
 *
 * ORDERED_STAGED: clusters of a few dozen members leave a work-group of eight wavefronts nothing to overlap, the more so the more clusters there are
 * (all of the update, us, staged and not: N = 80k, d = 32, k = 1024 31, 37; N = 40k 31, 30; d = 4, k = 4096: N = 1M 114, 116; N = 270k 77, 64).
 * Blocks of 32 coordinates are whole cache lines; of 16, twice as many work-groups and half the pieces per member, which long
 * chains want (N = 2M, d = 32, k = 1024 261 -> 231; N = 1M, d = 64, k = 100 388 -> 274) and the others do not (N = 500k, d = 500,
 * k = 200 432 -> 479; N = 100k, d = 32, k = 1024 34 -> 38).
 */
inline OrderedSumRoute ordered_sum_route(uint32_t value_bytes, bool whole_pieces, uint32_t dim, uint32_t k, uint32_t n)
{
	const uint32_t members = n / k;
	if (whole_pieces) {
		const uint32_t pieces = dim / (16 / value_bytes), block_dims = STREAM_BLOCK_BYTES / value_bytes, blocks = (dim + block_dims - 1) / block_dims;
		if (members >= (pieces <= 2 ? 128u : 32u)) {
			if (members < ORDERED_LARGE && (uint64_t)k * blocks > STREAM_GROUPS) {
				if (n >= ORDERED_LARGE && ordered_launch_holds((uint64_t)ordered_most_large(n) * blocks, STREAM_THREADS)) return OrderedSumRoute{ ORDERED_SPLIT, block_dims, blocks };
			}
			else if (ordered_launch_holds((uint64_t)k * blocks, STREAM_THREADS)) return OrderedSumRoute{ ORDERED_STREAM, block_dims, blocks };
		}
	}
	const uint32_t block_dims = members >= 512 && (uint64_t)k * ((dim + 31) / 32) <= 1024 ? 16 : 32, blocks = (dim + block_dims - 1) / block_dims;
	if (members >= ((uint64_t)k * blocks <= 2048 ? 64u : 256u) && ordered_launch_holds((uint64_t)k * blocks, STAGED_THREADS)) return OrderedSumRoute{ ORDERED_STAGED, block_dims, blocks };
	return OrderedSumRoute{ ORDERED_LANES, 0, 0 };
}

} // namespace kmx

#endif
