/*
 * KMX_UPDATE_SERIAL_ORDER: the update step with the bits of the serial loop, in O(n dim) work.
 *
 * The reference's CPU k-means adds the members of a cluster in ascending point order, one fp32 (or fp64) addition per
 * member and coordinate, starting from zero, and divides by the member count (serial.hpp:44-73). Floating-point
 * addition is not associative, so only that very order gives those very bits -- but the order only matters INSIDE a
 * cluster and coordinate: the k x dim chains are independent. This variant therefore
 *   1. sorts the point numbers by cluster with a STABLE counting sort (points of one cluster stay in ascending order):
 *      per-chunk histograms -> exclusive scan over (cluster, chunk) -> a wavefront per chunk (or part of one) walks its points in
 *      order, 64 at a time, and ranks the lanes that share a cluster by their lane number (ballots, no returning
 *      atomics, whose order would be arbitrary);
 *   2. gives every (cluster, coordinate) chain to one lane, which adds the rows of the sorted list one after the other
 *      with plain additions (no fused operations, no tree) and divides like divideMeansKernel.
 * A whole Lloyd run with this update and any assignment variant (all return the serial index) is bit-identical to the
 * reference's serial run. The price is the length of the longest chain: a cluster of m members is m dependent
 * additions, whatever the machine.
 *
 * Kernels: ordered_histogram_kernel, ordered_offsets_kernel, ordered_starts_kernel, ordered_scatter_kernel / ordered_scatter_group_kernel, ordered_large_kernel,
 * ordered_stream_sum_kernel / ordered_staged_sum_kernel / ordered_sum_kernel.
 */
#include "kmx_internal.h"
#include "update_ordered_route.h"

#include <algorithm>
#include <type_traits>

namespace kmx {

constexpr uint32_t ORDERED_LDS_CLUSTERS = 16384; /* up to here a chunk's counters live in LDS (64 KB per wavefront-sized work-group) */
constexpr uint32_t ORDERED_HIST_WORDS = 1u << 21; /* bound of chunks x k */
constexpr uint32_t ORDERED_MAX_CHUNKS = 4096;
/* wavefronts that share a chunk's row of the histogram, each with counters of its own in LDS while it scatters: 64 KB of them at most */
constexpr uint32_t ordered_group(uint32_t k) { return k <= 2048 ? 8 : k <= 4096 ? 4 : 1; }

/*
 * Histogram of one chunk of points: hist[chunk][cluster]. One work-group per chunk, the same chunks as the scatter.
 * IN_LDS: counters in LDS, the row is written out whole (nothing to clear beforehand); otherwise (one wavefront) the row in global
 * memory is the counter array (cleared by the launcher) and takes the atomics directly -- it belongs to this wavefront,
 * but two lanes may hold the same cluster.
 */
template <bool IN_LDS>
__global__ void __launch_bounds__(512)
ordered_histogram_kernel(const uint32_t* __restrict__ assignment, uint32_t* __restrict__ hist, uint32_t k, uint32_t n, uint32_t chunk_points)
{
	extern __shared__ uint32_t counters[];
	const uint32_t tid = threadIdx.x, threads = blockDim.x;
	uint32_t* row = hist + (size_t)blockIdx.x * k;
	const uint32_t begin = blockIdx.x * chunk_points;          /* chunks * chunk_points < 2^32: the launcher keeps n below 2^32 - 2^20 */
	const uint32_t end = min(n, begin + chunk_points);
	if (IN_LDS) {
		for (uint32_t c = tid; c < k; c += threads) counters[c] = 0u;
		__syncthreads();
	}
	constexpr uint32_t BATCH = 8; /* loads in flight */
	for (uint32_t i0 = begin + tid; i0 < end; i0 += BATCH * threads) {
		uint32_t c[BATCH];
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u) c[u] = i0 + u * threads < end ? assignment[i0 + u * threads] : 0xFFFFFFFFu;
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u) {
			if (c[u] >= k) continue; /* not a cluster: the point is left out, as by the scatter */
			if (IN_LDS) atomicAdd(&counters[c[u]], 1u);
			else atomicAdd(&row[c[u]], 1u);
		}
	}
	if (IN_LDS) {
		__syncthreads();
		for (uint32_t c = tid; c < k; c += threads) row[c] = counters[c];
	}
}

/*
 * hist[chunk][c] := number of members of cluster c in the chunks before `chunk` (exclusive scan along the chunks, in place), and the
 * sizes. A work-group takes 16 clusters (64 bytes of every row), 64 lanes share out the rows of a cluster: each adds its share,
 * the shares are scanned in LDS, each walks its share again (from L2). Loads go out SCAN_BATCH at a time: what bounds it is their
 * latency (one lane per cluster and 128 rows, one load after the other, in two launches: 52 us at 2048 chunks, k = 1024).
 */
constexpr uint32_t SCAN_COLUMNS = 16, SCAN_SHARES = 64, SCAN_BATCH = 16;

__global__ void __launch_bounds__(SCAN_COLUMNS * SCAN_SHARES)
ordered_offsets_kernel(uint32_t* __restrict__ hist, uint32_t* __restrict__ sizes, uint32_t k, uint32_t chunks)
{
	__shared__ uint32_t share_sum[SCAN_SHARES][SCAN_COLUMNS];
	const uint32_t column = threadIdx.x % SCAN_COLUMNS, share = threadIdx.x / SCAN_COLUMNS;
	const uint32_t c = min(blockIdx.x * SCAN_COLUMNS + column, k - 1);
	const bool mine = blockIdx.x * SCAN_COLUMNS + column < k;
	const uint32_t per = (chunks + SCAN_SHARES - 1) / SCAN_SHARES;
	const uint32_t c0 = min(chunks, share * per), c1 = min(chunks, c0 + per);
	uint32_t sum = 0;
	for (uint32_t base = c0; base < c1; base += SCAN_BATCH) {
		uint32_t v[SCAN_BATCH];
#pragma unroll
		for (uint32_t u = 0; u < SCAN_BATCH; ++u) v[u] = hist[(size_t)min(base + u, c1 - 1) * k + c];
#pragma unroll
		for (uint32_t u = 0; u < SCAN_BATCH; ++u) sum += base + u < c1 ? v[u] : 0u;
	}
	uint32_t upto = sum; /* of this share and those before it */
	share_sum[share][column] = sum;
#pragma unroll
	for (uint32_t off = 1; off < SCAN_SHARES; off <<= 1) {
		__syncthreads();
		const uint32_t before = share >= off ? share_sum[share - off][column] : 0u;
		__syncthreads();
		upto += before;
		share_sum[share][column] = upto;
	}
	if (mine && share == SCAN_SHARES - 1) sizes[c] = upto;
	uint32_t running = upto - sum;
	for (uint32_t base = c0; base < c1; base += SCAN_BATCH) {
		uint32_t v[SCAN_BATCH];
#pragma unroll
		for (uint32_t u = 0; u < SCAN_BATCH; ++u) v[u] = hist[(size_t)min(base + u, c1 - 1) * k + c];
#pragma unroll
		for (uint32_t u = 0; u < SCAN_BATCH; ++u) {
			if (base + u < c1 && mine) hist[(size_t)(base + u) * k + c] = running;
			running += base + u < c1 ? v[u] : 0u;
		}
	}
}

/* starts[c] = sizes[0] + ... + sizes[c - 1]: one work-group, 1024 clusters per step, wavefront sums meet in LDS */
__global__ void __launch_bounds__(1024)
ordered_starts_kernel(const uint32_t* __restrict__ sizes, uint32_t* __restrict__ starts, uint32_t k)
{
	__shared__ uint32_t wave_sum[2][16];
	const uint32_t lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
	uint32_t running = 0, buffer = 0;
	for (uint32_t base = 0; base < k; base += 1024, buffer ^= 1) {
		const uint32_t c = base + threadIdx.x;
		const uint32_t members = c < k ? sizes[c] : 0u;
		uint32_t upto = members; /* inclusive within the wavefront */
#pragma unroll
		for (uint32_t off = 1; off < WAVE; off <<= 1) {
			const uint32_t below = (uint32_t)__shfl_up((int)upto, off);
			if (lane >= off) upto += below;
		}
		if (lane == WAVE - 1) wave_sum[buffer][wave] = upto;
		__syncthreads(); /* (two buffers: the next step writes the other one) */
		uint32_t before = running;
		for (uint32_t v = 0; v < 16; ++v) {
			const uint32_t sum = wave_sum[buffer][v];
			before += v < wave ? sum : 0u;
			running += sum;
		}
		if (c < k) starts[c] = before + upto - members;
	}
}

/*
 * sorted[starts[c] + members of c in earlier chunks + rank inside the chunk] = point number. One wavefront per chunk
 * walks its points in ascending order, 64 per step. Inside a step the lanes that share a cluster are ranked by lane
 * number: one ballot per bit of the cluster number leaves every lane the mask of the lanes with its cluster, a lane's rank is
 * the number of those below it (naming the clusters of a step one after the other took up to 64 ballots, 48 instead of 32 us at
 * N = 2M, k = 1024). The cluster's counter then moves on by the size of the group (written
 * by its last lane, after every lane of the group has read it: one wavefront, in program order). The order inside a
 * cluster is therefore the point order, which no returning atomic would promise.
 */
template <bool IN_LDS>
__global__ void __launch_bounds__(64)
ordered_scatter_kernel(const uint32_t* __restrict__ assignment, uint32_t* __restrict__ hist, const uint32_t* __restrict__ starts,
                       uint32_t* __restrict__ sorted, uint32_t k, uint32_t n, uint32_t chunk_points)
{
	extern __shared__ uint32_t counters[];
	const uint32_t lane = threadIdx.x;
	uint32_t* row = hist + (size_t)blockIdx.x * k;
	if (IN_LDS) {
		constexpr uint32_t BATCH = 8; /* loads in flight (one pair of loads at a time was a third of the kernel) */
		for (uint32_t c0 = lane; c0 < k; c0 += BATCH * WAVE) {
			uint32_t first[BATCH];
#pragma unroll
			for (uint32_t u = 0; u < BATCH; ++u) {
				const uint32_t c = min(c0 + u * WAVE, k - 1);
				first[u] = starts[c] + row[c];
			}
#pragma unroll
			for (uint32_t u = 0; u < BATCH; ++u)
				if (c0 + u * WAVE < k) counters[c0 + u * WAVE] = first[u];
		}
	}
	else
		for (uint32_t c = lane; c < k; c += WAVE) __hip_atomic_store(&row[c], starts[c] + row[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
	if (!IN_LDS) __threadfence();
	__syncthreads();
	uint32_t* next = IN_LDS ? counters : row;
	const unsigned long long below = (1ull << lane) - 1ull;
	const uint32_t bits = 32 - (uint32_t)__builtin_clz(k - 1 | 1u);
	const uint32_t begin = blockIdx.x * chunk_points;
	const uint32_t end = min(n, begin + chunk_points);
	uint32_t cluster = begin + lane < end ? assignment[begin + lane] : 0xFFFFFFFFu;
	for (uint32_t base = begin; base < end; base += WAVE) {
		const uint32_t i = base + lane, c = cluster;
		if (base + WAVE < end) cluster = i + WAVE < end ? assignment[i + WAVE] : 0xFFFFFFFFu; /* of the next step */
		/* the lanes with this lane's cluster: those that agree in every bit of it */
		unsigned long long same = __ballot(c < k);
		for (uint32_t bit = 0; bit < bits; ++bit) {
			const bool set = (c >> bit) & 1u;
			const unsigned long long with = __ballot(set);
			same &= set ? with : ~with;
		}
		const uint32_t rank = (uint32_t)__popcll(same & below), group = (uint32_t)__popcll(same);
		if (c < k) {
			/* counters in global memory: read and written past the vector cache, and fenced below, so that the lanes of the
			 * next step see what this step wrote */
			const uint32_t slot = (IN_LDS ? next[c] : __hip_atomic_load(&next[c], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) + rank;
			sorted[slot] = i;
			if (rank + 1 == group) {
				if (IN_LDS) next[c] = slot + 1;
				else __hip_atomic_store(&next[c], slot + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
		}
		if (!IN_LDS) __threadfence();
	}
}

/*
 * The same by work-groups of GROUP wavefronts, which share a row of the histogram: each counts its part of the chunk first (so there is an
 * eighth of the rows to write, scan and read; N = 2M, k = 1024, us, a row per wavefront -> this: counting 11 -> 4.6, scanning 13 -> 4.9, starts 4.7 -> 0, scattering
 * 29 -> 18) and starts behind the wavefronts before it. Every work-group finds the clusters' starts for itself from their sizes, the first one leaves them for the sums.
 * Neighbouring chunks go to the same XCD, whose L2 then holds whole lines of the sorted list before they are written back.
 */
template <uint32_t GROUP>
__global__ void __launch_bounds__(GROUP * WAVE)
ordered_scatter_group_kernel(const uint32_t* __restrict__ assignment, const uint32_t* __restrict__ hist, const uint32_t* __restrict__ sizes, uint32_t* __restrict__ starts,
                             uint32_t* __restrict__ sorted, uint32_t k, uint32_t n, uint32_t chunk_points)
{
	constexpr uint32_t THREADS = GROUP * WAVE, XCDS = 8;
	extern __shared__ uint32_t counters[]; /* GROUP rows of k */
	__shared__ uint32_t wave_sum[GROUP];
	const uint32_t tid = threadIdx.x, lane = tid % WAVE, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t xcd = blockIdx.x % XCDS, chunk = xcd * (gridDim.x / XCDS) + min(xcd, gridDim.x % XCDS) + blockIdx.x / XCDS;
	const uint32_t* row = hist + (size_t)chunk * k;
	const uint32_t part = chunk_points / GROUP; /* (whole steps of 64 points) */
	const uint32_t begin = min(n, chunk * chunk_points + wave * part), end = min(n, begin + part);
	/* this lane's share of the clusters: neighbours */
	const uint32_t each = (k + THREADS - 1) / THREADS, c0 = min(k, tid * each), c1 = min(k, c0 + each);
	uint32_t members = 0;
	for (uint32_t c = c0; c < c1; ++c) members += sizes[c];
	for (uint32_t c = tid; c < GROUP * k; c += THREADS) counters[c] = 0u;
	uint32_t upto = members; /* inclusive within the wavefront */
#pragma unroll
	for (uint32_t off = 1; off < WAVE; off <<= 1) {
		const uint32_t below = (uint32_t)__shfl_up((int)upto, off);
		if (lane >= off) upto += below;
	}
	if (lane == WAVE - 1) wave_sum[wave] = upto;
	__syncthreads();
	uint32_t* next = counters + wave * k;
	constexpr uint32_t BATCH = 8; /* loads in flight */
	for (uint32_t i0 = begin + lane; i0 < end; i0 += BATCH * WAVE) {
		uint32_t c[BATCH];
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u) c[u] = i0 + u * WAVE < end ? assignment[i0 + u * WAVE] : 0xFFFFFFFFu;
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u)
			if (c[u] < k) atomicAdd(&next[c[u]], 1u);
	}
	__syncthreads();
	uint32_t start = upto - members;
	for (uint32_t v = 0; v < wave; ++v) start += wave_sum[v];
	for (uint32_t c = c0; c < c1; ++c) {
		if (chunk == 0) starts[c] = start;
		uint32_t running = start + row[c];
		start += sizes[c];
#pragma unroll
		for (uint32_t v = 0; v < GROUP; ++v) {
			const uint32_t count = counters[v * k + c];
			counters[v * k + c] = running;
			running += count;
		}
	}
	__syncthreads();
	const unsigned long long below = (1ull << lane) - 1ull;
	const uint32_t bits = 32 - (uint32_t)__builtin_clz(k - 1 | 1u);
	uint32_t cluster = begin + lane < end ? assignment[begin + lane] : 0xFFFFFFFFu;
	for (uint32_t base = begin; base < end; base += WAVE) {
		const uint32_t i = base + lane, c = cluster;
		if (base + WAVE < end) cluster = i + WAVE < end ? assignment[i + WAVE] : 0xFFFFFFFFu; /* of the next step */
		unsigned long long same = __ballot(c < k);
		for (uint32_t bit = 0; bit < bits; ++bit) {
			const bool set = (c >> bit) & 1u;
			const unsigned long long with = __ballot(set);
			same &= set ? with : ~with;
		}
		const uint32_t rank = (uint32_t)__popcll(same & below), group = (uint32_t)__popcll(same);
		if (c < k) {
			const uint32_t slot = next[c] + rank;
			sorted[slot] = i;
			if (rank + 1 == group) next[c] = slot + 1;
		}
	}
}

/* large[0] = how many clusters have at least `least` members, then their numbers in no particular order: one work-group, 1024 clusters per step */
__global__ void __launch_bounds__(1024)
ordered_large_kernel(const uint32_t* __restrict__ sizes, uint32_t* __restrict__ large, uint32_t k, uint32_t least)
{
	__shared__ uint32_t count;
	if (threadIdx.x == 0) count = 0u;
	__syncthreads();
	constexpr uint32_t BATCH = 4; /* loads in flight */
	for (uint32_t c0 = threadIdx.x; c0 < k; c0 += BATCH * 1024) {
		uint32_t members[BATCH];
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u) members[u] = c0 + u * 1024 < k ? sizes[c0 + u * 1024] : 0u;
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u)
			if (members[u] >= least) large[1 + atomicAdd(&count, 1u)] = c0 + u * 1024;
	}
	__syncthreads();
	if (threadIdx.x == 0) large[0] = count;
}

/*
 * One lane per cluster and piece of VEC consecutive coordinates (VEC = 1, or a 16-byte piece of an AoS row): the members'
 * coordinates added one after the other in the order of the sorted list, i.e. in ascending point number, starting from
 * zero like the serial loop (serial.hpp:57-63), then the guarded divide (serial.hpp:65-71). The additions of a
 * coordinate are a chain; what can overlap are the loads: the pieces of UNROLL rows are in flight together, and the
 * point numbers of the next UNROLL rows are requested before the current ones are added (a chain is as many sums as
 * the machine runs at once here, so the time is the latency of a load divided by the loads in flight). Clusters of `most` members and more
 * are left out.
 */
template <typename F, int VEC> struct alignas(sizeof(F) * VEC) OrderedPiece { F v[VEC]; };

template <typename F, int LD, int LM, int VEC, int UNROLL>
__global__ void __launch_bounds__(64)
ordered_sum_kernel(const F* __restrict__ data, size_t stride, const uint32_t* __restrict__ sorted, const uint32_t* __restrict__ starts,
                   const uint32_t* __restrict__ sizes, F* __restrict__ means, size_t stride_means, uint32_t dim, uint32_t k, uint32_t divide, uint32_t most)
{
	static_assert(VEC == 1 || LD == KMX_AOS, "pieces of several coordinates are pieces of AoS rows");
	typedef OrderedPiece<F, VEC> piece_t;
	const uint32_t pieces = dim / VEC; /* the launcher picks VEC among the divisors of dim */
	const size_t e = (size_t)blockIdx.x * WAVE + threadIdx.x;
	if (e >= (size_t)k * pieces) return;
	const uint32_t c = (uint32_t)(e / pieces), d = (uint32_t)(e % pieces) * VEC;
	const uint32_t members = sizes[c];
	if (members >= most) return; /* left to ordered_stream_sum_kernel */
	const uint32_t begin = starts[c], end = begin + members;
	piece_t sum;
#pragma unroll
	for (int i = 0; i < VEC; ++i) sum.v[i] = (F)0;
	if (members) {
		uint32_t point[UNROLL];
#pragma unroll
		for (int u = 0; u < UNROLL; ++u) point[u] = sorted[min(begin + u, end - 1)];
		for (uint32_t j = begin; j < end; j += UNROLL) {
			piece_t v[UNROLL];
#pragma unroll
			for (int u = 0; u < UNROLL; ++u) v[u] = *(const piece_t*)(data + elem<LD>(stride, point[u], d));
#pragma unroll
			for (int u = 0; u < UNROLL; ++u) point[u] = sorted[min(j + UNROLL + u, end - 1)];
#pragma unroll
			for (int u = 0; u < UNROLL; ++u) {
				if (j + u < end) {
#pragma unroll
					for (int i = 0; i < VEC; ++i) sum.v[i] = sum.v[i] + v[u].v[i];
				}
			}
		}
	}
#pragma unroll
	for (int i = 0; i < VEC; ++i)
		means[elem<LM>(stride_means, c, d + i)] = !divide ? sum.v[i] : (members ? sum.v[i] / (F)members : (F)0);
}

/*
 * The same for clusters of many members: a work-group per cluster and block of up to 32 coordinates. All eight wavefronts fetch the
 * members' pieces (16 bytes each, STAGED_PIECES per lane) of the next few hundred rows into registers while the first one adds
 * the last fetch from LDS, a lane per coordinate, four members per LDS read. The chain then runs at the latency of an addition and an LDS read
 * instead of a trip to memory per 32 rows. What bounds it: with clusters far larger than a fetch that chain (N = 4M, d = 16, k = 16, all of
 * it 33 -> 7.5 ms); with clusters of a few fetches the trips to memory, which nothing hides then (N = 2M, d = 32, k = 1024: 389 -> 125 us, 2.1 TB/s;
 * 2048 work-groups, two per compute unit and so four rounds, of two fetches each: 36 cycles per addition, with 16 of 512 lanes adding).
 * ELEMENTS: SoA points, rows shorter than a piece: single coordinates, consecutive lanes take consecutive members.
 */
constexpr uint32_t STAGED_PIECES = 8;

template <typename F, int LD, int LM, bool ELEMENTS>
__global__ void __launch_bounds__(STAGED_THREADS, 4)
ordered_staged_sum_kernel(const F* __restrict__ data, size_t stride, const uint32_t* __restrict__ sorted, const uint32_t* __restrict__ starts,
                          const uint32_t* __restrict__ sizes, F* __restrict__ means, size_t stride_means, uint32_t dim, uint32_t blocks, uint32_t block_dims, uint32_t divide)
{
	constexpr uint32_t PIECE = ELEMENTS ? 1 : 16 / sizeof(F), QUAD = 16 / sizeof(F); /* (QUAD: members per LDS read) */
	typedef F piece_any __attribute__((ext_vector_type(PIECE), aligned(sizeof(F))));
	typedef F quad_t __attribute__((ext_vector_type(QUAD)));
	extern __shared__ __attribute__((aligned(16))) char staged_lds[];
	F* columns = (F*)staged_lds;
	const uint32_t c = blockIdx.x / blocks, block = blockIdx.x % blocks;
	const uint32_t d0 = block * block_dims, width = min(block_dims, dim - d0); /* (ELEMENTS = false: width >= PIECE, see the launcher) */
	const uint32_t members = sizes[c], begin = starts[c];
	const uint32_t tid = threadIdx.x;
	const uint32_t pieces = (width + PIECE - 1) / PIECE;
	const uint32_t step = STAGED_THREADS * STAGED_PIECES / pieces / QUAD * QUAD; /* members per fetch */
	const uint32_t column = step + QUAD;                                         /* (the padding spreads the columns over the banks) */
	/* piece q of a fetch: its member there and its coordinate; the last piece ends with the block */
	uint32_t member_of[STAGED_PIECES], at_of[STAGED_PIECES];
#pragma unroll
	for (uint32_t i = 0; i < STAGED_PIECES; ++i) {
		const uint32_t q = tid + i * STAGED_THREADS;
		member_of[i] = ELEMENTS ? q % step : q / pieces;
		const uint32_t piece = ELEMENTS ? q / step : q % pieces;
		at_of[i] = min(piece * PIECE, width - PIECE);
		if (member_of[i] >= step || piece >= pieces) member_of[i] = 0xFFFFFFFFu; /* beyond the fetch */
	}
	uint32_t point[STAGED_PIECES];
	piece_any v[STAGED_PIECES];
	auto name = [&](uint32_t first) { /* the points of the fetch that starts with member `first` */
#pragma unroll
		for (uint32_t i = 0; i < STAGED_PIECES; ++i)
			if (member_of[i] < step && first + member_of[i] < members) point[i] = sorted[begin + first + member_of[i]];
	};
	auto fetch = [&](uint32_t first) {
#pragma unroll
		for (uint32_t i = 0; i < STAGED_PIECES; ++i)
			if (member_of[i] < step && first + member_of[i] < members) v[i] = *(const piece_any*)(data + elem<LD>(stride, point[i], d0 + at_of[i]));
	};
	F sum = (F)0;
	if (members) {
		name(0);
		fetch(0);
		if (step < members) name(step);
	}
	for (uint32_t first = 0; first < members; first += step) {
		__syncthreads(); /* the members in LDS have been added */
#pragma unroll
		for (uint32_t i = 0; i < STAGED_PIECES; ++i)
			if (member_of[i] < step && first + member_of[i] < members) {
#pragma unroll
				for (uint32_t e = 0; e < PIECE; ++e) columns[(at_of[i] + e) * column + member_of[i]] = v[i][e];
			}
		__syncthreads();
		if (first + step < members) {
			fetch(first + step);
			if (first + 2 * step < members) name(first + 2 * step);
		}
		if (tid < width) {
			const uint32_t here = min(step, members - first);
			const F* mine = columns + tid * column;
			constexpr uint32_t READS = 4;
			uint32_t r = 0;
			for (; r + READS * QUAD <= here; r += READS * QUAD) {
				quad_t x[READS];
#pragma unroll
				for (uint32_t u = 0; u < READS; ++u) x[u] = *(const quad_t*)(mine + r + u * QUAD);
#pragma unroll
				for (uint32_t u = 0; u < READS; ++u)
#pragma unroll
					for (uint32_t e = 0; e < QUAD; ++e) sum = sum + x[u][e];
			}
			for (; r < here; ++r) sum = sum + mine[r];
		}
	}
	if (tid < width) means[elem<LM>(stride_means, c, d0 + tid)] = !divide ? sum : (members ? sum / (F)members : (F)0);
}

/*
 * The same for AoS rows of whole 16-byte pieces: a work-group per cluster (`large`: of that list only) and block of 128 bytes of the row. One wavefront requests the members'
 * rows straight to LDS, AHEAD batches of eight requests before they are added, and the members' numbers AHEAD batches before that; the other one
 * adds, a lane per coordinate, two members per LDS read, three parts of eight to 16 members on their way from LDS, across the barrier between two batches too.
 * What bounds it is the longest cluster's chain, at 1.5 to 1.6 instructions a member, which a wavefront alone issues every five cycles (rows of 16 bytes 2.9 ns a
 * member, of 128 bytes 4.0; with one part on its way, from anew in every batch, 3.6 and 4.9; with one wavefront that requests and adds 7.8), then the memory
 * (N = 2M, d = 32, k = 1024: 64 us, with one part 77; one wavefront 107, the staged kernel above 169). AHEAD of 1, 2, 3, 4 with one wavefront: 133, 106,
 * 107, 122 us (four work-groups fit a compute unit with up to 3).
 */
constexpr uint32_t STREAM_REQUESTS = 8, STREAM_SLOT_BYTES = STREAM_REQUESTS * WAVE * 16;
static_assert(STREAM_THREADS == 2 * WAVE, "one wavefront requests, one adds");
constexpr uint32_t stream_rows(uint32_t pieces) { return WAVE / pieces; }                     /* per request */
constexpr uint32_t stream_batch(uint32_t pieces) { return STREAM_REQUESTS * stream_rows(pieces); }
constexpr uint32_t stream_names(uint32_t pieces) { return (stream_batch(pieces) + WAVE - 1) / WAVE; } /* requests for a batch's numbers */
/* (a wavefront's wait can leave up to 63 requests on their way) */
constexpr uint32_t stream_ahead(uint32_t pieces, bool deep) { return !deep ? 3 : std::min(6u, 63 / (STREAM_REQUESTS + stream_names(pieces)) + 1); }
constexpr uint32_t stream_lds_bytes(uint32_t pieces, bool deep) { return (stream_ahead(pieces, deep) + 1) * (STREAM_SLOT_BYTES + stream_names(pieces) * WAVE * 4); }

/* straight to LDS: 16 (4) bytes per lane, lane by lane behind `to`, a uniform byte offset. Waits are the caller's (vmcnt) */
__device__ __forceinline__ void stream_request16(const void* from, uint32_t to)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(to), "v"(from) : "m0", "memory");
}
__device__ __forceinline__ void stream_request4(const void* from, uint32_t to)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" : : "s"(to), "v"(from) : "m0", "memory");
}

template <typename F, int LM, uint32_t P, bool DEEP>
__global__ void __launch_bounds__(STREAM_THREADS)
ordered_stream_sum_kernel(const F* __restrict__ data, size_t stride, const uint32_t* __restrict__ sorted, const uint32_t* __restrict__ starts,
                          const uint32_t* __restrict__ sizes, const uint32_t* __restrict__ large, F* __restrict__ means, size_t stride_means, uint32_t dim, uint32_t blocks, uint32_t divide)
{
	constexpr uint32_t PIECE = 16 / sizeof(F), BLOCK = STREAM_BLOCK_BYTES / sizeof(F), ROWS = stream_rows(P), BATCH = stream_batch(P), NAMES = stream_names(P);
	constexpr uint32_t AHEAD = stream_ahead(P, DEEP), SLOTS = AHEAD + 1, EACH = STREAM_REQUESTS + NAMES;
	extern __shared__ __attribute__((aligned(16))) char stream_lds[];
	if (large && blockIdx.x / blocks >= large[0]) return;
	const uint32_t c = large ? large[1 + blockIdx.x / blocks] : blockIdx.x / blocks, d0 = blockIdx.x % blocks * BLOCK, width = min(BLOCK, dim - d0); /* (whole pieces, no more than P) */
	const uint32_t members = sizes[c], begin = starts[c], lane = threadIdx.x % WAVE;
	if (__builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE)) != 0) { /* requests */
		if (members == 0) return;
		const uint32_t rows_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)stream_lds, names_at = rows_at + SLOTS * STREAM_SLOT_BYTES;
		/* this lane's row of a request (lanes without one repeat the last) and its piece (a narrower last block repeats its last one) */
		const uint32_t row = min(lane / P, ROWS - 1);
		const F* piece = data + d0 + min(lane % P * PIECE, width - PIECE);
		const uint32_t row_bytes = (uint32_t)(stride * sizeof(F)); /* (below 2^32, see the launcher) */
		uint32_t named = 0, name_slot = 0, row_slot = 0; /* the next batch to be named, and the slots names and rows go to (rows: by the names of that slot) */
		auto request_names = [&]() {
#pragma unroll
			for (uint32_t i = 0; i < NAMES; ++i) /* (behind the last member, the last again: as many requests each time) */
				stream_request4(sorted + begin + min(named + i * WAVE + lane, members - 1), names_at + (name_slot * NAMES + i) * (WAVE * 4));
			named += BATCH;
			name_slot = name_slot + 1 < SLOTS ? name_slot + 1 : 0;
		};
		uint32_t point[STREAM_REQUESTS];
		auto read_names = [&]() {
			const uint32_t* names = (const uint32_t*)(stream_lds + SLOTS * STREAM_SLOT_BYTES) + row_slot * (NAMES * WAVE) + row;
#pragma unroll
			for (uint32_t j = 0; j < STREAM_REQUESTS; ++j) point[j] = names[j * ROWS];
		};
		auto request_rows = [&]() {
#pragma unroll
			for (uint32_t j = 0; j < STREAM_REQUESTS; ++j) stream_request16((const char*)piece + (uint64_t)point[j] * row_bytes, rows_at + row_slot * STREAM_SLOT_BYTES + j * (WAVE * 16));
			row_slot = row_slot + 1 < SLOTS ? row_slot + 1 : 0;
		};
		if (members <= AHEAD * BATCH) { /* all of it at once, and no more requests than there are members for */
			for (uint32_t i = 0; i * WAVE < members; ++i) stream_request4(sorted + begin + min(i * WAVE + lane, members - 1), names_at + i * (WAVE * 4));
			asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
			const uint32_t* names = (const uint32_t*)(stream_lds + SLOTS * STREAM_SLOT_BYTES);
			for (uint32_t j = 0; j * ROWS < members; ++j)
				stream_request16((const char*)piece + (uint64_t)names[min(j * ROWS + row, members - 1)] * row_bytes, rows_at + j * (WAVE * 16));
			asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
			for (uint32_t first = 0; first < members; first += BATCH) __syncthreads();
			return;
		}
#pragma unroll
		for (uint32_t i = 0; i < AHEAD; ++i) request_names();
		asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#pragma unroll
		for (uint32_t i = 0; i < AHEAD; ++i) { request_names(); read_names(); request_rows(); }
#pragma unroll 1
		for (uint32_t first = 0; first < members; first += BATCH) {
			/* the rows of this batch and the names of the one requested now are here (what was requested after them may not be) */
			asm volatile("s_waitcnt vmcnt(%0)" : : "n"((AHEAD - 1) * EACH) : "memory");
			read_names();
			__syncthreads(); /* the rows may be added, and those of the batch before have been */
			request_names();
			request_rows();
		}
		asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); /* (nothing may arrive in LDS that is no longer this work-group's) */
		return;
	}
	F sum = (F)0;
	const uint32_t own = min(lane, width - 1); /* this lane's coordinate */
	uint32_t from = 0;
	/* parts of a request's rows (a part behind the last row is read, not added) */
	constexpr uint32_t PART = ROWS <= 16 ? ROWS : ROWS % 16 == 0 ? 16 : 7, PARTS = ROWS / PART, ALL = STREAM_REQUESTS * PARTS;
	static_assert(ROWS % PART == 0 && ALL % 4 == 0, "whole parts, whole rounds");
	/* three parts are on their way while one is added, across the barrier between two batches too (the first time round zeros, which the sum of nothing takes
	 * without a trace) */
	F x[4][PART];
#pragma unroll
	for (uint32_t u = 1; u < 4; ++u)
#pragma unroll
		for (uint32_t r = 0; r < PART; ++r) x[u][r] = (F)0;
	auto add = [&](const F (&part)[PART]) {
#pragma unroll
		for (uint32_t r = 0; r < PART; ++r) sum = sum + part[r];
	};
	uint32_t first = 0;
#pragma unroll 1
	for (; first + BATCH <= members; first += BATCH) {
		__syncthreads();
		const F* mine = (const F*)(stream_lds + from * STREAM_SLOT_BYTES) + own;
		from = from + 1 < SLOTS ? from + 1 : 0;
#pragma unroll
		for (uint32_t at = 0; at < ALL; ++at) {
#pragma unroll
			for (uint32_t r = 0; r < PART; ++r) x[at % 4][r] = mine[at / PARTS * (WAVE * PIECE) + (at % PARTS * PART + r) * (P * PIECE)];
			__builtin_amdgcn_sched_barrier(0);
			add(x[(at + 1) % 4]);
			__builtin_amdgcn_sched_barrier(0);
		}
	}
	add(x[1]); add(x[2]); add(x[3]);
	if (first < members) { /* the last batch, not full */
		__syncthreads();
		const F* mine = (const F*)(stream_lds + from * STREAM_SLOT_BYTES) + own;
		const uint32_t here = members - first;
		auto read = [&](F (&into)[PART], uint32_t at) {
			at = min(at, ALL - 1);
#pragma unroll
			for (uint32_t r = 0; r < PART; ++r) into[r] = mine[at / PARTS * (WAVE * PIECE) + (at % PARTS * PART + r) * (P * PIECE)];
		};
		read(x[0], 0);
#pragma unroll 1
		for (uint32_t at = 0; at * PART < here; at += 2) {
#pragma unroll
			for (uint32_t u = 0; u < 2; ++u) {
				read(x[(u + 1) % 2], at + u + 1);
				__builtin_amdgcn_sched_barrier(0);
#pragma unroll
				for (uint32_t r = 0; r < PART; ++r) sum = (at + u) * PART + r < here ? sum + x[u][r] : sum;
				__builtin_amdgcn_sched_barrier(0);
			}
		}
	}
	if (lane < width) means[elem<LM>(stride_means, c, d0 + lane)] = !divide ? sum : (members ? sum / (F)members : (F)0);
}

/* Work-groups of one wavefront: what bounds this kernel is the number of cache lines a compute unit keeps in flight, so
 * the chains are spread over as many compute units as there are wavefronts (measured at N = 2M, d = 32, k = 1024: 32
 * work-groups of four wavefronts with 16-byte pieces 0.85 ms). The 16-byte pieces, which need a quarter of the lanes, are
 * taken only where they still leave two wavefronts per compute unit. */
template <typename F, int LD, int LM>
static int launch_ordered_sum(const F* data, size_t stride, const uint32_t* sorted, const uint32_t* starts, const uint32_t* sizes, uint32_t* large,
                              F* means, size_t stride_means, uint32_t dim, uint32_t k, uint32_t n, bool divide, const DeviceInfo& dev)
{
	constexpr int WIDE = 16 / sizeof(F);
	const bool fits = LD == KMX_AOS && dim % WIDE == 0 && stride % WIDE == 0 && ((uintptr_t)data & 15) == 0;
	const OrderedSumRoute route = ordered_sum_route(sizeof(F), fits && stride <= 0xFFFFFFFFu / sizeof(F), dim, k, n);
	uint32_t most = 0xFFFFFFFFu; /* members of a cluster that ordered_sum_kernel does not take */
	if constexpr (LD == KMX_AOS) {
		if (route.kernel == ORDERED_STREAM || route.kernel == ORDERED_SPLIT) {
			const bool split = route.kernel == ORDERED_SPLIT;
			if (split) {
				most = ORDERED_LARGE;
				KMX_LAUNCH_KERNEL(ordered_large_kernel, dim3(1), dim3(1024), 0, stream(), sizes, large, k, most);
				KMX_LAUNCH_CHECK("ordered_large_kernel");
			}
			const uint32_t pieces = std::min<uint32_t>(dim / WIDE, STREAM_BLOCK_BYTES / 16), groups = (split ? ordered_most_large(n) : k) * route.blocks;
			const bool deep = groups <= 2 * dev.compute_units;
			void (*kernel)(const F*, size_t, const uint32_t*, const uint32_t*, const uint32_t*, const uint32_t*, F*, size_t, uint32_t, uint32_t, uint32_t) = nullptr;
			uint32_t lds = 0;
			auto take = [&](auto tag) {
				constexpr uint32_t P = decltype(tag)::value;
				if (pieces != P) return;
				kernel = deep ? ordered_stream_sum_kernel<F, LM, P, true> : ordered_stream_sum_kernel<F, LM, P, false>;
				lds = stream_lds_bytes(P, deep);
			};
			take(std::integral_constant<uint32_t, 1>{}); take(std::integral_constant<uint32_t, 2>{}); take(std::integral_constant<uint32_t, 3>{}); take(std::integral_constant<uint32_t, 4>{});
			take(std::integral_constant<uint32_t, 5>{}); take(std::integral_constant<uint32_t, 6>{}); take(std::integral_constant<uint32_t, 7>{}); take(std::integral_constant<uint32_t, 8>{});
			KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
			KMX_LAUNCH_KERNEL(kernel, dim3(groups), dim3(STREAM_THREADS), lds, stream(), data, stride, sorted, starts, sizes, split ? (const uint32_t*)large : nullptr, means, stride_means, dim, route.blocks, divide ? 1u : 0u);
			KMX_LAUNCH_CHECK("ordered_stream_sum_kernel");
			if (!split) return KMX_OK;
		}
	}
	if (route.kernel == ORDERED_STAGED) {
		const uint32_t block_dims = route.block_dims, groups = k * route.blocks;
		const bool elements = LD == KMX_SOA || dim < (uint32_t)WIDE || (dim % block_dims != 0 && dim % block_dims < (uint32_t)WIDE);
		const uint32_t lds = STAGED_THREADS * STAGED_PIECES * (elements ? sizeof(F) : 16) + std::min(dim, block_dims) * 16;
		auto kernel = elements ? ordered_staged_sum_kernel<F, LD, LM, true> : ordered_staged_sum_kernel<F, KMX_AOS, LM, false>;
		KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
		KMX_LAUNCH_KERNEL(kernel, dim3(groups), dim3(STAGED_THREADS), lds, stream(), data, stride, sorted, starts, sizes, means, stride_means, dim, route.blocks, block_dims, divide ? 1u : 0u);
		KMX_LAUNCH_CHECK("ordered_staged_sum_kernel");
		return KMX_OK;
	}
	const bool wide = fits && (size_t)k * (dim / WIDE) >= (size_t)2 * WAVE * dev.compute_units;
	const size_t total = (size_t)k * (wide ? dim / WIDE : dim);
	const dim3 grid((uint32_t)((total + WAVE - 1) / WAVE));
	if (wide)
		KMX_LAUNCH_KERNEL((ordered_sum_kernel<F, KMX_AOS, LM, WIDE, 32>), grid, dim3(WAVE), 0, stream(),
		                   data, stride, sorted, starts, sizes, means, stride_means, dim, k, divide ? 1u : 0u, most);
	else
		KMX_LAUNCH_KERNEL((ordered_sum_kernel<F, LD, LM, 1, 32>), grid, dim3(WAVE), 0, stream(),
		                   data, stride, sorted, starts, sizes, means, stride_means, dim, k, divide ? 1u : 0u, most);
	KMX_LAUNCH_CHECK("ordered_sum_kernel");
	return KMX_OK;
}

template <typename F>
int launch_update_serial_order(const F* data, int layout, size_t stride, const uint32_t* assignment,
                               F* means, int layout_means, size_t stride_means, uint32_t* cluster_sizes,
                               uint32_t dim, uint32_t k, uint32_t n, bool divide, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	if (n > 0xFFFFFFFFu - (1u << 20)) return fail(KMX_ERR_UNSUPPORTED, "the serial-order update takes fewer than 2^32 - 2^20 points");
	if ((uint64_t)k * dim > 0xFFFFFFFFull * WAVE) return fail(KMX_ERR_UNSUPPORTED, "the serial-order update: k * dim is too large for one launch");
	/* chunks: `group` wavefronts each, a multiple of 64 points per wavefront, few enough that chunks x k counters stay small */
	const uint32_t group = ordered_group(k);
	uint32_t chunks = 0, chunk_points = WAVE;
	if (n > 0) {
		const uint32_t by_memory = std::max<uint32_t>(1, ORDERED_HIST_WORDS / k);
		chunks = (std::min<uint32_t>({ by_memory, ORDERED_MAX_CHUNKS, (n + 255) / 256 }) + group - 1) / group;
		chunk_points = ((n + chunks - 1) / chunks + group * WAVE - 1) / (group * WAVE) * (group * WAVE);
		chunks = (n + chunk_points - 1) / chunk_points;
	}
	const size_t hist_words = (size_t)std::max(chunks, 1u) * k;
	int rc = reserve_partials(ws, hist_words + k + n);
	if (rc) return rc;
	uint32_t* hist = (uint32_t*)ws->partials;
	uint32_t* starts = hist + hist_words;
	uint32_t* sorted = starts + k;
	const bool in_lds = k <= ORDERED_LDS_CLUSTERS;
	const uint32_t lds_bytes = in_lds ? k * 4 : 0;

	if constexpr (std::is_same<F, float>::value) {
		/* members are read row by row: SoA points go through an AoS copy like those of the other updates */
		UpdateArgs u{ data, layout, stride, assignment, means, layout_means, stride_means, cluster_sizes, dim, k, n };
		if (update_wants_rows(KMX_UPDATE_ATOMIC_SHM, u, exec, ws, dev)) {
			if ((rc = launch_rows_from_soa(data, stride, dim, n, ws, dev))) return rc;
			data = ws->rows_copy; layout = KMX_AOS; stride = dim;
		}
	}
	if ((rc = profile_begin(1))) return rc;
	exec->block_count = chunks;
	if (chunks > 0) {
		if (in_lds) {
			KMX_HIP(hipFuncSetAttribute((const void*)ordered_histogram_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
			KMX_LAUNCH_KERNEL((ordered_histogram_kernel<true>), dim3(chunks), dim3(group * WAVE), lds_bytes, stream(), assignment, hist, k, n, chunk_points);
		}
		else {
			rc = kmx_fill_zero_u32(hist, hist_words);
			if (rc) return rc;
			KMX_LAUNCH_KERNEL((ordered_histogram_kernel<false>), dim3(chunks), dim3(WAVE), 0, stream(), assignment, hist, k, n, chunk_points);
		}
		KMX_LAUNCH_CHECK("ordered_histogram_kernel");
	}
	KMX_LAUNCH_KERNEL(ordered_offsets_kernel, dim3((k + SCAN_COLUMNS - 1) / SCAN_COLUMNS), dim3(SCAN_COLUMNS * SCAN_SHARES), 0, stream(), hist, cluster_sizes, k, chunks);
	KMX_LAUNCH_CHECK("ordered_offsets_kernel");
	if (group == 1 || chunks == 0) {
		KMX_LAUNCH_KERNEL(ordered_starts_kernel, dim3(1), dim3(1024), 0, stream(), cluster_sizes, starts, k);
		KMX_LAUNCH_CHECK("ordered_starts_kernel");
	}
	if (chunks > 0) {
		if (group > 1) {
			auto kernel = group == 8 ? ordered_scatter_group_kernel<8> : ordered_scatter_group_kernel<4>;
			KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(group * lds_bytes)));
			KMX_LAUNCH_KERNEL(kernel, dim3(chunks), dim3(group * WAVE), group * lds_bytes, stream(), assignment, hist, cluster_sizes, starts, sorted, k, n, chunk_points);
		}
		else if (in_lds) {
			KMX_HIP(hipFuncSetAttribute((const void*)ordered_scatter_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
			KMX_LAUNCH_KERNEL((ordered_scatter_kernel<true>), dim3(chunks), dim3(WAVE), lds_bytes, stream(), assignment, hist, starts, sorted, k, n, chunk_points);
		}
		else
			KMX_LAUNCH_KERNEL((ordered_scatter_kernel<false>), dim3(chunks), dim3(WAVE), 0, stream(), assignment, hist, starts, sorted, k, n, chunk_points);
		KMX_LAUNCH_CHECK("ordered_scatter_kernel");
	}
	/* (the histograms are no longer needed: their first words take the list of the large clusters) */
	if (layout == KMX_AOS && layout_means == KMX_AOS) rc = launch_ordered_sum<F, KMX_AOS, KMX_AOS>(data, stride, sorted, starts, cluster_sizes, hist, means, stride_means, dim, k, n, divide, dev);
	else if (layout == KMX_AOS) rc = launch_ordered_sum<F, KMX_AOS, KMX_SOA>(data, stride, sorted, starts, cluster_sizes, hist, means, stride_means, dim, k, n, divide, dev);
	else if (layout_means == KMX_AOS) rc = launch_ordered_sum<F, KMX_SOA, KMX_AOS>(data, stride, sorted, starts, cluster_sizes, hist, means, stride_means, dim, k, n, divide, dev);
	else rc = launch_ordered_sum<F, KMX_SOA, KMX_SOA>(data, stride, sorted, starts, cluster_sizes, hist, means, stride_means, dim, k, n, divide, dev);
	if (rc) return rc;
	return profile_end(1);
}

template int launch_update_serial_order<float>(const float*, int, size_t, const uint32_t*, float*, int, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, bool, kmx_exec_params*, Workspace*, const DeviceInfo&);
template int launch_update_serial_order<double>(const double*, int, size_t, const uint32_t*, double*, int, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, bool, kmx_exec_params*, Workspace*, const DeviceInfo&);

} // namespace kmx
