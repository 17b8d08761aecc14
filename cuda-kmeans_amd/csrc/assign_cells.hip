/*
 * Assignment of rows of 2 to 4 dimensions through a grid of cells.
 *
 * The sweeps compare every point with every centroid; with so few dimensions what they spend is not the products but the search for
 * the smallest of k results (N = 4M, d = 4, k = 4096: 710 us, 0.04 ns per pair, four fifths of it vector instructions). Here the box around the
 * centroids (and some way beyond) is divided into 2^15 or 2^16 cells, every cell gets the list of the centroids that can be the
 * nearest of a point in it, and a point is compared with the twenty or so of its cell's list, in the serial arithmetic and in
 * ascending order: the result is the serial scan's, no certificate needed.
 *
 * A centroid stays off a cell's list if its smallest distance to the cell's box, squared, exceeds the smallest of all centroids'
 * largest ones by more than CELL_SLACK: the serial distances of any point of the box then compare the same way (they are off by at
 * most (d + 4) 2^-24 each). Boxes and centroids are taken relative to the grid's corner, where all coordinates are small, and a box
 * reaches CELL_MARGIN of its width beyond its edges, which covers the roundings of a point's coordinates there and of its cell.
 *
 * Points outside the grid, and those of cells without a list of their own (the lists take CELL_POOL_UNITS x 16 bytes; coordinates that
 * are not finite, squares that would overflow or underflow make the whole grid one of those), get a bound from the
 * list of the nearest cell, or a sample of the centroids, and go to the exact pass of rank16_exact_impl.h with it as their threshold.
 */
#include "rank16_exact_impl.h"

namespace kmx {

constexpr float CELL_SLACK = 1e-5f;
constexpr float CELL_MARGIN = 1e-3f;
/*
 * A centroid whose square, by fused multiply-adds, is less than 1 / CELL_CLEAR of all the others' is the serial scan's: both sums of squares are of the
 * same differences and off by at most 4 x 2^-24 each, so the serial ones differ by more than (33 - 4 x 4) 2^-24 of themselves, and their
 * square roots by more than a rounding (2 x 2^-24 of the square).
 */
constexpr float CELL_CLEAR = 1.000002f;
/*
 * A wavefront that has met this many points whose two smallest squares are not clear of each other stays with the serial arithmetic. On a raster (whole
 * numbers, colours, quantised measurements) every batch has some, and going through the lists twice costs more than the fused sums save (N = 4M, us
 * per call, the serial arithmetic alone, both for such points' wavefronts, this: d = 3, k = 4096, 16 places a dimension: 107, 142, 109; d = 4: 185, 237,
 * 189; 64 places 193, 215, 194; normal points rounded to 1/40 of their deviation, d = 3: 248, 300, 255). Other data have a dozen such points in all of
 * N = 4M: with 1 their wavefronts, which the others wait for at the end, cost half of what the fused sums save (normal points, d = 3, k = 4096: 254, 231, 248;
 * with 2 level with 231); with 4 the rounded normal points take 265.
 */
constexpr uint32_t CELL_TIES = 2;
constexpr uint32_t CELL_MAX_K = 6144;              /* what the building kernel's LDS holds */
constexpr uint32_t CELL_UNIT = 8;                  /* entries (16 bits) of a list that are read together */
/*
 * A building work-group's lists go to a region of its own if they fit, else to what all share, by an addition to one counter (256 additions that come
 * together take 2 us or more: all by the counter, d = 2, k = 1000: 67.2 instead of 65.5 us for the call, d = 3: 74.5 instead of 72.1).
 */
constexpr uint32_t CELL_SHARED_UNITS = 1u << 20, CELL_OWN_UNITS = 1u << 18;
constexpr uint32_t CELL_POOL_UNITS = CELL_SHARED_UNITS + CELL_OWN_UNITS;
constexpr uint32_t CELL_SAMPLE = 64;               /* centroids of the list for points without one, at the start of the pool */
constexpr uint32_t CELL_TRUNCATED = 1u << 31;      /* table entry: list start in units (21 bits), length in units (10), this flag */
constexpr uint32_t CELL_START_BITS = 21, CELL_MOST_UNITS = (1u << 10) - 1;
static_assert(CELL_POOL_UNITS <= 1u << CELL_START_BITS, "table entries");
constexpr uint32_t BUILD_THREADS = 1024;
constexpr uint32_t BUILD_WAVES = BUILD_THREADS / WAVE;
constexpr uint32_t BUILD_SHORT = 1024;             /* most centroids on the list of a second-level cell */
static_assert(BUILD_SHORT <= CELL_MOST_UNITS * CELL_UNIT, "a list's length");
constexpr uint32_t BUILD_OWN = CELL_MAX_K / BUILD_THREADS; /* most centroids of a thread */

/* cells per dimension: TOP of the first level (a work-group each), times MID (a wavefront each), times LOW */
template <int D> struct CellShape;
template <> struct CellShape<2> { static constexpr uint32_t TOP = 16, MID = 4, LOW = 4; };
template <> struct CellShape<3> { static constexpr uint32_t TOP = 8, MID = 2, LOW = 2; };
template <> struct CellShape<4> { static constexpr uint32_t TOP = 4, MID = 2, LOW = 2; };
template <int D> constexpr uint32_t cells_per_dim() { return CellShape<D>::TOP * CellShape<D>::MID * CellShape<D>::LOW; }
constexpr uint32_t power(uint32_t b, int e) { return e == 0 ? 1 : b * power(b, e - 1); }
template <int D> constexpr uint32_t cell_count() { return power(cells_per_dim<D>(), D); }

/* the grid: corner, cells per unit of length, cell widths (four floats each) */
struct Grid {
	float corner[4], inverse[4], width[4];
};

struct CellArgs {
	const float* means; size_t stride_means;
	Grid* grid; uint32_t* table; uint16_t* pool; uint32_t* counters;
	_Float16* packed; float* rows; float* norms;  /* operands, rows and norms of the exact pass (rank16_impl.h) */
	float* packed_form; float* form_norms;        /* of the packed sweep (assign_bf16_impl.h) */
	uint32_t k, kp, pool_units;
};

template <int D>
__device__ __forceinline__ void cell_distances(const float (&c)[D], const float (&lo)[D], const float (&hi)[D], float& least, float& most)
{
	least = 0.0f;
	most = 0.0f;
#pragma unroll
	for (int q = 0; q < D; ++q) {
		const float below = lo[q] - c[q], above = c[q] - hi[q]; /* (hi > lo) */
		const float out = fmaxf(fmaxf(below, above), 0.0f), far = fmaxf(-below, -above);
		least = __builtin_fmaf(out, out, least);
		most = __builtin_fmaf(far, far, most);
	}
}

/* all sums of one value per dimension, the last dimension's numbered fastest: sums of both halves of the dimensions first */
template <int D, uint32_t EACH>
__device__ __forceinline__ void all_sums(const float (&v)[D][EACH], float (&sums)[power(EACH, D)])
{
	constexpr int LEFT = D / 2, RIGHT = D - LEFT;
	static_assert(D >= 2 && D <= 4, "halves of one or two dimensions");
	float left[power(EACH, LEFT)], right[power(EACH, RIGHT)];
#pragma unroll
	for (uint32_t i = 0; i < power(EACH, LEFT); ++i) left[i] = LEFT == 1 ? v[0][i] : v[0][i / EACH] + v[1][i % EACH];
#pragma unroll
	for (uint32_t i = 0; i < power(EACH, RIGHT); ++i) right[i] = RIGHT == 1 ? v[D - 1][i] : v[D - 2][i / EACH] + v[D - 1][i % EACH];
#pragma unroll
	for (uint32_t c = 0; c < power(EACH, D); ++c) sums[c] = left[c / power(EACH, RIGHT)] + right[c % power(EACH, RIGHT)];
}

template <int CONTROL>
__device__ __forceinline__ float other_lane(float v) { return __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), CONTROL, 0xF, 0xF, true)); }
constexpr int ROW_ROR_8 = 0x128, ROW_HALF_MIRROR = 0x141, QUAD_XOR_2 = 0x4E, QUAD_XOR_1 = 0xB1;

/*
 * M values per lane: the least of number lane / (WAVE / M) over the wavefront. (Not through LDS, as shuffles are; a mirrored half row's lanes pair all of one
 * half of it with all of the other, which is as good as lanes 4 apart.)
 */
template <uint32_t M, uint32_t OFF = WAVE / 2>
__device__ __forceinline__ float least_of_each(const float (&v)[M], uint32_t lane)
{
	constexpr uint32_t H = M > 1 ? M / 2 : 1;
	float half[H];
#pragma unroll
	for (uint32_t i = 0; i < H; ++i) {
		const float first = v[i], second = v[M > 1 ? i + H : i]; /* for the lanes whose bit OFF is clear, is set */
		if constexpr (OFF == 32 || OFF == 16) {
			const auto both = OFF == 32 ? __builtin_amdgcn_permlane32_swap(__float_as_uint(first), __float_as_uint(second), false, false)
			                            : __builtin_amdgcn_permlane16_swap(__float_as_uint(first), __float_as_uint(second), false, false);
			half[i] = fminf(__uint_as_float(both[0]), __uint_as_float(both[1]));
		}
		else {
			constexpr int CONTROL = OFF == 8 ? ROW_ROR_8 : OFF == 4 ? ROW_HALF_MIRROR : OFF == 2 ? QUAD_XOR_2 : QUAD_XOR_1;
			const bool upper = M > 1 && (lane & OFF) != 0;
			half[i] = fminf(upper ? second : first, other_lane<CONTROL>(upper ? first : second));
		}
	}
	if constexpr (OFF > 1) return least_of_each<H, OFF / 2>(half, lane);
	else return half[0];
}

/* the least of 2 OFF neighbouring lanes */
template <uint32_t OFF = WAVE / 2>
__device__ __forceinline__ float least_of_lanes(float v)
{
	const float one[1] = { v };
	return least_of_each<1, OFF>(one, 0);
}

/* lanes of the mask below this one */
__device__ __forceinline__ uint32_t lanes_before(unsigned long long mask)
{
	return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ float of_lane(float v, uint32_t lane) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane)); }

/*
 * One work-group per first-level cell. All of them find the box of the centroids (they have to read them anyway), then three levels of
 * lists, each filtered from the one above: the work-group's, one per wavefront, one per cell. On the way a wavefront packs a row for
 * the exact pass and the packed sweep (as a kernel of its own ahead of this one that took 5 to 7 us and a launch).
 * What bounds it: the slowest work-group (uniform centroids, k = 4096, d = 4: half of the work-groups are done after 22 us, the last one, whose lists are
 * twice as long, after 31), in it the second level's box distances (9 us) and the writing of the lists (6), then the barriers. One level of lists,
 * every cell from all centroids, would be 65536 x k boxes, a millisecond. A thread's centroids stay in registers from the box to the first list, and a
 * wavefront's cells are filtered together (below): 50 -> 31 us; k = 1000, d = 3: the call 79 -> 72 us. (The second level's cells together as well, all
 * wavefronts on one list: its slowest work-group as slow, the others by 2 us, d = 3, k = 1000: 76 -> 80 us for the call.)
 */
template <int D, int LM>
__global__ void __launch_bounds__(BUILD_THREADS)
build_cells_kernel(const CellArgs w)
{
	constexpr uint32_t TOP = CellShape<D>::TOP, MID = CellShape<D>::MID, LOW = CellShape<D>::LOW, N = cells_per_dim<D>();
	constexpr uint32_t MIDS = power(MID, D), LOWS = power(LOW, D), LANES = WAVE / LOWS; /* second-level cells, cells of one, lanes per cell */
	static_assert(MIDS <= BUILD_WAVES && LOWS * LANES == WAVE, "shape");
	extern __shared__ __attribute__((aligned(16))) float lds[];
	float* coords = lds;                                        /* k x D, relative to the corner */
	uint16_t* first_list = (uint16_t*)(lds + w.k * D);          /* k */
	uint16_t* second_lists = first_list + (w.k + 1) / 2 * 2;    /* BUILD_WAVES x BUILD_SHORT */
	__shared__ __attribute__((aligned(16))) float reduce[8][BUILD_WAVES];
	__shared__ __attribute__((aligned(16))) uint32_t wave_count[BUILD_WAVES];
	__shared__ uint32_t wave_units[BUILD_WAVES], pool_start;
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));

	/* the frame of the packed rows: the mean of 16 centroids spread evenly; and this wavefront's (first) row, a coordinate per lane */
	float frame[D], member[D];
	{
		const uint32_t r = even_row(lane % 16, 4, w.k);
#pragma unroll
		for (int q = 0; q < D; ++q) member[q] = w.means[elem<LM>(w.stride_means, r, q)];
	}
	const uint32_t first_row = blockIdx.x * BUILD_WAVES + wave;
	float exact = w.means[elem<LM>(w.stride_means, min(first_row, w.k - 1), min(lane, (uint32_t)D - 1))];

	/* the box of the centroids (of their finite coordinates); a thread's own stay in registers, a wavefront's are consecutive */
	const uint32_t rounds = (w.k + BUILD_THREADS - 1) / BUILD_THREADS, first_own = wave * rounds * WAVE + lane;
	float own[BUILD_OWN][D];
#pragma unroll
	for (uint32_t i = 0; i < BUILD_OWN; ++i)
		if (i < rounds) {
			const uint32_t j = min(first_own + i * WAVE, w.k - 1);
			if constexpr (LM == KMX_AOS) __builtin_memcpy(own[i], w.means + elem<LM>(w.stride_means, j, 0), sizeof(own[i])); /* (one load, which need not be aligned) */
			else
#pragma unroll
				for (int q = 0; q < D; ++q) own[i][q] = w.means[elem<LM>(w.stride_means, j, q)];
		}
	bool odd = false;
	float ends[8]; /* least coordinates, least negative ones */
#pragma unroll
	for (uint32_t u = 0; u < 8; ++u) ends[u] = __builtin_inff();
#pragma unroll
	for (uint32_t i = 0; i < BUILD_OWN; ++i)
		if (i < rounds)
#pragma unroll
			for (int q = 0; q < D; ++q) {
				const float v = own[i][q];
				const bool finite = __builtin_fabsf(v) < __builtin_inff();
				ends[q] = finite ? fminf(ends[q], v) : ends[q];
				ends[4 + q] = finite ? fminf(ends[4 + q], -v) : ends[4 + q];
				odd = odd || !finite;
			}
	const float end = least_of_each(ends, lane);
	if (lane % 8 == 0) reduce[lane / 8][wave] = end;
#pragma unroll
	for (int q = 0; q < D; ++q) {
		float sum = __builtin_fabsf(member[q]) < __builtin_inff() ? member[q] : 0.0f;
		for (int off = 8; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
		sum = sum / 16.0f;
		frame[q] = __builtin_fabsf(sum) < __builtin_inff() ? sum : 0.0f; /* (the sum of finite values may overflow) */
	}
	bool usable = !__syncthreads_or(odd ? 1 : 0);
	float corner[D], width[D], inverse[D], far = 0.0f, size = 0.0f;
	{
		const float all = least_of_lanes<4>(fminf(reduce[lane / 8][lane % 8 * 2], reduce[lane / 8][lane % 8 * 2 + 1]));
		const float share = fmaxf(0.75f * __builtin_powf((float)w.k, -1.0f / D), 0.05f); /* of the extent, added on either side */
		float extent2 = 0.0f;
#pragma unroll
		for (int q = 0; q < D; ++q) {
			const float lo = of_lane(all, 8 * q), hi = -of_lane(all, 8 * (4 + q));
			far = fmaxf(far, fmaxf(hi - frame[q], frame[q] - lo));
			size = fmaxf(size, fmaxf(__builtin_fabsf(lo), __builtin_fabsf(hi)));
			const float half = fmaxf(0.5f * (hi - lo) * (1.0f + 2.0f * share), 1e-6f * (__builtin_fabsf(lo) + __builtin_fabsf(hi)) + 1e-16f);
			corner[q] = 0.5f * lo + 0.5f * hi - half;
			width[q] = 2.0f * half / (float)N;
			inverse[q] = (float)N / (2.0f * half);
			extent2 += half * half;
			usable = usable && width[q] * width[q] > 1e-30f;
		}
		usable = usable && extent2 < 1e36f;
	}
	if (blockIdx.x == 0 && tid < D) {
		float c = corner[0], i = inverse[0], s = width[0];
#pragma unroll
		for (int q = 1; q < D; ++q) {
			c = tid == (uint32_t)q ? corner[q] : c;
			i = tid == (uint32_t)q ? inverse[q] : i;
			s = tid == (uint32_t)q ? width[q] : s;
		}
		w.grid->corner[tid] = c; w.grid->inverse[tid] = i; w.grid->width[tid] = s;
	}
	if (blockIdx.x == 0 && tid < CELL_SAMPLE) w.pool[tid] = (uint16_t)((uint64_t)tid * w.k / CELL_SAMPLE);
	const uint32_t nothing = CELL_TRUNCATED | (CELL_SAMPLE / CELL_UNIT) << CELL_START_BITS; /* the sample */

	/* the packed rows, as pack_means16_kernel and pack_means_bf16_kernel make them */
	{
		const bool any = size < __builtin_inff(); /* (of finite coordinates) */
		const float scale = rank16_scale(any ? far : 0.0f, any ? size : 0.0f);
		float m = 0.0f;
#pragma unroll
		for (int q = 0; q < D; ++q) m = lane == (uint32_t)q ? frame[q] : m;
		for (uint32_t j = first_row; j < w.kp; j += gridDim.x * BUILD_WAVES) {
			if (j != first_row) exact = w.means[elem<LM>(w.stride_means, min(j, w.k - 1), min(lane, (uint32_t)D - 1))];
			const bool there = j < w.k && lane < (uint32_t)D;
			const float v = there ? __builtin_fmaf(exact, scale, -(m * scale)) : 0.0f;
			const float cv = -2.0f * v;
			const _Float16 half = (_Float16)cv;
			const float low_part = cv - (float)half;
			__bf16 hi, mid;
			const float rest = split_bf16(cv, hi, mid);
			float sums[7] = { v * v, low_part * low_part, (float)mid * (float)mid, rest * rest, 0.0f, 0.0f, 0.0f };
			const float moved = __shfl(there ? exact - m : 0.0f, (int)(lane % 4)); /* (by all lanes; zeros behind the row) */
			if (lane < KBLOCK) {
				w.rows[(size_t)j * KBLOCK + lane] = there ? exact : 0.0f;
				w.packed[((size_t)(j / TILE) * WAVE + lane / 8 * TILE + j % TILE) * 8 + lane % 8] = half;
				pack_packed_row(w.packed_form, j, lane, moved, sums[4], sums[5], sums[6]);
			}
#pragma unroll
			for (int u = 0; u < 7; ++u) { sums[u] += __shfl_xor(sums[u], 2); sums[u] += __shfl_xor(sums[u], 1); }
			if (lane == 0) {
				w.norms[norm_at(j)] = j < w.k ? sums[0] : 1.7e38f;
				w.form_norms[norm_at(j)] = j < w.k ? sums[4] : __builtin_inff();
#pragma unroll
				for (int u = 0; u < 3; ++u) w.norms[rank16_low_offset(w.kp) + u * w.kp + j] = sums[1 + u];
#pragma unroll
				for (int u = 0; u < 2; ++u) w.form_norms[split_norms_offset(w.kp) + u * w.kp + j] = sums[5 + u];
			}
			if (lane < NORM_TILE - TILE && j % TILE == 0) {
				w.norms[(j / TILE) * NORM_TILE + TILE + lane] = 1.7e38f;
				w.form_norms[(j / TILE) * NORM_TILE + TILE + lane] = __builtin_inff();
			}
		}
		if (blockIdx.x == 0 && wave == 0) {
			if (lane < KBLOCK) w.norms[rank16_frame_offset(w.kp) + lane] = m; /* (zeros behind the row) */
			if (lane < 4) w.form_norms[frame_offset(w.kp) + lane] = m;
			if (lane == 0) {
				w.norms[rank16_scale_offset(w.kp)] = scale;
				w.norms[rank16_scale_offset(w.kp) + 1] = 1.0f / (scale * scale);
				w.counters[0] = 0u; w.counters[LISTED_COUNTER] = 0u; /* (CELLS_COUNTER: cleared by the last search) */
			}
		}
	}

	/* this lane's cell */
	uint32_t top[D], mid[D], at[D];
	{
		uint32_t t = blockIdx.x, m = min(wave, MIDS - 1), l = lane / LANES;
#pragma unroll
		for (int q = D - 1; q >= 0; --q) {
			top[q] = t % TOP; t /= TOP;
			mid[q] = m % MID; m /= MID;
			at[q] = (top[q] * MID + mid[q]) * LOW + l % LOW; l /= LOW;
		}
	}
	uint32_t cell = 0;
#pragma unroll
	for (int q = 0; q < D; ++q) cell = cell * N + at[q];
	const bool writes = wave < MIDS && lane % LANES == 0;
	if (!usable) {
		if (writes) w.table[cell] = nothing;
		return; /* (the whole work-group) */
	}
	auto box = [&](float (&lo)[D], float (&hi)[D], const uint32_t (&first)[D], uint32_t cells) {
#pragma unroll
		for (int q = 0; q < D; ++q) {
			lo[q] = ((float)first[q] - CELL_MARGIN) * width[q];
			hi[q] = ((float)(first[q] + cells) + CELL_MARGIN) * width[q];
		}
	};
	auto measure = [&](uint32_t j, const float (&lo)[D], const float (&hi)[D], float& least, float& most) {
		float c[D];
#pragma unroll
		for (int q = 0; q < D; ++q) c[q] = coords[j * D + q];
		cell_distances<D>(c, lo, hi, least, most);
	};
	auto enough = [](float bound) { return bound * (1.0f + CELL_SLACK); };
	float lo[D], hi[D];

	/* the work-group's list */
	uint32_t first_count = 0;
	{
		uint32_t start[D];
#pragma unroll
		for (int q = 0; q < D; ++q) start[q] = top[q] * MID * LOW;
		box(lo, hi, start, MID * LOW);
		float bound = __builtin_inff(), least[BUILD_OWN];
#pragma unroll
		for (uint32_t i = 0; i < BUILD_OWN; ++i)
			if (i < rounds) {
				const uint32_t j = first_own + i * WAVE;
				float most;
#pragma unroll
				for (int q = 0; q < D; ++q) own[i][q] -= corner[q];
				cell_distances<D>(own[i], lo, hi, least[i], most);
				bound = fminf(bound, most); /* (behind the last centroid: that one again) */
				if (j < w.k)
#pragma unroll
					for (int q = 0; q < D; ++q) coords[j * D + q] = own[i][q];
			}
		bound = least_of_lanes(bound);
		__syncthreads(); /* (the box has been read) */
		if (lane == 0) reduce[0][wave] = bound;
		__syncthreads();
		bound = enough(least_of_lanes<BUILD_WAVES / 2>(reduce[0][lane % BUILD_WAVES]));
		unsigned long long masks[BUILD_OWN];
		uint32_t count = 0;
#pragma unroll
		for (uint32_t i = 0; i < BUILD_OWN; ++i)
			if (i < rounds) {
				masks[i] = __ballot(first_own + i * WAVE < w.k && least[i] <= bound);
				count += (uint32_t)__popcll(masks[i]);
			}
		if (lane == 0) wave_count[wave] = count;
		__syncthreads();
		uint32_t to = 0;
#pragma unroll
		for (uint32_t v = 0; v < BUILD_WAVES; ++v) {
			const uint32_t c = wave_count[v];
			to += v < wave ? c : 0u;
			first_count += c;
		}
#pragma unroll
		for (uint32_t i = 0; i < BUILD_OWN; ++i)
			if (i < rounds) {
				if (masks[i] >> lane & 1) first_list[to + lanes_before(masks[i])] = (uint16_t)(first_own + i * WAVE);
				to += (uint32_t)__popcll(masks[i]);
			}
		__syncthreads();
	}

	/* the wavefront's list */
	uint16_t* second_list = second_lists + wave * BUILD_SHORT;
	uint32_t second_count = 0;
	if (wave < MIDS) {
		uint32_t start[D];
#pragma unroll
		for (int q = 0; q < D; ++q) start[q] = (top[q] * MID + mid[q]) * LOW;
		box(lo, hi, start, LOW);
		float bound = __builtin_inff();
#pragma unroll 4
		for (uint32_t i = lane; i < first_count; i += WAVE) {
			float least, most;
			measure(first_list[i], lo, hi, least, most);
			bound = fminf(bound, most);
		}
		bound = enough(least_of_lanes(bound));
#pragma unroll 4
		for (uint32_t base = 0; base < first_count; base += WAVE) {
			const uint32_t i = base + lane;
			const uint16_t j = first_list[min(i, first_count - 1)];
			float least, most;
			measure(j, lo, hi, least, most);
			const bool keep = i < first_count && least <= bound;
			const unsigned long long mask = __ballot(keep);
			const uint32_t to = second_count + lanes_before(mask);
			if (keep && to < BUILD_SHORT) second_list[to] = j;
			second_count += (uint32_t)__popcll(mask);
		}
	}
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
	const bool too_long = second_count > BUILD_SHORT;

	/*
	 * The cells' lists, of all the wavefront's cells at once: a lane per centroid of the list, whose distances from a cell are sums of one of LOW values per
	 * dimension: 24 additions for the 16 cells of d = 4 (LANES lanes to a cell, a part of the list each and every distance by itself: 16 us of the slowest
	 * work-group instead of 3.6 at k = 4096).
	 */
	const uint32_t turns = too_long ? 0u : (second_count + WAVE - 1) / WAVE;
	float low_end[D][LOW], high_end[D][LOW];
#pragma unroll
	for (int q = 0; q < D; ++q)
#pragma unroll
		for (uint32_t l = 0; l < LOW; ++l) {
			const uint32_t first = (top[q] * MID + mid[q]) * LOW + l;
			low_end[q][l] = ((float)first - CELL_MARGIN) * width[q];
			high_end[q][l] = ((float)(first + 1) + CELL_MARGIN) * width[q];
		}
	float bounds[LOWS];
#pragma unroll
	for (uint32_t c = 0; c < LOWS; ++c) bounds[c] = __builtin_inff();
	for (uint32_t i = 0; i < turns; ++i) {
		const uint32_t j = second_list[min(i * WAVE + lane, second_count - 1)];
		float far[D][LOW], sums[LOWS];
#pragma unroll
		for (int q = 0; q < D; ++q) {
			const float v = coords[j * D + q];
#pragma unroll
			for (uint32_t l = 0; l < LOW; ++l) {
				const float most = fmaxf(v - low_end[q][l], high_end[q][l] - v);
				far[q][l] = most * most;
			}
		}
		all_sums<D, LOW>(far, sums);
#pragma unroll
		for (uint32_t c = 0; c < LOWS; ++c) bounds[c] = fminf(bounds[c], sums[c]);
	}
	const float bound = enough(least_of_each(bounds, lane)); /* of cell lane / LANES */
#pragma unroll
	for (uint32_t c = 0; c < LOWS; ++c) bounds[c] = of_lane(bound, c * LANES);
	uint32_t counts[LOWS], kept[BUILD_SHORT / WAVE / 2]; /* 16 bits a turn, the last turn's lowest: which cells keep this lane's centroid */
#pragma unroll
	for (uint32_t c = 0; c < LOWS; ++c) counts[c] = 0;
#pragma unroll
	for (uint32_t u = 0; u < BUILD_SHORT / WAVE / 2; ++u) kept[u] = 0;
	for (uint32_t i = 0; i < turns; ++i) {
		const bool there = i * WAVE + lane < second_count;
		const uint32_t j = second_list[min(i * WAVE + lane, second_count - 1)];
		float out[D][LOW], sums[LOWS];
#pragma unroll
		for (int q = 0; q < D; ++q) {
			const float v = coords[j * D + q];
#pragma unroll
			for (uint32_t l = 0; l < LOW; ++l) {
				const float least = fmaxf(fmaxf(low_end[q][l] - v, v - high_end[q][l]), 0.0f);
				out[q][l] = least * least;
				if (q == 0) out[q][l] = there ? out[q][l] : __builtin_inff();
			}
		}
		all_sums<D, LOW>(out, sums);
		uint32_t bits = 0;
#pragma unroll
		for (uint32_t c = 0; c < LOWS; ++c) {
			const bool keep = sums[c] <= bounds[c];
			counts[c] += (uint32_t)__popcll(__ballot(keep));
			bits |= keep ? 1u << c : 0u;
		}
#pragma unroll
		for (uint32_t u = BUILD_SHORT / WAVE / 2 - 1; u > 0; --u) kept[u] = kept[u] << 16 | kept[u - 1] >> 16;
		kept[0] = kept[0] << 16 | bits;
	}
	const uint32_t part = lane % LANES;
	uint32_t total = 0; /* entries of cell lane / LANES */
#pragma unroll
	for (uint32_t c = 0; c < LOWS; ++c) total = lane / LANES == c ? counts[c] : total;
	uint32_t units = wave < MIDS ? (total + CELL_UNIT - 1) / CELL_UNIT : 0u;
	const bool fits = units <= CELL_MOST_UNITS && !too_long;
	if (!fits) units = 0;
	uint32_t upto = part == 0 ? units : 0u; /* inclusive over the wavefront's cells */
#pragma unroll
	for (uint32_t off = 1; off < WAVE; off <<= 1) {
		const uint32_t v = (uint32_t)__shfl_up((int)upto, off);
		if (lane >= off) upto += v;
	}
	if (lane == WAVE - 1) wave_units[wave] = upto;
	__syncthreads();
	if (tid == 0) {
		uint32_t all = 0;
		for (uint32_t v = 0; v < BUILD_WAVES; ++v) { const uint32_t u = wave_units[v]; wave_units[v] = all; all += u; }
		constexpr uint32_t GROUPS = power(TOP, D), OWN = (CELL_OWN_UNITS - CELL_SAMPLE / CELL_UNIT) / GROUPS;
		pool_start = CELL_SAMPLE / CELL_UNIT + (all <= OWN ? blockIdx.x * OWN : GROUPS * OWN + atomicAdd(w.counters + CELLS_COUNTER, all));
	}
	__syncthreads();
	const uint32_t start = pool_start + wave_units[wave] + upto - units; /* (lanes of a cell behind its first: upto counts the cell already) */
	const bool listed = fits && units > 0 && (uint64_t)start + units <= w.pool_units;
	if (writes) w.table[cell] = listed ? start | units << CELL_START_BITS : nothing;
	if (listed) /* the last unit is filled up with the row behind the last centroid (which is infinitely far) */
		for (uint32_t to = total + part; to < units * CELL_UNIT; to += LANES) w.pool[(size_t)start * CELL_UNIT + to] = (uint16_t)w.k;
	const unsigned long long has_list = __ballot(listed);
	uint32_t cells = 0; /* that have a list */
#pragma unroll
	for (uint32_t c = 0; c < LOWS; ++c) {
		cells |= (uint32_t)(has_list >> (c * LANES) & 1) << c;
		counts[c] += (uint32_t)__builtin_amdgcn_readlane((int)(start * CELL_UNIT), (int)(c * LANES)); /* the end of what is still to be written */
	}
	for (uint32_t i = turns; i-- > 0;) {
		const uint16_t j = second_list[min(i * WAVE + lane, second_count - 1)];
		const uint32_t bits = kept[0] & cells;
#pragma unroll
		for (uint32_t u = 0; u < BUILD_SHORT / WAVE / 2; ++u) kept[u] = kept[u] >> 16 | (u + 1 < BUILD_SHORT / WAVE / 2 ? kept[u + 1] << 16 : 0u);
#pragma unroll
		for (uint32_t c = 0; c < LOWS; ++c) {
			const bool keep = bits >> c & 1;
			const unsigned long long mask = __ballot(keep);
			counts[c] -= (uint32_t)__popcll(mask);
			if (keep) w.pool[counts[c] + lanes_before(mask)] = j;
		}
	}
}

struct CellAssignArgs {
	const float* data; size_t stride;
	const float* means; size_t stride_means;
	const Grid* grid; const uint32_t* table; const uint16_t* pool;
	const float* norms; const float* low2; const float* frame; float* scale; /* of the exact pass */
	uint32_t* assignment; uint32_t* list;
	uint32_t* counters; /* LISTED_COUNTER: the list's length; CELLS_COUNTER: cleared for the next call; WAY_BACK_COUNTER: 0 or 1 is left there */
	uint32_t k, kp, n, choose;
	float kd;
};

constexpr uint32_t CELL_THREADS = 1024;
constexpr uint32_t CELL_WAVES = CELL_THREADS / WAVE;
constexpr uint32_t CHOICE_EACH = 2, CHOICE_GROUPS = CHOICE_EACH * CELL_WAVES; /* groups of 64 points that the choice between cells and sweep looks at */
constexpr uint32_t CELL_LIST = 64; /* points per wavefront that wait for the list */
constexpr uint32_t CELL_STATIC = CELL_WAVES * (2 * CELL_LIST + 6) * 4 + 128; /* LDS of assign_cells_kernel beside the centroids: the infinite row, flag_list, wave_max */

/*
 * A lane per point, the centroids in LDS. What bounds it: the gathers from LDS and the vector ALU, which are both close to full (N = 4M, d = 4, k = 4096,
 * uniform points: a wavefront goes through the longest list of its 64 points, 70 entries of 29 on average, and 16 bytes at 64 unrelated addresses take
 * 11 cycles with their bank conflicts: 179 000 of the 242 000 cycles of a compute unit; 61 600 vector instructions on a SIMD, one in 3.9 cycles: minima and
 * medians take 4.4 of them, fused sums two). A comparison is 13 instructions and no branch: the sums are fused, the
 * two smallest are kept (one v_med3), and the few points whose two smallest are not CELL_CLEAR of each other go through their list again in the
 * serial arithmetic (see CELL_TIES). Against that arithmetic for all, with its branches (17 instructions, and each row waited for by itself): 122 -> 112 us;
 * normal points, d = 4, k = 1000: 246 -> 216 us per call; d = 3, k = 6000: 119 -> 108 us. Sorting a wavefront's 256 points by the length of their
 * lists takes a quarter of the instructions out, but
 * fuller wavefronts have more bank conflicts: 122 -> 136 us. Two work-groups share a compute unit, eight wavefronts
 * a SIMD, which takes 64 vector registers; with more than 80 scalar registers (and the 16 the hardware adds) only seven fit, which is one
 * work-group (d = 3, k = 4096, normal points: 162 -> 220 us).
 */
template <int D, int LD, int LM>
__global__ void __launch_bounds__(CELL_THREADS) __attribute__((amdgpu_num_sgpr(80), amdgpu_waves_per_eu(8)))
assign_cells_kernel(const CellAssignArgs w)
{
	constexpr uint32_t N = cells_per_dim<D>();
	extern __shared__ __attribute__((aligned(16))) float lds[]; /* (k + 1) x 4 */
	/* (all of it is dynamic, so a row's address is 16 times its number) */
	uint32_t (*const wave_max)[CELL_WAVES] = (uint32_t (*)[CELL_WAVES])(lds + 4 * (w.k + 1));
	uint32_t (*const flag_list)[2 * CELL_LIST] = (uint32_t (*)[2 * CELL_LIST])(wave_max + 6);
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const float scale = w.scale[0];
	float corner[D], inverse[D];
#pragma unroll
	for (int q = 0; q < D; ++q) { corner[q] = w.grid->corner[q]; inverse[q] = w.grid->inverse[q]; }
	auto locate = [&](const float (&x)[D], bool& inside) -> uint32_t {
		inside = true;
		uint32_t cell = 0;
#pragma unroll
		for (int q = 0; q < D; ++q) {
			const float y = (x[q] - corner[q]) * inverse[q];
			inside = inside && y >= 0.0f && y < (float)N;
			cell = cell * N + (uint32_t)fminf(fmaxf(y, 0.0f), (float)(N - 1)); /* (NaN: 0) */
		}
		return cell;
	};

	/* the sample of the choice below is on its way while the centroids are */
	const bool choose = w.choose != 0;
	float sample[CHOICE_EACH][D];
	if (choose) {
#pragma unroll
		for (uint32_t i = 0; i < CHOICE_EACH; ++i) {
			const uint32_t pt = min((uint32_t)((uint64_t)(w.n / WAVE) * (wave * CHOICE_EACH + i) / CHOICE_GROUPS) * WAVE + lane, w.n - 1);
#pragma unroll
			for (int q = 0; q < D; ++q) sample[i][q] = w.data[elem<LD>(w.stride, pt, q)];
		}
	}
	for (uint32_t j = tid; j < w.k; j += CELL_THREADS) {
		f32x4 c = { 0.0f, 0.0f, 0.0f, 0.0f };
#pragma unroll
		for (int q = 0; q < D; ++q) c[q] = w.means[elem<LM>(w.stride_means, j, q)];
		*(f32x4*)(lds + 4 * j) = c;
	}
	if (tid < 4) lds[4 * w.k + tid] = __builtin_inff();
	/* the maxima of the certificate; the first work-group leaves them and those of the exact pass's own (rank16_leave_bounds) */
	uint32_t most[6] = { 0u, 0u, 0u, 0u, 0u, 0u }; /* of |c|^2, low^2, mid^2, rest^2; then two sums: entries, points without a list */
	for (uint32_t j = tid; j < w.k; j += CELL_THREADS) {
		most[0] = max(most[0], __float_as_uint(w.norms[norm_at(j)]));
		most[1] = max(most[1], __float_as_uint(w.low2[j]));
		if (blockIdx.x == 0) {
			most[2] = max(most[2], __float_as_uint(w.low2[w.kp + j]));
			most[3] = max(most[3], __float_as_uint(w.low2[2 * w.kp + j]));
		}
	}
	if (choose) {
#pragma unroll
		for (uint32_t i = 0; i < CHOICE_EACH; ++i) {
			bool inside;
			const uint32_t entry = w.table[locate(sample[i], inside)];
			uint32_t units = (entry >> CELL_START_BITS) & CELL_MOST_UNITS;
			for (int off = WAVE / 2; off > 0; off >>= 1) units = max(units, (uint32_t)__shfl_xor((int)units, off));
			most[4] += units * CELL_UNIT;
			most[5] += (uint32_t)__popcll(__ballot(!inside || (entry & CELL_TRUNCATED)));
		}
	}
#pragma unroll
	for (int q = 0; q < 6; ++q) {
		if (q < 4)
			for (int off = WAVE / 2; off > 0; off >>= 1) most[q] = max(most[q], (uint32_t)__shfl_xor((int)most[q], off));
		if (lane == 0) wave_max[q][wave] = most[q];
	}
	__syncthreads();
#pragma unroll
	for (int q = 0; q < 6; ++q) {
		most[q] = 0;
		for (uint32_t v = 0; v < CELL_WAVES; ++v) most[q] = q < 4 ? max(most[q], wave_max[q][v]) : most[q] + wave_max[q][v];
	}
	if (blockIdx.x == 0 && tid == 0) {
		w.counters[CELLS_COUNTER] = 0u;
		w.scale[2] = __uint_as_float(most[0]); w.scale[3] = __uint_as_float(most[2]);
		w.scale[4] = __uint_as_float(most[3]); w.scale[5] = __uint_as_float(most[1]);
	}
	const CertCoeffs cert = cert_coeffs_level1(CentroidBounds{ __uint_as_float(most[0]), __uint_as_float(most[1]), 0.0f });

	/*
	 * Are the cells any good for these points? The sample (CHOICE_GROUPS wavefronts' worth, spread evenly over the points) says what
	 * they would cost: a wavefront its longest list, N = 4M points 60 us and 1 us per entry (d = 4; 75 and 1.45 in the serial arithmetic alone, which
	 * rasters keep to: CELL_TIES); a point without a list as much as k to 2 k entries in the exact pass. The packed sweep costs those points 110 us + 0.14
	 * per centroid, its exact pass what the data make of it, and the lists have been built by then. So it is left to that sweep (all work-groups
	 * come to the same answer) if
	 *   - the lists are longer than k / 8 + 70 (d = 4, k = 1000: normal points, 168 entries, 261 us through the cells, 340 after all by the sweep; exponential,
	 *     474, 661 and 397: level at some 280, the line lies below since rasters cost the cells half as much again; points along a line 189, 450 and 2490 in the
	 *     serial arithmetic, the sweep certifies few of those) or k / 8 + 320 (d = 2, 3: skewed data, which
	 *     has such lists, costs the sweep more too: lognormal, k = 1000: 423 entries, 549 against 1044 us);
	 *   - or the points without a list cost more than half of the first of these (normal, d = 4, k = 4096: 65 % of the points, 4329
	 *     against 825 us; all outside the grid, d = 4, k = 1000: 1690 against 287).
	 */
	if (choose) {
		const uint32_t entries = most[4], unlisted = most[5];
		const bool sweep = 8 * entries > CHOICE_GROUPS * (w.k + 8 * (D == 4 ? 70 : 320)) ||
		                   3 * w.k * unlisted * 8 > CHOICE_GROUPS * WAVE * (w.k + 8 * 70);
		if (blockIdx.x == 0 && tid == 0) w.counters[WAY_BACK_COUNTER] = sweep ? 1u : 0u;
		if (sweep) return; /* the whole grid */
	}

	uint32_t flagged = 0; /* wave-uniform */
	uint32_t ties = 0;    /* wave-uniform: points whose nearest two were not clear of each other */
	for (uint32_t base = blockIdx.x * CELL_THREADS; base < w.n; base += gridDim.x * CELL_THREADS) {
		const uint32_t pt = base + tid;
		const bool mine = pt < w.n;
		float x[D];
#pragma unroll
		for (int q = 0; q < D; ++q) x[q] = w.data[elem<LD>(w.stride, min(pt, w.n - 1), q)];
		bool inside;
		const uint32_t entry = w.table[locate(x, inside)];
		const uint32_t units = (entry >> CELL_START_BITS) & CELL_MOST_UNITS;
		const uint4* list = (const uint4*)w.pool + (entry & ((1u << CELL_START_BITS) - 1));
		float best = __builtin_inff();
		uint32_t winner = 0; /* as an LDS address */
		auto compare = [&](const f32x4& c, uint32_t at) {
#pragma clang fp contract(off)
			float sum = 0.0f;
#pragma unroll
			for (int q = 0; q < D; ++q) {
				const float diff = x[q] - c[q];
				const float sq = diff * diff;
				sum = sum + sq;
			}
			/* the serial scan compares square roots: a smaller square may have the same one */
			if (sum < best && (sum < best * 0.9999995f || __builtin_sqrtf(sum) < __builtin_sqrtf(best))) { best = sum; winner = at; }
		};
		auto walk = [&](auto&& take) {
			uint4 next = list[0];
			for (uint32_t u = 0; u < units; ++u) {
				const uint4 now = next;
				next = list[min(u + 1, units - 1)];
				asm volatile("" ::: "memory"); /* (the next unit is requested here, not where it is used) */
				const uint32_t word[4] = { now.x, now.y, now.z, now.w };
#pragma unroll
				for (uint32_t h = 0; h < 4; h += 2) {
					uint32_t at[4]; /* LDS addresses: 16 times an entry */
					f32x4 c[4];
#pragma unroll
					for (uint32_t i = 0; i < 4; ++i) {
						if (i % 2) asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_1" : "=v"(at[i]) : "v"(4u), "v"(word[h + i / 2]));
						else asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0" : "=v"(at[i]) : "v"(4u), "v"(word[h + i / 2]));
						c[i] = *(const __attribute__((address_space(3))) f32x4*)at[i];
					}
					asm volatile("" : "+v"(c[0]), "+v"(c[1]), "+v"(c[2]), "+v"(c[3])); /* (all four are on their way before the first is used) */
#pragma unroll
					for (uint32_t i = 0; i < 4; ++i) take(c[i], at[i]);
				}
			}
		};
		const bool flag = mine && (!inside || (entry & CELL_TRUNCATED));
		bool open = true;
		if (ties < CELL_TIES) {
			float second = __builtin_inff();
			walk([&](const f32x4& c, uint32_t at) {
				float sum = 0.0f;
#pragma unroll
				for (int q = 0; q < D; ++q) {
					const float diff = x[q] - c[q];
					sum = q ? __builtin_fmaf(diff, diff, sum) : diff * diff;
				}
				second = __builtin_amdgcn_fmed3f(sum, best, second);
				const bool less = sum < best;
				best = less ? sum : best;
				winner = less ? at : winner;
			});
			/* (smaller squares may have lost bits; a sum of 0 is 0 in either arithmetic, and the first one wins) */
			const bool clear = best == 0.0f || (best > 1e-30f && second > best * CELL_CLEAR);
			ties += (uint32_t)__popcll(__ballot(!clear && !flag));
			open = flag || !clear; /* (a flagged point's distance becomes its threshold: the serial one) */
		}
		if (open) {
			best = __builtin_inff();
			winner = 0;
			walk(compare);
		}
		if (mine) w.assignment[pt] = winner / 16;
		const unsigned long long mask = __ballot(flag);
		if (mask) {
			const uint32_t add = (uint32_t)__popcll(mask);
			if (flagged + add > CELL_LIST) {
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				__builtin_amdgcn_wave_barrier();
				uint32_t slot = 0;
				if (lane == 0) slot = atomicAdd(w.counters + LISTED_COUNTER, flagged);
				slot = (uint32_t)__shfl((int)slot, 0);
				for (uint32_t i = lane; i < 2 * flagged; i += WAVE) w.list[2 * (size_t)slot + i] = flag_list[wave][i];
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				__builtin_amdgcn_wave_barrier();
				flagged = 0;
			}
			if (flag) {
				/* every centroid as near as the winner ranks at or below its distance, within the certificate of the ranking */
				float x2 = 0.0f, low2 = 0.0f;
#pragma unroll
				for (int q = 0; q < D; ++q) {
					const float v = __builtin_fmaf(x[q], scale, -(w.frame[q] * scale));
					const float r = v - (float)(_Float16)v;
					x2 = __builtin_fmaf(v, v, x2);
					low2 = __builtin_fmaf(r, r, low2);
				}
				const float nearest2 = best * (scale * scale);
				const bool extreme = !(best > 1e-30f && best < 1e37f && nearest2 < 1e37f && x2 < 1e37f);
				const float tau = cert_tau(w.kd, x2, low2, cert) + 64.0f * CERT_UNIT * nearest2;
				const uint32_t at = 2 * (flagged + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull)));
				flag_list[wave][at] = pt;
				flag_list[wave][at + 1] = screening_threshold(extreme ? __builtin_inff() : nearest2 - x2, tau);
			}
			flagged += add;
		}
	}
	/* what is left in the lists: one addition per work-group */
	__syncthreads();
	if (lane == 0) wave_max[0][wave] = flagged;
	__syncthreads();
	uint32_t before = 0, all = 0;
#pragma unroll
	for (uint32_t v = 0; v < CELL_WAVES; ++v) {
		before += v < wave ? wave_max[0][v] : 0u;
		all += wave_max[0][v];
	}
	if (all == 0) return;
	if (tid == 0) wave_max[1][0] = atomicAdd(w.counters + LISTED_COUNTER, all);
	__syncthreads();
	const size_t slot = 2 * (size_t)(wave_max[1][0] + before);
	for (uint32_t i = lane; i < 2 * flagged; i += WAVE) w.list[slot + i] = flag_list[wave][i];
}

template <int D>
static int launch_cells_d(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, const Cells16& half, bool choose)
{
	constexpr uint32_t CELLS = cell_count<D>();
	const size_t table_words = sizeof(Grid) / 4 + CELLS;
	int rc = reserve_cells(ws, table_words + (size_t)CELL_POOL_UNITS * CELL_UNIT / 2);
	if (rc) return rc;
	if ((rc = reserve_listed(ws, 2 * (size_t)a.n))) return rc;
	Grid* grid = (Grid*)ws->cells;
	uint32_t* table = ws->cells + sizeof(Grid) / 4;
	uint16_t* pool = (uint16_t*)(ws->cells + table_words);
	static_assert(sizeof(Grid) % 16 == 0 && CELLS % 4 == 0, "the pool is read in units of 16 bytes");
	const uint32_t build_lds = a.k * D * 4 + (a.k + 1) / 2 * 4 + BUILD_WAVES * BUILD_SHORT * 2;
	const CellArgs b = { a.means, a.stride_means, grid, table, pool, ws->counters, (_Float16*)ws->packed16, ws->packed16 + rank16_rows_offset(half.kp, KBLOCK), ws->norms16,
	                     ws->packed_means, ws->norms, a.k, half.kp, CELL_POOL_UNITS };
	if (!sizing_only() && ((size_t)half.kp * KBLOCK * 3 / 2 > ws->packed16_cap || rank16_norms_floats(half.kp) > ws->norms16_cap ||
	                       (size_t)half.kp / TILE * tile_floats(row_floats<1, true>()) > ws->packed_cap || split_norms_floats(half.kp) > ws->norms_cap))
		return fail(KMX_ERR_DEVICE, "assign (cells): launch refused, the packed rows of k %u do not fit their buffers", a.k);
	void (*build)(CellArgs) = a.layout_means == KMX_AOS ? build_cells_kernel<D, KMX_AOS> : build_cells_kernel<D, KMX_SOA>;
	KMX_HIP(hipFuncSetAttribute((const void*)build, hipFuncAttributeMaxDynamicSharedMemorySize, (int)build_lds));
	KMX_LAUNCH_KERNEL(build, dim3(power(CellShape<D>::TOP, D)), dim3(BUILD_THREADS), build_lds, stream(), b);
	KMX_LAUNCH_CHECK("build_cells_kernel");

	const CellAssignArgs w = { a.data, a.stride, a.means, a.stride_means, grid, table, pool, half.norms, half.low2, half.frame, half.scale,
	                           a.assignment, ws->listed, ws->counters, a.k, half.kp, a.n, choose ? 1u : 0u, half.kd };
	void (*assign)(CellAssignArgs) = a.layout == KMX_AOS ? (a.layout_means == KMX_AOS ? assign_cells_kernel<D, KMX_AOS, KMX_AOS> : assign_cells_kernel<D, KMX_AOS, KMX_SOA>)
	                                                     : (a.layout_means == KMX_AOS ? assign_cells_kernel<D, KMX_SOA, KMX_AOS> : assign_cells_kernel<D, KMX_SOA, KMX_SOA>);
	const uint32_t lds = a.k * 16 + CELL_STATIC, per_cu = std::max<uint32_t>(1, std::min<uint32_t>(2, dev.lds_bytes / lds));
	const uint32_t blocks = std::min((a.n + CELL_THREADS - 1) / CELL_THREADS, per_cu * dev.compute_units);
	exec->block_count = blocks;
	if ((rc = profile_begin(0))) return rc; /* (ended behind the packed sweep: one of the two does the work) */
	KMX_HIP(hipFuncSetAttribute((const void*)assign, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
	KMX_LAUNCH_KERNEL(assign, dim3(blocks), dim3(CELL_THREADS), lds, stream(), w);
	KMX_LAUNCH_CHECK("assign_cells_kernel");
	return KMX_OK;
}

bool cells_support(const AssignArgs& a, uint32_t lds_budget)
{
	if (a.dim < 2 || a.dim > 4 || a.k > CELL_MAX_K || a.k < 2 || a.n > (1u << 31) || a.ranking_only) return false;
	const uint32_t build_lds = a.k * a.dim * 4 + (a.k + 1) / 2 * 4 + BUILD_WAVES * BUILD_SHORT * 2 + 1024;
	const uint32_t assign_lds = a.k * 16 + CELL_STATIC;
	return std::max(build_lds, assign_lds) <= lds_budget && exact_dynamic_bytes(1, EXACT_GROUPS) + exact_static_bytes(false) <= lds_budget;
}

int launch_cells(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, const Cells16& half, bool choose)
{
	switch (a.dim) {
	case 2: return launch_cells_d<2>(a, exec, ws, dev, half, choose);
	case 3: return launch_cells_d<3>(a, exec, ws, dev, half, choose);
	case 4: return launch_cells_d<4>(a, exec, ws, dev, half, choose);
	default: return fail(KMX_ERR_UNSUPPORTED, "assign (cells): dim %u is not supported", a.dim);
	}
}

} // namespace kmx
