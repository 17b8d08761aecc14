/*
 * The update for clusters whose sums fit LDS as doubles: one pass over the rows in the order they lie in, every coordinate one ds_add_f64.
 *
 * ds_add_f64 takes 8 cycles for a wavefront on rows of 16 sums (two sums side by side in every bank of 8 bytes), as a plain read, addition and write would;
 * ds_add_f32 takes 194 whatever the addresses. So the sums are doubles, and nothing has to be sorted, listed or owned: the sorted chunks (update.hip) read rows
 * in the order of their clusters after a sort during which the memory idles, this kernel as a copy would. us per call, sorted chunks -> this:
 *   N = 8,388,608, d = 32, k = 1024 239 -> 208; N = 2M, d = 32, k = 1024 63 -> 55; N = 4M, d = 4, k = 4096 59 -> 26; N = 4M, d = 8, k = 1024 77 -> 31;
 *   N = 4M, d = 16, k = 512 85 -> 50; N = 1M, d = 64, k = 1024 65 -> 57; N = 1M, d = 128, k = 1024 135 -> 126.
 */
#include "kmx_internal.h"

#include <algorithm>
#include <type_traits>

namespace kmx {

constexpr uint32_t SUMS64_THREADS = 1024, SUMS64_WAVES = SUMS64_THREADS / WAVE;
constexpr uint32_t SUMS64_LANES = 64;      /* most coordinates of a slice: a lane each */
constexpr uint32_t SUMS64_XCDS = 8;

template <int LW> struct Sums64 {
	static constexpr uint32_t ROWS = WAVE / LW;                   /* rows of a request */
	static constexpr uint32_t SPAN = LW >= 16 ? 16 : LW >= 4 ? 4 : LW; /* consecutive rows of a group of LW lanes, whose memberships lie in the lanes of one register */
	static constexpr uint32_t REQUESTS = 16;                      /* of a step */
	static constexpr uint32_t REGS = REQUESTS / SPAN;             /* registers of memberships */
	static constexpr uint32_t POINTS = REQUESTS * ROWS;           /* of a step */
	static constexpr int STEPS = LW >= 16 ? 3 : 2;                /* under way */
};

/* the value that lane U of this lane's 16 (SPAN = 16), 4 or 2 lanes has */
template <int SPAN, int U> __device__ __forceinline__ uint32_t sums64_member(uint32_t v)
{
	if constexpr (SPAN == 1) return v;
	else return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, SPAN == 16 ? 0x150 + U /* row_newbcast */ : SPAN == 4 ? U * 0x55 : U * 0x05 + (U + 2) * 0x50 /* quad_perm */, 0xF, 0xF, true);
}

template <int LW, bool FULL, typename F>
__global__ void __launch_bounds__(SUMS64_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
update_sums64_kernel(const F* __restrict__ data, size_t stride, const uint32_t* __restrict__ assignment, F* __restrict__ partial, uint32_t* __restrict__ partial_counts,
                     uint32_t dim, uint32_t k, uint32_t n, uint32_t chunk_points, uint32_t chunks, uint32_t slices, uint32_t width, uint32_t copies)
{
	typedef Sums64<LW> S;
	/* copies of k + 1 rows of `width` sums (the last row takes what is no cluster's), then copies of k + 1 counts */
	extern __shared__ __attribute__((aligned(16))) double sums64[];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	/* the slices of a chunk share lines of memory: they lie on one XCD, whose second level of cache sees them side by side */
	const uint32_t at = blockIdx.x / SUMS64_XCDS, slice = at % slices, chunk = blockIdx.x % SUMS64_XCDS + SUMS64_XCDS * (at / slices);
	if (chunk >= chunks) return;
	const uint32_t copy = (k + 1) * width;
	uint32_t* counts = (uint32_t*)(sums64 + copies * copy);
	const uint32_t d0 = slice * width, mine = min(width, dim - d0);
	const uint32_t p_begin = (uint32_t)min((uint64_t)chunk * chunk_points, (uint64_t)n), count = min(chunk_points, n - p_begin);
	for (uint32_t i = tid; i < copies * copy; i += SUMS64_THREADS) sums64[i] = 0.0;
	for (uint32_t i = tid; i < copies * (k + 1); i += SUMS64_THREADS) counts[i] = 0u;
	__syncthreads();

	const uint32_t gl = lane % LW, group = lane / LW;
	const bool lane_on = gl < mine;
	const F* src = data + (size_t)p_begin * stride + d0 + min(gl, mine - 1);
	const uint32_t* members = assignment + p_begin;
	const uint32_t steps = (count + S::POINTS - 1) / S::POINTS;
	const bool counting = slice == 0 && gl < S::SPAN;
	const uint32_t which = group % copies;
	const uint32_t sums_at = (which * copy + gl) * 8, nowhere = (which * copy + k * width + gl % width) * 8;
	uint32_t* counts_at = counts + which * (k + 1);
	struct Step { F x[S::REQUESTS]; uint32_t member[S::REGS]; };
	auto request = [&](Step& s, uint32_t step) {
		const uint32_t first = step * S::POINTS;
#pragma unroll
		for (uint32_t r = 0; r < S::REGS; ++r) {
			const uint32_t p = first + (r * S::ROWS + group) * S::SPAN + gl % S::SPAN;
			s.member[r] = p < count ? members[p] : k;
		}
#pragma unroll
		for (uint32_t u = 0; u < S::REQUESTS; ++u) {
			const uint32_t p = first + (u / S::SPAN * S::ROWS + group) * S::SPAN + u % S::SPAN;
			s.x[u] = src[(size_t)min(p, count - 1) * stride];
		}
	};
	auto add = [&](Step& s) {
#pragma unroll
		for (uint32_t r = 0; r < S::REGS; ++r) {
			const uint32_t c = min(s.member[r], k);
			if (counting) atomicAdd(&counts_at[c], 1u);
			s.member[r] = c * (width * 8);
		}
		auto put = [&](auto tag) {
			constexpr uint32_t U = decltype(tag)::value;
			const uint32_t row = sums64_member<S::SPAN, U % S::SPAN>(s.member[U / S::SPAN]);
			unsafeAtomicAdd((double*)((char*)sums64 + (FULL || lane_on ? row + sums_at : nowhere)), (double)s.x[U]);
		};
#define KMX_PUT4(U) put(std::integral_constant<uint32_t, U>{}); put(std::integral_constant<uint32_t, U + 1>{}); put(std::integral_constant<uint32_t, U + 2>{}); put(std::integral_constant<uint32_t, U + 3>{});
		KMX_PUT4(0) KMX_PUT4(4) KMX_PUT4(8) KMX_PUT4(12)
#undef KMX_PUT4
	};
	constexpr int STEPS = S::STEPS;
	Step ring[STEPS];
#pragma unroll
	for (int i = 0; i < STEPS - 1; ++i)
		if (wave + SUMS64_WAVES * i < steps) request(ring[i], wave + SUMS64_WAVES * i);
	for (uint32_t step = wave; step < steps; step += SUMS64_WAVES * STEPS) {
#pragma unroll
		for (int i = 0; i < STEPS; ++i) {
			const uint32_t now = step + SUMS64_WAVES * i, then = now + SUMS64_WAVES * (STEPS - 1);
			if (then < steps) request(ring[(i + STEPS - 1) % STEPS], then);
			if (now < steps) add(ring[i]);
		}
	}
	__syncthreads();
	F* out = partial + (size_t)chunk * k * dim + d0 + gl;
	for (uint32_t c = tid / LW; c < k; c += SUMS64_THREADS / LW)
		if (lane_on) {
			double sum = sums64[c * width + gl];
			for (uint32_t i = 1; i < copies; ++i) sum += sums64[i * copy + c * width + gl];
			out[(size_t)c * dim] = (F)sum;
		}
	if (slice == 0)
		for (uint32_t c = tid; c < k; c += SUMS64_THREADS) {
			uint32_t size = counts[c];
			for (uint32_t i = 1; i < copies; ++i) size += counts[i * (k + 1) + c];
			partial_counts[(size_t)chunk * k + c] = size;
		}
}

/*
 * Where the sorted chunks (update.hip) are ahead of slices (floats; us per call, slices / sorted chunks):
 *   - wide slices whose sums to write are an eighth of what is read and more (N = 140625, d = 128, k = 300 29.3 / 24.1; N = 162500, d = 80, k = 500 28.9 / 23.9; N = 250000, d = 128,
 *     k = 300, a seventh, 37.0 / 33.4; N = 400000, d = 70, k = 300, a tenth, 34.8 / 40.7), of 32 coordinates and fewer nearly a half (N = 82000, d = 110, k = 600
 *     22.4 / 20.5; N = 102000, d = 127, k = 600, three eighths, 25.5 / 25.8);
 *   - slices that are parts of a line, from 2^26 floats on, which the caches do not hold: of 16 that begin inside lines, up to 2^27 floats, and while they leave a tenth of the compute units
 *     over up to 200 million (sorted chunks in shares of the slices' time: d = 100, k = 1000, seven slices x 32 chunks: N = 720000 0.87, 900000 0.85, 1.8M 0.94, 2.4M 1.18; d = 90,
 *     six x 40: N = 1M 0.91, 1.3M 1.00, 2.2M 1.05; d = 120, eight x 32: N = 600000 1.02, 1M 1.02); of 8 of rows of whole lines (N = 6.25M, d = 32, k = 2000 0.90; N = 1.9M, d = 48
 *     0.92; but d = 36 1.05) and of 4 (N = 6.25M, d = 32, k = 4000 0.78; N = 2.5M, d = 36 0.88; but N = 7.1M, d = 28 1.11).
 */
static bool sorted_pays(uint32_t dim, uint32_t k, uint32_t n, uint32_t width, uint32_t slices, uint32_t chunks, uint32_t compute_units)
{
	const uint64_t written = (uint64_t)chunks * k; /* rows of sums */
	if (width > 32 ? slices >= 2 && written * 8 > n : width > 16 && written * 20 > (uint64_t)n * 9) return true;
	const uint64_t floats = (uint64_t)n * dim;
	if (floats < (1u << 26)) return false;
	if (width == 16 && dim > 64 && dim % 16 != 0) {
		const uint32_t busy = slices * chunks;
		return floats < (busy * 10 < compute_units * 9 ? 200000000u : busy < compute_units ? 1u << 27 : 0u);
	}
	return dim >= 32 && (width <= 4 || (width == 8 && dim % 16 == 0));
}

/*
 * A work-group per compute unit: slices of the coordinates x chunks of the points, as few slices as let their sums fit LDS, ten at most (d = 160, k = 600: ten
 * 139 us, five 129, sorted chunks 158; d = 256, k = 1024: sixteen 277, sorted chunks 242; N = 1M here and below). Slices are equal, or, in floats, of whole 64
 * bytes up to 32 coordinates (sorted chunks / equal / these: d = 33, k = 1000 54 / 41 / 35; d = 80, k = 1000 86 / 101 / 77; wider ones d = 100, k = 100,
 * N = 500000: 50 + 50 38, 64 + 36 46; d = 112, N = 392857 56 + 56 34.5, 64 + 48 36.6), and of whole 64 bytes where rows consist of such in three slices and more (d = 160, k = 100: N = 412500
 * 54 + 54 + 52 60, 64 + 64 + 32 49.5, sorted chunks 53; N = 1.25M 180, 156, 164). Rows of up to 48 floats go in slices of 16, doubles in slices of 32 or two, even where the whole row fits (d = 40,
 * k = 300: 34, whole 37; doubles, N = 2M, d = 32, k = 500: 103, 113): the sums to write are fewer. But from some 60 million floats on, which the memory-side cache
 * does not hold, a row that begins anywhere is read once (slices of 16 / whole: d = 36, k = 18, N = 1.6M 43.6 / 42.8, N = 1.9M 64.6 / 53.4, N = 2.8M 113 / 86; d = 18 58.8 / 58.6
 * at 68 million, 81 / 75 at 80; d = 44, N = 1.3M 41 / 44, N = 1.5M 64 / 53; d = 48, k = 200, N = 3.3M 135 / 129; d = 32, N = 5M 128 / 126). Of rows with a gap
 * of 16 floats and more behind them, which share fewer lines, the memory that they span counts, from 45 million floats on where the last slice has eight coordinates and fewer (stride dim + 32:
 * d = 17, N = 1.6M 72 / 55; d = 20, N = 1.5M 65 / 52; d = 34, N = 1.4M, stride 50, 72 / 51; d = 20, N = 577000 level), else from 75 (d = 26, N = 1.2M 1.1; d = 42, N = 1.1M 1.07; d = 30 0.98). Doubles whose sums do not fit as a whole: 16 at a time (N = 500000,
 * d = 128, k = 1024: 123, slices of 19 142, sums of ranges of clusters 204), equal where the last would be narrow (N = 1M, d = 33, k = 1000: 73,
 * 16 + 16 + 1 86, ranges 77), eight at a time where rows are odd multiples of 32 bytes and short (N = 1M, d = 24, k = 1200: 43, 12 + 12 47, ranges 53).
 * Seven slices leave an eighth of the compute units over: where rows begin inside lines and the caches do not hold them, the ranges (d = 100, k = 600: N = 500000 103, ranges 91,
 * N = 1M 192, 176, but N = 300000 48, 52, N = 150000 30, 34; d = 105 105, 93, 197, 180, but 51, 54 and 31, 35). Rows of more than 192 floats in slices of 32 and less lose
 * (N = 500000, d = 256, k = 600: 123 against 121).
 * As many chunks per XCD as it has compute units for: one more somewhere comes alone at the end (d = 48, k = 1024: 85 chunks of three slices 62, 80 42).
 * A chunk has as many points as there are clusters, 512 at least: its sums are written and read once more (N = 200000, d = 4, k = 4000: 256 chunks 17 us, 50
 * 14, sorted chunks 31; N = 50000, d = 32, k = 1000: 17, 14, 16); where that leaves compute units over and a slice is wide, more slices (N = 100000, d = 32,
 * k = 500: one slice 16, two 13). Sums of doubles are twice as dear: four times as many points, and few points are left to the kernels that add to the means
 * where they lie (N = 400000, d = 32, k = 1000 33.2, those 34.2; N = 100000, k = 500 17.4, 17.1; N = 200000, d = 4, k = 4000 19.0, 16.2;
 * rows of one slice, whose work-groups are as few as the chunks, unless they are 4 or 8 doubles, which a group of lanes reads without a gap: d = 11, N = 225824, k = 1105 24.2, 16.0; N = 300000
 * 24.3, 20.9; N = 400000, k = 2000 28.2, 28.7; d = 6, N = 400000, k = 2000 26.3, 16.2; d = 13, N = 225824, k = 700 18.8, 21.1; but d = 8, N = 225824, k = 1105 15.7, 18.5;
 * d = 4, N = 300000, k = 2000 15.4, 18.3).
 * Few clusters: the rows of a request mostly meet at the same sums, which costs an LDS cycle each; copies of them, as many as rows (N = 16M, d = 2,
 * k = 2: 90 us without, 34 with).
 */
struct Sums64Plan { uint32_t width, slices, copies, chunks, chunk_points, lds_bytes; };
constexpr uint32_t SUMS64_SLICES = 10;

static bool plan_sums64(uint32_t dim, size_t stride, uint32_t k, uint32_t n, bool doubles, uint32_t budget, uint32_t compute_units, Sums64Plan* plan)
{
	auto bytes = [&](uint32_t width) -> uint64_t { return ((uint64_t)k + 1) * (8 * width + 4); };
	auto slices_of = [&](uint32_t width) -> uint32_t { return (dim - 1) / width + 1; };
	auto chunks_of = [&](uint32_t width) -> uint32_t { return std::max<uint32_t>(1, compute_units / SUMS64_XCDS / slices_of(width)) * SUMS64_XCDS; };
	if (dim > SUMS64_SLICES * SUMS64_LANES || (doubles && n / 200 < k && (uint64_t)k * dim > 8192)) return false;
	if (doubles && dim <= 16 && dim != 4 && dim != 8 && n / 300 < k && (uint64_t)k * dim > 6144) return false; /* (one slice: as many work-groups as chunks) */
	const uint64_t least_points = std::max<uint64_t>(512, (uint64_t)k * (doubles ? 4 : 1));
	/* doubles whose sums do not fit as a whole */
	const bool parts = doubles && bytes(dim) > budget, eights = parts && dim <= 56 && dim % 4 == 0 && dim % 16 != 0;
	if (parts && slices_of(16) == 7 && dim % 16 != 0 && (uint64_t)n * dim >= 40000000) return false;
	const bool beyond_caches = (uint64_t)n * dim >= 60000000 || (stride >= dim + 16 && n * std::min<uint64_t>(stride, dim + 32) >= ((dim - 1) % 16 < 8 ? 45000000 : 75000000));
	const bool whole_row = !doubles && dim > 16 && dim <= 48 && bytes(dim) <= budget && beyond_caches;
	const uint32_t fewest = dim <= 16 || whole_row ? 1 : parts ? slices_of(eights ? 8 : 16) : doubles ? std::max<uint32_t>(2, slices_of(32)) : dim <= 48 ? slices_of(16) : slices_of(SUMS64_LANES);
	uint32_t width = 0;
	for (uint32_t slices = fewest; slices <= SUMS64_SLICES && (width == 0 || width > 16); ++slices) {
		const uint32_t equal = (dim - 1) / slices + 1, whole = equal > 8 ? (equal + 15) / 16 * 16 : equal > 4 ? 8 : 4;
		const bool as_is = doubles ? !eights && !(parts && equal > 8 && (dim - 1) % 16 >= 7) : equal > 32 && !(dim % 16 == 0 && slices >= 3);
		const uint32_t w = dim <= 16 || slices == 1 || as_is ? equal : whole;
		if (bytes(w) > budget || (dim > 192 && w <= 32 && !doubles)) continue;
		if (width != 0 && least_points * 2 * chunks_of(width) <= n) break; /* enough points for this many work-groups */
		width = w;
	}
	if (width == 0) return false;
	uint32_t lanes = 1, copies = 1;
	while (lanes < width) lanes *= 2;
	while (copies * 2 <= WAVE / lanes && 2 * copies * bytes(width) <= std::min<uint32_t>(budget, 48 * 1024)) copies *= 2;
	const uint64_t points = (std::max<uint64_t>(least_points, ((uint64_t)n + chunks_of(width) - 1) / chunks_of(width)) + WAVE - 1) / WAVE * WAVE;
	const uint32_t chunk_points = (uint32_t)std::min<uint64_t>(points, 1u << 31);
	*plan = { width, slices_of(width), copies, (uint32_t)(((uint64_t)n + chunk_points - 1) / chunk_points), chunk_points, (uint32_t)(copies * bytes(width)) };
	return true;
}

/* the sum of a row of 16 lanes */
__device__ __forceinline__ double sums64_of_16(double v)
{
	auto turned = [](double x, auto by) -> double { /* row_ror */
		const int low = __builtin_amdgcn_update_dpp(0, __double2loint(x), 0x120 + decltype(by)::value, 0xF, 0xF, true);
		const int high = __builtin_amdgcn_update_dpp(0, __double2hiint(x), 0x120 + decltype(by)::value, 0xF, 0xF, true);
		return __hiloint2double(high, low);
	};
	v += turned(v, std::integral_constant<int, 8>{});
	v += turned(v, std::integral_constant<int, 4>{});
	v += turned(v, std::integral_constant<int, 2>{});
	return v + turned(v, std::integral_constant<int, 1>{});
}

/*
 * The same for SoA points: a lane takes a point, W columns of 64 points are W requests, and nothing is copied into rows first. Lanes that meet in a column's
 * sums have any clusters, so a column's sums lie side by side (rows of sums would leave whole banks unused), each in `copies` places for neighbouring
 * lanes. Points that come sorted by cluster are added up in registers first, 16 at a time: lanes that meet at a sum take turns of 3 cycles each.
 * What bounds it: memory (N = 8.4M, d = 32, k = 1024 208 us, 5.2 TB/s; AoS 219 on that card) or, from the caches, the conflicts of 64 lanes at random
 * sums, 26 cycles an addition (N = 2M 72 us). us per update, rows copied first or (d < 8) ds_add_f32 -> this:
 *   N = 8.4M, d = 32, k = 1024 752 -> 208; N = 250007, d = 50, k = 300 51 -> 22; N = 2M, d = 128, k = 1024 785 -> 212; N = 4M, d = 4, k = 4096 123 -> 29;
 *   N = 16M, d = 2, k = 2 204 -> 37; N = 1M, d = 64, k = 4000 247 -> 72; N = 2M, d = 32, k = 1024, points sorted by cluster 249 -> 74 (without the sums of 16 355);
 *   doubles: N = 2M, d = 32, k = 1024 350 -> 131; N = 500000, d = 128, k = 1024 865 -> 116; N = 250000, d = 50, k = 300 143 -> 26.
 */
template <int W, typename F>
__global__ void __launch_bounds__(SUMS64_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
update_columns64_kernel(const F* __restrict__ data, size_t stride, const uint32_t* __restrict__ assignment, F* __restrict__ partial, uint32_t* __restrict__ partial_counts,
                        uint32_t dim, uint32_t k, uint32_t n, uint32_t chunk_points, uint32_t chunks, uint32_t slices, uint32_t copies, uint32_t xcds)
{
	constexpr uint32_t SUBS = W >= 8 ? 1 : W >= 4 ? 2 : 4, POINTS = SUBS * WAVE;
	constexpr int STEPS = sizeof(F) == 8 ? 2 : 3; /* under way */
	/* W columns of (k + 1) * copies sums (the last ones take what is no cluster's), then as many counts as a column has sums */
	extern __shared__ __attribute__((aligned(16))) double sums64[];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	/* few slices: those of a chunk, which write to the same lines, on one XCD */
	const uint32_t at = blockIdx.x / xcds, slice = at % slices, chunk = blockIdx.x % xcds + xcds * (at / slices), column = (k + 1) * copies;
	if (chunk >= chunks) return;
	uint32_t* counts = (uint32_t*)(sums64 + W * column);
	const uint32_t d0 = slice * W, mine = min((uint32_t)W, dim - d0);
	const uint32_t p_begin = (uint32_t)min((uint64_t)chunk * chunk_points, (uint64_t)n), count = min(chunk_points, n - p_begin);
	for (uint32_t i = tid; i < W * column; i += SUMS64_THREADS) sums64[i] = 0.0;
	for (uint32_t i = tid; i < column; i += SUMS64_THREADS) counts[i] = 0u;
	__syncthreads();

	const char* from[W];
#pragma unroll
	for (uint32_t j = 0; j < W; ++j) from[j] = (const char*)(data + (size_t)(d0 + min(j, mine - 1)) * stride + p_begin); /* (behind the row's last column that one again, to sums nobody reads) */
	const uint32_t* members = assignment + p_begin;
	const uint32_t steps = (count + POINTS - 1) / POINTS;
	struct Step { F x[SUBS][W]; uint32_t member[SUBS]; };
	auto request = [&](Step& s, uint32_t step) {
#pragma unroll
		for (uint32_t sub = 0; sub < SUBS; ++sub) {
			const uint32_t p = step * POINTS + sub * WAVE + lane, inside = min(p, count - 1);
			s.member[sub] = p < count ? members[p] : k;
#pragma unroll
			for (uint32_t j = 0; j < W; ++j) s.x[sub][j] = *(const F*)(from[j] + inside * (uint32_t)sizeof(F));
		}
	};
	auto add = [&](Step& s) {
#pragma unroll
		for (uint32_t sub = 0; sub < SUBS; ++sub) {
			const uint32_t c = min(s.member[sub], k) * copies + lane % copies;
#pragma unroll
			for (uint32_t j = 0; j < W; ++j) asm volatile("" : "+v"(s.x[sub][j])); /* (all here before the paths part, so that neither waits for later steps too) */
			if (slice == 0) atomicAdd(&counts[c], 1u);
			if (__builtin_amdgcn_ballot_w64(s.member[sub] == sums64_member<16, 0>(s.member[sub])) == ~0ull) {
				/* 16 neighbours in one cluster, and so all over the wavefront: lanes that meet at a sum would take turns of 3 cycles each */
#pragma unroll
				for (uint32_t j = 0; j < W; ++j) {
					const double sum = sums64_of_16((double)s.x[sub][j]);
					if (lane % 16 == 0) unsafeAtomicAdd(&sums64[j * column + c], sum);
				}
			}
			else
#pragma unroll
				for (uint32_t j = 0; j < W; ++j) unsafeAtomicAdd(&sums64[j * column + c], (double)s.x[sub][j]);
		}
	};
	Step ring[STEPS];
#pragma unroll
	for (int i = 0; i < STEPS - 1; ++i)
		if (wave + SUMS64_WAVES * i < steps) request(ring[i], wave + SUMS64_WAVES * i);
	for (uint32_t step = wave; step < steps; step += SUMS64_WAVES * STEPS) {
#pragma unroll
		for (int i = 0; i < STEPS; ++i) {
			const uint32_t now = step + SUMS64_WAVES * i, then = now + SUMS64_WAVES * (STEPS - 1);
			if (then < steps) request(ring[(i + STEPS - 1) % STEPS], then);
			if (now < steps) add(ring[i]);
		}
	}
	__syncthreads();
	F* out = partial + (size_t)chunk * k * dim + d0;
	for (uint32_t i = tid; i < k * W; i += SUMS64_THREADS) {
		const uint32_t c = i / W, j = i % W;
		if (j >= mine) continue;
		const double* sums = sums64 + j * column + c * copies;
		double sum = sums[0];
		for (uint32_t q = 1; q < copies; ++q) sum += sums[q];
		out[(size_t)c * dim + j] = (F)sum;
	}
	if (slice == 0)
		for (uint32_t c = tid; c < k; c += SUMS64_THREADS) {
			uint32_t size = counts[c * copies];
			for (uint32_t q = 1; q < copies; ++q) size += counts[c * copies + q];
			partial_counts[(size_t)chunk * k + c] = size;
		}
}

/*
 * Slices of up to 16 columns, equal as far as they can be. Up to eight of them: as many chunks per XCD as it has compute units for; more: as many chunks as fill
 * the compute units in one to four rounds (17 slices, 15 chunks). Chunks of as many points as there are clusters at least, as above. Copies while
 * two points of a wavefront would often meet in one place.
 */
constexpr uint32_t COLUMNS64 = 16, COLUMNS64_TOGETHER = 8;

static bool plan_columns64(uint32_t dim, uint32_t k, uint32_t n, bool doubles, uint32_t budget, uint32_t compute_units, Sums64Plan* plan)
{
	if ((uint64_t)(k + 1) * 12 > budget || dim > 8192 || (doubles && n / 200 < k && (uint64_t)k * dim > 8192)) return false;
	const uint32_t most = std::min<uint32_t>(COLUMNS64, (budget / (k + 1) - 4) / 8), slices = (dim - 1) / most + 1, width = (dim - 1) / slices + 1;
	const uint32_t bytes = (k + 1) * (8 * width + 4);
	uint32_t copies = 1, chunks = 0, rounds = 0;
	while (copies < 32 && copies * k < 256 && 2 * copies * bytes <= std::min<uint32_t>(budget, 64 * 1024)) copies *= 2;
	if (slices <= COLUMNS64_TOGETHER) chunks = std::max<uint32_t>(1, compute_units / SUMS64_XCDS / slices) * SUMS64_XCDS;
	else for (uint32_t r = 1; r <= 4; ++r) {
		const uint32_t fit = compute_units * r / slices;
		if (fit > 0 && (chunks == 0 || (uint64_t)fit * 20 * rounds > (uint64_t)chunks * 21 * r)) { chunks = fit; rounds = r; }
	}
	const uint64_t least_points = std::max<uint64_t>(512, (uint64_t)k * (doubles ? 4 : 1));
	const uint64_t points = (std::max<uint64_t>(least_points, ((uint64_t)n + std::max(chunks, 1u) - 1) / std::max(chunks, 1u)) + WAVE - 1) / WAVE * WAVE;
	const uint32_t chunk_points = (uint32_t)std::min<uint64_t>(points, 1u << 28); /* (offsets of 32 bits) */
	*plan = { width, (dim - 1) / width + 1, copies, (uint32_t)(((uint64_t)n + chunk_points - 1) / chunk_points), chunk_points, copies * bytes };
	return true;
}

template <int W, typename F>
static int launch_columns64(uint32_t width, const F* data, size_t stride, const uint32_t* assignment, F* partial, uint32_t* partial_counts, uint32_t dim, uint32_t k, uint32_t n, const Sums64Plan& p)
{
	if constexpr (W > 1)
		if (width < W) return launch_columns64<W - 1, F>(width, data, stride, assignment, partial, partial_counts, dim, k, n, p);
	auto kernel = update_columns64_kernel<W, F>;
	KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds_bytes));
	const uint32_t xcds = p.slices <= COLUMNS64_TOGETHER ? SUMS64_XCDS : 1;
	KMX_LAUNCH_KERNEL(kernel, dim3((p.chunks + xcds - 1) / xcds * xcds * p.slices), dim3(SUMS64_THREADS), p.lds_bytes, stream(),
	                  data, stride, assignment, partial, partial_counts, dim, k, n, p.chunk_points, p.chunks, p.slices, p.copies, xcds);
	KMX_LAUNCH_CHECK("update_columns64_kernel");
	return KMX_OK;
}

/*
 * Rows of more coordinates than slices are worth it: a work-group takes the clusters c = range (modulo `ranges`, a power of two) of its part of the points, up to 256
 * of their coordinates. A wavefront looks through the memberships of its share, lists the points that are the work-group's, and then reads their rows, four
 * coordinates per lane, eight rows under way while eight are added.
 * A compute unit reads 50 GB/s at most, twice what all of them together get from memory: a range with many points has to have many work-groups. Each
 * work-group counts the ranges in the same sample of the memberships (16384 of them, 16 at a place) and finds from that which range it
 * has and which part of the points (in equal parts, N = 1M, d = 256, k = 1024: 190 us on equal clusters, 758 an iteration on normal ones, 1246 with all points
 * in one; now 202, 741, 230). What bounds it: memory, 1.07 GB in 188 us of the kernel's 193 (5.6 TB/s), then the fold, 6.
 */
constexpr uint32_t RANGES64_LIST = 384, RANGES64_SCAN = 4 * WAVE, RANGES64_ROWS = 8; /* entries of a wavefront's list; points looked at together; rows of a step */
constexpr uint32_t RANGES64_MOST = 32, RANGES64_SAMPLES = 16;                         /* ranges; places of the sample per 16 lanes */
typedef float f32x4_row __attribute__((ext_vector_type(4), aligned(4)));

/* partial: [work-group of a slice][its clusters][dim], partial_counts: [work-group][its clusters], starts: a range's first work-group, then their number */
__global__ void __launch_bounds__(SUMS64_THREADS) __attribute__((amdgpu_waves_per_eu(4)))
update_ranges64_kernel(const float* __restrict__ data, size_t stride, const uint32_t* __restrict__ assignment, float* __restrict__ partial, uint32_t* __restrict__ partial_counts,
                       uint32_t* __restrict__ starts, uint32_t dim, uint32_t k, uint32_t n, uint32_t groups, uint32_t log_ranges, uint32_t width)
{
	/* per cluster of the range four times width / 4 sums (a lane's coordinates lie in each of them), a row more for what fills up a step; counts; lists */
	extern __shared__ __attribute__((aligned(16))) double sums64[];
	__shared__ uint32_t in_range[RANGES64_MOST], begin[RANGES64_MOST + 1];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t ranges = 1u << log_ranges, most = (k + ranges - 1) >> log_ranges;
	const uint32_t me = blockIdx.x % groups, slice = blockIdx.x / groups, d0 = slice * width, lanes = min(width, dim - d0) / 4, row = width; /* (whole pieces of four) */
	uint32_t* counts = (uint32_t*)(sums64 + (most + 1) * row);
	uint32_t* lists = counts + most;
	uint32_t* list = lists + wave * (RANGES64_LIST + RANGES64_ROWS);
	{
		uint32_t sample[RANGES64_SAMPLES];
		constexpr uint32_t PLACES = SUMS64_THREADS / 16 * RANGES64_SAMPLES;
		const bool all = n <= PLACES * 16;
		const uint32_t whole = (n - min(n, 16u)) / PLACES, rest = (n - min(n, 16u)) % PLACES; /* (n <= 2^24, 2^10 places) */
#pragma unroll
		for (uint32_t i = 0; i < RANGES64_SAMPLES; ++i) {
			const uint32_t place = i * (SUMS64_THREADS / 16) + tid / 16, p = (all ? place * 16 : place * whole + place * rest / PLACES) + tid % 16;
			sample[i] = p < n ? assignment[p] : ~0u;
		}
		for (uint32_t i = tid; i < (most + 1) * row; i += SUMS64_THREADS) sums64[i] = 0.0;
		for (uint32_t i = tid; i < most; i += SUMS64_THREADS) counts[i] = 0u;
		for (uint32_t i = tid; i < ranges * WAVE; i += SUMS64_THREADS) lists[i] = 0u; /* a range's points by the lane that saw them */
		__syncthreads();
#pragma unroll
		for (uint32_t i = 0; i < RANGES64_SAMPLES; ++i)
			if (sample[i] < k) atomicAdd(&lists[(sample[i] & (ranges - 1)) * WAVE + lane], 1u);
		__syncthreads();
		for (uint32_t r = wave; r < ranges; r += SUMS64_WAVES) {
			uint32_t seen = lists[r * WAVE + lane];
			for (int off = WAVE / 2; off > 0; off >>= 1) seen += (uint32_t)__shfl_xor((int)seen, off);
			if (lane == 0) in_range[r] = seen;
		}
		__syncthreads();
	}
	if (wave == 0) {
		const uint32_t seen = lane < ranges ? in_range[lane] : 0;
		uint32_t total = seen;
		for (int off = WAVE / 2; off > 0; off >>= 1) total += (uint32_t)__shfl_xor((int)total, off);
		/* one work-group each, the others in proportion, those that the rounding leaves to the first ranges */
		uint32_t share = lane < ranges ? 1 + (uint32_t)((uint64_t)(groups - ranges) * seen / max(total, 1u)) : 0, given = share;
		for (int off = WAVE / 2; off > 0; off >>= 1) given += (uint32_t)__shfl_xor((int)given, off);
		const uint32_t left = groups - given;
		if (lane < ranges) share += left / ranges + (lane < left % ranges ? 1 : 0);
		uint32_t up_to = share;
		for (int off = 1; off < WAVE; off <<= 1) {
			const uint32_t up = (uint32_t)__shfl_up((int)up_to, off);
			if (lane >= (uint32_t)off) up_to += up;
		}
		if (lane < ranges) begin[lane + 1] = up_to;
		if (lane == 0) begin[0] = 0;
	}
	__syncthreads();
	if (blockIdx.x == 0 && tid <= ranges) starts[tid] = begin[tid];
	uint32_t range = 0;
	while (range + 1 < ranges && begin[range + 1] <= me) ++range;
	const uint32_t parts = begin[range + 1] - begin[range], part = me - begin[range];
	const uint32_t p_begin = (uint32_t)((uint64_t)part * n / parts), count = (uint32_t)((uint64_t)(part + 1) * n / parts) - p_begin;

	const uint32_t* members = assignment + p_begin;
	const uint32_t piece = min(lane, lanes - 1);
	const char* rows = (const char*)(data + (size_t)p_begin * stride + d0) + piece * 16;
	const bool lane_on = lane < lanes;
	const uint32_t sums_at = piece * 8;
	const uint32_t scans = (count + RANGES64_SCAN - 1) / RANGES64_SCAN;
	uint32_t scan = wave;
	while (scan < scans) {
		uint32_t listed = 0;
		bool room = true;
		while (room && scan < scans) {
			uint32_t member[2][4];
#pragma unroll
			for (uint32_t s = 0; s < 2; ++s)
#pragma unroll
				for (uint32_t q = 0; q < 4; ++q) {
					const uint32_t p = (scan + s * SUMS64_WAVES) * RANGES64_SCAN + q * WAVE + lane;
					member[s][q] = p < count ? members[p] : ~0u;
				}
#pragma unroll
			for (uint32_t s = 0; s < 2; ++s) {
				room = room && listed + RANGES64_SCAN <= RANGES64_LIST;
				if (!room) continue;
#pragma unroll
				for (uint32_t q = 0; q < 4; ++q) {
					const bool mine = member[s][q] < k && (member[s][q] & (ranges - 1)) == range;
					const unsigned long long mask = __builtin_amdgcn_ballot_w64(mine);
					if (mine) {
						const uint32_t c = member[s][q] >> log_ranges;
						if (slice == 0) atomicAdd(&counts[c], 1u);
						list[listed + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = c << 24 | (scan * RANGES64_SCAN + q * WAVE + lane);
					}
					listed += (uint32_t)__popcll(mask);
				}
				scan += SUMS64_WAVES;
			}
		}
		if (listed == 0) continue;
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		const uint32_t last = list[listed - 1] & 0xFFFFFFu;
		if (lane < RANGES64_ROWS) list[listed + lane] = most << 24 | last; /* the last step's rows beyond the list */
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		struct Step { f32x4_row x[RANGES64_ROWS]; uint32_t to[RANGES64_ROWS]; };
		auto request = [&](Step& s, uint32_t first) {
#pragma unroll
			for (uint32_t u = 0; u < RANGES64_ROWS; ++u) {
				const uint32_t e = (uint32_t)__builtin_amdgcn_readfirstlane((int)list[first + u]);
				s.to[u] = e >> 24;
				s.x[u] = *(const f32x4_row*)(rows + (size_t)(e & 0xFFFFFFu) * stride * sizeof(float));
			}
		};
		auto add = [&](Step& s) {
#pragma unroll
			for (uint32_t u = 0; u < RANGES64_ROWS; ++u) {
				char* to = (char*)sums64 + s.to[u] * (row * 8) + sums_at;
				if (lane_on) {
#pragma unroll
					for (uint32_t e = 0; e < 4; ++e) unsafeAtomicAdd((double*)(to + e * (row * 2)), (double)s.x[u][e]);
				}
			}
		};
		Step a, b;
		request(a, 0);
		for (uint32_t first = 0; first < listed; first += 2 * RANGES64_ROWS) {
			request(b, min(first + RANGES64_ROWS, listed));
			add(a);
			request(a, min(first + 2 * RANGES64_ROWS, listed));
			add(b);
		}
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
	}
	__syncthreads();
	float* out = partial + (size_t)me * most * dim + d0 + piece * 4;
	for (uint32_t i = wave; i < most; i += SUMS64_WAVES) {
		const double* sums = sums64 + i * row + piece;
		if (lane_on) *(f32x4_row*)(out + (size_t)i * dim) = f32x4_row{ (float)sums[0], (float)sums[row / 4], (float)sums[row / 2], (float)sums[row / 4 * 3] };
	}
	if (slice == 0)
		for (uint32_t i = tid; i < most; i += SUMS64_THREADS) partial_counts[(size_t)me * most + i] = counts[i];
}

/* means and sizes from what update_ranges64_kernel left: a work-group per cluster, four wavefronts share out its range's work-groups */
template <int LM>
__global__ void __launch_bounds__(4 * WAVE)
fold_ranges64_kernel(const float* __restrict__ partial, const uint32_t* __restrict__ partial_counts, const uint32_t* __restrict__ starts, float* __restrict__ means, size_t stride_means,
                     uint32_t* __restrict__ sizes, uint32_t dim, uint32_t k, uint32_t log_ranges, uint32_t divide)
{
	__shared__ double part[4][4][WAVE];
	const uint32_t c = blockIdx.x, lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE, ranges = 1u << log_ranges, most = (k + ranges - 1) >> log_ranges;
	const uint32_t first = starts[c & (ranges - 1)], last = starts[(c & (ranges - 1)) + 1], local = c >> log_ranges;
	uint32_t size = 0;
	for (uint32_t g = first + lane; g < last; g += WAVE) size += partial_counts[(size_t)g * most + local];
	for (int off = WAVE / 2; off > 0; off >>= 1) size += (uint32_t)__shfl_xor((int)size, off);
	if (threadIdx.x == 0) sizes[c] = size;
	for (uint32_t q0 = 0; q0 < dim / 4; q0 += WAVE) {
		const uint32_t q = min(q0 + lane, dim / 4 - 1);
		double sum[4] = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll 4
		for (uint32_t g = first + wave; g < last; g += 4) {
			const f32x4_row v = *(const f32x4_row*)(partial + ((size_t)g * most + local) * dim + q * 4);
#pragma unroll
			for (uint32_t e = 0; e < 4; ++e) sum[e] += (double)v[e];
		}
#pragma unroll
		for (uint32_t e = 0; e < 4; ++e) part[wave][e][lane] = sum[e];
		__syncthreads();
		/* wavefront `wave` has coordinate `wave` of the lanes' four */
		const float total = (float)(part[0][wave][lane] + part[1][wave][lane] + part[2][wave][lane] + part[3][wave][lane]);
		if (q0 + lane < dim / 4) means[elem<LM>(stride_means, c, q * 4 + wave)] = !divide ? total : size ? total / (float)size : 0.0f;
		__syncthreads();
	}
}

/*
 * Where ranges beat the sorted chunks (update.hip) or slices of 16 coordinates (us per update, those -> ranges; the sample and the fold cost 8 us): from 600 clusters on.
 * Up to 256 dimensions from 25 million floats on: N = 1M, d = 256, k = 1024 234 -> 202; d = 192 191 -> 162; N = 500000, d = 200, k = 1000 104 -> 92; d = 224, k = 2000 135 -> 113;
 * N = 100000, d = 256, k = 1000 34.7 -> 33.4, but d = 200, k = 600 28 -> 31; N = 190000, d = 148, k = 354 34 -> 37. More,
 * of whose clusters the sorted chunks write 32 sets of partial sums and more: N = 100000, d = 300, k = 2000 71 -> 45; N = 131071, d = 512, k = 1000 79 -> 60, k = 600 65 -> 58, k = 400 57 -> 59. Half of the points in
 * one cluster, N = 1M, d = 256, k = 1024 448 -> 216; all of them 702 -> 230; sorted by cluster 292 -> 225. Slices of 16: N = 1M, d = 160, k = 600 128.7 -> 128.3,
 * N = 300000, d = 144, k = 1000 37.6 -> 40.7: stay. More than 256 dimensions, few points: the sorted chunks' sums are fewer (802 shapes of 1 to 26 million floats; N = 8830, d = 372, k = 606
 * 18.1 -> 22.6, N = 16343, d = 304, k = 717 19.9 -> 23.3, but N = 6706, d = 400, k = 1585 27.9 -> 21.2): ranges from 280000 sums or 5 million floats on; below 1.10 in the mean, from there 0.75.
 */
static bool ranges64_pays(uint32_t dim, uint32_t k, uint32_t n, bool planned)
{
	const size_t floats = (size_t)n * dim;
	return !planned && k >= 600 && (dim > 256 ? floats >= 5000000 || (size_t)k * dim >= 280000 : floats >= (3u << 23));
}

struct Ranges64Plan { uint32_t width, slices, log_ranges, groups, lds_bytes; };

static size_t ranges64_words(const Ranges64Plan& p, uint32_t dim, uint32_t k)
{
	const size_t rows = (size_t)p.groups * (((size_t)k + (1u << p.log_ranges) - 1) >> p.log_ranges);
	return rows * (dim + 1) + RANGES64_MOST + 1;
}

static bool plan_ranges64(uint32_t dim, uint32_t k, uint32_t n, uint32_t budget, uint32_t compute_units, Ranges64Plan* plan)
{
	if (dim % 4 != 0 || dim <= 128 || dim > 1024 || n > (1u << 24)) return false; /* (numbers of points of 24 bits) */
	const uint32_t slices = (dim - 1) / 256 + 1, width = ((dim - 1) / slices + 4) / 4 * 4;
	const uint32_t tables = (2 * RANGES64_MOST + 1) * 4 + 64;
	static_assert(SUMS64_WAVES * (RANGES64_LIST + RANGES64_ROWS) >= RANGES64_MOST * WAVE, "the sample's counts lie in the lists");
	for (uint32_t log_ranges = 0; (1u << log_ranges) <= RANGES64_MOST; ++log_ranges) {
		const uint32_t ranges = 1u << log_ranges, most = (k + ranges - 1) >> log_ranges;
		const uint64_t bytes = ((uint64_t)most + 1) * width * 8 + (uint64_t)most * 4 + SUMS64_WAVES * (RANGES64_LIST + RANGES64_ROWS) * 4;
		if (most > 255 || bytes + tables > budget) continue; /* (clusters of eight bits) */
		const uint64_t wanted = (uint64_t)ranges * std::max<uint64_t>(1, n / std::max<uint32_t>(k, 512));
		const uint32_t groups = (uint32_t)std::min<uint64_t>(wanted, compute_units / slices);
		if (groups < ranges) return false;
		*plan = { width, slices, log_ranges, groups, (uint32_t)bytes };
		return true;
	}
	return false;
}

static int launch_ranges64(const float* data, size_t stride, const uint32_t* assignment, float* means, int layout_means, size_t stride_means, uint32_t* sizes,
                           uint32_t dim, uint32_t k, uint32_t n, bool divide, const Ranges64Plan& p, float* partials)
{
	const size_t rows = (size_t)p.groups * ((k + (1u << p.log_ranges) - 1) >> p.log_ranges);
	uint32_t* counts = (uint32_t*)(partials + rows * dim);
	KMX_HIP(hipFuncSetAttribute((const void*)update_ranges64_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds_bytes));
	KMX_LAUNCH_KERNEL(update_ranges64_kernel, dim3(p.groups * p.slices), dim3(SUMS64_THREADS), p.lds_bytes, stream(),
	                  data, stride, assignment, partials, counts, counts + rows, dim, k, n, p.groups, p.log_ranges, p.width);
	KMX_LAUNCH_CHECK("update_ranges64_kernel");
	auto fold = layout_means == KMX_AOS ? fold_ranges64_kernel<KMX_AOS> : fold_ranges64_kernel<KMX_SOA>;
	KMX_LAUNCH_KERNEL(fold, dim3(k), dim3(4 * WAVE), 0, stream(), partials, counts, counts + rows, means, stride_means, sizes, dim, k, p.log_ranges, divide ? 1u : 0u);
	KMX_LAUNCH_CHECK("fold_ranges64_kernel");
	return KMX_OK;
}

template <int LW, bool FULL, typename F>
static int launch_sums64(const F* data, size_t stride, const uint32_t* assignment, F* partial, uint32_t* partial_counts, uint32_t dim, uint32_t k, uint32_t n, const Sums64Plan& p)
{
	auto kernel = update_sums64_kernel<LW, FULL, F>;
	KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)p.lds_bytes));
	KMX_LAUNCH_KERNEL(kernel, dim3((p.chunks + SUMS64_XCDS - 1) / SUMS64_XCDS * SUMS64_XCDS * p.slices), dim3(SUMS64_THREADS), p.lds_bytes, stream(),
	                  data, stride, assignment, partial, partial_counts, dim, k, n, p.chunk_points, p.chunks, p.slices, p.width, p.copies);
	KMX_LAUNCH_CHECK("update_sums64_kernel");
	return KMX_OK;
}

static size_t sums64_words(const Sums64Plan& p, uint32_t dim, uint32_t k, size_t item) { return (size_t)p.chunks * k * dim * (item / sizeof(float)) + (size_t)p.chunks * k; }

/*
 * Where the partial sums of a call lie (null: a kernel without any has to do). A recording keeps the addresses of its moment, and the work space moves when a
 * later call needs more of it: recorded sums lie in the static scratch array, which holds all but those of SoA points with thousands of dimensions. Those of
 * floats take the work space (as the copied rows did), doubles the kernels of f64.hip, which need none.
 */
static bool recorded_sums_fit(size_t words)
{
	const Workspace* fixed = fixed_scratch();
	return fixed && words <= fixed->partials_cap;
}

template <typename F>
static int place_sums(Workspace* ws, size_t words, float** partials)
{
	*partials = nullptr;
	if (launches_recorded()) {
		if (recorded_sums_fit(words)) {
			*partials = fixed_scratch()->partials;
			scratch_recorded();
			return KMX_OK;
		}
		if (sizeof(F) == 8) return KMX_OK;
	}
	const int rc = reserve_partials(ws, words);
	*partials = ws->partials;
	return rc;
}

bool sums64_takes_columns(uint32_t dim, uint32_t k, uint32_t n, const kmx_exec_params* exec, const Workspace* ws, const DeviceInfo& dev)
{
	Sums64Plan p;
	if (n == 0 || ws->fixed || !plan_columns64(dim, k, n, false, lds_budget_of(exec, dev), dev.compute_units, &p)) return false;
	const size_t words = sums64_words(p, dim, k, sizeof(float));
	return !launches_recorded() || recorded_sums_fit(words) || words <= ws->partials_cap;
}

template <typename F>
int launch_update_sums64(const F* data, int layout, size_t stride, const uint32_t* assignment, F* means, int layout_means, size_t stride_means, uint32_t* sizes,
                         uint32_t dim, uint32_t k, uint32_t n, bool divide, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, bool* done)
{
	*done = false;
	Sums64Plan p;
	float* partials = nullptr;
	const bool columns = layout == KMX_SOA;
	if (n == 0 || (columns && ws && ws->fixed)) return KMX_OK; /* (SoA points are taken there whatever their number of partial sums) */
	const uint32_t budget = lds_budget_of(exec, dev);
	bool planned = columns ? plan_columns64(dim, k, n, sizeof(F) == 8, budget, dev.compute_units, &p) : plan_sums64(dim, stride, k, n, sizeof(F) == 8, budget, dev.compute_units, &p);
	/* (the sorted chunks' partial sums may be several times as many, and would not fit the scratch array) */
	if (planned && !columns && sizeof(F) == 4 && !ws->fixed && !launches_recorded()) planned = !sorted_pays(dim, k, n, p.width, p.slices, p.chunks, dev.compute_units);
	if constexpr (sizeof(F) == 4) {
		Ranges64Plan r;
		if (!columns && ranges64_pays(dim, k, n, planned) && plan_ranges64(dim, k, n, budget, dev.compute_units, &r)) {
			const int rc = place_sums<F>(ws, ranges64_words(r, dim, k), &partials);
			if (rc) return rc;
			*done = true;
			exec->block_count = r.groups * r.slices;
			return launch_ranges64(data, stride, assignment, means, layout_means, stride_means, sizes, dim, k, n, divide, r, partials);
		}
	}
	if (!planned) return KMX_OK;
	if (sizing_only() && !columns && sizeof(F) == 4) {
		/* the stride may decide whether rows go as a whole, and the room is for calls with any */
		Sums64Plan spread;
		if (plan_sums64(dim, (size_t)dim + 32, k, n, false, budget, dev.compute_units, &spread)) {
			const int rc = reserve_partials(ws, sums64_words(spread, dim, k, sizeof(F)));
			if (rc) return rc;
		}
	}
	const size_t sums = (size_t)p.chunks * k * dim;
	int rc = place_sums<F>(ws, sums64_words(p, dim, k, sizeof(F)), &partials);
	if (rc || !partials) return rc;
	*done = true;
	exec->block_count = p.chunks * p.slices;
	F* partial = (F*)partials;
	uint32_t* partial_counts = (uint32_t*)(partial + sums);
#define KMX_SUMS64(LW) (dim % p.width == 0 && p.width == LW ? launch_sums64<LW, true, F>(data, stride, assignment, partial, partial_counts, dim, k, n, p) \
	                                                        : launch_sums64<LW, false, F>(data, stride, assignment, partial, partial_counts, dim, k, n, p))
	if (columns) rc = launch_columns64<COLUMNS64, F>(p.width, data, stride, assignment, partial, partial_counts, dim, k, n, p);
	else rc = p.width <= 1 ? launch_sums64<1, true, F>(data, stride, assignment, partial, partial_counts, dim, k, n, p)
	   : p.width <= 2 ? KMX_SUMS64(2) : p.width <= 4 ? KMX_SUMS64(4) : p.width <= 8 ? KMX_SUMS64(8) : p.width <= 16 ? KMX_SUMS64(16)
	   : p.width <= 32 ? KMX_SUMS64(32) : KMX_SUMS64(64);
#undef KMX_SUMS64
	if (rc) return rc;
	return launch_reduce_partials<F>(partial, partial_counts, p.chunks, means, layout_means, stride_means, sizes, dim, k, divide);
}

template int launch_update_sums64<float>(const float*, int, size_t, const uint32_t*, float*, int, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, bool, kmx_exec_params*, Workspace*, const DeviceInfo&, bool*);
template int launch_update_sums64<double>(const double*, int, size_t, const uint32_t*, double*, int, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, bool, kmx_exec_params*, Workspace*, const DeviceInfo&, bool*);

} // namespace kmx
