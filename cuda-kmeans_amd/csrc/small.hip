/*
 * Small inputs, floats and doubles: what a call costs there is launches and latency, not arithmetic. The general paths take five
 * to seven dependent launches (pack, sweep, exact pass, clear, accumulate, fold or divide), each of them a few microseconds of
 * its own; N = 10240, d = 20, k = 128 was 34 us per iteration for 26 M multiply-adds. Two kernels instead:
 *
 *   assign_small_kernel  the serial arithmetic for every pair, nothing to pack, certify or re-evaluate. With `sums` it also adds
 *                        up its points (rows are still in LDS) into per-work-group partial sums for reduce_partials_kernel:
 *                        the single-pass iteration of small inputs.
 *   update_small_kernel  a work-group per range of clusters reads ALL memberships, lists its members, adds their rows and writes
 *                        finished centroids and sizes: no partial sums, nothing cleared before, nothing divided after.
 *
 * Where the general paths take over is measured; see small_assign_accepts (small_plan.h) and small_update_fits.
 */
#include "kmx_internal.h"
#include "small_plan.h"

#include <algorithm>
#include <type_traits>

#pragma clang fp contract(off)

namespace kmx {

template <typename F> struct SmallVec;
template <> struct SmallVec<float> { typedef float type __attribute__((ext_vector_type(4))); };
template <> struct SmallVec<double> { typedef double type __attribute__((ext_vector_type(4))); };

template <typename F> __device__ __forceinline__ F small_sqrt(F v);
template <> __device__ __forceinline__ float small_sqrt<float>(float v) { return __builtin_sqrtf(v); }
template <> __device__ __forceinline__ double small_sqrt<double>(double v) { return __builtin_sqrt(v); }

/* a root and its centroid's number (0xFFFFFFFF: none), ordered as the serial scan decides */
template <typename F> struct SmallKey {
	F root; uint32_t at;
	SmallKey() = default;
	__device__ __forceinline__ SmallKey(F root, uint32_t at) : root(root), at(at) {}
	__device__ __forceinline__ SmallKey of_lane(int off) const { return SmallKey(__shfl_xor(root, off), (uint32_t)__shfl_xor((int)at, off)); }
	__device__ __forceinline__ uint32_t number() const { return at; }
	__device__ __forceinline__ void take(const SmallKey& o)
	{
		const bool pinned = at == 0 && root != root, other_pinned = o.at == 0 && o.root != o.root;
		const bool wins = other_pinned || (!pinned && o.at != 0xFFFFFFFFu && (at == 0xFFFFFFFFu || o.root < root || (o.root == root && o.at < at)));
		root = wins ? o.root : root;
		at = wins ? o.at : at;
	}
};
template <> struct SmallKey<float> { /* roots are not negative: their bits are in their order, NaN behind infinity */
	unsigned long long bits;
	SmallKey() = default;
	__device__ __forceinline__ SmallKey(float root, uint32_t at)
	    : bits(at == 0xFFFFFFFFu ? ~0ull : at == 0 && root != root ? 0ull : (unsigned long long)__float_as_uint(root) << 32 | at) {}
	__device__ __forceinline__ SmallKey of_lane(int off) const { SmallKey o; o.bits = __shfl_xor(bits, off); return o; }
	__device__ __forceinline__ uint32_t number() const { return (uint32_t)bits; }
	__device__ __forceinline__ void take(const SmallKey& o) { bits = o.bits < bits ? o.bits : bits; }
};

/* The serial scan compares correctly rounded square roots. Two sums whose ratio is below this differ in their roots by more
 * than one unit in the last place, so comparing the sums decides; between this and 1 the roots themselves are compared. (Below
 * `tiny` the sums may be subnormal and their ratio means nothing.) */
template <typename F> struct SqrtMargin;
template <> struct SqrtMargin<float> { static constexpr float ratio = 0.9999995f, tiny = 1e-30f; };
template <> struct SqrtMargin<double> { static constexpr double ratio = 1.0 - 1e-15, tiny = 1e-290; };

/*
 * A work-group owns 64 points (or 32, see small_shape), whose rows it stages in LDS next to a chunk of the centroids. A wavefront is 16 x 4 lanes with
 * T points times T centroids each, so it covers 16 T points and 4 T centroids at a time; of 64 points, the eight wavefronts are 4 / T groups of
 * points times 2 T shares of the centroids. Per four dimensions a lane reads 2 T pieces of 16 bytes for its T^2 pairs: with T = 2
 * (192 ALU cycles against 128 of the LDS that four SIMDs share) the vector ALU sets the pace, T = 1 (48 against 64) is for a
 * dozen centroids at most, which would leave most of the larger tile empty. (A lane per point with the centroids broadcast is
 * bound by the LDS; with the centroids as scalar operands every scalar load waits for all earlier ones: N = 2588, d = 60, k = 1288
 * 135 us.) A few dozen centroids leave most of the time to the trips to memory and the barriers in front of that (N = 65536, d = 8, k = 64: 3 us
 * of vector instructions in 11 us): the first four pieces a lane has of points and of centroids are requested together, and no lane asks for more than there
 * is. With one after the other, each in eight loads a lane whatever there was to load, that call was 25.0 instead of 22.0 us; d = 100, k = 40, N = 30000:
 * 17.2 against 15.6; N = 10240, d = 20, k = 128: 19.5 against 18.9. Floats are held to 64 vector registers, so that a compute unit takes four work-groups
 * where their LDS lets it (40 KB each: up to 20 dimensions with a full chunk of centroids, 120 with a dozen; with 76 registers three: N = 50000, d = 2,
 * k = 10 14.0 against 13.4 us, N = 65000, d = 5, k = 50 10.0 against 9.5). The row stride is an odd number of 16-byte pieces: rows read together start in
 * different banks. Every sum runs in ascending dimension, every operation rounded separately.
 *
 * SUMS: the rows, which are still in LDS, added up in doubles where the centroids were, one ds_add_f64 per coordinate (8 cycles of a wavefront; memberships
 * times rows on the fp32 matrix instruction, which keeps the vector ALU, took 2.1 instead of 0.5 us of a work-group: N = 10240, d = 20, k = 128 17.7 -> 16.4 us per
 * iteration, N = 65536, d = 8, k = 64 20.5 -> 18.4, N = 20000, d = 20, k = 100 22.3 -> 19.4).
 */

/*
 * `count` rows of dim elements on their way to LDS rows of row_stride: AoS rows `stride` apart, or columns (row r of column q at src[q * stride + r];
 * a wavefront takes 64 rows of one column at a time). vec4: rows of whole, aligned pieces of four. Rows behind `last` repeat it.
 * magic = ceil(2^32 / dim): i / dim = umulhi(i, magic) for the few ten thousand elements of a work-group.
 */
template <typename F>
struct SmallRows {
	F* to; const F* src; size_t stride;
	uint32_t count, last, dim, row_stride, magic; bool vec4;
};
/* AoS: pieces of four or single coordinates */
template <typename F> __device__ __forceinline__ uint32_t small_items(const SmallRows<F>& s) { return s.vec4 ? s.count * (s.dim / 4) : s.count * s.dim; }

/* AoS: up to B items of every lane, all of them requested before the first is placed. Lanes without an item ask for nothing: a repeated one costs the
 * caches as much as any (N = 65536, d = 8, k = 64: seven of eight were). For the first items only: with any number of them in such batches and their
 * branches N = 94 doubles, d = 186, k = 3 took 9.3 us, with stage_items 7.9; N = 675 doubles, d = 195, k = 108: 58.6, 53.8. */
template <typename F, int B, uint32_t THREADS>
struct SmallBatch {
	typedef typename SmallVec<F>::type F4;
	F4 v[B];
	uint32_t at[B];
	static __device__ __forceinline__ bool holds(const SmallRows<F>& s) { return small_items(s) <= B * THREADS; }
	__device__ __forceinline__ void request(const SmallRows<F>& s)
	{
		const uint32_t items = small_items(s);
#pragma unroll
		for (int u = 0; u < B; ++u) {
			const uint32_t i = u * THREADS + threadIdx.x;
			if (i >= items) continue;
			const uint32_t e = s.vec4 ? i * 4 : i, r = s.dim == 1 ? e : __umulhi(e, s.magic), q = e - r * s.dim;
			const F* from = s.src + (size_t)min(r, s.last) * s.stride + q;
			at[u] = r * s.row_stride + q;
			if (s.vec4) v[u] = *(const F4*)from;
			else v[u].x = *from;
		}
	}
	__device__ __forceinline__ void place(const SmallRows<F>& s) const
	{
		const uint32_t items = small_items(s);
#pragma unroll
		for (int u = 0; u < B; ++u) {
			if (u * THREADS + threadIdx.x >= items) continue;
			if (s.vec4) *(F4*)(s.to + at[u]) = v[u];
			else s.to[at[u]] = v[u].x;
		}
	}
};

/*
 * AoS: the items from the one of that number per lane on, any number of them. A lane's pieces of four: four at a time, none beyond the last (the second and
 * later chunks of centroids have a piece or two for a lane: N = 8000 doubles, d = 48, k = 300 42.8 us, with repeated ones 44.7). Single coordinates: six at a
 * time, which is what 64 registers hold, the last one again behind the end: no branches between the loads.
 */
template <typename F, bool VEC, uint32_t THREADS>
__device__ __forceinline__ void stage_items(const SmallRows<F>& s, uint32_t from)
{
	typedef typename std::conditional<VEC, typename SmallVec<F>::type, F>::type V;
	constexpr int BATCH = VEC ? 4 : 6;
	const uint32_t last = small_items(s) - 1, one = s.dim == 1 ? 1u : 0u; /* (magic is 0 for rows of one) */
	for (uint32_t i0 = from * THREADS + threadIdx.x; i0 <= last; i0 += THREADS * BATCH) {
		V v[BATCH];
		uint32_t at[BATCH];
#pragma unroll
		for (int u = 0; u < BATCH; ++u) {
			const uint32_t i = i0 + u * THREADS;
			if (VEC && i > last) continue;
			const uint32_t e = min(i, last) * (VEC ? 4 : 1), r = __umulhi(e, s.magic) + e * one, q = e - r * s.dim;
			at[u] = r * s.row_stride + q;
			v[u] = *(const V*)(s.src + (size_t)min(r, s.last) * s.stride + q);
		}
#pragma unroll
		for (int u = 0; u < BATCH; ++u)
			if (!VEC || i0 + u * THREADS <= last) *(V*)(s.to + at[u]) = v[u];
	}
}

/*
 * Columns: a wavefront takes 64 rows of one at a time. Wide rows: eight columns under way, the last one again behind the end. Rows of fewer than two columns per
 * wavefront: blocks of 64 rows follow one another without a pause, and wavefronts beyond the columns take blocks of their own (the first way and this,
 * us: N = 21376, d = 2, k = 287 18.7, 17.6; N = 2550, d = 8, k = 284 15.0, 13.6; N = 43539, d = 9, k = 111 14.5, 13.6; but N = 53567, d = 42, k = 32 12.4, 13.3;
 * N = 3895, d = 252, k = 2 10.0, and 15.7 in batches of four).
 */
template <typename F, uint32_t WAVES>
__device__ __forceinline__ void stage_columns(const SmallRows<F>& s)
{
	constexpr uint32_t BATCH = 8;
	const uint32_t lane = threadIdx.x % WAVE, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x / WAVE));
	if (s.dim >= 2 * WAVES) {
		for (uint32_t r0 = 0; r0 < s.count; r0 += WAVE) {
			const uint32_t r = min(r0 + lane, s.count - 1);
			const F* src = s.src + min(r, s.last);
			for (uint32_t q0 = wave; q0 < s.dim; q0 += WAVES * BATCH) {
				F v[BATCH];
#pragma unroll
				for (uint32_t u = 0; u < BATCH; ++u) v[u] = src[(size_t)min(q0 + u * WAVES, s.dim - 1) * s.stride];
#pragma unroll
				for (uint32_t u = 0; u < BATCH; ++u) s.to[r * s.row_stride + min(q0 + u * WAVES, s.dim - 1)] = v[u];
			}
		}
		return;
	}
	/* groups of wavefronts, each with all columns of its blocks (one group where the columns are as many as wavefronts) */
	const bool few = s.dim < WAVES;
	const uint32_t group = !few ? 0 : s.dim == 1 ? wave : __umulhi(wave, s.magic), groups = !few ? 1 : s.dim == 1 ? WAVES : __umulhi(WAVES, s.magic);
	const uint32_t first = wave - group * s.dim;
	uint32_t q = first, r0 = group < groups ? group * WAVE : s.count;
	while (r0 < s.count) {
		F v[BATCH];
		uint32_t at[BATCH], got = 0;
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u) {
			if (r0 >= s.count) continue;
			const uint32_t r = min(r0 + lane, s.count - 1);
			at[u] = r * s.row_stride + q;
			v[u] = s.src[(size_t)q * s.stride + min(r, s.last)];
			got = u + 1;
			q += WAVES;
			const bool wrap = q >= s.dim;
			q = wrap ? first : q;
			r0 += wrap ? groups * WAVE : 0u;
		}
#pragma unroll
		for (uint32_t u = 0; u < BATCH; ++u)
			if (u < got) s.to[at[u]] = v[u];
	}
}

template <typename F, int L, uint32_t THREADS>
__device__ __forceinline__ void stage_rows(const SmallRows<F>& s, uint32_t from)
{
	if (L == KMX_SOA) stage_columns<F, THREADS / WAVE>(s);
	else if (s.vec4) stage_items<F, true, THREADS>(s, from);
	else stage_items<F, false, THREADS>(s, from);
}

template <typename F, int T, int POINTS, uint32_t THREADS, int LD, int LM, bool SUMS>
__global__ void __launch_bounds__(THREADS) __attribute__((amdgpu_waves_per_eu(sizeof(F) == 4 && THREADS == 512 ? 8 : 4)))
assign_small_kernel(const F* __restrict__ data, size_t stride, const F* __restrict__ means, size_t stride_means,
                    uint32_t* __restrict__ assignment, uint32_t dim, uint32_t k, uint32_t n, uint32_t row_stride, uint32_t chunk,
                    uint32_t magic, uint32_t vec4, uint32_t* __restrict__ counters, F* __restrict__ partial, uint32_t* __restrict__ partial_counts,
                    uint32_t sums_width, uint32_t magic_width)
{
	typedef typename SmallVec<F>::type F4;
	constexpr uint32_t PG = POINTS / 16 / T, CW = small_shares(T, POINTS, THREADS); /* groups of points, shares of the centroids */
	extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
	F* rows = (F*)lds_raw;
	F* cents = rows + (size_t)POINTS * row_stride; /* chunk rows; with SUMS later k * sums_width doubles and k counts */
	__shared__ SmallKey<F> cand[CW][POINTS];
	__shared__ __attribute__((aligned(16))) uint32_t member[POINTS];
	static_assert(sizeof(cand) + sizeof(member) == small_static_bytes(sizeof(F), T, POINTS, THREADS), "the plan's static arrays");
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t pg = wave % PG, cw = wave / PG;
	const uint32_t lp = lane & 15, lc = lane >> 4; /* points lp + 16 p of the group, centroids T lc + u of the wavefront's 4 T */
	const uint32_t first = blockIdx.x * POINTS;
	const uint32_t here = min((uint32_t)POINTS, n - first);
	if (blockIdx.x == 0 && tid == 0) counters[0] = 0u; /* nothing is left to an exact pass */

	auto centroids = [&](uint32_t base) -> SmallRows<F> {
		const uint32_t count = min(chunk, k - base);
		return SmallRows<F>{ cents, LM == KMX_AOS ? means + (size_t)base * stride_means : means + base, stride_means, count, count - 1, dim, row_stride, magic, (vec4 & 2u) != 0 };
	};
	{
		const SmallRows<F> points = { rows, LD == KMX_AOS ? data + (size_t)first * stride : data + first, stride, POINTS, here - 1, dim, row_stride, magic, (vec4 & 1u) != 0 };
		const SmallRows<F> start = centroids(0);
		uint32_t staged = 0; /* items of a lane */
		bool rest = true;
		if constexpr (LD == KMX_AOS && LM == KMX_AOS) {
			/* points and centroids travel together where all of them do, or where both are whole pieces: one trip to memory instead of two */
			typedef SmallBatch<F, 4, THREADS> Batch;
			rest = !(Batch::holds(points) && Batch::holds(start));
			if (!rest || (points.vec4 && start.vec4)) {
				Batch some, others;
				some.request(points);
				others.request(start);
				some.place(points);
				others.place(start);
				staged = 4;
			}
		}
		if (rest) {
			stage_rows<F, LD, THREADS>(points, staged);
			stage_rows<F, LM, THREADS>(start, staged);
		}
	}

	F low[T];
	uint32_t at[T];
#pragma unroll
	for (int p = 0; p < T; ++p) { low[p] = (F)__builtin_inff(); at[p] = 0xFFFFFFFFu; }
	const F* mine = rows + (pg * (16 * T) + lp) * row_stride;
	for (uint32_t base = 0; base < k; base += chunk) {
		const uint32_t count = min(chunk, k - base);
		if (base) {
			__syncthreads(); /* the previous chunk is no longer needed */
			stage_rows<F, LM, THREADS>(centroids(base), 0);
		}
		__syncthreads();
		for (uint32_t c0 = cw * (4 * T); c0 < count; c0 += CW * (4 * T)) {
			F sum[T][T];
			uint32_t centre[T];
#pragma unroll
			for (int u = 0; u < T; ++u) {
				centre[u] = min(c0 + T * lc + u, count - 1) * row_stride; /* beyond the last centroid: the last one again */
#pragma unroll
				for (int p = 0; p < T; ++p) sum[u][p] = (F)0;
			}
			auto add = [&](uint32_t q, auto width) {
				constexpr int W = decltype(width)::value;
				F x[T][W], cv[T][W];
				auto fetch = [&](F (&to)[W], const F* from) {
					if constexpr (W == 4) {
						const F4 v = *(const F4*)from;
						to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
					}
					else to[0] = from[0];
				};
#pragma unroll
				for (int p = 0; p < T; ++p) fetch(x[p], mine + p * (16 * row_stride) + q);
#pragma unroll
				for (int u = 0; u < T; ++u) fetch(cv[u], cents + centre[u] + q);
#pragma unroll
				for (int e = 0; e < W; ++e)
#pragma unroll
					for (int u = 0; u < T; ++u)
#pragma unroll
						for (int p = 0; p < T; ++p) {
							const F diff = x[p][e] - cv[u][e];
							const F sq = diff * diff;
							sum[u][p] = sum[u][p] + sq;
						}
			};
			uint32_t q = 0;
#pragma unroll 4
			for (; q + 4 <= dim; q += 4) add(q, std::integral_constant<int, 4>());
			for (; q < dim; ++q) add(q, std::integral_constant<int, 1>());
#pragma unroll
			for (int u = 0; u < T; ++u) {
				const uint32_t c = base + min(c0 + T * lc + u, count - 1);
#pragma unroll
				for (int p = 0; p < T; ++p) {
					const F s = sum[u][p];
					const bool start = c == 0; /* where the serial scan starts: a NaN stays */
					bool less = s < low[p];
					const bool close = less && !(s < low[p] * SqrtMargin<F>::ratio && low[p] > SqrtMargin<F>::tiny);
					if (__builtin_amdgcn_ballot_w64(close)) less = close ? small_sqrt(s) < small_sqrt(low[p]) : less;
					less = less || start;
					low[p] = less ? s : low[p];
					at[p] = less ? c : at[p];
				}
			}
		}
	}
	/* the four lanes of a point, then the wavefronts: the smaller root, then the smaller number; centroid 0 keeps a NaN root against everything, any other loses
	 * with one. Floats: as one comparison of 64 bits (N = 10240, d = 20, k = 128 15.2 -> 14.6 us per iteration, N = 65536, d = 8, k = 64 18.4 -> 17.7). */
	typedef SmallKey<F> Key;
#pragma unroll
	for (int p = 0; p < T; ++p) {
		Key key(small_sqrt(low[p]), at[p]);
#pragma unroll
		for (int off = 16; off < WAVE; off <<= 1) key.take(key.of_lane(off));
		if (lc == 0) cand[cw][pg * (16 * T) + lp + 16 * p] = key;
	}
	__syncthreads();
	double* sums = (double*)cents; /* SUMS: k * sums_width of them, then k counts; the centroids are no longer needed */
	uint32_t* counts = (uint32_t*)(sums + k * sums_width);
	if constexpr (SUMS) {
		for (uint32_t i = tid; i < k * sums_width; i += THREADS) sums[i] = 0.0;
		for (uint32_t i = tid; i < k; i += THREADS) counts[i] = 0u;
	}
	if (tid < POINTS) {
		Key best = cand[0][tid];
#pragma unroll
		for (uint32_t w = 1; w < CW; ++w) best.take(cand[w][tid]);
		const uint32_t idx = best.number();
		if (tid < here) assignment[first + tid] = idx;
		if (SUMS) member[tid] = tid < here ? idx : 0xFFFFFFFFu;
	}

	if constexpr (SUMS) {
		F* out = partial + (size_t)blockIdx.x * k * dim;
		if (sums_width == dim) {
			__syncthreads();
			for (uint32_t e = tid; e < here * dim; e += THREADS) {
				const uint32_t p = dim == 1 ? e : __umulhi(e, magic), q = e - p * dim;
				unsafeAtomicAdd(&sums[member[p] * dim + q], (double)rows[p * row_stride + q]);
			}
			if (tid < here) atomicAdd(&counts[member[tid]], 1u);
			__syncthreads();
			for (uint32_t e = tid; e < k * dim; e += THREADS) out[e] = (F)sums[e];
		}
		else { /* parts of two coordinates and more, the last one may be narrower (small_shape) */
			for (uint32_t from = 0; from < dim; from += sums_width) {
				__syncthreads();
				for (uint32_t e = tid; e < here * sums_width; e += THREADS) {
					const uint32_t p = __umulhi(e, magic_width), q = e - p * sums_width;
					if (from + q < dim) unsafeAtomicAdd(&sums[member[p] * sums_width + q], (double)rows[p * row_stride + from + q]);
				}
				if (from == 0 && tid < here) atomicAdd(&counts[member[tid]], 1u);
				__syncthreads();
				for (uint32_t e = tid; e < k * sums_width; e += THREADS) {
					const uint32_t c = __umulhi(e, magic_width), q = e - c * sums_width;
					if (from + q < dim) out[c * dim + from + q] = (F)sums[e];
					sums[e] = 0.0;
				}
			}
		}
		for (uint32_t i = tid; i < k; i += THREADS) partial_counts[(size_t)blockIdx.x * k + i] = counts[i];
	}
}

/*
 * blockIdx.x owns the clusters [per * blockIdx.x, + per). Its 1024 lanes read all n memberships (ITEMS 16-byte pieces each, one
 * round trip to the caches); every wavefront lists the points of its share that belong to these clusters in a region of LDS of
 * its own (ballots, no atomics), the lists are joined, sorted by cluster where there are several, and the listed rows are added:
 * groups of gw lanes (a lane: VEC consecutive coordinates) take equal shares of the list, 8 rows in flight, and add what they
 * have of a cluster to its sums in LDS when the cluster changes. Rows wider than a group go by in slices.
 * One hot cluster holding everything is bound by what one compute unit reads (about 0.1 TB/s), which small_update_fits bounds.
 */
constexpr uint32_t UPDATE_SMALL_THREADS = 1024;
constexpr uint32_t UPDATE_SMALL_WAVES = UPDATE_SMALL_THREADS / WAVE;
constexpr uint32_t UPDATE_SMALL_MAX_PER = 64;

template <typename F, int ITEMS, int VEC, int LD, int LM>
__global__ void __launch_bounds__(UPDATE_SMALL_THREADS)
update_small_kernel(const F* __restrict__ data, size_t stride, const uint32_t* __restrict__ assignment, F* __restrict__ means, size_t stride_means,
                    uint32_t* __restrict__ sizes, uint32_t dim, uint32_t k, uint32_t n, uint32_t per, uint32_t gw, uint32_t divide, uint32_t vec4)
{
	typedef uint32_t u4 __attribute__((ext_vector_type(4)));
	extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
	F* acc = (F*)lds_raw;                                                     /* per x dim sums */
	constexpr uint32_t REGION = WAVE * 4 * ITEMS;                             /* points a wavefront looks at */
	unsigned short* found = (unsigned short*)(acc + (size_t)per * dim);       /* UPDATE_SMALL_WAVES regions */
	unsigned short* list = found + UPDATE_SMALL_WAVES * REGION;               /* all of them, sorted by cluster */
	__shared__ uint32_t count[UPDATE_SMALL_MAX_PER], cursor[UPDATE_SMALL_MAX_PER], begin[UPDATE_SMALL_MAX_PER + 1];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE;
	const uint32_t c0 = blockIdx.x * per, mine = min(per, k - c0);

	u4 a[ITEMS];
#pragma unroll
	for (int i = 0; i < ITEMS; ++i) {
		const uint32_t p = (i * UPDATE_SMALL_THREADS + tid) * 4;
		a[i] = u4{ 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFFFFFFu };
		if (vec4 && p + 4 <= n) a[i] = *(const u4*)(assignment + p);
		else {
#pragma unroll
			for (int e = 0; e < 4; ++e)
				if (p + e < n) a[i][e] = assignment[p + e];
		}
	}
	if (tid < per) count[tid] = 0u;
	for (uint32_t i = tid; i < per * dim; i += UPDATE_SMALL_THREADS) acc[i] = (F)0;
	uint32_t have = 0; /* wave-uniform */
	unsigned short* region = found + wave * REGION;
#pragma unroll
	for (int i = 0; i < ITEMS; ++i)
#pragma unroll
		for (int e = 0; e < 4; ++e) {
			const bool match = a[i][e] - c0 < mine; /* (a membership beyond k belongs to nobody) */
			const unsigned long long mask = __builtin_amdgcn_ballot_w64(match);
			if (mask == 0) continue;
			if (match) region[have + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] = (unsigned short)((i * UPDATE_SMALL_THREADS + tid) * 4 + e);
			have += (uint32_t)__popcll(mask);
		}
	__syncthreads();
	for (uint32_t i = lane; i < have; i += WAVE) atomicAdd(&count[mine > 1 ? assignment[region[i]] - c0 : 0u], 1u);
	__syncthreads();
	if (tid < WAVE) {
		const uint32_t v = tid < mine ? count[tid] : 0u;
		uint32_t incl = v;
		for (int off = 1; off < WAVE; off <<= 1) {
			const uint32_t up = (uint32_t)__shfl_up((int)incl, off);
			if (tid >= (uint32_t)off) incl += up;
		}
		if (tid < mine) { begin[tid] = incl - v; cursor[tid] = incl - v; }
		if (tid == mine - 1) begin[mine] = incl;
	}
	__syncthreads();
	for (uint32_t i = lane; i < have; i += WAVE) list[atomicAdd(&cursor[mine > 1 ? assignment[region[i]] - c0 : 0u], 1u)] = region[i];
	__syncthreads();

	const uint32_t groups = UPDATE_SMALL_THREADS / gw, group = tid / gw, gl = tid % gw;
	const uint32_t entries = begin[mine];
	const uint32_t e_begin = (uint32_t)((uint64_t)group * entries / groups), e_end = (uint32_t)((uint64_t)(group + 1) * entries / groups);
	for (uint32_t slice = 0; slice < dim; slice += gw * VEC) {
		const uint32_t d0 = slice + gl * VEC;
		const bool on = d0 < dim;
		/* (the last piece of a row that is no multiple of VEC starts early enough to end with the row; its first coordinates are the previous lane's) */
		const uint32_t d = on ? (VEC > 1 ? min(d0, dim - VEC) : d0) : 0u;
		if (!on || e_begin == e_end) continue;
		F s[VEC];
#pragma unroll
		for (int v = 0; v < VEC; ++v) s[v] = (F)0;
		uint32_t cl = 0;
		while (begin[cl + 1] <= e_begin) ++cl;
		auto flush = [&]() {
#pragma unroll
			for (int v = 0; v < VEC; ++v) {
				if (VEC == 1 || d + v >= d0) unsafeAtomicAdd(&acc[cl * dim + d + v], s[v]);
				s[v] = (F)0;
			}
		};
		constexpr int AHEAD = 8;
		for (uint32_t e = e_begin; e < e_end; e += AHEAD) {
			F x[AHEAD][VEC];
#pragma unroll
			for (int u = 0; u < AHEAD; ++u) {
				const uint32_t p = list[min(e + u, e_end - 1)];
#pragma unroll
				for (int v = 0; v < VEC; ++v) x[u][v] = data[elem<LD>(stride, p, d + v)];
			}
#pragma unroll
			for (int u = 0; u < AHEAD; ++u) {
				if (e + u < e_end) {
					while (begin[cl + 1] <= e + u) { flush(); ++cl; }
#pragma unroll
					for (int v = 0; v < VEC; ++v) s[v] += x[u][v];
				}
			}
		}
		flush();
	}
	__syncthreads();
	for (uint32_t i = tid; i < mine * dim; i += UPDATE_SMALL_THREADS) {
		const uint32_t cl = i / dim, d = i - cl * dim;
		const uint32_t members = count[cl];
		const F s = acc[i];
		means[elem<LM>(stride_means, c0 + cl, d)] = !divide ? s : (members ? s / (F)members : (F)0);
	}
	if (tid < mine) sizes[c0 + tid] = count[tid];
}

template <typename F>
bool small_assign_fits(int layout, uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget) { return small_assign_accepts(sizeof(F), layout == KMX_SOA, dim, k, n, lds_budget); }

template <typename F, bool SUMS>
static int launch_assign_small_t(const F* data, int layout, size_t stride, const F* means, int layout_means, size_t stride_means, uint32_t* assignment,
                                 uint32_t dim, uint32_t k, uint32_t n, uint32_t* counters, F* partial, uint32_t* partial_counts, uint32_t* blocks, uint32_t lds_budget)
{
	const SmallShape shape = small_shape(sizeof(F), dim, k, n, SUMS, lds_budget);
	*blocks = (n + shape.points - 1) / shape.points;
	const uint32_t align = 4 * sizeof(F) - 1;
	const uint32_t vec4 = (dim % 4 == 0 && stride % 4 == 0 && ((uintptr_t)data & align) == 0 ? 1u : 0u) | (dim % 4 == 0 && stride_means % 4 == 0 && ((uintptr_t)means & align) == 0 ? 2u : 0u);
	void (*kernel)(const F*, size_t, const F*, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t*, F*, uint32_t*, uint32_t, uint32_t) = nullptr;
#define KMX_PICK(P, Q, W) (layout == KMX_AOS ? (layout_means == KMX_AOS ? assign_small_kernel<F, P, Q, W, KMX_AOS, KMX_AOS, SUMS> : assign_small_kernel<F, P, Q, W, KMX_AOS, KMX_SOA, SUMS>) \
                                       : (layout_means == KMX_AOS ? assign_small_kernel<F, P, Q, W, KMX_SOA, KMX_AOS, SUMS> : assign_small_kernel<F, P, Q, W, KMX_SOA, KMX_SOA, SUMS>))
	const bool few = shape.tile == 1;
	kernel = shape.points == 32 ? (few ? KMX_PICK(1, 32, 512) : KMX_PICK(2, 32, 512)) : shape.threads == 1024 ? (few ? KMX_PICK(1, 64, 1024) : KMX_PICK(2, 64, 1024)) : few ? KMX_PICK(1, 64, 512) : KMX_PICK(2, 64, 512);
#undef KMX_PICK
	if (shape.lds_bytes > 48 * 1024) KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shape.lds_bytes));
	KMX_LAUNCH_KERNEL(kernel, dim3(*blocks), dim3(shape.threads), shape.lds_bytes, stream(), data, stride, means, stride_means, assignment, dim, k, n,
	                   small_row_stride(dim), assign_small_chunk(sizeof(F), dim, k), (uint32_t)((0x100000000ull + dim - 1) / dim), vec4, counters, partial, partial_counts,
	                   shape.sums_width, shape.sums_width ? (uint32_t)((0x100000000ull + shape.sums_width - 1) / shape.sums_width) : 0u);
	KMX_LAUNCH_CHECK("assign_small_kernel");
	return KMX_OK;
}

template <typename F>
int launch_assign_small(const F* data, int layout, size_t stride, const F* means, int layout_means, size_t stride_means, uint32_t* assignment,
                        uint32_t dim, uint32_t k, uint32_t n, uint32_t* counters, uint32_t* blocks, uint32_t lds_budget)
{
	return launch_assign_small_t<F, false>(data, layout, stride, means, layout_means, stride_means, assignment, dim, k, n, counters, nullptr, nullptr, blocks, lds_budget);
}

/* the single-pass iteration of small inputs: partial sums and counts of *blocks work-groups, at most assign_small_max_blocks(n), for launch_reduce_partials */
int launch_assign_small_sums(const AssignArgs& a, float* partial, uint32_t* partial_counts, uint32_t* blocks, uint32_t* counters, uint32_t lds_budget)
{
	return launch_assign_small_t<float, true>(a.data, a.layout, a.stride, a.means, a.layout_means, a.stride_means, a.assignment, a.dim, a.k, a.n,
	                                          counters, partial, partial_counts, blocks, lds_budget);
}
bool small_iteration_fits(int layout, uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget) { return small_iteration_accepts(layout == KMX_SOA, dim, k, n, lds_budget); }

/*
 * The members of a cluster come from one compute unit, so the largest cluster sets the time: everything in one cluster is
 * n * dim * sizeof(F) bytes at about 0.1 TB/s. 2 MB keeps that worst case near 20 us, what the general path takes anyway.
 */
constexpr uint32_t SMALL_UPDATE_POINTS = 1u << 15;
constexpr uint64_t SMALL_UPDATE_BYTES = 2u << 20;

static uint32_t update_small_per(uint32_t k, const DeviceInfo& dev) { return (k + dev.compute_units - 1) / dev.compute_units; }
static uint32_t update_small_items(uint32_t n)
{
	const uint32_t items = (n + 4 * UPDATE_SMALL_THREADS - 1) / (4 * UPDATE_SMALL_THREADS);
	return items <= 1 ? 1 : items <= 3 ? 3 : 8;
}
template <typename F> static uint64_t update_small_lds(uint32_t dim, uint32_t k, uint32_t n, const DeviceInfo& dev)
{
	return (uint64_t)update_small_per(k, dev) * dim * sizeof(F) + (uint64_t)update_small_items(n) * UPDATE_SMALL_THREADS * 4 * 2 * 2;
}

template <typename F>
bool small_update_fits(uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget, const DeviceInfo& dev)
{
	return n > 0 && n <= SMALL_UPDATE_POINTS && (uint64_t)n * dim * sizeof(F) <= SMALL_UPDATE_BYTES && update_small_per(k, dev) <= UPDATE_SMALL_MAX_PER &&
	       update_small_lds<F>(dim, k, n, dev) + 1024 <= lds_budget;
}

template <typename F>
int launch_update_small(const F* data, int layout, size_t stride, const uint32_t* assignment, F* means, int layout_means, size_t stride_means, uint32_t* sizes,
                        uint32_t dim, uint32_t k, uint32_t n, bool divide, uint32_t* blocks, const DeviceInfo& dev)
{
	const uint32_t per = update_small_per(k, dev);
	*blocks = (k + per - 1) / per;
	const uint32_t lds = (uint32_t)update_small_lds<F>(dim, k, n, dev);
	constexpr int VEC = sizeof(F) == 4 ? 4 : 2;
	const bool vec = layout == KMX_AOS && dim >= (uint32_t)VEC;
	uint32_t gw = 1;
	while (gw < 64 && gw * (vec ? VEC : 1) < dim) gw <<= 1;
	const uint32_t items = update_small_items(n);
	void (*kernel)(const F*, size_t, const uint32_t*, F*, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) = nullptr;
#define KMX_PICK_LM(I, V, L) (layout_means == KMX_AOS ? update_small_kernel<F, I, V, L, KMX_AOS> : update_small_kernel<F, I, V, L, KMX_SOA>)
#define KMX_PICK(I) (layout == KMX_SOA ? KMX_PICK_LM(I, 1, KMX_SOA) : vec ? KMX_PICK_LM(I, VEC, KMX_AOS) : KMX_PICK_LM(I, 1, KMX_AOS))
	kernel = items == 1 ? KMX_PICK(1) : items == 3 ? KMX_PICK(3) : KMX_PICK(8);
#undef KMX_PICK
#undef KMX_PICK_LM
	if (lds > 48 * 1024) KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
	KMX_LAUNCH_KERNEL(kernel, dim3(*blocks), dim3(UPDATE_SMALL_THREADS), lds, stream(), data, stride, assignment, means, stride_means, sizes, dim, k, n, per, gw,
	                   divide ? 1u : 0u, ((uintptr_t)assignment & 15) == 0 ? 1u : 0u);
	KMX_LAUNCH_CHECK("update_small_kernel");
	return KMX_OK;
}

#define KMX_SMALL_INSTANCES(F)                                                                                                                                   \
	template bool small_assign_fits<F>(int, uint32_t, uint32_t, uint32_t, uint32_t);                                                                             \
	template bool small_update_fits<F>(uint32_t, uint32_t, uint32_t, uint32_t, const DeviceInfo&);                                                               \
	template int launch_assign_small<F>(const F*, int, size_t, const F*, int, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, uint32_t*, uint32_t*, uint32_t); \
	template int launch_update_small<F>(const F*, int, size_t, const uint32_t*, F*, int, size_t, uint32_t*, uint32_t, uint32_t, uint32_t, bool, uint32_t*, const DeviceInfo&);
KMX_SMALL_INSTANCES(float)
KMX_SMALL_INSTANCES(double)

} // namespace kmx
