/*
 * The exact pass behind the half-precision sweep (rank16_impl.h): the serial result for the points it listed. Device code,
 * instantiated per row width (rank16_inst.hip).
 */
#ifndef KMX_RANK16_EXACT_IMPL_H
#define KMX_RANK16_EXACT_IMPL_H

#include "rank16_impl.h"

namespace kmx {

constexpr uint32_t EXACT_THREADS = 512;
constexpr uint32_t EXACT_WAVES = EXACT_THREADS / WAVE;
constexpr uint32_t EXACT_GROUPS = 4;                       /* most groups of 32 points per unit */
constexpr uint32_t EXACT_ROWS = EXACT_GROUPS * TILE;
constexpr uint32_t EXACT_HITS = 256;                       /* pairs per wavefront and unit that wait for the common evaluation */
constexpr uint32_t EXACT_SQUARES_BYTES = EXACT_WAVES * WAVE * (KBLOCK + 4) * 4; /* (doubles: half as many pairs) */
constexpr uint32_t exact_static_bytes(bool doubles)
{
	return (7 * EXACT_ROWS + EXACT_WAVES * EXACT_HITS + EXACT_WAVES) * 4 + 96 + (doubles ? EXACT_WAVES * EXACT_HITS * 8 + EXACT_ROWS * 4 : 0);
}

template <typename F>
struct ExactArgs {
	/* coordinate d of point p: data[p * stride + d * step]; step 1: rows of row_dim coordinates (zeros behind the first dim). Other
	 * steps (SoA points) are for KB <= 1 only. */
	const float* data; size_t stride, step; uint32_t row_dim;
	/* the same of the points the serial arithmetic is for (doubles: data is their float copy) */
	const F* points; size_t points_stride, points_step; uint32_t points_dim;
	const F* means;                         /* rows of KB * 16 values, zeros behind the coordinates */
	const f16x8* packed; const float* norms; const float* frame; const float* scale;
	uint32_t* assignment; const uint32_t* list; const uint32_t* length; uint32_t* undecided;
	uint32_t dim, k, kp;
	float kd_split;
	uint32_t blocks, most_groups; /* KB = 0: blocks of 16 dimensions per row; groups whose operands fit LDS */
};

/* four coordinates of a row at its coordinate d, as they come from memory: d brought inside the row (row_dim >= 4), or, strided, zeros beyond it */
template <typename F>
__device__ __forceinline__ void exact_request(F __attribute__((ext_vector_type(4)))& v, const F* src, uint32_t d, uint32_t dim, uint32_t row_dim, size_t step, bool strided)
{
	typedef F F4_any __attribute__((ext_vector_type(4), aligned(sizeof(F))));
	if (strided) {
#pragma unroll
		for (uint32_t e = 0; e < 4; ++e) v[e] = d + e < dim ? src[(size_t)(d + e) * step] : (F)0;
	}
	else v = *(const F4_any*)(src + min(d, row_dim - 4));
}

/* ... and in their places, zeros beyond the row (masks: the compiler makes branches of selections) */
template <typename F>
__device__ __forceinline__ void exact_place(F __attribute__((ext_vector_type(4)))& v, uint32_t d, uint32_t row_dim)
{
	typedef typename std::conditional<sizeof(F) == 8, unsigned long long, uint32_t>::type bits_t;
	const uint32_t shift = d + 4 > row_dim ? d + 4 - row_dim : 0;
	const bits_t m0 = (bits_t)0 - (bits_t)(shift == 0), m1 = (bits_t)0 - (bits_t)(shift == 1), m2 = (bits_t)0 - (bits_t)(shift == 2), m3 = (bits_t)0 - (bits_t)(shift == 3);
	const bits_t x = __builtin_bit_cast(bits_t, (F)v.x), y = __builtin_bit_cast(bits_t, (F)v.y), z = __builtin_bit_cast(bits_t, (F)v.z), t = __builtin_bit_cast(bits_t, (F)v.w);
	v.x = __builtin_bit_cast(F, (x & m0) | (y & m1) | (z & m2) | (t & m3));
	v.y = __builtin_bit_cast(F, (y & m0) | (z & m1) | (t & m2));
	v.z = __builtin_bit_cast(F, (z & m0) | (t & m1));
	v.w = __builtin_bit_cast(F, t & m0);
}

/* the value of lane Q (0..3) of this lane's four */
template <int Q> __device__ __forceinline__ float lane_of_four(float v)
{
	return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), Q * 0x55, 0xF, 0xF, true)); /* quad_perm [Q Q Q Q] */
}
template <int Q> __device__ __forceinline__ double lane_of_four(double v)
{
	const unsigned long long bits = __builtin_bit_cast(unsigned long long, v);
	const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)bits, Q * 0x55, 0xF, 0xF, true);
	const uint32_t up = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(bits >> 32), Q * 0x55, 0xF, 0xF, true);
	return __builtin_bit_cast(double, (unsigned long long)up << 32 | lo);
}

/* doubles: the bits of a serial distance as they are compared, like exact_key without the centroid */
__device__ __forceinline__ unsigned long long exact_bits(double sum, uint32_t c)
{
	const double dist = __builtin_sqrt(sum);
	return (c == 0 && dist != dist) ? 0ull : (unsigned long long)__double_as_longlong(dist);
}

__device__ __forceinline__ unsigned long long exact_key(float sum, uint32_t c)
{
	const float dist = __builtin_sqrtf(sum);
	return (c == 0 && dist != dist) ? 0ull : (((unsigned long long)__float_as_uint(dist) << 32) | c); /* see evaluate_pair */
}

/*
 * KB: blocks of 16 dimensions per row, 0: any number (their operands do not stay in registers, the accumulators of the groups do).
 * A unit is 32, 64 or 128 listed points of a work-group of eight wavefronts: as many as leave every work-group something to do, since
 * all of a unit's points share one reading of the centroids' operands (512 KB at k = 1024, d = 256).
 *   1. The rows, moved, scaled and rounded as in the sweep, go to LDS as operands of the ranking.
 *   2. The wavefronts share out the centroid tiles: operands from the caches to registers, then one chain of matrix instructions per
 *      group of points. A centroid at or below the point's threshold is noted in the wavefront's list; NaN passes.
 *   3. The lists are evaluated together, up to 64 pairs per wavefront: for a block of 16 dimensions four lanes per pair fetch 16
 *      bytes each of point and centroid and square the differences (64 consecutive bytes per row: a lane of its own per row would
 *      touch 64 lines per load), the squares go through LDS to the pair's lane, which adds them in order. The results merge into
 *      the point's two smallest keys (distance bits << 32 | centroid, see evaluate_pair) in LDS.
 * F: the type of the serial arithmetic; doubles are ranked by float copies.
 * A wavefront whose list fills up (ties, duplicated centroids, data that the thresholds tell nothing about) evaluates it on the spot, 16
 * pairs at a time (N = 262144, d = 256, k = 1024, 32 copies each of 32 centroids: 1.00 ms a call, with a lane per pair 6.85).
 *
 * counters[0] receives the number of points whose two smallest serial distances are closer than the three-product certificate.
 */
template <int KB, typename F>
__global__ void __launch_bounds__(EXACT_THREADS, 4)
listed_exact_kernel(const ExactArgs<F> w)
{
	const uint32_t blocks = KB ? KB : w.blocks, DP = blocks * KBLOCK;
	extern __shared__ __attribute__((aligned(16))) float lds[];
	f16x8* ops = (f16x8*)lds;                                   /* groups x KB x 64 lanes; the squares afterwards */
	__shared__ unsigned long long best[EXACT_ROWS], second[EXACT_ROWS];
	__shared__ float threshold[EXACT_ROWS], tau3[EXACT_ROWS];
	__shared__ uint32_t point[EXACT_ROWS];
	__shared__ uint32_t hits[EXACT_WAVES][EXACT_HITS];          /* row << 25 | centroid (supports: k < 2^25) */
	__shared__ uint32_t noted_by[EXACT_WAVES];
	constexpr bool DOUBLES = sizeof(F) == 8; /* keys of 96 bits: the smallest distances first, then who has them */
	__shared__ unsigned long long pair_bits[DOUBLES ? EXACT_WAVES * EXACT_HITS : 1];
	__shared__ uint32_t winner[DOUBLES ? EXACT_ROWS : 1];
	constexpr uint32_t PASS = DOUBLES ? 32 : 64; /* pairs a wavefront evaluates at a time */
	typedef F F4 __attribute__((ext_vector_type(4)));
	constexpr uint32_t PAIR = KBLOCK + 16 / sizeof(F); /* a pair's squares of a block in LDS; the padding spreads 16 lanes' reads over all banks */
	constexpr uint32_t CENTROID = (1u << 25) - 1u;
	const uint32_t count = w.length[0];
	if (count == 0) return;
	uint32_t groups = 1;
	while (2 * groups <= w.most_groups && groups * TILE * gridDim.x < count) groups *= 2;
	const uint32_t unit_rows = groups * TILE, units = (count + unit_rows - 1) / unit_rows;
	if (blockIdx.x >= units) return;
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t col = lane & 31, h = lane >> 5;
	const float scale = w.scale[0], unscale = w.scale[1];
	const uint32_t tiles = w.kp / TILE;
	/* (rows of fewer than four coordinates are read one by one, like those of SoA points) */
	const bool strided = KB <= 1 && (w.step != 1 || w.row_dim < 4), ragged = w.row_dim < DP && !strided;
	const bool points_strided = (KB <= 1 || DOUBLES) && (w.points_step != 1 || w.points_dim < 4), points_ragged = w.points_dim < DP && !points_strided;

	/* of the three-product ranking: only what is counted depends on it (the sweep left the maxima behind the scale) */
	const CertCoeffs cert = cert_coeffs_split(CentroidBounds{ w.scale[2], w.scale[3], w.scale[4] });

	/* four coordinates of a row at its coordinate d, as they come from memory (d brought inside the row), see exact_place */
	auto source = [&](uint32_t row) -> const float* { return w.data + (size_t)point[row] * w.stride; };
	auto serial_source = [&](uint32_t row) -> const F* { return w.points + (size_t)point[row] * w.points_stride; };
	auto request = [&](f32x4& v, const float* src, uint32_t d) { exact_request<float>(v, src, d, w.dim, w.row_dim, w.step, strided); };
	uint32_t close_here = 0;
	for (uint32_t unit = blockIdx.x; unit < units; unit += gridDim.x) {
		const uint32_t first = unit * unit_rows;
		__syncthreads(); /* the previous unit has been written out */
		if (tid < unit_rows) {
			const uint32_t e = min(first + tid, count - 1);
			point[tid] = w.list[2 * (size_t)e];
			threshold[tid] = first + tid < count ? __uint_as_float(w.list[2 * (size_t)e + 1]) : -__builtin_inff(); /* rows beyond the list pass nothing */
			best[tid] = ~0ull;
			if constexpr (DOUBLES) winner[tid] = ~0u;
			second[tid] = ~0ull;
		}
		__syncthreads();

		{
			uint32_t me = tid;
			asm volatile("" : "+v"(me)); /* (what follows is not worth keeping in registers from one unit to the next) */
			const uint32_t lanes = EXACT_THREADS / unit_rows; /* per row: 16, 8 or 4, a piece of four coordinates each */
			const uint32_t row = me / lanes, sub = me % lanes;
			const float* src = source(row);
			f16x8* dst = ops + (row / TILE) * (blocks * WAVE) + row % TILE;
			float x2 = 0.0f, xmid2 = 0.0f;
#pragma unroll 1
			for (uint32_t f0 = sub; f0 < DP / 4; f0 += 4 * lanes) {
				f32x4 v[4];
#pragma unroll
				for (int i = 0; i < 4; ++i) request(v[i], src, (f0 + i * lanes) * 4);
#pragma unroll
				for (int i = 0; i < 4; ++i) {
					const uint32_t d = (f0 + i * lanes) * 4;
					if (d >= DP) break;
					if (ragged) exact_place<float>(v[i], d, w.row_dim);
					const f32x4 m = *(const f32x4*)(w.frame + d);
					typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
					f16x4 half;
#pragma unroll
					for (int e = 0; e < 4; ++e) {
						const float s = __builtin_fmaf(v[i][e], scale, -(m[e] * scale));
						half[e] = (_Float16)s;
						__bf16 hi, mid;
						split_bf16(s, hi, mid);
						x2 += s * s;
						xmid2 += (float)mid * (float)mid;
					}
					/* block d / 16, half-wave (d % 16) / 8: four of its eight values */
					*(f16x4*)((char*)(dst + (d / KBLOCK) * WAVE + (d % KBLOCK) / 8 * TILE) + (d % 8) * 2) = half;
				}
			}
			for (uint32_t off = lanes / 2; off > 0; off >>= 1) { x2 += __shfl_xor(x2, off); xmid2 += __shfl_xor(xmid2, off); }
			if (sub == 0) tau3[row] = cert_tau(w.kd_split, x2, xmid2, cert);
		}
		__syncthreads();

		/*
		 * The serial sum of a point and a centroid, by four lanes (the same pair in all of them; all lanes of the wavefront call): each
		 * fetches and squares four of a block's 16 differences, then the running sum goes round the four, which add their squares in order.
		 */
		auto serial_sum = [&](uint32_t row, uint32_t c, uint32_t lane) -> F {
#pragma clang fp contract(off)
			const F* src = serial_source(row);
			const F* mean = w.means + (size_t)c * DP + lane % 4 * 4;
			/* blocks requested together: often one wavefront has all the pairs and nobody to wait beside (wide rows are whole chunks of four blocks) */
			constexpr uint32_t AT_ONCE = KB == 1 ? 1 : KB == 3 || KB == 6 ? 3 : KB == 2 || DOUBLES ? 2 : 4;
			static_assert(KB % AT_ONCE == 0, "whole steps");
			F sum = (F)0;
#pragma unroll 1
			for (uint32_t kb = 0; kb < blocks; kb += AT_ONCE) {
				F4 x[AT_ONCE], m[AT_ONCE];
#pragma unroll
				for (uint32_t u = 0; u < AT_ONCE; ++u) {
					exact_request<F>(x[u], src, (kb + u) * KBLOCK + lane % 4 * 4, w.dim, w.points_dim, w.points_step, points_strided);
					m[u] = *(const F4*)(mean + (kb + u) * KBLOCK);
				}
#pragma unroll
				for (uint32_t u = 0; u < AT_ONCE; ++u) {
					if (points_ragged && (kb + u + 1) * KBLOCK > w.points_dim) exact_place<F>(x[u], (kb + u) * KBLOCK + lane % 4 * 4, w.points_dim);
					F4 sq;
#pragma unroll
					for (int e = 0; e < 4; ++e) {
						const F diff = x[u][e] - m[u][e];
						sq[e] = diff * diff;
					}
					auto add = [&]() { return (((sum + sq[0]) + sq[1]) + sq[2]) + sq[3]; };
					sum = lane_of_four<0>(add()); /* (zeros behind the row change nothing) */
					sum = lane_of_four<1>(add());
					sum = lane_of_four<2>(add());
					sum = lane_of_four<3>(add());
				}
			}
			return sum;
		};
		/* doubles: who has the smallest distance is settled when it is known; `at`: where the pair's distance waits for that */
		auto merge = [&](uint32_t row, uint32_t c, F sum, uint32_t at) {
			if constexpr (DOUBLES) {
				pair_bits[at] = exact_bits(sum, c);
				atomicMin(&best[row], pair_bits[at]);
			}
			else {
				const unsigned long long key = exact_key(sum, c), before = atomicMin(&best[row], key);
				atomicMin(&second[row], before < key ? key : before);
			}
		};
		uint32_t noted = 0;                      /* wave-uniform */
		[[maybe_unused]] uint32_t kept = 0;      /* doubles: of those, evaluated before and kept */
		constexpr bool INSIDE = KB >= 1 && KB <= (DOUBLES ? 2 : 4); /* full lists are evaluated where they are found full */
		/* a list that is full: 16 pairs at a time (their rows and the tile's centroids are in the caches), or, rows of one block, a pair per lane */
		auto evaluate_here = [&]() {
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			__builtin_amdgcn_wave_barrier();
			[[maybe_unused]] const uint32_t full = noted;
			if constexpr (KB == 1) {
#pragma clang fp contract(off)
				for (uint32_t i = kept + lane; i < noted; i += WAVE) {
					const uint32_t hit = hits[wave][i], row = hit >> 25, c = hit & CENTROID;
					const F* src = serial_source(row);
					const F* mean = w.means + (size_t)c * DP;
					F sum = (F)0;
#pragma unroll 1
					for (uint32_t d = 0; d < w.dim; d += 4) {
						F4 x;
						exact_request<F>(x, src, d, w.dim, w.points_dim, w.points_step, points_strided);
						const F4 m = *(const F4*)(mean + d);
						if (points_ragged && d + 4 > w.points_dim) exact_place<F>(x, d, w.points_dim);
#pragma unroll
						for (int e = 0; e < 4; ++e) {
							const F diff = x[e] - m[e];
							const F sq = diff * diff;
							sum = sum + sq; /* (zeros behind the row change nothing) */
						}
					}
					merge(row, c, sum, wave * EXACT_HITS + i);
				}
			}
			else
			{
				uint32_t me = lane;
				asm volatile("" : "+v"(me)); /* (rare: nothing of this is worth keeping in registers meanwhile) */
#pragma unroll 1
				for (uint32_t i = kept; i < noted; i += WAVE / 4) {
					const uint32_t hit = hits[wave][min(i + me / 4, noted - 1)], row = hit >> 25, c = hit & CENTROID;
					const F sum = serial_sum(row, c, me);
					if (i + me / 4 < noted && me % 4 == 0) merge(row, c, sum, wave * EXACT_HITS + i + me / 4);
				}
			}
			auto in_order = [&]() {
				__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
				__builtin_amdgcn_wave_barrier();
			};
			in_order();
			noted = 0;
			if constexpr (DOUBLES) {
				/* what stays in the list is, per row, the first centroid of those at the row's smallest distance so far: at most one per row */
				constexpr uint32_t EACH = EXACT_HITS / WAVE;
				uint32_t hit[EACH];
				unsigned long long bits[EACH];
#pragma unroll
				for (uint32_t q = 0; q < EACH; ++q) {
					hit[q] = hits[wave][lane + q * WAVE];
					bits[q] = pair_bits[wave * EXACT_HITS + lane + q * WAVE];
				}
				in_order();
				uint32_t* lowest = (uint32_t*)&pair_bits[wave * EXACT_HITS]; /* per row; the distances are in registers */
				for (uint32_t row = lane; row < EXACT_ROWS; row += WAVE) lowest[row] = ~0u;
				in_order();
				bool keep[EACH];
#pragma unroll
				for (uint32_t q = 0; q < EACH; ++q) {
					keep[q] = lane + q * WAVE < full && bits[q] == best[hit[q] >> 25];
					if (keep[q]) atomicMin(&lowest[hit[q] >> 25], hit[q] & CENTROID);
				}
				in_order();
#pragma unroll
				for (uint32_t q = 0; q < EACH; ++q) {
					keep[q] = keep[q] && lowest[hit[q] >> 25] == (hit[q] & CENTROID);
					if (lane + q * WAVE < full && !keep[q]) atomicMin(&second[hit[q] >> 25], bits[q]);
				}
				in_order();
#pragma unroll
				for (uint32_t q = 0; q < EACH; ++q) {
					const unsigned long long mask = __builtin_amdgcn_ballot_w64(keep[q]);
					const uint32_t to = noted + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
					if (keep[q]) { hits[wave][to] = hit[q]; pair_bits[wave * EXACT_HITS + to] = bits[q]; }
					noted += (uint32_t)__popcll(mask);
				}
				kept = noted;
				in_order();
			}
		};
		uint32_t rounds = 0; /* of the tile and group at hand, noted before the list was full */
		auto screen = [&](const f32x16& a, uint32_t t, uint32_t g) -> bool { /* false: the list is full */
			const float limit = threshold[g * TILE + col];
			float low = a[0]; /* NaN-propagating minimum */
#pragma unroll
			for (int r = 1; r < 16; ++r) low = __builtin_elementwise_minimum(low, a[r]);
			const bool near = !(low > limit);
			if (__builtin_amdgcn_ballot_w64(near) == 0) return true;
			uint32_t passed = 0; /* bit r: result r */
#pragma unroll
			for (int r = 0; r < 16; ++r) passed |= !(a[r] > limit) ? 1u << r : 0u;
			if (t + 1 == tiles) { /* rows that do not exist */
#pragma unroll
				for (int r = 0; r < 16; ++r)
					if (t * TILE + 8 * (r / 4) + 4 * h + (r % 4) >= w.k) passed &= ~(1u << r);
			}
			for (uint32_t r = 0; r < rounds; ++r) passed &= passed - 1;
			for (;;) { /* the lanes' next results */
				const unsigned long long mask = __builtin_amdgcn_ballot_w64(passed != 0);
				if (mask == 0) break;
				const uint32_t more = (uint32_t)__popcll(mask);
				if (noted + more > EXACT_HITS) {
					/* (evaluated here it takes registers from the loops over tiles and groups, which narrow rows have to spare; being able to take
					 * those loops up again costs them more: N = 1M, d = 16, k = 1024, coordinates of 0 and 1: 249 against 233 us a call; N = 2M,
					 * d = 32, k = 1024: this kernel 64 against 60; N = 1M, d = 64, k = 512, small whole numbers: 1.6 % of a call. Doubles of 3 and 4
					 * blocks would spill 72 registers instead of 31) */
					if constexpr (INSIDE) evaluate_here();
					else return false;
				}
				if (passed) {
					const uint32_t r = (uint32_t)__builtin_ctz(passed);
					hits[wave][noted + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull))] = (g * TILE + col) << 25 | (t * TILE + 8 * (r / 4) + 4 * h + r % 4);
					passed &= passed - 1;
				}
				noted += more;
				++rounds;
			}
			rounds = 0;
			return true;
		};
		auto start_of = [&](uint32_t t) {
			f32x16 start;
#pragma unroll
			for (int q = 0; q < 4; ++q) {
				const f32x4 n0 = *(const f32x4*)(w.norms + t * NORM_TILE + 8 * q + 4 * h);
				start[4 * q] = n0.x; start[4 * q + 1] = n0.y; start[4 * q + 2] = n0.z; start[4 * q + 3] = n0.w;
			}
			return start;
		};
		/* few tiles: the wavefronts share out the groups of points as well */
		const uint32_t parts = tiles < EXACT_WAVES ? groups : 1;
		uint32_t t = wave / parts, g = wave % parts;
		for (;;) {
			bool room = true;
#pragma unroll 1
			while (t < tiles) {
				const f16x8* operand = w.packed + (size_t)t * (blocks * WAVE) + lane;
				if constexpr (KB > 0) {
					const f32x16 start = start_of(t);
					f16x8 c[KB];
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) c[kb] = operand[kb * WAVE];
#pragma unroll 1
					for (; g < groups; g += parts) {
						f32x16 a = start;
						const f16x8* x = ops + g * (KB * WAVE) + lane;
#pragma unroll
						for (int kb = 0; kb < KB; ++kb) a = __builtin_amdgcn_mfma_f32_32x32x16_f16(c[kb], x[kb * WAVE], a, 0, 0, 0);
						room = screen(a, t, g);
						if (!room) break;
					}
				}
				else {
					const uint32_t g0 = wave % parts;
					f32x16 a[EXACT_GROUPS];
					a[0] = start_of(t);
#pragma unroll
					for (uint32_t q = 1; q < EXACT_GROUPS; ++q) a[q] = a[0];
					for (uint32_t kb = 0; kb < blocks; kb += 4) { /* (rows are padded to whole chunks of four blocks) */
						f16x8 four[4];
#pragma unroll
						for (uint32_t i = 0; i < 4; ++i) four[i] = operand[(kb + i) * WAVE];
#pragma unroll
						for (uint32_t q = 0; q < EXACT_GROUPS; ++q)
							if (g0 + q * parts < groups) {
								const f16x8* x = ops + ((g0 + q * parts) * blocks + kb) * WAVE + lane;
#pragma unroll
								for (uint32_t i = 0; i < 4; ++i) a[q] = __builtin_amdgcn_mfma_f32_32x32x16_f16(four[i], x[i * WAVE], a[q], 0, 0, 0);
							}
					}
#pragma unroll
					for (uint32_t q = 0; q < EXACT_GROUPS; ++q)
						if (room && g0 + q * parts == g && g < groups) {
							room = screen(a[q], t, g);
							if (room) g += parts;
						}
				}
				if (!room) break;
				t += EXACT_WAVES / parts;
				g = wave % parts;
			}
			if (room) break;
			evaluate_here(); /* then this tile and group again, from where the list was full */
		}
		if (lane == 0) noted_by[wave] = noted;
		__syncthreads(); /* all pairs are listed, the operands are no longer needed */

		{
#pragma clang fp contract(off)
			uint32_t total = 0;
#pragma unroll
			for (uint32_t v = 0; v < EXACT_WAVES; ++v) total += noted_by[v];
			auto pair_of = [&](uint32_t at) -> uint32_t { /* pair `at` of all the lists */
				uint32_t list = 0;
				while (at >= noted_by[list]) at -= noted_by[list++];
				return hits[list][at];
			};
			/* equal shares of the pairs, in groups of 16 */
			const uint32_t share = ((total + 15) / 16 + EXACT_WAVES - 1) / EXACT_WAVES * 16;
			const uint32_t end = min((wave + 1) * share, total);
			F* squares = (F*)lds + wave * (PASS * PAIR);
#pragma unroll 1
			for (uint32_t p0 = wave * share; p0 < end; p0 += PASS) {
				/* this lane's pair (the last one again behind the end), and those it fetches for */
				const uint32_t hit = pair_of(min(p0 + lane % PASS, end - 1));
				F sum = (F)0;
				/* GROUPS of 16 pairs (those beyond the last repeat it), DEPTH blocks on their way while one is squared and added */
				auto evaluate = [&](auto groups_tag, auto depth_tag) {
					constexpr uint32_t GROUPS = decltype(groups_tag)::value, DEPTH = decltype(depth_tag)::value;
					const F* x[GROUPS]; const F* m[GROUPS];
#pragma unroll
					for (uint32_t g = 0; g < GROUPS; ++g) {
						const uint32_t other = (uint32_t)__shfl((int)hit, (int)(16 * g + lane / 4));
						x[g] = serial_source(other >> 25);
						m[g] = w.means + (size_t)(other & CENTROID) * DP + lane % 4 * 4;
					}
					F4 xv[DEPTH][GROUPS], mv[DEPTH][GROUPS];
					auto fetch = [&](uint32_t u, uint32_t kb) {
						kb = min(kb, blocks - 1);
#pragma unroll
						for (uint32_t g = 0; g < GROUPS; ++g) {
							exact_request<F>(xv[u][g], x[g], kb * KBLOCK + lane % 4 * 4, w.dim, w.points_dim, w.points_step, points_strided);
							mv[u][g] = *(const F4*)(m[g] + kb * KBLOCK);
						}
					};
#pragma unroll
					for (uint32_t u = 0; u < DEPTH; ++u) fetch(u, u);
#pragma unroll 1
					for (uint32_t kb0 = 0; kb0 < blocks; kb0 += DEPTH) {
#pragma unroll
						for (uint32_t u = 0; u < DEPTH; ++u) {
							const uint32_t kb = kb0 + u;
							if (DEPTH > 1 && kb >= blocks) break;
							if (points_ragged && (kb + 1) * KBLOCK > w.points_dim) {
#pragma unroll
								for (uint32_t g = 0; g < GROUPS; ++g) exact_place<F>(xv[u][g], kb * KBLOCK + lane % 4 * 4, w.points_dim);
							}
#pragma unroll
							for (uint32_t g = 0; g < GROUPS; ++g) {
								F4 sq;
#pragma unroll
								for (int e = 0; e < 4; ++e) {
									const F diff = xv[u][g][e] - mv[u][g][e];
									sq[e] = diff * diff;
								}
								*(F4*)(squares + (16 * g + lane / 4) * PAIR + lane % 4 * 4) = sq;
							}
							fetch(u, kb + DEPTH);
							__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
							__builtin_amdgcn_wave_barrier();
							const F* mine = squares + lane % (16 * GROUPS) * PAIR;
							F4 s[4];
#pragma unroll
							for (int q = 0; q < 4; ++q) s[q] = *(const F4*)(mine + 4 * q);
#pragma unroll
							for (int q = 0; q < 4; ++q)
#pragma unroll
								for (int e = 0; e < 4; ++e) sum = sum + s[q][e]; /* (zeros behind the row change nothing) */
							__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
							__builtin_amdgcn_wave_barrier();
						}
					}
				};
				if (end - p0 <= 16) evaluate(std::integral_constant<uint32_t, 1>{}, std::integral_constant<uint32_t, DOUBLES ? 2 : 4>{});
				else evaluate(std::integral_constant<uint32_t, PASS / 16>{}, std::integral_constant<uint32_t, 1>{});
				if (lane < PASS && p0 + lane < end) merge(hit >> 25, hit & CENTROID, sum, p0 + lane);
			}
			if constexpr (DOUBLES) {
				__syncthreads();
				auto settle = [&](uint32_t row, uint32_t c, unsigned long long bits) {
					if (bits != best[row]) atomicMin(&second[row], bits);
					else if (atomicMin(&winner[row], c) != ~0u) atomicMin(&second[row], bits);
				};
				for (uint32_t i = tid; i < total; i += EXACT_THREADS) {
					const uint32_t hit = pair_of(i), row = hit >> 25;
					settle(row, hit & CENTROID, pair_bits[i]);
				}
			}
		}
		__syncthreads();
		if (tid < unit_rows && first + tid < count) {
			const unsigned long long key = best[tid], next = second[tid];
			uint32_t c;
			double d1, d2;
			if constexpr (DOUBLES) {
				c = winner[tid];
				d1 = __longlong_as_double((long long)key); d2 = __longlong_as_double((long long)next);
			}
			else {
				c = (uint32_t)key;
				d1 = __uint_as_float((uint32_t)(key >> 32)); d2 = __uint_as_float((uint32_t)(next >> 32));
			}
			w.assignment[point[tid]] = key == ~0ull ? 0u : c;
			if (next != ~0ull && !((float)(d2 * d2 - d1 * d1) / unscale > tau3[tid])) ++close_here;
		}
	}
	if (wave < EXACT_ROWS / WAVE) {
		for (int off = WAVE / 2; off > 0; off >>= 1) close_here += (uint32_t)__shfl_xor((int)close_here, off);
		if (lane == 0 && close_here) atomicAdd(w.undecided, close_here);
	}
}

/* operands of the groups; the squares take their place */
constexpr uint32_t exact_dynamic_bytes(uint32_t blocks, uint32_t groups) { return std::max<uint32_t>(groups * blocks * WAVE * 16, EXACT_SQUARES_BYTES); }

template <int KB, typename F>
static int launch_listed_exact_kb(const AssignArgs& a, const ExactArgs<F>& w, const DeviceInfo& dev)
{
	void (*kernel)(ExactArgs<F>) = listed_exact_kernel<KB, F>;
	const uint32_t lds = exact_dynamic_bytes(KB ? KB : w.blocks, w.most_groups);
	KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
	const uint32_t grid = std::min<uint32_t>((a.n + TILE - 1) / TILE, 2 * dev.compute_units);
	KMX_LAUNCH_KERNEL(kernel, dim3(grid), dim3(EXACT_THREADS), lds, stream(), w);
	KMX_LAUNCH_CHECK("listed_exact_kernel");
	return KMX_OK;
}

} // namespace kmx

#endif
