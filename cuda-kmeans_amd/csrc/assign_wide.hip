/*
 * Assignment of rows of more than 256 dimensions on the matrix cores. The sweeps of the narrower rows (assign_bf16_impl.h)
 * keep the split operands of whole point rows in registers; a row of 512 dimensions does not fit there. Here a work-group
 * stages the rows of its points in LDS instead, 64 dimensions at a time, converted once on the way, and its eight wavefronts
 * share them: every wavefront owns centroid tiles of its own, whose packed operands it reads straight from the caches (no two
 * wavefronts of a work-group want the same ones, so LDS would only add a copy).
 *
 * Ranking, operands and certificates are those of rank16.hip, one product per dimension in half precision, and the points it lists get
 * their serial result from the exact pass of that file (rank16_exact_impl.h). Rows of more than 2304 dimensions, whose operands that
 * pass cannot keep in LDS, and kmx_set_two_level_sweep(0) take the three bf16 products of assign_bf16.hip and its exact pass.
 *
 * Split of the work. Per block of 16 dimensions a wavefront reads the operands of its NT centroid tiles (1 KB each, global)
 * and of the PT point tiles (1 KB each, LDS) for NT * PT MFMAs of 32 cycles; with NT = 2, PT = 4 the four SIMDs of a compute
 * unit ask the LDS for 64 and the vector cache for 32 of their 128 / 64 bytes per cycle, and all centroids pass by 128 points
 * at a time. The alternatives: PT = 2 doubles the cache traffic (at its limit), NT = 4 does not fit the registers.
 * The rows of a unit are read from memory once while 512 centroids go by; with more centroids the converted rows stay in LDS
 * if they fit (d <= 512), otherwise they are staged again per group of 512.
 *
 * What bounds it: latencies, between one barrier per 64 dimensions and the next, of one work-group of eight wavefronts per compute unit
 * (N = 131071, d = 512, k = 400: 85 us; the matrix cores are busy 32 % of the time, 13 tiles for eight wavefronts; the vector ALU 46 %, half of it the
 * search for the smallest results; the rows alone take 44 us to read). A wavefront converts its share of the next 64 dimensions piece by piece between
 * its matrix instructions of a block, while the SIMD's other wavefront has its own under way, and the last 64 of a unit bring the first of the next one
 * with them, so six of the eight wavefronts go on while two decide over the unit's points. With the conversion behind the 64
 * dimensions' products, and each unit started with a conversion of its own and a barrier: 111 us; columns of points, N = 65536: 175 -> 135 us per
 * call; k = 8, d = 257: 120 -> 101 us.
 * N = 131071, d = 512, k = 400, one iteration: the lane-per-point kernel that took these rows before needed 147 ms, two levels of bf16
 * products and a pass over the slices of the queued points (234 us of the assignment) 0.29 ms, this one 0.18 ms.
 */
#include "rank16_exact_impl.h"

namespace kmx {

constexpr uint32_t WIDE_THREADS = 512;
constexpr uint32_t WIDE_WAVES = WIDE_THREADS / WAVE;
constexpr uint32_t WIDE_CHUNK = 64;                       /* dimensions staged at a time */
constexpr uint32_t WIDE_BLOCKS = WIDE_CHUNK / KBLOCK;     /* MFMA blocks of a chunk */
constexpr uint32_t WIDE_LIST = 512;                       /* points waiting for the queue, per work-group */
constexpr uint32_t WIDE_ROW_PAD = 4;                      /* 16-byte units: the two half-waves' units of a block start 64 bytes apart modulo the banks */

/* the norms array: tiles of |c - m|^2, per row sum c'mid^2 and sum c'rest^2, the frame m (dp floats, |m|^2, an upper bound of |m|), tiles of |c|^2 */
__host__ __device__ __forceinline__ size_t wide_exact_norms_offset(uint32_t kp, uint32_t dp) { return frame_offset(kp) + dp + 4; }
__host__ __device__ __forceinline__ size_t wide_norms_floats(uint32_t kp, uint32_t dp) { return wide_exact_norms_offset(kp, dp) + split_norms_offset(kp); }
/* the packed centroids: plane of hi parts, plane of mid parts of -2 (c - m); inside a plane per tile and block the 64 lanes' 16-byte operands */
__host__ __device__ __forceinline__ size_t wide_plane_units(uint32_t kp, uint32_t dp) { return (size_t)(kp / TILE) * (dp / KBLOCK) * WAVE; }

struct WideArgs {
	const float* data; size_t stride;
	const bf16x8* packed;   /* bf16 parts, or half-precision values of S (c - m) */
	const float* norms;     /* tiles of |c - m|^2 (S^2 |c - m|^2) */
	const float* part_norms; /* per row the squared norm of the mid parts, then of the rest (of what half precision leaves out) */
	const float* frame;     /* dp floats: m; bf16: then |m|^2 and an upper bound of |m| */
	float* scale;           /* half precision: S (rank16_leave_bounds) */
	uint32_t* assignment; uint32_t* queue; uint32_t* counters;
	uint32_t dim, dp, k, kp, n, buffers;
	float kd, kd_unmoved;
};

/* One wavefront per (padded) centroid row; the frame as in sweep_frame, for any row length, computed by every work-group into LDS. */
template <int LM>
__global__ void __launch_bounds__(256)
pack_means_wide_kernel(const float* __restrict__ means, size_t stride_means, __bf16* __restrict__ packed, float* __restrict__ norms,
                       float* __restrict__ means_t, uint32_t dim, uint32_t k, uint32_t kp, uint32_t dp, uint32_t moved, uint32_t* __restrict__ counters)
{
	extern __shared__ float m[]; /* dp floats */
	constexpr uint32_t SAMPLE = 16;
	const uint32_t lane = threadIdx.x & (WAVE - 1);
	if (blockIdx.x == 0 && threadIdx.x == 0) { counters[0] = 0u; counters[LISTED_COUNTER] = 0u; }
	const uint32_t sample = min(k, SAMPLE);
	for (uint32_t q = threadIdx.x; q < dp; q += 256) {
		float sum = 0.0f;
		if (moved && q < dim) {
			float v[SAMPLE];
#pragma unroll
			for (uint32_t r = 0; r < SAMPLE; ++r) v[r] = r < sample ? means[elem<LM>(stride_means, r, q)] : 0.0f;
#pragma unroll
			for (uint32_t r = 0; r < SAMPLE; ++r) sum += __builtin_fabsf(v[r]) < __builtin_inff() ? v[r] : 0.0f;
			sum = sum / (float)sample;
			sum = __builtin_fabsf(sum) < __builtin_inff() ? sum : 0.0f;
		}
		m[q] = sum;
	}
	__syncthreads();
	if (blockIdx.x == 0) {
		float* stored = norms + frame_offset(kp);
		for (uint32_t q = threadIdx.x; q < dp; q += 256) stored[q] = m[q];
		if (threadIdx.x < WAVE) {
			float m2 = 0.0f;
			for (uint32_t q = threadIdx.x; q < dp; q += WAVE) m2 += m[q] * m[q];
			for (int off = 32; off > 0; off >>= 1) m2 += __shfl_xor(m2, off);
			if (threadIdx.x == 0) { stored[dp] = m2; stored[dp + 1] = __builtin_sqrtf(m2) * 1.0001f; }
		}
	}
	const uint32_t j = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
	if (j >= kp) return;
	const size_t plane = wide_plane_units(kp, dp) * 8;
	float c2 = 0.0f, mid2 = 0.0f, rest2 = 0.0f, exact2 = 0.0f;
	for (uint32_t q = lane; q < dp; q += WAVE) {
		const bool there = j < k && q < dim;
		const float exact = there ? means[elem<LM>(stride_means, j, q)] : 0.0f;
		const float v = there ? exact - m[q] : 0.0f;
		exact2 += exact * exact;
		c2 += v * v;
		__bf16 hi, mid;
		const float rest = split_bf16(-2.0f * v, hi, mid);
		mid2 += (float)mid * (float)mid;
		rest2 += rest * rest;
		const size_t at = (((size_t)(j / TILE) * (dp / KBLOCK) + q / KBLOCK) * WAVE + (q % KBLOCK) / 8 * TILE + j % TILE) * 8 + q % 8;
		packed[at] = hi;
		packed[plane + at] = mid;
		if (q < dim) means_t[(size_t)q * kp + j] = exact; /* exact copy for the exact pass */
	}
	for (int off = WAVE / 2; off > 0; off >>= 1) {
		c2 += __shfl_xor(c2, off);
		mid2 += __shfl_xor(mid2, off);
		rest2 += __shfl_xor(rest2, off);
		exact2 += __shfl_xor(exact2, off);
	}
	if (lane == 0) {
		norms[norm_at(j)] = j < k ? c2 : __builtin_inff();
		norms[wide_exact_norms_offset(kp, dp) + norm_at(j)] = j < k ? exact2 : __builtin_inff();
		norms[split_norms_offset(kp) + j] = mid2;
		norms[split_norms_offset(kp) + kp + j] = rest2;
	}
	if (lane < NORM_TILE - TILE && j % TILE == 0) {
		norms[(j / TILE) * NORM_TILE + TILE + lane] = __builtin_inff();
		norms[wide_exact_norms_offset(kp, dp) + (j / TILE) * NORM_TILE + TILE + lane] = __builtin_inff();
	}
}

/* ws->norms16 of wide rows: tiles of S^2 |c - m|^2; per row the squared norms of what half precision leaves out and of the bf16 mid
 * and rest parts (all of S (c - m)); m; S, 1 / S^2 and (rank16_leave_bounds) three maxima */
__host__ __device__ __forceinline__ size_t wide16_part_offset(uint32_t kp) { return (size_t)(kp / TILE) * NORM_TILE; }
__host__ __device__ __forceinline__ size_t wide16_frame_offset(uint32_t kp) { return wide16_part_offset(kp) + 3 * (size_t)kp; }
__host__ __device__ __forceinline__ size_t wide16_scale_offset(uint32_t kp, uint32_t dp) { return wide16_frame_offset(kp) + dp; }
static size_t wide16_norms_floats(uint32_t kp, uint32_t dp) { return wide16_scale_offset(kp, dp) + 8; }

/* groups of 32 listed points whose operands fit the LDS of the exact pass (0: none) */
static uint32_t wide16_groups(uint32_t dp, bool doubles, uint32_t lds_budget)
{
	for (uint32_t groups : { 4u, 2u, 1u })
		if (exact_dynamic_bytes(dp / KBLOCK, groups) + exact_static_bytes(doubles) <= lds_budget) return groups;
	return 0;
}

/*
 * pack_means16_kernel (rank16.hip) for any row length: one wavefront per (padded) centroid row. A chain of latencies: eight loads of a lane are
 * on their way together, the first eight while the frame is found (k = 400, d = 512: 6.9 us; one after the other 11.0 us).
 */
template <int LM>
__global__ void __launch_bounds__(256)
pack_means16_wide_kernel(const float* __restrict__ means, const double* __restrict__ means64, size_t stride_means, _Float16* __restrict__ packed, float* __restrict__ rows, float* __restrict__ norms,
                         uint32_t dim, uint32_t k, uint32_t kp, uint32_t dp, uint32_t* __restrict__ counters)
{
	extern __shared__ float m[]; /* dp floats */
	__shared__ float wave_far[2][4];
	constexpr uint32_t SAMPLE = 16, EACH = 8;
	const uint32_t lane = threadIdx.x & (WAVE - 1);
	if (blockIdx.x == 0 && threadIdx.x == 0) { counters[0] = 0u; counters[LISTED_COUNTER] = 0u; }
	const uint32_t sample = min(k, SAMPLE);
	const uint32_t j = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE; /* (below kp: whole tiles) */
	float own[EACH];
	auto request = [&](uint32_t base) {
#pragma unroll
		for (uint32_t i = 0; i < EACH; ++i) own[i] = means[elem<LM>(stride_means, min(j, k - 1), min(base + i * WAVE + lane, dim - 1))];
	};
	request(0); /* (on its way while the frame is found) */
	float far = 0.0f, size = 0.0f;
	for (uint32_t q = threadIdx.x; q < dp; q += 256) {
		float sum = 0.0f;
		if (q < dim) {
			float v[SAMPLE];
#pragma unroll
			for (uint32_t r = 0; r < SAMPLE; ++r) v[r] = r < sample ? means[elem<LM>(stride_means, even_row(r, 4, k), q)] : 0.0f;
#pragma unroll
			for (uint32_t r = 0; r < SAMPLE; ++r) sum += __builtin_fabsf(v[r]) < __builtin_inff() ? v[r] : 0.0f;
			sum = sum / (float)sample;
			sum = __builtin_fabsf(sum) < __builtin_inff() ? sum : 0.0f;
#pragma unroll
			for (uint32_t r = 0; r < SAMPLE; ++r) {
				const float d = __builtin_fabsf(v[r] - sum);
				if (r < sample && d < __builtin_inff()) { far = fmaxf(far, d); size = fmaxf(size, __builtin_fabsf(v[r])); }
			}
		}
		m[q] = sum;
	}
	for (int off = WAVE / 2; off > 0; off >>= 1) { far = fmaxf(far, __shfl_xor(far, off)); size = fmaxf(size, __shfl_xor(size, off)); }
	if (lane == 0) { wave_far[0][threadIdx.x / WAVE] = far; wave_far[1][threadIdx.x / WAVE] = size; }
	__syncthreads();
	const float scale = rank16_scale(fmaxf(fmaxf(wave_far[0][0], wave_far[0][1]), fmaxf(wave_far[0][2], wave_far[0][3])),
	                                 fmaxf(fmaxf(wave_far[1][0], wave_far[1][1]), fmaxf(wave_far[1][2], wave_far[1][3])));
	if (blockIdx.x == 0) {
		for (uint32_t q = threadIdx.x; q < dp; q += 256) norms[wide16_frame_offset(kp) + q] = m[q];
		if (threadIdx.x == 0) {
			norms[wide16_scale_offset(kp, dp)] = scale;
			norms[wide16_scale_offset(kp, dp) + 1] = 1.0f / (scale * scale);
		}
	}
	float c2 = 0.0f, low2 = 0.0f, mid2 = 0.0f, rest2 = 0.0f;
	for (uint32_t base = 0; base < dp; base += EACH * WAVE) {
		if (base) request(base);
		double own64[EACH];
		if (means64) {
#pragma unroll
			for (uint32_t i = 0; i < EACH; ++i) own64[i] = means64[elem<LM>(stride_means, min(j, k - 1), min(base + i * WAVE + lane, dim - 1))];
		}
#pragma unroll
		for (uint32_t i = 0; i < EACH; ++i) {
			const uint32_t q = base + i * WAVE + lane;
			if (base + i * WAVE >= dp) break;
			const bool there = j < k && q < dim;
			const float exact = there ? own[i] : 0.0f;
			const float v = there ? __builtin_fmaf(exact, scale, -(m[q] * scale)) : 0.0f;
			c2 += v * v;
			const float cv = -2.0f * v;
			const _Float16 half = (_Float16)cv;
			const float low = cv - (float)half;
			low2 += low * low;
			__bf16 hi, mid;
			const float rest = split_bf16(cv, hi, mid);
			mid2 += (float)mid * (float)mid;
			rest2 += rest * rest;
			if (means64) ((double*)rows)[(size_t)j * dp + q] = there ? own64[i] : 0.0;
			else rows[(size_t)j * dp + q] = exact;
			packed[(((size_t)(j / TILE) * (dp / KBLOCK) + q / KBLOCK) * WAVE + (q % KBLOCK) / 8 * TILE + j % TILE) * 8 + q % 8] = half;
		}
	}
	for (int off = WAVE / 2; off > 0; off >>= 1) {
		c2 += __shfl_xor(c2, off);
		low2 += __shfl_xor(low2, off);
		mid2 += __shfl_xor(mid2, off);
		rest2 += __shfl_xor(rest2, off);
	}
	if (lane == 0) {
		norms[norm_at(j)] = j < k ? c2 : 1.7e38f;
		norms[wide16_part_offset(kp) + j] = low2;
		norms[wide16_part_offset(kp) + kp + j] = mid2;
		norms[wide16_part_offset(kp) + 2 * kp + j] = rest2;
	}
	if (lane < NORM_TILE - TILE && j % TILE == 0) norms[(j / TILE) * NORM_TILE + TILE + lane] = 1.7e38f;
}

/*
 * PT point tiles of 32 per unit, NT centroid tiles per wavefront and group (a group: the WIDE_WAVES * NT tiles that go by together),
 * X3: three bf16 products instead of one in half precision.
 *
 * Order of a step (one chunk of 64 dimensions against one group), per block of 16: the MFMAs of the first tile, the conversion of a quarter of
 * the rows requested a step ago into the next buffer and the request of their successors, the MFMAs of the second tile, each followed by the
 * request from LDS of its point tile's next operand, and the request of the centroid operands of the block RING blocks on. Loads retire in
 * order, so the rows have until then to arrive. RESIDENT: all chunks of a unit stay in LDS, staged once.
 *
 * Ranking values carry the number of their result (4 or 5 bits) in the lowest mantissa bits, as in the single-pass kernels
 * (cert_kd_keyed): three operations per value for the two smallest and the place of the smallest. A NaN anywhere makes the smallest
 * NaN (v_minimum3_f32 passes it on), which certifies nothing.
 */
template <int PT, int NT, bool X3, int LD, bool VEC, bool RESIDENT>
__global__ void __launch_bounds__(WIDE_THREADS)
wide_sweep_kernel(const WideArgs w)
{
	constexpr uint32_t ROWS = PT * TILE;
	constexpr uint32_t SUBS = WIDE_THREADS / ROWS;          /* lanes that stage one row */
	constexpr uint32_t VECS = WIDE_CHUNK / 4 / SUBS;        /* 4-dimension pieces per lane and chunk */
	constexpr uint32_t UNIT_STRIDE = ROWS + WIDE_ROW_PAD;   /* 16-byte units between the half-blocks of a chunk */
	constexpr uint32_t PART_UNITS = 2 * WIDE_BLOCKS * UNIT_STRIDE;
	constexpr uint32_t BUFFER_UNITS = (X3 ? 2 : 1) * PART_UNITS;
	constexpr uint32_t GROUP_TILES = WIDE_WAVES * NT;
	constexpr uint32_t KEY_MASK = NT * 16 - 1;
	constexpr uint32_t SUMS = X3 ? 3 : 2;                   /* of a row: |x|^2, the part left out; X3: (x - m) . m */
	static_assert(VECS * SUBS * 4 == WIDE_CHUNK && NT <= 2 && SUMS * WIDE_THREADS <= BUFFER_UNITS * 4, "shape");

	extern __shared__ __attribute__((aligned(16))) float dyn[];
	float* frame = dyn;                            /* dp floats (a multiple of 64) */
	bf16x8* rows_lds = (bf16x8*)(dyn + w.dp);      /* w.buffers buffers of BUFFER_UNITS */
	__shared__ float cand_first[WIDE_WAVES][ROWS], cand_second[WIDE_WAVES][ROWS];
	__shared__ uint32_t cand_idx[WIDE_WAVES][ROWS];
	__shared__ float row_info[3][ROWS];            /* |x|^2, squared norm of the part the products drop, (x - m) . m */
	__shared__ __attribute__((aligned(16))) float norm_stage[WIDE_WAVES][NT * TILE];
	__shared__ uint32_t flags[2 * WIDE_LIST];
	__shared__ uint32_t flag_count, flag_base;
	__shared__ uint32_t wave_max[3][WIDE_WAVES];

	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t col = lane & 31, h = lane >> 5;
	const uint32_t n = w.n;
	const float scale = X3 ? 1.0f : w.scale[0];
	const uint32_t units = (n + ROWS - 1) / ROWS;
	const uint32_t tiles = w.kp / TILE;
	const uint32_t groups = (tiles + GROUP_TILES - 1) / GROUP_TILES;
	const uint32_t chunks = w.dp / WIDE_CHUNK;
	const uint32_t blocks = w.dp / KBLOCK;
	const uint32_t steps = groups * chunks;
	const uint32_t staged_steps = RESIDENT ? chunks : steps;
	if (blockIdx.x >= units) return; /* the whole work-group */

	/* the certificate's maxima over the centroids (bit patterns: NaN and infinity win) and the frame */
	if (tid == 0) flag_count = 0u;
	for (uint32_t q = tid; q < w.dp; q += WIDE_THREADS) frame[q] = w.frame[q] * scale; /* S m */
	const float m2 = X3 ? w.frame[w.dp] : 0.0f, mnorm = X3 ? w.frame[w.dp + 1] : 0.0f;
	CertCoeffs cert;
	{
		uint32_t most[3] = { 0u, 0u, 0u };
		for (uint32_t j = tid; j < w.k; j += WIDE_THREADS) {
			most[0] = max(most[0], __float_as_uint(w.norms[norm_at(j)]));
			most[1] = max(most[1], __float_as_uint(w.part_norms[j]));
			if (X3) most[2] = max(most[2], __float_as_uint(w.part_norms[w.kp + j]));
		}
#pragma unroll
		for (int q = 0; q < 3; ++q) {
			for (int off = WAVE / 2; off > 0; off >>= 1) most[q] = max(most[q], (uint32_t)__shfl_xor((int)most[q], off));
			if (lane == 0) wave_max[q][wave] = most[q];
		}
		__syncthreads();
#pragma unroll
		for (int q = 0; q < 3; ++q) {
			most[q] = 0;
			for (uint32_t v = 0; v < WIDE_WAVES; ++v) most[q] = max(most[q], wave_max[q][v]);
		}
		const CentroidBounds cb{ __uint_as_float(most[0]), __uint_as_float(most[1]), __uint_as_float(most[2]) };
		if (!X3 && blockIdx.x == 0) rank16_leave_bounds(w.scale, most[0], most[1], w.part_norms, w.k, w.kp);
		cert = X3 ? cert_coeffs_split(cb) : cert_coeffs_level1(cb);
	}

	/* staging: this lane's row of the unit and its pieces of a chunk */
	const uint32_t row = LD == KMX_AOS ? tid / SUBS : tid % ROWS;
	const uint32_t sub = LD == KMX_AOS ? tid % SUBS : tid / ROWS;
	f32x4 piece[VECS];
	auto point_of = [&](uint32_t unit) -> uint32_t { /* rows beyond the end repeat the last one */
		const uint32_t slot = min(unit * ROWS + row, n - 1);
		return slot;
	};
	auto request_piece = [&](uint32_t i, uint32_t pt, uint32_t chunk) {
		const uint32_t d = chunk * WIDE_CHUNK + (i * SUBS + sub) * 4;
		f32x4 v = { 0.0f, 0.0f, 0.0f, 0.0f };
		/* (pieces beyond the row repeat its end: no branches around the loads; store_piece puts zeros there) */
		if (LD == KMX_AOS) {
			typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4))); /* 16-byte loads need no more than 4-byte alignment */
			const float* at = w.data + (size_t)pt * w.stride + min(d, w.dim - 4);
			if constexpr (VEC) v = *(const f32x4*)at;
			else v = *(const f32x4_any*)at;
		}
		else {
#pragma unroll
			for (uint32_t e = 0; e < 4; ++e) v[e] = w.data[elem<LD>(w.stride, pt, min(d + e, w.dim - 1))];
		}
		piece[i] = v;
	};
	float xx = 0.0f, xpart = 0.0f, xalong = 0.0f;
	auto store_piece = [&](uint32_t i, uint32_t buffer, uint32_t chunk, bool first_pass) {
		typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
		char* base = (char*)(rows_lds + (size_t)buffer * BUFFER_UNITS);
		const uint32_t f = i * SUBS + sub, d = chunk * WIDE_CHUNK + f * 4;
		const f32x4 mv = *(const f32x4*)(frame + d);
		if constexpr (LD == KMX_AOS && !VEC) {
			/* the piece that holds the end of a row whose length is no multiple of four came from up to three places before */
			if ((chunk + 1) * WIDE_CHUNK > w.dim && d + 4 > w.dim && d < w.dim) {
				const f32x4 p = piece[i];
				const uint32_t s = d + 4 - w.dim;
				piece[i].x = s == 1 ? p.y : s == 2 ? p.z : p.w;
				piece[i].y = s == 1 ? p.z : p.w;
				piece[i].z = p.w;
			}
		}
		bf16x4 hi, mid;
		float a = 0.0f, b = 0.0f, c = 0.0f;
#pragma unroll
		for (uint32_t e = 0; e < 4; ++e) {
			const bool there = d + (VEC ? 0 : e) < w.dim;
			if constexpr (X3) {
				const float v = there ? piece[i][e] - mv[e] : 0.0f;
				__bf16 vh, vm;
				split_bf16(v, vh, vm);
				hi[e] = vh;
				mid[e] = vm;
				a += v * v;
				b += (float)vm * (float)vm;
				c += v * mv[e];
			}
			else {
				const float v = there ? __builtin_fmaf(piece[i][e], scale, -mv[e]) : 0.0f;
				const _Float16 half = (_Float16)v;
				const float low = v - (float)half;
				hi[e] = __builtin_bit_cast(__bf16, half);
				a += v * v;
				b += low * low;
			}
		}
		xx += first_pass ? a : 0.0f;
		xpart += first_pass ? b : 0.0f;
		if constexpr (X3) xalong += first_pass ? c : 0.0f;
		asm volatile("" : "+v"(xx), "+v"(xpart)); /* (summed here: left alone the compiler keeps all pieces' values until after the matrix instructions) */
		char* at = base + ((f / 2) * UNIT_STRIDE + row) * 16 + (f % 2) * 8;
		*(bf16x4*)at = hi;
		if constexpr (X3) *(bf16x4*)(at + PART_UNITS * 16) = mid;
	};

	/* this wavefront's tile of a group (beyond the last tile: the last one again, with infinite norms) */
	auto tile_of = [&](uint32_t group, int nt) -> uint32_t { return group * GROUP_TILES + nt * WIDE_WAVES + wave; };
	const size_t plane = wide_plane_units(w.kp, w.dp);
	const bf16x8* next_ops[NT]; /* operands of the next step */
	uint32_t next_chunk = 0, next_group = 0;
	auto seek = [&]() {
#pragma unroll
		for (int nt = 0; nt < NT; ++nt)
			next_ops[nt] = w.packed + ((size_t)min(tile_of(next_group, nt), tiles - 1) * blocks + next_chunk * WIDE_BLOCKS) * WAVE;
	};
	auto advance = [&]() {
		if (++next_chunk == chunks) {
			next_chunk = 0;
			if (++next_group == groups) next_group = 0;
		}
		seek();
	};
	/* Blocks that a centroid tile's operands are requested ahead, and buffers of the points'. Units of 128 points have no registers left for more (4 blocks
	 * ahead: 88 -> 98 us at N = 131071, d = 512, k = 400); units of 32 are all latency (n = 3000, k = 300: 45 us with these, 49 with the others). */
	constexpr int RING = PT == 1 ? WIDE_BLOCKS : 2, SLOTS = PT == 1 ? 2 : 1;
	bf16x8 ahi[RING][NT], amid[X3 ? RING : 1][NT];
	auto fetch_ops = [&](int slot, int b) {
#pragma unroll
		for (int nt = 0; nt < NT; ++nt) {
			ahi[slot][nt] = next_ops[nt][b * WAVE + lane];
			if constexpr (X3) amid[slot][nt] = (next_ops[nt] + plane)[b * WAVE + lane];
		}
	};
	/* |c|^2 of this wavefront's tiles of a group, one per lane; requested a group ahead */
	float norm_reg = 0.0f;
	auto request_norms = [&](uint32_t group) {
		const uint32_t tile = tile_of(group, NT == 2 ? (int)h : 0);
		/* rows that do not exist: beyond all values, but finite (a number in the low bits would make infinity a NaN) */
		norm_reg = tile * TILE + col < w.k ? w.norms[tile * NORM_TILE + col] : 1.7e38f;
	};

	uint32_t unit = blockIdx.x;
	uint32_t pt = point_of(unit);
	request_norms(0);
	seek();
#pragma unroll
	for (int b = 0; b < RING; ++b) fetch_ops(b, b);
#pragma unroll
	for (uint32_t i = 0; i < VECS; ++i) request_piece(i, pt, 0);
	const uint32_t uniform_n = n;
#pragma unroll
	for (uint32_t i = 0; i < VECS; ++i) {
		store_piece(i, 0, 0, true);
		request_piece(i, pt, 1);
	}
	uint32_t write_chunk = 1, write_buffer = 1, read_buffer = 0;
	__syncthreads();

	for (; unit < units; unit += gridDim.x) {
		const uint32_t next_pt = unit + gridDim.x < units ? point_of(unit + gridDim.x) : pt;
		float best[PT], second[PT];
		uint32_t best_idx[PT];
#pragma unroll
		for (int p = 0; p < PT; ++p) { best[p] = __builtin_inff(); second[p] = __builtin_inff(); best_idx[p] = 0; }
		float unit_xx = 0.0f, unit_xpart = 0.0f, unit_xalong = 0.0f;

		uint32_t step = 0;
		for (uint32_t group = 0; group < groups; ++group) {
			f32x16 acc[NT][PT];
			norm_stage[wave][NT == 2 ? lane : col] = norm_reg;
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			__builtin_amdgcn_wave_barrier();
#pragma unroll
			for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
				for (int g = 0; g < 4; ++g) {
					const f32x4 v = *(const f32x4*)&norm_stage[wave][nt * TILE + 8 * g + 4 * h];
					acc[nt][0][4 * g] = v.x; acc[nt][0][4 * g + 1] = v.y; acc[nt][0][4 * g + 2] = v.z; acc[nt][0][4 * g + 3] = v.w;
				}
#pragma unroll
				for (int p = 1; p < PT; ++p) acc[nt][p] = acc[nt][0];
			}
			request_norms(group + 1 < groups ? group + 1 : 0);
			bool busy[NT]; /* uniform: which tiles of this wavefront exist in this group */
#pragma unroll
			for (int nt = 0; nt < NT; ++nt) busy[nt] = tile_of(group, nt) < tiles;

			for (uint32_t chunk = 0; chunk < chunks; ++chunk, ++step) {
				const bf16x8* rows_at = rows_lds + (size_t)read_buffer * BUFFER_UNITS + h * UNIT_STRIDE + col;
				bf16x8 bhi[SLOTS][PT], bmid[SLOTS][X3 ? PT : 1];
				auto fetch_point = [&](int b, int p) {
					bhi[b % SLOTS][p] = rows_at[2 * b * UNIT_STRIDE + p * TILE];
					if constexpr (X3) bmid[b % SLOTS][p] = rows_at[PART_UNITS + 2 * b * UNIT_STRIDE + p * TILE];
				};
				/* the last step stages the first chunk of the next unit, so that its products follow without a wait */
				const bool last_step = step + 1 == steps;
				const bool stages = (!RESIDENT && PT > 1) || step + 1 < staged_steps || (last_step && (PT > 1 || unit + gridDim.x < units)), first_pass = step + 1 < chunks || last_step;
				const uint32_t request_pt = step + 2 < staged_steps ? pt : next_pt, request_chunk = write_chunk + 1 < chunks ? write_chunk + 1 : 0;
				if (last_step) {
					if (RESIDENT) __syncthreads(); /* (all are past the unit's first chunk) */
					unit_xx = xx; unit_xpart = xpart; unit_xalong = xalong;
					xx = xpart = xalong = 0.0f;
				}
#pragma unroll
				for (int p = 0; p < PT; ++p) fetch_point(0, p);
#pragma unroll
				for (int b = 0; b < (int)WIDE_BLOCKS; ++b) {
					if constexpr (SLOTS > 1)
						if (b + 1 < (int)WIDE_BLOCKS)
#pragma unroll
							for (int p = 0; p < PT; ++p) fetch_point(b + 1, p);
					__builtin_amdgcn_sched_barrier(0);
					auto products = [&](int nt) {
						const bool ahead = SLOTS == 1 && nt == NT - 1 && b + 1 < (int)WIDE_BLOCKS;
						if (!busy[nt]) {
							if (ahead)
#pragma unroll
								for (int p = 0; p < PT; ++p) fetch_point(b + 1, p);
							return;
						}
						if constexpr (X3) {
#pragma unroll
							for (int p = 0; p < PT; ++p) acc[nt][p] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahi[b % RING][nt], bmid[b % SLOTS][p], acc[nt][p], 0, 0, 0);
#pragma unroll
							for (int p = 0; p < PT; ++p) acc[nt][p] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(amid[X3 ? b % RING : 0][nt], bhi[b % SLOTS][p], acc[nt][p], 0, 0, 0);
						}
#pragma unroll
						for (int p = 0; p < PT; ++p) {
							if constexpr (X3) acc[nt][p] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ahi[b % RING][nt], bhi[b % SLOTS][p], acc[nt][p], 0, 0, 0);
							else acc[nt][p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, ahi[b % RING][nt]), __builtin_bit_cast(f16x8, bhi[b % SLOTS][p]), acc[nt][p], 0, 0, 0);
							if (ahead) {
								fetch_point(b + 1, p);
								__builtin_amdgcn_sched_barrier(0);
							}
						}
					};
					products(0);
					__builtin_amdgcn_sched_barrier(0);
					if (stages) {
#pragma unroll
						for (uint32_t i = 0; i < VECS; ++i)
							if ((int)((i + 1) * WIDE_BLOCKS / VECS) == b + 1) {
								store_piece(i, write_buffer, write_chunk, first_pass);
								request_piece(i, request_pt, request_chunk);
							}
					}
					__builtin_amdgcn_sched_barrier(0);
					if constexpr (NT == 2) products(NT - 1);
					__builtin_amdgcn_sched_barrier(0);
					if ((b + RING) % (int)WIDE_BLOCKS == 0) advance();
					fetch_ops(b % RING, (b + RING) % (int)WIDE_BLOCKS);
					__builtin_amdgcn_sched_barrier(0);
				}
				if (stages) {
					write_chunk = write_chunk + 1 == chunks ? 0 : write_chunk + 1;
					write_buffer = write_buffer + 1 == w.buffers ? 0 : write_buffer + 1;
					__syncthreads();
				}
				read_buffer = read_buffer + 1 == w.buffers ? 0 : read_buffer + 1;
			}

			if (busy[0]) {
#pragma unroll
				for (int p = 0; p < PT; ++p) {
					__builtin_amdgcn_sched_barrier(0); /* one point tile at a time: the keyed values of all of them do not fit the registers */
					float g1 = __builtin_inff(), g2 = __builtin_inff();
#pragma unroll
					for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
						for (int r = 0; r < 16; ++r) {
							const float v = __uint_as_float((__float_as_uint(acc[nt][p][r]) & ~KEY_MASK) | (uint32_t)(nt * 16 + r));
							g2 = __builtin_amdgcn_fmed3f(g1, g2, v);
							g1 = __builtin_elementwise_minimum(g1, v);
							asm volatile("" : "+v"(g1), "+v"(g2)); /* value by value: left alone the compiler takes all minima first and spills the values for the medians */
						}
					}
					const uint32_t key = __float_as_uint(g1) & KEY_MASK, r = key % 16;
					const uint32_t idx = (group * GROUP_TILES + (key / 16) * WIDE_WAVES + wave) * TILE + 8 * (r / 4) + 4 * h + r % 4;
					const bool wins = g1 < best[p];
					second[p] = fminf(fminf(second[p], g2), fmaxf(best[p], g1));
					best_idx[p] = wins ? idx : best_idx[p];
					best[p] = __builtin_elementwise_minimum(best[p], g1);
				}
			}
		}

		/* the two half-waves of a wavefront, then the wavefronts */
#pragma unroll
		for (int p = 0; p < PT; ++p) {
			const float ob = __shfl_xor(best[p], 32), os = __shfl_xor(second[p], 32);
			const uint32_t oi = (uint32_t)__shfl_xor((int)best_idx[p], 32);
			if (h == 0) {
				cand_second[wave][p * TILE + col] = fminf(fminf(second[p], os), fmaxf(best[p], ob));
				cand_idx[wave][p * TILE + col] = ob < best[p] ? oi : best_idx[p];
				cand_first[wave][p * TILE + col] = __builtin_elementwise_minimum(best[p], ob);
			}
		}
		if (LD == KMX_AOS) {
			for (int off = SUBS / 2; off > 0; off >>= 1) {
				unit_xx += __shfl_xor(unit_xx, off);
				unit_xpart += __shfl_xor(unit_xpart, off);
				unit_xalong += __shfl_xor(unit_xalong, off);
			}
			if (sub == 0) { row_info[0][row] = unit_xx; row_info[1][row] = unit_xpart; if constexpr (X3) row_info[2][row] = unit_xalong; }
		}
		else {
			/* the lanes of a row sit in different wavefronts: their shares meet in LDS, in a fixed order, where the unit's last chunk was */
			if (PT == 1) __syncthreads(); /* (its last step need not have ended with a barrier) */
			float* share = (float*)(rows_lds + (size_t)(read_buffer ? read_buffer - 1 : w.buffers - 1) * BUFFER_UNITS);
			share[(0 * SUBS + sub) * ROWS + row] = unit_xx;
			share[(1 * SUBS + sub) * ROWS + row] = unit_xpart;
			if constexpr (X3) share[(2 * SUBS + sub) * ROWS + row] = unit_xalong;
			__syncthreads();
			if (tid < ROWS) {
				for (uint32_t q = 0; q < SUMS; ++q) {
					float s = 0.0f;
					for (uint32_t i = 0; i < SUBS; ++i) s += share[(q * SUBS + i) * ROWS + tid];
					row_info[q][tid] = s;
				}
			}
		}
		const bool full = flag_count + ROWS > WIDE_LIST; /* (the same in every lane: no one adds to the list between the last step's barrier and the next one) */
		__syncthreads();
		if (full) {
			if (tid == 0) { flag_base = atomicAdd(&w.counters[0], flag_count); }
			__syncthreads();
			for (uint32_t i = tid; i < 2 * flag_count; i += WIDE_THREADS) w.queue[2 * (size_t)flag_base + i] = flags[i];
			__syncthreads();
			if (tid == 0) flag_count = 0u;
			__syncthreads();
		}
		/* the other wavefronts go on with the next unit */
		if (tid < ROWS) {
			float first = cand_first[0][tid], next = cand_second[0][tid];
			uint32_t idx = cand_idx[0][tid];
#pragma unroll
			for (uint32_t v = 1; v < WIDE_WAVES; ++v) {
				const float cf = cand_first[v][tid];
				next = fminf(fminf(next, cand_second[v][tid]), fmaxf(first, cf));
				idx = cf < first ? cand_idx[v][tid] : idx;
				first = __builtin_elementwise_minimum(first, cf);
			}
			const float x2 = row_info[0][tid], along = X3 ? row_info[2][tid] : 0.0f;
			const float tau = cert_tau(w.kd, x2, row_info[1][tid], cert);
			const uint32_t slot = unit * ROWS + tid;
			const bool mine = slot < uniform_n;
			/* squares of the data as given underflow or overflow: no ranking says anything about the serial sums (in the frame of the
			 * data as it is, an overflow makes the values infinite or NaN) */
			const bool extreme = !(x2 + cert.c2max > 1e-30f * (scale * scale)) || (!X3 && !(x2 + cert.c2max < 1e37f * (scale * scale)));
			const bool decided = (next - first > tau) && !extreme && idx < w.k;
			if (mine) w.assignment[slot] = idx < w.k ? idx : 0u;
			if (mine && !decided) {
				const uint32_t at = atomicAdd(&flag_count, 1u);
				flags[2 * at] = slot;
				flags[2 * at + 1] = !X3 ? screening_threshold(extreme ? __builtin_inff() : first, tau) : w.kd_unmoved > 0.0f
					? screening_threshold(cert_unmoved_threshold(first, tau, x2, along, cert.c2max, m2, mnorm, w.kd_unmoved), 0.0f)
					: screening_threshold(first, tau);
			}
		}
		pt = next_pt;
	}
	__syncthreads();
	if (flag_count) {
		if (tid == 0) flag_base = atomicAdd(&w.counters[0], flag_count);
		__syncthreads();
		for (uint32_t i = tid; i < 2 * flag_count; i += WIDE_THREADS) w.queue[2 * (size_t)flag_base + i] = flags[i];
	}
}

constexpr uint32_t WIDE_MAX_DIM = 2560; /* what the exact pass takes */

static uint32_t wide_buffer_bytes(uint32_t pt, bool x3) { return (x3 ? 2u : 1u) * 2 * WIDE_BLOCKS * (pt * TILE + WIDE_ROW_PAD) * 16; }
static uint32_t wide_static_bytes(uint32_t pt, uint32_t nt) { return (3 * WIDE_WAVES * pt * TILE + 3 * pt * TILE + WIDE_WAVES * nt * TILE + 2 * WIDE_LIST + 3 * WIDE_WAVES + 64) * 4; }

/* LDS of a sweep with units of 32 pt points, nt tiles per wavefront, two buffers */
static uint32_t wide_sweep_bytes(uint32_t dp, uint32_t pt, uint32_t nt, bool x3) { return dp * 4 + 2 * wide_buffer_bytes(pt, x3) + wide_static_bytes(pt, nt); }

bool wide_supports(const AssignArgs& a, uint32_t lds_budget)
{
	return a.dim > 256 && a.dim <= WIDE_MAX_DIM && (wide16_supports(a, lds_budget) || wide_sweep_bytes(round_up(a.dim, WIDE_CHUNK), 1, 1, true) <= lds_budget);
}

template <int PT, int NT, bool X3>
static int launch_wide_sweep(const AssignArgs& a, WideArgs w, uint32_t lds_budget, const DeviceInfo& dev, kmx_exec_params* exec)
{
	const bool vec = a.dim % 4 == 0 && a.stride % 4 == 0 && ((uintptr_t)a.data & 15) == 0;
	const uint32_t chunks = w.dp / WIDE_CHUNK, groups = (w.kp / TILE + WIDE_WAVES * NT - 1) / (WIDE_WAVES * NT);
	const uint32_t buffer = wide_buffer_bytes(PT, X3);
	const uint32_t room = lds_budget - wide_static_bytes(PT, NT) - w.dp * 4; /* (wide_sweep_bytes fits) */
	/* all chunks of a unit stay in LDS where another group of centroids wants them again */
	const bool resident = groups > 1 && (uint64_t)chunks * buffer <= room;
	w.buffers = resident ? chunks : 2u;
	void (*kernel)(WideArgs) = a.layout == KMX_SOA ? (resident ? wide_sweep_kernel<PT, NT, X3, KMX_SOA, false, true> : wide_sweep_kernel<PT, NT, X3, KMX_SOA, false, false>)
	                           : vec ? (resident ? wide_sweep_kernel<PT, NT, X3, KMX_AOS, true, true> : wide_sweep_kernel<PT, NT, X3, KMX_AOS, true, false>)
	                                 : (resident ? wide_sweep_kernel<PT, NT, X3, KMX_AOS, false, true> : wide_sweep_kernel<PT, NT, X3, KMX_AOS, false, false>);
	const uint32_t lds_bytes = w.dp * 4 + w.buffers * buffer;
	const uint32_t units = (a.n + PT * TILE - 1) / (PT * TILE);
	const uint32_t grid = std::min(units, dev.compute_units);
	exec->block_count = grid;
	KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
	KMX_LAUNCH_KERNEL(kernel, dim3(grid), dim3(WIDE_THREADS), lds_bytes, stream(), w);
	KMX_LAUNCH_CHECK("wide_sweep_kernel");
	return KMX_OK;
}

/* every offset the kernels form must lie inside its allocation (see check_sweep_plan) */
static int check_wide_plan(const AssignArgs& a, const WideArgs& w, const Workspace* ws, bool half)
{
#define KMX_PLAN(cond) do { if (!(cond)) return fail(KMX_ERR_DEVICE, "assign (wide rows): launch refused, the plan breaks \"%s\" (dim %u, k %u, kp %u, n %u)", #cond, a.dim, a.k, w.kp, a.n); } while (0)
	KMX_PLAN(w.dp % WIDE_CHUNK == 0 && w.dp >= a.dim && w.kp % TILE == 0 && w.kp >= a.k && w.kp - a.k < TILE && a.n >= 1);
	if (half) {
		KMX_PLAN(ws->packed16 && wide_plane_units(w.kp, w.dp) * 4 + (size_t)w.kp * w.dp * (a.points64 ? 2 : 1) <= ws->packed16_cap);
		KMX_PLAN(ws->norms16 && wide16_norms_floats(w.kp, w.dp) <= ws->norms16_cap);
		KMX_PLAN(ws->listed && 2 * (size_t)a.n <= ws->listed_cap && ws->counters);
		return KMX_OK;
	}
	KMX_PLAN(ws->packed_means && wide_plane_units(w.kp, w.dp) * 2 * 4 <= ws->packed_cap);
	KMX_PLAN(ws->norms && wide_norms_floats(w.kp, w.dp) <= ws->norms_cap);
	KMX_PLAN(ws->means_t && (size_t)w.kp * a.dim <= ws->means_t_cap);
	KMX_PLAN(ws->queue && 2 * (size_t)a.n <= ws->queue_cap && ws->counters);
#undef KMX_PLAN
	return KMX_OK;
}

/* one half-precision product per dimension, then the exact pass for what that lists */
static int launch_assign_wide16(const AssignArgs& a, uint32_t dp, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	const uint32_t kp = round_up(a.k, TILE);
	const size_t operand_floats = wide_plane_units(kp, dp) * 4;
	int rc = reserve_packed16(ws, operand_floats + (size_t)kp * dp * (a.points64 ? 2 : 1), wide16_norms_floats(kp, dp));
	if (rc) return rc;
	if ((rc = reserve_listed(ws, 2 * (size_t)a.n))) return rc;
	float* rows = ws->packed16 + operand_floats;
	auto pack = a.layout_means == KMX_AOS ? pack_means16_wide_kernel<KMX_AOS> : pack_means16_wide_kernel<KMX_SOA>;
	KMX_LAUNCH_KERNEL(pack, dim3((kp * WAVE + 255) / 256), dim3(256), dp * 4, stream(),
	                   a.means, a.means64, a.stride_means, (_Float16*)ws->packed16, rows, ws->norms16, a.dim, a.k, kp, dp, ws->counters);
	KMX_LAUNCH_CHECK("pack_means16_wide_kernel");
	const float* norms = ws->norms16;
	const WideArgs w = { a.data, a.stride, (const bf16x8*)ws->packed16, norms, norms + wide16_part_offset(kp), norms + wide16_frame_offset(kp), ws->norms16 + wide16_scale_offset(kp, dp),
	                     a.assignment, ws->listed, ws->counters + LISTED_COUNTER, a.dim, dp, a.k, kp, a.n, 0,
	                     cert_kd_level1(a.dim) + cert_kd_keyed(5) + 8.0f * CERT_UNIT + a.kd_extra, 0.0f };
	if (!sizing_only() && (rc = check_wide_plan(a, w, ws, true))) return rc;
	if ((rc = profile_begin(0))) return rc;
	/* units of 128 points, or, where those do not reach half of the compute units or do not fit, of 32 */
	const uint32_t budget = lds_budget_of(exec, dev);
	const bool large = a.n >= 64 * dev.compute_units && wide_sweep_bytes(dp, 4, 2, false) <= budget;
	rc = large ? launch_wide_sweep<4, 2, false>(a, w, budget, dev, exec) : launch_wide_sweep<1, 1, false>(a, w, budget, dev, exec);
	if (rc) return rc;
	if ((rc = profile_end(0))) return rc;
	const size_t stride = a.layout == KMX_AOS ? a.stride : 1, step = a.layout == KMX_AOS ? 1 : a.stride;
	const uint32_t groups = wide16_groups(dp, a.points64 != nullptr, budget);
	auto exact = [&](auto* points, auto* centroids) -> int {
		typedef typename std::remove_const<typename std::remove_pointer<decltype(points)>::type>::type F;
		const ExactArgs<F> e = { a.data, stride, step, a.dim, points, stride, step, a.dim, centroids, (const f16x8*)ws->packed16, norms,
		                         norms + wide16_frame_offset(kp), norms + wide16_scale_offset(kp, dp), a.assignment, ws->listed, ws->counters + LISTED_COUNTER, ws->counters,
		                         a.dim, a.k, kp, cert_kd_split(a.dim) + 8.0f * CERT_UNIT, dp / KBLOCK, groups };
		return launch_listed_exact_kb<0, F>(a, e, dev);
	};
	rc = a.points64 ? exact(a.points64, (const double*)rows) : exact(a.data, (const float*)rows);
	if (rc) return rc;
	if (a.settled) *a.settled = true;
	return KMX_OK;
}

bool wide16_supports(const AssignArgs& a, uint32_t lds_budget)
{
	const uint32_t dp = round_up(a.dim, WIDE_CHUNK);
	return two_level_mode() != 0 && a.k < (1u << 25) && (!a.ranking_only || a.points64) && wide_sweep_bytes(dp, 1, 1, false) <= lds_budget &&
	       wide16_groups(dp, a.points64 != nullptr, lds_budget) > 0;
}

int launch_assign_wide(const AssignArgs& args, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	AssignArgs a = args;
	const uint32_t dp = round_up(a.dim, WIDE_CHUNK), kp = round_up(a.k, TILE);
	const uint32_t budget = lds_budget_of(exec, dev);
	if (wide16_supports(a, budget))
		return launch_assign_wide16(a, dp, exec, ws, dev);
	const bool moved = !a.ranking_only; /* (the double path hands over copies it has moved itself) */
	int rc = reserve_packed(ws, wide_plane_units(kp, dp) * 2 * 4, wide_norms_floats(kp, dp), (size_t)kp * a.dim);
	if (rc) return rc;
	if ((rc = reserve_queue(ws, 2 * (size_t)a.n))) return rc;
	auto pack = a.layout_means == KMX_AOS ? pack_means_wide_kernel<KMX_AOS> : pack_means_wide_kernel<KMX_SOA>;
	KMX_LAUNCH_KERNEL(pack, dim3((kp * WAVE + 255) / 256), dim3(256), dp * 4, stream(),
	                   a.means, a.stride_means, (__bf16*)ws->packed_means, ws->norms, ws->means_t, a.dim, a.k, kp, dp, moved ? 1u : 0u, ws->counters);
	KMX_LAUNCH_CHECK("pack_means_wide_kernel");

	const WideArgs w = { a.data, a.stride, (const bf16x8*)ws->packed_means, ws->norms, ws->norms + split_norms_offset(kp), ws->norms + frame_offset(kp), nullptr,
	                     a.assignment, ws->queue, ws->counters, a.dim, dp, a.k, kp, a.n, 0,
	                     cert_kd_split(a.dim) + cert_kd_keyed(4) + (moved ? 8.0f * CERT_UNIT : 0.0f) + a.kd_extra, moved ? cert_kd_unmoved(a.dim) : 0.0f };
	if (!sizing_only() && (rc = check_wide_plan(a, w, ws, false))) return rc;
	if ((rc = profile_begin(0))) return rc;
	const bool large = a.n >= 128 * dev.compute_units && wide_sweep_bytes(dp, 4, 1, true) <= budget;
	rc = large ? launch_wide_sweep<4, 1, true>(a, w, budget, dev, exec) : launch_wide_sweep<1, 1, true>(a, w, budget, dev, exec);
	if (rc) return rc;
	if ((rc = profile_end(0))) return rc;
	if (a.ranking_only) return KMX_OK; /* the caller resolves the queued points */
	ws->exact_norms = ws->norms + wide_exact_norms_offset(kp, dp);
	rc = launch_recheck(a, ws, kp);
	ws->exact_norms = nullptr;
	return rc;
}

} // namespace kmx
