/*
 * The ranking sweep on half-precision operands: a[j] = |c_j|^2 - 2 c_j . x, one v_mfma_f32_32x32x16_f16 per 16 dimensions and tile of
 * 32 x 32, for every point; what it cannot settle is listed. Device code, instantiated per row width (rank16_inst.hip); the design
 * and the launch rules are in rank16.hip.
 */
#ifndef KMX_RANK16_IMPL_H
#define KMX_RANK16_IMPL_H

#include "assign_bf16_impl.h"

namespace kmx {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr uint32_t RANK16_WAVES = 8;
constexpr uint32_t RANK16_THREADS = RANK16_WAVES * WAVE;
constexpr int RANK16_P = 2; /* point tiles per wavefront: an operand read serves two instructions */
constexpr uint32_t RANK16_LIST = 128;

struct Rank16Args {
	const float* data; size_t stride;
	const f16x8* packed;   /* per tile and block of 16 dimensions the 64 lanes' operands of -2 S (c - m), 16 bytes each */
	const float* norms;    /* tiles of S^2 |c - m|^2 */
	const float* low2;     /* per padded row the squared norm of what the half-precision parts leave out */
	const float* frame;    /* m */
	float* scale;          /* S, 1 / S^2; the first work-group puts the maxima of the norms and of the bf16 mid and rest parts behind them */
	uint32_t* assignment; uint32_t* list; uint32_t* length;
	float* copies; uint32_t copy_stride; /* SoA: the rows as AoS, zeros behind the coordinates */
	uint32_t dim, k, kp, n, chunk_tiles;
	float kd;
};

/* ws->packed16: the operands, then the centroids' rows as they are, padded with zeros to whole blocks */
inline size_t rank16_rows_offset(uint32_t kp, uint32_t dp) { return (size_t)kp * dp / 2; }
/* ws->norms16: tiles of S^2 |c - m|^2, then per row the squared norms of what half precision leaves out, of the bf16 mid and of the rest
 * parts, then the frame m, S, 1 / S^2 and (rank16_leave_bounds) four maxima */
__host__ __device__ __forceinline__ size_t rank16_low_offset(uint32_t kp) { return (size_t)(kp / TILE) * NORM_TILE; }
__host__ __device__ __forceinline__ size_t rank16_frame_offset(uint32_t kp) { return rank16_low_offset(kp) + 3 * (size_t)kp; }
__host__ __device__ __forceinline__ size_t rank16_scale_offset(uint32_t kp) { return rank16_frame_offset(kp) + FRAME_FLOATS; }
inline size_t rank16_norms_floats(uint32_t kp) { return rank16_scale_offset(kp) + 8; }

/* 16 tile bytes per block of 16 dimensions and lane, then the tile's norms */
template <int KB> constexpr uint32_t rank16_tile_floats() { return KB * WAVE * 4; }
template <int KB> constexpr uint32_t rank16_static_bytes() { return (2 * RANK16_LIST * RANK16_WAVES + 4 * RANK16_WAVES + KB * KBLOCK) * 4 + 64; }

/*
 * S for centroids whose coordinates are up to `far` from the frame and up to `size` from the origin, both of a sample: the power of two
 * that puts far into [2^-5, 2^-4), kept inside what S and 1 / S^2 can be as normal numbers. A coordinate may then be half a million
 * times larger before it overflows (which would certify nothing any more), and what half precision loses below its smallest normal
 * number, 2^-25 at most, is a 256th of the rounding of a coordinate as large as far. Less than 2^-12 of `size` is taken for that: a
 * sample of equal rows differs from their mean by its roundings only. (With far in [16, 32) from the first 16 centroids a quiet start of
 * 5e-3 before centroids of 20 overflowed: N = 1M, d = 32, k = 512 in 29 ms; now 0.31.)
 */
__device__ __forceinline__ float rank16_scale(float far, float size)
{
	far = fmaxf(far, size * 0x1p-12f);
	const int shift = far > 0.0f ? min(max(122 - (int)(__float_as_uint(far) >> 23), -60), 60) : 0;
	return __uint_as_float((uint32_t)(127 + shift) << 23);
}

/* row r of 2^log >= 4 rows spread evenly over k: four neighbours (of SoA centroids, in one line) at each place, the places multiples of the
 * golden ratio (equal steps would meet the same row again and again where rows repeat) */
__device__ __forceinline__ uint32_t even_row(uint32_t r, uint32_t log, uint32_t k)
{
	return min(k <= (1u << log) ? r : __umulhi(r / 4 * 0x9E3779B9u, k) + r % 4, k - 1);
}

/* the exact pass's certificate, by one work-group (first wavefront): max |c|^2, max |mid|^2, max |rest|^2 and max |low|^2 to scale[2 .. 5] */
__device__ __forceinline__ void rank16_leave_bounds(float* scale, uint32_t c2max, uint32_t low2max, const float* part_norms, uint32_t k, uint32_t kp)
{
	if (threadIdx.x >= WAVE) return;
	uint32_t mid = 0, rest = 0; /* (bit patterns: NaN and infinity win) */
	for (uint32_t j = threadIdx.x; j < k; j += WAVE) {
		mid = max(mid, __float_as_uint(part_norms[kp + j]));
		rest = max(rest, __float_as_uint(part_norms[2 * kp + j]));
	}
	for (int off = WAVE / 2; off > 0; off >>= 1) {
		mid = max(mid, (uint32_t)__shfl_xor((int)mid, off));
		rest = max(rest, (uint32_t)__shfl_xor((int)rest, off));
	}
	if (threadIdx.x == 0) { scale[2] = __uint_as_float(c2max); scale[3] = __uint_as_float(mid); scale[4] = __uint_as_float(rest); scale[5] = __uint_as_float(low2max); }
}

/* the 8 coordinates of a half-wave of block kb as they come from memory, zeros beyond the row. Blocks inside the row (the same
 * for all lanes) are loaded without guards. */
template <int LD>
__device__ __forceinline__ void rank16_request(float (&v)[8], const float* __restrict__ data, size_t stride, uint32_t pt, uint32_t kb, uint32_t h, uint32_t dim)
{
	typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
	const uint32_t d0 = kb * KBLOCK + h * 8;
	if (LD == KMX_AOS) {
		const float* src = data + (size_t)pt * stride + d0;
		if ((kb + 1) * KBLOCK <= dim) {
			const f32x4 lo = *(const f32x4_any*)src, up = *(const f32x4_any*)(src + 4);
			v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = up.x; v[5] = up.y; v[6] = up.z; v[7] = up.w;
		}
		else {
			load_piece_any(v, src, true, d0, dim);
			load_piece_any(v + 4, src + 4, true, d0 + 4, dim);
		}
	}
	else {
		const float* src = data + (size_t)d0 * stride + pt;
		if ((kb + 1) * KBLOCK <= dim) {
#pragma unroll
			for (int j = 0; j < 8; ++j) { v[j] = *src; src += stride; }
		}
		else {
#pragma unroll
			for (int j = 0; j < 8; ++j) { v[j] = d0 + j < dim ? *src : 0.0f; src += stride; }
		}
	}
}

/*
 * SoA: the rows go out as AoS on the way, for the exact pass and whatever else reads single rows (coordinates of a listed point lie a
 * cache line each apart; with 9 % of N = 2M, d = 128 listed, gathering them read all data again, 430 us, and was no cheaper right
 * behind the sweep of the point, 360 us. The stores travel behind the matrix instructions).
 */
template <int LD>
__device__ __forceinline__ void rank16_copy(const Rank16Args& w, const float (&v)[8], uint32_t pt, uint32_t d0)
{
	if (LD == KMX_AOS || pt >= w.n || d0 >= w.copy_stride) return;
	float* dst = w.copies + (size_t)pt * w.copy_stride + d0;
	*(f32x4*)dst = f32x4{ v[0], v[1], v[2], v[3] };
	*(f32x4*)(dst + 4) = f32x4{ v[4], v[5], v[6], v[7] };
}

/* v = S (x - m) rounded once (S is a power of two), its half-precision part, and the shares of |v|^2 and of the squared norm of the rest */
__device__ __forceinline__ void rank16_convert(f16x8& b, const float (&raw)[8], const float* frame, float scale, float& part, float& low)
{
	const f32x4 m0 = *(const f32x4*)frame, m1 = *(const f32x4*)(frame + 4); /* S m */
	const float m[8] = { m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w };
#pragma unroll
	for (int j = 0; j < 8; ++j) {
		const float v = __builtin_fmaf(raw[j], scale, -m[j]);
		part = __builtin_fmaf(v, v, part);
		const _Float16 h = (_Float16)v;
		const float r = v - (float)h;
		low = __builtin_fmaf(r, r, low);
		b[j] = h;
	}
}

/*
 * A work-group of eight wavefronts around centroids in LDS: all of them (STREAM = false), or two buffers of chunk_tiles tiles that
 * go round (a barrier per chunk, all wavefronts sweep together). A wavefront sweeps 64 points at a time. With resident centroids the
 * wavefronts take items of 64 points from a counter in LDS (a SIMD serves its older wavefront first: equal shares leave the
 * younger ones sweeping alone at the end).
 *
 * Tracking is the snapshot of assign_bf16_impl.h: the minimum of a lane's 16 results per tile, the two smallest minima, and the 16
 * results of the leading tile, from which the winner and the runner-up inside that tile come at the end.
 * Rows of up to 64 dimensions and resident centroids: two accumulator sets, the tracking of one tile in pieces behind the matrix
 * instructions of the next (the fenced step). Otherwise one chain per tile whose tracking the partner wavefront of the SIMD covers.
 */
template <int KB, int LD, bool STREAM>
__global__ void __launch_bounds__(RANK16_THREADS)
rank16_kernel(const Rank16Args w)
{
	constexpr int P = RANK16_P;
	constexpr uint32_t TF = rank16_tile_floats<KB>();
	constexpr bool PIPE = !STREAM && KB <= 4;
	constexpr bool SNAP = KB < 12;          /* wider rows: their operands leave no registers for the snapshot, their instructions hide row-by-row tracking */
	constexpr bool PREFETCH = PIPE && KB <= 2; /* the next item's coordinates travel while the current one is swept */
	extern __shared__ __attribute__((aligned(16))) float lds[];
	__shared__ __attribute__((aligned(16))) float frame[KB * KBLOCK]; /* S m */
	__shared__ uint32_t wave_max[4][RANK16_WAVES];
	__shared__ uint32_t flag_list[RANK16_WAVES][2 * RANK16_LIST];
	uint32_t& claimed = wave_max[3][0];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t col = lane & 31, h = lane >> 5;
	const float scale = w.scale[0], smallest = 1e-30f * (scale * scale), largest = 1e37f * (scale * scale);
	if (tid == 0) claimed = 0u;
	for (uint32_t i = tid; i < KB * KBLOCK; i += RANK16_THREADS) frame[i] = w.frame[i] * scale;

	CertCoeffs cert;
	{
		uint32_t most[2] = { 0u, 0u };
		for (uint32_t j = tid; j < w.k; j += RANK16_THREADS) {
			most[0] = max(most[0], __float_as_uint(w.norms[norm_at(j)]));
			most[1] = max(most[1], __float_as_uint(w.low2[j]));
		}
#pragma unroll
		for (int q = 0; q < 2; ++q) {
			for (int off = WAVE / 2; off > 0; off >>= 1) most[q] = max(most[q], (uint32_t)__shfl_xor((int)most[q], off));
			if (lane == 0) wave_max[q][wave] = most[q];
		}
		__syncthreads();
#pragma unroll
		for (int q = 0; q < 2; ++q) {
			most[q] = 0;
			for (uint32_t v = 0; v < RANK16_WAVES; ++v) most[q] = max(most[q], wave_max[q][v]);
		}
		if (blockIdx.x == 0) rank16_leave_bounds(w.scale, most[0], most[1], w.low2, w.k, w.kp);
		cert = cert_coeffs_level1(CentroidBounds{ __uint_as_float(most[0]), __uint_as_float(most[1]), 0.0f });
		cert.c2max = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(cert.c2max)));
		cert.a = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(cert.a)));
		cert.b = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(cert.b)));
	}

	const uint32_t all_tiles = w.kp / TILE;
	const uint32_t buffer_floats = w.chunk_tiles * (TF + NORM_TILE); /* chunk_tiles tiles of operands, then their norms */
	const uint32_t chunks = (all_tiles + w.chunk_tiles - 1) / w.chunk_tiles;
	uint32_t cur = 0;
	{
		const uint32_t tiles = min(w.chunk_tiles, all_tiles);
		f32x4* dst = (f32x4*)lds;
		const f32x4* src = (const f32x4*)w.packed;
		for (uint32_t i = tid; i < tiles * (TF / 4); i += RANK16_THREADS) dst[i] = src[i];
		f32x4* ndst = (f32x4*)(lds + (size_t)w.chunk_tiles * TF);
		const f32x4* nsrc = (const f32x4*)w.norms;
		for (uint32_t i = tid; i < tiles * (NORM_TILE / 4); i += RANK16_THREADS) ndst[i] = nsrc[i];
	}
	__syncthreads();

	uint32_t flagged = 0; /* wave-uniform */
	auto flush_flags = [&]() {
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		uint32_t slot = 0;
		if (lane == 0) slot = atomicAdd(w.length, flagged);
		slot = (uint32_t)__shfl((int)slot, 0);
		for (uint32_t i = lane; i < 2 * flagged; i += WAVE) w.list[2 * (size_t)slot + i] = flag_list[wave][i];
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		flagged = 0;
	};

	/* the operands of a tile for this lane, and the norms of the 16 rows it receives */
	auto operand = [&](const float* tiles, uint32_t tile, int kb) -> f16x8 { return ((const f16x8*)(tiles + (size_t)tile * TF))[kb * WAVE + lane]; };

	f16x8 b[P][KB];
	float xx[P], xl[P]; /* this half-wave's shares of |v|^2 and of the squared norm of the rest */
	float m1[P], m2[P];
	uint32_t leader[P];
	float snap[P][SNAP ? SNAP_ROWS : 1];

	auto load_points = [&](uint32_t first) {
#pragma unroll
		for (int p = 0; p < P; ++p) { xx[p] = 0.0f; xl[p] = 0.0f; }
		constexpr int GROUP = KB <= 2 ? KB : KB <= 12 ? 4 : 2; /* blocks whose coordinates are in registers at a time */
		uint32_t dim = w.dim;
		asm volatile("" : "+s"(dim)); /* (the comparisons with it are not kept from one item to the next: they are as many as scalar registers) */
#pragma unroll
		for (int g = 0; g < KB; g += GROUP) {
#pragma unroll
			for (int p = 0; p < P; ++p) {
				float raw[GROUP][8];
				const uint32_t pt = min(first + p * TILE + col, w.n - 1); /* rows beyond the points repeat the last one */
#pragma unroll
				for (int i = 0; i < GROUP; ++i)
					if (g + i < KB) rank16_request<LD>(raw[i], w.data, w.stride, pt, g + i, h, dim);
#pragma unroll
				for (int i = 0; i < GROUP; ++i)
					if (g + i < KB) {
						rank16_copy<LD>(w, raw[i], first + p * TILE + col, (g + i) * KBLOCK + h * 8);
						rank16_convert(b[p][g + i], raw[i], frame + (g + i) * KBLOCK + h * 8, scale, xx[p], xl[p]);
						if constexpr (KB > 2) asm volatile("" : "+v"(b[p][g + i]));
					}
				if constexpr (KB > 2) {
					/* the sums exist here: left alone the compiler moves them behind the sweep and keeps the coordinates alive */
					asm volatile("" : "+v"(xx[p]), "+v"(xl[p]));
					__builtin_amdgcn_sched_barrier(0);
				}
			}
		}
	};

	auto finish = [&](uint32_t first_pt) {
#pragma unroll
		for (int p = 0; p < P; ++p) {
			/* the two smallest of the leading tile's 16 results, the number of a result in its lowest four bits (cert_kd_keyed) */
			float v1 = __builtin_inff(), v2 = __builtin_inff();
			if constexpr (!SNAP) { v1 = m1[p]; v2 = m2[p]; }
			else
#pragma unroll
			for (int r = 0; r < SNAP_ROWS; ++r) {
				const float v = __uint_as_float((__float_as_uint(snap[p][r]) & ~15u) | (uint32_t)r);
				v2 = __builtin_amdgcn_fmed3f(v1, v2, v);
				v1 = __builtin_elementwise_minimum(v1, v);
			}
			const uint32_t r = __float_as_uint(v1) & 15u;
			const uint32_t mine_idx = leader[p] * TILE + 8 * (r / 4) + 4 * h + r % 4;
			const float o1 = __shfl_xor(m1[p], 32), o2 = __shfl_xor(m2[p], 32);
			const float ov1 = __shfl_xor(v1, 32), ov2 = __shfl_xor(v2, 32);
			const uint32_t oi = (uint32_t)__shfl_xor((int)mine_idx, 32);
			const bool win = m1[p] < o1 || (m1[p] == o1 && h == 0);
			const float others = win ? fminf(o1, m2[p]) : fminf(m1[p], o2); /* everything outside the leading 16 rows */
			const uint32_t idx = win ? mine_idx : oi;
			const float lowest = win ? v1 : ov1;
			const float next = fminf(win ? v2 : ov2, others); /* (!SNAP: v2 is m2) */
			const float x2 = xx[p] + __shfl_xor(xx[p], 32), low = xl[p] + __shfl_xor(xl[p], 32);
			const float tau = cert_tau(w.kd, x2, low, cert);
			const uint32_t pt = first_pt + p * TILE + col;
			const bool mine = h == 0 && pt < w.n;
			/* squares of the data as given underflow or overflow: no ranking says anything about the serial sums */
			const bool extreme = !(x2 + cert.c2max > smallest && x2 + cert.c2max < largest);
			const bool decided = (next - lowest > tau) && !extreme && idx < w.k;
			if (mine) w.assignment[pt] = idx < w.k ? idx : 0u;
			const bool flag = mine && !decided;
			const unsigned long long mask = __ballot(flag);
			if (mask) {
				const uint32_t add = (uint32_t)__builtin_popcountll(mask);
				if (flagged + add > RANK16_LIST) flush_flags();
				if (flag) {
					const uint32_t at = 2 * (flagged + (uint32_t)__builtin_popcountll(mask & ((1ull << lane) - 1ull)));
					flag_list[wave][at] = pt;
					flag_list[wave][at + 1] = screening_threshold(extreme ? __builtin_inff() : lowest, tau); /* (scaled, like the values) */
				}
				flagged += add;
			}
		}
	};

	auto start = [&]() {
#pragma unroll
		for (int p = 0; p < P; ++p) {
			m1[p] = __builtin_inff(); m2[p] = __builtin_inff(); leader[p] = 0;
#pragma unroll
			for (int i = 0; i < (SNAP ? SNAP_ROWS : 0); ++i) asm volatile("" : "=v"(snap[p][i])); /* no value yet: tile 0 always takes the lead */
		}
	};

	auto lowest_of = [](float a, float c) { return __builtin_elementwise_minimum(a, c); };
	auto track = [&](const f32x16& acc, int p, uint32_t tile) {
		if constexpr (!SNAP) { /* every result keyed with its number: the two smallest so far, the tile of the smallest */
			const float before = m1[p];
#pragma unroll
			for (int r = 0; r < 16; ++r) {
				const float v = __uint_as_float((__float_as_uint(acc[r]) & ~15u) | (uint32_t)r);
				m2[p] = __builtin_amdgcn_fmed3f(m1[p], m2[p], v);
				m1[p] = __builtin_elementwise_minimum(m1[p], v);
				asm volatile("" : "+v"(m1[p]), "+v"(m2[p])); /* value by value (see wide_sweep_kernel) */
			}
			leader[p] = m1[p] < before ? tile : leader[p];
			return;
		}
		else {
		float t = acc[0];
#pragma unroll
		for (int i = 1; i < 16; ++i) t = lowest_of(t, acc[i]);
		m2[p] = __builtin_amdgcn_fmed3f(m1[p], m2[p], t);
		const uint64_t leads = settled_mask(tile == 0 ? ~0ull : __builtin_amdgcn_ballot_w64(t < m1[p]));
		take_lead_where(leads, m1[p], leader[p], t, tile, snap[p], acc);
		copy_second_half_where(leads, snap[p], acc);
		}
	};

	if constexpr (PIPE) {
		const float* norms = lds + (size_t)w.chunk_tiles * TF;
		const uint32_t tiles = all_tiles;
		struct Ops { f16x8 c[KB]; };
		auto fetch = [&](Ops& o, uint32_t tile) {
#pragma unroll
			for (int kb = 0; kb < KB; ++kb) o.c[kb] = operand(lds, tile, kb);
		};
		auto multiply = [&](f32x16 (&acc)[P], const Ops& o) { /* acc[0] holds the tile's norms: they start every accumulator, acc[0] itself last */
#pragma unroll
			for (int kb = 0; kb < KB; ++kb)
#pragma unroll
				for (int p = P - 1; p >= 0; --p) acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(o.c[kb], b[p][kb], kb == 0 ? acc[0] : acc[p], 0, 0, 0);
		};
		auto sweep = [&]() {
			start();
			f32x16 acc0[P], acc1[P];
			constexpr int MFMAS = KB * P, SLOTS = KB;
			constexpr int SNAP_OPS = 12 + SNAP_ROWS / 2;
			constexpr int OPS_PER_SLOT = (SNAP_OPS + SLOTS - 1) / SLOTS;
			/* one step: tile t_new into acc_new (which holds its norms), the tile after it requested, the tile in acc_old tracked in
			 * pieces behind the matrix instructions, then the norms of the tile after next into acc_old */
			auto step = [&](Ops& fetch_into, uint32_t t_new, f32x16 (&acc_new)[P], const Ops& use, f32x16 (&acc_old)[P], uint32_t tile_old) {
				fetch(fetch_into, min(t_new + 1, tiles - 1));
				__builtin_amdgcn_sched_barrier(0);
				float lowest[P];
				uint64_t leads[P];
				auto op = [&](int p, int u) {
					const f32x16& a = acc_old[p];
					if (u == 0) lowest[p] = lowest_of(a[0], a[1]);
					else if (u < 8) lowest[p] = lowest_of(lowest_of(lowest[p], a[2 * u]), a[2 * u + 1]);
					else if (u == 8) m2[p] = __builtin_amdgcn_fmed3f(m1[p], m2[p], lowest[p]);
					else if (u == 9) leads[p] = settled_mask(tile_old == 0 ? ~0ull : __builtin_amdgcn_ballot_w64(lowest[p] < m1[p]));
					else if (u == 12) take_lead_where(leads[p], m1[p], leader[p], lowest[p], tile_old, snap[p], a);
					else if (u == 16) copy_second_half_where(leads[p], snap[p], a);
				};
				int issued = 0;
#pragma unroll
				for (int kb = 0; kb < KB; ++kb)
#pragma unroll
					for (int p = P - 1; p >= 0; --p) {
						acc_new[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(use.c[kb], b[p][kb], kb == 0 ? acc_new[0] : acc_new[p], 0, 0, 0);
						__builtin_amdgcn_sched_barrier(0);
						const int tp = issued / SLOTS, first_op = (issued % SLOTS) * OPS_PER_SLOT;
#pragma unroll
						for (int u = first_op; u < first_op + OPS_PER_SLOT; ++u)
							if (u < SNAP_OPS) op(tp, u);
						__builtin_amdgcn_sched_barrier(0);
						if (issued == SLOTS - 1 || MFMAS == 1) { /* acc_old[0] has been tracked */
							fetch_norms(acc_old[0], norms, min(t_new + 1, tiles - 1), h);
							__builtin_amdgcn_sched_barrier(0);
						}
						++issued;
					}
			};
			Ops o0, o1;
			fetch(o0, 0);
			fetch_norms(acc0[0], norms, 0, h);
			fetch(o1, min(1u, tiles - 1));
			fetch_norms(acc1[0], norms, min(1u, tiles - 1), h);
			multiply(acc0, o0);
			uint32_t t = 0; /* acc0 holds tile t, not yet tracked; o1 and acc1[0] hold the operands and norms of tile t + 1 */
			while (t + 2 < tiles) {
				step(o0, t + 1, acc1, o1, acc0, t);
				step(o1, t + 2, acc0, o0, acc1, t + 1);
				t += 2;
			}
			if (t + 1 < tiles) {
				multiply(acc1, o1);
#pragma unroll
				for (int p = 0; p < P; ++p) track(acc0[p], p, t);
#pragma unroll
				for (int p = 0; p < P; ++p) track(acc1[p], p, t + 1);
			}
			else {
#pragma unroll
				for (int p = 0; p < P; ++p) track(acc0[p], p, t);
			}
		};
		const uint32_t items_all = (w.n + P * TILE - 1) / (P * TILE);
		const uint32_t item0 = (uint32_t)((uint64_t)blockIdx.x * items_all / gridDim.x), item1 = (uint32_t)((uint64_t)(blockIdx.x + 1) * items_all / gridDim.x);
		const uint32_t items = item1 - item0;
		auto claim = [&]() -> uint32_t {
			uint32_t item = 0;
			if (lane == 0) item = atomicAdd(&claimed, 1u);
			return item;
		};
		auto uniform = [&](uint32_t v) -> uint32_t { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); };
		auto first_point = [&](uint32_t item) -> uint32_t { return (item0 + item) * (P * TILE); };
		uint32_t item = uniform(claim());
		if constexpr (PREFETCH) {
			float raw[P][KB][8];
			auto request = [&](uint32_t first) {
#pragma unroll
				for (int p = 0; p < P; ++p)
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) {
						rank16_request<LD>(raw[p][kb], w.data, w.stride, min(first + p * TILE + col, w.n - 1), kb, h, w.dim);
					}
			};
			auto convert = [&](uint32_t first) {
#pragma unroll
				for (int p = 0; p < P; ++p) {
					xx[p] = 0.0f; xl[p] = 0.0f;
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) {
						rank16_copy<LD>(w, raw[p][kb], first + p * TILE + col, kb * KBLOCK + h * 8);
						rank16_convert(b[p][kb], raw[p][kb], frame + kb * KBLOCK + h * 8, scale, xx[p], xl[p]);
					}
				}
			};
			uint32_t next = uniform(claim());
			if (item < items) { request(first_point(item)); convert(first_point(item)); }
			while (item < items) {
				const uint32_t after = claim();
				if (next < items) request(first_point(next));
				sweep();
				finish(first_point(item));
				item = next;
				next = uniform(after);
				if (item < items) convert(first_point(item));
			}
		}
		else {
			while (item < items) {
				const uint32_t after = claim();
				load_points(first_point(item));
				sweep();
				finish(first_point(item));
				item = uniform(after);
			}
		}
	}
	else {
		/* one chain of KB instructions per tile and point tile; the operands of block kb + AHEAD are requested before the instructions of block kb */
		constexpr int AHEAD = 2;
		constexpr uint32_t PIECES = (TF / 4 + RANK16_THREADS - 1) / RANK16_THREADS; /* 16-byte pieces per lane that cover one tile */
		const uint32_t units = (w.n + RANK16_WAVES * P * TILE - 1) / (RANK16_WAVES * P * TILE);
		for (uint32_t unit = blockIdx.x; unit < units; unit += gridDim.x) {
			const uint32_t first = (unit * RANK16_WAVES + wave) * (P * TILE);
			load_points(first);
			start();
			for (uint32_t chunk = 0; chunk < chunks; ++chunk) {
				const uint32_t tile0 = chunk * w.chunk_tiles, tiles = min(w.chunk_tiles, all_tiles - tile0);
				const uint32_t next_tile0 = chunk + 1 < chunks ? tile0 + w.chunk_tiles : 0, next_tiles = min(w.chunk_tiles, all_tiles - next_tile0);
				const float* here = lds + (size_t)cur * buffer_floats;
				const float* norms = here + (size_t)w.chunk_tiles * TF;
				const f32x4* src = (const f32x4*)w.packed + (size_t)next_tile0 * (TF / 4);
				const f32x4* nsrc = (const f32x4*)(w.norms + (size_t)next_tile0 * NORM_TILE);
				f32x4* dst = (f32x4*)(lds + (size_t)(cur ^ 1u) * buffer_floats);
				f32x4* ndst = (f32x4*)(lds + (size_t)(cur ^ 1u) * buffer_floats + (size_t)w.chunk_tiles * TF);
				const uint32_t last_vec = next_tiles * (TF / 4) - 1, norm_vec = min(tid, next_tiles * (NORM_TILE / 4) - 1);
				uint32_t piece = tid;
				for (uint32_t t = 0; t < tiles; ++t) {
					f32x4 pv[PIECES], nv;
					if constexpr (STREAM) {
#pragma unroll
						for (uint32_t i = 0; i < PIECES; ++i) pv[i] = src[min(piece + i * RANK16_THREADS, last_vec)];
						nv = nsrc[norm_vec];
					}
					f32x16 acc[P];
					fetch_norms(acc[0], norms, t, h);
#pragma unroll
					for (int p = 1; p < P; ++p) acc[p] = acc[0];
					f16x8 c[KB];
#pragma unroll
					for (int kb = 0; kb < AHEAD && kb < KB; ++kb) c[kb] = operand(here, t, kb);
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) {
						if (kb + AHEAD < KB) c[kb + AHEAD] = operand(here, t, kb + AHEAD);
#pragma unroll
						for (int p = 0; p < P; ++p) acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(c[kb], b[p][kb], acc[p], 0, 0, 0);
					}
					__builtin_amdgcn_sched_group_barrier(0x020, STREAM ? PIECES + 1 : 0, 0);
					__builtin_amdgcn_sched_group_barrier(0x100, 4 + (AHEAD < KB ? AHEAD : KB), 0);
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) {
						__builtin_amdgcn_sched_group_barrier(0x008, P, 0);
						if (kb + AHEAD < KB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
					}
#pragma unroll
					for (int p = 0; p < P; ++p) track(acc[p], p, tile0 + t);
					if constexpr (STREAM) {
#pragma unroll
						for (uint32_t i = 0; i < PIECES; ++i) dst[min(piece + i * RANK16_THREADS, last_vec)] = pv[i];
						ndst[norm_vec] = nv;
						piece += PIECES * RANK16_THREADS;
					}
				}
				if constexpr (STREAM) {
					/* a short chunk has fewer steps than the next one has tiles: the remaining pieces */
					for (; piece - tid <= last_vec; piece += PIECES * RANK16_THREADS) {
#pragma unroll
						for (uint32_t i = 0; i < PIECES; ++i) {
							const uint32_t at = min(piece + i * RANK16_THREADS, last_vec);
							dst[at] = src[at];
						}
					}
					__syncthreads();
					cur ^= 1u;
				}
			}
			finish(first);
		}
	}
	/* what is left in the lists: one addition per work-group (one per wavefront took 12 us of a launch: 2048 of them to one address) */
	__syncthreads();
	if (lane == 0) wave_max[0][wave] = flagged;
	__syncthreads();
	uint32_t before = 0, all = 0;
#pragma unroll
	for (uint32_t v = 0; v < RANK16_WAVES; ++v) {
		before += v < wave ? wave_max[0][v] : 0u;
		all += wave_max[0][v];
	}
	if (all == 0) return;
	if (tid == 0) wave_max[1][0] = atomicAdd(w.length, all);
	__syncthreads();
	const size_t slot = 2 * (size_t)(wave_max[1][0] + before);
	for (uint32_t i = lane; i < 2 * flagged; i += WAVE) w.list[slot + i] = flag_list[wave][i];
}

template <int KB>
static int launch_rank16_kb(const AssignArgs& a, Rank16Args w, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	const uint32_t budget = lds_budget_of(exec, dev), static_bytes = rank16_static_bytes<KB>();
	const uint32_t tile_bytes = (rank16_tile_floats<KB>() + NORM_TILE) * 4;
	if (budget < static_bytes + 2 * tile_bytes) return fail(KMX_ERR_UNSUPPORTED, "assign (half-precision sweep): LDS budget of %u bytes is too small", budget);
	const uint32_t tiles = w.kp / TILE, fit = (budget - static_bytes) / tile_bytes;
	const bool stream_mode = tiles > fit;
	w.chunk_tiles = stream_mode ? std::min(fit / 2, RANK16_THREADS * 4 / NORM_TILE) : tiles;
	const uint32_t lds_bytes = (stream_mode ? 2 : 1) * w.chunk_tiles * tile_bytes;
	void (*kernel)(Rank16Args) = a.layout == KMX_AOS ? (stream_mode ? rank16_kernel<KB, KMX_AOS, true> : rank16_kernel<KB, KMX_AOS, false>)
	                                                 : (stream_mode ? rank16_kernel<KB, KMX_SOA, true> : rank16_kernel<KB, KMX_SOA, false>);
	const bool pipe = !stream_mode && KB <= 4;
	const uint32_t unit = (pipe ? 1 : RANK16_WAVES) * RANK16_P * TILE;
	const uint32_t grid = std::min((a.n + unit - 1) / unit, dev.compute_units);
	exec->block_count = grid;
#define KMX_PLAN(cond) do { if (!(cond)) return fail(KMX_ERR_DEVICE, "assign (half-precision sweep): launch refused, the plan breaks \"%s\" (dim %u, k %u, kp %u, n %u, chunk tiles %u, LDS %u)", \
	#cond, a.dim, a.k, w.kp, a.n, w.chunk_tiles, lds_bytes); } while (0)
	if (!sizing_only()) {
		KMX_PLAN(w.kp % TILE == 0 && w.kp >= a.k && w.kp - a.k < TILE && a.n >= 1 && KB * KBLOCK >= a.dim);
		KMX_PLAN(w.chunk_tiles >= 1 && (uint64_t)lds_bytes + static_bytes <= dev.lds_bytes && rank16_tile_floats<KB>() % 4 == 0);
		KMX_PLAN(ws->packed16 && (size_t)tiles * KB * WAVE * 4 <= ws->packed16_cap);
		KMX_PLAN(a.layout == KMX_AOS || (w.copies && w.copy_stride % 8 == 0 && w.copy_stride >= a.dim && w.copy_stride <= KB * KBLOCK && (size_t)a.n * w.copy_stride <= ws->queued_rows_cap));
		KMX_PLAN(w.list && w.length && w.norms && w.low2 && w.frame && w.scale);
	}
#undef KMX_PLAN
	KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
	KMX_LAUNCH_KERNEL(kernel, dim3(grid), dim3(RANK16_THREADS), lds_bytes, stream(), w);
	KMX_LAUNCH_CHECK("rank16_kernel");
	return KMX_OK;
}

} // namespace kmx

#endif
