/*
 * The ranking sweep on half-precision operands: a[j] = |c_j|^2 - 2 c_j . x, one v_mfma_f32_32x32x16_f16 per 16 dimensions and tile of
 * 32 x 32, for every point; what it cannot settle is listed. Device code, instantiated per row width (rank16_inst.hip); the design
 * and the launch rules are in rank16.hip.
 */
#ifndef KMX_RANK16_IMPL_H
#define KMX_RANK16_IMPL_H

#include "assign_bf16_impl.h"
#include "rank16_columns.h"

namespace kmx {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

/* SoA: which rows go out as AoS (copy_listed, rank16_copy): the listed points', or all of them; AoS: none */
enum Rank16Copies { RANK16_NONE, RANK16_LISTED, RANK16_ALL };

/*
 * Rows of up to 32 dimensions around resident centroids: three wavefronts on a SIMD, of which the third also covers the ends of the others'
 * sweeps. That takes tracking in fewer registers (RANK16_GROUPS). us per assignment (N = 2M, Gaussian mixture, centroids after two rounds), two wavefronts with
 * the snapshot -> three: d = 32, k = 1024 219 -> 204; d = 16 174 -> 150; d = 10, k = 100 74 -> 70. The same tracking with two: 220, 165, 78. Wider rows
 * would spill (N = 1M, d = 64, k = 512: 103 -> 114). SoA: d = 32, k = 1024 225 -> 215, around its first points 246 -> 230; N = 1M, d = 20, k = 300 70 -> 68.
 */
constexpr bool rank16_grouped(uint32_t kb) { return kb <= 2; }
/*
 * Wavefronts of a work-group: otherwise eight around centroids in LDS. Where the centroids stream by (slots of a chunk of tiles that go round, filled by
 * requests straight to LDS, a barrier per chunk), rows of up to 128 dimensions keep that form with two chunks as large as fit, since the
 * barriers are what costs (us per assignment, two work-groups of four wavefronts with four slots of 32 matrix instructions -> this: N = 2M,
 * d = 128, k = 1024 659 -> 627; N = 1M, d = 96, k = 2000 493 -> 440; d = 64, k = 3000 473 -> 424). Wider rows have a barrier's worth of matrix
 * instructions in a single tile: two work-groups of four wavefronts on a compute unit, one of which reads its points while the other has
 * the matrix cores, and four slots of a tile (N = 1M, d = 256, k = 1024: 549, with eight wavefronts and two chunks of four tiles 569).
 * With chunks through registers and eight wavefronts for all widths: 656, 655, 480, 464.
 */
constexpr uint32_t rank16_waves(uint32_t kb, bool stream) { return stream && kb >= 12 ? 4 : !stream && rank16_grouped(kb) ? 12 : 8; }
constexpr int RANK16_P = 2; /* point tiles per wavefront: an operand read serves two instructions */

struct Rank16Args {
	const float* data; size_t stride;
	const f16x8* packed;   /* per tile and block of 16 dimensions the 64 lanes' operands of -2 S (c - m), 16 bytes each */
	const float* norms;    /* tiles of S^2 |c - m|^2 */
	const float* low2;     /* per padded row the squared norm of what the half-precision parts leave out */
	const float* frame;    /* m */
	float* scale;          /* S, 1 / S^2; the first work-group puts the maxima of the norms and of the bf16 mid and rest parts behind them */
	uint32_t* assignment; uint32_t* list; uint32_t* length;
	float* copies; uint32_t copy_stride; /* SoA: the rows as AoS, zeros behind the coordinates */
	bool copy_all;         /* of all points, else of the listed ones */
	uint32_t dim, k, kp, n, chunk_tiles;
	float kd;
	uint32_t list_entries; /* of a wavefront's list, resident centroids */
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
/*
 * Listed points a wavefront keeps in LDS before they go out, 32 of a tile at most at a time. Going out is an addition to one word in memory, of which
 * the card makes one in 5.3 ns: where nearly every point is listed (coordinates that are all 0 or 1) that bounds the launch (N = 1M, d = 16, k = 256:
 * 156 us a call with lists of 80, which go out at 64; 125 with 128). Around resident centroids the lists take what the centroids leave of LDS, up to 128.
 */
constexpr uint32_t RANK16_LIST_STREAMED = 120, RANK16_LIST_MOST = 128;
/* the least, before the centroids stream by instead. Rows of more than 128 dimensions are no slower that way (N = 262144, d = 256, k = 285, SoA: 177
 * streamed, 193 resident, where the registers do not hold everything), rows of up to 128 are (d = 40, k = 1500, SoA: 86, 79) */
constexpr uint32_t rank16_list_least(uint32_t kb) { return kb >= 12 ? 120 : 64; }
constexpr uint32_t rank16_slots(uint32_t kb) { return kb >= 12 ? 4 : 2; }
__host__ __device__ constexpr uint32_t rank16_norm_blocks(uint32_t tiles) { return (tiles * NORM_TILE + WAVE - 1) / WAVE; }
/* what a chunk takes in LDS, its norms behind its operands as whole requests of 64 words */
__host__ __device__ constexpr uint32_t rank16_slot_bytes(uint32_t kb, uint32_t tiles) { return tiles * kb * WAVE * 16 + rank16_norm_blocks(tiles) * WAVE * 4; }
/*
 * SoA points requested 64 of a column at a time instead of 32 of two columns, from scalar addresses (rank16_request_columns): 128 dimensions, where eight wavefronts
 * wait for points between streams of centroids, and 256, whose registers hold no vector addresses beside the operands. us per assignment,
 * N = 2M, d = 128, k = 1024 738 -> 693 (9 % listed 816 -> 782; addresses kept 795); N = 400000, d = 250, k = 130 357 -> 213; N = 262144, d = 256, k = 285 147 -> 133;
 * but N = 500000, d = 200, k = 1024 330 -> 334; N = 1M, d = 90, k = 300 157 -> 161; d = 40, k = 200 77 -> 81; N = 2M, d = 32, k = 1024 225 -> 230.
 */
constexpr bool rank16_whole_columns(uint32_t kb, int layout) { return layout == KMX_SOA && (kb == 8 || kb == 16); }
constexpr uint32_t RANK16_EXCHANGE = 256; /* words per wavefront in which the lanes exchange a block of a tile of points */
constexpr bool rank16_shared_rows(uint32_t kb, int layout) { return layout == KMX_AOS && kb >= 12; }
constexpr uint32_t rank16_exchange(uint32_t kb, int layout, Rank16Copies copies) { return rank16_shared_rows(kb, layout) || copies == RANK16_ALL ? RANK16_EXCHANGE : 0; }
constexpr uint32_t rank16_static_bytes(uint32_t kb, int layout, bool stream, Rank16Copies copies) { return ((2 * (stream ? RANK16_LIST_STREAMED : 0) + rank16_exchange(kb, layout, copies) + 4) * rank16_waves(kb, stream) + kb * KBLOCK) * 4 + 64; }
/* the lists of a work-group around resident centroids, lying behind them */
constexpr uint32_t rank16_list_bytes(uint32_t kb, uint32_t entries) { return rank16_waves(kb, false) * entries * 8; }
constexpr uint32_t rank16_least_bytes(uint32_t kb, int layout) { return rank16_static_bytes(kb, layout, true, layout == KMX_SOA ? RANK16_ALL : RANK16_NONE) + rank16_slots(kb) * rank16_slot_bytes(kb, 1); }

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

/*
 * How the coordinates come from memory. AoS: four lanes take 64 consecutive bytes of a row, lane 4 r + q the piece q (four coordinates) of
 * rows r and 16 + r of the tile, and the rounded values go through LDS to the lanes that hold them as operands: a lane per row would make
 * every 16 bytes an access of their own to the vector cache, 64 a load instead of 16 (N = 1M, d = 256, k = 1024: 104 M accesses a launch,
 * the cache busy for half of it). SoA: lane (col, h) takes eight coordinates of point col, which are its operand.
 * Without branches, so that many blocks travel together: blocks that the row does not fill (ragged rows only) read what lies inside it, and
 * rank16_place puts that into its places. WHOLE: no such blocks.
 */
struct Rank16Source { const float* row[2]; }; /* AoS: the lane's two rows; SoA: row[0], the lane's point at coordinate 0 */

template <int LD, bool SHARED>
__device__ __forceinline__ Rank16Source rank16_source(const float* __restrict__ data, size_t stride, uint32_t tile_first, uint32_t n, uint32_t lane)
{
	if (!SHARED) return Rank16Source{ { data + (size_t)min(tile_first + lane % TILE, n - 1) * (LD == KMX_AOS ? stride : 1), nullptr } }; /* rows beyond the points repeat the last one */
	return Rank16Source{ { data + (size_t)min(tile_first + lane / 4, n - 1) * stride, data + (size_t)min(tile_first + 16 + lane / 4, n - 1) * stride } };
}

template <int LD, bool SHARED, bool WHOLE>
__device__ __forceinline__ void rank16_request(float (&v)[8], const Rank16Source& from, size_t stride, uint32_t kb, uint32_t lane, uint32_t dim)
{
	typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));
	if (LD == KMX_AOS) {
		const uint32_t d = kb * KBLOCK + (SHARED ? lane % 4 * 4 : lane / TILE * 8), at = WHOLE ? d : min(d, dim - 4), at2 = SHARED ? at : WHOLE ? d + 4 : min(d + 4, dim - 4);
		const f32x4 lo = *(const f32x4_any*)(from.row[0] + at), up = *(const f32x4_any*)(from.row[SHARED] + at2);
		v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w; v[4] = up.x; v[5] = up.y; v[6] = up.z; v[7] = up.w;
	}
	else {
		asm volatile("" : "+v"(lane)); /* (addresses are formed here: 64 of them kept for the next tile of points would be spilled) */
		const uint32_t d0 = kb * KBLOCK + lane / TILE * 8;
		const float* src = from.row[0] + (size_t)(WHOLE ? d0 : min(d0, dim - 1)) * stride;
#pragma unroll
		for (uint32_t j = 0; j < 8; ++j) {
			v[j] = *src;
			src += WHOLE || d0 + j + 1 < dim ? stride : 0;
		}
	}
}

/*
 * SoA, both tiles of a wavefront's 64 points: lane l requests point l's coordinates j and 8 + j of block kb, 256 consecutive bytes of a column each, from an
 * address that is the same for all lanes, and the half-waves change places (rank16_halves). `inside`: the lane's point, from rank16_column_base on; `column`: that
 * point's coordinate 0. FRESH: addresses are formed here and not kept (spilled) from one unit of points to the next.
 */
template <bool WHOLE, bool FRESH>
__device__ __forceinline__ void rank16_request_columns(float (&low)[8], float (&high)[8], const float* column, size_t stride, uint32_t inside, uint32_t kb, uint32_t dim)
{
	const uint32_t d0 = kb * KBLOCK;
	if (FRESH) asm volatile("" : "+s"(stride));
	const float* at = column + (size_t)(WHOLE ? d0 : min(d0, dim - 1)) * stride;
#pragma unroll
	for (uint32_t j = 0; j < 16; ++j) {
		(j < 8 ? low : high)[j % 8] = *(const float*)((const char*)at + inside * 4u);
		at += WHOLE || d0 + j + 1 < dim ? stride : 0;
	}
}
/* the requested coordinates as the two tiles' (first tile's to v0), zeros behind the row */
__device__ __forceinline__ void rank16_halves(float (&v0)[8], float (&v1)[8], uint32_t kb, uint32_t dim)
{
	const bool whole = (kb + 1) * KBLOCK <= dim;
#pragma unroll
	for (uint32_t j = 0; j < 8; ++j) {
		if (!whole) {
			v0[j] = kb * KBLOCK + j < dim ? v0[j] : 0.0f;
			v1[j] = kb * KBLOCK + 8 + j < dim ? v1[j] : 0.0f;
		}
		const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v0[j]), __float_as_uint(v1[j]), false, false);
		v0[j] = __uint_as_float(r[0]);
		v1[j] = __uint_as_float(r[1]);
	}
}

/* ragged rows: zeros behind the row (AoS: rows of at least 4 coordinates, pieces that end behind the row have been read up to its end) */
template <int LD, bool SHARED>
__device__ __forceinline__ void rank16_place(float (&v)[8], uint32_t kb, uint32_t lane, uint32_t dim)
{
	if ((kb + 1) * KBLOCK <= dim) return; /* (the same for all lanes) */
	if (LD == KMX_AOS) {
#pragma unroll
		for (uint32_t q = 0; q < 8; q += 4) {
			const uint32_t beyond = max(kb * KBLOCK + (SHARED ? lane % 4 * 4 : lane / TILE * 8 + q) + 4, dim) - dim; /* coordinates of the piece behind the row */
			const float x = v[q], y = v[q + 1], z = v[q + 2], t = v[q + 3];
			v[q] = beyond == 0 ? x : beyond == 1 ? y : beyond == 2 ? z : beyond == 3 ? t : 0.0f;
			v[q + 1] = beyond == 0 ? y : beyond == 1 ? z : beyond == 2 ? t : 0.0f;
			v[q + 2] = beyond == 0 ? z : beyond == 1 ? t : 0.0f;
			v[q + 3] = beyond == 0 ? t : 0.0f;
		}
	}
	else {
		const uint32_t d0 = kb * KBLOCK + lane / TILE * 8;
#pragma unroll
		for (uint32_t j = 0; j < 8; ++j) v[j] = d0 + j < dim ? v[j] : 0.0f;
	}
}

__device__ __forceinline__ void rank16_exchanged() /* LDS keeps the order of a wavefront's requests; the compiler has to as well */
{
	__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
	__builtin_amdgcn_wave_barrier();
}

/*
 * SoA: rows go out as AoS, for the exact pass (coordinates of a listed point lie a cache line each apart) and whatever else reads single rows: those of the
 * listed points, behind the sweep (LISTED, see copy_listed in the kernel). Writing as many bytes as are read, in the phase in which
 * the matrix cores wait for the points, cost more than reading the columns' lines of the listed points once more from the memory-side
 * cache. us per assignment, all rows -> listed ones: N = 2M, d = 128, k = 1024, 9 % listed 854 -> 812 (without any copies 643), 1 % 808 -> 732; d = 32
 * 256 -> 222; N = 1M, d = 64, k = 500 162 -> 119; d = 90, k = 300 222 -> 157; N = 500000, d = 200, k = 1024 392 -> 331; nearly all listed (coordinates 0 or 1),
 * d = 64, k = 256 145 -> 89, d = 128, k = 512 193 -> 189; 950 calls of 3000 to 300000 points and 24 to 256 dimensions 0.98 in the mean, 0.82 to 1.06, dearest where points that come
 * together are listed and a work-group has no further points meanwhile (N = 52692, d = 237, k = 300, uniform points 61 -> 64).
 * All of them (ALL), on the way in and through LDS, so that four lanes store 64 consecutive bytes of a row, where the update behind it reads whole rows: iterations
 * with more centroids than fit a column's sums. `exchange`: RANK16_EXCHANGE words of this wavefront's. Otherwise a lane stores its 32 bytes as they are.
 */
template <bool EXCHANGED>
__device__ __forceinline__ void rank16_copy(const Rank16Args& w, const float (&v)[8], uint32_t tile_first, uint32_t kb, uint32_t lane, float* exchange)
{
	if (!EXCHANGED) {
		const uint32_t pt = tile_first + lane % TILE, d = kb * KBLOCK + lane / TILE * 8;
		if (pt >= w.n || d >= w.copy_stride) return;
		float* to = w.copies + (size_t)pt * w.copy_stride + d;
		*(f32x4*)to = f32x4{ v[0], v[1], v[2], v[3] };
		*(f32x4*)(to + 4) = f32x4{ v[4], v[5], v[6], v[7] };
		return;
	}
	/* half of the tile at a time, 16 words a row in pieces of four; row r's piece q lies in the place q ^ (r / 2 % 4) of the row, which spreads a
	 * column over the banks */
	const uint32_t col = lane % TILE, h = lane / TILE, turn = col / 2 % 4, row = lane / 4, d = kb * KBLOCK + lane % 4 * 4;
#pragma unroll
	for (uint32_t half = 0; half < 2; ++half) {
		rank16_exchanged();
		if (col / 16 == half) {
			float* to = exchange + col % 16 * 16;
			*(f32x4*)(to + ((2 * h) ^ turn) * 4) = f32x4{ v[0], v[1], v[2], v[3] };
			*(f32x4*)(to + ((2 * h + 1) ^ turn) * 4) = f32x4{ v[4], v[5], v[6], v[7] };
		}
		rank16_exchanged();
		const f32x4 piece = *(const f32x4*)(exchange + row * 16 + ((lane % 4) ^ (row / 2 % 4)) * 4);
		const uint32_t pt = tile_first + half * 16 + row;
		if (pt < w.n && d < w.copy_stride) *(f32x4*)(w.copies + (size_t)pt * w.copy_stride + d) = piece;
	}
}

/* four coordinates v = S (x - m) rounded once (S is a power of two), in half precision, and their shares of |v|^2 and of the squared norm of
 * what half precision leaves out; m: S times the frame */
__device__ __forceinline__ void rank16_round(f16x2 (&out)[2], const float* raw, const f32x4& m, float scale, float& part, float& low)
{
	float minus_one = -1.0f;
	asm("" : "+s"(minus_one));
#pragma unroll
	for (int j = 0; j < 4; j += 2) {
		const float v0 = __builtin_fmaf(raw[j], scale, -m[j]), v1 = __builtin_fmaf(raw[j + 1], scale, -m[j + 1]);
		f16x2 pair = { (_Float16)v0, (_Float16)v1 };
		asm("" : "+v"(pair)); /* (the halves are read from the pair from here on: left alone the compiler rounds again for each use) */
		const float r0 = __builtin_fmaf((float)pair.x, minus_one, v0), r1 = __builtin_fmaf((float)pair.y, minus_one, v1); /* (one instruction each) */
		part = __builtin_fmaf(v0, v0, part);
		part = __builtin_fmaf(v1, v1, part);
		low = __builtin_fmaf(r0, r0, low);
		low = __builtin_fmaf(r1, r1, low);
		out[j / 2] = pair;
	}
}

/* what a lane sums up while it converts: AoS: of its two rows; SoA: of its eight coordinates of each block (the second entry stays zero) */
struct Rank16Sums { float part[2], low[2]; };

/* block kb of a tile of points as this lane's operand; frame: S m, in LDS */
template <bool SHARED>
__device__ __forceinline__ void rank16_convert(f16x8& b, const float (&raw)[8], const float* frame, float scale, uint32_t kb, uint32_t lane, Rank16Sums& sums, float* exchange)
{
	union { f16x8 all; f16x2 two[4]; } h;
	if (SHARED) {
		const f32x4 m = *(const f32x4*)(frame + kb * KBLOCK + lane % 4 * 4);
		f16x2* to = (f16x2*)exchange + 2 * lane;
		rank16_exchanged();
#pragma unroll
		for (int half = 0; half < 2; ++half) {
			union { f16x2 two[2]; uint2 all; } piece;
			rank16_round(piece.two, raw + 4 * half, m, scale, sums.part[half], sums.low[half]);
			*(uint2*)(to + 2 * WAVE * half) = piece.all; /* row 16 half + lane / 4, 32 bytes a row */
		}
		rank16_exchanged();
		b = *(const f16x8*)((const f16x2*)exchange + lane % TILE * 8 + lane / TILE * 4);
	}
	else {
#pragma unroll
		for (int half = 0; half < 2; ++half) {
			f16x2 two[2];
			rank16_round(two, raw + 4 * half, *(const f32x4*)(frame + kb * KBLOCK + lane / TILE * 8 + 4 * half), scale, sums.part[0], sums.low[0]);
			h.two[2 * half] = two[0]; h.two[2 * half + 1] = two[1];
		}
		b = h.all;
	}
}

/* SHARED: the sums of point lane % 32 of the tile, from the lanes that share its row; otherwise the two half-waves have a part each, which
 * rank16_whole adds up (at the end of a sweep, where nothing waits for it) */
template <bool SHARED>
__device__ __forceinline__ void rank16_total(float& x2, float& low2, const Rank16Sums& sums, uint32_t lane)
{
	if (!SHARED) { x2 = sums.part[0]; low2 = sums.low[0]; return; }
	float all[2];
#pragma unroll
	for (int q = 0; q < 2; ++q) {
		float a = q ? sums.low[0] : sums.part[0], c = q ? sums.low[1] : sums.part[1];
		a += __shfl_xor(a, 1); c += __shfl_xor(c, 1);
		a += __shfl_xor(a, 2); c += __shfl_xor(c, 2);
		const float first = __shfl(a, (int)(lane % 16 * 4)), second = __shfl(c, (int)(lane % 16 * 4));
		all[q] = lane % TILE < 16 ? first : second;
	}
	x2 = all[0]; low2 = all[1];
}
template <bool SHARED> __device__ __forceinline__ float rank16_whole(float sum) { return SHARED ? sum : sum + __shfl_xor(sum, 32); }

__device__ __forceinline__ uint32_t rank16_uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ const void* rank16_uniform(const void* p)
{
	const uint64_t v = (uint64_t)p;
	return (const void*)((uint64_t)rank16_uniform((uint32_t)(v >> 32)) << 32 | rank16_uniform((uint32_t)v));
}
__device__ __forceinline__ void stage_block(const void* from, uint32_t lane, uint32_t to)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(rank16_uniform(to)), "v"(lane * 16), "s"(rank16_uniform(from)) : "m0");
}
__device__ __forceinline__ void stage_words(const void* from, uint32_t lane, uint32_t to)
{
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(rank16_uniform(to)), "v"(lane * 4), "s"(rank16_uniform(from)) : "m0");
}
/* all but the last LATER requests of this wavefront have arrived (requests of other kinds among them make it wait longer, never shorter) */
template <uint32_t LATER> __device__ __forceinline__ void staged_but() { asm volatile("s_waitcnt vmcnt(%0)" : : "n"(LATER) : "memory"); }

/*
 * rank16_grouped: of the leading tile's 16 results only the minima of six groups are kept (the instructions that find the tile's minimum
 * produce them on the way), and the winning group's three centroids are looked at again at the end. Results of groups 0 to 3: 4 i, 4 i + 1, 4 i + 2; of group 4: 3, 7, 11; of group 5: 15. As rows of a tile: */
constexpr int RANK16_GROUPS = 6;
__device__ __forceinline__ uint32_t rank16_group_row(uint32_t group) { return group < 4 ? 8 * group : group == 4 ? 3 : 27; } /* + 4 h: the first */
__device__ __forceinline__ uint32_t rank16_group_step(uint32_t group) { return group < 4 ? 1 : 8; }

/* In the lanes of `mask` (settled_mask; see take_lead_where): the smallest value so far becomes `lowest`, its tile `tile`, and the minima of the
 * tile's groups replace those kept */
__device__ __forceinline__ void take_groups_where(uint64_t mask, float& m1, uint32_t& leader, float lowest, uint32_t tile, f32x2 (&kept)[3], const f32x2 (&now)[2], float g4, float g5)
{
	uint64_t saved;
	float k4 = kept[2].x, k5 = kept[2].y;
	asm volatile("s_and_saveexec_b64 %[saved], %[mask]\n\tv_mov_b32 %[m1], %[lowest]\n\tv_mov_b32 %[leader], %[tile]\n\t"
	             "v_mov_b64 %[d0], %[s0]\n\tv_mov_b64 %[d1], %[s1]\n\tv_mov_b32 %[d4], %[s4]\n\tv_mov_b32 %[d5], %[s5]\n\ts_mov_b64 exec, %[saved]"
	             : [m1] "+v"(m1), [leader] "+v"(leader), [d0] "+v"(kept[0]), [d1] "+v"(kept[1]), [d4] "+v"(k4), [d5] "+v"(k5), [saved] "=&s"(saved)
	             : [lowest] "v"(lowest), [tile] "s"(tile), [s0] "v"(now[0]), [s1] "v"(now[1]), [s4] "v"(g4), [s5] "v"(g5), [mask] "s"(mask)
	             : "scc");
	kept[2] = f32x2{ k4, k5 };
}

/* sum + the products of eight half-precision values, one rounding each */
__device__ __forceinline__ float rank16_dot(const f16x8& c, const f16x8& x, float sum)
{
#pragma unroll
	for (int e = 0; e < 8; ++e) sum = __builtin_fmaf((float)c[e], (float)x[e], sum);
	return sum;
}

/* the sum of the two half-waves' values, without a trip through LDS */
__device__ __forceinline__ float rank16_both(float v)
{
	const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
	return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

/*
 * A work-group around centroids in LDS: all of them (STREAM = false), or slots that go round (rank16_waves). A wavefront sweeps 64 points at
 * a time. Rows of up to 64 dimensions around resident centroids: the wavefronts take items of 64 points from a counter in LDS (a SIMD
 * serves its older wavefront first: equal shares leave the younger ones sweeping alone at the end). Otherwise a work-group takes units of
 * 64 points per wavefront, its wavefronts side by side, every gridDim.x-th unit.
 *
 * What bounds the sweep of wide rows (N = 1M, d = 256, k = 1024: 505 us, 1.09 PFLOP/s): the power the matrix cores may take -- at 58 % of their
 * cycles the clock has come down to 1.73 GHz, without the points' fetches they reach 76 % at 1.51 -- and the fetches and conversions themselves.
 *
 * Tracking is the snapshot of assign_bf16_impl.h: the minimum of a lane's 16 results per tile, the two smallest minima, and the 16
 * results of the leading tile, from which the winner and the runner-up inside that tile come at the end; rank16_grouped: six minima of those.
 * Rows of up to 64 dimensions and resident centroids: two accumulator sets, the tracking of one tile in pieces behind the matrix
 * instructions of the next (the fenced step). Otherwise one chain per tile whose tracking the partner wavefront of the SIMD covers.
 */
template <int KB, int LD, bool STREAM, Rank16Copies COPIES>
__global__ void __launch_bounds__(rank16_waves(KB, STREAM) * WAVE, rank16_waves(KB, STREAM) == 12 ? 3 : 2)
rank16_kernel(const Rank16Args w)
{
	constexpr uint32_t WAVES = rank16_waves(KB, STREAM), THREADS = WAVES * WAVE;
	constexpr int P = RANK16_P;
	constexpr uint32_t TF = rank16_tile_floats<KB>();
	constexpr bool PIPE = !STREAM && KB <= 4;
	constexpr bool SHARED = rank16_shared_rows(KB, LD);
	constexpr bool GROUPED = PIPE && rank16_grouped(KB);
	constexpr bool PREFETCH = PIPE && (KB == 1 || (KB == 2 && !GROUPED)); /* the next item's coordinates travel while the current one is swept */
	extern __shared__ __attribute__((aligned(16))) float lds[];
	__shared__ __attribute__((aligned(16))) float frame[KB * KBLOCK]; /* S m */
	__shared__ uint32_t wave_max[4][WAVES];
	__shared__ uint32_t streamed_lists[STREAM ? WAVES : 1][STREAM ? 2 * RANK16_LIST_STREAMED : 1];
	__shared__ __attribute__((aligned(16))) float exchanges[WAVES][rank16_exchange(KB, LD, COPIES) ? RANK16_EXCHANGE : 1];
	uint32_t& claimed = wave_max[3][0];
	const uint32_t tid = threadIdx.x, lane = tid & (WAVE - 1);
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid / WAVE));
	const uint32_t col = lane & 31, h = lane >> 5;
	const float scale = w.scale[0], smallest = 1e-30f * (scale * scale), largest = 1e37f * (scale * scale);
	if (tid == 0) claimed = 0u;
	for (uint32_t i = tid; i < KB * KBLOCK; i += THREADS) frame[i] = w.frame[i] * scale;

	CertCoeffs cert;
	{
		uint32_t most[2] = { 0u, 0u };
		for (uint32_t j = tid; j < w.k; j += THREADS) {
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
			for (uint32_t v = 0; v < WAVES; ++v) most[q] = max(most[q], wave_max[q][v]);
		}
		if (blockIdx.x == 0) rank16_leave_bounds(w.scale, most[0], most[1], w.low2, w.k, w.kp);
		cert = cert_coeffs_level1(CentroidBounds{ __uint_as_float(most[0]), __uint_as_float(most[1]), 0.0f });
		cert.c2max = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(cert.c2max)));
		cert.a = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(cert.a)));
		cert.b = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(cert.b)));
	}

	const uint32_t all_tiles = w.kp / TILE;
	if constexpr (!STREAM) {
		const uint32_t tiles = all_tiles;
		f32x4* dst = (f32x4*)lds;
		const f32x4* src = (const f32x4*)w.packed;
		for (uint32_t i = tid; i < tiles * (TF / 4); i += THREADS) dst[i] = src[i];
		f32x4* ndst = (f32x4*)(lds + (size_t)w.chunk_tiles * TF);
		const f32x4* nsrc = (const f32x4*)w.norms;
		for (uint32_t i = tid; i < tiles * (NORM_TILE / 4); i += THREADS) ndst[i] = nsrc[i];
	}
	__syncthreads();

	const uint32_t list_entries = STREAM ? RANK16_LIST_STREAMED : w.list_entries;
	uint32_t* const flag_list = STREAM ? streamed_lists[wave] : (uint32_t*)lds + (size_t)w.chunk_tiles * (TF + NORM_TILE) + wave * 2 * list_entries;
	uint32_t flagged = 0; /* wave-uniform */
	auto flush_flags = [&]() {
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		uint32_t slot = 0;
		if (lane == 0) slot = atomicAdd(w.length, flagged);
		slot = (uint32_t)__shfl((int)slot, 0);
		for (uint32_t i = lane; i < 2 * flagged; i += WAVE) w.list[2 * (size_t)slot + i] = flag_list[i];
		__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
		__builtin_amdgcn_wave_barrier();
		flagged = 0;
	};

	/* the operands of a tile for this lane, and the norms of the 16 rows it receives */
	auto operand = [&](const float* tiles, uint32_t tile, int kb) -> f16x8 { return ((const f16x8*)(tiles + (size_t)tile * TF))[kb * WAVE + lane]; };

	f16x8 b[P][KB];
	float xx[P], xl[P]; /* of this lane's point: |v|^2 and the squared norm of what half precision leaves out (rank16_whole) */
	float* const exchange = exchanges[wave];
	float m1[P], m2[P];
	uint32_t leader[P];
	float snap[P][GROUPED ? 1 : SNAP_ROWS];
	f32x2 kept[P][RANK16_GROUPS / 2]; /* GROUPED: the minima of the leading tile's groups */

	/*
	 * RANK16_LISTED: the listed points' rows, read again once the sweep has left them: `late`, a bit for each of the 64 points from late_first on.
	 * Eight lanes a row, LATE_EACH consecutive coordinates each (in LATE_TURNS turns), so that a load touches eight columns: with a lane per
	 * column every lane had a page of its own (N = 2M, d = 128, k = 1024: 905 against 812 us a call). Up to eight
	 * rows are requested (request_listed) ahead of the next points and stored
	 * behind them (store_listed). Many of the 64: their tiles as a whole (copy_tiles).
	 */
	constexpr bool LISTED = COPIES == RANK16_LISTED;
	static_assert(COPIES == RANK16_NONE ? LD == KMX_AOS : LD == KMX_SOA && (LISTED || STREAM), "all rows go out around centroids that stream by");
	constexpr uint32_t LATE_TURNS = KB > 8 ? 2 : 1, LATE_EACH = KB * KBLOCK / 8 / LATE_TURNS, LATE_VEC = LATE_EACH % 4 == 0 ? 4 : 2, LATE_MANY = 24;
	static_assert(P == 2 && LATE_EACH % LATE_VEC == 0, "whole stores");
	uint64_t late = 0;
	uint32_t late_first = 0;
	struct Late { float v[LATE_EACH]; uint32_t point; }; /* point: 64 for none */
	auto late_rows = [&](Late& l) { /* the next eight */
		l.point = 64;
#pragma unroll
		for (uint32_t g = 0; g < 8; ++g) {
			const uint32_t bit = late ? (uint32_t)__builtin_ctzll(late) : 64u;
			late &= late - 1; /* (of zero: zero) */
			l.point = lane / 8 == g ? bit : l.point;
		}
	};
	auto request_listed = [&](Late& l, uint32_t turn) {
		uint32_t d0 = (turn * 8 + lane % 8) * LATE_EACH;
		asm volatile("" : "+v"(d0));
		if (l.point < 64) {
			const float* src = w.data + late_first + l.point + (size_t)min(d0, w.dim - 1) * w.stride;
#pragma unroll
			for (uint32_t q = 0; q < LATE_EACH; ++q) {
				l.v[q] = *src;
				src += d0 + q + 1 < w.dim ? w.stride : 0;
			}
		}
	};
	auto store_listed = [&](const Late& l, uint32_t turn) {
		uint32_t d0 = (turn * 8 + lane % 8) * LATE_EACH;
		asm volatile("" : "+v"(d0));
		if (l.point < 64) {
			float* to = w.copies + (size_t)(late_first + l.point) * w.copy_stride + d0;
#pragma unroll
			for (uint32_t q = 0; q < LATE_EACH; q += LATE_VEC) {
				typedef float Part __attribute__((ext_vector_type(LATE_VEC)));
				Part part;
#pragma unroll
				for (uint32_t e = 0; e < LATE_VEC; ++e) part[e] = d0 + q + e < w.dim ? l.v[q + e] : 0.0f;
				if (d0 + q < w.copy_stride) *(Part*)(to + q) = part;
			}
		}
	};
	auto copy_tiles = [&]() {
#pragma unroll 1
		for (uint32_t p = 0; p < P; ++p) {
			const Rank16Source from = rank16_source<LD, SHARED>(w.data, w.stride, late_first + p * TILE, w.n, lane);
#pragma unroll 1
			for (uint32_t kb = 0; kb < KB; ++kb) {
				float v[8];
				rank16_request<LD, SHARED, false>(v, from, w.stride, kb, lane, w.dim);
				rank16_place<LD, SHARED>(v, kb, lane, w.dim);
				rank16_copy<false>(w, v, late_first + p * TILE, kb, lane, exchange);
			}
		}
		late = 0;
	};
	/* copy the listed rows around what fetches the next points */
	auto copy_listed = [&](auto&& fetch_next) {
		if constexpr (LISTED) {
			if (__builtin_popcountll(late) > LATE_MANY) copy_tiles();
			const bool some = late != 0;
			Late l;
			if (some) {
				late_rows(l);
				if (LATE_TURNS > 1) {
					request_listed(l, 1);
					store_listed(l, 1);
				}
				request_listed(l, 0);
			}
			fetch_next();
			if (some) store_listed(l, 0);
			while (late) {
				late_rows(l);
#pragma unroll
				for (uint32_t turn = 0; turn < LATE_TURNS; ++turn) {
					request_listed(l, turn);
					store_listed(l, turn);
				}
			}
		}
		else fetch_next();
	};
	/* A block is converted while the next DEPTH ones are on their way. (Requesting the first of them while the unit before is swept was no gain:
	 * N = 2M, d = 128, k = 1024: 653 against 618 us, d = 96 440 against 442.) */
	constexpr int BLOCKS = P * KB, DEPTH = BLOCKS < 8 ? BLOCKS : 8;
	auto load_points_of = [&](auto whole, uint32_t first, uint32_t dim) {
		constexpr bool WHOLE = decltype(whole)::value;
		Rank16Sums sums[P];
		if constexpr (rank16_whole_columns(KB, LD)) {
			constexpr int PAIRS = 4; /* blocks of both tiles under way */
			constexpr bool FRESH = KB == 8;
			float raw[PAIRS][P][8];
			const uint32_t base = rank16_column_base(rank16_uniform(first), w.n), inside = rank16_column_inside(base, lane, w.n);
			const float* column = w.data + base;
#pragma unroll
			for (int p = 0; p < P; ++p) sums[p] = Rank16Sums{ { 0.0f, 0.0f }, { 0.0f, 0.0f } };
#pragma unroll
			for (int kb = 0; kb < PAIRS; ++kb) rank16_request_columns<WHOLE, FRESH>(raw[kb][0], raw[kb][1], column, w.stride, inside, kb, dim);
#pragma unroll
			for (int kb = 0; kb < KB; ++kb) {
				__builtin_amdgcn_sched_barrier(0);
				float (&v)[P][8] = raw[kb % PAIRS];
				rank16_halves(v[0], v[1], kb, WHOLE ? KB * KBLOCK : dim);
#pragma unroll
				for (int p = 0; p < P; ++p) {
					if (COPIES == RANK16_ALL) rank16_copy<true>(w, v[p], first + p * TILE, kb, lane, exchange);
					rank16_convert<SHARED>(b[p][kb], v[p], frame, scale, kb, lane, sums[p], exchange);
					asm volatile("" : "+v"(b[p][kb]));
					asm volatile("" : "+v"(sums[p].part[0]), "+v"(sums[p].low[0]));
				}
				__builtin_amdgcn_sched_barrier(0);
				if (kb + PAIRS < KB) rank16_request_columns<WHOLE, FRESH>(raw[kb % PAIRS][0], raw[kb % PAIRS][1], column, w.stride, inside, kb + PAIRS, dim);
			}
			__builtin_amdgcn_sched_barrier(0);
#pragma unroll
			for (int p = 0; p < P; ++p) rank16_total<SHARED>(xx[p], xl[p], sums[p], lane);
			return;
		}
		float raw[DEPTH][8];
		Rank16Source from[P];
#pragma unroll
		for (int p = 0; p < P; ++p) {
			from[p] = rank16_source<LD, SHARED>(w.data, w.stride, first + p * TILE, w.n, lane);
			sums[p] = Rank16Sums{ { 0.0f, 0.0f }, { 0.0f, 0.0f } };
		}
		auto request = [&](int at) { rank16_request<LD, SHARED, WHOLE>(raw[at % DEPTH], from[at / KB], w.stride, at % KB, lane, dim); };
#pragma unroll
		for (int at = 0; at < DEPTH; ++at) request(at);
#pragma unroll
		for (int at = 0; at < BLOCKS; ++at) {
			const int p = at / KB, kb = at % KB;
			__builtin_amdgcn_sched_barrier(0);
			float (&v)[8] = raw[at % DEPTH];
			if (!WHOLE) rank16_place<LD, SHARED>(v, kb, lane, dim);
			if (COPIES == RANK16_ALL) rank16_copy<true>(w, v, first + p * TILE, kb, lane, exchange);
			rank16_convert<SHARED>(b[p][kb], v, frame, scale, kb, lane, sums[p], exchange);
			if (!SHARED) asm volatile("" : "+v"(b[p][kb]));
			/* the sums exist here: left alone the compiler moves them behind the sweep and keeps the coordinates alive */
			asm volatile("" : "+v"(sums[p].part[0]), "+v"(sums[p].part[1]), "+v"(sums[p].low[0]), "+v"(sums[p].low[1]));
			__builtin_amdgcn_sched_barrier(0);
			if (at + DEPTH < BLOCKS) request(at + DEPTH);
		}
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int p = 0; p < P; ++p) rank16_total<SHARED>(xx[p], xl[p], sums[p], lane);
	};
	auto load_points = [&](uint32_t first) {
		uint32_t dim = w.dim;
		asm volatile("" : "+v"(dim)); /* (the comparisons with it are not kept from one item to the next: they are as many as scalar registers) */
		dim = (uint32_t)__builtin_amdgcn_readfirstlane((int)dim);
		if (dim == KB * KBLOCK) load_points_of(std::true_type{}, first, dim);
		else load_points_of(std::false_type{}, first, dim);
	};

	auto finish = [&](uint32_t first_pt) {
#pragma unroll
		for (int p = 0; p < P; ++p) {
			/* the two smallest of the leading tile's 16 results, the number of a result in its lowest four bits (cert_kd_keyed) */
			float v1 = __builtin_inff(), v2 = __builtin_inff();
			constexpr int VALUES = GROUPED ? RANK16_GROUPS : SNAP_ROWS;
			constexpr uint32_t NUMBER = GROUPED ? 7u : 15u;
#pragma unroll
			for (int r = 0; r < VALUES; ++r) {
				const float v = __uint_as_float((__float_as_uint(GROUPED ? kept[p][r / 2 % (RANK16_GROUPS / 2)][r % 2] : snap[p][GROUPED ? 0 : r]) & ~NUMBER) | (uint32_t)r);
				v2 = __builtin_amdgcn_fmed3f(v1, v2, v);
				v1 = __builtin_elementwise_minimum(v1, v);
			}
			const uint32_t r = __float_as_uint(v1) & NUMBER;
			/* GROUPED: the first centroid of the group, and the group */
			const uint32_t mine_idx = GROUPED ? (leader[p] * TILE + rank16_group_row(r) + 4 * h) * 8 + r : leader[p] * TILE + 8 * (r / 4) + 4 * h + r % 4;
			const float o1 = __shfl_xor(m1[p], 32), o2 = __shfl_xor(m2[p], 32);
			const float ov1 = __shfl_xor(v1, 32), ov2 = __shfl_xor(v2, 32);
			const uint32_t oi = (uint32_t)__shfl_xor((int)mine_idx, 32);
			const bool win = m1[p] < o1 || (m1[p] == o1 && h == 0);
			const float others = win ? fminf(o1, m2[p]) : fminf(m1[p], o2); /* everything outside the leading 16 rows */
			uint32_t idx = win ? mine_idx : oi;
			float lowest = win ? v1 : ov1;
			float next = fminf(win ? v2 : ov2, others);
			if constexpr (GROUPED) {
				/* the group's centroids again, on the vector ALU: half of the dimensions in each half-wave, chains of half as many roundings as the
				 * matrix instructions' (cert_kd_level1 covers them) */
				const uint32_t group = idx % 8, first = idx / 8, tile = first / TILE, row = first % TILE, step = rank16_group_step(group);
				const f16x8* at = (const f16x8*)(lds + (size_t)tile * TF) + h * TILE + row;
				const float* norms = lds + (size_t)w.chunk_tiles * TF + tile * NORM_TILE + row;
				float r1 = __builtin_inff(), r2 = __builtin_inff();
#pragma unroll
				for (uint32_t q = 0; q < 3; ++q) {
					const uint32_t on = group == 5 ? 0 : q * step;
					float sum = 0.0f;
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) {
						const f16x8 c = at[kb * WAVE + on];
						sum = rank16_dot(c, b[p][kb], sum);
					}
					float a = norms[on] + rank16_both(sum);
					if (q > 0) a = group == 5 ? 1.7e38f : a;
					const float v = __uint_as_float((__float_as_uint(a) & ~3u) | q);
					r2 = __builtin_amdgcn_fmed3f(r1, r2, v);
					r1 = __builtin_elementwise_minimum(r1, v);
				}
				idx = first + (__float_as_uint(r1) & 3u) * step;
				lowest = r1;
				next = fminf(next, r2);
			}
			const float x2 = rank16_whole<SHARED>(xx[p]), tau = cert_tau(w.kd, x2, rank16_whole<SHARED>(xl[p]), cert);
			const uint32_t pt = first_pt + p * TILE + col;
			const bool mine = h == 0 && pt < w.n;
			/* squares of the data as given underflow or overflow: no ranking says anything about the serial sums */
			const bool extreme = !(x2 + cert.c2max > smallest && x2 + cert.c2max < largest);
			const bool decided = (next - lowest > tau) && !extreme && idx < w.k;
			if (mine) w.assignment[pt] = idx < w.k ? idx : 0u;
			const bool flag = mine && !decided;
			const unsigned long long mask = __ballot(flag);
			if (LISTED) {
				late |= (uint64_t)mask << (p * TILE);
				late_first = first_pt;
			}
			if (mask) {
				const uint32_t add = (uint32_t)__builtin_popcountll(mask);
				if (flagged + add > list_entries) flush_flags();
				if (flag) {
					const uint32_t at = 2 * (flagged + (uint32_t)__builtin_popcountll(mask & ((1ull << lane) - 1ull)));
					flag_list[at] = pt;
					flag_list[at + 1] = screening_threshold(extreme ? __builtin_inff() : lowest, tau); /* (scaled, like the values) */
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
			for (int i = 0; i < (GROUPED ? 0 : SNAP_ROWS); ++i) asm volatile("" : "=v"(snap[p][i])); /* no value yet: tile 0 always takes the lead */
#pragma unroll
			for (int i = 0; i < (GROUPED ? RANK16_GROUPS / 2 : 0); ++i) asm volatile("" : "=v"(kept[p][i]));
		}
	};

	auto lowest_of = [](float a, float c) { return __builtin_elementwise_minimum(a, c); };
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
			constexpr int TRACK_OPS = GROUPED ? 11 : 20, OPS_PER_SLOT = (TRACK_OPS + SLOTS - 1) / SLOTS;
			f32x2 group[P][2];
			float group4[P], lowest[P];
			uint64_t leads[P];
			auto track = [&](const f32x16& a, int p, uint32_t tile, int u) {
				auto lowest_of_three = [&](float x, float y, float z) { return lowest_of(lowest_of(x, y), z); };
				const int minima = 8;
				if (u >= minima) {
					if (u == minima) m2[p] = __builtin_amdgcn_fmed3f(m1[p], m2[p], lowest[p]);
					else if (u == minima + 1) leads[p] = settled_mask(tile == 0 ? ~0ull : __builtin_amdgcn_ballot_w64(lowest[p] < m1[p]));
					else if constexpr (GROUPED) {
						if (u == minima + 2) take_groups_where(leads[p], m1[p], leader[p], lowest[p], tile, kept[p], group[p], group4[p], a[15]);
					}
					else if (u == 12) take_lead_where(leads[p], m1[p], leader[p], lowest[p], tile, snap[p], a);
					else if (u == 16) copy_second_half_where(leads[p], snap[p], a);
				}
				else if constexpr (GROUPED) {
					if (u < 4) group[p][u / 2][u % 2] = lowest_of_three(a[4 * u], a[4 * u + 1], a[4 * u + 2]);
					else if (u == 4) group4[p] = lowest_of_three(a[3], a[7], a[11]);
					else if (u == 5) lowest[p] = lowest_of_three(group[p][0].x, group[p][0].y, group[p][1].x);
					else if (u == 6) lowest[p] = lowest_of_three(lowest[p], group[p][1].y, group4[p]);
					else lowest[p] = lowest_of(lowest[p], a[15]);
				}
				else lowest[p] = u == 0 ? lowest_of(a[0], a[1]) : lowest_of_three(lowest[p], a[2 * u], a[2 * u + 1]);
			};
			auto track_all = [&](const f32x16 (&a)[P], uint32_t tile) {
#pragma unroll
				for (int p = 0; p < P; ++p)
#pragma unroll
					for (int u = 0; u < TRACK_OPS; ++u) track(a[p], p, tile, u);
			};
			/* one step: tile t_new into acc_new (which holds its norms), the tile after it requested, the tile in acc_old tracked in
			 * pieces behind the matrix instructions, then the norms of the tile after next into acc_old */
			auto step = [&](Ops& fetch_into, uint32_t t_new, f32x16 (&acc_new)[P], const Ops& use, f32x16 (&acc_old)[P], uint32_t tile_old) {
				fetch(fetch_into, min(t_new + 1, tiles - 1));
				__builtin_amdgcn_sched_barrier(0);
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
							if (u < TRACK_OPS) track(acc_old[tp], tp, tile_old, u);
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
				track_all(acc0, t);
				track_all(acc1, t + 1);
			}
			else track_all(acc0, t);
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
				for (int p = 0; p < P; ++p) {
					const Rank16Source from = rank16_source<LD, SHARED>(w.data, w.stride, first + p * TILE, w.n, lane);
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) rank16_request<LD, SHARED, false>(raw[p][kb], from, w.stride, kb, lane, w.dim);
				}
			};
			auto convert = [&](uint32_t first) {
#pragma unroll
				for (int p = 0; p < P; ++p) {
					Rank16Sums sums = { { 0.0f, 0.0f }, { 0.0f, 0.0f } };
#pragma unroll
					for (int kb = 0; kb < KB; ++kb) {
						rank16_place<LD, SHARED>(raw[p][kb], kb, lane, w.dim);
						rank16_convert<SHARED>(b[p][kb], raw[p][kb], frame, scale, kb, lane, sums, exchange);
					}
					rank16_total<SHARED>(xx[p], xl[p], sums, lane);
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
				copy_listed([&]() { if (item < items) convert(first_point(item)); });
			}
		}
		else {
			while (item < items) {
				const uint32_t after = claim();
				copy_listed([&]() { load_points(first_point(item)); });
				sweep();
				finish(first_point(item));
				item = uniform(after);
			}
			copy_listed([]() {});
		}
	}
	else {
		/* one chain of KB instructions per tile and point tile; the operands of block kb + OPERANDS are requested before the instructions of block kb */
		constexpr int OPERANDS = 2;
		auto track = [&](const f32x16& acc, int p, uint32_t tile) {
			float t = acc[0];
#pragma unroll
			for (int i = 1; i < 16; ++i) t = lowest_of(t, acc[i]);
			m2[p] = __builtin_amdgcn_fmed3f(m1[p], m2[p], t);
			const uint64_t leads = settled_mask(tile == 0 ? ~0ull : __builtin_amdgcn_ballot_w64(t < m1[p]));
			take_lead_where(leads, m1[p], leader[p], t, tile, snap[p], acc);
			copy_second_half_where(leads, snap[p], acc);
		};
		auto sweep_tile = [&](const float* operands, const float* norms, uint32_t t, uint32_t tile) {
			f32x16 acc[P];
			fetch_norms(acc[0], norms, t, h);
#pragma unroll
			for (int p = 1; p < P; ++p) acc[p] = acc[0];
			f16x8 c[KB];
#pragma unroll
			for (int kb = 0; kb < OPERANDS && kb < KB; ++kb) c[kb] = operand(operands, t, kb);
#pragma unroll
			for (int kb = 0; kb < KB; ++kb) {
				if (kb + OPERANDS < KB) c[kb + OPERANDS] = operand(operands, t, kb + OPERANDS);
#pragma unroll
				for (int p = 0; p < P; ++p) acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(c[kb], b[p][kb], acc[p], 0, 0, 0);
			}
			__builtin_amdgcn_sched_group_barrier(0x100, 4 + (OPERANDS < KB ? OPERANDS : KB), 0);
#pragma unroll
			for (int kb = 0; kb < KB; ++kb) {
				__builtin_amdgcn_sched_group_barrier(0x008, P, 0);
				if (kb + OPERANDS < KB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
			}
#pragma unroll
			for (int p = 0; p < P; ++p) track(acc[p], p, tile);
		};
		/* the ring of chunks: the one whose turn it is has arrived, the others are on their way */
		constexpr uint32_t SLOTS = rank16_slots(KB), EACH = (KB + WAVES - 1) / WAVES + (rank16_norm_blocks(1) + WAVES - 1) / WAVES; /* a wavefront's requests for a chunk of one tile (more than two slots) */
		const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) float*)lds;
		const uint32_t slot_bytes = rank16_slot_bytes(KB, w.chunk_tiles), norm_blocks = rank16_norm_blocks(w.chunk_tiles);
		const uint32_t chunks = STREAM ? (all_tiles + w.chunk_tiles - 1) / w.chunk_tiles : 1;
		uint32_t coming = 0, into = 0, from = 0; /* the chunk requested next, the slot it goes to, and the slot whose turn it is */
		auto request_chunk = [&]() { /* as many requests each time: a short last chunk repeats its last block */
			const uint32_t tile0 = coming * w.chunk_tiles, blocks = min(w.chunk_tiles, all_tiles - tile0) * KB, to = lds_base + into * slot_bytes;
			const char* src = (const char*)(w.packed + (size_t)tile0 * (KB * WAVE));
			for (uint32_t i = wave; i < w.chunk_tiles * KB + wave; i += WAVES) {
				const uint32_t block = min(i, blocks - 1);
				stage_block(src + (size_t)block * (WAVE * 16), lane, to + block * (WAVE * 16));
			}
			for (uint32_t i = wave; i < norm_blocks + wave; i += WAVES) {
				const uint32_t block = min(i, norm_blocks - 1);
				stage_words(w.norms + (size_t)tile0 * NORM_TILE + block * WAVE, lane, to + w.chunk_tiles * (KB * WAVE * 16) + block * (WAVE * 4));
			}
			coming = coming + 1 < chunks ? coming + 1 : 0;
			into = into + 1 < SLOTS ? into + 1 : 0;
		};
		if constexpr (STREAM)
			for (uint32_t i = 0; i + 1 < SLOTS; ++i) request_chunk();
		auto sweep_chunk = [&](uint32_t chunk) {
			if constexpr (!STREAM) {
				for (uint32_t t = 0; t < all_tiles; ++t) sweep_tile(lds, lds + (size_t)all_tiles * TF, t, t);
				return;
			}
			const uint32_t tile0 = chunk * w.chunk_tiles, tiles = min(w.chunk_tiles, all_tiles - tile0);
			const float* here = lds + (size_t)from * (slot_bytes / 4);
			for (uint32_t t = 0; t < tiles; ++t) sweep_tile(here, here + w.chunk_tiles * TF, t, tile0 + t);
			from = from + 1 < SLOTS ? from + 1 : 0;
		};
		auto next_chunk = [&]() {
			if constexpr (!STREAM) return;
			staged_but<(SLOTS - 2) * EACH>();
			__syncthreads(); /* everybody's part of this chunk is here, and nobody reads the one before it any more */
			request_chunk();
		};
		const uint32_t units = (w.n + WAVES * P * TILE - 1) / (WAVES * P * TILE);
		for (uint32_t unit = blockIdx.x; unit < units; unit += gridDim.x) {
			const uint32_t first = (unit * WAVES + wave) * (P * TILE);
			copy_listed([&]() { load_points(first); });
			start();
			for (uint32_t chunk = 0; chunk < chunks; ++chunk) { next_chunk(); sweep_chunk(chunk); }
			finish(first);
		}
		copy_listed([]() {});
	}
	if constexpr (STREAM) staged_but<0>(); /* (nothing may arrive in LDS that is no longer this work-group's) */
	/* what is left in the lists: one addition per work-group (one per wavefront took 12 us of a launch: 2048 of them to one address) */
	__syncthreads();
	if (lane == 0) wave_max[0][wave] = flagged;
	__syncthreads();
	uint32_t before = 0, all = 0;
#pragma unroll
	for (uint32_t v = 0; v < WAVES; ++v) {
		before += v < wave ? wave_max[0][v] : 0u;
		all += wave_max[0][v];
	}
	if (all == 0) return;
	if (tid == 0) wave_max[1][0] = atomicAdd(w.length, all);
	__syncthreads();
	const size_t slot = 2 * (size_t)(wave_max[1][0] + before);
	for (uint32_t i = lane; i < 2 * flagged; i += WAVE) w.list[slot + i] = flag_list[i];
}

template <int KB>
static int launch_rank16_kb(const AssignArgs& a, Rank16Args w, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	const uint32_t tile_bytes = (rank16_tile_floats<KB>() + NORM_TILE) * 4, tiles = w.kp / TILE, budget = lds_budget_of(exec, dev);
	if (budget < rank16_least_bytes(KB, a.layout)) return fail(KMX_ERR_UNSUPPORTED, "assign (half-precision sweep): LDS budget of %u bytes is too small", budget);
	const Rank16Copies copies = a.layout == KMX_AOS ? RANK16_NONE : w.copy_all ? RANK16_ALL : RANK16_LISTED;
	auto resident = [&](Rank16Copies room, uint32_t entries) { return (uint64_t)tiles * tile_bytes + rank16_static_bytes(KB, a.layout, false, room) + rank16_list_bytes(KB, entries) <= budget; };
	/*
	 * All rows go out only where the update has no columns' sums: more centroids than those fit LDS, and so than fit it here (or a recording without room for them). Without room to exchange rows, SoA points have a tile more in LDS.
	 * Beyond 128 dimensions that is too dear: what is left holds short lists, where the streamed form has two work-groups of four wavefronts and whole ones (us per assignment,
	 * resident -> streamed: N = 192644, d = 133, k = 375 110 -> 79; N = 56454, d = 169, k = 368 66 -> 49; N = 28000, d = 204, k = 274 1.13 of the time; up to 128 dimensions
	 * 0.90 to 1.06).
	 */
	const bool stream_mode = copies == RANK16_ALL || !resident(KB >= 12 && copies == RANK16_LISTED ? RANK16_ALL : copies, rank16_list_least(KB));
	w.chunk_tiles = tiles;
	w.list_entries = RANK16_LIST_MOST;
	while (!stream_mode && !resident(copies, w.list_entries)) --w.list_entries;
	uint32_t lds_bytes = tiles * tile_bytes + rank16_list_bytes(KB, w.list_entries);
	const uint32_t static_bytes = rank16_static_bytes(KB, a.layout, stream_mode, copies);
	if (stream_mode) {
		w.chunk_tiles = 1;
		while (rank16_slots(KB) == 2 && w.chunk_tiles < tiles && static_bytes + 2 * rank16_slot_bytes(KB, w.chunk_tiles + 1) <= budget) ++w.chunk_tiles;
		lds_bytes = rank16_slots(KB) * rank16_slot_bytes(KB, w.chunk_tiles);
	}
	void (*kernel)(Rank16Args) = a.layout == KMX_AOS ? (stream_mode ? rank16_kernel<KB, KMX_AOS, true, RANK16_NONE> : rank16_kernel<KB, KMX_AOS, false, RANK16_NONE>)
	                           : copies == RANK16_ALL ? rank16_kernel<KB, KMX_SOA, true, RANK16_ALL>
	                           : stream_mode ? rank16_kernel<KB, KMX_SOA, true, RANK16_LISTED> : rank16_kernel<KB, KMX_SOA, false, RANK16_LISTED>;
	const uint32_t waves = rank16_waves(KB, stream_mode), unit = (stream_mode || KB > 4 ? waves : 1) * RANK16_P * TILE;
	const uint32_t grid = std::min((a.n + unit - 1) / unit, (waves == 4 ? 2 : 1) * dev.compute_units);
	exec->block_count = grid;
#define KMX_PLAN(cond) do { if (!(cond)) return fail(KMX_ERR_DEVICE, "assign (half-precision sweep): launch refused, the plan breaks \"%s\" (dim %u, k %u, kp %u, n %u, chunk tiles %u, LDS %u)", \
	#cond, a.dim, a.k, w.kp, a.n, w.chunk_tiles, lds_bytes); } while (0)
	if (!sizing_only()) {
		KMX_PLAN(w.kp % TILE == 0 && w.kp >= a.k && w.kp - a.k < TILE && a.n >= 1 && KB * KBLOCK >= a.dim);
		KMX_PLAN(w.chunk_tiles >= 1 && (uint64_t)lds_bytes + static_bytes <= dev.lds_bytes && rank16_tile_floats<KB>() % 4 == 0);
		KMX_PLAN(stream_mode || (w.list_entries >= RANK16_P * TILE / 2 && rank16_waves(KB, false) * 2 * w.list_entries + tiles * (tile_bytes / 4) <= lds_bytes / 4));
		KMX_PLAN(ws->packed16 && (size_t)tiles * KB * WAVE * 4 <= ws->packed16_cap);
		KMX_PLAN(!stream_mode || ((rank16_slots(KB) == 2 || w.chunk_tiles == 1) && /* whole requests of norms, the last chunk's too */
		                          (size_t)(tiles - 1) / w.chunk_tiles * w.chunk_tiles * NORM_TILE + rank16_norm_blocks(w.chunk_tiles) * WAVE <= ws->norms16_cap));
		KMX_PLAN(a.layout == KMX_AOS || (w.copies && w.copy_stride % 8 == 0 && w.copy_stride >= a.dim && w.copy_stride <= KB * KBLOCK && (size_t)a.n * w.copy_stride <= ws->queued_rows_cap));
		KMX_PLAN(w.list && w.length && w.norms && w.low2 && w.frame && w.scale);
	}
#undef KMX_PLAN
	KMX_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes));
	KMX_LAUNCH_KERNEL(kernel, dim3(grid), dim3(waves * WAVE), lds_bytes, stream(), w);
	KMX_LAUNCH_CHECK("rank16_kernel");
	return KMX_OK;
}

} // namespace kmx

#endif
