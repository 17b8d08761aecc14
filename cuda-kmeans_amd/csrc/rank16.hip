/*
 * Assignment of rows of 5 to 256 dimensions by one half-precision product per dimension, and the exact pass behind it.
 *
 * Ranking. Points and centroids are moved to the middle of the centroids and scaled by a power of two S that brings the centroids'
 * coordinates to about 2^-5 (rank16_scale), then rounded to half precision (11 significant bits): a[j] = S^2 (|c_j|^2 - 2 c_j . x) is one
 * v_mfma_f32_32x32x16_f16 per 16 dimensions, a third of what three bf16 products cost. The certificate is the one-product form of
 * certificate.h with the norms of what the roundings actually dropped, |x - x_half| of the point and max_j |c'_j - c'_half| of the
 * centroids; overflow to infinity and values lost below the smallest half-precision number are covered by the same norms (an
 * infinite one certifies nothing). Eleven bits instead of the eight of a bf16 make it eight times narrower: at N = 2M, d = 32,
 * k = 1024 it leaves 0.5 to 4 % of the points, where hi * hi in bf16 left 12 to 26 % to a second sweep with three products.
 *
 * Exact pass (rank16_exact_impl.h). One kernel for the listed points: it ranks them again with the same instruction on the same
 * operands, notes the centroids within the point's threshold (two or three of k) and evaluates the serial arithmetic for those.
 * Gather, screen, evaluate and scatter were four launches (63 us at N = 1M, d = 256, k = 1024, behind a second sweep of 188).
 *
 * What bounds it: the sweep by the matrix instructions and the tracking of the minima that shares the issue slots with them, at a clock that
 * gives way to the power they take (N = 1M, d = 256, k = 1024: 475 to 505 us, 1.09 to 1.16 PFLOP/s; d = 32, k = 1024, N = 2M: 151 to 169 us); the
 * exact pass by the latencies of one unit, list, rows, ranking and pairs in turn (1 to 4 % listed: 26 to 35 us; 9 % of N = 2M, d = 128: 110).
 * Whole calls, two bf16 levels -> this kernel at first -> now: N = 1M, d = 256, k = 1024 1713 -> 743 -> 520 us; N = 2M, d = 128, k = 1024, SoA
 * 1629 -> 940 -> 845; N = 2M, d = 32, k = 1024 332 -> 230 -> 204 (Gaussian mixture, centroids after two rounds; 218 around its first points).
 */
#include "rank16_exact_impl.h"

namespace kmx {

/* blocks of 16 dimensions the sweep is built for */
static uint32_t rank16_kb(uint32_t dim)
{
	const uint32_t need = (dim + KBLOCK - 1) / KBLOCK;
	for (uint32_t o : { 1u, 2u, 3u, 4u, 6u, 8u, 12u, 16u })
		if (need <= o) return o;
	return 0;
}

#define KMX_DECLARE_RANK16(W) int launch_rank16_##W(const AssignArgs& a, const Rank16Args& w, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);
KMX_DECLARE_RANK16(1) KMX_DECLARE_RANK16(2) KMX_DECLARE_RANK16(3) KMX_DECLARE_RANK16(4)
KMX_DECLARE_RANK16(6) KMX_DECLARE_RANK16(8) KMX_DECLARE_RANK16(12) KMX_DECLARE_RANK16(16)
#define KMX_DECLARE_EXACT16(W) int launch_listed_exact_##W(const AssignArgs& a, const ExactArgs<float>& w, const DeviceInfo& dev); \
	int launch_listed_exact_##W(const AssignArgs& a, const ExactArgs<double>& w, const DeviceInfo& dev);
KMX_DECLARE_EXACT16(1) KMX_DECLARE_EXACT16(2) KMX_DECLARE_EXACT16(3) KMX_DECLARE_EXACT16(4)
KMX_DECLARE_EXACT16(6) KMX_DECLARE_EXACT16(8) KMX_DECLARE_EXACT16(12) KMX_DECLARE_EXACT16(16)

/*
 * One wavefront per (padded) centroid row: its half-precision operands, S^2 |c|^2, the squared norms of what half precision and the
 * bf16 parts leave out. Every work-group computes the frame m and S (rank16_scale) from centroids spread evenly over
 * all of them: the first ones are often the first points, and those may be unlike the rest (blank rows ahead of an image, the quiet start
 * of a recording).
 */
template <int LM>
__global__ void __launch_bounds__(256)
pack_means16_kernel(const float* __restrict__ means, const double* __restrict__ means64, size_t stride_means, _Float16* __restrict__ packed, float* __restrict__ rows, float* __restrict__ norms,
                    uint32_t dim, uint32_t k, uint32_t kp, uint32_t dp, uint32_t* __restrict__ counters)
{
	__shared__ float frame[FRAME_DIMS];
	__shared__ float wave_far[2][4];
	const uint32_t lane = threadIdx.x & (WAVE - 1);
	if (blockIdx.x == 0 && threadIdx.x == 0) { counters[0] = 0u; counters[LISTED_COUNTER] = 0u; }
	const uint32_t j = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
	/* this row's coordinates are requested ahead of the frame they will be moved to */
	float exact[FRAME_DIMS / WAVE];
#pragma unroll
	for (uint32_t i = 0; i < FRAME_DIMS / WAVE; ++i) {
		const uint32_t q = lane + i * WAVE;
		exact[i] = (j < k && q < dim) ? means[elem<LM>(stride_means, j, q)] : 0.0f;
	}
	/* 16 coordinates per lane, of as many rows spread evenly over the centroids: 16 rows of 129 to 256 dimensions, 128 of 17 to 32 */
	const uint32_t log_columns = 32 - __builtin_clz(max(dim, 2u) - 1), log_groups = 8 - log_columns; /* (dim <= 256) */
	const uint32_t column = min(threadIdx.x & ((1u << log_columns) - 1u), dim - 1), group = threadIdx.x >> log_columns;
	float sample[16];
#pragma unroll
	for (uint32_t i = 0; i < 16; ++i) sample[i] = means[elem<LM>(stride_means, even_row(group * 16 + i, 4 + log_groups, k), column)];
	/* the frame m: the mean of the first lanes' 16 rows, finite coordinates only (any vector would do; this one lies inside the data) */
	if (group == 0 && threadIdx.x < dim) {
		float sum = 0.0f;
#pragma unroll
		for (uint32_t i = 0; i < 16; ++i) sum += __builtin_fabsf(sample[i]) < __builtin_inff() ? sample[i] : 0.0f;
		sum = sum / 16.0f;
		frame[column] = __builtin_fabsf(sum) < __builtin_inff() ? sum : 0.0f; /* (the sum of finite values may overflow) */
	}
	if (threadIdx.x >= dim && threadIdx.x < dp) frame[threadIdx.x] = 0.0f;
	__syncthreads();
	if (blockIdx.x == 0 && threadIdx.x < dp) norms[rank16_frame_offset(kp) + threadIdx.x] = frame[threadIdx.x];
	float far = 0.0f, size = 0.0f; /* (infinities and NaN drop out) */
#pragma unroll
	for (uint32_t i = 0; i < 16; ++i) {
		const float d = __builtin_fabsf(sample[i] - frame[column]);
		if (d < __builtin_inff()) { far = fmaxf(far, d); size = fmaxf(size, __builtin_fabsf(sample[i])); }
	}
	for (int off = WAVE / 2; off > 0; off >>= 1) { far = fmaxf(far, __shfl_xor(far, off)); size = fmaxf(size, __shfl_xor(size, off)); }
	if (lane == 0) { wave_far[0][threadIdx.x / WAVE] = far; wave_far[1][threadIdx.x / WAVE] = size; }
	__syncthreads();
	const float scale = rank16_scale(fmaxf(fmaxf(wave_far[0][0], wave_far[0][1]), fmaxf(wave_far[0][2], wave_far[0][3])),
	                                 fmaxf(fmaxf(wave_far[1][0], wave_far[1][1]), fmaxf(wave_far[1][2], wave_far[1][3])));
	if (blockIdx.x == 0 && threadIdx.x == 0) {
		norms[rank16_scale_offset(kp)] = scale;
		norms[rank16_scale_offset(kp) + 1] = 1.0f / (scale * scale);
	}
	if (j >= kp) return;
	float c2 = 0.0f, low2 = 0.0f, mid2 = 0.0f, rest2 = 0.0f;
#pragma unroll
	for (uint32_t i = 0; i < FRAME_DIMS / WAVE; ++i) {
		const uint32_t q = lane + i * WAVE;
		if (q >= dp) break;
		const float v = (j < k && q < dim) ? __builtin_fmaf(exact[i], scale, -(frame[q] * scale)) : 0.0f;
		c2 += v * v;
		const float cv = -2.0f * v;
		const _Float16 half = (_Float16)cv;
		const float low = cv - (float)half;
		low2 += low * low;
		__bf16 hi, mid;
		const float rest = split_bf16(cv, hi, mid);
		mid2 += (float)mid * (float)mid;
		rest2 += rest * rest;
		if (means64) ((double*)rows)[(size_t)j * dp + q] = (j < k && q < dim) ? means64[elem<LM>(stride_means, j, q)] : 0.0;
		else rows[(size_t)j * dp + q] = exact[i];
		packed[(((size_t)(j / TILE) * (dp / KBLOCK) + q / KBLOCK) * WAVE + (q % KBLOCK) / 8 * TILE + j % TILE) * 8 + q % 8] = half;
	}
	for (int off = WAVE / 2; off > 0; off >>= 1) {
		c2 += __shfl_xor(c2, off);
		low2 += __shfl_xor(low2, off);
		mid2 += __shfl_xor(mid2, off);
		rest2 += __shfl_xor(rest2, off);
	}
	if (lane == 0) {
		norms[norm_at(j)] = j < k ? c2 : 1.7e38f; /* rows that do not exist: beyond all values, but finite (keyed values) */
		norms[rank16_low_offset(kp) + j] = low2;
		norms[rank16_low_offset(kp) + kp + j] = mid2;
		norms[rank16_low_offset(kp) + 2 * kp + j] = rest2;
	}
	if (lane < NORM_TILE - TILE && j % TILE == 0) norms[(j / TILE) * NORM_TILE + TILE + lane] = 1.7e38f;
}

bool rank16_supports(const AssignArgs& a, uint32_t lds_budget)
{
	const uint32_t kb = rank16_kb(a.dim);
	if (a.dim <= 4 || kb == 0 || a.k >= (1u << 25) || a.n > (1u << 31)) return false;
	return rank16_least_bytes(kb, a.layout) <= lds_budget && exact_dynamic_bytes(kb, EXACT_GROUPS) + exact_static_bytes(a.points64 != nullptr) <= lds_budget;
}

/* the centroids for launch_rank16_sweep */
static int launch_pack16(const AssignArgs& a, Workspace* ws)
{
	const uint32_t dp = rank16_kb(a.dim) * KBLOCK, kp = round_up(a.k, TILE);
	const int rc = reserve_packed16(ws, rank16_rows_offset(kp, dp) + (size_t)kp * dp * (a.points64 ? 2 : 1), rank16_norms_floats(kp));
	if (rc) return rc;
	auto pack = a.layout_means == KMX_AOS ? pack_means16_kernel<KMX_AOS> : pack_means16_kernel<KMX_SOA>;
	KMX_LAUNCH_KERNEL(pack, dim3((kp * WAVE + 255) / 256), dim3(256), 0, stream(),
	                   a.means, a.means64, a.stride_means, (_Float16*)ws->packed16, ws->packed16 + rank16_rows_offset(kp, dp), ws->norms16, a.dim, a.k, kp, dp, ws->counters);
	KMX_LAUNCH_CHECK("pack_means16_kernel");
	return KMX_OK;
}

/* sweeps the points; what is left goes to ws->listed (length in counters[LISTED_COUNTER]), the rows of SoA points to ws->queued_rows: those of listed points, or (copy_all) all */
static int launch_rank16_sweep(const AssignArgs& a, bool copy_all, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	const uint32_t kb = rank16_kb(a.dim), kp = round_up(a.k, TILE), copy_stride = round_up(a.dim, 8);
	int rc = reserve_listed(ws, 2 * (size_t)a.n);
	if (rc) return rc;
	if (a.layout == KMX_SOA && (rc = reserve_queued_rows(ws, a.n, copy_stride, 0))) return rc;
	const float* norms = ws->norms16;
	const Rank16Args w = { a.data, a.stride, (const f16x8*)ws->packed16, norms, norms + rank16_low_offset(kp), norms + rank16_frame_offset(kp), ws->norms16 + rank16_scale_offset(kp),
	                       a.assignment, ws->listed, ws->counters + LISTED_COUNTER, ws->queued_rows, copy_stride, copy_all, a.dim, a.k, kp, a.n, 0,
	                       cert_kd_level1(a.dim) + cert_kd_keyed(4) + 8.0f * CERT_UNIT + a.kd_extra, 0 };
	switch (kb) {
	case 1: return launch_rank16_1(a, w, exec, ws, dev);
	case 2: return launch_rank16_2(a, w, exec, ws, dev);
	case 3: return launch_rank16_3(a, w, exec, ws, dev);
	case 4: return launch_rank16_4(a, w, exec, ws, dev);
	case 6: return launch_rank16_6(a, w, exec, ws, dev);
	case 8: return launch_rank16_8(a, w, exec, ws, dev);
	case 12: return launch_rank16_12(a, w, exec, ws, dev);
	case 16: return launch_rank16_16(a, w, exec, ws, dev);
	default: return fail(KMX_ERR_UNSUPPORTED, "assign (half-precision sweep): dim %u is not supported", a.dim);
	}
}

/* the serial result for the points in ws->listed, after launch_rank16_sweep; F: what the serial arithmetic is done in */
template <typename F>
static int launch_listed_exact(const AssignArgs& a, const F* points, size_t points_stride, size_t points_step, uint32_t points_dim, Workspace* ws, const DeviceInfo& dev)
{
	const uint32_t kb = rank16_kb(a.dim), dp = kb * KBLOCK, kp = round_up(a.k, TILE);
	const float* norms = ws->norms16;
	const bool aos = a.layout == KMX_AOS, copied = !aos && a.dim > 4; /* (narrow rows have not been copied) */
	const uint32_t row_dim = copied ? round_up(a.dim, 8) : a.dim;
	const ExactArgs<F> w = { copied ? ws->queued_rows : a.data, aos ? a.stride : copied ? row_dim : 1, aos || copied ? 1 : a.stride, row_dim, points, points_stride, points_step, points_dim,
	                         (const F*)(ws->packed16 + rank16_rows_offset(kp, dp)), (const f16x8*)ws->packed16, norms,
	                         norms + rank16_frame_offset(kp), norms + rank16_scale_offset(kp), a.assignment, ws->listed, ws->counters + LISTED_COUNTER, ws->counters,
	                         a.dim, a.k, kp, cert_kd_split(a.dim) + 8.0f * CERT_UNIT, kb, EXACT_GROUPS };
	switch (kb) {
	case 1: return launch_listed_exact_1(a, w, dev);
	case 2: return launch_listed_exact_2(a, w, dev);
	case 3: return launch_listed_exact_3(a, w, dev);
	case 4: return launch_listed_exact_4(a, w, dev);
	case 6: return launch_listed_exact_6(a, w, dev);
	case 8: return launch_listed_exact_8(a, w, dev);
	case 12: return launch_listed_exact_12(a, w, dev);
	case 16: return launch_listed_exact_16(a, w, dev);
	default: return fail(KMX_ERR_UNSUPPORTED, "assign (half-precision sweep): dim %u is not supported", a.dim);
	}
}

static __global__ void clear_word_kernel(uint32_t* word) { *word = 0u; }

int launch_assign_rank16(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	int rc = launch_pack16(a, ws);
	if (rc) return rc;
	/* SoA points go in parts whose copied rows fit the bound of the workspace (1 GiB unless it was set) */
	const size_t row_bytes = round_up(a.dim, 8) * sizeof(float);
	const uint32_t part = a.layout == KMX_AOS ? a.n : (uint32_t)std::min<size_t>(a.n, std::max<size_t>(1024, queued_rows_limit() / row_bytes));
	const bool copy_all = a.rows_out && a.layout == KMX_SOA && part == a.n; /* somebody reads all of them */
	for (uint32_t first = 0; first < a.n; first += std::min(part, a.n - first)) {
		AssignArgs p = a;
		p.n = std::min(part, a.n - first);
		p.data = a.data + first;
		p.assignment = a.assignment + first;
		if (first) {
			KMX_LAUNCH_KERNEL(clear_word_kernel, dim3(1), dim3(1), 0, stream(), ws->counters + LISTED_COUNTER);
			KMX_LAUNCH_CHECK("clear_word_kernel");
		}
		if (first == 0 && (rc = profile_begin(0))) return rc;
		if ((rc = launch_rank16_sweep(p, copy_all, exec, ws, dev))) return rc;
		if (first == 0 && (rc = profile_end(0))) return rc;
		const bool aos = a.layout == KMX_AOS;
		if (a.points64) rc = launch_listed_exact<double>(p, a.points64 + first, aos ? a.stride : 1, aos ? 1 : a.stride, a.dim, ws, dev);
		else if (aos) rc = launch_listed_exact<float>(p, p.data, p.stride, 1, p.dim, ws, dev);
		else rc = launch_listed_exact<float>(p, ws->queued_rows, round_up(a.dim, 8), 1, round_up(a.dim, 8), ws, dev);
		if (rc) return rc;
	}
	if (a.settled) *a.settled = true;
	if (copy_all) *a.rows_out = AosRows{ ws->queued_rows, round_up(a.dim, 8) };
	return KMX_OK;
}

int launch_bf16_behind_cells(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, uint32_t kp, float kd, const WayBack& way);

int launch_assign_cells(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev)
{
	const bool choose = two_level_mode() != 2; /* (tests of the cells take them whatever the points) */
	const uint32_t kp = round_up(a.k, TILE);
	int rc = reserve_packed16(ws, rank16_rows_offset(kp, KBLOCK) + (size_t)kp * KBLOCK, rank16_norms_floats(kp));
	if (rc) return rc;
	if ((rc = reserve_packed(ws, (size_t)(kp / TILE) * tile_floats(row_floats<1, true>()), split_norms_floats(kp), 0))) return rc;
	const Cells16 half = { ws->norms16, ws->norms16 + rank16_low_offset(kp), ws->norms16 + rank16_frame_offset(kp), ws->norms16 + rank16_scale_offset(kp), kp,
	                       cert_kd_level1(a.dim) + 8.0f * CERT_UNIT };
	if ((rc = launch_cells(a, exec, ws, dev, half, choose))) return rc;
	if (choose) {
		/* the sweep those points get for which the search thinks little of the cells */
		Workspace view = *ws; /* (the launcher only reads the pointers) */
		view.queue = ws->listed; view.queue_cap = ws->listed_cap; view.counters = ws->counters + LISTED_COUNTER;
		AssignArgs p = a;
		p.shift_rows = true;
		kmx_exec_params other = *exec;
		if ((rc = launch_bf16_behind_cells(p, &other, &view, dev, kp, cert_kd_packed(a.dim), WayBack{ ws->counters + WAY_BACK_COUNTER, half.scale, half.kd }))) return rc;
	}
	if ((rc = profile_end(0))) return rc;
	const bool aos = a.layout == KMX_AOS;
	return launch_listed_exact<float>(a, a.data, aos ? a.stride : 1, aos ? 1 : a.stride, a.dim, ws, dev);
}

} // namespace kmx
