/*
 * Internal declarations shared by the HIP sources of libkmx_hip.so (not part of the C ABI).
 */
#ifndef KMX_INTERNAL_H
#define KMX_INTERNAL_H

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <cstdio>

#include "kmx.h"

namespace kmx {

constexpr int WAVE = 64; /* gfx950 wavefront width */

typedef float f32x4 __attribute__((ext_vector_type(4)));

/* Records the message returned by kmx_last_error() and passes `code` through. */
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
void clear_error();

/* The stream every kernel of the library is launched on. */
hipStream_t stream();

/* Brackets the dominant kernel of a call with events when kmx_set_profiling(1) is active (which: 0 assign, 1 update). */
int profile_begin(int which);
int profile_end(int which);
/* while set, profile_begin / profile_end do nothing (they create events on first use: not for the entry point that allocates nothing) */
void suspend_profiling(bool suspended);

/* Properties of the current device, queried once. */
struct DeviceInfo {
	int device = -1;
	uint32_t compute_units = 0;
	uint32_t lds_bytes = 0;      /* LDS available to one work-group */
	uint32_t max_threads = 0;
};
int device_info(const DeviceInfo** out);

/*
 * Work space owned by the library (grown on demand, released by kmx_shutdown):
 *   recheck queue : indices of the points the fast assignment kernels hand to the exact pass
 *   counters      : [0] = queue length of the current call, [4] = length of the list of the half-precision sweep
 *   packed means  : centroids re-laid-out (scaled by -2, padded) for the fast assignment kernels
 *   norms         : |c|^2 per (padded) centroid followed by max_j |c_j|^2
 *   partials      : per-work-group partial sums/counts of the update kernels that need them
 *   queued rows   : the rows of the queued points as a compact AoS block for the exact pass, with a
 *                   queue and an assignment vector of their own (counters[1] = rows taken, counters[2] = entries left
 *                   over); the split-bf16 sweep uses the block for every layout
 */
struct Workspace {
	uint32_t* queue = nullptr;      size_t queue_cap = 0;      /* entries */
	uint32_t* counters = nullptr;                               /* 16 words */
	float* packed_means = nullptr;  size_t packed_cap = 0;     /* floats  */
	float* packed16 = nullptr;      size_t packed16_cap = 0;   /* floats: half-precision operands of the centroids (rank16.hip) */
	float* norms = nullptr;         size_t norms_cap = 0;      /* floats  */
	uint32_t* cells = nullptr;      size_t cells_cap = 0;      /* words: grid, table and lists of assign_cells.hip */
	float* norms16 = nullptr;       size_t norms16_cap = 0;    /* floats: norms, frame and scale of the half-precision sweep */
	float* means_t = nullptr;       size_t means_t_cap = 0;    /* floats: exact transposed centroids [dim][kp] */
	float* partials = nullptr;      size_t partials_cap = 0;   /* floats  */
	uint32_t* fused_assignment = nullptr; size_t fused_cap = 0; /* entries: assignment vector of kmx_fused_f32 */
	uint32_t* bucket_sizes = nullptr;     size_t bucket_cap = 0; /* entries: member counts nobody asked for (kmx_bucket_sum_f32) */
	float* rows_copy = nullptr;           size_t rows_copy_cap = 0;     /* floats: AoS copy of SoA points for the tuned update */
	float* queued_rows = nullptr;         size_t queued_rows_cap = 0;   /* floats */
	uint32_t* queued_index = nullptr;     size_t queued_index_cap = 0;  /* words: per row 2 (queue) + 2 (assignment or 64-bit key), then the screen's pair counters and pairs */
	uint32_t* carried = nullptr;          size_t carried_cap = 0;       /* words: per point the leader and the two smallest ranking values over the slices of centroids swept so far */
	uint32_t* listed = nullptr;           size_t listed_cap = 0;        /* words: two per point the half-precision sweep could not settle (its length: counters[LISTED_COUNTER]) */
	const float* exact_norms = nullptr; /* |c|^2 of the centroids as given, in the layout of `norms`, for the exact pass of a sweep that moved its frame (points into `norms`; null: `norms` holds them) */
	bool fixed = false; /* the work space of the entry point that allocates nothing: its buffers never grow, a call that needs more is refused */
};
int workspace(Workspace** ws);
int reserve_queue(Workspace* ws, size_t entries);
int reserve_packed(Workspace* ws, size_t packed_floats, size_t norm_floats, size_t transposed_floats);
int reserve_cells(Workspace* ws, size_t words);
int reserve_packed16(Workspace* ws, size_t packed_floats, size_t norm_floats);
int reserve_partials(Workspace* ws, size_t floats);
int reserve_fused_assignment(Workspace* ws, size_t entries);
int reserve_bucket_sizes(Workspace* ws, size_t entries);
int reserve_rows_copy(Workspace* ws, size_t floats);
int reserve_queued_rows(Workspace* ws, size_t rows, size_t dim, size_t extra_words);
int reserve_carried(Workspace* ws, size_t words);
int reserve_listed(Workspace* ws, size_t words);
int two_level_mode(); /* kmx_set_two_level_sweep */
constexpr uint32_t CELLS_COUNTER = 5;  /* word of Workspace::counters that counts the list units handed out by build_cells_kernel */
constexpr uint32_t FINISH_COUNTER = 6; /* and the one that counts the work-groups fused_finish_kernel has behind it */
constexpr uint32_t WAY_BACK_COUNTER = 7; /* not zero: the points are left to the packed sweep (assign_cells_kernel) */
constexpr uint32_t LISTED_COUNTER = 4; /* word of Workspace::counters that holds the length of Workspace::listed */

#define KMX_HIP(call)                                                                                         \
	do {                                                                                                      \
		hipError_t kmx_e_ = (call);                                                                           \
		if (kmx_e_ != hipSuccess)                                                                             \
			return ::kmx::fail(KMX_ERR_DEVICE, "%s failed: %s", #call, hipGetErrorString(kmx_e_));           \
	} while (0)

/* Every kernel of the library is launched through this: while kmx_reserve_f32 walks the launchers to size the work space
 * (sizing_only()), the reservations happen and the kernels do not run. */
bool sizing_only();
#define KMX_LAUNCH_KERNEL(...)                                                                                \
	do {                                                                                                      \
		if (!::kmx::sizing_only()) hipLaunchKernelGGL(__VA_ARGS__);                                           \
	} while (0)

#define KMX_LAUNCH_CHECK(name)                                                                                \
	do {                                                                                                      \
		hipError_t kmx_e_ = hipGetLastError();                                                                \
		if (kmx_e_ != hipSuccess)                                                                             \
			return ::kmx::fail(KMX_ERR_DEVICE, "launch of %s failed: %s", name, hipGetErrorString(kmx_e_));  \
	} while (0)

/* Element address in either layout (layout_policies.hpp:22-25 SoA, :46-49 AoS of the reference). */
template <int LAYOUT>
__host__ __device__ __forceinline__ size_t elem(size_t stride, size_t idx, size_t dim)
{
	return LAYOUT == KMX_AOS ? idx * stride + dim : dim * stride + idx;
}

/* AoS copy of SoA points in the work space */
struct AosRows {
	const float* data; size_t stride;
};

/* Argument bundle of one assignment call after validation. */
struct AssignArgs {
	const float* data; int layout; size_t stride;
	const float* means; int layout_means; size_t stride_means;
	uint32_t* assignment;
	uint32_t dim, k, n;
	/* The double-precision entry point runs the float sweeps on rounded copies of its inputs as a ranking stage:
	 * kd_extra widens the certificate by the effect of that rounding, and ranking_only leaves the queue of
	 * uncertified points (pairs of point number and threshold, length in counters[0]) to the caller. */
	float kd_extra = 0.0f;
	bool ranking_only = false;
	/* The split-bf16 sweep may work in a frame moved to the middle of the centroids (shift_rows). Where the screen follows,
	 * the thresholds of the queue stay values of that frame, which only the screen shares, so entries from position
	 * shifted_cap on -- those the screen has no rows for -- get an infinite threshold; where the other kernels of the exact
	 * pass follow, the sweep takes the thresholds back to the frame of the data (unmoved_thresholds). */
	bool shift_rows = false;
	uint32_t shifted_cap = 0xFFFFFFFFu;
	bool unmoved_thresholds = false;
	/* the single-pass fused kernel: write the result of every point to `assignment`, not only those of the exact pass */
	bool emit_assignment = false;
	/* ranking_only: the doubles behind the float copies (layouts and strides of the copies). A sweep whose exact pass takes doubles leaves
	 * nothing to the caller and says so in *settled. */
	const double* points64 = nullptr; const double* means64 = nullptr; bool* settled = nullptr;
	/* SoA points: filled in by a sweep that wrote all rows as AoS on the way (left alone by the others) */
	AosRows* rows_out = nullptr;
};

struct UpdateArgs {
	const float* data; int layout; size_t stride;
	const uint32_t* assignment;
	float* means; int layout_means; size_t stride_means;
	uint32_t* cluster_sizes;
	uint32_t dim, k, n;
	bool divide = true; /* false: leave the member sums in `means` (the update micro-benchmark) */
};

/* kmx_runtime.hip: runs one assignment variant (KMX_ASSIGN_BEST: chosen by shape); *chosen receives the concrete variant */
int dispatch_assign(int variant, const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, int* chosen);

/* assign_exact.hip */
int launch_assign_base(const AssignArgs& a, kmx_exec_params* exec);
/* Re-evaluates the points listed in ws->queue[0 .. counters[0]) with the serial arithmetic, reading the
 * exact transposed centroids ws->means_t ([dim][kp]) that pack_means wrote for this call. */
int launch_recheck(const AssignArgs& a, Workspace* ws, uint32_t kp);
void set_queued_rows_limit(size_t bytes); /* bound of the block of copied rows */
size_t queued_rows_limit();
/* The exact pass behind the split-bf16 sweep for k >= 128 and rows of more than 32 dimensions: the queued rows are copied into a compact block, a second
 * split-bf16 sweep over them notes the (row, centroid) pairs within the threshold (assign_bf16.hip), and one lane
 * per pair evaluates the serial arithmetic. */
int launch_recheck_screened(const AssignArgs& a, Workspace* ws, uint32_t kp, const DeviceInfo& dev);
uint32_t screened_rows_cap(const AssignArgs& a); /* queue entries the screened exact pass has rows for */
int launch_screen_bf16(const float* rows, const Workspace* ws, const uint32_t* row_queue, const uint32_t* row_count,
                       uint32_t* pairs, uint32_t* item_pairs, unsigned long long* keys, uint32_t dim, uint32_t k, uint32_t kp,
                       const DeviceInfo& dev, uint32_t* waves);
uint32_t screen_unit_rows(uint32_t dim);

/* assign_mfma.hip / assign_lds_fma.hip: return KMX_ERR_UNSUPPORTED (without message side effects
 * beyond kmx_last_error) when the shape does not fit the variant. */
/* shared by both fast variants: packed centroids (-2c rows of dp floats, kp rows), norms, transposed copy, empty queue */
struct ClearOutputs { float* means; size_t words; uint32_t* sizes; }; /* outputs to clear on the way (means: nullptr: none) */
int launch_pack_means(const AssignArgs& a, Workspace* ws, uint32_t dp, uint32_t kp, uint32_t moved, const ClearOutputs& clear = {}); /* FRAME_KEPT, FRAME_MOVED, FRAME_MOVED_IF_FAR (assign_mfma_impl.h) */
bool mfma_supports(const AssignArgs& a, const DeviceInfo& dev);
int launch_assign_mfma(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);
bool bf16_supports(const AssignArgs& a, uint32_t lds_budget, const DeviceInfo& dev); /* (the budget decides for rows of more than 256 dimensions; the launchers of narrower ones say what they need) */
int launch_assign_bf16(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);
/* rank16.hip: one half-precision product per dimension for all points, the serial result for what that leaves */
bool rank16_supports(const AssignArgs& a, uint32_t lds_budget);
/* assign_cells.hip: rows of 2 to 4 dimensions through a grid; half: where the exact pass finds its norms, frame and scale */
struct Cells16 {
	const float* norms; const float* low2; const float* frame; float* scale;
	uint32_t kp; float kd;
};
bool takes_cells(const AssignArgs& a, uint32_t lds_budget); /* KMX_ASSIGN_MFMA_BF16X3 runs as cells (assign_bf16.hip) */
bool cells_support(const AssignArgs& a, uint32_t lds_budget);
int launch_cells(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, const Cells16& half, bool choose); /* choose: may leave all points to the packed sweep (WAY_BACK_COUNTER) */
int launch_assign_cells(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev); /* rank16.hip: all of it */
bool sweep_writes_rows(const AssignArgs& a, const kmx_exec_params* exec, const DeviceInfo& dev); /* KMX_ASSIGN_BEST would write a.rows_out */
int launch_assign_rank16(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);
/* assign_wide.hip: rows of more than 256 dimensions (the split-bf16 variant's launcher passes them on) */
bool wide_supports(const AssignArgs& a, uint32_t lds_budget);
bool wide16_supports(const AssignArgs& a, uint32_t lds_budget); /* ... in half precision, nothing left to the caller */
int launch_assign_wide(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);
bool lds_fma_supports(const AssignArgs& a, const DeviceInfo& dev);
bool lds_fma_reads_through_scalar_cache(const AssignArgs& a); /* a handful of centroids: no LDS staging */
int launch_assign_lds_fma(const AssignArgs& a, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);

/* small.hip: small inputs in one launch each (assignment, update), floats and doubles */
template <typename F> bool small_assign_fits(int layout, uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget);
template <typename F> bool small_update_fits(uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget, const DeviceInfo& dev);
/* lds_budget: the one that small_assign_fits or small_iteration_fits was asked with */
template <typename F>
int launch_assign_small(const F* data, int layout, size_t stride, const F* means, int layout_means, size_t stride_means, uint32_t* assignment,
                        uint32_t dim, uint32_t k, uint32_t n, uint32_t* counters, uint32_t* blocks, uint32_t lds_budget);
template <typename F>
int launch_update_small(const F* data, int layout, size_t stride, const uint32_t* assignment, F* means, int layout_means, size_t stride_means, uint32_t* sizes,
                        uint32_t dim, uint32_t k, uint32_t n, bool divide, uint32_t* blocks, const DeviceInfo& dev);
/* the assignment of small inputs that also adds its points up: partial sums and counts of *blocks work-groups (at most
 * assign_small_max_blocks(n), small_plan.h), for launch_reduce_partials */
int launch_assign_small_sums(const AssignArgs& a, float* partial, uint32_t* partial_counts, uint32_t* blocks, uint32_t* counters, uint32_t lds_budget);
bool small_iteration_fits(int layout, uint32_t dim, uint32_t k, uint32_t n, uint32_t lds_budget);
inline uint32_t lds_budget_of(const kmx_exec_params* exec, const DeviceInfo& dev)
{
	return exec->shared_mem_bytes && exec->shared_mem_bytes < dev.lds_bytes ? exec->shared_mem_bytes : dev.lds_bytes;
}

/* update.hip */
/* means and sizes from the partial sums [chunks][k][dim] and counts [chunks][k] */
template <typename F>
int launch_reduce_partials(const F* partial, const uint32_t* partial_counts, uint32_t chunks, F* means, int layout_means, size_t stride_means, uint32_t* sizes, uint32_t dim, uint32_t k, bool divide);
/* update_sums64.hip: the update where the clusters' sums fit LDS as doubles. *done: means and sizes are finished; otherwise it is not for this shape.
 * Doubles whose launches are recorded take no work space (ws may be null) */
template <typename F>
int launch_update_sums64(const F* data, int layout, size_t stride, const uint32_t* assignment, F* means, int layout_means, size_t stride_means, uint32_t* sizes,
                         uint32_t dim, uint32_t k, uint32_t n, bool divide, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev, bool* done);
/* floats: whether it takes SoA points as they are */
bool sums64_takes_columns(uint32_t dim, uint32_t k, uint32_t n, const kmx_exec_params* exec, const Workspace* ws, const DeviceInfo& dev);
/* the work space of kmx_update_f32_noalloc on the current device: `partials` is the library's static scratch array */
int noalloc_workspace(Workspace** ws);
Workspace* fixed_scratch(); /* the same where its address is known, else null */
bool recording_graph(); /* between kmx_graph_begin and kmx_graph_end */
bool launches_recorded(); /* the same, or the caller records the stream it has set */
void scratch_recorded(); /* the launches that are recorded use the static scratch array */
int launch_update(int variant, const UpdateArgs& u, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);
/* whether launch_update would copy the SoA points of u into AoS rows first, and that copy: ws->rows_copy, rows of dim floats */
bool update_wants_rows(int variant, const UpdateArgs& u, const kmx_exec_params* exec, const Workspace* ws, const DeviceInfo& dev);
int launch_rows_from_soa(const float* data, size_t stride, uint32_t dim, uint32_t n, Workspace* ws, const DeviceInfo& dev);

/* update_ordered.hip: KMX_UPDATE_SERIAL_ORDER for floats and doubles -- stable counting sort of the point numbers by
 * cluster, then one lane per (cluster, coordinate) adds the members in ascending point order and divides: the bits of
 * the serial loop. Scratch (chunk histograms, cluster starts, the sorted point numbers: about n + 2^21 words) is taken
 * from ws->partials. */
template <typename F>
int launch_update_serial_order(const F* data, int layout, size_t stride, const uint32_t* assignment,
                               F* means, int layout_means, size_t stride_means, uint32_t* cluster_sizes,
                               uint32_t dim, uint32_t k, uint32_t n, bool divide, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);

/* f64.hip: the double-precision calls keep their own transposed centroids; the runtime grows the buffer under the
 * rules of the work space (not while a graph is recorded, after the stream has drained) and releases it on shutdown */
int reserve_f64(double** ptr, size_t* cap, size_t doubles);
int release_f64_workspace();
/* [dst, dst + bytes) is about to be written or released (bytes = 0: extent unknown): if the points announced by
 * kmx_prepare_points_f64 lie there, their float copy is forgotten */
void forget_prepared_points_f64(const void* dst, size_t bytes);

/* fused_small.hip: one pass over the points for a handful of centroids. a.assignment is a scratch vector of n entries
 * (only the entries of the points left to the exact pass are written); means_out and sizes are zero on entry and hold
 * sums and counts on return (the caller divides). */
bool fused_small_supports(uint32_t dim, uint32_t k, int layout, size_t stride, uint32_t n);
int launch_fused_small(const AssignArgs& a, float* means_out, uint32_t* sizes, size_t clear_words, kmx_exec_params* exec, Workspace* ws, const DeviceInfo& dev);

} // namespace kmx

#endif
