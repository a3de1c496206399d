// Ahead of the one-kernel reverse sweep, for a batch with a long row of evaluation times in no order: every sample's points ordered by
// the iteration that wrote them.  The sweep makes such lists by itself where it meets such a row, one thread to a sample; what
// bounds it there is the chain of loads of one search after the other, so for long rows they are made here, a thread to a point.  (Eight
// searches side by side in the sweep's own code were as quick, but moved its scalar registers about: -11 to +13 % for float64 rows
// in order.)  Van der Pol, two points of every row swapped, lists and sweep, before and after: B = 65 536, 65 points 0.76 and 0.60 ms
// in float32, 1.01 and 0.75 in float64; 400 points 4.22 and 2.79, 4.95 and 3.26; B = 64, 4000 points 20.9 and 16.1, 23.6 and 19.5.
#include "tode_internal.h"

namespace tode {

// Which iteration wrote which evaluation point (adjoints.py:215-234: the first whose new time has reached it; none for
// a point at t_start, which the loop's set-up writes, and for one the solve never reached): one thread per point, a
// binary search over the sample's recorded times.
template <typename T>
__global__ void __launch_bounds__(256) backward_hits_kernel(long long B, int E, long long L, const T *t_start, long long ts_stride, const T *t_end, long long te_stride,
                                                            const T *t_eval, const T *rec_t, int32_t *iterations_sorted, int32_t *points_by_iteration) {
    const long long at_point = (long long)blockIdx.x * 256 + threadIdx.x;
    if (at_point >= B * E) return;
    const long long b = at_point / E;
    const int e = (int)(at_point - b * E);
    const T ts = t_start[b * ts_stride], dir = t_end[b * te_stride] > ts ? (T)1 : (T)-1;
    const T at = t_eval[at_point], v = dir * at;
    long long lo = 0, hi = L;
    while (lo < hi) {
        const long long mid = (lo + hi) / 2;
        if (dir * rec_t[(mid + 1) * B + b] < v) lo = mid + 1;
        else hi = mid;
    }
    int32_t hit = lo < L ? (int32_t)lo : -1;
    if (e == 0 && at == ts) hit = -1;
    iterations_sorted[at_point] = hit, points_by_iteration[at_point] = e;
}

// Each sample's points ordered by that iteration (stable: points of one iteration stay in their order).  One thread per sample.
// Rows that run in the direction of the solve are in order already, which a look along the row shows; the others are
// sorted by insertion.
static __global__ void __launch_bounds__(64) backward_order_kernel(long long B, int E, int32_t *iterations_sorted, int32_t *points_by_iteration) {
    const long long b = (long long)blockIdx.x * 64 + threadIdx.x;
    if (b >= B) return;
    int32_t *its = iterations_sorted + b * E, *pts = points_by_iteration + b * E;
    bool ordered = true;
    for (int e = 1; e < E; ++e) ordered = ordered && its[e - 1] <= its[e];
    if (ordered) return;
    for (int e = 1; e < E; ++e) {
        const int32_t hit = its[e], point = pts[e];
        int j = e - 1;
        for (; j >= 0 && its[j] > hit; --j) its[j + 1] = its[j], pts[j + 1] = pts[j];
        its[j + 1] = hit, pts[j + 1] = point;
    }
}

// Whether some row does not run in the direction of its solve (as the sweep sees it: a time that is not a number is in no order).
template <typename T>
__global__ void __launch_bounds__(256) unordered_rows_kernel(long long B, int E, const T *t_start, long long ts_stride, const T *t_end, long long te_stride, const T *t_eval, int32_t *flags) {
    const long long at_point = (long long)blockIdx.x * 256 + threadIdx.x;
    if (at_point >= B * E) return;
    const long long b = at_point / E;
    if (at_point == b * E) return;
    const T dir = t_end[b * te_stride] > t_start[b * ts_stride] ? (T)1 : (T)-1;
    if (!(dir * t_eval[at_point - 1] <= dir * t_eval[at_point])) flags[TODE_FLAG_NON_MONOTONE] = 1;
}

template <typename T> static int unordered_rows(const tode_solve_args &a, hipStream_t s) {
    hipLaunchKernelGGL((unordered_rows_kernel<T>), dim3((unsigned)((a.batch * a.n_eval + 255) / 256)), dim3(256), 0, s, (long long)a.batch, a.n_eval, (const T *)a.t_start,
                       (long long)a.t_start_stride, (const T *)a.t_end, (long long)a.t_end_stride, (const T *)a.t_eval, a.flags);
    return check_hip(hipGetLastError(), "tode_mark_unordered_rows launch");
}

template <typename T> static int backward_lists(const tode_solve_args &a, const tode_solve_adjoint &adj, hipStream_t s) {
    const long long B = a.batch, points = B * a.n_eval;
    int32_t *its = (int32_t *)adj.scratch, *pts = its + points;
    hipLaunchKernelGGL((backward_hits_kernel<T>), dim3((unsigned)((points + 255) / 256)), dim3(256), 0, s, B, a.n_eval, (long long)adj.iterations, (const T *)a.t_start,
                       (long long)a.t_start_stride, (const T *)a.t_end, (long long)a.t_end_stride, (const T *)a.t_eval, (const T *)a.record->t, its, pts);
    hipLaunchKernelGGL(backward_order_kernel, dim3((unsigned)((B + 63) / 64)), dim3(64), 0, s, B, a.n_eval, its, pts);
    return check_hip(hipGetLastError(), "tode_solve_backward_lists launch");
}

}  // namespace tode

namespace tode {
// what both entry points read of the arguments, and that one launch takes the points
static int check_rows(const tode_solve_args *a) {
    if (a->batch < 0 || a->n_features <= 0 || a->n_eval < 1) return fail(TODE_E_INVALID, "bad sizes");
    if (a->t_start_stride < 1 || a->t_end_stride < 1) return fail(TODE_E_INVALID, "t_start_stride / t_end_stride must be >= 1");
    if (!known_dtype(a->dtype)) return fail(TODE_E_INVALID, "unknown dtype %d", a->dtype);
    if (a->dtype & TODE_DTYPE_PAIR) return fail(TODE_E_UNSUPPORTED, "the whole reverse sweep is built for time and data in one dtype");
    if (a->batch > 0 && (!a->t_start || !a->t_end || !a->t_eval)) return fail(TODE_E_INVALID, "null pointer");
    if (a->batch > 0xffffff00ll / a->n_eval) return fail(TODE_E_UNSUPPORTED, "too many evaluation points for one launch: leave the lists to the sweep");
    return TODE_OK;
}
}  // namespace tode

extern "C" {

int tode_mark_unordered_rows(const tode_solve_args *a, void *stream) {
    using namespace tode;
    if (!a) return fail(TODE_E_INVALID, "null argument struct");
    const int rc = check_rows(a);
    if (rc || a->batch == 0) return rc;
    if (!a->flags) return fail(TODE_E_INVALID, "null pointer");
    return a->dtype == TODE_F32 ? unordered_rows<float>(*a, (hipStream_t)stream) : unordered_rows<double>(*a, (hipStream_t)stream);
}

int tode_solve_backward_lists(const tode_solve_args *a, const tode_solve_adjoint *adj, void *stream) {
    using namespace tode;
    if (!a || !adj) return fail(TODE_E_INVALID, "null argument struct");
    const int rc = check_rows(a);
    if (rc) return rc;
    if (!a->record || !a->record->t || adj->iterations < 0 || a->record->capacity < adj->iterations + 1) return fail(TODE_E_INVALID, "no record of that many iterations");
    if (!adj->scratch || adj->scratch_bytes < tode_solve_backward_scratch_bytes(a))
        return fail(TODE_E_INVALID, "the scratch buffer holds %lld bytes, these lists need %lld (tode_solve_backward_scratch_bytes)", (long long)(adj->scratch ? adj->scratch_bytes : 0),
                    (long long)tode_solve_backward_scratch_bytes(a));
    if (a->batch == 0) return TODE_OK;
    return a->dtype == TODE_F32 ? backward_lists<float>(*a, *adj, (hipStream_t)stream) : backward_lists<double>(*a, *adj, (hipStream_t)stream);
}

}  // extern "C"
