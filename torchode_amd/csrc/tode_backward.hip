// Reverse sweep over a whole recorded solve with a built-in right-hand side, in one kernel.
//
// The reference differentiates its loop through the graph of torch operations that autograd kept of it
// (adjoints.py:33-40, 111-113, 135-260).  Here the forward pass left a record of the loop state before every
// iteration (tode_solve_record).  One thread per sample walks its iterations from the last to the first: it forms
// the six stages again from the recorded state (registers, the right-hand side evaluated in the kernel), pulls the
// cotangents of the state after the iteration and of the evaluation points the iteration wrote through everything
// after the stages, then through the stages from the last to the first, with the
// right-hand side's own vector-Jacobian product in closed form where the per-iteration path asks autograd for it.
// Everything a sample's thread works on -- stage derivatives, their cotangents, the cotangents of the state -- is an
// array private to the thread, indexed by constants (registers).  What an iteration reads is loaded while the one before is
// worked on: its entry of the record, and the evaluation points it may have written.
#include "tode_adjoint.h"

// Largest number of groups of 64 samples that take two wavefronts each (launch_backward); half as many in float64.
#ifndef TODE_PAIRED_SWEEP_GROUPS
#define TODE_PAIRED_SWEEP_GROUPS 1024
#endif

namespace tode {

template <typename T> struct WholeBackward {
    long long batch, iterations;  // iterations: L, the record holds entries 0..L
    int E, through_control;
    const T *t_start, *t_end, *t_eval, *grad_ys;
    T *g_t_start, *g_t_end, *g_t_eval;
    CtrlParams<T> cp;
    T dt_min, dt_max;
    const T *rec_t, *rec_dt, *rec_y, *rec_k0, *rec_prev, *rec_pprev;
    const int32_t *rec_running, *rec_n_accepted;
    const T *params;
    double scalars[4];
    T *a_y, *a_k0, *a_t, *a_dt, *a_prev, *a_pprev;  // results: cotangents of the state before the first iteration
    T *g_params;  // [B,P] result
    // the evaluation points of every sample ordered by the iteration that wrote them, where the caller hands them in: [B,E]
    // point indices and, in the same order, the iterations (-1 first: points no iteration wrote)
    const int32_t *points_by_iteration, *iterations_sorted;
    int32_t *lists;  // room for both, for wavefronts with a row of times in no order (list_points)
    long long ts_stride, te_stride;  // t_start / t_end: sample b at element b * stride
    int through_start;  // also carry the cotangents through the start of the loop (start_backward); 2: and a point at t_start's
    int dt0_given;      // the first step was the caller's, not the start rule's
    int plain;          // tolerances and exponents in the ranges of the short forms
};

template <typename T, int F> struct RecordEntry {
    T t, dt, prev, pprev, y[F], k0[F];
    int32_t running, n_accepted;
};

template <typename T, int F> __device__ __forceinline__ RecordEntry<T, F> load_entry(const WholeBackward<T> &w, long long entry, long long sample) {
    const long long at = entry * w.batch + sample;
    RecordEntry<T, F> r;
    r.t = w.rec_t[at], r.dt = w.rec_dt[at], r.prev = w.rec_prev[at], r.pprev = w.rec_pprev[at];
#pragma unroll
    for (int f = 0; f < F; ++f) r.y[f] = w.rec_y[at * F + f], r.k0[f] = w.rec_k0[at * F + f];
    r.running = w.rec_running[at], r.n_accepted = w.rec_n_accepted[at];
    return r;
}

// A loaded entry waited for here and not where its values are copied at the end of the iteration: there the wait is behind the
// loads of the next evaluation points, and would be for those too.
template <typename T, int F> __device__ __forceinline__ void entry_is_here(RecordEntry<T, F> &r) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(r.t), "+v"(r.dt), "+v"(r.prev), "+v"(r.pprev), "+v"(r.running), "+v"(r.n_accepted));
#pragma unroll
    for (int f = 0; f < F; ++f) asm volatile("" : "+v"(r.y[f]), "+v"(r.k0[f]));
#endif
}

// cotangent shares of minimum(a, b) (or maximum with the comparison turned round) for operand a: all of it where a
// is the one taken, half on a tie (torch.minimum / torch.maximum)
template <typename T> __device__ __forceinline__ T share_of_min(T a, T b) { return a < b ? (T)1 : (a == b ? (T)0.5 : (T)0); }
template <typename T> __device__ __forceinline__ T share_of_max(T a, T b) { return a > b ? (T)1 : (a == b ? (T)0.5 : (T)0); }

// cotangent of v given that of rms(v) = |v / sqrt(F)|_2 (zero where the norm is zero, as torch.linalg.vector_norm)
template <typename T, int F> __device__ __forceinline__ void rms_backward(const T (&v)[F], T norm, T g, T (&gv)[F]) {
    const T sf = (T)__builtin_sqrt((double)F);
#pragma unroll
    for (int f = 0; f < F; ++f) gv[f] = norm != (T)0 ? (g * ((v[f] / sf) / norm)) / sf : (T)0;
}

// The start of the loop reversed: y = y0, k0 = f(t_start, y0) and, unless the caller gave the first step, the step of
// the start rule (step_size_controllers.py:431-490 / 776-835, written out in initial_step) clamped to the time range
// (adjoints.py:86-93).  In: the cotangents a_y, a_k0, a_dt of that first loop state.  Out: a_y becomes the cotangent
// of y0, gpar gains the right-hand side's parameters' share.  The times are constants here (a caller that wants their
// gradients takes the first state's cotangents and does this part itself), and the right-hand side does not depend
// on t (none of the built-in ones does).
template <typename T, int CTRL, typename Term>
__device__ __forceinline__ void start_backward(const CtrlParams<T> &cp, const Term &rhs, const bool through_rule, const T ts, const T te,
                                               const T (&y0)[Term::F], const T (&f0)[Term::F], T (&a_y)[Term::F], const T (&a_k0)[Term::F],
                                               const T a_dt, T (&gpar)[Term::P]) {
    constexpr int F = Term::F;
    T g_y0[F], g_f0[F];
#pragma unroll
    for (int f = 0; f < F; ++f) g_y0[f] = a_y[f], g_f0[f] = a_k0[f];
    if (through_rule && a_dt != (T)0) {
        // ---- forward values (initial_step) ----
        const T dir = te > ts ? (T)1 : (T)-1, span = abs_(te - ts);
        T inv[F], u[F], v[F], w[F], y1[F], f1[F];
#pragma unroll
        for (int f = 0; f < F; ++f) inv[f] = (T)1 / fma_(cp.rtol, abs_(y0[f]), cp.atol), u[f] = y0[f] * inv[f], v[f] = f0[f] * inv[f];
        const T d0 = rms<T, F>(u), d1 = rms<T, F>(v);
        const bool small = d0 < (T)1e-5 || d1 < (T)1e-5;
        const T h0a = small ? (T)1e-6 : ((T)0.01 * d0) / d1;
        const T h0 = tmin(h0a, span);
        const T dh = dir * h0;
#pragma unroll
        for (int f = 0; f < F; ++f) y1[f] = fma_(dh, f0[f], y0[f]);
        const T t1 = fma_(dir, h0, ts);
        rhs(t1, y1, f1);
#pragma unroll
        for (int f = 0; f < F; ++f) w[f] = (f1[f] - f0[f]) * inv[f];
        const T r2 = rms<T, F>(w);
        const bool blocked = CTRL == 0 && h0 == (T)0;  // (the integral controller's copy of the rule: d2 = inf)
        const T d2 = blocked ? (T)__builtin_huge_val() : r2 / h0;
        const T m = tmax(d1, d2);
        const bool tiny = m <= (T)1e-15;
        const T z = ((T)1 / m) * (T)0.01;
        const T h1 = tiny ? tmax((T)1e-6, h0 * (T)1e-3) : rpow<T>(z, 1.0 / 5.0);
        const T first = dir * tmin((T)100 * h0, h1);
        const T lo = tmin(ts, te) - ts, hi = tmax(te, ts) - ts;
        // ---- reversed ----
        // torch.clamp(first, lo, hi) (adjoints.py:107): the whole cotangent stays with the step where it lies within
        // the bounds, the bounds included (another rule than minimum / maximum, which halve it on a tie)
        const T g_first = (first >= lo && first <= hi) ? a_dt : (T)0;
        const T g_min = g_first * dir;
        T g_h0 = (T)100 * (g_min * share_of_min<T>((T)100 * h0, h1));
        const T g_h1 = g_min * share_of_min<T>(h1, (T)100 * h0);
        T g_d1 = 0, g_d2 = 0;
        if (tiny) {
            g_h0 += (h0 * (T)1e-3 >= (T)1e-6) ? g_h1 * (T)1e-3 : (T)0;
        } else {
            const T g_z = g_h1 * ((T)(1.0 / 5.0) * rpow<T>(z, 1.0 / 5.0 - 1.0));
            const T rm = (T)1 / m;
            const T g_m = -(g_z * (T)0.01) * rm * rm;
            g_d1 = g_m * share_of_max<T>(d1, d2);
            g_d2 = g_m * share_of_max<T>(d2, d1);
        }
        T g_inv[F];
#pragma unroll
        for (int f = 0; f < F; ++f) g_inv[f] = 0;
        if (!blocked && g_d2 != (T)0) {
            const T g_r2 = g_d2 / h0;
            g_h0 += -g_d2 * r2 / (h0 * h0);
            T g_w[F], g_f1[F], g_y1[F];
            rms_backward<T, F>(w, r2, g_r2, g_w);
#pragma unroll
            for (int f = 0; f < F; ++f) g_f1[f] = g_w[f] * inv[f], g_f0[f] -= g_w[f] * inv[f], g_inv[f] += g_w[f] * (f1[f] - f0[f]);
            rhs.vjp(t1, y1, g_f1, g_y1, gpar);
            T g_step = 0;
#pragma unroll
            for (int f = 0; f < F; ++f) g_y0[f] += g_y1[f], g_f0[f] += g_y1[f] * dh, g_step += g_y1[f] * f0[f];
            g_h0 += g_step * dir;
        }
        const T g_h0a = g_h0 * share_of_min<T>(h0a, span);
        if (!small) {
            const T q = (T)0.01 * d0;
            g_d1 += -g_h0a * q / (d1 * d1);
            const T g_d0 = (T)0.01 * (g_h0a / d1);
            T g_u[F];
            rms_backward<T, F>(u, d0, g_d0, g_u);
#pragma unroll
            for (int f = 0; f < F; ++f) g_y0[f] += g_u[f] * inv[f], g_inv[f] += g_u[f] * y0[f];
        }
        {
            T g_v[F];
            rms_backward<T, F>(v, d1, g_d1, g_v);
#pragma unroll
            for (int f = 0; f < F; ++f) g_f0[f] += g_v[f] * inv[f], g_inv[f] += g_v[f] * f0[f];
        }
#pragma unroll
        for (int f = 0; f < F; ++f) g_y0[f] += (-g_inv[f] * inv[f] * inv[f]) * cp.rtol * sign_(y0[f]);
    }
    T g_from_f0[F];
    rhs.vjp(ts, y0, g_f0, g_from_f0, gpar);
#pragma unroll
    for (int f = 0; f < F; ++f) a_y[f] = g_y0[f] + g_from_f0[f];
}

// Which iteration wrote which evaluation point (adjoints.py:215-234: the first whose new time has reached it; none for
// a point at t_start, which the loop's set-up writes, and for one the solve never reached), for a row of times in no order:
// a binary search over the sample's recorded times for each point, and the points sorted by insertion (stable: points of one
// iteration stay in their order).  One thread per sample; rows whose times run in the direction of the solve, nearly all
// there are, never come here (the sweep meets their points in order), and long ones in no order have their lists handed in
// (tode_solve_backward_lists).
template <typename T>
__device__ __forceinline__ void list_points(const WholeBackward<T> &w, const long long sample, const T ts, const T dir, const T *t_eval, int32_t *its, int32_t *pts) {
    for (int e = 0; e < w.E; ++e) {
        const T at = t_eval[e], v = dir * at;
        long long lo = 0, hi = w.iterations;
        while (lo < hi) {
            const long long mid = (lo + hi) / 2;
            if (dir * w.rec_t[(mid + 1) * w.batch + sample] < v) lo = mid + 1;
            else hi = mid;
        }
        int32_t hit = lo < w.iterations ? (int32_t)lo : -1;
        if (e == 0 && at == ts) hit = -1;
        int j = e - 1;
        for (; j >= 0 && its[j] > hit; --j) its[j + 1] = its[j], pts[j + 1] = pts[j];
        its[j + 1] = hit, pts[j + 1] = e;
    }
}

// Dividends of short-form quotients (quotient_with): zero, or from 2^-90 to 2^80 (float64: 2^-700 to 2^700), with divisors from
// 2^-40 to 2^20, so that no quotient and no remainder is subnormal.  outside(): the lanes, of those that run, with one that is
// not; those that are not numbers count among them.
template <typename T> struct Dividends {
    static constexpr int smallest = sizeof(T) == 4 ? -90 : -700, largest = sizeof(T) == 4 ? 80 : 700;
    unsigned least = 0xffffffffu, most = 0;
    __device__ __forceinline__ Dividends() {}
    __device__ __forceinline__ Dividends(T a) { add(a); }
    __device__ __forceinline__ Dividends(T a, T b) { add(a), add(b); }
    __device__ __forceinline__ void add(T a) {
        const unsigned bits = high_bits(abs_(a));
        least = min(least, bits - 1u), most = max(most, bits);  // (zero wraps round to the largest)
    }
    __device__ __forceinline__ lanes_t outside() const {
        return lanes_where(least < power_of_two_bits<T>(smallest) - 1u) | lanes_where(most >= power_of_two_bits<T>(largest));
    }
};

// What the reverse of an iteration needs of the iteration itself: the stages again (runge_kutta.py:255-263), the error ratio
// and the step factor before its clip.  None of it waits for a cotangent.
template <typename T, int F> struct Formed {
    T k[7][F], yi[7][F], y1[F];
    T err[F], eb[F], per_eb[F], q[F], x[F], r, ratio, F0;
    bool bounds_outside;  // this lane's error bounds or history are outside the short forms' ranges
};
// With the sum of the errors' squares in front of the rest, for the kernels that form the errors later (LATER below).
template <typename T> struct KeptSum {
    T acc;
};
template <typename T, int F> struct FormedLater : KeptSum<T>, Formed<T, F> {};
template <typename T, int F> __device__ __forceinline__ T &sum_of_squares(Formed<T, F> &, T &own) { return own; }
template <typename T, int F> __device__ __forceinline__ T &sum_of_squares(FormedLater<T, F> &o, T &) { return o.acc; }

template <typename T, int METHOD, typename Term>
__device__ __forceinline__ void form_stages(const Term &rhs, const RecordEntry<T, Term::F> &here, Formed<T, Term::F> &o) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    constexpr int F = Term::F;
    const T t0 = here.t, dt = here.dt;
    const T(&y)[F] = here.y;
#pragma unroll
    for (int f = 0; f < F; ++f) o.k[0][f] = here.k0[f];
#pragma unroll
    for (int s = 1; s < 7; ++s) {
#pragma unroll
        for (int f = 0; f < F; ++f) {
            T sum = 0;
#pragma unroll
            for (int j = 0; j < s; ++j) sum = fma_((T)Tab::a[s][j], o.k[j][f], sum);
            o.yi[s][f] = fma_(dt, sum, y[f]);
        }
        rhs(fma_((T)Tab::c[s], dt, t0), o.yi[s], o.k[s]);
    }
#pragma unroll
    for (int f = 0; f < F; ++f) o.y1[f] = o.yi[6][f];
}

// Returns bounds_outside of all lanes.
template <typename T, int METHOD, int CTRL, typename Term, typename O>
__device__ __forceinline__ lanes_t form_errors(const WholeBackward<T> &w, const RecordEntry<T, Term::F> &here, const bool running_new, O &o) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    constexpr int F = Term::F;
    constexpr bool SHORT = F * sizeof(T) <= 32;
    const CtrlParams<T> &cp = w.cp;
    const T sf = (T)__builtin_sqrt((double)F);
    const T dt = here.dt, prev = here.prev, pprev = here.pprev;
    const T(&y)[F] = here.y;
    using Div = DivSqrtFeatures<T, F>;
    // error ratio and step factor, in the short forms where every lane's operands are in their ranges (control_common's,
    // over a wider range of the errors: their squares may vanish in the sum, as they do in the general form).  A sample
    // that sits through an iteration with a zero step has an error of zero; its controller's results reach nothing.
    T own, &acc = sum_of_squares<T, F>(o, own);
    acc = 0;
    lanes_t outside = 0, bounds_outside = 0;
    unsigned smallest = 0xffffffffu;
    T largest_eb = 0;
#pragma unroll
    for (int f = 0; f < F; ++f) {
        o.err[f] = 0;
#pragma unroll
        for (int s = 0; s < 7; ++s) o.err[f] = fma_(dt * (T)Tab::b_err[s], o.k[s][f], o.err[f]);
        if constexpr (SHORT) {
            o.eb[f] = fma_(cp.rtol, max_abs(y[f], o.y1[f]), cp.atol);
            o.per_eb[f] = reciprocal_estimate(o.eb[f]);
            o.q[f] = quotient_with(abs_(o.err[f]), o.eb[f], o.per_eb[f]);
            o.x[f] = Div::fast(o.q[f]);
            smallest = min(smallest, min(high_bits(abs_(o.err[f])) - 1u, high_bits(o.q[f]) - 1u));  // (zero wraps round to the largest)
            largest_eb = f == 0 ? o.eb[f] : max_ordered(largest_eb, o.eb[f]);
            acc = fma_(o.x[f], o.x[f], acc);
        }
    }
    if constexpr (SHORT) {
        constexpr unsigned from = power_of_two_bits<T>(-40), width = power_of_two_bits<T>(16) - from;
        const bool idle = acc == (T)0 && !running_new;
        acc = idle ? (T)1 : acc;
        bounds_outside = lanes_where(!(largest_eb <= (T)0x1p+20));
        outside = lanes_where(smallest < power_of_two_bits<T>(Dividends<T>::smallest) - 1u) | lanes_where(high_bits(acc) - from >= width) | bounds_outside;
        o.r = o.ratio = sqrt_plain(acc);
        o.F0 = cp.safety * expk<true>(dw_mul(logk<true>(o.ratio), (T)cp.e1));
        if (CTRL == 1 && !cp.skip2) o.F0 = o.F0 * expk<true>(dw_mul(logk<true>(prev), (T)cp.e2));
        if (CTRL == 1 && !cp.skip3) o.F0 = o.F0 * expk<true>(dw_mul(logk<true>(pprev), (T)cp.e3));
        constexpr unsigned history = power_of_two_bits<T>(-20), history_width = power_of_two_bits<T>(20) - history;
        lanes_t history_outside = 0;
        if (CTRL == 1 && !cp.skip2) history_outside |= lanes_where(high_bits(prev) - history >= history_width);
        if (CTRL == 1 && !cp.skip3) history_outside |= lanes_where(high_bits(pprev) - history >= history_width);
        outside |= history_outside, bounds_outside |= history_outside;
    }
    if (!SHORT || !w.plain || outside) {
        acc = 0;
#pragma unroll
        for (int f = 0; f < F; ++f) {
            o.eb[f] = fma_(cp.rtol, tmax(abs_(y[f]), abs_(o.y1[f])), cp.atol);
            o.q[f] = abs_(o.err[f]) / o.eb[f];
            o.x[f] = o.q[f] / sf;
            acc = fma_(o.x[f], o.x[f], acc);
        }
        o.r = sqrt_(acc), o.ratio = tmax(o.r, (T)1e-38);
        o.F0 = cp.safety * rpow<T>(o.ratio, cp.e1);
        if (CTRL == 1) {
            o.F0 = o.F0 * (cp.skip2 ? (T)1 : rpow<T>(prev, cp.e2));
            o.F0 = o.F0 * (cp.skip3 ? (T)1 : rpow<T>(pprev, cp.e3));
        }
    }
    o.bounds_outside = holds(bounds_outside);
    return bounds_outside;
}

// Coefficients of the dense output's derivative, lowest power first.
template <typename T, int METHOD, int F>
__device__ __forceinline__ void form_slope(T dt, const T (&y)[F], const T (&y1)[F], const T (&k)[7][F], int f, T (&slope)[4]) {
    const T ks[7] = {k[0][f], k[1][f], k[2][f], k[3][f], k[4][f], k[5][f], k[6][f]};
    T q[5][1];
    quartic_elem<T, METHOD>(dt, y[f], y1[f], ks, true, q);
    slope[0] = q[1][0], slope[1] = (T)2 * q[2][0], slope[2] = (T)3 * q[3][0], slope[3] = (T)4 * q[4][0];
}

// What one wavefront forms and another one uses, by way of LDS: 16 bytes of a lane's values at a time, lanes side by side, two
// iterations' worth.  The stage inputs are left out: the user has their sums in hand when it needs them.
template <typename T, int F> struct HandOver {
    static constexpr int PER = 16 / (int)sizeof(T), VALUES = 16 * F + 4, CHUNKS = (VALUES + PER - 1) / PER;
    struct alignas(16) Chunk {
        T v[PER];
    };
    static constexpr size_t bytes() { return 2 * sizeof(Chunk) * CHUNKS * 64; }
    Chunk *lane;  // [2][CHUNKS][64], at this lane
    int phase = 0;
    __device__ __forceinline__ HandOver(unsigned char *lds) : lane(reinterpret_cast<Chunk *>(lds) + (threadIdx.x & 63)) {}
    // every value in its place: the slopes last, which only iterations with an evaluation point read
    template <typename Each> static __device__ __forceinline__ void each(Formed<T, F> &o, Each each) {
        int at = 0;
#pragma unroll
        for (int f = 0; f < F; ++f) {
#pragma unroll
            for (int s = 1; s < 7; ++s) each(at++, o.k[s][f]);
            each(at++, o.y1[f]), each(at++, o.err[f]), each(at++, o.eb[f]), each(at++, o.per_eb[f]), each(at++, o.q[f]), each(at++, o.x[f]);
        }
        each(at++, o.r), each(at++, o.ratio), each(at++, o.F0);
    }
    static constexpr int SLOPES = 12 * F + 4, FIRST_SLOPE_CHUNK = SLOPES / PER;
    __device__ __forceinline__ void write(Formed<T, F> &o, const T (&slope)[F][4]) {
        T v[CHUNKS * PER] = {};
        each(o, [&](int at, T &value) { v[at] = value; });
        v[12 * F + 3] = o.bounds_outside ? (T)1 : (T)0;
#pragma unroll
        for (int f = 0; f < F; ++f)
#pragma unroll
            for (int j = 0; j < 4; ++j) v[SLOPES + 4 * f + j] = slope[f][j];
        Chunk *const to = lane + phase * CHUNKS * 64;
#pragma unroll
        for (int c = 0; c < CHUNKS; ++c) {
            Chunk chunk;
#pragma unroll
            for (int j = 0; j < PER; ++j) chunk.v[j] = v[c * PER + j];
            to[c * 64] = chunk;
        }
        phase ^= 1;
    }
    __device__ __forceinline__ void read(Formed<T, F> &o) {
        T v[(SLOPES + PER - 1) / PER * PER];
        const Chunk *const from = lane + phase * CHUNKS * 64;
#pragma unroll
        for (int c = 0; c * PER < SLOPES; ++c) {
            const Chunk chunk = from[c * 64];
#pragma unroll
            for (int j = 0; j < PER; ++j) v[c * PER + j] = chunk.v[j];
        }
        each(o, [&](int at, T &value) { value = v[at]; });
        o.bounds_outside = v[12 * F + 3] != (T)0;
        phase ^= 1;
    }
    __device__ __forceinline__ void read_slopes(T (&slope)[F][4]) {  // (after read)
        const Chunk *const from = lane + (phase ^ 1) * CHUNKS * 64;
#pragma unroll
        for (int c = FIRST_SLOPE_CHUNK; c < CHUNKS; ++c) {
            const Chunk chunk = from[c * 64];
#pragma unroll
            for (int j = 0; j < PER; ++j) {
                const int at = c * PER + j - SLOPES;
                if (at >= 0 && at < 4 * F) slope[at / 4][at % 4] = chunk.v[j];
            }
        }
    }
};

// What bounds this kernel is one thread's chain: B = 65536 is one wavefront per SIMD, and the slowest sample's 107
// iterations follow one another.  The evaluation points of an iteration are in registers before the iteration begins: AHEAD
// of them, from the last one that no iteration has met yet downwards, are loaded as soon as the iteration before has taken
// its own.  (Looked up in lists that two kernels in front of this one made, an iteration waited for memory two or three
// times, first for the number of its points, then for each point's index, then for its time and cotangent: Van der Pol float32,
// B = 65536, 50 points: 0.76 ms and 0.05 ms for the two kernels; 0.66 ms this way.)  What remains is instructions: the
// divisions, the square root and the two powers in the short forms of tode_math.h wherever the wavefront's operands allow
// them, 0.66 -> 0.53 ms; and the waits for what was loaded ahead only where it is used (they stood behind each point's index,
// and at the end of the iteration behind the copies of the record's entry): 0.53 -> 0.46, float64, B = 20 000, 0.56 -> 0.49.
// What does not wait for a cotangent -- the stages, the error ratio and the step factor's powers, the dense output's
// coefficients, 500 of 1800 instructions -- is formed by a second wavefront one iteration ahead (PAIR, form_stages, form_errors, HandOver; one
// barrier of LDS between them an iteration) where the SIMD has an issue slot to spare: 0.45 -> 0.355 ms at B = 65536.
// What is held for all this costs registers (one wavefront for everything): float32 rows of two take up to 182 (two wavefronts per SIMD; three before), rows of four
// 256 and 7 to 12 accumulation registers (one; two before), float64 rows of eight all 512 and 800 to 900 bytes of scratch.  It pays all the
// same where a SIMD has wavefronts to choose from.  Backward passes, before and now: Van der Pol float32, B = 262 144, 2.41 -> 1.11 ms,
// a million 7.9 -> 4.1; decay, float32 rows of four, 262 144, 1.00 -> 0.75, a million 3.00 -> 2.75; float64 rows of eight, 262 144,
// Dopri5 4.45 -> 4.17 and Tsit5 4.42 -> 3.81, a million 16.3 -> 15.8 and 16.3 -> 14.2.
template <typename T, int METHOD, int CTRL, typename Term, bool PAIR>
__global__ void __launch_bounds__(PAIR ? 128 : 64) whole_backward_kernel(const WholeBackward<T> w) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    constexpr int F = Term::F, P = Term::P;
    constexpr bool SHORT = F * sizeof(T) <= 32;  // the short forms (rows of eight doubles have no registers left for what they keep)
    constexpr int AHEAD = F <= 4 ? 4 : (SHORT ? 2 : 1);  // points held: a step of these systems passes one to four
    const long long B = w.batch;
    const long long g = (long long)blockIdx.x * 64 + (threadIdx.x & 63);  // this thread's sample
    if (g >= B) return;
    Term rhs;
    rhs.load(w.params + g * P, w.scalars);
    T gpar[P];
#pragma unroll
    for (int j = 0; j < P; ++j) gpar[j] = 0;

    // One wavefront for everything, float64, Tsit5 and PID, systems of several equations with one parameter: the errors are formed
    // behind the new time instead of right behind the stages.  It is the same arithmetic; what differs is the compiler's allocation,
    // which elsewhere is the better one with both in one place.  Right behind and later, B = 65 536, us: Van der Pol 482 and 467,
    // Lorenz 335 and 302; with a rate per value, rows of three and four, 270 and 288, 287 and 297.
    constexpr bool LATER = !PAIR && sizeof(T) == 8 && METHOD == 1 && CTRL == 1 && F > 1 && P == 1;

    const CtrlParams<T> &cp = w.cp;
    const int E = w.E;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    HandOver<T, F> hand(smem_raw);
    if constexpr (PAIR) {
        static_assert(SHORT, "built for the short forms");
        // The group's first wavefront forms; for rows of four doubles the second one.  Which of them does was measured to matter where
        // groups share a compute unit, and to the registers the compiler chooses; roles that take turns by the group's number are
        // slower (which SIMDs two groups' wavefronts share is not known here).  Taking turns and so, us: Van der Pol float32, 512 groups, 340 and 322, 768 339 and 316, 1024
        // 360 and 355; float64, 256 387 and 389, 313 468 and 400, 511 484 and 431.  Decay, rows of four doubles, first and second
        // wavefront: 5 groups 178 and 172, 256 187 and 183, 511 199 and 196.
        constexpr unsigned FORMS = F * sizeof(T) == 32 ? 1 : 0;
        if (threadIdx.x >> 6 == FORMS) {
            const long long L = w.iterations;
            RecordEntry<T, F> here = load_entry<T, F>(w, L > 0 ? L - 1 : 0, g);
            bool running_new = w.rec_running[L * B + g] != 0;
            for (long long i = L - 1; i >= 0; --i) {
                RecordEntry<T, F> before = load_entry<T, F>(w, i > 0 ? i - 1 : 0, g);
                if ((E == 0 && i == L - 1) || lanes_where(here.running != 0)) {  // (the iterations that the other wavefront asks for)
                    Formed<T, F> formed;
                    form_stages<T, METHOD, Term>(rhs, here, formed);
                    form_errors<T, METHOD, CTRL, Term>(w, here, running_new, formed);
                    T slope[F][4];
#pragma unroll
                    for (int f = 0; f < F; ++f) form_slope<T, METHOD, F>(here.dt, here.y, formed.y1, formed.k, f, slope[f]);
                    hand.write(formed, slope);
                    entry_is_here(before);
                    lds_barrier();
                }
                running_new = here.running != 0;
                here = before;
            }
            return;
        }
    }
    const T ts = w.t_start[g * w.ts_stride], te = w.t_end[g * w.te_stride];
    const T tlo = tmin(ts, te), thi = tmax(te, ts);
    const T sf = (T)__builtin_sqrt((double)F);
    const T *t_eval = E > 0 ? w.t_eval + g * E : nullptr;
    const T *grad_ys = w.grad_ys + g * (long long)(E > 0 ? E : 1) * F;

    T a_y[F], a_k0[F], a_t = 0, a_dt = 0, a_prev = 0, a_pprev = 0;  // cotangents of the state after the iteration: zeros behind the last one
#pragma unroll
    for (int f = 0; f < F; ++f) a_y[f] = 0, a_k0[f] = 0;

    const long long L = w.iterations;
    RecordEntry<T, F> after = load_entry<T, F>(w, L, g), here = load_entry<T, F>(w, L > 0 ? L - 1 : 0, g);

    // ---- the evaluation points, walked from the last to the first as the iterations are ----
    // Where every row of the wavefront runs in the direction of its solve, a point belongs to the iteration at hand if it
    // lies behind the time before it: those behind the time after it have been taken.  Elsewhere the lists say.
    const T dir = te > ts ? (T)1 : (T)-1;
    const int32_t *its = nullptr, *pts = nullptr;
    int lowest = 0, cursor = E - 1;
    bool listed = false;  // (a mask's truth, the same in all lanes: a scalar branch)
    if (E > 0) {
        bool in_order = w.points_by_iteration == nullptr;
        T last = t_eval[0];
        for (int e = 1; in_order && e < E; e += 8) {  // (eight loads on the way at a time: one by one they were fifty trips to memory)
            T next[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) next[j] = t_eval[min(e + j, E - 1)];
#pragma unroll
            for (int j = 0; j < 8; ++j) {  // (false for a time that is not a number)
                in_order = in_order && dir * last <= dir * next[j];
                last = next[j];
            }
        }
        listed = lanes_where(!in_order) != 0;
        if (listed) {
            its = w.iterations_sorted + g * E, pts = w.points_by_iteration + g * E;
            if (w.points_by_iteration == nullptr) {
                int32_t *const own = w.lists + g * E, *const own_points = own + B * E;
                list_points<T>(w, g, ts, dir, t_eval, own, own_points);
                its = own, pts = own_points;
            }
        } else {
            lowest = t_eval[0] == ts ? 1 : 0;  // (written by the loop's set-up)
            while (cursor >= lowest && dir * after.t < dir * t_eval[cursor]) --cursor;  // (never reached)
        }
    }
    T at[AHEAD], g_at[AHEAD][F];
    int32_t written_by[AHEAD];
    // (All indices before all values: an index taken from the lists, or the bare chance of one, is waited for where it is used, and
    // one at a time those waits stood behind the values of the point before.)
    auto load_ahead = [&]() {
        int e[AHEAD];
#pragma unroll
        for (int p = 0; p < AHEAD; ++p) e[p] = max(cursor - p, 0), written_by[p] = 0;
        if (listed) {
#pragma unroll
            for (int p = 0; p < AHEAD; ++p) written_by[p] = its[e[p]], e[p] = pts[e[p]];
        }
#pragma unroll
        for (int p = 0; p < AHEAD; ++p) {
            at[p] = t_eval[e[p]];
#pragma unroll
            for (int f = 0; f < F; ++f) g_at[p][f] = grad_ys[(long long)e[p] * F + f];
        }
    };
    if (E > 0) {
        load_ahead();
    } else {  // (the end point, written by the batch's last iteration)
        at[0] = te;
#pragma unroll
        for (int f = 0; f < F; ++f) g_at[0][f] = grad_ys[f];
    }

    for (long long i = L - 1; i >= 0; --i) {
        RecordEntry<T, F> before = load_entry<T, F>(w, i > 0 ? i - 1 : 0, g);  // (used by the next pass of this loop)
        const bool end_point = E == 0 && i == L - 1;
        // An iteration that none of the wavefront's samples took part in (all had finished before it) changes nothing for
        // them -- no move, no point written, the step and the history kept -- so its reverse hands every cotangent on as
        // it is.  (Without evaluation points the batch's last iteration is the one whose interpolant gives the result.)
        if (!end_point && !lanes_where(here.running != 0)) {
            if constexpr (SHORT) entry_is_here(before);
            after = here, here = before;
            continue;
        }
        const T t0 = here.t, dt = here.dt, prev = here.prev, pprev = here.pprev;
        const bool move = after.n_accepted > here.n_accepted, running_new = after.running != 0;

        T y[F];
#pragma unroll
        for (int f = 0; f < F; ++f) y[f] = here.y[f];
        typename std::conditional<LATER, FormedLater<T, F>, Formed<T, F>>::type o;
        if constexpr (PAIR) {
            lds_barrier();
            hand.read(o);
#pragma unroll
            for (int f = 0; f < F; ++f) o.k[0][f] = here.k0[f];
        } else {
            form_stages<T, METHOD, Term>(rhs, here, o);
            if constexpr (!LATER) form_errors<T, METHOD, CTRL, Term>(w, here, running_new, o);
        }
        const T(&k)[7][F] = o.k, (&y1)[F] = o.y1;

        // ---- everything after the stages, reversed: the operations of finish_backward_sample, in its order ----
        const T t_new = move ? (t0 + dt) : t0;
        const T lo = tlo - t_new, hi = thi - t_new;
        T g_t, g_dt, g_prev = 0, g_pprev = 0, g_h, g_lo, g_hi, g_k[7][F], g_y[F], g_y1[F];
        {
            using Div = DivSqrtFeatures<T, F>;
            lanes_t bounds_outside;
            if constexpr (LATER) bounds_outside = form_errors<T, METHOD, CTRL, Term>(w, here, running_new, o);
            else bounds_outside = lanes_where(o.bounds_outside);
            const T(&err)[F] = o.err, (&eb)[F] = o.eb, (&per_eb)[F] = o.per_eb, (&q)[F] = o.q, (&x)[F] = o.x;
            const T r = o.r, ratio = o.ratio, F0 = o.F0;
            // Quotients of cotangents: the divisors' ranges are known, the dividends are looked at.  divisors_outside: lanes
            // (of those that take part) whose divisor is outside.
            const T per_ratio = reciprocal_estimate(ratio);
            const lanes_t ratio_outside = lanes_where(!(ratio >= (T)0x1p-20)) | lanes_where(!(ratio <= (T)0x1p+20));
            if (SHORT && !w.plain) bounds_outside = ~(lanes_t)0;

            const T factor = tclamp(F0, cp.fmin, cp.fmax);
            const T raw = dt * factor;
            T dt_next = raw;
            (void)limit_step<T, T>(cp, w.dt_min, w.dt_max, ratio, dt_next);
            const T dtn = running_new ? dt_next : dt;

            // clamp of the step to the time range, and the new time
            const T g_self = (dtn >= lo && dtn <= hi) ? a_dt : (T)0;
            g_lo = (dtn < lo && lo < hi) ? a_dt : (T)0;
            g_hi = (dtn > hi || hi < lo) ? a_dt : (T)0;
            const T g_tnew = a_t - (g_lo + g_hi), g_dt_next = running_new ? g_self : (T)0;
            g_dt = running_new ? (T)0 : g_self;
            g_t = g_tnew;
            if (move) g_dt += g_tnew;

            // controller history and step proposal
            T g_ratio = 0;
            if (CTRL == 1) {
                const bool keep = running_new && move;
                g_ratio = keep ? a_prev : (T)0;
                g_prev = keep ? a_pprev : a_prev;
                g_pprev = keep ? (T)0 : a_pprev;
            }
            if (w.through_control) {
                T g_raw = g_dt_next;
                if (cp.has_dt_min || cp.has_dt_max) {
                    const T mag = abs_(raw);
                    const bool inside = (!cp.has_dt_min || mag >= w.dt_min) && (!cp.has_dt_max || mag <= w.dt_max);
                    g_raw = (inside && raw != (T)0) ? g_dt_next : (T)0;
                }
                g_dt += g_raw * factor;
                const T g_factor = g_raw * dt;
                const T g_F0 = (F0 >= cp.fmin && F0 <= cp.fmax) ? g_factor : (T)0;
                const T g_powers = g_F0 * F0;
                // (times an exponent of 2^-10 to 1/2: dividends a little below the smallest, of divisors between 2^-20 and 2^20)
                const Dividends<T> d(g_powers);
                if (SHORT && !(d.outside() | ratio_outside | bounds_outside)) {
                    g_ratio += quotient_with(g_powers * (T)cp.e1, ratio, per_ratio);
                    if (CTRL == 1) {
                        if (!cp.skip2) g_prev += quotient_plain(g_powers * (T)cp.e2, prev);
                        if (!cp.skip3) g_pprev += quotient_plain(g_powers * (T)cp.e3, pprev);
                    }
                } else {
                    g_ratio += g_powers * (T)cp.e1 / ratio;
                    if (CTRL == 1) {
                        if (!cp.skip2) g_prev += g_powers * (T)cp.e2 / prev;
                        if (!cp.skip3) g_pprev += g_powers * (T)cp.e3 / pprev;
                    }
                }
            }

            // error ratio and error estimate; state update
            const T tiny = (T)1e-38;
            const T g_r = r > tiny ? g_ratio : (r == tiny ? g_ratio / (T)2 : (T)0);
            g_h = 0;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                g_y[f] = move ? (T)0 : a_y[f], g_y1[f] = move ? a_y[f] : (T)0;
#pragma unroll
                for (int s = 0; s < 7; ++s) g_k[s][f] = 0;
                g_k[0][f] = move ? (T)0 : a_k0[f], g_k[6][f] = move ? a_k0[f] : (T)0;
            }
            if (g_r != (T)0 && r > (T)0) {
                T g_q[F], g_err[F], g_m[F];
                lanes_t general = ~(lanes_t)0;
                if constexpr (SHORT) {  // (r is the ratio where it is in range)
                    Dividends<T> d;
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        const T g_x = g_r * x[f], over_r = quotient_with(g_x, r, per_ratio);
                        g_q[f] = Div::fast(over_r);
                        const T g_eb = -g_q[f] * q[f];
                        g_err[f] = quotient_with(g_q[f], eb[f], per_eb[f]);
                        g_m[f] = quotient_with(g_eb, eb[f], per_eb[f]);
                        d.add(g_x), d.add(over_r), d.add(g_q[f]), d.add(g_eb);
                    }
                    general = d.outside() | ((ratio_outside | bounds_outside) & lanes_where(true));
                }
                if (general) {
#pragma unroll
                    for (int f = 0; f < F; ++f) {
                        g_q[f] = g_r * x[f] / r / sf;
                        g_err[f] = g_q[f] / eb[f];
                        g_m[f] = -g_q[f] * q[f] / eb[f];
                    }
                }
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    T bk = 0;
#pragma unroll
                    for (int s = 0; s < 7; ++s) bk = fma_((T)Tab::b_err[s], k[s][f], bk);
                    const T g_e = g_err[f] * sign_(err[f]);
                    T ga, gb;
                    max_backward<T>(abs_(y[f]), abs_(y1[f]), g_m[f] * cp.rtol, ga, gb);
                    g_y[f] += ga * sign_(y[f]);
                    g_y1[f] += gb * sign_(y1[f]);
#pragma unroll
                    for (int s = 0; s < 7; ++s) g_k[s][f] += g_e * (dt * (T)Tab::b_err[s]);
                    g_h += g_e * bk;
                }
            }
        }
        if (w.g_t_start || w.g_t_end) {
            T g_ts_lo, g_te_lo, g_ts_hi, g_te_hi;
            // tlo = minimum(t_start, t_end), thi = maximum(t_start, t_end) (problems.py:58-64)
            max_backward<T>(-ts, -te, g_lo, g_ts_lo, g_te_lo);  // minimum(a, b) = -maximum(-a, -b): same split
            max_backward<T>(ts, te, g_hi, g_ts_hi, g_te_hi);
            if (w.g_t_start) w.g_t_start[g] += g_ts_lo + g_ts_hi;
            if (w.g_t_end) w.g_t_end[g] += g_te_lo + g_te_hi;
        }

        // dense output: the evaluation points this iteration wrote, one by one in their order (see finish_backward_sample)
        T den = (t0 + dt) - t0;
        const bool flat = !(abs_(den) > (T)0);
        if (flat) den = (T)1;
        const T per_den = reciprocal_estimate(den);
        const lanes_t den_outside = SHORT ? lanes_where(!(abs_(den) >= (T)0x1p-20)) | lanes_where(!(abs_(den) <= (T)0x1p+20)) : ~(lanes_t)0;
        T slope[F][4];  // the polynomial's coefficients, lowest power first, differentiated
        auto build_slopes = [&](int first, int last) {
#pragma unroll
            for (int f = first; f < last; ++f) {
                form_slope<T, METHOD, F>(dt, y, y1, k, f, slope[f]);
            }
        };
        auto slopes_of_all = [&] {
            if constexpr (PAIR) hand.read_slopes(slope);
            else build_slopes(0, F);
        };
        auto add_point = [&](const T t, const T(&cotangent)[F], T *g_time) {
            const T from_t0 = t - t0;
            T x = quotient_with(from_t0, den, per_den);
            if (Dividends<T>(from_t0).outside() | (den_outside & lanes_where(true))) x = from_t0 / den;
            T g_x = 0;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const T g0 = cotangent[f];
                if (g0 == (T)0) continue;
                if (!SHORT) build_slopes(f, f + 1);
                const T ks[7] = {k[0][f], k[1][f], k[2][f], k[3][f], k[4][f], k[5][f], k[6][f]};
                g_x += g0 * (slope[f][0] + x * (slope[f][1] + x * (slope[f][2] + x * slope[f][3])));
                const T g1 = g0 * x, g2 = g1 * x, g3 = g2 * x, g4 = g3 * x;
                if (METHOD == 1) {
                    g_y[f] += g0;
                    g_k[0][f] += g1 * dt;
                    g_h += g1 * ks[0];
#pragma unroll
                    for (int s = 0; s < 7; ++s) {
                        const T u = g2 * (T)Tsit5Tab::w[0][s] + g3 * (T)Tsit5Tab::w[1][s] + g4 * (T)Tsit5Tab::w[2][s];
                        g_k[s][f] += u * dt;
                        g_h += u * ks[s];
                    }
                } else {
                    const T g_f0 = (T)-2 * g4 + (T)5 * g3 - (T)4 * g2 + g1, g_f1 = (T)2 * g4 - (T)3 * g3 + g2;
                    const T g_mid = (T)16 * g4 - (T)32 * g3 + (T)16 * g2;
                    g_y[f] += (T)-8 * g4 + (T)18 * g3 - (T)11 * g2 + g0 + g_mid;
                    g_y1[f] += (T)-8 * g4 + (T)14 * g3 - (T)5 * g2;
                    g_k[0][f] += g_f0 * dt;
                    g_k[6][f] += g_f1 * dt;
                    g_h += g_f0 * ks[0] + g_f1 * ks[6];
#pragma unroll
                    for (int s = 0; s < 7; ++s) {
                        g_k[s][f] += g_mid * (dt * (T)Dopri5Tab::w[0][s]);
                        g_h += g_mid * (T)Dopri5Tab::w[0][s] * ks[s];
                    }
                }
            }
            // x = (t - t0) / ((t0 + dt) - t0)
            const T g_xx = g_x * x;
            T g_at = quotient_with(g_x, den, per_den), g_den = quotient_with(g_xx, den, per_den);
            if (Dividends<T>(g_x, g_xx).outside() | (den_outside & lanes_where(true))) g_at = g_x / den, g_den = g_xx / den;
            if (g_time) *g_time += g_at;
            g_t -= g_at;
            if (!flat) g_dt -= g_den;
        };
        lanes_t takes[AHEAD];
        int n = 0;
        if (E > 0) {
            auto wrote = [&](int p, T time, int32_t by) {
                return cursor - p >= lowest && (listed ? by == (int32_t)i : (i == 0 || dir * t0 < dir * time));
            };
#pragma unroll
            for (int p = 0; p < AHEAD; ++p) {
                const bool more = wrote(p, at[p], written_by[p]);
                takes[p] = lanes_where(more), n += more ? 1 : 0;
            }
            if (SHORT && takes[0]) slopes_of_all();
            if (takes[AHEAD - 1]) {  // (some sample's step passed more points than are held)
                for (bool more = n == AHEAD; lanes_where(more);) {
                    const int e = max(cursor - n, 0);
                    more = more && wrote(n, t_eval[listed ? pts[e] : e], listed ? its[e] : 0);
                    n += more ? 1 : 0;
                }
                for (int p = n - 1; lanes_where(p >= AHEAD); --p) {
                    if (p < AHEAD) continue;
                    const int e = listed ? pts[cursor - p] : cursor - p;
                    T cotangent[F];
#pragma unroll
                    for (int f = 0; f < F; ++f) cotangent[f] = grad_ys[(long long)e * F + f];
                    add_point(t_eval[e], cotangent, w.g_t_eval ? w.g_t_eval + g * E + e : nullptr);
                }
            }
        } else {
            takes[0] = lanes_where(end_point);
#pragma unroll
            for (int p = 1; p < AHEAD; ++p) takes[p] = 0;
            if (SHORT && end_point) slopes_of_all();
        }
#pragma unroll
        for (int p = AHEAD - 1; p >= 0; --p) {
            if (!takes[p]) continue;
            if (holds(takes[p])) {
                T *g_time = E > 0 ? w.g_t_eval : w.g_t_end;
                if (g_time) g_time += E == 0 ? g : g * E + (listed ? pts[cursor - p] : cursor - p);
                add_point(at[p], g_at[p], g_time);
            }
        }
        if constexpr (SHORT) entry_is_here(before);  // (eight doubles a row: no registers for it)
        if (E > 0) {
            cursor -= n;
            load_ahead();
        }
        g_dt += g_h;

        // ---- the stages reversed ----
#pragma unroll
        for (int s = 6; s >= 1; --s) {
            T gk[F], gy[F], sums[F], yi[F];
#pragma unroll
            for (int f = 0; f < F; ++f) {
                gk[f] = g_k[s][f], sums[f] = 0;
#pragma unroll
                for (int j = 0; j < s; ++j) sums[f] = fma_((T)Tab::a[s][j], k[j][f], sums[f]);
                yi[f] = PAIR ? fma_(dt, sums[f], y[f]) : o.yi[s][f];
            }
            rhs.vjp(fma_((T)Tab::c[s], dt, t0), yi, gk, gy, gpar);
            T g_step = 0;
#pragma unroll
            for (int f = 0; f < F; ++f) {
                const T g_in = s == 6 ? gy[f] + g_y1[f] : gy[f];
                g_y[f] += g_in;
#pragma unroll
                for (int j = 0; j < s; ++j) g_k[j][f] += (T)Tab::a[s][j] * dt * g_in;
                g_step += g_in * sums[f];
            }
            g_dt += g_step;
        }

        // ---- the cotangents of the state before this iteration are those behind the one before it ----
#pragma unroll
        for (int f = 0; f < F; ++f) a_y[f] = g_y[f], a_k0[f] = g_k[0][f];
        a_t = g_t, a_dt = g_dt, a_prev = g_prev, a_pprev = g_pprev;
        after = here, here = before;
    }
    // (no iteration: nothing flows back through the loop, and the cotangents are still the zeros they started as)
    if (w.through_start)  // (`here` is the record's first entry now: t_start, y0, f(t_start, y0))
        start_backward<T, CTRL, Term>(cp, rhs, w.through_control && !w.dt0_given, ts, te, here.y, here.k0, a_y, a_k0, a_dt, gpar);
    if (w.through_start == 2 && E > 0 && t_eval[0] == ts) {
#pragma unroll
        for (int f = 0; f < F; ++f) a_y[f] += grad_ys[f];
    }
#pragma unroll
    for (int f = 0; f < F; ++f) w.a_y[g * F + f] = a_y[f], w.a_k0[g * F + f] = a_k0[f];
    w.a_t[g] = a_t, w.a_dt[g] = a_dt, w.a_prev[g] = a_prev, w.a_pprev[g] = a_pprev;
#pragma unroll
    for (int j = 0; j < P; ++j) w.g_params[g * P + j] = gpar[j];
}

template <typename T, int METHOD, int CTRL, typename Term>
static int launch_backward(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t stream) {
    const long long B = a.batch;
    WholeBackward<T> w = {};
    w.batch = B, w.E = a.n_eval, w.through_control = adj.through_control;
    w.t_start = (const T *)a.t_start, w.t_end = (const T *)a.t_end, w.t_eval = (const T *)a.t_eval, w.grad_ys = (const T *)adj.grad_ys;
    w.g_t_start = (T *)adj.g_t_start, w.g_t_end = (T *)adj.g_t_end, w.g_t_eval = (T *)adj.g_t_eval;
    w.cp = make_ctrl<T>(c);
    w.dt_min = (T)c.dt_min, w.dt_max = (T)c.dt_max;
    const auto counts = [](double e) { return e >= 0x1p-10 || e <= -0x1p-10; };  // (a cotangent times an exponent)
    w.plain = w.cp.plain && !w.cp.shortcut_exponent() && counts(w.cp.e1) && (w.cp.skip2 || counts(w.cp.e2)) && (w.cp.skip3 || counts(w.cp.e3));
    w.a_y = (T *)adj.a_y, w.a_k0 = (T *)adj.a_k0, w.a_t = (T *)adj.a_t, w.a_dt = (T *)adj.a_dt, w.a_prev = (T *)adj.a_prev, w.a_pprev = (T *)adj.a_pprev;
    const tode_solve_record &r = *a.record;
    w.iterations = adj.iterations;
    w.rec_t = (const T *)r.t, w.rec_dt = (const T *)r.dt, w.rec_y = (const T *)r.y, w.rec_k0 = (const T *)r.k0;
    w.rec_prev = (const T *)r.prev, w.rec_pprev = (const T *)r.pprev, w.rec_running = r.running, w.rec_n_accepted = r.n_accepted;
    w.params = (const T *)a.params;
    for (int i = 0; i < 4; ++i) w.scalars[i] = a.term_scalars[i];
    w.g_params = (T *)adj.g_params;
    w.points_by_iteration = adj.points_by_iteration, w.iterations_sorted = adj.iterations_sorted;
    w.lists = (int32_t *)adj.scratch;
    w.through_start = adj.through_start, w.dt0_given = a.dt0 != nullptr;
    w.ts_stride = a.t_start_stride, w.te_stride = a.t_end_stride;
    // Two wavefronts to a group while a SIMD has no second group to issue for: up to one group per SIMD in float32, half of that in
    // float64, whose hand-over takes twice the LDS (rows of four: 70 KB, two groups to a compute unit).  Kernel in us with Tsit5 and
    // PID, one wavefront and two: Van der Pol float32, 5 groups 390 and 322, 256 375 and 311, 512 388 and 314, 1024 455 and 356,
    // beyond the line 1280 450 and 417, 2048 544 and 720; Lorenz float32, 938 206 and 158, beyond it 1563 227 and 298; decay, rows of
    // four, 938 170 and 147, beyond it 1563 320 and 278.  float64: Van der Pol 256 531 and 391, 511 552 and 418, beyond it 1024 535 and 500;
    // Lorenz 511 288 and 195, 1024 297 and 363; decay, rows of four, 511 253 and 197, 1024 265 and 380.
    const long long groups = (B + 63) / 64;
    constexpr bool paired = Term::F <= 4;
    if (paired && groups <= TODE_PAIRED_SWEEP_GROUPS * 4 / (long long)sizeof(T))
        hipLaunchKernelGGL((whole_backward_kernel<T, METHOD, CTRL, Term, paired>), dim3((unsigned)groups), dim3(128), (HandOver<T, Term::F>::bytes()), stream, w);
    else
        hipLaunchKernelGGL((whole_backward_kernel<T, METHOD, CTRL, Term, false>), dim3((unsigned)groups), dim3(64), 0, stream, w);
    return check_hip(hipGetLastError(), "tode_solve_builtin_backward launch");
}

template <typename T, typename Term> static int backward_mc(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s) {
    if (a.method == TODE_DOPRI5 && c.kind == TODE_CTRL_INTEGRAL) return launch_backward<T, 0, 0, Term>(a, c, adj, s);
    if (a.method == TODE_DOPRI5 && c.kind == TODE_CTRL_PID) return launch_backward<T, 0, 1, Term>(a, c, adj, s);
    if (a.method == TODE_TSIT5 && c.kind == TODE_CTRL_INTEGRAL) return launch_backward<T, 1, 0, Term>(a, c, adj, s);
    if (a.method == TODE_TSIT5 && c.kind == TODE_CTRL_PID) return launch_backward<T, 1, 1, Term>(a, c, adj, s);
    return fail(TODE_E_INVALID, "unknown method %d or controller kind %d", a.method, c.kind);
}

template <typename T> static int backward_term(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s) {
    switch (a.term) {
    case TODE_TERM_VAN_DER_POL:
        if (a.n_features != 2 || a.n_params != 1) return fail(TODE_E_INVALID, "Van der Pol needs F=2, P=1");
        return backward_mc<T, VanDerPolTerm<T>>(a, c, adj, s);
    case TODE_TERM_LORENZ63:
        if (a.n_features != 3 || a.n_params != 1) return fail(TODE_E_INVALID, "Lorenz-63 needs F=3, P=1");
        return backward_mc<T, Lorenz63Term<T>>(a, c, adj, s);
    case TODE_TERM_LINEAR_DECAY:
        if (a.n_params != a.n_features) return fail(TODE_E_INVALID, "linear decay needs P == F");
        switch (a.n_features) {
        case 1: return backward_mc<T, LinearDecayTerm<T, 1>>(a, c, adj, s);
        case 2: return backward_mc<T, LinearDecayTerm<T, 2>>(a, c, adj, s);
        case 3: return backward_mc<T, LinearDecayTerm<T, 3>>(a, c, adj, s);
        case 4: return backward_mc<T, LinearDecayTerm<T, 4>>(a, c, adj, s);
        case 8: return backward_mc<T, LinearDecayTerm<T, 8>>(a, c, adj, s);
        default: return fail(TODE_E_UNSUPPORTED, "linear decay is built for F in {1,2,3,4,8}, got %d", a.n_features);
        }
    default:
        return fail(TODE_E_UNSUPPORTED, "the whole reverse sweep is built for the three small systems (term %d)", a.term);
    }
}

int solve_backward_f32(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s);
int solve_backward_f64(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s);
#if TODE_INSTANTIATE_F32
int solve_backward_f32(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s) { return backward_term<float>(a, c, adj, s); }
#endif
#if TODE_INSTANTIATE_F64
int solve_backward_f64(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s) { return backward_term<double>(a, c, adj, s); }
#endif

}  // namespace tode

#if TODE_INSTANTIATE_F32
extern "C" {

int64_t tode_solve_backward_scratch_bytes(const tode_solve_args *a) {
    if (!a || a->n_features <= 0 || a->batch < 0 || a->n_eval < 0) return -1;
    return 2 * a->batch * a->n_eval * (int64_t)sizeof(int32_t);  // (the two lists of evaluation points, where the caller does not hand them in)
}

int tode_solve_builtin_backward(const tode_solve_args *a, const tode_controller *c, const tode_solve_adjoint *adj, void *stream) {
    using namespace tode;
    if (!a || !c || !adj) return fail(TODE_E_INVALID, "null argument struct");
    if (a->batch < 0 || a->n_features <= 0 || a->n_eval < 0 || a->n_params < 0) return fail(TODE_E_INVALID, "bad sizes");
    if (!known_dtype(a->dtype)) return fail(TODE_E_INVALID, "unknown dtype %d", a->dtype);
    if (a->dtype & TODE_DTYPE_PAIR) return fail(TODE_E_UNSUPPORTED, "the whole reverse sweep is built for time and data in one dtype");
    if (c->kind != TODE_CTRL_INTEGRAL && c->kind != TODE_CTRL_PID) return fail(TODE_E_INVALID, "unknown controller kind %d", c->kind);
    if (!a->record) return fail(TODE_E_INVALID, "args->record is null: the sweep starts from the record of the forward pass");
    if (adj->iterations < 0 || a->record->capacity < adj->iterations + 1)
        return fail(TODE_E_INVALID, "the record holds %lld entries, %lld iterations need %lld", (long long)a->record->capacity, (long long)adj->iterations, (long long)adj->iterations + 1);
    if (a->t_start_stride < 1 || a->t_end_stride < 1) return fail(TODE_E_INVALID, "t_start_stride / t_end_stride must be >= 1");
    if ((a->t_start_stride != 1 && adj->g_t_start) || (a->t_end_stride != 1 && adj->g_t_end)) return fail(TODE_E_INVALID, "g_t_start / g_t_end are dense arrays: ask for them with dense t_start / t_end");
    if (a->batch == 0) return TODE_OK;
    const tode_solve_record &r = *a->record;
    if (!r.t || !r.dt || !r.y || !r.k0 || !r.prev || !r.pprev || !r.running || !r.n_accepted) return fail(TODE_E_INVALID, "a null array in the record");
    if (!a->t_start || !a->t_end || (a->n_eval > 0 && (!a->t_eval || !adj->points_by_iteration != !adj->iterations_sorted)) || (a->n_params > 0 && !a->params) || !adj->grad_ys || !adj->a_y ||
        !adj->a_k0 || !adj->a_t || !adj->a_dt || !adj->a_prev || !adj->a_pprev || !adj->g_params)
        return fail(TODE_E_INVALID, "null pointer");
    const bool own_lists = a->n_eval > 0 && !adj->points_by_iteration;
    if (own_lists && (!adj->scratch || adj->scratch_bytes < tode_solve_backward_scratch_bytes(a)))
        return fail(TODE_E_INVALID, "the scratch buffer holds %lld bytes, this sweep needs %lld (tode_solve_backward_scratch_bytes)", (long long)(adj->scratch ? adj->scratch_bytes : 0),
                    (long long)tode_solve_backward_scratch_bytes(a));
    hipStream_t s = (hipStream_t)stream;
    return a->dtype == TODE_F32 ? solve_backward_f32(*a, *c, *adj, s) : solve_backward_f64(*a, *c, *adj, s);
}

}  // extern "C"
#endif
