// Two-wavefront variant of the fast whole-solve kernel, for batches that would
// otherwise leave the SIMDs with a single wavefront each (B <= 2 * 65536 on an
// MI355X: 256 CUs x 4 SIMDs x 64 lanes).
//
// A single in-order wavefront cannot keep a SIMD busy: every instruction costs an
// issue slot and every dependent result is waited for (measured: one dependent fp32
// FMA every 7.7 cycles with one wave per SIMD, one every 5.3 per SIMD with two).  The solve
// loop has exactly one piece of work that the next step does not depend on -- the
// dense output -- so each group of 64 samples gets two wavefronts:
//   * the STEPPER runs the adaptive loop (stages, error ratio, step size control,
//     state update) and, after every attempted step, leaves the step's
//     (t0, dt, y0, y1, k_0..k_6, new time) in LDS;
//   * the EVALUATOR picks that record up one barrier later, builds the quartic
//     interpolant and writes the evaluation points the step passed, while the
//     stepper is already computing the next step.
// Records are double-buffered; one s_barrier per loop iteration orders the
// hand-over.  Stepper and evaluator roles alternate between neighbouring pairs of
// workgroups, meant to give every SIMD one of each.
//
// In the smallest batches a sample's features get a lane each (the ...Lanes systems of tode_solve.h), 64 / L samples per
// wavefront: the same kernel with one feature per lane.
//
// Same arithmetic, bit for bit, and same contract as tode_fast.hip
// (TODE_FLAG_NEEDS_GENERAL when the batch leaves the common case).
//
// RECORD: the stepper also writes the loop state before every iteration to p.rec_* (tode_solve_record), as
// tode_fast.hip's recording variant does, for the reverse sweep of a differentiable solve.
#include "tode_solve.h"

#if TODE_INSTANTIATE_LANES
#define TODE_PAIR_TERM(name) name##Lanes
#else
#define TODE_PAIR_TERM(name) name##Term
#endif

namespace tode {

template <typename T> struct PairOut {
    int64_t *n_steps, *n_accepted, *n_initialized, *status;
};

template <typename T, int METHOD, int CTRL, int NHIST, typename Term, bool STAGE_TE, bool RECORD = false>
__global__ void __launch_bounds__(128) solve_pair_kernel(const SolveParams<T> p, const PairOut<T> o) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    // F features per sample, K of them per lane, L lanes per sample, S samples per wavefront
    constexpr int F = Term::F, K = Term::K, L = Term::L, S = 64 / L;
    constexpr int P = Term::P;
    constexpr int NF = 3 + 9 * K;  // record: t0, dt, dir*t_new (-inf once the sample has finished), y[K], y1[K], k[7][K]
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const bool stepper = ((wave + (blockIdx.x >> 1)) & 1) == 0;
    const long long b0 = (long long)blockIdx.x * S;
    const int group = lane / L;  // the lane's sample among the wavefront's
    const long long b = b0 + group;
    const int rows = (int)min((long long)S, p.batch - b0);
    const bool live = group < rows;
    // the features of the lane (a lane beyond the last feature repeats it and stores nothing), and the lane that stores what
    // the sample has one of
    auto feature = [&](int i) { return L == 1 ? i : min(lane_feature<L>(), F - 1); };
    const bool owns = L == 1 || lane_feature<L>() < F;
    const bool first_lane = L == 1 || lane_feature<L>() == 0;
    const long long bs = live ? b : b0;
    const CtrlParams<T> &cp = p.cp;
    // Without evaluation points the reference reports the end point alone (adjoints.py:296-311): the
    // interpolant of the batch's last iteration at t_end.  Here: t_end as the one evaluation point of
    // every sample, and the final state next to it in y_idle; which of the two a sample gets depends on
    // whether its last step was the batch's last iteration, known only when all samples are done
    // (tode_select_end_point).
    const bool end_only = p.n_eval == 0;
    const int E = end_only ? 1 : p.n_eval;

    T *rec = reinterpret_cast<T *>(smem_raw);                // [2][NF][64]
    int *ctl = reinterpret_cast<int *>(rec + 2 * NF * 64);   // [2] "stepper is done", by phase
    T *te_s = reinterpret_cast<T *>(ctl + 4);                // [E + 1][S] when STAGE_TE

    const T ts = p.t_start[bs * p.ts_stride], te = p.t_end[bs * p.te_stride];
    const bool fwd = te > ts;
    const T dir = fwd ? (T)1 : (T)-1;

    if (stepper) {
        // =============================== stepper ===============================
        Term rhs;
        rhs.load(p.params + bs * P, p.scalars);
        T y[K], k[7][K];
#pragma unroll
        for (int f = 0; f < K; ++f) y[f] = p.y0[bs * F + feature(f)];
        const T tlo = tmin(ts, te), thi = tmax(te, ts);
        T t = ts, dt;
        if (p.dt0) {
            dt = p.dt0[bs];
            rhs(ts, y, k[0]);
        } else {
            dt = initial_step<T, CTRL, Term>(cp, rhs, ts, y, dir, abs_(te - ts), k[0]);
        }
        dt = tclamp(dt, tlo - t, thi - t);
        StepFactor<T, NHIST, L> step_factor;  // with the logarithms of the previous two accepted error ratios (both start at 1)
        const T dte_end = dir * te;
        int n_steps = 0, n_acc = 0;
        // The loop below uses the hardware's minimum and maximum, which is the reference's arithmetic as long as no
        // operand is NaN: a sample that starts with a NaN or infinite time, step or state goes to the general kernel,
        // and so does one that produces a non-finite error ratio, step factor or step later.
        bool odd_start = !finite_(dt) || !finite_(ts) || !finite_(te);
#pragma unroll
        for (int f = 0; f < K; ++f) odd_start = odd_start || !finite_(y[f]) || !finite_(k[0][f]);
        // lanes whose sample is still stepping, and lanes whose sample needs the general kernel
        lanes_t active = lanes_where(live && !odd_start), bail_lanes = lanes_where(live && odd_start);
        const int step_limit = p.max_steps < TODE_HARD_STEP_LIMIT ? p.max_steps : TODE_HARD_STEP_LIMIT;
        const T e1 = (T)cp.e1, e2 = (T)cp.e2, e3 = (T)cp.e3;

        // (RECORD) the last two accepted error ratios as values (the step factor keeps their logarithms)
        T ratio_prev = 1, ratio_prev_prev = 1;
        bool record_full = false;
        auto keep = [&](long long at, bool running) {
            if (at >= p.rec_capacity) {
                record_full = true;
                return;
            }
            if (!live) return;
            if constexpr (L == 1) {
                record_entry<T, T, F>(p, at, b, t, dt, y, k[0], ratio_prev, ratio_prev_prev, running, n_acc);
            } else {
                const long long i = at * p.batch + b;
                if (owns) p.rec_y[i * F + feature(0)] = y[0], p.rec_k0[i * F + feature(0)] = k[0][0];
                if (first_lane) {
                    p.rec_t[i] = t, p.rec_dt[i] = dt;
                    p.rec_prev[i] = ratio_prev, p.rec_pprev[i] = ratio_prev_prev;
                    p.rec_running[i] = running ? 1 : 0, p.rec_n_accepted[i] = n_acc;
                }
            }
        };

        // A sample that has landed past t_end (t + (t_end - t) rounded upwards) keeps stepping in the reference's
        // later iterations with the clamped step t_end - t: with evaluation points that is seen only in the status of
        // that step, a success unless its error ratio is not finite.  The sample sits through one more iteration here,
        // as an inactive lane whose error ratio is looked at.
        lanes_t idle = 0;
        int phase = 0;
        if (lane == 0) ctl[0] = ctl[1] = 0;
        for (;; ++phase) {
            const lanes_t counted = active | idle;
            if (counted) {
                if (RECORD) keep(phase, holds(active));
                // ---- stages (runge_kutta.py:255-263) ----
                const T t0 = t;
                T y1[K];
#pragma unroll
                for (int i = 1; i < 7; ++i) {
                    T tn = fma_((T)Tab::c[i], dt, t0);
                    T yi[K];
#pragma unroll
                    for (int f = 0; f < K; ++f) {
                        T s = 0;
#pragma unroll
                        for (int j = 0; j < i; ++j)
                            if (Tab::a[i][j] != 0.0) s = fma_((T)Tab::a[i][j], k[j][f], s);  // (a zero weight: weighted_k's FINITE)
                        yi[f] = fma_(dt, s, y[f]);
                    }
                    rhs(tn, yi, k[i]);
                    if (i == 6) {
#pragma unroll
                        for (int f = 0; f < K; ++f) y1[f] = yi[f];
                    }
                }
                // hand the attempted step to the evaluator (everything it needs is known now)
                T *r = rec + (phase & 1) * NF * 64 + lane;
                r[0 * 64] = t0;
                r[1 * 64] = dt;
#pragma unroll
                for (int f = 0; f < K; ++f) {
                    r[(3 + f) * 64] = y[f];
                    if (METHOD != 1) r[(3 + K + f) * 64] = y1[f];  // (Tsit5's interpolant does not look at the step's result)
                }
#pragma unroll
                for (int s = 0; s < 7; ++s)
#pragma unroll
                    for (int f = 0; f < K; ++f) r[(3 + 2 * K + s * K + f) * 64] = k[s][f];

                // ---- error estimate and step size control (step_size_controllers.py:370-429, 715-774) ----
                lanes_t insane;  // (a NaN or infinite ratio is a non-success status: left to the general kernel)
                T factor;
                const T ratio = control_common<T, F, K, L, NHIST, Tab>(cp, dt, k, y, y1, counted, step_factor, e1, e2, e3, factor, insane);
                const lanes_t accept = lanes_where(ratio < (T)1), move = accept & active;
                bail_lanes |= idle & insane;
                idle = 0;
                factor = clamp_ordered(factor, cp.fmin, cp.fmax);
                const T dt_next = dt * factor;

                t = holds(move) ? (t0 + dt) : t0;
                const T dt_new = dir * t;
                const lanes_t running = lanes_where(dt_new < dte_end);
                n_acc += holds(move) ? 1 : 0;
                r[2 * 64] = holds(active) ? dt_new : (T)-__builtin_huge_val();  // (a finished sample passes no point)

                // ---- state update (adjoints.py:150-155, 247-255) ----
#pragma unroll
                for (int f = 0; f < K; ++f) {
                    y[f] = holds(move) ? y1[f] : y[f];
                    k[0][f] = holds(move) ? k[6][f] : k[0][f];
                }
                // (a finished sample no longer runs: its step stays what this clamp made it)
                dt = clamp_ordered(holds(running) ? dt_next : dt, tlo - t, thi - t);
                if (NHIST >= 1) step_factor.shift(holds(running & accept));
                if (RECORD && CTRL == 1) {
                    const bool shift = holds(running & accept);
                    ratio_prev_prev = shift ? ratio_prev : ratio_prev_prev;
                    ratio_prev = shift ? ratio : ratio_prev;
                }
                const lanes_t failed = active & (phase + 1 >= step_limit ? ~(lanes_t)0 : insane);
                const lanes_t ended = active & (failed | ~running);
                if (ended) {
                    n_steps = holds(ended) ? phase + 1 : n_steps;
                    // a sample whose state or derivative at the end is not finite shows up in later iterations of
                    // the reference loop with another status, and so does, without evaluation points, one that
                    // landed past t_end (in the interpolant of the batch's last step); with evaluation points
                    // such a sample is looked at in the next iteration
                    bool odd = end_only && !(t == te);
#pragma unroll
                    for (int f = 0; f < K; ++f) odd = odd || !settles_(y[f], k[0][f]);
                    const lanes_t finished = ended & ~failed, odd_lanes = lanes_where(odd);
                    bail_lanes |= failed | (finished & odd_lanes);
                    idle = finished & ~odd_lanes & ~lanes_where(t == te);
                    active &= ~ended;
                }
            }
            if (!counted && lane == 0) ctl[phase & 1] = 1;  // (the evaluator may still be about to look at the other word)
            __syncthreads();
            if (!counted) break;
        }
        bool bail = holds(bail_lanes);

        if (RECORD) {  // the state every sample is left in, for every later iteration of the batch
            for (long long at = phase; at < p.rec_capacity; ++at) keep(at, false);
            if (phase >= p.rec_capacity) record_full = true;
            bail = bail || record_full;
        }
        if (live && first_lane) {
            o.n_steps[b] = n_steps;
            o.n_accepted[b] = n_acc;
            o.status[b] = 0;
        }
        if (live && owns && end_only) {
#pragma unroll
            for (int f = 0; f < K; ++f) p.y_idle[b * F + feature(f)] = y[f];
        }
        int my_steps = live ? n_steps : 0, my_bail = (live && bail) ? 1 : 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            my_steps = max(my_steps, __shfl_xor(my_steps, off));
            my_bail = max(my_bail, __shfl_xor(my_bail, off));
        }
        if (lane == 0) {
            if (my_steps > 0) atomicMax(&p.flags[TODE_FLAG_MAX_ITERATIONS], my_steps);
            if (my_bail) atomicMax(&p.flags[TODE_FLAG_NEEDS_GENERAL], 1);
        }
    } else {
        // ============================== evaluator ==============================
        const T *tev_g = p.t_eval + bs * (long long)E;
        if (STAGE_TE && !end_only) {
            // this group's block of t_eval (rows * E contiguous values), transposed into LDS
            const T *src = p.t_eval + b0 * E;
            const int n = rows * E;
            int row = lane / E, e = lane - row * E;
            const int drow = 64 / E, de = 64 - drow * E;
            for (int g = lane; g < n; g += 64) {
                te_s[e * S + row] = src[g];
                e += de;
                row += drow;
                if (e >= E) {
                    e -= E;
                    row += 1;
                }
            }
        }
        // (LDS accesses of one wavefront complete in order; te_s is private to this wave)
        // From here on times are multiplied by the sample's direction (exact), and behind the last point lies one that no
        // time reaches, not even the infinite one that a step without a finite result may lead to: not a number.  Whether a
        // step has passed the next point is one comparison.
        const T never = nan_<T>();
        bool bail = false;
        const T te_first = end_only ? te : (STAGE_TE ? te_s[group] : tev_g[0]);
        if (!end_only) {
            T prev_te = dir * te_first;
            if (STAGE_TE) te_s[group] = prev_te;
            for (int e = 1; e < E; ++e) {
                const T cur = dir * (STAGE_TE ? te_s[e * S + group] : tev_g[e]);
                if (STAGE_TE) te_s[e * S + group] = cur;
                if (!(cur >= prev_te)) bail = true;
                prev_te = cur;
            }
            if (STAGE_TE) te_s[E * S + group] = never;
        }
        auto point = [&](int e) -> T {
            if (end_only) return e == 0 ? dir * te : never;
            if (STAGE_TE) return te_s[e * S + group];
            return e < E ? dir * tev_g[e] : never;
        };
        // (a workgroup's block of ys holds fewer than 2^32 values: launch_pair)
        T *ys_block = p.ys + b0 * (long long)E * F;
        const unsigned ys_row = (unsigned)(live ? group : 0) * (unsigned)E;
        int cursor = 0;
        if (te_first == ts) {
            if (live && owns) {
#pragma unroll
                for (int f = 0; f < K; ++f) ys_block[ys_row * F + feature(f)] = p.y0[bs * F + feature(f)];
            }
            cursor = 1;
        }
        T dte_next = live ? point(cursor) : never;

        for (int phase = 0;; ++phase) {
            __syncthreads();
            const T *r = rec + (phase & 1) * NF * 64 + lane;
            const int done = ctl[phase & 1];
            const T dt_new = r[2 * 64];
            if (done) break;
            if (dt_new >= dte_next) {
                const T t0 = r[0 * 64], dt = r[1 * 64];
                T y[K], y1[K], k[7][K], q[5][K];
#pragma unroll
                for (int f = 0; f < K; ++f) {
                    y[f] = r[(3 + f) * 64];
                    y1[f] = METHOD != 1 ? r[(3 + K + f) * 64] : (T)0;
                }
#pragma unroll
                for (int s = 0; s < 7; ++s)
#pragma unroll
                    for (int f = 0; f < K; ++f) k[s][f] = r[(3 + 2 * K + s * K + f) * 64];
                quartic<T, K, METHOD, true>(dt, y, y1, k, q);
                const StepPosition<T> position(t0, dt, dir, dte_next);
                auto write_points = [&](auto plain) {
                    do {
                        T out[K];
                        quartic_at_unit<T, K>(q, position.template at<decltype(plain)::value>(dir, dte_next), out);
                        T *row = ys_block + (ys_row + (unsigned)cursor) * F;
#pragma unroll
                        for (int f = 0; f < K; ++f)
                            if (owns) row[feature(f)] = out[f];
                        ++cursor;
                        dte_next = point(cursor);
                    } while (dt_new >= dte_next);
                };
                if (position.plain == lanes_where(true))
                    write_points(std::true_type());
                else
                    write_points(std::false_type());
            }
        }

        if (live && first_lane) o.n_initialized[b] = cursor;
        int my_bail = (live && bail) ? 1 : 0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) my_bail = max(my_bail, __shfl_xor(my_bail, off));
        if (lane == 0 && my_bail) atomicMax(&p.flags[TODE_FLAG_NEEDS_GENERAL], 1);
    }
    publish_flags(p);
}

// The largest batch that takes this form.  One sample per lane: up to 2048 groups of 64 samples, above which the
// single-wavefront kernel has three wavefronts per SIMD by itself.
template <typename Term> constexpr long long pair_batch_limit() {
    if constexpr (Term::L == 1)
        return 2048 * 64;
    else
        return Term::most_samples;
}

template <typename T, int METHOD, int CTRL, typename Term>
static int launch_pair(const tode_solve_args &a, const tode_controller &c, const PairOut<T> &o, hipStream_t stream, bool *used) {
    *used = false;
    constexpr int L = Term::L, S = 64 / L, NF = 3 + 9 * Term::K;
    const long long blocks = (a.batch + S - 1) / S;
    if (blocks == 0 || a.batch > pair_batch_limit<Term>()) return TODE_OK;
    const size_t rec_bytes = (size_t)2 * NF * 64 * sizeof(T) + 16;
    const size_t te_bytes = a.n_eval > 0 ? ((size_t)a.n_eval + 1) * S * sizeof(T) : 0;
    if ((size_t)a.n_eval * Term::F * S > 0xffffffffu) return TODE_OK;  // (32-bit offsets into a workgroup's block of ys)
    // LDS: up to four workgroups per compute unit for every 64 samples of theirs, fewer in a batch that does not have them
    const long long per_cu = (blocks + 255) / 256;
    const size_t budget = (size_t)(160 * 1024) / (size_t)(per_cu < 4 * L ? per_cu : 4 * L) - 512;
    if (rec_bytes > 36 * 1024) return TODE_OK;  // (four features in float64, one sample per lane: the records alone would fill a quarter of it)
    // (the same problem without evaluation points stays with the general kernel)
    if (L > 1 && a.n_eval == 0 && Term::F * sizeof(T) > 24) return TODE_OK;
    const bool stage_te = rec_bytes + te_bytes <= budget;
    const size_t lds = rec_bytes + (stage_te ? te_bytes : 0);
    constexpr bool RECORD = TODE_INSTANTIATE_RECORD != 0;
    if (RECORD != (a.record != nullptr)) return fail(TODE_E_INVALID, "internal: record variant mismatch");
    SolveParams<T> p = make_params<T>(a, c);
    if (p.cp.shortcut_exponent()) return TODE_OK;  // left to the caller's other kernels
    const int nhist = CTRL == 0 ? 0 : (p.cp.skip3 ? 1 : 2);
    const dim3 grid((unsigned)blocks), block(128);
    reset_flags(a.flags, stream);
    timing_before(stream, "tode::solve_pair_kernel");
#define TODE_PAIR_LAUNCH(NH, ST) hipLaunchKernelGGL((solve_pair_kernel<T, METHOD, CTRL, NH, Term, ST, RECORD>), grid, block, lds, stream, p, o)
    if (nhist == 0) {
        if (stage_te) TODE_PAIR_LAUNCH(0, true); else TODE_PAIR_LAUNCH(0, false);
    } else if (nhist == 1) {
        if (stage_te) TODE_PAIR_LAUNCH(CTRL == 0 ? 0 : 1, true); else TODE_PAIR_LAUNCH(CTRL == 0 ? 0 : 1, false);
    } else {
        if (stage_te) TODE_PAIR_LAUNCH(CTRL == 0 ? 0 : 2, true); else TODE_PAIR_LAUNCH(CTRL == 0 ? 0 : 2, false);
    }
#undef TODE_PAIR_LAUNCH
    timing_after(stream);
    *used = true;
    return check_hip(hipGetLastError(), "tode_solve_builtin_fast (pair kernel) launch");
}

template <typename T, typename Term>
static int pair_mc(const tode_solve_args &a, const tode_controller &c, const PairOut<T> &o, hipStream_t s, bool *used) {
    if (a.method == TODE_DOPRI5 && c.kind == TODE_CTRL_INTEGRAL) return launch_pair<T, 0, 0, Term>(a, c, o, s, used);
    if (a.method == TODE_DOPRI5 && c.kind == TODE_CTRL_PID) return launch_pair<T, 0, 1, Term>(a, c, o, s, used);
    if (a.method == TODE_TSIT5 && c.kind == TODE_CTRL_INTEGRAL) return launch_pair<T, 1, 0, Term>(a, c, o, s, used);
    if (a.method == TODE_TSIT5 && c.kind == TODE_CTRL_PID) return launch_pair<T, 1, 1, Term>(a, c, o, s, used);
    *used = false;
    return TODE_OK;
}

// Tries the two-wavefront kernel; *used tells whether it was launched (otherwise the caller
// falls through to the single-wavefront kernel).
template <typename T>
static int pair_term(const tode_solve_args &a, const tode_controller &c, int64_t *ns, int64_t *na, int64_t *ni, int64_t *st, hipStream_t s,
                     bool *used) {
    PairOut<T> o{ns, na, ni, st};
    *used = false;
    switch (a.term) {
    case TODE_TERM_VAN_DER_POL:
        if (a.n_features != 2 || a.n_params != 1) return TODE_OK;
        return pair_mc<T, TODE_PAIR_TERM(VanDerPol)<T>>(a, c, o, s, used);
    case TODE_TERM_LORENZ63:
        if (a.n_features != 3 || a.n_params != 1) return TODE_OK;
        return pair_mc<T, TODE_PAIR_TERM(Lorenz63)<T>>(a, c, o, s, used);
    case TODE_TERM_LINEAR_DECAY:
        if (a.n_params != a.n_features) return TODE_OK;
        switch (a.n_features) {
#if !TODE_INSTANTIATE_LANES
        case 1: return pair_mc<T, TODE_PAIR_TERM(LinearDecay)<T, 1>>(a, c, o, s, used);
#endif
        case 2: return pair_mc<T, TODE_PAIR_TERM(LinearDecay)<T, 2>>(a, c, o, s, used);
        case 3: return pair_mc<T, TODE_PAIR_TERM(LinearDecay)<T, 3>>(a, c, o, s, used);
        case 4:
            // (with the record, four float64 features stay with the single-wavefront kernel in either form)
            if (TODE_INSTANTIATE_LANES && TODE_INSTANTIATE_RECORD && sizeof(T) == 8) return TODE_OK;
            return pair_mc<T, TODE_PAIR_TERM(LinearDecay)<T, 4>>(a, c, o, s, used);
        default: return TODE_OK;
        }
    default:
        return TODE_OK;
    }
}

// (each translation unit instantiates one type and form, with or without the record: TODE_INSTANTIATE_LANES, ..._RECORD)
#if TODE_INSTANTIATE_RECORD
#define TODE_PAIR_ENTRY(name) TODE_PAIR_FORM(name, _record)
#else
#define TODE_PAIR_ENTRY(name) TODE_PAIR_FORM(name, )
#endif
#if TODE_INSTANTIATE_LANES
#define TODE_PAIR_FORM(name, suffix) name##_lanes##suffix
#else
#define TODE_PAIR_FORM(name, suffix) name##suffix
#endif
#if TODE_INSTANTIATE_F32
int TODE_PAIR_ENTRY(solve_pair_f32)(const tode_solve_args &a, const tode_controller &c, int64_t *ns, int64_t *na, int64_t *ni, int64_t *st, hipStream_t s, bool *used) {
    return pair_term<float>(a, c, ns, na, ni, st, s, used);
}
#endif
#if TODE_INSTANTIATE_F64
int TODE_PAIR_ENTRY(solve_pair_f64)(const tode_solve_args &a, const tode_controller &c, int64_t *ns, int64_t *na, int64_t *ni, int64_t *st, hipStream_t s, bool *used) {
    return pair_term<double>(a, c, ns, na, ni, st, s, used);
}
#endif

}  // namespace tode
