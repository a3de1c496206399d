// The one-kernel reverse sweep of the small systems on the host (hip/hip_runtime.h here), against its own operations in their general
// forms: the reverse of an iteration and of a stage that the per-iteration kernels run, iteration by iteration, with the
// points found by looking at every recorded time.  Records and points are drawn at random, ordinary ones and such as leave the ranges
// of the short forms: tiny and zero cotangents, errors and states, states that are not finite, times in no order, repeated
// or beyond the end.
//     sweep first last
// prints the number of runs and of runs with a value that differs.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>

#include <algorithm>
#include <random>

#define TODE_INSTANTIATE_F32 1
#include "tode_backward.hip"

namespace host {
thread_local dim3 thread_idx, block_idx, grid_dim;
unsigned char *lds;
Barrier barrier;
}  // namespace host

namespace tode {
int fail(int code, const char *, ...) { return code; }
int check_hip(hipError_t, const char *) { return TODE_OK; }
const FlagTarget *flag_target() { return nullptr; }
int solve_backward_f64(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, hipStream_t s) { return backward_term<double>(a, c, adj, s); }

// one sample's sweep, in the order of whole_backward_kernel
template <typename T, int METHOD, int CTRL, typename Term>
static void reference(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, std::vector<T> &result) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    constexpr int F = Term::F, P = Term::P;
    const tode_solve_record &rec = *a.record;
    const T ts = *(const T *)a.t_start, te = *(const T *)a.t_end, dir = te > ts ? (T)1 : (T)-1;
    const int E = a.n_eval, L = (int)adj.iterations;
    const T *rt = (const T *)rec.t;
    Term rhs;
    rhs.load((const T *)a.params, a.term_scalars);
    std::vector<int32_t> hit(E);
    for (int e = 0; e < E; ++e) {
        const T at = ((const T *)a.t_eval)[e], v = dir * at;
        int i = 0;
        while (i < L && dir * rt[i + 1] < v) ++i;
        hit[e] = i < L && !(e == 0 && at == ts) ? i : -1;
    }
    T k[7][F], g_k[7][F], y1[F], g_ystage[F], g_y[F], g_y1[F], a_y[F] = {}, a_k0[F] = {}, g_t, g_dt, g_prev, g_pprev;
    T a_t = 0, a_dt = 0, a_prev = 0, a_pprev = 0, gpar[P] = {};
    AdjointParams<T, T> q = {};
    q.batch = 1, q.F = F, q.E = E, q.through_control = adj.through_control, q.t_start = &ts, q.t_end = &te, q.t_eval = (const T *)a.t_eval;
    q.grad_ys = (const T *)adj.grad_ys, q.hit_iteration = hit.data();
    q.g_t_start = (T *)adj.g_t_start, q.g_t_end = (T *)adj.g_t_end, q.g_t_eval = (T *)adj.g_t_eval;
    q.cp = make_ctrl<T>(c), q.dt_min = (T)c.dt_min, q.dt_max = (T)c.dt_max;
    for (int s = 0; s < 7; ++s) q.k[s] = k[s], q.g_k[s] = g_k[s];
    q.y1 = y1, q.g_y = g_y, q.g_y1 = g_y1, q.g_t = &g_t, q.g_dt = &g_dt, q.g_prev = &g_prev, q.g_pprev = &g_pprev;
    q.a_y = a_y, q.a_k0 = a_k0, q.a_t = &a_t, q.a_dt = &a_dt, q.a_prev = &a_prev, q.a_pprev = &a_pprev;
    for (int i = L - 1; i >= 0; --i) {
        q.iteration = i, q.end_point = E == 0 && i == L - 1;
        if (!q.end_point && !rec.running[i]) continue;
        const int32_t moved = rec.n_accepted[i + 1] > rec.n_accepted[i], running_next = rec.running[i + 1] != 0;
        const T *y = (const T *)rec.y + i * F, t0 = rt[i], dt = ((const T *)rec.dt)[i];
        q.t = rt + i, q.dt = (const T *)rec.dt + i, q.y = y, q.prev = (const T *)rec.prev + i, q.pprev = (const T *)rec.pprev + i;
        q.moved = &moved, q.running_next = &running_next;
        T yi[7][F];
        for (int f = 0; f < F; ++f) k[0][f] = ((const T *)rec.k0)[i * F + f];
        for (int s = 1; s < 7; ++s) {
            for (int f = 0; f < F; ++f) {
                T sum = 0;
                for (int j = 0; j < s; ++j) sum = fma_((T)Tab::a[s][j], k[j][f], sum);
                yi[s][f] = fma_(dt, sum, y[f]);
            }
            rhs(fma_((T)Tab::c[s], dt, t0), yi[s], k[s]);
        }
        for (int f = 0; f < F; ++f) y1[f] = yi[6][f];
        finish_backward_sample<T, T, METHOD, CTRL, false>(q, 0, 0, 1);
        for (int s = 6; s >= 1; --s) {
            T gk[F], gy[F];
            for (int f = 0; f < F; ++f) gk[f] = g_k[s][f];
            rhs.vjp((T)0, yi[s], gk, gy, gpar);
            for (int f = 0; f < F; ++f) g_ystage[f] = gy[f] + (s == 6 ? g_y1[f] : (T)0);
            stage_backward_sample<T, T, METHOD, false>(q, 0, s, g_ystage, (const T *)nullptr, 0, 1);
        }
        for (int f = 0; f < F; ++f) a_y[f] = g_y[f], a_k0[f] = g_k[0][f];
        a_t = g_t, a_dt = g_dt, a_prev = g_prev, a_pprev = g_pprev;
    }
    result.insert(result.end(), a_y, a_y + F), result.insert(result.end(), a_k0, a_k0 + F);
    for (T x : {a_t, a_dt, a_prev, a_pprev}) result.push_back(x);
    result.insert(result.end(), gpar, gpar + P);
}

template <typename T, typename Term> static void reference_mc(const tode_solve_args &a, const tode_controller &c, const tode_solve_adjoint &adj, std::vector<T> &result) {
    if (a.method == TODE_TSIT5) return c.kind == TODE_CTRL_PID ? reference<T, 1, 1, Term>(a, c, adj, result) : reference<T, 1, 0, Term>(a, c, adj, result);
    return c.kind == TODE_CTRL_PID ? reference<T, 0, 1, Term>(a, c, adj, result) : reference<T, 0, 0, Term>(a, c, adj, result);
}
}  // namespace tode

template <typename T> static bool same(unsigned seed) {
    std::mt19937_64 rng(seed);
    auto uniform = [&](double lo, double hi) { return (T)(lo + (hi - lo) * (double)(rng() >> 11) * 0x1p-53); };
    auto pick = [&](int lo, int hi) { return lo + (int)(rng() % (unsigned)(hi - lo + 1)); };
    const int kinds[][3] = {{TODE_TERM_VAN_DER_POL, 2, 1}, {TODE_TERM_LORENZ63, 3, 1}, {TODE_TERM_LINEAR_DECAY, 1, 1}, {TODE_TERM_LINEAR_DECAY, 4, 4}, {TODE_TERM_LINEAR_DECAY, 8, 8}};
    const auto *kind = kinds[pick(0, 4)];
    const int F = kind[1], P = kind[2], L = pick(0, 12) ? pick(1, 25) : 0, n = L + 1, E = pick(0, 5) ? pick(1, 40) : 0, times = pick(0, 6), scale = pick(0, 6);
    const double cotangents = scale == 0 ? 1e-30 : scale == 1 ? 1e-12 : 1, states = scale == 2 ? 1e-12 : 1, dir = pick(0, 1) ? 1 : -1;
    std::vector<T> t_eval(E), rt(n), rdt(n), ry(n * F), rk(n * F), prev(n), pprev(n), par(P), g(std::max(E, 1) * F);
    std::vector<int32_t> running(n), accepted(n);
    T ts = pick(0, 2) ? uniform(-2, 2) : (T)0, t = ts, te, ratio = 1, before = 1;
    int n_accepted = 0;
    const int last = pick(1, L + 1);
    for (int i = 0; i < n; ++i) {
        running[i] = i < last, rt[i] = t, rdt[i] = running[i] ? (T)(dir * (double)uniform(0.01, 0.6)) : (T)0, prev[i] = ratio, pprev[i] = before, accepted[i] = n_accepted;
        for (int f = 0; f < F; ++f) ry[i * F + f] = pick(0, 9) ? uniform(-2, 2) * (T)states : (T)0, rk[i * F + f] = uniform(-3, 3) * (T)states;
        if (scale == 3 && pick(0, 60) == 0) ry[i * F] = (T)INFINITY;
        if (running[i] && pick(0, 4)) t = t + rdt[i], ++n_accepted, before = ratio, ratio = pick(0, 20) ? (T)exp((double)uniform(-7, 2)) : (T)1e-38;
    }
    te = pick(0, 3) ? t : (T)(t + dir * 0.3);
    if (te == ts) te = (T)(ts + dir);
    for (int e = 0; e < E; ++e) {
        const double x = times == 1 ? (double)uniform(-0.3, 1.3) : times == 2 && pick(0, 3) == 0 ? 0.0 : E > 1 ? (double)e / (E - 1) : pick(0, 1);
        t_eval[e] = (T)(ts + x * ((double)te - ts) * (times == 3 ? 1.5 : 1));
        if (times == 4 && pick(0, 2) == 0) t_eval[e] = rt[pick(0, L)];
        if (times == 5 && pick(0, 20) == 0) t_eval[e] = (T)NAN;
    }
    if (times == 4) std::sort(t_eval.begin(), t_eval.end(), [&](T a, T b) { return dir * a < dir * b; });
    for (auto &p : par) p = kind[0] == TODE_TERM_LORENZ63 ? uniform(20, 30) : uniform(0.1, 5);
    for (auto &x : g) x = pick(0, 9) ? uniform(-1, 1) * (T)cotangents : (T)0;
    tode_solve_record r = {n, rt.data(), rdt.data(), ry.data(), rk.data(), prev.data(), pprev.data(), running.data(), accepted.data()};
    tode_solve_args a;
    memset(&a, 0, sizeof a);
    a.dtype = sizeof(T) == 4 ? TODE_F32 : TODE_F64, a.method = pick(0, 1) ? TODE_TSIT5 : TODE_DOPRI5, a.term = kind[0], a.n_features = F, a.n_params = P, a.n_eval = E, a.batch = 1;
    a.term_scalars[0] = 10, a.term_scalars[1] = 8.0 / 3, a.t_start = &ts, a.t_end = &te, a.t_start_stride = a.t_end_stride = 1, a.t_eval = t_eval.data(), a.params = par.data(), a.record = &r;
    tode_controller c;
    memset(&c, 0, sizeof c);
    c.kind = pick(0, 1) ? TODE_CTRL_PID : TODE_CTRL_INTEGRAL, c.atol = pick(0, 3) ? 1e-6 : 1e-2, c.rtol = 1e-4, c.pcoeff = 0.2, c.icoeff = pick(0, 5) ? 0.5 : 2.5, c.dcoeff = pick(0, 1) ? 0.05 : 0;
    c.safety = 0.9, c.factor_min = 0.2, c.factor_max = 10.0;
    if (pick(0, 4) == 0) c.has_dt_max = 1, c.dt_max = 0.4;
    if (pick(0, 4) == 0) c.has_dt_min = 1, c.dt_min = 0.05;
    tode_solve_adjoint adj;
    memset(&adj, 0, sizeof adj);
    adj.grad_ys = g.data(), adj.iterations = L, adj.through_control = pick(0, 3) != 0;
    std::vector<int32_t> scratch(2 * std::max(E, 1));
    adj.scratch = scratch.data(), adj.scratch_bytes = 4 * (int64_t)scratch.size();
    const bool wants_times = pick(0, 1);
    std::vector<T> found, expected;
    for (auto *result : {&found, &expected}) {
        std::vector<T> state(2 * F + 4 + P), of_times(2 + E);
        if (wants_times) adj.g_t_start = &of_times[0], adj.g_t_end = &of_times[1], adj.g_t_eval = &of_times[2];
        if (result == &found) {
            adj.a_y = &state[0], adj.a_k0 = &state[F], adj.a_t = &state[2 * F], adj.a_dt = &state[2 * F + 1], adj.a_prev = &state[2 * F + 2], adj.a_pprev = &state[2 * F + 3];
            adj.g_params = &state[2 * F + 4];
            if (tode_solve_builtin_backward(&a, &c, &adj, nullptr)) return false;
            *result = state;
        } else if (kind[0] == TODE_TERM_VAN_DER_POL) {
            tode::reference_mc<T, tode::VanDerPolTerm<T>>(a, c, adj, *result);
        } else if (kind[0] == TODE_TERM_LORENZ63) {
            tode::reference_mc<T, tode::Lorenz63Term<T>>(a, c, adj, *result);
        } else if (F == 1) {
            tode::reference_mc<T, tode::LinearDecayTerm<T, 1>>(a, c, adj, *result);
        } else if (F == 4) {
            tode::reference_mc<T, tode::LinearDecayTerm<T, 4>>(a, c, adj, *result);
        } else {
            tode::reference_mc<T, tode::LinearDecayTerm<T, 8>>(a, c, adj, *result);
        }
        result->insert(result->end(), of_times.begin(), of_times.end());
    }
    for (size_t i = 0; i < found.size(); ++i)
        if (!(found[i] == expected[i] || (found[i] != found[i] && expected[i] != expected[i]))) {
            fprintf(stderr, "seed %u: F %d, L %d, E %d, value %zu: %a instead of %a\n", seed, F, L, E, i, (double)found[i], (double)expected[i]);
            return false;
        }
    return found.size() == expected.size();
}

int main(int, char **v) {
    int runs = 0, wrong = 0;
    for (unsigned seed = atoi(v[1]); seed < (unsigned)atoi(v[2]); ++seed) runs += 2, wrong += !same<float>(2 * seed), wrong += !same<double>(2 * seed + 1);
    printf("%d %d\n", runs, wrong);
}
