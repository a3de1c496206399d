// One sample with one evaluation point through the whole-solve kernels of the small systems on the host (hip/hip_runtime.h
// here): ys is a heap block of exactly its size, so that the address sanitizer sees a write past it.
//     main {fast|pair} {f32|f64} {dopri5|tsit5} rate y0 t_start t_eval t_end
// prints: flag for the general kernel, steps, initialized points, the point's value.
#include <stdarg.h>
#include <stdio.h>
#include <stdlib.h>

#include "tode_fast.hip"
#include "tode_pair.hip"

namespace host {
thread_local dim3 thread_idx, block_idx, grid_dim;
unsigned char *lds;
Barrier barrier;
}  // namespace host

namespace tode {
int fail(int code, const char *fmt, ...) {
    va_list args;
    va_start(args, fmt);
    vfprintf(stderr, fmt, args);
    va_end(args);
    return code;
}
int check_hip(hipError_t, const char *) { return TODE_OK; }
const FlagTarget *flag_target() { return nullptr; }
void timing_before(hipStream_t, const char *) {}
void timing_after(hipStream_t) {}
}  // namespace tode

template <typename T> static int run(char **v) {
    const T rate = (T)atof(v[4]), y0 = (T)atof(v[5]), times[3] = {(T)atof(v[6]), (T)atof(v[7]), (T)atof(v[8])};
    std::vector<T> ys(1);
    int32_t flags[TODE_FLAG_WORDS];
    int64_t stats[4] = {0, 0, 0, 0};
    tode_solve_args a;
    memset(&a, 0, sizeof a);
    a.dtype = sizeof(T) == 4 ? TODE_F32 : TODE_F64;
    a.method = !strcmp(v[3], "tsit5") ? TODE_TSIT5 : TODE_DOPRI5;
    a.term = TODE_TERM_LINEAR_DECAY, a.n_features = a.n_params = a.n_eval = 1, a.batch = 1, a.max_steps = -1, a.iteration_cap = -1;
    a.y0 = &y0, a.t_start = times, a.t_eval = times + 1, a.t_end = times + 2, a.t_start_stride = a.t_end_stride = 1;
    a.params = &rate, a.ys = ys.data(), a.flags = flags;
    tode_controller c;
    memset(&c, 0, sizeof c);
    c.kind = TODE_CTRL_INTEGRAL, c.atol = 1e-6, c.rtol = 1e-4, c.safety = 0.9, c.factor_min = 0.2, c.factor_max = 10.0;
    const bool tsit5 = a.method == TODE_TSIT5;
    bool used = true;
    int rc;
    if (!strcmp(v[1], "fast")) {
        const tode::FastOut<T> o{stats, stats + 1, stats + 2, stats + 3};
        rc = tsit5 ? tode::launch_fast<T, 1, 0, tode::LinearDecayTerm<T, 1>>(a, c, o, nullptr) : tode::launch_fast<T, 0, 0, tode::LinearDecayTerm<T, 1>>(a, c, o, nullptr);
    } else {
        const tode::PairOut<T> o{stats, stats + 1, stats + 2, stats + 3};
        rc = tsit5 ? tode::launch_pair<T, 1, 0, tode::LinearDecayTerm<T, 1>>(a, c, o, nullptr, &used) : tode::launch_pair<T, 0, 0, tode::LinearDecayTerm<T, 1>>(a, c, o, nullptr, &used);
    }
    if (rc || !used) return 2;
    printf("%d %lld %lld %.17g\n", flags[TODE_FLAG_NEEDS_GENERAL], (long long)stats[0], (long long)stats[2], (double)ys[0]);
    return 0;
}

int main(int n, char **v) { return n != 9 ? 3 : (!strcmp(v[2], "f32") ? run<float>(v) : run<double>(v)); }
