// Reverse sweep of a solve with the two-layer perceptron as right-hand side (float32, up to 64 state values and 256 hidden
// units): what lies on either side of tode_step_finish_backward for one recorded iteration, and the gradients of the
// weights.  The reference leaves all of it to autograd over its loop (adjoints.py:135-260); through autograd it is, per
// iteration, six evaluations of the network and six vector-Jacobian products of some fifteen launches each.  Here:
//
//   mlp_stages_kernel           all six stages of an iteration again (a tile of 16 samples per workgroup, laid out as in
//                               the whole-solve kernel), keeping stage inputs, derivatives and hidden activations; of all
//                               iterations in one launch where their rows fit, since they depend on the record alone, and
//                               then the sums of the squares of the scaled errors for the sweep of a whole record as well;
//   mlp_sweep_control_kernel    ahead of that sweep: an iteration's step factor and the points it wrote, a thread each;
//   mlp_stages_backward_kernel  the six stages in reverse: the network's vector-Jacobian product and the stage sums' reverse,
//                               the cotangents of all stage derivatives in registers between them;
//   mlp_sweep_kernel            the iterations of a whole record in reverse, where the times want no gradient and the rows of all
//                               evaluations fit: the step rule's and the dense output's reverse between the iterations too;
//   mlp_weight_gradient_kernel  the two outer products over the rows of all evaluations of several iterations, split over
//                               the rows;
//   mlp_weight_gradient_sum_kernel  the splits' sums added in order, once per sweep.
//
// What bounds them, network of 64 and 256 at B = 4096 (one workgroup per compute unit, one wavefront per SIMD): six
// evaluations forward 28 us (three iterations in one launch 63 us, two workgroups to a compute unit), back 29 us, of which the
// matrix cores are busy 10.6 and 10.2 us -- the rest are the round trips through LDS between two products, the stage sums and
// 150 KB of weights loaded per workgroup; the outer products of 20 evaluations 69 us (34 us of matrix instructions at 2.4 GHz,
// 200 MB of rows at 2.9 TB/s).  A solve and its backward pass: 9.75 ms through autograd, 0.61 to 0.80 ms by the host's speed with the
// launches per iteration (0.42 ms of kernels), 0.46 to 0.54 in the one kernel, one call of it and one launch for
// the weights (0.38 ms).  Against float64 over the same record, 60 solves with rows shorter than 64, the one kernel and
// the launches per iteration (geometric means): y0 4.5e-7 and 4.6e-7, W1 8.5e-7 and 8.6e-7 with the steps held constant; y0 4.8e-5 and
// 4.8e-5, W1 1.00e-5 and 1.01e-5 through the step sizes.
//
// All products are on v_mfma_f32_16x16x4_f32.  For the vector-Jacobian product the weights are packed a second time,
// transposed (tode_mlp_pack_weights_reverse), so that the same two facts hold as in the forward kernel: every lane keeps its
// A operands in registers, and the first product's result, lane (q, c) holding the cotangents of hidden units 4q..4q+3 of
// sample c, is after (1 - h^2) already the second product's B operand.
#include "tode_adjoint.h"
#include "tode_mlp.h"

namespace tode {

constexpr int MLP_REVERSE_REGS = 64 + 64 + 16;  // packed values per thread: W2 transposed, W1 transposed, W1's time column
// sums per split: W1 without its time column as [64 inputs][256 units] | time column | b1 | W2 [64][256] | b2
constexpr int MLP_SUM_W1T = MLP_F * MLP_H, MLP_SUM_B1 = MLP_SUM_W1T + MLP_H, MLP_SUM_W2 = MLP_SUM_B1 + MLP_H, MLP_SUM_B2 = MLP_SUM_W2 + MLP_F * MLP_H;
constexpr int MLP_SUMS = MLP_SUM_B2 + MLP_F;

// Where value i of the transposed order comes from in W1 | b1 | W2 | b2, or -1 for zero.
__device__ __forceinline__ long long mlp_reverse_source(int i, int H, int FR) {
    const int tid = (i / 4) % 256, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15;
    int j = 4 * (i / 1024) + i % 4;
    const long long o_w2 = (long long)H * (FR + 1) + H;
    long long src = -1;
    if (j < 64) {  // W2[16q + kk][64w + 16 tile + c]
        const int f = 16 * q + j / 4, unit = 64 * w + 16 * (j % 4) + c;
        if (f < FR && unit < H) src = o_w2 + (long long)f * H + unit;
    } else if (j < 128) {  // W1[64w + 16 tile + 4q + r][16 it + c]
        j -= 64;
        const int input = 16 * (j / 16) + c, unit = 64 * w + 16 * ((j / 4) % 4) + 4 * q + j % 4;
        if (input < FR && unit < H) src = (long long)unit * (FR + 1) + input;
    } else {  // W1[64w + 16 tile + 4q + r][time]
        j -= 128;
        const int unit = 64 * w + 16 * (j / 4) + 4 * q + j % 4;
        if (unit < H) src = (long long)unit * (FR + 1) + FR;
    }
    return src;
}

static __global__ void mlp_pack_reverse_kernel(const float *raw, float *packed, int H, int FR) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= MLP_REVERSE_REGS * 256) return;
    const long long src = mlp_reverse_source(i, H, FR);
    packed[i] = src < 0 ? 0.0f : raw[src];
}

// Both orders (tode_mlp_pack_weights_for's for float32 and the transposed one behind it) straight from the four tensors, in one
// launch: a solve whose gradient is wanted packs its weights anew every time, and putting the tensors one behind the other and
// packing them in two more launches, then all of it again ahead of the reverse sweep, left the GPU waiting for the host five times.
static __global__ void mlp_pack_both_kernel(const float *W1, const float *b1, const float *W2, const float *b2, float *packed, int H, int FR) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (MLP_REGS + MLP_REVERSE_REGS) * 256) return;
    long long src;
    if (i < MLP_REGS * 256) {
        const int tid = (i / 4) % 256, j = 4 * (i / 1024) + i % 4;  // (16-byte chunks: lane-contiguous loads of four values per thread)
        src = mlp_packed_source(j, tid, H, FR);
    } else {
        src = mlp_reverse_source(i - MLP_REGS * 256, H, FR);
    }
    const long long o_b1 = (long long)H * (FR + 1), o_w2 = o_b1 + H, o_b2 = o_w2 + (long long)FR * H;
    packed[i] = src < 0 ? 0.0f : src < o_b1 ? W1[src] : src < o_w2 ? b1[src - o_b1] : src < o_b2 ? W2[src - o_w2] : b2[src - o_b2];
}

// The lane's four features f0 .. f0 + 3 of a row of FR values: 16 bytes at a time where rows are whole groups of four.
__device__ __forceinline__ void mlp_get(const float *row, int f0, int FR, float (&v)[4]) {
    if ((FR & 3) == 0) {
        const float4 u = f0 < FR ? *reinterpret_cast<const float4 *>(row + f0) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = f0 + r < FR ? row[f0 + r] : 0.0f;
    }
}

__device__ __forceinline__ void mlp_put(float *row, int f0, int FR, const float (&v)[4]) {
    if ((FR & 3) == 0) {
        if (f0 < FR) *reinterpret_cast<float4 *>(row + f0) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (f0 + r < FR) row[f0 + r] = v[r];
    }
}

// error_sums: where not null, the sum over a row of the squares of its scaled errors, as the solve formed it.
template <int METHOD>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) mlp_stages_kernel(const tode_mlp_reverse p, float atol, float rtol, float *error_sums) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    __shared__ MlpShared sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15, FR = p.n_features, f0 = 16 * w + 4 * q;
    const long long B = p.batch, tiles = (B + MLP_TILE - 1) / MLP_TILE;
    const float sf = (float)__builtin_sqrt((double)FR);
    MlpWeights W;
    mlp_load(W, (const float *)p.packed, tid);
    for (int i = tid; i < MLP_TILE * MLP_XS; i += 256) sh.x[i] = 0.0f;  // also the zero columns from 65 on
    __syncthreads();
    int slot = 0;
    for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const bool live = tile * MLP_TILE + c < B;
        const long long b = live ? tile * MLP_TILE + c : B - 1;
        const float t = ((const float *)p.t)[b], dt = ((const float *)p.dt)[b];
        float y[4], k[7][4];
        mlp_get((const float *)p.y + b * FR, f0, FR, y);
        mlp_get((const float *)p.k0 + b * FR, f0, FR, k[0]);
#pragma unroll
        for (int s = 1; s < 7; ++s) {
            float yi[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                float sum = 0;
#pragma unroll
                for (int j = 0; j < s; ++j) sum = fma_((float)Tab::a[s][j], k[j][r], sum);
                yi[r] = fma_(dt, sum, y[r]);
            }
            const float tn = fma_((float)Tab::c[s], dt, t);
            const long long row = (s - 1) * B + b;
            if (live) {
                mlp_put((float *)p.stage_inputs + row * FR, f0, FR, yi);
                if (w == 0 && q == 0) ((float *)p.stage_times)[row] = tn;
            }
            mlp_rhs<true>(sh, W, tn, yi, k[s], live ? (float *)p.hidden + row * MLP_H : nullptr);
            if (live) mlp_put((float *)p.k + row * FR, f0, FR, k[s]);
            if (s == 6 && error_sums) {
                float part[4], none[4] = {0, 0, 0, 0}, acc, unused;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float err = 0;
#pragma unroll
                    for (int j = 0; j < 7; ++j) err = fma_(dt * (float)Tab::b_err[j], k[j][r], err);
                    const float m = tmax(abs_(y[r]), abs_(yi[r]));
                    const float x = (abs_(err) / fma_(rtol, m, atol)) / sf;
                    part[r] = f0 + r < FR ? x * x : 0.0f;
                }
                mlp_sum2(sh, slot, part, none, acc, unused);
                if (live && w == 0 && q == 0) error_sums[b] = acc;
            }
        }
    }
}

struct __align__(16) MlpReverseShared {
    float g[MLP_TILE * MLP_XS];   // cotangent of the stage derivative: [sample][feature]
    float part[4][4][64][4];      // [16 inputs][wavefront it comes from][lane][4 inputs]
    float red[2][4][MLP_TILE][2]; // sums over a sample's features (mlp_sum2)
};

struct MlpReverseWeights {
    float w2t[16][4];   // W2[16q + kk][64w + 16 tile + c]
    float w1t[4][16];   // W1[64w + 16 tile + 4q + r][16 it + c]
    float wt[16];       // W1[64w + 16 tile + 4q + r][time]
};

__device__ __forceinline__ void mlp_load(MlpReverseWeights &W, const float *packed, int tid) {
    const float4 *src = reinterpret_cast<const float4 *>(packed) + tid;
#pragma unroll
    for (int i = 0; i < MLP_REVERSE_REGS / 4; ++i) {
        const float4 u = src[i * 256];
        const float v[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (i < 16) W.w2t[i][r] = v[r];
            else if (i < 32) W.w1t[(i - 16) / 4][4 * ((i - 16) % 4) + r] = v[r];
            else W.wt[4 * (i - 32) + r] = v[r];
        }
    }
}

// The network's vector-Jacobian product for the lane's sample: g (cotangent of f, the lane's four features) to gi (of y) and
// gt (of t: this lane's share, to be summed over the sample's lanes).  hidden: the sample's row of hidden activations;
// cotangents: its row of the cotangents in front of tanh, to be written, or null.
__device__ __forceinline__ void mlp_vjp(MlpReverseShared &sh, const MlpReverseWeights &W, const float (&gf)[4], const float *hidden, float *cotangents, float (&gi)[4], float &gt) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, c = lane & 15;
    *reinterpret_cast<float4 *>(sh.g + c * MLP_XS + 16 * w + 4 * q) = make_float4(gf[0], gf[1], gf[2], gf[3]);
    float4 h[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) h[u] = *reinterpret_cast<const float4 *>(hidden + 64 * w + 16 * u + 4 * q);
    lds_barrier();
    float g[16];
    {
        const float4 *at = reinterpret_cast<const float4 *>(sh.g + c * MLP_XS + 16 * q);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 v = at[j];
            g[4 * j] = v.x, g[4 * j + 1] = v.y, g[4 * j + 2] = v.z, g[4 * j + 3] = v.w;
        }
    }
    mfma_acc d[4], acc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) d[u] = {0.0f, 0.0f, 0.0f, 0.0f}, acc[u] = {0.0f, 0.0f, 0.0f, 0.0f};
    gt = 0;
    const auto in_front_of_tanh = [&](int n) {
        const int u = n / 4, r = n % 4;
        const float hv = r == 0 ? h[u].x : r == 1 ? h[u].y : r == 2 ? h[u].z : h[u].w;
        const float v = d[u][r] * fma_(-hv, hv, 1.0f);
        gt = fma_(W.wt[n], v, gt);
        return v;
    };
    // (in the order of mlp_rhs: two tiles of hidden units at a time, the first two's way through tanh's derivative behind the
    // other two's products and theirs behind the first two's part of the second product)
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
#pragma unroll
        for (int u = 0; u < 2; ++u) d[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w2t[kk][u], g[kk], d[u], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
#pragma unroll
        for (int kk = 2 * n; kk < 2 * n + 2; ++kk)
#pragma unroll
            for (int u = 2; u < 4; ++u) d[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w2t[kk][u], g[kk], d[u], 0, 0, 0);
        float v = in_front_of_tanh(n);
        if (n < 7) asm volatile("" : "+v"(v), "+v"(g[2 * n + 2]), "+v"(g[2 * n + 3]));  // (the next group behind this value)
        d[n / 4][n % 4] = v;
        mlp_interleave<3>();
    }
#pragma unroll
    for (int n = 0; n < 8; ++n) {
#pragma unroll
        for (int it = 0; it < 4; ++it) acc[it] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w1t[it][n], d[n / 4][n % 4], acc[it], 0, 0, 0);
        d[2 + n / 4][n % 4] = in_front_of_tanh(8 + n);
        mlp_interleave<3>();
    }
    if (cotangents) {
#pragma unroll
        for (int u = 0; u < 4; ++u) *reinterpret_cast<float4 *>(cotangents + 64 * w + 16 * u + 4 * q) = make_float4(d[u][0], d[u][1], d[u][2], d[u][3]);
    }
#pragma unroll
    for (int n = 8; n < 16; ++n)
#pragma unroll
        for (int it = 0; it < 4; ++it) acc[it] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w1t[it][n], d[n / 4][n % 4], acc[it], 0, 0, 0);
#pragma unroll
    for (int it = 0; it < 4; ++it) *reinterpret_cast<float4 *>(sh.part[it][w][lane]) = make_float4(acc[it][0], acc[it][1], acc[it][2], acc[it][3]);
    lds_barrier();
    float4 v[4];
#pragma unroll
    for (int from = 0; from < 4; ++from) v[from] = *reinterpret_cast<const float4 *>(sh.part[w][from][lane]);
    gi[0] = (v[0].x + v[1].x) + (v[2].x + v[3].x);
    gi[1] = (v[0].y + v[1].y) + (v[2].y + v[3].y);
    gi[2] = (v[0].z + v[1].z) + (v[2].z + v[3].z);
    gi[3] = (v[0].w + v[1].w) + (v[2].w + v[3].w);
}

// One wavefront per SIMD: 144 registers of weights, 28 + 24 of stage derivatives and their cotangents.  A workgroup takes
// several tiles where the batch has more than the grid, so that the weights are loaded once.
template <int METHOD> __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) mlp_stages_backward_kernel(const tode_mlp_reverse p) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    __shared__ MlpReverseShared sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15, FR = p.n_features, f0 = 16 * w + 4 * q;
    const long long B = p.batch, R = p.stage_rows > 0 ? p.stage_rows : B, tiles = (B + MLP_TILE - 1) / MLP_TILE;
    MlpReverseWeights W;
    mlp_load(W, (const float *)p.packed_reverse, tid);
    int slot = 0;
    for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const bool live = tile * MLP_TILE + c < B;
        const long long b = live ? tile * MLP_TILE + c : B - 1;
        const float dt = ((const float *)p.dt)[b];
        float k[6][4], gk[7][4], gy[4], gy1[4], g_t = 0, g_dt = 0;
        mlp_get((const float *)p.k0 + b * FR, f0, FR, k[0]);
#pragma unroll
        for (int s = 1; s < 6; ++s) mlp_get((const float *)p.k + ((s - 1) * R + b) * FR, f0, FR, k[s]);
#pragma unroll
        for (int s = 0; s < 7; ++s) mlp_get((const float *)p.g_k + (s * B + b) * FR, f0, FR, gk[s]);
        mlp_get((const float *)p.g_y + b * FR, f0, FR, gy);
        mlp_get((const float *)p.g_y1 + b * FR, f0, FR, gy1);
#pragma unroll
        for (int s = 6; s >= 1; --s) {
            const long long row = (s - 1) * R + b;
            if (live && p.stage_cotangents) mlp_put((float *)p.stage_cotangents + row * FR, f0, FR, gk[s]);  // (final: the weights' gradients read it)
            float gi[4], gt;
            mlp_vjp(sh, W, gk[s], (const float *)p.hidden + row * MLP_H, live && p.hidden_cotangents ? (float *)p.hidden_cotangents + row * MLP_H : nullptr, gi, gt);
            g_t += gt;
            g_dt = fma_((float)Tab::c[s], gt, g_dt);
            // the stage's sum reversed (stage_backward_sample)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (s == 6) gi[r] += gy1[r];
                gy[r] += gi[r];
                float sum = 0;
#pragma unroll
                for (int j = 0; j < s; ++j) {
                    sum = fma_((float)Tab::a[s][j], k[j][r], sum);
                    gk[j][r] += (float)Tab::a[s][j] * dt * gi[r];
                }
                g_dt = fma_(gi[r], sum, g_dt);
            }
        }
        const float share_t[4] = {g_t, 0, 0, 0}, share_dt[4] = {g_dt, 0, 0, 0};
        mlp_sum2(sh, slot, share_t, share_dt, g_t, g_dt);
        if (live) {
            mlp_put((float *)p.g_y + b * FR, f0, FR, gy);
            mlp_put((float *)p.g_k + b * FR, f0, FR, gk[0]);
            if (w == 0 && q == 0) {
                ((float *)p.g_t)[b] += g_t;
                ((float *)p.g_dt)[b] += g_dt;
            }
        }
    }
}

// What an iteration of a sample is to the sweep below, ahead of it (one thread per iteration and sample; none of it waits for a
// cotangent): the error ratio's root mean square from the stages' sum, the step factor before its clip, and the evaluation points
// the iteration wrote (adjoints.py:215-234: those that its new time has reached and the time before it had not; times run in the
// direction of the solve).  In a kernel of its own because powers and searches branch lane by lane, and the sweep holds more
// registers than this compiler keeps whole across such branches (copies_ahead_of_the_exec_restore in build.py).
struct MlpIteration {
    float rms, F0;
    int first, end;
};

template <int CTRL> __global__ void __launch_bounds__(256) mlp_sweep_control_kernel(const tode_mlp_sweep s, long long B, const CtrlParams<float> cp) {
    const long long at = (long long)blockIdx.x * 256 + threadIdx.x;
    if (at >= s.iterations * B) return;
    const long long n = at / B, b = at - n * B;
    const tode_solve_record &rec = s.record;
    MlpIteration *const out = (MlpIteration *)s.control + at;
    const float te = ((const float *)s.t_end)[b * s.t_end_stride], ts = ((const float *)s.t_start)[b * s.t_start_stride], dir = te > ts ? 1.0f : -1.0f;
    const float rms = sqrt_(((const float *)s.error_sums)[at]), ratio = tmax(rms, 1e-38f);
    float F0 = cp.safety * rpow_common<float>(ratio, cp.e1);
    if (CTRL == 1) {
        F0 = F0 * (cp.skip2 ? 1.0f : rpow_common<float>(((const float *)rec.prev)[at], cp.e2));
        F0 = F0 * (cp.skip3 ? 1.0f : rpow_common<float>(((const float *)rec.pprev)[at], cp.e3));
    }
    const float *const times = (const float *)s.t_eval + b * s.n_eval;
    const int lowest = times[0] == ts ? 1 : 0;  // (written by the loop's set-up)
    auto reached = [&](float t) {  // how many points lie no further than t
        int lo = 0, hi = s.n_eval;
        while (lo < hi) {
            const int mid = (lo + hi) / 2;
            if (dir * t < dir * times[mid]) hi = mid;
            else lo = mid + 1;
        }
        return max(lo, lowest);
    };
    out->rms = rms, out->F0 = F0;
    out->first = n == 0 ? lowest : reached(((const float *)rec.t)[at]), out->end = reached(((const float *)rec.t)[at + B]);
    if (n == 0) ((float *)s.t_end_dense)[b] = te;
}

// The whole loop of a recorded solve in reverse, a tile of 16 samples from its last iteration to its first: what
// finish_backward_kernel and mlp_stages_backward_kernel do for one iteration, launch by launch, with the cotangents of the state
// between the iterations in registers and the transposed weights loaded once.  A sample's row lies across sixteen lanes as in the
// products: lane (q, c) of wavefront w holds features 16w + 4q .. + 3 of sample c, and every lane its sample's scalars.
//
// What a feature's cotangents are made of keeps the operations and the order of the two kernels (points in ascending order, five
// sums a feature, spread once; shorter rows than 64 the former sweeps point by point), so that gradients with the step sizes held
// constant are theirs bit for bit; sums over a
// sample's features are the solve kernel's (mlp_sum2).  B = 4096, three iterations: 101 us, where three times the two kernels took 138.
template <int METHOD, int CTRL>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) mlp_sweep_kernel(const tode_mlp_reverse p, const tode_mlp_sweep s, const CtrlParams<float> cp) {
    using Tab = typename std::conditional<METHOD == 1, Tsit5Tab, Dopri5Tab>::type;
    __shared__ MlpReverseShared sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15, FR = p.n_features, f0 = 16 * w + 4 * q, E = s.n_eval;
    const long long B = p.batch, L = s.iterations, R = L * B, tiles = (B + MLP_TILE - 1) / MLP_TILE;
    const float sf = (float)__builtin_sqrt((double)FR);
    const tode_solve_record &rec = s.record;
    MlpReverseWeights W;
    mlp_load(W, (const float *)p.packed_reverse, tid);
    int slot = 0;
    for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const bool live = tile * MLP_TILE + c < B;
        const long long b = live ? tile * MLP_TILE + c : B - 1;
        const float ts = ((const float *)s.t_start)[b * s.t_start_stride], te = ((const float *)s.t_end)[b * s.t_end_stride];
        const float tlo = tmin(ts, te), thi = tmax(te, ts);
        const float *const times = (const float *)s.t_eval + b * E;
        const float *const grad_ys = (const float *)s.grad_ys + b * E * FR;
        float a_y[4] = {0, 0, 0, 0}, a_k0[4] = {0, 0, 0, 0}, a_t = 0, a_dt = 0, a_prev = 0, a_pprev = 0;
        int running_after = rec.running[L * B + b], accepted_after = rec.n_accepted[L * B + b];
        for (long long n = L - 1; n >= 0; --n) {
            const long long at = n * B + b;
            const float t0 = ((const float *)rec.t)[at], dt = ((const float *)rec.dt)[at], prev = ((const float *)rec.prev)[at], pprev = ((const float *)rec.pprev)[at];
            const int running = rec.running[at], accepted = rec.n_accepted[at];
            const bool move = accepted_after > accepted, running_new = running_after != 0;
            float y[4], y1[4], k[7][4];
            mlp_get((const float *)rec.y + at * FR, f0, FR, y);
            mlp_get((const float *)rec.k0 + at * FR, f0, FR, k[0]);
            mlp_get((const float *)p.stage_inputs + (5 * R + at) * FR, f0, FR, y1);
#pragma unroll
            for (int j = 1; j < 7; ++j) mlp_get((const float *)p.k + ((j - 1) * R + at) * FR, f0, FR, k[j]);

            const MlpIteration it = ((const MlpIteration *)s.control)[at];
            const int n_points = it.end - it.first;
            const float rms = it.rms, F0 = it.F0, ratio = tmax(rms, 1e-38f);
            const float factor = tclamp(F0, cp.fmin, cp.fmax);
            const float t_new = move ? (t0 + dt) : t0, lo = tlo - t_new, hi = thi - t_new, dtn = running_new ? dt * factor : dt;

            // ---- clamp of the step to the time range, and the new time ----
            const float g_self = (dtn >= lo && dtn <= hi) ? a_dt : 0.0f, g_lo = (dtn < lo && lo < hi) ? a_dt : 0.0f, g_hi = (dtn > hi || hi < lo) ? a_dt : 0.0f;
            const float g_tnew = a_t - (g_lo + g_hi), g_dt_next = running_new ? g_self : 0.0f;
            float g_t = g_tnew, g_dt = running_new ? 0.0f : g_self;
            if (move) g_dt += g_tnew;

            // ---- controller history and step proposal ----
            float g_ratio = 0, g_prev = 0, g_pprev = 0;
            if (CTRL == 1) {
                const bool keep = running_new && move;
                g_ratio = keep ? a_prev : 0.0f;
                g_prev = keep ? a_pprev : a_prev;
                g_pprev = keep ? 0.0f : a_pprev;
            }
            if (s.through_control) {
                g_dt += g_dt_next * factor;
                const float g_factor = g_dt_next * dt, g_F0 = (F0 >= cp.fmin && F0 <= cp.fmax) ? g_factor : 0.0f;
                g_ratio += g_F0 * F0 * (float)cp.e1 / ratio;
                if (CTRL == 1) {
                    if (!cp.skip2) g_prev += g_F0 * F0 * (float)cp.e2 / prev;
                    if (!cp.skip3) g_pprev += g_F0 * F0 * (float)cp.e3 / pprev;
                }
            }

            // ---- error ratio and error estimate; state update ----
            const float tiny = 1e-38f, g_r = rms > tiny ? g_ratio : (rms == tiny ? g_ratio / 2.0f : 0.0f);
            float share_t = 0, share_dt = 0;  // (this lane's, summed over the sample's lanes at the end)
            float gk[7][4], gy[4], gy1[4];
            const bool through_error = g_r != 0.0f && rms > 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                gy[r] = move ? 0.0f : a_y[r], gy1[r] = move ? a_y[r] : 0.0f;
#pragma unroll
                for (int j = 0; j < 7; ++j) gk[j][r] = 0;
                gk[0][r] = move ? 0.0f : a_k0[r], gk[6][r] = move ? a_k0[r] : 0.0f;
            }
            if (lanes_where(through_error)) {  // (what a lane does not have is selected away, as everywhere here)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const bool on = through_error && f0 + r < FR;
                    float err = 0, bk = 0;
#pragma unroll
                    for (int j = 0; j < 7; ++j) err = fma_(dt * (float)Tab::b_err[j], k[j][r], err), bk = fma_((float)Tab::b_err[j], k[j][r], bk);
                    const float ay = abs_(y[r]), ay1 = abs_(y1[r]);
                    const float eb = fma_(cp.rtol, tmax(ay, ay1), cp.atol);
                    const float x = abs_(err) / eb;
                    const float g_q = g_r * (x / sf) / rms / sf;
                    const float g_err = on ? g_q / eb * sign_(err) : 0.0f;
                    const float g_m = on ? -g_q * x / eb * cp.rtol : 0.0f;
                    float ga, gb;
                    max_backward<float>(ay, ay1, g_m, ga, gb);
                    gy[r] += ga * sign_(y[r]);
                    gy1[r] += gb * sign_(y1[r]);
#pragma unroll
                    for (int j = 0; j < 7; ++j) gk[j][r] += g_err * (dt * (float)Tab::b_err[j]);
                    share_dt += on ? g_err * bk : 0.0f;
                }
            }

            // ---- dense output: five sums a feature over the points, then their shares ----
            float den = (t0 + dt) - t0;
            const bool flat = !(abs_(den) > 0.0f);
            if (flat) den = 1.0f;
            float G[4][5];
            bool any[4] = {false, false, false, false};
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < 5; ++i) G[r][i] = 0;
            for (int j = 0; lanes_where(j < n_points); j += 4) {  // (the cotangents of four points are on their way together)
                float cotangent[4][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) mlp_get(grad_ys + (long long)max(min(it.first + j + i, it.end - 1), 0) * FR, f0, FR, cotangent[i]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool taken = j + i < n_points;
                    const float x = (times[max(min(it.first + j + i, it.end - 1), 0)] - t0) / den;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        float g = cotangent[i][r];
                        const bool adds = taken && g != 0.0f;  // (zero adds nothing, wherever the point lies: its position may be an infinity)
                        any[r] = any[r] || adds;
#pragma unroll
                        for (int m = 0; m < 5; ++m) G[r][m] = adds ? G[r][m] + g : G[r][m], g = g * x;
                    }
                }
            }
            float g_points = 0, g_points_x = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float ks[7] = {k[0][r], k[1][r], k[2][r], k[3][r], k[4][r], k[5][r], k[6][r]};
                float co[5][1], more_dt = 0;
                quartic_elem<float, METHOD>(dt, y[r], y1[r], ks, true, co);
                const float *g = G[r];
                const bool on = any[r];  // (a state that is not finite adds nothing where no cotangent came)
                g_points += on ? g[0] * co[1][0] + 2.0f * (g[1] * co[2][0]) + 3.0f * (g[2] * co[3][0]) + 4.0f * (g[3] * co[4][0]) : 0.0f;
                g_points_x += on ? g[1] * co[1][0] + 2.0f * (g[2] * co[2][0]) + 3.0f * (g[3] * co[3][0]) + 4.0f * (g[4] * co[4][0]) : 0.0f;
                auto add = [&](float &to, float v) { to = on ? to + v : to; };
                if (METHOD == 1) {
                    add(gy[r], g[0]);
                    add(gk[0][r], g[1] * dt);
                    more_dt += g[1] * ks[0];
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const float u = g[2] * (float)Tsit5Tab::w[0][j] + g[3] * (float)Tsit5Tab::w[1][j] + g[4] * (float)Tsit5Tab::w[2][j];
                        add(gk[j][r], u * dt);
                        more_dt += u * ks[j];
                    }
                } else {
                    const float g_f0 = -2.0f * g[4] + 5.0f * g[3] - 4.0f * g[2] + g[1], g_f1 = 2.0f * g[4] - 3.0f * g[3] + g[2];
                    const float g_mid = 16.0f * g[4] - 32.0f * g[3] + 16.0f * g[2];
                    add(gy[r], -8.0f * g[4] + 18.0f * g[3] - 11.0f * g[2] + g[0] + g_mid);
                    add(gy1[r], -8.0f * g[4] + 14.0f * g[3] - 5.0f * g[2]);
                    add(gk[0][r], g_f0 * dt);
                    add(gk[6][r], g_f1 * dt);
                    more_dt += g_f0 * ks[0] + g_f1 * ks[6];
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        add(gk[j][r], g_mid * (dt * (float)Dopri5Tab::w[0][j]));
                        more_dt += g_mid * (float)Dopri5Tab::w[0][j] * ks[j];
                    }
                }
                share_dt += on ? more_dt : 0.0f;
            }
            share_t -= g_points / den;
            share_dt -= flat ? 0.0f : g_points_x / den;

            // ---- the stages reversed (mlp_stages_backward_kernel) ----
#pragma unroll
            for (int j = 6; j >= 1; --j) {
                const long long row = (j - 1) * R + at;
                if (live && p.stage_cotangents) mlp_put((float *)p.stage_cotangents + row * FR, f0, FR, gk[j]);
                float gi[4], gt;
                mlp_vjp(sh, W, gk[j], (const float *)p.hidden + row * MLP_H, live && p.hidden_cotangents ? (float *)p.hidden_cotangents + row * MLP_H : nullptr, gi, gt);
                share_t += gt;
                share_dt = fma_((float)Tab::c[j], gt, share_dt);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (j == 6) gi[r] += gy1[r];
                    gy[r] += gi[r];
                    float sum = 0;
#pragma unroll
                    for (int i = 0; i < j; ++i) {
                        sum = fma_((float)Tab::a[j][i], k[i][r], sum);
                        gk[i][r] += (float)Tab::a[j][i] * dt * gi[r];
                    }
                    share_dt = fma_(gi[r], sum, share_dt);
                }
            }
            const float of_t[4] = {share_t, 0, 0, 0}, of_dt[4] = {share_dt, 0, 0, 0};
            float sum_t, sum_dt;
            mlp_sum2(sh, slot, of_t, of_dt, sum_t, sum_dt);
#pragma unroll
            for (int r = 0; r < 4; ++r) a_y[r] = gy[r], a_k0[r] = gk[0][r];
            a_t = g_t + sum_t, a_dt = g_dt + sum_dt, a_prev = g_prev, a_pprev = g_pprev;
            running_after = running, accepted_after = accepted;
        }
        if (live) {
            mlp_put((float *)s.a_y + b * FR, f0, FR, a_y);
            mlp_put((float *)s.a_k0 + b * FR, f0, FR, a_k0);
            if (w == 0 && q == 0) ((float *)s.a_dt)[b] = a_dt;
        }
    }
}

// The start of the loop (y = y0, k0 = f(t_start, y0) and, with THROUGH, the step of the start rule clamped to the time range,
// step_size_controllers.py:431-490 / 776-835, adjoints.py:86-107), its evaluations of the network again: slot 0 of the stage
// buffers f(t_start, y0), slot 1 (THROUGH) the start rule's probe, whose value goes to p.k.
__device__ __forceinline__ void mlp_start_scale(const CtrlParams<float> &cp, int f0, int FR, float sf, const float (&y)[4], const float (&k0)[4], float (&inv)[4], float (&a0)[4],
                                                float (&a1)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        inv[r] = f0 + r < FR ? 1.0f / fma_(cp.rtol, abs_(y[r]), cp.atol) : 0.0f;  // (features beyond the problem's add nothing to the norms)
        const float u = (y[r] * inv[r]) / sf, v = (k0[r] * inv[r]) / sf;
        a0[r] = u * u, a1[r] = v * v;
    }
}

__device__ __forceinline__ float mlp_start_probe_step(float d0, float d1, float span, bool &small, float &h0a) {
    small = d0 < 1e-5f || d1 < 1e-5f;
    h0a = small ? 1e-6f : (0.01f * d0) / d1;
    return tmin(h0a, span);
}

template <bool THROUGH>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) mlp_start_kernel(const tode_mlp_reverse p, const tode_mlp_start st, const CtrlParams<float> cp) {
    __shared__ MlpShared sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15, FR = p.n_features, f0 = 16 * w + 4 * q;
    const long long B = p.batch, tiles = (B + MLP_TILE - 1) / MLP_TILE;
    const float sf = (float)__builtin_sqrt((double)FR);
    MlpWeights W;
    mlp_load(W, (const float *)p.packed, tid);
    for (int i = tid; i < MLP_TILE * MLP_XS; i += 256) sh.x[i] = 0.0f;
    __syncthreads();
    int slot = 0;
    for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const bool live = tile * MLP_TILE + c < B;
        const long long b = live ? tile * MLP_TILE + c : B - 1;
        float y[4], k0[4], out[4];
        mlp_get((const float *)p.y + b * FR, f0, FR, y);
        mlp_get((const float *)p.k0 + b * FR, f0, FR, k0);
        const auto evaluate = [&](int at, float t, const float (&x)[4]) {
            const long long row = at * B + b;
            if (live) {
                mlp_put((float *)p.stage_inputs + row * FR, f0, FR, x);
                if (w == 0 && q == 0) ((float *)p.stage_times)[row] = t;
            }
            mlp_rhs<true>(sh, W, t, x, out, live ? (float *)p.hidden + row * MLP_H : nullptr);
        };
        const float ts = ((const float *)p.t)[b], te = ((const float *)st.t_end)[b];
        evaluate(0, ts, y);
        if (THROUGH) {
            float inv[4], a0[4], a1[4], d0, d1, h0a, y1[4];
            mlp_start_scale(cp, f0, FR, sf, y, k0, inv, a0, a1);
            mlp_sum2(sh, slot, a0, a1, d0, d1);
            bool small;
            const float dir = te > ts ? 1.0f : -1.0f, h0 = mlp_start_probe_step(sqrt_(d0), sqrt_(d1), abs_(te - ts), small, h0a);
#pragma unroll
            for (int r = 0; r < 4; ++r) y1[r] = fma_(dir * h0, k0[r], y[r]);
            evaluate(1, fma_(dir, h0, ts), y1);
            if (live) mlp_put((float *)p.k + b * FR, f0, FR, out);
        }
    }
}

// The same reversed: the cotangents a_y, a_k0, a_dt of the first loop state to that of y0 (p.g_y), those of the two evaluations of
// the network left in p.stage_cotangents for the weights' gradients.  The times are constants here.  (start_backward of
// the small systems, a sample's row spread over sixteen lanes; a term that a sample does not have is selected away, since
// all lanes meet at the barriers of the sums and products.)
template <bool THROUGH>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) mlp_start_backward_kernel(const tode_mlp_reverse p, const tode_mlp_start st, const CtrlParams<float> cp,
                                                                                                           const bool integral) {
    __shared__ MlpReverseShared sh;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15, FR = p.n_features, f0 = 16 * w + 4 * q;
    const long long B = p.batch, tiles = (B + MLP_TILE - 1) / MLP_TILE;
    const float sf = (float)__builtin_sqrt((double)FR);
    const auto share_of_min = [](float a, float b) { return a < b ? 1.0f : (a == b ? 0.5f : 0.0f); };
    const auto share_of_max = [](float a, float b) { return a > b ? 1.0f : (a == b ? 0.5f : 0.0f); };
    MlpReverseWeights W;
    mlp_load(W, (const float *)p.packed_reverse, tid);
    int slot = 0;
    for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const bool live = tile * MLP_TILE + c < B;
        const long long b = live ? tile * MLP_TILE + c : B - 1;
        float g_y0[4], g_k0[4], gi[4], gt;
        mlp_get((const float *)st.a_y + b * FR, f0, FR, g_y0);
        mlp_get((const float *)st.a_k0 + b * FR, f0, FR, g_k0);
        const auto product = [&](int at, const float (&g)[4]) {
            const long long row = at * B + b;
            if (live && p.stage_cotangents) mlp_put((float *)p.stage_cotangents + row * FR, f0, FR, g);
            mlp_vjp(sh, W, g, (const float *)p.hidden + row * MLP_H, live && p.hidden_cotangents ? (float *)p.hidden_cotangents + row * MLP_H : nullptr, gi, gt);
        };
        if (THROUGH) {
            // ---- forward values ----
            float y[4], k0[4], f1[4], inv[4], a0[4], a1[4], a2[4], none[4] = {0, 0, 0, 0}, A0, A1, A2, unused;
            mlp_get((const float *)p.y + b * FR, f0, FR, y);
            mlp_get((const float *)p.k0 + b * FR, f0, FR, k0);
            mlp_get((const float *)p.k + b * FR, f0, FR, f1);
            const float ts = ((const float *)p.t)[b], te = ((const float *)st.t_end)[b], a_dt = ((const float *)st.a_dt)[b];
            mlp_start_scale(cp, f0, FR, sf, y, k0, inv, a0, a1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = ((f1[r] - k0[r]) * inv[r]) / sf;
                a2[r] = x * x;
            }
            mlp_sum2(sh, slot, a0, a1, A0, A1);
            mlp_sum2(sh, slot, a2, none, A2, unused);
            const float d0 = sqrt_(A0), d1 = sqrt_(A1), r2 = sqrt_(A2), dir = te > ts ? 1.0f : -1.0f, span = abs_(te - ts);
            bool small;
            float h0a;
            const float h0 = mlp_start_probe_step(d0, d1, span, small, h0a), dh = dir * h0;
            const bool blocked = integral && h0 == 0.0f;  // (the integral controller's copy of the rule: d2 = inf)
            const float d2 = blocked ? __builtin_huge_valf() : r2 / h0, m = tmax(d1, d2);
            const bool tiny = m <= 1e-15f;
            const float rm = 1.0f / m, z = rm * 0.01f;
            const float h1 = tiny ? tmax(1e-6f, h0 * 1e-3f) : rpow<float>(z, 1.0 / 5.0);
            const float first = dir * tmin(100.0f * h0, h1), lo = tmin(ts, te) - ts, hi = tmax(te, ts) - ts;
            // ---- reversed ----
            const bool on = a_dt != 0.0f;
            const float g_min = (on && first >= lo && first <= hi) ? a_dt * dir : 0.0f;
            float g_h0 = 100.0f * (g_min * share_of_min(100.0f * h0, h1)), g_d1 = 0, g_d2 = 0;
            const float g_h1 = g_min * share_of_min(h1, 100.0f * h0);
            if (on && tiny) g_h0 += (h0 * 1e-3f >= 1e-6f) ? g_h1 * 1e-3f : 0.0f;
            if (on && !tiny) {
                const float g_z = g_h1 * (0.2f * rpow<float>(z, 1.0 / 5.0 - 1.0)), g_m = -(g_z * 0.01f) * rm * rm;
                g_d1 = g_m * share_of_max(d1, d2), g_d2 = g_m * share_of_max(d2, d1);
            }
            const bool probe = on && !blocked && g_d2 != 0.0f;
            float g_inv[4], g_f1[4], g_step[4];
            const float g_r2 = probe ? g_d2 / h0 : 0.0f;
            if (probe) g_h0 += -g_d2 * r2 / (h0 * h0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float diff = f1[r] - k0[r], g_w = (probe && r2 != 0.0f) ? (g_r2 * (((diff * inv[r]) / sf) / r2)) / sf : 0.0f;
                g_f1[r] = probe ? g_w * inv[r] : 0.0f;
                g_inv[r] = probe ? g_w * diff : 0.0f;
                g_k0[r] -= g_f1[r];
            }
            product(1, g_f1);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                g_y0[r] += probe ? gi[r] : 0.0f;
                g_k0[r] += probe ? gi[r] * dh : 0.0f;
                g_step[r] = probe ? gi[r] * k0[r] : 0.0f;
            }
            g_step[0] += probe ? gt : 0.0f;  // (the probe's time moves with its step as well)
            float steps;
            mlp_sum2(sh, slot, g_step, none, steps, unused);
            g_h0 += steps * dir;
            const float g_h0a = on ? g_h0 * share_of_min(h0a, span) : 0.0f;
            float g_d0 = 0;
            if (on && !small) {
                g_d1 += -g_h0a * (0.01f * d0) / (d1 * d1);
                g_d0 = 0.01f * (g_h0a / d1);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float g_u = (on && !small && d0 != 0.0f) ? (g_d0 * (((y[r] * inv[r]) / sf) / d0)) / sf : 0.0f;
                const float g_v = (on && d1 != 0.0f) ? (g_d1 * (((k0[r] * inv[r]) / sf) / d1)) / sf : 0.0f;
                g_y0[r] += on ? g_u * inv[r] : 0.0f;
                g_k0[r] += on ? g_v * inv[r] : 0.0f;
                g_inv[r] += on ? g_u * y[r] + g_v * k0[r] : 0.0f;
                const float sign = y[r] > 0.0f ? 1.0f : (y[r] < 0.0f ? -1.0f : 0.0f);
                g_y0[r] += on ? (-g_inv[r] * inv[r] * inv[r]) * cp.rtol * sign : 0.0f;
            }
        }
        product(0, g_k0);
#pragma unroll
        for (int r = 0; r < 4; ++r) g_y0[r] += gi[r];
        if (st.grad_ys && ((const float *)st.t_eval)[b * st.n_eval] == ((const float *)p.t)[b]) {
            const float *first = (const float *)st.grad_ys + b * st.n_eval * FR;
#pragma unroll
            for (int r = 0; r < 4; ++r) g_y0[r] += f0 + r < FR ? first[f0 + r] : 0.0f;
        }
        if (live) mlp_put((float *)p.g_y + b * FR, f0, FR, g_y0);
    }
}

// Ahead of a sweep (tode_mlp_sweep_begin): a point's iteration by binary search over its sample's recorded times, one thread per
// point; a sample's move and its dense times by further uses of the same threads.  A few microseconds, where the same in torch
// operations took fifteen launches.
__global__ void __launch_bounds__(256) mlp_sweep_begin_kernel(long long B, int E, long long L, const float *t_start, long long ts_stride, const float *t_end, long long te_stride,
                                                              const float *t_eval, const float *rec_t, const int32_t *rec_n_accepted, int32_t *hit_iteration, int32_t *moved,
                                                              float *t_start_out, float *t_end_out) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < B) t_start_out[i] = t_start[i * ts_stride], t_end_out[i] = t_end[i * te_stride];
    if (i < L * B) moved[i] = rec_n_accepted[i + B] > rec_n_accepted[i] ? 1 : 0;
    if (i >= B * E) return;
    const long long b = i / E;
    const float ts = t_start[b * ts_stride], dir = t_end[b * te_stride] > ts ? 1.0f : -1.0f, at = t_eval[i], v = dir * at;
    long long lo = 0, hi = L;
    while (lo < hi) {
        const long long mid = (lo + hi) / 2;
        if (dir * rec_t[(mid + 1) * B + b] >= v) hi = mid;
        else lo = mid + 1;
    }
    hit_iteration[i] = lo < L && !(i == b * E && at == ts) ? (int32_t)lo : -1;
}

// The operands of four rows (k of the matrix instructions) for one wavefront: lane (q, c) holds row 4 step + q, and of it the
// hidden units 64w + 4c + u and the features 4c + i (which of them is which row or column of a tile is free, and four
// neighbours are one load).  Rows past the end repeat the last one with cotangents of zero.
constexpr int MLP_OUTER_AHEAD = 4;
struct MlpOuterRows {
    float h[4], d[4], g[4], x[4], t;
};

// The lane's four features of a row, without a branch; those past the problem's repeat the first ones (their sums go nowhere).
// QUADS: rows are whole groups of four.
template <bool QUADS> __device__ __forceinline__ void mlp_outer_get(const float *row, int f0, int FR, float (&v)[4]) {
    if (QUADS) {
        const float4 u = *reinterpret_cast<const float4 *>(row + (f0 < FR ? f0 : 0));
        v[0] = u.x, v[1] = u.y, v[2] = u.z, v[3] = u.w;
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = row[f0 + r < FR ? f0 + r : 0];
    }
}

// The rows row .. row + 3 (the same for the whole wavefront) of a share that ends at `end`; those past it repeat the last one.
// (Nothing is done to the values here: that would be the place where their loads are waited for.)
template <bool QUADS> __device__ __forceinline__ void mlp_outer_rows(const tode_mlp_reverse &p, long long row, long long end, int w, int q, int c, MlpOuterRows &v) {
    const long long from = min(row, end - 1);
    const int at = min(q, (int)min(end - 1 - from, 3ll)), FR = p.n_features;
    const float4 h = *reinterpret_cast<const float4 *>((const float *)p.hidden + from * MLP_H + (at * MLP_H + 64 * w + 4 * c));
    const float4 d = *reinterpret_cast<const float4 *>((const float *)p.hidden_cotangents + from * MLP_H + (at * MLP_H + 64 * w + 4 * c));
    v.h[0] = h.x, v.h[1] = h.y, v.h[2] = h.z, v.h[3] = h.w;
    v.d[0] = d.x, v.d[1] = d.y, v.d[2] = d.z, v.d[3] = d.w;
    mlp_outer_get<QUADS>((const float *)p.stage_cotangents + from * FR + at * FR, 4 * c, FR, v.g);
    mlp_outer_get<QUADS>((const float *)p.stage_inputs + from * FR + at * FR, 4 * c, FR, v.x);
    v.t = ((const float *)p.stage_times + from)[at];
}

// dW2[f][u] = sum over rows g[f] h[u],  dW1[u][i] = sum over rows d[u] x[i],  and the biases' and the time column's sums:
// every workgroup takes a share of the rows and holds all sums of it in registers (wavefront w: units 64w .. 64w + 63, 128
// accumulators), 32 matrix instructions (0.43 us at 2.4 GHz) per four rows with the operands of the next four such steps on their way:
// one wavefront per SIMD has nothing else to cover the memory's latency with.  82 000 rows: 69 us, of which the matrix
// instructions are 34; 92 with a load per value, half of whose instructions were addresses.  The sums of a share go to the workgroup's
// own slot, added to those of earlier calls (`accumulate`).
template <bool QUADS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) mlp_weight_gradient_kernel(const tode_mlp_reverse p, long long rows, long long rows_per_split, int accumulate) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15;
    const long long first = (long long)blockIdx.x * rows_per_split, end = min(rows, first + rows_per_split);
    mfma_acc a2[4][4], a1[4][4];
    float at[4], ab[4], ag[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        at[i] = ab[i] = ag[i] = 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) a2[i][u] = {0.0f, 0.0f, 0.0f, 0.0f}, a1[i][u] = {0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (first < end) {
        MlpOuterRows ring[MLP_OUTER_AHEAD];
#pragma unroll
        for (int n = 0; n < MLP_OUTER_AHEAD; ++n) mlp_outer_rows<QUADS>(p, first + 4 * n, end, w, q, c, ring[n]);
        for (long long row = first; row < end; row += 4 * MLP_OUTER_AHEAD) {
#pragma unroll
            for (int n = 0; n < MLP_OUTER_AHEAD; ++n) {
                MlpOuterRows here = ring[n];
                if (row + 4 * n + 4 > end) {  // (the share's last rows: cotangents of zero for those past its end)
                    const bool in = row + 4 * n + q < end;
#pragma unroll
                    for (int u = 0; u < 4; ++u) here.d[u] = in ? here.d[u] : 0.0f, here.g[u] = in ? here.g[u] : 0.0f;
                }
                mlp_outer_rows<QUADS>(p, row + 4 * (MLP_OUTER_AHEAD + n), end, w, q, c, ring[n]);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        a2[i][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(here.g[i], here.h[u], a2[i][u], 0, 0, 0);
                        a1[i][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(here.x[i], here.d[u], a1[i][u], 0, 0, 0);
                    }
                    at[u] = fma_(here.t, here.d[u], at[u]);
                    ab[u] += here.d[u];
                    ag[u] += here.g[u];
                }
            }
        }
    }
    float *out = (float *)p.sums + (long long)blockIdx.x * MLP_SUMS;
    auto put = [&](int i, float v) { out[i] = accumulate ? out[i] + v : v; };
    auto put_four = [&](int i, float a, float b, float c, float d) {
        float4 *to = reinterpret_cast<float4 *>(out + i);
        float4 v = make_float4(a, b, c, d);
        if (accumulate) {
            const float4 before = *to;
            v = make_float4(before.x + a, before.y + b, before.z + c, before.w + d);
        }
        *to = v;
    };
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int feature = 4 * (4 * q + r) + i;
            put_four(feature * MLP_H + 64 * w + 4 * c, a1[i][0][r], a1[i][1][r], a1[i][2][r], a1[i][3][r]);
            put_four(MLP_SUM_W2 + feature * MLP_H + 64 * w + 4 * c, a2[i][0][r], a2[i][1][r], a2[i][2][r], a2[i][3][r]);
        }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int unit = 64 * w + 4 * c + u;
#pragma unroll
        for (int off = 16; off < 64; off <<= 1) at[u] += __shfl_xor(at[u], off), ab[u] += __shfl_xor(ab[u], off), ag[u] += __shfl_xor(ag[u], off);
        if (q == 0) {
            put(MLP_SUM_W1T + unit, at[u]);
            put(MLP_SUM_B1 + unit, ab[u]);
            if (w == 0) put(MLP_SUM_B2 + 4 * c + u, ag[u]);
        }
    }
}

// The splits of 64 sums per workgroup, a quarter of the splits per wavefront with 32 loads in flight (one thread per sum over
// all splits waited for memory 64 times in a row: 68 us for 34 MB; eight loads in flight: 20 us); always in the same order.  out in the order of
// the weights: W1 [H x (F + 1)] | b1 | W2 [F x H] | b2.
static __global__ void __launch_bounds__(256) mlp_weight_gradient_sum_kernel(const float *sums, int splits, int H, int FR, float *out) {
    __shared__ float part[4][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, i = blockIdx.x * 64 + lane;
    const int share = (splits + 3) / 4, first = w * share, end = min(splits, first + share);
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    if (i < MLP_SUMS) {
        for (int k = first; k < end; k += 32) {
            float v[32];
#pragma unroll
            for (int j = 0; j < 32; ++j) v[j] = k + j < end ? sums[(long long)(k + j) * MLP_SUMS + i] : 0.0f;
#pragma unroll
            for (int j = 0; j < 32; ++j) s[j % 8] += v[j];
        }
    }
    part[w][lane] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    if (w != 0 || i >= MLP_SUMS) return;
    const long long o_b1 = (long long)H * (FR + 1), o_w2 = o_b1 + H, o_b2 = o_w2 + (long long)FR * H;
    long long to = -1;
    const int row = i / MLP_H, unit = i % MLP_H;  // (of the first part; the others start at multiples of MLP_H as well)
    if (i < MLP_SUM_W1T) to = (unit < H && row < FR) ? (long long)unit * (FR + 1) + row : -1;
    else if (i < MLP_SUM_B1) to = unit < H ? (long long)unit * (FR + 1) + FR : -1;
    else if (i < MLP_SUM_W2) to = unit < H ? o_b1 + unit : -1;
    else if (i < MLP_SUM_B2) to = (unit < H && row - MLP_F - 2 < FR) ? o_w2 + (long long)(row - MLP_F - 2) * H + unit : -1;
    else to = i - MLP_SUM_B2 < FR ? o_b2 + (i - MLP_SUM_B2) : -1;
    if (to >= 0) out[to] = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
}

static int check_mlp_reverse(const tode_mlp_reverse *p) {
    if (!p) return fail(TODE_E_INVALID, "null tode_mlp_reverse");
    if (p->method != TODE_DOPRI5 && p->method != TODE_TSIT5) return fail(TODE_E_INVALID, "unknown method %d", p->method);
    if (p->n_features < 1 || p->n_features > MLP_F || p->n_hidden < 1 || p->n_hidden > MLP_H)
        return fail(TODE_E_UNSUPPORTED, "the network's kernels take 1 to %d features and 1 to %d hidden units, got %d and %d", MLP_F, MLP_H, p->n_features, p->n_hidden);
    if (p->batch < 0 || p->batch > (1ll << 40)) return fail(TODE_E_INVALID, "batch %lld", (long long)p->batch);
    if (p->stage_rows != 0 && p->stage_rows < p->batch) return fail(TODE_E_INVALID, "stage_rows %lld for a batch of %lld", (long long)p->stage_rows, (long long)p->batch);
    if (p->splits < 1 || p->splits > TODE_MLP_MAX_SPLITS) return fail(TODE_E_INVALID, "splits %d", p->splits);
    if (p->batch > 0 && (!p->packed || !p->packed_reverse || !p->t || !p->dt || !p->y || !p->k0 || !p->k || !p->stage_inputs || !p->stage_times || !p->hidden ||
                         !p->g_k || !p->g_y || !p->g_y1 || !p->g_t || !p->g_dt))
        return fail(TODE_E_INVALID, "null pointer");
    if (!p->hidden_cotangents != !p->sums || !p->stage_cotangents != !p->sums) return fail(TODE_E_INVALID, "hidden_cotangents, stage_cotangents and sums go together");
    return TODE_OK;
}

// A workgroup of the reverse kernel fills its compute unit (one wavefront per SIMD), of the stages' kernel half of one:
// beyond that they take several tiles each and load the weights once (133 KB per workgroup, as long as a stage takes).
static unsigned mlp_tiles_grid(const tode_mlp_reverse &p, int per_unit) {
    const long long tiles = (p.batch + MLP_TILE - 1) / MLP_TILE;
    return (unsigned)(tiles < 256ll * per_unit ? tiles : 256ll * per_unit);
}

static int launch_stages(const tode_mlp_reverse &p, float atol, float rtol, float *error_sums, hipStream_t stream) {
    const dim3 grid(mlp_tiles_grid(p, 2));
    if (p.method == TODE_TSIT5) hipLaunchKernelGGL((mlp_stages_kernel<1>), grid, dim3(256), 0, stream, p, atol, rtol, error_sums);
    else hipLaunchKernelGGL((mlp_stages_kernel<0>), grid, dim3(256), 0, stream, p, atol, rtol, error_sums);
    return check_hip(hipGetLastError(), "tode_mlp_stages");
}

}  // namespace tode

extern "C" {

int tode_mlp_pack_weights_reverse(const void *raw, int64_t n_raw, int32_t n_features, void *packed, void *stream) {
    using namespace tode;
    static_assert(TODE_MLP_REVERSE_PACKED_SIZE == MLP_REVERSE_REGS * 256 && TODE_MLP_SUMS_SIZE == MLP_SUMS, "sizes");
    if (!raw || !packed) return fail(TODE_E_INVALID, "null pointer");
    const long long FR = n_features;
    if (FR < 1 || FR > MLP_F) return fail(TODE_E_UNSUPPORTED, "the network's kernels take 1 to %d features, got %lld", MLP_F, FR);
    const long long H = (n_raw - FR) / (2 * FR + 2);
    if (n_raw < FR || H * (2 * FR + 2) + FR != n_raw || H < 1 || H > MLP_H) return fail(TODE_E_UNSUPPORTED, "%lld weights do not make a network of up to %d hidden units", (long long)n_raw, MLP_H);
    hipLaunchKernelGGL(mlp_pack_reverse_kernel, dim3(MLP_REVERSE_REGS), dim3(256), 0, (hipStream_t)stream, (const float *)raw, (float *)packed, (int)H, (int)FR);
    return check_hip(hipGetLastError(), "tode_mlp_pack_weights_reverse");
}

int tode_mlp_pack_weights_both(const void *W1, const void *b1, const void *W2, const void *b2, int32_t n_hidden, int32_t n_features, void *packed, void *stream) {
    using namespace tode;
    static_assert(TODE_MLP_PACKED_SIZE == MLP_REGS * 256, "sizes");
    if (!W1 || !b1 || !W2 || !b2 || !packed) return fail(TODE_E_INVALID, "null pointer");
    if (n_features < 1 || n_features > MLP_F || n_hidden < 1 || n_hidden > MLP_H)
        return fail(TODE_E_UNSUPPORTED, "the network's kernels take 1 to %d features and 1 to %d hidden units, got %d and %d", MLP_F, MLP_H, n_features, n_hidden);
    hipLaunchKernelGGL(mlp_pack_both_kernel, dim3(MLP_REGS + MLP_REVERSE_REGS), dim3(256), 0, (hipStream_t)stream, (const float *)W1, (const float *)b1, (const float *)W2, (const float *)b2,
                       (float *)packed, n_hidden, n_features);
    return check_hip(hipGetLastError(), "tode_mlp_pack_weights_both");
}

int tode_mlp_stages(const tode_mlp_reverse *p, void *stream) {
    using namespace tode;
    const int rc = check_mlp_reverse(p);
    if (rc || p->batch == 0) return rc;
    return launch_stages(*p, 0, 0, nullptr, (hipStream_t)stream);
}

int tode_mlp_stages_backward(const tode_mlp_reverse *p, void *stream) {
    using namespace tode;
    const int rc = check_mlp_reverse(p);
    if (rc || p->batch == 0) return rc;
    const dim3 grid(mlp_tiles_grid(*p, 1));
    if (p->method == TODE_TSIT5) hipLaunchKernelGGL((mlp_stages_backward_kernel<1>), grid, dim3(256), 0, (hipStream_t)stream, *p);
    else hipLaunchKernelGGL((mlp_stages_backward_kernel<0>), grid, dim3(256), 0, (hipStream_t)stream, *p);
    return check_hip(hipGetLastError(), "tode_mlp_stages_backward");
}

int tode_mlp_start_backward(const tode_mlp_reverse *p, const tode_mlp_start *start, const tode_controller *c, void *stream) {
    using namespace tode;
    const int rc = check_mlp_reverse(p);
    if (rc || p->batch == 0) return rc;
    if (!start || !c || !start->t_end || !start->a_y || !start->a_k0 || !start->a_dt) return fail(TODE_E_INVALID, "null pointer");
    if (start->grad_ys && (!start->t_eval || start->n_eval < 1)) return fail(TODE_E_INVALID, "grad_ys without evaluation points");
    if (c->kind != TODE_CTRL_INTEGRAL && c->kind != TODE_CTRL_PID) return fail(TODE_E_INVALID, "unknown controller kind %d", c->kind);
    const CtrlParams<float> cp = make_ctrl<float>(*c);
    const bool integral = c->kind == TODE_CTRL_INTEGRAL;
    const dim3 grid(mlp_tiles_grid(*p, 2)), grid_back(mlp_tiles_grid(*p, 1));
    hipStream_t s = (hipStream_t)stream;
    if (start->through_rule) {
        hipLaunchKernelGGL((mlp_start_kernel<true>), grid, dim3(256), 0, s, *p, *start, cp);
        hipLaunchKernelGGL((mlp_start_backward_kernel<true>), grid_back, dim3(256), 0, s, *p, *start, cp, integral);
    } else {
        hipLaunchKernelGGL((mlp_start_kernel<false>), grid, dim3(256), 0, s, *p, *start, cp);
        hipLaunchKernelGGL((mlp_start_backward_kernel<false>), grid_back, dim3(256), 0, s, *p, *start, cp, integral);
    }
    return check_hip(hipGetLastError(), "tode_mlp_start_backward");
}

int tode_mlp_sweep_begin(int64_t batch, int32_t n_eval, int64_t iterations, const void *t_start, int64_t t_start_stride, const void *t_end, int64_t t_end_stride,
                         const void *t_eval, const void *rec_t, const int32_t *rec_n_accepted, int32_t *hit_iteration, int32_t *moved, void *t_start_out, void *t_end_out,
                         void *stream) {
    using namespace tode;
    if (batch < 0 || n_eval < 1 || iterations < 0 || t_start_stride < 1 || t_end_stride < 1) return fail(TODE_E_INVALID, "bad sizes");
    if (batch == 0) return TODE_OK;
    if (!t_start || !t_end || !t_eval || !rec_t || !rec_n_accepted || !hit_iteration || (iterations > 0 && !moved) || !t_start_out || !t_end_out) return fail(TODE_E_INVALID, "null pointer");
    const long long threads = batch * (n_eval > iterations ? n_eval : iterations);
    if ((threads + 255) / 256 > 2147483647) return fail(TODE_E_UNSUPPORTED, "batch too large");
    hipLaunchKernelGGL(mlp_sweep_begin_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (long long)batch, n_eval, (long long)iterations,
                       (const float *)t_start, (long long)t_start_stride, (const float *)t_end, (long long)t_end_stride, (const float *)t_eval, (const float *)rec_t, rec_n_accepted,
                       hit_iteration, moved, (float *)t_start_out, (float *)t_end_out);
    return check_hip(hipGetLastError(), "tode_mlp_sweep_begin");
}

int tode_mlp_outer_products(const tode_mlp_reverse *p, int64_t rows, int32_t accumulate, void *stream) {
    using namespace tode;
    const int rc = check_mlp_reverse(p);
    if (rc || p->batch == 0) return rc;
    if (!p->sums) return fail(TODE_E_INVALID, "null pointer");
    if (rows < 0) return fail(TODE_E_INVALID, "rows %lld", (long long)rows);
    const long long per_split = ((rows + p->splits - 1) / p->splits + 3) / 4 * 4;
    // (rows of the features as 16-byte values, as everywhere in these kernels, where they are whole groups of four)
    if ((p->n_features & 3) == 0) hipLaunchKernelGGL((mlp_weight_gradient_kernel<true>), dim3(p->splits), dim3(256), 0, (hipStream_t)stream, *p, (long long)rows, per_split, accumulate);
    else hipLaunchKernelGGL((mlp_weight_gradient_kernel<false>), dim3(p->splits), dim3(256), 0, (hipStream_t)stream, *p, (long long)rows, per_split, accumulate);
    return check_hip(hipGetLastError(), "tode_mlp_outer_products");
}

int tode_mlp_sweep_record(const tode_mlp_reverse *p, const tode_mlp_sweep *s, const tode_controller *c, void *stream) {
    using namespace tode;
    if (!p || !s || !c) return fail(TODE_E_INVALID, "null argument");
    tode_mlp_reverse q = *p;
    q.batch = p->batch * s->iterations, q.stage_rows = 0;
    q.t = s->record.t, q.dt = s->record.dt, q.y = s->record.y, q.k0 = s->record.k0;
    q.g_k = q.g_y1 = q.g_t = q.g_dt = p->g_y;  // (not used by the stages; the sweep keeps them in registers)
    int rc = check_mlp_reverse(&q);
    if (rc) return rc;
    if (s->iterations < 1 || s->record.capacity < s->iterations + 1) return fail(TODE_E_INVALID, "%lld iterations, a record of %lld entries", (long long)s->iterations, (long long)s->record.capacity);
    if (s->n_eval < 1) return fail(TODE_E_INVALID, "n_eval=%d", s->n_eval);
    if (q.batch > (1ll << 38)) return fail(TODE_E_UNSUPPORTED, "batch too large");
    if (s->t_start_stride < 1 || s->t_end_stride < 1) return fail(TODE_E_INVALID, "t_start_stride / t_end_stride must be >= 1");
    if (c->kind != TODE_CTRL_INTEGRAL && c->kind != TODE_CTRL_PID) return fail(TODE_E_INVALID, "unknown controller kind %d", c->kind);
    if (c->has_dt_min || c->has_dt_max) return fail(TODE_E_UNSUPPORTED, "limits of the step size");
    if (p->batch == 0) return TODE_OK;
    const tode_solve_record &r = s->record;
    if (!r.t || !r.dt || !r.y || !r.k0 || !r.prev || !r.pprev || !r.running || !r.n_accepted || !s->t_start || !s->t_end || !s->t_eval || !s->grad_ys || !s->a_y || !s->a_k0 || !s->a_dt ||
        !s->t_end_dense || !s->control || !s->error_sums || !p->sums != !s->weight_gradients)
        return fail(TODE_E_INVALID, "null pointer");
    if ((p->n_features & 3) == 0 && ((uintptr_t)s->grad_ys & 15)) return fail(TODE_E_INVALID, "grad_ys is not aligned to 16 bytes");  // (as every array whose rows are read so)
    hipStream_t stream_ = (hipStream_t)stream;
    const CtrlParams<float> cp = make_ctrl<float>(*c);
    if ((rc = launch_stages(q, cp.atol, cp.rtol, (float *)s->error_sums, stream_))) return rc;
    const dim3 blocks((unsigned)((q.batch + 255) / 256));
    if (c->kind == TODE_CTRL_PID) hipLaunchKernelGGL((mlp_sweep_control_kernel<1>), blocks, dim3(256), 0, stream_, *s, (long long)p->batch, cp);
    else hipLaunchKernelGGL((mlp_sweep_control_kernel<0>), blocks, dim3(256), 0, stream_, *s, (long long)p->batch, cp);
    if ((rc = check_hip(hipGetLastError(), "tode_mlp_sweep_record launch"))) return rc;

    q.batch = p->batch;
    const dim3 grid(mlp_tiles_grid(q, 1));
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream_, q, *s, cp); };
    const bool pid = c->kind == TODE_CTRL_PID;
    if (p->method == TODE_TSIT5) pid ? launch(mlp_sweep_kernel<1, 1>) : launch(mlp_sweep_kernel<1, 0>);
    else pid ? launch(mlp_sweep_kernel<0, 1>) : launch(mlp_sweep_kernel<0, 0>);
    if ((rc = check_hip(hipGetLastError(), "tode_mlp_sweep_record launch"))) return rc;

    // the start of the loop: its evaluations' rows lie behind those of the iterations
    const long long rows = 6 * s->iterations * p->batch, FR = p->n_features;
    tode_mlp_reverse first = q;
    first.stage_inputs = (float *)p->stage_inputs + rows * FR, first.stage_times = (float *)p->stage_times + rows, first.hidden = (float *)p->hidden + rows * MLP_H;
    if (p->sums) first.stage_cotangents = (float *)p->stage_cotangents + rows * FR, first.hidden_cotangents = (float *)p->hidden_cotangents + rows * MLP_H;
    const tode_mlp_start start = {s->t_end_dense, s->a_y, s->a_k0, s->a_dt, s->through_rule, s->n_eval, s->grad_ys, s->t_eval};
    if ((rc = tode_mlp_start_backward(&first, &start, c, stream))) return rc;
    if (!p->sums) return TODE_OK;
    if ((rc = tode_mlp_outer_products(&q, rows + (s->through_rule ? 2 : 1) * p->batch, 0, stream))) return rc;
    return tode_mlp_weight_gradients(&q, s->weight_gradients, stream);
}

int tode_mlp_weight_gradients(const tode_mlp_reverse *p, void *out, void *stream) {
    using namespace tode;
    const int rc = check_mlp_reverse(p);
    if (rc) return rc;
    if (!p->sums || !out) return fail(TODE_E_INVALID, "null pointer");
    hipLaunchKernelGGL(mlp_weight_gradient_sum_kernel, dim3((MLP_SUMS + 63) / 64), dim3(256), 0, (hipStream_t)stream, (const float *)p->sums, p->splits, p->n_hidden,
                       p->n_features, (float *)out);
    return check_hip(hipGetLastError(), "tode_mlp_weight_gradients");
}

}  // extern "C"
