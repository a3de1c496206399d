// Two-layer perceptron on the matrix cores: the tile of 16 samples, the order of the weights in registers, the evaluation of
// f and the per-sample sums, shared by the whole-solve kernel (tode_mlp.hip, which describes the layout) and the
// reverse sweep's kernels (tode_mlp_reverse.hip).
#pragma once
#include "tode_solve.h"

namespace tode {

typedef float mfma_acc __attribute__((ext_vector_type(4)));

struct MlpOut {
    int64_t *n_steps, *n_accepted, *n_initialized, *status;
    int n_features;  // features of the problem: at most 64 (the kernel's others stay zero)
};

constexpr int MLP_F = 64, MLP_H = 256, MLP_TILE = 16;
// LDS row of the stage input: 64 features, t, zeros up to column 79; padded to 100 values = 4 banks past a multiple of
// 32, so that the 16-byte reads and writes of eight lanes that differ in their sample fall on 32 different banks
constexpr int MLP_XS = 100;
constexpr int MLP_REGS = 68 + 16 + 64 + 4;       // packed values per thread: W1, b1, W2, b2
constexpr int MLP_REGS_BF16 = 40 + 16 + 32 + 4;  // the same with W1 (80 inputs) and W2 as pairs of bfloat16

struct __align__(16) MlpShared {
    float x[MLP_TILE * MLP_XS];
    float part[4][4][64][4];        // [output tile][wavefront it comes from][lane][4 features]
    float red[2][4][MLP_TILE][2];   // per-wavefront partial sums of up to two per-sample reductions
    int vote[2][4];                 // per-wavefront bits of the workgroup-wide "or"
    float b1[MLP_H], b2[MLP_F];     // (bfloat16 variant) the biases
};

struct MlpWeights {
    float w1[17][4];    // W1[64w + 16 tile + c][input of (kk, q)]
    float b1[4][4];     // b1[64w + 16 tile + 4q + r]
    float w2[4][4][4];  // W2[16 ft + c][64w + 16 tile + 4q + r]
    float b2[4];        // b2[16w + 4q + r]
};

// The variant with bfloat16 inputs to the matrix cores (v_mfma_f32_16x16x16_bf16: 16 k per
// instruction, a lane supplies k = 4q..4q+3): float32 accumulation, biases, tanh and solver state.
typedef __bf16 mlp_bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned mlp_u32x2 __attribute__((ext_vector_type(2)));

// Four values rounded to nearest even, two by one instruction.  Put together as words: a vector of four bfloat16 that goes to a
// matrix instruction the compiler makes of four conversions and two permutations.
typedef __bf16 mlp_bf16x2 __attribute__((ext_vector_type(2)));
typedef float mlp_f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned mlp_round(float a, float b) { return __builtin_bit_cast(unsigned, __builtin_convertvector(mlp_f32x2{a, b}, mlp_bf16x2)); }
__device__ __forceinline__ mlp_bf16x4 mlp_round(float a, float b, float c, float d) { return __builtin_bit_cast(mlp_bf16x4, mlp_u32x2{mlp_round(a, b), mlp_round(c, d)}); }

struct MlpWeightsBf16 {
    mlp_bf16x4 w1[5][4];  // W1[64w + 16 tile + c][16 ks + 4q + j], inputs 65..79 are zero
    mlp_bf16x4 w2[4][4];  // [ft][tile]: W2[16 ft + c][64w + 16 tile + 4q + j]
};

// Which input column lane group q feeds at k-step kk of the first layer: 16 features each for
// the first 16 steps (contiguous in LDS), then t and three zero columns.
__host__ __device__ __forceinline__ int mlp_input_of(int kk, int q) { return kk < 16 ? 16 * q + kk : 64 + q; }

// Source index (in W1 | b1 | W2 | b2, row-major) of packed value j of thread tid, or -1 for zero.  H: hidden units of
// the network at hand, at most MLP_H; the kernel's units from H on get zero weights and a zero bias, so that they
// add tanh(0) * 0 = 0 to every sum in the same places as before (a narrower network in the same arithmetic).
// FR: features of the network at hand (at most MLP_F): W1 is [H x (FR + 1)] with the time in its last
// column, W2 [FR x H]; the kernel's features from FR on get zero weights on both sides and stay zero throughout.
__host__ __device__ inline long long mlp_packed_source(int j, int tid, int H, int FR) {
    const int lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15;
    const long long o_b1 = (long long)H * (FR + 1), o_w2 = o_b1 + H, o_b2 = o_w2 + (long long)FR * H;
    // column of W1 for the kernel's input k (features 0..63, then the time at 64), or -1
    auto w1_column = [&](int k) { return k < FR ? k : (k == MLP_F ? FR : -1); };
    if (j < 68) {
        const int kk = j / 4, tile = j % 4, col = w1_column(mlp_input_of(kk, q)), unit = 64 * w + 16 * tile + c;
        return (col >= 0 && unit < H) ? (long long)unit * (FR + 1) + col : -1;
    }
    j -= 68;
    if (j < 16) {
        const int unit = 64 * w + 16 * (j / 4) + 4 * q + (j % 4);
        return unit < H ? o_b1 + unit : -1;
    }
    j -= 16;
    if (j < 64) {
        const int ft = j / 16, tile = (j / 4) % 4, r = j % 4, unit = 64 * w + 16 * tile + 4 * q + r;
        return (unit < H && 16 * ft + c < FR) ? o_w2 + (long long)(16 * ft + c) * H + unit : -1;
    }
    j -= 64;
    return 16 * w + 4 * q + j < FR ? o_b2 + 16 * w + 4 * q + j : -1;
}

// The same for the bfloat16 variant: packed word j of thread tid holds the values of sources
// (lo, hi) as bfloat16 in its low and high half (words of b1 and b2: one float32, hi = -2).
__host__ __device__ inline void mlp_packed_source_bf16(int j, int tid, int H, int FR, long long &lo, long long &hi) {
    const int lane = tid & 63, w = tid >> 6, q = lane >> 4, c = lane & 15;
    const long long o_b1 = (long long)H * (FR + 1), o_w2 = o_b1 + H, o_b2 = o_w2 + (long long)FR * H;
    auto w1_column = [&](int k) { return k < FR ? k : (k == MLP_F ? FR : -1); };
    hi = -2;
    if (j < 40) {
        const int ks = j / 8, tile = (j / 2) % 4, k = 16 * ks + 4 * q + 2 * (j % 2), unit = 64 * w + 16 * tile + c;
        const long long row = (long long)unit * (FR + 1);
        lo = (w1_column(k) >= 0 && unit < H) ? row + w1_column(k) : -1;
        hi = (w1_column(k + 1) >= 0 && unit < H) ? row + w1_column(k + 1) : -1;
        return;
    }
    j -= 40;
    if (j < 16) {
        const int unit = 64 * w + 16 * (j / 4) + 4 * q + (j % 4);
        lo = unit < H ? o_b1 + unit : -1;
        hi = -3;  // (one float32 word, zero where lo < 0)
        return;
    }
    j -= 16;
    if (j < 32) {
        const int ft = j / 8, tile = (j / 2) % 4, unit = 64 * w + 16 * tile + 4 * q + 2 * (j % 2);
        const long long at = o_w2 + (long long)(16 * ft + c) * H + unit;
        lo = (unit < H && 16 * ft + c < FR) ? at : -1;
        hi = (unit + 1 < H && 16 * ft + c < FR) ? at + 1 : -1;
        return;
    }
    j -= 32;
    lo = 16 * w + 4 * q + j < FR ? o_b2 + 16 * w + 4 * q + j : -1;
}

// Bitwise "or" of `bits` over the workgroup (four wavefronts).  Consecutive calls alternate between
// two sets of LDS words, so a wavefront that runs ahead into the next call cannot overwrite what
// a slower one still has to read.
__device__ __forceinline__ int block_or(MlpShared &sh, int &vslot, int bits) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) bits |= __shfl_xor(bits, off);
    if (lane == 0) sh.vote[vslot][w] = bits;
    lds_barrier();
    const int all = (sh.vote[vslot][0] | sh.vote[vslot][1]) | (sh.vote[vslot][2] | sh.vote[vslot][3]);
    vslot ^= 1;
    return all;
}

// tanh(x) = 1 - 2 / (exp(2x) + 1) on the hardware exp2 and reciprocal: absolute error about 2e-7
// (the library tanhf costs several times the matrix products of a layer).  exp2 overflows to inf
// and underflows to 0 exactly where tanh saturates, so no range checks are needed.
__device__ __forceinline__ float mlp_tanh(float x) {
    const float e = __builtin_amdgcn_exp2f(x * 2.8853900817779268f);  // 2 / ln 2
    return fma_(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f);  // (2 r is exact)
}

// tanh(x) to an ulp and a half: up to 1 an odd polynomial of degree 15 (fitted to the smallest relative error, 5e-9), beyond it
// the form above; 0.31 ulp in the mean over normal arguments.  No branch, so that the compiler can place it between matrix
// instructions: the math library's tanhf branches on |x|, and each of its sixteen values of an evaluation stood by itself between
// the two products.
__device__ __forceinline__ float mlp_tanh_accurate(float x) {
    const float e = __builtin_amdgcn_exp2f(__builtin_fabsf(x) * 2.8853900817779268f);
    const float far = __builtin_copysignf(fma_(-2.0f, __builtin_amdgcn_rcpf(e + 1.0f), 1.0f), x);
    const float z = x * x;
    float p = -0x1.77dcb2p-12f;
    p = fma_(p, z, 0x1.2da4c0p-9f);
    p = fma_(p, z, -0x1.0460b0p-7f);
    p = fma_(p, z, 0x1.60098cp-6f);
    p = fma_(p, z, -0x1.b96222p-5f);
    p = fma_(p, z, 0x1.110be2p-3f);
    p = fma_(p, z, -0x1.55553cp-2f);
    const float near = fma_(x * z, p, x);
    return __builtin_fabsf(x) < 1.0f ? near : far;  // (not a number: e is, and far with it)
}

// One of sixteen groups of four matrix instructions with the VALUES instructions of a tanh spread between them: a wavefront
// issues in order, and a group's worth of tanh behind the fourth instruction leaves the matrix cores idle for most of it.
template <int VALUES> __device__ __forceinline__ void mlp_interleave() {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // matrix instruction
        __builtin_amdgcn_sched_group_barrier(0x2 | 0x400, (VALUES + 3) / 4, 0);  // vector instructions
    }
    __builtin_amdgcn_sched_barrier(0);
}

// out[r] = f(tn, yi)[16w + 4q + r] for the lane's sample.
// ACCURATE_TANH: for the gradient's kernels, whose f stands where torch's was.  hidden: where not null, the sample's row of 256
// hidden activations in memory.
// The order of the matrix instructions hides tanh behind them: layer 1 for two of the four tiles of hidden units, then for the
// other two while the first two go through tanh, then layer 2 over the first two while the other two do (each sum in the
// order of its inputs all the same).
template <bool ACCURATE_TANH = false>
__device__ __forceinline__ void mlp_rhs(MlpShared &sh, const MlpWeights &W, float tn, const float (&yi)[4], float (&out)[4], float *hidden = nullptr) {
    constexpr int TANH = ACCURATE_TANH ? 17 : 6;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, c = lane & 15;
    *reinterpret_cast<float4 *>(sh.x + c * MLP_XS + 16 * w + 4 * q) = make_float4(yi[0], yi[1], yi[2], yi[3]);
    if (w == 0 && q == 0) sh.x[c * MLP_XS + MLP_F] = tn;
    lds_barrier();
    // all B operands of the layer into registers first, so that the matrix cores never wait for LDS
    float a1[17];
    {
        const float4 *row = reinterpret_cast<const float4 *>(sh.x + c * MLP_XS + 16 * q);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float4 v = row[j];
            a1[4 * j] = v.x, a1[4 * j + 1] = v.y, a1[4 * j + 2] = v.z, a1[4 * j + 3] = v.w;
        }
        a1[16] = sh.x[c * MLP_XS + MLP_F + q];
    }
    asm volatile("" ::: "memory");
    const auto hidden_unit = [](float x) { return ACCURATE_TANH ? mlp_tanh_accurate(x) : mlp_tanh(x); };
    mfma_acc h[4], acc[4];
#pragma unroll
    for (int tile = 0; tile < 4; ++tile) h[tile] = {W.b1[tile][0], W.b1[tile][1], W.b1[tile][2], W.b1[tile][3]}, acc[tile] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < 17; ++kk) {
#pragma unroll
        for (int tile = 0; tile < 2; ++tile) h[tile] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w1[kk][tile], a1[kk], h[tile], 0, 0, 0);
    }
#pragma unroll
    for (int tile = 2; tile < 4; ++tile) h[tile] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w1[0][tile], a1[0], h[tile], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 8; ++n) {
#pragma unroll
        for (int kk = 1 + 2 * n; kk < 3 + 2 * n; ++kk)
#pragma unroll
            for (int tile = 2; tile < 4; ++tile) h[tile] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w1[kk][tile], a1[kk], h[tile], 0, 0, 0);
        float unit = hidden_unit(h[n / 4][n % 4]);
        if (n < 7) asm volatile("" : "+v"(unit), "+v"(a1[3 + 2 * n]), "+v"(a1[4 + 2 * n]));  // (the next group behind this value)
        h[n / 4][n % 4] = unit;
        mlp_interleave<TANH>();
    }
#pragma unroll
    for (int n = 0; n < 8; ++n) {
#pragma unroll
        for (int ft = 0; ft < 4; ++ft) acc[ft] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w2[ft][n / 4][n % 4], h[n / 4][n % 4], acc[ft], 0, 0, 0);
        h[2 + n / 4][n % 4] = hidden_unit(h[2 + n / 4][n % 4]);
        mlp_interleave<TANH>();
    }
    if (hidden) {
#pragma unroll
        for (int tile = 0; tile < 4; ++tile)
            *reinterpret_cast<float4 *>(hidden + 64 * w + 16 * tile + 4 * q) = make_float4(h[tile][0], h[tile][1], h[tile][2], h[tile][3]);
    }
#pragma unroll
    for (int n = 8; n < 16; ++n)
#pragma unroll
        for (int ft = 0; ft < 4; ++ft) acc[ft] = __builtin_amdgcn_mfma_f32_16x16x4f32(W.w2[ft][n / 4][n % 4], h[n / 4][n % 4], acc[ft], 0, 0, 0);
#pragma unroll
    for (int ft = 0; ft < 4; ++ft) *reinterpret_cast<float4 *>(sh.part[ft][w][lane]) = make_float4(acc[ft][0], acc[ft][1], acc[ft][2], acc[ft][3]);
    lds_barrier();
    float4 s[4];
#pragma unroll
    for (int from = 0; from < 4; ++from) s[from] = *reinterpret_cast<const float4 *>(sh.part[w][from][lane]);
    out[0] = ((s[0].x + s[1].x) + (s[2].x + s[3].x)) + W.b2[0];
    out[1] = ((s[0].y + s[1].y) + (s[2].y + s[3].y)) + W.b2[1];
    out[2] = ((s[0].z + s[1].z) + (s[2].z + s[3].z)) + W.b2[2];
    out[3] = ((s[0].w + s[1].w) + (s[2].w + s[3].w)) + W.b2[3];
}

__device__ __forceinline__ void mlp_rhs(MlpShared &sh, const MlpWeightsBf16 &W, float tn, const float (&yi)[4], float (&out)[4]) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, c = lane & 15;
    *reinterpret_cast<float4 *>(sh.x + c * MLP_XS + 16 * w + 4 * q) = make_float4(yi[0], yi[1], yi[2], yi[3]);
    if (w == 0 && q == 0) sh.x[c * MLP_XS + MLP_F] = tn;
    lds_barrier();
    mlp_bf16x4 a1[5];
    {
        const float *row = sh.x + c * MLP_XS + 4 * q;
#pragma unroll
        for (int ks = 0; ks < 5; ++ks) {
            const float4 v = *reinterpret_cast<const float4 *>(row + 16 * ks);
            a1[ks] = mlp_round(v.x, v.y, v.z, v.w);
        }
    }
    mfma_acc h[4];
#pragma unroll
    for (int tile = 0; tile < 4; ++tile) h[tile] = *reinterpret_cast<const mfma_acc *>(sh.b1 + 64 * w + 16 * tile + 4 * q);
    asm volatile("" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < 5; ++ks) {
#pragma unroll
        for (int tile = 0; tile < 4; ++tile) h[tile] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(W.w1[ks][tile], a1[ks], h[tile], 0, 0, 0);
    }
    mlp_bf16x4 hb[4];
#pragma unroll
    for (int tile = 0; tile < 4; ++tile)
        hb[tile] = mlp_round(mlp_tanh(h[tile][0]), mlp_tanh(h[tile][1]), mlp_tanh(h[tile][2]), mlp_tanh(h[tile][3]));
    mfma_acc acc[4];
#pragma unroll
    for (int ft = 0; ft < 4; ++ft) acc[ft] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int tile = 0; tile < 4; ++tile)
#pragma unroll
        for (int ft = 0; ft < 4; ++ft) acc[ft] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(W.w2[ft][tile], hb[tile], acc[ft], 0, 0, 0);
#pragma unroll
    for (int ft = 0; ft < 4; ++ft) *reinterpret_cast<float4 *>(sh.part[ft][w][lane]) = make_float4(acc[ft][0], acc[ft][1], acc[ft][2], acc[ft][3]);
    lds_barrier();
    float4 s[4];
#pragma unroll
    for (int from = 0; from < 4; ++from) s[from] = *reinterpret_cast<const float4 *>(sh.part[w][from][lane]);
    const float4 b2 = *reinterpret_cast<const float4 *>(sh.b2 + 16 * w + 4 * q);
    out[0] = ((s[0].x + s[1].x) + (s[2].x + s[3].x)) + b2.x;
    out[1] = ((s[0].y + s[1].y) + (s[2].y + s[3].y)) + b2.y;
    out[2] = ((s[0].z + s[1].z) + (s[2].z + s[3].z)) + b2.z;
    out[3] = ((s[0].w + s[1].w) + (s[2].w + s[3].w)) + b2.w;
}

// Packed weights (tode_mlp_pack_weights) into the registers of thread tid.
__device__ __forceinline__ void mlp_load(MlpWeights &W, const float *packed, int tid) {
    const float4 *src = reinterpret_cast<const float4 *>(packed) + tid;
    float v[MLP_REGS];
#pragma unroll
    for (int i = 0; i < MLP_REGS / 4; ++i) {
        const float4 u = src[i * 256];
        v[4 * i] = u.x, v[4 * i + 1] = u.y, v[4 * i + 2] = u.z, v[4 * i + 3] = u.w;
    }
#pragma unroll
    for (int j = 0; j < 68; ++j) W.w1[j / 4][j % 4] = v[j];
#pragma unroll
    for (int j = 0; j < 16; ++j) W.b1[j / 4][j % 4] = v[68 + j];
#pragma unroll
    for (int j = 0; j < 64; ++j) W.w2[j / 16][(j / 4) % 4][j % 4] = v[84 + j];
#pragma unroll
    for (int j = 0; j < 4; ++j) W.b2[j] = v[148 + j];
}

__device__ __forceinline__ void mlp_load(MlpWeightsBf16 &W, const float *packed, int tid) {
    const uint4 *src = reinterpret_cast<const uint4 *>(packed) + tid;
#pragma unroll
    for (int i = 0; i < 10; ++i) {
        const uint4 u = src[i * 256];
        W.w1[i / 2][2 * (i % 2)] = __builtin_bit_cast(mlp_bf16x4, (mlp_u32x2){u.x, u.y});
        W.w1[i / 2][2 * (i % 2) + 1] = __builtin_bit_cast(mlp_bf16x4, (mlp_u32x2){u.z, u.w});
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint4 u = src[(14 + i) * 256];
        W.w2[i / 2][2 * (i % 2)] = __builtin_bit_cast(mlp_bf16x4, (mlp_u32x2){u.x, u.y});
        W.w2[i / 2][2 * (i % 2) + 1] = __builtin_bit_cast(mlp_bf16x4, (mlp_u32x2){u.z, u.w});
    }
}

// The bfloat16 variant's biases to LDS: b1[64w + 16 tile + 4q ..] from one lane of the sixteen that hold it, b2[16w + 4q ..] likewise.
__device__ __forceinline__ void mlp_load_biases(MlpShared &sh, const float *packed, int tid) {
    const int lane = tid & 63, w = tid >> 6, q = lane >> 4;
    if ((lane & 15) != 0) return;
    const float4 *src = reinterpret_cast<const float4 *>(packed) + tid;
#pragma unroll
    for (int tile = 0; tile < 4; ++tile) *reinterpret_cast<float4 *>(sh.b1 + 64 * w + 16 * tile + 4 * q) = src[(10 + tile) * 256];
    *reinterpret_cast<float4 *>(sh.b2 + 16 * w + 4 * q) = src[22 * 256];
}

// Per-sample sums over the 64 features of two quantities at once: the lane's four features, the
// four lane groups of a wavefront by shuffles, the four wavefronts through LDS.
template <typename Shared> __device__ __forceinline__ void mlp_sum2(Shared &sh, int &slot, const float (&a)[4], const float (&b)[4], float &A, float &B) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, q = lane >> 4, c = lane & 15;
    float u = (a[0] + a[1]) + (a[2] + a[3]), v = (b[0] + b[1]) + (b[2] + b[3]);
    u = add_from<32>(add_from<16>(u)), v = add_from<32>(add_from<16>(v));
    if (q == 0) {
        sh.red[slot][w][c][0] = u;
        sh.red[slot][w][c][1] = v;
    }
    lds_barrier();
    A = (sh.red[slot][0][c][0] + sh.red[slot][1][c][0]) + (sh.red[slot][2][c][0] + sh.red[slot][3][c][0]);
    B = (sh.red[slot][0][c][1] + sh.red[slot][1][c][1]) + (sh.red[slot][2][c][1] + sh.red[slot][3][c][1]);
    slot ^= 1;
}

}  // namespace tode
