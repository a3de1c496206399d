// The short forms of tode_math.h against the compiler's own division and square root, on the device that runs them: their
// results rest on the hardware's estimates of reciprocals and roots (a unit more or less for a few dozen operands would
// show), which nothing but the hardware knows.  float32 operands exhaustively over the forms' ranges, pairs and
// float64 operands pseudo-randomly.  A hook for tests; nothing of it runs in a solve.
#include "tode_internal.h"
#include "tode_math.h"
#include "tode_solve.h"

namespace tode {

enum ShortForm { RECIPROCAL_F32, ROOT_F32, OVER_ROOT2_F32, OVER_ROOT3_F32, QUOTIENT_F32, RECIPROCAL_F64, ROOT_F64, OVER_ROOT2_F64, OVER_ROOT3_F64, QUOTIENT_F64, POWER_F32, POWER_F64, SUM_F32, SUM_F64, SHORT_FORMS };

__device__ __forceinline__ unsigned long long scramble(unsigned long long i) {  // (the finaliser of splitmix64)
    i = (i ^ (i >> 30)) * 0xbf58476d1ce4e5b9ull;
    i = (i ^ (i >> 27)) * 0x94d049bb133111ebull;
    return i ^ (i >> 31);
}
// a value of random mantissa with an exponent of lo ... hi - 1
__device__ __forceinline__ float random_value(float, unsigned long long r, int lo, int hi) {
    return __uint_as_float((unsigned)(r & 0x7fffff) | (unsigned)(127 + lo + (int)((r >> 40) % (unsigned)(hi - lo))) << 23);
}
__device__ __forceinline__ double random_value(double, unsigned long long r, int lo, int hi) {
    return __longlong_as_double((long long)((r & 0xfffffffffffffull) | (unsigned long long)(1023 + lo + (int)((r >> 52) % (unsigned)(hi - lo))) << 52));
}

template <typename T> __device__ __forceinline__ bool short_form_differs(int form, T x, T other) {
    switch (form) {
    case 0: return reciprocal_plain(x) != (T)1 / x;
    case 1: return sqrt_plain(x) != sqrt_(x);
    case 2: return DivSqrtFeatures<T, 2>::fast(x) != DivSqrtFeatures<T, 2>::exact(x);
    case 3: return DivSqrtFeatures<T, 3>::fast(x) != DivSqrtFeatures<T, 3>::exact(x);
    default: return quotient_plain(x * other, other) != (x * other) / other;  // (x is about their quotient)
    }
}

// rpow_common against rpow: exponents inside and outside the short forms' range and such as are not computed as powers;
// every other x from around their range, the rest any bits at all
template <typename T> __device__ __forceinline__ bool power_differs(unsigned long long i) {
    constexpr double exponents[] = {-0.2, 0.2, 0.04, -0.14, 0.5, -0.5, 0.4999, -0.5001, 1.0, -1.0, 2.0, 0.7, 1e-60, 0.0};
    const unsigned long long r = scramble(2 * i + 1), s = scramble(2 * i + 2);
    T x = random_value((T)0, r, -53, 53);
    if (s & 1) x = sizeof(T) == 4 ? (T)__uint_as_float((unsigned)r) : (T)__longlong_as_double((long long)r);
    if ((s >> 1) % 1024 == 0) x = (T)((s >> 12) % 2);
    const double p = exponents[(s >> 20) % (sizeof exponents / sizeof exponents[0])];
    const T a = rpow_common<T>(x, p), b = rpow<T>(x, p);
    return !(a == b || (a != a && b != b));
}

// wave_sum against the butterfly of shuffles whose order it keeps (whole wavefronts run the caller's loop together)
template <typename T> __device__ __forceinline__ bool sum_differs(unsigned long long i) {
    const T x = random_value((T)0, scramble(i), -20, 20) * ((i & 3) ? (T)1 : (T)-1);
    T v = x;
    for (int off = 32; off > 0; off >>= 1) v = v + __shfl_xor(v, off);
    return v != wave_sum(x);
}

__global__ void __launch_bounds__(256) check_short_forms_kernel(int form, unsigned first, unsigned long long count, int *mismatches) {
    const unsigned long long start = (unsigned long long)blockIdx.x * 256 + threadIdx.x, step = (unsigned long long)gridDim.x * 256;
    int wrong = 0;
    for (unsigned long long i = start; i < count; i += step) {
        if (form < QUOTIENT_F32) {
            wrong += short_form_differs<float>(form, __uint_as_float(first + (unsigned)i), 1.0f) ? 1 : 0;
        } else if (form == QUOTIENT_F32) {
            const unsigned long long r = scramble(2 * i + 1), s = scramble(2 * i + 2);
            wrong += short_form_differs<float>(4, random_value(0.0f, r, -59, 60), random_value(0.0f, s, -40, 64)) ? 1 : 0;
        } else if (form >= SUM_F32) {
            wrong += (form == SUM_F32 ? sum_differs<float>(i) : sum_differs<double>(i)) ? 1 : 0;
        } else if (form >= POWER_F32) {
            wrong += (form == POWER_F32 ? power_differs<float>(i) : power_differs<double>(i)) ? 1 : 0;
        } else {
            const unsigned long long r = scramble(2 * i + 1), s = scramble(2 * i + 2);
            const int f = form - RECIPROCAL_F64;
            const double x = f == 0 ? random_value(0.0, r, 0, 2) : (f == 1 ? random_value(0.0, r, -100, 100) : random_value(0.0, r, -59, 60));
            wrong += short_form_differs<double>(f, x, random_value(0.0, s, -40, 64)) ? 1 : 0;
        }
    }
    if (wrong) atomicAdd(mismatches, wrong);
}

}  // namespace tode

extern "C" int tode_check_short_forms(int32_t form, int64_t samples, void *mismatches, void *stream) {
    using namespace tode;
    if (form < 0 || form >= SHORT_FORMS || samples < 1 || samples > (1ll << 40) || !mismatches) return fail(TODE_E_INVALID, "form %d of %d, %lld samples, or a null pointer", form, (int)SHORT_FORMS, (long long)samples);
    // float32: every value of the form's range (the reciprocal's is a divisor's; the other two divide scaled errors)
    const int lo = form == RECIPROCAL_F32 ? -40 : (form == ROOT_F32 ? -100 : -60), hi = form == RECIPROCAL_F32 ? 124 : (form == ROOT_F32 ? 100 : 60);
    const unsigned first = (unsigned)(127 + lo) << 23;
    const unsigned long long count = form < QUOTIENT_F32 ? (unsigned long long)(hi - lo) << 23 : ((unsigned long long)samples + 63) / 64 * 64;
    hipLaunchKernelGGL(check_short_forms_kernel, dim3(4096), dim3(256), 0, (hipStream_t)stream, form, first, count, (int *)mismatches);
    return check_hip(hipGetLastError(), "tode_check_short_forms");
}
