// Shared helpers for the libfeelmri_hip kernels (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <string>

#include "../../include/feelmri_hip.h"

namespace fm {

// Per-thread message behind fm_last_error().
void set_error(const char *fmt, ...);

#define FM_CHECK_ARG(cond, ...)          \
    do {                                 \
        if (!(cond)) {                   \
            ::fm::set_error(__VA_ARGS__); \
            return FM_ERR_ARG;           \
        }                                \
    } while (0)

#define FM_HIP(call)                                                                     \
    do {                                                                                 \
        hipError_t fm_e_ = (call);                                                       \
        if (fm_e_ != hipSuccess) {                                                       \
            ::fm::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(fm_e_),   \
                            __FILE__, __LINE__);                                         \
            return FM_ERR_HIP;                                                           \
        }                                                                                \
    } while (0)

// Launch-status check after a <<<>>> launch.
#define FM_LAUNCH_CHECK(name)                                                           \
    do {                                                                                \
        hipError_t fm_e_ = hipGetLastError();                                           \
        if (fm_e_ != hipSuccess) {                                                      \
            ::fm::set_error("launch of %s failed: %s", name, hipGetErrorString(fm_e_)); \
            return FM_ERR_HIP;                                                          \
        }                                                                               \
    } while (0)

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

__host__ __device__ inline int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// A phase u in cycles reduced for the FP32 hardware sine and cosine, which
// take revolutions and want an argument in [0, 1]: one fract (u - floor(u),
// exact) and, from FP64, one conversion.  The result can round to 1.0f, which
// the periodic functions take as 0.
__device__ inline float turns_f32(double u) { return (float)__builtin_amdgcn_fract(u); }
__device__ inline float turns_f32(float u) { return __builtin_amdgcn_fractf(u); }

// Workgroup b of a launch of ceil(n / 8) * 8 workgroups takes range
// (b % 8) * ceil(n / 8) + b / 8 of n ranges: workgroups are dealt onto the
// 8 XCDs round-robin, so each XCD runs one contiguous eighth of the ranges.
__device__ inline int64_t xcd_range(int64_t n_ranges)
{
    const int64_t per = (n_ranges + 7) / 8;
    return (int64_t)(blockIdx.x % 8) * per + blockIdx.x / 8;
}

inline unsigned xcd_grid(int64_t n_ranges) { return (unsigned)(((n_ranges + 7) / 8) * 8); }

// (h + l) v less a whole number of turns, l far below h: the product's rounding
// is that of the fraction left, 2^-54 of a turn, not of the product.
__device__ inline double turns_f64(double h, double l, double v)
{
    return fma(l, v, fma(h, v, -__builtin_rint(h * v)));
}

// sin 2 pi r, |r| <= 3/4, in FP64: r is reduced exactly to t in [-1/4, 1/4] (sin(pi - x)
// = sin x) and the Taylor series in t summed to t^21 (the next term is below
// 2e-18): with the reductions below about 20 FP64 instructions, where a sine and
// cosine pair takes about 45.
__device__ inline double sin_fraction_f64(double r)
{
    const double t = __builtin_fabs(r) > 0.25 ? __builtin_copysign(0.5, r) - r : r;
    const double q = t * t;
    double p = 0.0011309237482517963;
    p = fma(p, q, -0.012031585942120627);
    p = fma(p, q, 0.10422916220813984);
    p = fma(p, q, -0.71812230177850056);
    p = fma(p, q, 3.819952584848282);
    p = fma(p, q, -15.09464257682299);
    p = fma(p, q, 42.058693944897655);
    p = fma(p, q, -76.705859753061389);
    p = fma(p, q, 81.605249276075057);
    p = fma(p, q, -41.341702240399762);
    p = fma(p, q, 6.2831853071795862);
    return t * p;
}
// sin 2 pi (u + quarter), quarter 0 or 1/4 (a cosine; what the sum rounds then lies
// at the top of the sine).
__device__ inline double sin_cycles_f64(double u, double quarter)
{
    return sin_fraction_f64((u - __builtin_rint(u + quarter)) + quarter);
}
// The same of (h + l) v + quarter, the product as turns_f64 takes it.
__device__ inline double sin_turns_f64(double h, double l, double v, double quarter)
{
    return sin_fraction_f64(fma(l, v, fma(h, v, quarter - __builtin_rint(fma(h, v, quarter)))));
}

// Coefficients of the series below, in t: s t + s[7] t^3 + ... and 1 + c[7] t^2 + ...
struct TrigCoefs {
    double s[9] = {0.10422916220813984, -0.71812230177850056, 3.819952584848282,   -15.09464257682299, 42.058693944897655,
                   -76.705859753061389, 81.605249276075057,   -41.341702240399762, 6.2831853071795862};
    double c[8] = {0.28200596845579123, -1.714390711088672,  7.9035363713184692, -26.426256783374399,
                   60.244641371876661,  -85.456817206693728, 64.939394022668296, -19.739208802178716};
};
// The same held in scalar registers: the compiler keeps the constants of a loop in
// vector registers, 30 or more of them.  Where registers bound the waves that pays
// (Bloch, FP64: 128 with 19 spilled -> 121 with none, 0.367 -> 0.345 ms for the
// sequence named there); where they do not it costs (spiral, FP64: 3.03 -> 3.32 ms;
// radial runs 0.94 -> 1.08 ms).  Formed once, before the loop: an operand pinned in
// the loop is copied before each use, which one wave alone on a SIMD waits for.
__device__ inline TrigCoefs scalar_trig_coefs()
{
    TrigCoefs k;
#pragma unroll
    for (int i = 0; i < 9; ++i) asm volatile("" : "+s"(k.s[i]));
#pragma unroll
    for (int i = 0; i < 8; ++i) asm volatile("" : "+s"(k.c[i]));
    return k;
}

// sin and cos of 2 pi u in FP64, u in cycles: u reduced exactly to t in
// [-1/8, 1/8] and the octant's quarter turn, both Taylor series summed to t^17
// and t^16 (the next terms are below 3e-18), swapped and signed by the quarter.
// About 35 instructions, where the library's sincospi takes about 55.
__device__ inline void sincos_cycles_f64(double u, double &s, double &c, const TrigCoefs &k = TrigCoefs())
{
    const double r = u - __builtin_rint(u);
    constexpr double kWhole = 6755399441055744.0;  // 1.5 2^52: the sum's low bits are the integer
    const double qw = fma(4.0, r, kWhole);
    const double t = fma(-0.25, qw - kWhole, r);
    const int iq = (int)__builtin_bit_cast(unsigned long long, qw);
    const double w = t * t;
    double ps = k.s[0], pc = k.c[0];
#pragma unroll
    for (int i = 1; i < 8; ++i) {
        ps = fma(ps, w, k.s[i]);
        pc = fma(pc, w, k.c[i]);
    }
    ps = fma(ps, w, k.s[8]);
    pc = fma(pc, w, 1.0);
    ps *= t;
    const bool odd = iq & 1;
    const unsigned long long ss = (unsigned long long)(iq & 2) << 62, sc = (unsigned long long)((iq + 1) & 2) << 62;
    s = __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, odd ? pc : ps) ^ ss);
    c = __builtin_bit_cast(double, __builtin_bit_cast(unsigned long long, odd ? ps : pc) ^ sc);
}

// The same in FP32, u reduced in FP64: Taylor series to t^9 and t^10 (the next
// terms are below 2e-9), within an ulp or so of the rounded result where the
// hardware sine and cosine have an absolute error of a few 1e-8.
__device__ inline void sincos_cycles_f32(double u, float &s, float &c)
{
    const double r = u - __builtin_rint(u);
    const double q = __builtin_rint(4.0 * r);
    const float t = (float)fma(-0.25, q, r);
    const int iq = (int)q;
    const float w = t * t;
    float ps = 42.0586939f, pc = -26.4262568f;
    pc = fmaf(pc, w, 60.2446414f);
    ps = fmaf(ps, w, -76.7058598f);
    pc = fmaf(pc, w, -85.4568172f);
    ps = fmaf(ps, w, 81.6052493f);
    pc = fmaf(pc, w, 64.939394f);
    ps = fmaf(ps, w, -41.3417022f);
    pc = fmaf(pc, w, -19.7392088f);
    ps = fmaf(ps, w, 6.28318531f);
    pc = fmaf(pc, w, 1.0f);
    ps *= t;
    const bool odd = iq & 1;
    s = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, odd ? pc : ps) ^ ((unsigned)(iq & 2) << 30));
    c = __builtin_bit_cast(float, __builtin_bit_cast(unsigned, odd ? ps : pc) ^ ((unsigned)((iq + 1) & 2) << 30));
}

// (double)(float)pi / pi: the reference forms 2*pi from a float constant
// (cpp/feelmri/MRI.h:13), so every k.x phase carries this factor.
constexpr double kPiFOverPi = static_cast<double>(static_cast<float>(3.14159265358979323846)) /
                              3.14159265358979323846;
constexpr double kTwoPi = 6.283185307179586476925286766559;

// Number of CUs on the current device (cached per device).
int device_cu_count();

// Sum of n split partials, `stride` apart, in FP64 and in order, 8 loads in
// flight together (past the last: + 0).
template <typename P>
__device__ inline double2 sum_splits(const P *__restrict__ p, int64_t stride, int64_t n)
{
    double re = 0.0, im = 0.0;
    for (int64_t s = 0; s < n; s += 8) {
        P v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            v[u].x = v[u].y = 0;
            if (s + u < n) v[u] = p[(s + u) * stride];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            re += (double)v[u].x;
            im += (double)v[u].y;
        }
    }
    return make_double2(re, im);
}

// Reductions over splits: G threads of a workgroup of 256 share an output, each
// sums a contiguous range of its splits, and the ranges are added in order.
// Few outputs of many splits leave most CUs idle and a thread waits for one
// round of loads after the other, so G is 8 where the outputs alone fill less
// than 4 waves a CU and there are splits to share.  Radial, mixed, 342 x 55
// samples of 52 splits, 19 838 nodes, both in turn: the call 54.9 -> 43.4 us.
inline int reduce_group(int64_t n_out, int64_t n_splits)
{
    return n_splits >= 16 && n_out < (int64_t)256 * device_cu_count() ? 8 : 1;
}
inline unsigned reduce_grid(int64_t n_out, int G) { return (unsigned)cdiv(n_out, 256 / G); }
// The output of this thread, and its sum: of all splits in the thread with
// tid < 256 / G, whose result it is.
template <int G>
__device__ inline int64_t reduce_output() { return (int64_t)blockIdx.x * (256 / G) + threadIdx.x % (256 / G); }
template <int G, typename P>
__device__ inline double2 reduce_sum(const P *__restrict__ p, int64_t stride, int64_t n, bool live)
{
    if constexpr (G == 1) return live ? sum_splits(p, stride, n) : make_double2(0.0, 0.0);
    constexpr int kOut = 256 / G;
    __shared__ double2 sums[G][kOut];
    const int g = threadIdx.x / kOut, o = threadIdx.x % kOut;
    const int64_t share = (n + G - 1) / G, s0 = g * share, s1 = s0 + share < n ? s0 + share : n;
    sums[g][o] = live && s0 < s1 ? sum_splits(p + s0 * stride, stride, s1 - s0) : make_double2(0.0, 0.0);
    __syncthreads();
    double2 t = sums[0][o];
#pragma unroll
    for (int q = 1; q < G; ++q) {
        t.x += sums[q][o].x;
        t.y += sums[q][o].y;
    }
    return t;
}

// Workgroups of `kernel` (a __global__ function) that one CU holds at once
// with `threads` threads and `dyn` bytes of dynamic LDS; 1 when the runtime
// cannot tell.
template <typename F>
int blocks_per_cu(F kernel, int threads, size_t dyn)
{
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, dyn) != hipSuccess || n < 1) n = 1;
    return n;
}

inline int blocks_per_cu(const void *kernel, int threads, size_t dyn)
{
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, dyn) != hipSuccess || n < 1) n = 1;
    return n;
}

// Node splits of a grid of `base` workgroups per split, each split a whole
// number of `chunk`-node chunks: the count in [s_min, 2 s_min] (and at most
// s_max, 0 = one chunk per split) that minimises (rounds of `capacity`
// concurrent workgroups) x (nodes per split), the fewest on a tie.
// Workgroups of one grid take the same time, so a last round that is only
// partly filled leaves the rest of the device idle.
int64_t balanced_splits(int64_t N, int64_t chunk, int64_t base, int64_t s_min, int64_t capacity,
                        int64_t s_max = 0);

// Zero n doubles on the stream with a kernel (not a memset node, so the
// call can be captured into a HIP graph and replayed).
int zero_f64_async(double *x, int64_t n, hipStream_t st);

}  // namespace fm
