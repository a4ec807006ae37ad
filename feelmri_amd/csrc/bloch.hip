// Per-node Bloch integrator (Cayley-Klein rotation, then T1/T2 relaxation).
//
// reference: cpp/feelmri/BlochSimulator.cpp:151-276 (static nodes) and
// :12-148 (moving nodes), solve_mri<T>.
//
// One lane per node; node attributes come from an SoA table (coalesced).
// The event table is walked in chunks of 256 events: each lane of the
// workgroup stages one event (rf, |rf|^2, G, dt, flags and, for
// moving nodes, the POD weights of that step) into LDS, then every lane
// integrates its node through the chunk reading the events by broadcast.
// Step i -> i+1 uses event i+1; e1/e2 are refreshed only when dt changes;
// |B| is floored at 1e-12; rotation first, then relaxation toward M0.
//
// Events without RF (rf = 0, the same for every lane) take the precession
// the rotation reduces to: beta = 0 and conj(alpha)^2 = exp(-i gamma dt Bz),
// so Mxy turns by -gamma dt Bz and the rotation leaves Mz alone.  This skips
// |B|, its reciprocal and the Cayley-Klein products; the result departs from
// the general step by rounding only (|alpha|^2 is 1 to an ulp).
//
// What an event needs is found once, by the thread that stages it, and stored
// as flags that every lane branches on together:
//   * the gradient axes that are on: with more than two modes a position along an
//     axis is formed only where its gradient is not 0, since the other products
//     are 0 (all three axes where a coefficient or a position is not finite,
//     whose products are not); with fewer the tests cost more than they save;
//   * whether dt is the previous step's;
//   * whether RF and field repeat the previous step's (hard pulses, gradient
//     plateaus and delays; moving nodes: no gradient): the lane then keeps the
//     rotation it formed.  FP32 form: where dt is the same, to the last bit the
//     same results.  FP64 form: dt = diff(times) varies by roundings (~1e-15
//     ms) within such a run; to 1e-12 ms the kept sine and cosine and the decay
//     factors are corrected to first order (the second order is below 1e-16).
// A run's steps are an inner loop that applies the rotation and relaxes: the
// rotation is local to it (kept across the outer loop it was copied on every
// path).  FP64 rotations are formed as a 3 x 3 matrix and applied in 9
// instructions; formed and applied as (alpha, beta) products they took 45 a
// step.  The next event's record is read from LDS in wide reads while the current
// one relaxes.
//
// Finding out whether the next step is of the run costs a single event more than
// forming its rotation again would (30 000 nodes, 400 events that all differ: 134
// against 85 us in FP64, 95 against 87 in FP32), so a chunk with few like steps takes a
// loop without runs.  Few is less than a half in FP64 (runs of 2: 92 against 85 us at
// 30 000 nodes, 258 against 308 at 400 000) and less than a sixth in FP32 (runs of 2: 63
// against 87 us; all different 210 against 187 at 400 000).
//
// Bound by VALU issue, and by the latency of one event's chain of operations where
// the nodes do not fill the device.  The mode loop is unrolled for some mode counts
// (it was one loop of 16 with a test each).
// Before: one loop over the events, every rotation formed and applied as products.
// 1 948 800 moving nodes, 1 mode, 11 255 events, FP32: 21.0-22.1 ms (before: 52.6);
// 512 000 nodes, 33 blocks, 419 steps in all, FP64: 0.29 ms (0.929).  1000 events
// that all differ: 512 000 nodes, FP64 0.88 ms (1.10), with RF 1.63 (2.19), FP32 0.52
// (0.56), 0.95 (1.00); 30 000 nodes, FP64 0.22 (0.23), 0.30 (0.37), FP32 0.22 (0.22), 0.29
// (0.29); 20-event plateaus instead: 0.14 (0.23), 0.08 (0.22).  Slower than before: events
// of which every one has another dt, FP64, 30 000 nodes, 0.35 (0.33; at 512 000 1.67
// against 1.78).
#include <algorithm>
#include <type_traits>

#include "fm_common.h"

namespace fm {

constexpr int kBlochThreads = 256;
constexpr int kBlochChunk = 256;
constexpr int kBlochMaxModes = 16;
constexpr int kChainMaxBlocks = 128;  // blocks per chained launch

// A chain of blocks in one launch (static nodes, final state): the blocks'
// event tables are concatenated; offset[b] is block b's first event.  That
// event is not a step (step i of a block uses its event i + 1): it ends
// block b - 1 instead, applying code[b - 1] = spoil | (store column + 1) << 1
// -- the store of the state into column `col` of the (n_store, N) stores,
// then the artificial spoiling Mxy = 0 (Bloch.py:355-368).  code[n - 1] is
// applied after the last event.
struct ChainDesc {
    int64_t offset[kChainMaxBlocks + 1];
    int32_t code[kChainMaxBlocks];
    int32_t n;
};
struct NoChain {};

template <typename T>
struct alignas(16) Event {
    T rf_re, rf_im, rf2, dt;
    T gx, gy, gz;
    int flags;  // kEv...; of a block's end 1 + its code, negated
};
// Event flags: axes with a gradient, RF on, rotation as the previous step's,
// dt as the previous step's.
constexpr int kEvAxes = 7, kEvRf = 8, kEvSame = 16, kEvDt = 32;
// FP64: largest departure of dt (ms) that is corrected to first order, and the
// largest 1/T1, 1/T2 (1/ms) of a wave that does so: the second order of the decay
// is then below 1e-16.  (At T = 0 the rate is infinite and has no first order.)
constexpr double kDtNear = 1e-12, kRateNear = 1e4;

// FP32 form: the hardware sine/cosine, which take revolutions, after
// reducing the argument to [-1/2, 1/2] revolution.  Their error is absolute
// (a few 1e-7), which is large relative to the small per-event rotations of
// an RF pulse (e.g. 0.013 rad per 10 us step of a 15 deg, 0.2 ms pulse) and
// accumulates over the pulse; below 0.25 rad the Taylor series to x^7 / x^6
// (truncation < 1e-10) is used instead.  The choice is per lane; the wave
// evaluates only the form(s) its lanes need (series only, hardware only, or
// both and a select).
__device__ inline void sincos_f32(float x, float *s, float *c)
{
    float r = x * 0.159154943091895336f;
    r -= __builtin_rintf(r);
    const float a = r * 6.28318530717958648f;
    const bool small = __builtin_fabsf(a) < 0.25f;
    auto series = [&](float &ps, float &pc) {
        const float a2 = a * a;
        ps = a * (1.0f - a2 * (1.0f / 6.0f) * (1.0f - a2 * (1.0f / 20.0f) * (1.0f - a2 * (1.0f / 42.0f))));
        pc = 1.0f - a2 * 0.5f * (1.0f - a2 * (1.0f / 12.0f) * (1.0f - a2 * (1.0f / 30.0f)));
    };
    if (__all(small)) {
        series(*s, *c);
    } else if (!__any(small)) {
        *s = __builtin_amdgcn_sinf(r);
        *c = __builtin_amdgcn_cosf(r);
    } else {
        float ps, pc;
        series(ps, pc);
        const float hs = __builtin_amdgcn_sinf(r), hc = __builtin_amdgcn_cosf(r);
        *s = small ? ps : hs;
        *c = small ? pc : hc;
    }
}

template <typename T>
__device__ inline T dev_exp(T x);
template <>
__device__ inline double dev_exp<double>(double x) { return exp(x); }
template <>
__device__ inline float dev_exp<float>(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }

// An FP64 constant of the FP32 form's seldom taken decay update, in scalar registers:
// left to the compiler these are hoisted into some 20 vector registers of the event
// loop, which then spills (static nodes: 14 of 64).
__device__ inline double seldom(double c)
{
    asm("" : "+s"(c));
    return c;
}

// T1 recovery Mz' = Mz e1 + (1 - e1) M0.  FP64 form: exactly the reference's
// expression (BlochSimulator.cpp:271).  FP32 form: Mz - om1 (Mz - M0) with
// om1 = 1 - e1 = -expm1(x) evaluated in FP64 and rounded once.  The spoiled
// steady state (1 - E1) / (1 - E1 cos a) magnifies a relative error in E1 by
// E1 / (1 - E1) (~200 for TR 5 ms, T1 1 s), so e1 rounded to FP32 (or 1 - e1
// formed in FP32) would bias Mz by ~1e-5; om1 carries the recovery with full
// FP32 relative precision.  Evaluated only when dt changes.
// Every lane takes the form its own x asks for, so that a node's result does not
// depend on its neighbours in the wave.
__device__ inline float one_minus_exp(float x)
{
    const double w = (double)x;
    const bool small = __builtin_fabsf(x) < 1.0f / 64.0f;  // an event against T1: the series to w^7, within 3e-15
    double p = fma(w, seldom(1.0 / 5040.0), seldom(1.0 / 720.0));
    p = fma(w, p, seldom(1.0 / 120.0));
    p = fma(w, p, seldom(1.0 / 24.0));
    p = fma(w, p, seldom(1.0 / 6.0));
    p = fma(w, p, 0.5);
    p = w * fma(w, p, 1.0);
    if (!__all(small)) {
        // x = n ln 2 + r, |r| <= ln 2 / 2, the series of exp(r) to r^13; exp(x) - 1
        // loses no more than 6 of 53 bits.  0 or infinity beyond +-800.
        const double v = w < -800.0 ? -800.0 : w > 800.0 ? 800.0 : w;
        const double n = __builtin_rint(v * seldom(1.4426950408889634));
        const double r = fma(-n, seldom(2.3190468138462996e-17), fma(-n, seldom(0.6931471805599453), v));
        double e = 1.0;
#pragma unroll
        for (int i = 13; i > 0; --i) e = fma(r * seldom(1.0 / i), e, 1.0);
        e = __builtin_amdgcn_ldexp(e, (int)n) - 1.0;
        p = small ? p : e;
    }
    return (float)-p;
}

// The FP32 rotation of an event with RF: alpha = c - i nz s, beta = -i (rf/|B|)
// s (BlochSimulator.cpp:251-262), as the coefficients of Mz, Mxy and conj(Mxy).
// The Mz coefficient is 1 - 2 |beta|^2, equal to |alpha|^2 - |beta|^2 for a
// unitary (alpha, beta): in FP32 c^2 + s^2 misses 1 by up to an ulp, the same
// way on every event of a readout.
struct NoCoefs {};
struct Rot32 {
    float zr, zi;      // 2 conj(alpha) beta: Mz into Mxy
    float ar, ai;      // conj(alpha)^2: Mxy into Mxy
    float br, bi;      // beta^2: conj(Mxy) into Mxy (subtracted)
    float m, abr, abi; // Mz into Mz; alpha beta: 2 Re(alpha beta conj(Mxy)) out of Mz
};
__device__ inline void rot_make(Rot32 &r, float Bz, float rf_re, float rf_im, float rf2, float gamma, float dt, NoCoefs)
{
    float Bn = __builtin_amdgcn_sqrtf(fmaf(Bz, Bz, rf2));
    if (Bn < 1e-12f) Bn = 1e-12f;
    const float inv = __builtin_amdgcn_rcpf(Bn);
    const float nz = Bz * inv;
    float s, c;
    sincos_f32(Bn * (-0.5f * gamma * dt), &s, &c);
    const float ar = c, ai = -nz * s;
    const float br = rf_im * inv * s, bi = -rf_re * inv * s;
    // every sum of two products is written as one fma and one product, so that
    // each instantiation of the kernel rounds alike (a free contraction may
    // fuse either product)
    const float b2 = fmaf(br, br, bi * bi);
    const float car = ar, cai = -ai;
    r.zr = 2.0f * fmaf(car, br, -(cai * bi));
    r.zi = 2.0f * fmaf(car, bi, cai * br);
    r.ar = fmaf(car, car, -(cai * cai));
    r.ai = (2.0f * car) * cai;
    r.br = fmaf(br, br, -(bi * bi));
    r.bi = (2.0f * br) * bi;
    r.m = fmaf(-2.0f, b2, 1.0f);
    r.abr = fmaf(ar, br, -(ai * bi));
    r.abi = fmaf(ar, bi, ai * br);
}
__device__ inline void rot_apply(const Rot32 &r, bool, float, float &mxr, float &mxi, float &mz)
{
    const float cmr = mxr, cmi = -mxi;
    const float nmr = fmaf(r.zr, mz, fmaf(r.ar, mxr, -(r.ai * mxi)) - fmaf(r.br, cmr, -(r.bi * cmi)));
    const float nmi = fmaf(r.zi, mz, fmaf(r.ar, mxi, r.ai * mxr) - fmaf(r.br, cmi, r.bi * cmr));
    mz = fmaf(r.m, mz, -(2.0f * fmaf(r.abr, cmr, -(r.abi * cmi))));
    mxr = nmr;
    mxi = nmi;
}
// Free precession: Mxy exp(-i gamma dt Bz).
struct Pre32 {
    float s, c;
};
__device__ inline void pre_make(Pre32 &r, float Bz, float gamma, float dt, NoCoefs)
{
    sincos_f32(-gamma * dt * Bz, &r.s, &r.c);
}
__device__ inline void pre_apply(const Pre32 &r, bool, float, float &mxr, float &mxi)
{
    const float nmr = fmaf(r.c, mxr, -(r.s * mxi));
    mxi = fmaf(r.c, mxi, r.s * mxr);
    mxr = nmr;
}

// 1 / sqrt(x) for x in [1e-24, 1e24]: the hardware's estimate and two Newton
// steps (error below an ulp or so).
__device__ inline double rsqrt_f64(double x)
{
    double r = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const double e = fma(-x * r, r, 1.0);
        r = fma(0.5 * r, e, r);
    }
    return r;
}

// FP64: the rotation matrix about the axis n = (rf, Bz) / |B|, and the angle's
// rate om per ms of dt: for a dt that is off by d the rotation by om d about n
// follows, to first order.
struct Rot64 {
    double m[9], nx, ny, nz, om;
};
// -gamma dt B in cycles.  gamma / 2 pi enters as two doubles: its rounding
// would be the same on every event, and add up over a sequence.
__device__ inline double cycles_f64(double B, double gamma, double dt)
{
    constexpr double kHi = 0.15915494309189535, kLo = -9.839338337591243e-18;  // 1 / 2 pi
    const double hi = gamma * kHi, lo = fma(gamma, kLo, fma(gamma, kHi, -hi));
    const double u = -dt * B;
    return fma(u, hi, u * lo);
}
__device__ inline void rot_make(Rot64 &r, double Bz, double rf_re, double rf_im, double rf2, double gamma, double dt,
                                const TrigCoefs &trig)
{
    const double B2 = fma(Bz, Bz, rf2);
    const double B2c = B2 < 1e-24 ? 1e-24 : B2;  // |B| floored at 1e-12
    const double inv = rsqrt_f64(B2c), B0 = B2c * inv;
    const double Bn = fma(0.5 * inv, fma(-B0, B0, B2c), B0);
    double sh, ch;
    sincos_cycles_f64(0.5 * cycles_f64(Bn, gamma, dt), sh, ch, trig);  // of the half angle
    const double x = rf_re * inv, y = rf_im * inv, z = Bz * inv;
    r.nx = x;
    r.ny = y;
    r.nz = z;
    const double s = 2.0 * sh * ch, k = 2.0 * sh * sh;  // v + s n x v + k n x (n x v)
    const double kx = k * x, ky = k * y, kz = k * z;
    r.m[0] = 1.0 - fma(ky, y, kz * z);
    r.m[1] = fma(kx, y, -(s * z));
    r.m[2] = fma(kx, z, s * y);
    r.m[3] = fma(kx, y, s * z);
    r.m[4] = 1.0 - fma(kx, x, kz * z);
    r.m[5] = fma(ky, z, -(s * x));
    r.m[6] = fma(kx, z, -(s * y));
    r.m[7] = fma(ky, z, s * x);
    r.m[8] = 1.0 - fma(kx, x, ky * y);
    r.om = -gamma * Bn;
}
__device__ inline void rot_apply(const Rot64 &r, bool off, double d, double &mxr, double &mxi, double &mz)
{
    const double a = fma(r.m[0], mxr, fma(r.m[1], mxi, r.m[2] * mz));
    const double b = fma(r.m[3], mxr, fma(r.m[4], mxi, r.m[5] * mz));
    const double c = fma(r.m[6], mxr, fma(r.m[7], mxi, r.m[8] * mz));
    mxr = a;
    mxi = b;
    mz = c;
    if (off) {
        asm volatile("");  // a branch, not a select
        const double th = r.om * d;
        mxr = fma(th, fma(r.ny, c, -(r.nz * b)), a);
        mxi = fma(th, fma(r.nz, a, -(r.nx * c)), b);
        mz = fma(th, fma(r.nx, b, -(r.ny * a)), c);
    }
}
struct Pre64 {
    double s, c, om;
};
__device__ inline void pre_make(Pre64 &r, double Bz, double gamma, double dt, const TrigCoefs &trig)
{
    sincos_cycles_f64(cycles_f64(Bz, gamma, dt), r.s, r.c, trig);
    r.om = -gamma * Bz;
}
__device__ inline void pre_apply(const Pre64 &r, bool off, double d, double &mxr, double &mxi)
{
    const double a = fma(r.c, mxr, -(r.s * mxi)), b = fma(r.c, mxi, r.s * mxr);
    mxr = a;
    mxi = b;
    if (off) {
        asm volatile("");
        const double th = r.om * d;
        mxr = fma(-th, b, a);
        mxi = fma(th, a, b);
    }
}

template <typename T>
struct Cplx2;
template <>
struct Cplx2<double> {
    using type = double2;
    using Rot = Rot64;
    using Pre = Pre64;
};
template <>
struct Cplx2<float> {
    using type = float2;
    using Rot = Rot32;
    using Pre = Pre32;
};

// Chained blocks: kChainHost takes the block boundaries from a ChainDesc
// passed by value, kChainMarks from per-event marks in device memory
// (marks[e] = 1 + code of the block ending before event e, 0 inside a
// block; marks[n_time] = 1 + code of the last block) with the event count
// read from device memory as well.
constexpr int kChainNone = 0, kChainHost = 1, kChainMarks = 2;

// Modes above which a gradient axis that is off is skipped.
constexpr int kSkipFrom = 2;

// Waves per SIMD: one event is a chain of dependent operations that waves overlap,
// until registers spill.  400 events that all differ, with one wave fewer and one
// more (us, 200 000 nodes unless named):
//   FP64, static  192, 195, 196; 800 000 nodes 559, 551, 544; chained blocks spill 22
//                 registers at 5 (33 blocks: 0.297 ms at 5, 0.291 at 4);
//   FP64, 1 mode  222, 221, 224;  2 modes 256, 233, 236;  5 modes 290, 269 (3, 4 waves);
//   FP64, 10      392, 358, 391;  16 445, 445, 445;
//   FP32, 1 mode  139, 137;  2 modes 144, 144 (7, 8: the most there are);
//   FP32, 5       174, 173, 171 and 800 000 nodes 453, 455, 434;
//   FP32, 10      210, 209, 210;  16 249, 245, 264.
constexpr int bloch_waves(bool f64, int RB, bool chain)
{
    return f64 ? (RB == 0 && !chain ? 5 : RB <= 5 ? 4 : RB <= 10 ? 3 : 2) : (RB <= 2 ? 8 : RB <= 5 ? 7 : 4);
}

// RB: modes per component, 0 for static nodes (R <= RB; the rest are zero).
template <typename T, int RB, bool HISTORY, int CHAIN = kChainNone>
__global__ __launch_bounds__(kBlochThreads, bloch_waves(sizeof(T) == 8, RB, CHAIN != kChainNone)) void k_bloch(
    const double *__restrict__ packed, int64_t N, int64_t n_time, double M0d, double gammad,
    const double *__restrict__ rf, const double *__restrict__ G, const double *__restrict__ dt,
    const double *mxy_in, const double *mz_in,  // may alias mxy_fin / mz_fin
    const float *__restrict__ modes, int R, const double *__restrict__ mcoef,
    typename Cplx2<T>::type *__restrict__ mxy_out, T *__restrict__ mz_out,
    double2 *mxy_fin, double *mz_fin, const std::conditional_t<CHAIN == kChainHost, ChainDesc, NoChain> chain = {},
    float2 *__restrict__ store_xy = nullptr, float *__restrict__ store_z = nullptr,
    const int32_t *__restrict__ marks = nullptr, const int64_t *__restrict__ n_events = nullptr,
    int64_t n_store = 0)
{
    using C2 = typename Cplx2<T>::type;
    constexpr bool MOTION = RB > 0, F64 = sizeof(T) == 8, kSkip = RB > kSkipFrom;
    static_assert(CHAIN == kChainNone || !HISTORY, "chained blocks keep the final state only");
    constexpr int kRow = RB + 3;                     // mode weights, translation
    __shared__ Event<T> sev[kBlochChunk + 1];        // one more: the read ahead
    __shared__ T scoef[MOTION ? (kBlochChunk + 1) * kRow : 1];
    __shared__ int slike[kBlochThreads / 64];
    if constexpr (CHAIN == kChainMarks) {
        // the event count is produced on the device; n_time is the capacity
        const int64_t ne = *n_events;
        n_time = ne < n_time ? ne : n_time;
    }

    const int tid = threadIdx.x;
    const int64_t p = (int64_t)blockIdx.x * kBlochThreads + tid;
    const bool active = p < N;
    const T M0 = (T)M0d, gamma = (T)gammad;
    std::conditional_t<F64, TrigCoefs, NoCoefs> trig;
    if constexpr (F64) trig = scalar_trig_coefs();

    T pos[3] = {0, 0, 0}, invT1 = 0, invT2 = 0, dB = 0;
    T mxr = 0, mxi = 0, mz = 0;
    float md[MOTION ? 3 * RB : 1];
    bool finite = true;  // position and modes: a gradient of 0 leaves nothing of them
    if (active) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            pos[c] = (T)packed[c * N + p];
            finite = finite && __builtin_isfinite(pos[c]);
        }
        invT1 = (T)packed[3 * N + p];
        invT2 = (T)packed[4 * N + p];
        dB = (T)packed[5 * N + p];
        mxr = (T)mxy_in[2 * p];
        mxi = (T)mxy_in[2 * p + 1];
        mz = (T)mz_in[p];
        if constexpr (MOTION) {
#pragma unroll
            for (int r = 0; r < RB; ++r)
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    md[c * RB + r] = r < R ? modes[(int64_t)(c * R + r) * N + p] : 0.0f;
                    finite = finite && __builtin_isfinite(md[c * RB + r]);
                }
        }
        if (HISTORY) {
            C2 o;
            o.x = mxr;
            o.y = mxi;
            mxy_out[p] = o;
            mz_out[p] = mz;
        }
    }
    const int all_axes = __all(finite) ? 0 : kEvAxes;  // the same for the wave
    const T dt_near = __all(__builtin_fabs(invT1) <= kRateNear && __builtin_fabs(invT2) <= kRateNear) ? (T)kDtNear : (T)0;
    // decay factors (FP32: e1 is 1 - exp(-dt / T1); FP64: om1 = (1 - e1) M0) and their dt
    T e1 = 0, e2 = 0, om1 = 0, dt_e = (T)-1;
    T dt_r = (T)-1;                                    // dt of the rotation
    const int64_t n_steps = n_time > 0 ? n_time - 1 : 0;
    const int RC = R + 3;
    if (tid == 0) sev[kBlochChunk].flags = 0;

    int64_t kept = p + N;                              // HISTORY: where the next state goes
    for (int64_t base = 0; base < n_steps; base += kBlochChunk) {
        __syncthreads();
        bool like;  // a step like the one before
        {
            const int64_t i = base + tid;  // step i uses event i + 1
            Event<T> ev;
            int mk = 0, fl = 0;
            if (i < n_steps) {
                const double rr = rf[2 * (i + 1)], ri = rf[2 * (i + 1) + 1];
                const double g0 = G[3 * (i + 1)], g1 = G[3 * (i + 1) + 1], g2 = G[3 * (i + 1) + 2];
                // the event before, loaded with it (one wait for both)
                const double pr = rf[2 * i], pi = rf[2 * i + 1], p0 = G[3 * i], p1 = G[3 * i + 1], p2 = G[3 * i + 2];
                const T pdt = (T)dt[i];
                ev.rf_re = (T)rr;
                ev.rf_im = (T)ri;
                ev.rf2 = ev.rf_re * ev.rf_re + ev.rf_im * ev.rf_im;
                ev.dt = (T)dt[i + 1];
                ev.gx = (T)g0;
                ev.gy = (T)g1;
                ev.gz = (T)g2;
                fl = (ev.gx != (T)0 ? 1 : 0) | (ev.gy != (T)0 ? 2 : 0) | (ev.gz != (T)0 ? 4 : 0) |
                     (ev.rf2 != (T)0 ? kEvRf : 0);
                // the previous event (a step unless it starts a block or is the first)
                bool prev_step = i >= 1;
                if constexpr (CHAIN == kChainMarks) {
                    mk = marks[i + 1];
                    prev_step = prev_step && marks[i] == 0;
                }
                if constexpr (CHAIN == kChainHost) {
                    // event q starts block b > 0: it ends block b - 1
                    auto starts = [&](int64_t q) {
                        int lo = 1, hi = chain.n - 1;
                        while (lo <= hi) {
                            const int mid = (lo + hi) / 2;
                            if (chain.offset[mid] == q) return 1 + chain.code[mid - 1];
                            if (chain.offset[mid] < q) lo = mid + 1;
                            else hi = mid - 1;
                        }
                        return 0;
                    };
                    mk = starts(i + 1);
                    prev_step = prev_step && starts(i) == 0;
                }
                if (prev_step & (pdt == ev.dt)) fl |= kEvDt;
                const bool same = (pr == rr) & (pi == ri) & (p0 == g0) & (p1 == g1) & (p2 == g2);
                if (prev_step & same & (F64 || (fl & kEvDt)) & (!MOTION || (fl & kEvAxes) == 0)) fl |= kEvSame;
            } else {
                ev.rf_re = ev.rf_im = ev.rf2 = ev.gx = ev.gy = ev.gz = ev.dt = 0;
            }
            if constexpr (MOTION) {
                bool fin = true;
                for (int q = 0; q < kRow; ++q) {
                    // weights 0 .. R - 1, zeros up to RB, translation
                    const int src = q < R ? q : (q >= RB ? q - RB + R : -1);
                    const T w = i < n_steps && src >= 0 ? (T)mcoef[i * RC + src] : (T)0;
                    scoef[tid * kRow + q] = w;
                    fin = fin && __builtin_isfinite(w);
                }
                if (!fin) fl = (fl | kEvAxes) & ~kEvSame;
            }
            ev.flags = mk != 0 ? -mk : fl;
            sev[tid] = ev;
            like = mk == 0 && (fl & kEvSame);
        }
        {   // how many of the chunk's steps are like the one before: a wave's count each
            const int wave_like = __builtin_popcountll(__ballot(like));
            if (tid % 64 == 0) slike[tid / 64] = wave_like;
        }
        __syncthreads();
        int n_like = 0;
#pragma unroll
        for (int w = 0; w < kBlochThreads / 64; ++w) n_like += slike[w];
        n_like = __builtin_amdgcn_readfirstlane(n_like);
        const int cnt = (n_steps - base < kBlochChunk) ? (int)(n_steps - base) : kBlochChunk;
        // field along z: rounded as the sum over all three axes would be
        auto field = [&](const Event<T> &ev, int fl, const T *w) {
#pragma clang fp contract(off)
            auto at = [&](auto axis) {
                constexpr int c = decltype(axis)::value;
                T q = pos[c];
                if constexpr (MOTION) {
                    T dq = w[RB + c];
#pragma unroll
                    for (int r = 0; r < RB; ++r) dq = fma((T)md[c * RB + r], w[r], dq);
                    q += dq;
                }
                return q;
            };
            using X = std::integral_constant<int, 0>;
            using Y = std::integral_constant<int, 1>;
            using Z = std::integral_constant<int, 2>;
            T Bz = 0;
            if (!kSkip || (fl & kEvAxes) == kEvAxes) {
                Bz = fma(at(Z{}), ev.gz, fma(at(Y{}), ev.gy, at(X{}) * ev.gx));
            } else {  // only the axes that are on
                if (fl & 1) Bz = at(X{}) * ev.gx;
                if (fl & 2) Bz = fma(at(Y{}), ev.gy, Bz);
                if (fl & 4) Bz = fma(at(Z{}), ev.gz, Bz);
            }
            return Bz + dB;
        };
        // a block ends at an event whose flags are the negated mark (the same for every lane)
        auto block_end = [&](int mk) {
            const int col = ((mk - 1) >> 1) - 1;
            if (col >= 0 && (CHAIN == kChainHost || col < n_store)) {
                store_xy[p + col * N] = make_float2((float)mxr, (float)mxi);
                store_z[p + col * N] = (float)mz;
            }
            if ((mk - 1) & 1) mxr = mxi = 0;
        };
        auto keep = [&]() {  // the state after one more event
            if constexpr (HISTORY) {
                C2 v;
                v.x = mxr;
                v.y = mxi;
                mxy_out[kept] = v;
                mz_out[kept] = mz;
                kept += N;
            }
        };
        if (active && n_like * (F64 ? 2 : 6) < cnt) {
            // few like steps: every event by itself
            T de = 0;
            bool off_e = false;
            auto step = [&](int e, const Event<T> &ev) {
                const int flags = __builtin_amdgcn_readfirstlane(ev.flags);
                if constexpr (CHAIN != kChainNone) {
                    if (flags < 0) {
                        block_end(-flags);
                        return;
                    }
                }
                const int fl = flags | all_axes;
                if constexpr (F64) {
                    if (!(fl & kEvDt) || e == 0) {
                        de = ev.dt - dt_e;
                        if (!__all(__builtin_fabs(de) <= dt_near)) {
                            e1 = dev_exp<T>(-ev.dt * invT1);
                            e2 = dev_exp<T>(-ev.dt * invT2);
                            om1 = (1.0 - e1) * M0;
                            dt_e = ev.dt;
                            de = 0;
                            off_e = false;
                        } else {
                            off_e = __any(de != 0);
                        }
                    }
                } else if (!(fl & kEvDt)) {
                    e1 = one_minus_exp(-ev.dt * invT1);
                    e2 = dev_exp<T>(-ev.dt * invT2);
                }
                const T Bz = field(ev, fl, &scoef[MOTION ? e * kRow : 0]);
                if (fl & kEvRf) {
                    typename Cplx2<T>::Rot rot;
                    rot_make(rot, Bz, ev.rf_re, ev.rf_im, ev.rf2, gamma, ev.dt, trig);
                    rot_apply(rot, false, (T)0, mxr, mxi, mz);
                } else {
                    typename Cplx2<T>::Pre pre;
                    pre_make(pre, Bz, gamma, ev.dt, trig);
                    pre_apply(pre, false, (T)0, mxr, mxi);
                }
                if constexpr (F64) {
                    if (off_e) {
                        asm volatile("");
                        const T f2 = fma(-de * invT2, e2, e2), f1 = fma(-de * invT1, e1, e1);
                        mxr *= f2;
                        mxi *= f2;
                        mz = fma(mz, f1, (1.0 - f1) * M0);
                    } else {
                        mxr *= e2;
                        mxi *= e2;
                        mz = fma(mz, e1, om1);
                    }
                } else {
                    mxr *= e2;
                    mxi *= e2;
                    mz = mz - e1 * (mz - M0);
                }
                keep();
            };
            if constexpr (F64 || HISTORY) {
                for (int e = 0; e < cnt; ++e) {
                    const Event<T> a = sev[e];
                    step(e, a);
                }
            } else {
                // two events read at a time: the second's latency passes behind the first's step
                for (int e = 0; e < cnt; e += 2) {
                    const Event<T> a = sev[e], b = sev[e + 1];
                    asm volatile("");
                    step(e, a);
                    if (e + 1 < cnt) step(e + 1, b);
                }
            }
        } else if (active) {
            int e = 0;
            Event<T> ev;
            T cf[RB > 0 && RB <= 2 ? kRow : 1];
            // event e, and its weights where they are few, in wide reads kept together
            auto fetch = [&]() {
                ev = sev[e];
                if constexpr (RB > 0 && RB <= 2)
#pragma unroll
                    for (int q = 0; q < kRow; ++q) cf[q] = scoef[e * kRow + q];
            };
            auto fetched = [&]() {
                {
                    asm volatile("" : "+v"(ev.rf_re), "+v"(ev.rf_im), "+v"(ev.rf2), "+v"(ev.dt), "+v"(ev.gx), "+v"(ev.gy),
                                 "+v"(ev.gz), "+v"(ev.flags));
                    if constexpr (RB > 0 && RB <= 2)
#pragma unroll
                        for (int q = 0; q < kRow; ++q) asm volatile("" : "+v"(cf[q]));
                }
            };
            fetch();
            fetched();
            T de = 0, d = 0;  // FP64: departures of dt from that of the decay factors and of the rotation
            bool off = false, off_e = false;  // either, the first is not 0
            // the end of a step: the next event's record, then relaxation
            auto relax = [&]() {
                ++e;
                fetch();  // one past the last: the spare entry, which is not a step
                if constexpr (F64) {
                    if (off) {
                        asm volatile("");
                        const T f2 = fma(-de * invT2, e2, e2), f1 = fma(-de * invT1, e1, e1);
                        mxr *= f2;
                        mxi *= f2;
                        mz = fma(mz, f1, (1.0 - f1) * M0);
                    } else {
                        mxr *= e2;
                        mxi *= e2;
                        mz = fma(mz, e1, om1);
                    }
                } else {
                    mxr *= e2;
                    mxi *= e2;
                    mz = mz - e1 * (mz - M0);
                }
                fetched();
                keep();
            };
            // the next step has the rotation and decay at hand
            auto more = [&]() {
                const int fl = __builtin_amdgcn_readfirstlane(ev.flags);
                if (fl < 0 || !(fl & kEvSame)) return false;
                if (F64 && !(fl & kEvDt)) {
                    de = ev.dt - dt_e;
                    d = ev.dt - dt_r;
                    const T m = __builtin_fabs(de) + __builtin_fabs(d);
                    off = __any(m != 0);
                    off_e = __any(de != 0);
                    return __all(m <= dt_near) != 0;
                }
                return true;
            };
            while (e < cnt) {
                const int flags = __builtin_amdgcn_readfirstlane(ev.flags);
                const int fl = flags | all_axes;
                if constexpr (CHAIN != kChainNone) {
                    if (flags < 0) {
                        block_end(-flags);
                        ++e;
                        fetch();
                        fetched();
                        continue;
                    }
                }
                // BlochSimulator.cpp:207-214: e1/e2 only when dt changes.  dt
                // is the same for every lane, so these are real branches.
                if constexpr (F64) {
                    // (a chunk begins without the departure of the one before)
                    if (!(fl & kEvDt) || e == 0) {
                        de = ev.dt - dt_e;
                        if (!__all(__builtin_fabs(de) <= dt_near)) {
                            e1 = dev_exp<T>(-ev.dt * invT1);
                            e2 = dev_exp<T>(-ev.dt * invT2);
                            om1 = (1.0 - e1) * M0;
                            dt_e = ev.dt;
                            de = 0;
                            off_e = false;
                        } else {
                            off_e = __any(de != 0);
                        }
                    }
                    // a run of equal steps that a chunk cuts keeps its dt
                    off = off_e;
                    const T dr = ev.dt - dt_r;
                    if ((fl & kEvSame) && __all(__builtin_fabs(dr) <= dt_near)) {
                        d = dr;
                        off = true;
                    } else {
                        dt_r = ev.dt;
                        d = 0;
                    }
                } else {
                    if (!(fl & kEvDt)) {
                        e1 = one_minus_exp(-ev.dt * invT1);
                        e2 = dev_exp<T>(-ev.dt * invT2);
                    }
                    dt_r = ev.dt;
                }
                const T Bz = field(ev, fl, RB > 0 && RB <= 2 ? cf : &scoef[MOTION ? e * kRow : 0]);
                if (fl & kEvRf) {
                    typename Cplx2<T>::Rot rot;
                    rot_make(rot, Bz, ev.rf_re, ev.rf_im, ev.rf2, gamma, dt_r, trig);
                    do {
                        rot_apply(rot, off, d, mxr, mxi, mz);
                        relax();
                    } while (more());
                } else {  // the precession leaves Mz alone
                    typename Cplx2<T>::Pre pre;
                    pre_make(pre, Bz, gamma, dt_r, trig);
                    do {
                        pre_apply(pre, off, d, mxr, mxi);
                        relax();
                    } while (more());
                }
            }
        }
    }
    if constexpr (CHAIN != kChainNone) {
        if (active) {  // the last block's end
            int code;
            if constexpr (CHAIN == kChainHost) code = chain.code[chain.n - 1];
            else code = marks[n_time] - 1;
            const int col = (code >> 1) - 1;
            if (col >= 0 && (CHAIN == kChainHost || col < n_store)) {
                store_xy[p + col * N] = make_float2((float)mxr, (float)mxi);
                store_z[p + col * N] = (float)mz;
            }
            if (code & 1) mxr = mxi = 0;
        }
    }
    if (!HISTORY && active) {
        mxy_fin[p] = make_double2((double)mxr, (double)mxi);
        mz_fin[p] = (double)mz;
    }
}

template <typename T>
__global__ void k_bloch_pack(int64_t N, const T *__restrict__ r0, const T *__restrict__ T1,
                             const T *__restrict__ T2, const T *__restrict__ dB, double *__restrict__ out)
{
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    out[n] = (double)r0[3 * n];
    out[N + n] = (double)r0[3 * n + 1];
    out[2 * N + n] = (double)r0[3 * n + 2];
    out[3 * N + n] = 1.0 / (double)T1[n];
    out[4 * N + n] = 1.0 / (double)T2[n];
    out[5 * N + n] = (double)dB[n];
}

__global__ void k_store_spoil(int64_t N, double2 *__restrict__ mxy, const double *__restrict__ mz,
                              float2 *__restrict__ mxy_store, float *__restrict__ mz_store, int64_t col,
                              int spoil)
{
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    const double2 v = mxy[n];
    if (col >= 0) {
        mxy_store[n + col * N] = make_float2((float)v.x, (float)v.y);
        mz_store[n + col * N] = (float)mz[n];
    }
    if (spoil) mxy[n] = make_double2(0.0, 0.0);
}

// Instantiated mode counts: the smallest that holds R.  The counts between run the
// next one's zero modes too, which costs less than the tests of a loop over them did:
// 1000 events, 300 000 nodes, FP64, 3 modes (as 5) 0.82 ms (1.63 before), 6 (as 10) 1.05
// (1.95), 11 (as 16) 1.39 (2.45); FP32 0.49 (1.07), 0.60 (1.28), 0.81 (1.64).  More
// counts would save up to a third of that and cost a kernel for each of the
// six forms.
#define FM_BLOCH_MODES(R, CALL)             \
    do {                                    \
        if ((R) <= 0) CALL(0);              \
        else if ((R) <= 1) CALL(1);         \
        else if ((R) <= 2) CALL(2);         \
        else if ((R) <= 5) CALL(5);         \
        else if ((R) <= 10) CALL(10);       \
        else CALL(16);                      \
    } while (0)

template <typename T>
static int launch_bloch(bool motion, bool history, int64_t N, int64_t n_time, const double *packed,
                        double M0, double gamma, const double *rf, const double *G, const double *dt,
                        const double *mxy_in, const double *mz_in, const float *modes, int R,
                        const double *mcoef, void *mxy_out, void *mz_out, hipStream_t st)
{
    using C2 = typename Cplx2<T>::type;
    const unsigned blocks = (unsigned)cdiv(N, kBlochThreads);
    C2 *mo = reinterpret_cast<C2 *>(mxy_out);
    T *zo = reinterpret_cast<T *>(mz_out);
    double2 *mf = reinterpret_cast<double2 *>(mxy_out);
    double *zf = reinterpret_cast<double *>(mz_out);
    const int RR = motion ? R : 0;
#define FM_BLOCH_ARGS packed, N, n_time, M0, gamma, rf, G, dt, mxy_in, mz_in, modes, RR, mcoef, mo, zo, mf, zf
#define FM_BLOCH_H(RB) k_bloch<T, RB, true><<<blocks, kBlochThreads, 0, st>>>(FM_BLOCH_ARGS)
#define FM_BLOCH_F(RB) k_bloch<T, RB, false><<<blocks, kBlochThreads, 0, st>>>(FM_BLOCH_ARGS)
    if (history) FM_BLOCH_MODES(RR, FM_BLOCH_H);
    else FM_BLOCH_MODES(RR, FM_BLOCH_F);
#undef FM_BLOCH_H
#undef FM_BLOCH_F
#undef FM_BLOCH_ARGS
    FM_LAUNCH_CHECK("k_bloch");
    return FM_OK;
}

template <typename T>
static void launch_bloch_chain(int64_t N, int64_t n_time, const double *packed, double M0, double gamma,
                               const double *rf, const double *G, const double *dt, const double *mxy_in,
                               const double *mz_in, double *mxy_out, double *mz_out, const ChainDesc &cd,
                               float2 *store_xy, float *store_z, hipStream_t st)
{
    const unsigned blocks = (unsigned)cdiv(N, kBlochThreads);
    k_bloch<T, 0, false, kChainHost><<<blocks, kBlochThreads, 0, st>>>(
        packed, N, n_time, M0, gamma, rf, G, dt, mxy_in, mz_in, nullptr, 0, nullptr, nullptr, nullptr,
        reinterpret_cast<double2 *>(mxy_out), mz_out, cd, store_xy, store_z);
}

template <typename T>
static void launch_bloch_marked(bool motion, int64_t N, int64_t capacity, const int64_t *n_events,
                                const double *packed, double M0, double gamma, const double *rf, const double *G,
                                const double *dt, const int32_t *marks, const float *modes, int R,
                                const double *mcoef, const double *mxy_in, const double *mz_in, double *mxy_out,
                                double *mz_out, float2 *store_xy, float *store_z, int64_t n_store, hipStream_t st)
{
    const unsigned blocks = (unsigned)cdiv(N, kBlochThreads);
    double2 *mf = reinterpret_cast<double2 *>(mxy_out);
    const int RR = motion ? R : 0;
#define FM_BLOCH_M(RB)                                                                                             \
    k_bloch<T, RB, false, kChainMarks><<<blocks, kBlochThreads, 0, st>>>(                                         \
        packed, N, capacity, M0, gamma, rf, G, dt, mxy_in, mz_in, modes, RR, mcoef, nullptr, nullptr, mf, mz_out, \
        NoChain{}, store_xy, store_z, marks, n_events, n_store)
    FM_BLOCH_MODES(RR, FM_BLOCH_M);
#undef FM_BLOCH_M
}

}  // namespace fm

using namespace fm;

extern "C" int fm_bloch_nodes_pack(int64_t n_pos, int dtype, const void *r0, const void *T1,
                                   const void *T2, const void *delta_B, double *packed, void *stream)
{
    FM_CHECK_ARG(n_pos >= 0, "negative n_pos");
    FM_CHECK_ARG(dtype == FM_DTYPE_F32 || dtype == FM_DTYPE_F64, "unknown dtype %d", dtype);
    if (n_pos == 0) return FM_OK;
    FM_CHECK_ARG(r0 && T1 && T2 && delta_B && packed, "NULL array");
    const unsigned blocks = (unsigned)cdiv(n_pos, 256);
    hipStream_t st = as_stream(stream);
    if (dtype == FM_DTYPE_F64)
        k_bloch_pack<double><<<blocks, 256, 0, st>>>(n_pos, (const double *)r0, (const double *)T1,
                                                    (const double *)T2, (const double *)delta_B, packed);
    else
        k_bloch_pack<float><<<blocks, 256, 0, st>>>(n_pos, (const float *)r0, (const float *)T1,
                                                   (const float *)T2, (const float *)delta_B, packed);
    FM_LAUNCH_CHECK("k_bloch_pack");
    return FM_OK;
}

extern "C" int fm_bloch_execute(int precision, int64_t n_pos, int64_t n_time, const double *packed,
                                double M0, double gamma, const double *rf, const double *G,
                                const double *dt, const double *mxy_in, const double *mz_in,
                                const float *modes, int n_modes, const double *motion_coef,
                                void *mxy_out, void *mz_out, int history, void *stream)
{
    FM_CHECK_ARG(precision == FM_PREC_F64 || precision == FM_PREC_F32,
                 "Bloch precision must be FM_PREC_F64 or FM_PREC_F32 (got %d)", precision);
    FM_CHECK_ARG(n_pos >= 0 && n_time >= 0, "negative size");
    FM_CHECK_ARG(n_modes >= 0 && n_modes <= kBlochMaxModes, "n_modes must be in [0, %d]", kBlochMaxModes);
    if (n_pos == 0) return FM_OK;
    FM_CHECK_ARG(packed && mxy_in && mz_in && mxy_out && mz_out, "NULL array");
    FM_CHECK_ARG(n_time == 0 || (rf && G && dt), "NULL event table");
    const bool motion = modes != nullptr && n_modes > 0;
    FM_CHECK_ARG(!motion || motion_coef != nullptr, "motion_coef is NULL");
    if (n_time == 0) {
        set_error("empty event table (n_time = 0)");
        return FM_ERR_ARG;
    }
    hipStream_t st = as_stream(stream);
    if (precision == FM_PREC_F64)
        return launch_bloch<double>(motion, history != 0, n_pos, n_time, packed, M0, gamma, rf, G, dt, mxy_in,
                                    mz_in, modes, n_modes, motion_coef, mxy_out, mz_out, st);
    return launch_bloch<float>(motion, history != 0, n_pos, n_time, packed, M0, gamma, rf, G, dt, mxy_in,
                               mz_in, modes, n_modes, motion_coef, mxy_out, mz_out, st);
}

extern "C" int fm_bloch_store_spoil(int64_t n_pos, double *mxy_state, const double *mz_state,
                                    void *mxy_store, void *mz_store, int64_t store_col, int spoil,
                                    void *stream)
{
    FM_CHECK_ARG(n_pos >= 0, "negative n_pos");
    if (n_pos == 0) return FM_OK;
    FM_CHECK_ARG(mxy_state && mz_state, "NULL state");
    FM_CHECK_ARG(store_col < 0 || (mxy_store && mz_store), "NULL store");
    k_store_spoil<<<(unsigned)cdiv(n_pos, 256), 256, 0, as_stream(stream)>>>(
        n_pos, reinterpret_cast<double2 *>(mxy_state), mz_state, reinterpret_cast<float2 *>(mxy_store),
        reinterpret_cast<float *>(mz_store), store_col, spoil);
    FM_LAUNCH_CHECK("k_store_spoil");
    return FM_OK;
}

extern "C" int fm_bloch_chain(int precision, int64_t n_pos, const double *packed, double M0, double gamma,
                              int64_t n_blocks, const int64_t *block_len, const int32_t *store_col,
                              const int32_t *spoil, const double *rf, const double *G, const double *dt,
                              const double *mxy_in, const double *mz_in, void *mxy_store, void *mz_store,
                              int64_t n_store, double *mxy_out, double *mz_out, void *stream)
{
    FM_CHECK_ARG(precision == FM_PREC_F64 || precision == FM_PREC_F32,
                 "Bloch precision must be FM_PREC_F64 or FM_PREC_F32 (got %d)", precision);
    FM_CHECK_ARG(n_pos >= 0 && n_blocks >= 0 && n_store >= 0, "negative size");
    if (n_pos == 0) return FM_OK;
    FM_CHECK_ARG(mxy_in && mz_in && mxy_out && mz_out, "NULL state");
    hipStream_t st = as_stream(stream);
    if (n_blocks == 0) {  // no block: the state passes through
        hipError_t e = hipSuccess;
        if (mxy_out != mxy_in)
            e = hipMemcpyAsync(mxy_out, mxy_in, 2 * sizeof(double) * (size_t)n_pos, hipMemcpyDeviceToDevice, st);
        if (e == hipSuccess && mz_out != mz_in)
            e = hipMemcpyAsync(mz_out, mz_in, sizeof(double) * (size_t)n_pos, hipMemcpyDeviceToDevice, st);
        if (e != hipSuccess) {
            set_error("fm_bloch_chain: %s", hipGetErrorString(e));
            return FM_ERR_HIP;
        }
        return FM_OK;
    }
    FM_CHECK_ARG(block_len && store_col && spoil, "NULL block description");
    FM_CHECK_ARG(packed && rf && G && dt, "NULL array");
    for (int64_t b = 0; b < n_blocks; ++b) {
        FM_CHECK_ARG(block_len[b] >= 1, "block %lld has no event", (long long)b);
        FM_CHECK_ARG(store_col[b] >= -1 && store_col[b] < n_store, "block %lld: store column %d outside [-1, %lld)",
                     (long long)b, store_col[b], (long long)n_store);
    }
    FM_CHECK_ARG(n_store == 0 || (mxy_store && mz_store), "NULL store");
    int64_t ev0 = 0;
    for (int64_t b0 = 0; b0 < n_blocks; b0 += kChainMaxBlocks) {
        const int nb = (int)std::min<int64_t>(kChainMaxBlocks, n_blocks - b0);
        ChainDesc cd;
        cd.n = nb;
        int64_t o = 0;
        for (int k = 0; k < nb; ++k) {
            cd.offset[k] = o;
            cd.code[k] = (spoil[b0 + k] ? 1 : 0) | ((store_col[b0 + k] + 1) << 1);
            o += block_len[b0 + k];
        }
        cd.offset[nb] = o;
        // later launches continue from the state the previous one left
        const double *xin = b0 == 0 ? mxy_in : mxy_out;
        const double *zin = b0 == 0 ? mz_in : mz_out;
        if (precision == FM_PREC_F64)
            launch_bloch_chain<double>(n_pos, o, packed, M0, gamma, rf + 2 * ev0, G + 3 * ev0, dt + ev0, xin, zin,
                                       mxy_out, mz_out, cd, reinterpret_cast<float2 *>(mxy_store),
                                       reinterpret_cast<float *>(mz_store), st);
        else
            launch_bloch_chain<float>(n_pos, o, packed, M0, gamma, rf + 2 * ev0, G + 3 * ev0, dt + ev0, xin, zin,
                                      mxy_out, mz_out, cd, reinterpret_cast<float2 *>(mxy_store),
                                      reinterpret_cast<float *>(mz_store), st);
        FM_LAUNCH_CHECK("k_bloch (chained blocks)");
        ev0 += o;
    }
    return FM_OK;
}

extern "C" int fm_bloch_chain_marked(int precision, int64_t n_pos, const double *packed, double M0, double gamma,
                                     const int64_t *n_events, int64_t capacity, const double *rf, const double *G,
                                     const double *dt, const int32_t *marks, const float *modes, int n_modes,
                                     const double *motion_coef, const double *mxy_in, const double *mz_in,
                                     void *mxy_store, void *mz_store, int64_t n_store, double *mxy_out,
                                     double *mz_out, void *stream)
{
    FM_CHECK_ARG(precision == FM_PREC_F64 || precision == FM_PREC_F32,
                 "Bloch precision must be FM_PREC_F64 or FM_PREC_F32 (got %d)", precision);
    FM_CHECK_ARG(n_pos >= 0 && capacity >= 1 && n_store >= 0, "negative size or capacity < 1");
    FM_CHECK_ARG(n_modes >= 0 && n_modes <= kBlochMaxModes, "n_modes must be in [0, %d]", kBlochMaxModes);
    if (n_pos == 0) return FM_OK;
    FM_CHECK_ARG(packed && n_events && rf && G && dt && marks, "NULL array");
    FM_CHECK_ARG(mxy_in && mz_in && mxy_out && mz_out, "NULL state");
    FM_CHECK_ARG(n_store == 0 || (mxy_store && mz_store), "NULL store");
    const bool motion = modes != nullptr && n_modes > 0;
    FM_CHECK_ARG(!motion || motion_coef != nullptr, "motion_coef is NULL");
    hipStream_t st = as_stream(stream);
    float2 *sx = reinterpret_cast<float2 *>(mxy_store);
    float *sz = reinterpret_cast<float *>(mz_store);
    if (precision == FM_PREC_F64)
        launch_bloch_marked<double>(motion, n_pos, capacity, n_events, packed, M0, gamma, rf, G, dt, marks, modes,
                                    n_modes, motion_coef, mxy_in, mz_in, mxy_out, mz_out, sx, sz, n_store, st);
    else
        launch_bloch_marked<float>(motion, n_pos, capacity, n_events, packed, M0, gamma, rf, G, dt, marks, modes,
                                   n_modes, motion_coef, mxy_in, mz_in, mxy_out, mz_out, sx, sz, n_store, st);
    FM_LAUNCH_CHECK("k_bloch (marked chain)");
    return FM_OK;
}
