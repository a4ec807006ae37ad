// Direct non-uniform k-space sum (any trajectory), FP64 and mixed forms.
//
//   S[s, v] = sum_n exp(i(-2 pi_f k_s . r_n + phi_n t_s)) exp(-t_s / T2_n) b[n, v]
//
// reference: cpp/feelmri/MRI.cpp:196-297 (static nodes), :38-159 (moving).
//
// Work decomposition.  A workgroup owns a tile of samples and one contiguous
// split of the nodes, which stream through LDS in chunks; all lanes read the
// same LDS node at the same time (broadcast).  Node splits write partial sums
// that a second kernel adds in a fixed order, so results do not depend on
// scheduling.  Four kernels:
//   * samples grouped by t (the reference's t cache): k_signal_groups
//     (signal_groups.hip), all moving nodes, and static nodes whose t-groups
//     are not tiny;
//   * samples in any order, per-sample t: k_signal_consec, static nodes;
//   * readouts linear in k and t: k_signal_runs and k_signal_runs_f64, static
//     nodes;
//   * whole lines linear in k and t: the per-line GEMM (signal_lines_bf16.hip).
//
// Phase handling.  u = k'.x is accumulated in FP64 in cycles (k' carries the
// reference's float-pi factor).  FP64 form: exact range reduction, FP64 sine
// and cosine.  Mixed form: fract(u) in [0, 1) (one instruction, exact),
// rounded to FP32 and fed to the hardware v_sin_f32 / v_cos_f32, which take
// revolutions; partial sums over a 256-node chunk are kept in FP32 and added
// into FP64.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <type_traits>
#include <unordered_map>

#include "signal_plan.h"

namespace fm {

template <bool MIXED>
struct CoefT;
template <>
struct CoefT<true> {
    using T = float;
};
template <>
struct CoefT<false> {
    using T = double;
};

// A node staged in LDS.
template <int VB, bool MIXED>
struct alignas(16) StagedNode {
    using CT = typename CoefT<MIXED>::T;
    double x, y, z;
    double dwc;  // phi/(2 pi), cycles/ms
    double r2;   // 1/T2, 1/ms
    CT b[2 * VB];
};

// Static nodes, tiles of up to 512 consecutive samples of any t (lane l takes
// samples offset + l and offset + l + 256): the decay and the off-resonance
// phase are formed per (node, sample).
template <int VB, bool MIXED>
__global__ __launch_bounds__(kDirectThreads) void k_signal_consec(
    const double *__restrict__ packed, int64_t N, int V, int v0, const double4 *__restrict__ ks,
    const SignalTile *__restrict__ tiles, int64_t nodes_per_split, double2 *__restrict__ dst, int64_t S,
    int write_final)
{
    using CT = typename CoefT<MIXED>::T;
    __shared__ StagedNode<VB, MIXED> snode[kDirectThreads];
    const int64_t split = blockIdx.y;
    const int64_t n_begin = split * nodes_per_split;
    const int64_t n_end = (n_begin + nodes_per_split < N) ? n_begin + nodes_per_split : N;
    const int tid = threadIdx.x;
    const SignalTile tl = tiles[blockIdx.x];

    int sid[kDirectSPL];
    bool valid[kDirectSPL];
    double kxs[kDirectSPL], kys[kDirectSPL], kzs[kDirectSPL], ts[kDirectSPL];
#pragma unroll
    for (int j = 0; j < kDirectSPL; ++j) {
        const int idx = tid + j * kDirectThreads;
        valid[j] = idx < tl.count;
        sid[j] = valid[j] ? tl.offset + idx : 0;
        const double4 k = ks[sid[j]];
        kxs[j] = k.x;
        kys[j] = k.y;
        kzs[j] = k.z;
        ts[j] = k.w;
    }
    double tot_re[kDirectSPL][VB], tot_im[kDirectSPL][VB];
#pragma unroll
    for (int j = 0; j < kDirectSPL; ++j)
#pragma unroll
        for (int v = 0; v < VB; ++v) tot_re[j][v] = tot_im[j][v] = 0.0;

    for (int64_t base = n_begin; base < n_end; base += kDirectThreads) {
        __syncthreads();  // previous chunk fully consumed
        {
            const int64_t n = base + tid;
            const bool ok = n < n_end;
            StagedNode<VB, MIXED> &nd = snode[tid];
            nd.x = ok ? packed[n] : 0.0;
            nd.y = ok ? packed[N + n] : 0.0;
            nd.z = ok ? packed[2 * N + n] : 0.0;
            nd.dwc = (ok ? packed[3 * N + n] : 0.0) * (1.0 / kTwoPi);
            nd.r2 = ok ? packed[4 * N + n] : 0.0;
#pragma unroll
            for (int v = 0; v < VB; ++v) {
                nd.b[2 * v] = ok ? (CT)packed[(int64_t)(5 + 2 * (v0 + v)) * N + n] : (CT)0;
                nd.b[2 * v + 1] = ok ? (CT)packed[(int64_t)(6 + 2 * (v0 + v)) * N + n] : (CT)0;
            }
        }
        __syncthreads();
        const int cnt = (n_end - base < kDirectThreads) ? (int)(n_end - base) : kDirectThreads;

        CT acc_re[kDirectSPL][VB], acc_im[kDirectSPL][VB];
#pragma unroll
        for (int j = 0; j < kDirectSPL; ++j)
#pragma unroll
            for (int v = 0; v < VB; ++v) acc_re[j][v] = acc_im[j][v] = (CT)0;
#pragma unroll 2
        for (int m = 0; m < cnt; ++m) {
            const StagedNode<VB, MIXED> &nd = snode[m];
#pragma unroll
            for (int j = 0; j < kDirectSPL; ++j) {
                // phase - phi t, in cycles
                const double u = fma(-nd.dwc, ts[j], fma(kxs[j], nd.x, fma(kys[j], nd.y, kzs[j] * nd.z)));
                CT cs, sn, d;
                if constexpr (MIXED) {
                    const float rf = turns_f32(u);
                    sn = __builtin_amdgcn_sinf(rf);
                    cs = __builtin_amdgcn_cosf(rf);
                    d = __builtin_amdgcn_exp2f((float)(-ts[j] * nd.r2 * 1.4426950408889634));
                } else {
                    sincos_cycles_f64(u, sn, cs);
                    d = exp(-ts[j] * nd.r2);
                }
                cs *= d;
                sn *= d;
                // e = cs - i sn ; acc += e * b
#pragma unroll
                for (int v = 0; v < VB; ++v) {
                    const CT cr = nd.b[2 * v], ci = nd.b[2 * v + 1];
                    acc_re[j][v] = fma(cs, cr, fma(sn, ci, acc_re[j][v]));
                    acc_im[j][v] = fma(cs, ci, fma(-sn, cr, acc_im[j][v]));
                }
            }
        }
#pragma unroll
        for (int j = 0; j < kDirectSPL; ++j)
#pragma unroll
            for (int v = 0; v < VB; ++v) {
                tot_re[j][v] += (double)acc_re[j][v];
                tot_im[j][v] += (double)acc_im[j][v];
            }
    }
#pragma unroll
    for (int j = 0; j < kDirectSPL; ++j) {
        if (!valid[j]) continue;
        const int64_t row = write_final ? (int64_t)sid[j] : split * S + sid[j];
#pragma unroll
        for (int v = 0; v < VB; ++v) dst[row * V + v0 + v] = make_double2(tot_re[j][v], tot_im[j][v]);
    }
}

// Mixed form, static nodes, readout runs.  Lane l of a workgroup owns run
// blockIdx.x * 256 + l (kRunLen samples of one readout line).  Per staged
// node the lane forms
//   e0 = exp(-t0/T2) exp(-2 pi i (k0.x - phi t0 / 2 pi))      (FP64 phase,
//        range-reduced, FP32 hardware sine/cosine)
//   q  = exp(-dt/T2) exp(-2 pi i (dk.x - phi dt / 2 pi))       (FP32)
// and accumulates e0 q^m c for m = 0 .. kRunLen-1, advancing e (one
// encoding: y = e c) by one complex multiply per sample.  FP32 partial sums over a 256-node chunk are
// added into FP64, as in k_signal_consec.
template <int VB>
struct alignas(16) RunNode {
    double x, y, z, dwc, r2;
    float xf, yf, zf, dwcf, r2f;
    float c[2 * VB];
};

// SHQ: the tile's runs share at most kRunSteps steps (dk, dt); the staging
// threads form each node's step factor once per step into LDS, and the lanes
// read it instead of forming their own.
constexpr int kSqStride = kDirectThreads + 1;  // LDS row of step factors (+1 entry)

template <int VB, bool SHQ = false>
__global__ __launch_bounds__(kDirectThreads) void k_signal_runs(
    const double *__restrict__ packed, int64_t N, int V, int v0, const RunDesc *__restrict__ runs,
    int64_t n_runs, int64_t stride, int64_t nodes_per_split, double2 *__restrict__ dst, int64_t S,
    int write_final, const double *__restrict__ run_steps = nullptr, const int32_t *__restrict__ run_nsteps = nullptr)
{
    __shared__ RunNode<VB> snode[kDirectThreads];
    extern __shared__ float2 sq32[];  // SHQ: (step, node) factors, rows of kSqStride
    const int nst = SHQ ? run_nsteps[blockIdx.x] : 0;
    const int64_t split = blockIdx.y;
    const int64_t n_begin = split * nodes_per_split;
    const int64_t n_end = (n_begin + nodes_per_split < N) ? n_begin + nodes_per_split : N;
    const int tid = threadIdx.x;
    const int64_t rid = (int64_t)blockIdx.x * kDirectThreads + tid;
    const bool valid = rid < n_runs;
    const RunDesc rd = runs[valid ? rid : 0];
    const float dkx = (float)rd.dkx, dky = (float)rd.dky, dkz = (float)rd.dkz, dtf = (float)rd.dt;

    const double *px = packed;
    const double *py = packed + N;
    const double *pz = packed + 2 * N;
    const double *pphi = packed + 3 * N;
    const double *pr2 = packed + 4 * N;
    const double *pb = packed + 5 * N;

    double tot_re[kRunLen][VB], tot_im[kRunLen][VB];
#pragma unroll
    for (int m = 0; m < kRunLen; ++m)
#pragma unroll
        for (int v = 0; v < VB; ++v) tot_re[m][v] = tot_im[m][v] = 0.0;

    for (int64_t base = n_begin; base < n_end; base += kDirectThreads) {
        __syncthreads();
        {
            const int64_t n = base + tid;
            RunNode<VB> nd;
            if (n < n_end) {
                nd.x = px[n];
                nd.y = py[n];
                nd.z = pz[n];
                nd.dwc = pphi[n] * (1.0 / kTwoPi);
                nd.r2 = pr2[n];
#pragma unroll
                for (int v = 0; v < VB; ++v) {
                    nd.c[2 * v] = (float)pb[(int64_t)(2 * (v0 + v)) * N + n];
                    nd.c[2 * v + 1] = (float)pb[(int64_t)(2 * (v0 + v) + 1) * N + n];
                }
            } else {
                nd.x = nd.y = nd.z = nd.dwc = nd.r2 = 0.0;
#pragma unroll
                for (int v = 0; v < 2 * VB; ++v) nd.c[v] = 0.0f;
            }
            nd.xf = (float)nd.x;
            nd.yf = (float)nd.y;
            nd.zf = (float)nd.z;
            nd.dwcf = (float)nd.dwc;
            nd.r2f = (float)nd.r2;
            snode[tid] = nd;
            if constexpr (SHQ) {
                for (int j = 0; j < nst; ++j) {
                    const double *st = &run_steps[((int64_t)blockIdx.x * kRunSteps + j) * 4];
                    const float sdkx = (float)st[0], sdky = (float)st[1], sdkz = (float)st[2], sdt = (float)st[3];
                    const float du = turns_f32(fmaf(sdkx, nd.xf, fmaf(sdky, nd.yf, fmaf(sdkz, nd.zf, -nd.dwcf * sdt))));
                    const float ds = __builtin_amdgcn_exp2f(-sdt * nd.r2f * 1.44269504f);
                    sq32[j * kSqStride + tid] = make_float2(ds * __builtin_amdgcn_cosf(du), -ds * __builtin_amdgcn_sinf(du));
                }
            }
        }
        __syncthreads();
        const int cnt = (n_end - base < kDirectThreads) ? (int)(n_end - base) : kDirectThreads;

        float acc_re[kRunLen][VB], acc_im[kRunLen][VB];
#pragma unroll
        for (int m = 0; m < kRunLen; ++m)
#pragma unroll
            for (int v = 0; v < VB; ++v) acc_re[m][v] = acc_im[m][v] = 0.0f;

        for (int i = 0; i < cnt; ++i) {
            const RunNode<VB> &nd = snode[i];
            // anchor: FP64 phase in cycles, range-reduced
            const double u = fma(rd.k0x, nd.x, fma(rd.k0y, nd.y, fma(rd.k0z, nd.z, -nd.dwc * rd.t0)));
            const float r = turns_f32(u);
            const float d0 = __builtin_amdgcn_exp2f((float)(-rd.t0 * nd.r2) * 1.44269504f);
            float er = d0 * __builtin_amdgcn_cosf(r);
            float ei = -d0 * __builtin_amdgcn_sinf(r);
            // step factor
            float qr, qi;
            if constexpr (SHQ) {
                const float2 q = sq32[rd.step * kSqStride + i];
                qr = q.x;
                qi = q.y;
            } else {
                const float du = turns_f32(fmaf(dkx, nd.xf, fmaf(dky, nd.yf, fmaf(dkz, nd.zf, -nd.dwcf * dtf))));
                const float ds = __builtin_amdgcn_exp2f(-dtf * nd.r2f * 1.44269504f);
                qr = ds * __builtin_amdgcn_cosf(du);
                qi = -ds * __builtin_amdgcn_sinf(du);
            }
            if constexpr (VB == 1) {
                // y = e c advances by q: one complex multiply and one complex
                // add per sample
                float yr = fmaf(er, nd.c[0], -ei * nd.c[1]);
                float yi = fmaf(er, nd.c[1], ei * nd.c[0]);
#pragma unroll
                for (int m = 0; m < kRunLen; ++m) {
                    acc_re[m][0] += yr;
                    acc_im[m][0] += yi;
                    const float nr = fmaf(yr, qr, -yi * qi);
                    yi = fmaf(yr, qi, yi * qr);
                    yr = nr;
                }
            } else {
#pragma unroll
                for (int m = 0; m < kRunLen; ++m) {
#pragma unroll
                    for (int v = 0; v < VB; ++v) {
                        const float cr = nd.c[2 * v], ci = nd.c[2 * v + 1];
                        acc_re[m][v] = fmaf(er, cr, fmaf(-ei, ci, acc_re[m][v]));
                        acc_im[m][v] = fmaf(er, ci, fmaf(ei, cr, acc_im[m][v]));
                    }
                    const float nr = er * qr - ei * qi;
                    ei = fmaf(er, qi, ei * qr);
                    er = nr;
                }
            }
        }
#pragma unroll
        for (int m = 0; m < kRunLen; ++m)
#pragma unroll
            for (int v = 0; v < VB; ++v) {
                tot_re[m][v] += (double)acc_re[m][v];
                tot_im[m][v] += (double)acc_im[m][v];
            }
    }

    if (!valid) return;
#pragma unroll
    for (int m = 0; m < kRunLen; ++m) {
        if (m >= rd.len) continue;
        const int64_t sid = (int64_t)rd.s0 + m * stride;
        const int64_t row = write_final ? sid : split * S + sid;
#pragma unroll
        for (int v = 0; v < VB; ++v) dst[row * V + v0 + v] = make_double2(tot_re[m][v], tot_im[m][v]);
    }
}

// FP64 form, static nodes, readout runs: the same recurrence in FP64
// (FP64 phase, sine and cosine for the anchor and the step, FP64 products and
// accumulators).  Taken only when every run is linear to 1e-14 of the
// largest |k'| and |t|; 15 FP64 complex products then leave the result
// ~1e-15 from the per-sample sum of MRI.cpp:260-288.  Bound by FP64 issue: 96
// instructions for a run's 16 samples, 35 for a sine and cosine, an exponential.
// 212 765 nodes, 150 x 188, radial: 3.52 ms (3.88 with the library's sincospi);
// 70 479 nodes, 140 x 118: 0.94 (1.07).
template <int VB>
struct alignas(16) RunNode64 {
    double x, y, z, dwc, r2, pad;
    double c[2 * VB];
};

template <int VB, bool SHQ = false>
__global__ __launch_bounds__(kDirectThreads) void k_signal_runs_f64(
    const double *__restrict__ packed, int64_t N, int V, int v0, const RunDesc *__restrict__ runs,
    int64_t n_runs, int64_t stride, int64_t nodes_per_split, double2 *__restrict__ dst, int64_t S,
    int write_final, const double *__restrict__ run_steps = nullptr, const int32_t *__restrict__ run_nsteps = nullptr)
{
    __shared__ RunNode64<VB> snode[kDirectThreads];
    extern __shared__ double2 sq64[];  // SHQ: (step, node) factors, rows of kSqStride
    const int nst = SHQ ? run_nsteps[blockIdx.x] : 0;
    const int64_t split = blockIdx.y;
    const int64_t n_begin = split * nodes_per_split;
    const int64_t n_end = (n_begin + nodes_per_split < N) ? n_begin + nodes_per_split : N;
    const int tid = threadIdx.x;
    const int64_t rid = (int64_t)blockIdx.x * kDirectThreads + tid;
    const bool valid = rid < n_runs;
    const RunDesc rd = runs[valid ? rid : 0];

    double tot_re[kRunLen][VB], tot_im[kRunLen][VB];
#pragma unroll
    for (int m = 0; m < kRunLen; ++m)
#pragma unroll
        for (int v = 0; v < VB; ++v) tot_re[m][v] = tot_im[m][v] = 0.0;

    for (int64_t base = n_begin; base < n_end; base += kDirectThreads) {
        __syncthreads();
        {
            const int64_t n = base + tid;
            RunNode64<VB> nd;
            nd.pad = 0.0;
            if (n < n_end) {
                nd.x = packed[n];
                nd.y = packed[N + n];
                nd.z = packed[2 * N + n];
                nd.dwc = packed[3 * N + n] * (1.0 / kTwoPi);
                nd.r2 = packed[4 * N + n];
#pragma unroll
                for (int v = 0; v < VB; ++v) {
                    nd.c[2 * v] = packed[(int64_t)(5 + 2 * (v0 + v)) * N + n];
                    nd.c[2 * v + 1] = packed[(int64_t)(6 + 2 * (v0 + v)) * N + n];
                }
            } else {
                nd.x = nd.y = nd.z = nd.dwc = nd.r2 = 0.0;
#pragma unroll
                for (int v = 0; v < 2 * VB; ++v) nd.c[v] = 0.0;
            }
            snode[tid] = nd;
            if constexpr (SHQ) {
                for (int j = 0; j < nst; ++j) {
                    const double *st = &run_steps[((int64_t)blockIdx.x * kRunSteps + j) * 4];
                    const double du = fma(st[0], nd.x, fma(st[1], nd.y, fma(st[2], nd.z, -nd.dwc * st[3])));
                    double qs, qc;
                    sincos_cycles_f64(du, qs, qc);
                    const double ds = exp(-st[3] * nd.r2);
                    sq64[j * kSqStride + tid] = make_double2(ds * qc, -ds * qs);
                }
            }
        }
        __syncthreads();
        const int cnt = (n_end - base < kDirectThreads) ? (int)(n_end - base) : kDirectThreads;
        for (int i = 0; i < cnt; ++i) {
            const RunNode64<VB> &nd = snode[i];
            // anchor: the first sample's term, as the per-sample sum forms it
            const double u = fma(rd.k0x, nd.x, fma(rd.k0y, nd.y, fma(rd.k0z, nd.z, -nd.dwc * rd.t0)));
            double sn, cs;
            sincos_cycles_f64(u, sn, cs);
            const double d0 = exp(-rd.t0 * nd.r2);
            double er = d0 * cs, ei = -d0 * sn;
            // step factor
            double qr, qi;
            if constexpr (SHQ) {
                const double2 q = sq64[rd.step * kSqStride + i];
                qr = q.x;
                qi = q.y;
            } else {
                const double du = fma(rd.dkx, nd.x, fma(rd.dky, nd.y, fma(rd.dkz, nd.z, -nd.dwc * rd.dt)));
                double qs, qc;
                sincos_cycles_f64(du, qs, qc);
                const double ds = exp(-rd.dt * nd.r2);
                qr = ds * qc;
                qi = -ds * qs;
            }
            if constexpr (VB == 1) {
                // y = e c advances by q, as in k_signal_runs
                double yr = fma(er, nd.c[0], -ei * nd.c[1]);
                double yi = fma(er, nd.c[1], ei * nd.c[0]);
#pragma unroll
                for (int m = 0; m < kRunLen; ++m) {
                    tot_re[m][0] += yr;
                    tot_im[m][0] += yi;
                    const double nr = fma(yr, qr, -yi * qi);
                    yi = fma(yr, qi, yi * qr);
                    yr = nr;
                }
            } else {
#pragma unroll
                for (int m = 0; m < kRunLen; ++m) {
#pragma unroll
                    for (int v = 0; v < VB; ++v) {
                        const double cr = nd.c[2 * v], ci = nd.c[2 * v + 1];
                        tot_re[m][v] = fma(er, cr, fma(-ei, ci, tot_re[m][v]));
                        tot_im[m][v] = fma(er, ci, fma(ei, cr, tot_im[m][v]));
                    }
                    const double nr = er * qr - ei * qi;
                    ei = fma(er, qi, ei * qr);
                    er = nr;
                }
            }
        }
    }

    if (!valid) return;
#pragma unroll
    for (int m = 0; m < kRunLen; ++m) {
        if (m >= rd.len) continue;
        const int64_t sid = (int64_t)rd.s0 + m * stride;
        const int64_t row = write_final ? sid : split * S + sid;
#pragma unroll
        for (int v = 0; v < VB; ++v) dst[row * V + v0 + v] = make_double2(tot_re[m][v], tot_im[m][v]);
    }
}

// out[s, v] = sum over splits, in split order.
template <int G>
__global__ __launch_bounds__(256) void k_reduce_splits(const double2 *__restrict__ part, int64_t n_splits, int64_t SV,
                                                       double2 *__restrict__ out)
{
    const int64_t i = reduce_output<G>();
    const double2 sum = reduce_sum<G>(part + i, SV, n_splits, i < SV);
    if (i < SV && threadIdx.x < 256 / G) out[i] = sum;
}

template <typename T>
__global__ void k_nodes_pack(int64_t N, int V, const T *__restrict__ r0, const T *__restrict__ phi,
                             const T *__restrict__ T2, const T *__restrict__ mxy,
                             const double *__restrict__ w, double *__restrict__ out)
{
    const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    out[n] = (double)r0[3 * n];
    out[N + n] = (double)r0[3 * n + 1];
    out[2 * N + n] = (double)r0[3 * n + 2];
    out[3 * N + n] = (double)phi[n];
    out[4 * N + n] = 1.0 / (double)T2[n];
    const double ww = w ? w[n] : 1.0;
    for (int v = 0; v < V; ++v) {
        out[(int64_t)(5 + 2 * v) * N + n] = ww * (double)mxy[2 * (n * V + v)];
        out[(int64_t)(6 + 2 * v) * N + n] = ww * (double)mxy[2 * (n * V + v) + 1];
    }
}

// Sum over the 16 lanes of a row group by a fixed butterfly (lane ^ 8, 4, 2,
// 1; a rotation by 8, 4, 2, 1 reaches the same value, as lanes that far apart
// hold equal sums by then).
__device__ inline double sum_group16(double v)
{
    auto step = [&](auto ctrl) {
        const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
        const unsigned lo = __builtin_amdgcn_update_dpp(0u, (unsigned)b, decltype(ctrl)::value, 0xf, 0xf, true);
        const unsigned hi = __builtin_amdgcn_update_dpp(0u, (unsigned)(b >> 32), decltype(ctrl)::value, 0xf, 0xf, true);
        v += __builtin_bit_cast(double, (unsigned long long)hi << 32 | lo);
    };
    step(std::integral_constant<int, 0x128>{});  // row_ror:8
    step(std::integral_constant<int, 0x124>{});
    step(std::integral_constant<int, 0x122>{});
    step(std::integral_constant<int, 0x121>{});
    return v;
}

// CSR SpMV, 16 lanes per row (P1 mass rows hold ~15 entries on tetrahedral
// meshes): lane j of a row's group adds the row's terms j, j + 16, ... for VB
// encodings at a time (the row's values and column indices read once per pass,
// coalesced across the group), then the group sums its lanes in a fixed
// butterfly, so a result does not depend on the launch.  Rows past the last
// one work on it and write nothing.
// Bound by the latency of three dependent loads (row, entry, x).  The rows of a
// workgroup's XCD are one range, whose part of x stays in that L2.  215 940 rows
// of 15, two encodings: 16.6 us, 4 TB/s (38.7 us with sums for four encodings
// through LDS and the rows dealt over the XCDs).  The x of all encodings is loaded before
// it is used: 200 000 rows of 40, four encodings 205 -> 139 us.
// ROWS: rows of a lane group, whose loads overlap; csr_two_rows tells when that is two.
template <int VB, int ROWS>
__global__ __launch_bounds__(256) void k_csr_spmv_c128(int64_t n_rows, int V, const int64_t *__restrict__ indptr,
                                                       const int64_t *__restrict__ indices,
                                                       const double *__restrict__ data,
                                                       const double2 *__restrict__ x, double2 *__restrict__ y)
{
    const int64_t row = xcd_range(cdiv(n_rows, 16 * ROWS)) * 16 * ROWS + threadIdx.x / 16;
    const int j = threadIdx.x % 16;
    int64_t k0[ROWS], k1[ROWS], longest = 0;
#pragma unroll
    for (int q = 0; q < ROWS; ++q) {
        const int64_t r = row + 16 * q < n_rows ? row + 16 * q : n_rows - 1;
        k0[q] = indptr[r] + j;
        k1[q] = indptr[r + 1];
        longest = k1[q] - k0[q] > longest ? k1[q] - k0[q] : longest;
    }
    for (int v0 = 0; v0 < V; v0 += VB) {
        double re[ROWS][VB], im[ROWS][VB];
#pragma unroll
        for (int q = 0; q < ROWS; ++q)
#pragma unroll
            for (int u = 0; u < VB; ++u) re[q][u] = im[q][u] = 0.0;
        for (int64_t t = 0; t < longest; t += 16) {
            double a[ROWS];
            int64_t c[ROWS];
            double2 xv[ROWS][VB];  // loaded together
#pragma unroll
            for (int q = 0; q < ROWS; ++q) {
                c[q] = -1;
                if (ROWS == 1 || k0[q] + t < k1[q]) {
                    a[q] = data[k0[q] + t];
                    c[q] = indices[k0[q] + t];
                }
            }
#pragma unroll
            for (int q = 0; q < ROWS; ++q)
#pragma unroll
                for (int u = 0; u < VB; ++u)
                    if ((ROWS == 1 || c[q] >= 0) && v0 + u < V) xv[q][u] = x[c[q] * V + v0 + u];
                    else xv[q][u] = make_double2(0.0, 0.0);
#pragma unroll
            for (int q = 0; q < ROWS; ++q)
                if (ROWS == 1 || c[q] >= 0)
#pragma unroll
                    for (int u = 0; u < VB; ++u) {
                        re[q][u] = fma(a[q], xv[q][u].x, re[q][u]);
                        im[q][u] = fma(a[q], xv[q][u].y, im[q][u]);
                    }
        }
#pragma unroll
        for (int q = 0; q < ROWS; ++q)
#pragma unroll
            for (int u = 0; u < VB; ++u) {
                const double sr = sum_group16(re[q][u]), si = sum_group16(im[q][u]);
                if (j == 0 && v0 + u < V && row + 16 * q < n_rows)
                    y[(row + 16 * q) * V + v0 + u] = make_double2(sr, si);
            }
    }
}

// Two rows a lane group: up to two encodings (with more a lane has loads enough in
// flight) and two rounds of the workgroups the device holds (8 a CU).  One encoding, 512 000 mesh
// rows: 30.6 -> 23.7 us, 216 000: 14.0 -> 11.8, 200 000 rows of 40: 28.6 -> 23.5; two
// encodings: 36.1 -> 33.6, 17.1 -> 15.6, 32.1 -> 31.0.  Four: 57.3 -> 54.4, but 125 000 rows 15.6
// -> 16.1.  Fewer rows leave CUs idle (27 000, two encodings: 3.5 -> 3.7 us; 2000 rows of
// 500, one: 8.5 -> 15.4).
static bool csr_two_rows(int64_t n_rows, int n_enc)
{
    return n_enc <= 2 && cdiv(n_rows, 32) >= (int64_t)16 * device_cu_count();
}

// ---------------------------------------------------------------------------
// Launch helpers
// ---------------------------------------------------------------------------
struct DirectLaunch {
    int64_t n_splits;
    int64_t nodes_per_split;
};

// Tilings of the direct path: 0 consecutive, 1 t-grouped, 2 readout runs.
static int64_t direct_tiles(const fm_signal_plan *p, int tiling)
{
    if (tiling == 2) return cdiv(p->n_runs, kDirectThreads);
    return tiling == 1 ? p->n_tiles_pairs : p->n_tiles_consec;
}

static DirectLaunch direct_launch_shape(const fm_signal_plan *p, int64_t N, int tiling)
{
    // Aim for ~8 workgroups per CU over the whole grid; keep >= 2048 nodes
    // per split so the staging cost stays amortised.
    const int64_t target = 8 * (int64_t)device_cu_count();
    const int64_t nt = direct_tiles(p, tiling);
    int64_t splits = cdiv(target, nt > 0 ? nt : 1);
    const int64_t max_splits = cdiv(N, 2048);
    if (splits > max_splits) splits = max_splits;
    if (splits < 1) splits = 1;
    int64_t nps = cdiv(N, splits);
    nps = cdiv(nps, kDirectThreads) * kDirectThreads;
    splits = cdiv(N, nps);
    return {splits, nps};
}

// Workspace that the t-grouped tiles may take for node splits beyond the least
// (below the array of fm_signal_execute_noalloc).
constexpr size_t kFineSplitBytes = size_t(32) << 20;

// The t-grouped tiles' splits.  The least, which the workspace has to hold: whole
// rounds of the workgroups the device holds, of at least 2048 nodes, no more
// splits than the consecutive tiles (the fewest tiles) would take.  Where that
// leaves the device idle (few tiles, small meshes) the splits are as fine as 256
// nodes, as far as kFineSplitBytes and the workspace at hand go: tiles of many
// groups are few, and one workgroup alone on a CU waits for its loads.
// Mixed form, 20 011 nodes: 40 x 31 moving, 32 modes: 1.04 -> 0.13 ms (one group to
// a slot, more tiles: 0.24); 200 x 16, 4 encodings: 0.52 -> 0.11 ms (0.31 with per-sample
// t); 64 x 64 of one t: 0.16 -> 0.05 ms.  200 003 nodes, 200 x 17: 0.52 -> 0.40 ms.
static DirectLaunch groups_launch_shape(const fm_signal_plan *p, bool mixed, bool motion, int64_t N, int V, int R,
                                        size_t ws_bytes)
{
    const int64_t most = direct_launch_shape(p, N, 0).n_splits;
    const int64_t nt = p->n_tiles_pairs;
    const int64_t capacity = (int64_t)groups_blocks_per_cu(p, mixed, motion, V, R) * device_cu_count();
    const size_t per_split = (size_t)p->n_samples * (size_t)V * sizeof(double2);
    auto shape = [&](int64_t s_max) -> DirectLaunch {
        const int64_t splits = balanced_splits(N, kDirectThreads, nt, cdiv(capacity, nt), capacity, s_max);
        const int64_t nps = cdiv(cdiv(N, splits), kDirectThreads) * kDirectThreads;
        return {cdiv(N, nps), nps};
    };
    const DirectLaunch least = shape(std::min(most, cdiv(N, 2048)));
    const int64_t fits = (int64_t)(std::min(ws_bytes, kFineSplitBytes) / per_split);
    if (fits <= least.n_splits) return least;
    return shape(std::min(cdiv(N, kDirectThreads), fits));
}

// Workspace of the t-grouped tiles with the finest splits they may take
// (balanced_splits takes at most twice its least count).
static size_t groups_fine_workspace(const fm_signal_plan *p, int64_t N, int V)
{
    const size_t per_split = (size_t)p->n_samples * (size_t)V * sizeof(double2);
    const int64_t most = 2 * cdiv(8 * (int64_t)device_cu_count(), std::max<int64_t>(p->n_tiles_pairs, 1));
    const int64_t fits = (int64_t)(kFineSplitBytes / per_split);
    const int64_t splits = std::min({cdiv(N, kDirectThreads), most, fits});
    return splits > 1 ? (size_t)splits * per_split : 0;
}

template <bool MIXED>
static void launch_consec(const fm_signal_plan *p, dim3 grid, const double *packed, int64_t N, int V, int v0, int vb,
                          int64_t nps, double2 *dst, int write_final, hipStream_t st)
{
#define FM_LD(VBV)                                                                                                  \
    k_signal_consec<VBV, MIXED><<<grid, kDirectThreads, 0, st>>>(packed, N, V, v0, p->d_ks, p->d_tiles_consec, nps, \
                                                                 dst, p->n_samples, write_final)
    switch (vb) {
    case 1: FM_LD(1); break;
    case 2: FM_LD(2); break;
    case 3: FM_LD(3); break;
    default: FM_LD(4); break;
    }
#undef FM_LD
}

static size_t direct_workspace(const fm_signal_plan *p, int64_t N, int V)
{
    if (N <= 0 || p->n_samples == 0) return 0;
    // the largest of the tilings' needs (the t-grouped tiles' least is no more
    // than the consecutive ones') and of the per-line GEMM's partial samples
    // (one encoding at a time)
    size_t need = std::max(lines_workspace(p, N), groups_fine_workspace(p, N, V));
    for (int g = 0; g < 3; g += 2) {
        if (g == 2 && p->n_runs == 0) continue;
        const DirectLaunch L = direct_launch_shape(p, N, g);
        if (L.n_splits > 1)
            need = std::max(need, (size_t)L.n_splits * (size_t)p->n_samples * (size_t)V * sizeof(double2));
    }
    return need;
}

// The direct kernels' route.  Mixed form, static nodes, whole linear lines: the
// per-line GEMM.  Positions depend on t, so moving nodes always take the t-grouped
// tiles; static nodes take the readout runs when the plan has them (the FP64
// form only when they are linear to 1e-14).
static int direct_route(const fm_signal_plan *p, int precision, int64_t N, bool motion)
{
    const bool mixed = precision != FM_PREC_F64;
    if (!motion && mixed && lines_usable(p, N)) return FM_ROUTE_LINES;
    if (!motion && p->n_runs > 0 && (mixed || p->runs_exact)) return FM_ROUTE_RUNS;
    if (!motion && !p->prefer_grouped) return FM_ROUTE_CONSECUTIVE;
    return groups_in_pairs(p, mixed) ? FM_ROUTE_GROUP_PAIRS : FM_ROUTE_GROUPS;
}

static DirectLaunch direct_launch(const fm_signal_plan *p, int route, int precision, int64_t N, int V, int R,
                                  size_t ws_bytes)
{
    if (route == FM_ROUTE_RUNS) return direct_launch_shape(p, N, 2);
    if (route == FM_ROUTE_CONSECUTIVE) return direct_launch_shape(p, N, 0);
    return groups_launch_shape(p, precision != FM_PREC_F64, R > 0, N, V, R, ws_bytes);
}

static int direct_execute(const fm_signal_plan *p, int precision, int64_t N, int V,
                          const double *packed, const float *modes, int R, const double *mcoef,
                          void *ws, size_t ws_bytes, double *out, hipStream_t st)
{
    const int64_t S = p->n_samples;
    if (S == 0) return FM_OK;
    if (N == 0) {
        return zero_f64_async(out, 2 * S * V, st);
    }
    const bool motion = modes != nullptr && R > 0;
    const int route = direct_route(p, precision, N, motion);
    if (route == FM_ROUTE_LINES) return lines_execute(p, N, V, packed, ws, ws_bytes, out, st);
    const bool use_runs = route == FM_ROUTE_RUNS, grouped = !use_runs && route != FM_ROUTE_CONSECUTIVE;
    const int tiling = use_runs ? 2 : (grouped ? 1 : 0);
    const DirectLaunch L = direct_launch(p, route, precision, N, V, motion ? R : 0, ws ? ws_bytes : 0);
    const size_t need = L.n_splits > 1 ? (size_t)L.n_splits * (size_t)S * (size_t)V * sizeof(double2) : 0;
    if (need > ws_bytes) {
        set_error("signal workspace too small: need %zu bytes, got %zu", need, ws_bytes);
        return FM_ERR_WORKSPACE;
    }
    double2 *dst = L.n_splits > 1 ? reinterpret_cast<double2 *>(ws) : reinterpret_cast<double2 *>(out);
    const int write_final = L.n_splits > 1 ? 0 : 1;
    dim3 grid((unsigned)direct_tiles(p, tiling), (unsigned)L.n_splits);
    plan_timing_start(p, st);
    if (use_runs) {
        // one encoding per launch: 16 samples x 1 encoding of accumulators
        // keeps the kernel at ~130 VGPRs (3 waves per SIMD)
        for (int v0 = 0; v0 < V; ++v0) {
            if (precision == FM_PREC_F64)
                if (p->run_steps > 0)
                    k_signal_runs_f64<1, true><<<grid, kDirectThreads, sizeof(double2) * kSqStride * p->run_steps, st>>>(
                        packed, N, V, v0, p->d_runs, p->n_runs, p->run_stride, L.nodes_per_split, dst, S, write_final,
                        p->d_run_steps, p->d_run_nsteps);
                else
                    k_signal_runs_f64<1><<<grid, kDirectThreads, 0, st>>>(packed, N, V, v0, p->d_runs, p->n_runs,
                                                                          p->run_stride, L.nodes_per_split, dst, S,
                                                                          write_final);
            else if (p->run_steps > 0)
                k_signal_runs<1, true><<<grid, kDirectThreads, sizeof(float2) * kSqStride * p->run_steps, st>>>(
                    packed, N, V, v0, p->d_runs, p->n_runs, p->run_stride, L.nodes_per_split, dst, S, write_final,
                    p->d_run_steps, p->d_run_nsteps);
            else
                k_signal_runs<1><<<grid, kDirectThreads, 0, st>>>(packed, N, V, v0, p->d_runs, p->n_runs,
                                                                  p->run_stride, L.nodes_per_split, dst, S,
                                                                  write_final);
            FM_LAUNCH_CHECK("k_signal_runs");
        }
    }
    for (int v0 = 0; v0 < V && !use_runs; v0 += kMaxVB) {
        const int vb = (V - v0 < kMaxVB) ? V - v0 : kMaxVB;
        if (grouped) {
            const int rc = groups_launch(p, precision != FM_PREC_F64, motion, N, V, v0, vb, packed, modes, R, mcoef,
                                         L.n_splits, L.nodes_per_split, dst, write_final, st);
            if (rc != FM_OK) return rc;
            continue;
        }
        if (precision == FM_PREC_F64)
            launch_consec<false>(p, grid, packed, N, V, v0, vb, L.nodes_per_split, dst, write_final, st);
        else
            launch_consec<true>(p, grid, packed, N, V, v0, vb, L.nodes_per_split, dst, write_final, st);
        FM_LAUNCH_CHECK("k_signal_consec");
    }
    plan_timing_stop(p, st);
    if (L.n_splits > 1) {
        const int64_t SV = S * V;
        const int G = reduce_group(SV, L.n_splits);
        auto *reduce = G == 8 ? k_reduce_splits<8> : k_reduce_splits<1>;
        reduce<<<reduce_grid(SV, G), 256, 0, st>>>(dst, L.n_splits, SV, reinterpret_cast<double2 *>(out));
        FM_LAUNCH_CHECK("k_reduce_splits");
    }
    return FM_OK;
}

}  // namespace fm

using namespace fm;

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
namespace fm {
// Host tables of a plan before upload.
struct PlanHost {
    std::vector<SignalTile> tiles_c;
    std::vector<int2> pairs;             // per lane: samples
    std::vector<uint8_t> lane_group;     // per lane: group of its tile
    std::vector<int4> tiles_p;
    std::vector<double4> ks;
    std::vector<RunDesc> runs;
    std::vector<RunDesc> lines;       // whole linear lines (per-line GEMM)
    std::vector<double> run_steps;    // (tiles, kRunSteps, 4)
    std::vector<int32_t> run_nsteps;  // (tiles)
};

// Host analysis of a trajectory: distinct-t groups, Cartesian
// factorisation, tilings, readout runs.  No device calls.
static int plan_analyse(fm_signal_plan *p, const double *kx, const double *ky, const double *kz,
                        const double *t, int method, PlanHost &h)
{
    const int64_t S = p->n_samples, n_meas = p->n_meas, n_lines = p->n_lines, n_kz = p->n_kz;
    // distinct t in first-appearance order (equal values share decay/phase)
    std::unordered_map<uint64_t, int32_t> gid;
    p->sample_group.resize((size_t)S);
    for (int64_t s = 0; s < S; ++s) {
        double tv = t[s];
        if (tv == 0.0) tv = 0.0;  // -0.0 and 0.0 compare equal in the reference's cache
        uint64_t key;
        std::memcpy(&key, &tv, sizeof key);
        auto it = gid.find(key);
        int32_t g;
        if (it == gid.end()) {
            g = (int32_t)p->tg_t.size();
            gid.emplace(key, g);
            p->tg_t.push_back(t[s]);
        } else {
            g = it->second;
        }
        p->sample_group[(size_t)s] = g;
    }
    p->n_tgroups = (int64_t)p->tg_t.size();

    if (method != FM_METHOD_DIRECT && S > 0) {
        const bool ok = cartesian_analyse(p, kx, ky, kz, t);
        if (method == FM_METHOD_CARTESIAN && !ok) {
            set_error("k-space sampling does not factorise as a Cartesian grid "
                      "(k not additively separable per axis, or t not a function of the readout index)");
            return FM_ERR_UNSUPPORTED;
        }
        p->method = ok ? FM_METHOD_CARTESIAN : FM_METHOD_DIRECT;
    }

    std::vector<double4> &ks = h.ks;
    ks.resize((size_t)S);
    for (int64_t s = 0; s < S; ++s)
        ks[(size_t)s] = make_double4(kx[s] * kPiFOverPi, ky[s] * kPiFOverPi, kz[s] * kPiFOverPi, t[s]);
    p->planar = 1;
    for (int64_t s = 0; s < S && p->planar; ++s) p->planar = ks[(size_t)s].z == 0.0;

    // Tilings.  Consecutive: plain runs of samples, per-sample t.  Grouped:
    // lanes of two samples of one t-group, in the order of the groups, cut
    // into tiles of 256 lanes and at most kGroupCap groups, so the t-dependent
    // node factors are staged once per tile and group.
    for (int64_t o = 0; o < S; o += kDirectTile)
        h.tiles_c.push_back({(int32_t)o, (int32_t)std::min<int64_t>(kDirectTile, S - o)});
    p->n_tiles_consec = (int64_t)h.tiles_c.size();
    std::vector<int64_t> first((size_t)p->n_tgroups + 1, 0);  // group g: perm[first[g] .. first[g + 1])
    std::vector<int32_t> perm((size_t)S);
    {
        for (int64_t s = 0; s < S; ++s) first[(size_t)p->sample_group[(size_t)s] + 1]++;
        for (int64_t g = 0; g < p->n_tgroups; ++g) first[(size_t)g + 1] += first[(size_t)g];
        std::vector<int64_t> fill(first.begin(), first.end() - 1);
        for (int64_t s = 0; s < S; ++s) perm[(size_t)fill[(size_t)p->sample_group[(size_t)s]]++] = (int32_t)s;
    }
    const double avg_group = p->n_tgroups ? (double)S / (double)p->n_tgroups : 0.0;
    p->prefer_grouped = avg_group >= kGroupMin;

    // Pairs and runs are found to a tolerance taken from the largest |k'| and
    // |t|.  Where a coordinate is infinite or NaN nothing is: every sample is
    // then summed by itself, and only those coordinates' samples are not finite.
    double kmax = 0.0, tmax = 0.0;
    bool finite = true;
    for (int64_t s = 0; s < S; ++s) {
        const double4 v = ks[(size_t)s];
        kmax = std::max({kmax, std::fabs(v.x), std::fabs(v.y), std::fabs(v.z)});
        tmax = std::max(tmax, std::fabs(v.w));
        finite = finite && std::isfinite(v.x) && std::isfinite(v.y) && std::isfinite(v.z) && std::isfinite(v.w);
    }

    // Conjugate pairs: in every t-group pair each sample with one whose k' is
    // its negative, to 1e-12 of the largest |k'| (an O(g^2) search per group
    // of at most 128 samples, given up at the first sample without a partner;
    // k' = 0 pairs with another k' = 0).  All groups or none.
    std::vector<int32_t> mate;  // partner of perm[i] for the first of each pair, else -1
    double worst = 0.0;
    p->pairs_conj = S > 0 && finite;
    {
        const double tol = 1e-12 * (kmax > 0.0 ? kmax : 1.0);
        std::vector<char> used;
        for (int64_t g = 0; g < p->n_tgroups && p->pairs_conj; ++g) {
            const int64_t n = first[(size_t)g + 1] - first[(size_t)g];
            const int32_t *mem = &perm[(size_t)first[(size_t)g]];
            p->pairs_conj = n % 2 == 0 && n <= 128;
            if (!p->pairs_conj) break;
            if (mate.empty()) mate.assign((size_t)S, -1);
            used.assign((size_t)n, 0);
            auto apart = [&](int64_t i, int64_t j) {
                const double4 u = ks[(size_t)mem[i]], v = ks[(size_t)mem[j]];
                return std::fabs(u.x + v.x) + std::fabs(u.y + v.y) + std::fabs(u.z + v.z);
            };
            for (int64_t a = 0; a < n && p->pairs_conj; ++a) {
                if (used[(size_t)a]) continue;
                int64_t best = -1;
                double bd = 0.0;
                // the sample half the group on (interleaves in order) at once
                // where it is exact, else the nearest of the rest
                const int64_t h = a + n / 2;
                const bool opposite = h < n && !used[(size_t)h] && apart(a, h) <= 4e-15 * kmax;
                if (opposite) {
                    best = h;
                    bd = apart(a, h);
                }
                for (int64_t b = a + 1; b < n && !opposite; ++b) {
                    if (used[(size_t)b]) continue;
                    const double d = apart(a, b);
                    if (d <= tol && (best < 0 || d < bd)) {
                        best = b;
                        bd = d;
                    }
                }
                if (best < 0) {
                    p->pairs_conj = false;
                    break;
                }
                used[(size_t)a] = used[(size_t)best] = 1;
                mate[(size_t)(first[(size_t)g] + a)] = mem[best];
                worst = std::max(worst, bd);
            }
        }
    }
    p->pairs_exact = p->pairs_conj && worst <= 4e-15 * kmax;
    // lanes and tiles
    {
        int32_t lane0 = 0, group0 = 0;
        h.pairs.reserve((size_t)((S + p->n_tgroups) / 2));
        h.lane_group.reserve((size_t)((S + p->n_tgroups) / 2));
        auto close = [&](int64_t g_end) {  // the tile of groups [group0, g_end)
            const int32_t n = (int32_t)h.pairs.size() - lane0;
            if (n == 0) return;
            h.tiles_p.push_back(make_int4(lane0, n, group0, (int32_t)g_end - group0));
            p->groups_per_tile = std::max(p->groups_per_tile, (int)(g_end - group0));
            lane0 = (int32_t)h.pairs.size();
        };
        for (int64_t g = 0; g < p->n_tgroups; ++g) {
            const int64_t n = first[(size_t)g + 1] - first[(size_t)g], o = first[(size_t)g], half = (n + 1) / 2;
            if (g - group0 >= kGroupCap) {
                close(g);
                group0 = (int32_t)g;
            }
            int64_t l = 0;  // lanes of the group so far
            for (int64_t a = 0; l < half; ++a) {
                int32_t s0 = perm[(size_t)(o + a)], s1 = a + half < n ? perm[(size_t)(o + a + half)] : -1;
                if (p->pairs_conj) {
                    s1 = mate[(size_t)(o + a)];
                    if (s1 < 0) continue;  // the second of a pair
                }
                if ((int32_t)h.pairs.size() - lane0 == kDirectThreads) {
                    close(l > 0 ? g + 1 : g);
                    group0 = (int32_t)g;
                }
                h.pairs.push_back(make_int2(s0, s1));
                h.lane_group.push_back((uint8_t)(g - group0));
                ++l;
            }
        }
        close(p->n_tgroups);
        p->n_tiles_pairs = (int64_t)h.tiles_p.size();
    }
    // facts reported by the analysis: slots of up to 256 samples of one group, two to a tile;
    // groups of one size of 32, 64 or 128 samples and how many fill 256 lanes,
    // singly and as conjugate pairs
    {
        int64_t slots = 0;
        const int64_t g0 = p->n_tgroups > 0 ? first[1] : 0;
        bool uniform = g0 == 32 || g0 == 64 || g0 == 128;
        for (int64_t g = 0; g < p->n_tgroups; ++g) {
            const int64_t n = first[(size_t)g + 1] - first[(size_t)g];
            slots += cdiv(n, kDirectThreads);
            uniform = uniform && n == g0;
        }
        p->n_tiles_grouped = cdiv(slots, 2);
        p->group_pack = uniform ? (int)(kDirectThreads / g0) : 1;
        p->conj_pack = uniform && p->pairs_conj ? (int)(2 * kDirectThreads / g0) : 1;
    }

    // Readout runs: kRunLen consecutive readout samples of a line (stride
    // lines * kz in the sample index) whose k' and t are linear in the
    // readout index to 1e-12 of the largest |k'| / |t|.  All runs or none.
    std::vector<RunDesc> &runs = h.runs;
    if (n_meas >= 2 && S > 0 && finite) {
        const int64_t stride = n_lines * n_kz;
        const double tolk = 1e-12 * (kmax > 0.0 ? kmax : 1.0), tolt = 1e-12 * (tmax > 0.0 ? tmax : 1.0);
        bool linear = true;
        double devk = 0.0, devt = 0.0;  // largest departure from the linear model
        runs.reserve((size_t)(stride * cdiv(n_meas, kRunLen)));
        for (int64_t line = 0; line < stride && linear; ++line) {
            // one slope per line (first to last sample), so that the runs of
            // a line share their step factor
            const double4 f = ks[(size_t)line], l = ks[(size_t)((n_meas - 1) * stride + line)];
            const double inv = 1.0 / (double)(n_meas - 1);
            const double4 d = make_double4((l.x - f.x) * inv, (l.y - f.y) * inv, (l.z - f.z) * inv, (l.w - f.w) * inv);
            for (int64_t i0 = 0; i0 < n_meas && linear; i0 += kRunLen) {
                const int64_t len = std::min<int64_t>(kRunLen, n_meas - i0);
                const int64_t s0 = i0 * stride + line;
                const double4 a = ks[(size_t)s0];
                for (int64_t m = 1; m < len && linear; ++m) {
                    const double4 c = ks[(size_t)(s0 + m * stride)];
                    const double ek = std::max({std::fabs(c.x - a.x - m * d.x), std::fabs(c.y - a.y - m * d.y),
                                                std::fabs(c.z - a.z - m * d.z)});
                    const double et = std::fabs(c.w - a.w - m * d.w);
                    devk = std::max(devk, ek);
                    devt = std::max(devt, et);
                    linear = ek <= tolk && et <= tolt;
                }
                RunDesc r{};
                r.k0x = a.x;
                r.k0y = a.y;
                r.k0z = a.z;
                r.t0 = a.w;
                r.dkx = d.x;
                r.dky = d.y;
                r.dkz = d.z;
                r.dt = d.w;
                r.s0 = (int32_t)s0;
                r.len = (int32_t)len;
                runs.push_back(r);
            }
        }
        if (linear) {
            p->n_runs = (int64_t)runs.size();
            p->run_stride = stride;
            p->runs_exact = devk <= 1e-2 * tolk && devt <= 1e-2 * tolt;
            // the distinct steps of each 256-run tile (bitwise)
            const int64_t n_tiles = cdiv(p->n_runs, kDirectThreads);
            h.run_steps.assign((size_t)(n_tiles * kRunSteps * 4), 0.0);
            h.run_nsteps.assign((size_t)n_tiles, 0);
            int most = 0;
            for (int64_t b = 0; b < n_tiles && most <= kRunSteps; ++b) {
                int cnt = 0;
                for (int64_t r = b * kDirectThreads; r < std::min<int64_t>(p->n_runs, (b + 1) * kDirectThreads); ++r) {
                    RunDesc &rd = runs[(size_t)r];
                    const double v[4] = {rd.dkx, rd.dky, rd.dkz, rd.dt};
                    int j = 0;
                    for (; j < cnt; ++j)
                        if (std::memcmp(&h.run_steps[(size_t)((b * kRunSteps + j) * 4)], v, sizeof v) == 0) break;
                    if (j == cnt) {
                        if (cnt == kRunSteps) {
                            most = kRunSteps + 1;
                            break;
                        }
                        std::memcpy(&h.run_steps[(size_t)((b * kRunSteps + j) * 4)], v, sizeof v);
                        ++cnt;
                    }
                    rd.step = j;
                }
                h.run_nsteps[(size_t)b] = cnt;
                most = std::max(most, cnt);
            }
            p->run_steps = most <= kRunSteps ? most : 0;
            if (p->run_steps == 0) {
                h.run_steps.clear();
                h.run_nsteps.clear();
            }
            // whole lines: every sample within 1e-12 of the line's first
            // sample plus m times its slope (the per-line GEMM's model)
            bool whole = true;
            std::vector<RunDesc> &lines = h.lines;
            lines.reserve((size_t)stride);
            for (int64_t line = 0; line < stride && whole; ++line) {
                const double4 f = ks[(size_t)line], l = ks[(size_t)((n_meas - 1) * stride + line)];
                const double inv = 1.0 / (double)(n_meas - 1);
                const double4 d = make_double4((l.x - f.x) * inv, (l.y - f.y) * inv, (l.z - f.z) * inv, (l.w - f.w) * inv);
                for (int64_t m = 1; m < n_meas && whole; ++m) {
                    const double4 c = ks[(size_t)(m * stride + line)];
                    const double ek = std::max({std::fabs(c.x - f.x - m * d.x), std::fabs(c.y - f.y - m * d.y),
                                                std::fabs(c.z - f.z - m * d.z)});
                    whole = ek <= tolk && std::fabs(c.w - f.w - m * d.w) <= tolt;
                }
                RunDesc r{};
                r.k0x = f.x;
                r.k0y = f.y;
                r.k0z = f.z;
                r.t0 = f.w;
                r.dkx = d.x;
                r.dky = d.y;
                r.dkz = d.z;
                r.dt = d.w;
                r.s0 = (int32_t)line;
                r.len = (int32_t)n_meas;
                lines.push_back(r);
            }
            if (whole) p->n_line_tabs = stride;
            else lines.clear();
        } else {
            runs.clear();
        }
    }

    return FM_OK;
}
}  // namespace fm

extern "C" int fm_signal_plan_create(fm_signal_plan **plan, int64_t n_meas, int64_t n_lines,
                                     int64_t n_kz, const double *kx, const double *ky,
                                     const double *kz, const double *t, int method)
{
    FM_CHECK_ARG(plan != nullptr, "plan pointer is NULL");
    *plan = nullptr;
    FM_CHECK_ARG(n_meas >= 0 && n_lines >= 0 && n_kz >= 0, "negative k-space dimension");
    FM_CHECK_ARG(method == FM_METHOD_AUTO || method == FM_METHOD_DIRECT || method == FM_METHOD_CARTESIAN,
                 "unknown method %d", method);
    const int64_t S = n_meas * n_lines * n_kz;
    FM_CHECK_ARG(S < (int64_t(1) << 31), "too many k-space samples (%lld)", (long long)S);
    FM_CHECK_ARG(S == 0 || (kx && ky && kz && t), "NULL k-space array");

    auto *p = new fm_signal_plan();
    p->n_meas = n_meas;
    p->n_lines = n_lines;
    p->n_kz = n_kz;
    p->n_samples = S;
    {
        const hipError_t e = hipGetDevice(&p->device);
        if (e != hipSuccess) {
            delete p;
            set_error("hipGetDevice failed: %s", hipGetErrorString(e));
            return FM_ERR_HIP;
        }
    }
    PlanHost h;
    {
        const int rc = plan_analyse(p, kx, ky, kz, t, method, h);
        if (rc != FM_OK) {
            delete p;
            return rc;
        }
    }
    const std::vector<double4> &ks = h.ks;
    const std::vector<RunDesc> &runs = h.runs;

    auto fail = [&](hipError_t e, const char *what) {
        set_error("%s failed: %s", what, hipGetErrorString(e));
        fm_signal_plan_destroy(p);
        return FM_ERR_HIP;
    };
    hipError_t e;
    if (S > 0) {
        if ((e = hipMalloc(&p->d_ks, sizeof(double4) * (size_t)S)) != hipSuccess) return fail(e, "hipMalloc");
        if ((e = hipMalloc(&p->d_pairs, sizeof(int2) * h.pairs.size())) != hipSuccess) return fail(e, "hipMalloc");
        if ((e = hipMalloc(&p->d_lane_group, h.lane_group.size())) != hipSuccess) return fail(e, "hipMalloc");
        if ((e = hipMalloc(&p->d_tiles_pairs, sizeof(int4) * h.tiles_p.size())) != hipSuccess) return fail(e, "hipMalloc");
        if ((e = hipMalloc(&p->d_tiles_consec, sizeof(SignalTile) * h.tiles_c.size())) != hipSuccess) return fail(e, "hipMalloc");
        if ((e = hipMalloc(&p->d_tg_t, sizeof(double) * (size_t)p->n_tgroups)) != hipSuccess) return fail(e, "hipMalloc");
        if ((e = hipMemcpy(p->d_ks, ks.data(), sizeof(double4) * (size_t)S, hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        if ((e = hipMemcpy(p->d_pairs, h.pairs.data(), sizeof(int2) * h.pairs.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        if ((e = hipMemcpy(p->d_lane_group, h.lane_group.data(), h.lane_group.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        if ((e = hipMemcpy(p->d_tiles_pairs, h.tiles_p.data(), sizeof(int4) * h.tiles_p.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        if ((e = hipMemcpy(p->d_tiles_consec, h.tiles_c.data(), sizeof(SignalTile) * h.tiles_c.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        if ((e = hipMemcpy(p->d_tg_t, p->tg_t.data(), sizeof(double) * (size_t)p->n_tgroups, hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        if (p->n_runs > 0) {
            if ((e = hipMalloc(&p->d_runs, sizeof(RunDesc) * runs.size())) != hipSuccess) return fail(e, "hipMalloc");
            if ((e = hipMemcpy(p->d_runs, runs.data(), sizeof(RunDesc) * runs.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        }
        if (p->n_line_tabs > 0) {
            if ((e = hipMalloc(&p->d_lines, sizeof(RunDesc) * h.lines.size())) != hipSuccess) return fail(e, "hipMalloc");
            if ((e = hipMemcpy(p->d_lines, h.lines.data(), sizeof(RunDesc) * h.lines.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        }
        if (p->run_steps > 0) {
            if ((e = hipMalloc(&p->d_run_steps, sizeof(double) * h.run_steps.size())) != hipSuccess) return fail(e, "hipMalloc");
            if ((e = hipMemcpy(p->d_run_steps, h.run_steps.data(), sizeof(double) * h.run_steps.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
            if ((e = hipMalloc(&p->d_run_nsteps, sizeof(int32_t) * h.run_nsteps.size())) != hipSuccess) return fail(e, "hipMalloc");
            if ((e = hipMemcpy(p->d_run_nsteps, h.run_nsteps.data(), sizeof(int32_t) * h.run_nsteps.size(), hipMemcpyHostToDevice)) != hipSuccess) return fail(e, "hipMemcpy");
        }
        if (p->method == FM_METHOD_CARTESIAN) {
            const int rc = cartesian_upload(p);
            if (rc != FM_OK) {
                fm_signal_plan_destroy(p);
                return rc;
            }
        }
    }
    *plan = p;
    return FM_OK;
}

extern "C" int fm_signal_plan_analyse(int64_t n_meas, int64_t n_lines, int64_t n_kz, const double *kx,
                                      const double *ky, const double *kz, const double *t, int method,
                                      int *method_out, int64_t *n_tgroups, int64_t *n_runs,
                                      int64_t *n_tiles_grouped, int *runs_exact, int *group_pack,
                                      int *conj_pack)
{
    FM_CHECK_ARG(n_meas >= 0 && n_lines >= 0 && n_kz >= 0, "negative k-space dimension");
    FM_CHECK_ARG(method == FM_METHOD_AUTO || method == FM_METHOD_DIRECT || method == FM_METHOD_CARTESIAN,
                 "unknown method %d", method);
    const int64_t S = n_meas * n_lines * n_kz;
    FM_CHECK_ARG(S < (int64_t(1) << 31), "too many k-space samples (%lld)", (long long)S);
    FM_CHECK_ARG(S == 0 || (kx && ky && kz && t), "NULL k-space array");
    fm_signal_plan p;
    p.n_meas = n_meas;
    p.n_lines = n_lines;
    p.n_kz = n_kz;
    p.n_samples = S;
    PlanHost h;
    const int rc = plan_analyse(&p, kx, ky, kz, t, method, h);
    if (rc != FM_OK) return rc;
    if (method_out) *method_out = p.method;
    if (n_tgroups) *n_tgroups = p.n_tgroups;
    if (n_runs) *n_runs = p.n_runs;
    if (n_tiles_grouped) *n_tiles_grouped = p.n_tiles_grouped;
    if (runs_exact) *runs_exact = p.runs_exact ? 1 : 0;
    if (group_pack) *group_pack = p.group_pack;
    if (conj_pack) *conj_pack = p.conj_pack;
    return FM_OK;
}

extern "C" int fm_signal_plan_set_timing(fm_signal_plan *p, int max_launches)
{
    FM_CHECK_ARG(p != nullptr, "plan is NULL");
    FM_CHECK_ARG(max_launches >= 0 && max_launches <= 1 << 16, "max_launches out of range");
    for (hipEvent_t e : p->ev_start) (void)hipEventDestroy(e);
    for (hipEvent_t e : p->ev_stop) (void)hipEventDestroy(e);
    p->ev_start.clear();
    p->ev_stop.clear();
    p->ev_used = 0;
    for (int i = 0; i < max_launches; ++i) {
        hipEvent_t a, b;
        FM_HIP(hipEventCreate(&a));
        FM_HIP(hipEventCreate(&b));
        p->ev_start.push_back(a);
        p->ev_stop.push_back(b);
    }
    return FM_OK;
}

extern "C" int fm_signal_plan_kernel_ms(fm_signal_plan *p, double *total_ms, int *n_timed)
{
    FM_CHECK_ARG(p != nullptr && total_ms != nullptr && n_timed != nullptr, "NULL argument");
    double sum = 0.0;
    const int n = p->ev_used;
    if (n > 0) FM_HIP(hipEventSynchronize(p->ev_stop[(size_t)n - 1]));
    for (int i = 0; i < n; ++i) {
        float ms = 0.0f;
        FM_HIP(hipEventElapsedTime(&ms, p->ev_start[(size_t)i], p->ev_stop[(size_t)i]));
        sum += ms;
    }
    p->ev_used = 0;
    *total_ms = sum;
    *n_timed = n;
    return FM_OK;
}

extern "C" int fm_signal_plan_destroy(fm_signal_plan *p)
{
    if (!p) return FM_OK;
    // executes still in flight on any stream read the plan's tables: wait
    // for the device before they are freed
    {
        int cur = 0;
        (void)hipGetDevice(&cur);
        if (cur != p->device) (void)hipSetDevice(p->device);
        (void)hipDeviceSynchronize();
        if (cur != p->device) (void)hipSetDevice(cur);
    }
    for (hipEvent_t e : p->ev_start) (void)hipEventDestroy(e);
    for (hipEvent_t e : p->ev_stop) (void)hipEventDestroy(e);
    (void)hipFree(p->d_ks);
    (void)hipFree(p->d_pairs);
    (void)hipFree(p->d_lane_group);
    (void)hipFree(p->d_tiles_pairs);
    (void)hipFree(p->d_runs);
    (void)hipFree(p->d_lines);
    (void)hipFree(p->d_run_steps);
    (void)hipFree(p->d_run_nsteps);
    (void)hipFree(p->d_tiles_consec);
    (void)hipFree(p->d_tg_t);
    cartesian_free(p);
    delete p;
    return FM_OK;
}

extern "C" int fm_signal_plan_info(const fm_signal_plan *p, int64_t *n_samples, int64_t *n_tgroups,
                                   int *method, double *tgroup_t)
{
    FM_CHECK_ARG(p != nullptr, "plan is NULL");
    if (n_samples) *n_samples = p->n_samples;
    if (n_tgroups) *n_tgroups = p->n_tgroups;
    if (method) *method = p->method;
    if (tgroup_t && p->n_tgroups) std::memcpy(tgroup_t, p->tg_t.data(), sizeof(double) * (size_t)p->n_tgroups);
    return FM_OK;
}

extern "C" int fm_signal_plan_runs(const fm_signal_plan *p, int64_t *n_runs, int *run_len, int *runs_exact)
{
    FM_CHECK_ARG(p != nullptr, "plan is NULL");
    if (n_runs) *n_runs = p->n_runs;
    if (run_len) *run_len = kRunLen;
    if (runs_exact) *runs_exact = p->runs_exact ? 1 : 0;
    return FM_OK;
}

extern "C" int fm_signal_plan_lines(const fm_signal_plan *p, int64_t *n_lines, int *line_gemm)
{
    FM_CHECK_ARG(p != nullptr, "plan is NULL");
    if (n_lines) *n_lines = p->n_line_tabs;
    if (line_gemm) *line_gemm = lines_usable(p, 0) ? 1 : 0;
    return FM_OK;
}

extern "C" int fm_signal_workspace_size(const fm_signal_plan *p, int precision, int64_t n_nodes,
                                        int n_enc, int moving, size_t *bytes)
{
    FM_CHECK_ARG(p != nullptr && bytes != nullptr, "NULL argument");
    FM_CHECK_ARG(n_nodes >= 0 && n_enc >= 1, "bad sizes");
    // the path fm_signal_execute takes: a Cartesian plan runs static nodes
    // on its GEMM and moving nodes on the per-readout moving GEMM (either
    // form, up to kMovMaxV encodings) or the direct kernels
    if (p->method == FM_METHOD_CARTESIAN && !moving)
        *bytes = cartesian_workspace(p, precision, n_nodes, n_enc);
    else if (p->method == FM_METHOD_CARTESIAN && n_enc <= kMovMaxV)
        *bytes = cartesian_moving_workspace(p, precision, n_nodes, n_enc);
    else
        *bytes = direct_workspace(p, n_nodes, n_enc);
    return FM_OK;
}

extern "C" int fm_signal_route(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc, int n_modes,
                               int *route, int64_t *n_splits)
{
    FM_CHECK_ARG(p != nullptr && route != nullptr && n_splits != nullptr, "NULL argument");
    FM_CHECK_ARG(precision == FM_PREC_F64 || precision == FM_PREC_MIXED,
                 "signal precision must be FM_PREC_F64 or FM_PREC_MIXED (got %d)", precision);
    FM_CHECK_ARG(n_nodes >= 1 && n_enc >= 1 && p->n_samples >= 1, "no nodes, encodings or samples");
    FM_CHECK_ARG(n_modes >= 0 && n_modes <= kMaxModes, "n_modes must be in [0, %d]", kMaxModes);
    const bool motion = n_modes > 0;
    if (p->method == FM_METHOD_CARTESIAN && (!motion || n_enc <= kMovMaxV)) {
        *route = cartesian_route(p, precision, n_nodes, n_enc, motion, n_splits);
        return FM_OK;
    }
    *route = direct_route(p, precision, n_nodes, motion);
    *n_splits = *route == FM_ROUTE_LINES
                    ? lines_splits(p, n_nodes)
                    : direct_launch(p, *route, precision, n_nodes, n_enc, n_modes, direct_workspace(p, n_nodes, n_enc)).n_splits;
    return FM_OK;
}

extern "C" int fm_signal_nodes_pack(int64_t n_nodes, int n_enc, int dtype, const void *r0,
                                    const void *phi_dB0, const void *T2, const void *mxy,
                                    const double *weights, double *packed, void *stream)
{
    FM_CHECK_ARG(n_nodes >= 0 && n_enc >= 1, "bad sizes (n_nodes=%lld, n_enc=%d)", (long long)n_nodes, n_enc);
    FM_CHECK_ARG(dtype == FM_DTYPE_F32 || dtype == FM_DTYPE_F64, "unknown dtype %d", dtype);
    if (n_nodes == 0) return FM_OK;
    FM_CHECK_ARG(r0 && phi_dB0 && T2 && mxy && packed, "NULL array");
    const unsigned blocks = (unsigned)cdiv(n_nodes, 256);
    hipStream_t st = as_stream(stream);
    if (dtype == FM_DTYPE_F64)
        k_nodes_pack<double><<<blocks, 256, 0, st>>>(n_nodes, n_enc, (const double *)r0, (const double *)phi_dB0,
                                                    (const double *)T2, (const double *)mxy, weights, packed);
    else
        k_nodes_pack<float><<<blocks, 256, 0, st>>>(n_nodes, n_enc, (const float *)r0, (const float *)phi_dB0,
                                                   (const float *)T2, (const float *)mxy, weights, packed);
    FM_LAUNCH_CHECK("k_nodes_pack");
    return FM_OK;
}

extern "C" int fm_signal_execute(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc,
                                 const double *packed, const float *modes, int n_modes,
                                 const double *motion_coef, void *workspace, size_t workspace_bytes,
                                 double *out, void *stream)
{
    FM_CHECK_ARG(p != nullptr, "plan is NULL");
    FM_CHECK_ARG(precision == FM_PREC_F64 || precision == FM_PREC_MIXED,
                 "signal precision must be FM_PREC_F64 or FM_PREC_MIXED (got %d)", precision);
    FM_CHECK_ARG(n_nodes >= 0 && n_enc >= 1, "bad sizes (n_nodes=%lld, n_enc=%d)", (long long)n_nodes, n_enc);
    FM_CHECK_ARG(p->n_samples == 0 || out != nullptr, "out is NULL");
    FM_CHECK_ARG(n_nodes == 0 || packed != nullptr, "packed is NULL");
    FM_CHECK_ARG(n_modes >= 0 && n_modes <= kMaxModes, "n_modes must be in [0, %d]", kMaxModes);
    FM_CHECK_ARG(!(modes != nullptr && n_modes > 0) || motion_coef != nullptr, "motion_coef is NULL");
    int dev = 0;
    FM_HIP(hipGetDevice(&dev));
    FM_CHECK_ARG(dev == p->device, "plan was created on device %d, current device is %d", p->device, dev);
    hipStream_t st = as_stream(stream);
    const bool motion = modes != nullptr && n_modes > 0;
    if (p->method == FM_METHOD_CARTESIAN && !motion)
        return cartesian_execute(p, precision, n_nodes, n_enc, packed, workspace, workspace_bytes, out, st);
    // moving nodes on a Cartesian plan: the per-readout GEMM in either form
    // (up to kMovMaxV encodings), otherwise the direct kernels
    if (p->method == FM_METHOD_CARTESIAN && motion && n_enc <= kMovMaxV)
        return cartesian_moving_execute(p, precision, n_nodes, n_enc, packed, modes, n_modes, motion_coef,
                                        workspace, workspace_bytes, out, st);
    return direct_execute(p, precision, n_nodes, n_enc, packed, modes, n_modes, motion_coef, workspace,
                          workspace_bytes, out, st);
}

extern "C" int fm_csr_spmv_c128(int64_t n_rows, int n_enc, const int64_t *indptr, const int64_t *indices,
                                const double *data, const double *x, double *y, void *stream)
{
    FM_CHECK_ARG(n_rows >= 0 && n_enc >= 1, "bad sizes");
    if (n_rows == 0) return FM_OK;
    FM_CHECK_ARG(indptr && indices && data && x && y, "NULL array");
    FM_CHECK_ARG(cdiv(n_rows * 16, 256) <= 0x7fffffff, "too many rows for one launch");
    using One = std::integral_constant<int, 1>;
    using Two = std::integral_constant<int, 2>;
    auto launch = [&](auto vb, auto rows) {
        constexpr int kRows = decltype(rows)::value;
        k_csr_spmv_c128<decltype(vb)::value, kRows><<<xcd_grid(cdiv(n_rows, 16 * kRows)), 256, 0, as_stream(stream)>>>(
            n_rows, n_enc, indptr, indices, data, reinterpret_cast<const double2 *>(x), reinterpret_cast<double2 *>(y));
    };
    const bool two = csr_two_rows(n_rows, n_enc);
    if (n_enc == 1 && two) launch(One{}, Two{});
    else if (n_enc == 2 && two) launch(Two{}, Two{});
    else if (n_enc == 1) launch(One{}, One{});
    else if (n_enc == 2) launch(Two{}, One{});
    else if (n_enc == 3) launch(std::integral_constant<int, 3>{}, One{});
    else launch(std::integral_constant<int, 4>{}, One{});
    FM_LAUNCH_CHECK("k_csr_spmv_c128");
    return FM_OK;
}
