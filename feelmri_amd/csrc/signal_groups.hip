// Direct sum over samples grouped by t: static nodes and moving nodes, FP64
// and mixed form (signal_direct.hip chooses it for t-groups of some size, and
// for moving nodes always).
//
//   S[s, v] = sum_n exp(-2 pi i k_s . r_n(t_s)) c_n[v](t_s),
//   c_n[v](t) = b[n, v] exp(-t / T2_n) exp(i phi_n t)
//
// Samples of one t share each node's position, decay and off-resonance.  A tile is up to
// 256 lanes of two samples each, the two of one t-group, lanes in the order of
// the groups, up to kGroupCap groups to a tile: small groups (the interleaves
// of a spiral, the spokes of a radial set) fill the lanes together.  Nodes
// pass through LDS in chunks: the threads stage, per (node, group of the
// tile), b exp(-t/T2), the off-resonance phase and for moving nodes the
// position (one loop over the modes for up to four groups at a time); the lanes then
// read one record for their two samples, whose phases start from the staged
// one (no instruction more than the product k.x, and one sine and cosine less
// to round than with a staged factor).
//
// CONJ: the two samples of a lane have k' = m and -m (every group pairs up,
// e.g. spiral interleaves half a turn apart); c is staged, so that one phase and one sine and
// cosine serve both: P = sum cos c and Q = sum sin c are accumulated, 4 FMAs
// per node and encoding, and the samples are P -+ i Q.  The mixed form takes k' to be
// +-m; in FP64 the pair's k' are mid +- m with a mid of a few roundings, whose phase
// turns c (to first order: its square is below 1e-24), and m is held in two
// doubles: without either the error against the sums in 80 bits is 2.1 times that of
// single samples (spiral, 300 x 32, 600 nodes: 2.8e-15 against 1.3e-15), with both 0.97
// times, for 8 % of the time.
//
// Phases are FP64, in cycles (k' carries the reference's float-pi factor).
// PLANAR: every kz is 0, so z is neither staged nor multiplied; 0 z joins x where
// it is staged, which makes a node with an infinite z what the product would (NaN).
// FP64 form: sincos_cycles_f64.  Mixed form: one fract, FP32 hardware sine and
// cosine, partial sums of a chunk in FP32, added into FP64.
//
// Bound by VALU issue.  LDS is kept small (chunks of 16 to 128 nodes, group_chunk)
// so that several waves share a SIMD.  Measured, whole calls (before: tiles of two
// 256-sample slots, one group to a slot or 32, 64, 128-sample groups packed,
// 3 waves per SIMD):
//   spiral, 973 000 nodes, 2048 x 32, mixed: 15.06 -> 13.2-13.5 ms (the staged factors by
//   FP32 series and their product in FP64, 0.5-0.9 ms of it less with the hardware sine and
//   cosine, take the error against 64 bits from 7.8e-8 to 3.6e-8);
//   spiral, 120 011 nodes, 1024 x 32, FP64: 6.54 -> 3.23-3.28 ms;
//   radial, 200 003 moving nodes, 256 x 96, 8 modes, 2 encodings, mixed: 5.70 ->
//   2.65 ms;
//   spiral, 138 519 nodes, 1504 x 48, mixed (per-sample t before): 5.49 -> 1.9 ms.
#include <algorithm>
#include <type_traits>

#include "signal_plan.h"

namespace fm {

// Static nodes: (x, y) per node, z per node unless planar; c and, unless conj,
// the phase per (node, group).
// Moving nodes: all per (node, group).  Rows of a node's groups have an odd
// number of entries: the staging threads write neighbouring nodes at once.
struct GroupLds {
    int xy, z, ph, c, t, coef;  // byte offsets
    int ps, cs;             // entries from node to node: positions, c
    int total;
};
__host__ __device__ constexpr GroupLds group_lds(int vb, bool mixed, bool motion, bool conj, bool planar, int chunk,
                                              int gs, int R)
{
    GroupLds l{};
    l.ps = motion ? gs | 1 : 1;
    l.cs = (gs * vb) | 1;
    const int pos = chunk * l.ps;
    int off = 0;
    l.xy = off;
    off += pos * 16;
    l.z = off;
    off += planar ? 0 : pos * 8;
    l.ph = off;
    off += conj ? 0 : chunk * (gs | 1) * 8;
    l.t = off;
    off += gs * 8;
    l.coef = off;
    off += motion ? gs * (R + 3) * 8 : 0;
    off = (off + 15) & ~15;
    l.c = off;
    off += chunk * l.cs * 2 * (mixed ? 4 : 8);
    l.total = off;
    return l;
}

// The most a tile can ask for, at the fewest nodes to a chunk: 59 136 bytes.
constexpr int kGroupChunkMin = 16, kGroupChunkMax = 128;
static_assert(group_lds(kMaxVB, false, true, false, false, kGroupChunkMin, kGroupCap, kMaxModes).total <= 64 * 1024,
              "the records of the fewest nodes fit the LDS of a workgroup");

template <bool MIXED>
struct GroupCT;
template <>
struct GroupCT<true> {
    using T = float;
    using T2 = float2;
};
template <>
struct GroupCT<false> {
    using T = double;
    using T2 = double2;
};

// u in cycles -> sin, cos of 2 pi u
template <bool MIXED>
__device__ inline void group_sincos(double u, typename GroupCT<MIXED>::T &s, typename GroupCT<MIXED>::T &c)
{
    if constexpr (MIXED) {
        const float r = turns_f32(u);
        s = __builtin_amdgcn_sinf(r);
        c = __builtin_amdgcn_cosf(r);
    } else {
        sincos_cycles_f64(u, s, c);
    }
}

// m + lo = (a - b) / 2 exactly (the rounding of a - b is a double), and (a + b) / 2.
__device__ inline void half_difference(double a, double b, double &m, double &lo, double &mid)
{
    const double s = a - b, t = s - a;
    m = 0.5 * s;
    lo = 0.5 * ((a - (s - t)) - (b + t));
    mid = 0.5 * (a + b);
}

template <int VB, bool MIXED, bool MOTION, bool CONJ, bool PLANAR>
__global__ __launch_bounds__(kDirectThreads, MIXED ? 4 : 3) void k_signal_groups(
    const double *__restrict__ packed, int64_t N, int V, int v0, const double4 *__restrict__ ks,
    const int2 *__restrict__ pairs, const uint8_t *__restrict__ lane_group, const int4 *__restrict__ tiles, const double *__restrict__ tg_t,
    const float *__restrict__ modes, int R, const double *__restrict__ mcoef, int chunk, int gs,
    int64_t nodes_per_split, double2 *__restrict__ dst, int64_t S, int write_final)
{
    using CT = typename GroupCT<MIXED>::T;
    using CT2 = typename GroupCT<MIXED>::T2;
    extern __shared__ char lds[];
    const GroupLds off = group_lds(VB, MIXED, MOTION, CONJ, PLANAR, chunk, gs, R);
    double2 *const sxy = reinterpret_cast<double2 *>(lds + off.xy);
    double *const sz = reinterpret_cast<double *>(lds + off.z);
    double *const sph = reinterpret_cast<double *>(lds + off.ph);
    double *const st = reinterpret_cast<double *>(lds + off.t);
    double *const scoef = reinterpret_cast<double *>(lds + off.coef);
    CT2 *const sc = reinterpret_cast<CT2 *>(lds + off.c);

    const int64_t split = blockIdx.y;
    const int64_t n_begin = split * nodes_per_split;
    const int64_t n_end = (n_begin + nodes_per_split < N) ? n_begin + nodes_per_split : N;
    const int tid = threadIdx.x;
    const int4 tile = tiles[blockIdx.x];  // first lane entry, count, first group, groups
    const int ng = tile.w;
    for (int g = tid; g < ng; g += kDirectThreads) st[g] = tg_t[tile.z + g];
    if (MOTION)
        for (int q = tid; q < ng * (R + 3); q += kDirectThreads) scoef[q] = mcoef[(int64_t)tile.z * (R + 3) + q];

    const bool live = tid < tile.y;
    const int2 pr = pairs[tile.x + (live ? tid : 0)];  // samples (second -1: none)
    const int lg = lane_group[tile.x + (live ? tid : 0)];
    double kx[2], ky[2], kz[2];
    constexpr int kFix = CONJ && !MIXED ? 3 : 0;
    double klo[kFix ? kFix : 1], kmid[kFix ? kFix : 1];  // FP64 pairs: of m, of the middle
    {
        const double4 a = ks[pr.x], b = ks[pr.y >= 0 ? pr.y : pr.x];
        if (CONJ) {
            double m[3], lo[3], sum[3];
            half_difference(a.x, b.x, m[0], lo[0], sum[0]);
            half_difference(a.y, b.y, m[1], lo[1], sum[1]);
            half_difference(a.z, b.z, m[2], lo[2], sum[2]);
            kx[0] = m[0];
            ky[0] = m[1];
            kz[0] = m[2];
            kx[1] = ky[1] = kz[1] = 0.0;
#pragma unroll
            for (int d = 0; d < kFix; ++d) {
                klo[d] = lo[d];
                kmid[d] = kTwoPi * sum[d];
            }
        } else {
            kx[0] = a.x;
            ky[0] = a.y;
            kz[0] = a.z;
            kx[1] = b.x;
            ky[1] = b.y;
            kz[1] = b.z;
        }
    }

    double tot_re[2][VB], tot_im[2][VB];  // CONJ: [0] P, [1] Q
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int v = 0; v < VB; ++v) tot_re[j][v] = tot_im[j][v] = 0.0;

    // staging: thread -> node tid % chunk, groups tid / chunk, + 256 / chunk, ...
    const int nl = tid & (chunk - 1), g0 = tid / chunk, gstep = kDirectThreads / chunk;

    for (int64_t base = n_begin; base < n_end; base += chunk) {
        __syncthreads();  // previous chunk consumed; times and coefficients visible
        {
            const int64_t n = base + nl;
            const bool ok = n < n_end;
            const double x0 = ok ? packed[n] : 0.0, y0 = ok ? packed[N + n] : 0.0, z0 = ok ? packed[2 * N + n] : 0.0;
            const double phc = (ok ? packed[3 * N + n] : 0.0) * (1.0 / kTwoPi), r2 = ok ? packed[4 * N + n] : 0.0;
            double br[VB], bi[VB];
#pragma unroll
            for (int v = 0; v < VB; ++v) {
                br[v] = ok ? packed[(int64_t)(5 + 2 * (v0 + v)) * N + n] : 0.0;
                bi[v] = ok ? packed[(int64_t)(6 + 2 * (v0 + v)) * N + n] : 0.0;
            }
            if constexpr (!MOTION) {
                if (g0 == 0) {
                    sxy[nl] = make_double2(PLANAR ? fma(0.0, z0, x0) : x0, y0);
                    if (!PLANAR) sz[nl] = z0;
                }
            } else {
                // one pass over the modes for B groups of the thread (gb, gb + gstep, ...)
                auto place = [&](int gb, auto count) {
                    constexpr int B = decltype(count)::value;
                    double dx[B], dy[B], dz[B];
                    int cg[B];
#pragma unroll
                    for (int q = 0; q < B; ++q) {
                        const int g = gb + q * gstep;
                        cg[q] = (g < ng ? g : ng - 1) * (R + 3);
                        dx[q] = scoef[cg[q] + R];
                        dy[q] = scoef[cg[q] + R + 1];
                        dz[q] = scoef[cg[q] + R + 2];
                    }
                    if (ok) {
                        for (int r = 0; r < R; ++r) {
                            const double mx = (double)modes[(int64_t)(0 * R + r) * N + n];
                            const double my = (double)modes[(int64_t)(1 * R + r) * N + n];
                            const double mz = (double)modes[(int64_t)(2 * R + r) * N + n];
#pragma unroll
                            for (int q = 0; q < B; ++q) {
                                const double w = scoef[cg[q] + r];
                                dx[q] = fma(mx, w, dx[q]);
                                dy[q] = fma(my, w, dy[q]);
                                dz[q] = fma(mz, w, dz[q]);
                            }
                        }
                    }
#pragma unroll
                    for (int q = 0; q < B; ++q) {
                        const int g = gb + q * gstep;
                        if (g < ng) {
                            const double x = x0 + dx[q], z = z0 + dz[q];
                            sxy[nl * off.ps + g] =
                                ok ? make_double2(PLANAR ? fma(0.0, z, x) : x, y0 + dy[q]) : make_double2(0.0, 0.0);
                            if (!PLANAR) sz[nl * off.ps + g] = ok ? z : 0.0;
                        }
                    }
                };
                // the same passes for every thread of the workgroup: 4, 2 or 1 groups by what is left
                for (int k0 = 0; k0 < ng;) {
                    if (ng - k0 > 2 * gstep) {
                        place(k0 + g0, std::integral_constant<int, 4>{});
                        k0 += 4 * gstep;
                    } else if (ng - k0 > gstep) {
                        place(k0 + g0, std::integral_constant<int, 2>{});
                        k0 += 2 * gstep;
                    } else {
                        place(k0 + g0, std::integral_constant<int, 1>{});
                        k0 += gstep;
                    }
                }
            }
            // b exp(-t/T2) and phi t, or c = b exp(-t/T2) exp(i phi t)   (MRI.cpp:264-271);
            // products in FP64, rounded once
            for (int g = g0; g < ng; g += gstep) {
                const double t = st[g];
                CT d;
                if constexpr (MIXED) d = __builtin_amdgcn_exp2f((float)(-t * r2 * 1.4426950408889634));
                else d = exp(-t * r2);
                double fr = (double)d, fi = 0.0;
                if constexpr (CONJ) {
                    CT so, co;
                    if constexpr (MIXED) sincos_cycles_f32(phc * t, so, co);
                    else sincos_cycles_f64(phc * t, so, co);
                    fr = (double)(d * co);
                    fi = (double)(d * so);
                } else {
                    sph[nl * (gs | 1) + g] = -phc * t;
                }
#pragma unroll
                for (int v = 0; v < VB; ++v) {
                    double cr = br[v] * fr, ci = bi[v] * fr;
                    if constexpr (CONJ) {
                        cr = fma(-bi[v], fi, cr);
                        ci = fma(br[v], fi, ci);
                    }
                    CT2 c;
                    c.x = ok ? (CT)cr : (CT)0;
                    c.y = ok ? (CT)ci : (CT)0;
                    sc[nl * off.cs + g * VB + v] = c;
                }
            }
        }
        __syncthreads();
        const int cnt = (n_end - base < chunk) ? (int)(n_end - base) : chunk;

        CT acc_re[2][VB], acc_im[2][VB];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < VB; ++v) acc_re[j][v] = acc_im[j][v] = (CT)0;

        const double2 *pxy = sxy + (MOTION ? lg : 0);
        const double *pz = sz + (MOTION ? lg : 0);
        const double *pp = sph + lg;
        const CT2 *pc = sc + lg * VB;
#pragma unroll (MIXED ? 4 : 2)
        for (int m = 0; m < cnt; ++m) {
            const double2 xy = *pxy;
            const double z = PLANAR ? 0.0 : *pz;
            CT2 c[VB];
#pragma unroll
            for (int v = 0; v < VB; ++v) c[v] = pc[v];
            pxy += MOTION ? off.ps : 1;
            pz += MOTION ? off.ps : 1;
            pc += off.cs;
            double ph = 0.0;
            if constexpr (!CONJ) {
                ph = *pp;
                pp += gs | 1;
            }
#pragma unroll
            for (int j = 0; j < (CONJ ? 1 : 2); ++j) {
                double u;
                if constexpr (kFix) {
                    double lo = fma(klo[0], xy.x, klo[1] * xy.y), eps = fma(kmid[0], xy.x, kmid[1] * xy.y);
                    if (!PLANAR) {
                        lo = fma(klo[2], z, lo);
                        eps = fma(kmid[2], z, eps);
                        lo = fma(kz[j], z, lo);
                    }
                    u = fma(kx[j], xy.x, fma(ky[j], xy.y, lo));
#pragma unroll
                    for (int v = 0; v < VB; ++v) {
                        const CT2 w = c[v];
                        c[v].x = fma(eps, w.y, w.x);
                        c[v].y = fma(-eps, w.x, w.y);
                    }
                } else if constexpr (CONJ) {
                    u = PLANAR ? fma(kx[j], xy.x, ky[j] * xy.y) : fma(kx[j], xy.x, fma(ky[j], xy.y, kz[j] * z));
                } else {
                    u = PLANAR ? fma(kx[j], xy.x, fma(ky[j], xy.y, ph))
                               : fma(kx[j], xy.x, fma(ky[j], xy.y, fma(kz[j], z, ph)));
                }
                CT sn, cs;
                group_sincos<MIXED>(u, sn, cs);
#pragma unroll
                for (int v = 0; v < VB; ++v) {
                    if constexpr (CONJ) {
                        acc_re[0][v] = fma(cs, c[v].x, acc_re[0][v]);
                        acc_im[0][v] = fma(cs, c[v].y, acc_im[0][v]);
                        acc_re[1][v] = fma(sn, c[v].x, acc_re[1][v]);
                        acc_im[1][v] = fma(sn, c[v].y, acc_im[1][v]);
                    } else {
                        acc_re[j][v] = fma(cs, c[v].x, fma(sn, c[v].y, acc_re[j][v]));
                        acc_im[j][v] = fma(cs, c[v].y, fma(-sn, c[v].x, acc_im[j][v]));
                    }
                }
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < VB; ++v) {
                tot_re[j][v] += (double)acc_re[j][v];
                tot_im[j][v] += (double)acc_im[j][v];
            }
    }

    if (!live) return;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int s = j == 0 ? pr.x : pr.y;
        if (s < 0) continue;
        const int64_t row = write_final ? (int64_t)s : split * S + s;
#pragma unroll
        for (int v = 0; v < VB; ++v) {
            double re = tot_re[j][v], im = tot_im[j][v];
            if constexpr (CONJ) {  // P - i Q and P + i Q
                re = j == 0 ? tot_re[0][v] + tot_im[1][v] : tot_re[0][v] - tot_im[1][v];
                im = j == 0 ? tot_im[0][v] - tot_re[1][v] : tot_im[0][v] + tot_re[1][v];
            }
            dst[row * V + v0 + v] = make_double2(re, im);
        }
    }
}

// Conjugate pairs serve the FP64 form where they are exact to a few roundings.

bool groups_in_pairs(const fm_signal_plan *p, bool mixed) { return p->pairs_conj && (mixed || p->pairs_exact); }

// Nodes per chunk: the most, a power of two from 16 to 128, whose records take
// at most 24 KB (6 workgroups of 4 waves per CU).  16 where even those take
// more: FP64 moving nodes, 4 encodings, 32 groups and modes ask for 58 KB and run 2
// workgroups per CU.
static int group_chunk(const fm_signal_plan *p, int vb, bool mixed, bool motion, int R)
{
    const bool conj = groups_in_pairs(p, mixed);
    int c = kGroupChunkMax;
    while (c > kGroupChunkMin && group_lds(vb, mixed, motion, conj, p->planar != 0, c, p->groups_per_tile, R).total > 24 * 1024) c /= 2;
    return c;
}

template <int VB, bool MIXED, bool MOTION, bool CONJ>
static const void *group_kernel(bool planar)
{
    return planar ? reinterpret_cast<const void *>(k_signal_groups<VB, MIXED, MOTION, CONJ, true>)
                  : reinterpret_cast<const void *>(k_signal_groups<VB, MIXED, MOTION, CONJ, false>);
}

template <int VB, bool MIXED>
static const void *group_kernel_vm(bool motion, bool conj, bool planar)
{
    if (motion) return conj ? group_kernel<VB, MIXED, true, true>(planar) : group_kernel<VB, MIXED, true, false>(planar);
    return conj ? group_kernel<VB, MIXED, false, true>(planar) : group_kernel<VB, MIXED, false, false>(planar);
}

static const void *group_kernel_of(int vb, bool mixed, bool motion, bool conj, bool planar)
{
    switch (vb) {
    case 1: return mixed ? group_kernel_vm<1, true>(motion, conj, planar) : group_kernel_vm<1, false>(motion, conj, planar);
    case 2: return mixed ? group_kernel_vm<2, true>(motion, conj, planar) : group_kernel_vm<2, false>(motion, conj, planar);
    case 3: return mixed ? group_kernel_vm<3, true>(motion, conj, planar) : group_kernel_vm<3, false>(motion, conj, planar);
    default: return mixed ? group_kernel_vm<4, true>(motion, conj, planar) : group_kernel_vm<4, false>(motion, conj, planar);
    }
}

// Workgroups of encodings [0, min(V, kMaxVB)) that one CU holds at once.
int groups_blocks_per_cu(const fm_signal_plan *p, bool mixed, bool motion, int V, int R)
{
    const int vb = std::min(V, kMaxVB);
    const int chunk = group_chunk(p, vb, mixed, motion, R);
    const int lds = group_lds(vb, mixed, motion, groups_in_pairs(p, mixed), p->planar != 0, chunk, p->groups_per_tile, R).total;
    return blocks_per_cu(group_kernel_of(vb, mixed, motion, groups_in_pairs(p, mixed), p->planar != 0), kDirectThreads,
                         (size_t)lds);
}

int groups_launch(const fm_signal_plan *p, bool mixed, bool motion, int64_t N, int V, int v0, int vb,
                  const double *packed, const float *modes, int R, const double *mcoef, int64_t n_splits,
                  int64_t nodes_per_split, double2 *dst, int write_final, hipStream_t st)
{
    int chunk = group_chunk(p, vb, mixed, motion, R), gs = p->groups_per_tile, vv = V, vfirst = v0, RR = R;
    const int lds = group_lds(vb, mixed, motion, groups_in_pairs(p, mixed), p->planar != 0, chunk, gs, R).total;
    int64_t S = p->n_samples, nn = N, nps = nodes_per_split;
    const double4 *ks = p->d_ks;
    const int2 *pairs = p->d_pairs;
    const uint8_t *lane_group = p->d_lane_group;
    const int4 *tiles = p->d_tiles_pairs;
    const double *tg = p->d_tg_t;
    void *args[] = {&packed, &nn, &vv, &vfirst, &ks, &pairs, &lane_group, &tiles, &tg, &modes, &RR, &mcoef, &chunk, &gs, &nps,
                    &dst, &S, &write_final};
    FM_HIP(hipLaunchKernel(group_kernel_of(vb, mixed, motion, groups_in_pairs(p, mixed), p->planar != 0),
                           dim3((unsigned)p->n_tiles_pairs, (unsigned)n_splits), dim3(kDirectThreads), args,
                           (size_t)lds, st));
    return FM_OK;
}

}  // namespace fm
