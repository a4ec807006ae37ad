// Cartesian factorised signal: a complex GEMM on the matrix cores.
//
// When every k-space coordinate splits additively over the three sample
// indices, k(i,j,k) = F(i) + G(j) + H(k) per axis, and t depends on the
// readout index i only (Cartesian stacks with one line per shot,
// python/feelmri/KSpaceTraj.py:183-220), the direct sum of
// cpp/feelmri/MRI.cpp:196-297 factorises:
//
//   S[i, (j,k,v)] = sum_n E[i,n] A[n,(j,k,v)]
//   E[i,n]        = exp(-t_i/T2_n) exp(i phi_n t_i) exp(-2 pi i F_i . x_n)
//   A[n,(j,k,v)]  = Ey[j,n] Ezb[(k,v),n]
//   Ey[j,n]       = exp(-2 pi i G_j . x_n),  Ezb[(k,v),n] = b[n,v] exp(-2 pi i H_k . x_n)
//
// (2 pi carries the reference's float-pi factor, MRI.h:13).  Per execute the
// E, Ey and Ezb tables are computed once (O((n_ro + n_ln + n_kz V) N)
// transcendentals); the GEMM then streams E through LDS and builds the A
// operand in registers from Ey and Ezb, so the (N x lines*kz*V) matrix A is
// never stored.
//
// Lines that pair up about a centre are taken as real rows (PairAxis,
// signal_plan.h): the roles turn, S[r, (i,k,v)] = sum_n A[r,n] (Ex[i,n]
// Ezb[(k,v),n]) with A the lines' cosine and sine rows and Ex the readout
// factors, half the products, and the reduction forms each pair's samples.
//
// Mixed form: E and A are split into bf16 hi + lo parts and each real product
// x*y is formed as xh*yh + xh*yl + xl*yh on v_mfma_f32_32x32x16_bf16 with
// FP32 accumulation (12 MFMAs per 16 nodes per 32x32 complex tile).  FP64
// form: v_mfma_f64_16x16x4_f64 (4 MFMAs per 4 nodes per 16x16 complex tile).
// Nodes are split across workgroups; per-split partial tiles are summed in
// FP64 in a fixed order by a second kernel.  Workgroups that share a node
// split (and so the same E tiles) are mapped onto the same XCD so the tiles
// are fetched from HBM once per split and served from that XCD's L2.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "cart_gemm.h"

namespace fm {


// ---------------------------------------------------------------------------
// Sampling analysis (host)
// ---------------------------------------------------------------------------
// k as the kernels' phases take it, k' = k (float)pi / pi, in extended precision.
static long double kprime(double k)
{
    return (long double)k * ((long double)(float)3.14159265358979323846 / 3.14159265358979323846264338327950288L);
}

// A value as two doubles.
static void two_doubles(long double v, double &hi, double &lo)
{
    hi = (double)v;
    lo = std::isfinite(hi) ? (double)(v - (long double)hi) : 0.0;
}

// Rows of the entities in a.ent (index, partner or -1): first the cosines, then the
// sines; the centre a.c is that of the pairs (their middles' mean), or as given.
static void pair_rows(PairAxis &a, const std::vector<double> &k, double tol)
{
    const int64_t n = a.n_ent = (int64_t)a.ent.size() / 4;
    auto at = [&](int32_t j, int d) { return kprime(k[(size_t)(3 * j + d)]); };
    int64_t n_pair = 0;
    long double mid[3] = {0.0L, 0.0L, 0.0L};
    for (int64_t e = 0; e < n; ++e) {
        const int32_t p = a.ent[(size_t)(4 * e)], q = a.ent[(size_t)(4 * e + 1)];
        if (q < 0) continue;
        ++n_pair;
        for (int d = 0; d < 3; ++d) mid[d] += 0.5L * (at(p, d) + at(q, d));
    }
    for (int d = 0; d < 3 && n_pair; ++d) a.c[d] = mid[d] / (long double)n_pair;
    std::vector<long double> D;
    int64_t n_lines = 0;
    long double departs = 0.0L;
    std::vector<char> centred;
    for (int64_t e = 0; e < n; ++e) {
        const int32_t p = a.ent[(size_t)(4 * e)], q = a.ent[(size_t)(4 * e + 1)];
        bool zero = q < 0;
        for (int d = 0; d < 3; ++d) {
            const long double v = q < 0 ? at(p, d) - a.c[d] : 0.5L * (at(p, d) - at(q, d));
            zero = zero && std::fabs((double)v) <= tol;
            D.push_back(v);
            const long double off = q < 0 ? 0.0L : 0.5L * (at(p, d) + at(q, d)) - a.c[d];
            departs += 2.0L * off * off;  // of both
        }
        if (zero)
            for (int d = 0; d < 3; ++d) {
                departs += D[D.size() - 3 + (size_t)d] * D[D.size() - 3 + (size_t)d];
                D[D.size() - 3 + (size_t)d] = 0.0L;
            }
        centred.push_back(zero);
        n_lines += q < 0 ? 1 : 2;
    }
    a.departs2 = (double)(departs / (long double)std::max<int64_t>(n_lines, 1));
    auto row = [&](int64_t e, double quarter) {
        double lo[3];
        for (int d = 0; d < 3; ++d) {
            double hi;
            two_doubles(D[(size_t)(3 * e + d)], hi, lo[d]);
            a.rows.push_back(hi);
        }
        a.rows.push_back(quarter);
        a.rows_lo.insert(a.rows_lo.end(), {lo[0], lo[1], lo[2], 0.0});
        return (int32_t)a.n_rows++;
    };
    a.n_rows = 0;
    for (int64_t e = 0; e < n; ++e) a.ent[(size_t)(4 * e + 2)] = row(e, 0.25);
    for (int64_t e = 0; e < n; ++e) a.ent[(size_t)(4 * e + 3)] = centred[(size_t)e] ? -1 : row(e, 0.0);
}

// Real rows of the n offsets of one axis (PairAxis; g as k', k as given) about the
// centre c: the offsets sorted, partners found from both ends.  Partners' middles
// lie within 2e-15 of the largest |offset| of c.
static PairAxis pair_axis_about(const std::vector<double> &g, const std::vector<double> &k, int64_t n, const double (&c)[3])
{
    PairAxis a;
    double gmax = 0.0;
    for (double v : g) gmax = std::max(gmax, std::fabs(v));
    const double tol = 4e-15 * gmax;
    std::vector<int32_t> order((size_t)n);
    for (int64_t j = 0; j < n; ++j) order[(size_t)j] = (int32_t)j;
    std::sort(order.begin(), order.end(), [&](int32_t p, int32_t q) {
        for (int d = 0; d < 3; ++d) {
            const double vp = g[(size_t)(3 * p + d)], vq = g[(size_t)(3 * q + d)];
            if (vp != vq) return vp < vq;
        }
        return p < q;
    });
    auto add = [&](int32_t p, int32_t q) { a.ent.insert(a.ent.end(), {p, q, 0, 0}); };  // q = -1: no partner
    int64_t lo = 0, hi = n - 1;
    while (lo <= hi) {
        const int32_t p = order[(size_t)lo], q = order[(size_t)hi];
        if (lo == hi) {
            add(p, -1);
            break;
        }
        bool match = true;
        int side = 0;                      // sign of the first component off the centre
        for (int d = 0; d < 3; ++d) {
            const double s = g[(size_t)(3 * p + d)] + g[(size_t)(3 * q + d)] - 2.0 * c[d];
            match = match && std::fabs(s) <= tol;
            if (side == 0 && std::fabs(s) > tol) side = s > 0.0 ? 1 : -1;
        }
        if (match) {
            add(p, q);
            ++lo;
            --hi;
        } else if (side < 0) {             // p lies further out than q
            add(p, -1);
            ++lo;
        } else {
            add(q, -1);
            --hi;
        }
    }
    for (int d = 0; d < 3; ++d) a.c[d] = c[d];
    pair_rows(a, k, tol);
    return a;
}

// The centre that leaves the fewest rows: the middle of the offsets (an even
// count -n/2 .. n/2 - 1 pairs up completely about its half step), or 0 (where
// single-precision offsets are symmetric to the last bit).
static PairAxis pair_axis(const std::vector<double> &g, const std::vector<double> &k, int64_t n)
{
    double mid[3] = {0.0, 0.0, 0.0};
    const double zero[3] = {0.0, 0.0, 0.0};
    // an offset that is not finite has no partner, and no tolerance can be
    // taken from it: no pairs, every offset with rows of its own about 0
    for (double v : g)
        if (!std::isfinite(v)) {
            PairAxis a;
            for (int64_t j = 0; j < n; ++j) a.ent.insert(a.ent.end(), {(int32_t)j, -1, 0, 0});
            pair_rows(a, k, -1.0);
            return a;
        }
    for (int d = 0; d < 3; ++d) {
        double lo = g[(size_t)d], hi = lo;
        for (int64_t j = 1; j < n; ++j) {
            lo = std::min(lo, g[(size_t)(3 * j + d)]);
            hi = std::max(hi, g[(size_t)(3 * j + d)]);
        }
        mid[d] = 0.5 * (lo + hi);
    }
    PairAxis a = pair_axis_about(g, k, n, mid), b = pair_axis_about(g, k, n, zero);
    return b.n_rows < a.n_rows ? b : a;
}

// What complex rows round on the offsets k (mean square, as an offset): k' to a
// double, and the product with a position, 0.42 of 2^-53 of it (rms over the mantissas).
static double complex_rounding2(const std::vector<double> &k, int64_t n)
{
    long double sum = 0.0L;
    for (double v : k) {
        const long double e = kprime(v) - (long double)(v * kPiFOverPi), r = 0.42L * 0x1p-53L * kprime(v);
        sum += e * e + r * r;
    }
    return (double)(sum / (long double)std::max<int64_t>(n, 1));
}

bool cartesian_analyse(fm_signal_plan *p, const double *kx, const double *ky, const double *kz,
                       const double *t)
{
    const int64_t R = p->n_meas, L = p->n_lines, K = p->n_kz;
    auto at = [&](const double *a, int64_t i, int64_t j, int64_t k) { return a[(i * L + j) * K + k]; };
    // t must be a function of the readout index only
    for (int64_t i = 0; i < R; ++i)
        for (int64_t j = 0; j < L; ++j)
            for (int64_t k = 0; k < K; ++k)
                if (!(at(t, i, j, k) == at(t, i, 0, 0))) return false;
    CartesianTables &c = p->cart;
    c.n_ro = R;
    c.n_ln = L;
    c.n_kz = K;
    c.F.assign((size_t)R * 3, 0.0);
    c.G.assign((size_t)L * 3, 0.0);
    c.H.assign((size_t)K * 3, 0.0);
    c.t.resize((size_t)R);
    for (int64_t i = 0; i < R; ++i) c.t[(size_t)i] = at(t, i, 0, 0);
    c.ro_group.resize((size_t)R);
    for (int64_t i = 0; i < R; ++i) c.ro_group[(size_t)i] = p->sample_group[(size_t)(i * L * K)];
    const double *ax[3] = {kx, ky, kz};
    for (int a = 0; a < 3; ++a) {
        const double *k3 = ax[a];
        double kmax = 0.0;
        bool only_i = true, only_j = true, only_k = true;
        for (int64_t i = 0; i < R; ++i)
            for (int64_t j = 0; j < L; ++j)
                for (int64_t k = 0; k < K; ++k) {
                    const double v = at(k3, i, j, k);
                    kmax = std::max(kmax, std::fabs(v));
                    only_i &= v == at(k3, i, 0, 0);
                    only_j &= v == at(k3, 0, j, 0);
                    only_k &= v == at(k3, 0, 0, k);
                }
        if (only_i) {
            for (int64_t i = 0; i < R; ++i) c.F[(size_t)(3 * i + a)] = at(k3, i, 0, 0);
        } else if (only_j) {
            for (int64_t j = 0; j < L; ++j) c.G[(size_t)(3 * j + a)] = at(k3, 0, j, 0);
        } else if (only_k) {
            for (int64_t k = 0; k < K; ++k) c.H[(size_t)(3 * k + a)] = at(k3, 0, 0, k);
        } else {
            // general additive split (e.g. a rotated Cartesian grid)
            const double k0 = at(k3, 0, 0, 0);
            for (int64_t i = 0; i < R; ++i) c.F[(size_t)(3 * i + a)] = at(k3, i, 0, 0);
            for (int64_t j = 0; j < L; ++j) c.G[(size_t)(3 * j + a)] = at(k3, 0, j, 0) - k0;
            for (int64_t k = 0; k < K; ++k) c.H[(size_t)(3 * k + a)] = at(k3, 0, 0, k) - k0;
            const double tol = 1e-12 * std::max(kmax, 1.0);
            for (int64_t i = 0; i < R; ++i)
                for (int64_t j = 0; j < L; ++j)
                    for (int64_t k = 0; k < K; ++k) {
                        const double s = c.F[(size_t)(3 * i + a)] + c.G[(size_t)(3 * j + a)] + c.H[(size_t)(3 * k + a)];
                        if (!(std::fabs(at(k3, i, j, k) - s) <= tol)) return false;
                    }
        }
    }
    const std::vector<double> kF = c.F, kG = c.G, kH = c.H;
    for (auto *v : {&c.F, &c.G, &c.H})
        for (double &x : *v) x *= kPiFOverPi;
    c.axis_aligned = true;
    for (int64_t j = 0; j < L; ++j) c.axis_aligned &= c.G[(size_t)(3 * j)] == 0.0 && c.G[(size_t)(3 * j + 2)] == 0.0;
    for (int64_t k = 0; k < K; ++k) c.axis_aligned &= c.H[(size_t)(3 * k)] == 0.0 && c.H[(size_t)(3 * k + 1)] == 0.0;
    c.lines = pair_axis(c.G, kG, L);
    c.kzs = pair_axis(c.H, kH, K);
    c.F_pairs.assign((size_t)R * 6, 0.0);
    c.F_pairs_lo.assign((size_t)R * 6, 0.0);
    for (int64_t i = 0; i < R; ++i)
        for (int d = 0; d < 3; ++d) {
            const long double f = kprime(kF[(size_t)(3 * i + d)]) + c.lines.c[d];
            two_doubles(f, c.F_pairs[(size_t)(3 * i + d)], c.F_pairs_lo[(size_t)(3 * i + d)]);
            two_doubles(f + c.kzs.c[d], c.F_pairs[(size_t)(3 * (R + i) + d)], c.F_pairs_lo[(size_t)(3 * (R + i) + d)]);
        }
    c.H_lo.assign((size_t)K * 3, 0.0);
    for (size_t q = 0; q < c.H_lo.size(); ++q) c.H_lo[q] = std::isfinite(c.H[q]) ? (double)(kprime(kH[q]) - (long double)c.H[q]) : 0.0;
    // (the box of the nodes is taken to be as wide along each axis)
    const double rounds = complex_rounding2(kF, R) + complex_rounding2(kG, L) + complex_rounding2(kH, K);
    c.pairs_f64 = c.lines.departs2 <= rounds;
    c.pairs_f64_moving = c.lines.departs2 + c.kzs.departs2 <= rounds;
    c.ok = true;
    return true;
}

int cartesian_upload(fm_signal_plan *p)
{
    CartesianTables &c = p->cart;
    FM_HIP(hipMalloc(&c.d_F, sizeof(double) * c.F.size()));
    FM_HIP(hipMalloc(&c.d_G, sizeof(double) * c.G.size()));
    FM_HIP(hipMalloc(&c.d_H, sizeof(double) * c.H.size()));
    FM_HIP(hipMalloc(&c.d_t, sizeof(double) * c.t.size()));
    FM_HIP(hipMemcpy(c.d_F, c.F.data(), sizeof(double) * c.F.size(), hipMemcpyHostToDevice));
    FM_HIP(hipMemcpy(c.d_G, c.G.data(), sizeof(double) * c.G.size(), hipMemcpyHostToDevice));
    FM_HIP(hipMemcpy(c.d_H, c.H.data(), sizeof(double) * c.H.size(), hipMemcpyHostToDevice));
    FM_HIP(hipMemcpy(c.d_t, c.t.data(), sizeof(double) * c.t.size(), hipMemcpyHostToDevice));
    {   // the pair tables in one allocation: rows (32 B each), entities (16 B), F, H
        const std::vector<double> *src[7] = {&c.lines.rows, &c.lines.rows_lo, &c.kzs.rows, &c.kzs.rows_lo,
                                             &c.F_pairs, &c.F_pairs_lo, &c.H_lo};
        const std::vector<int32_t> *ent[2] = {&c.lines.ent, &c.kzs.ent};
        size_t off[9], total = 0;
        auto place = [&](size_t bytes) {
            const size_t o = total;
            total += (bytes + 31) & ~size_t(31);
            return o;
        };
        for (int q = 0; q < 7; ++q) off[q] = place(sizeof(double) * src[q]->size());
        for (int q = 0; q < 2; ++q) off[7 + q] = place(sizeof(int32_t) * ent[q]->size());
        std::vector<char> host(total);
        for (int q = 0; q < 7; ++q) std::memcpy(host.data() + off[q], src[q]->data(), sizeof(double) * src[q]->size());
        for (int q = 0; q < 2; ++q) std::memcpy(host.data() + off[7 + q], ent[q]->data(), sizeof(int32_t) * ent[q]->size());
        FM_HIP(hipMalloc(&c.d_pairs, total));
        FM_HIP(hipMemcpy(c.d_pairs, host.data(), total, hipMemcpyHostToDevice));
        char *d = reinterpret_cast<char *>(c.d_pairs);
        c.lines.d_rows = reinterpret_cast<double4 *>(d + off[0]);
        c.lines.d_rows_lo = reinterpret_cast<double4 *>(d + off[1]);
        c.kzs.d_rows = reinterpret_cast<double4 *>(d + off[2]);
        c.kzs.d_rows_lo = reinterpret_cast<double4 *>(d + off[3]);
        c.d_F_lines = reinterpret_cast<double *>(d + off[4]);
        c.d_F_pairs = c.d_F_lines + 3 * c.n_ro;
        c.d_F_lines_lo = reinterpret_cast<double *>(d + off[5]);
        c.d_F_pairs_lo = c.d_F_lines_lo + 3 * c.n_ro;
        c.d_H_lo = reinterpret_cast<double *>(d + off[6]);
        c.lines.d_ent = reinterpret_cast<int4 *>(d + off[7]);
        c.kzs.d_ent = reinterpret_cast<int4 *>(d + off[8]);
    }
    FM_HIP(hipMalloc(&c.d_ro_group, sizeof(int32_t) * c.ro_group.size()));
    FM_HIP(hipMemcpy(c.d_ro_group, c.ro_group.data(), sizeof(int32_t) * c.ro_group.size(), hipMemcpyHostToDevice));
    return FM_OK;
}

void cartesian_free(fm_signal_plan *p)
{
    CartesianTables &c = p->cart;
    (void)hipFree(c.d_F);
    (void)hipFree(c.d_G);
    (void)hipFree(c.d_H);
    (void)hipFree(c.d_t);
    (void)hipFree(c.d_ro_group);
    (void)hipFree(c.d_pairs);
    c.d_pairs = nullptr;
    c.d_F = c.d_G = c.d_H = c.d_t = nullptr;
    c.d_ro_group = nullptr;
}


// mixed: row block 32, K stage 16 nodes, column block 32 per wave (4 per WG)
// f64:   row block 16, K stage 16 nodes (4 MFMA k-steps), column block 16 per wave
// Complex rows (pairs = false): rows are the readout indices, columns (line,
// kz, encoding).  Real rows: the lines' cosine and sine rows, columns
// (readout index, kz, encoding).
// max_total: workspace that real rows may take (they fall back on fewer node
// splits, and report total > max_total where even one does not fit).
static GemmShape gemm_shape_of(const CartesianTables &c, bool mixed, int64_t N, int V, bool pairs, size_t max_total)
{
    GemmShape s{};
    s.mixed = mixed;
    s.pairs = pairs;
    const int rowblk = s.mixed ? 32 : 16;
    const int colblk = s.mixed ? 32 : 16;
    const int max_rb = !mixed && pairs ? 8 : 4;
    const int64_t outer = pairs ? c.n_ro : c.n_ln;  // the columns' outer index
    s.N = N;
    s.Np = cdiv(std::max<int64_t>(N, 1), 16) * 16;
    s.M = pairs ? c.lines.n_rows : c.n_ro;
    const int64_t nrb = cdiv(s.M, rowblk);
    s.rb_per_wave = (int)std::min<int64_t>(max_rb, nrb);
    s.n_rt = cdiv(nrb, s.rb_per_wave);
    if (pairs) s.rb_per_wave = (int)cdiv(nrb, s.n_rt);  // tiles of equal height
    s.Mp = s.n_rt * s.rb_per_wave * rowblk;
    s.NC = outer * c.n_kz * V;
    s.n_ct = cdiv(s.NC, 4 * colblk);
    s.NCp = s.n_ct * 4 * colblk;
    s.ksteps = s.Np / 16;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        size_t o = off;
        off += (bytes + 255) & ~size_t(255);
        return o;
    };
    const size_t real = s.mixed ? sizeof(float) : sizeof(double);
    // E: Re (and Im) planes, in the mixed form each as bf16 hi, lo
    s.off_E = take((size_t)s.Mp * s.Np * (pairs ? 1 : 2) * real);
    s.off_Ey = take((size_t)outer * s.Np * 2 * real);
    s.off_Ez = take((size_t)c.n_kz * V * s.Np * 2 * real);
    const size_t per_split = (size_t)s.M * s.NC * 2 * real;
    const int64_t base = s.n_rt * s.n_ct;
    // mixed: one round of workgroups (one 8-wave or two 4-wave workgroups
    // per CU); FP64: two rounds (two 4-wave workgroups per CU, measured faster)
    const int64_t target = (s.mixed ? 2 : 4) * (int64_t)device_cu_count();
    int64_t splits = cdiv(target, base);
    // mixed: FP32 accumulators sum at most 8192 steps (131 072 nodes) per
    // split before the FP64 split reduction, bounding the accumulation error
    // for large meshes
    const int64_t s_acc = s.mixed ? cdiv(s.ksteps, 8192) : 1;
    splits = std::max(splits, s_acc);
    // small meshes: a split keeps at least 8 steps, with real rows 3 (half as
    // long a step, and more workgroups hide more of the memory latency: 4 110
    // nodes, 45 x 123, 3 encodings: GEMM 18.0 -> 15.3 us; 10 007 nodes, 64 x 64: 11.5
    // -> 8.1 us)
    splits = std::max<int64_t>(1, std::min<int64_t>(splits, cdiv(s.ksteps, pairs ? 3 : 8)));
    if (pairs) {
        const int64_t fit = off < max_total ? (int64_t)((max_total - off) / std::max<size_t>(per_split, 1)) : 0;
        splits = std::max(s_acc, std::min(splits, std::max<int64_t>(fit, 1)));
    }
    s.steps_per_split = cdiv(s.ksteps, splits);
    s.n_splits = cdiv(s.ksteps, s.steps_per_split);
    s.off_part = take((size_t)s.n_splits * per_split);
    s.total = off;
    return s;
}

// Real rows where they take fewer MFMAs (half as many per row and column
// block: 2.64 against 4.67 ms at 512 000 nodes, 128 x 128 x 32; FP64 5.93
// against 11.69 ms at 150 001 nodes, 125 x 127 x 31) and no more workspace than
// complex rows do; the FP64 form where they are no less exact (pairs_f64).
static GemmShape gemm_shape(const fm_signal_plan *p, int precision, int64_t N, int V)
{
    const CartesianTables &c = p->cart;
    const bool mixed = precision != FM_PREC_F64;
    const GemmShape g = gemm_shape_of(c, mixed, N, V, false, 0);
    if (!mixed && !c.pairs_f64) return g;
    const GemmShape s = gemm_shape_of(c, mixed, N, V, true, g.total);
    const bool fits = s.total <= g.total && s.NCp < (int64_t(1) << 31);  // column indexes in 32 bits
    return fits && s.Mp * s.NCp < 2 * g.Mp * g.NCp ? s : g;
}

size_t cartesian_workspace(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc)
{
    if (p->n_samples == 0 || n_nodes == 0) return 0;
    return gemm_shape(p, precision, n_nodes, n_enc).total;
}

// ---------------------------------------------------------------------------
// Operand tables
// ---------------------------------------------------------------------------
// exp(-2 pi i u) for u in cycles: in FP64 (FP64 form), or reduced in FP64 for the
// hardware FP32 sine/cosine, which take revolutions.
template <bool MIXED>
__device__ inline void cis_neg_cycles(double u, double &c, double &s)
{
    if (MIXED) {
        const float rf = (float)(u - __builtin_rint(u));
        c = (double)__builtin_amdgcn_cosf(rf);
        s = -(double)__builtin_amdgcn_sinf(rf);
    } else {
        sincos_cycles_f64(u, s, c);
        s = -s;
    }
}

// E tables.  Mixed: tiles of (32 rows x 16 nodes) per 4 planes (Er_h, Er_l,
// Ei_h, Ei_l), each plane in MFMA lane order: lane l holds row l%32 and
// nodes 8*(l/32) .. +7 (8 bf16 = 16 bytes).  Tile index (kstep, rowblock).
// FP64: tiles of (16 rows x 16 nodes) per 2 planes (Er, Ei), plane layout
// [kstep4 (4)][lane (64)] with lane l holding row l%16, node l/16 of that
// 4-node step.  Padding rows/nodes are zero.
//
// FP64 E table, one thread per (k-step, 4-node step, lane): the thread owns
// node n = 16 kb + 4 st + l/16 and walks the row blocks (row 16 rb + l%16),
// so a wave writes 512 contiguous bytes per plane.
__device__ __forceinline__ void cart_E_f64(int64_t t, const double *__restrict__ packed, int64_t N, int64_t Np,
                                           int64_t M, int64_t Mp, int64_t rb0, int64_t rb1, const double *__restrict__ F,
                                           const double *__restrict__ tr, double *__restrict__ E)
{
    // t over (Np / 16) * 4 * 64
    if (t >= (Np / 16) * 256) return;
    const int lane = (int)(t % 64);
    const int st = (int)((t / 64) % 4);
    const int64_t kb = t / 256;
    const int64_t nrb = Mp / 16;
    const int64_t n = kb * 16 + 4 * st + lane / 16;
    const bool ok = n < N;
    const double x = ok ? packed[n] : 0.0, y = ok ? packed[N + n] : 0.0, z = ok ? packed[2 * N + n] : 0.0;
    const double phi = ok ? packed[3 * N + n] : 0.0, r2 = ok ? packed[4 * N + n] : 0.0;
    for (int64_t rb = rb0; rb < rb1; ++rb) {
        const int64_t i = rb * 16 + (lane % 16);
        double er = 0.0, ei = 0.0;
        if (ok && i < M) {
            const double ti = tr[i];
            // total phase in cycles: -(F.x) + phi t / (2 pi)
            const double u = fma(F[3 * i], x, fma(F[3 * i + 1], y, F[3 * i + 2] * z)) - phi * ti * (1.0 / kTwoPi);
            double c, s;
            cis_neg_cycles<false>(u, c, s);
            const double d = exp(-ti * r2);
            er = d * c;
            ei = d * s;
        }
        const int64_t tile = (kb * nrb + rb) * 2;
        E[((tile + 0) * 4 + st) * 64 + lane] = er;
        E[((tile + 1) * 4 + st) * 64 + lane] = ei;
    }
}

// Mixed E table, one thread per lane fragment column: the thread owns the 8
// nodes n0..n0+7 that lane l (row l%32, node group l/32) of k-step kb feeds
// to the MFMA, keeps their attributes in registers and walks the row blocks,
// writing each of the 4 planes of a tile as one 16-byte store (a wave writes
// 1 KB contiguous per plane).  Phase in FP64 with range reduction, then the
// hardware FP32 sine/cosine and exp2.
__device__ __forceinline__ void cart_E_bf16(int64_t t, const double *__restrict__ packed, int64_t N, int64_t Np,
                                            int64_t M, int64_t Mp, int64_t rb0, int64_t rb1, const double *__restrict__ F,
                                            const double *__restrict__ tr, uint4 *__restrict__ E)
{
    // t over (Np / 16) * 64
    if (t >= (Np / 16) * 64) return;
    const int lane = (int)(t % 64);
    const int64_t kb = t / 64;
    const int64_t nrb = Mp / 32;
    const int64_t n0 = kb * 16 + 8 * (lane / 32);
    double x[8], y[8], z[8], ph[8], r2[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int64_t n = n0 + q;
        const bool ok = n < N;
        x[q] = ok ? packed[n] : 0.0;
        y[q] = ok ? packed[N + n] : 0.0;
        z[q] = ok ? packed[2 * N + n] : 0.0;
        ph[q] = ok ? packed[3 * N + n] : 0.0;
        r2[q] = ok ? packed[4 * N + n] : 0.0;
    }
    const int nvalid = (int)(N - n0 < 8 ? (N - n0 > 0 ? N - n0 : 0) : 8);
    for (int64_t rb = rb0; rb < rb1; ++rb) {
        const int64_t i = rb * 32 + (lane % 32);
        const bool row_ok = i < M;
        const double fx = row_ok ? F[3 * i] : 0.0, fy = row_ok ? F[3 * i + 1] : 0.0,
                     fz = row_ok ? F[3 * i + 2] : 0.0;
        const double ti = row_ok ? tr[i] : 0.0;
        unsigned short h[4][8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            float er = 0.0f, ei = 0.0f;
            if (row_ok && q < nvalid) {
                const double u = fma(fx, x[q], fma(fy, y[q], fz * z[q])) - ph[q] * ti * (1.0 / kTwoPi);
                const float rf = turns_f32(u);
                const float d = __builtin_amdgcn_exp2f((float)(-ti * r2[q] * 1.4426950408889634));
                er = d * __builtin_amdgcn_cosf(rf);
                ei = -d * __builtin_amdgcn_sinf(rf);
            }
            const __bf16 erh = (__bf16)er, eih = (__bf16)ei;
            const __bf16 erl = (__bf16)(er - (float)erh), eil = (__bf16)(ei - (float)eih);
            h[0][q] = __builtin_bit_cast(unsigned short, erh);
            h[1][q] = __builtin_bit_cast(unsigned short, erl);
            h[2][q] = __builtin_bit_cast(unsigned short, eih);
            h[3][q] = __builtin_bit_cast(unsigned short, eil);
        }
        const int64_t tile = kb * nrb + rb;
#pragma unroll
        for (int pl = 0; pl < 4; ++pl) {
            uint4 v;
            v.x = (unsigned)h[pl][0] | ((unsigned)h[pl][1] << 16);
            v.y = (unsigned)h[pl][2] | ((unsigned)h[pl][3] << 16);
            v.z = (unsigned)h[pl][4] | ((unsigned)h[pl][5] << 16);
            v.w = (unsigned)h[pl][6] | ((unsigned)h[pl][7] << 16);
            E[(tile * 4 + pl) * 64 + lane] = v;
        }
    }
}

// Real rows, mixed: tiles of (32 rows x 16 nodes) per 2 planes (hi, lo) in the
// lane order of cart_E_bf16; row r holds sin 2 pi (D_r . x + quarter turn of a
// cosine row).
__device__ __forceinline__ void cart_rows_bf16(int64_t t, const double *__restrict__ packed, int64_t N, int64_t Np,
                                               int64_t M, int64_t Mp, int64_t rb0, int64_t rb1, const double4 *__restrict__ rows,
                                               uint4 *__restrict__ E)
{
    // t over (Np / 16) * 64
    if (t >= (Np / 16) * 64) return;
    const int lane = (int)(t % 64);
    const int64_t kb = t / 64;
    const int64_t nrb = Mp / 32;
    const int64_t n0 = kb * 16 + 8 * (lane / 32);
    double x[8], y[8], z[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
        const int64_t n = n0 + q;
        const bool ok = n < N;
        x[q] = ok ? packed[n] : 0.0;
        y[q] = ok ? packed[N + n] : 0.0;
        z[q] = ok ? packed[2 * N + n] : 0.0;
    }
    const int nvalid = (int)(N - n0 < 8 ? (N - n0 > 0 ? N - n0 : 0) : 8);
    for (int64_t rb = rb0; rb < rb1; ++rb) {
        const int64_t i = rb * 32 + (lane % 32);
        const bool row_ok = i < M;
        const double4 d = rows[row_ok ? i : 0];
        unsigned short h[2][8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            float e = 0.0f;
            if (row_ok && q < nvalid)
                e = __builtin_amdgcn_sinf(turns_f32(fma(d.x, x[q], fma(d.y, y[q], fma(d.z, z[q], d.w)))));
            const __bf16 eh = (__bf16)e;
            const __bf16 el = (__bf16)(e - (float)eh);
            h[0][q] = __builtin_bit_cast(unsigned short, eh);
            h[1][q] = __builtin_bit_cast(unsigned short, el);
        }
        const int64_t tile = kb * nrb + rb;
#pragma unroll
        for (int pl = 0; pl < 2; ++pl) {
            uint4 v;
            v.x = (unsigned)h[pl][0] | ((unsigned)h[pl][1] << 16);
            v.y = (unsigned)h[pl][2] | ((unsigned)h[pl][3] << 16);
            v.z = (unsigned)h[pl][4] | ((unsigned)h[pl][5] << 16);
            v.w = (unsigned)h[pl][6] | ((unsigned)h[pl][7] << 16);
            E[(tile * 2 + pl) * 64 + lane] = v;
        }
    }
}

// Real rows, FP64: tiles of (16 rows x 16 nodes), one plane in the lane order
// of cart_E_f64.  Offsets in two doubles, products to about 2^-54 of a cycle
// (turns_f64), which takes the rounding of the phases (2e-15 cycles at 16 cycles)
// out of the sum.
__device__ __forceinline__ void cart_rows_f64(int64_t t, const double *__restrict__ packed, int64_t N, int64_t Np,
                                              int64_t M, int64_t Mp, int64_t rb0, int64_t rb1, const double4 *__restrict__ rows,
                                              const double4 *__restrict__ rows_lo, double *__restrict__ E)
{
    // t over (Np / 16) * 4 * 64
    if (t >= (Np / 16) * 256) return;
    const int lane = (int)(t % 64);
    const int st = (int)((t / 64) % 4);
    const int64_t kb = t / 256;
    const int64_t nrb = Mp / 16;
    const int64_t n = kb * 16 + 4 * st + lane / 16;
    const bool ok = n < N;
    const double x = ok ? packed[n] : 0.0, y = ok ? packed[N + n] : 0.0, z = ok ? packed[2 * N + n] : 0.0;
    for (int64_t rb = rb0; rb < rb1; ++rb) {
        const int64_t i = rb * 16 + (lane % 16);
        double e = 0.0;
        if (ok && i < M) {
            const double4 d = rows[i], l = rows_lo[i];
            e = sin_cycles_f64(turns_f64(d.x, l.x, x) + turns_f64(d.y, l.y, y) + turns_f64(d.z, l.z, z), d.w);
        }
        E[((kb * nrb + rb) * 4 + st) * 64 + lane] = e;
    }
}

// The columns' outer rows -- complex rows: Ey, exp(-2 pi i (G_j . x_n)) of the
// lines; real rows: Ex, exp(-t_i/T2) exp(i phi t_i) exp(-2 pi i F_i . x) of the
// readout indices -- and Ezb rows exp(-2 pi i (H_k . x_n)) b_v[n] (the
// encoding's weighted magnetisation folded into the kz factor).  One thread
// per node keeps its position in registers and walks a block of rows_blk rows
// (outer rows first, then Ezb).
template <bool MIXED, bool PAIRS>
__device__ __forceinline__ void cart_yz(int64_t n, int64_t rblk, int rows_blk, const double *__restrict__ packed, int64_t N,
                                        int64_t Np, int V, int64_t n_out, int64_t n_kz,
                                        const double *__restrict__ G, const double *__restrict__ G_lo,
                                        const double *__restrict__ tr, const double *__restrict__ H,
                                        const double *__restrict__ H_lo, void *__restrict__ Ey, void *__restrict__ Ez)
{
    if (n >= Np) return;
    const int64_t r0 = rblk * rows_blk;
    const int64_t r1 = (r0 + rows_blk < n_out + n_kz) ? r0 + rows_blk : n_out + n_kz;
    const bool ok = n < N;
    const double x = ok ? packed[n] : 0.0, y = ok ? packed[N + n] : 0.0, z = ok ? packed[2 * N + n] : 0.0;
    double phi = 0.0, r2 = 0.0;
    if (PAIRS && ok) {
        phi = packed[3 * N + n];
        r2 = packed[4 * N + n];
    }
    for (int64_t row = r0; row < r1; ++row) {
        const bool outer = row < n_out;
        const double *kv = outer ? &G[3 * row] : &H[3 * (row - n_out)];
        double c = 0.0, s = 0.0;
        if (ok) {
            double u;
            if constexpr (PAIRS && !MIXED) {
                const double *lv = outer ? &G_lo[3 * row] : &H_lo[3 * (row - n_out)];
                u = turns_f64(kv[0], lv[0], x) + turns_f64(kv[1], lv[1], y) + turns_f64(kv[2], lv[2], z);
            } else {
                u = fma(kv[0], x, fma(kv[1], y, kv[2] * z));
            }
            const double ti = PAIRS && outer ? tr[row] : 0.0;
            if (PAIRS && outer) u -= phi * ti * (1.0 / kTwoPi);
            cis_neg_cycles<MIXED>(u, c, s);
            if (PAIRS && outer) {
                const double d = MIXED ? (double)__builtin_amdgcn_exp2f((float)(-ti * r2 * 1.4426950408889634))
                                       : exp(-ti * r2);
                c *= d;
                s *= d;
            }
        }
        if (outer) {
            if (MIXED)
                reinterpret_cast<float2 *>(Ey)[row * Np + n] = make_float2((float)c, (float)s);
            else
                reinterpret_cast<double2 *>(Ey)[row * Np + n] = make_double2(c, s);
        } else {
            const int64_t k = row - n_out;
            for (int v = 0; v < V; ++v) {
                double br = 0.0, bi = 0.0;
                if (ok) {
                    br = packed[(int64_t)(5 + 2 * v) * N + n];
                    bi = packed[(int64_t)(6 + 2 * v) * N + n];
                }
                const double ar = br * c - bi * s, ai = br * s + bi * c;
                if (MIXED)
                    reinterpret_cast<float2 *>(Ez)[(k * V + v) * Np + n] = make_float2((float)ar, (float)ai);
                else
                    reinterpret_cast<double2 *>(Ez)[(k * V + v) * Np + n] = make_double2(ar, ai);
            }
        }
    }
}

// Both operand tables in one launch: blocks [0, nb_E) build the E table,
// the rest the outer and Ezb rows (nb_n node blocks x row blocks), so the two
// memory-bound jobs overlap instead of running back to back.
template <bool MIXED, bool PAIRS>
__global__ __launch_bounds__(256) void k_cart_tables(const double *__restrict__ packed, int64_t N, int64_t Np,
                                                     int64_t M, int64_t Mp, const double *__restrict__ F,
                                                     const double *__restrict__ F_lo, const double4 *__restrict__ lrows,
                                                     const double4 *__restrict__ lrows_lo,
                                                     const double *__restrict__ tr, void *__restrict__ E,
                                                     int64_t nb_E, int V, int64_t n_out, int64_t n_kz,
                                                     const double *__restrict__ G, const double *__restrict__ H,
                                                     const double *__restrict__ H_lo, void *__restrict__ Ey,
                                                     void *__restrict__ Ez, int64_t nb_n,
                                                     int e_parts, int rows_blk)
{
    // the grid is below 2^31 blocks: 32-bit divisions
    const unsigned b = blockIdx.x, nE = (unsigned)nb_E;
    if (b < nE * (unsigned)e_parts) {
        const int64_t t = (int64_t)(b % nE) * 256 + threadIdx.x;
        // this block's share of the row blocks
        const int64_t nrb = Mp / (MIXED ? 32 : 16), ep = b / nE;
        const int64_t rb0 = (unsigned)(nrb * ep) / (unsigned)e_parts, rb1 = (unsigned)(nrb * (ep + 1)) / (unsigned)e_parts;
        if (MIXED && PAIRS)
            cart_rows_bf16(t, packed, N, Np, M, Mp, rb0, rb1, lrows, reinterpret_cast<uint4 *>(E));
        else if (MIXED)
            cart_E_bf16(t, packed, N, Np, M, Mp, rb0, rb1, F, tr, reinterpret_cast<uint4 *>(E));
        else if (PAIRS)
            cart_rows_f64(t, packed, N, Np, M, Mp, rb0, rb1, lrows, lrows_lo, reinterpret_cast<double *>(E));
        else
            cart_E_f64(t, packed, N, Np, M, Mp, rb0, rb1, F, tr, reinterpret_cast<double *>(E));
        return;
    }
    const unsigned c = b - nE * (unsigned)e_parts, nn = (unsigned)nb_n;
    cart_yz<MIXED, PAIRS>((int64_t)(c % nn) * 256 + threadIdx.x, c / nn, rows_blk, packed, N, Np, V, n_out, n_kz, PAIRS ? F : G,
                          F_lo, tr, H, H_lo, Ey, Ez);
}

template <typename P, int G>
__global__ __launch_bounds__(256) void k_cart_reduce(const P *__restrict__ part, int64_t n_splits, int64_t MNC,
                                                     double2 *__restrict__ out)
{
    const int64_t i = reduce_output<G>();
    const double2 sum = reduce_sum<G>(part + i, MNC, n_splits, i < MNC);
    if (i < MNC && threadIdx.x < 256 / G) out[i] = sum;
}

template <typename P>
static void launch_cart_reduce(const void *part, int64_t n_splits, int64_t MNC, void *out, hipStream_t st)
{
    const int G = reduce_group(MNC, n_splits);
    auto *reduce = G == 8 ? k_cart_reduce<P, 8> : k_cart_reduce<P, 1>;
    reduce<<<reduce_grid(MNC, G), 256, 0, st>>>(reinterpret_cast<const P *>(part), n_splits, MNC,
                                                reinterpret_cast<double2 *>(out));
}

// Samples from the partial sums over real rows: Lr cosine and sine rows of the
// lines and, KPAIR, Kr rows of the kz planes (else Kr = K planes with their own
// complex columns); readout index i, line row r, column q V + v of one split
// at i si + r sr + q V + v, M Lr Kr V to a split.  One thread
// group of G sums the splits of one (readout, line entity, kz entity,
// encoding) in FP64, each thread a contiguous share of them, the shares added
// in order, and writes the entity's up to four samples:
//   (C_a -+ i S_a) (C_b -+ i S_b) = CC - s_a s_b SS - i (s_b CS + s_a SC).
template <typename P, int OL, bool KPAIR>
__global__ __launch_bounds__(256) void k_cart_reduce_pairs(
    const P *__restrict__ part, int64_t n_splits, int64_t M, int64_t per_split, int64_t si, int64_t sr, int64_t V,
    const int4 *__restrict__ lent, int64_t n_lent, const int4 *__restrict__ kent, int64_t n_kent, int64_t L, int64_t K,
    double2 *__restrict__ out)
{
    constexpr int GL = 64 / OL, G = 4 * GL;  // shares in a wave, in the workgroup
    constexpr int NC = KPAIR ? 4 : 2;        // sums per group: (line cosine, sine) x (kz cosine, sine)
    __shared__ double2 sum[4][NC][OL];
    const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
    const int o = lane % OL, g = wave * GL + lane / OL;
    const int64_t t = (int64_t)blockIdx.x * OL + o;
    const int64_t n_out = M * n_lent * n_kent * V;
    const bool live = t < n_out;
    // the index that is contiguous in `part` runs first (7 434 nodes, 121 x 140,
    // 4 encodings: 22.5 -> 14.4 us): after (kz, encoding)
    // the line rows of a readout index (KPAIR), or the readout indices of a row
    const int64_t na = KPAIR ? n_lent : M;
    int64_t v, e, a, b;
    if (n_out < (int64_t(1) << 31)) {  // 32-bit division: a fifth of the instructions
        unsigned r = live ? (unsigned)t : 0u;
        v = r % (unsigned)V;
        r /= (unsigned)V;
        e = r % (unsigned)n_kent;
        r /= (unsigned)n_kent;
        a = r % (unsigned)na;
        b = r / (unsigned)na;
    } else {
        const int64_t r = live ? t : 0;
        v = r % V;
        e = (r / V) % n_kent;
        a = (r / (V * n_kent)) % na;
        b = r / (V * n_kent * na);
    }
    const int64_t f = KPAIR ? a : b, i = KPAIR ? b : a;
    const int4 le = lent[f];
    const int4 ke = KPAIR ? kent[e] : make_int4((int)e, -1, (int)e, -1);
    const int rows[2] = {le.z, le.w}, cols[2] = {ke.z, ke.w};
    const int64_t s0 = n_splits * g / G, s1 = n_splits * (g + 1) / G;
    // the sums advance together, so their loads overlap
    double re[NC], im[NC];
    const P *src[NC];
    bool on[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int r = rows[KPAIR ? c / 2 : c], q = cols[KPAIR ? c % 2 : 0];
        re[c] = im[c] = 0.0;
        on[c] = live && r >= 0 && q >= 0;
        src[c] = part + (on[c] ? i * si + r * sr + q * V + v : 0) + s0 * per_split;
    }
#pragma unroll 4
    for (int64_t s = s0; s < s1; ++s) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if (on[c]) {
                const P x = *src[c];
                re[c] += (double)x.x;
                im[c] += (double)x.y;
                src[c] += per_split;
            }
        }
    }
    // shares of a wave, then of the four waves, each in a fixed order
#pragma unroll
    for (int c = 0; c < NC; ++c) {
#pragma unroll
        for (int d = OL; d < 64; d *= 2) {
            re[c] += __shfl_xor(re[c], d, 64);
            im[c] += __shfl_xor(im[c], d, 64);
        }
        if (lane < OL) sum[wave][c][o] = make_double2(re[c], im[c]);
    }
    __syncthreads();
    // one thread per sample of the group
    const int c = threadIdx.x / OL;
    if (c >= 4 || !live) return;
    const int j = c / 2 ? le.y : le.x, k = c % 2 ? ke.y : ke.x;
    if (j < 0 || k < 0) return;
    double2 w[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        w[q] = make_double2(0.0, 0.0);
        if (!KPAIR && q % 2) continue;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const double2 y = sum[x][KPAIR ? q : q / 2][o];
            w[q].x += y.x;
            w[q].y += y.y;
        }
    }
    // w: CC, CS (kz sine), SC (line sine), SS
    const double sa = c / 2 ? -1.0 : 1.0, sb = c % 2 ? -1.0 : 1.0;
    const double ar = w[0].x - sa * sb * w[3].x, ai = w[0].y - sa * sb * w[3].y;
    const double br = sb * w[1].x + sa * w[2].x, bi = sb * w[1].y + sa * w[2].y;
    out[((i * L + j) * K + k) * V + v] = make_double2(ar + bi, ai - br);
}

// 16 groups of samples to a workgroup (16 shares of the splits) where the
// samples alone would leave most of the device idle in a long chain of loads,
// else 64 (4 shares).  Whole calls of 10 007 nodes, mixed, 16 against 64 groups: 32 x 32
// (512 groups of samples) 22 against 41 us, 128 x 128 (8192) 37 and 48, 128 x 128 x 4 (32 768) 38 and
// 44, x 8 (65 536) 52 and 50, x 16 64 and 61.
template <typename P, bool KPAIR>
static void launch_reduce_pairs(const P *part, int64_t n_splits, int64_t si, int64_t sr, int64_t V,
                                const CartesianTables &c, double2 *out, hipStream_t st)
{
    const int64_t M = c.n_ro;
    const int64_t per_split = M * c.lines.n_rows * (KPAIR ? c.kzs.n_rows : c.n_kz) * V;
    const int64_t n_kent = KPAIR ? c.kzs.n_ent : c.n_kz;
    const int64_t n = M * c.lines.n_ent * n_kent * V;
    if (n < 64 * 1024)
        k_cart_reduce_pairs<P, 16, KPAIR><<<(unsigned)cdiv(n, 16), 256, 0, st>>>(
            part, n_splits, M, per_split, si, sr, V, c.lines.d_ent, c.lines.n_ent, c.kzs.d_ent, n_kent, c.n_ln, c.n_kz,
            out);
    else
        k_cart_reduce_pairs<P, 64, KPAIR><<<(unsigned)cdiv(n, 64), 256, 0, st>>>(
            part, n_splits, M, per_split, si, sr, V, c.lines.d_ent, c.lines.n_ent, c.kzs.d_ent, n_kent, c.n_ln, c.n_kz,
            out);
}

int cartesian_execute(const fm_signal_plan *p, int precision, int64_t N, int V, const double *packed, void *wsv,
                      size_t ws_bytes, double *out, hipStream_t st)
{
    const CartesianTables &c = p->cart;
    const int64_t S = p->n_samples;
    if (S == 0) return FM_OK;
    if (N == 0) {
        return zero_f64_async(out, 2 * S * V, st);
    }
    const GemmShape s = gemm_shape(p, precision, N, V);
    if (s.total > ws_bytes) {
        set_error("signal workspace too small: need %zu bytes, got %zu", s.total, ws_bytes);
        return FM_ERR_WORKSPACE;
    }
    char *ws = reinterpret_cast<char *>(wsv);
    const int64_t n_kzV = c.n_kz * V;
    {
        const int64_t nb_E = s.mixed ? cdiv(s.Np / 16 * 64, 256) : cdiv(s.Np / 16 * 256, 256);
        const int64_t nb_n = cdiv(s.Np, 256);
        const int64_t n_out = s.pairs ? c.n_ro : c.n_ln;
        // small meshes: the row blocks and rows shared among more blocks, until
        // there are some 4 per CU (4 110 nodes, 45 x 123: 9.9 -> 6.0 us)
        const int64_t nrb = s.Mp / (s.mixed ? 32 : 16), want = 4 * (int64_t)device_cu_count();
        const int e_parts = (int)std::max<int64_t>(1, std::min(nrb, want / std::max<int64_t>(2 * nb_E, 1)));
        int rows_blk = 16;
        while (rows_blk > 2 && nb_n * cdiv(n_out + c.n_kz, rows_blk) < want) rows_blk /= 2;
        const int64_t nb = nb_E * e_parts + nb_n * cdiv(n_out + c.n_kz, rows_blk);
        if (nb > (int64_t)0x7fffffff) {
            set_error("Cartesian operand tables exceed the launch grid (%lld blocks)", (long long)nb);
            return FM_ERR_UNSUPPORTED;
        }
#define FM_TABLES(MX, PR)                                                                                            \
    k_cart_tables<MX, PR><<<(unsigned)nb, 256, 0, st>>>(packed, N, s.Np, s.M, s.Mp, PR ? c.d_F_lines : c.d_F,       \
                                                        c.d_F_lines_lo, c.lines.d_rows, c.lines.d_rows_lo, c.d_t,    \
                                                        ws + s.off_E, nb_E, V, n_out, c.n_kz, c.d_G, c.d_H, c.d_H_lo, \
                                                        ws + s.off_Ey, ws + s.off_Ez, nb_n, e_parts, rows_blk)
        if (s.mixed && s.pairs) FM_TABLES(true, true);
        else if (s.mixed) FM_TABLES(true, false);
        else if (s.pairs) FM_TABLES(false, true);
        else FM_TABLES(false, false);
#undef FM_TABLES
        FM_LAUNCH_CHECK("k_cart_tables");
    }
    if (s.mixed) {
        plan_timing_start(p, st);
        launch_cart_gemm_bf16(s, ws, n_kzV, st);
        plan_timing_stop(p, st);
        FM_LAUNCH_CHECK("k_cart_gemm_bf16");
        const int64_t MNC = s.M * s.NC;
        if (s.pairs)
            launch_reduce_pairs<float2, false>(reinterpret_cast<const float2 *>(ws + s.off_part), s.n_splits, n_kzV,
                                               s.NC, V, c, reinterpret_cast<double2 *>(out), st);
        else launch_cart_reduce<float2>(ws + s.off_part, s.n_splits, MNC, out, st);
    } else {
        plan_timing_start(p, st);
        launch_cart_gemm_f64(s, ws, n_kzV, st);
        plan_timing_stop(p, st);
        FM_LAUNCH_CHECK("k_cart_gemm_f64");
        const int64_t MNC = s.M * s.NC;
        if (s.pairs)
            launch_reduce_pairs<double2, false>(reinterpret_cast<const double2 *>(ws + s.off_part), s.n_splits, n_kzV,
                                                s.NC, V, c, reinterpret_cast<double2 *>(out), st);
        else launch_cart_reduce<double2>(ws + s.off_part, s.n_splits, MNC, out, st);
    }
    FM_LAUNCH_CHECK("k_cart_reduce");
    return FM_OK;
}

// The moving form a shape takes: real rows where the plan has them.
static MovingShape moving_form(const CartesianTables &c, bool f64, int64_t N, int V)
{
    const MovingShape s = f64 ? moving_pairs_shape_f64(c, N, V) : moving_pairs_shape(c, N, V);
    return s.pairs ? s : (f64 ? moving_shape_f64(c, N, V) : moving_shape(c, N, V));
}

int cartesian_route(const fm_signal_plan *p, int precision, int64_t N, int V, bool moving, int64_t *n_splits)
{
    bool pairs;
    if (moving) {
        const MovingShape s = moving_form(p->cart, precision == FM_PREC_F64, N, V);
        pairs = s.pairs;
        *n_splits = s.n_splits;
    } else {
        const GemmShape s = gemm_shape(p, precision, N, V);
        pairs = s.pairs;
        *n_splits = s.n_splits;
    }
    return pairs ? FM_ROUTE_CARTESIAN_REAL : FM_ROUTE_CARTESIAN;
}

size_t cartesian_moving_workspace(const fm_signal_plan *p, int precision, int64_t N, int V)
{
    if (p->n_samples == 0 || N == 0 || V > kMovMaxV) return 0;
    return moving_form(p->cart, precision == FM_PREC_F64, N, V).part_bytes;
}

int cartesian_moving_execute(const fm_signal_plan *p, int precision, int64_t N, int V, const double *packed,
                             const float *modes, int R, const double *mcoef, void *ws, size_t ws_bytes, double *out,
                             hipStream_t st)
{
    const CartesianTables &c = p->cart;
    const int64_t S = p->n_samples;
    if (S == 0) return FM_OK;
    if (N == 0) {
        return zero_f64_async(out, 2 * S * V, st);
    }
    if (V > kMovMaxV) {
        set_error("moving Cartesian GEMM takes at most %d encodings per call (got %d)", kMovMaxV, V);
        return FM_ERR_UNSUPPORTED;
    }
    const bool f64 = precision == FM_PREC_F64;
    const MovingShape s = moving_form(c, f64, N, V);
    if (s.part_bytes > ws_bytes) {
        set_error("signal workspace too small: need %zu bytes, got %zu", s.part_bytes, ws_bytes);
        return FM_ERR_WORKSPACE;
    }
    const int64_t grid = s.n_splits * s.M * s.n_rt * s.n_ct;
    if (grid > (int64_t)0x7fffffff) {
        set_error("moving Cartesian GEMM exceeds the launch grid (%lld workgroups)", (long long)grid);
        return FM_ERR_UNSUPPORTED;
    }
    const int64_t MNC = s.M * s.L * s.KV;
    plan_timing_start(p, st);
    if (f64) {
        double2 *part = reinterpret_cast<double2 *>(ws);
        launch_cart_moving_f64(s, c, packed, N, modes, R, mcoef, part, st);
        plan_timing_stop(p, st);
        FM_LAUNCH_CHECK("k_cart_moving_f64");
        if (s.pairs)
            launch_reduce_pairs<double2, true>(part, s.n_splits, s.L * s.KV, s.KV, s.V, c,
                                               reinterpret_cast<double2 *>(out), st);
        else launch_cart_reduce<double2>(part, s.n_splits, MNC, out, st);
    } else {
        float2 *part = reinterpret_cast<float2 *>(ws);
        if (s.pairs) launch_cart_moving_pairs_bf16(s, c, packed, N, modes, R, mcoef, part, st);
        else launch_cart_moving_bf16(s, c, packed, N, modes, R, mcoef, part, st);
        plan_timing_stop(p, st);
        FM_LAUNCH_CHECK("k_cart_moving_bf16");
        if (s.pairs)
            launch_reduce_pairs<float2, true>(part, s.n_splits, s.L * s.KV, s.KV, s.V, c,
                                              reinterpret_cast<double2 *>(out), st);
        else launch_cart_reduce<float2>(part, s.n_splits, MNC, out, st);
    }
    FM_LAUNCH_CHECK("k_cart_reduce");
    return FM_OK;
}

}  // namespace fm
