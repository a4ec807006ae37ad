// Moving nodes on a Cartesian stack whose lines (along y) and kz planes
// (along z) pair up about a centre: the per-readout product of
// cart_moving_bf16.hip with real rows (PairAxis), mixed form.
//
//   P[i, r, (q,v)] = sum_n A_i[r,n] B_i[n,(q,v)]              (per readout index i)
//   A_i[r,n]       = cos or sin of 2 pi D_r y_n(t_i)           (line rows, real)
//   B_i[n,(q,v)]   = (cos or sin of 2 pi D_q z_n(t_i)) c_i[n,v]  (kz rows, complex by c)
//   c_i[n,v]       = b_v[n] exp(-t_i/T2_n) exp(i phi_n t_i) exp(-2 pi i F'_i . x_n(t_i))
//
// with F' = F + the centres.  The sample at line c +- D_a, plane c +- D_b is a
// signed sum of the four partial sums (cos or sin) x (cos or sin)
// (k_cart_reduce_pairs).  Against complex rows this halves the matrix
// products (6 MFMAs per 32 x 32 block and 16 nodes instead of 12) and the
// operand build (one sine and one hi/lo split per row and node instead of a
// sine, a cosine and two splits; two products per B entry instead of four).
//
// Per chunk of 64 W nodes each thread forms one node record in LDS (y, z in
// FP64, c_i in FP32).  Per 16-node step:
//   * kz rows of the step after the next into LDS (FP64 phase plus a quarter
//     turn for cosine rows, one fract, FP32 hardware sine);
//   * B fragments of the next step, bf16 hi + lo planes, into the other of
//     two LDS buffers; A fragments of the next step in registers (lane l: row
//     32 (W rt + w) + l%32, nodes 8 (l/32) .. +7);
//   * 6 v_mfma_f32_32x32x16_bf16 per column block on this step's operands:
//     Re += A Re B, Im += A Im B, each as hh + hl + lh;
//   * one barrier.
//
// Bound: VALU and MFMA issue, which add up on a SIMD (counters: VALU issue 54 %
// of the cycles, MFMA 43 %).  1 948 800 nodes, 96 x 96 x 24, 4 encodings, 10
// modes: 23.0 ms per call against 35.5 ms with complex rows, 600 against 390
// TFLOP/s of 8 flops per node * sample * encoding; error against 64 bits
// 6.7e-7 against 9.7e-7.
// Rows and columns past the last are computed on clamped indices and not
// written; nodes past the last have c = 0.
#include <algorithm>
#include <type_traits>

#include "cart_gemm.h"

namespace fm {

typedef __attribute__((ext_vector_type(2))) float mp_f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 mp_bf16x2;

// bf16 hi + lo planes of 8 values.
__device__ inline void split8_real(const float (&x)[8], bf16x8 &h, bf16x8 &l)
{
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const mp_f32x2 v = {x[2 * p], x[2 * p + 1]};
        const mp_bf16x2 vh = __builtin_convertvector(v, mp_bf16x2);
        const mp_bf16x2 vl = __builtin_convertvector(v - __builtin_convertvector(vh, mp_f32x2), mp_bf16x2);
        h[2 * p] = vh[0];
        h[2 * p + 1] = vh[1];
        l[2 * p] = vl[0];
        l[2 * p + 1] = vl[1];
    }
}

// sin 2 pi u, u in cycles: FP64 range reduction, FP32 hardware sine.
__device__ inline float sin_turns_f32(double u) { return __builtin_amdgcn_sinf(turns_f32(u)); }

// floats per kz row of the kz buffer: 16 nodes + 4 of pad (rows 16-byte aligned)
constexpr int kKzStride = 20;

template <int W, int CB>
__global__ __launch_bounds__(64 * W, (CB <= 3 ? 3 : 2)) void k_cart_moving_pairs_bf16(
    const double *__restrict__ packed, int64_t N, int V, const float *__restrict__ modes, int R,
    const double *__restrict__ mcoef, const int32_t *__restrict__ ro_group, const double *__restrict__ F,
    const double4 *__restrict__ lrows, const double4 *__restrict__ krows, const double *__restrict__ tr, int64_t M,
    int64_t L, int64_t K, int64_t n_rt, int64_t n_ct, int64_t n_splits, int64_t nodes_per_split, int kz_rows,
    float2 *__restrict__ part)
{
    constexpr int kThreads = 64 * W;
    constexpr int kChunk = kThreads;       // nodes per record chunk
    constexpr int kSteps = kChunk / 16;    // 16-node steps per chunk (even)
    constexpr int kCols = 32 * CB;         // columns of the workgroup tile
    constexpr int kBF = (CB + W - 1) / W;  // B fragments per thread
    __shared__ double sy[kChunk], sz[kChunk];
    __shared__ float2 sc[kMovMaxV][kChunk + 2];
    __shared__ uint4 sB0[CB * 4 * 64], sB1[CB * 4 * 64];
    __shared__ double2 sH[kCols + 1];      // (D, quarter) of the tile's kz rows
    __shared__ double scoef[kMaxModes + 3];
    extern __shared__ float4 sKz4[];       // 2 buffers of kz_rows rows of kKzStride floats
    float *const sKz = reinterpret_cast<float *>(sKz4);

    // workgroup -> (split, readout index, row tile, column tile); the ids of
    // one split are contiguous and dealt onto one XCD
    const int64_t total = n_splits * M * n_rt * n_ct;
    const int64_t h = blockIdx.x;
    int64_t lg = h;
    if (total % kXcds == 0) lg = (h % kXcds) * (total / kXcds) + h / kXcds;
    const int64_t ct = lg % n_ct;
    int64_t rest = lg / n_ct;
    const int64_t rt = rest % n_rt;
    rest /= n_rt;
    const int64_t i = rest % M;
    const int64_t split = rest / M;

    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int64_t KV = K * V;
    const int64_t n_begin = split * nodes_per_split;
    const int64_t n_end = (n_begin + nodes_per_split < N) ? n_begin + nodes_per_split : N;

    const double ti = tr[i];
    const double Fx = F[3 * i], Fy = F[3 * i + 1], Fz = F[3 * i + 2];
    const int64_t grp = ro_group[i];
    for (int q = tid; q < R + 3; q += kThreads) scoef[q] = mcoef[grp * (R + 3) + q];

    // this lane's A row
    const int64_t row = (rt * W + wave) * 32 + (lane % 32);
    const double4 lr = lrows[row < L ? row : L - 1];
    const double Dy = lr.y, qy = lr.w;

    // the column tile's kz rows
    const int64_t c0 = ct * kCols;
    const int64_t kmin = c0 / V;
    const int64_t kmax = std::min<int64_t>(K - 1, (c0 + kCols - 1) / V);
    const int nk = (int)(kmax - kmin + 1);  // <= kz_rows
    for (int q = tid; q < nk; q += kThreads) {
        const double4 kr = krows[kmin + q];
        sH[q] = make_double2(kr.z, kr.w);
    }

    // this thread's B fragments: fragment f = tid + r kThreads feeds lane
    // f % 64 (= lane) of column block f / 64
    int bkk[kBF], bv[kBF];
#pragma unroll
    for (int r = 0; r < kBF; ++r) {
        const int f = tid + r * kThreads;
        const int64_t c = c0 + (f / 64) * 32 + (lane % 32);
        const bool ok = f < CB * 64 && c < KV;
        bkk[r] = ok ? (int)(c / V - kmin) * kKzStride : 0;
        bv[r] = ok ? (int)(c % V) : 0;
    }

    f32x16 acc_re[CB], acc_im[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int q = 0; q < 16; ++q) acc_re[cb][q] = acc_im[cb][q] = 0.0f;

    const int kz_buf = kz_rows * kKzStride;
    const int half = lane / 32;

    // kz rows of step s's 16 nodes into kz buffer s % 2
    auto kz_gen = [&](int s) {
        float *dst = sKz + (s & 1) * kz_buf;
        for (int e = tid; e < nk * 16; e += kThreads) {
            const int kk = e / 16, m = e % 16;
            const double2 hk = sH[kk];
            dst[kk * kKzStride + m] = sin_turns_f32(fma(hk.x, sz[s * 16 + m], hk.y));
        }
    };
    // B fragments of step s into `dst0`
    auto b_gen = [&](int s, uint4 *dst0) {
        const float *kz = sKz + (s & 1) * kz_buf;
#pragma unroll
        for (int r = 0; r < kBF; ++r) {
            const int f = tid + r * kThreads;
            if (CB % W == 0 || f < CB * 64) {
                float br[8], bi[8];
                const float4 *a4 = reinterpret_cast<const float4 *>(kz + bkk[r] + 8 * half);
                const float4 *c4 = reinterpret_cast<const float4 *>(&sc[bv[r]][s * 16 + 8 * half]);
                const float4 a0 = a4[0], a1 = a4[1];
                const float a[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 c = c4[q];
                    br[2 * q] = a[2 * q] * c.x;
                    bi[2 * q] = a[2 * q] * c.y;
                    br[2 * q + 1] = a[2 * q + 1] * c.z;
                    bi[2 * q + 1] = a[2 * q + 1] * c.w;
                }
                bf16x8 rh, rl, ih, il;
                split8_real(br, rh, rl);
                split8_real(bi, ih, il);
                uint4 *dst = dst0 + (f / 64) * 4 * 64 + lane;
                dst[0 * 64] = __builtin_bit_cast(uint4, rh);
                dst[1 * 64] = __builtin_bit_cast(uint4, rl);
                dst[2 * 64] = __builtin_bit_cast(uint4, ih);
                dst[3 * 64] = __builtin_bit_cast(uint4, il);
            }
        }
    };
    // A fragment of step s
    auto a_gen = [&](int s, bf16x8 &ah, bf16x8 &al) {
        float a[8];
        const double *y = &sy[s * 16 + 8 * half];
#pragma unroll
        for (int q = 0; q < 8; ++q) a[q] = sin_turns_f32(fma(Dy, y[q], qy));
        split8_real(a, ah, al);
    };
    auto products = [&](const uint4 *src0, const bf16x8 ah, const bf16x8 al) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const uint4 *src = src0 + cb * 4 * 64 + lane;
            const bf16x8 brh = __builtin_bit_cast(bf16x8, src[0 * 64]);
            const bf16x8 brl = __builtin_bit_cast(bf16x8, src[1 * 64]);
            const bf16x8 bih = __builtin_bit_cast(bf16x8, src[2 * 64]);
            const bf16x8 bil = __builtin_bit_cast(bf16x8, src[3 * 64]);
            acc_re[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, brh, acc_re[cb], 0, 0, 0);
            acc_im[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bih, acc_im[cb], 0, 0, 0);
            acc_re[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, brl, acc_re[cb], 0, 0, 0);
            acc_im[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah, bil, acc_im[cb], 0, 0, 0);
            acc_re[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, brh, acc_re[cb], 0, 0, 0);
            acc_im[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al, bih, acc_im[cb], 0, 0, 0);
        }
    };

    for (int64_t base = n_begin; base < n_end; base += kChunk) {
        __syncthreads();  // previous chunk consumed; scoef and sH visible
        {
            const int64_t n = base + tid;
            double x = 0.0, y = 0.0, z = 0.0;
            float2 cv[kMovMaxV];
#pragma unroll
            for (int v = 0; v < kMovMaxV; ++v) cv[v] = make_float2(0.0f, 0.0f);
            if (n < n_end) {
                double dx = scoef[R], dy = scoef[R + 1], dz = scoef[R + 2];
                for (int r = 0; r < R; ++r) {
                    const double w = scoef[r];
                    dx += (double)modes[(int64_t)(0 * R + r) * N + n] * w;
                    dy += (double)modes[(int64_t)(1 * R + r) * N + n] * w;
                    dz += (double)modes[(int64_t)(2 * R + r) * N + n] * w;
                }
                x = packed[n] + dx;
                y = packed[N + n] + dy;
                z = packed[2 * N + n] + dz;
                const double phi = packed[3 * N + n], r2 = packed[4 * N + n];
                // c = b exp(-t/T2) exp(i phi t) exp(-2 pi i F'.x)   (MRI.cpp:124-146)
                const double u = fma(Fx, x, fma(Fy, y, Fz * z)) - phi * ti * (1.0 / kTwoPi);
                const float rf = turns_f32(u);
                const float d = __builtin_amdgcn_exp2f((float)(-ti * r2 * 1.4426950408889634));
                const float er = d * __builtin_amdgcn_cosf(rf), ei = -d * __builtin_amdgcn_sinf(rf);
#pragma unroll
                for (int v = 0; v < kMovMaxV; ++v) {
                    if (v < V) {
                        const float br = (float)packed[(int64_t)(5 + 2 * v) * N + n];
                        const float bi = (float)packed[(int64_t)(6 + 2 * v) * N + n];
                        cv[v] = make_float2(br * er - bi * ei, br * ei + bi * er);
                    }
                }
            }
            sy[tid] = y;
            sz[tid] = z;
#pragma unroll
            for (int v = 0; v < kMovMaxV; ++v) sc[v][tid] = cv[v];
        }
        __syncthreads();
        kz_gen(0);
        __syncthreads();
        bf16x8 ah, al;
        kz_gen(1);
        b_gen(0, sB0);
        a_gen(0, ah, al);
        __syncthreads();
        // step s: products on buffer s % 2, operands of s + 1 into the other
        // (AHEAD: how many further steps there are, at most 2)
        auto step = [&](int s, const uint4 *cur, uint4 *nxt, auto ahead) {
            constexpr int AHEAD = decltype(ahead)::value;
            bf16x8 nh, nl;
            if constexpr (AHEAD >= 2) kz_gen(s + 2);
            if constexpr (AHEAD >= 1) {
                b_gen(s + 1, nxt);
                a_gen(s + 1, nh, nl);
            }
            products(cur, ah, al);
            if constexpr (AHEAD >= 1) {
                ah = nh;
                al = nl;
            }
            __syncthreads();
        };
        using I0 = std::integral_constant<int, 0>;
        using I1 = std::integral_constant<int, 1>;
        using I2 = std::integral_constant<int, 2>;
        for (int s = 0; s < kSteps - 2; s += 2) {
            step(s, sB0, sB1, I2{});
            step(s + 1, sB1, sB0, I2{});
        }
        step(kSteps - 2, sB0, sB1, I1{});
        step(kSteps - 1, sB1, sB0, I0{});
    }

    // acc register q of lane l holds row 8 (q/4) + 4 (l/32) + q%4 and column
    // l%32 of its 32x32 block
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        const int64_t col = c0 + cb * 32 + (lane % 32);
        if (col >= KV) continue;
#pragma unroll
        for (int q = 0; q < 16; ++q) {
            const int64_t r = (rt * W + wave) * 32 + 8 * (q / 4) + 4 * half + (q % 4);
            if (r < L) part[((split * M + i) * L + r) * KV + col] = make_float2(acc_re[cb][q], acc_im[cb][q]);
        }
    }
}

static size_t pairs_dyn_lds(const MovingShape &s) { return 2 * (size_t)s.ez_rows * kKzStride * sizeof(float); }

template <int W>
static int pairs_blocks_w(int CB, size_t dyn)
{
    switch (CB) {
    case 1: return blocks_per_cu(k_cart_moving_pairs_bf16<W, 1>, 64 * W, dyn);
    case 2: return blocks_per_cu(k_cart_moving_pairs_bf16<W, 2>, 64 * W, dyn);
    case 3: return blocks_per_cu(k_cart_moving_pairs_bf16<W, 3>, 64 * W, dyn);
    default: return blocks_per_cu(k_cart_moving_pairs_bf16<W, 4>, 64 * W, dyn);
    }
}

// Workgroups of the shape's instantiation that one CU holds at once.
static int pairs_blocks_per_cu(const MovingShape &s)
{
    const size_t dyn = pairs_dyn_lds(s);
    switch (s.W) {
    case 1: return pairs_blocks_w<1>(s.CB, dyn);
    case 2: return pairs_blocks_w<2>(s.CB, dyn);
    case 3: return pairs_blocks_w<3>(s.CB, dyn);
    default: return pairs_blocks_w<4>(s.CB, dyn);
    }
}

MovingShape moving_pairs_shape(const CartesianTables &c, int64_t N, int V)
{
    MovingShape s{};
    const MovingShape g = moving_shape(c, N, V);
    s.M = c.n_ro;
    s.L = c.lines.n_rows;
    s.K = c.kzs.n_rows;
    s.V = V;
    s.KV = s.K * V;
    const int64_t nrb = cdiv(s.L, 32), ncb = cdiv(s.KV, 32);
    s.W = (int)std::min<int64_t>(4, nrb);
    s.CB = (int)std::min<int64_t>(4, ncb);
    s.n_rt = cdiv(nrb, s.W);
    s.n_ct = cdiv(ncb, s.CB);
    // used where it runs fewer MFMAs, 6 per 32 x 32 block against 12 (the time
    // follows them: 23.0 against 35.5 ms at half the products): sets with many
    // unpaired lines or planes keep the complex rows, as do rotated stacks,
    // whose phases take three products instead of one
    if (!c.axis_aligned || s.n_rt * s.W * s.n_ct * s.CB >= 2 * g.n_rt * g.W * g.n_ct * g.CB) return s;
    const int64_t n1 = std::max<int64_t>(N, 1);
    const int64_t chunk = 64 * s.W;
    const int64_t base = s.M * s.n_rt * s.n_ct;
    const int64_t cols = 32 * (int64_t)s.CB;
    s.ez_rows = (int)std::min<int64_t>(cols, (cols - 1) / V + 2);
    // splits as the general form chooses them (FP32 accumulation over at most
    // ~16 384 nodes, whole rounds of workgroups), within its workspace
    const size_t per_split = (size_t)s.M * (size_t)s.L * (size_t)s.KV * sizeof(float2);
    const int64_t s_max = (int64_t)(g.part_bytes / std::max<size_t>(per_split, 1));
    const int64_t s_acc = cdiv(n1, 16384);
    if (s_max < s_acc || s_max < 1) return s;
    const int64_t s_min = std::max(cdiv(4 * (int64_t)device_cu_count(), base), s_acc);
    const int64_t capacity = (int64_t)pairs_blocks_per_cu(s) * device_cu_count();
    const int64_t splits = balanced_splits(N, chunk, base, s_min, capacity, s_max);
    s.nodes_per_split = cdiv(cdiv(n1, splits), chunk) * chunk;
    s.n_splits = cdiv(n1, s.nodes_per_split);
    s.part_bytes = (size_t)s.n_splits * per_split;
    s.pairs = true;
    return s;
}

template <int W>
static void launch_pairs_w(const MovingShape &s, const CartesianTables &c, const double *packed, int64_t N,
                           const float *modes, int R, const double *mcoef, float2 *part, hipStream_t st)
{
    const unsigned grid = (unsigned)(s.n_splits * s.M * s.n_rt * s.n_ct);
    const size_t dyn = pairs_dyn_lds(s);
#define FM_MP(CBV)                                                                                                  \
    k_cart_moving_pairs_bf16<W, CBV><<<grid, 64 * W, dyn, st>>>(                                                   \
        packed, N, (int)s.V, modes, R, mcoef, c.d_ro_group, c.d_F_pairs, c.lines.d_rows, c.kzs.d_rows, c.d_t, s.M, \
        s.L, s.K, s.n_rt, s.n_ct, s.n_splits, s.nodes_per_split, s.ez_rows, part)
    switch (s.CB) {
    case 1: FM_MP(1); break;
    case 2: FM_MP(2); break;
    case 3: FM_MP(3); break;
    default: FM_MP(4); break;
    }
#undef FM_MP
}

void launch_cart_moving_pairs_bf16(const MovingShape &s, const CartesianTables &c, const double *packed, int64_t N,
                                   const float *modes, int R, const double *mcoef, float2 *part, hipStream_t st)
{
    switch (s.W) {
    case 1: launch_pairs_w<1>(s, c, packed, N, modes, R, mcoef, part, st); break;
    case 2: launch_pairs_w<2>(s, c, packed, N, modes, R, mcoef, part, st); break;
    case 3: launch_pairs_w<3>(s, c, packed, N, modes, R, mcoef, part, st); break;
    default: launch_pairs_w<4>(s, c, packed, N, modes, R, mcoef, part, st); break;
    }
}

}  // namespace fm
