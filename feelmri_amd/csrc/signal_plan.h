// Internal layout of fm_signal_plan (shared by the direct and Cartesian paths).
#pragma once
#include <vector>

#include "fm_common.h"

namespace fm {

// Samples handled by one workgroup of the direct kernels (256 lanes x 2).
constexpr int kDirectThreads = 256;
constexpr int kDirectSPL = 2;
constexpr int kDirectTile = kDirectThreads * kDirectSPL;
// Encodings handled per direct launch (register-resident accumulators).
constexpr int kMaxVB = 4;
// Upper bound on POD modes fused into the loaders.
constexpr int kMaxModes = 32;
// Encodings per launch of the moving-node Cartesian GEMM (node records in LDS).
constexpr int kMovMaxV = 4;

// t-groups of one tile, at most.
constexpr int kGroupCap = 32;
// Static nodes take the t-grouped tiles from this many samples per group on
// average (32 groups then fill a tile's 256 lanes), else per-sample t (spiral,
// 61 394 nodes, 568 x 16, FP64: 0.71 ms grouped, 1.80 ms per-sample t).
constexpr double kGroupMin = 16.0;

// Readout runs (mixed-form direct kernel for static nodes): kRunLen
// consecutive readout samples of one line whose k and t are linear in the
// readout index, so exp(-2 pi i k.x) exp((i phi - 1/T2) t) advances by one
// complex factor per sample.
constexpr int kRunLen = 16;

struct RunDesc {
    double k0x, k0y, k0z, t0;  // first sample (k' in cycles/m, t in ms)
    double dkx, dky, dkz, dt;  // step per sample (the line's slope)
    int32_t s0;                // first sample index; sample m is s0 + m * run_stride
    int32_t len;               // samples in the run (<= kRunLen)
    int32_t step;              // index of (dk, dt) in its tile's step table
    int32_t pad;
};
// distinct (dk, dt) steps a 256-run tile may share through LDS
constexpr int kRunSteps = 8;
// Lines linear in k and t over their whole length take the per-line GEMM
// (mixed form, static nodes) from this many samples per line.
constexpr int kLineMinLen = 128;
// ... and up to this many nodes (32-bit byte offsets into the node arrays).
constexpr int64_t kLineMaxNodes = int64_t(1) << 28;

struct SignalTile {
    int32_t offset;  // first sample
    int32_t count;   // samples in the tile
};

// One axis of a Cartesian stack (its lines or its kz planes) as real rows.
// Offsets that lie symmetrically about a centre c pair up as c + D and c - D,
// and
//   exp(-2 pi i (c +- D).x) = exp(-2 pi i c.x) (cos 2 pi D.x -+ i sin 2 pi D.x):
// the pair's two sums over the nodes are P -+ i Q with P and Q the sums over
// one cosine and one sine row.  A contraction with real rows takes half the
// multiplications of one with the complex factors; the centre's phase joins
// another factor.  An offset without a partner takes both rows for itself, an
// offset at the centre the cosine row only.
//
// The centre and D are held in two doubles each, formed in extended precision from
// the given offsets; the mixed form uses the first of them.  What is left of an
// offset is the pair's departure from the common centre.  The FP64 form takes the
// rows where that departure (rms) is no larger than what complex rows round
// (pairs_f64): k' and the products are then the less exact way.
struct PairAxis {
    long double c[3] = {0.0L, 0.0L, 0.0L};
    int64_t n_rows = 0, n_ent = 0;
    std::vector<double> rows;    // (n_rows, 4): D, then the quarter turn added to D.x: 1/4 cosine, 0 sine
    std::vector<double> rows_lo; // (n_rows, 4): what D is more than that, 0
    std::vector<int32_t> ent;    // (n_ent, 4): index of c + D, of c - D or -1, cosine row, sine row or -1
    double departs2 = 0.0;       // mean square of the departures
    double4 *d_rows = nullptr, *d_rows_lo = nullptr;
    int4 *d_ent = nullptr;
};

struct CartesianTables {
    bool ok = false;
    int64_t n_ro = 0, n_ln = 0, n_kz = 0;
    // Additive split k(i,j,k) = F(i) + G(j) + H(k) per axis, cycles/m,
    // already multiplied by (double)(float)pi / pi.
    std::vector<double> F, G, H;  // (n_ro,3), (n_ln,3), (n_kz,3)
    std::vector<double> t;        // (n_ro)
    std::vector<int32_t> ro_group;  // (n_ro) t-group of each readout index
    // a standard stack: G varies along y only and H along z only (their
    // other components are exactly 0), so a line or kz phase is one product
    bool axis_aligned = false;
    double *d_F = nullptr, *d_G = nullptr, *d_H = nullptr, *d_t = nullptr;
    int32_t *d_ro_group = nullptr;
    // lines and kz planes as real rows, and F plus the lines' centre (R
    // entries), then F plus both centres
    PairAxis lines, kzs;
    std::vector<double> F_pairs, F_pairs_lo, H_lo;  // _lo: second doubles (H as it is: first double c.H)
    double *d_F_lines = nullptr, *d_F_pairs = nullptr, *d_F_lines_lo = nullptr, *d_F_pairs_lo = nullptr, *d_H_lo = nullptr;
    // the FP64 form's choice of real rows: for the lines (static nodes), for lines
    // and kz planes (moving nodes)
    bool pairs_f64 = false, pairs_f64_moving = false;
    void *d_pairs = nullptr;     // one allocation behind the pair tables
};

}  // namespace fm

struct fm_signal_plan {
    int device = 0;
    int64_t n_meas = 0, n_lines = 0, n_kz = 0, n_samples = 0;
    int method = FM_METHOD_DIRECT;
    bool prefer_grouped = true;   // static nodes: take the t-grouped tiles
    int64_t n_tgroups = 0;
    std::vector<double> tg_t;     // distinct t, first-appearance order
    std::vector<int32_t> sample_group;
    // Tilings of the samples: consecutive tiles (any t per sample) and tiles
    // of lanes with two samples of one t-group each, in the order of the groups
    // (signal_groups.hip; always used for moving nodes).
    int64_t n_tiles_consec = 0, n_tiles_pairs = 0;
    int groups_per_tile = 0;      // the most groups of one tile
    // every lane's samples have k'_b = -k'_a: to 1e-12 of the largest |k'|
    // (mixed form), to 4e-15 (FP64 form too)
    bool pairs_conj = false, pairs_exact = false;
    int planar = 0;               // every kz is 0
    // reported by fm_signal_plan_analyse
    int64_t n_tiles_grouped = 0;
    int group_pack = 1, conj_pack = 1;
    // device tables
    double4 *d_ks = nullptr;      // per sample: kx', ky', kz' (cycles/m, pi_f-scaled), t
    fm::SignalTile *d_tiles_consec = nullptr;  // offsets are sample indices
    int2 *d_pairs = nullptr;        // per lane: samples a, b (-1: none)
    uint8_t *d_lane_group = nullptr;  // per lane: group within the tile
    int4 *d_tiles_pairs = nullptr;  // first lane, lanes, first group, groups
    double *d_tg_t = nullptr;
    // readout runs (empty when some run is not linear in k and t)
    int64_t n_runs = 0, run_stride = 0;
    // every run linear to 1e-14 of the largest |k'| and |t| (not only the
    // 1e-12 of run detection): the FP64 form may then take the runs too
    bool runs_exact = false;
    fm::RunDesc *d_runs = nullptr;
    // whole lines linear in k and t (to 1e-12 of the largest |k'| / |t|
    // from the line's first sample): one RunDesc per line, len = n_meas,
    // s0 = the line's first sample; 0 when some line is not
    int64_t n_line_tabs = 0;
    fm::RunDesc *d_lines = nullptr;
    // per 256-run tile, its distinct steps (kRunSteps x (dkx, dky, dkz, dt))
    // and their count; run_steps = the largest count, 0 when some tile has
    // more than kRunSteps (each lane then forms its own step factor)
    int run_steps = 0;
    double *d_run_steps = nullptr;
    int32_t *d_run_nsteps = nullptr;
    fm::CartesianTables cart;
    // optional timing of the dominant kernel (fm_signal_plan_set_timing)
    std::vector<hipEvent_t> ev_start, ev_stop;
    mutable int ev_used = 0;
};

namespace fm {
// Record the start / stop event of the dominant kernel when timing is on.
inline void plan_timing_start(const fm_signal_plan *p, hipStream_t st)
{
    if (p->ev_used < (int)p->ev_start.size()) (void)hipEventRecord(p->ev_start[(size_t)p->ev_used], st);
}
inline void plan_timing_stop(const fm_signal_plan *p, hipStream_t st)
{
    if (p->ev_used < (int)p->ev_stop.size()) (void)hipEventRecord(p->ev_stop[(size_t)p->ev_used++], st);
}
}  // namespace fm

namespace fm {
// Cartesian path (signal_gemm.hip).
bool cartesian_analyse(fm_signal_plan *p, const double *kx, const double *ky, const double *kz,
                       const double *t);
int cartesian_upload(fm_signal_plan *p);
void cartesian_free(fm_signal_plan *p);
size_t cartesian_workspace(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc);
int cartesian_execute(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc,
                      const double *packed, void *ws, size_t ws_bytes, double *out,
                      hipStream_t stream);
// Static nodes on linear lines, per-line GEMM, mixed form
// (signal_lines_bf16.hip).
bool lines_usable(const fm_signal_plan *p, int64_t n_nodes);
size_t lines_workspace(const fm_signal_plan *p, int64_t n_nodes);
int64_t lines_splits(const fm_signal_plan *p, int64_t n_nodes);
int lines_execute(const fm_signal_plan *p, int64_t n_nodes, int n_enc, const double *packed, void *ws,
                  size_t ws_bytes, double *out, hipStream_t stream);
// Samples grouped by t (signal_groups.hip).
int groups_blocks_per_cu(const fm_signal_plan *p, bool mixed, bool motion, int n_enc, int n_modes);
int groups_launch(const fm_signal_plan *p, bool mixed, bool motion, int64_t n_nodes, int n_enc, int v0, int vb,
                  const double *packed, const float *modes, int n_modes, const double *motion_coef, int64_t n_splits,
                  int64_t nodes_per_split, double2 *dst, int write_final, hipStream_t stream);
bool groups_in_pairs(const fm_signal_plan *p, bool mixed);
// Route and splits of the Cartesian GEMM (fm_signal_route), static or moving.
int cartesian_route(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc, bool moving, int64_t *n_splits);
// Moving nodes, per-readout GEMM in either form (n_enc <= kMovMaxV).
size_t cartesian_moving_workspace(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc);
int cartesian_moving_execute(const fm_signal_plan *p, int precision, int64_t n_nodes, int n_enc,
                             const double *packed, const float *modes, int n_modes, const double *motion_coef,
                             void *ws, size_t ws_bytes, double *out, hipStream_t stream);
}  // namespace fm
