// Fused direct log-likelihood of a ragged template batch on gfx950 (no
// counterpart entry point in the reference; it computes what
// Likelihood.get_ll does, likelihood.py:140-225, for templates whose sparse
// frequency grids have different lengths, in one launch sequence with no host
// synchronisation, so a caller can capture it in a hipGraph).
//
// Per binary b with sparse length L_b (layout: points of all binaries
// concatenated, offset off_b; within a binary [i][mode] for the grid and
// [i][mode] segment records: the knots x_i, x_{i+1} that bound segment i, then
// per quantity [y, c1, c2, c3], so that one segment of one quantity is 32
// contiguous bytes and one record read both checks and evaluates the segment):
//   k_dir_setup   one lane per (binary, mode): coefficient records
//   k_dir_grid    one workgroup per (binary, mode): default grid
//                 Mf in [mf_min, mf_max] * m / 2, t(f) there, the crossings of
//                 t = 0 and t = Tobs, the grid refitted to that window
//                 (phenomhm.py:208-224, :509-614), then amplitude, phase, t(f)
//                 and the TDI response on the refitted grid (phenomhm.py:487-507,
//                 Response.cu), written compact: nine values per (knot, mode)
//   k_dir_spline  one workgroup per block of a (binary, mode)'s knots, or for several
//                 short grids, one lane per knot: not-a-knot spline coefficients (Interpolate.cu:15-359)
//                 of the nine quantities by parallel cyclic reduction, from the
//                 compact values; each record written once
//   k_dir_band    dense band [st, et) of each binary (waveformbuild.py:139-156)
//                 and the exclusive prefix of its chunks of dense bins (chunks
//                 aligned to absolute multiples of the chunk size)
//   k_dir_cnt_zero, k_dir_cnt, k_dir_cnt_scan, k_dir_perm
//                 chunk-major execution order of the work items (counting sort)
//   k_dir_like    persistent: wavefronts take the (binary, chunk) work
//                 items in that order; each lane evaluates dense bins (spline segment per
//                 mode, WaveformBuild.cu:80-143, window and mode sum :48-60)
//                 and accumulates the noise-weighted inner products
//                 (Likelihood.cu:357-471); one partial sum per work item
//   k_dir_reduce  one wavefront per binary: its partials in a fixed order (deterministic)

#include <algorithm>
#include <memory>
#include <new>
#include <vector>

#include "bbhx_hip.h"
#include "common.h"
#include "fused_device.h"
#include "grad_device.h"
#include "spline_device.h"

using namespace bbhx;
using namespace bbhx::fused;

namespace bbhx {
bool response_orbit_tab(const bbhx_response* r, resp::OrbitTab& o);
}

// A part of a plan's work table: the entries of one launch
struct TablePart {
    int threads = 0;  // lanes per workgroup
    int lmax = 0;     // longest grid
    long first = 0, count = 0;
};

struct bbhx_direct_plan {
    int device = -1;
    int B = 0, M = 0, N = 0, Lmax = 0;
    int min_chunk = 0;   // smallest chunk a caller may ask for
    int min_item = 0;    // dense bins of the smallest work item the buffers are sized for
    long S = 0;          // total sparse points
    long max_items = 0;  // bound on (binary, chunk) work items
    // device buffers
    long* off = nullptr;   // (B,) first point of each binary
    int* len = nullptr;    // (B,)
    std::vector<int> lengths;  // the same on the host
    // Work tables of the launches whose workgroups go by grid length: laid out for the
    // longest grid, most of them start for nothing in an uneven batch. 4096 templates of 64
    // knots and one of 4096, as many workgroups for each of them and the tables: k_dirg_knots
    // 10.4 and 0.42 ms, k_dir_grid 0.65 and 0.29, k_dirg_spline_adj 0.55 and 0.41.
    int* grid_b = nullptr;     // (B,) binaries by size of their k_dir_grid workgroup
    int4* spl = nullptr;       // workgroups of the spline kernels (SplineRows): blocks, then packs
    int4* knots = nullptr;     // {b M + m, first knot, row of gpart} of each of k_dirg_knots'
    int* gpart_b = nullptr;    // (B + 1,) first row of gpart of each binary
    TablePart grid_parts[3], knot_parts[4];
    long nspl = 0, nblocks = 0, nknots = 0;
    FusedRec* recs = nullptr;
    double* X = nullptr;   // (S, M)
    double* Cf = nullptr;  // (S, M, RS): segment records (bounds, value and cubic coefficients)
    double* Yc = nullptr;  // (S, M, NQ): the grid pass's nine values per knot, compact
    double* grid_lo = nullptr;    // (B, M) log2 of the first refitted grid point
    double* grid_istep = nullptr; // (B, M) 1 / log2 step (0 for a degenerate grid)
    int* band = nullptr;          // (B, 3): st, et, chunk_begin
    int* total = nullptr;         // (1,) number of work items
    double* partial = nullptr;    // (max_items, 4)
    int* perm = nullptr;          // (max_items,) execution order of the work items
    int* cnt = nullptr;           // (max_chunks + 1,) items per absolute chunk, then offsets
    int* next = nullptr;          // (1,) next entry of perm for the dense-band kernel
    // gradient buffers (bbhx_hip_direct_plan_enable_grad)
    double* Yadj = nullptr;              // (S, M, 9, 4) adjoint records
    bbhx::gradk::GradRec* grecs = nullptr;  // (B, M) records with tangents
    double* gpart = nullptr;             // (rows, 11) gradients of the workgroups of k_dirg_knots
    int max_chunks = 0;           // absolute chunks of min_item bins
};

namespace {

constexpr int NQ = 9;


// one spline segment of one quantity: value at the knot and c1, c2, c3
struct alignas(32) Cubic {
    double y, c1, c2, c3;
};

// Whether t(f) stays inside the observation window over a whole segment: then
// (or if it stays outside) the dense pass need not evaluate t(f) bin by bin.
enum SegWin : int { WIN_MIXED = 0, WIN_ALL = 1, WIN_NONE = 2 };

// segment i of one (binary, mode): it covers x_lo <= f < x_hi (x_hi = x_lo for
// the last knot, which starts no segment). The cubics in the order A, phase,
// T1..T3 re/im, t_f (seg_slot): the 288 B in front of t_f's are what a segment
// inside the window needs.
struct alignas(32) SegRec {
    double x_lo, x_hi;
    int win, pad0;  // SegWin
    double pad1;
    Cubic q[NQ];
};
constexpr int RS = sizeof(SegRec) / sizeof(double);  // 40 doubles
constexpr int RQ = 4;                                 // offset of q[0] in doubles
static_assert(sizeof(SegRec) == 320, "segment record layout");
constexpr int S_A = 0, S_PH = 1, S_T = 2, S_TF = 8;  // slots of q
// slot of quantity q of the grid pass (A, phase, t_f, T1..T3 re/im)
__host__ __device__ constexpr int seg_slot(int q) { return q < 2 ? q : (q == 2 ? S_TF : q - 1); }

__global__ __launch_bounds__(64) void k_dir_setup(FusedRec* __restrict__ recs, const double* __restrict__ params, int B, ModeList modes,
                            int M, const double* __restrict__ qnm, int table_len, double dspin)
{
    setup_split(recs, params, B, modes, M, qnm, table_len, dspin);
}

// numpy.logspace point i of num between 10^lo and 10^hi (start + i step, the
// last point exactly 10^hi)
__device__ inline double logspace_pt(double lo, double step, double hi, int i, int num)
{
    return pow(10.0, i == num - 1 ? hi : lo + i * step);
}

__device__ inline int wsum_i(int v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

__device__ inline int wmax_i(int v)
{
    for (int o = 32; o > 0; o >>= 1) v = max(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline double wmin_d(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}

__device__ inline double wmax_d(double v)
{
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// One workgroup per (binary, mode), one lane per knot of each pass. LDS: t(f) of the
// default grid (L_b doubles).
//
// Bound by the FP64 work of a knot, some 4000 instructions over both grids, at the
// two wavefronts per SIMD that its 251 VGPRs leave (three and four spill: 1.41 and
// 1.92 ms). 16 templates of 1024 knots: 33 us, 1024 uneven ones: 0.95 ms. One
// wavefront per (binary, mode): 78 us, a chain of 16 knots per lane and pass, and
// 1.18 ms, as the LDS for the longest grid then allows five wavefronts per CU. 512
// lanes: 30 us and 1.18 ms.
constexpr int GRID_T = 256;
__global__ __launch_bounds__(GRID_T) void k_dir_grid(double* __restrict__ X, double* __restrict__ Yc,
                                                 double* __restrict__ grid_lo, double* __restrict__ grid_istep,
                                                 int* __restrict__ flags, const FusedRec* __restrict__ recs,
                                                 const int* __restrict__ bins, const long* __restrict__ off,
                                                 const int* __restrict__ len, const double* __restrict__ params,
                                                 const double* __restrict__ t_start,
                                                 const double* __restrict__ t_end, int B, int M, ModeList modes,
                                                 resp::OrbitTab orb, int TDItag, int rescaled, int tdi2,
                                                 double initial_t_val, double mf_min, double mf_max)
{
    extern __shared__ double tfs[];
    __shared__ double2 s_t[GRID_T / 64];
    __shared__ int4 s_n[GRID_T / 64];
    const int b = bins[blockIdx.x / M], m = blockIdx.x % M, bm = b * M + m;
    const int t = threadIdx.x, T = blockDim.x;
    const int L = len[b];
    const long base = off[b];
    const FusedRec& r = recs[bm];
    const double t_ref = params[P_TREF * B + b];
    const double Tobs = t_end[b] - t_start[b];
    const double Msec = (params[P_M1 * B + b] + params[P_M2 * B + b]) * MTSUN_SI;
    const double mm = modes.mm[m];

    // default grid (phenomhm.py:208-224) and t(f) on it; the frequencies go to X for now
    const double lo = log10(mf_min), hi = log10(mf_max), step = (hi - lo) / (L - 1);
    for (int i = t; i < L; i += T) {
        const double f = logspace_pt(lo, step, hi, i, L) / Msec * mm / 2;
        double amp, phase, tf;
        phm::phm_eval(r.w, f, amp, phase, tf);
        tfs[i] = tf + t_ref;
        X[(base + i) * M + m] = f;
    }
    __syncthreads();

    // window search (phenomhm.py:520-614): the single segment where t crosses 0 / Tobs
    double tmin = 1e300, tmax = -1e300;
    int n0 = 0, nT = 0, s0 = -1, sT = -1;
    for (int i = t; i < L; i += T) {
        const double t0 = tfs[i];
        tmin = fmin(tmin, t0);
        tmax = fmax(tmax, t0);
        if (i + 1 < L) {
            const double t1 = tfs[i + 1];
            if ((0.0 < t1) && (0.0 > t0)) {
                n0++;
                s0 = i;
            }
            if ((Tobs < t1) && (Tobs > t0)) {
                nT++;
                sT = i;
            }
        }
    }
    tmin = wmin_d(tmin);
    tmax = wmax_d(tmax);
    n0 = wsum_i(n0);
    nT = wsum_i(nT);
    s0 = wmax_i(s0);
    sT = wmax_i(sT);
    if ((t & 63) == 0) {
        s_t[t >> 6] = {tmin, tmax};
        s_n[t >> 6] = {n0, nT, s0, sT};
    }
    __syncthreads();
    for (int w = 0; w < T / 64; w++) {
        if (w == t >> 6) continue;
        tmin = fmin(tmin, s_t[w].x);
        tmax = fmax(tmax, s_t[w].y);
        n0 += s_n[w].x;
        nT += s_n[w].y;
        s0 = max(s0, s_n[w].z);
        sT = max(sT, s_n[w].w);
    }
    const double* xf = X + base * M + m;
    double f_min = xf[0], f_max = xf[(long)(L - 1) * M];
    int flag = 0;
    if (tmin < 0.0) {
        if (n0 != 1) flag |= 1;
        else {
            const double y1 = xf[(long)s0 * M], y2 = xf[(long)(s0 + 1) * M];
            const double x1 = tfs[s0], x2 = tfs[s0 + 1];
            f_min = (y2 - y1) / (x2 - x1) * (0.0 - x1) + y1;
        }
    }
    if (tmax > Tobs) {
        if (nT != 1) flag |= 2;
        else {
            const double y1 = xf[(long)sT * M], y2 = xf[(long)(sT + 1) * M];
            const double x1 = tfs[sT], x2 = tfs[sT + 1];
            f_max = (y2 - y1) / (x2 - x1) * (Tobs - x1) + y1;
        }
    }
    if (t == 0 && flag) atomicOr(&flags[b], flag);
    __syncthreads();  // every lane has read the default grid before it is overwritten

    // refitted grid and the nine quantities on it
    const double lo2 = log10(f_min), hi2 = log10(f_max), step2 = (hi2 - lo2) / (L - 1);
    if (t == 0) {
        // log2 units: the dense kernel estimates the segment from an FP32 log2
        grid_lo[bm] = lo2 * LOG2_10;
        grid_istep[bm] = step2 > 0.0 ? 1.0 / (step2 * LOG2_10) : 0.0;
    }
    const double dt_shift = t_ref - initial_t_val;
    for (int i = t; i < L; i += T) {
        const double f = logspace_pt(lo2, step2, hi2, i, L);
        double amp, phase, tf;
        phm::phm_eval(r.w, f, amp, phase, tf);
        phase = phase + ((f * dt_shift) * 2) * PI;
        tf = tf + t_ref;
        cd T[3];
        double dphi;
        resp::resp_eval(r.s, orb, f, tf, TDItag, rescaled, tdi2, T, dphi);
        phase = phase + dphi;
        const long p = (base + i) * M + m;
        X[p] = f;
        double* y = Yc + p * NQ;
        y[0] = amp;
        y[1] = phase;
        y[2] = tf;
        y[3] = T[0].re;
        y[4] = T[0].im;
        y[5] = T[1].re;
        y[6] = T[1].im;
        y[7] = T[2].re;
        y[8] = T[2].im;
    }
}

// SegWin of the cubic c over [0, h]: a cubic lies between the least and the
// greatest of its four Bernstein coefficients there; the margin (1e-12 of the
// terms' magnitudes, and 1 microsecond) covers the rounding of those and of the
// bin-by-bin evaluation, so WIN_ALL and WIN_NONE are what every bin would find.
__device__ inline int segment_window(const Cubic& c, double h, double ts, double te)
{
    const double t1 = c.c1 * h, t2 = c.c2 * (h * h), t3 = c.c3 * (h * h * h);
    const double b1 = c.y + t1 * (1.0 / 3.0), b2 = c.y + (2.0 * t1 + t2) * (1.0 / 3.0), b3 = c.y + t1 + t2 + t3;
    const double m = 1e-6 + 1e-12 * (fabs(c.y) + fabs(t1) + fabs(t2) + fabs(t3));
    const double lo = fmin(fmin(c.y, b1), fmin(b2, b3)) - m, hi = fmax(fmax(c.y, b1), fmax(b2, b3)) + m;
    if (!(m < 1e300)) return WIN_MIXED;  // not finite: bin by bin
    if (lo >= ts && (hi <= te || te <= 0.0)) return WIN_ALL;
    if (hi < ts || (te > 0.0 && lo > te)) return WIN_NONE;
    return WIN_MIXED;
}

// ---------------------------------------------------------------- splines (see spline_device.h)
//
// Bound by the solves' exchange through LDS for few templates (16 of 1024 knots: 25
// us), by the records' writes (320 B per (knot, mode)) for many (1024 uneven ones,
// 9.4 M records: 1.7 ms; 64 of 4096 knots: 0.2 ms). Thomas sweeps, one lane per (mode,
// quantity), are one chain over all knots: 537 us, 3.1 ms and 2.24 ms.

// This lane's row in a spline kernel, by the workgroup's entry of the plan's table.
// A block {b M + m, 1, T, block}: T rows of one (binary, mode). A pack {b M + m, sets, lanes
// per set, 0}: whole grids of at most T / 2 knots, of (binary, mode) pairs from b M + m on,
// side by side; with a workgroup for each of them, 16384 templates of 16 knots take 1.71
// ms instead of 0.15 (a lane per (mode, quantity), by Thomas sweeps: 0.26).
struct SplineRow {
    int b, m, n, i, s;  // knot i of the n of (binary b, mode m); set s of the workgroup
    int t0, t1;         // lanes of the set
    int row0, row1;     // rows of the grid that this workgroup finishes
    bool any, out;      // i is a row of the grid; one of those
};
template <bool PACK>
__device__ inline SplineRow spline_row(const int4* __restrict__ spl, const int* __restrict__ len, int M)
{
    constexpr int T = SPL_T;
    const int4 e = spl[blockIdx.x];
    const int t = threadIdx.x;
    SplineRow w;
    w.s = PACK ? t / e.z : 0;
    const bool set = !PACK || w.s < e.y;
    const int bm = PACK && set ? e.x + w.s : e.x;
    w.b = bm / M;
    w.m = bm % M;
    w.n = len[w.b];
    w.t0 = w.s * e.z;
    w.t1 = PACK ? min(w.t0 + e.z, T) : T;
    const int first = PACK ? 0 : e.w * SPL_U;
    w.i = set ? first + t - w.t0 : w.n;
    w.row0 = PACK || e.w == 0 ? 0 : first + SPL_W;
    w.row1 = PACK || e.w == spline_blocks(w.n) - 1 ? w.n : first + T - SPL_W;
    w.any = w.i < w.n;
    w.out = w.i >= w.row0 && w.i < w.row1;
    return w;
}
constexpr int SPL_SETS = SPL_T / 4;  // sets of a pack

// Not-a-knot splines of the nine quantities of one (binary, mode) (the system of
// spline.hip), one lane per knot. The two end rows are folded into their
// neighbours, which leaves every row dominant: s_0 = (b_0 - (h_0 + h_1) s_1) / h_1.
template <bool PACK>
__global__ __launch_bounds__(SPL_T) __attribute__((amdgpu_waves_per_eu(4))) void k_dir_spline(const double* __restrict__ X, const double* __restrict__ Yc,
                                                    SegRec* __restrict__ Cf, const int4* __restrict__ spl,
                                                    const long* __restrict__ off, const int* __restrict__ len,
                                                    const double* __restrict__ t_start,
                                                    const double* __restrict__ t_end, int M)
{
    constexpr int T = SPL_T;
    __shared__ __align__(16) double sh[(NQ + 2) * T];
    __shared__ double ends[2][NQ][PACK ? SPL_SETS : 1];  // right sides of the sets' two end rows
    const int t = threadIdx.x;
    const SplineRow w = spline_row<PACK>(spl, len, M);
    const int i = w.i, n = w.n, s = w.s;
    const long base = off[w.b];
    const long p = (base + (w.any ? i : n - 1)) * M + w.m;
    const double x = X[p];
    double y[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) y[q] = Yc[p * NQ + q];
    sh[t] = x;
#pragma unroll
    for (int q = 0; q < NQ; q++) sh[(1 + q) * T + t] = y[q];
    __syncthreads();
    const int tl = t > 0 ? t - 1 : 0, th = t + 1 < T ? t + 1 : t;
    const double hl = x - sh[tl], xr = sh[th], hr = xr - x;
    const double il = rcp_pos(hl), ir = rcp_pos(hr);
    // rows to solve: the interior ones with both neighbours in the block
    const bool solve = i > 0 && i < n - 1 && t > 0 && t + 1 < T;
    const bool low = solve && i == 1, high = solve && i == n - 2;
    const double d = hl + hr;
    double a = low ? 0.0 : hr, c = high ? 0.0 : hl;
    double diag = 2.0 * d;
    if (low) diag -= d;
    if (high) diag -= d;
    const double id = rcp_pos(d), ib = rcp_pos(diag);
    a = solve ? a * ib : 0.0;
    c = solve ? c * ib : 0.0;
    double mr[NQ], r[NQ];
    // right sides of the end rows, as multiples of the slopes on either side
    const double e0l = (hl + 2.0 * d) * hr * id, e0r = hl * hl * id;
    const double e1l = hr * hr * id, e1r = (2.0 * d + hr) * hl * id;
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const double ml = (y[q] - sh[(1 + q) * T + tl]) * il;
        mr[q] = (sh[(1 + q) * T + th] - y[q]) * ir;
        double v = 3.0 * (hr * ml + hl * mr[q]);
        if (low) {
            ends[0][q][s] = e0l * ml + e0r * mr[q];
            v -= ends[0][q][s];
        }
        if (high) {
            ends[1][q][s] = e1l * ml + e1r * mr[q];
            v -= ends[1][q][s];
        }
        r[q] = solve ? v * ib : 0.0;
    }
    __syncthreads();
    pcr_solve(a, c, r, sh, t, w.t0, w.t1);
    // slopes to the neighbours, the end ones from their rows
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        if (i != 0 && i < n - 1) sh[q * T + t] = r[q];
        if (low) sh[q * T + t - 1] = (ends[0][q][s] - d * r[q]) * ir;
        if (high) sh[q * T + t + 1] = (ends[1][q][s] - d * r[q]) * il;
    }
    __syncthreads();
    const bool end = i == n - 1;
    int win = WIN_MIXED;
    Cubic k[NQ];
#pragma unroll
    for (int q = 0; q < NQ; q++) {
        const double sl = sh[q * T + t], sn = sh[q * T + th];
        const double u = (sl + sn - 2.0 * mr[q]) * ir;
        k[q] = end ? Cubic{y[q], 0.0, 0.0, 0.0} : Cubic{y[q], sl, (mr[q] - sl) * ir - u, u * ir};
        if (q == 2 && !end) win = segment_window(k[q], hr, t_start[w.b], t_end[w.b]);
    }
    __syncthreads();
    // The records leave through LDS, 16 of a wavefront's at a time, so that a
    // store covers whole records (written by their own lanes, 16 B to a line each,
    // the kernel waits on the number of requests: 2.1 against 1.7 ms at 1024)
    constexpr int PER = 16, PITCH = RS + 2;  // doubles, padded against bank conflicts
    static_assert(4 * PER * PITCH <= (NQ + 2) * T, "the records of a workgroup's wavefronts fit in sh");
    const int lane = t & 63;
    __shared__ long rec[PACK ? T : 1];  // the rows' records, -1: none
    if (PACK) rec[t] = w.out ? p : -1;
    double* own = sh + (t >> 6) * PER * PITCH;
    for (int g = 0; g < 64; g += PER) {
        if (lane >= g && lane < g + PER) {
            double* o = own + (lane - g) * PITCH;
            o[0] = x;
            o[1] = end ? x : xr;
            o[2] = __hiloint2double(0, win);
            o[3] = 0.0;
#pragma unroll
            for (int q = 0; q < NQ; q++) {
                double* v = o + RQ + 4 * seg_slot(q);
                v[0] = k[q].y;
                v[1] = k[q].c1;
                v[2] = k[q].c2;
                v[3] = k[q].c3;
            }
        }
        __syncthreads();
        for (int e = lane; e < PER * RS / 2; e += 64) {
            const int j = e / (RS / 2), c = e - j * (RS / 2);
            const int ij = i - lane + g + j;
            const long pj = PACK ? rec[(t & ~63) + g + j] : (ij >= w.row0 && ij < w.row1 ? (base + ij) * M + w.m : -1);
            if (pj >= 0)
                reinterpret_cast<double2*>(Cf + pj)[c] = *reinterpret_cast<const double2*>(own + j * PITCH + 2 * c);
        }
        __syncthreads();
    }
}

// number of entries of the sorted array a[0..n) that are <= v (searchsorted side='right')
__device__ inline int search_right(const double* __restrict__ a, int n, double v)
{
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (a[mid] <= v) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// Dense band of each binary and the exclusive prefix of its chunks; one
// workgroup of 1024 threads, each owning a contiguous run of binaries. Chunks
// are aligned to absolute multiples of 'chunk' dense bins, so that the work
// items of different binaries over the same dense bins read the same data.
__global__ __launch_bounds__(1024) void k_dir_band(int* __restrict__ band, int* __restrict__ total,
                                                   const double* __restrict__ X, const long* __restrict__ off,
                                                   const int* __restrict__ len, const double* __restrict__ freqs,
                                                   int N, int B, int M, int chunk)
{
    __shared__ int part[1024];
    const int t = threadIdx.x;
    const int per = (B + 1023) / 1024;
    const int b0 = t * per, b1 = min(B, b0 + per);
    int sum = 0;
    for (int b = b0; b < b1; b++) {
        const long base = off[b];
        const int L = len[b];
        double lo = 1e300, hi = -1e300;
        for (int m = 0; m < M; m++) {
            lo = fmin(lo, X[base * M + m]);
            hi = fmax(hi, X[(base + L - 1) * M + m]);
        }
        const int st = search_right(freqs, N, lo), et = search_right(freqs, N, hi);
        const int nch = et > st ? (et - 1) / chunk - st / chunk + 1 : 0;
        band[3 * b] = st;
        band[3 * b + 1] = et;
        band[3 * b + 2] = nch;  // count for now
        sum += nch;
    }
    part[t] = sum;
    __syncthreads();
    // inclusive scan of the 1024 partial counts (Hillis-Steele)
    for (int o = 1; o < 1024; o <<= 1) {
        const int v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = t > 0 ? part[t - 1] : 0;
    for (int b = b0; b < b1; b++) {
        const int nch = band[3 * b + 2];
        band[3 * b + 2] = run;
        run += nch;
    }
    if (t == 1023) total[0] = part[1023];
}

// Execution order of the work items, chunk-major: perm lists the items of
// absolute chunk 0, then of chunk 1, ... (a counting sort; the order inside a
// chunk is whatever the atomics give, which does not affect any result: each
// item writes its own partial, reduced per binary in item order). Concurrent
// workgroups then work on the same dense bins for different binaries, so the
// data and noise weights of a chunk come from L2 instead of being fetched again
// for every binary. cnt has nchunks + 1 entries.
__global__ void k_dir_cnt_zero(int* __restrict__ cnt, int n, int* __restrict__ next)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) cnt[i] = 0;
    if (i == 0) next[0] = 0;
}

// binary owning work item 'it' (largest b with chunk_begin <= it)
__device__ inline int owner(const int* __restrict__ band, int B, int it)
{
    int lo = 0, hi = B - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (band[3 * mid + 2] <= it) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// absolute chunk of work item it
__device__ inline int item_chunk(const int* __restrict__ band, int B, int it, int chunk, int& b)
{
    b = owner(band, B, it);
    return band[3 * b] / chunk + (it - band[3 * b + 2]);
}

// one lane per work item
__global__ void k_dir_cnt(int* __restrict__ cnt, const int* __restrict__ band, const int* __restrict__ total, int B,
                          int chunk)
{
    const int it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= total[0]) return;
    int b;
    atomicAdd(&cnt[item_chunk(band, B, it, chunk, b)], 1);
}

// exclusive scan of cnt[0, n) in place; one workgroup of 1024 threads
__global__ __launch_bounds__(1024) void k_dir_cnt_scan(int* __restrict__ cnt, int n)
{
    __shared__ int part[1024];
    const int t = threadIdx.x;
    const int per = (n + 1023) / 1024;
    const int g0 = t * per, g1 = min(n, g0 + per);
    int sum = 0;
    for (int g = g0; g < g1; g++) sum += cnt[g];
    part[t] = sum;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        const int v = t >= o ? part[t - o] : 0;
        __syncthreads();
        part[t] += v;
        __syncthreads();
    }
    int run = t > 0 ? part[t - 1] : 0;
    for (int g = g0; g < g1; g++) {
        const int c = cnt[g];
        cnt[g] = run;
        run += c;
    }
}

__global__ void k_dir_perm(int* __restrict__ perm, int* __restrict__ cnt, const int* __restrict__ band,
                           const int* __restrict__ total, int B, int chunk)
{
    const int it = blockIdx.x * blockDim.x + threadIdx.x;
    if (it >= total[0]) return;
    int b;
    perm[atomicAdd(&cnt[item_chunk(band, B, it, chunk, b)], 1)] = it;
}

// h[ch] += conj(T_ch A e^{i phase}) of one mode at x = f - x_i into its segment
// (WaveformBuild.cu:48-60, :80-143)
__device__ inline void add_mode(cd h[3], const Cubic* q, double x, const double2* tab)
{
    auto ev = [&](int k) { return fma(fma(fma(q[k].c3, x, q[k].c2), x, q[k].c1), x, q[k].y); };
    const cd ap = ev(S_A) * cexpi_tab1k(ev(S_PH), tab);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const double tr = ev(S_T + 2 * c), ti = ev(S_T + 2 * c + 1);
        h[c].re = fma(tr, ap.re, fma(-ti, ap.im, h[c].re));
        h[c].im = fma(-tr, ap.im, fma(-ti, ap.re, h[c].im));
    }
}

// t_start <= t_f <= t_end (t_end <= 0: no upper limit) at x into a segment whose
// 'win' does not say so already (WaveformBuild.cu:50)
__device__ inline bool bin_in_window(const Cubic& c, double x, double ts, double te)
{
    const double tf = fma(fma(fma(c.c3, x, c.c2), x, c.c1), x, c.y);
    return (tf >= ts) && ((tf <= te) || (te <= 0.0));
}

// add_mode where the window may cut the segment: q is the record at rc with all
// but t_f's cubic loaded
__device__ inline void add_mode_window(cd h[3], const SegRec& q, const SegRec* rc, double x, double ts, double te,
                                       const double2* tab)
{
    if (q.win != WIN_ALL && (q.win == WIN_NONE || !bin_in_window(rc->q[S_TF], x, ts, te))) return;
    add_mode(h, q.q, x, tab);
}

// Segment of one lane's dense frequency f in the grid of one mode, searched by
// that lane, and its contribution (lanes of a wavefront in many different
// segments): from the FP32 log2 estimate the index moves until x_lo <= f < x_hi
// or leaves [0, L - 2] (no contribution, WaveformBuild.cu:92-93).
__device__ inline void mode_per_lane(cd h[3], const SegRec* __restrict__ rm, int M, int L,
                                     double f, int i, double ts, double te, const double2* tab)
{
    double2 bnd = *reinterpret_cast<const double2*>(rm + (long)i * M);
    while (f < bnd.x && i > 0) bnd = *reinterpret_cast<const double2*>(rm + (long)--i * M);
    while (f >= bnd.y && i < L - 2) bnd = *reinterpret_cast<const double2*>(rm + (long)++i * M);
    if (!(bnd.x <= f && f < bnd.y)) return;
    const SegRec* rc = rm + (long)i * M;
    add_mode_window(h, *rc, rc, f - bnd.x, ts, te, tab);
}

// ---------------------------------------------------------------- adjoint helpers

// Adjoint record of one (knot, mode): for each of the nine quantities, the
// adjoints of its segment's (y, c1, c2, c3).
constexpr int NA = NQ * 4;  // 36 doubles

// quantity of adjoint j (0..7): A, phase, then the six transfer-function parts
// (t_f carries none: the observation window is held fixed)
__device__ inline int adj_q(int j) { return j < 2 ? j : j + 1; }

// Adjoints of the eight interpolated quantities of one mode at one dense bin (A,
// phase, T1..T3 re/im), given Lam_c = 4 w_c (d~_c - h~_c) (d logL =
// Re sum_c conj(Lam_c) dh_c with h_c = sum_m conj(T_c A e^{i phase});
// Likelihood.cu:357-375 differentiated). The adjoint of coefficient p of a
// quantity's cubic is its adjoint times x^p.
__device__ inline void mode_adjoint(double (&a)[8], const Cubic* q, double x, const cd Lam[3], const double2* tab)
{
    auto ev = [&](int k) { return fma(fma(fma(q[k].c3, x, q[k].c2), x, q[k].c1), x, q[k].y); };
    const double A = ev(S_A);
    const cd E = cexpi_tab1k(ev(S_PH), tab);
    const cd AE = A * E;
    cd P = mk(0.0, 0.0);
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const cd T = mk(ev(S_T + 2 * c), ev(S_T + 2 * c + 1));
        P.re = fma(Lam[c].re, T.re, fma(-Lam[c].im, T.im, P.re));
        P.im = fma(Lam[c].re, T.im, fma(Lam[c].im, T.re, P.im));
        const cd LAE = Lam[c] * AE;
        a[2 + 2 * c] = LAE.re;
        a[3 + 2 * c] = -LAE.im;
    }
    const cd PE = P * E;
    a[0] = PE.re;
    a[1] = -A * PE.im;
}

// v of the lane whose index differs in the bits of a quad permutation
template <int CTRL>
__device__ inline double quad_swap(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}

// 4 x 4 transpose within each quad of lanes: v[s] of lane i <- v[i] of lane s
__device__ inline void quad_transpose(double (&v)[4], int lane)
{
    const bool odd = (lane & 1) != 0, up = (lane & 2) != 0;
#pragma unroll
    for (int k = 0; k < 4; k += 2) {
        const double t0 = quad_swap<0xB1>(v[k]), t1 = quad_swap<0xB1>(v[k + 1]);  // lanes 1 0 3 2
        v[k] = odd ? t1 : v[k];
        v[k + 1] = odd ? v[k + 1] : t0;
    }
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const double t0 = quad_swap<0x4E>(v[k]), t2 = quad_swap<0x4E>(v[k + 2]);  // lanes 2 3 0 1
        v[k] = up ? t2 : v[k];
        v[k + 2] = up ? v[k + 2] : t0;
    }
}

// Sums over the bins of a wavefront of (quantity adjoint) x (power of x): an
// (8 x bins) (bins x 4) product on the matrix cores, four blocks of 4 x 4 x 4
// (v_mfma_f64_4x4x4: lane i + 4 b + 16 k gives A[i][k] and B[k][i] of block b and
// holds D[k][i]). The quad of lanes 4 Q + s gives, in step s, the four quantities
// and the four powers of one bin, that of lane 4 Q + s: a transpose within quads,
// no exchange through LDS. acc[g] of lane j + 4 b + 16 i: quantity i + 4 g, power
// j, the bins of block b.
__device__ inline void adjoint_accumulate(double (&acc)[2], const double (&a)[8], double x, int lane)
{
    double v0[4] = {a[0], a[1], a[2], a[3]}, v1[4] = {a[4], a[5], a[6], a[7]};
    double w[4] = {1.0, x, x * x, x * (x * x)};
    quad_transpose(v0, lane);
    quad_transpose(v1, lane);
    quad_transpose(w, lane);
#pragma unroll
    for (int k = 0; k < 4; k++) {
        acc[0] = __builtin_amdgcn_mfma_f64_4x4x4f64(v0[k], w[k], acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f64_4x4x4f64(v1[k], w[k], acc[1], 0, 0, 0);
    }
}

// adjoint of one lane's bin for one mode, segment searched by the lane (as
// mode_per_lane), added to the segment's adjoint record
__device__ inline void mode_adjoint_per_lane(double* __restrict__ Ym, const SegRec* __restrict__ rm, int M, int L,
                                             double f, int i, double ts, double te, const cd Lam[3],
                                             const double2* tab)
{
    double2 bnd = *reinterpret_cast<const double2*>(rm + (long)i * M);
    while (f < bnd.x && i > 0) bnd = *reinterpret_cast<const double2*>(rm + (long)--i * M);
    while (f >= bnd.y && i < L - 2) bnd = *reinterpret_cast<const double2*>(rm + (long)++i * M);
    if (!(bnd.x <= f && f < bnd.y)) return;
    const SegRec* rc = rm + (long)i * M;
    const double x = f - bnd.x;
    if (rc->win != WIN_ALL && (rc->win == WIN_NONE || !bin_in_window(rc->q[S_TF], x, ts, te))) return;
    double a[8];
    mode_adjoint(a, rc->q, x, Lam, tab);
    double* y = Ym + (long)i * M * NA;
#pragma unroll
    for (int k = 0; k < 8; k++) {
        double v = a[k];
#pragma unroll
        for (int c = 0; c < 4; c++, v *= x) unsafeAtomicAdd(y + adj_q(k) * 4 + c, v);
    }
}

// Persistent dense-band kernel, each wavefront taking work items of its own (the
// wavefronts of a workgroup share the table of e^{i theta} and no barrier):
// partial[it] = (Re, Im of sum conj(d~) h~, sum |h~|^2, 0)
// over the dense bins of work item it, where h~ = w h (Likelihood.cu:357-375).
//
// A work item's bins go in blocks of RB x 64 consecutive bins (lane l: bins
// kb + 64 r + l), the modes of a block summed mode by mode. The segment of bin f in a mode's grid is
// searchsorted(x, f, 'right') - 1 (waveformbuild.py:139-156), found with the
// exact FP64 comparisons x_lo <= f < x_hi against the stored knots.
//
// Dense bins are much finer than the sparse grid over most of a band, so a block
// usually lies in the segment that the mode's previous block ended in (kept in
// lane m of 'curv'): a wavefront-uniform walker reads its record in one round of
// scalar loads, evaluates every bin in [x_lo, x_hi) (t_f only where 'win' leaves
// the window open) and moves to the next segment until all bins are placed. After
// WALK_STEPS segments (low frequencies, where a block spans many) each lane left
// over searches its own (mode_per_lane).
//
// Bound by FP64 issue: 55 vector instructions per (bin, mode) evaluation (24 of
// the eight cubics, 14 of e^{i phase}, 12 of the mode sum), 83 with the walker and
// the inner products, the SIMDs issuing 84 % of the cycles (counters). 1024 uneven templates,
// 1.58 M bins: 44.3 -> 20 ms (145 instructions per evaluation before, 65 %
// busy: two rounds of scalar loads per segment and iteration, t_f for every bin,
// a copy of one coefficient per cubic and bin, a 24-operation e^{i phase}).
// RB = 4 measured best: the whole step 25.9 (RB = 2), 24.9 (3), 24.5 ms (4);
// fewer iterations pay the record loads and the walker more often.
//
// ADJ: also the adjoint pass of the direct log-likelihood's gradient: after the
// mode sum of a block, Lam = 4 w (d~ - h~) per bin and channel, then the modes
// again, each bin's quantity adjoints (mode_adjoint) contracted over the bins
// that share a segment (adjoint_accumulate) and added to the segment's adjoint record
// where the walker leaves it. At least 4 wavefronts per SIMD (at most 128 VGPRs), 3
// with the adjoint pass, which takes one iteration per block: it holds Lam as well,
// and more iterations spill (256 uneven templates of 1.58 M bins, 1, 2, 3 and 4 of
// them: 23.4, 24.1, 33 and 37 ms). Bound by instruction issue, 82 % of the cycles: 396
// vector instructions per (mode, 64 bins), 134 of them FP64 arithmetic, 8 matrix
// instructions, the rest moves, selections and the walker's. 32 sums over the wavefront by
// exchanges between lanes in place of the matrix product, and a record loaded per
// lane: 43.5 ms.

constexpr int DENSE_RB = 4, ADJ_RB = 1;  // iterations of 64 dense bins per block of a wavefront

// A record at a wavefront-uniform address, its bounds and cubics (t_f's apart)
// loaded in one round: the statements keep the compiler from sinking the
// cubics' loads below the bounds check, which would serialise two rounds of
// memory latency.
__device__ inline SegRec load_uniform(const SegRec* rc)
{
    SegRec q;
    q.x_lo = rc->x_lo;
    q.x_hi = rc->x_hi;
    q.win = rc->win;
#pragma unroll
    for (int k = 0; k < S_TF; k++) q.q[k] = rc->q[k];
#pragma unroll
    for (int k = 0; k < S_TF; k++)
        asm volatile("" ::"s"(q.q[k].y), "s"(q.q[k].c1), "s"(q.q[k].c2), "s"(q.q[k].c3));
    // an instruction takes one scalar operand: the c2 are copied to vector
    // registers here, once for the iterations that share the record, where each
    // cubic would otherwise copy one of its first two coefficients for every bin
#pragma unroll
    for (int k = 0; k < S_TF; k++) asm volatile("" : "+v"(q.q[k].c2));
    return q;
}

// Steps of the walker before the lanes left over search for themselves.
constexpr int WALK_STEPS = 4;

// segment of f in a log-spaced grid, from an FP32 log2 (within one or two)
__device__ inline int segment_estimate(double f, double glo, double gis, int L)
{
    return (int)fmin(fmax(((double)__log2f((float)f) - glo) * gis, 0.0), (double)(L - 2));
}

// The walker over one mode's segments for a block of RB x 64 bins. 'cur': the
// segment to start from (-1: not known); returns the one it ended in, or -1 if bins
// are left over (todo) for their lanes to search. todo[r] says on entry whether
// the lane holds a bin.
//   guess(f)             segment near f
//   visit(r, in, q, rc)  lanes 'in' of iteration r lie in segment q (record rc)
//   leave(i)             segment i is done
template <int RB, class Guess, class Visit, class Leave>
__device__ inline int walk_block(int cur, const SegRec* rm, int M, int L, const double (&f)[RB], bool (&todo)[RB],
                                 Guess guess, Visit visit, Leave leave)
{
    if (cur < 0) cur = __builtin_amdgcn_readfirstlane(guess(f[0]));
    // lanes below the current segment send the walker down, else lanes above it up;
    // a sorted block needs one step per segment it spans
    bool open = true;
    for (int step = 0; step < WALK_STEPS; step++) {
        cur = __builtin_amdgcn_readfirstlane(cur);
        const SegRec* rc = rm + (unsigned)(cur * M);
        const SegRec q = load_uniform(rc);
        bool rest = false;
#pragma unroll
        for (int r = 0; r < RB; r++) {
            const bool in = todo[r] && f[r] >= q.x_lo && f[r] < q.x_hi;
            visit(r, in, q, rc);
            todo[r] = todo[r] && !in;
            rest = rest || todo[r];
        }
        leave(cur);
        if (!__any(rest)) { open = false; break; }
        bool below = false, above = false;
#pragma unroll
        for (int r = 0; r < RB; r++) {
            below = below || (todo[r] && f[r] < q.x_lo);
            above = above || (todo[r] && f[r] >= q.x_hi);
        }
        if (__any(below) && cur > 0) cur--;
        else if (__any(above) && cur < L - 2) cur++;
        else { open = false; break; }  // beyond the grid's ends: no contribution
    }
    return open ? -1 : cur;
}

template <bool ADJ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ADJ ? 3 : 4, 8))) void k_dir_like_t(double* __restrict__ partial, double* __restrict__ Yadj,
                                                    const int* __restrict__ band,
                                                  const int* __restrict__ total, const int* __restrict__ perm,
                                                  int* __restrict__ next, const SegRec* __restrict__ R,
                                                  const double* __restrict__ grid_lo,
                                                  const double* __restrict__ grid_istep,
                                                  const long* __restrict__ off, const int* __restrict__ len,
                                                  const double* __restrict__ t_start,
                                                  const double* __restrict__ t_end, const double* __restrict__ freqs,
                                                  const cd* __restrict__ dch, const double* __restrict__ wts, int N,
                                                  int B, int M, int chunk)
{
    constexpr int RB = ADJ ? ADJ_RB : DENSE_RB;
    __shared__ double2 s_tab[1024];
    const int nitems = total[0];
    const int lane = threadIdx.x & 63;
    fill_etab1k(s_tab, threadIdx.x, blockDim.x);
    __syncthreads();
    // The wavefront's items in the chunk-major order: the first by its number, the
    // following from a counter (dynamic: the items running at any time stay a window of
    // consecutive entries, i.e. the same dense bins). The counter takes some 8 ns per
    // wavefront, so with none left beyond the first ones it is not asked: 16 templates of
    // 65536 bins in 4096 items, 8192 wavefronts: 180 -> 72 us (56 in item_bins' items).
    const int waves = gridDim.x * (blockDim.x >> 6);
    int pi = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    for (bool first = true;; first = false) {
        // The barrier (no instruction) is convergent: without one in this block the
        // compiler may thread the branch on lane 0 with one at the end of the loop, and
        // the other lanes would go round it on their own
        __builtin_amdgcn_wave_barrier();
        if (!first) {
            if (waves >= nitems) break;
            pi = 0;
            if (lane == 0) pi = atomicAdd(next, 1);
            pi = waves + __builtin_amdgcn_readfirstlane(pi);
        }
        if (pi >= nitems) break;
        const int it = perm[pi];
        int b;
        const int g = item_chunk(band, B, it, chunk, b);
        const int kw0 = max(band[3 * b], g * chunk), kw1 = min(band[3 * b + 1], (g + 1) * chunk);
        const long base = off[b];
        const int L = len[b];
        const double ts = t_start[b], te = t_end[b];
        double a0 = 0.0, a1 = 0.0, a2 = 0.0;
        // lane m: the segment that mode m's last block ended in (at first an estimate);
        // -1: not known, -2: a degenerate grid, no segment holds any f
        int curv = -1;
        if (lane < M) {
            const double gis = grid_istep[b * M + lane];
            curv = gis > 0.0 ? segment_estimate(freqs[kw0], grid_lo[b * M + lane], gis, L) : -2;
        }
        for (int kb = kw0; kb < kw1; kb += RB * 64) {
            const int curs = curv;  // where the modes' walkers start, for the adjoint pass
            double f[RB];
            cd h[RB][3];
#pragma unroll
            for (int r = 0; r < RB; r++) {
                // bins past the item repeat its last one (not summed below)
                f[r] = freqs[min((unsigned)(kb + 64 * r + lane), (unsigned)(kw1 - 1))];
#pragma unroll
                for (int ch = 0; ch < 3; ch++) h[r][ch] = mk(0.0, 0.0);
            }
            for (int m = 0; m < M; m++) {
                int cur = __builtin_amdgcn_readlane(curv, m);
                if (cur == -2) continue;
                const SegRec* rm = R + base * M + m;
                // loads the grid's parameters only where they are needed
                auto guess = [&](double fr) {
                    return segment_estimate(fr, grid_lo[b * M + m], grid_istep[b * M + m], L);
                };
                bool todo[RB];
#pragma unroll
                for (int r = 0; r < RB; r++) todo[r] = kb + 64 * r + lane < kw1;
                cur = walk_block<RB>(
                    cur, rm, M, L, f, todo, guess,
                    [&](int r, bool in, const SegRec& q, const SegRec* rc) {
                        if (in) add_mode_window(h[r], q, rc, f[r] - q.x_lo, ts, te, s_tab);
                    },
                    [](int) {});
                if (cur < 0) {
#pragma unroll
                    for (int r = 0; r < RB; r++)
                        if (todo[r]) mode_per_lane(h[r], rm, M, L, f[r], guess(f[r]), ts, te, s_tab);
                }
                curv = lane == m ? cur : curv;
            }
            // bins past the item repeat its last one with weight 0 (no branch, so
            // that the loads of all iterations can go ahead of the arithmetic)
#pragma unroll
            for (int r = 0; r < RB; r++) {
                const bool mine = kb + 64 * r + lane < kw1;
                const unsigned k = min((unsigned)(kb + 64 * r + lane), (unsigned)(kw1 - 1));
#pragma unroll
                for (int ch = 0; ch < 3; ch++) {
                    const double wk = (wts + (long)ch * N)[k];
                    const cd d = (dch + (long)ch * N)[k];
                    const double w = mine ? wk : 0.0;
                    const cd ht = h[r][ch] * w;
                    a0 = fma(d.re, ht.re, fma(d.im, ht.im, a0));
                    a1 = fma(d.re, ht.im, fma(-d.im, ht.re, a1));
                    a2 = fma(ht.re, ht.re, fma(ht.im, ht.im, a2));
                    if constexpr (ADJ) h[r][ch] = (4.0 * w) * (d - ht);  // Lam
                }
            }
            if constexpr (ADJ) {
                for (int m = 0; m < M; m++) {
                    int cur = __builtin_amdgcn_readlane(curs, m);
                    if (cur == -2) continue;
                    const SegRec* rm = R + base * M + m;
                    auto guess = [&](double fr) {
                        return segment_estimate(fr, grid_lo[b * M + m], grid_istep[b * M + m], L);
                    };
                    double* Ym = Yadj + (base * M + m) * (long)NA;
                    bool todo[RB];
#pragma unroll
                    for (int r = 0; r < RB; r++) todo[r] = kb + 64 * r + lane < kw1;
                    double acc[2] = {0.0, 0.0};
                    bool used = false;
                    cur = walk_block<RB>(
                        cur, rm, M, L, f, todo, guess,
                        [&](int r, bool in, const SegRec& q, const SegRec* rc) {
                            const double x = in ? f[r] - q.x_lo : 0.0;
                            in = in && (q.win == WIN_ALL || (q.win == WIN_MIXED && bin_in_window(rc->q[S_TF], x, ts, te)));
                            if (!__any(in)) return;
                            used = true;
                            // every lane evaluates (the others at x = 0), so that a block
                            // within the segment needs no selection
                            double a[8];
                            mode_adjoint(a, q.q, x, h[r], s_tab);
                            if (!__all(in)) {
#pragma unroll
                                for (int k = 0; k < 8; k++) a[k] = in ? a[k] : 0.0;
                            }
                            adjoint_accumulate(acc, a, x, lane);
                        },
                        [&](int i) {
                            if (!used) return;
                            // the four blocks of bins, then one lane per coefficient
                            double* y = Ym + (long)i * M * NA;
#pragma unroll
                            for (int g = 0; g < 2; g++) {
                                double v = acc[g];
                                v += __shfl_xor(v, 4, 64);
                                v += __shfl_xor(v, 8, 64);
                                if ((lane & 12) == 0) unsafeAtomicAdd(y + adj_q(4 * g + (lane >> 4)) * 4 + (lane & 3), v);
                                acc[g] = 0.0;
                            }
                            used = false;
                        });
                    if (cur < 0) {
#pragma unroll
                        for (int r = 0; r < RB; r++)
                            if (todo[r]) mode_adjoint_per_lane(Ym, rm, M, L, f[r], guess(f[r]), ts, te, h[r], s_tab);
                    }
                }
            }
        }
        a0 = wsum(a0);
        a1 = wsum(a1);
        a2 = wsum(a2);
        // every lane holds the sums: lanes l, l + 4, ... write the same value l
        const int c = lane & 3;
        partial[4 * (long)it + c] = c == 0 ? a0 : (c == 1 ? a1 : (c == 2 ? a2 : 0.0));
    }
}

// One wavefront per binary: lane l adds the binary's items l, l + 64, ... (in
// item order), then the wavefront adds the 64 lane sums in a fixed tree; the
// result does not depend on the schedule of the dense-band kernel.
__global__ __launch_bounds__(64) void k_dir_reduce(double* __restrict__ d_h, double* __restrict__ h_h,
                                                   const double* __restrict__ partial, const int* __restrict__ band,
                                                   const int* __restrict__ total, int B)
{
    const int b = blockIdx.x;
    const int c0 = band[3 * b + 2];
    const int c1 = b + 1 < B ? band[3 * (b + 1) + 2] : total[0];
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
    for (int c = c0 + (int)threadIdx.x; c < c1; c += 64) {
        s0 += partial[4 * (long)c];
        s1 += partial[4 * (long)c + 1];
        s2 += partial[4 * (long)c + 2];
    }
    s0 = wsum(s0);
    s1 = wsum(s1);
    s2 = wsum(s2);
    if (threadIdx.x == 0) {
        d_h[2 * b] = 4.0 * s0;
        d_h[2 * b + 1] = 4.0 * s1;
        h_h[2 * b] = 4.0 * s2;
        h_h[2 * b + 1] = 0.0;
    }
}

// ---------------------------------------------------------------- gradient kernels

__global__ void k_dirg_zero(double* __restrict__ y, long n)
{
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) y[i] = 0.0;
}

// records with tangents, one lane per (binary, mode)
__global__ __launch_bounds__(64) void k_dirg_setup(gradk::GradRec* __restrict__ grecs,
                                                   const double* __restrict__ params, int B, ModeList modes, int M,
                                                   const double* __restrict__ qnm, int table_len, double dspin)
{
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= B * M) return;
    const int b = idx / M, mi = idx % M;
    gradk::grad_setup_one(grecs[idx], params, B, b, modes.ell[mi], modes.mm[mi], qnm, table_len, dspin);
}

// Adjoint of the not-a-knot spline construction (k_dir_spline): segment-coefficient
// adjoints (Yadj) -> adjoints Ya (S, M, NQ) of the knot values, of one (binary, mode)
// and the eight quantities that have them, one lane per knot, in the blocks of
// k_dir_spline. Row j of the transposed system couples by h_{j-2} and h_{j+1} against
// 2 (h_{j-1} + h_j) (h_i: interval i); the end rows are folded like the system's
// (z_0 = s_0 / h_1 - z_1, and the same at the other end). A solution forgets like
// the system's own, the inverse being the transpose.
//
// Bound by the records' reads (288 B per (knot, mode), one lane's at a time) and the
// exchanges: 256 uneven templates, 2.36 M records: 0.66 ms (0.16 ms at the rate of a
// copy). Thomas sweeps, one lane per (mode, quantity): 8.7 ms.
template <bool PACK>
__global__ __launch_bounds__(SPL_T) __attribute__((amdgpu_waves_per_eu(4))) void k_dirg_spline_adj(
    double* __restrict__ Ya, const double* __restrict__ Yadj, const double* __restrict__ X,
    const int4* __restrict__ spl, const long* __restrict__ off, const int* __restrict__ len, int M)
{
    constexpr int T = SPL_T, NA8 = 8;
    __shared__ double sh[(NA8 + 2) * T];
    const int t = threadIdx.x;
    const SplineRow w = spline_row<PACK>(spl, len, M);
    const int i = w.i, n = w.n;
    const long base = off[w.b];
    const bool seg = i < n - 1;  // segment i
    const long p = (base + (w.any ? i : n - 1)) * M + w.m;
    const double x = X[p];
    sh[t] = x;
    __syncthreads();
    auto at = [&](int d) { return min(max(t + d, 0), T - 1); };
    // h[k]: interval i - 2 + k
    double h[4], xk = sh[at(-2)];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const double xn = sh[at(k - 1)];
        h[k] = xn - xk;
        xk = xn;
    }
    const double ih = rcp_pos(h[2]);
    // this segment's share of the value and slope adjoints of its two knots
    double yb[NA8], sb[NA8], cy[NA8];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA8; q++) {
        const double* c = Yadj + p * NA + adj_q(q) * 4;
        const double tb = (c[3] * ih - c[2]) * ih, sl = c[2] * ih - 2.0 * tb;
        cy[q] = seg ? sl * ih : 0.0;
        yb[q] = seg ? c[0] - cy[q] : 0.0;
        sb[q] = seg ? c[1] - c[2] * ih + tb : 0.0;
        sh[q * T + t] = seg ? tb : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA8; q++)
        if (t > 0) sb[q] += sh[q * T + t - 1];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA8; q++) sh[q * T + t] = cy[q];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA8; q++)
        if (t > 0) yb[q] += sh[q * T + t - 1];
    __syncthreads();
    // the transposed system; rows with all their neighbours in the block
    const bool solve = i > 0 && i < n - 1 && t > 0 && t + 1 < T && (i == 1 || t > 1) && (i == n - 2 || t + 2 < T);
    const bool low = solve && i == 1, high = solve && i == n - 2;
    const double d = h[1] + h[2];
    const double diag = 2.0 * d - (low ? d : 0.0) - (high ? d : 0.0), ib = rcp_pos(diag);
    const double a = solve && !low ? h[0] * ib : 0.0, c = solve && !high ? h[3] * ib : 0.0;
    double z[NA8];
#pragma unroll
    for (int q = 0; q < NA8; q++) sh[q * T + t] = sb[q];
    __syncthreads();
    const double iel = rcp_pos(h[2]), ieh = rcp_pos(h[1]);  // pivots of the end rows
#pragma unroll
    for (int q = 0; q < NA8; q++) {
        double v = sb[q];
        if (low) v -= d * (sh[q * T + t - 1] * iel);
        if (high) v -= d * (sh[q * T + t + 1] * ieh);
        z[q] = solve ? v * ib : 0.0;
    }
    double zl[NA8];  // the end rows' own terms, by their neighbours
#pragma unroll
    for (int q = 0; q < NA8; q++) zl[q] = low ? sh[q * T + t - 1] * iel : (high ? sh[q * T + t + 1] * ieh : 0.0);
    // (a grid of four knots has two such rows, in different lanes)
    __syncthreads();
    pcr_solve(a, c, z, sh, t, w.t0, w.t1);
#pragma unroll
    for (int q = 0; q < NA8; q++) {
        if (i != 0 && i < n - 1) sh[q * T + t] = z[q];
        if (low) sh[q * T + t - 1] = zl[q] - z[q];
        if (high) sh[q * T + t + 1] = zl[q] - z[q];
    }
    __syncthreads();
    // adjoint of the segment's slope (y_{i+1} - y_i) / h_i from the right sides of rows
    // i and i + 1 (3 (h_r m_l + h_l m_r)) and of the end rows
    double k0 = i > 0 && i < n - 1 ? 3.0 * h[1] : 0.0;      // row i
    double k1 = i + 1 < n - 1 ? 3.0 * h[3] : 0.0;           // row i + 1
    double km = 0.0, k2 = 0.0;                              // rows i - 1, i + 2
    if (i == 0) k0 = (h[2] + 2.0 * (h[2] + h[3])) * h[3] * rcp_pos(h[2] + h[3]);
    if (i == 1) km = h[1] * h[1] * rcp_pos(h[1] + h[2]);
    if (i == n - 3) k2 = h[3] * h[3] * rcp_pos(h[2] + h[3]);
    if (i == n - 2) k1 = (2.0 * (h[1] + h[2]) + h[2]) * h[1] * rcp_pos(h[1] + h[2]);
#pragma unroll
    for (int q = 0; q < NA8; q++) {
        double g = k0 * sh[q * T + t] + k1 * sh[q * T + at(1)];
        if (i == 1) g += km * sh[q * T + t - 1];
        if (i == n - 3) g += k2 * sh[q * T + at(2)];
        cy[q] = seg ? g * ih : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NA8; q++) sh[q * T + t] = cy[q];
    __syncthreads();
    if (!w.out) return;
#pragma unroll
    for (int q = 0; q < NA8; q++)
        Ya[p * NQ + adj_q(q)] = yb[q] - cy[q] + (i > 0 ? sh[q * T + t - 1] : 0.0);
}

// Knot-level contraction, a workgroup per (binary, mode) and up to GRAD_T knots, by its
// entry of the plan's table; the
// knot-value adjoints of A, phase and T weight the waveform's and response's
// tangents at the knot's frequency (grad_point_core, no window rule: the
// window acts on the dense bins).
__global__ __launch_bounds__(gradk::GRAD_T) __attribute__((amdgpu_waves_per_eu(2))) void k_dirg_knots(
    double* __restrict__ gpart, const gradk::GradRec* __restrict__ grecs, const double* __restrict__ Ya,
    const double* __restrict__ X, const int4* __restrict__ knots, const long* __restrict__ off,
    const int* __restrict__ len, const double* __restrict__ params, int B, int M, resp::OrbitTab orb, int TDItag,
    int rescaled, int tdi2, double initial_t_val)
{
    __shared__ gradk::GradShared sh;
    const int4 w = knots[blockIdx.x];
    const int bm = w.x, b = bm / M, m = bm % M;
    const int n = len[b], i = w.y + threadIdx.x;
    Window win;
    win.t_ref = params[P_TREF * B + b];
    win.ts = 0.0;
    win.te = 0.0;
    win.dt_shift = win.t_ref - initial_t_val;
    const double dist = params[P_DIST * B + b];
    const gradk::GradRec& G = gradk::grad_stage(sh, grecs + bm);
    double acc[gradk::NGRAD];
    for (int p = 0; p < gradk::NGRAD; p++) acc[p] = 0.0;
    if (i < n) {
        const long rec = (off[b] + i) * M + m;
        const double* y = Ya + rec * NQ;
        auto weights = [&](const cd*, cd, double, cd W[3], double& a_A, double& a_Ph) {
            for (int c = 0; c < 3; c++) W[c] = mk(y[3 + 2 * c], -y[4 + 2 * c]);
            a_A = y[0];
            a_Ph = y[1];
        };
        gradk::grad_point_core(G, orb, X[rec], win, false, weights, TDItag, rescaled, tdi2, dist, acc, sh.tab,
                               sh.tan + threadIdx.x, blockDim.x);
    }
    gradk::grad_sum(sh, acc, gpart + (long)w.z * gradk::NGRAD);
}

// grad[p B + b] = sum over the binary's rows of gpart: one wavefront per binary
__global__ __launch_bounds__(64) void k_dirg_reduce(double* __restrict__ grad, const double* __restrict__ gpart,
                                                    const int* __restrict__ gpart_b, int B)
{
    const int b = blockIdx.x, r1 = gpart_b[b + 1];
    double acc[gradk::NGRAD];
    for (int p = 0; p < gradk::NGRAD; p++) acc[p] = 0.0;
    for (int r = gpart_b[b] + threadIdx.x; r < r1; r += 64)
        for (int p = 0; p < gradk::NGRAD; p++) acc[p] += gpart[(long)r * gradk::NGRAD + p];
    for (int p = 0; p < gradk::NGRAD; p++) {
        const double v = wsum(acc[p]);
        if (threadIdx.x == 0) grad[(long)p * B + b] = v;
    }
}

template <class T>
T* dalloc(size_t n, bool& ok)
{
    void* p = nullptr;
    if (!ok || hipMalloc(&p, n * sizeof(T) + 256) != hipSuccess) {
        ok = false;
        return nullptr;
    }
    return static_cast<T*>(p);
}

void plan_free(bbhx_direct_plan* p)
{
    void* bufs[] = {p->off, p->len, p->recs, p->X, p->Cf, p->Yc, p->grid_lo, p->grid_istep, p->band,
                    p->total, p->partial, p->perm, p->cnt, p->next, p->Yadj, p->grecs, p->gpart, p->grid_b,
                    p->spl, p->knots, p->gpart_b};
    for (void* b : bufs)
        if (b) (void)hipFree(b);
}

// a host table on the device
template <class T>
T* upload(const std::vector<T>& v, bool& ok)
{
    T* d = dalloc<T>(v.size(), ok);
    ok = ok && (v.empty() || hipMemcpy(d, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice) == hipSuccess);
    return d;
}

// Binaries by the lanes that k_dir_grid takes for their knots, 64, 128 or GRID_T, and the
// workgroups of the spline kernels; false: more of these than a table holds.
bool lay_out_forward(bbhx_direct_plan* p, std::vector<int>& grid_b, std::vector<int4>& spl)
{
    for (int c = 0; c < 3; c++) {
        TablePart& part = p->grid_parts[c];
        part.threads = 64 << c;
        part.first = (long)grid_b.size();
        for (int b = 0; b < p->B; b++) {
            const int n = p->lengths[b];
            if (std::min(GRID_T, n <= 64 ? 64 : (n <= 128 ? 128 : GRID_T)) != part.threads) continue;
            grid_b.push_back(b);
            part.lmax = std::max(part.lmax, n);
        }
        part.count = (long)grid_b.size() - part.first;
    }
    for (int b = 0; b < p->B; b++)
        for (int m = 0; m < p->M && 2 * p->lengths[b] > SPL_T; m++)
            for (int blk = 0; blk < spline_blocks(p->lengths[b]); blk++) spl.push_back({b * p->M + m, 1, SPL_T, blk});
    p->nblocks = (long)spl.size();
    for (int b = 0; b < p->B; b++)
        for (int m = 0; m < p->M && 2 * p->lengths[b] <= SPL_T; m++) {
            const int bm = b * p->M + m, n = p->lengths[b];
            int4* last = (long)spl.size() > p->nblocks ? &spl.back() : nullptr;
            if (last && last->x + last->y == bm && (last->y + 1) * std::max(last->z, n) <= SPL_T) {
                last->y++;
                last->z = std::max(last->z, n);
            } else
                spl.push_back({bm, 1, n, 0});
        }
    p->nspl = (long)spl.size();
    return p->nspl <= 2147483647L;
}

// The workgroups of k_dirg_knots, by their lanes; false: as above.
bool lay_out_knots(bbhx_direct_plan* p, std::vector<int4>& knots, std::vector<int>& gpart_b)
{
    long rows = 0;
    for (int b = 0; b < p->B; b++) {
        gpart_b.push_back((int)rows);
        rows += (long)p->M * gradk::grad_chunks(p->lengths[b]);
        if (rows > 2147483647L) return false;
    }
    gpart_b.push_back((int)rows);
    for (int c = 0; c < 4; c++) {
        TablePart& part = p->knot_parts[c];
        part.threads = 64 * (c + 1);
        part.first = (long)knots.size();
        for (int b = 0; b < p->B; b++) {
            const int n = p->lengths[b], chunks = gradk::grad_chunks(n);
            if (gradk::grad_threads(n) != part.threads) continue;
            for (int m = 0; m < p->M; m++)
                for (int k = 0; k < chunks; k++)
                    knots.push_back({b * p->M + m, k * part.threads, gpart_b[b] + m * chunks + k, 0});
        }
        part.count = (long)knots.size() - part.first;
    }
    return true;
}

}  // namespace

// ---- dense bins per work item
//
// A work item is what one wavefront takes: a caller's chunk (bins per workgroup
// and pass) split over the workgroup's wavefronts, and less than that for a small
// batch, down to ITEM_MIN bins (half a block). Up to FEW bins in all about ITEMS_ONCE
// items, the wavefronts of the default launch on 256 CUs: if the bands hold no more than
// that, each has a first item and no other, and the counter of the following ones, 8 ns
// a time, is not asked. Above, twice as many, for the dynamic order to balance. Plans of
// up to SMALL_ITEMS such items have buffers for them. The whole call with at least 256
// bins and 16384 items at any size, and with this rule: 16 templates of 65536 bins 321 and
// 303 us, 48 of them 440 and 395, 64 499 and 433; with ITEMS_ONCE at 128 and 256 of
// them 630 became 657 and 1005 became 1174 us. At 1024 templates of 1.58 M bins the item
// size does not matter (items of 4096, 8192 and 16384 bins: 25.4, 25.5 and 26.3 ms).
//
// The size does not follow the caller's launch: counted for its own wavefronts, 4096
// instead of 8192 of them took 171 instead of 222 us for 16 such templates, but 861 instead
// of 682 for 200 (fewer items balance worse), 2048 took 224 instead of 210 for 16. Nor does
// it count the items of a whole data set exactly: 16 templates of 65537 bins, 8208 items at
// most and 8192 at hand, 156 us, 171 with the next larger size.
constexpr long ITEM_MIN = 128, SMALL_ITEMS = 1L << 19, ITEMS_ONCE = 8192, FEW = ITEMS_ONCE * 512;

static int item_bins(const bbhx_direct_plan* p, int chunk, int block)
{
    long n = chunk / (block / 64);
    const long all = (long)p->B * p->N;  // the whole data set of every binary
    const long fine = all / (all <= FEW ? ITEMS_ONCE : 2 * ITEMS_ONCE);
    n = std::min(n, std::max(fine, ITEM_MIN));
    n = n <= ITEM_MIN ? ITEM_MIN : (n + 255) / 256 * 256;  // half a block, or whole ones
    return (int)std::max(n, (long)p->min_item);
}

static int plan_create(bbhx_direct_plan** out, int numBinAll, const int* lengths_host, int numModes, int data_length,
                       int min_chunk)
{
    std::vector<long> off(numBinAll);
    long S = 0;
    int Lmax = 0;
    for (int b = 0; b < numBinAll; b++) {
        if (lengths_host[b] < 4) return ERR_ARGS;
        off[b] = S;
        S += lengths_host[b];
        Lmax = lengths_host[b] > Lmax ? lengths_host[b] : Lmax;
    }
    // the default-grid t(f) of one (binary, mode) lives in LDS
    if ((size_t)Lmax * sizeof(double) > 48 * 1024) return ERR_ARGS;
    auto p = std::make_unique<bbhx_direct_plan>();
    (void)hipGetDevice(&p->device);
    p->lengths.assign(lengths_host, lengths_host + numBinAll);
    p->B = numBinAll;
    p->M = numModes;
    p->N = data_length;
    p->Lmax = Lmax;
    p->min_chunk = min_chunk;
    // small batches are cut finer than the caller's chunks (item_bins)
    p->min_item = (long)numBinAll * data_length <= ITEM_MIN * SMALL_ITEMS ? std::min(min_chunk, (int)ITEM_MIN)
                                                                         : min_chunk;
    p->S = S;
    p->max_items = (long)numBinAll * ((data_length + p->min_item - 1) / p->min_item) + numBinAll;
    if (p->max_items > 2147483647L) return ERR_ARGS;
    std::vector<int> grid_b;
    std::vector<int4> spl;
    if (!lay_out_forward(p.get(), grid_b, spl)) return ERR_ARGS;
    bool ok = true;
    const size_t SM = (size_t)S * numModes;
    p->grid_b = upload(grid_b, ok);
    p->spl = upload(spl, ok);
    p->off = dalloc<long>(numBinAll, ok);
    p->len = dalloc<int>(numBinAll, ok);
    p->recs = dalloc<FusedRec>((size_t)numBinAll * numModes, ok);
    p->X = dalloc<double>(SM, ok);
    p->Cf = dalloc<double>(SM * RS, ok);
    p->Yc = dalloc<double>(SM * NQ, ok);
    p->grid_lo = dalloc<double>((size_t)numBinAll * numModes, ok);
    p->grid_istep = dalloc<double>((size_t)numBinAll * numModes, ok);
    p->band = dalloc<int>((size_t)numBinAll * 3, ok);
    p->total = dalloc<int>(1, ok);
    p->partial = dalloc<double>((size_t)p->max_items * 4, ok);
    p->max_chunks = (data_length + p->min_item - 1) / p->min_item;
    p->perm = dalloc<int>((size_t)p->max_items, ok);
    p->cnt = dalloc<int>((size_t)p->max_chunks + 1, ok);
    p->next = dalloc<int>(1, ok);
    if (!ok) {
        plan_free(p.get());
        return ERR_ALLOC;
    }
    if (hipMemcpy(p->off, off.data(), sizeof(long) * numBinAll, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemcpy(p->len, lengths_host, sizeof(int) * numBinAll, hipMemcpyHostToDevice) != hipSuccess) {
        plan_free(p.get());
        return ERR_LAUNCH;
    }
    *out = p.release();
    return OK;
}

extern "C" int bbhx_hip_direct_plan_create(bbhx_direct_plan** out, int numBinAll, const int* lengths_host,
                                           int numModes, int data_length, int min_chunk)
{
    if (!out || numBinAll < 1 || !lengths_host || numModes < 1 || numModes > MAX_MODES || data_length < 1 ||
        min_chunk < 64)
        return ERR_ARGS;
    try {
        return plan_create(out, numBinAll, lengths_host, numModes, data_length, min_chunk);
    } catch (const std::bad_alloc&) {
        return ERR_ALLOC;
    }
}
extern "C" int bbhx_hip_direct_plan_destroy(bbhx_direct_plan* p)
{
    if (!p) return ERR_ARGS;
    (void)hipDeviceSynchronize();
    plan_free(p);
    delete p;
    return OK;
}

extern "C" long bbhx_hip_direct_plan_bytes(const bbhx_direct_plan* p)
{
    if (!p) return -1;
    const long SM = p->S * p->M;
    long bytes = SM * 8 * (1 + RS + NQ) + (long)p->B * p->M * (sizeof(FusedRec) + 16) + p->max_items * 36 + p->B * 28 +
                 16 * p->nspl + 4L * (p->max_chunks + 1);
    if (p->Yadj)
        bytes += SM * 8 * NA + (long)p->B * p->M * sizeof(gradk::GradRec) + p->B * 4 + p->nknots * (16 + 8 * gradk::NGRAD);
    return bytes;
}

extern "C" int bbhx_hip_direct_plan_band(const bbhx_direct_plan* p, int* band_host)
{
    if (!p || !band_host) return ERR_ARGS;
    std::vector<int> b3((size_t)p->B * 3);
    if (hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(b3.data(), p->band, sizeof(int) * b3.size(), hipMemcpyDeviceToHost) != hipSuccess)
        return ERR_LAUNCH;
    for (int b = 0; b < p->B; b++) {
        band_host[2 * b] = b3[3 * b];
        band_host[2 * b + 1] = b3[3 * b + 1];
    }
    return OK;
}

namespace {

// The launches of a spline kernel, for blocks and for packs
template <class Kernel, class Launch>
int spline_launches(const bbhx_direct_plan* p, Kernel blocks, Kernel packs, Launch launch)
{
    const int rc = launch_rows(p->nblocks, 1, SPL_T, [&](long r, dim3 g) { launch(blocks, p->spl + r, g); });
    if (rc != OK) return rc;
    return launch_rows(p->nspl - p->nblocks, 1, SPL_T,
                       [&](long r, dim3 g) { launch(packs, p->spl + p->nblocks + r, g); });
}

// The launch sequence of the fused direct likelihood; with grad != nullptr
// also its gradient (the plan's gradient buffers must exist).
int direct_launch(bbhx_direct_plan* p, double* d_h, double* h_h, double* grad, int* flags, const double* params,
                  const double* t_start, const double* t_end, const int* ells_host, const int* mms_host,
                  int numModes, const double* dataFreqs, const double* dataChannels, const double* noiseFactors,
                  const double* qnm, int table_len, double dspin, double initial_t_val, double mf_min, double mf_max,
                  const bbhx_response* orbits, int TDItag, int rescaled, int tdi2, int chunk, int block, int grid,
                  void* stream)
{
    if (!p) return ERR_ARGS;
    if (chunk < p->min_chunk || (block != 64 && block != 128 && block != 256) || grid < 1) return ERR_ARGS;
    chunk = item_bins(p, chunk, block);
    int dev = -1;
    (void)hipGetDevice(&dev);
    if (dev != p->device || numModes != p->M) return ERR_ARGS;
    resp::OrbitTab orb;
    if (!response_orbit_tab(orbits, orb)) return ERR_ARGS;
    ModeList ml;
    const int mst = check_modes(ells_host, mms_host, numModes, ml);
    if (mst != OK) return mst;
    if (!d_h || !h_h || !flags || !params || !t_start || !t_end || !dataFreqs || !dataChannels || !noiseFactors ||
        !qnm || table_len < 2 || !(mf_min > 0.0) || !(mf_max > mf_min))
        return ERR_ARGS;
    if (grad && !p->Yadj) return ERR_ARGS;  // bbhx_hip_direct_plan_enable_grad first
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const int B = p->B, M = p->M;
    hipEvent_t ev[3];
    const bool timed = timer_take3(ev);
    if (timed) (void)hipEventRecord(ev[0], st);
    hipLaunchKernelGGL(k_dir_setup, dim3(setup_blocks(B, M)), dim3(64), 0, st, p->recs, params, B,
                       ml, M, qnm,
                       table_len, dspin);
    int rc = OK;
    for (const TablePart& part : p->grid_parts) {
        if (rc != OK) return rc;
        rc = launch_rows(part.count, M, part.threads, [&](long r, dim3 g) {
            hipLaunchKernelGGL(k_dir_grid, g, dim3(part.threads), sizeof(double) * (size_t)part.lmax, st, p->X, p->Yc,
                               p->grid_lo, p->grid_istep, flags, p->recs, p->grid_b + part.first + r, p->off, p->len,
                               params, t_start, t_end, B, M, ml, orb, TDItag, rescaled, tdi2, initial_t_val, mf_min,
                               mf_max);
        });
    }
    if (rc == OK)
        rc = spline_launches(p, k_dir_spline<false>, k_dir_spline<true>, [&](auto kernel, const int4* spl, dim3 g) {
            hipLaunchKernelGGL(kernel, g, dim3(SPL_T), 0, st, p->X, p->Yc, reinterpret_cast<SegRec*>(p->Cf), spl,
                               p->off, p->len, t_start, t_end, M);
        });
    if (rc != OK) return rc;
    hipLaunchKernelGGL(k_dir_band, dim3(1), dim3(1024), 0, st, p->band, p->total, p->X, p->off, p->len, dataFreqs,
                       p->N, B, M, chunk);
    const int nchunks = (p->N + chunk - 1) / chunk;  // <= max_chunks since chunk >= min_item
    hipLaunchKernelGGL(k_dir_cnt_zero, dim3(ceil_div(nchunks + 1, 256)), dim3(256), 0, st, p->cnt, nchunks + 1,
                       p->next);
    // one lane per possible work item (those past the batch's count exit)
    const long items = std::min(p->max_items, (long)B * nchunks + B);
    const int item_blocks = ceil_div(items, 256);
    hipLaunchKernelGGL(k_dir_cnt, dim3(item_blocks), dim3(256), 0, st, p->cnt, p->band, p->total, B, chunk);
    hipLaunchKernelGGL(k_dir_cnt_scan, dim3(1), dim3(1024), 0, st, p->cnt, nchunks);
    hipLaunchKernelGGL(k_dir_perm, dim3(item_blocks), dim3(256), 0, st, p->perm, p->cnt, p->band, p->total, B, chunk);
    if (grad) {
        hipLaunchKernelGGL(k_dirg_zero, dim3(4096), dim3(256), 0, st, p->Yadj, p->S * (long)M * NA);
        hipLaunchKernelGGL(k_dirg_setup, dim3(ceil_div((long)B * M, 64)), dim3(64), 0, st, p->grecs, params, B, ml, M,
                           qnm, table_len, dspin);
    }
    if (timed) (void)hipEventRecord(ev[1], st);
    if (grad)
        hipLaunchKernelGGL((k_dir_like_t<true>), dim3(grid), dim3(block), 0, st, p->partial, p->Yadj, p->band, p->total,
                           p->perm, p->next, reinterpret_cast<const SegRec*>(p->Cf), p->grid_lo, p->grid_istep,
                           p->off, p->len, t_start, t_end, dataFreqs, reinterpret_cast<const cd*>(dataChannels),
                           noiseFactors, p->N, B, M, chunk);
    else
        hipLaunchKernelGGL((k_dir_like_t<false>), dim3(grid), dim3(block), 0, st, p->partial, nullptr,
                           p->band, p->total, p->perm, p->next, reinterpret_cast<const SegRec*>(p->Cf), p->grid_lo,
                           p->grid_istep, p->off, p->len, t_start, t_end, dataFreqs,
                           reinterpret_cast<const cd*>(dataChannels), noiseFactors, p->N, B, M, chunk);
    hipLaunchKernelGGL(k_dir_reduce, dim3(B), dim3(64), 0, st, d_h, h_h, p->partial, p->band,
                       p->total, B);
    if (grad) {
        // the knot values' adjoints take the place of the values, which are not read again
        rc = spline_launches(p, k_dirg_spline_adj<false>, k_dirg_spline_adj<true>,
                             [&](auto kernel, const int4* spl, dim3 g) {
                                 hipLaunchKernelGGL(kernel, g, dim3(SPL_T), 0, st, p->Yc, p->Yadj, p->X, spl, p->off,
                                                    p->len, M);
                             });
        for (const TablePart& part : p->knot_parts) {
            if (rc != OK) return rc;
            rc = launch_rows(part.count, 1, part.threads, [&](long r, dim3 g) {
                hipLaunchKernelGGL(k_dirg_knots, g, dim3(part.threads), 0, st, p->gpart, p->grecs, p->Yc, p->X,
                                   p->knots + part.first + r, p->off, p->len, params, B, M, orb, TDItag, rescaled,
                                   tdi2, initial_t_val);
            });
        }
        if (rc != OK) return rc;
        hipLaunchKernelGGL(k_dirg_reduce, dim3(B), dim3(64), 0, st, grad, p->gpart, p->gpart_b, B);
    }
    if (timed) (void)hipEventRecord(ev[2], st);
    return hipGetLastError() == hipSuccess ? OK : ERR_LAUNCH;
}

}  // namespace

extern "C" int bbhx_hip_direct_fused(bbhx_direct_plan* p, double* d_h, double* h_h, int* flags, const double* params,
                                     const double* t_start, const double* t_end, const int* ells_host,
                                     const int* mms_host, int numModes, const double* dataFreqs,
                                     const double* dataChannels, const double* noiseFactors, const double* qnm,
                                     int table_len, double dspin, double initial_t_val, double mf_min, double mf_max,
                                     const bbhx_response* orbits, int TDItag, int rescaled, int tdi2, int chunk,
                                     int block, int grid, void* stream)
{
    return direct_launch(p, d_h, h_h, nullptr, flags, params, t_start, t_end, ells_host, mms_host, numModes,
                         dataFreqs, dataChannels, noiseFactors, qnm, table_len, dspin, initial_t_val, mf_min, mf_max,
                         orbits, TDItag, rescaled, tdi2, chunk, block, grid, stream);
}

// 0 and 1 are evaluated alike, in FP64, the faster form: FP32 instructions issue at
// the FP64 rate without packed arithmetic, and an FP32 pass over the quiet
// templates needs its own records, the split of the items and a second pass for the
// loud ones. 1024 uneven templates: 27.7 ms with such a pass, which had the FP64 pass's
// walker but not its later changes, 25.0 then without it, 23 now.
extern "C" int bbhx_hip_direct_plan_set_precision(bbhx_direct_plan* p, int precision)
{
    return p && (precision == 0 || precision == 1) ? OK : ERR_ARGS;
}

static int plan_enable_grad(bbhx_direct_plan* p)
{
    bool ok = true;
    std::vector<int4> knots;
    std::vector<int> gpart_b;
    if (!lay_out_knots(p, knots, gpart_b)) return ERR_ARGS;
    p->nknots = (long)knots.size();
    p->Yadj = dalloc<double>((size_t)p->S * p->M * NA, ok);
    p->grecs = dalloc<gradk::GradRec>((size_t)p->B * p->M, ok);
    p->gpart = dalloc<double>(knots.size() * gradk::NGRAD, ok);
    p->knots = upload(knots, ok);
    p->gpart_b = upload(gpart_b, ok);
    if (!ok) {
        for (void* b : {(void*)p->Yadj, (void*)p->grecs, (void*)p->gpart, (void*)p->knots, (void*)p->gpart_b})
            if (b) (void)hipFree(b);
        p->Yadj = nullptr;
        p->grecs = nullptr;
        p->gpart = nullptr;
        p->knots = nullptr;
        p->gpart_b = nullptr;
        return ERR_ALLOC;
    }
    return OK;
}

extern "C" int bbhx_hip_direct_plan_enable_grad(bbhx_direct_plan* p)
{
    if (!p) return ERR_ARGS;
    if (p->Yadj) return OK;
    try {
        return plan_enable_grad(p);
    } catch (const std::bad_alloc&) {
        return ERR_ALLOC;
    }
}

extern "C" int bbhx_hip_direct_fused_grad(bbhx_direct_plan* p, double* d_h, double* h_h, double* grad, int* flags,
                                          const double* params, const double* t_start, const double* t_end,
                                          const int* ells_host, const int* mms_host, int numModes,
                                          const double* dataFreqs, const double* dataChannels,
                                          const double* noiseFactors, const double* qnm, int table_len, double dspin,
                                          double initial_t_val, double mf_min, double mf_max,
                                          const bbhx_response* orbits, int TDItag, int rescaled, int tdi2, int chunk,
                                          int block, int grid, void* stream)
{
    if (!grad) return ERR_ARGS;
    return direct_launch(p, d_h, h_h, grad, flags, params, t_start, t_end, ells_host, mms_host, numModes, dataFreqs,
                         dataChannels, noiseFactors, qnm, table_len, dspin, initial_t_val, mf_min, mf_max, orbits,
                         TDItag, rescaled, tdi2, chunk, block, grid, stream);
}
