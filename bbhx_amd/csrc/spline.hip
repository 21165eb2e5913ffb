// Batched not-a-knot cubic spline (the reference's CubicSplineInterpolant,
// Interpolate.cu:15-359, which solves with cuSPARSE gtsv2StridedBatch).
//
// The system for the knot slopes s_i is the reference's (identical to scipy
// CubicSpline, bc_type='not-a-knot'): interior rows dx_i s_{i-1} +
// 2(dx_{i-1}+dx_i) s_i + dx_{i-1} s_{i+1} = 3(dx_i m_{i-1} + dx_{i-1} m_i), with the
// not-a-knot end rows folded into their neighbours. It is solved by parallel
// cyclic reduction (spline_device.h), one lane per knot, the quantities on the same
// knots SPL_NR at a time, building each row from x and y, so no band matrix is ever
// materialised; then the segment coefficients
//   c1 = s_i, c2 = (m_i - s_i)/dx - t, c3 = t/dx, t = (s_i + s_{i+1} - 2 m_i)/dx
// written to upper_diag (c1), diag (c2), lower_diag (c3) as in the reference
// (Interpolate.cu:245-261, :332-334). The last knot's c1..c3 entries are set to 0.
//
// Bound by the arrays' reads and writes (40 B per knot and system, all unit-stride) for
// large batches, by the latency of the steps for small ones: 54 systems of 8096 knots 12
// us, 864 of 1024 14 us, 3456 of 4096 0.14 ms, 27648 of 4096 1.3 ms (3.5 TB/s). Thomas
// sweeps took 206 and 159 us (a wavefront per system, 64 row blocks), 2.4 and 6.6 ms (a lane
// per system).

#include "bbhx_hip.h"
#include "common.h"
#include "spline_device.h"

using namespace bbhx;

namespace {

constexpr int SPL_NR = 3;  // systems of one set of knots per workgroup

// Workgroup g of the launch: block g % nb of the knots of item e = e0 + g / nb, which is
// the G sets from G (e % packs) on and the quantities NR (e / packs) and following of P;
// system = quantity * nsub + set. PACK: sets of at most half a workgroup's lanes, which take
// n lanes each, one after another. With a workgroup for each of them, 100000 sets of 4, 16
// and 64 knots and nine quantities took 1036, 1040 and 1066 us instead of 29, 119 and 465
// (a lane per system, by a Thomas sweep: 76, 1287 and 4922). Otherwise G = 1, in a kernel of
// its own, without the room for the sets' end rows.
template <int NR, bool PACK>
__global__ __launch_bounds__(SPL_T) void k_spline(const double* __restrict__ x, const double* __restrict__ y,
                                                  double* __restrict__ Bs, double* __restrict__ c1,
                                                  double* __restrict__ c2, double* __restrict__ c3, int n, int nsub,
                                                  int P, int nb, int G, int e0)
{
    constexpr int T = SPL_T;
    __shared__ double sh[(NR + 2) * T];
    __shared__ double ends[2][NR][PACK ? T / 3 : 1];  // right sides of the sets' two end rows
    const int t = threadIdx.x;
    const int blk = blockIdx.x % nb, e = e0 + blockIdx.x / nb, packs = PACK ? (nsub - 1) / G + 1 : nsub;
    const int set0 = PACK ? e % packs * G : e % packs, q0 = e / packs * NR;
    // this lane's set in the workgroup and its lanes
    const int s = PACK ? t / n : 0, t0 = s * n, t1 = PACK ? min(t0 + n, T) : T;
    const bool any = !PACK || (s < G && set0 + s < nsub);
    const int sub = any ? set0 + s : set0;
    const int first = blk * SPL_U, i = any ? first + t - t0 : n, iy = min(i, n - 1);
    const int row0 = blk == 0 ? 0 : first + SPL_W, row1 = blk == nb - 1 ? n : first + T - SPL_W;
    const double xi = x[(long)sub * n + iy];
    long at[NR];
    double v[NR];
#pragma unroll
    for (int q = 0; q < NR; q++) {
        at[q] = ((long)min(q0 + q, P - 1) * nsub + sub) * n + iy;
        v[q] = y[at[q]];
        sh[(1 + q) * T + t] = v[q];
    }
    sh[t] = xi;
    __syncthreads();
    const int tl = t > 0 ? t - 1 : 0, th = t + 1 < T ? t + 1 : t;
    const double hl = xi - sh[tl], hr = sh[th] - xi;
    const double il = rcp_pos(hl), ir = rcp_pos(hr);
    // rows to solve: the interior ones with both neighbours in the block
    const bool solve = i > 0 && i < n - 1 && t > 0 && t + 1 < T;
    const bool low = solve && i == 1, high = solve && i == n - 2;
    const double d = hl + hr, id = rcp_pos(d);
    double diag = 2.0 * d;
    if (low) diag -= d;
    if (high) diag -= d;
    double ib = rcp_pos(diag);
    const double a = solve && !low ? hr * ib : 0.0, c = solve && !high ? hl * ib : 0.0;
    // three knots: the end rows leave the middle slope open; the parabola's
    const bool parabola = low && high;
    if (parabola) ib = id;
    const double e0l = (hl + 2.0 * d) * hr * id, e0r = hl * hl * id;
    const double e1l = hr * hr * id, e1r = (2.0 * d + hr) * hl * id;
    double mr[NR], r[NR];
#pragma unroll
    for (int q = 0; q < NR; q++) {
        const double ml = (v[q] - sh[(1 + q) * T + tl]) * il;
        mr[q] = (sh[(1 + q) * T + th] - v[q]) * ir;
        double w = 3.0 * (hr * ml + hl * mr[q]);
        if (low) {
            ends[0][q][s] = e0l * ml + e0r * mr[q];
            w -= ends[0][q][s];
        }
        if (high) {
            ends[1][q][s] = e1l * ml + e1r * mr[q];
            w -= ends[1][q][s];
        }
        if (parabola) w = hr * ml + hl * mr[q];
        r[q] = solve ? w * ib : 0.0;
    }
    __syncthreads();
    pcr_solve(a, c, r, sh, t, t0, t1);
    // slopes to the neighbours, the end ones from their rows
#pragma unroll
    for (int q = 0; q < NR; q++) {
        if (i != 0 && i < n - 1) sh[q * T + t] = r[q];
        if (low) sh[q * T + t - 1] = (ends[0][q][s] - d * r[q]) * ir;
        if (high) sh[q * T + t + 1] = (ends[1][q][s] - d * r[q]) * il;
    }
    __syncthreads();
    if (i < row0 || i >= row1) return;
    const bool end = i == n - 1;
#pragma unroll
    for (int q = 0; q < NR; q++) {
        if (q0 + q >= P) break;
        const double sl = sh[q * T + t], u = (sl + sh[q * T + th] - 2.0 * mr[q]) * ir;
        Bs[at[q]] = sl;
        c1[at[q]] = end ? 0.0 : sl;
        c2[at[q]] = end ? 0.0 : (mr[q] - sl) * ir - u;
        c3[at[q]] = end ? 0.0 : u * ir;
    }
}

}  // namespace

extern "C" int bbhx_hip_interpolate(const double* freqs, const double* propArrays, double* B, double* upper_diag,
                                    double* diag, double* lower_diag, int length, int numInterpParams, int numModes,
                                    int numBinAll, void* stream)
{
    if (length < 3 || numInterpParams < 1 || numModes < 1 || numBinAll < 0) return ERR_ARGS;
    if (numBinAll == 0) return OK;
    if (!freqs || !propArrays || !B || !upper_diag || !diag || !lower_diag) return ERR_ARGS;
    long nsys = (long)numInterpParams * numModes * numBinAll;
    if (nsys > 2147483647L) return ERR_ARGS;
    const int nsub = numModes * numBinAll, nb = spline_blocks(length);
    const bool one = numInterpParams < SPL_NR, pack = length <= SPL_T / 2;
    const int groups = one ? numInterpParams : (numInterpParams + SPL_NR - 1) / SPL_NR;
    const int G = pack ? SPL_T / length : 1;
    const auto kernel = one ? (pack ? k_spline<1, true> : k_spline<1, false>)
                            : (pack ? k_spline<SPL_NR, true> : k_spline<SPL_NR, false>);
    return launch_rows((long)((nsub - 1) / G + 1) * groups, nb, SPL_T, [&](long e0, dim3 grid) {
        hipLaunchKernelGGL(kernel, grid, dim3(SPL_T), 0,
                           reinterpret_cast<hipStream_t>(stream), freqs, propArrays, B, upper_diag, diag, lower_diag,
                           length, nsub, numInterpParams, nb, G, (int)e0);
    });
}
