// Not-a-knot spline systems by parallel cyclic reduction in a workgroup.
//
// One knot per lane, several quantities on the same knots together, the systems
// and their transposes: with every row scaled to a unit diagonal, a step at distance d
// replaces the couplings to rows i -+ d by ones to rows i -+ 2d, so that grids of up to 66
// knots (64 rows) are solved exactly in six steps. In a longer one the system's inner
// rows are diagonally dominant by two or more (the couplings' magnitudes add up to at most
// half of the diagonal), and the couplings fall from 1/2 to at most 1/4, 1/16, 1/256,
// 2^-16, 2^-32 and 2^-64 (evenly spaced knots: 5e-37), after which each row is its
// solution. A row that a folded end row went into couples by h_end / (h_end + h), up to 1
// where the end interval is much the longer, and by at most a half after the first step.
// The transposed rows need not be dominant (8 on four knots over the default range of
// frequencies), but a step of the transposed system is the transpose of the system's own:
// its couplings are those times the ratio of the two rows' diagonals, below 10^4 on any
// grid here and 10^(4 64 / n) on a log-spaced one of n knots over 4 decades. What lies
// farther does not count either, so a grid longer than a workgroup is cut into blocks
// that overlap by SPL_W rows on each side: a solution forgets by a factor of about 0.27
// per row (0.5 at worst) what a block's end leaves out, and on a log-spaced grid over 4
// decades the end's slopes, steeper by at most r^(11/3) per row (r = the knots' ratio),
// weigh (0.28 r^(11/3))^48 < 1e-16 there.
#pragma once

#include "common.h"

namespace bbhx {

constexpr int SPL_W = 48;
constexpr int SPL_STEPS = 6;

// Rows per block = lanes of a workgroup (384 and 512 overlap less and measured the
// same at 1024 uneven templates, slower for few).
constexpr int SPL_T = 256;
constexpr int SPL_U = SPL_T - 2 * SPL_W;  // rows between the starts of two blocks
__host__ __device__ inline int spline_blocks(int n) { return n <= SPL_T ? 1 : 1 + (n - SPL_T + SPL_U - 1) / SPL_U; }

// Solves x_i + a x_{i-1} + c x_{i+1} = r_i for NR right sides over rows [t0, t1) of a
// workgroup (this lane's row t = threadIdx.x among them; rows outside are left out); sh:
// (NR + 2) SPL_T doubles of LDS, free on entry and on exit.
template <int NR>
__device__ inline void pcr_solve(double a, double c, double (&r)[NR], double* sh, int t, int t0, int t1)
{
    constexpr int T = SPL_T;
    for (int k = 0, d = 1; k < SPL_STEPS; k++, d *= 2) {
        sh[t] = a;
        sh[T + t] = c;
#pragma unroll
        for (int q = 0; q < NR; q++) sh[(2 + q) * T + t] = r[q];
        __syncthreads();
        const bool lo = t - d >= t0, hi = t + d < t1;
        const int tl = lo ? t - d : t, th = hi ? t + d : t;
        // couplings to rows outside are dropped
        const double fl = lo ? a : 0.0, fh = hi ? c : 0.0;
        const double ib = rcp_pos(1.0 - fl * sh[T + tl] - fh * sh[th]);
        a = -(fl * sh[tl]) * ib;
        c = -(fh * sh[T + th]) * ib;
#pragma unroll
        for (int q = 0; q < NR; q++) r[q] = (r[q] - fl * sh[(2 + q) * T + tl] - fh * sh[(2 + q) * T + th]) * ib;
        __syncthreads();
    }
}

}  // namespace bbhx
