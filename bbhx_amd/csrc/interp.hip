// Dense-grid template build from the sparse spline coefficients
// (the reference's InterpTDI / TDI kernel, WaveformBuild.cu:41-189).
//
// The reference launches one kernel per binary on its own stream. Here all
// binaries go in ONE launch: each binary's band [start, start + n_b) is cut
// into tiles of TILE dense bins; block -> (binary, tile) by a binary search
// over the per-binary tile offsets (ragged CSR). One lane per dense bin sums
// the modes:
//   h_ch(f) = sum_m conj(T_ch,m(f) A_m(f) e^{i phi_m(f)})  if t_start <= t_m(f) <= t_end
// with every quantity a cubic in (f - f_k) on the segment k = inds[m][i].
// A first pass repacks the 36 spline coefficients and the knot of each
// (binary, mode, segment), spread over nine arrays each in the reference's
// layout, into one 320-B record (library workspace): the lanes of a wavefront
// mostly share a segment, and one base address lets the wavefront read it with
// a few wide scalar loads instead of 37 separately addressed ones.

#include <vector>

#include "bbhx_hip.h"
#include "common.h"
#include "interp_device.h"
#include "workspace.h"

using namespace bbhx;

namespace {

// Segment records are built for a chunk of binaries at a time, at most this
// many bytes (at least one binary), so that the workspace stays bounded for
// batches whose spline arrays already fill much of the device.
constexpr size_t INTERP_REC_CAP = size_t(256) << 20;

// Repack the spline arrays of segments [s0, s0 + ns) into one InterpSeg each
// (R[s - s0]): lane t -> (part p, segment s) with s fastest, so the reads of
// each spline array are unit-stride; part 9 is the knot.
__global__ __launch_bounds__(256) void k_interp_pack(InterpSeg* __restrict__ R, const double* __restrict__ freqs,
                                                     const double* __restrict__ y, const double* __restrict__ c1,
                                                     const double* __restrict__ c2, const double* __restrict__ c3,
                                                     long nper, long s0, long ns)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= 10 * ns) return;
    const int p = (int)(t / ns);
    const long s = t - p * ns;
    if (p == 9) {
        R[s].x = freqs[s0 + s];
        return;
    }
    const long q = p * nper + s0 + s;
    R[s].c[p][0] = y[q];
    R[s].c[p][1] = c1[q];
    R[s].c[p][2] = c2[q];
    R[s].c[p][3] = c3[q];
}

// Tiles [tile0, tile0 + gridDim.x) of binaries [b0, b0 + nb), whose segment
// records start at R.
__global__ __launch_bounds__(INTERP_TILE) void k_interp_tdi(const InterpBin* __restrict__ bins, int b0, int nb,
                                                            int tile0, const double* __restrict__ dataFreqs,
                                                            const InterpSeg* __restrict__ R, int length,
                                                            int numModes)
{
    // e^{i phi} table in LDS: its lookups are per-lane gathers
    __shared__ double2 s_tab[129];
    fill_etab(s_tab, (int)threadIdx.x, INTERP_TILE);
    __syncthreads();
    const int tile = tile0 + (int)blockIdx.x;
    const int bl = find_bin(bins + b0, nb, tile);
    const InterpBin& d = bins[b0 + bl];
    const int i = (tile - d.tile_begin) * INTERP_TILE + threadIdx.x;
    if (i >= d.len) return;
    const double f = dataFreqs[d.start + i];
    cd h[3];
    interp_point(h, f, i, d, bl, R, length, numModes, s_tab);
    cd* out = reinterpret_cast<cd*>(d.tmpl);
    out[0 * (long)d.len + i] = h[0];
    out[1 * (long)d.len + i] = h[1];
    out[2 * (long)d.len + i] = h[2];
}

// number of entries of the sorted a[0, n) that are <= v (n if v is not a number)
__device__ inline int upper_bound(const double* __restrict__ a, int n, double v)
{
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (a[mid] > v) hi = mid;
        else lo = mid + 1;
    }
    return lo;
}

// the same by a wavefront: 64 entries a round
__device__ inline int wave_upper_bound(const double* __restrict__ a, int n, double v)
{
    const int lane = threadIdx.x & 63;
    int lo = 0;
    while (n > 0) {
        const int step = (n + 63) >> 6;
        const long p = (long)lane * step;
        const int c = __popcll(__ballot(p < n && !(a[lo + (p < n ? p : 0)] > v)));
        if (c == 0) break;
        lo += (c - 1) * step + 1;
        n = min(step, n - (c - 1) * step) - 1;
    }
    return lo;
}

// band[b] = [start, end) of the data grid that binary b's sparse grids cover: one
// workgroup per binary, least and greatest of its n sparse frequencies
__global__ __launch_bounds__(256) void k_interp_bands(int2* __restrict__ band, const double* __restrict__ freqs, long n,
                                                      const double* __restrict__ dataFreqs, int N)
{
    __shared__ double s_lo[4], s_hi[4];
    const double* x = freqs + (long)blockIdx.x * n;
    double lo = x[0], hi = x[0];
    auto least = [](double a, double b) { return (b < a || b != b) && a == a ? b : a; };  // not a number if any is
    auto most = [](double a, double b) { return (b > a || b != b) && a == a ? b : a; };
    for (long i = threadIdx.x; i < n; i += 256) {
        lo = least(lo, x[i]);
        hi = most(hi, x[i]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        lo = least(lo, __shfl_xor(lo, o, 64));
        hi = most(hi, __shfl_xor(hi, o, 64));
    }
    if ((threadIdx.x & 63) == 0) {
        s_lo[threadIdx.x >> 6] = lo;
        s_hi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x >= 128) return;
    lo = s_lo[0];
    hi = s_hi[0];
    for (int w = 1; w < 4; w++) {
        lo = least(lo, s_lo[w]);
        hi = most(hi, s_hi[w]);
    }
    // one wavefront per end
    const bool end = threadIdx.x >= 64;
    const int k = wave_upper_bound(dataFreqs, N, end ? hi : lo);
    if ((threadIdx.x & 63) == 0) (end ? band[blockIdx.x].y : band[blockIdx.x].x) = k;
}

// off[b]: bins of the bands before b's (one workgroup)
__global__ __launch_bounds__(256) void k_interp_offsets(int64_t* __restrict__ off, const int2* __restrict__ band, int B)
{
    __shared__ int64_t part[256];
    const int t = threadIdx.x, per = (B + 255) / 256, b0 = min(B, t * per), b1 = min(B, b0 + per);
    int64_t sum = 0;
    for (int b = b0; b < b1; b++) sum += max(0, band[b].y - band[b].x);
    part[t] = sum;
    __syncthreads();
    int64_t run = 0;
    for (int w = 0; w < t; w++) run += part[w];
    for (int b = b0; b < b1; b++) {
        off[b] = run;
        run += max(0, band[b].y - band[b].x);
    }
}

// Spline segment of every (binary, mode, dense bin): block -> (binary, mode) from bm0 on,
// tile of SEG_TILE bins. The grids are log-spaced, so the segment is estimated from an FP32
// logarithm and checked, its neighbours next; whatever they do not hold is searched.
// Bound by instruction issue, the estimate and its checks, and the writes. Up to 38 M
// (binary, mode, bin): 0.062 ms (0.112 with a lane's bins one after another, 0.23 by a
// binary search per bin); torch's searchsorted and its conversions, binary by binary:
// 0.49 ms and seven launches for each.
constexpr int SEG_TILE = 1024;
__global__ __launch_bounds__(256) void k_interp_segments(int* __restrict__ inds, const int2* __restrict__ band,
                                                         const int64_t* __restrict__ off,
                                                         const double* __restrict__ dataFreqs,
                                                         const double* __restrict__ freqs, int M, int L, int tiles,
                                                         int bm0)
{
    const int tile = blockIdx.x % tiles, bm = bm0 + blockIdx.x / tiles, b = bm / M, m = bm - b * M;
    const int2 r = band[b];
    const int len = r.y - r.x;
    const double* x = freqs + (long)bm * L;
    int* o = inds + off[b] * M + (long)m * len;
    const int i0 = tile * SEG_TILE, n = min(len - i0, SEG_TILE);
    if (L < 2) {
        for (int i = threadIdx.x; i < n; i += 256) o[i0 + i] = upper_bound(x, L, dataFreqs[r.x + i0 + i]) - 1;
        return;
    }
    if (n <= 0) return;
    const double x0 = x[0], x1 = x[L - 1];
    const float g0 = __log2f((float)x0), gs = (float)(L - 1) / (__log2f((float)x1) - g0);
    // the estimates' bounds of all of the lane's bins first, so that their loads overlap
    constexpr int U = SEG_TILE / 256;
    double f[U], xa[U], xb[U];
    int k[U];
#pragma unroll
    for (int u = 0; u < U; u++) f[u] = dataFreqs[r.x + i0 + min((int)threadIdx.x + 256 * u, n - 1)];
#pragma unroll
    for (int u = 0; u < U; u++) {
        k[u] = (int)fminf(fmaxf((__log2f((float)f[u]) - g0) * gs, 0.0f), (float)(L - 2));
        xa[u] = x[k[u]];
        xb[u] = x[k[u] + 1];
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int i = threadIdx.x + 256 * u;
        if (i >= n) return;
        int j = k[u];
        if (!(xa[u] <= f[u] && f[u] < xb[u])) {
            if (f[u] >= x1) j = L - 1;
            else if (f[u] < x0) j = -1;
            else {
                j = f[u] < xa[u] ? max(j - 1, 0) : min(j + 1, L - 2);
                if (!(x[j] <= f[u] && f[u] < x[j + 1])) j = upper_bound(x, L, f[u]) - 1;
            }
        }
        o[i0 + i] = j;
    }
}

// out[b][ch][k]: the template on b's band, zero elsewhere; block -> (binary, tile), one
// pass over the output (bound by its writes; a fill, then a copy per binary, writes the
// bands twice)
__global__ __launch_bounds__(256) void k_fill_bands(double2* __restrict__ out, const double2* __restrict__ tmpl,
                                                    const int2* __restrict__ band, const int64_t* __restrict__ off,
                                                    int N, int tiles)
{
    const int tile = blockIdx.x % tiles, b = blockIdx.x / tiles;
    if ((unsigned)tile * 256 + threadIdx.x >= (unsigned)N) return;
    const int k = tile * 256 + threadIdx.x;
    const int2 r = band[b];
    const int len = r.y - r.x;
    const bool in = k >= r.x && k < r.y;
    const double2* t = tmpl + off[b] * 3 + (k - r.x);
    double2* o = out + (long)b * 3 * N + k;
#pragma unroll
    for (int ch = 0; ch < 3; ch++) o[(long)ch * N] = in ? t[(long)ch * len] : make_double2(0.0, 0.0);
}

}  // namespace

extern "C" int bbhx_hip_interp_bands(int* band, int64_t* off, const double* freqs, const double* dataFreqs, int length,
                                     int data_length, int numBinAll, int numModes, void* stream)
{
    if (length < 1 || data_length < 0 || numBinAll < 0 || numModes < 1) return ERR_ARGS;
    if (numBinAll == 0) return OK;
    if (!band || !off || !freqs || (!dataFreqs && data_length > 0)) return ERR_ARGS;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int2* r = reinterpret_cast<int2*>(band);
    const long n = (long)numModes * length;
    const int rc = launch_rows(numBinAll, 1, 256, [&](long b0, dim3 grid) {
        hipLaunchKernelGGL(k_interp_bands, grid, dim3(256), 0, st, r + b0, freqs + b0 * n, n, dataFreqs, data_length);
    });
    if (rc != OK) return rc;
    hipLaunchKernelGGL(k_interp_offsets, dim3(1), dim3(256), 0, st, off, r, numBinAll);
    return hipGetLastError() == hipSuccess ? OK : ERR_LAUNCH;
}

extern "C" int bbhx_hip_interp_segments(int* inds, const int* band, const int64_t* off, const double* freqs,
                                        const double* dataFreqs, int length, int max_len, int numBinAll, int numModes,
                                        void* stream)
{
    if (length < 1 || max_len < 0 || numBinAll < 0 || numModes < 1) return ERR_ARGS;
    if (numBinAll == 0 || max_len == 0) return OK;
    if (!inds || !band || !off || !freqs || !dataFreqs) return ERR_ARGS;
    const int tiles = (int)(((long)max_len + SEG_TILE - 1) / SEG_TILE);
    const long rows = (long)numBinAll * numModes;
    if (rows > 2147483647L) return ERR_ARGS;
    return launch_rows(rows, tiles, 256, [&](long bm0, dim3 grid) {
        hipLaunchKernelGGL(k_interp_segments, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), inds,
                           reinterpret_cast<const int2*>(band), off, dataFreqs, freqs, numModes, length, tiles,
                           (int)bm0);
    });
}

extern "C" int bbhx_hip_fill_bands(double* out, const double* templates, const int* band, const int64_t* off,
                                   int data_length, int numBinAll, void* stream)
{
    if (data_length < 0 || numBinAll < 0) return ERR_ARGS;
    if (numBinAll == 0 || data_length == 0) return OK;
    if (!out || !templates || !band || !off) return ERR_ARGS;
    const int tiles = (int)(((long)data_length + 255) / 256);
    return launch_rows(numBinAll, tiles, 256, [&](long b0, dim3 grid) {
        hipLaunchKernelGGL(k_fill_bands, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                           reinterpret_cast<double2*>(out) + b0 * 3 * data_length,
                           reinterpret_cast<const double2*>(templates), reinterpret_cast<const int2*>(band) + b0,
                           off + b0, data_length, tiles);
    });
}

namespace bbhx {
// Uploads a host table of per-binary descriptors to the table workspace.
// Synchronises the stream so the host vector may be released on return.
InterpBin* upload_table(const std::vector<InterpBin>& h, hipStream_t stream)
{
    InterpBin* d = static_cast<InterpBin*>(workspace_get(WS_TABLE, sizeof(InterpBin) * (h.size() + 1), stream));
    if (!d) return nullptr;
    if (hipMemcpyAsync(d, h.data(), sizeof(InterpBin) * h.size(), hipMemcpyHostToDevice, stream) != hipSuccess)
        return nullptr;
    if (hipStreamSynchronize(stream) != hipSuccess) return nullptr;
    return d;
}

// Host table for ragged bands cut in tiles of 'tile' dense bins; returns the
// number of tiles, or -1 when a band is invalid.
long build_table(std::vector<InterpBin>& h, const int64_t* tmpl_ptrs, const int64_t* inds_ptrs,
                 const int* inds_start, const int* ind_lengths, const double* t_start, const double* t_end,
                 int numBinAll, int tile)
{
    h.resize(numBinAll);
    long tiles = 0;
    for (int b = 0; b < numBinAll; b++) {
        if (ind_lengths[b] < 0 || inds_start[b] < 0) return -1;
        h[b].tmpl = reinterpret_cast<double*>(tmpl_ptrs ? tmpl_ptrs[b] : 0);
        h[b].inds = reinterpret_cast<const int*>(inds_ptrs ? inds_ptrs[b] : 0);
        h[b].start = inds_start[b];
        h[b].len = ind_lengths[b];
        h[b].t_start = t_start ? t_start[b] : 0.0;
        h[b].t_end = t_end ? t_end[b] : 0.0;
        h[b].tile_begin = (int)tiles;
        h[b].pad = 0;
        tiles += (ind_lengths[b] + tile - 1) / tile;
        if (tiles > 2147483647L) return -1;
    }
    return tiles;
}
}  // namespace bbhx

extern "C" int bbhx_hip_InterpTDI(const int64_t* templateChannels_ptrs, const double* dataFreqs, const double* freqs,
                                  const double* propArrays, const double* c1, const double* c2, const double* c3,
                                  const double* t_start, const double* t_end, int length, int data_length,
                                  int numBinAll, int numModes, const int64_t* inds_ptrs, const int* inds_start,
                                  const int* ind_lengths, void* stream)
{
    if (length < 2 || data_length < 0 || numBinAll < 0 || numModes < 1 || numModes > MAX_MODES) return ERR_ARGS;
    if (numBinAll == 0) return OK;
    if (!templateChannels_ptrs || !dataFreqs || !freqs || !propArrays || !c1 || !c2 || !c3 || !t_start || !t_end ||
        !inds_ptrs || !inds_start || !ind_lengths)
        return ERR_ARGS;
    for (int b = 0; b < numBinAll; b++)
        if ((long)inds_start[b] + ind_lengths[b] > data_length) return ERR_ARGS;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    std::vector<InterpBin> h;
    long tiles = build_table(h, templateChannels_ptrs, inds_ptrs, inds_start, ind_lengths, t_start, t_end, numBinAll,
                             INTERP_TILE);
    if (tiles < 0) return ERR_ARGS;
    if (tiles == 0) return OK;
    InterpBin* bins = upload_table(h, st);
    if (!bins) return ERR_ALLOC;
    const long nper = (long)numBinAll * numModes * length;
    const long per_bin = (long)numModes * length;  // segment records per binary
    long chunk = (long)(INTERP_REC_CAP / (sizeof(InterpSeg) * (size_t)per_bin));
    chunk = chunk < 1 ? 1 : (chunk > numBinAll ? numBinAll : chunk);
    InterpSeg* R = static_cast<InterpSeg*>(workspace_get(WS_INTERP, sizeof(InterpSeg) * (size_t)(per_bin * chunk), st));
    if (!R) return ERR_ALLOC;
    for (long b0 = 0; b0 < numBinAll; b0 += chunk) {
        const long b1 = b0 + chunk < numBinAll ? b0 + chunk : numBinAll;
        const int t0 = h[b0].tile_begin;
        const int t1 = b1 < numBinAll ? h[b1].tile_begin : (int)tiles;
        if (t1 == t0) continue;  // empty bands only
        const long ns = (b1 - b0) * per_bin;
        hipLaunchKernelGGL(k_interp_pack, dim3((unsigned)ceil_div(10 * ns, 256)), dim3(256), 0, st, R, freqs,
                           propArrays, c1, c2, c3, nper, b0 * per_bin, ns);
        hipLaunchKernelGGL(k_interp_tdi, dim3((unsigned)(t1 - t0)), dim3(INTERP_TILE), 0, st, bins, (int)b0,
                           (int)(b1 - b0), t0, dataFreqs, R, length, numModes);
        if (hipGetLastError() != hipSuccess) return ERR_LAUNCH;
    }
    return OK;
}
