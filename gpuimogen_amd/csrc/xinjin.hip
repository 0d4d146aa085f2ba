// xinjin.hip -- Xin-Jin relaxing TVD sweeps (second order) for gfx950.
//
// One directional sweep is four steps, in the reference's order
// (gpuclass/cudaFluidStep.cu:357-475):
//   freeze(Q) -> predict U = floor(Q - lambda/4 dF(Q))
//   freeze(U) -> correct Q = floor(Q - lambda/2 dF_tvd(U))
// The freezing speed of a line is max |p_x|/rho + sqrt(gamma P/rho) over that
// line (cukern_PressureFreezeSolverHydro, :2868-2941); the stage arithmetic,
// including the Ospre flux limiter of the corrector and the density/energy
// floors, follows cukern_XinJinHydro_step (:2427-2654) for cartesian geometry.
// The data movement is this library's: lines that a block can hold take all
// four steps in one launch, in registers (xj_lines). Longer ones take four
// launches with U in memory: X lines by waves whose lanes hold consecutive
// cells (neighbours by cross-lane shuffle, 60 outputs per 64 lanes), Y/Z lines
// by lanes marching along their column with a register window. The corrector
// reads U and writes Q, and each lane reads Q only at the cell it writes, so it
// runs in place without hazards.
#include "sweep_device.h"
#include "imogen_internal.h"

namespace imogen {

struct XjConsts {
    double gamma, gm1, rhomin, emin;
};

// Ospre flux limiter, gpuclass/limiter_functions.h:36-42
__device__ __forceinline__ double xj_ospre(double a, double b)
{
    // a^2 + ab + b^2 below the normal range (|a|, |b| < 1.5e-154, numerator
    // already +-0) is raised to the smallest normal: its hardware reciprocal
    // would be infinite and the quotient NaN instead of +-0
    const double r = a * b;
    const double v = div_nr(1.5 * r * (a + b), fmax(a * a + r + b * b, 0x1p-1022));
    return (r <= 0.0) ? 0.0 : v;
}

// Left- and right-going fluxes (C_f q - w, C_f q + w) of one cell for every
// slab; NS is the slab of the normal momentum (2, 3, 4).
template <int NS>
__device__ __forceinline__ void xj_cell(const XjConsts &k, double cf, const double (&q)[5], double (&wl)[5],
                                        double (&wr)[5])
{
    const double ir = rcp_nr(q[0]);
    const double P = k.gm1 * (q[1] - .5 * (q[4] * q[4] + q[3] * q[3] + q[2] * q[2]) * ir);
    const double vx = q[NS] * ir;
#pragma unroll
    for (int v = 0; v < 5; v++) {
        double w;
        if (v == 0) w = q[NS];
        else if (v == 1) w = vx * (q[1] + P);
        else if (v == NS) w = vx * q[v] + P;
        else w = vx * q[v];
        wl[v] = cf * q[v] - w;
        wr[v] = cf * q[v] + w;
    }
}

// density and internal-energy floors of a new state (:2620-2628)
__device__ __forceinline__ void xj_floor(const XjConsts &k, double (&p)[5])
{
    p[0] = (p[0] < k.rhomin) ? k.rhomin : p[0];
    const double w = .5 * (p[2] * p[2] + p[3] * p[3] + p[4] * p[4]) * rcp_nr(p[0]);
    if ((p[1] - w) < p[0] * k.emin) p[1] = w + p[0] * k.emin;
}

__device__ __forceinline__ double xj_wave_max(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(v, off, 64);
        v = (o > v) ? o : v;
    }
    return v;
}

// freezing speed contribution of one cell (:2887-2896)
__device__ __forceinline__ double xj_cf_cell(const XjConsts &k, const double *__restrict__ c, int64_t pitch)
{
    const double invrho = rcp_nr(c[0]);
    double psq = c[3 * pitch];
    double px = c[4 * pitch];
    psq = psq * psq + px * px;
    px = c[2 * pitch];
    psq += px * px;
    const double P = (c[pitch] - .5 * psq * invrho) * k.gm1;
    return fabs(px) * invrho + sqrt_nr(k.gamma * P * invrho);
}

// X lines: one wave per line, lanes strided along x
__global__ __launch_bounds__(256) void xj_freeze_x(const double *__restrict__ q, int64_t pitch, int N,
                                                   int64_t nlines, XjConsts k, double *__restrict__ cf)
{
    const int64_t line = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (line >= nlines) return;
    const int lane = threadIdx.x & 63;
    const double *row = q + line * (int64_t)N;
    double cmax = 0.0;
    for (int x = lane; x < N; x += 64) {
        const double loc = xj_cf_cell(k, row + x, pitch);
        cmax = (loc > cmax) ? loc : cmax;
    }
    cmax = xj_wave_max(cmax);
    if (lane == 0) cf[line] = cmax;
}

// Y/Z lines: a block takes 64 columns, its 16 waves a sixteenth of the line
// each. (With one lane per column most of the chip was idle: the Y sweep of a
// 1024 x 1024 plane took 1315 us in the staged form, 655 with the split.)
__global__ __launch_bounds__(1024) void xj_freeze_march(const double *__restrict__ q, int64_t pitch, int nx,
                                                        int64_t sstride, int64_t ostride, int N, XjConsts k,
                                                        double *__restrict__ cf)
{
    __shared__ double part[16][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t x = (int64_t)blockIdx.x * 64 + lane;
    const int64_t xc = x < nx ? x : nx - 1;
    const double *col = q + xc + (int64_t)blockIdx.y * ostride;
    const int j1 = (int)((int64_t)N * (w + 1) / 16);
    double cmax = 0.0;
    for (int j = (int)((int64_t)N * w / 16); j < j1; j++) {
        const double loc = xj_cf_cell(k, col + (int64_t)j * sstride, pitch);
        cmax = (loc > cmax) ? loc : cmax;
    }
    part[w][lane] = cmax;
    __syncthreads();
    if (w == 0 && x < nx) {
        for (int i = 1; i < 16; i++) cmax = (part[i][lane] > cmax) ? part[i][lane] : cmax;
        cf[x + (int64_t)nx * blockIdx.y] = cmax;
    }
}

// ---------------------------------------------------------------------------
// whole lines
// ---------------------------------------------------------------------------
// A sweep of lines that fit a block: C lines of N cells, T threads a line, K
// consecutive cells (periodic) a thread, so the freezing speed, the predictor,
// the freezing speed of its result and the corrector run in one launch and the
// state is read and written once (and read once more by the corrector, from
// the caches: holding it costs a wave per SIMD and was no faster). Adjacent X
// lines lie behind one another, and a line's threads are neighbours; adjacent
// Y/Z columns lie side by side, and threads of one cell row are neighbours.
// Two fluxes per cell and variable pass through LDS, in two buffers, so one
// barrier per variable separates writes from reads. 110-126 VGPRs: four waves
// per SIMD. Bound by FP64 issue (about 400 instructions per cell) and memory
// in turn, which two blocks per CU only partly overlap.
// Sweeps along X, Y, Z, four launches -> one: 131 x 120 x 113 cells 96, 216,
// 209 -> 58, 67, 55 us; 64^3 31, 66, 68 -> 22 us each; 256^3 914, 1161, 1125 ->
// 425, 414, 497 us; 1024 x 1024 59, 1315 -> 37, 70 us.
__device__ __forceinline__ unsigned long long xj_line_max(unsigned long long *slot, double v, int t, int T, bool xline,
                                                          bool run)
{
    if (xline) {
        // the lanes of one line are neighbours: their maximum first
        const int lane = threadIdx.x & 63;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double o = __shfl_down(v, off, 64);
            if (lane + off < 64 && t + off < T && o > v) v = o;
        }
        run = run && (t == 0 || lane == 0);
    }
    // v >= 0: its bits order as the values do
    if (run) atomicMax(slot, (unsigned long long)__double_as_longlong(v));
    __syncthreads();
    return *slot;
}

// the freezing speed's cell maximum over a thread's cells
template <int K>
__device__ __forceinline__ double xj_cells_max(const XjConsts &k, const double (&q)[5][K])
{
    double cmax = 0.0;
#pragma unroll
    for (int i = 0; i < K; i++) {
        const double c[5] = {q[0][i], q[1][i], q[2][i], q[3][i], q[4][i]};
        const double loc = xj_cf_cell(k, c, 1);
        cmax = (loc > cmax) ? loc : cmax;
    }
    return cmax;
}

template <int NS, int K, int BLOCK>
__global__ __launch_bounds__(BLOCK) void xj_lines(double *__restrict__ state, int64_t pitch, int N, int T, int C,
                                                  unsigned nlines, unsigned nx, unsigned sstride, unsigned ostride,
                                                  double lambda, const double *__restrict__ lamp, XjConsts k)
{
    __shared__ double2 w[2][BLOCK * K];  // (wl, wr) of C N cells
    __shared__ unsigned long long speed[2][BLOCK];
    if (lamp) lambda = lamp[0];  // time step kept on the device
    constexpr bool xline = NS == 2;
    const int tid = threadIdx.x;
    const bool run = tid < C * T;
    const int id = run ? tid : 0;
    const int t = xline ? id % T : id / C;
    const int c = xline ? id / T : id - t * C;
    unsigned line = blockIdx.x * C + c;
    const bool live = run && line < nlines;
    line = line < nlines ? line : nlines - 1;
    const unsigned q0 = xline ? line * N : line % nx + line / nx * ostride;
    const int j0 = t * K;
    const int n = N - j0 < K ? N - j0 : K;  // cells of this thread's own; the rest repeat the line's first
    auto wrap = [&](int j) { return j < 0 ? j + N : (j >= N ? j - N : j); };
    // X: slot j mod K of thread j / K, so that a wave's 16-byte accesses are
    // contiguous; Y/Z: rows of C cells
    auto at = [&](int j) {
        j = wrap(j);
        return xline ? (j & (K - 1)) * BLOCK + c * T + j / K : j * C + c;
    };
    // cell i, variable v; 32-bit byte offsets, so a slab ends below 4 GiB
    unsigned off[K];
#pragma unroll
    for (int i = 0; i < K; i++) off[i] = 8 * (q0 + wrap(j0 + i) * (xline ? 1 : sstride));
    auto cell = [&](int v, int i) -> double & {
        return *reinterpret_cast<double *>(reinterpret_cast<char *>(state + v * pitch) + off[i]);
    };

    if (tid < C) speed[0][tid] = speed[1][tid] = 0;
    double q[5][K];
#pragma unroll
    for (int i = 0; i < K; i++)
#pragma unroll
        for (int v = 0; v < 5; v++) q[v][i] = cell(v, i);
    __syncthreads();

#pragma unroll
    for (int stage = 0; stage < 2; stage++) {
        const double cf = __longlong_as_double(xj_line_max(&speed[stage][c], xj_cells_max<K>(k, q), t, T, xline, run));
        const double lam = (stage ? 0.5 : 0.25) * lambda;
        double vx[K], P[K];
#pragma unroll
        for (int i = 0; i < K; i++) {
            const double ir = rcp_nr(q[0][i]);
            P[i] = k.gm1 * (q[1][i] - .5 * (q[4][i] * q[4][i] + q[3][i] * q[3][i] + q[2][i] * q[2][i]) * ir);
            vx[i] = q[NS][i] * ir;
        }
#pragma unroll
        for (int v = 0; v < 5; v++) {
            // slots 2 .. K + 1 are this thread's cells
            double wl[K + 4], wr[K + 4];
#pragma unroll
            for (int i = 0; i < K; i++) {
                double f;
                if (v == 0) f = q[NS][i];
                else if (v == 1) f = vx[i] * (q[1][i] + P[i]);
                else if (v == NS) f = vx[i] * q[v][i] + P[i];
                else f = vx[i] * q[v][i];
                wl[i + 2] = cf * q[v][i] - f;
                wr[i + 2] = cf * q[v][i] + f;
            }
            double2 *buf = w[(stage * 5 + v) & 1];
#pragma unroll
            for (int i = 0; i < K; i++)
                if (run && i < n) buf[at(j0 + i)] = double2{wl[i + 2], wr[i + 2]};
            double b[K];
            if (stage) {
#pragma unroll
                for (int i = 0; i < K; i++) {
                    asm volatile("" : "+v"(off[i]));  // read again: the first reading is not kept
                    b[i] = cell(v, i);
                }
            }
            __syncthreads();
            const double2 m1 = buf[at(j0 - 1)], p1 = buf[at(j0 + K)];
            wl[1] = m1.x;
            wr[1] = m1.y;
            wl[K + 2] = p1.x;
            wr[K + 2] = p1.y;
            if (stage) {
                wr[0] = buf[at(j0 - 2)].y;
                wl[K + 3] = buf[at(j0 + K + 1)].x;
                // corrected fluxes, in place: cells 0 .. K to the left, -1 .. K - 1 to the right
                double dl = .5 * (wl[2] - wl[1]), dr = .5 * (wr[1] - wr[0]);
#pragma unroll
                for (int i = 0; i <= K; i++) {
                    const double dln = .5 * (wl[i + 3] - wl[i + 2]);
                    const double drn = .5 * (wr[i + 2] - wr[i + 1]);
                    wl[i + 2] -= xj_ospre(dl, dln);
                    wr[i + 1] += xj_ospre(dr, drn);
                    dl = dln;
                    dr = drn;
                }
            }
#pragma unroll
            for (int i = 0; i < K; i++) {
                q[v][i] = (stage ? b[i] : q[v][i]) - lam * (wr[i + 2] - wr[i + 1] - wl[i + 3] + wl[i + 2]);
                asm volatile("" : "+v"(q[v][i]));  // done here: put off, the fluxes of all five would be held
            }
        }
#pragma unroll
        for (int i = 0; i < K; i++) {
            double p[5] = {q[0][i], q[1][i], q[2][i], q[3][i], q[4][i]};
            xj_floor(k, p);
            q[0][i] = p[0];
            q[1][i] = p[1];
        }
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < K; i++) {
            if (i < n) {
#pragma unroll
                for (int v = 0; v < 5; v++) cell(v, i) = q[v][i];
            }
        }
    }
}

// One stage along X. Lane l of a wave holds cell x0 - 2 + l (periodic); lanes
// 2..61 produce outputs. src: state the fluxes are taken of (Q or U); base:
// state the update starts from; dst: where the new state goes.
template <bool CORRECT>
__global__ __launch_bounds__(256) void xj_stage_x(const double *__restrict__ src, const double *base,
                                                  double *dst, int64_t pitch, int N, int64_t nlines, int nseg,
                                                  double lambda, const double *__restrict__ lamp, double lscale,
                                                  XjConsts k, const double *__restrict__ cf)
{
    if (lamp) lambda = lscale * lamp[0];  // time step kept on the device
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (wave >= nlines * nseg) return;
    const int lane = threadIdx.x & 63;
    const int64_t line = wave / nseg;
    const int seg = (int)(wave - line * nseg);
    const int xr = seg * 60 - 2 + lane;  // >= -2
    int x = xr % N;
    if (x < 0) x += N;
    const int64_t off = line * (int64_t)N + x;
    const double cfl = cf[line];
    double q[5];
#pragma unroll
    for (int v = 0; v < 5; v++) q[v] = src[off + v * pitch];
    double wl[5], wr[5];
    xj_cell<2>(k, cfl, q, wl, wr);
    const bool delivers = lane >= 2 && lane <= 61 && xr < N;
    double p[5];
#pragma unroll
    for (int v = 0; v < 5; v++) {
        double WL = wl[v], WR = wr[v];
        if (CORRECT) {
            const double dl = .5 * (wl[v] - __shfl(wl[v], lane - 1, 64));
            const double dr = .5 * (wr[v] - __shfl(wr[v], lane - 1, 64));
            WL -= xj_ospre(dl, __shfl(dl, lane + 1, 64));
            WR += xj_ospre(dr, __shfl(dr, lane + 1, 64));
        }
        const double WRm = __shfl(WR, lane - 1, 64);
        const double WLp = __shfl(WL, lane + 1, 64);
        const double b = CORRECT ? base[off + v * pitch] : q[v];
        p[v] = b - lambda * (WR - WRm - WLp + WL);
    }
    xj_floor(k, p);
    if (delivers) {
#pragma unroll
        for (int v = 0; v < 5; v++) dst[off + v * pitch] = p[v];
    }
}

// One stage along Y (DIR 2) or Z (DIR 3): each lane marches one segment of a
// column. At load k the window gains cell m = j0 - 2 + k; the corrected
// fluxes of cell m-1 complete and cell m-2 is written (from k = 4 on).
template <int DIR, bool CORRECT>
__global__ __launch_bounds__(256) void xj_stage_march(const double *__restrict__ src, const double *base,
                                                      double *dst, int64_t pitch, int nx, int64_t sstride,
                                                      int64_t ostride, int N, int S, int seglen, double lambda,
                                                      const double *__restrict__ lamp, double lscale, XjConsts k,
                                                      const double *__restrict__ cf)
{
    if (lamp) lambda = lscale * lamp[0];  // time step kept on the device
    constexpr int NS = DIR + 1;
    const int lane = threadIdx.x & 63;
    const int W = 64 / S;
    const int s = lane / W;
    const int64_t x = (int64_t)blockIdx.x * (blockDim.x / S) + (threadIdx.x >> 6) * W + (lane - s * W);
    if (x >= nx || s >= S) return;
    const int j0 = s * seglen;
    int L = N - j0;
    L = L < seglen ? L : seglen;
    if (L <= 0) return;
    const int64_t colOff = x + (int64_t)blockIdx.y * ostride;
    const double cfl = cf[x + (int64_t)nx * blockIdx.y];
    int mw = j0 - 2;
    if (mw < 0) mw += N;
    int ow = j0;  // wrapped index of the next output cell (never wraps: j0 + L <= N)

    double wlp[5], wrp[5], dlp[5], drp[5], WLp[5], WRp[5], WRpp[5];
#pragma unroll
    for (int v = 0; v < 5; v++) wlp[v] = wrp[v] = dlp[v] = drp[v] = WLp[v] = WRp[v] = WRpp[v] = 0.0;

    for (int t = 0; t < L + 4; t++) {
        double q[5];
        const int64_t o = colOff + (int64_t)mw * sstride;
#pragma unroll
        for (int v = 0; v < 5; v++) q[v] = src[o + v * pitch];
        mw = (mw + 1 == N) ? 0 : mw + 1;
        double wl[5], wr[5];
        xj_cell<NS>(k, cfl, q, wl, wr);
        double p[5];
#pragma unroll
        for (int v = 0; v < 5; v++) {
            const double dl = .5 * (wl[v] - wlp[v]);
            const double dr = .5 * (wr[v] - wrp[v]);
            // corrected fluxes of cell m-1
            double WL = wlp[v], WR = wrp[v];
            if (CORRECT) {
                WL -= xj_ospre(dlp[v], dl);
                WR += xj_ospre(drp[v], dr);
            }
            // flux difference at cell m-2
            p[v] = WRp[v] - WRpp[v] - WL + WLp[v];
            wlp[v] = wl[v];
            wrp[v] = wr[v];
            dlp[v] = dl;
            drp[v] = dr;
            WRpp[v] = WRp[v];
            WRp[v] = WR;
            WLp[v] = WL;
        }
        if (t >= 4) {
            const int64_t oo = colOff + (int64_t)ow * sstride;
            ow++;
            double r[5];
#pragma unroll
            for (int v = 0; v < 5; v++) r[v] = base[oo + v * pitch] - lambda * p[v];
            xj_floor(k, r);
#pragma unroll
            for (int v = 0; v < 5; v++) dst[oo + v * pitch] = r[v];
        }
    }
}

static int xj_freeze(const double *q, int64_t pitch, int nx, int ny, int nz, int dir, const XjConsts &k,
                     double *cf, hipStream_t s)
{
    if (dir == 1) {
        const int64_t nlines = (int64_t)ny * nz;
        hipLaunchKernelGGL(xj_freeze_x, dim3((unsigned)((nlines + 3) / 4)), dim3(256), 0, s, q, pitch, nx, nlines,
                           k, cf);
    } else {
        const int N = (dir == 2) ? ny : nz;
        const int64_t sstride = (dir == 2) ? (int64_t)nx : (int64_t)nx * ny;
        const int64_t ostride = (dir == 2) ? (int64_t)nx * ny : (int64_t)nx;
        const int nother = (dir == 2) ? nz : ny;
        hipLaunchKernelGGL(xj_freeze_march, dim3((unsigned)((nx + 63) / 64), (unsigned)nother), dim3(1024), 0, s,
                           q, pitch, nx, sstride, ostride, N, k, cf);
    }
    return IM_LAUNCHED("xj_freeze");
}

template <bool CORRECT>
static int xj_stage(const double *src, const double *base, double *dst, int64_t pitch, int nx, int ny, int nz,
                    int dir, double lambda, const double *lamp, double lscale, const XjConsts &k, const double *cf,
                    hipStream_t s)
{
    if (dir == 1) {
        const int64_t nlines = (int64_t)ny * nz;
        const int nseg = (nx + 59) / 60;
        const int64_t waves = nlines * nseg;
        hipLaunchKernelGGL((xj_stage_x<CORRECT>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, src, base,
                           dst, pitch, nx, nlines, nseg, lambda, lamp, lscale, k, cf);
        return IM_LAUNCHED("xj_stage_x");
    }
    const int N = (dir == 2) ? ny : nz;
    const int64_t sstride = (dir == 2) ? (int64_t)nx : (int64_t)nx * ny;
    const int64_t ostride = (dir == 2) ? (int64_t)nx * ny : (int64_t)nx;
    const int nother = (dir == 2) ? nz : ny;
    const int64_t columns = (int64_t)nx * nother;
    int S = 1;
    while (S < 4 && columns * S < 2048 * 64 && N >= 32 * S) S *= 2;
    const int seglen = (N + S - 1) / S;
    const int colsPerBlock = 256 / S;
    dim3 grid((unsigned)((nx + colsPerBlock - 1) / colsPerBlock), (unsigned)nother), block(256);
    if (dir == 2)
        hipLaunchKernelGGL((xj_stage_march<2, CORRECT>), grid, block, 0, s, src, base, dst, pitch, nx, sstride,
                           ostride, N, S, seglen, lambda, lamp, lscale, k, cf);
    else
        hipLaunchKernelGGL((xj_stage_march<3, CORRECT>), grid, block, 0, s, src, base, dst, pitch, nx, sstride,
                           ostride, N, S, seglen, lambda, lamp, lscale, k, cf);
    return IM_LAUNCHED("xj_stage_march");
}

template <int K, int BLOCK>
static void xj_lines_launch(int dir, unsigned blocks, int threads, double *base, int64_t pitch, int N, int T, int C,
                            int64_t nlines, int64_t cx, int64_t sstride, int64_t ostride, double lambda,
                            const double *lamp, const XjConsts &k, hipStream_t s)
{
    auto f = dir == 1 ? xj_lines<2, K, BLOCK> : (dir == 2 ? xj_lines<3, K, BLOCK> : xj_lines<4, K, BLOCK>);
    hipLaunchKernelGGL(f, dim3(blocks), dim3((unsigned)threads), 0, s, base, pitch, N, T, C, (unsigned)nlines,
                       (unsigned)cx, (unsigned)sstride, (unsigned)ostride, lambda, lamp, k);
}

// Whole lines in one launch where a block of up to 1024 threads holds them: an
// X line of up to 4096 cells, 16 Y/Z columns (a full cache line of each row) of
// up to 256, 8 of 512 or 4 of 1024. The narrower rows fetch their cache lines
// from several blocks, and are still far ahead of four launches: Y of 1024 x
// 1024 70 against 655 us, of 400 x 300 x 300 1251 against 2200 us. false: the
// lines are longer.
static bool xj_whole_lines(double *base, int64_t pitch, int nx, int ny, int nz, int dir, double lambda,
                           const double *lamp, const XjConsts &k, hipStream_t s, int *rc)
{
    const int N = (dir == 1) ? nx : (dir == 2 ? ny : nz);
    const int64_t ncells = (int64_t)nx * ny * nz, nlines = ncells / N;
    const int64_t sstride = (dir == 1) ? 1 : (dir == 2 ? (int64_t)nx : (int64_t)nx * ny);
    // Y columns: nx side by side, then the next plane; Z columns are one run
    const int64_t cx = (dir == 3) ? (int64_t)nx * ny : nx;
    const int64_t ostride = (int64_t)nx * ny;
    const int unit = (dir == 1) ? 1 : (N <= 256 ? 16 : (N <= 512 ? 8 : 4));
    if (((int64_t)N + 3) / 4 * unit > 1024 || ncells > (1ll << 29)) return false;
    // four cells a thread; two, for a shorter chain, while four leave SIMDs without a wave
    const int K = (nlines * ((N + 3) / 4) < 1024 * 64 && (N + 1) / 2 * unit <= 512) ? 2 : 4;
    const int T = (N + K - 1) / K;
    int C = unit;
    // several short lines to a block, while there are blocks for every CU; along
    // X 256 threads, whose blocks overlap better (58 against 62 us for 131 cells)
    const int threads0 = (dir == 1) ? 256 : 512, blocks0 = (dir == 1) ? 1024 : 512;
    while ((C + unit) * T <= threads0 && nlines >= (int64_t)(C + unit) * blocks0) C += unit;
    const unsigned blocks = (unsigned)((nlines + C - 1) / C);
    const int threads = (C * T + 63) / 64 * 64;
    if (K == 2)
        xj_lines_launch<2, 512>(dir, blocks, threads, base, pitch, N, T, C, nlines, cx, sstride, ostride, lambda, lamp,
                                k, s);
    else if (threads <= 256)
        xj_lines_launch<4, 256>(dir, blocks, threads, base, pitch, N, T, C, nlines, cx, sstride, ostride, lambda, lamp,
                                k, s);
    else if (threads <= 512)
        xj_lines_launch<4, 512>(dir, blocks, threads, base, pitch, N, T, C, nlines, cx, sstride, ostride, lambda, lamp,
                                k, s);
    else
        xj_lines_launch<4, 1024>(dir, blocks, threads, base, pitch, N, T, C, nlines, cx, sstride, ostride, lambda,
                                 lamp, k, s);
    *rc = IM_LAUNCHED("xj_lines");
    return true;
}

// The staged form's block. Counted for every sweep, so the grids that the
// allocation-free step admits do not depend on their lines' lengths.
int64_t xinjin_scratch_bytes(int64_t pitch, int nx, int ny, int nz, int dir)
{
    const int N = (dir == 1) ? nx : (dir == 2 ? ny : nz);
    if (dir < 1 || dir > 3 || N < 3) return 0;
    const int64_t nlines = (dir == 1) ? (int64_t)ny * nz : (dir == 2 ? (int64_t)nx * nz : (int64_t)nx * ny);
    return (5 * pitch + nlines + 32) * (int64_t)sizeof(double);
}

int launch_xinjin_sweep(double *base, int64_t pitch, int nx, int ny, int nz, int dir, double lambda,
                        double gamma, double rhomin, hipStream_t s, const double *lamp)
{
    if (dir < 1 || dir > 3) return IM_FAIL(ERROR_INVALID_ARGS, "sweep direction %d", dir);
    const int N = (dir == 1) ? nx : (dir == 2 ? ny : nz);
    if (N < 3) return SUCCESSFUL;  // cudaFluidStep.cu:301
    if ((int64_t)nx * ny * nz > pitch) return IM_FAIL(ERROR_INVALID_ARGS, "slab pitch below the cell count");
    XjConsts k{gamma, gamma - 1.0, rhomin, 1e-5 / (gamma - 1.0)};
    const int slot = prof_begin(PROF_SWEEP_X + dir - 1, s);
    int rc = SUCCESSFUL;
    if (xj_whole_lines(base, pitch, nx, ny, nz, dir, lambda, lamp, k, s, &rc)) {
        prof_end(slot, s);
        return rc;
    }
    // temporary: 5 slabs of U at the fluid's pitch, then the per-line freezing speeds
    double *U = (double *)scratch_block((size_t)xinjin_scratch_bytes(pitch, nx, ny, nz, dir));
    if (!U) {
        prof_end(slot, s);
        return IM_FAIL(ERROR_NOMEM, "no scratch for the Xin-Jin stages");
    }
    double *cf = U + 5 * pitch;
    rc = xj_freeze(base, pitch, nx, ny, nz, dir, k, cf, s);
    if (!rc) rc = xj_stage<false>(base, base, U, pitch, nx, ny, nz, dir, 0.25 * lambda, lamp, 0.25, k, cf, s);
    if (!rc) rc = xj_freeze(U, pitch, nx, ny, nz, dir, k, cf, s);
    if (!rc) rc = xj_stage<true>(U, base, base, pitch, nx, ny, nz, dir, 0.5 * lambda, lamp, 0.5, k, cf, s);
    prof_end(slot, s);
    return rc;
}

}  // namespace imogen
