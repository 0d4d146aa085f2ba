// sweep_kernels.h -- the HLLC / HLL sweep kernels (templates) shared by the
// single-array sweeps (fluid_sweep.hip) and the batched ensemble sweeps
// (ensemble.hip). See fluid_sweep.hip for the data-movement design.
#pragma once
#include "cfl_device.h"
#include "imogen_internal.h"
#include "sweep_device.h"

namespace imogen {

// ---------------------------------------------------------------------------
// cross-lane helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ double shfl_d(double v, int src)
{
    return __shfl(v, src, 64);
}

__device__ __forceinline__ V5 shfl5(const V5 &v, int src)
{
    return V5{shfl_d(v.a, src), shfl_d(v.b, src), shfl_d(v.c, src), shfl_d(v.d, src),
              shfl_d(v.e, src)};
}

// v of the lane before (after) in the wave, the first (last) lane's from the
// other end: one VALU move per word where a shuffle goes through the LDS unit
// and its address holds registers (sweep_x of 4 cells per lane 226 -> 156 by
// this alone; X at 256^3 308 -> 302 us, 1024^2 34.2 -> 32.4).
template <int CTRL>
__device__ __forceinline__ double rot_d(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
template <int CTRL>
__device__ __forceinline__ V5 rot5(const V5 &v)
{
    return V5{rot_d<CTRL>(v.a), rot_d<CTRL>(v.b), rot_d<CTRL>(v.c), rot_d<CTRL>(v.d), rot_d<CTRL>(v.e)};
}

// The neighbour lanes' values: ROT: the lines or windows fill the wave, so they
// are those of the adjacent lanes; otherwise lane src's.
template <bool ROT>
__device__ __forceinline__ V5 left5(const V5 &v, int src)
{
    return ROT ? rot5<0x13c>(v) : shfl5(v, src);  // wave_ror:1
}
template <bool ROT>
__device__ __forceinline__ V5 right5(const V5 &v, int src)
{
    return ROT ? rot5<0x134>(v) : shfl5(v, src);  // wave_rol:1
}

__device__ __forceinline__ V5 sel5(bool c, const V5 &x, const V5 &y)
{
    return c ? x : y;
}

__device__ __forceinline__ V5 axpy5(const V5 &q, double c, const V5 &d)
{
    return V5{fma(c, d.a, q.a), fma(c, d.b, q.b), fma(c, d.c, q.c), fma(c, d.d, q.d), fma(c, d.e, q.e)};
}

// The SSP-RK2 stages (cudaFluidStep.cu:1510-1516, 1555-1561): with dF = F_{i+1/2}
// - F_{i-1/2}, U1 = Q - lambda dF(Q) and Qout = (Q + U1)/2 - lambda/2 dF(U1).
// The half sum (Q + U1)/2 is Q - lambda/2 dF(Q) where the method has no floors
// that change U1.
template <class M>
__device__ __forceinline__ V5 half_sum(const V5 &q, const V5 &u, const V5 &dF, double mhl)
{
    if (!M::floors) return axpy5(q, mhl, dF);
    return V5{.5 * (q.a + u.a), .5 * (q.b + u.b), .5 * (q.c + u.c), .5 * (q.d + u.d), .5 * (q.e + u.e)};
}

// NT: loads and stores with the nontemporal hint. The single-grid Y/Z
// marches over rows of a multiple of 16 cells read and write whole 128-byte
// cache lines once per sweep and use it (Sedov 256^3 device loop 1 % faster,
// measured). The X sweep's lanes hold K consecutive cells, so one of its
// store instructions covers each cache line only in part: nontemporal stores
// there doubled its time. Rows that start at other 8-byte offsets (the
// ensemble's) are 10 % faster without the hint.
template <class Meth, int DIR, bool NT = false>
__device__ __forceinline__ V5 load_cell(const double *__restrict__ p, int64_t pitch)
{
    using M = MomSlabs<Meth, DIR>;
    if (NT)
        return V5{__builtin_nontemporal_load(p), __builtin_nontemporal_load(p + pitch),
                  __builtin_nontemporal_load(p + M::n * pitch), __builtin_nontemporal_load(p + M::t1 * pitch),
                  __builtin_nontemporal_load(p + M::t2 * pitch)};
    return V5{p[0], p[pitch], p[M::n * pitch], p[M::t1 * pitch], p[M::t2 * pitch]};
}

template <class Meth, int DIR, bool NT = false>
__device__ __forceinline__ void store_cell(double *__restrict__ p, int64_t pitch, const V5 &v)
{
    using M = MomSlabs<Meth, DIR>;
    if (NT) {
        __builtin_nontemporal_store(v.a, p);
        __builtin_nontemporal_store(v.b, p + pitch);
        __builtin_nontemporal_store(v.c, p + M::n * pitch);
        __builtin_nontemporal_store(v.d, p + M::t1 * pitch);
        __builtin_nontemporal_store(v.e, p + M::t2 * pitch);
        return;
    }
    p[0] = v.a;
    p[pitch] = v.b;
    p[M::n * pitch] = v.c;
    p[M::t1 * pitch] = v.d;
    p[M::t2 * pitch] = v.e;
}

// time-step limit of a stored cell (physical x, y, z momentum order, as the
// CFL kernel reads the slabs)
template <class Meth, int DIR>
__device__ __forceinline__ double cfl_of_cell(const CflArgs &a, const V5 &o)
{
    using M = MomSlabs<Meth, DIR>;
    const double px = (M::n == 2) ? o.c : ((M::t1 == 2) ? o.d : o.e);
    const double py = (M::n == 3) ? o.c : ((M::t1 == 3) ? o.d : o.e);
    const double pz = (M::n == 4) ? o.c : ((M::t1 == 4) ? o.d : o.e);
    return cfl_cell(a, o.a, o.b, px, py, pz, 0.0);
}

// ---------------------------------------------------------------------------
// ghost cells of the swept direction, set as the sweep stores them
// ---------------------------------------------------------------------------
// Const and mirror faces of depth kGhost with the memory-x conventions
// (cudaStatics.cu:1308-1366), which the fluid step applies along the direction
// it has just swept: a copy of cell kGhost (N - 1 - kGhost), or the mirror image
// about it with the normal momentum turned. As launches of their own the two
// faces cost 4.5 us at 64^3 (a quarter of an iteration), and 30 us along X at
// 256^3, where they rewrite parts of every row's cache lines.
// The cell whose value cell g takes; turned: with the normal momentum turned.
__device__ __forceinline__ int ghost_source(int g, int N, const GhostFill &gf, bool &turned)
{
    const int lo = kGhost, hi = N - 1 - kGhost;
    turned = false;
    if (gf.lo && g < lo) {
        turned = gf.lo == kFillMirror;
        return turned ? 2 * lo - g : lo;
    }
    if (gf.hi && g > hi) {
        turned = gf.hi == kFillMirror;
        return turned ? 2 * hi - g : hi;
    }
    return g;
}

// Q[i] of a uniform i
template <int K>
__device__ __forceinline__ V5 pick5(const V5 (&Q)[K], int i)
{
    V5 v = Q[0];
#pragma unroll
    for (int k = 1; k < K; k++) v = sel5(k == i, Q[k], v);
    return v;
}

// The ghosts among a lane's K cells from the lanes that hold their sources. Slot
// k is cell w0 + k of its line's (or window's) numbering, whose cell 0 is lane
// lbase's first; wlo, whi: the innermost cells next to the two faces in that
// numbering (filled where gf says so), slotHi = whi mod K. All lanes reach it.
template <int K>
__device__ __forceinline__ void fill_ghosts(V5 (&Q)[K], int w0, int lbase, int wlo, int whi, int slotHi,
                                            const GhostFill &gf)
{
    if (!(gf.lo | gf.hi)) return;
    if (K == 1) {
        int w = w0;
        bool turned = false;
        if (gf.lo && w0 < wlo) {
            turned = gf.lo == kFillMirror;
            w = turned ? 2 * wlo - w0 : wlo;
        } else if (gf.hi && w0 > whi) {
            turned = gf.hi == kFillMirror;
            w = turned ? 2 * whi - w0 : whi;
        }
        V5 v = shfl5(Q[0], lbase + w);
        v.c = turned ? -v.c : v.c;
        Q[0] = v;
        return;
    }
    if (gf.lo != kFillMirror && gf.hi != kFillMirror) {
        // one exchange for both faces: each lane's source is its nearer face's
        const bool upper = 2 * w0 > wlo + whi;
        const bool src = w0 <= whi && w0 + K > whi;  // holds the upper face's source
        const V5 v = shfl5(sel5(src, pick5<K>(Q, slotHi), pick5<K>(Q, wlo % K)), lbase + (upper ? whi : wlo) / K);
        const bool fill = upper ? gf.hi : gf.lo;
#pragma unroll
        for (int k = 0; k < K; k++) Q[k] = sel5(fill && (upper ? w0 + k > whi : w0 + k < wlo), v, Q[k]);
        return;
    }
#pragma unroll
    for (int side = 0; side < 2; side++) {
        const int fill = side ? gf.hi : gf.lo, we = side ? whi : wlo, out = side ? 1 : -1;
        if (!fill) continue;
#pragma unroll
        for (int i = 1; i <= kGhost; i++) {
            const int ws = fill == kFillMirror ? we - out * i : we;
            V5 v = shfl5(pick5<K>(Q, ws % K), lbase + ws / K);
            v.c = fill == kFillMirror ? -v.c : v.c;
#pragma unroll
            for (int k = 0; k < K; k++) Q[k] = sel5(w0 + k == we + out * i, v, Q[k]);
        }
    }
}

// ---------------------------------------------------------------------------
// X sweep: lanes own K consecutive cells of a line
// ---------------------------------------------------------------------------

// Interface fluxes of the cells a lane owns. F[k] is the flux at k+1/2 for
// k < cnt; Fm is the flux at -1/2 (the left lane's last interface). The
// method's floors are applied to U in place first.
template <class M, int K, int LIM, int DIR, bool ROT>
__device__ __forceinline__ void x_fluxes(const HydroConsts &hc, int rt, V5 (&U)[K], int cnt, int srcL,
                                         int srcR, V5 (&F)[K], V5 &Fm)
{
    V5 w[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        const double e = M::template floor<DIR>(hc, U[k]);
        w[k] = M::template prims<LIM>(hc, U[k], e);
    }

    V5 wlast = w[0];
#pragma unroll
    for (int k = 1; k < K; k++) wlast = sel5(k == cnt - 1, w[k], wlast);
    const V5 wl = left5<ROT>(wlast, srcL);
    const V5 wr = right5<ROT>(w[0], srcR);

    // backward differences d[k] = w[k] - w[k-1]; d[cnt] uses the right neighbour
    V5 d[K + 1];
    d[0] = w[0] - wl;
#pragma unroll
    for (int k = 1; k < K; k++) d[k] = sel5(k < cnt, w[k], wr) - w[k - 1];
    d[K] = wr - w[K - 1];

    V5 Lf[K], Rf[K];
#pragma unroll
    for (int k = 0; k < K; k++) M::template face<LIM>(hc, w[k], d[k], d[k + 1], rt, Lf[k], Rf[k]);

    const V5 LfR = right5<ROT>(Lf[0], srcR);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const V5 right = (k + 1 < K) ? sel5(k + 1 < cnt, Lf[(k + 1 < K) ? k + 1 : 0], LfR) : LfR;
        F[k] = M::flux(hc, Rf[k], right);
        // keep the cells' fluxes apart: interleaved they spill at 4 cells per lane
        if (K >= 4) __builtin_amdgcn_sched_barrier(0);
    }
    V5 Flast = F[0];
#pragma unroll
    for (int k = 1; k < K; k++) Flast = sel5(k == cnt - 1, F[k], Flast);
    Fm = left5<ROT>(Flast, srcL);
}

// Both stages of the cells a lane owns, Q in, the new state out (in Q).
template <class M, int K, int LIM, bool ROT, int DIR = 1>
__device__ __forceinline__ void x_stages(const HydroConsts &hc, int rt, V5 (&Q)[K], int cnt, int srcL, int srcR,
                                         double lambda)
{
    const double ml = -lambda, mhl = -.5 * lambda;
    V5 F[K], Fm, U1[K];
    x_fluxes<M, K, LIM, DIR, ROT>(hc, rt, Q, cnt, srcL, srcR, F, Fm);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const V5 dF = F[k] - (k == 0 ? Fm : F[k > 0 ? k - 1 : 0]);
        U1[k] = axpy5(Q[k], ml, dF);
        if (!M::floors) Q[k] = half_sum<M>(Q[k], U1[k], dF, mhl);
    }
    x_fluxes<M, K, LIM, DIR, ROT>(hc, rt, U1, cnt, srcL, srcR, F, Fm);
#pragma unroll
    for (int k = 0; k < K; k++) {
        const V5 dF = F[k] - (k == 0 ? Fm : F[k > 0 ? k - 1 : 0]);
        if (M::floors) Q[k] = half_sum<M>(Q[k], U1[k], dF, mhl);  // U1 as its floors left it
        Q[k] = axpy5(Q[k], mhl, dF);
    }
}

// Whole lines, 64 / nl of them per wave (nl lanes of K cells each). FULL: every
// line is exactly nl*K cells and nl divides 64, so every lane holds K cells.
// A wave takes one group of lines: fresh waves hide the load latency better
// than a wave that prefetched its next group, whose second register set cost
// spills (256^3: 347 us against 475 prefetching; 128^3 49 against 56).
template <class M, int K, int LIM, bool FULL, bool CFL>
__global__ __launch_bounds__(256, (K <= 4) ? 2 : 1) void sweep_x(const double *src, double *dst, int64_t pitch, int N,
                                               int64_t nlines, int nl, double lambda,
                                               const double *__restrict__ lamp, HydroConsts hc, int rt, CflFuse cf,
                                               GhostFill gf)
{
    if (lamp) lambda = lamp[0];  // time step kept on the device
    const int lane = threadIdx.x & 63;
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int lpw = 64 / nl;
    const int sub = lane / nl;
    const int j = lane - sub * nl;
    const bool laneUsed = sub < lpw;
    const int lbase = sub * nl;
    const int srcL = laneUsed ? lbase + (j == 0 ? nl - 1 : j - 1) : lane;
    const int srcR = laneUsed ? lbase + (j == nl - 1 ? 0 : j + 1) : lane;
    const int x0 = laneUsed ? j * K : 0;
    int cnt = N - x0;
    cnt = cnt < K ? cnt : K;
    if (FULL) cnt = K;
    else if (!laneUsed) cnt = 0;
    const int64_t line = wave * lpw + (laneUsed ? sub : 0);
    const bool own = laneUsed && line < nlines;
    const int64_t off = (line < nlines ? line : nlines - 1) * (int64_t)N + x0;
    V5 Q[K];
#pragma unroll
    for (int k = 0; k < K; k++) Q[k] = (k < cnt) ? load_cell<M, 1>(src + off + k, pitch) : V5{1.0, 1.0, 0.0, 0.0, 0.0};
    x_stages<M, K, LIM, (FULL && K > 1)>(hc, rt, Q, cnt, srcL, srcR, lambda);
    fill_ghosts<K>(Q, laneUsed ? x0 : lane, laneUsed ? lbase : 0, kGhost, N - 1 - kGhost,
                   FULL ? (5 * K - 1 - kGhost) % K : (N - 1 - kGhost) % K, gf);
    double cmin = kCflNone;
#pragma unroll
    for (int k = 0; k < K; k++) {
        if (own && k < cnt) {
            store_cell<M, 1>(dst + off + k, pitch, Q[k]);
            if (CFL && x0 + k >= cf.lo && x0 + k < cf.hi) {
                const double u = cfl_of_cell<M, 1>(cf.a, Q[k]);
                cmin = (u < cmin) ? u : cmin;
            }
        }
    }
    if (CFL) cfl_fold(cf, wave, cmin);
}

// One wave's part of an X line: part `part` of `parts` (near-equal runs of
// cells), K consecutive cells per lane. The wave's window is its part and the
// 4 cells beyond each end (the two stages' stencil, periodic within the line),
// so it forms its outputs alone; the window's outer cells only feed discarded
// values. inplace: the waves of a line share a workgroup and every load of the
// workgroup precedes the barrier while every store follows it, so no wave
// overwrites a cell another has still to read.
// CFL: cmin takes the minimum CFL limit of the outputs at cells [cf.lo, cf.hi),
// nanc counts the NaN limits. gf: K = 1 only (with K = 3 the parts of a mirrored
// 321 x 287 x 305 box took 906 us instead of 793 and its launch of 42, and a
// periodic 1024 x 1024 plane, which fills nothing, 40 us instead of 33).
template <class M, int K, int LIM, bool CFL>
__device__ __forceinline__ void xp_body(const double *src, double *dst, int64_t pitch, int N, int part, int parts,
                                        bool inplace, double lambda, const HydroConsts &hc, int rt,
                                        const CflFuse &cf, const GhostFill &gf, double &cmin, unsigned &nanc)
{
    const int lane = threadIdx.x & 63;
    const int s0 = (int)((int64_t)N * part / parts);  // first output cell of this part
    const int Wn = (int)((int64_t)N * (part + 1) / parts) - s0 + 8;
    const int w0 = lane * K;
    V5 Q[K];
#pragma unroll
    for (int k = 0; k < K; k++) {
        int g = s0 - 4 + w0 + k;  // window cell -> line cell, periodic
        g = (g < 0) ? g + N : g;
        g = (g >= N) ? g - N : g;
        g = (g < N) ? g : N - 1;
        // every lane of the window has K cells (the last one's run past it);
        // idle lanes compute on a constant state
        Q[k] = (w0 < Wn) ? load_cell<M, 1>(src + g, pitch) : V5{1.0, 1.0, 0.0, 0.0, 0.0};
    }
    if (inplace) __syncthreads();
    x_stages<M, K, LIM, true>(hc, rt, Q, K, (lane + 63) & 63, (lane + 1) & 63, lambda);
    // window cell 4 is the part's first
    if (K == 1)
        fill_ghosts<K>(Q, w0, 0, kGhost + 4, N - 1 - kGhost - s0 + 4, 0,
                       GhostFill{part == 0 ? gf.lo : kFillNone, part == parts - 1 ? gf.hi : kFillNone});
#pragma unroll
    for (int k = 0; k < K; k++) {
        const int w = w0 + k;
        if (w >= 4 && w < Wn - 4) {
            const int x = s0 + w - 4;
            const V5 &o = Q[k];
            store_cell<M, 1>(dst + x, pitch, o);
            if (CFL && x >= cf.lo && x < cf.hi) {
                const double u = cfl_of_cell<M, 1>(cf.a, o);
                cmin = (u < cmin) ? u : cmin;
                nanc += (u != u);
            }
        }
    }
}

// X sweep of lines split into parts: one wave per part, one line per
// workgroup of 64 parts threads (two lines per workgroup measured 1-20 %
// slower: the barrier then waits for both).
template <class M, int K, int LIM, bool CFL>
__global__ __launch_bounds__(512, 2) void sweep_xp(const double *src, double *dst, int64_t pitch, int N, int parts,
                                                  double lambda, const double *__restrict__ lamp, HydroConsts hc,
                                                  int rt, CflFuse cf, GhostFill gf)
{
    if (lamp) lambda = lamp[0];  // time step kept on the device
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // in a scalar register
    const int64_t line = blockIdx.x;
    double cmin = kCflNone;
    unsigned nanc = 0;  // not reported by the single-array fold
    xp_body<M, K, LIM, CFL>(src + line * (int64_t)N, dst + line * (int64_t)N, pitch, N, wib, parts, src == dst,
                            lambda, hc, rt, cf, gf, cmin, nanc);
    if (CFL) cfl_fold(cf, (int64_t)blockIdx.x * (blockDim.x >> 6) + wib, cmin);
}

// ---------------------------------------------------------------------------
// Y/Z sweep: register-window march along strided columns
// ---------------------------------------------------------------------------
// One wave-uniform march: lane `lane` walks cells [j0, j0+L) of the column
// starting at `col` (stride sstride, N cells, periodic), the wave's stencil
// ring in LDS at `ring`, and writes to the column starting at `out`. In place
// (out == col) the segments of a column belong to one wave and first = 4: a
// segment's first 4 outputs, which its neighbours' halo reads and the periodic
// wrap still need, wait in this lane's deferred slots (defer/gtid/nthr) until
// the wave has finished reading. Out of place first = 0. seglen is uniform
// over the wave. CFL: cmin takes the minimum CFL limit of the outputs at
// column cells [cf.lo, cf.hi), nanc counts the NaN limits among them.
template <class M, int DIR, int LIM, bool CFL = false, bool NT = false>
__device__ __forceinline__ void march_body(const double *col, double *out, int64_t pitch, int64_t sstride, int N,
                                           int seglen, int j0, int L, int first, double lambda,
                                           const HydroConsts &hc, int rt, double *__restrict__ defer, int64_t gtid,
                                           int64_t nthr, double (*ring)[5][64], int lane, const CflFuse &cf,
                                           const GhostFill &gf, double &cmin, unsigned &nanc)
{
    // wrapped sweep index of the first load (m = j0 - 4), in [0, N)
    int mw = (j0 - 4) % N;
    if (mw < 0) mw += N;
    double *outp = out + (int64_t)(j0 - 9) * sstride;  // address of output t - 9
    double *const dfr = defer + gtid;
    const int64_t dstride = 5 * nthr;
    const double ml = -lambda, mhl = -.5 * lambda;

    const V5 one = V5{1.0, 1.0, 0.0, 0.0, 0.0};
    const V5 zero = V5{0.0, 0.0, 0.0, 0.0, 0.0};
    // Every window variable lives in two slots that trade roles on even and
    // odd steps (prev <-> new), so the loop carries no register moves.
    V5 QA = one, QB = one;    // Q_{m-2} in, Q_m out
    V5 U1A = one, U1B = one;  // U1 (floored) of the previous step in, this step's out
    double eA = 1.0, eB = 1.0;  // internal energy the floors left in U1A / U1B
    V5 wA = one, wB = one, dA = zero, dB = zero, RA = one, RB = one, FAA = zero, FAB = zero;
    V5 w1A = one, w1B = one, d1A = zero, d1B = zero, R1A = one, R1B = one, FBA = zero, FBB = zero;

    // Stage B runs one step behind stage A (it consumes the previous step's
    // U1), so the two long dependency chains of a step are independent.
    // (U1+Q)/2 of a cell is needed three steps after it is formed:
    // it waits in a 4-slot ring in LDS, private to the lane.

    auto step = [&](int t, V5 &Qcur, V5 &Qs, const V5 &U1p, V5 &U1n, const double &ep, double &en,
                    const V5 &wp, V5 &wn, const V5 &dp, V5 &dn, const V5 &Rp, V5 &Rn, const V5 &FAp, V5 &FAn,
                    const V5 &w1p, V5 &w1n, const V5 &d1p, V5 &d1n, const V5 &R1p, V5 &R1n, const V5 &FBp,
                    V5 &FBn) {
        // stage A at cell m-2
        {
            const double e = M::template floor<DIR>(hc, Qcur);
            wn = M::template prims<LIM>(hc, Qcur, e);
        }
        dn = wn - wp;
        V5 Lc;
        M::template face<LIM>(hc, wp, dp, dn, rt, Lc, Rn);  // faces of cell m-1
        FAn = M::flux(hc, Rp, Lc);                           // interface (m-2)+1/2
        const V5 dA = FAn - FAp;
        U1n = axpy5(Qs, ml, dA);
        en = M::template floor<DIR>(hc, U1n);
        {
            const V5 S2 = half_sum<M>(Qs, U1n, dA, mhl);  // (U1+Q)/2 of cell m-2, used at step m+3
            double *r = &ring[t & 3][0][lane];
            r[0] = S2.a;
            r[64] = S2.b;
            r[128] = S2.c;
            r[192] = S2.d;
            r[256] = S2.e;
        }
        Qs = Qcur;

        // stage B at cell m-5, from the previous step's U1 (cell m-3). Its code
        // stays behind stage A's: scheduled into one another the two hold more
        // than two waves' registers (the ensembles' march spilled 16 of them:
        // 60 problems of 64..512 cells 664 us an iteration, 604 so; 200^3 step
        // with van Leer 580, 571).
        __builtin_amdgcn_sched_barrier(0);
        w1n = M::template prims<LIM>(hc, U1p, ep);
        d1n = w1n - w1p;
        V5 L1c;
        M::template face<LIM>(hc, w1p, d1p, d1n, rt, L1c, R1n);  // faces of cell m-4
        FBn = M::flux(hc, R1p, L1c);                              // interface (m-5)+1/2
        const double *r = &ring[(t + 1) & 3][0][lane];  // slot of step t-3
        const V5 S5{r[0], r[64], r[128], r[192], r[256]};
        const V5 o = axpy5(S5, mhl, FBn - FBp);  // cell m-5

        // Every step stores exactly 5 doubles: to the cell (outputs first..L-1),
        // to a deferred slot (earlier ones) or to this lane's dummy slot (no
        // output yet / past the segment). With a fixed store count per step the
        // compiler can wait for a prefetched load without waiting for stores
        // (stores share the vector-memory counter on gfx9).
        // outp walks the column one cell per step (it points at output oi);
        // the deferred slots are wave-uniform offsets of this lane's block.
        const int oi = t - 9;  // output index within the segment
        if (CFL && oi >= 0 && oi < L && j0 + oi >= cf.lo && j0 + oi < cf.hi) {
            const double u = cfl_of_cell<M, DIR>(cf.a, o);
            cmin = (u < cmin) ? u : cmin;
            nanc += (u != u);
        }
        const bool direct = (oi >= first) & (oi < L);
        const int slot = ((oi >= 0) & (oi < first) & (oi < L)) ? oi : first;
        double *dq = dfr + (int64_t)slot * dstride;
        double *dst = direct ? outp : dq;
        const int64_t st = direct ? pitch : nthr;
        outp += sstride;
        store_cell<M, DIR, NT>(dst, st, o);
    };

    const int maxsteps = seglen + 9;
    // Prefetch slots for even / odd steps. The loads are unconditional (a lane
    // past its segment, or of an inactive column, reads a valid cell it then
    // ignores: mw always wraps into [0, N) and `col` of an inactive column is
    // element 0), so the compiler neither copies slots nor waits for a load it
    // has just issued.
    V5 N0 = load_cell<M, DIR, NT>(col + (int64_t)mw * sstride, pitch);
    V5 N1;
    // Enter the loop with the same vector-memory counter pattern as the
    // back-edge (load group, then 5 stores) so the wait at the loop head can
    // leave stores outstanding: the stores write the loaded cell into this
    // lane's dummy slot, which also pins them after the load.
    store_cell<M, DIR, NT>(dfr + (int64_t)first * dstride, nthr, N0);

    // Steps go in pairs. When maxsteps is odd the last pair's second step is
    // one past the segment: it loads a valid (wrapped) cell and stores to the
    // dummy slot, so running it unconditionally changes no output and keeps
    // the loop to one path (no register copies at the back edge).
    for (int t = 0; t < maxsteps; t += 2) {
        mw = (mw + 1 == N) ? 0 : mw + 1;
        N1 = load_cell<M, DIR, NT>(col + (int64_t)mw * sstride, pitch);
        step(t, N0, QA, U1A, U1B, eA, eB, wA, wB, dA, dB, RA, RB, FAA, FAB, w1A, w1B, d1A, d1B, R1A, R1B, FBA,
             FBB);
        mw = (mw + 1 == N) ? 0 : mw + 1;
        N0 = load_cell<M, DIR, NT>(col + (int64_t)mw * sstride, pitch);
        step(t + 1, N1, QB, U1B, U1A, eB, eA, wB, wA, dB, dA, RB, RA, FAB, FAA, w1B, w1A, d1B, d1A, R1B, R1A, FBB,
             FBA);
    }

    // every lane of the wave has finished reading: release the deferred outputs
    const int nd = L < first ? L : first;
    for (int oi = 0; oi < nd; oi++) {
        const V5 o = load_cell<M, DIR, NT>(defer + gtid + (int64_t)oi * 5 * nthr, nthr);
        store_cell<M, DIR, NT>(out + (int64_t)(j0 + oi) * sstride, pitch, o);
    }

    // the faces' ghosts from the cells this lane has stored: a segment at a face
    // holds the ghosts and their sources (the launcher sees to it)
    if (gf.lo && j0 == 0 && L > 0) {
        for (int g = 0; g < kGhost; g++) {
            bool turned;
            V5 v = load_cell<M, DIR, NT>(out + (int64_t)ghost_source(g, N, gf, turned) * sstride, pitch);
            if (turned) v.c = -v.c;
            store_cell<M, DIR, NT>(out + (int64_t)g * sstride, pitch, v);
        }
    }
    if (gf.hi && j0 + L == N && L > 0) {
        for (int g = N - kGhost; g < N; g++) {
            bool turned;
            V5 v = load_cell<M, DIR, NT>(out + (int64_t)ghost_source(g, N, gf, turned) * sstride, pitch);
            if (turned) v.c = -v.c;
            store_cell<M, DIR, NT>(out + (int64_t)g * sstride, pitch, v);
        }
    }
}

// Columns are numbered x + nx * o (o: the other direction), so a wave's
// columns run on across rows and every lane but the last wave's has one.
// In place: a wave holds W = 64/S columns, their S segments side by side in
// its lanes. Out of place (dst != src): a wave holds one segment of 64 columns
// and the segments of a column are waves of their own, segment-major.
template <class M, int DIR, int LIM, bool CFL, bool NT>
__global__ __launch_bounds__(256) void sweep_march(const double *src, double *dst, int64_t pitch, int nx,
                                                   int64_t sstride, int64_t ostride, int64_t columns, int N, int S,
                                                   int seglen, double lambda, const double *__restrict__ lamp,
                                                   HydroConsts hc, int rt, double *__restrict__ defer, CflFuse cf,
                                                   GhostFill gf)
{
    if (lamp) lambda = lamp[0];  // time step kept on the device
    const int lane = threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // in a scalar register
    const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + wib;
    const bool inplace = src == dst;
    const int W = inplace ? 64 / S : 64;
    const int64_t colWaves = (columns + W - 1) / W;
    if (wave >= (inplace ? colWaves : colWaves * S)) return;
    const int64_t cw = inplace ? wave : wave % colWaves;
    const int s = inplace ? lane / W : (int)(wave / colWaves);
    const int64_t cid = cw * W + lane % W;
    const bool colValid = (cid < columns) && (s < S);
    // lanes of no column (past the last, or s >= S when S does not divide
    // 64) march a zero-length segment from row 0: their unconditional loads
    // then stay inside the column
    const int j0 = colValid ? s * seglen : 0;
    int L = N - j0;
    L = L < seglen ? L : seglen;
    if (!colValid || L < 0) L = 0;

    const int64_t other = cid / nx;
    const int64_t off = colValid ? (cid - other * nx) + other * ostride : 0;
    const int64_t gtid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nthr = (int64_t)gridDim.x * blockDim.x;
    __shared__ double sring[4][4][5][64];  // [wave in block][slot][variable][lane]
    double cmin = kCflNone;
    unsigned nanc = 0;  // not reported by the single-array fold
    march_body<M, DIR, LIM, CFL, NT>(src + off, dst + off, pitch, sstride, N, seglen, j0, L, inplace ? 4 : 0, lambda,
                                     hc, rt, defer, gtid, nthr, sring[wib], lane, cf, gf, cmin, nanc);
    if (CFL) cfl_fold(cf, wave, cmin);
}

// ---------------------------------------------------------------------------
// Y/Z sweep of few columns: the X scheme on a tile turned in LDS
// ---------------------------------------------------------------------------
// A block takes 16 columns (a full cache line of each row) of up to 64 cells,
// reads them row by row, and its waves take them out of the tile as the X sweep
// takes its lines: one cell per lane, neighbours by cross-lane shuffle. Rows
// are 17 doubles apart, so neither way of reading the tile meets a bank twice.
// Columns of up to 64 cells are held whole (64 / N of them in a wave), in place
// or not; longer ones go out of place in parts of up to 56 cells, with the 4
// cells beyond each end as the X sweep's parts (part = blockIdx.y).
constexpr int kTileCols = 16;

template <class M, int DIR, int LIM, bool CFL>
__global__ __launch_bounds__(1024) void sweep_tile(const double *src, double *dst, int64_t pitch, int nx,
                                                   int64_t sstride, int64_t ostride, int64_t columns, int N, int parts,
                                                   double lambda, const double *__restrict__ lamp, HydroConsts hc,
                                                   int rt, CflFuse cf, GhostFill gf)
{
    if (lamp) lambda = lamp[0];  // time step kept on the device
    constexpr int kLd = kTileCols + 1, kSlab = 64 * kLd;
    __shared__ double tile[5 * kSlab];
    // rows [0, Wn) of the tile are the column's cells r0 + row (periodic); the
    // part's outputs are its rows [halo, Wn - halo)
    const int halo = parts > 1 ? 4 : 0;
    const int r0 = (int)((int64_t)N * blockIdx.y / parts) - halo;
    const int Wn = (int)((int64_t)N * (blockIdx.y + 1) / parts) - r0 + halo;
    const int64_t col0 = (int64_t)blockIdx.x * kTileCols;
    // this thread's column and first row on the tile's global side
    const int gc = threadIdx.x % kTileCols, g0 = threadIdx.x / kTileCols, gstep = blockDim.x / kTileCols;
    const int64_t cid = col0 + gc;
    const bool gown = cid < columns;
    const int64_t other = cid / nx;
    const int64_t goff = (cid - other * nx) + other * ostride;
    for (int r = g0; r < Wn; r += gstep) {
        int g = r0 + r;
        g = (g < 0) ? g + N : ((g >= N) ? g - N : g);
        if (gown) store_cell<M, DIR>(tile + r * kLd + gc, kSlab, load_cell<M, DIR>(src + goff + g * sstride, pitch));
    }
    __syncthreads();

    const int lane = threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // in a scalar register
    const int lpw = 64 / Wn;
    const int sub = lane / Wn;
    const int j = lane - sub * Wn;
    const bool laneUsed = sub < lpw;
    const int srcL = laneUsed ? sub * Wn + (j == 0 ? Wn - 1 : j - 1) : lane;
    const int srcR = laneUsed ? sub * Wn + (j == Wn - 1 ? 0 : j + 1) : lane;
    const int c = wib * lpw + sub;
    const bool own = laneUsed && c < kTileCols && col0 + c < columns;
    double *cell = tile + (own ? j * kLd + c : 0);
    V5 Q[1] = {own ? load_cell<M, DIR>(cell, kSlab) : V5{1.0, 1.0, 0.0, 0.0, 0.0}};
    x_stages<M, 1, LIM, false, DIR>(hc, rt, Q, 1, srcL, srcR, lambda);
    double cmin = kCflNone;
    if (own) {
        store_cell<M, DIR>(cell, kSlab, Q[0]);
        const int g = r0 + j;
        if (CFL && j >= halo && j < Wn - halo && g >= cf.lo && g < cf.hi) cmin = cfl_of_cell<M, DIR>(cf.a, Q[0]);
    }
    __shared__ double least[16];
    if (CFL) {
        cmin = wave_min(cmin < kCflNone ? cmin : kCflNone);
        if (lane == 0) least[wib] = cmin;
    }
    __syncthreads();
    if (CFL && wib == 0) {
        // one key for the block: 4096 waves of 64^3 cells on the keys took 8 us
        cmin = wave_min(lane < (int)(blockDim.x >> 6) ? least[lane] : kCflNone);
        if (lane == 0) fold_min(cf.slots + ((blockIdx.x + blockIdx.y * gridDim.x) & (kCflSlots - 1)), cmin);
    }
    for (int r = halo + g0; r < Wn - halo; r += gstep) {
        if (gown) {
            bool turned;
            V5 q = load_cell<M, DIR>(tile + (ghost_source(r0 + r, N, gf, turned) - r0) * kLd + gc, kSlab);
            if (turned) q.c = -q.c;
            store_cell<M, DIR>(dst + goff + (r0 + r) * sstride, pitch, q);
        }
    }
}

}  // namespace imogen
