// fluid_sweep.hip -- fused HLLC / HLL SSP-RK2 directional sweeps for gfx950.
//
// One kernel launch performs both SSP-RK2 stages of one directional sweep
// (the reference runs them as two or more launches through a 5-slab temporary
// plus a physical transpose, gpuclass/cudaFluidStep.cu:485-627 and :630-700,
// gpuclass/flux.cu:92-116). For HLL the pressure solver's floors, which the
// reference applies in place before each stage (:646-690), are applied to
// each cell as it is read: Q before stage A, U1 before stage B; the floored
// values feed both the fluxes and the SSP-RK2 combination. The fluid is updated in place in the reference's
// 5-slab layout (rho, E, px, py, pz; x fastest), with the reference's periodic
// wrap along the swept line (cudaFluidStep.cu:1159-1162).
//
// Three data-movement schemes, all free of transposes through memory:
//  * X (contiguous) lines: a wave owns whole lines or, for long or few lines,
//    a part of one. Each lane holds K consecutive cells in registers; the
//    one-cell neighbours it needs from the adjacent lanes (primitives, left
//    face, flux) come by cross-lane shuffle. No LDS.
//  * Few Y/Z (strided) lines: a block turns 16 columns of up to 64 cells in LDS
//    and takes them as the X sweep does.
//  * Other Y/Z lines: each lane marches along one column (coalesced over
//    x across the wave) keeping a register window of the two-stage stencil.
//    Columns are split into segments for occupancy. A sweep whose output goes
//    to a second state array (update_3d pairs such sweeps) may cut them
//    anywhere; one that works in place keeps a column's segments in one wave,
//    and each segment its first 4 outputs in a scratch buffer until the whole
//    wave has finished reading, so the update (and the periodic wrap) is
//    race-free.
#include "sweep_kernels.h"
#include "imogen_internal.h"

namespace imogen {


// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------

// Segments per column of an in-place Y/Z march, S in {1, 2, 4} (W = 64/S
// columns per wave, so every lane has a column slot). The kernel's time follows
// the busiest SIMD: with w waves over 1024 SIMDs (256 CUs x 4, up to 2 resident
// waves each) it runs ceil(w / 1024) waves of seglen + 9 steps, and a launch
// with fewer waves than SIMDs runs about 1.8x slower per step (idle SIMDs,
// no latency hiding). Segments shorter than 16 cells are not used. Measured
// Y / Z times (HLLC, ms) and the rule's pick:
//   96^3  S=1 0.140  S=2 0.077  S=4 0.051  -> 4     320^3 S=1 1.04  S=2 0.79  S=4 0.79  -> 4
//   160^3 S=1 0.216  S=2 0.201  S=4 0.125  -> 4     384^3 S=1 1.37  S=2 1.24  S=4 1.26  -> 4
//   192^3 S=1 0.249  S=2 0.236  S=4 0.203  -> 4     256^3 S=1 0.315 S=2 0.309..0.329 S=4 0.324 -> 1
// Counts that do not divide 64 leave a wave's row segment off the 128-byte
// lines: S = 3, 6 (21, 10 columns) ran 1.5-2x slower than S = 2 or 4 (smooth
// state, 160^3-384^3; 192^3: S=3 0.374, S=6 0.395 against S=4 0.197), and
// S = 8 (8 columns, 64 bytes) 1.3-1.5x slower.
static int segments_in_place(int64_t columns, int N)
{
    int best = 1;
    double bestCost = 0.0;
    for (int S = 1; S <= 4; S *= 2) {
        if (S > 1 && N < 16 * S) break;
        const int64_t waves = (columns * S + 63) / 64;
        const int64_t rounds = (waves + 1023) / 1024;
        const double cost = (double)rounds * ((N + S - 1) / S + 9) * (waves < 1024 ? 1.8 : 1.0);
        if (S == 1 || cost < bestCost) {
            best = S;
            bestCost = cost;
        }
    }
    return best;
}

// Segments per column of an out-of-place march, any count: a wave holds one
// segment of 64 columns, a segment of L cells takes L + 9 steps, and a step
// of one wave is bound by its issue (about 1.0 us alone on a SIMD, 1.15 us
// per wave with two), so the time is about ceil(waves / 1024) (L + 9); a lone
// wave per SIMD also waits for memory (the 5 %). Measured (HLLC, van Leer,
// smooth states, us; in place in brackets):
//   1024^2 L=8 61  L=16 46  L=32 57 (305)      64^3  L=4 22.5  L=8 26  L=16 34 (35)
//   600^2  L=4 37  L=6 26   L=16 35 (193)      128^3 L=16 72   L=32 60 L=64 94 (65)
//   160^3  L=16 133 L=32 105 L=80 136 (124)    192^3 L=32 195  L=64 174 L=192 268 (212)
//   256^3  Y: L=64 363  L=128 341  L=256 355 (409-480)  Z: 353, 329, 345 (336-353)
static int segments_out_of_place(int64_t columns, int N)
{
    const int64_t colWaves = (columns + 63) / 64;
    int best = 1;
    double bestCost = 0.0;
    for (int S = 1; S == 1 || S * 4 <= N; S++) {
        const int64_t rounds = (colWaves * S + 1023) / 1024;
        const double cost = (double)rounds * ((N + S - 1) / S + 9) * (rounds == 1 ? 1.05 : 1.0);
        if (S == 1 || cost < bestCost) {
            best = S;
            bestCost = cost;
        }
        if (rounds > 16) break;
    }
    return best;
}

// Launch shape of an X sweep over nlines lines of N cells: K cells per lane;
// parts = 0: whole lines (sweep_x, nl lanes per line, 256-thread blocks),
// otherwise one line per block, split over `parts` waves (sweep_xp).
// K = 0 when N is above 1024.
struct XGeom {
    int K = 0, nl = 0, parts = 0;
    int64_t blocks = 0;
    int threads = 256;
};

// A part's window is its cells and 8 more, so K cells per lane take parts of
// at most 64 K - 8 cells. Measured (HLLC, van Leer, smooth states, us):
//  * Lines that fill their lanes (64, 128, 192, 256 cells) stay whole (16384 of
//    128: 49, K=1 parts 64; 65536 of 256: 347, K=3 parts 477), as do lines of
//    less than 64.
//  * So do many lines of 384 where six cells a lane stay in registers (`wide`:
//    HLLC with Ospre or van Leer; 36864 lines: 341, K=4 parts 375). HLL and the
//    limiters chosen at run time hold more per cell: whole steps of 384 x 384 x
//    96 cells with whole lines 1307 and 1354, with K=4 parts 1155 and 1129.
//    Fewer lines go the way of their neighbours (steps of 384 x 200 cells: HLLC
//    23.1, K=1 parts 17.1; HLL 27.7, 17.7).
//  * Others of up to 256 cells: K=1 parts, whose lanes need no select at a
//    line's end and leave room for four waves per SIMD (13560 of 131: 54,
//    whole 68; 20000 of 150: 77, 92), while the last-level cache holds the
//    state and gives the parts' overlap for nothing (62500 of 250: 521, whole
//    375; 40000 of 200: 240, 215).
//  * Longer ones: K=3 (28700 of 321: 250, K=2 263, K=1 283; 1024 of 1024: 34,
//    K=4 46, whole lines of 16 cells per lane, whose arrays left the
//    registers, 130), but K=4 where two parts of it replace three (369..496).
//    Many lines of 497..552 are three parts of K=3 (whole HLLC steps of N x 512 x
//    64 cells, in place with whole lines of 8 or 9 cells per lane -> as here: 497
//    1334 -> 1195, 512 1276 -> 1202, 530 2770 -> 1300, 552 2810 -> 1338).
//  * Too few lines to fill the 1024 SIMDs: smaller K for a shorter chain per
//    wave (17 lines of 300: K=1 5.3, K=2 5.7, K=3 6.6; 400 x 400: K=1 8.8,
//    K=2 8.9, K=3 10.8), as far as 8 waves reach.
static XGeom x_geom(int N, int64_t nlines, bool wide)
{
    XGeom g;
    if (N > 1024) return g;
    const auto parts = [N](int K) { return (N + 64 * K - 9) / (64 * K - 8); };
    if (N > 64 && N <= 256) {
        const bool cached = (int64_t)N * nlines * 5 * (int64_t)sizeof(double) <= (int64_t)256 << 20;
        if ((N % 64 != 0 && cached) || nlines * parts(1) <= 1024) g.K = 1;
    } else if (N > 256) {
        if (nlines * parts(3) >= 1536) g.K = (N == 384 && wide) ? 0 : ((N > 368 && N <= 496) ? 4 : 3);
        else g.K = parts(1) <= 8 ? 1 : (parts(2) <= 8 ? 2 : 3);
    }
    if (g.K) {
        g.parts = parts(g.K);
        g.threads = 64 * g.parts;
        g.blocks = nlines;
        return g;
    }
    g.K = (N == 384) ? 6 : (N + 63) / 64;
    g.nl = (N + g.K - 1) / g.K;
    const int lpw = 64 / g.nl;
    g.blocks = ((nlines + lpw - 1) / lpw + 3) / 4;
    return g;
}

// Launch shape of a Y (dir 2) or Z (dir 3) march: S segments per column,
// blocks of 256 threads (nthr in all).
struct MarchGeom {
    int N = 0, S = 1, seglen = 0;
    int64_t columns = 0, blocks = 0, nthr = 0;
};

static MarchGeom march_geom(int nx, int ny, int nz, int dir, bool inplace)
{
    MarchGeom g;
    g.N = (dir == 2) ? ny : nz;
    g.columns = (int64_t)nx * ((dir == 2) ? nz : ny);
    g.S = inplace ? segments_in_place(g.columns, g.N) : segments_out_of_place(g.columns, g.N);
    g.seglen = (g.N + g.S - 1) / g.S;
    if (!inplace) g.S = (g.N + g.seglen - 1) / g.seglen;  // no empty segment
    const int W = inplace ? 64 / g.S : 64;
    const int64_t colWaves = (g.columns + W - 1) / W;
    g.blocks = ((inplace ? colWaves : colWaves * g.S) + 3) / 4;
    g.nthr = g.blocks * 256;
    return g;
}

// Scratch doubles per marching lane: a dummy slot of 5 and, in place, 4
// deferred outputs.
static int march_slots(bool inplace)
{
    return inplace ? 25 : 5;
}

// Scratch of one launch: past the first `off` bytes of the library's block,
// which update_3d keeps a second state array in.
static void *sweep_scratch(size_t off, size_t bytes)
{
    char *p = (char *)scratch_block(off + bytes);
    return p ? p + off : nullptr;
}

template <class M, int LIM>
static int launch_x(const double *src, double *dst, int64_t pitch, int N, int64_t nlines, double lambda,
                    const double *lamp, const HydroConsts &hc, int rt, const CflFuse &cf, GhostFill gf,
                    bool *filled, hipStream_t s)
{
    constexpr bool wide = !M::floors && LIM >= 0;
    const XGeom g = x_geom(N, nlines, wide);
    if (g.K == 0) return IM_FAIL(ERROR_NOIMPLEMENT, "X sweep supports lines of at most 1024 cells (got %d)", N);
    const int K = g.K, nl = g.nl;
    if (g.blocks > INT32_MAX) return IM_FAIL(ERROR_INVALID_ARGS, "too many lines for one X launch");
    dim3 grid((unsigned)g.blocks), block((unsigned)g.threads);
    if (g.parts) {
        if (K > 1 && (gf.lo | gf.hi)) *filled = false;
#define IM_XP(KK, C)                                                                                          \
    hipLaunchKernelGGL((sweep_xp<M, KK, LIM, C>), grid, block, 0, s, src, dst, pitch, N, g.parts, lambda, \
                       lamp, hc, rt, cf, gf)
#define IM_XP_CASE(KK)                  \
    case KK:                            \
        if (cf.slots) IM_XP(KK, true);  \
        else IM_XP(KK, false);          \
        break;
        switch (K) {
            IM_XP_CASE(1)
            IM_XP_CASE(2)
            IM_XP_CASE(3)
            IM_XP_CASE(4)
        }
#undef IM_XP_CASE
#undef IM_XP
        return IM_LAUNCHED("sweep_xp");
    }
    const bool full = (nl * K == N) && (64 % nl == 0);
#define IM_X(KK, F, C)                                                                                        \
    hipLaunchKernelGGL((sweep_x<M, KK, LIM, F, C>), grid, block, 0, s, src, dst, pitch, N, nlines, nl, lambda, lamp, \
                       hc, rt, cf, gf)
#define IM_X_CASE(KK)                               \
    case KK:                                        \
        if (full && cf.slots) IM_X(KK, true, true); \
        else if (full) IM_X(KK, true, false);       \
        else if (cf.slots) IM_X(KK, false, true);   \
        else IM_X(KK, false, false);                \
        break;
    switch (K) {
        IM_X_CASE(1)
        IM_X_CASE(2)
        IM_X_CASE(3)
        IM_X_CASE(4)
    case 6:  // 384 cells: every lane full
        if constexpr (wide) {
            if (cf.slots) IM_X(6, true, true);
            else IM_X(6, true, false);
        }
        break;
    }
#undef IM_X_CASE
#undef IM_X
    return IM_LAUNCHED("sweep_x");
}

// Parts per column of a tiled Y/Z sweep, 0: the sweep marches. A march of few
// columns is bound by its serial chain, at least 13 steps of about 1 us however
// short its segments, and a tile by its waves' issue: about 8 us, and twice as
// long once each SIMD has 8 waves. So tiles where their waves are few: 16384 of
// whole columns, or 8192 of parts, which compute their 8 halo cells twice.
// Device loop (HLLC, van Leer), us per iteration, march -> tile:
//   whole: 16^3 107 -> 51   32^3 111 -> 59   48^3 133 -> 85   64^3 143 -> 104
//          200 x 200 x 32 (20000 waves) 282 -> 257   128 x 128 x 64 (16384) 233 -> 227
//          256 x 256 x 64 (65536) 635 -> 717   512 x 512 x 32 (131072) 1233 -> 1277
//   parts: 64 x 100 66 -> 45   300^2 81 -> 60   512^2 (5120) 101 -> 89   700^2 (9100) 115 -> 111
//          80^3 (12800) 174 -> 183   1024^2 (19456) 166 -> 168   128^3 (49152) 345 -> 412
static int tile_parts(int64_t columns, int N, bool inplace)
{
    if (N <= 64) {
        const int lpw = 64 / N;
        return (columns + lpw - 1) / lpw <= 16384 ? 1 : 0;
    }
    const int parts = (N + 55) / 56;
    return !inplace && columns * parts <= 8192 ? parts : 0;
}

bool sweep_cuts(int nx, int ny, int nz, int dir)
{
    const int N = (dir == 2) ? ny : nz;
    return dir != 1 && tile_parts((int64_t)nx * ((dir == 2) ? nz : ny), N, false) != 1;
}

template <class M, int LIM>
static int launch_tile(const double *src, double *dst, int64_t pitch, int nx, int ny, int nz, int dir, int parts,
                       double lambda, const double *lamp, const HydroConsts &hc, int rt, const CflFuse &cf,
                       GhostFill gf, hipStream_t s)
{
    const int N = (dir == 2) ? ny : nz;
    const int64_t sstride = (dir == 2) ? (int64_t)nx : (int64_t)nx * ny;
    const int64_t ostride = (dir == 2) ? (int64_t)nx * ny : (int64_t)nx;
    const int64_t columns = (int64_t)nx * ((dir == 2) ? nz : ny);
    const int lpw = parts == 1 ? 64 / N : 1;
    const int waves = (kTileCols + lpw - 1) / lpw;
    dim3 grid((unsigned)((columns + kTileCols - 1) / kTileCols), (unsigned)parts), block((unsigned)(64 * waves));
#define IM_TILE(D, C)                                                                                        \
    hipLaunchKernelGGL((sweep_tile<M, D, LIM, C>), grid, block, 0, s, src, dst, pitch, nx, sstride, ostride, \
                       columns, N, parts, lambda, lamp, hc, rt, cf, gf)
    if (dir == 2) {
        if (cf.slots) IM_TILE(2, true);
        else IM_TILE(2, false);
    } else {
        if (cf.slots) IM_TILE(3, true);
        else IM_TILE(3, false);
    }
#undef IM_TILE
    return IM_LAUNCHED("sweep_tile");
}

template <class M, int LIM>
static int launch_march(const double *src, double *dst, size_t scratchOff, int64_t pitch, int nx, int ny, int nz,
                        int dir, double lambda, const double *lamp, const HydroConsts &hc, int rt, const CflFuse &cf,
                        GhostFill gf, bool *filled, hipStream_t s)
{
    const int64_t sstride = (dir == 2) ? (int64_t)nx : (int64_t)nx * ny;
    const int64_t ostride = (dir == 2) ? (int64_t)nx * ny : (int64_t)nx;
    const MarchGeom g = march_geom(nx, ny, nz, dir, src == dst);
    if (g.blocks > INT32_MAX) return IM_FAIL(ERROR_INVALID_ARGS, "too many columns for one march launch");
    const int lastlen = g.N - (g.S - 1) * g.seglen;
    if ((g.seglen < lastlen ? g.seglen : lastlen) < gf.reach()) {
        if (gf.lo | gf.hi) *filled = false;
        gf = GhostFill{};
    }
    dim3 grid((unsigned)g.blocks), block(256);
    double *defer = (double *)sweep_scratch(scratchOff, (size_t)g.nthr * march_slots(src == dst) * sizeof(double));
    if (!defer) return IM_FAIL(ERROR_NOMEM, "no scratch for deferred outputs");
    // rows of a multiple of 16 cells in a 256-byte-aligned slab: every segment
    // row (16, 32 or 64 columns) is whole 128-byte lines -> nontemporal hint,
    // for states beyond the 256 MB last-level cache (256^3: 341 us with it,
    // 347 without; 192^3: 174 and 170, 1024^2: 46 and 43)
    const bool lines = (nx % 16) == 0 && (pitch % 32) == 0 && (((uintptr_t)src | (uintptr_t)dst) % 256) == 0 &&
                       pitch * 5 * (int64_t)sizeof(double) > (int64_t)256 << 20;
#define IM_MARCH(D, C, T)                                                                                      \
    hipLaunchKernelGGL((sweep_march<M, D, LIM, C, T>), grid, block, 0, s, src, dst, pitch, nx, sstride, ostride, \
                       g.columns, g.N, g.S, g.seglen, lambda, lamp, hc, rt, defer, cf, gf)
#define IM_MARCH_NT(D, C)             \
    do {                              \
        if (lines) IM_MARCH(D, C, true);  \
        else IM_MARCH(D, C, false);       \
    } while (0)
    if (dir == 2) {
        if (cf.slots) IM_MARCH_NT(2, true);
        else IM_MARCH_NT(2, false);
    } else {
        if (cf.slots) IM_MARCH_NT(3, true);
        else IM_MARCH_NT(3, false);
    }
#undef IM_MARCH_NT
#undef IM_MARCH
    return IM_LAUNCHED("sweep_march");
}

template <class M, int LIM>
static int launch_dir(const double *src, double *dst, size_t off, int64_t pitch, int nx, int ny, int nz, int dir,
                      double lambda, const double *lamp, const HydroConsts &hc, int rt, const CflFuse &cf,
                      GhostFill gf, bool *filled, hipStream_t s)
{
    const int slot = prof_begin(PROF_SWEEP_X + dir - 1, s);
    int rc;
    *filled = true;
    if (dir == 1) rc = launch_x<M, LIM>(src, dst, pitch, nx, (int64_t)ny * nz, lambda, lamp, hc, rt, cf, gf, filled, s);
    else if (const int parts = tile_parts((int64_t)nx * ((dir == 2) ? nz : ny), (dir == 2) ? ny : nz, src == dst))
        rc = launch_tile<M, LIM>(src, dst, pitch, nx, ny, nz, dir, parts, lambda, lamp, hc, rt, cf, gf, s);
    else rc = launch_march<M, LIM>(src, dst, off, pitch, nx, ny, nz, dir, lambda, lamp, hc, rt, cf, gf, filled, s);
    prof_end(slot, s);
    return rc;
}

template <class M>
static int launch_method(const double *src, double *dst, size_t off, int64_t pitch, int nx, int ny, int nz, int dir,
                         double lambda, const double *lamp, const HydroConsts &hc, int limiter, const CflFuse &cf,
                         const GhostFill &gf, bool *filled, hipStream_t s)
{
    switch (limiter) {
    case LIMITER_OSPRE:
        return launch_dir<M, 0>(src, dst, off, pitch, nx, ny, nz, dir, lambda, lamp, hc, 0, cf, gf, filled, s);
    case LIMITER_VANLEER:
        return launch_dir<M, 1>(src, dst, off, pitch, nx, ny, nz, dir, lambda, lamp, hc, 1, cf, gf, filled, s);
    case LIMITER_MINMOD:
    case LIMITER_SUPERBEE:
    case LIMITER_VANALBADA:
    case LIMITER_MC:
    case LIMITER_ZERO:
        return launch_dir<M, -1>(src, dst, off, pitch, nx, ny, nz, dir, lambda, lamp, hc, limiter, cf, gf, filled, s);
    default: return IM_FAIL(ERROR_INVALID_ARGS, "unknown slope limiter %d", limiter);
    }
}

// The march's, also where a tiled sweep takes none: the grids that the
// allocation-free step admits do not depend on that choice.
int64_t sweep_scratch_bytes(int nx, int ny, int nz, int dir, bool inplace)
{
    const int N = (dir == 1) ? nx : (dir == 2 ? ny : nz);
    if (dir < 1 || dir > 3 || N < 3) return 0;
    if (dir == 1) return 0;
    return march_geom(nx, ny, nz, dir, inplace).nthr * march_slots(inplace) * (int64_t)sizeof(double);
}

int launch_fluid_sweep(const double *src, double *dst, size_t scratchOff, int64_t pitch, int nx, int ny, int nz,
                       int dir, int method, double lambda, double gamma, double rhomin, double ciso, int limiter,
                       hipStream_t s, const double *lamp, const CflFuse *cfl, const GhostFill &gf, bool *filled)
{
    if (dir < 1 || dir > 3) return IM_FAIL(ERROR_INVALID_ARGS, "sweep direction %d", dir);
    const int N = (dir == 1) ? nx : (dir == 2 ? ny : nz);
    *filled = false;
    if (N < 3) return SUCCESSFUL;  // cudaFluidStep.cu:301
    HydroConsts hc;
    hc.gamma = gamma;
    hc.gm1 = gamma - 1.0;
    hc.hgm1 = .5 * (gamma - 1.0);
    hc.igm1 = 1.0 / (gamma - 1.0);
    hc.govergm1 = gamma / (gamma - 1.0);
    hc.rhomin = rhomin;
    hc.emin = 1e-5 / (gamma - 1.0);  // cudaFluidStep.cu:298
    hc.ciso = ciso;
    hc.cisosq = ciso * ciso;
    const CflFuse cf = cfl ? *cfl : CflFuse{};
    if (method == METHOD_HLLC)
        return launch_method<Hllc>(src, dst, scratchOff, pitch, nx, ny, nz, dir, lambda, lamp, hc, limiter, cf, gf,
                                   filled, s);
    if (method == METHOD_HLL)
        return launch_method<Hll>(src, dst, scratchOff, pitch, nx, ny, nz, dir, lambda, lamp, hc, limiter, cf, gf,
                                  filled, s);
    return IM_FAIL(ERROR_INVALID_ARGS, "sweep kernel for method %d", method);
}

}  // namespace imogen
