// cfl_device.h -- per-cell sound speed and CFL time-step limit (FP64).
// cukern_Soundspeed_hd (gpuclass/cudaSoundspeed.cu:178-195) and
// cukern_CFLtimestep (gpuclass/cflTimestep.cu:262-377, SQUARE geometry).
#pragma once
#include <hip/hip_runtime.h>

#include <cstring>

namespace imogen {

// The CFL arithmetic is evaluated exactly as written (no FMA contraction), so
// the limit of a cell is bitwise the same in the CFL kernel and in a sweep
// that folds the CFL in, whatever the surrounding code lets the compiler fuse.
__device__ __forceinline__ double cs_of(double rho, double E, double px, double py, double pz, double gg1)
{
#pragma clang fp contract(off)
    double rhoinv = 1 / rho;
    double csq = gg1 * (E - .5 * (px * px + py * py + pz * pz) * rhoinv) * rhoinv;
    if (csq < 0.0) csq = 0.0;
    return sqrt(csq);
}

__device__ __forceinline__ double wave_min(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        double o = __shfl_xor(v, off, 64);
        v = (o < v) ? o : v;
    }
    return v;
}

// Adds the wave's total of the lanes' counts to *slot with one atomic (none
// when the total is 0). Must be reached by all 64 lanes; slot null: no-op.
__device__ __forceinline__ void wave_count(unsigned long long *slot, unsigned v)
{
    if (!slot) return;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    if ((threadIdx.x & 63) == 0 && v) atomicAdd(slot, (unsigned long long)v);
}

// dim = simulation dimension (1..3), xinjin selects the per-direction form.
// fused != 0: sound speed computed in-line from gamma instead of read from cs.
struct CflArgs {
    double gg1, hx, hy, hz, hmin;
    int fused, dim, xinjin;
};

// time-step limit of one cell (cflTimestep.cu:292-335)
__device__ __forceinline__ double cfl_cell(const CflArgs &a, double rho, double E, double px, double py,
                                           double pz, double cIn)
{
#pragma clang fp contract(off)
    const double c = a.fused ? cs_of(rho, E, px, py, pz, a.gg1) : cIn;
    double u;
    if (!a.xinjin) {
        double pm;
        if (a.dim == 1) {
            pm = fabs(px);
        } else {
            double p = px * px;
            p = p + py * py;
            if (a.dim > 2) p = p + pz * pz;
            pm = sqrt(p);
        }
        u = pm / rho + c;
        u = a.hmin / u;
    } else {
        u = a.hx / (fabs(px) / rho + c);
        double v = a.hy / (fabs(py) / rho + c);
        u = (u < v) ? u : v;
        if (a.dim > 2) {
            v = a.hz / (fabs(pz) / rho + c);
            u = (u < v) ? u : v;
        }
    }
    return u;
}

constexpr double kCflNone = 1e37;  // CFL minimum of a set with no limiting cell

// Order-preserving map of doubles (NaN aside) to unsigned 64-bit keys, so that
// any wave can take a minimum with one integer atomic.
__host__ __device__ inline unsigned long long order_key(double v)
{
    unsigned long long b;
    memcpy(&b, &v, sizeof b);
    return (b >> 63) ? ~b : (b | 0x8000000000000000ull);
}

__device__ __forceinline__ double order_value(unsigned long long k)
{
    const unsigned long long b = (k >> 63) ? (k & 0x7fffffffffffffffull) : ~k;
    return __longlong_as_double((long long)b);
}

// CFL minimum folded into a sweep: each wave takes the minimum time-step limit
// over the cells it stores whose value survives the direction's boundary
// conditions (cells [lo, hi) of the swept direction; the ghost cells the
// boundary then overwrites are copies or mirror images of kept cells, with the
// same limit) into one of kCflSlots keys, which the next CFL reduction reads and
// resets. slots = null: off.
constexpr int kCflSlots = 256;
struct CflFuse {
    unsigned long long *slots;
    CflArgs a;
    int lo, hi;
};

// A wave's minimum into a key, by one lane. The look before the atomic leaves
// out nearly all of them once the first waves have been there: 70 thousand
// waves of an ensemble on 60 keys took 469 us for a sweep of 91 without it.
__device__ __forceinline__ void fold_min(unsigned long long *slot, double cmin)
{
    if (!(cmin < kCflNone)) return;
    const unsigned long long k = order_key(cmin);
    if (k < __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMin(slot, k);
}

// A wave's minimum into one of the slots. All 64 lanes reach it.
__device__ __forceinline__ void cfl_fold(const CflFuse &cf, int64_t wave, double cmin)
{
    cmin = wave_min(cmin);
    if ((threadIdx.x & 63) == 0) fold_min(cf.slots + (wave & (kCflSlots - 1)), cmin);
}

}  // namespace imogen
