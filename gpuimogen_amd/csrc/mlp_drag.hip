// mlp_drag.hip -- learned drag surrogate: BF16 MFMA inference fused into the
// drag source with a per-cell residual check and exact fallback, plus the
// FP32 kernels that train the network on the GPU.
//
// Network 5 -> 64 -> 64 -> 3 with GELU (tanh form). Inference keeps the cells
// of a wave on the N side of the BF16 MFMAs (16 cells per tile; K = 16 for
// layer 1, gfx950's K = 32 for layers 2 and 3) and the hidden units on M/K,
// so a layer's D tiles are, lane for lane, the B operand of the next layer: no
// data moves between layers, the FP32 accumulators only pass through GELU and
// a BF16 rounding. Biases enter as the accumulator's initial value. Weights
// and biases are read from an LDS copy each block makes once; rejected cells
// reach the fallback queue through per-wave LDS batches.
//
// Per cell the surrogate replaces the adaptive integrator of the relaxation
// problem (drag_device.h). With k0 = k(|dv_0|, u_0), tau = dt k0 and the
// analytic initial slope g = d ln k / d tau at tau = 0, the rates along the
// exact path are written k/k0 = 1 + tau (c g + tau r) with c = 1/2 for the
// mean rate kbar and the midpoint rate and c = 1 for the end rate; the network
// predicts the three second-order remainders r (standardised). Cells whose
// features leave the training box use r = 0. The cell is accepted when
//   |dt (k(end state implied by kbar) - predicted end rate)|   and
//   |dt (kbar - Simpson(k0, predicted mid rate, true end rate))|
// are both below the model's residual tolerance, and its features lie inside
// the training box; otherwise that cell runs the adaptive integrator.
#include <cstring>
#include <vector>

#include "cfl_device.h"
#include "drag_device.h"
#include "imogen_internal.h"
#include "sweep_device.h"

namespace imogen {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bfv4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef short bf16x8s __attribute__((ext_vector_type(8)));
typedef __bf16 bfv8 __attribute__((ext_vector_type(8)));

constexpr int kIn = 5, kHid = 64, kOut = 3;
constexpr int kOffW1 = 0, kOffB1 = kIn * kHid, kOffW2 = kOffB1 + kHid, kOffB2 = kOffW2 + kHid * kHid,
              kOffW3 = kOffB2 + kHid, kOffB3 = kOffW3 + kHid * kOut, kNParams = kOffB3 + kOut;
static_assert(kNParams == IMOGEN_MLP_NPARAMS, "parameter layout");

// Device copy of a model: BF16 transposed weights in MFMA A-operand order
// (row = output unit, padded), FP32 biases (padded), and the standardisation.
struct MlpDev {
    const unsigned short *w1t;  // [64][16]
    const unsigned short *w2t;  // [64][64]
    const unsigned short *w3t;  // [16][64]
    const float *b1, *b2, *b3;  // [64], [64], [16]
    DragModelNorm norm;
};

__device__ __forceinline__ unsigned short f2bf(float f)
{
    // round to nearest even
    unsigned u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return 0x7fc0;
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

__device__ __forceinline__ float bf2f(unsigned short b)
{
    return __uint_as_float((unsigned)b << 16);
}

// GELU, tanh form: 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3))), with
// tanh(a) = 1 - 2 / (exp(2a) + 1)
__device__ __forceinline__ float gelu_f(float x)
{
    const float a = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    const float t = 1.0f - 2.0f / (__expf(2.0f * a) + 1.0f);
    return 0.5f * x * (1.0f + t);
}

__device__ __forceinline__ float gelu_grad(float x)
{
    const float a = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    const float t = 1.0f - 2.0f / (__expf(2.0f * a) + 1.0f);
    return 0.5f * (1.0f + t) + 0.5f * x * (1.0f - t * t) * 0.7978845608028654f * (1.0f + 3.0f * 0.044715f * x * x);
}

// Eight BF16 K-values of a 16x16x32 MFMA operand from two 16x16x16 ones:
// elements 0..3 from the lower K-tile, 4..7 from the upper. A and B operands
// are built alike, so each product pairs the same hidden unit whatever K
// index the hardware gives each element.
__device__ __forceinline__ bfv8 cat8(const bf16x4 &a, const bf16x4 &b)
{
    const bf16x8s v = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return __builtin_bit_cast(bfv8, v);
}

__device__ __forceinline__ bf16x4 load_frag(const unsigned short *w, int ld, int row, int col)
{
    const uint2 v = *reinterpret_cast<const uint2 *>(w + (int64_t)row * ld + col);
    bf16x4 r;
    r[0] = (short)(v.x & 0xffff);
    r[1] = (short)(v.x >> 16);
    r[2] = (short)(v.y & 0xffff);
    r[3] = (short)(v.y >> 16);
    return r;
}

// four FP32 values to BF16 (round to nearest even: v_cvt_pk_bf16_f32)
__device__ __forceinline__ bf16x4 to_bf16x4(const f32x4 &v)
{
    return __builtin_bit_cast(bf16x4, __builtin_convertvector(v, bfv4));
}

// Inference GELU: the same tanh form as x * sigmoid(2 sqrt(2/pi) (x + 0.044715 x^3)),
// from the hardware 2^x and reciprocal (about 1 ulp of FP32 each); the result
// is rounded to BF16 right after, 2^-9 relative, far coarser. (A linearly
// interpolated table in LDS took as many VALU issue cycles: more operations,
// fewer transcendentals.)
__device__ __forceinline__ float gelu_fast(float x)
{
    const float c1 = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
    const float c3 = c1 * 0.044715f;
    const float e = __builtin_amdgcn_exp2f(x * fmaf(c3, x * x, c1));
    return x * __builtin_amdgcn_rcpf(1.0f + e);
}

__device__ __forceinline__ bf16x4 act_to_b(const f32x4 &d)
{
    const f32x4 a = {gelu_fast(d[0]), gelu_fast(d[1]), gelu_fast(d[2]), gelu_fast(d[3])};
    return to_bf16x4(a);
}

// One block's LDS copy of the model: the BF16 weights (w1t, w2t, w3t back to
// back, as in the device block) and the biases (b1, b2, b3). Read from LDS,
// the weight fragments of the 96 MFMAs per 64 cells wait tens of cycles
// instead of a global-memory round trip.
struct alignas(16) MlpLds {
    unsigned short w[64 * 16 + 64 * 64 + 16 * 64];
    float b[64 + 64 + 16];
};

// Copies the model into LDS. Every thread of the block must call it (it
// ends with a barrier).
__device__ __forceinline__ void stage_model(MlpLds &L, const MlpDev &m)
{
    const uint4 *src = reinterpret_cast<const uint4 *>(m.w1t);
    uint4 *dst = reinterpret_cast<uint4 *>(L.w);
    constexpr int nw = (int)sizeof(MlpLds::w) / 16;
    for (int k = threadIdx.x; k < nw; k += blockDim.x) dst[k] = src[k];
    for (int k = threadIdx.x; k < 144; k += blockDim.x) L.b[k] = m.b1[k];
    __syncthreads();
}

// Network outputs for the 64 cells of a wave: every lane passes its own
// standardised features f[5] and receives its own outputs. Must be called by
// all 64 lanes together. The weights and biases come from LDS.
__device__ __forceinline__ void mlp_wave(const MlpLds &L, const float (&f)[5], float (&o)[3])
{
    const unsigned short *w1t = L.w, *w2t = L.w + 64 * 16, *w3t = L.w + 64 * 16 + 64 * 64;
    const float *b1 = L.b, *b2 = L.b + 64, *b3 = L.b + 128;
    const int lane = threadIdx.x & 63;
    const int q = lane >> 4;   // which group of 4 K (or M) rows this lane holds
    const int col = lane & 15; // which of the 16 cells of a tile
    float res[4][3];
#pragma unroll
    for (int g = 0; g < 4; g++) {
        // B operand of layer 1: features 4q..4q+3 of cell 16g + col (K padded to 16)
        const int src = 16 * g + col;
        float x[5];
#pragma unroll
        for (int j = 0; j < 5; j++) x[j] = __shfl(f[j], src, 64);
        const f32x4 xf = {q == 0 ? x[0] : (q == 1 ? x[4] : 0.0f), q == 0 ? x[1] : 0.0f, q == 0 ? x[2] : 0.0f,
                          q == 0 ? x[3] : 0.0f};
        const bf16x4 xb = to_bf16x4(xf);
        // layer 1: 4 tiles of 16 hidden units
        bf16x4 h1[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            const int u = 16 * mt + 4 * q;
            f32x4 acc = {b1[u], b1[u + 1], b1[u + 2], b1[u + 3]};
            acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(load_frag(w1t, 16, 16 * mt + col, 4 * q), xb, acc, 0, 0,
                                                           0);
            h1[mt] = act_to_b(acc);
        }
        // layer 2 with gfx950's K = 32 MFMA: hidden tiles 2b and 2b+1 form one
        // K block (B operand: this lane's two D fragments of layer 1, as they
        // are); the four output tiles' accumulators advance together, so
        // consecutive MFMAs never wait on each other's results
        f32x4 acc2[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            const int u = 16 * mt + 4 * q;
            acc2[mt] = f32x4{b2[u], b2[u + 1], b2[u + 2], b2[u + 3]};
        }
#pragma unroll
        for (int b = 0; b < 2; b++) {
            const bfv8 hb = cat8(h1[2 * b], h1[2 * b + 1]);
#pragma unroll
            for (int mt = 0; mt < 4; mt++)
                acc2[mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    cat8(load_frag(w2t, 64, 16 * mt + col, 32 * b + 4 * q),
                         load_frag(w2t, 64, 16 * mt + col, 32 * b + 16 + 4 * q)),
                    hb, acc2[mt], 0, 0, 0);
        }
        bf16x4 h2[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++) h2[mt] = act_to_b(acc2[mt]);
        // layer 3: one tile, outputs 0..2 in rows 0..2 (lanes 0..15)
        f32x4 acc = {b3[4 * q], b3[4 * q + 1], b3[4 * q + 2], b3[4 * q + 3]};
#pragma unroll
        for (int b = 0; b < 2; b++)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                cat8(load_frag(w3t, 64, col, 32 * b + 4 * q), load_frag(w3t, 64, col, 32 * b + 16 + 4 * q)),
                cat8(h2[2 * b], h2[2 * b + 1]), acc, 0, 0, 0);
        res[g][0] = acc[0];
        res[g][1] = acc[1];
        res[g][2] = acc[2];
    }
    // cell `lane` = column lane%16 of group lane/16, held by lane lane%16
    const int g = lane >> 4;
#pragma unroll
    for (int j = 0; j < 3; j++) {
        const float v0 = __shfl(res[0][j], col, 64);
        const float v1 = __shfl(res[1][j], col, 64);
        const float v2 = __shfl(res[2][j], col, 64);
        const float v3 = __shfl(res[3][j], col, 64);
        o[j] = (g == 0) ? v0 : ((g == 1) ? v1 : ((g == 2) ? v2 : v3));
    }
}

// ---------------------------------------------------------------------------
// features of a cell
// ---------------------------------------------------------------------------
struct DragRate {
    double k, Re, Kn;
    double g;    // d ln k / d tau at tau = 0 along the relaxation path
    double lRe;  // ln Re
    double lT;   // ln(alpha u), the rate's temperature logarithm
};

// The surrogate path restates drag_load and drag_apply on register cells, with
// the densities' reciprocals kept between them.

// |dv| and u_0 of a register cell, with 1/rho_g and 1/rho_d
__device__ __forceinline__ DragCell learned_load(const double (&G)[5], const double (&D)[5], double &irg,
                                                 double &ird)
{
    DragCell s;
    s.rg = G[0];
    s.rd = D[0];
    irg = rcp_nr(s.rg);
    ird = rcp_nr(s.rd);
    double dv = G[2] * irg - D[2] * ird;
    double dvsq = dv * dv;
    dv = G[3] * irg - D[3] * ird;
    dvsq += dv * dv;
    dv = G[4] * irg - D[4] * ird;
    dvsq += dv * dv;
    s.s0 = sqrt_nr(dvsq);
    s.u0 = (G[1] - .5 * (G[2] * G[2] + G[3] * G[3] + G[4] * G[4]) * irg) * irg;
    return s;
}

// drag_apply's update about the barycentric velocity (dv scaled by f)
__device__ __forceinline__ void learned_apply(double (&G)[5], double (&D)[5], const DragCell &s, double irg,
                                              double ird, double f)
{
    const double irs = rcp_nr(s.rg + s.rd);
    const double mu = s.rd * irs * s.rg;
    double pdustsq = 0.0;
#pragma unroll
    for (int c = 2; c <= 4; c++) {
        const double pg = G[c], pd = D[c];
        pdustsq -= pd * pd;
        const double vstick = (pg + pd) * irs;
        const double dv_t = (pg * irg - pd * ird) * f;
        G[c] = s.rg * vstick + dv_t * mu;
        const double q = s.rd * vstick - dv_t * mu;
        D[c] = q;
        pdustsq += q * q;
    }
    G[1] -= .5 * pdustsq * ird;
}

// k0, Re0, Kn0 and the initial slope. With k = C_d(Re, Kn) |dv| (rho_g +
// rho_d) eps, Re ~ |dv| T^viscpow, Kn ~ T^lampow, T ~ u, and along the path
// d ln|dv|/d tau = -1, d ln u/d tau = (rho_d/(rho_g+rho_d)) |dv_0|^2/u_0:
//   g = -(1 + a) + (a viscpow + b lampow) rho_d |dv_0|^2 / ((rho_g+rho_d) u_0)
// with a = d ln N/d ln Re, b = -d ln Cu/d ln Kn for C_d = N(Re)/Cu(Kn).
__device__ __forceinline__ DragRate drag_k_parts(const DragConsts &c, const DragPre &pre, double rhog, double rhod,
                                                 double magdv, double u)
{
    DragRate r;
    r.lT = log_fast(c.alpha * u);
    const double lTv = scaled_log(c.viscpow, r.lT);
    r.lRe = pre.ls + log_fast(magdv) + lTv;
    r.Re = pre.dr * magdv * exp_fast(lTv);
    r.Kn = pre.brg * exp_fast(scaled_log(c.lampow, r.lT));
    const double E = cunningham_exp(r.Kn);
    const double cunningham = 1 + r.Kn * (1.142 + 0.558 * E);
    const double p319 = exp_fast(-.319 * r.lRe);
    const double iRe = rcp_nr(r.Re);
    const double q = 8710 + r.Re;
    const double iq = rcp_nr(q);
    const double N = 3 * iRe + .45 * p319 + .0509 * r.Re * iq;
    const double icun = rcp_nr(cunningham);
    r.k = N * icun * magdv * pre.C;
    const double a = (-3 * iRe - .319 * .45 * p319 + .0509 * 8710 * r.Re * iq * iq) * rcp_nr(N);
    const double b = -(1.142 * r.Kn + 0.558 * E * (r.Kn + 0.999)) * icun;
    r.g = -(1.0 + a) + (a * c.viscpow + b * c.lampow) * rhod * magdv * magdv * rcp_nr((rhog + rhod) * u);
    return r;
}

// raw features: ln(dt k0), ln(rho_d/rho_g), ln(|dv|/c_s), ln Re0, ln Kn0
__device__ __forceinline__ void drag_features(const DragConsts &c, const DragCell &s, const DragRate &r, double dt,
                                              float (&f)[5])
{
    f[0] = __logf((float)(dt * r.k));
    f[1] = __logf((float)s.rd) - __logf((float)s.rg);
    f[2] = __logf((float)s.s0) - 0.5f * __logf((float)((c.gm1 + 1.0) * c.gm1 * s.u0));
    f[3] = (float)r.lRe;
    f[4] = __logf((float)r.Kn);
}

// ---------------------------------------------------------------------------
// learned drag source
// ---------------------------------------------------------------------------
// Cells the surrogate does not accept are appended to a queue (one atomic
// per wave) and integrated by the fallback kernels in dense waves, so a few
// rejected lanes do not hold their whole wave in the adaptive integrator.
// A queue entry is qtag | cell index, with kQueueSecond set when the cell
// still owes a second learned call after its exact one (a source's two
// half-interval calls applied in one pass, below).
constexpr int64_t kQueueSecond = (int64_t)1 << 62;
constexpr int64_t kQueueIndex = ((int64_t)1 << 32) - 1;

// One learned drag call on cell s (register copy): features, network,
// residual check. Must be called by all 64 lanes of the wave together (the
// network runs on the wave). ok: the surrogate's factor `fac` is accepted;
// a cell the problem is not defined on is never accepted (the exact
// integrator flags it, drag_exact_ratio).
__device__ __forceinline__ void learned_step(const DragConsts &c, const DragCell &s, double dt, const MlpDev &m,
                                             const MlpLds &Lm, bool &ok, double &fac)
{
    const bool defined = drag_cell_defined(s.rg, s.rd, s.s0, s.u0);
    const bool moving = defined && s.s0 >= 1e-9;
    DragRate r0 = {0.0, 1.0, 1.0, 0.0};
    DragPre pre = {0.0, 0.0, 0.0, 0.0};
    if (moving) {
        pre = drag_pre(c, s.rg, s.rd);
        r0 = drag_k_parts(c, pre, s.rg, s.rd, s.s0, s.u0);
    }
    float f[5];
    drag_features(c, s, r0, dt, f);
    bool inside = moving;
    float z[5];
#pragma unroll
    for (int j = 0; j < 5; j++) {
        inside = inside && (f[j] >= m.norm.flo[j]) && (f[j] <= m.norm.fhi[j]);
        z[j] = inside ? (f[j] - m.norm.fmean[j]) / m.norm.fstd[j] : 0.0f;
    }
    float o[3];
    mlp_wave(Lm, z, o);
    fac = 1.0;
    ok = defined;  // a cell below the rate's |dv| cut-off stays as it is
    if (moving) {
        const double tau = dt * r0.k;
        const double q0 = inside ? (double)(o[0] * m.norm.tstd[0] + m.norm.tmean[0]) : 0.0;
        const double q1 = inside ? (double)(o[1] * m.norm.tstd[1] + m.norm.tmean[1]) : 0.0;
        const double q2 = inside ? (double)(o[2] * m.norm.tstd[2] + m.norm.tmean[2]) : 0.0;
        const double kbar = r0.k * (1.0 + tau * (.5 * r0.g + tau * q0));
        const double kmid = r0.k * (1.0 + tau * (.5 * r0.g + tau * q1));
        const double kend = r0.k * (1.0 + tau * (r0.g + tau * q2));
        // end state implied by kbar; its true rate checks the prediction
        const double x = kbar * dt;
        fac = exp_decay(-x);
        const double s1 = s.s0 * fac;
        const double u1 = s.u0 + .5 * s.rd * rcp_nr(s.rg + s.rd) * (s.s0 * s.s0 - s1 * s1);
        // ln Re follows the decay: ln(delta rho_g s1) = ln Re0 - viscpow ln T0 - x
        const double k1 = drag_rate(c, pre, s1, r0.lRe - scaled_log(c.viscpow, r0.lT) - x, u1);
        const double ksimp = (r0.k + 4.0 * kmid + k1) * (1.0 / 6.0);
        const double e1 = fabs(dt * (k1 - kend));
        const double e2 = fabs(dt * (kbar - ksimp));
        ok = (e1 <= m.norm.residTol) && (e2 <= m.norm.residTol) && kbar > 0.0;
        if (!ok) fac = 1.0;
    }
}

// The nine values a drag call reads and writes, as a pitch-1 cell (the dust
// energy is neither read nor written: D[1] stays 0).
__device__ __forceinline__ void cell_in(const double *g, const double *d, int64_t pitch, double (&G)[5],
                                        double (&D)[5])
{
#pragma unroll
    for (int k = 0; k < 5; k++) G[k] = g[k * pitch];
    D[0] = d[0];
    D[1] = 0.0;
#pragma unroll
    for (int k = 2; k < 5; k++) D[k] = d[k * pitch];
}

__device__ __forceinline__ void cell_out(double *g, double *d, int64_t pitch, const double (&G)[5],
                                         const double (&D)[5])
{
    g[pitch] = G[1];
#pragma unroll
    for (int k = 2; k < 5; k++) {
        g[k * pitch] = G[k];
        d[k * pitch] = D[k];
    }
}

// One learned drag call on a register cell, applied when accepted. Not
// inlined: the learned and the fallback kernels run these very instructions,
// so a call gives bitwise the same result whichever kernel takes it (copies
// inlined into different code can contract their FMAs differently). Must be
// called by all 64 lanes of the wave together.
__device__ __forceinline__ bool learned_call(double (&G)[5], double (&D)[5], const DragConsts &c,
                                                       double dt, const MlpDev &m, const MlpLds &Lm)
{
    double irg, ird;
    const DragCell s = learned_load(G, D, irg, ird);
    bool ok;
    double fac;
    learned_step(c, s, dt, m, Lm, ok, fac);
    if (ok) learned_apply(G, D, s, irg, ird, fac);
    return ok;
}

// One exact (adaptive integrator) drag call on a register cell; counts
// invalid cells and budget overruns when `count`. Not inlined, as learned_call.
__device__ __forceinline__ void exact_call(double (&G)[5], double (&D)[5], const DragConsts &c,
                                                     double dt, bool count, unsigned &invalid, unsigned &overrun)
{
    const DragCell s = drag_load(G, D, 1);
    int steps;
    const double fac = drag_exact_ratio(c, s.rg, s.rd, s.s0, s.u0, dt, &steps);
    if (count) {
        invalid += (steps == kDragInvalid);
        overrun += (steps < 0 && steps != kDragInvalid);
    }
    drag_apply(G, D, 1, s, fac);
}

// Rejected cells are collected per wave in LDS and appended to the global
// fallback queue in batches: one atomic per batch of up to kWaveQueue entries
// instead of one per wave of cells (a single counter that every wave hits
// serialises the waves on the atomic's round trip).
constexpr int kWaveQueue = 448;

struct WaveQueue {
    int64_t *buf;  // this wave's kWaveQueue LDS entries
    int count;     // entries held (wave-uniform)
};

__device__ __forceinline__ void wq_flush(WaveQueue &w, int64_t *__restrict__ queue,
                                         unsigned long long *__restrict__ qcount)
{
    if (w.count == 0) return;
    const int lane = threadIdx.x & 63;
    unsigned long long slot = 0;
    if (lane == 0) slot = atomicAdd(qcount, (unsigned long long)w.count);
    slot = __shfl(slot, 0, 64);
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // other lanes' LDS entries
    for (int k = lane; k < w.count; k += 64) queue[slot + k] = w.buf[k];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // read before the buffer is reused
    w.count = 0;
}

__device__ __forceinline__ void wq_push(WaveQueue &w, bool reject, int64_t tag, int64_t *__restrict__ queue,
                                        unsigned long long *__restrict__ qcount)
{
    const unsigned long long mask = __ballot(reject);
    if (!mask) return;
    const int n = __popcll(mask);
    if (w.count + n > kWaveQueue) wq_flush(w, queue, qcount);
    const int lane = threadIdx.x & 63;
    if (reject) w.buf[w.count + __popcll(mask & ((1ull << lane) - 1ull))] = tag;
    w.count += n;
}

// One wave of learned drag calls: lane cells i (live lanes; the others work
// on cell ic and store nothing). `calls` (1 or 2) calls of dt each are taken
// in registers. A cell that one call does not accept is stored as the
// accepted calls left it and queued: the fallback kernel integrates the
// rejected call exactly and, when the cell's first call was the rejected one
// (kQueueSecond), lists the cell for a second pass of this kernel (list
// mode) that takes its second call, so every call of every cell runs the same
// instructions as in two separate launches and gives the same result.
__device__ __forceinline__ void learned_cells(double *__restrict__ g, double *__restrict__ d, int64_t pitch,
                                              int64_t i, int64_t ic, bool live, const DragConsts &c, double dt,
                                              const MlpDev &m, const MlpLds &Lm, WaveQueue &wq,
                                              int64_t *__restrict__ queue, unsigned long long *__restrict__ qcount,
                                              int64_t qtag, int calls)
{
    double G[5], D[5];
    cell_in(g + ic, d + ic, pitch, G, D);
    int done = 0;  // calls accepted before the first rejection
    bool rejected = false;
#pragma unroll 1
    for (int r = 0; r < calls; r++) {
        // a rejected lane's copy is left as it was: the call only keeps the
        // wave together for the network
        double G2[5], D2[5];
#pragma unroll
        for (int k = 0; k < 5; k++) {
            G2[k] = G[k];
            D2[k] = D[k];
        }
        const bool ok = learned_call(G2, D2, c, dt, m, Lm);
        if (!rejected) {
            if (ok) {
#pragma unroll
                for (int k = 0; k < 5; k++) {
                    G[k] = G2[k];
                    D[k] = D2[k];
                }
                done++;
            } else {
                rejected = true;
            }
        }
    }
    const bool reject = live && rejected;
    wq_push(wq, reject, qtag | i | ((done == 0 && calls == 2) ? kQueueSecond : 0), queue, qcount);
    if (live && done > 0) cell_out(g + i, d + i, pitch, G, D);
}

// The exact call of one queued cell; returns whether the cell is listed for
// a learned second call.
__device__ __forceinline__ void fallback_cell(double *gi, double *di, int64_t pitch, bool live, const DragConsts &c,
                                              double dt, unsigned &invalid, unsigned &overrun)
{
    double G[5], D[5];
    cell_in(gi, di, pitch, G, D);
    exact_call(G, D, c, dt, live, invalid, overrun);
    if (live) cell_out(gi, di, pitch, G, D);
}

// Appends the live lanes' entries to a global list (one atomic per wave).
__device__ __forceinline__ void wave_append(bool put, int64_t v, int64_t *__restrict__ list,
                                            unsigned long long *__restrict__ count)
{
    const unsigned long long mask = __ballot(put);
    if (!mask) return;
    const int lane = threadIdx.x & 63;
    unsigned long long slot = 0;
    if (lane == 0) slot = atomicAdd(count, (unsigned long long)__popcll(mask));
    slot = __shfl(slot, 0, 64);
    if (put) list[slot + __popcll(mask & ((1ull << lane) - 1ull))] = v;
}

// Dense mode (list null): cells [0, n). List mode: the *listCount cells of
// list (every entry valid).
__global__ __launch_bounds__(256, 2) void learned_drag_kernel(double *__restrict__ g, double *__restrict__ d,
                                                              int64_t pitch, int64_t n, DragConsts c, DragDt dtv,
                                                              MlpDev m, int calls, int64_t *__restrict__ queue,
                                                              unsigned long long *__restrict__ qcount,
                                                              const int64_t *__restrict__ list,
                                                              const unsigned long long *__restrict__ listCount)
{
    __shared__ MlpLds Lm;
    __shared__ int64_t qbuf[4][kWaveQueue];
    stage_model(Lm, m);
    WaveQueue wq{qbuf[threadIdx.x >> 6], 0};
    const double dt = drag_dt(dtv);
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    const int64_t total = list ? (int64_t)*listCount : n;
    for (int64_t base = wave * 64; base < total; base += nwaves * 64) {
        const int64_t t = base + lane;
        const bool live = t < total;
        int64_t i, ic;
        if (list) {
            i = list[live ? t : base];
            ic = i;
        } else {
            i = t;
            ic = live ? t : n - 1;
        }
        learned_cells(g, d, pitch, i, ic, live, c, dt, m, Lm, wq, queue, qcount, 0, calls);
    }
    wq_flush(wq, queue, qcount);
}

// Exact integration of the queued cells in dense waves. cells: the calls'
// cell count to add to counts[0]; entries marked kQueueSecond are appended to
// listOut for the learned second call.
__global__ __launch_bounds__(256) void fallback_drag_kernel(double *__restrict__ g, double *__restrict__ d,
                                                            int64_t pitch, int64_t cells, DragConsts c, DragDt dtv,
                                                            const int64_t *__restrict__ queue,
                                                            const unsigned long long *__restrict__ qcount,
                                                            unsigned long long *__restrict__ counts,
                                                            unsigned long long *__restrict__ err,
                                                            int64_t *__restrict__ listOut,
                                                            unsigned long long *__restrict__ listCount)
{
    const double dt = drag_dt(dtv);
    const unsigned long long nq = *qcount;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (cells) atomicAdd(counts, (unsigned long long)cells);
        if (nq) atomicAdd(counts + 1, nq);
    }
    unsigned invalid = 0, overrun = 0;
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (unsigned long long base = (unsigned long long)wave * 64; base < nq; base += (unsigned long long)nwaves * 64) {
        const unsigned long long t = base + lane;
        const bool live = t < nq;
        const int64_t e = queue[live ? t : base];
        const int64_t i = e & ~kQueueSecond;
        fallback_cell(g + i, d + i, pitch, live, c, dt, invalid, overrun);
        if (listOut) wave_append(live && (e & kQueueSecond), i, listOut, listCount);
    }
    wave_count(err + ERRW_DRAG_INVALID, invalid);
    wave_count(err + ERRW_DRAG_BUDGET, overrun);
}

__global__ void zero_counters(unsigned long long *p, int n)
{
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0;
}

// ---------------------------------------------------------------------------
// drag over the dusty problems of an ensemble: persistent waves over 64-cell
// items, dt = frac * dTime of the item's problem (read on the device), `calls`
// (1 or 2) calls of dt each applied in one pass
// ---------------------------------------------------------------------------
// Learned list mode (list not null): the *listCount queue entries of list
// ((table entry << 32) | cell, every entry valid), one call each; the lanes of
// a wave may then belong to different problems. Both modes run the same
// learned_cells code.
template <bool LEARNED>
__global__ __launch_bounds__(256, 2) void ens_drag_kernel(const EnsDragTable *__restrict__ tab,
                                                          const EnsDragItem *__restrict__ items, int nitems,
                                                          const double *__restrict__ dtp, double frac, DragConsts c,
                                                          int method, int calls, MlpDev m,
                                                          int64_t *__restrict__ queue,
                                                          unsigned long long *__restrict__ qcount,
                                                          unsigned long long *__restrict__ err,
                                                          const int64_t *__restrict__ list,
                                                          const unsigned long long *__restrict__ listCount)
{
    __shared__ MlpLds Lm;
    __shared__ int64_t qbuf[LEARNED ? 4 : 1][LEARNED ? kWaveQueue : 1];
    if (LEARNED) stage_model(Lm, m);
    WaveQueue wq{qbuf[LEARNED ? threadIdx.x >> 6 : 0], 0};
    const int lane = threadIdx.x & 63;
    const int wave0 = (int)(((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int nwaves = (int)(((int64_t)gridDim.x * blockDim.x) >> 6);
    unsigned invalid = 0, overrun = 0;
    if (LEARNED) {
        const int64_t total = list ? (int64_t)*listCount : (int64_t)nitems * 64;
        for (int64_t base = (int64_t)wave0 * 64; base < total; base += (int64_t)nwaves * 64) {
            int tt;
            int64_t i;
            bool live;
            if (list) {
                const int64_t t = base + lane;
                live = t < total;
                const int64_t e = list[live ? t : base];
                tt = (int)(e >> 32);
                i = e & kQueueIndex;
            } else {
                const EnsDragItem it = items[base >> 6];
                tt = it.t;
                i = it.base + lane;
                live = i < tab[tt].n;
            }
            const EnsDragTable T = tab[tt];
            learned_cells(T.g, T.d, T.pitch, i, live ? i : T.n - 1, live, c, frac * dtp[T.p], m, Lm, wq, queue,
                          qcount, (int64_t)tt << 32, list ? 1 : calls);
        }
        wq_flush(wq, queue, qcount);
        return;
    }
    for (int wave = wave0; wave < nitems; wave += nwaves) {
        const EnsDragItem it = items[wave];
        const EnsDragTable T = tab[it.t];
        const double dt = frac * dtp[T.p];
        const int64_t i = it.base + lane;
        if (i >= T.n) continue;
        double G[5], D[5];
        cell_in(T.g + i, T.d + i, T.pitch, G, D);
        for (int r = 0; r < calls; r++) {
            const DragCell s = drag_load(G, D, 1);
            double f;
            if (method == DRAG_EXACT) {
                int k;
                f = drag_exact_ratio(c, s.rg, s.rd, s.s0, s.u0, dt, &k);
                invalid += (k == kDragInvalid);
                overrun += (k < 0 && k != kDragInvalid);
            } else {
                invalid += !drag_cell_defined(s.rg, s.rd, s.s0, s.u0);
                f = exp_decay(-dt * drag_logtrap_rate(c, s.rg, s.rd, s.s0, s.u0, dt, method == DRAG_LOGTRAP3 ? 3 : 2));
            }
            drag_apply(G, D, 1, s, f);
        }
        cell_out(T.g + i, T.d + i, T.pitch, G, D);
    }
    wave_count(err + ERRW_DRAG_INVALID, invalid);
    wave_count(err + ERRW_DRAG_BUDGET, overrun);
}

// Exact integration of the queued calls; entries marked kQueueSecond are
// appended to listOut for the learned second call (listOut null: none are).
__global__ __launch_bounds__(256) void ens_fallback_kernel(const EnsDragTable *__restrict__ tab,
                                                           const double *__restrict__ dtp, double frac, DragConsts c,
                                                           const int64_t *__restrict__ queue,
                                                           const unsigned long long *__restrict__ qcount,
                                                           int64_t cells, unsigned long long *__restrict__ counts,
                                                           unsigned long long *__restrict__ err,
                                                           int64_t *__restrict__ listOut,
                                                           unsigned long long *__restrict__ listCount)
{
    const unsigned long long nq = *qcount;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (cells) atomicAdd(counts, (unsigned long long)cells);
        if (nq) atomicAdd(counts + 1, nq);
    }
    unsigned invalid = 0, overrun = 0;
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (unsigned long long base = (unsigned long long)wave * 64; base < nq; base += (unsigned long long)nwaves * 64) {
        const unsigned long long t = base + lane;
        const bool live = t < nq;
        const int64_t e = queue[live ? t : base];
        const EnsDragTable T = tab[(int)((e & ~kQueueSecond) >> 32)];
        const int64_t i = e & kQueueIndex;
        fallback_cell(T.g + i, T.d + i, T.pitch, live, c, frac * dtp[T.p], invalid, overrun);
        if (listOut) wave_append(live && (e & kQueueSecond), e & ~kQueueSecond, listOut, listCount);
    }
    wave_count(err + ERRW_DRAG_INVALID, invalid);
    wave_count(err + ERRW_DRAG_BUDGET, overrun);
}

// standalone BF16 inference (tests)
__global__ __launch_bounds__(256) void mlp_infer_kernel(int64_t batch, const float *__restrict__ x,
                                                        float *__restrict__ y, MlpDev m)
{
    __shared__ MlpLds Lm;
    stage_model(Lm, m);
    const int lane = threadIdx.x & 63;
    const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (int64_t base = wave * 64; base < batch; base += nwaves * 64) {
        const int64_t i = base + lane;
        const int64_t ic = i < batch ? i : batch - 1;
        float f[5], o[3];
#pragma unroll
        for (int j = 0; j < 5; j++) f[j] = x[ic * 5 + j];
        mlp_wave(Lm, f, o);
        if (i < batch) {
#pragma unroll
            for (int j = 0; j < 3; j++) y[i * 3 + j] = o[j];
        }
    }
}

// ---------------------------------------------------------------------------
// training set from the exact integrator
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void drag_samples_kernel(int64_t n, const double *__restrict__ cells, DragConsts c,
                                                           float *__restrict__ feat, float *__restrict__ targ)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        DragCell s;
        s.rg = cells[i * 5 + 0];
        s.rd = cells[i * 5 + 1];
        s.s0 = cells[i * 5 + 2];
        s.u0 = cells[i * 5 + 3];
        const double tau_in = cells[i * 5 + 4];
        float f[5];
        float t[3];
        const DragRate r0 = (s.s0 < 1e-9) ? DragRate{0.0, 1.0, 1.0, 0.0}
                                               : drag_k_parts(c, drag_pre(c, s.rg, s.rd), s.rg, s.rd, s.s0, s.u0);
        const double dt = (r0.k > 0.0) ? tau_in / r0.k : 0.0;
        if (s.s0 < 1e-9 || !(dt > 0)) {
#pragma unroll
            for (int j = 0; j < 5; j++) f[j] = __int_as_float(0x7fc00000);
            t[0] = t[1] = t[2] = __int_as_float(0x7fc00000);
        } else {
            drag_features(c, s, r0, dt, f);
            int st;
            const double hc = .5 * s.rd / (s.rg + s.rd);
            const double rend = drag_exact_ratio(c, s.rg, s.rd, s.s0, s.u0, dt, &st);
            const double rmid = drag_exact_ratio(c, s.rg, s.rd, s.s0, s.u0, .5 * dt, &st);
            const double smid = s.s0 * rmid, send = s.s0 * rend;
            const double kmid = drag_k(c, s.rg, s.rd, smid, s.u0 + hc * (s.s0 * s.s0 - smid * smid));
            const double kend = drag_k(c, s.rg, s.rd, send, s.u0 + hc * (s.s0 * s.s0 - send * send));
            const double kbar = -log(rend) / dt;
            const double tau = dt * r0.k;
            t[0] = (float)(((kbar / r0.k - 1.0) / tau - .5 * r0.g) / tau);
            t[1] = (float)(((kmid / r0.k - 1.0) / tau - .5 * r0.g) / tau);
            t[2] = (float)(((kend / r0.k - 1.0) / tau - r0.g) / tau);
        }
#pragma unroll
        for (int j = 0; j < 5; j++) feat[i * 5 + j] = f[j];
#pragma unroll
        for (int j = 0; j < 3; j++) targ[i * 3 + j] = t[j];
    }
}

// ---------------------------------------------------------------------------
// FP32 training kernels, blocks of 256 threads
// ---------------------------------------------------------------------------
// The 64 x 64 products run on the FP32 MFMA (16x16x4, FP32 operands and
// accumulation), every sum one accumulator in the order of a plain loop over
// its terms (step i, lane group q = lane / 16 holds term 4 i + q). The forward
// pass takes 16 rows per block, wave w the hidden units 16 w .. 16 w + 15; the
// backward one 64 rows and 16 hidden units, four blocks per row group, so a
// batch of 2048 makes 128 blocks of each (64 rows per block in VALU loops over
// global activations: 32 blocks, forward 20 us and backward 126 us at that
// batch, now 5 and 8). The launches are bound by their latency, not by the
// 0.06 GFLOP.
constexpr int kRows = 16;        // rows of a forward block
constexpr int kBwdRows = 64;     // rows of a backward group: one partial gradient each
constexpr int kPadH = kHid + 4;  // LDS row of hidden units

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // four floats of a caller's buffer

__device__ __forceinline__ f32x4 mfma_f32(float a, float b, f32x4 c)
{
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__global__ __launch_bounds__(256) void mlp_fwd_kernel(const float *__restrict__ P, int64_t batch,
                                                      const float *__restrict__ x, float *__restrict__ act,
                                                      float *__restrict__ y)
{
    __shared__ float H[kRows][kPadH];
    __shared__ float H2[kRows][kPadH];
    __shared__ float W3[kHid * kOut];
    const int t = threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.x * kRows;
    const int lane = t & 63, w = t >> 6, q = lane >> 4, n = lane & 15;
    // W2's column 16 w + n at rows 4 i + q
    float b[16];
#pragma unroll
    for (int i = 0; i < 16; i++) b[i] = P[kOffW2 + (4 * i + q) * kHid + 16 * w + n];
    const float b2 = P[kOffB2 + 16 * w + n];
    if (t < kHid * kOut) W3[t] = P[kOffW3 + t];
    const int r = t >> 4;         // row of layer 1
    const int j0 = (t & 15) * 4;  // its 4 hidden units
    const int64_t row = r0 + r;
    float xv[kIn];
#pragma unroll
    for (int k = 0; k < kIn; k++) xv[k] = row < batch ? x[row * kIn + k] : 0.0f;
    float z[4], h[4];
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
        z[jj] = P[kOffB1 + j0 + jj];
#pragma unroll
        for (int k = 0; k < kIn; k++) z[jj] += xv[k] * P[kOffW1 + k * kHid + j0 + jj];
        h[jj] = gelu_f(z[jj]);
        H[r][j0 + jj] = h[jj];
    }
    if (row < batch) {
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            act[row * 256 + j0 + jj] = z[jj];
            act[row * 256 + 64 + j0 + jj] = h[jj];
        }
    }
    __syncthreads();
    f32x4 d = {b2, b2, b2, b2};
#pragma unroll
    for (int i = 0; i < 16; i++) d = mfma_f32(H[n][4 * i + q], b[i], d);
#pragma unroll
    for (int i = 0; i < 4; i++) {  // D: row 4 q + i, column n
        const int rr = 4 * q + i;
        const float h2 = gelu_f(d[i]);
        H2[rr][16 * w + n] = h2;
        if (r0 + rr < batch) {
            act[(r0 + rr) * 256 + 128 + 16 * w + n] = d[i];
            act[(r0 + rr) * 256 + 192 + 16 * w + n] = h2;
        }
    }
    __syncthreads();
    if (t < kRows * kOut) {
        const int rr = t / kOut, o = t % kOut;
        float v = P[kOffB3 + o];
#pragma unroll 16
        for (int k = 0; k < kHid; k++) v += H2[rr][k] * W3[k * kOut + o];
        if (r0 + rr < batch) y[(r0 + rr) * kOut + o] = v;
    }
}

// Gradient partials per group of 64 rows (deterministic); added up by
// mlp_grad_reduce. Block (group, c) forms those of hidden units 16 c ..
// 16 c + 15 (rows of W2 and W3, columns of W1).
__global__ __launch_bounds__(256) void mlp_bwd_kernel(const float *__restrict__ P, int64_t batch,
                                                      const float *__restrict__ x, const float *__restrict__ act,
                                                      const float *__restrict__ dy, float *__restrict__ part)
{
    __shared__ alignas(16) float DZ2[kBwdRows][kPadH];
    __shared__ alignas(16) float W2[16][kPadH];      // rows 16 c ..
    __shared__ alignas(16) float H1[kBwdRows][20], H2[kBwdRows][20], DZ1[kBwdRows][20];  // units 16 c ..
    __shared__ float DY[kBwdRows][kOut], X[kBwdRows][kIn];
    const int t = threadIdx.x, c = blockIdx.y;
    const int lane = t & 63, w = t >> 6, q = lane >> 4, n = lane & 15;
    const int64_t r0 = (int64_t)blockIdx.x * kBwdRows;
    const int r = t >> 2, j0 = (t & 3) * 16, u0 = (t & 3) * 4;
    const int64_t row = r0 + r;
    const bool live = row < batch;
    // rows past the batch: zero activations and zero gradients
    const float *ar = act + (live ? row : 0) * 256;
    f32x4 z2[4];
#pragma unroll
    for (int k = 0; k < 4; k++) z2[k] = *reinterpret_cast<const f32x4u *>(ar + 128 + j0 + 4 * k);
    const f32x4 z1 = *reinterpret_cast<const f32x4u *>(ar + 16 * c + u0);
    f32x4 h1 = *reinterpret_cast<const f32x4u *>(ar + 64 + 16 * c + u0);
    f32x4 h2 = *reinterpret_cast<const f32x4u *>(ar + 192 + 16 * c + u0);
    if (!live) h1 = h2 = f32x4{0, 0, 0, 0};
    *reinterpret_cast<f32x4 *>(&W2[t >> 4][(t & 15) * 4]) =
        *reinterpret_cast<const f32x4u *>(P + kOffW2 + (16 * c + (t >> 4)) * kHid + (t & 15) * 4);
    if (t < kBwdRows * kOut) (&DY[0][0])[t] = (r0 * kOut + t < batch * kOut) ? dy[r0 * kOut + t] : 0.0f;
    for (int k = t; k < kBwdRows * kIn; k += 256) (&X[0][0])[k] = (r0 * kIn + k < batch * kIn) ? x[r0 * kIn + k] : 0.0f;
    *reinterpret_cast<f32x4 *>(&H1[r][u0]) = h1;
    *reinterpret_cast<f32x4 *>(&H2[r][u0]) = h2;
    __syncthreads();
    // dz2 = (dy W3^T) * gelu'(z2), all 64 units
#pragma unroll
    for (int jj = 0; jj < 16; jj++) {
        const int j = j0 + jj;
        float dh = 0.0f;
#pragma unroll
        for (int o = 0; o < kOut; o++) dh += DY[r][o] * P[kOffW3 + j * kOut + o];
        DZ2[r][j] = live ? dh * gelu_grad(z2[jj >> 2][jj & 3]) : 0.0f;
    }
#pragma unroll
    for (int jj = 0; jj < 4; jj++) DZ1[r][u0 + jj] = live ? gelu_grad(z1[jj]) : 0.0f;
    __syncthreads();
    // dz1 = (dz2 W2^T) * gelu'(z1): wave w's rows 16 w .., columns the block's units
    f32x4 d = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) d = mfma_f32(DZ2[16 * w + n][4 * i + q], W2[n][4 * i + q], d);
    // dW2 = h1^T dz2: rows the block's units, wave w's columns 16 w ..
    f32x4 g = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 16; i++) g = mfma_f32(H1[4 * i + q][n], DZ2[4 * i + q][16 * w + n], g);
#pragma unroll
    for (int i = 0; i < 4; i++) DZ1[16 * w + 4 * q + i][n] *= d[i];
    float *pp = part + (int64_t)blockIdx.x * kNParams;
#pragma unroll
    for (int i = 0; i < 4; i++) pp[kOffW2 + (16 * c + 4 * q + i) * kHid + 16 * w + n] = g[i];
    __syncthreads();
    // the rest, one output per thread: dW1 (80), db1, db2 (16 each), dW3 (48), db3 (3, by c = 0)
    float s = 0.0f;
    int out = -1;
    if (t < 80) {
        const int k = t >> 4, u = t & 15;
        for (int rr = 0; rr < kBwdRows; rr++) s += X[rr][k] * DZ1[rr][u];
        out = kOffW1 + k * kHid + 16 * c + u;
    } else if (t < 96) {
        for (int rr = 0; rr < kBwdRows; rr++) s += DZ1[rr][t - 80];
        out = kOffB1 + 16 * c + t - 80;
    } else if (t >= 128 && t < 144) {
        for (int rr = 0; rr < kBwdRows; rr++) s += DZ2[rr][16 * c + t - 128];
        out = kOffB2 + 16 * c + t - 128;
    } else if (t >= 144 && t < 147 && c == 0) {
        for (int rr = 0; rr < kBwdRows; rr++) s += DY[rr][t - 144];
        out = kOffB3 + t - 144;
    } else if (t >= 192 && t < 240) {
        const int k = (t - 192) / kOut, o = (t - 192) % kOut;
        for (int rr = 0; rr < kBwdRows; rr++) s += H2[rr][k] * DY[rr][o];
        out = kOffW3 + (16 * c + k) * kOut + o;
    }
    if (out >= 0) pp[out] = s;
}

// 64 parameters per block: its 16 waves load the partials side by side, the
// first adds them in group order (a thread per parameter loading them one
// after another: 8.6 us at 32 of them)
constexpr int kReduceChunk = 128;
__global__ __launch_bounds__(1024) void mlp_grad_reduce(const float *__restrict__ part, int nblocks,
                                                        float *__restrict__ grads)
{
    __shared__ float S[kReduceChunk][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int e = blockIdx.x * 64 + lane;
    float s = 0.0f;
    for (int b0 = 0; b0 < nblocks; b0 += kReduceChunk) {
        const int m = nblocks - b0 < kReduceChunk ? nblocks - b0 : kReduceChunk;
        if (e < kNParams)
            for (int b = w; b < m; b += 16) S[b][lane] = part[(int64_t)(b0 + b) * kNParams + e];
        __syncthreads();
        if (w == 0 && e < kNParams)
            for (int b = 0; b < m; b++) s += S[b][lane];
        __syncthreads();
    }
    if (w == 0 && e < kNParams) grads[e] = s;
}

__global__ __launch_bounds__(256) void mlp_adam_kernel(float *__restrict__ p, const float *__restrict__ gr,
                                                       float *__restrict__ m, float *__restrict__ v, int64_t n,
                                                       float lr, float b1, float b2, float eps, float c1, float c2)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gr[i];
    const float mi = b1 * m[i] + (1.0f - b1) * g;
    const float vi = b2 * v[i] + (1.0f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

__global__ __launch_bounds__(256) void mlp_mse_grad_kernel(int64_t n, const float *__restrict__ y,
                                                           const float *__restrict__ t, float *__restrict__ dy,
                                                           float scale, double *__restrict__ loss)
{
    double acc = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float e = y[i] - t[i];
        dy[i] = 2.0f * scale * e;
        acc += (double)e * (double)e;
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
    if ((threadIdx.x & 63) == 0 && acc != 0.0) atomicAdd(loss, acc * (double)scale);
}

__global__ __launch_bounds__(256) void gather_rows_kernel(const float *__restrict__ src,
                                                          const int64_t *__restrict__ idx, int64_t nrows, int ncols,
                                                          float *__restrict__ dst)
{
    const int64_t total = nrows * ncols;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e / ncols;
        const int c = (int)(e - r * ncols);
        dst[e] = src[idx[r] * ncols + c];
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
struct HostModel {
    void *buf = nullptr;  // device: w1t | w2t | w3t | b1 | b2 | b3
    MlpDev dev{};
    bool loaded = false;
    unsigned long long *counts = nullptr;  // device [learned cells, fallbacks, queue length, unused]
};
static HostModel g_model;
static uint64_t g_modelGeneration = 0;  // bumped by every imogen_drag_set_model

static int ensure_counts()
{
    if (g_model.counts) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    if (IM_HIP(hipMalloc(&g_model.counts, 8 * sizeof(unsigned long long)))) return ERROR_CUDA_BLEW_UP;
    if (IM_HIP(hipMemsetAsync(g_model.counts, 0, 8 * sizeof(unsigned long long), st->stream)))
        return ERROR_CUDA_BLEW_UP;
    return IM_HIP(hipStreamSynchronize(st->stream));
}

// counts: [0] cells, [1] fallbacks (imogen_drag_learned_stats), [2] queue
// length, [3] second-call list length, [4] the second pass's queue length.
// Two calls: learned (both calls) -> fallback (exact; first-call rejections
// listed) -> learned over the list (second call) -> fallback.
int launch_learned_drag(double *g, double *d, int64_t pitch, int64_t n, const DragConsts &c, DragDt dt,
                        int64_t *queue, hipStream_t s, int calls)
{
    if (calls < 1 || calls > 2) return IM_FAIL(ERROR_INVALID_ARGS, "drag calls per pass: %d", calls);
    if (!g_model.loaded) return IM_FAIL(ERROR_INVALID_ARGS, "learned drag: no model (imogen_drag_set_model)");
    if (ensure_counts()) return ERROR_CUDA_BLEW_UP;
    if (queue && calls == 2) return IM_FAIL(ERROR_INVALID_ARGS, "a caller's queue serves one call per pass");
    int64_t waves = (n + 63) / 64;
    if (waves > 8192) waves = 8192;
    const int64_t blocks = (waves + 3) / 4;
    if (!queue) queue = (int64_t *)scratch_block((size_t)n * calls * sizeof(int64_t));
    if (!queue) return IM_FAIL(ERROR_NOMEM, "no scratch for the drag fallback queue");
    int64_t *list = calls == 2 ? queue + n : nullptr;
    unsigned long long *cnt = g_model.counts;
    unsigned long long *err = state()->err;
    const int slot = prof_begin(PROF_MLP, s);
    hipLaunchKernelGGL(zero_counters, dim3(1), dim3(64), 0, s, cnt + 2, 3);
    int rc = IM_LAUNCHED("zero_counters");
    if (rc) return rc;
    hipLaunchKernelGGL(learned_drag_kernel, dim3((unsigned)blocks), dim3(256), 0, s, g, d, pitch, n, c, dt,
                       g_model.dev, calls, queue, cnt + 2, (const int64_t *)nullptr,
                       (const unsigned long long *)nullptr);
    if ((rc = IM_LAUNCHED("learned_drag_kernel"))) return rc;
    hipLaunchKernelGGL(fallback_drag_kernel, dim3(1024), dim3(256), 0, s, g, d, pitch, n * calls, c, dt, queue,
                       cnt + 2, cnt, err, list, cnt + 3);
    if ((rc = IM_LAUNCHED("fallback_drag_kernel"))) return rc;
    if (calls == 2) {
        hipLaunchKernelGGL(learned_drag_kernel, dim3(256), dim3(256), 0, s, g, d, pitch, n, c, dt, g_model.dev, 1,
                           queue, cnt + 4, (const int64_t *)list, (const unsigned long long *)(cnt + 3));
        if ((rc = IM_LAUNCHED("learned_drag_kernel"))) return rc;
        hipLaunchKernelGGL(fallback_drag_kernel, dim3(1024), dim3(256), 0, s, g, d, pitch, (int64_t)0, c, dt, queue,
                           cnt + 4, cnt, err, (int64_t *)nullptr, (unsigned long long *)nullptr);
        if ((rc = IM_LAUNCHED("fallback_drag_kernel"))) return rc;
    }
    prof_end(slot, s);
    return SUCCESSFUL;
}

int launch_ens_drag(const EnsDragTable *tab, const EnsDragItem *items, int nitems, int64_t ncells,
                    const double *dtp, double frac, const DragConsts &c, int method, int64_t *queue,
                    unsigned long long *qcount, hipStream_t s, int calls)
{
    if (calls < 1 || calls > 2) return IM_FAIL(ERROR_INVALID_ARGS, "drag calls per pass: %d", calls);
    if (method != DRAG_LOGTRAP2 && method != DRAG_LOGTRAP3 && method != DRAG_EXACT && method != DRAG_LEARNED)
        return IM_FAIL(ERROR_NOIMPLEMENT, "ensemble drag method %d", method);
    if (method == DRAG_LEARNED && !g_model.loaded)
        return IM_FAIL(ERROR_INVALID_ARGS, "learned drag: no model (imogen_drag_set_model)");
    if (nitems <= 0) return SUCCESSFUL;
    const bool learned = method == DRAG_LEARNED;
    if (learned && !g_model.counts)
        return IM_FAIL(ERROR_INVALID_ARGS, "learned drag counters not prepared (learned_drag_prepare)");
    if (learned) {
        hipLaunchKernelGGL(zero_counters, dim3(1), dim3(64), 0, s, qcount, 3);
        int rc = IM_LAUNCHED("zero_counters");
        if (rc) return rc;
    }
    unsigned long long *err = state()->err;
    // persistent waves (a block stages the model once for many items)
    const int blocks = (nitems + 3) / 4 < 2048 ? (nitems + 3) / 4 : 2048;
    const int64_t *noList = nullptr;
    const unsigned long long *noCount = nullptr;
    if (learned)
        hipLaunchKernelGGL(ens_drag_kernel<true>, dim3((unsigned)blocks), dim3(256), 0, s, tab, items, nitems, dtp,
                           frac, c, method, calls, g_model.dev, queue, qcount, err, noList, noCount);
    else
        hipLaunchKernelGGL(ens_drag_kernel<false>, dim3((unsigned)blocks), dim3(256), 0, s, tab, items, nitems, dtp,
                           frac, c, method, calls, g_model.dev, queue, qcount, err, noList, noCount);
    int rc = IM_LAUNCHED("ens_drag_kernel");
    if (rc || !learned) return rc;
    // calls = 2: the first pass left cells whose first call was rejected
    // without their second call; the fallback lists them, a list-mode pass
    // gives them a learned second call and a second fallback takes its rejects
    int64_t *list = calls == 2 ? queue + ncells : nullptr;
    hipLaunchKernelGGL(ens_fallback_kernel, dim3(1024), dim3(256), 0, s, tab, dtp, frac, c, queue, qcount,
                       ncells * calls, g_model.counts, err, list, qcount + 1);
    if ((rc = IM_LAUNCHED("ens_fallback_kernel")) || calls == 1) return rc;
    hipLaunchKernelGGL(ens_drag_kernel<true>, dim3(256), dim3(256), 0, s, tab, items, 0, dtp, frac, c, method, 1,
                       g_model.dev, queue, qcount + 2, err, (const int64_t *)list,
                       (const unsigned long long *)(qcount + 1));
    if ((rc = IM_LAUNCHED("ens_drag_kernel"))) return rc;
    hipLaunchKernelGGL(ens_fallback_kernel, dim3(1024), dim3(256), 0, s, tab, dtp, frac, c, queue, qcount + 2,
                       (int64_t)0, g_model.counts, err, (int64_t *)nullptr, (unsigned long long *)nullptr);
    return IM_LAUNCHED("ens_fallback_kernel");
}

int learned_drag_prepare()
{
    return ensure_counts();
}

uint64_t learned_model_generation()
{
    return g_modelGeneration;
}

}  // namespace imogen

using namespace imogen;

extern "C" {

int imogen_drag_set_model(const float *params, const DragModelNorm *norm)
{
    if (!params || !norm) return IM_FAIL(ERROR_NULL_POINTER, "null model");
    for (int j = 0; j < 5; j++)
        if (!(norm->fstd[j] > 0)) return IM_FAIL(ERROR_INVALID_ARGS, "feature std %d must be positive", j);
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    // host-side layout of the device block
    const size_t n1 = 64 * 16, n2 = 64 * 64, n3 = 16 * 64;
    std::vector<unsigned short> w(n1 + n2 + n3, 0);
    auto bf = [](float f) {
        unsigned u;
        memcpy(&u, &f, 4);
        if ((u & 0x7fffffffu) > 0x7f800000u) return (unsigned short)0x7fc0;
        u += 0x7fffu + ((u >> 16) & 1u);
        return (unsigned short)(u >> 16);
    };
    for (int o = 0; o < 64; o++)
        for (int i = 0; i < kIn; i++) w[o * 16 + i] = bf(params[kOffW1 + i * kHid + o]);
    for (int o = 0; o < 64; o++)
        for (int i = 0; i < 64; i++) w[n1 + o * 64 + i] = bf(params[kOffW2 + i * kHid + o]);
    for (int o = 0; o < kOut; o++)
        for (int i = 0; i < 64; i++) w[n1 + n2 + o * 64 + i] = bf(params[kOffW3 + i * kOut + o]);
    std::vector<float> b(64 + 64 + 16, 0.0f);
    for (int j = 0; j < 64; j++) b[j] = params[kOffB1 + j];
    for (int j = 0; j < 64; j++) b[64 + j] = params[kOffB2 + j];
    for (int j = 0; j < kOut; j++) b[128 + j] = params[kOffB3 + j];
    const size_t wbytes = w.size() * sizeof(unsigned short), bbytes = b.size() * sizeof(float);
    if (!g_model.buf && IM_HIP(hipMalloc(&g_model.buf, wbytes + bbytes))) return ERROR_CUDA_BLEW_UP;
    // ordered after any learned-drag kernel still reading the previous model
    if (IM_HIP(hipMemcpyAsync(g_model.buf, w.data(), wbytes, hipMemcpyHostToDevice, st->stream)))
        return ERROR_CUDA_BLEW_UP;
    if (IM_HIP(hipMemcpyAsync((char *)g_model.buf + wbytes, b.data(), bbytes, hipMemcpyHostToDevice, st->stream)))
        return ERROR_CUDA_BLEW_UP;
    if (IM_HIP(hipStreamSynchronize(st->stream))) return ERROR_CUDA_BLEW_UP;
    const unsigned short *wd = (const unsigned short *)g_model.buf;
    const float *bd = (const float *)((char *)g_model.buf + wbytes);
    g_model.dev.w1t = wd;
    g_model.dev.w2t = wd + n1;
    g_model.dev.w3t = wd + n1 + n2;
    g_model.dev.b1 = bd;
    g_model.dev.b2 = bd + 64;
    g_model.dev.b3 = bd + 128;
    g_model.dev.norm = *norm;
    g_model.loaded = true;
    g_modelGeneration++;
    return SUCCESSFUL;
}

int imogen_drag_learned_stats(int64_t *cells, int64_t *fallbacks)
{
    if (ensure_counts()) return ERROR_CUDA_BLEW_UP;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    unsigned long long h[2];
    // read and clear in order with the kernels on the library stream
    if (IM_HIP(hipMemcpyAsync(h, g_model.counts, sizeof(h), hipMemcpyDeviceToHost, st->stream)))
        return ERROR_CUDA_BLEW_UP;
    if (IM_HIP(hipMemsetAsync(g_model.counts, 0, sizeof(h), st->stream))) return ERROR_CUDA_BLEW_UP;
    if (IM_HIP(hipStreamSynchronize(st->stream))) return ERROR_CUDA_BLEW_UP;
    if (cells) *cells = (int64_t)h[0];
    if (fallbacks) *fallbacks = (int64_t)h[1];
    return SUCCESSFUL;
}

int imogen_drag_training_samples(const ThermoDetails *gas, const ThermoDetails *dust, int64_t n,
                                 const double *cells, float *features, float *targets)
{
    if (!gas || !dust || !cells || !features || !targets) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (n <= 0) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    DragConsts c = drag_consts(gas, dust);
    // targets are second-order remainders (divided by tau^3 relative to ln r):
    // integrate the training paths well below the product tolerance
    c.tol = 1e-14;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(drag_samples_kernel, dim3((unsigned)blocks), dim3(256), 0, st->stream, n, cells, c, features,
                       targets);
    return IM_LAUNCHED("drag_samples_kernel");
}

int imogen_mlp_forward(const float *params, int64_t batch, const float *x, float *act, float *y)
{
    if (!params || !x || !act || !y) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (batch <= 0) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    const int64_t blocks = (batch + kRows - 1) / kRows;
    hipLaunchKernelGGL(mlp_fwd_kernel, dim3((unsigned)blocks), dim3(256), 0, st->stream, params, batch, x, act, y);
    return IM_LAUNCHED("mlp_fwd_kernel");
}

int imogen_mlp_backward(const float *params, int64_t batch, const float *x, const float *act, const float *dy,
                        float *grads)
{
    if (!params || !x || !act || !dy || !grads) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (batch <= 0) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    const int64_t blocks = (batch + kBwdRows - 1) / kBwdRows;
    float *part = (float *)scratch_block((size_t)blocks * kNParams * sizeof(float));
    if (!part) return IM_FAIL(ERROR_NOMEM, "no scratch for gradient partials");
    hipLaunchKernelGGL(mlp_bwd_kernel, dim3((unsigned)blocks, 4), dim3(256), 0, st->stream, params, batch, x, act, dy,
                       part);
    int rc = IM_LAUNCHED("mlp_bwd_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(mlp_grad_reduce, dim3((kNParams + 63) / 64), dim3(1024), 0, st->stream, part, (int)blocks,
                       grads);
    return IM_LAUNCHED("mlp_grad_reduce");
}

int imogen_mlp_adam(float *params, const float *grads, float *m, float *v, int64_t n, float lr, float beta1,
                    float beta2, float eps, int step)
{
    if (!params || !grads || !m || !v) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (step < 1) return IM_FAIL(ERROR_INVALID_ARGS, "Adam step counts from 1");
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    const float c1 = 1.0f - powf(beta1, (float)step), c2 = 1.0f - powf(beta2, (float)step);
    hipLaunchKernelGGL(mlp_adam_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st->stream, params, grads,
                       m, v, n, lr, beta1, beta2, eps, c1, c2);
    return IM_LAUNCHED("mlp_adam_kernel");
}

int imogen_mlp_mse_grad(int64_t batch, const float *y, const float *t, float *dy, double *lossAccum)
{
    if (!y || !t || !dy || !lossAccum) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (batch <= 0) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    const int64_t n = batch * kOut;
    int64_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(mlp_mse_grad_kernel, dim3((unsigned)blocks), dim3(256), 0, st->stream, n, y, t, dy,
                       1.0f / (float)n, lossAccum);
    return IM_LAUNCHED("mlp_mse_grad_kernel");
}

int imogen_gather_rows(const float *src, const int64_t *idx, int64_t nrows, int ncols, float *dst)
{
    if (!src || !idx || !dst) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (nrows <= 0 || ncols <= 0) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    int64_t blocks = (nrows * ncols + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    hipLaunchKernelGGL(gather_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, st->stream, src, idx, nrows, ncols,
                       dst);
    return IM_LAUNCHED("gather_rows_kernel");
}

int imogen_mlp_infer_bf16(int64_t batch, const float *x, float *y)
{
    if (!g_model.loaded) return IM_FAIL(ERROR_INVALID_ARGS, "no model loaded (imogen_drag_set_model)");
    if (!x || !y) return IM_FAIL(ERROR_NULL_POINTER, "null argument");
    if (batch <= 0) return SUCCESSFUL;
    DeviceState *st = state();
    if (!st) return ERROR_CUDA_BLEW_UP;
    int64_t waves = (batch + 63) / 64;
    if (waves > 8192) waves = 8192;
    hipLaunchKernelGGL(mlp_infer_kernel, dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st->stream, batch, x, y,
                       g_model.dev);
    return IM_LAUNCHED("mlp_infer_kernel");
}

}  // extern "C"
