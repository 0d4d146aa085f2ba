// drag_device.h -- per-cell arithmetic of the gas-dust drag source (FP64).
//
// Drag rate: cukern_GasDustDrag_GeneralLinearCore + allregimeCdrag
// (gpuclass/cudaSource2FluidDrag.cu:819-890). Powers of the normalised
// temperature and of Re share their logarithms: x^a = exp(a ln x), off by about
// |a ln x| roundings.
//
// The drag kernels are bound by the issue of these functions (the adaptive
// integrator spent 98 % of its issue slots): exp and log below are half the
// instructions of the math library's, which carry a second word through and
// treat overflow, subnormals and signed zeros, and quotients are products with
// refined reciprocals and a residual correction. One LogTrap2 call on 2.99e6
// cells: 130 -> 71 us; two adaptive calls on 96^3 cells: 304 -> 140 us; the
// learned source's fallback in a 192^3 run: 190 -> 132 us a launch.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/imogen_abi.h"
#include "sweep_device.h"

namespace imogen {

// absolute tolerance on ln|dv| of the adaptive reference integrator
constexpr double kDragExactTol = 1e-12;

struct DragConsts {
    double visc0, viscpow, lampow, alpha, beta, delta, epsilon, gm1;
    double tol;
};

struct DragCell {
    double rg, rd;   // gas and dust density
    double s0, u0;   // |dv| and gas specific internal energy
};

// e^x - 1 = 2^n (1 + p) - 1 with n = round(x / ln 2) and p = r + r^2 Q(r) on the
// remainder |r| <= ln 2 / 2; Q is a degree-9 Chebyshev fit of (e^r - 1 - r)/r^2
// (p within 1e-16). ln 2 is split so that n ln2hi is exact. Overflow gives inf
// and underflow 0 through the exponent up to |x| = 1e12; NaN stays.
__device__ __forceinline__ double exp_parts(double x, int &n)
{
    const double f = rint(x * 0x1.71547652b82fep+0);
    const double r = fma(-f, 0x1.d1cf79ac00000p-32, fma(-f, 0x1.62e42fec00000p-1, x));
    n = (int)f;
    double q = 0x1.ae5b5adb47a68p-26;
    q = fma(q, r, 0x1.287e80b64b99ep-22);
    q = fma(q, r, 0x1.71de80ebc2248p-19);
    q = fma(q, r, 0x1.a019c8b3fdbdcp-16);
    q = fma(q, r, 0x1.a01a018d205fbp-13);
    q = fma(q, r, 0x1.6c16c174b881ap-10);
    q = fma(q, r, 0x1.111111110e1c4p-7);
    q = fma(q, r, 0x1.5555555554696p-5);
    q = fma(q, r, 0x1.5555555555555p-3);
    q = fma(q, r, 0.5);
    return fma(r * r, q, r);
}

__device__ __forceinline__ double exp_fast(double x)
{
    int n;
    const double p = exp_parts(x, n);
    return ldexp(1.0 + p, n);
}

// e^x for an exponent of any size (a decay over a very long time): 0 below -1100,
// and for a trial stage thrown far off, inf above 1100
__device__ __forceinline__ double exp_decay(double x)
{
    return exp_fast(x < -1100.0 ? -1100.0 : x);
}
__device__ __forceinline__ double exp_any(double x)
{
    return exp_decay(x > 1100.0 ? 1100.0 : x);
}

// e^x and e^x - 1 for a decay exponent, the latter to full relative precision near 0 (n = 0: p itself)
__device__ __forceinline__ double exp_fast(double x, double &em1)
{
    int n;
    const double p = exp_parts(x < -1100.0 ? -1100.0 : x, n);
    em1 = ldexp(p, n) + (ldexp(1.0, n) - 1.0);
    return ldexp(1.0 + p, n);
}

// ln x for normal x > 0, NaN otherwise: x = 2^e m, sqrt(1/2) <= m < sqrt(2),
// ln m = 2 atanh(s) with s = (m - 1)/(m + 1); q(s^2) = (2 atanh(s)/s - 2)/s^2 is a
// degree-6 Chebyshev fit (within 7e-18 of ln m). With f = m - 1, which is exact,
// 2 s = f - s f, so ln m = f - s (f - s^2 q): the rounding of s is scaled by f.
__device__ __forceinline__ double log_fast(double x)
{
    double m = __builtin_amdgcn_frexp_mant(x);
    int e = __builtin_amdgcn_frexp_exp(x);
    const bool low = m < 0x1.6a09e667f3bcdp-1;
    m = low ? m + m : m;
    e -= low ? 1 : 0;
    const double f = m - 1.0;
    const double s = div_cr(f, m + 1.0);
    const double z = s * s;
    double q = 0x1.2a30988db636ap-3;
    q = fma(q, z, 0x1.3a1a8e48fafadp-3);
    q = fma(q, z, 0x1.7461ad42ed849p-3);
    q = fma(q, z, 0x1.c71c6777b76fcp-3);
    q = fma(q, z, 0x1.24924929220f5p-2);
    q = fma(q, z, 0x1.999999999933cp-2);
    q = fma(q, z, 0x1.5555555555555p-1);
    const double d = (double)e;
    const double l = fma(d, 0x1.62e42fec00000p-1, fma(-s, fma(-z, q, f), fma(d, 0x1.d1cf79ac00000p-32, f)));
    return x > 0 ? l : __builtin_nan("");
}

// a / b with rb = rcp_nr(b) at hand (div_cr's residual correction)
__device__ __forceinline__ double quot(double a, double b, double rb)
{
    const double q = a * rb;
    return fma(fma(-q, b, a), rb, q);
}

// What a cell's rates share.
struct DragPre {
    double dr;   // delta rho_g: Re = dr |dv| T^viscpow
    double ls;   // ln dr: ln Re = ls + ln|dv| + viscpow ln T
    double brg;  // beta / rho_g
    double C;    // (rho_g + rho_d) epsilon
};
__device__ __forceinline__ DragPre drag_pre(const DragConsts &c, double rhog, double rhod)
{
    const double dr = c.delta * rhog;
    return DragPre{dr, log_fast(dr), div_cr(c.beta, rhog), (rhog + rhod) * c.epsilon};
}

// a ln T; T^0 = 1 for any T
__device__ __forceinline__ double scaled_log(double a, double lT)
{
    return (a == 0.0) ? 0.0 : a * lT;
}

// e^{-0.999/Kn} of the Cunningham factor. Below Kn = 0.024 it is under 1e-18 and
// changes no bit of what it is added to, so a wave whose cells all lie there
// (dense gas: Kn is about 1e-3 in the gas-dust configuration) leaves it out: a
// fifth of a rate's instructions (adaptive gas-dust run at 96^3 2674 -> 2600 us).
// The floor keeps the quotient finite at Kn = 0.
__device__ __forceinline__ double cunningham_exp(double Kn)
{
    double e = 0.0;
    if (__any(!(Kn < 0.024))) e = exp_fast(-0.999 * rcp_nr(fmax(Kn, 1e-3)));
    return e;
}

// C_d |dv| (rho_g + rho_d) epsilon at |dv| = s, ls1 = ln(delta rho_g s) and gas
// internal energy u. With q = 8710 + Re the drag coefficient's sum is
// .45 Re^-.319 + [3 q + .0509 Re^2] / (Re q). Re itself is the product, not
// e^{ln Re}: the logarithm's terms are of order 10, and their rounding would be
// the rate's largest error; Re^-.319 is the larger term and is kept out of the
// quotient. Mean relative error of a rate in the gas-dust configuration 1.6e-16,
// as with the library's functions and divisions throughout (3.8e-16 with
// e^{ln Re}, e^{.681 ln Re} and one reciprocal for everything).
__device__ __forceinline__ double drag_rate(const DragConsts &c, const DragPre &pre, double s, double ls1, double u)
{
    const double lT = log_fast(c.alpha * u);
    const double lTv = scaled_log(c.viscpow, lT);
    const double Re = pre.dr * s * exp_fast(lTv);
    const double Kn = pre.brg * exp_fast(scaled_log(c.lampow, lT));
    const double cunningham = fma(Kn, fma(0.558, cunningham_exp(Kn), 1.142), 1.0);
    const double q = 8710 + Re;
    const double N = fma(.45, exp_fast(-.319 * (ls1 + lTv)), fma(.0509 * Re, Re, 3 * q) * rcp_nr(Re * q));
    return div_cr(N * s * pre.C, cunningham);
}

// drag_rate where T = alpha u may be 0 or infinite (a gas without internal
// energy: its cells are reported, and updated as the formula falls). log_fast
// has no such limit, so the powers take theirs here: T^a is 0, 1 or infinite.
// The adaptive integrator refuses such cells and needs no look.
__device__ __forceinline__ double drag_rate_any(const DragConsts &c, const DragPre &pre, double s, double ls1, double u)
{
    const double T = c.alpha * u, inf = __builtin_inf();
    if (!(T == 0.0 || T == inf)) return drag_rate(c, pre, s, ls1, u);
    auto power = [&](double a) { return a == 0.0 ? 1.0 : ((a > 0) == (T == 0.0) ? 0.0 : inf); };
    const double Re = pre.dr * s * power(c.viscpow);
    const double Kn = pre.brg * power(c.lampow);
    const double cunningham = 1 + Kn * (1.142 + 0.558 * exp_decay(-0.999 / Kn));
    const double E = Re > 0 ? exp_fast(-.319 * log_fast(Re)) : inf;
    return (3 / Re + .45 * E + .0509 * Re / (8710 + Re)) / cunningham * s * pre.C;
}

// drag rate k(|dv|, u); no drag below |dv| = 1e-9 (:853-859)
__device__ __forceinline__ double drag_k(const DragConsts &c, double rhog, double rhod, double magdv, double u)
{
    if (magdv < 1e-9) return 0.0;
    const DragPre pre = drag_pre(c, rhog, rhod);
    return drag_rate_any(c, pre, magdv, pre.ls + log_fast(magdv), u);
}

// |dv| and u_0 of a cell (cukern_prepareForERK_h0, :1883-1908)
__device__ __forceinline__ DragCell drag_load(const double *g, const double *d, int64_t p)
{
    DragCell s;
    s.rg = g[0];
    s.rd = d[0];
    const double irg = rcp_nr(s.rg), ird = rcp_nr(s.rd);
    const double E = g[p], gx = g[2 * p], gy = g[3 * p], gz = g[4 * p];
    const double dx = d[2 * p], dy = d[3 * p], dz = d[4 * p];
    double dv = quot(gx, s.rg, irg) - quot(dx, s.rd, ird);
    double dvsq = dv * dv;
    dv = quot(gy, s.rg, irg) - quot(dy, s.rd, ird);
    dvsq += dv * dv;
    dv = quot(gz, s.rg, irg) - quot(dz, s.rd, ird);
    dvsq += dv * dv;
    s.s0 = sqrt_nr(dvsq);
    s.u0 = quot(E - quot(.5 * (gx * gx + gy * gy + gz * gz), s.rg, irg), s.rg, irg);
    return s;
}

// New momenta about the barycentric velocity, dv scaled by f, and the gas
// energy change conserving total energy (:1632-1676).
__device__ __forceinline__ void drag_apply(double *g, double *d, int64_t p, const DragCell &s, double f)
{
    const double rs = s.rg + s.rd, irs = rcp_nr(rs);
    const double mu = quot(s.rd, rs, irs) * s.rg;
    const double rhoginv = rcp_nr(s.rg), rhodinv = rcp_nr(s.rd);
    double pdustsq = 0.0;
#pragma unroll
    for (int c = 2; c <= 4; c++) {
        const double pg = g[c * p], pd = d[c * p];
        pdustsq -= pd * pd;
        const double vstick = quot(pg + pd, rs, irs);
        const double dv_t = (quot(pg, s.rg, rhoginv) - quot(pd, s.rd, rhodinv)) * f;
        g[c * p] = s.rg * vstick + dv_t * mu;
        const double q = s.rd * vstick - dv_t * mu;
        d[c * p] = q;
        pdustsq += q * q;
    }
    g[p] -= quot(.5 * pdustsq, s.rd, rhodinv);
}

// Exponential Euler update (cukern_ETDRK1, :1426-1530, with ACCOUNT_GRADP
// undefined, :63): every dv component decays by exp(-t k0) about the
// barycentric velocity, in the reference's driven form dpdt/k + (dv - dpdt/k)
// e^{-kt} with dpdt = 0 (NaN when k0 = 0, as there)
__device__ __forceinline__ void drag_etd1_apply(double *g, double *d, int64_t p, double t, double k)
{
    const double rs = g[0] + d[0];
    const double rhoginv = rcp_nr(g[0]), rhodinv = rcp_nr(d[0]), irs = rcp_nr(rs);
    const double mu = quot(g[0] * d[0], rs, irs);
    const double e = exp_decay(-t * k);
    // dpdt/k: 0, and NaN where the rate is cut to 0
    const double driven = (k == 0.0) ? __builtin_nan("") : 0.0;
    double pdustsq = 0.0;
#pragma unroll
    for (int c = 2; c <= 4; c++) {
        const double pg = g[c * p], pd = d[c * p];
        pdustsq -= pd * pd;
        const double vstick = quot(pg + pd, rs, irs);
        const double dv_i = quot(pg, g[0], rhoginv) - quot(pd, d[0], rhodinv);
        const double dv_t = driven + (dv_i - driven) * e;
        g[c * p] = g[0] * vstick + dv_t * mu;
        const double q = d[0] * vstick - dv_t * mu;
        d[c * p] = q;
        pdustsq += q * q;
    }
    g[p] -= quot(.5 * pdustsq, d[0], rhodinv);
}

// path-averaged drag rate of LogTrap2 / LogTrap3 (cukern_LogTrapSolve, :1546-1630)
__device__ __forceinline__ double drag_logtrap_rate(const DragConsts &c, double rhog, double rhod, double dv0,
                                                    double u0, double t, int order)
{
    const DragPre pre = drag_pre(c, rhog, rhod);
    const double heat = -.5 * dv0 * dv0 * div_cr(rhod, rhog + rhod);
    const double l0 = pre.ls + log_fast(dv0);
    // the rate at |dv| = dv0 e^{-t a} and the energy its decay at rate a leaves
    auto end_rate = [&](double a) {
        double em1;
        const double e = exp_fast(-t * a, em1);
        const double s = dv0 * e;
        return s < 1e-9 ? 0.0 : drag_rate_any(c, pre, s, l0 - t * a, u0 + heat * (em1 * (1.0 + e)));
    };
    const double k0 = dv0 < 1e-9 ? 0.0 : drag_rate_any(c, pre, dv0, l0, u0);
    const double ksum = k0 + end_rate(k0);
    if (order == 3) return 0.16666666666666666667 * ksum + 0.66666666666666666667 * end_rate(.25 * ksum);
    return .5 * ksum;
}

// d ln|dv| / dt along the relaxation path, with the gas heated by the
// dissipated relative kinetic energy
__device__ __forceinline__ double drag_exact_rhs(const DragConsts &c, const DragPre &pre, double s0sq, double u0,
                                                 double h, double y)
{
    const double s = exp_any(y);
    return s < 1e-9 ? 0.0 : -drag_rate(c, pre, s, pre.ls + y, u0 + h * (s0sq - s * s));
}

// Whether the relaxation problem is defined on a cell: positive finite
// densities, a finite |dv| and, when the cell moves (|dv| >= 1e-9, the rate's
// cut-off), a positive finite gas internal energy.
__device__ __forceinline__ bool drag_cell_defined(double rhog, double rhod, double s0, double u0)
{
    const double big = 1.7976931348623157e308;
    return (rhog > 0 && rhog <= big) && (rhod > 0 && rhod <= big) && (s0 <= big) &&
           (s0 < 1e-9 || (u0 > 0 && u0 <= big));
}

// drag_exact_ratio's step count for a cell the problem is not defined on
constexpr int kDragInvalid = -(1 << 30);

// |dv(t)|/|dv(0)|: adaptive Dormand-Prince 5(4) (J. Comput. Appl. Math. 6
// (1980) 19) on y = ln|dv|, absolute tolerance c.tol on y, first trial step t.
// *steps receives the number of steps tried (negative if the budget ran out).
// A cell the problem is not defined on (drag_cell_defined), or whose rate is
// not finite, returns NaN at once with *steps = kDragInvalid; a trial step
// whose error estimate is not finite (an overflowing stage of a too-long
// step) is rejected and shrunk by the minimum factor.
__device__ __forceinline__ double drag_exact_ratio(const DragConsts &c, double rhog, double rhod, double s0,
                                                   double u0, double t, int *steps)
{
    const double big = 1.7976931348623157e308;
    *steps = 0;
    if (!drag_cell_defined(rhog, rhod, s0, u0)) {
        *steps = kDragInvalid;
        return __builtin_nan("");
    }
    if (s0 < 1e-9 || t <= 0) return 1.0;
    const DragPre pre = drag_pre(c, rhog, rhod);
    const double hc = div_cr(.5 * rhod, rhog + rhod);
    const double s0sq = s0 * s0;
    const double y0 = log_fast(s0);
    double y = y0, tt = 0.0, h = t;
    double k1 = drag_exact_rhs(c, pre, s0sq, u0, hc, y);
    if (!(fabs(k1) <= big)) {
        *steps = kDragInvalid;
        return __builtin_nan("");
    }
    const double itol = 1.0 / c.tol;
    int n = 0;
    while (tt < t) {
        if (n >= 4096) {
            *steps = -n;
            return exp_decay(y - y0);
        }
        if (h > t - tt) h = t - tt;
        const double k2 = drag_exact_rhs(c, pre, s0sq, u0, hc, y + h * (1.0 / 5) * k1);
        const double k3 = drag_exact_rhs(c, pre, s0sq, u0, hc, y + h * ((3.0 / 40) * k1 + (9.0 / 40) * k2));
        const double k4 = drag_exact_rhs(c, pre, s0sq, u0, hc,
                                         y + h * ((44.0 / 45) * k1 - (56.0 / 15) * k2 + (32.0 / 9) * k3));
        const double k5 = drag_exact_rhs(c, pre, s0sq, u0, hc,
                                         y + h * ((19372.0 / 6561) * k1 - (25360.0 / 2187) * k2 +
                                                  (64448.0 / 6561) * k3 - (212.0 / 729) * k4));
        const double k6 = drag_exact_rhs(c, pre, s0sq, u0, hc,
                                         y + h * ((9017.0 / 3168) * k1 - (355.0 / 33) * k2 + (46732.0 / 5247) * k3 +
                                                  (49.0 / 176) * k4 - (5103.0 / 18656) * k5));
        const double yn = y + h * ((35.0 / 384) * k1 + (500.0 / 1113) * k3 + (125.0 / 192) * k4 -
                                   (2187.0 / 6784) * k5 + (11.0 / 84) * k6);
        const double k7 = drag_exact_rhs(c, pre, s0sq, u0, hc, yn);
        double err = h * ((71.0 / 57600) * k1 - (71.0 / 16695) * k3 + (71.0 / 1920) * k4 -
                          (17253.0 / 339200) * k5 + (22.0 / 525) * k6 - (1.0 / 40) * k7);
        err = fabs(err) * itol;
        n++;
        if (!(err <= big)) err = 1e300;  // reject, shrink by the minimum factor
        if (err <= 1.0) {
            if (!(fabs(k7) <= big)) {
                *steps = kDragInvalid;
                return __builtin_nan("");
            }
            tt += h;
            y = yn;
            k1 = k7;
            if (!(tt < t)) break;  // most cells take one step: no next one to size
        }
        double f = (err > 0) ? 0.9 * exp_fast(-0.2 * log_fast(err)) : 5.0;
        f = (f < 0.2) ? 0.2 : ((f > 5.0) ? 5.0 : f);
        h *= f;
    }
    *steps = n;
    return exp_decay(y - y0);
}

// ---- explicit midpoint / RK4 on |dv| (solveDragEMP :305-370, solveDragRK4 :372-467) ----

// d|dv|/dt of cukern_GasDustDrag_GeneralAccel (:898-946); unlike the linear
// core it has no small-|dv| cut-off
__device__ __forceinline__ double drag_rk_accel(const DragConsts &c, const DragPre &pre, double magdv, double u)
{
    return -(drag_rate_any(c, pre, magdv, pre.ls + log_fast(magdv), u) * magdv);
}

// |dv| after dt; the stage and accumulator updates of cukern_SolveRK_single /
// _final (:1062-1100) in the reference's order, the gas heated by the
// dissipated relative kinetic energy at every later stage (:921-924)
template <int METHOD>
__device__ __forceinline__ double drag_rk_magdv(const DragConsts &c, double rhog, double rhod, double s0,
                                                double u0, double dt)
{
    const DragPre pre = drag_pre(c, rhog, rhod);
    const double hc = div_cr(.5 * rhod, rhog + rhod);
    auto u_at = [&](double s) { return u0 + hc * (s0 * s0 - s * s); };
    double k = drag_rk_accel(c, pre, s0, u0);
    if (METHOD == DRAG_EMP) {
        const double acc = 0.0 * k;
        const double s = s0 + (.5 * dt) * k;
        k = drag_rk_accel(c, pre, s, u_at(s));
        return s0 + dt * (acc + 1.0 * k);
    }
    double acc = 1.0 * k;
    double s = s0 + (.5 * dt) * k;
    k = drag_rk_accel(c, pre, s, u_at(s));
    s = s0 + (.5 * dt) * k;
    acc += 2.0 * k;
    k = drag_rk_accel(c, pre, s, u_at(s));
    s = s0 + (1.0 * dt) * k;
    acc += 2.0 * k;
    k = drag_rk_accel(c, pre, s, u_at(s));
    return s0 + (dt / 6.0) * (acc + 1.0 * k);
}

// cukern_findInitialDeltaV (:1014-1056): |dv| and u_0 with reciprocal densities
__device__ __forceinline__ DragCell drag_rk_load(const double *g, const double *d, int64_t p)
{
    DragCell s;
    s.rg = g[0];
    s.rd = d[0];
    const double rgi = rcp_nr(s.rg), rdi = rcp_nr(s.rd);
    double q = g[2 * p];
    double u = quot(q, s.rg, rgi) - quot(d[2 * p], s.rd, rdi);
    double momsq = q * q;
    double dvsq = u * u;
    q = g[3 * p];
    u = quot(q, s.rg, rgi) - quot(d[3 * p], s.rd, rdi);
    momsq += q * q;
    dvsq += u * u;
    q = g[4 * p];
    u = quot(q, s.rg, rgi) - quot(d[4 * p], s.rd, rdi);
    momsq += q * q;
    dvsq += u * u;
    s.s0 = sqrt_nr(dvsq);
    s.u0 = quot(g[p] - quot(.5 * momsq, s.rg, rgi), s.rg, rgi);
    return s;
}

// cukern_applyFinalDeltaV (:1160-1237): dv rescaled to |dv| = s1, momenta about
// the barycentric velocity, gas E + dust KE conserved, and the dust energy
// reset to its kinetic energy plus 1e-4 rho_d as the reference does
__device__ __forceinline__ void drag_rk_apply(double *g, double *d, int64_t p, double s1)
{
    const double rhog = g[0], rhod = d[0];
    const double rs = rhog + rhod, irg = rcp_nr(rhog), ird = rcp_nr(rhod), irs = rcp_nr(rs);
    double vs[3], dv[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double p1 = g[(k + 2) * p], p2 = d[(k + 2) * p];
        vs[k] = quot(p1 + p2, rs, irs);
        dv[k] = quot(p1, rhog, irg) - quot(p2, rhod, ird);
    }
    const double a = s1 / sqrt_nr(dv[0] * dv[0] + dv[1] * dv[1] + dv[2] * dv[2]);
    const double b = quot(rhog * rhod, rs, irs);
    double dustmom = 0.0, dustmomfin = 0.0;
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const double pd = d[(k + 2) * p];
        dustmom = (k == 0) ? pd * pd : dustmom + pd * pd;
        const double dvk = dv[k] * a;
        g[(k + 2) * p] = rhog * vs[k] + dvk * b;
        const double q = rhod * vs[k] - dvk * b;
        d[(k + 2) * p] = q;
        dustmomfin = (k == 0) ? q * q : dustmomfin + q * q;
    }
    g[p] += quot(.5 * (dustmom - dustmomfin), rhod, ird);
    d[p] = quot(.5 * dustmomfin, rhod, ird) + 1e-4 * rhod;
}

// The time interval of a drag call: a host value, or frac * dTime read on the
// device (loops that keep dTime in device memory). Scaling by frac = 1/4 or
// 1/2 is exact, so both forms give the same dt for the same dTime.
struct DragDt {
    double dt;
    const double *p;
    double frac;
};
__device__ __forceinline__ double drag_dt(const DragDt &t)
{
    return t.p ? t.frac * t.p[0] : t.dt;
}
inline DragDt host_dt(double dt)
{
    return DragDt{dt, nullptr, 0.0};
}

DragConsts drag_consts(const ThermoDetails *tg, const ThermoDetails *td);
// Every drag kernel counts the cells the method cannot be applied to (and the
// adaptive integrator's budget overruns) into the device error word. calls:
// 1, or 2 for two back-to-back drag calls of dt each applied in one pass.
int launch_drag(double *g, double *d, int64_t pitch, int64_t n, const DragConsts &c, DragDt dt, int method,
                hipStream_t s, int calls = 1);
// queue: one int64 per cell, or null for the library's scratch block; calls
// as launch_drag (two calls: the same result as two launches)
int launch_learned_drag(double *g, double *d, int64_t pitch, int64_t n, const DragConsts &c, DragDt dt,
                        int64_t *queue, hipStream_t s, int calls = 1);

// Drag over many gas/dust array pairs (the dusty problems of an ensemble):
// table entry t = (gas, dust, slab pitch, cells, problem index for dtp), items
// = 64-cell chunks (t, first cell). Each cell gets dt = frac * dtp[problem].
// Methods 4, 5, 6 and 7 (learned, with the queue of rejected cells integrated
// exactly). queue: one entry per cell of all tables per call (2 x cells for
// calls = 2); qcount: 3 counters.
struct EnsDragTable {
    double *g, *d;
    int64_t pitch, n;
    int p, pad;
};
struct EnsDragItem {
    int t, pad;
    int64_t base;
};
int launch_ens_drag(const EnsDragTable *tab, const EnsDragItem *items, int nitems, int64_t ncells,
                    const double *dtp, double frac, const DragConsts &c, int method, int64_t *queue,
                    unsigned long long *qcount, hipStream_t s, int calls = 1);
// changes whenever imogen_drag_set_model loads a model (captured graphs hold it by value)
uint64_t learned_model_generation();
// Allocates the learned drag's device counters (cells, fallbacks, queue
// length) if needed. Call at setup, outside any graph capture: the launchers
// of captured loops never allocate.
int learned_drag_prepare();

}  // namespace imogen
