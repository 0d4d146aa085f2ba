// sweep_device.h -- per-cell arithmetic of the HLLC and HLL sweeps (gfx950, FP64).
//
// Same formulas as the reference kernels
// cukern_HLLC_2ndorder (gpuclass/cudaFluidStep.cu:1124-1716) and
// cukern_HLL_step + cukern_PressureSolverHydro (:1801-2422, 2813-2864):
// primitive recovery (RECONSTRUCT_VELOCITY, gpuclass/Makefile:5), half-slope
// limiters (gpuclass/limiter_functions.h:50-117), Einfeldt speed bounds
// (:1728-1799), the HLLC contact speed and four-way flux selection
// (:1357-1431), the HLL flux (:2124-2196) and the HLL density/energy floors.
// Divisions and square roots use refined hardware estimates: 1-2 ulp for the
// densities' reciprocals and HLL's quotients, 3e-15 and 5e-15 elsewhere.
// The data movement around these functions (which lane owns which cell, how
// neighbours are exchanged) is this library's own.
#pragma once
#include <hip/hip_runtime.h>

namespace imogen {

// Variables of one cell or face, ordered (rho, e|P, vN, vT1, vT2): normal
// velocity first, then the two tangential components in the order the
// reference kernels read them (X: y,z; Y: x,z; Z: y,x).
struct V5 {
    double a, b, c, d, e;
};

struct HydroConsts {
    double gamma;     // adiabatic index
    double gm1;       // gamma - 1
    double hgm1;      // (gamma - 1) / 2
    double igm1;      // 1 / (gamma - 1)
    double govergm1;  // gamma / (gamma - 1)
    double rhomin;    // density floor (HLL)
    double emin;      // specific internal energy floor 1e-5/(gamma-1) (cudaFluidStep.cu:298)
    double ciso;      // isothermal sound speed, -1 = adiabatic (HLL)
    double cisosq;    // ciso^2
};

__device__ __forceinline__ V5 operator-(const V5 &x, const V5 &y)
{
    return V5{x.a - y.a, x.b - y.b, x.c - y.c, x.d - y.d, x.e - y.e};
}

// ---- fast FP64 reciprocal, quotient and square root ------------------------
// The IEEE-exact sequences the compiler emits for '/' and sqrt() handle
// denormal and overflow scaling that the fluid variables never need; these
// use the hardware estimates (v_rcp_f64, v_rsq_f64) with Newton/Goldschmidt
// refinement to full double precision (within 1-2 ulp). Arguments are finite,
// non-zero normals (rcp, quotient) or >= 0 normals (sqrt).
// v_rcp_f64 / v_rsq_f64 are accurate to ~4.6e-8 and ~5.2e-8 relative
// (measured on gfx950 over 4M values spanning 2^-30..2^30).
__device__ __forceinline__ double rcp_nr(double x)
{
    // third-order refinement r0 (1 + e + e^2), e = 1 - x r0: error ~ e^3
    const double r = __builtin_amdgcn_rcp(x);
    const double e = fma(-x, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

__device__ __forceinline__ double div_nr(double a, double b)
{
    return a * rcp_nr(b);
}

// Quotient with one residual correction: q + (a - q b) / b. With a correctly
// rounded reciprocal this is the correctly rounded quotient (Markstein,
// IBM J. Res. Dev. 34 (1990) 111), i.e. what the reference's `a / b` gives.
__device__ __forceinline__ double div_cr(double a, double b)
{
    const double r = rcp_nr(b);
    const double q = a * r;
    return fma(fma(-q, b, a), r, q);
}

__device__ __forceinline__ double sqrt_nr(double x)
{
    // One Goldschmidt step and one Newton correction reach full precision from
    // the hardware estimate. The 1e-300 offset keeps rsq finite at x = 0 (so
    // sqrt(0) = 0) without changing any argument >= 1e-284; x < 0 stays NaN.
    const double y = __builtin_amdgcn_rsq(x + 1e-300);
    double g = x * y;
    double h = 0.5 * y;
    const double r = fma(-g, h, 0.5);
    g = fma(g, r, g);
    h = fma(h, r, h);
    const double d = fma(-g, g, x);
    return fma(d, h, g);
}

// Reduced-refinement variants for the sweeps' quotients and roots: one quadratic Newton
// step for the reciprocal (relative error ~ e^2 + 1 ulp ~ 3e-15) and one
// Goldschmidt step for the square root (~5e-15). The sweep results stay far
// inside the 1e-12 parity bar; the correctly rounded quotient (div_cr) keeps
// the full-precision reciprocal.
__device__ __forceinline__ double rcp_fast(double x)
{
    const double r = __builtin_amdgcn_rcp(x);
    return fma(r, fma(-x, r, 1.0), r);
}

__device__ __forceinline__ double div_fast(double a, double b)
{
    // the Newton step on the quotient: q (2 - b r), q = a r
    const double r = __builtin_amdgcn_rcp(b);
    const double q = a * r;
    return fma(q, fma(-b, r, 1.0), q);
}

// sqrt(x), x > 0. Callers add the smallest step kTinySq to a sum that may be
// exactly 0 (in an FMA they need anyway), so that its root is ~0 and not NaN;
// it changes no sum >= 1e-284, and negative ones stay NaN.
constexpr double kTinySq = 1e-300;
__device__ __forceinline__ double sqrt_fast_pos(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double g = x * y;
    const double r = fma(-g, 0.5 * y, 0.5);
    return fma(g, r, g);
}

// sqrt(x), x > 0, as a product g t: a sum v +- g t is then one FMA
struct Root {
    double g, t;
};
__device__ __forceinline__ Root root_fast(double x)
{
    const double y = __builtin_amdgcn_rsq(x);
    const double g = x * y;
    return Root{g, fma(.5, fma(-g, y, 1.0), 1.0)};
}

// ---- half-slope limiters (limiter_functions.h) ----------------------------
__device__ __forceinline__ double flux_minmod(double a, double b)
{
    if (a * b < 0) return 0.0;
    return (fabs(a) > fabs(b)) ? b : a;
}

// The limited half slope is slope_scale<LIM> * slope_limit<LIM>(a, b). Ospre and
// van Leer select on a b > 0, as the reference does: a NaN difference gives no
// slope, so a bad cell spoils its own faces and fluxes and not its neighbours'
// other faces. (Raising the product to 0 instead left a + b NaN.)
template <int LIM>
__device__ __forceinline__ double slope_limit(double a, double b, int rt)
{
    const int which = (LIM >= 0) ? LIM : rt;
    switch (which) {
    case 0: {  // Ospre: .75 A B (A+B) / (A^2 + AB + B^2)
        // Where A B is positive but below the normal range, the numerator
        // underflows and the slope is 0 (the hardware reciprocal of so small a
        // denominator would be infinite); otherwise the denominator is at least
        // 3 A B, a normal.
        const double r = a * b;
        const double s = a + b;
        const double v = div_fast(((LIM >= 0) ? 1.0 : .75) * r * s, fma(s, s, -r));
        return (r >= 0x1p-1022) ? v : 0.0;
    }
    case 1: {  // van Leer: A B / (A+B)
        const double r = a * b;
        const double v = div_fast(r, a + b);
        return (r > 0) ? v : 0.0;
    }
    case 2: {  // minmod, returned through float as the reference does (:70)
        if (a * b < 0) return 0.0;
        return (double)(float)((fabs(a) > fabs(b)) ? .5 * b : .5 * a);
    }
    case 3: {  // superbee (first branch without the 1/2, :80-86)
        if (a * b < 0) return 0.0;
        if (b < a) return flux_minmod(a, 2 * b);
        return .5 * flux_minmod(2 * a, b);
    }
    case 4: {  // van Albada
        double r = a * b;
        if (r < 0) return 0;
        return .5 * r * (a + b) / (a * a + b * b);
    }
    case 5: {  // monotonized central
        if (a * b <= 0) return 0;
        double r = b / a;
        double s = .25 + .25 * r;
        s = (s < r) ? s : r;
        s = (s < 1) ? s : 1.0;
        return s * a;
    }
    default:
        return 0.0;
    }
}

template <int LIM>
constexpr double slope_scale = (LIM == 0) ? .75 : 1.0;

// w -+ the limited half slope, one FMA each
template <int LIM>
__device__ __forceinline__ void face_pair(double w, double dl, double dr, int rt, double &L, double &R)
{
    const double s = slope_limit<LIM>(dl, dr, rt);
    L = fma(-slope_scale<LIM>, s, w);
    R = fma(slope_scale<LIM>, s, w);
}

// Limiters with lim(c a, c b) = c lim(a, b): pressure and internal energy then
// reconstruct alike, and the pressure is formed once per cell instead of on
// both faces. (Minmod's pass through float is not of these.)
template <int LIM>
constexpr bool slope_homogeneous = (LIM == 0 || LIM == 1);

// Conserved (rho, E, pN, pT1, pT2) -> primitive (rho, e_int, vN, vT1, vT2),
// cudaFluidStep.cu:1218-1234; with a homogeneous limiter P in place of e_int.
// The densities' reciprocals here and in roe_terms are refined in full: their
// error enters every flux of a cell, and through the hottest cell's sound speed
// the time step (12 iterations of a Sedov blast of 36^3 and 44^3 cells, mean
// relative error against 80-bit arithmetic over 16 seeds and two limiters:
// 6.9e-16 with one Newton step, 4.8e-16 so; no measurable time).
template <int LIM>
__device__ __forceinline__ V5 to_prim(const HydroConsts &k, const V5 &q)
{
    const double F = rcp_nr(q.a);
    const double u = q.c * F, v = q.d * F, w = q.e * F;
    const double e = fma(-.5, fma(q.e, w, fma(q.d, v, q.c * u)), q.b);
    return V5{q.a, slope_homogeneous<LIM> ? k.gm1 * e : e, u, v, w};
}

// Left/right face states of a cell from its primitive w and the backward
// differences dl = w_i - w_{i-1}, dr = w_{i+1} - w_i. The energy slot holds
// pressure (gm1 * e) on the faces (cudaFluidStep.cu:1277-1278).
template <int LIM>
__device__ __forceinline__ void faces(const HydroConsts &k, const V5 &w, const V5 &dl, const V5 &dr,
                                      int rt, V5 &L, V5 &R)
{
    face_pair<LIM>(w.a, dl.a, dr.a, rt, L.a, R.a);
    face_pair<LIM>(w.b, dl.b, dr.b, rt, L.b, R.b);
    if (!slope_homogeneous<LIM>) {
        L.b *= k.gm1;
        R.b *= k.gm1;
    }
    face_pair<LIM>(w.c, dl.c, dr.c, rt, L.c, R.c);
    face_pair<LIM>(w.d, dl.d, dr.d, rt, L.d, R.d);
    face_pair<LIM>(w.e, dl.e, dr.e, rt, L.e, R.e);
}

// Roe weights and sound speeds of an interface from its face densities and
// pressures. A reciprocal per side: one reciprocal root of the product of the
// densities would give both with fewer instructions, but a NaN of one side then
// reaches the other side's sound speed (and the plain flux of a side whose
// waves all leave the bad cell), and the product leaves the double range for
// densities below 1.5e-154 or above 1.3e154.
struct RoeTerms {
    double csql, csqr;  // gamma P / rho
    double Fa, Fb;      // sqrt(rhoR / rhoL), 1 / (1 + Fa)
};
__device__ __forceinline__ RoeTerms roe_terms(const HydroConsts &k, double rl, double rr, double Pl, double Pr)
{
    const double il = rcp_nr(rl);
    RoeTerms t;
    t.csql = fma(k.gamma * Pl, il, kTinySq);
    t.csqr = fma(k.gamma * Pr, rcp_nr(rr), kTinySq);
    t.Fa = sqrt_fast_pos(rr * il);  // NaN where the densities differ in sign, as the reference's
    t.Fb = rcp_fast(1.0 + t.Fa);
    return t;
}

// Einfeldt bounds (cudaFluidStep.cu:1728-1754) of normal velocities vl, vr and
// squared velocity jump dvsq. The reference's selects, not fmin/fmax: a NaN
// bound (negative face pressure) must propagate as it does there.
__device__ __forceinline__ void einfeldt(const HydroConsts &k, const RoeTerms &t, double vl, double vr, double dvsq,
                                         double &sl, double &sr)
{
    const double Vroe = fma(t.Fa, vr, vl) * t.Fb;
    const double x = fma(k.hgm1 * dvsq, t.Fa * t.Fb, fma(t.Fa, t.csqr, t.csql));
    const Root C = root_fast(fma(x, t.Fb, kTinySq)), cl = root_fast(t.csql), cr = root_fast(t.csqr);
    const double sroe = fma(-C.g, C.t, Vroe), rroe = fma(C.g, C.t, Vroe);
    sl = fma(-cl.g, cl.t, vl);
    sr = fma(cr.g, cr.t, vr);
    sl = (sroe < sl) ? sroe : sl;
    sr = (rroe > sr) ? rroe : sr;
}

// HLLC flux through the interface between face state L (right face of cell i)
// and R (left face of cell i+1). Returns (mass, energy, pN, pT1, pT2) fluxes.
// The four reference cases are evaluated without divergence: the upwind side
// and its wave speed are selected first; that side's plain flux (cases 0/1,
// cudaFluidStep.cu:1372-1383, 1416-1430) is its star flux (cases 2/3,
// :1384-1415) with the contact speed replaced by the side's own velocity and
// rho beta by rho, so two selects choose between them. With mass flux m the
// energy flux is m (c^2/(gamma-1) + |v|^2/2 + S_K (S_M - v)) and the
// tangential ones are v_t m.
__device__ __forceinline__ V5 hllc_flux(const HydroConsts &k, const V5 &L, const V5 &R)
{
    // velocity jump squared (cudaFluidStep.cu:1318-1322)
    const double C = L.c - R.c;
    const double D = L.d - R.d;
    const double E = L.e - R.e;
    const RoeTerms t = roe_terms(k, L.a, R.a, L.b, R.b);
    double sl, sr;
    einfeldt(k, t, L.c, R.c, fma(E, E, fma(D, D, C * C)), sl, sr);

    // contact speed, Batten et al. eq. 34 (cudaFluidStep.cu:1352-1357)
    const double A = L.a * (sl - L.c);
    const double B = R.a * (sr - R.c);
    const double sm = div_fast(fma(B, R.c, fma(-A, L.c, L.b - R.b)), B - A);

    // case selection (cudaFluidStep.cu:1363-1369)
    const bool left = sm > 0;
    const bool star = left ? !(sl > 0) : (sr > 0);
    const V5 S = left ? L : R;
    const double sk = left ? sl : sr;
    const double csq = left ? t.csql : t.csqr;
    const double AS = left ? A : B;

    double rb = div_fast(AS, sk - sm);  // rho beta
    // the empty asm keeps the quotient out of a branch on `star` (which the
    // compiler would form around its one use): nearly every interface is a
    // star one, and a branch per interface splits the code the two stages'
    // chains interleave in
    asm("" : "+v"(rb));
    rb = star ? rb : S.a;
    const double vm = star ? sm : S.c;
    const double ksum = fma(S.e, S.e, fma(S.d, S.d, S.c * S.c));  // |v|^2 of the upwind face
    // 0 in the plain case also where the bound of the other side is NaN
    const double Cc = (star ? sk : 0.0) * (vm - S.c);
    const double m = rb * vm;
    V5 out;
    out.a = m;
    out.b = m * fma(csq, k.igm1, fma(.5, ksum, Cc));
    out.c = fma(rb, fma(vm, S.c, Cc), S.b);
    out.d = S.d * m;
    out.e = S.e * m;
    return out;
}

// ---------------------------------------------------------------------------
// Method policies used by the sweep kernels
// ---------------------------------------------------------------------------
// floor(q): applies the method's pointwise floors to the conserved cell q in
// place (the floored q is what the SSP-RK2 combination uses) and returns the
// internal energy density the floors settled on. prims(q, e): reconstruction
// variables of a floored cell. face(): limited left/right face states.
// flux(): interface flux in slab order (mass, energy, normal, t1, t2).

struct Hllc {
    static constexpr bool floors = false;  // floor() leaves the cell as it is
    template <int DIR>
    __device__ static __forceinline__ double floor(const HydroConsts &, V5 &)
    {
        return 0.0;
    }
    template <int LIM>
    __device__ static __forceinline__ V5 prims(const HydroConsts &k, const V5 &q, double)
    {
        return to_prim<LIM>(k, q);
    }
    template <int LIM>
    __device__ static __forceinline__ void face(const HydroConsts &k, const V5 &w, const V5 &dl, const V5 &dr,
                                                int rt, V5 &L, V5 &R)
    {
        faces<LIM>(k, w, dl, dr, rt, L, R);
    }
    __device__ static __forceinline__ V5 flux(const HydroConsts &k, const V5 &L, const V5 &R)
    {
        return hllc_flux(k, L, R);
    }
};

struct Hll {
    static constexpr bool floors = true;
    // q = (rho, E, pN, pT1, pT2) in HLL's component order for direction DIR:
    // X (px,py,pz), Y (py,px,pz), Z (pz,px,py) (cudaFluidStep.cu:1869-1885).
    // The floors accumulate |p|^2 in physical x,y,z order (:2821-2843).
    template <int DIR>
    __device__ static __forceinline__ double floor(const HydroConsts &k, V5 &q)
    {
        double rho = q.a;
        if (rho < k.rhomin) {
            const double f = k.rhomin / rho;
            rho = q.a = k.rhomin;
            q.b = f * q.b;
            q.c = f * q.c;
            q.d = f * q.d;
            q.e = f * q.e;
        }
        const double px = (DIR == 1) ? q.c : q.d;
        const double py = (DIR == 1) ? q.d : ((DIR == 2) ? q.c : q.e);
        const double pz = (DIR == 3) ? q.c : q.e;
        double momsq = px * px;
        momsq += py * py;
        momsq += pz * pz;
        const double ke = div_cr(.5 * momsq, rho);
        double e = q.b - ke;
        if (e < rho * k.emin) {
            e = k.emin * rho;
            q.b = ke + e;
        }
        return e;
    }
    // (rho, vN, P, vT1, vT2); velocities are quotients, as in the reference (:1887-1889)
    template <int LIM>
    __device__ static __forceinline__ V5 prims(const HydroConsts &k, const V5 &q, double e)
    {
        return V5{q.a, div_cr(q.c, q.a), e * k.gm1, div_cr(q.d, q.a), div_cr(q.e, q.a)};
    }
    template <int LIM>
    __device__ static __forceinline__ void face(const HydroConsts &, const V5 &w, const V5 &dl, const V5 &dr,
                                                int rt, V5 &L, V5 &R)
    {
        face_pair<LIM>(w.a, dl.a, dr.a, rt, L.a, R.a);
        face_pair<LIM>(w.b, dl.b, dr.b, rt, L.b, R.b);
        face_pair<LIM>(w.c, dl.c, dr.c, rt, L.c, R.c);
        face_pair<LIM>(w.d, dl.d, dr.d, rt, L.d, R.d);
        face_pair<LIM>(w.e, dl.e, dr.e, rt, L.e, R.e);
    }
    // L, R = (rho, vN, P, vT1, vT2), the reference's A..E (cudaFluidStep.cu:2124-2196)
    __device__ static __forceinline__ V5 flux(const HydroConsts &k, const V5 &L, const V5 &R)
    {
        const double Ut = R.b - L.b, St1 = R.d - L.d, St2 = R.e - L.e;
        const RoeTerms t = roe_terms(k, L.a, R.a, L.c, R.c);
        double sl, sr;
        if (k.ciso == -1) {
            einfeldt(k, t, L.b, R.b, fma(St2, St2, fma(St1, St1, Ut * Ut)), sl, sr);
        } else {
            // computeEinfeldtBounds_isothermal, passed C_iso^2 for the sound speed (:2131)
            const double Vroe = fma(t.Fa, R.b, L.b) * t.Fb;
            double cs = Vroe - k.cisosq;
            sl = L.b - cs;
            sr = R.b + cs;
            sl = (cs < sl) ? cs : sl;
            cs = 2 * Vroe - cs;
            sr = (cs > sr) ? cs : sr;
        }
        const double At = rcp_fast(sr - sl);
        const double Fl = L.a * L.b, Fr = R.a * R.b;
        V5 o;
        if (sl >= 0 || sr <= 0) {  // one-sided (left unless the right case also holds)
            const bool right = sr <= 0;
            const V5 S = right ? R : L;
            const double F = right ? Fr : Fl;
            const double ke = .5 * S.a * (S.b * S.b + S.d * S.d + S.e * S.e);
            o.a = F;
            if (k.ciso == -1) {
                o.b = S.b * (k.govergm1 * S.c + ke);
                o.c = F * S.b + S.c;
            } else {
                o.b = S.b * (S.c + ke);
                o.c = F * S.b + (right ? k.ciso : k.cisosq) * S.a;  // C_iso on the right side (:2191)
            }
            o.d = F * S.d;
            o.e = F * S.e;
        } else {
            const double wl = sr * (L.b - sl);
            const double wr = sl * (R.b - sr);
            o.a = (wl * L.a - wr * R.a) * At;
            if (k.ciso == -1) o.c = (wl * Fl - wr * Fr + sr * L.c - sl * R.c) * At;
            else o.c = (wl * Fl - wr * Fr + k.cisosq * (sr * L.a - sl * R.a)) * At;
            o.d = (wl * L.a * L.d - wr * R.a * R.d) * At;
            o.e = (wl * L.a * L.e - wr * R.a * R.e) * At;
            if (k.ciso == -1) {
                const double kl = .5 * L.a * (L.b * L.b + L.d * L.d + L.e * L.e);
                const double kr = .5 * R.a * (R.b * R.b + R.d * R.d + R.e * R.e);
                const double e = (wl * kl - wr * kr);
                o.b = (e + (k.govergm1 * (sr * L.c * L.b - sl * R.c * R.b) + sl * sr * (R.c - L.c) * k.igm1)) * At;
            } else {
                // no 1/(Sr-Sl) on the isothermal energy flux in the reference (:2185-2189)
                const double kl = .5 * L.a * (L.b * L.b + L.d * L.d + L.e * L.e) + L.c;
                const double kr = .5 * R.a * (R.b * R.b + R.d * R.d + R.e * R.e) + R.c;
                o.b = (wl * kl - wr * kr);
            }
        }
        return o;
    }
};

// Slabs holding (normal, t1, t2) momentum per method and direction.
template <class M, int DIR>
struct MomSlabs;
template <>
struct MomSlabs<Hllc, 1> {
    static constexpr int n = 2, t1 = 3, t2 = 4;
};
template <>
struct MomSlabs<Hllc, 2> {
    static constexpr int n = 3, t1 = 2, t2 = 4;
};
template <>
struct MomSlabs<Hllc, 3> {
    static constexpr int n = 4, t1 = 3, t2 = 2;
};
template <>
struct MomSlabs<Hll, 1> {
    static constexpr int n = 2, t1 = 3, t2 = 4;
};
template <>
struct MomSlabs<Hll, 2> {
    static constexpr int n = 3, t1 = 2, t2 = 4;
};
template <>
struct MomSlabs<Hll, 3> {
    static constexpr int n = 4, t1 = 2, t2 = 3;
};

}  // namespace imogen
