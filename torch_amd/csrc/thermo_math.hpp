// thermo_math.hpp -- Henney et al. (2009) heating/cooling functions and the
// subcycled explicit source step of the reference's Thermodynamics operator
// (hgsteggles/TORCH src/Integrators/Thermodynamics.cpp), FP64, for the HIP
// kernels.  Operand order follows the reference except inside the cooling
// sum, whose exponentials share one reciprocal and one log of T (see
// subtract_cooling).  exp, log and pow of the rates are the table-driven
// forms below (the heating output keeps the device library's), so agreement
// with the x86 build is to within rounding rather than bitwise.
#pragma once

#include <hip/hip_runtime.h>

namespace tg {

// Constants in code units, as Thermodynamics::initialise computes them
// (Thermodynamics.cpp:24-57) plus the switches of ThermoParameters.
struct ThermoConsts {
    double thermo_hii_switch, heating_amplification, X, gamma, pfloor;
    double hydrogen_mass, spec_gas_const, dust_xsec, pi;
    double z0, T1, T2, T3, T4, imlc, nmlc, ciec_minT, ciec, cxhi_damp, n0, nmc;
    double fuvh_a, fuvh_b, fuvh_c, irh_a, irh_b, crh;
    double spl_min_slope, spl_max_slope;
    double icxhi;  // 1 / cxhi_damp
    double spl_k0; // 1 - 10 spl_x[0]: the spline piece at log10 T is 10 log10 T + spl_k0
    int subcycling;
    int pad;
};

// The constants as the rate functions take them.  EVEN: the spline's abscissae
// are spl_x[0] + k / 10 to 1e-9.  A kernel is built for both (chosen at
// launch): the test and its uneven branch inside the rate took 3 % of a lone
// wave's subcycle.
template <bool EVEN>
struct RateConsts : ThermoConsts {
    static constexpr bool even = EVEN;
};

// ---------------------------------------------------------------------------
// Tables of the rate functions, staged in LDS by every kernel that evaluates
// rates (load_tables; filled by fill_rate_tables in thermo.hip):
//   exp2   2^(j/128) as the double and what it is short of
//   c, lhi, llo  for mantissas m in [0.5, 1) of leading fraction bits j:
//                c ~ 1/m, lhi + llo = -ln c with lhi a multiple of 2^-40
//   spl    the cubic of each spline interval as (origin, a, b, c, d), with a
//          linear piece beyond either end
// The library's exp takes 23 FP64 operations and its log 85 in one dependent
// chain (double-double); these take 16 and 17 and keep an error of 0.53 and
// 0.51 ulp, and the spline's three divides go.  A subcycle (the integrator's
// whole trip: rate, floors, bookkeeping) went from about 650 vector
// instructions to 150, and 210 above ciec_minT (225 and 300 with the scalar and
// LDS ones).
// ---------------------------------------------------------------------------
constexpr int TT_EXP = 0, TT_EXP_LO = 128, TT_C = 256, TT_LHI = 384, TT_LLO = 512, TT_SPL = 640, TT_NSPL = 27;
constexpr int TT_N = TT_SPL + 5 * TT_NSPL;
constexpr double TT_LN2_HI = 0x1.62e42fefap-1;  // ln 2 to a multiple of 2^-40; times an exponent, exact
constexpr double TT_LN2_LO = 0x1.cf79abc9e3b3ap-40;

// e^x[i] for |x[i]| < 2^40; underflows to zero, overflows to infinity, NaN
// stays NaN.  x = k ln2/128 + r: 2^(k/128) from the table and a degree-5
// polynomial in |r| <= 0.0027.  N values step by step, so that their
// dependent chains overlap where few waves are in flight.
template <int N>
__device__ __forceinline__ void exp_n(const double* tab, double (&x)[N]) {
    const double magic = 0x1.8p52;
    double r[N], p[N];
    int k[N];
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = __builtin_fma(x[i], 0x1.71547652b82fep7, magic);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        k[i] = __double2loint(p[i]);
        p[i] -= magic;
    }
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = __builtin_fma(-p[i], 0x1.62e42fefa39efp-8, x[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = __builtin_fma(-p[i], 0x1.abc9e3b39803fp-63, r[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = __builtin_fma(r[i], 0x1.1111111111111p-7, 0x1.5555555555555p-5);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = __builtin_fma(p[i], r[i], 0x1.5555555555555p-3);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = __builtin_fma(p[i], r[i], 0.5);
#pragma unroll
    for (int i = 0; i < N; ++i) p[i] = __builtin_fma(p[i], r[i] * r[i], r[i]);
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const double* s = tab + TT_EXP + (k[i] & 127);
        x[i] = __builtin_amdgcn_ldexp(s[0] + __builtin_fma(s[0], p[i], s[TT_EXP_LO - TT_EXP]), k[i] >> 7);
    }
}

// arguments of -800 and less give 0 (the tables' range reduction needs |x| < 2^40)
__device__ __forceinline__ double exp_floor(double x) { return fmax(x, -800.0); }

__device__ __forceinline__ double exp_t(const double* tab, double x) {
    double v[1] = {x};
    exp_n<1>(tab, v);
    return v[0];
}

// e^x for any x (NaN stays NaN)
__device__ __forceinline__ double exp_any(const double* tab, double x) {
    x = x < -800.0 ? -800.0 : x;
    return exp_t(tab, x > 800.0 ? 800.0 : x);
}

// ln x = hi + lo for a positive finite x; hi is a multiple of 2^-40, |lo| < 0.005
__device__ __forceinline__ void log_t(const double* tab, double x, double& hi, double& lo) {
    const double m = __builtin_amdgcn_frexp_mant(x);
    const double e = (double)__builtin_amdgcn_frexp_exp(x);
    const int j = (__double2hiint(m) >> 13) & 127;
    const double r = __builtin_fma(m, tab[TT_C + j], -1.0);
    double p = __builtin_fma(r, 1.0 / 7.0, -1.0 / 6.0);
    p = __builtin_fma(p, r, 0.2);
    p = __builtin_fma(p, r, -0.25);
    p = __builtin_fma(p, r, 1.0 / 3.0);
    p = __builtin_fma(p, r, -0.5);
    p = __builtin_fma(p, r * r, r);
    hi = __builtin_fma(e, TT_LN2_HI, tab[TT_LHI + j]);
    lo = __builtin_fma(e, TT_LN2_LO, tab[TT_LLO + j]) + p;
}

// x^y, y > 0, from the two parts of ln x; 0, infinity, and NaN for a
// negative x as pow gives them for a fractional y
__device__ __forceinline__ double pow_t(const double* tab, double x, double y) {
    if (!(x > 0.0 && x <= 0x1.fffffffffffffp1023)) return x >= 0.0 ? x : __builtin_nan("");
    double hi, lo;
    log_t(tab, x, hi, lo);
    const double ph = y * hi;
    const double pl = __builtin_fma(y, lo, __builtin_fma(y, hi, -ph));
    const double x1 = ph + pl, x2 = (ph - x1) + pl;  // y ln x as a rounded sum and its error
    const double e = exp_any(tab, x1);
    return __builtin_fma(e, x2, e);
}

// 1/x for a normal x of magnitude 2^-900 .. 2^900 (T within 1e-100 .. 1e100
// and its power 1.63), within one ulp: the
// hardware reciprocal and two Newton steps
__device__ __forceinline__ double rcp_t(double x) {
    double r = __builtin_amdgcn_rcp(x);
    r = __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
    return __builtin_fma(__builtin_fma(-x, r, 1.0), r, r);
}

// The cooling spline (LogSplineData::interpolate) at log10 T for ln T = hi +
// lo: the piece from the 0.1 spacing of the abscissae (two pieces agree at
// their knot to rounding, so a neighbour chosen by rounding there changes
// nothing), corrected by one against the stored ones, as log_spline does,
// where they are not that even.  The spline is steep (20 decades in 1.5 of T):
// the offset from the knot is formed from both parts, or the rounding of log10
// T alone would be 2e-14 of the rate.
template <bool EVEN>
__device__ __forceinline__ double log_spline_t(const RateConsts<EVEN>& t, const double* tab, double hi, double lo) {
    const double x = hi * 0x1.bcb7b1526e50ep-2;
    const double xl = __builtin_fma(lo, 0x1.bcb7b1526e50ep-2,
                                    __builtin_fma(hi, 0x1.95355baaafad3p-57, __builtin_fma(hi, 0x1.bcb7b1526e50ep-2, -x)));
    int k = (int)__builtin_fma(x + xl, 10.0, t.spl_k0);  // 0 below the first knot, 26 from the last on
    k = k < 0 ? 0 : (k > TT_NSPL - 1 ? TT_NSPL - 1 : k);
    if (!EVEN) {  // piece 0 starts at knot 0, piece j at knot j - 1
        const double* knot = tab + TT_SPL + 1;
        const double v = x + xl;
        k = k < 1 ? 1 : (k > TT_NSPL - 2 ? TT_NSPL - 2 : k);
        if (knot[k - 1] > v) --k;
        else if (knot[k] <= v) ++k;
        if (knot[0] > v) k = 0;
        if (knot[TT_NSPL - 2] < v) k = TT_NSPL - 1;
    }
    const double* p = tab + TT_SPL + k;
    const double s = (x - p[0]) + xl;
    double r = __builtin_fma(p[4 * TT_NSPL], s, p[3 * TT_NSPL]);
    r = __builtin_fma(r, s, p[2 * TT_NSPL]);
    return __builtin_fma(r, s, p[TT_NSPL]);
}

// Natural cubic spline in log10 space: LogSplineData::interpolate +
// SplineData::splint (SplineData.cpp:57-81,142-151).  x, y, y2 are 26-entry
// tables (LDS) whose abscissae are 0.1 apart (log10 T = 3.5, 3.6, ..., 6.0, the
// operator's own) up to rounding: the bracketing interval of the reference's bisection (largest
// klo <= 24 with x[klo] <= x) is found from the spacing and corrected by one
// step against the stored abscissae, which gives the same klo.
__device__ __forceinline__ double log_spline(const ThermoConsts& t, const double* sx, const double* sy,
                                             const double* sy2, double x) {
    if (x > sx[25]) return sy[25] + t.spl_max_slope * (x - sx[25]);
    if (x < sx[0]) return sy[0] + t.spl_min_slope * (x - sx[0]);
    int klo = (int)((x - sx[0]) * 10.0);
    klo = klo < 0 ? 0 : (klo > 24 ? 24 : klo);
    if (sx[klo] > x) --klo;
    else if (klo < 24 && sx[klo + 1] <= x) ++klo;
    const int khi = klo + 1;
    double h = sx[khi] - sx[klo];
    double a = (sx[khi] - x) / h;
    double b = (x - sx[klo]) / h;
    return a * sy[klo] + b * sy[khi] + ((a * a * a - a) * sy2[klo] + (b * b * b - b) * sy2[khi]) * (h * h) / 6.0;
}

__device__ __forceinline__ double soft_landing(double rate, double T, double T_min) {
    double result = rate;
    if (rate < 0.0) {
        if (T <= T_min) result = 0;
        else if (T <= T_min + 200) {
            // rate (T - T_min) / 200, rounded as the division rounds it; an
            // infinite product's remainder, NaN, is replaced by a finite value
            const double x = rate * (T - T_min), q = x * 0.005;
            result = __builtin_fma(fmin(__builtin_fma(-200.0, q, x), 1.0e300), 0.005, q);
        }
    }
    return result;
}

// Per-cell factors of the cooling functions that do not depend on T; each
// is the left-to-right prefix of the reference's product, so hoisting it
// out of the subcycle loop does not change the rounding.
struct CoolingCell {
    double imlc_k;   // m_imlc*m_z0*ne*ne                (:122)
    double nmlc_k;   // m_nmlc*m_z0*ne*nn                (:127)
    double ciec_k;   // m_ciec*ne*ne*m_z0                (:133)
    double cehi_k;   // HIIFRAC*(1-HIIFRAC)*nH*nH        (:159)
    double nmc_k;    // m_nmc*(1-x)*(1-x)*pow(nH,1.6)    (:144)
    double nmc_T0;   // 70 + 220*pow(nH/m_n0, 0.2)       (:143)
};

__device__ __forceinline__ CoolingCell cooling_cell(const ThermoConsts& t, const double* tab, double nH, double x) {
    CoolingCell c;
    const double ne = nH * (x), nn = nH * (1.0 - x);
    c.imlc_k = t.imlc * t.z0 * ne * ne;
    c.nmlc_k = t.nmlc * t.z0 * ne * nn;
    c.ciec_k = t.ciec * ne * ne * t.z0;
    c.cehi_k = x * (1.0 - x) * nH * nH;
    c.nmc_k = t.nmc * (1.0 - x) * (1.0 - x) * pow_t(tab, nH, 1.6);
    c.nmc_T0 = 70.0 + 220.0 * pow_t(tab, nH / t.n0, 0.2);
    return c;
}

// subtract_cooling where its shared forms end: outside 1e-100 .. 1e100 K a
// reciprocal, a square or e^(1.63 ln T) leaves the double range and meets its
// opposite as 0 x infinity.  Each term by its own exponential, whose exponent
// is clamped where the result is 0 or infinity anyway.
template <bool EVEN>
__device__ __forceinline__ double subtract_cooling_far(const RateConsts<EVEN>& t, const CoolingCell& c,
                                                       const double* tab, double rate, double T) {
    if (!(T > 0.0)) return T == 0.0 ? rate : __builtin_nan("");  // all terms vanish towards 0; no rate below it, or of NaN
    if (T > 0x1.fffffffffffffp1023) return rate - c.imlc_k - c.nmlc_k - c.nmc_k * T;
    const double iT = 1.0 / T;
    double hi, lo;
    log_t(tab, T, hi, lo);
    const double ln = hi + lo, a1 = t.T2 * iT, a2 = t.T4 * iT, a3 = T * t.icxhi;
    rate -= c.imlc_k * exp_any(tab, -t.T1 * iT - a1 * a1);
    rate -= c.nmlc_k * exp_any(tab, -t.T3 * iT - a2 * a2);
    rate -= c.cehi_k * exp_any(tab, 2.302585093 * log_spline_t(t, tab, hi, lo) - a3 * a3);
    if (T > t.ciec_minT) {
        const double p163 = exp_any(tab, 1.63 * (ln - 11.512925464970228420));
        const double smoothing = (T - 5.0e4) / 2.0e4;
        rate -= c.ciec_k * exp_any(tab, -0.63 * ln) * (1.0 - exp_any(tab, -p163)) * (smoothing < 1.0 ? smoothing : 1.0);
    }
    return rate - c.nmc_k * exp_any(tab, 0.5 * ln - c.nmc_T0 * iT);
}

// Sum of the five cooling terms, subtracted in the reference's order from
// `rate` (Thermodynamics.cpp:255-259 / 315-319).  The transcendental work is
// shared between the terms: one reciprocal and one natural log of T feed
// every exponent (x/T = x * (1/T); log10 T = ln T / ln 10; sqrt(T) e^-a =
// e^(ln T / 2 - a); pow(1e-5 T, 1.63) = e^(1.63 (ln T + ln 1e-5)) and T^-0.63
// = T / T^1.63), leaving four exponentials per evaluation (six above
// ciec_minT) instead of ten libm calls.  The values differ from the
// reference's by rounding of the exponents only (relative ~1e-15 on each
// term).
template <bool EVEN>
__device__ __forceinline__ double subtract_cooling(const RateConsts<EVEN>& t, const CoolingCell& c, const double* tab,
                                                   double rate, double T) {
    if (!(T >= 1e-100 && T <= 1e100)) return subtract_cooling_far(t, c, tab, rate, T);
    const double iT = rcp_t(T);
    double hi, lo;
    log_t(tab, T, hi, lo);
    const double a1 = t.T2 * iT, a2 = t.T4 * iT, a3 = T * t.icxhi;
    double e[4] = {exp_floor(__builtin_fma(-a1, a1, -t.T1 * iT)), exp_floor(__builtin_fma(-a2, a2, -t.T3 * iT)),
                   exp_floor(__builtin_fma(2.302585093, log_spline_t(t, tab, hi, lo), -(a3 * a3))),
                   exp_floor(__builtin_fma(0.5, lo, __builtin_fma(-c.nmc_T0, iT, 0.5 * hi)))};
    exp_n<4>(tab, e);
    rate -= c.imlc_k * e[0];
    rate -= c.nmlc_k * e[1];
    rate -= c.cehi_k * e[2];
    if (T > t.ciec_minT) {
        // ln (1e-5 T), ln 1e5 being a multiple of 2^-40 and a rest
        const double l5 = (hi - 0x1.7069e2aa2aap3) + (lo - 0x1.6b8e527645db3p-43);
        const double p163 = exp_t(tab, exp_floor(1.63 * l5));
        // T^-0.63 = T (1e5)^-1.63 / (1e-5 T)^1.63
        const double cie_rate = c.ciec_k * (T * 7.0794578438413791080e-9 * rcp_t(p163)) *
                                (1.0 - exp_t(tab, exp_floor(-p163)));
        const double x = T - 5.0e4, q = x * 5.0e-5;  // x / 2e4, rounded as the division rounds it
        double smoothing = __builtin_fma(__builtin_fma(-2.0e4, q, x), 5.0e-5, q);
        smoothing = (smoothing < 1.0) ? smoothing : 1.0;
        rate -= cie_rate * smoothing;
    }
    rate -= c.nmc_k * e[3];
    return rate;
}

// Heating terms FUVH + IRH + CRH (Thermodynamics.cpp:178-191, 249-251);
// e^(-2 ln u) is 1 / u^2.
__device__ __forceinline__ double heating(const ThermoConsts& t, const double* tab, double nH, double Av, double F) {
    double rate = 0;
    const double ea = exp_any(tab, -1.9 * Av);
    const double iu = 1.0 / (1.0 + t.irh_b / nH);
    rate += t.fuvh_a * nH * F * ea / (t.fuvh_b + t.fuvh_c * F * ea / nH);
    rate += t.irh_a * nH * F * exp_any(tab, -0.05 * Av) * (iu * iu);
    rate += t.crh * nH;
    return rate;
}

// The heating and cooling terms one by one, as Thermodynamics::
// fillHeatingArrays writes them into GridCell::H (Thermodynamics.cpp:445-457,
// the term functions :121-191): ionised and neutral metal lines, HI
// collisional excitation, collisional ionisation equilibrium and neutral /
// molecular cooling (negated), FUV, IR and cosmic-ray heating.  Written with
// the reference's own operations (one libm call per exponential), not the
// shared-log form of subtract_cooling.  Order of H: IMLC, NMLC, RHII, CEHI,
// CIEC, NMC, EUVH, FUVH, IRH, CRH, TOT (Common.hpp:32-34); RHII, EUVH and
// TOT are left to the caller.
__device__ __forceinline__ void heating_terms(const ThermoConsts& t, const double* sx, const double* sy,
                                              const double* sy2, double nH, double x, double T, double Av,
                                              double F, double H[11]) {
    const double ne = x * nH, nn = (1.0 - x) * nH;
    H[7] = t.fuvh_a * nH * F * exp(-1.9 * Av) / (t.fuvh_b + t.fuvh_c * F * exp(-1.9 * Av) / nH);
    H[8] = t.irh_a * nH * F * exp(-0.05 * Av) * exp(-2.0 * log(1.0 + t.irh_b / nH));
    H[9] = t.crh * nH;
    H[0] = -(t.imlc * t.z0 * ne * ne * exp(-t.T1 / T - (t.T2 / T) * (t.T2 / T)));
    H[1] = -(t.nmlc * t.z0 * ne * nn * exp(-t.T3 / T - (t.T4 / T) * (t.T4 / T)));
    {
        const double r = log_spline(t, sx, sy, sy2, log10(T));
        H[3] = -(x * (1.0 - x) * nH * nH * exp((2.302585093 * r) - ((T / t.cxhi_damp) * (T / t.cxhi_damp))));
    }
    if (T > t.ciec_minT) {
        const double cie = t.ciec * ne * ne * t.z0 * exp(-0.63 * log(T)) * (1.0 - exp(-pow(1.0e-5 * T, 1.63)));
        double smoothing = (T - 5.0e4) / (2.0e4);
        smoothing = (smoothing < 1.0) ? smoothing : 1.0;
        H[4] = -(cie * smoothing);
    } else {
        H[4] = -0.0;
    }
    {
        const double T0 = 70.0 + 220.0 * pow(nH / t.n0, 0.2);
        H[5] = -(t.nmc * (1.0 - x) * (1.0 - x) * pow(nH, 1.6) * sqrt(T) * exp(-T0 / T));
    }
}

}  // namespace tg
