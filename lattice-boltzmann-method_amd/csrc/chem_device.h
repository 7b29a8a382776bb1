// Thermo, kinetics, transport and unit conversions of the multicomponent
// path, as __host__ __device__ functions over the generated mechanism tables
// (mech.h).
//
// These replace the Cantera calls the reference makes per cell (ideal-gas
// NASA7 thermo, setState_UV / TD / TP, getNetProductionRates with
// Arrhenius, third-body, Troe and Lindemann falloff and pressure-dependent
// Arrhenius (PLOG) reactions and reverse rates from equilibrium constants,
// mixture-averaged transport) and the binary32
// Units_Conv crossings between lattice and SI units (units.hpp:75-131).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>

#include "mech.h"

namespace lbm {
namespace chem {

using namespace mech;
constexpr double SPECIES_MIN = 1e-8;  // defines.hpp:96

// 1 / W_a, for products in place of divisions by the molar masses
struct InvW {
    double v[NS];
};
constexpr InvW make_inv_w()
{
    InvW r{};
    for (int a = 0; a < NS; ++a) r.v[a] = 1.0 / W[a];
    return r;
}
constexpr InvW INV_W_TABLE = make_inv_w();
__host__ __device__ inline double inv_w(int a) { return INV_W_TABLE.v[a]; }

// Reciprocal of the FP32 path's binary32 transport: the hardware's, within 1 ulp.
__host__ __device__ inline float rcp_r(float x)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return __builtin_amdgcn_rcpf(x);
#else
    return 1.0f / x;
#endif
}

// ------------------------------------------------------------ quotients
// The binary64 kernels are bound by their arithmetic, and a division is the
// dearest of it: the compiled sequence (scaling, reciprocal, Newton steps,
// residual, fix-up) issues 11 operations, and divisions made up half to two
// thirds of the binary64 operations of the chemistry, transport, collide and
// moment kernels.  Most of their divisors are constants (molar masses) or shared
// by many quotients (rho, T, a pivot), so a divisor carries its reciprocal
// and a quotient takes three: the approximate quotient, its exact residual by
// fused multiply-add and the correction (Markstein 1990).  With y the correctly
// rounded 1 / b the result is the correctly rounded quotient, bit for bit that of
// `/`, for divisors and quotients in the normal range.  (With y the other
// neighbour of 1 / b it is not for three in ten of the quotients that lie as close
// to the middle of two numbers as they come.)  The Newton steps of divisor() give
// the correctly rounded y unless 1 / b lies within 2^-88 of itself of a middle:
// for a few divisors less than 2^-42 below a power of two, over which a quotient
// next to a middle may round to the other side (1 over 2 - 2^-52 does).  Tested
// on the host and on the device.  A zero or infinite divisor and an infinite
// quotient give NaN, and -0 gives 0: a division that may meet one is written `/`.
// Host code divides.
struct Divisor {
    double b, y;  // the divisor and 1 / b, correctly rounded
};
// a / d.b by the residual correction
__host__ __device__ inline double quotient_fma(double a, const Divisor& d)
{
    const double q = a * d.y;
    const double r = __builtin_fma(-q, d.b, a);
    return __builtin_fma(r, d.y, q);
}
// 1 / b: the hardware's approximate reciprocal (2^-22 or better) and two Newton
// steps, 2^-88 before the last rounding
__host__ __device__ inline Divisor divisor(double b)
{
#if defined(__HIP_DEVICE_COMPILE__)
    double y = __builtin_amdgcn_rcp(b);
    y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
    y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
    return {b, y};
#else
    return {b, 1.0 / b};
#endif
}
__host__ __device__ inline double quot(double a, const Divisor& d)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return quotient_fma(a, d);
#else
    return a / d.b;
#endif
}
__host__ __device__ inline double quot(double a, double b) { return quot(a, divisor(b)); }
// a / b of binary32 numbers through the binary64 reciprocal y of b: a
// quotient of two 24-bit numbers is at least 2^-50 of itself away from the middle
// of two binary32 numbers, so rounding a y (2^-52 off) gives the rounded quotient
__host__ __device__ inline float quotf(float a, float b, double y)
{
#if defined(__HIP_DEVICE_COMPILE__)
    return (float)((double)a * y);
#else
    return a / b;
#endif
}
// quotients by constants
__host__ __device__ inline double third(double x) { return quot(x, Divisor{3.0, 1.0 / 3.0}); }
__host__ __device__ inline double fifth(double x) { return quot(x, Divisor{5.0, 1.0 / 5.0}); }
__host__ __device__ inline double over_w(double x, int k) { return quot(x, Divisor{W[k], INV_W_TABLE.v[k]}); }

// ---------------------------------------------------------------- units
// Units_Conv after set_m_kg_s(dx, dt): m, kg, s, K stored as float; every
// conversion rounds its argument to float and computes in float, or in
// double where the reference's double cb()/sq() enters, then returns float.
// The y_ members are the reciprocals of the conversions' divisors for device
// code (make_units sets them).
struct Units {
    float m, kg, s, K;
    double y_K = 0, y_mm = 0, y_ss = 0, y_m = 0, y_kg = 0, y_kgm = 0;  // binary32 divisors K, m m, s s, m, kg, kg m
    double y_m3 = 0, y_m2 = 0, y_mss = 0;                              // binary64 divisors m^3, m^2, m s^2

    __host__ __device__ float temp(double x) const { return quotf((float)x, K, y_K); }
    __host__ __device__ float si_temp(double x) const { return (float)x * K; }
    __host__ __device__ float energy_mass(double x) const { return quotf((float)x * (s * s), m * m, y_mm); }
    __host__ __device__ float si_energy_mass(double x) const { return quotf((float)x * (m * m), s * s, y_ss); }
    __host__ __device__ float u(double x) const { return quotf((float)x * s, m, y_m); }  // velocity
    __host__ __device__ float rho(double x) const
    {
        const double md = m;
        return (float)quot((double)(float)x * (md * md * md), Divisor{(double)kg, y_kg});
    }
    __host__ __device__ float si_rho(double x) const
    {
        const double md = m;
        return (float)quot((double)((float)x * kg), Divisor{md * md * md, y_m3});
    }
    __host__ __device__ float rho_dot(double x) const
    {
        const double md = m;
        return (float)quot((double)(float)x * (md * md * md) * (double)s, Divisor{(double)kg, y_kg});
    }
    __host__ __device__ float nu(double x) const
    {
        const double md = m;
        return (float)quot((double)((float)x * s), Divisor{md * md, y_m2});
    }
    __host__ __device__ float mu(double x) const { return quotf((float)x * s * m, kg, y_kg); }
    __host__ __device__ float thermal_conductivity(double x) const
    {
        return quotf((float)x * s * s * s * K, kg * m, y_kgm);
    }
    __host__ __device__ float cp(double x) const { return quotf((float)x * s * s * K, m * m, y_mm); }
    __host__ __device__ float p(double x) const
    {
        const double sd = s;
        return (float)quot((double)(float)x * ((double)m * (sd * sd)), Divisor{(double)kg, y_kg});
    }
    __host__ __device__ float si_p(double x) const
    {
        const double sd = s;
        return (float)quot((double)((float)x * kg), Divisor{(double)m * (sd * sd), y_mss});
    }
};

// set_m_kg_s(dx, dt) of units.hpp:32-44.
inline Units make_units(double dx, double dt)
{
    Units u;
    u.m = (float)((double)(float)dx / 1.0);
    const double md = u.m;
    u.kg = (float)(1.0 / 1.0 * (md * md * md));
    u.s = (float)((double)(float)dt / 1.0);
    u.K = 12000.0f;
    const float mm = u.m * u.m, ss = u.s * u.s, kgm = u.kg * u.m;
    const double sd = u.s;
    u.y_K = 1.0 / (double)u.K;
    u.y_mm = 1.0 / (double)mm;
    u.y_ss = 1.0 / (double)ss;
    u.y_m = 1.0 / (double)u.m;
    u.y_kg = 1.0 / (double)u.kg;
    u.y_kgm = 1.0 / (double)kgm;
    u.y_m3 = 1.0 / (md * md * md);
    u.y_m2 = 1.0 / (md * md);
    u.y_mss = 1.0 / ((double)u.m * (sd * sd));
    return u;
}

// --------------------------------------------------------------- thermo
// Rows of the coefficients a0..a6 and a2 / 3.
struct NasaRows {
    double v[NS][8];
};
constexpr NasaRows nasa_rows(const double (&t)[NS][7])
{
    NasaRows r{};
    for (int k = 0; k < NS; ++k) {
        for (int i = 0; i < 7; ++i) r.v[k][i] = t[k][i];
        r.v[k][7] = t[k][2] / 3;
    }
    return r;
}
constexpr NasaRows ROWS_LO = nasa_rows(NASA_LO), ROWS_HI = nasa_rows(NASA_HI);
__host__ __device__ inline const double* nasa(int k, double T) { return T < T_MID[k] ? ROWS_LO.v[k] : ROWS_HI.v[k]; }

// Which side of T_MID the temperature lies on, as a branch.  Chosen by address,
// a species' row is eight vector loads and as many register pairs per lane;
// on either side of a branch the rows are constants in scalar registers, and
// a wavefront runs both sides only when its lanes straddle T_MID.  Mechanisms
// whose species differ in T_MID keep the choice by address.
enum : int { SIDE_LO = 0, SIDE_HI = 1, SIDE_MIXED = 2 };
template <int S>
struct Side {
    static constexpr int side = S;
};
constexpr bool one_t_mid()
{
    for (int k = 1; k < NS; ++k)
        if (T_MID[k] != T_MID[0]) return false;
    return true;
}
template <int S>
__host__ __device__ inline const double* nasa_row(int k, double T)
{
    if constexpr (S == SIDE_LO) return ROWS_LO.v[k];
    if constexpr (S == SIDE_HI) return ROWS_HI.v[k];
    return nasa(k, T);
}
template <typename Body>
__host__ __device__ inline void by_side(double T, Body body)
{
    if constexpr (one_t_mid()) {
        if (T < T_MID[0]) body(Side<SIDE_LO>{});
        else body(Side<SIDE_HI>{});
    } else {
        body(Side<SIDE_MIXED>{});
    }
}

template <int S = SIDE_MIXED>
__host__ __device__ inline double cp_R(int k, double T)
{
    const double* a = nasa_row<S>(k, T);
    return a[0] + T * (a[1] + T * (a[2] + T * (a[3] + T * a[4])));
}

template <int S = SIDE_MIXED>
__host__ __device__ inline double h_RT(int k, double T)
{
    const double* a = nasa_row<S>(k, T);
    const double t4 = fifth(T * a[4]);
    return a[0] + T * (a[1] / 2 + T * (a[7] + T * (a[3] / 4 + t4))) + quot(a[5], T);
}

template <int S = SIDE_MIXED>
__host__ __device__ inline double s_R(int k, double T, double lnT)
{
    const double* a = nasa_row<S>(k, T);
    return a[0] * lnT + T * (a[1] + T * (a[2] / 2 + T * (third(a[3]) + T * a[4] / 4))) + a[6];
}

// Cantera's setMassFractions: negatives clipped, then normalised.
__host__ __device__ inline void normalize(double Y[NS])
{
    double s = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        Y[k] = Y[k] > 0.0 ? Y[k] : 0.0;
        s += Y[k];
    }
    const double inv = quot(1.0, s);
#pragma unroll
    for (int k = 0; k < NS; ++k) Y[k] *= inv;
}

// FAST = true (the FP32 path): products with 1/W and one reciprocal in place
// of a division per species (each result within a few ulp of the exact
// form, which the plain path keeps).
template <bool FAST = false>
__host__ __device__ inline double mean_W(const double Y[NS])
{
    double s = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) s += FAST ? Y[k] * inv_w(k) : over_w(Y[k], k);
    return quot(1.0, s);
}

template <bool FAST = false>
__host__ __device__ inline void X_from_Y(const double Y[NS], double X[NS])
{
    double s = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        X[k] = FAST ? Y[k] * inv_w(k) : over_w(Y[k], k);
        s += X[k];
    }
    if constexpr (FAST) {
        const double is = quot(1.0, s);
#pragma unroll
        for (int k = 0; k < NS; ++k) X[k] *= is;
    } else {
        const Divisor ds = divisor(s);
#pragma unroll
        for (int k = 0; k < NS; ++k) X[k] = quot(X[k], ds);
    }
}

__host__ __device__ inline void Y_from_X(const double X[NS], double Y[NS])
{
    double s = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        Y[k] = (X[k] > 0.0 ? X[k] : 0.0) * W[k];
        s += Y[k];
    }
    const Divisor ds = divisor(s);
#pragma unroll
    for (int k = 0; k < NS; ++k) Y[k] = quot(Y[k], ds);
}

template <bool FAST = false>
__host__ __device__ inline double cp_mass(double T, const double Y[NS])
{
    double s = 0;
    by_side(T, [&](auto sd) {
#pragma unroll
        for (int k = 0; k < NS; ++k)
            s += FAST ? Y[k] * cp_R<sd.side>(k, T) * inv_w(k) : over_w(Y[k] * cp_R<sd.side>(k, T), k);
    });
    return s * R_UNIV;
}

// h / RT with the reciprocal temperature given (one division per state
// instead of one per species)
template <int S = SIDE_MIXED>
__host__ __device__ inline double h_RT_inv(int k, double T, double invT)
{
    const double* a = nasa_row<S>(k, T);
    const double t4 = fifth(T * a[4]);
    return a[0] + T * (a[1] / 2 + T * (a[7] + T * (a[3] / 4 + t4))) + a[5] * invT;
}

__host__ __device__ inline double u_mass(double T, const double Y[NS])
{
    double s = 0;
    by_side(T, [&](auto sd) {
#pragma unroll
        for (int k = 0; k < NS; ++k) s += over_w(Y[k] * (h_RT<sd.side>(k, T) - 1.0), k);
    });
    return s * R_UNIV * T;
}

// setState_UV at fixed composition (tolerance 1e-15 as the reference asks):
// Newton on u(T) = u_target from the current temperature T0.
// (FAST: Y/W hoisted as products with 1/W, one reciprocal of T per
// iteration; the same Newton and stopping rule.)
template <bool FAST = false>
__host__ __device__ inline double T_from_UV(double u_target, const double Y[NS], double T0)
{
    double T = T0;
    if constexpr (FAST) {
        double yw[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) yw[k] = Y[k] * inv_w(k);
        for (int it = 0; it < 60; ++it) {
            const double invT = quot(1.0, T);
            double u = 0, cv = 0;
            by_side(T, [&](auto sd) {
#pragma unroll
                for (int k = 0; k < NS; ++k) {
                    u += yw[k] * (h_RT_inv<sd.side>(k, T, invT) - 1.0);
                    cv += yw[k] * (cp_R<sd.side>(k, T) - 1.0);
                }
            });
            const double dT = quot(-(u * R_UNIV * T - u_target), cv * R_UNIV);
            T += dT;
            if (fabs(dT) <= 1e-15 * fabs(T)) break;
        }
        return T;
    }
    double yw[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) yw[k] = over_w(Y[k], k);
    for (int it = 0; it < 60; ++it) {
        double u = 0, cv = 0;
        by_side(T, [&](auto sd) {
#pragma unroll
            for (int k = 0; k < NS; ++k) {
                u += yw[k] * (h_RT<sd.side>(k, T) - 1.0);
                cv += yw[k] * (cp_R<sd.side>(k, T) - 1.0);
            }
        });
        const double dT = quot(-(u * R_UNIV * T - u_target), cv * R_UNIV);
        T += dT;
        if (fabs(dT) <= 1e-15 * fabs(T)) break;
    }
    return T;
}

template <bool FAST = false>
__host__ __device__ inline double pressure(double T, double rho, const double Y[NS])
{
    if constexpr (FAST) {
        double s = 0;
#pragma unroll
        for (int k = 0; k < NS; ++k) s += Y[k] * inv_w(k);
        return rho * R_UNIV * T * s;
    }
    return quot(rho * R_UNIV * T, mean_W(Y));
}

// ------------------------------------------------------------ kinetics
// Concentration factor C^o of a rate of progress: plain products for the
// exponents 0-3 (any sign of C), otherwise (fractional reaction orders) C^o
// when C > 0, else 0 (Cantera's rule for non-integer exponents).  The
// exponents are table constants, so the branches fold at compile time.
__host__ __device__ inline double conc_power(double c, double o)
{
    if (o == 0.0) return 1.0;
    if (o == 1.0) return c;
    if (o == 2.0) return c * c;
    if (o == 3.0) return c * c * c;
    return c > 0.0 ? pow(c, o) : 0.0;
}

// Pressure-dependent Arrhenius (PLOG) rate of reaction r at ln P [Pa]:
// ln k interpolated linearly in ln P between the two bracketing levels, the
// first (last) level's rate below (above) the table (Cantera's PlogRate).
__host__ __device__ inline double plog_rate(int r, double lnT, double invT, double lnP)
{
    const int n = PLOG_N[r];
    auto lnk = [&](int i) { return PLOG_LNA[r][i] + PLOG_B[r][i] * lnT - PLOG_EA_R[r][i] * invT; };
    if (lnP <= PLOG_LNP[r][0]) return exp(lnk(0));
    for (int i = 0; i + 1 < n; ++i) {
        if (lnP < PLOG_LNP[r][i + 1]) {
            const double w = (lnP - PLOG_LNP[r][i]) * (1.0 / (PLOG_LNP[r][i + 1] - PLOG_LNP[r][i]));
            const double l1 = lnk(i);
            return exp(l1 + (lnk(i + 1) - l1) * w);
        }
    }
    return exp(lnk(n - 1));
}

constexpr bool any_plog()
{
    for (int r = 0; r < NR; ++r)
        if (PLOG_N[r] > 0) return true;
    return false;
}

// log10 of Troe's broadening factor from log10 of the reduced pressure and of
// the factor at its centre.  Plain divisions: where the inner divisor passes
// through zero its quotient is infinite and the factor 1, and through a
// reciprocal it would be NaN.
__host__ __device__ inline double troe_log_f(double lPr, double lFc)
{
    const double cc = -0.4 - 0.67 * lFc;
    const double nn = 0.75 - 1.27 * lFc;
    const double f1 = (lPr + cc) / (nn - 0.14 * (lPr + cc));
    return lFc / (1.0 + f1 * f1);
}

// Net molar production rates [kmol/m^3/s] at (T, rho, Y), SI units.
__host__ __device__ inline void net_production(double T, double rho, const double Y[NS], double wdot[NS])
{
    double C[NS], gRT[NS];
    const double lnT = log(T), invT = quot(1.0, T);
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        C[k] = over_w(rho * Y[k], k);
        wdot[k] = 0.0;
    }
    by_side(T, [&](auto sd) {
#pragma unroll
        for (int k = 0; k < NS; ++k) gRT[k] = h_RT<sd.side>(k, T) - s_R<sd.side>(k, T, lnT);
    });
    const double ln_pref_RT = log(quot(P_REF, R_UNIV * T));
    // ln p of the PLOG rates, p = R T sum_k C_k
    double lnP = 0.0;
    if constexpr (any_plog()) {
        double Ct = 0.0;
#pragma unroll
        for (int k = 0; k < NS; ++k) Ct += C[k];
        lnP = log(R_UNIV * T * Ct);
    }
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        // (a rate with b = 0 and Ea = 0 is A: exp(0) = 1 is not evaluated)
        double kf = KIND[r] == 3                                ? plog_rate(r, lnT, invT, lnP)
                    : ARR_B[r] == 0.0 && ARR_EA_R[r] == 0.0 ? ARR_A[r]
                                                              : ARR_A[r] * exp(ARR_B[r] * lnT - ARR_EA_R[r] * invT);
        if (KIND[r] == 1 || KIND[r] == 2) {
            double M = 0;
#pragma unroll
            for (int k = 0; k < NS; ++k)
                if (EFF[r][k] != 0.0) M += EFF[r][k] * C[k];
            if (KIND[r] == 1) {
                kf *= M;
            } else {
                const double k0 = LOW_A[r] * exp(LOW_B[r] * lnT - LOW_EA_R[r] * invT);
                const double Pr = quot(k0 * M, kf);
                if (TROE_ON[r]) {
                    double Fc = (1.0 - TROE[r][0]) * exp(quot(-T, Divisor{TROE[r][1], 1.0 / TROE[r][1]})) +
                                TROE[r][0] * exp(quot(-T, Divisor{TROE[r][2], 1.0 / TROE[r][2]}));
                    if (TROE_HAS_T2[r]) Fc += exp(-TROE[r][3] * invT);
                    const double lPr = log10(Pr > 1e-300 ? Pr : 1e-300);
                    kf = quot(kf * Pr, 1.0 + Pr) * exp10(troe_log_f(lPr, log10(Fc)));
                } else {  // Lindemann: broadening factor 1
                    kf = quot(kf * Pr, 1.0 + Pr);
                }
            }
        }
        double dG = 0, dn = 0, cf = 1, cr = 1;
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            // species the reaction leaves alone add nothing (the table's zeros
            // do not fold by themselves: 0 x is not 0 for every x)
            if (NU_R[r][k] - NU_F[r][k] != 0.0) dG += (NU_R[r][k] - NU_F[r][k]) * gRT[k];
            dn += NU_R[r][k] - NU_F[r][k];
            cf *= conc_power(C[k], ORD_F[r][k]);
            cr *= conc_power(C[k], NU_R[r][k]);
        }
        // k_r = k_f / K_c, K_c = exp(-dG) (p_ref / RT)^dn; 0 for irreversible steps
        const double kr = REVERSIBLE[r] ? kf * exp(dG - dn * ln_pref_RT) : 0.0;
        const double q = kf * cf - kr * cr;
#pragma unroll
        for (int k = 0; k < NS; ++k)
            if (NU_R[r][k] - NU_F[r][k] != 0.0) wdot[k] += (NU_R[r][k] - NU_F[r][k]) * q;
    }
}

// ------------------------------------------------------------ transport
__host__ __device__ inline double poly4(const double c[5], double x)
{
    return c[0] + x * (c[1] + x * (c[2] + x * (c[3] + x * c[4])));
}

__host__ __device__ inline double species_viscosity(int k, double lnT) { return exp(poly4(VISC_FIT[k], lnT)); }
__host__ __device__ inline double species_conductivity(int k, double lnT) { return exp(poly4(COND_FIT[k], lnT)); }
// D_ab [m^2/s] at (T, p).
__host__ __device__ inline double binary_diff(int a, int b, double lnT, double p)
{
    return quot(exp(poly4(DIFF_FIT[a][b], lnT)), p);
}

// The same fits evaluated in arithmetic type R (double reproduces the
// functions above bit for bit; float is the FP32 path's binary32 transport).
template <typename R>
__host__ __device__ inline R poly4r(const double c[5], R x)
{
    return (R)c[0] + x * ((R)c[1] + x * ((R)c[2] + x * ((R)c[3] + x * (R)c[4])));
}
__host__ __device__ inline float species_viscosity_f(int k, float lnT) { return exp(poly4r<float>(VISC_FIT[k], lnT)); }

// Divisor sqrt(8 (1 + W_a / W_b)) of the Wilke weights
__host__ __device__ inline Divisor wilke_divisor(int a, int b)
{
    const double d = sqrt(8.0 * (1.0 + W[a] / W[b]));
    return {d, 1.0 / d};
}

// Wilke weight Phi_ab with sqrt(mu_a / mu_b) given: (1 + sqrt(mu_a/mu_b)
// (W_b/W_a)^(1/4))^2 / sqrt(8 (1 + W_a/W_b)), the W factors folded at compile time.
__host__ __device__ inline float wilke_phi(int a, int b, float sq_ratio)
{
    const float r = 1.0f + sq_ratio * (float)sqrt(sqrt(W[b] / W[a]));
    return r * r * (float)(1.0 / sqrt(8.0 * (1.0 + W[a] / W[b])));
}

// Wilke mixture viscosity with the direct Phi_ab formula.
__host__ __device__ inline double mix_viscosity(double lnT, const double X[NS])
{
    double mu[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) mu[k] = species_viscosity(k, lnT);
    double tot = 0;
#pragma unroll
    for (int a = 0; a < NS; ++a) {
        double den = 0;
#pragma unroll
        for (int b = 0; b < NS; ++b) {
            const double r = 1.0 + sqrt(mu[a] / mu[b]) * sqrt(sqrt(W[b] / W[a]));
            den += X[b] * (r * r / sqrt(8.0 * (1.0 + W[a] / W[b])));
        }
        tot += X[a] * mu[a] / den;
    }
    return tot;
}

template <typename R>
__host__ __device__ inline R mix_viscosity_r(R lnT, const double X[NS])
{
    if constexpr (sizeof(R) == 4) {
        // sqrt(mu_a / mu_b) = sqrt(mu_a) / sqrt(mu_b): 9 square roots and
        // reciprocals in place of 81 divisions and square roots
        float mu[NS], sm[NS], rsm[NS];
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            mu[k] = species_viscosity_f(k, lnT);
            sm[k] = sqrt(mu[k]);
            rsm[k] = rcp_r(sm[k]);
        }
        float tot = 0;
#pragma unroll
        for (int a = 0; a < NS; ++a) {
            float den = 0;
#pragma unroll
            for (int b = 0; b < NS; ++b) den += (float)X[b] * wilke_phi(a, b, sm[a] * rsm[b]);
            tot += (float)X[a] * mu[a] * rcp_r(den);
        }
        return tot;
    }
    double mu[NS];
    Divisor dmu[NS];
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        mu[k] = species_viscosity(k, lnT);
        dmu[k] = divisor(mu[k]);
    }
    double tot = 0;
#pragma unroll
    for (int a = 0; a < NS; ++a) {
        double den = 0;
#pragma unroll
        for (int b = 0; b < NS; ++b) {
            if (b == a) {  // Phi_aa = 1
                den += X[a];
                continue;
            }
            const double r = 1.0 + sqrt(quot(mu[a], dmu[b])) * sqrt(sqrt(W[b] / W[a]));
            den += X[b] * quot(r * r, wilke_divisor(a, b));
        }
        tot += quot(X[a] * mu[a], den);
    }
    return tot;
}

template <typename R, typename XT = double>
__host__ __device__ inline R mix_conductivity_r(R lnT, const XT X[NS])
{
    R s1 = 0, s2 = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const R l = exp(poly4r<R>(COND_FIT[k], lnT));
        s1 += (R)X[k] * l;
        if constexpr (sizeof(R) == 4)
            s2 += (R)X[k] * rcp_r(l);
        else
            s2 += quot((double)X[k], (double)l);
    }
    if constexpr (sizeof(R) == 4) return R(0.5) * (s1 + rcp_r(s2));
    return R(0.5) * (s1 + R(quot(1.0, (double)s2)));
}

// Combination-averaged mixture conductivity 1/2 (sum X l + 1 / sum X / l).
__host__ __device__ inline double mix_conductivity(double lnT, const double X[NS])
{
    double s1 = 0, s2 = 0;
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const double l = species_conductivity(k, lnT);
        s1 += X[k] * l;
        s2 += X[k] / l;
    }
    return 0.5 * (s1 + 1.0 / s2);
}

}  // namespace chem
}  // namespace lbm
