// obme_device.h — device-side building blocks of the gfx950 biogeochemistry
// step: Julia scalar semantics, precision-dispatched math, the
// NutrientsPlanktonDetritus tendencies (NPZD, LOBSTER + CarbonateSystem) and
// the FP64 carbonate chemistry (constants, alkalinity residual, damped
// Newton, pCO2, CO2 gas-exchange flux).
//
// FT = double is the plain FP64 path (the reference's arithmetic, operand
// order kept in the carbonate chemistry; the transitions agree to rounding).  FT = float is the
// FP32-mixed path: native v_exp/v_log/v_rcp based transcendentals and
// divisions on the vector ALUs; the carbonate chemistry is always FP64.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "../../include/obme.h"

namespace obme {

// ---------------------------------------------------------------- scalars

// Julia Base min/max for IEEE floats (NaN propagates; -0 < 0): the minimum and
// maximum of IEEE 754-2019.  FP32: one hardware instruction (a difference, its
// sign and two selects take five: a third of the PISCES transitions'
// comparisons and selects).  FP64: the hardware's minimum, which orders the
// zeros, a comparison and two selects for NaN.
template <typename FT>
__device__ __forceinline__ FT jmin(FT x, FT y) { return __builtin_elementwise_minimum(x, y); }
template <typename FT>
__device__ __forceinline__ FT jmax(FT x, FT y) { return __builtin_elementwise_maximum(x, y); }

// Precision-dispatched math.  FP64: the accurate device library.  FP32:
// the hardware instructions v_exp_f32 (2^x), v_log_f32 (log2 x),
// v_rcp_f32 and v_sqrt_f32 (about 1 ulp each).
__device__ __forceinline__ double m_div(double a, double b) { return a / b; }
__device__ __forceinline__ float m_div(float a, float b) { return a * __builtin_amdgcn_rcpf(b); }
__device__ __forceinline__ double m_exp2(double x) { return exp2(x); }
__device__ __forceinline__ float m_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ double m_log2(double x) { return log2(x); }
__device__ __forceinline__ float m_log2(float x) { return __builtin_amdgcn_logf(x); }
__device__ __forceinline__ double m_exp(double x) { return exp(x); }
__device__ __forceinline__ float m_exp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }
__device__ __forceinline__ double m_sqrt(double x) { return sqrt(x); }
__device__ __forceinline__ float m_sqrt(float x) { return __builtin_amdgcn_sqrtf(x); }
// 1/x: the hardware's estimate; FP64 with two Newton steps (36 cycles of a
// wave where the IEEE quotient takes 65; within 1 ulp, NaN for x = 0 or
// infinite).
__device__ __forceinline__ float m_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double m_rcp(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}
// 1/sqrt(x), x > 0 and finite: the same way.
__device__ __forceinline__ float m_rsqrt(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double m_rsqrt(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    y = fma(0.5 * y, fma(-(x * y), y, 1.0), y);
    return fma(0.5 * y, fma(-(x * y), y, 1.0), y);
}
// log x for a finite x > 0, within 1 ulp: x = 2^k (1 + f), 1 + f in
// [sqrt(1/2), sqrt(2)), s = f / (2 + f), log(1 + f) = 2 atanh s =
// f - (f^2/2 - s (f^2/2 + R(s^2))), R the series 2 (z/3 + z^2/5 + ...) to
// z^9 (z <= 0.0295: the rest is below 2^-55 of the logarithm).  About 150 cycles of a wave
// where the library's log takes 365.
__device__ __forceinline__ double log_positive(double x)
{
    double m = __builtin_amdgcn_frexp_mant(x);         // [1/2, 1)
    int k = __builtin_amdgcn_frexp_exp(x);
    const bool lo = m < 0.70710678118654752;
    m = lo ? m + m : m;
    k = lo ? k - 1 : k;
    const double f = m - 1.0;
    const double s = f * m_rcp(2.0 + f);
    const double z = s * s;
    double R = fma(z, 2.0 / 19, 2.0 / 17);
    R = fma(z, R, 2.0 / 15);
    R = fma(z, R, 2.0 / 13);
    R = fma(z, R, 2.0 / 11);
    R = fma(z, R, 2.0 / 9);
    R = fma(z, R, 2.0 / 7);
    R = fma(z, R, 2.0 / 5);
    R = fma(z, R, 2.0 / 3);
    R = z * R;
    const double h = 0.5 * f * f;
    const double dk = (double)k;
    // ln 2 in two parts, the first a multiple of 2^-42: k times it is exact
    const double ln2h = 0x1.62e42fefa3800p-1, ln2l = 0x1.ef35793c76730p-45;
    return fma(dk, ln2h, f - (h - fma(s, h + R, dk * ln2l)));
}
// log x with log's values at x <= 0, infinity and NaN.
__device__ __forceinline__ double m_log_any(double x)
{
    double l = log_positive(x);
    if (!(x > 0.0 && x < HUGE_VAL))
        l = x == 0.0 ? -HUGE_VAL : (x > 0.0 ? x : __longlong_as_double(0x7ff8000000000000ll));
    return l;
}
// 10^x and log10 x through e, the products' rounding errors put back (about
// 130 and 170 cycles of a wave; pow(10, x) takes 600, the library's log10 380).
__device__ __forceinline__ double m_exp10(double x)
{
    const double c = 0x1.26bb1bbb55516p+1, cl = -0x1.f48ad494ea3e9p-53;   // ln 10
    const double p = x * c;
    const double r = exp(p);
    const double q = fma(r, fma(x, c, -p) + x * cl, r);
    return q < HUGE_VAL ? q : r;    // (overflow: the correction is inf * 0)
}
__device__ __forceinline__ double m_log10(double x)
{
    const double c = 0x1.bcb7b1526e50ep-2, cl = 0x1.95355baaafad3p-57;    // 1 / ln 10
    const double L = m_log_any(x);
    const double p = L * c;
    return p + (fma(L, c, -p) + L * cl);
}
// Quotients by one denominator: its reciprocal once, then three instructions
// each, with one correction (the rounded quotient; an IEEE quotient each
// takes 13).  Denominators finite and not 0.
struct Divisor {
    double b, r;
    __device__ __forceinline__ explicit Divisor(double x) : b(x), r(m_rcp(x)) {}
    __device__ __forceinline__ double under(double a) const
    {
        const double q = a * r;
        return fma(r, fma(-b, q, a), q);
    }
};
// x^e from L = log |x| as exp(e L), the product's rounding error put back
// (exp would amplify it: |e L| is of order 10).  Where the power overflows or e
// is infinite it is not below infinity (NaN: infinity times a correction of 0),
// and pow_special takes it.
__device__ __forceinline__ double exp_product(double e, double L)
{
    const double p = e * L;
    const double r = exp(p);
    return fma(r, fma(e, L, -p), r);
}
// pow's value at x <= 0, infinite and NaN x, at e = 0 and (ANY) where it
// overflows, r = |x|^e elsewhere.
template <bool ANY = true>
__device__ __forceinline__ double pow_special(double x, double e, double r)
{
    if (e == 0.0) return 1.0;
    if (x != x || e != e) return x + e;
    const double inf = HUGE_VAL;
    if (ANY && !(r < inf)) r = fabs(x) == 1.0 ? 1.0 : ((e > 0.0) == (fabs(x) > 1.0) ? inf : 0.0);
    if (x == 0.0) r = e > 0.0 ? 0.0 : inf;
    if (fabs(x) == inf) r = e > 0.0 ? inf : 0.0;
    if (x < 0.0) {
        if (e != rint(e)) return x == -inf ? r : __longlong_as_double(0x7ff8000000000000ll);
        if (0.5 * e != rint(0.5 * e)) r = -r;
    }
    return r;
}
// Exponents with which the power of a finite base does not overflow.
__host__ __device__ __forceinline__ bool tame_exponents(double e1, double e2)
{
    return e1 >= 0.0 && e1 <= 1.0 && e2 >= 0.0 && e2 <= 1.0;
}
// x^e1 and x^e2 of one base in FP64, within a few ulp of pow: the logarithm
// shared, pow's special cases behind one branch.  ANY: the exponents (the same
// in every lane) need not be tame; with others every lane takes the branch.
// (Only kernels with the formulations read at run time have ANY: the branch's
// code alone cost the fused step of 512x512x64 697 -> 762 us.)
template <bool ANY>
__device__ __forceinline__ void pow_pair(double x, double e1, double e2, double& r1, double& r2)
{
    const bool plain = ANY ? tame_exponents(e1, e2) && e1 != 0.0 && e2 != 0.0 : e1 != 0.0 && e2 != 0.0;
    const double L = log_positive(fabs(x));
    r1 = exp_product(e1, L);
    r2 = exp_product(e2, L);
    if (!(x > 0.0 && x < HUGE_VAL && plain)) {
        r1 = pow_special<ANY>(x, e1, r1);
        r2 = pow_special<ANY>(x, e2, r2);
    }
}
// x^y: within a few ulp of pow (270 cycles of a wave where pow takes 600).
__device__ __forceinline__ double m_pow(double x, double y)
{
    double r = exp_product(y, log_positive(fabs(x)));
    if (!(x > 0.0 && x < HUGE_VAL && y != 0.0 && r < HUGE_VAL)) r = pow_special(x, y, r);
    return r;
}
// x^y for x >= 0 as 2^(y log2 x); a negative x gives NaN, as on the GPU
// reference path.
__device__ __forceinline__ float m_pow(float x, float y) { return m_exp2(y * m_log2(x)); }

// ---------------------------------------------------------------- buffer I/O

// Raw buffer access: a 128-bit descriptor in SGPRs per array plus a 32-bit
// byte offset per lane, shared by every array of the same layout.  Offsets
// at or beyond `bytes` read 0 and drop stores.
using rsrc_t = __amdgpu_buffer_rsrc_t;

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, unsigned bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ void buf_load(rsrc_t r, unsigned off, float& v)
{
    v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
}
__device__ __forceinline__ void buf_load(rsrc_t r, unsigned off, double& v)
{
    v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
__device__ __forceinline__ void buf_store(rsrc_t r, unsigned off, float v)
{
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, off, 0, 0);
}
__device__ __forceinline__ void buf_store(rsrc_t r, unsigned off, double v)
{
    using V2 = decltype(__builtin_amdgcn_raw_buffer_load_b64(r, 0, 0, 0));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(V2, v), r, off, 0, 0);
}

// Plain global access at a 32-bit byte offset from an array's base: the
// base stays in scalar registers and one per-lane offset serves every array
// of the same layout (global_load/store with a scalar base address).
template <typename FT>
__device__ __forceinline__ FT gload(const FT* p, unsigned boff)
{
    return *reinterpret_cast<const FT*>(reinterpret_cast<const char*>(p) + boff);
}
template <typename FT>
__device__ __forceinline__ void gstore(FT* p, unsigned boff, FT v)
{
    *reinterpret_cast<FT*>(reinterpret_cast<char*>(p) + boff) = v;
}

// ---------------------------------------------------------------- tendencies

// The NutrientsPlanktonDetritus transitions in the arithmetic type FT.  The
// products of parameters are formed once on the host in FP64 (the vector
// ALUs do all float arithmetic: there is no scalar float ALU), and the
// quotients are gathered: the Monod terms and the light limitation over one
// reciprocal (FP64 two: the ammonia term apart), the grazing over one.  The
// reference's expressions (plankton.jl, nutrients.jl, detritus.jl) hold 13
// quotients per cell; FP64 agrees with them to rounding.
template <typename FT>
struct FastParams {
    FT nPSI;           // FP32 -psi log2(e): exp(-psi NH4) = 2^(nPSI NH4); FP64 -psi
    FT kNO3, kNH4, kPAR, kPAR2;
    FT mu0h;           // mu0/2 (LOBSTER's (L_NO3 + L_NH4)/2)
    FT pref, prefc;    // pref, 1 - pref
    FT kGp, kGs, kG, kG2;   // kG pref, kG (1 - pref), kG, kG^2
    FT g;
    FT mP, mZ, muZ;
    FT growP;          // (1 - gamma) mu0/2
    FT axg;            // alpha_x gamma mu0/2
    FT nitrif;
    FT pinw_z;         // aZ_exc muZ
    FT pinw_p, solid_p;   // (1 - aP) , aP: the mortality's inorganic and solid shares
    FT s_rem, b_rem, d_rem, a_rem, one_m_arem;
    FT ponw_mu;        // (1 - alpha_x) gamma mu0/2
    FT ponw_z;         // (1 - aZ_exc) muZ
    FT solid_g, gainZ; // (1 - aZ_ass) g, aZ_ass g
    FT ss, one_m_ss;
    FT ppc;            // (1 + rho (1-gamma) - alpha_x gamma) R mu0/2
    FT R, Rd, rhoR, rhoRg, rhoR4;  // R, Rd, rho R, rho R g, 4 rho R mu0/2
    FT rem, small_frac;           // Detritus rate and fraction
    FT nGrowP, nUp, nPonw, nOx;   // NPZD: (1 - gamma) mu0, (1 - alpha_x gamma) mu0, (1 - alpha_x) gamma mu0, Rp mu0
    FT logQ10_10, logQ10_10l;   // Q10^(T/10): FP32 log2(Q10)/10; FP64 ln|Q10|/10 and its rounding error
                                // (use_Q10 = 2: a Q10 of 0 or less, and it in its place)
    FT oRp, oRpn, oRpm;           // Oxygen(): Rp, Rp - Rn, Rp mu0/2
    int light_form, use_Q10, mort_form, graz_form;
};

// (q10: with the temperature factor's constants; the ensemble has its factor per
// column, and 8192 columns' logarithms take 315 us)
template <typename FT>
inline FastParams<FT> make_fast_params(const obme_npd_params& p, double Rp = 0.0, double Rn = 0.0, bool q10 = true)
{
    FastParams<FT> f;
    const bool F32 = sizeof(FT) == 4;
    const double LOG2E = 1.4426950408889634;
    const double mu0 = p.phytoplankton_maximum_growth_rate, h = mu0 / 2;
    const double gam = p.phytoplankton_exudation_fraction, ax = p.ammonia_fraction_of_exudate;
    const double g = p.maximum_grazing_rate, kG = p.grazing_half_saturation, pr = p.preference_for_phytoplankton;
    const double R = p.redfield_ratio, rho = p.carbon_calcite_ratio;
    f.nPSI = (FT)(-p.nitrate_ammonia_inhibition * (F32 ? LOG2E : 1.0));
    f.kNO3 = (FT)p.nitrate_half_saturation;
    f.kNH4 = (FT)p.ammonia_half_saturation;
    f.kPAR = (FT)p.light_half_saturation;
    f.kPAR2 = (FT)(p.light_half_saturation * p.light_half_saturation);
    f.mu0h = (FT)h;
    f.pref = (FT)pr;
    f.prefc = (FT)(1 - pr);
    f.kGp = (FT)(kG * pr);
    f.kGs = (FT)(kG * (1 - pr));
    f.kG = (FT)kG;
    f.kG2 = (FT)(kG * kG);
    f.g = (FT)g;
    f.mP = (FT)p.phytoplankton_mortality_rate;
    f.mZ = (FT)p.zooplankton_mortality_rate;
    f.muZ = (FT)p.zooplankton_excretion_rate;
    f.growP = (FT)((1 - gam) * h);
    f.axg = (FT)(ax * gam * h);
    f.nitrif = (FT)p.nitrification_rate;
    f.pinw_z = (FT)(p.excretion_inorganic_fraction * p.zooplankton_excretion_rate);
    f.pinw_p = (FT)(1 - p.phytoplankton_solid_waste_fraction);
    f.solid_p = (FT)p.phytoplankton_solid_waste_fraction;
    f.s_rem = (FT)p.small_remineralisation_rate;
    f.b_rem = (FT)p.large_remineralisation_rate;
    f.d_rem = (FT)p.dissolved_remineralisation_rate;
    f.a_rem = (FT)p.remineralisation_inorganic_fraction;
    f.one_m_arem = (FT)(1 - p.remineralisation_inorganic_fraction);
    f.ponw_mu = (FT)((1 - ax) * gam * h);
    f.ponw_z = (FT)((1 - p.excretion_inorganic_fraction) * p.zooplankton_excretion_rate);
    f.solid_g = (FT)((1 - p.zooplankton_assimilation_fraction) * g);
    f.gainZ = (FT)(p.zooplankton_assimilation_fraction * g);
    f.ss = (FT)p.small_solid_waste_fraction;
    f.one_m_ss = (FT)(1 - p.small_solid_waste_fraction);
    f.ppc = (FT)((1 + rho * (1 - gam) - ax * gam) * R * h);
    f.R = (FT)R;
    f.Rd = (FT)p.detritus_redfield_ratio;
    f.rhoR = (FT)(rho * R);
    f.rhoRg = (FT)(rho * R * g);
    f.rhoR4 = (FT)(4 * rho * R * h);
    f.rem = (FT)p.remineralisation_rate;
    f.small_frac = (FT)p.small_particle_fraction;
    f.nGrowP = (FT)((1 - gam) * mu0);
    f.nUp = (FT)((1 - ax * gam) * mu0);
    f.nPonw = (FT)((1 - ax) * gam * mu0);
    f.nOx = (FT)(Rp * mu0);
    f.logQ10_10 = f.logQ10_10l = FT(0);
    if (q10 && F32) {
        // (a Q10 of 0 or less: FP32 none, FP64 pow's values)
        f.logQ10_10 = (FT)(std::log2(p.temperature_coefficient > 0 ? p.temperature_coefficient : 1.0) / 10);
    } else if (q10) {
        const long double lnQ = std::log((long double)std::fabs(p.temperature_coefficient)) / 10;
        f.logQ10_10 = (FT)lnQ;
        f.logQ10_10l = (FT)(lnQ - (long double)(double)lnQ);
    }
    const bool special = q10 && !F32 && p.use_temperature_coefficient && !(p.temperature_coefficient > 0);
    if (special) f.logQ10_10l = (FT)p.temperature_coefficient;
    f.oRp = (FT)Rp;
    f.oRpn = (FT)(Rp - Rn);
    f.oRpm = (FT)(Rp * h);
    f.light_form = p.light_limitation;
    f.use_Q10 = special ? 2 : p.use_temperature_coefficient;
    f.mort_form = p.phytoplankton_mortality_formulation;
    f.graz_form = p.grazing_concentration_formulation;
    return f;
}

// max(0, x), 0 for a NaN x.
__device__ __forceinline__ float max0(float x) { return fmaxf(x, 0.0f); }
__device__ __forceinline__ double max0(double x) { return fmax(x, 0.0); }
// the smallest normal number: keeps 0/0 away as the reference's eps(food) does
template <typename FT> struct Least;
template <> struct Least<float> { static constexpr float v = 1.17549435e-38f; };
template <> struct Least<double> { static constexpr double v = 2.2250738585072014e-308; };

// Formulation choices: FM < 0 reads them from FastParams at run time;
// otherwise they are compiled in, FM = light (bit 0: 0 Mondo, 1 analytical) |
// phytoplankton mortality << 1 (0 linear, 1 quadratic) | grazing
// concentration << 2 (0 linear, 1 quadratic) | Q10 in use << 3.
template <int FM, typename FT> __device__ __forceinline__ int fm_light(const FastParams<FT>& f) { if constexpr (FM < 0) return f.light_form; else return FM & 1; }
template <int FM, typename FT> __device__ __forceinline__ int fm_mort(const FastParams<FT>& f) { if constexpr (FM < 0) return f.mort_form; else return (FM >> 1) & 1; }
template <int FM, typename FT> __device__ __forceinline__ int fm_graz(const FastParams<FT>& f) { if constexpr (FM < 0) return f.graz_form; else return (FM >> 2) & 1; }
template <int FM, typename FT> __device__ __forceinline__ int fm_q10(const FastParams<FT>& f) { if constexpr (FM < 0) return f.use_Q10; else return (FM >> 3) & 1; }
inline int fm_code(const FastParams<float>& f)
{
    return (f.light_form & 1) | ((f.mort_form & 1) << 1) | ((f.graz_form & 1) << 2) | ((f.use_Q10 ? 1 : 0) << 3);
}

// Q10^(T/10) (plankton.jl:210-214); FP64 with the product's low part put back.
// (A Q10 of 0 or less: with the formulations read at run time, which such a
// handle takes.)
template <int FM, typename FT>
__device__ __forceinline__ FT q10_factor(const FastParams<FT>& f, FT T)
{
    if constexpr (sizeof(FT) == 4) {
        return m_exp2(T * f.logQ10_10);
    } else {
        const double p = T * f.logQ10_10;
        const double e = exp(p);
        if constexpr (FM < 0) {
            if (f.use_Q10 == 2) return pow_special(f.logQ10_10l, T / 10, fma(e, fma(T, f.logQ10_10, -p), e));
        }
        return fma(e, fma(T, f.logQ10_10, -p) + T * f.logQ10_10l, e);
    }
}

// Grazing of the PhytoZoo plankton (plankton.jl:118-135, :352-397) without
// the rate g: with n = pref P^2 + (1-pref) sPOM^2 and d = pref P + (1-pref)
// sPOM the preference-weighted food is n/d, so the total grazing is
// Z n^2 / (n^2 + kG^2 d^2) (quadratic) or Z n / (n + kG d) (linear), and the
// grazed shares of the total are pref P^2 / n and (1-pref) sPOM^2 / n.  FP64
// keeps the preference p = pref P / (d + ε) apart, as the reference has it: at
// P = 0 with pref = 1 (a rescaled cell) n and d vanish and p = 0 leaves the
// food to sPOM.
template <typename FT>
struct FGrazing {
    FT total, onP, onSmall;
};
template <int FM, typename FT>
__device__ __forceinline__ FGrazing<FT> fast_grazing(const FastParams<FT>& f, FT P2, FT P, FT Z, FT S)
{
    FGrazing<FT> G;
    if constexpr (sizeof(FT) == 8) {
        const FT pP = f.pref * P;
        const FT p = pP * m_rcp(fma(f.prefc, S, pP) + Least<FT>::v);
        const FT q = FT(1) - p;
        const FT food = fma(p, P, q * S);
        FT fr;
        if (fm_graz<FM>(f) == OBME_LINEAR) fr = Z * m_rcp(food + f.kG);
        else fr = (Z * food) * m_rcp(fma(food, food, f.kG2));
        G.total = fr * food;
        G.onP = fr * (p * P);
        G.onSmall = fr * (q * S);
        return G;
    }
    const FT onp = f.pref * P2, ons = f.prefc * (S * S);
    const FT n = onp + ons;
    const FT kd = fma(f.kGp, P, f.kGs * S);
    FT fr;
    if (fm_graz<FM>(f) == OBME_LINEAR) fr = Z * m_rcp(n + kd + Least<FT>::v);
    else fr = (Z * n) * m_rcp(fma(kd, kd, fma(n, n, Least<FT>::v)));
    G.total = fr * n;
    G.onP = fr * onp;
    G.onSmall = fr * ons;
    return G;
}

// LOBSTER (+ CarbonateSystem, Oxygen) transitions; v/out in tracer order
// NO3, NH4, P, Z, sPOM, bPOM, DOM[, DIC, Alk][, O2].  CARB: bit 1
// CarbonateSystem, bit 2 Oxygen.  The nitrate and ammonia uptakes are mu0/2
// L_PAR P times their own limitation (the reference forms them as fractions
// of the total production, plankton.jl:223-261, which is the same product);
// uN, uA and mu leave mu0/2 to the constants.
template <int CARB, int FM = -1, typename FT>
__device__ __forceinline__ void lobster_fast(const FastParams<FT>& f, const FT* v, FT PAR, FT* out)
{
    const FT NO3 = v[0], NH4 = v[1], P = v[2], Z = v[3], S = v[4], B = v[5], DOM = v[6];
    const FT a = NO3 + f.kNO3, b = NH4 + f.kNH4;
    FT inhibition;
    if constexpr (sizeof(FT) == 4) inhibition = m_exp2(f.nPSI * NH4);
    else inhibition = m_exp(f.nPSI * NH4);
    const FT nl = NO3 * inhibition;
    FT uN, uA;
    if constexpr (sizeof(FT) == 8) {
        const FT light = fm_light<FM>(f) == OBME_LIGHT_MONDO ? f.kPAR + PAR : FT(1);
        FT pp = fm_light<FM>(f) == OBME_LIGHT_MONDO ? PAR * P : PAR * P * m_rsqrt(fma(PAR, PAR, f.kPAR2));
        // an infinite NH4 has no limitation (infinity over infinity): NaN to
        // both uptakes.  (A NaN of max0's is then a denominator of 0 under a
        // negative NH4, whose quotient is -infinity.)
        pp = fma(FT(0), NH4, pp);
        const FT r = m_rcp(a * light);
        uN = pp * nl * r;
        uA = max0(NH4 * m_rcp(b)) * (pp * (a * r));
    } else if (fm_light<FM>(f) == OBME_LIGHT_MONDO) {
        // with c = kPAR + PAR > 0, 1/(a c) = b r and 1/(b c) = a r for
        // r = 1/(a b c), and max(0, x / c) = max(0, x) / c
        const FT r = m_rcp((a * b) * (f.kPAR + PAR));
        const FT pp = PAR * P;
        uN = nl * (b * (pp * r));
        uA = max0(NH4 * (a * r)) * pp;
    } else {
        const FT r = m_rcp(a * b);
        const FT pp = PAR * P * m_rsqrt(fma(PAR, PAR, f.kPAR2));
        uN = nl * (b * (pp * r));
        uA = max0(NH4 * (a * r)) * pp;
    }
    const FT mu = uN + uA;
    const FT P2 = P * P, Z2 = Z * Z;
    const FGrazing<FT> G = fast_grazing<FM>(f, P2, P, Z, S);
    const FT nuP = f.mP * (fm_mort<FM>(f) == OBME_LINEAR ? P : P2);
    const FT nit = f.nitrif * NH4;
    const FT sr = f.s_rem * S, br = f.b_rem * B, dd = f.d_rem * DOM;
    const FT sb = sr + br;
    const FT pinw = fma(f.pinw_z, Z, f.pinw_p * nuP);
    const FT dinw = fma(f.a_rem, sb, dd);
    const FT solid = fma(f.solid_g, G.total, fma(f.solid_p, nuP, f.mZ * Z2));
    const FT dNO3 = fma(-f.mu0h, uN, nit);
    const FT dNH4 = fma(f.axg, mu, fma(-f.mu0h, uA, (pinw + dinw) - nit));
    out[0] = dNO3;
    out[1] = dNH4;
    out[2] = fma(f.growP, mu, fma(-f.g, G.onP, -nuP));
    out[3] = fma(f.gainZ, G.total, fma(-f.mZ, Z2, -(f.muZ * Z)));
    out[4] = fma(f.ss, solid, fma(-f.g, G.onSmall, -sr));
    out[5] = fma(f.one_m_ss, solid, -br);
    out[6] = fma(f.ponw_mu, mu, fma(f.ponw_z, Z, fma(f.one_m_arem, sb, -dd)));
    if constexpr ((CARB & 1) != 0) {
        // calcite dissolution (G_P + ν) ρ R (plankton.jl:429-441), uptake 2 ρ μP R (:443-450)
        const FT cdis = fma(f.rhoRg, G.onP, f.rhoR * nuP);
        out[7] = fma(-f.ppc, mu, fma(f.R, pinw, fma(f.Rd, dinw, cdis)));
        out[8] = fma(FT(0.9375), dNH4, fma(FT(-1.0625), dNO3, fma(-f.rhoR4, mu, cdis + cdis)));
    }
    if constexpr ((CARB & 2) != 0) {
        // Rp (μP - nitrification) - (Rp - Rn) G_NH₄ (oxygen.jl:21-31: the NH₄
        // tendency stands for "nitrate_production")
        out[(CARB & 1) ? 9 : 7] = fma(f.oRpm, mu, fma(-f.oRp, nit, -(f.oRpn * dNH4)));
    }
}

// NPZD transitions (N, P, Z, D); Lt = Q10^(T/10).  With dO2 the O2 transition
// of the Oxygen component's Nutrient method (oxygen.jl:35-46): Rp μP -
// (Rp - Rn) respiration, where respiration is the plankton's inorganic
// nitrogen waste alone (the line that adds the detritus waste, oxygen.jl:42,
// begins with a unary + and is a separate, discarded expression in Julia).
template <int FM = -1, typename FT>
__device__ __forceinline__ void npzd_fast(const FastParams<FT>& f, FT N, FT P, FT Z, FT D, FT PAR, FT Lt, FT& dN,
                                          FT& dP, FT& dZ, FT& dD, FT* dO2 = nullptr)
{
    const FT S = D * f.small_frac;
    FT mu;   // without mu0
    if (fm_light<FM>(f) == OBME_LIGHT_MONDO) mu = (N * Lt) * (PAR * P) * m_rcp((N + f.kNO3) * (f.kPAR + PAR));
    else mu = (N * Lt) * (PAR * P) * (m_rcp(N + f.kNO3) * m_rsqrt(fma(PAR, PAR, f.kPAR2)));
    const FT P2 = P * P, Z2 = Z * Z;
    const FGrazing<FT> G = fast_grazing<FM>(f, P2, P, Z, S);
    const FT nuP = f.mP * (fm_mort<FM>(f) == OBME_LINEAR ? P : P2);
    const FT zz = f.mZ * Z2, rD = f.rem * D;
    const FT pinw = fma(f.pinw_z, Z, f.pinw_p * nuP);
    dP = fma(f.nGrowP, mu, fma(-f.g, G.onP, -nuP));
    dZ = fma(f.gainZ, G.total, -zz) - f.muZ * Z;
    dN = fma(-f.nUp, mu, rD + pinw);
    const FT solid = fma(f.solid_g, G.total, fma(f.solid_p, nuP, zz));
    dD = fma(f.nPonw, mu, fma(f.ponw_z, Z, solid)) - fma(f.g, G.onSmall, rD);
    if (dO2) *dO2 = fma(f.nOx, mu, -f.oRpn * pinw);
}

}  // namespace obme

#include "obme_sediment_order.h"

namespace obme {

// ScaleNegativeTracers groups for the kernels: members as bits of the
// tracer index and a scalefactor per tracer index (obme_negative_scaling
// converted on the host).
template <typename FT, int NTMAX>
struct NegScale {
    int n_groups;
    unsigned mask[OBME_MAX_SCALE_GROUPS];
    FT sf[OBME_MAX_SCALE_GROUPS][NTMAX];
    FT fill[OBME_MAX_SCALE_GROUPS];
};

// The scaling of one cell's NT tracer values x[] (src/Utils/negative_tracers.jl:
// 198-251): per group t = Σ s·c, p = Σ s·c over c > 0 (summed in tracer
// order: a reassociation of the reference's member order), t := fill where
// t < 0, then c := c·t/p where c > 0 or c is not finite, else 0.
template <int NT, typename FT, int NTMAX>
__device__ __forceinline__ void scale_negatives_cell(const NegScale<FT, NTMAX>& s, FT* x)
{
#pragma unroll 1
    for (int g = 0; g < s.n_groups; g++) {
        const unsigned mask = s.mask[g];
        FT t = FT(0), p = FT(0);
#pragma unroll
        for (int n = 0; n < NT; n++) {
            if (mask & (1u << n)) {
                const FT vs = x[n] * s.sf[g][n];
                t = t + vs;
                if (x[n] > FT(0)) p = p + vs;
            }
        }
        t = (t < FT(0)) ? s.fill[g] : t;
#pragma unroll
        for (int n = 0; n < NT; n++) {
            if (mask & (1u << n)) {
                const FT v = x[n];
                x[n] = (!isfinite(v) || v > FT(0)) ? v * t / p : FT(0);
            }
        }
    }
}

// ---------------------------------------------------------------- carbonate chemistry (FP64)

// teos10_polynomial_approximation (Models/seawater_density.jl:33-39) over
// SeawaterPolynomials' TEOS10 _ρ (Roquet et al. 2015 polynomial).
__device__ __forceinline__ double teos10_density(double T, double S, double Pbar)
{
    const double Sau = 40.0 * 35.16504 / 35.0;
    double t = T / 40.0;
    double s = sqrt((S + 32.0) / Sau);
    double z = -(10.0 * Pbar) / 1e4;
    double r0 = (((((-1.7243708991e-03 * z + 1.5616995503e-02) * z + 6.4326772569e-02) * z
                   + 2.2601900708e-01) * z - 5.2099962525e+00) * z + 4.6494977072e+01) * z;
    double n3 = 3.7969820455e-01 * t + -1.8507636718e-02 * s + -2.3342758797e-02;
    double n2 = (-1.2419983026e+00 * t + -2.1311365518e-01 * s + 2.0564311499e+00) * t
                + (2.5019633244e+00 * s + -4.9527603989e+00) * s + 2.0660924175e+00;
    double n1 = (((5.5927935970e-01 * t + -5.5077101279e-01 * s + -2.4649669534e+00) * t
                  + (-1.8795372996e+00 * s + 3.5063081279e+00) * s + 6.7080479603e+00) * t
                 + ((-6.5399043664e-01 * s + 5.0042598061e+00) * s + -4.4870114575e+00) * s + -1.3336301113e+01) * t
                + (((6.6051753097e+00 * s + -3.0938076334e+01) * s + 5.0774768218e+01) * s + -4.2549998214e+01) * s
                + 1.9681925209e+01;
    double n0 = (((((-1.9083568888e-01 * t + 4.8169980163e-01 * s + 5.4048723791e-01) * t
                    + (-5.3563304045e+00 * s + 1.1311538584e+01) * s + -8.3627885467e+00) * t
                   + ((-3.1742946532e+00 * s + 1.9717078466e+01) * s + -3.3449108469e+01) * s + 2.1661789529e+01) * t
                  + (((-5.4723692739e+00 * s + 2.9130021253e+01) * s + -6.0362551501e+01) * s + 6.1548258127e+01) * s
                  + -3.7074170417e+01) * t
                 + ((((-1.9193502195e+00 * s + 1.7681814114e+01) * s + -5.6888046321e+01) * s + 8.1770425108e+01) * s
                    + -6.5281885265e+01) * s + 2.6010145068e+01) * t
                + (((((-6.0579916612e+01 * s + 4.3227585684e+02) * s + -1.2849161071e+03) * s + 2.0375295546e+03) * s
                    + -1.7864682637e+03) * s + 8.6672408165e+02) * s + 8.0189615746e+02;
    return r0 + (((n3 * z + n2) * z + n1) * z + n0);
}

struct CarbonParams {
    double DIC, Alk, boron, sulfate, fluoride, silicate;
    double K1, K2, KB, KW, KS, KF, KSi, K0, Tk;
};

// Equilibrium constants at the surface (P = nothing): CarbonChemistry/
// equilibrium_constants.jl K0 :65-80, K1 :103-126, K2 :149-172, KB :202-250,
// KW :279-313, IonicStrength :335-341, KS :366-419, KF :451-488,
// KSi :674-713 (KP1-3 enter with phosphate, which is 0 here).  lT = log T, √S
// and √Is are computed once; the quotients by T share its reciprocal.
__device__ __forceinline__ double k0_constant(const Divisor& rT, double S, double lT)
{
    const double T = rT.b;
    return exp(-60.2409 + rT.under(93.4517 * 100) + 23.3585 * (lT - 4.605170185988092)
               + (0.023517 + (-0.023656 / 100) * T + (0.0047036 / 10000.0) * (T * T)) * S);
}

__device__ __forceinline__ void carbon_constants(const Divisor& rT, double lT, double S, CarbonParams& p)
{
    const double Tk = rT.b;
    auto over = [&](double a) { return rT.under(a); };
    double sS = sqrt(S);
    double Is = 19.924 * S / (1000.0 + -1.005 * S);
    double sIs = sqrt(Is);
    p.K0 = k0_constant(rT, S, lT);
    p.K1 = m_exp10(61.2172 + over(-3633.86) + -9.67770 * lT + 0.011555 * S + -0.0001152 * (S * S));
    p.K2 = m_exp10(-25.9290 + over(-471.78) + 0.01781 * S + -0.0001122 * (S * S) + 3.16967 * lT);
    p.KB = exp(148.0248 + over(-8966.90 + -2890.53 * sS + -77.942 * S + 1.728 * (S * sS) + -0.0996 * (S * S))
               + 137.1942 * sS + 1.62142 * S + (-24.4344 + -25.085 * sS + -0.2474 * S) * lT + 0.053105 * sS * Tk);
    p.KW = exp(148.9652 + over(-13847.26) + -23.6521 * lT + (-5.977 + over(118.67) + 1.0495 * lT) * sS + -0.01615 * S);
    double l1S = m_log_any(1 + -0.001005 * S);
    p.KS = exp(141.328 + over(-4276.1) + -23.093 * lT + (324.57 + over(-13856.0) + -47.986 * lT) * sIs
               + (-771.54 + over(35474.0) + 114.723 * lT) * Is + over(-2698.0 * (Is * sIs))
               + over(1776.0 * (Is * Is)) + l1S);
    // (the logarithms of 1 + 0 S and 1 + 0 S / KS of the form are 0)
    p.KF = exp(-9.68 + over(874.0) + 0.111 * sS);
    p.KSi = exp(117.385 + over(-8904.2) + -19.334 * lT + (3.5913 + over(-458.79)) * sIs + (-1.5998 + over(188.74)) * Is
                + (0.07871 + over(-12.1652)) * (Is * Is) + l1S);
}

// alkalinity_residual / ∂ₕ (CarbonChemistry/alkalinity_residual.jl:18-75)
// with phosphate = 0 and, unless SI, silicate = 0 (the defaults).  Those
// terms are then ±0 and adding them to the nonzero partial sums is exact, so
// they are left out; with SI the silicate term enters at its place in the sum.
template <bool SI = false>
__device__ __forceinline__ double alk_residual(double H, const CarbonParams& p)
{
    double cd = H * H + p.K1 * H + p.K1 * p.K2;
    double sd = 1 + p.sulfate / p.KS;
    double bicarbonate = p.K1 * H * p.DIC / cd;
    double carbonate = 2 * p.DIC * p.K1 * p.K2 / cd;
    double borate = p.boron / (1 + H / p.KB);
    double hydroxide = p.KW / H;
    double free_hydrogen = -H / sd;
    double hydrogen_sulfate = -p.sulfate / (1 + p.KS / H * sd);
    double hydrogen_fluoride = -p.fluoride / (1 + p.KF / H);
    double acc = bicarbonate + carbonate + borate + hydroxide;
    if constexpr (SI) acc = acc + p.silicate / (1 + H / p.KSi);
    return acc + free_hydrogen + hydrogen_sulfate + hydrogen_fluoride - p.Alk;
}

template <bool SI = false>
__device__ __forceinline__ double alk_residual_derivative(double H, const CarbonParams& p)
{
    double cd = H * H + p.K1 * H + p.K1 * p.K2;
    double sd = 1 + p.sulfate / p.KS;
    double dcd = 2 * H + p.K1;
    double d_bicarbonate = p.K1 * p.DIC * (p.K1 * p.K2 - H * H) / (cd * cd);
    double d_carbonate = -dcd * 2 * p.DIC * p.K1 * p.K2 / (cd * cd);
    double bd = 1 + H / p.KB;
    double d_borate = -p.boron / (bd * bd) / p.KB;
    double d_hydroxide = -p.KW / (H * H);
    double d_free_hydrogen = -1 / sd;
    double hsd = 1 + p.KS / H * sd;
    double d_hydrogen_sulfate = p.sulfate / (hsd * hsd) * (p.KS / H * 0.0 - p.KS / (H * H) * sd);
    double fd = 1 + p.KF / H;
    double d_hydrogen_fluoride = -p.fluoride / (fd * fd) * p.KF / (H * H);
    double acc = d_bicarbonate + d_carbonate + d_borate + d_hydroxide;
    if constexpr (SI) {
        const double sdn = 1 + H / p.KSi;
        acc = acc + -p.silicate / (sdn * sdn) / p.KSi;
    }
    return acc + d_free_hydrogen + d_hydrogen_sulfate + d_hydrogen_fluoride;
}

__device__ __forceinline__ double jsign(double x)
{
    return (x > 0) ? 1.0 : ((x < 0) ? -1.0 : x);
}

// DampedNewtonRaphsonSolver (Utils/solvers.jl:90-121) with bounded_λ for
// the lower bound 0 (:126-131).  An iteration that leaves x unchanged is an
// exact fixed point of the loop (same x, same f(x), same δ, same λ
// sequence), so the remaining iterations are skipped with the identical
// result.  evals counts residual evaluations.
template <bool SI = false>
__device__ __forceinline__ double solve_for_H(const CarbonParams& p, const obme_carbon_solver& s, double x0,
                                              int& evals)
{
    double x = x0;
    int N = 0;
    double fx = alk_residual<SI>(x, p);
    int ne = 1;
    while ((fabs(fx) > s.atol) && (N < s.max_iters)) {
        double delta = fx / alk_residual_derivative<SI>(x, p);
        double lb = (x - 0.0) / delta;
        lb = (lb < 0) ? 1.0 : lb;
        double lambda = jmin(1.0, lb);
        double trial = x - lambda * delta;
        double fnew = alk_residual<SI>(trial, p);
        ne++;
        while ((fabs(fnew) >= fabs(fx) - s.armijo_constant * lambda * fx * jsign(fx)) && (lambda > s.min_damping)) {
            lambda *= s.damping;
            // (at the root the halved steps round to the same trial point)
            const double t = x - lambda * delta;
            if (t != trial) {
                trial = t;
                fnew = alk_residual<SI>(trial, p);
                ne++;
            }
        }
        double xn = x - lambda * delta;
        N += 1;
        bool stuck = (xn == x);
        x = xn;
        fx = fnew;
        if (stuck) N = s.max_iters;
    }
    evals += ne;
    return x;
}

// The residual and its derivative together for the refinement: the same
// function as alk_residual / alk_residual_derivative, each fraction rewritten
// over one reciprocal of its denominator (bicarbonate + carbonate =
// DIC K1 (H + 2 K2) / cd, borate = boron KB / (KB + H), ...).  What does not
// depend on H is formed once per solve.
template <bool SI, typename FT = double>
struct AlkResidual {
    FT K1, K2, K12, KB, KW, KSsd, KF, KSi, DK1, bKB, sulfate, fluoride, sK, rsd, Alk;
    __device__ __forceinline__ explicit AlkResidual(const CarbonParams& p)
        : K1((FT)p.K1), K2((FT)(p.K2 + p.K2)), K12((FT)(p.K1 * p.K2)), KB((FT)p.KB), KW((FT)p.KW), KF((FT)p.KF),
          KSi((FT)(SI ? p.KSi : 0.0)), DK1((FT)(p.DIC * p.K1)), bKB((FT)(p.boron * p.KB)), sulfate((FT)p.sulfate),
          fluoride((FT)p.fluoride), sK((FT)(SI ? p.silicate * p.KSi : 0.0)), Alk((FT)p.Alk)
    {
        KSsd = (FT)(p.KS + p.sulfate);    // KS (1 + sulfate / KS)
        rsd = (FT)p.KS * m_rcp(KSsd);
    }
    __device__ __forceinline__ void operator()(FT H, FT& f, FT& df) const
    {
        const FT cd = fma(H, H + K1, K12);
        const FT rcd = m_rcp(cd), rH = m_rcp(H), rB = m_rcp(KB + H), rS = m_rcp(H + KSsd), rF = m_rcp(H + KF);
        const FT n = DK1 * rcd;
        const FT h2 = H + K2;
        const FT carb = n * h2;
        const FT dcarb = n * fma(-h2 * rcd, H + H + K1, FT(1));
        const FT bor = bKB * rB;
        const FT hyd = KW * rH;
        const FT qs = sulfate * rS, qf = fluoride * rF;
        FT acc = carb + bor + hyd;
        FT dacc = dcarb - bor * rB - hyd * rH;
        if constexpr (SI) {
            const FT rSi = m_rcp(KSi + H);
            const FT sil = sK * rSi;
            acc = acc + sil;
            dacc = fma(-sil, rSi, dacc);
        }
        f = acc - H * (rsd + qs + qf) - Alk;
        df = dacc - rsd - qs * (KSsd * rS) - qf * (KF * rF);
    }
};

// FP32 first guess for [H+]: Newton on the residual in FP32 from pH 8, each
// step limited to half the distance to the bound H = 0, to a step of 1e-3 (the
// next would be of order 1e-6).  first_step: the first step before the limit,
// in units of its H (positive towards 0).
template <bool SI = false>
__device__ __forceinline__ float guess_H_fp32(const CarbonParams& p, float& first_step)
{
    const AlkResidual<SI, float> residual(p);
    float x = 1e-8f;
    first_step = 0.0f;
#pragma unroll 1
    for (int it = 0; it < 20; it++) {
        float f, df;
        residual(x, f, df);
        const float d = f * m_rcp(df);
        if (it == 0) first_step = d * 1e8f;
        x = x - fminf(d, 0.5f * x);
        if (fabsf(d) <= 1e-3f * x) break;
    }
    return x;
}
template <bool SI = false>
__device__ __forceinline__ float guess_H_fp32(const CarbonParams& p)
{
    float first_step;
    return guess_H_fp32<SI>(p, first_step);
}

// Refinement of a close first guess by plain FP64 Newton on the same
// residual; returns false when it has not converged after 6 steps.  It
// stops after the step that is at most tol relative to the iterate: Newton
// converges quadratically here, so the error left after a step of relative
// size tol is of order tol^2.
// The stop of the FP32-mixed paths, whose [H+] feeds FP32 arithmetic: after
// a step below 1e-4 relative, H is within ~1e-8 of the root (measured on
// the CPU oracle from warm starts off by up to 1e-2: at most 9e-9).
constexpr double FP32_NEWTON_TOL = 1e-4;
// The stop of the FP64 refinements: after a step below 3e-9 relative the next
// would be of order 1e-17, below the rounding of H.
constexpr double FP64_NEWTON_TOL = 3e-9;
template <bool SI = false>
__device__ __forceinline__ bool refine_H(const CarbonParams& p, double& x, int& evals, double tol = FP64_NEWTON_TOL)
{
    const AlkResidual<SI> residual(p);
#pragma unroll 1
    for (int it = 0; it < 6; it++) {
        double f, df;
        residual(x, f, df);
        evals++;
        double d = f * m_rcp(df);
        double xn = x - d;
        if (!(xn > 0.0)) return false;
        x = xn;
        if (fabs(d) <= tol * x) return true;
    }
    return false;
}

// pCO2 from H (carbon_chemistry.jl:160-162 and selected_output(::Val{:pCO₂}) :170-193).
__device__ __forceinline__ double pco2_from_H(const CarbonParams& p, double H)
{
    double CO2 = p.DIC * (H * H) * m_rcp(H * H + p.K1 * H + p.K1 * p.K2);
    double fCO2 = (CO2 * m_rcp(p.K0)) * 1e6;
    double P = 101325.0;
    double Tk = p.Tk;
    double B = (-1636.75 + 12.0408 * Tk + (-3.27957 * 1e-2) * (Tk * Tk) + (3.16528 * 1e-5) * (Tk * Tk * Tk)) * 1e-6;
    double dl = (57.7 + -0.118 * Tk) * 1e-6;
    fCO2 *= 0.09807;
    // x = fCO2 / (φ P), φ = exp(...) from the x before: 1/φ is exp of minus it
    const double c = P * m_rcp(8.31446261815324 * Tk);
    const double fP = fCO2 / P;
    double x = fP, rphi = 1.0;
#pragma unroll
    for (int n = 0; n < 3; n++) {
        const double om = 1.0 - x;
        rphi = exp(-(B + 2.0 * (om * om) * dl) * c);
        x = fP * rphi;
    }
    return fCO2 * rphi / 0.09807;
}

// Julia's literal x^4 (compensated power by squaring).
__device__ __forceinline__ double pow4_compensated(double x)
{
    double hi2 = x * x;
    double lo2 = fma(x, x, -hi2);
    double err = hi2 * 2.0 * lo2;
    double hi4 = hi2 * hi2;
    double lo4 = fma(hi2, hi2, -hi4);
    double lo = lo4 + err;
    return (isfinite(hi4) && isfinite(lo)) ? fma(hi4, 1.0, lo) : hi4;
}

// Gas transfer velocity (gas_transfer_velocity.jl:33-34, :61; schmidt
// number gas_solubility.jl:211-212; solubility gas_solubility.jl:204).
// K0: the solubility at T and S.
__device__ __forceinline__ double transfer_velocity(const obme_co2_exchange& g, double u10, double T, double S,
                                                   double K0)
{
    double k660 = g.transfer_velocity[0] + g.transfer_velocity[1] * u10 + g.transfer_velocity[2] * (u10 * u10);
    double sc = g.schmidt[0] + g.schmidt[1] * T + g.schmidt[2] * (T * T) + g.schmidt[3] * (T * T * T)
                + g.schmidt[4] * pow4_compensated(T);
    double sol = K0 * teos10_density(T, S, 0.0) / 1000.0;
    return k660 / sqrt(sc / 660.0) * sol;
}

// Everything of the CO2 flux that depends on T and S only: the carbonate
// parameters without DIC/Alk, the mmol/m³ → mol/kg factor 1e-3/ρ and the
// transfer velocity k (a function of u10, T, S).
struct SurfaceCarbon {
    CarbonParams p;   // DIC and Alk unset
    double conv;      // 1e-3 / ρ(T, S, Pbar = 1)
    double k;         // transfer velocity
};

__device__ __forceinline__ void surface_carbon_setup(const obme_co2_exchange& g, double T, double S, double u10,
                                                     SurfaceCarbon& sc)
{
    CarbonParams& p = sc.p;
    p.boron = 0.000232 / 10.811 * S / 1.80655;
    p.sulfate = 0.14 / 96.06 * S / 1.80655;
    p.fluoride = 0.000067 / 18.9984 * S / 1.80655;
    double rho = teos10_density(T, S, 1.0);
    p.Tk = T + 273.15;
    sc.conv = 1e-3 / rho;
    p.silicate = 0.0;
    carbon_constants(Divisor(p.Tk), m_log_any(p.Tk), S, p);
    sc.k = transfer_velocity(g, u10, T, S, p.K0);
}

// Whether the damped Newton's settings are the reference's (solvers.jl:81-88):
// it then ends at the root to rounding, and so does a refined guess.
__device__ __forceinline__ bool reference_solver(const obme_carbon_solver& s)
{
    return s.max_iters == 100 && s.atol == 1e-20 && s.damping == 0.5 && s.armijo_constant == 0.5 &&
           s.min_damping == 0.0009765625 && s.initial_pH_guess == 8.0;
}
// The damped Newton's root from its initial guess.  With the reference's
// settings and DIC and silicate >= 0 (the residual then falls with H: one
// root), an FP32 Newton from the same pH 8 refined in FP64 ends at the same
// root in two FP64 iterations instead of 10 to 14, each a residual, a
// derivative and a line search (4 10^6 points of the ocean's range, with the
// constants: 1263 -> 151 us; 362 us with the guess in IEEE quotients to
// 2e-7).  The damped Newton runs where the refinement
// fails, and where the first step goes past 0 by more than 8 H: past
// 1 / min_damping its line search cannot shorten a step onto 0, which ends in
// NaN (hardly any salt or carbon under an ocean's alkalinity).
template <bool SI = false>
__device__ __forceinline__ double root_H(const CarbonParams& p, const obme_carbon_solver& s, int& evals)
{
    if (p.DIC >= 0.0 && reference_solver(s) && (!SI || p.silicate >= 0.0)) {
        float step;
        double H = (double)guess_H_fp32<SI>(p, step);
        if (step < 8.0f && refine_H<SI>(p, H, evals)) return H;
    }
    return solve_for_H<SI>(p, s, pow(10.0, -s.initial_pH_guess), evals);
}

// Solve for H and return the flux F = k (pCO2_w - pCO2_air)
// (GasExchange/gas_exchange.jl:26-38).  mode 0: the reference damped Newton's
// root; mode 1: FP32 first guess refined by FP64 Newton, whatever the
// solver's settings, with the mode-0 solve where that has not converged.
__device__ __forceinline__ double surface_flux(const SurfaceCarbon& sc, const obme_carbon_solver& s, double DIC,
                                               double Alk, double pCO2_air, int mode, double& H, int& evals)
{
    CarbonParams p = sc.p;
    p.Alk = Alk * sc.conv;
    p.DIC = DIC * sc.conv;
    if (mode == 1) {
        H = (double)guess_H_fp32(p);
        if (!refine_H(p, H, evals)) H = solve_for_H(p, s, pow(10.0, -s.initial_pH_guess), evals);
    } else {
        H = root_H(p, s, evals);
    }
    return sc.k * (pco2_from_H(p, H) - pCO2_air);
}

__device__ __forceinline__ double co2_flux(const obme_co2_exchange& g, const obme_carbon_solver& s, double DIC,
                                           double Alk, double T, double S, double u10, double pCO2_air, int mode,
                                           double& pH, int& evals)
{
    SurfaceCarbon sc;
    surface_carbon_setup(g, T, S, u10, sc);
    double H;
    const double F = surface_flux(sc, s, DIC, Alk, pCO2_air, mode, H, evals);
    pH = -m_log10(H);
    return F;
}

// Flux with a warm start: H from the previous stage (or an FP32 guess) refined
// by FP64 Newton (stopping after a step below tol relative, see refine_H),
// with the reference solve as fallback.
__device__ __forceinline__ double surface_flux_warm(const SurfaceCarbon& sc, const obme_carbon_solver& s,
                                                    double DIC, double Alk, double pCO2_air, double& H, int& evals,
                                                    double tol = FP64_NEWTON_TOL)
{
    CarbonParams p = sc.p;
    p.Alk = Alk * sc.conv;
    p.DIC = DIC * sc.conv;
    double x = (H > 0.0) ? H : (double)guess_H_fp32(p);
    bool done = refine_H(p, x, evals, tol);
    if (!done) {
        x = (double)guess_H_fp32(p);
        done = refine_H(p, x, evals, tol);
        if (!done) x = solve_for_H(p, s, pow(10.0, -s.initial_pH_guess), evals);
    }
    H = x;
    return sc.k * (pco2_from_H(p, x) - pCO2_air);
}

// OxygenGasExchangeBoundaryCondition (GasExchange/GasExchange.jl:127-146):
// F = k (O2 - C_air α), k = k660(u10) / sqrt(Sc(T) / 660) · 1
// (gas_transfer_velocity.jl:33-34), Sc the quartic of schmidt_number.jl:15-16
// (generic_parameterisations.jl:31-32), α = β / Tk with
// β = exp(A1 + A2/(Tk/100) + A3 log(Tk/100) + S (B1 + B2 Tk/100 + B2 (Tk/100)²))
// (gas_solubility.jl:37-48: B2 in both salinity terms, as there).
// The T- and S-dependent part: the transfer velocity k and the air-side
// concentration C_air α.
__device__ __forceinline__ void o2_exchange_coefficients(const obme_o2_exchange& g, double T, double S, double& k,
                                                         double& air)
{
    const double* c = g.schmidt;
    const double Sc = c[0] + c[1] * T + c[2] * (T * T) + c[3] * (T * T * T) + c[4] * pow4_compensated(T);
    const double* v = g.transfer_velocity;
    const double u = g.wind_speed;
    const double k660 = v[0] + v[1] * u + v[2] * (u * u);
    k = k660 / sqrt(Sc / 660.0) * 1.0;
    const double Tk = T + 273.15;
    const double Tk100 = Tk / 100.0;
    const double* a = g.solubility;
    const double beta = exp(a[0] + a[1] / Tk100 + a[2] * log(Tk100) + S * (a[3] + a[4] * Tk100 + a[4] * (Tk100 * Tk100)));
    air = g.air_concentration * (beta / Tk);
}

__device__ __forceinline__ double o2_flux(const obme_o2_exchange& g, double O2, double T, double S)
{
    double k, air;
    o2_exchange_coefficients(g, T, S, k, air);
    return k * (O2 - air);
}

// SurfaceCarbon (without DIC and Alk) and the O2 coefficients of a column
// as 17 doubles, for a stepper with T and S fixed.
constexpr int SURF_PACK = 17;
__device__ __forceinline__ void surface_pack(const SurfaceCarbon& sc, double kO2, double airO2, double* o)
{
    const CarbonParams& p = sc.p;
    const double f[SURF_PACK] = {p.boron, p.sulfate, p.fluoride, p.silicate, p.K1, p.K2, p.KB, p.KW, p.KS,
                                 p.KF, p.KSi, p.K0, p.Tk, sc.conv, sc.k, kO2, airO2};
#pragma unroll
    for (int q = 0; q < SURF_PACK; q++) o[q] = f[q];
}
__device__ __forceinline__ void surface_unpack(const double* o, SurfaceCarbon& sc, double& kO2, double& airO2)
{
    CarbonParams& p = sc.p;
    p.DIC = 0.0;
    p.Alk = 0.0;
    p.boron = o[0];
    p.sulfate = o[1];
    p.fluoride = o[2];
    p.silicate = o[3];
    p.K1 = o[4];
    p.K2 = o[5];
    p.KB = o[6];
    p.KW = o[7];
    p.KS = o[8];
    p.KF = o[9];
    p.KSi = o[10];
    p.K0 = o[11];
    p.Tk = o[12];
    sc.conv = o[13];
    sc.k = o[14];
    kO2 = o[15];
    airO2 = o[16];
}

// ---- wave-level helpers (the column sweeps)

// Cross-lane data movement with DPP (GFX9 family): row_shr:d shifts within
// rows of 16 lanes, row_bcast:15/31 carries row ends into later rows,
// wave_shr:1 shifts the whole wave by one lane.  bound_ctrl gives 0 for a
// source lane outside the row (or wave), so a shifted-in 0 is the identity
// of the sums below.
template <int CTRL, int ROWMASK, bool BC>
__device__ __forceinline__ float dpp(float x)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, ROWMASK,
                                                                 0xf, BC));
}
template <int CTRL, int ROWMASK, bool BC>
__device__ __forceinline__ double dpp(double x)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b & 0xffffffffull), CTRL, ROWMASK, 0xf, BC);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, ROWMASK, 0xf, BC);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// value of lane r-1 (lane 0 of the wave: 0)
template <typename T>
__device__ __forceinline__ T lane_shr1(T x)
{
    return dpp<0x138, 0xf, true>(x);
}

// Inclusive prefix sum over segments of W lanes (W = 16, 32 or 64).
template <int W, typename T>
__device__ __forceinline__ T seg_prefix(T x)
{
    x = x + dpp<0x111, 0xf, true>(x);
    x = x + dpp<0x112, 0xf, true>(x);
    x = x + dpp<0x114, 0xf, true>(x);
    x = x + dpp<0x118, 0xf, true>(x);
    if constexpr (W >= 32) x = x + dpp<0x142, 0xa, false>(x);
    if constexpr (W >= 64) x = x + dpp<0x143, 0xc, false>(x);
    return x;
}

// Tile of workgroup b of an nb-workgroup launch.  The dispatcher hands
// workgroup b to XCD b % 8 (round robin over the 8 XCDs of MI355X, each
// with its own L2).  Each XCD is given a contiguous run of tiles instead,
// so tiles that are neighbours along i, which share the 64-byte segments
// at their edges (a tile row is TXB values from an arbitrary offset), are
// read into and written back from one L2, by workgroups that run at about
// the same time.  A bijection of [0, nb).
__device__ __forceinline__ unsigned xcd_tile(unsigned b, unsigned nb)
{
    constexpr unsigned X = 8;
    const unsigned x = b % X, s = b / X, q = nb / X, rem = nb % X;
    return x * q + (x < rem ? x : rem) + s;
}

}  // namespace obme
