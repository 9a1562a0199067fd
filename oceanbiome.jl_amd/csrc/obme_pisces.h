// obme_pisces.h — PISCES (OceanBioME.jl src/Models/AdvectedPopulations/PISCES)
// on gfx950: the 24 per-cell transitions, the MultiBand light, euphotic
// depth and mixed-layer means of the update-state step, the per-cell calcite
// saturation (FP64 carbonate solve with silicate and pressure), and the
// sinking of the particle tracers.
//
// Kernels (one RK3 stage each):
//   k_pisces_columns  blocks of water columns: MultiBand PAR from the surface
//                     down (multi_band.jl:147-165), euphotic depth
//                     (compute_euphotic_depth.jl:3-33), mixed-layer mean PAR
//                     (mean_mixed_layer_properties.jl:25-47);
//   k_pisces_omega    thread per cell: calcite saturation (FP64,
//                     compute_calcite_saturation.jl:22-36);
//   k_pisces_cell     thread per cell: transitions, sinking divergence and
//                     the RK3 substep (or the tendency output).
// FT is the arithmetic type of the transitions (double: the reference's
// expressions in order; float: the FP32-mixed path).  Julia semantics:
// NaN-propagating min/max (jmin/jmax), eps(0.0) guards, x^2 as x*x.
#pragma once

#include "obme_device.h"

namespace obme {
namespace pisces {

constexpr double DAYS = 86400.0;
constexpr double EPS0 = 4.9406564584124654e-324;  // Julia eps(0.0)

template <typename FT>
__device__ __forceinline__ FT eps0()
{
    if constexpr (sizeof(FT) == 8) return EPS0;
    else return 1.17549435e-38f;  // the smallest normal float keeps the FP32 guards finite
}

// The quotients of the transitions.  FP64: the IEEE quotient (the
// reference's expressions, unchanged).  FP32-mixed: the dividend times the
// hardware reciprocal (within 2 ulp; two instructions, where the compiler's
// quotient scales both operands for denormal and huge divisors, which these
// divisors are not: tracer sums guarded by the smallest normal, parameters).
template <typename FT>
__device__ __forceinline__ FT qdiv(FT a, FT b)
{
    if constexpr (sizeof(FT) == 8) return a / b;
    else return a * __builtin_amdgcn_rcpf(b);
}

// a / k for a constant k: times 1/k, folded at compile time.
template <typename FT>
__device__ __forceinline__ FT qdivk(FT a, double k)
{
    return a * (FT)(1.0 / k);
}

template <typename FT>
__device__ __forceinline__ FT jmin3(FT a, FT b, FT c) { return jmin(jmin(a, b), c); }
template <typename FT>
__device__ __forceinline__ FT jmin4(FT a, FT b, FT c, FT d) { return jmin(jmin(jmin(a, b), c), d); }

template <typename FT>
__device__ __forceinline__ FT m_log(FT x)
{
    if constexpr (sizeof(FT) == 8) return m_log_any(x);
    else return __builtin_amdgcn_logf(x) * 0.693147180559945309f;
}

// sind / cosd with the argument reduced modulo 360 first
__device__ __forceinline__ double sind(double x) { return sin(fmod(x, 360.0) * (3.141592653589793 / 180.0)); }
__device__ __forceinline__ double cosd(double x) { return cos(fmod(x, 360.0) * (3.141592653589793 / 180.0)); }

// CBMDayLength()(t, φ) (src/Utils/Utils.jl:17-33) in seconds, FP64.
__device__ __forceinline__ double day_length(double t, double phi)
{
    const double p = 0.833;
    double J = floor(fmod(t, 365 * DAYS) / DAYS);
    if (fmod(t, 365 * DAYS) < 0) J = floor((fmod(t, 365 * DAYS) + 365 * DAYS) / DAYS);
    double theta = 0.216310 + 2 * atan(0.9671396 * tan(0.00860 * (J - 186)));
    double dec = asin(0.39795 * cos(theta)) * (180.0 / 3.141592653589793);
    double L = jmax(-1.0, jmin(1.0, (sind(p) + sind(phi) * sind(dec)) / (cosd(phi) * cosd(dec))));
    return (24 - 24.0 / 180 * (acos(L) * (180.0 / 3.141592653589793))) * 3600.0;
}

// Per-stage uniform inputs of the transitions, from the day lengths
// d = day_length(φ, t) (the argument order of growth_rate.jl:30) and
// d' = day_length(t, φ) (growth_rate.jl:128).  There is no scalar float
// arithmetic: what is the same for every cell is formed on the host (here, and
// below what depends on the parameters alone).
template <typename FT>
struct StageConst {
    FT f1;          // f₁(d) = 1.5 d / (d + 1/2 day)
    FT rl[2];       // 1 / (d (basal respiration + reference growth)): nanophytoplankton, diatoms
    FT chl;         // d' / f₁(d')
};

// Combinations of the parameters, behind them in the device's array.
enum {
    PD_KSI_N, PD_KSI_D,        // 7 Sc² / (pk² + Sc²) of the half saturation for silicate
    PD_RFE_N, PD_RFE_D,        // 1 / θFe optimum
    PD_RKAPPA,                 // 1 / κ
    PD_UTW,                    // m₀ / (1 - e₀) of the mesozooplankton
    PD_UT_KEEP,                // 1 - e₀ - σ
    PD_DOC_RATE,               // λ / Bact reference
    PD_RFIX_E,                 // 1 / E fixation
    PD_RAIN_ZM,                // min(1, -50 / zmxl)
    PD_O2_N,                   // θ nitrification / θN
    PD_COUNT
};
// (p: the OBME_PP_COUNT parameters)
inline void derived_parameters(const double* p, double* d)
{
    const double *n = p + OBME_PP_NANO, *m = p + OBME_PP_DIATOMS, *z = p + OBME_PP_MESO, *s = p + OBME_PP_SCALARS;
    const double c2 = s[OBME_PS_SILICATE_CLIMATOLOGY] * s[OBME_PS_SILICATE_CLIMATOLOGY];
    d[PD_KSI_N] = 7 * c2 / (n[OBME_PH_PK] * n[OBME_PH_PK] + c2);
    d[PD_KSI_D] = 7 * c2 / (m[OBME_PH_PK] * m[OBME_PH_PK] + c2);
    d[PD_RFE_N] = 1 / n[OBME_PH_THETA_FE_OPT];
    d[PD_RFE_D] = 1 / m[OBME_PH_THETA_FE_OPT];
    d[PD_RKAPPA] = 1 / s[OBME_PS_KAPPA];
    d[PD_UTW] = 1 / (1 - z[OBME_PZ_E0]) * z[OBME_PZ_M0];
    d[PD_UT_KEEP] = 1 - z[OBME_PZ_E0] - z[OBME_PZ_SIGMA];
    d[PD_DOC_RATE] = s[OBME_PS_DOC_LAMBDA] / s[OBME_PS_DOC_BACT_REF];
    d[PD_RFIX_E] = 1 / s[OBME_PS_FIX_E];
    const double q = -50 / s[OBME_PS_MIXED_LAYER_DEPTH];
    d[PD_RAIN_ZM] = q < 1 ? q : 1;     // (the depth is below 0, checked at create)
    d[PD_O2_N] = s[OBME_PS_O2_NITRIF] / s[OBME_PS_THETAN];
}

// Auxiliary values of one cell.
template <typename FT>
struct Aux {
    FT z, zmxl, zeu, mlPAR, Omega, PAR, PAR1, PAR2, PAR3, wPOCc, wGOCc;
};

// The factors of the transitions that depend on the temperature alone: the
// growth rates' bᵀ of the two phytoplankton and two zooplankton classes
// (growth_rate.jl:25, food_quality_dependant.jl:157), of DOC and POM
// degradation (dissolved_organic_carbon.jl:62, two_size_class.jl:154), the
// rain ratio's 1 + exp(-(T-10)²/25) (nano_diatom_coupling.jl), the ligand
// constant of the free iron (iron/iron.jl:29), the silicate equilibrium
// 10^(6.44 - 968/T_K) and (1 + T/400)^4 (silicate.jl:30-34).  The rain ratio's
// takes max(0, T / (T + 0.1)) with it, the silicate equilibrium enters as its
// reciprocal and t15 is 0.225 (1 + T/15).  The same expressions whether
// evaluated per stage or once per stepper call.
template <typename FT>
struct TFac {
    FT btN, btD, bZ, bM, doc, pom, rain, kfe, req, t4, t15;
};
constexpr int TFAC_FIELDS = 11;

template <typename FT>
__device__ __forceinline__ void temperature_factors(const FT* pp, FT T, TFac<FT>& f)
{
    const FT* sc = pp + OBME_PP_SCALARS;
    f.btN = m_pow(pp[OBME_PP_NANO + OBME_PH_BT], T);
    f.btD = m_pow(pp[OBME_PP_DIATOMS + OBME_PH_BT], T);
    f.bZ = m_pow(pp[OBME_PP_MICRO + OBME_PZ_B], T);
    f.bM = m_pow(pp[OBME_PP_MESO + OBME_PZ_B], T);
    f.doc = m_pow(sc[OBME_PS_DOC_B], T);
    f.pom = m_pow(sc[OBME_PS_POM_B], T);
    const FT Tm = T - 10;
    f.rain = jmax(FT(0), qdiv(T, T + FT(0.1))) * (1 + m_exp(qdivk(-(Tm * Tm), 25)));
    f.kfe = m_exp(FT(16.27) - qdiv(FT(1565.7), jmax(T + FT(273.15), FT(5))));
    f.req = m_pow(FT(10), qdiv(FT(968), T + FT(273.15)) - FT(6.44));
    const FT t = 1 + qdivk(T, 400), t2 = t * t;
    f.t4 = t2 * t2;
    f.t15 = FT(0.225) * (1 + qdivk(T, 15));
}

// One phytoplankton class (parameters at block b of pp).
template <typename FT>
struct Phyto {
    FT I, IChl, IFe;
    FT L, LFe, LPO4, LN, LNO3, LNH4;
    FT mu, muI;
    FT Kb, PAR, alpha;   // size factor, absorbed light, light sensitivity
};

template <typename FT>
__device__ __forceinline__ FT size_factor(const FT* ph, FT I)
{
    const FT Im = ph[OBME_PH_SIZE_THRESHOLD];
    FT I1 = jmin(I, Im);
    FT I2 = jmax(FT(0), I - Im);
    return qdiv(I1 + ph[OBME_PH_SIZE_RATIO] * I2, I1 + I2 + eps0<FT>());
}

template <typename FT>
__device__ __forceinline__ FT nitrogen_lim(FT N1, FT N2, FT K1, FT K2)
{
    return qdiv(K2 * N1, K1 * K2 + K1 * N2 + K2 * N1 + eps0<FT>());
}

// NitrogenIronPhosphateSilicateLimitation (nutrient_limitation.jl:20-71) and
// the growth rate (growth_rate.jl:3-47, GrowthRespirationLimitedProduction :104-111).
template <typename FT>
__device__ __forceinline__ void phyto_state(const FT* ph, const FT* sc, const FT* v, const Aux<FT>& A,
                                            const StageConst<FT>& sk, const FT* pd, int cls, FT btT, FT I, FT IChl, FT IFe,
                                            Phyto<FT>& s)
{
    const FT NO3 = v[OBME_PI_NO3], NH4 = v[OBME_PI_NH4], PO4 = v[OBME_PI_PO4], Si = v[OBME_PI_SI];
    s.I = I;
    s.IChl = IChl;
    s.IFe = IFe;
    const FT thFe = (I == FT(0)) ? FT(0) : qdiv(IFe, I + eps0<FT>());
    const FT thChl = (I == FT(0)) ? FT(0) : qdiv(IChl, 12 * I + eps0<FT>());
    const FT Kb = size_factor(ph, I);
    s.Kb = Kb;
    const FT Kno = ph[OBME_PH_KNO3] * Kb, Knh = ph[OBME_PH_KNH4] * Kb, Kp = ph[OBME_PH_KPO4] * Kb,
             Ksi = ph[OBME_PH_KSI_MIN] * Kb;
    s.LNO3 = nitrogen_lim(NO3, NH4, Kno, Knh);
    s.LNH4 = nitrogen_lim(NH4, NO3, Knh, Kno);
    s.LN = s.LNO3 + s.LNH4;
    s.LPO4 = qdiv(PO4, PO4 + Kp + eps0<FT>());
    const FT thm = FT(1000) * (FT(0.0016) / FT(55.85) * FT(12) * thChl
                               + FT(1.5) * FT(1.21e-5) * FT(14) / (FT(55.85) * FT(7.625)) * s.LN
                               + FT(1.15e-4) * FT(14) / (FT(55.85) * FT(7.625)) * s.LNO3);
    s.LFe = jmin(FT(1), jmax(FT(0), (thFe - thm) * pd[PD_RFE_N + cls]));
    const FT KSi = Ksi + pd[PD_KSI_N + cls];
    FT LSi = qdiv(Si, Si + KSi);
    if (ph[OBME_PH_SI_LIMITED] == FT(0)) LSi = FT(INFINITY);
    s.L = jmin4(s.LN, s.LPO4, s.LFe, LSi);
    // growth rate μ(L)
    const FT PAR = ph[OBME_PH_BETA1] * A.PAR1 + ph[OBME_PH_BETA2] * A.PAR2 + ph[OBME_PH_BETA3] * A.PAR3;
    const FT d = jmax(FT(0), A.zeu - A.zmxl);
    const FT drt = d * d * pd[PD_RKAPPA];
    const FT mui = ph[OBME_PH_MU0] * btT;
    const FT f2 = 1 - qdiv(drt, drt + ph[OBME_PH_DARK_TOLERANCE]);
    const FT alpha = ph[OBME_PH_ALPHA0] * (1 + ph[OBME_PH_BETA] * m_exp(-PAR));
    s.PAR = PAR;
    s.alpha = alpha;
    const FT theta = qdiv(IChl, 12 * I + eps0<FT>());
    const FT fl = 1 - m_exp(-alpha * theta * PAR * sk.rl[cls]);
    s.mu = mui * sk.f1 * f2 * fl * s.L;
    s.muI = s.mu * I;
}

// mortality (mixed_mondo.jl:115-133): linear, quadratic
template <typename FT>
__device__ __forceinline__ void phyto_mortality(const FT* ph, const FT* sc, const Phyto<FT>& s, const Aux<FT>& A,
                                                FT& lin, FT& quad)
{
    const FT I = s.I;
    lin = qdiv(ph[OBME_PH_MORT_LIN] * I, I + ph[OBME_PH_MORT_K]) * I;
    const FT L2 = s.L * s.L;
    const FT w = ph[OBME_PH_MORT_W0] + qdiv(ph[OBME_PH_MORT_W1] * FT(0.25) * (1 - L2), FT(0.25) + L2);
    const FT shear = (A.z < A.zmxl) ? sc[OBME_PS_BACKGROUND_SHEAR] : sc[OBME_PS_MIXED_LAYER_SHEAR];
    quad = shear * w * (I * I);
}

// chlorophyll growth (mixed_mondo.jl:84-97; growth_rate.jl:113-148)
template <typename FT>
__device__ __forceinline__ FT chlorophyll_growth(const FT* ph, const Phyto<FT>& s, const StageConst<FT>& sk)
{
    const FT mucheck = s.mu * sk.chl;
    const FT rho = qdiv(12 * mucheck * s.I, s.alpha * s.IChl * s.PAR + eps0<FT>()) * s.L;
    const FT th0 = ph[OBME_PH_CHL_MIN], th1 = ph[OBME_PH_CHL_MAX];
    return (1 - ph[OBME_PH_DELTA]) * 12 * (th0 + (th1 - th0) * rho) * s.mu * s.I;
}

// iron uptake (mixed_mondo.jl:161-181)
template <typename FT>
__device__ __forceinline__ FT iron_uptake(const FT* ph, const Phyto<FT>& s, FT btT, FT Fe)
{
    const FT fe_max = ph[OBME_PH_FE_MAX];
    const FT mui = ph[OBME_PH_MU0] * btT;
    const FT K = ph[OBME_PH_KFE_UPTAKE] * s.Kb;
    const FT L1 = qdiv(Fe, Fe + K + eps0<FT>());
    const FT L2 = 4 - qdiv(FT(4.5) * s.LFe, s.LFe + 1);
    // (1 - r) / (1.05 - r), r = θFe / θFe_max, θFe = IFe / (I + ε)
    FT pole;
    if constexpr (sizeof(FT) == 8) {
        const FT thFe = s.IFe / (s.I + eps0<FT>());
        const FT r = thFe / fe_max;
        pole = (1 - r) / (FT(1.05) - r);
    } else {
        // the same quotient times F / F, F = θFe_max (I + ε):
        // (F - IFe) / (1.05 F - IFe), with F's product exact inside the FMAs
        // and 1.05 split into two floats.  Near the pole (r -> 1.05) the
        // denominator is a small difference, and rounding r first would lose
        // its leading digits.
        const FT Ie = s.I + eps0<FT>();
        const FT Fh = fe_max * Ie, Fl = fmaf(fe_max, Ie, -Fh);
        const FT c = 1.05f, cl = (float)(1.05 - (double)1.05f);
        const FT num = fmaf(fe_max, Ie, -s.IFe);
        const FT den = fmaf(c, Fh, -s.IFe) + fmaf(c, Fl, cl * Fh);
        pole = qdiv(num, den);
    }
    return (1 - ph[OBME_PH_DELTA]) * fe_max * L1 * L2 * jmax(FT(0), pole) * mui * s.I;
}

// silicate uptake (mixed_mondo.jl:195-226)
template <typename FT>
__device__ __forceinline__ FT silicate_uptake(const FT* ph, const FT* sc, const Phyto<FT>& s, FT btT, FT Si)
{
    const FT mui = ph[OBME_PH_MU0] * btT;
    const FT L1 = qdiv(Si, Si + ph[OBME_PH_SI_K1] + eps0<FT>());
    const FT K2 = ph[OBME_PH_SI_K2];
    const FT L2 = (sc[OBME_PS_LATITUDE] < FT(0)) ? qdiv(Si * Si * Si, Si * Si * Si + K2 * K2 * K2) : FT(0);
    const FT F1 = jmin4(qdiv(s.mu, mui * s.L + eps0<FT>()), s.LFe, s.LPO4, s.LN);
    const FT F2 = jmin(FT(1), FT(2.2) * jmax(FT(0), L1 - FT(0.5)));
    const FT th1 = ph[OBME_PH_SI_THETA0] * L1 * jmin(FT(5.4), (FT(4.4) * m_exp(FT(-4.23) * F1) * F2 + 1) * (1 + 2 * L2));
    return (1 - ph[OBME_PH_DELTA]) * th1 * s.mu * s.I;
}

// QualityDependantZooplankton grazing of one class (food_quality_dependant.jl:138-183,
// iron_grazing.jl:1-36); prey order P, D, POC (, Z for the meso class).
template <typename FT>
struct Zoo {
    FT I, on, gI, ge, gIFe, ff, ffFe, tf;
};

template <typename FT, int NPREY>
__device__ __forceinline__ void zoo_state(const FT* zp, const FT* v, FT bT, FT micro_iron, FT wPOCc, FT wGOCc, FT I,
                                          Zoo<FT>& g)
{
    g.I = I;
    g.tf = bT;
    const FT base = zp[OBME_PZ_G0] * g.tf;
    const FT food[4] = {v[OBME_PI_P], v[OBME_PI_D], v[OBME_PI_POC], v[OBME_PI_Z]};
    const FT iron[4] = {qdiv(v[OBME_PI_PFE], v[OBME_PI_P] + eps0<FT>()), qdiv(v[OBME_PI_DFE], v[OBME_PI_D] + eps0<FT>()),
                        qdiv(v[OBME_PI_SFE], v[OBME_PI_POC] + eps0<FT>()), micro_iron};
    const FT pref[4] = {zp[OBME_PZ_PREF_P], zp[OBME_PZ_PREF_D], zp[OBME_PZ_PREF_POC], zp[OBME_PZ_PREF_Z]};
    const FT J = zp[OBME_PZ_J];
    FT total_food = food[0] * pref[0];
    FT avail = jmax(FT(0), food[0] - J) * pref[0];
    FT total_iron = iron[0] * pref[0];
    FT s = jmax(FT(0), food[0] - J) * pref[0] * iron[0];
#pragma unroll
    for (int n = 1; n < NPREY; n++) {
        total_food = total_food + food[n] * pref[n];
        avail = avail + jmax(FT(0), food[n] - J) * pref[n];
        total_iron = total_iron + iron[n] * pref[n];
        s = s + jmax(FT(0), food[n] - J) * pref[n] * iron[n];
    }
    const FT clg = jmax(FT(0), avail - jmin(avail / 2, zp[OBME_PZ_FOOD_THRESHOLD]));
    const FT tsg = qdiv(base * clg, zp[OBME_PZ_K] + total_food);
    const FT igr = qdiv(total_iron, zp[OBME_PZ_IRON_RATIO] * tsg + eps0<FT>());
    const FT fq = jmin(FT(1), igr);
    g.ge = fq * jmin(zp[OBME_PZ_E0], (1 - zp[OBME_PZ_SIGMA]) * igr);
    g.gI = tsg * I;
    // what is grazed per available prey: one quotient for every prey and its
    // iron (avail = 0 has tsg = 0)
    g.on = qdiv(g.gI, avail + eps0<FT>());
    g.gIFe = s * g.on;
    // flux feeding on the sinking particles (food_quality_dependant.jl:185-199, iron_grazing.jl:38-53)
    const FT ffb = zp[OBME_PZ_FF] * g.tf;
    g.ff = ffb * (v[OBME_PI_POC] * wPOCc + v[OBME_PI_GOC] * wGOCc) * I;
    g.ffFe = ffb * (v[OBME_PI_SFE] * wPOCc + v[OBME_PI_BFE] * wGOCc) * I;
}

// grazing of one class on one prey (food_quality_dependant.jl:215-243)
template <typename FT>
__device__ __forceinline__ FT zoo_on(const FT* zp, const Zoo<FT>& g, FT pref, FT prey)
{
    return pref * jmax(FT(0), prey - zp[OBME_PZ_J]) * g.on;
}

template <typename FT>
__device__ __forceinline__ FT anoxia(const FT* sc, FT O2)
{
    return jmin(FT(1), jmax(FT(0), qdiv(FT(0.4) * (sc[OBME_PS_ANOXIA1] - O2), sc[OBME_PS_ANOXIA2] + O2)));
}

// The parameters' pointer again, by an offset the compiler cannot see through
// and only once `after` is known: what follows loads them anew.
template <typename FT>
__device__ __forceinline__ const FT* reread(const FT* pp, FT after)
{
    int none;
    asm("s_mov_b32 %0, 0" : "=s"(none) : "v"(after));
    return pp + none;
}

// The 24 transitions of one cell (v: tracers in OBME_PI order).  SECTIONS (the
// fused step): each section loads its parameters anew, where the compiler keeps
// what a later one uses again in lanes of vector registers (256x256x64, 10
// steps: 4290 -> 4166 us).  Not in FP64, with two waves per SIMD to cover the
// loads (238 lanes fewer, but 1146 -> 1236 us at 120x100x48), nor in the hook
// (185 -> 192).
template <bool SECTIONS = false, typename FT>
__device__ __forceinline__ void pisces_tendencies(const FT* pp, const FT* v, const Aux<FT>& A,
                                                  const StageConst<FT>& sk, const TFac<FT>& tf, FT* G)
{
    const FT* phN = pp + OBME_PP_NANO;
    const FT* phD = pp + OBME_PP_DIATOMS;
    const FT* zpZ = pp + OBME_PP_MICRO;
    const FT* zpM = pp + OBME_PP_MESO;
    const FT* sc = pp + OBME_PP_SCALARS;
    const FT* pd = pp + OBME_PP_COUNT;
    const FT e0 = eps0<FT>();

    auto section = [&](FT after) {
        if constexpr (SECTIONS) {
            pp = reread(pp, after);
            phN = pp + OBME_PP_NANO;
            phD = pp + OBME_PP_DIATOMS;
            zpZ = pp + OBME_PP_MICRO;
            zpM = pp + OBME_PP_MESO;
            sc = pp + OBME_PP_SCALARS;
            pd = pp + OBME_PP_COUNT;
        }
    };

    Phyto<FT> sP, sD;
    phyto_state(phN, sc, v, A, sk, pd, 0, tf.btN, v[OBME_PI_P], v[OBME_PI_PCHL], v[OBME_PI_PFE], sP);
    section(sP.muI);
    phyto_state(phD, sc, v, A, sk, pd, 1, tf.btD, v[OBME_PI_D], v[OBME_PI_DCHL], v[OBME_PI_DFE], sD);
    section(sD.muI);
    Zoo<FT> gZ, gM;
    const FT micro_iron = zpZ[OBME_PZ_IRON_RATIO];
    zoo_state<FT, 3>(zpZ, v, tf.bZ, micro_iron, A.wPOCc, A.wGOCc, v[OBME_PI_Z], gZ);
    zoo_state<FT, 4>(zpM, v, tf.bM, micro_iron, A.wPOCc, A.wGOCc, v[OBME_PI_M], gM);
    section(gM.gIFe);
    const FT O2 = v[OBME_PI_O2];
    const FT an = anoxia(sc, O2);
    // zooplankton mortality (food_quality_dependant.jl:201-227)
    auto zmort = [&](const FT* zp, const Zoo<FT>& g, FT& mort, FT& lin) {
        const FT cf = qdiv(g.I, g.I + zp[OBME_PZ_KM]);
        mort = g.tf * g.I * (zp[OBME_PZ_M0] * g.I + zp[OBME_PZ_R] * (cf + 3 * an));
        lin = g.tf * zp[OBME_PZ_R] * (cf + 3 * an) * g.I;
    };
    FT mZ, linZ, mM, linM;
    zmort(zpZ, gZ, mZ, linZ);
    zmort(zpM, gM, mM, linM);
    (void)linZ;
    auto graz = [&](int prey_pref, FT prey) {
        return zoo_on(zpZ, gZ, zpZ[prey_pref], prey) + zoo_on(zpM, gM, zpM[prey_pref], prey);
    };
    const FT shear_lt = (A.z < A.zmxl) ? sc[OBME_PS_BACKGROUND_SHEAR] : sc[OBME_PS_MIXED_LAYER_SHEAR];

    // phytoplankton (mixed_mondo_nano_diatoms.jl:47-111)
    FT Plin, Pquad, Dlin, Dquad;
    phyto_mortality(phN, sc, sP, A, Plin, Pquad);
    phyto_mortality(phD, sc, sD, A, Dlin, Dquad);
    const FT grazP = graz(OBME_PZ_PREF_P, v[OBME_PI_P]);
    const FT grazD = graz(OBME_PZ_PREF_D, v[OBME_PI_D]);
    {
        const FT death = Plin + Pquad;
        G[OBME_PI_P] = (1 - phN[OBME_PH_DELTA]) * sP.muI - death - grazP;
        const FT thChl = qdiv(sP.IChl, 12 * sP.I + e0);
        G[OBME_PI_PCHL] = chlorophyll_growth(phN, sP, sk) - (death + grazP) * thChl * 12;
        const FT thFe = qdiv(sP.IFe, sP.I + e0);
        G[OBME_PI_PFE] = iron_uptake(phN, sP, tf.btN, v[OBME_PI_FE]) - (death + grazP) * thFe;
    }
    {
        const FT death = Dlin + Dquad;
        G[OBME_PI_D] = (1 - phD[OBME_PH_DELTA]) * sD.muI - death - grazD;
        const FT thChl = qdiv(sD.IChl, 12 * sD.I + e0);
        G[OBME_PI_DCHL] = chlorophyll_growth(phD, sD, sk) - (death + grazD) * thChl * 12;
        const FT thFe = qdiv(sD.IFe, sD.I + e0);
        G[OBME_PI_DFE] = iron_uptake(phD, sD, tf.btD, v[OBME_PI_FE]) - (death + grazD) * thFe;
    }
    const FT si_uptake = silicate_uptake(phD, sc, sD, tf.btD, v[OBME_PI_SI]);
    const FT thSi = qdiv(v[OBME_PI_DSI], v[OBME_PI_D] + e0);
    G[OBME_PI_DSI] = si_uptake - (Dlin + Dquad + grazD) * thSi;

    section(G[OBME_PI_DFE]);
    // zooplankton (micro_and_meso.jl:36-48)
    G[OBME_PI_Z] = gZ.ge * (gZ.gI + gZ.ff) - mZ - zoo_on(zpM, gM, zpM[OBME_PZ_PREF_Z], v[OBME_PI_Z]);
    G[OBME_PI_M] = gM.ge * (gM.gI + gM.ff) - mM;

    const FT sigZ = zpZ[OBME_PZ_SIGMA], sigM = zpM[OBME_PZ_SIGMA];
    const FT excZ = (1 - sigZ - gZ.ge) * (gZ.gI + gZ.ff);
    const FT excM = (1 - sigM - gM.ge) * (gM.gI + gM.ff);
    const FT inorg_exc = zpZ[OBME_PZ_GAMMA] * excZ + zpM[OBME_PZ_GAMMA] * excM;
    const FT org_exc = (1 - zpZ[OBME_PZ_GAMMA]) * excZ + (1 - zpM[OBME_PZ_GAMMA]) * excM;
    // upper trophic waste of the meso class (mortality_waste.jl)
    const FT utw = pd[PD_UTW] * gM.tf * (gM.I * gM.I);
    const FT R_ut = pd[PD_UT_KEEP] * utw;
    const FT fecal = zpM[OBME_PZ_SIGMA] * utw;
    const FT ut_excretion = (1 - zpM[OBME_PZ_GAMMA]) * R_ut;
    const FT ut_respiration = zpM[OBME_PZ_GAMMA] * R_ut;

    // bacteria (micro_and_meso.jl:85-132)
    const FT zm = jmin(A.zmxl, A.zeu);
    const FT surface_bact = jmin(sc[OBME_PS_BACT_MAX], sc[OBME_PS_BZ] * v[OBME_PI_Z] + sc[OBME_PS_BM] * v[OBME_PI_M]);
    const FT Bact = ((A.z >= zm) ? FT(1) : m_pow(qdiv(zm, A.z), sc[OBME_PS_BACT_EXP])) * surface_bact;
    const FT DOC = v[OBME_PI_DOC], NO3 = v[OBME_PI_NO3], NH4 = v[OBME_PI_NH4], PO4 = v[OBME_PI_PO4],
             Fe = v[OBME_PI_FE];
    const FT KNO = sc[OBME_PS_K_NO3_B], KNH = sc[OBME_PS_K_NH4_B];
    const FT LBact = jmin3(qdiv(KNO * NH4 + KNH * NO3, KNO * KNH + KNO * NH4 + KNH * NO3),
                           qdiv(PO4, PO4 + sc[OBME_PS_K_PO4_B]), qdiv(Fe, Fe + sc[OBME_PS_K_FE_B]))
                     * qdiv(DOC, DOC + sc[OBME_PS_K_DOC]);

    section(LBact);
    // DOC (dissolved_organic_carbon.jl:39-106)
    const FT doc_deg = pd[PD_DOC_RATE] * tf.doc * LBact * Bact * DOC;
    const FT POC = v[OBME_PI_POC], GOC = v[OBME_PI_GOC];
    const FT Phi1 = shear_lt * (sc[OBME_PS_DOC_A1] * DOC + sc[OBME_PS_DOC_A2] * POC) * DOC;
    const FT Phi2 = shear_lt * (sc[OBME_PS_DOC_A3] * GOC) * DOC;
    const FT Phi3 = (sc[OBME_PS_DOC_A4] * POC + sc[OBME_PS_DOC_A5] * DOC) * DOC;
    const FT doc_agg = Phi1 + Phi2 + Phi3;
    const FT lam_pom = sc[OBME_PS_POM_LAMBDA] * tf.pom * (1 - FT(0.45) * an);
    const FT pom_deg_POC = lam_pom * POC;
    const FT exudate = phN[OBME_PH_DELTA] * sP.muI + phD[OBME_PH_DELTA] * sD.muI;
    G[OBME_PI_DOC] = exudate + ut_excretion + org_exc + pom_deg_POC - doc_deg - doc_agg;
    const FT oxic = (1 - an) * doc_deg;
    const FT anoxic = an * doc_deg;

    // particles: aggregation, rain ratio and the mortality partitions
    // (two_size_class.jl:109-143, nano_diatom_coupling.jl)
    const FT pom_agg = shear_lt * (sc[OBME_PS_POM_A1] * (POC * POC) + sc[OBME_PS_POM_A2] * POC * GOC)
                       + sc[OBME_PS_POM_A3] * POC * GOC + sc[OBME_PS_POM_A4] * (POC * POC);
    const FT PAR = A.PAR;
    const FT L_CaCO3 = jmin3(sP.LN, qdiv(Fe, Fe + FT(0.05)), sP.LPO4);
    const FT R = sc[OBME_PS_RAIN_RATIO] * L_CaCO3 * jmax(FT(1), v[OBME_PI_P] / 2)
                 * qdiv(jmax(FT(0), PAR - 1), 4 + PAR) * qdiv(FT(30), 30 + PAR) * tf.rain * pd[PD_RAIN_ZM];
    const FT small_mort = (1 - R / 2) * (Plin + Pquad) + Dlin / 2;
    const FT large_mort = R / 2 * (Plin + Pquad) + Dlin / 2 + Dquad;
    const FT thP = qdiv(v[OBME_PI_PFE], v[OBME_PI_P] + e0);
    const FT thD = qdiv(v[OBME_PI_DFE], v[OBME_PI_D] + e0);
    const FT small_mort_fe = (1 - R / 2) * (Plin + Pquad) * thP + Dlin * thD / 2;
    const FT large_mort_fe = R / 2 * (Plin + Pquad) * thP + (Dlin / 2 + Dquad) * thD;
    const FT ffbZ = zpZ[OBME_PZ_FF] * gZ.tf, ffbM = zpM[OBME_PZ_FF] * gM.tf;
    const FT tot_graz_POC = graz(OBME_PZ_PREF_POC, POC) + (ffbZ * (POC * A.wPOCc) * gZ.I + ffbM * (POC * A.wPOCc) * gM.I);
    const FT tot_graz_GOC = ffbZ * (GOC * A.wGOCc) * gZ.I + ffbM * (GOC * A.wGOCc) * gM.I;

    // carbon.jl:3-50
    G[OBME_PI_POC] = (sigZ * (gZ.gI + gZ.ff) + small_mort + mZ + (Phi1 + Phi3) + lam_pom * GOC
                      - tot_graz_POC - pom_agg - pom_deg_POC);
    G[OBME_PI_GOC] = (sigM * (gM.gI + gM.ff) + large_mort + linM + fecal + pom_agg + Phi2
                      - tot_graz_GOC - lam_pom * GOC);

    section(G[OBME_PI_GOC]);
    // iron in particles (iron.jl:2-89) with the free iron of SimpleIron (iron/iron.jl:25-37)
    const FT ligands = jmax(FT(0.6), FT(0.09) * (DOC + 40) - 3);
    const FT Kfe = tf.kfe;
    const FT Dl = 1 + Kfe * ligands - Kfe * Fe;
    const FT Fef = qdiv(-Dl + m_sqrt(Dl * Dl + 4 * Kfe * Fe), 2 * Kfe);
    const FT colloidal = FT(0.5) * (Fe - Fef);
    const FT CgFe1 = qdiv((Phi1 + Phi3) * colloidal, DOC + e0);
    const FT CgFe2 = qdiv(Phi2 * colloidal, DOC + e0);
    const FT lamFe = sc[OBME_PS_FE_SCAV_MIN] + sc[OBME_PS_FE_SCAV_LOAD] * (POC + GOC + v[OBME_PI_CACO3] + v[OBME_PI_PSI]);
    const FT BactFe = qdiv(sc[OBME_PS_BACT_MU0] * tf.pom * LBact * sc[OBME_PS_BACT_FE_MAX] * Fe,
                           Fe + sc[OBME_PS_BACT_FE_K]) * Bact * sc[OBME_PS_BACT_FE_EFF];
    const FT thS = qdiv(v[OBME_PI_SFE], POC + e0);
    const FT thB = qdiv(v[OBME_PI_BFE], GOC + e0);
    G[OBME_PI_SFE] = (sigZ * (gZ.gIFe + gZ.ffFe) + small_mort_fe + mZ * zpZ[OBME_PZ_IRON_RATIO]
                      + lam_pom * v[OBME_PI_BFE] + lamFe * POC * Fef + sc[OBME_PS_SMALL_BACT_FE] * BactFe + CgFe1
                      - tot_graz_POC * thS - pom_agg * thS - lam_pom * v[OBME_PI_SFE]);
    G[OBME_PI_BFE] = (sigM * (gM.gIFe + gM.ffFe) + large_mort_fe + linM * zpM[OBME_PZ_IRON_RATIO]
                      + fecal * zpM[OBME_PZ_IRON_RATIO] + lamFe * GOC * Fef + sc[OBME_PS_LARGE_BACT_FE] * BactFe
                      + CgFe2 + pom_agg * thS - tot_graz_GOC * thB - lam_pom * v[OBME_PI_BFE]);

    section(G[OBME_PI_BFE]);
    // particulate silicate (silicate.jl:1-48)
    const FT chi = sc[OBME_PS_CHI0] * ((A.z >= zm) ? FT(1)
                                                   : m_exp(qdiv((sc[OBME_PS_SI_FAST] - sc[OBME_PS_SI_SLOW]) * (zm - A.z), A.wGOCc)));
    const FT lam0 = chi * sc[OBME_PS_SI_FAST] + (1 - chi) * sc[OBME_PS_SI_SLOW];
    const FT sat = 1 - v[OBME_PI_SI] * tf.req;
    const FT ts = tf.t4 * sat, ts2 = ts * ts, ts4 = ts2 * ts2;
    const FT lam_si = lam0 * (tf.t15 * sat + FT(0.775) * (ts4 * ts4 * ts));
    const FT si_diss = lam_si * v[OBME_PI_PSI];
    G[OBME_PI_PSI] = (grazD + Dlin + Dquad) * thSi - si_diss;

    // calcite (calcite.jl:1-19, nano_diatom_coupling.jl:96-104)
    const FT calc_loss = zpZ[OBME_PZ_ETA] * zoo_on(zpZ, gZ, zpZ[OBME_PZ_PREF_P], v[OBME_PI_P])
                         + zpM[OBME_PZ_ETA] * zoo_on(zpM, gM, zpM[OBME_PZ_PREF_P], v[OBME_PI_P]);
    const FT calc_prod = R * (calc_loss + (Plin + Pquad) / 2);
    const FT calc_diss = sc[OBME_PS_CACO3_LAMBDA] * m_pow(jmax(FT(0), 1 - A.Omega), sc[OBME_PS_CACO3_EXP])
                         * v[OBME_PI_CACO3];
    G[OBME_PI_CACO3] = calc_prod - calc_diss;

    section(G[OBME_PI_CACO3]);
    // nitrogen (nitrogen/nitrate_ammonia.jl:22-88)
    const FT thN = sc[OBME_PS_THETAN];
    const FT nitrif = qdiv(sc[OBME_PS_NITRIF] * NH4, 1 + A.mlPAR) * (1 - an);
    const FT fix_limit = (sP.LN >= FT(0.8)) ? FT(0.01) : 1 - sP.LN;
    const FT mu_nano = phN[OBME_PH_MU0] * tf.btN;
    const FT growth_req = jmax(FT(0), mu_nano - FT(2.15));
    const FT nut_lim = jmin(qdiv(Fe, Fe + sc[OBME_PS_FIX_KFE]), qdiv(PO4, PO4 + sc[OBME_PS_FIX_KPO4]));
    const FT light_lim = 1 - m_exp(-PAR * pd[PD_RFIX_E]);
    const FT fixation = sc[OBME_PS_FIX_MAX] * growth_req * fix_limit * nut_lim * light_lim;
    // (L <= LN: no uptake where LN = 0)
    const FT upP = qdiv(sP.muI, sP.LN + e0), upD = qdiv(sD.muI, sD.LN + e0);
    const FT up_NO3 = upP * sP.LNO3 + upD * sD.LNO3;
    const FT up_NH4 = upP * sP.LNH4 + upD * sD.LNH4;
    G[OBME_PI_NO3] = nitrif + thN * (oxic - up_NO3);
    G[OBME_PI_NH4] = fixation + thN * (anoxic + inorg_exc + ut_respiration - up_NH4) - nitrif;

    // phosphate (phosphate.jl:21-33)
    const FT total_prod = sP.muI + sD.muI;
    G[OBME_PI_PO4] = sc[OBME_PS_THETAP] * (inorg_exc + ut_respiration + doc_deg - total_prod);

    // iron (iron/simple_iron.jl:19-53)
    const FT ligand = jmax(sc[OBME_PS_FE_LIGAND_MAX], sc[OBME_PS_FE_LIGAND_RATIO] * DOC - sc[OBME_PS_FE_LIGAND_MAX]);
    const FT lig_agg = sc[OBME_PS_FE_EXCESS] * lamFe * jmax(FT(0), Fe - ligand) * Fef;
    const FT scav = lamFe * (POC + GOC) * Fef;
    const FT naZ = (gZ.gIFe + gZ.ffFe) - sigZ * (gZ.gIFe + gZ.ffFe) - zpZ[OBME_PZ_IRON_RATIO] * gZ.ge * (gZ.gI + gZ.ff);
    const FT naM = (gM.gIFe + gM.ffFe) - sigM * (gM.gIFe + gM.ffFe) - zpM[OBME_PZ_IRON_RATIO] * gM.ge * (gM.gI + gM.ff);
    const FT up_Fe = iron_uptake(phN, sP, tf.btN, Fe) + iron_uptake(phD, sD, tf.btD, Fe);
    G[OBME_PI_FE] = (lam_pom * v[OBME_PI_SFE] + (naZ + naM) + zpM[OBME_PZ_IRON_RATIO] * R_ut
                     - up_Fe - lig_agg - (CgFe1 + CgFe2) - scav - BactFe);

    // silicate (silicate.jl:20-26)
    G[OBME_PI_SI] = si_diss - si_uptake;

    // inorganic carbon (inorganic_carbon.jl:32-57)
    G[OBME_PI_DIC] = inorg_exc + ut_respiration + doc_deg + calc_diss - calc_prod - total_prod;
    G[OBME_PI_ALK] = G[OBME_PI_NH4] - G[OBME_PI_NO3] - 2 * G[OBME_PI_CACO3];

    // oxygen (oxygen.jl:30-50)
    const FT th_r = sc[OBME_PS_O2_RESP], th_n = sc[OBME_PS_O2_NITRIF];
    G[OBME_PI_O2] = (th_r * up_NH4 + (th_r + th_n) * up_NO3 + pd[PD_O2_N] * fixation
                     - ((th_r + th_n) * oxic + th_r * anoxic) - th_r * inorg_exc - th_r * ut_respiration
                     - pd[PD_O2_N] * nitrif);
}

// ---------------------------------------------------------------- calcite saturation (FP64)

// Millero (2007) pressure correction (equilibrium_constants.jl:29-38), a: a0 a1 a2 b0 b1
// (as the exponent, under the reciprocal of R T)
__device__ __forceinline__ double pressure_exponent(const double* a, double Tc, double P, double PRT)
{
    const double dV = a[0] + a[1] * Tc + a[2] * (Tc * Tc);
    const double dk = a[3] + a[4] * Tc;
    return (-dV + 0.5 * dk * P) * PRT;
}

// Constants of the calcite saturation that depend only on T, S and the
// pressure (fixed through a step of frozen physics): the unit conversion
// 1e-3/ρ(T, S, P), the pressure-corrected equilibrium constants that enter
// the residual (phosphate is 0, so KP1-3 do not), the salinity totals, the
// calcium concentration and KSP.
struct OmegaConst {
    double conv, K1, K2, KB, KW, KS, KF, KSi, boron, sulfate, fluoride, ca, KSP;
};
// stored per cell: conv to KSi and KSP (the salinity terms are formed from S,
// four multiplications against 32 B to read)
constexpr int OMEGA_CONST_FIELDS = 9;

// The salinity totals and the calcium concentration (functions of S alone).
__device__ __forceinline__ void omega_salinity_terms(double S, OmegaConst& c)
{
    c.boron = 0.000232 / 10.811 * S / 1.80655;
    c.sulfate = 0.14 / 96.06 * S / 1.80655;
    c.fluoride = 0.000067 / 18.9984 * S / 1.80655;
    c.ca = 0.0103 * S / 35;
}

// calcite_saturation (CarbonChemistry/calcite_concentration.jl:1-79) with
// silicate and the pressure P in bar: constants pressure-corrected, density
// at P.  First half: the constants.
__device__ __forceinline__ void omega_constants(double T, double S, double P, OmegaConst& c)
{
    static constexpr double PC_K1[5] = {-25.50, 0.1271, 0.0, -0.00308, 0.0000877};
    static constexpr double PC_K2[5] = {-15.82, -0.0219, 0.0, 0.00113, -0.0001475};
    static constexpr double PC_KB[5] = {-29.48, 0.1622, -0.0026080, -0.00284, 0.0};
    static constexpr double PC_KW[5] = {-20.02, 0.1119, -0.001409, -0.00513, 0.0000794};
    static constexpr double PC_KS[5] = {-18.03, 0.0466, 0.000316, -0.00453, 0.00009};
    static constexpr double PC_KF[5] = {-9.78, -0.0090, -0.000942, -0.00391, 0.000054};
    static constexpr double PC_CAL[5] = {-48.76, 0.5304, -0.0, -0.01176, 0.0003692};
    CarbonParams p;
    omega_salinity_terms(S, c);
    const double rho = teos10_density(T, S, P);
    const double Tk = T + 273.15;
    const Divisor rT(Tk);
    const double lT = m_log_any(Tk);
    c.conv = 1e-3 / rho;
    carbon_constants(rT, lT, S, p);
    const double Tc = Tk - 273.15;
    const double PRT = P * m_rcp(83.14472 * Tk);
    auto corrected = [&](double K, const double* a) { return K * exp(pressure_exponent(a, Tc, P, PRT)); };
    c.K1 = corrected(p.K1, PC_K1);
    c.K2 = corrected(p.K2, PC_K2);
    c.KB = corrected(p.KB, PC_KB);
    c.KW = corrected(p.KW, PC_KW);
    c.KS = corrected(p.KS, PC_KS);
    c.KF = corrected(p.KF, PC_KF);
    c.KSi = p.KSi;
    const double sS = sqrt(S);
    const double lnK_therm = -171.9065 + -0.077993 * Tk + rT.under(2839.319) + 71.595 * m_log10(Tk);
    const double lnK_sea = ((-0.77712 + 0.0028426 * Tk + rT.under(178.34)) * sS + -0.07711 * S + 0.0041249 * (S * sS));
    c.KSP = corrected(m_exp10(lnK_therm + lnK_sea), PC_CAL);
}

__device__ __forceinline__ CarbonParams omega_params(const OmegaConst& c, double DIC, double Alk, double Si)
{
    CarbonParams p;
    p.boron = c.boron;
    p.sulfate = c.sulfate;
    p.fluoride = c.fluoride;
    p.Alk = Alk * c.conv;
    p.DIC = DIC * c.conv;
    p.silicate = Si * c.conv;
    p.K1 = c.K1;
    p.K2 = c.K2;
    p.KB = c.KB;
    p.KW = c.KW;
    p.KS = c.KS;
    p.KF = c.KF;
    p.KSi = c.KSi;
    p.K0 = 0.0;
    p.Tk = 0.0;
    return p;
}

// Second half: Ω from [H+] (calcite_concentration.jl: CO3 from H, then
// Ca·CO3/KSP).
__device__ __forceinline__ double omega_from_H(const OmegaConst& c, const CarbonParams& p, double H)
{
    // DIC K1 K2 / (H (H + K1)) / (1 + K1 K2 / (H (H + K1))), over one denominator
    const double K12 = p.K1 * p.K2;
    return c.ca * p.DIC * K12 * m_rcp((H * (H + p.K1) + K12) * c.KSP);
}

// The root of the reference solve, the damped Newton from 10^-pH₀.
__device__ __forceinline__ double calcite_saturation(double DIC, double Alk, double T, double S, double Si, double P,
                                                     const obme_carbon_solver& s, int& evals)
{
    OmegaConst c;
    omega_constants(T, S, P, c);
    const CarbonParams p = omega_params(c, DIC, Alk, Si);
    const double H = root_H<true>(p, s, evals);
    return omega_from_H(c, p, H);
}

}  // namespace pisces
}  // namespace obme
