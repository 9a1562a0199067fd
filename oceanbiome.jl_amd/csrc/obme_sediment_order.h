// obme_sediment_order.h — the FP32 transitions of a model with a sediment.
//
// The sediment's storage is an FP64 sum of the FP32 flux through the bottom
// face.  A last bit of a particle tracer that rounds the other way is 6e-8
// of the flux, far above what the storage itself resolves, so a handle with a
// sediment keeps one fixed order of operations for its FP32 transitions:
// these.  (The transitions of obme_device.h round in another order, in 10
// operations less per cell and stage.)
#pragma once

namespace obme {

// Derived constants, formed once on the host in FP64 and rounded.
struct SedimentParams {
    float nPSI2;       // -psi * log2(e): exp(-psi NH4) = 2^(nPSI2 NH4)
    float kNO3, kNH4, kPAR, kPAR2;
    float mu0, mu0h;   // mu0, mu0/2 (LOBSTER's (L_NO3 + L_NH4)/2)
    float pref, prefc; // pref, 1 - pref
    float kG, kG2, g;
    float mP, mZ, muZ;
    float one_m_gamma, axg;
    float nitrif;
    float pinw_z;      // aZ_exc * muZ
    float one_m_aPs, aPs;
    float s_rem, b_rem, d_rem, a_rem, one_m_arem;
    float ponw_mu;     // (1 - alpha_x) gamma
    float ponw_z;      // (1 - aZ_exc) muZ
    float one_m_aZass, aZass;
    float ss, one_m_ss;
    float ppc;         // (1 + rho (1-gamma) - alpha_x gamma) R
    float R, Rd, rhoR2, rhoR4;  // R, Rd, 2 rho R, 4 rho R
    float rem, small_frac, uptake_N;  // Detritus rate, fraction, (1 - alpha_x gamma)
    float oRp, oRpn;   // Oxygen(): Rp, Rp - Rn (set from obme_oxygen)
    int light_form, mort_form, graz_form;
};

inline SedimentParams make_sediment_params(const obme_npd_params& p)
{
    SedimentParams f;
    f.oRp = f.oRpn = 0.0f;
    const double LOG2E = 1.4426950408889634;
    f.nPSI2 = (float)(-p.nitrate_ammonia_inhibition * LOG2E);
    f.kNO3 = (float)p.nitrate_half_saturation;
    f.kNH4 = (float)p.ammonia_half_saturation;
    f.kPAR = (float)p.light_half_saturation;
    f.kPAR2 = (float)(p.light_half_saturation * p.light_half_saturation);
    f.mu0 = (float)p.phytoplankton_maximum_growth_rate;
    f.mu0h = (float)(p.phytoplankton_maximum_growth_rate / 2);
    f.pref = (float)p.preference_for_phytoplankton;
    f.prefc = (float)(1 - p.preference_for_phytoplankton);
    f.kG = (float)p.grazing_half_saturation;
    f.kG2 = (float)(p.grazing_half_saturation * p.grazing_half_saturation);
    f.g = (float)p.maximum_grazing_rate;
    f.mP = (float)p.phytoplankton_mortality_rate;
    f.mZ = (float)p.zooplankton_mortality_rate;
    f.muZ = (float)p.zooplankton_excretion_rate;
    f.one_m_gamma = (float)(1 - p.phytoplankton_exudation_fraction);
    f.axg = (float)(p.ammonia_fraction_of_exudate * p.phytoplankton_exudation_fraction);
    f.nitrif = (float)p.nitrification_rate;
    f.pinw_z = (float)(p.excretion_inorganic_fraction * p.zooplankton_excretion_rate);
    f.one_m_aPs = (float)(1 - p.phytoplankton_solid_waste_fraction);
    f.aPs = (float)p.phytoplankton_solid_waste_fraction;
    f.s_rem = (float)p.small_remineralisation_rate;
    f.b_rem = (float)p.large_remineralisation_rate;
    f.d_rem = (float)p.dissolved_remineralisation_rate;
    f.a_rem = (float)p.remineralisation_inorganic_fraction;
    f.one_m_arem = (float)(1 - p.remineralisation_inorganic_fraction);
    f.ponw_mu = (float)((1 - p.ammonia_fraction_of_exudate) * p.phytoplankton_exudation_fraction);
    f.ponw_z = (float)((1 - p.excretion_inorganic_fraction) * p.zooplankton_excretion_rate);
    f.one_m_aZass = (float)(1 - p.zooplankton_assimilation_fraction);
    f.aZass = (float)p.zooplankton_assimilation_fraction;
    f.ss = (float)p.small_solid_waste_fraction;
    f.one_m_ss = (float)(1 - p.small_solid_waste_fraction);
    f.ppc = (float)((1 + p.carbon_calcite_ratio * (1 - p.phytoplankton_exudation_fraction)
                     - p.ammonia_fraction_of_exudate * p.phytoplankton_exudation_fraction) * p.redfield_ratio);
    f.R = (float)p.redfield_ratio;
    f.Rd = (float)p.detritus_redfield_ratio;
    f.rhoR2 = (float)(2 * p.carbon_calcite_ratio * p.redfield_ratio);
    f.rhoR4 = (float)(4 * p.carbon_calcite_ratio * p.redfield_ratio);
    f.rem = (float)p.remineralisation_rate;
    f.small_frac = (float)p.small_particle_fraction;
    f.uptake_N = (float)(1 - p.ammonia_fraction_of_exudate * p.phytoplankton_exudation_fraction);
    f.light_form = p.light_limitation;
    f.mort_form = p.phytoplankton_mortality_formulation;
    f.graz_form = p.grazing_concentration_formulation;
    return f;
}

__device__ __forceinline__ float frcp(float x) { return __builtin_amdgcn_rcpf(x); }
// max(0, x) that keeps a NaN x (Julia's max propagates NaN)
__device__ __forceinline__ float fmax0(float x) { return (x < 0.0f) ? 0.0f : x; }
constexpr float F_TINY = 1.17549435e-38f;  // smallest normal float

// Grazing of the PhytoZoo plankton (plankton.jl:118-135, :352-397) in FP32,
// reformulated over n = pref P^2 + (1-pref) sPOM^2 and d = pref P + (1-pref) sPOM:
// the preference-weighted food is n/d, so the total grazing is
// g Z n^2 / (n^2 + kG^2 d^2) (quadratic) or g Z n / (n + kG d) (linear), and
// the grazed fractions of the total are pref P^2 / n and (1-pref) sPOM^2 / n.
// With fr = total / n = g Z n / (n^2 + kG^2 d^2) (or g Z / (n + kG d)) the
// three terms are fr n, fr pref P^2 and fr (1-pref) sPOM^2: one reciprocal
// instead of the reference's three divisions; F_TINY keeps 0/0 away as the
// reference's eps(food) does.
struct SGrazing {
    float total, onP, onSmall;
};
template <int FM> __device__ __forceinline__ int fm_light(const SedimentParams& f) { if constexpr (FM < 0) return f.light_form; else return FM & 1; }
template <int FM> __device__ __forceinline__ int fm_mort(const SedimentParams& f) { if constexpr (FM < 0) return f.mort_form; else return (FM >> 1) & 1; }
template <int FM> __device__ __forceinline__ int fm_graz(const SedimentParams& f) { if constexpr (FM < 0) return f.graz_form; else return (FM >> 2) & 1; }
template <int FM = -1>
__device__ __forceinline__ SGrazing sediment_grazing(const SedimentParams& f, float P, float Z, float sPOM)
{
    const float pP = f.pref * P;
    const float cS = f.prefc * sPOM;
    const float sS = cS * sPOM;
    const float n = fmaf(pP, P, sS);
    const float d = pP + cS;
    const float gZ = f.g * Z;
    float fr;
    if (fm_graz<FM>(f) == OBME_LINEAR) fr = gZ * frcp(fmaf(f.kG, d, n) + F_TINY);
    else {
        const float kd = f.kG * d;
        fr = (gZ * n) * frcp(fmaf(kd, kd, n * n) + F_TINY);
    }
    SGrazing G;
    G.total = fr * n;
    G.onP = fr * (pP * P);
    G.onSmall = fr * sS;
    return G;
}

template <int FM = -1>
__device__ __forceinline__ float sediment_light(const SedimentParams& f, float PAR)
{
    if (fm_light<FM>(f) == OBME_LIGHT_MONDO) return PAR * frcp(f.kPAR + PAR);
    return PAR * __builtin_amdgcn_rsqf(fmaf(PAR, PAR, f.kPAR2));
}

// LOBSTER (+ CarbonateSystem) transitions in FP32; v/out in tracer order.
// The nitrate and ammonia uptakes are mu0/2 L_PAR P times their own
// limitation (the reference forms them as fractions of the total
// production, plankton.jl:223-261, which is the same product).
template <int CARB, int FM = -1>
__device__ __forceinline__ void lobster_sediment(const SedimentParams& f, const float* v, float PAR, float* out)
{
    const float NO3 = v[0], NH4 = v[1], P = v[2], Z = v[3], sPOM = v[4], bPOM = v[5], DOM = v[6];
    const float a = NO3 + f.kNO3, b = f.kNH4 + NH4;
    float up_NO3, muA;
    if (fm_light<FM>(f) == OBME_LIGHT_MONDO) {
        // one reciprocal for both Monod terms and the light limitation
        // PAR / (kPAR + PAR): with c = kPAR + PAR > 0, 1/(a c) = b r and
        // 1/(b c) = a r for r = 1/(a b c), and max(0, x / c) = max(0, x) / c
        const float r = frcp((a * b) * (f.kPAR + PAR));
        const float nlc = NO3 * __builtin_amdgcn_exp2f(f.nPSI2 * NH4) * (b * r);
        const float alc = fmax0(NH4 * (a * r));
        const float muLPc = f.mu0h * PAR * P;
        up_NO3 = muLPc * nlc;
        muA = muLPc * alc;
    } else {
        // one reciprocal for both Monod terms
        const float rab = frcp(a * b);
        const float nl = NO3 * __builtin_amdgcn_exp2f(f.nPSI2 * NH4) * (b * rab);
        const float al = fmax0(NH4 * (a * rab));
        const float muLP = f.mu0h * sediment_light<FM>(f, PAR) * P;
        up_NO3 = muLP * nl;
        muA = muLP * al;
    }
    const float muP = up_NO3 + muA;
    const SGrazing G = sediment_grazing<FM>(f, P, Z, sPOM);
    const float nuP = (fm_mort<FM>(f) == OBME_LINEAR) ? f.mP * P : f.mP * P * P;
    const float nit = f.nitrif * NH4;
    const float up_NH4 = fmaf(-f.axg, muP, muA);
    const float pinw = fmaf(f.pinw_z, Z, f.one_m_aPs * nuP);
    const float sb = fmaf(f.s_rem, sPOM, f.b_rem * bPOM);
    const float dinw = fmaf(f.a_rem, sb, f.d_rem * DOM);
    const float ponw = fmaf(f.ponw_mu, muP, f.ponw_z * Z);
    const float Z2 = Z * Z;
    const float solid = fmaf(f.one_m_aZass, G.total, fmaf(f.aPs, nuP, f.mZ * Z2));
    const float dNO3 = nit - up_NO3;
    const float dNH4 = pinw + dinw - nit - up_NH4;
    out[0] = dNO3;
    out[1] = dNH4;
    out[2] = fmaf(f.one_m_gamma, muP, -G.onP) - nuP;
    out[3] = fmaf(f.aZass, G.total, -f.mZ * Z2) - f.muZ * Z;
    out[4] = fmaf(f.ss, solid, -G.onSmall) - f.s_rem * sPOM;
    out[5] = fmaf(f.one_m_ss, solid, -f.b_rem * bPOM);
    out[6] = fmaf(f.one_m_arem, sb, ponw) - f.d_rem * DOM;
    if constexpr ((CARB & 1) != 0) {
        // calcite dissolution (G_P + ν) ρ R (plankton.jl:429-441), uptake 2 ρ μP R (:443-450)
        const float cdis2 = (G.onP + nuP) * f.rhoR2;            // 2 cdis
        out[7] = fmaf(-f.ppc, muP, fmaf(f.R, pinw, fmaf(f.Rd, dinw, 0.5f * cdis2)));
        out[8] = fmaf(0.9375f, dNH4, -1.0625f * dNO3) - f.rhoR4 * muP + cdis2;
    }
    if constexpr ((CARB & 2) != 0) {
        // Rp (μP - nitrification) - (Rp - Rn) G_NH4 (oxygen.jl:21-31)
        out[(CARB & 1) ? 9 : 7] = fmaf(f.oRp, muP - nit, -f.oRpn * dNH4);
    }
}

// NPZD transitions in FP32 (N, P, Z, D); Lt = Q10^(T/10); dO2 as in npzd_tendencies.
template <int FM = -1>
__device__ __forceinline__ void npzd_sediment(const SedimentParams& f, float N, float P, float Z, float D, float PAR,
                                          float Lt, float& dN, float& dP, float& dZ, float& dD,
                                          float* dO2 = nullptr)
{
    const float muP = f.mu0 * sediment_light<FM>(f, PAR) * (N * frcp(N + f.kNO3)) * Lt * P;
    const float sPOM = D * f.small_frac;
    const SGrazing G = sediment_grazing<FM>(f, P, Z, sPOM);
    float nuP = (fm_mort<FM>(f) == OBME_LINEAR) ? f.mP * P : f.mP * P * P;
    const float Z2 = Z * Z;
    dP = fmaf(f.one_m_gamma, muP, -G.onP) - nuP;
    dZ = fmaf(f.aZass, G.total, -f.mZ * Z2) - f.muZ * Z;
    const float pinw = fmaf(f.pinw_z, Z, f.one_m_aPs * nuP);
    dN = fmaf(D, f.rem, pinw) - muP * f.uptake_N;
    const float ponw = fmaf(f.ponw_mu, muP, f.ponw_z * Z);
    const float solid = fmaf(f.one_m_aZass, G.total, fmaf(f.aPs, nuP, f.mZ * Z2));
    dD = ponw + solid - G.onSmall - f.rem * D;
    if (dO2) *dO2 = fmaf(f.oRp, muP, -f.oRpn * pinw);
}

}  // namespace obme
