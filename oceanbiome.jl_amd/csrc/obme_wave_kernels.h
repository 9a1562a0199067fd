// obme_wave_kernels.h — the NPZD / LOBSTER step and hooks with the levels of a
// water column along the lanes of a wave, for gfx950.
//
// The column sweep (obme_npd_kernels.h) gives a lane a whole column: it needs
// a few hundred thousand columns to fill the chip, and a wave walks Nz levels
// x 3 stages in series.  Here a column takes lpc = ceil(Nz / L) lanes of one
// wave, lane r of it holding the L levels j = r L .. r L + L - 1 from the top
// (k = Nz - 1 - j), and a wave takes cpw = 64 / lpc columns side by side:
//  - the light's chlorophyll integral is a prefix sum from the top over the
//    column's lanes (DPP row shifts and row broadcasts; each step's source
//    is masked to the lane's own column, so that a NaN stays in its column);
//  - the sinking tracers' neighbours come from the neighbouring lanes, above
//    and, for the centred and WENO face values, below: those schemes need no
//    launch per stage here;
//  - the state stays in registers through the stages and through up to
//    WAVE_MAX_STEPS steps of a launch (T, S and the light at the surface are
//    given, columns are independent): each tracer is read and written once per
//    launch.  Between steps the state is rounded as a store and a load would.
// What it measured (us per call, the sweep of the columns, one launch a step |
// this): NPZD 160 x 32 FP64, one step 161 | 10.5; LOBSTER + DIC/Alk with the CO2
// flux, FP32 512 x 512 x 64, ten steps 2733 | 1755 (3.9 cycles of a SIMD per
// vector instruction: issue-bound), FP64 256 x 256 x 64, four steps 1158 | 624;
// WENO5 256 x 256 x 64, four steps 3491 (three launches a step) | 410; scaling,
// CO2 flux and sediment 240 x 180 x 50, four steps 1786 | 365.  (Where the
// sweep is the faster: wave_columns in obme_api.hip.)
//
// Loads and stores go through LDS: a workgroup moves its C = NW cpw columns
// (neighbours in the flattened (i, j) order) level by level, C values per run,
// into and out of the slots of the lanes that own the cells.
#pragma once

#include "obme_npd_kernels.h"

namespace obme {

// The model's default formulations (fm_code): LOBSTER Mondo light,
// quadratic mortality and grazing; NPZD analytical light, linear
// mortality, quadratic grazing, Q10 on.  The kernels are compiled for these
// with the choices folded in.
template <int MODEL>
constexpr int default_fm()
{
    return MODEL == OBME_LOBSTER ? (0 | (1 << 1) | (1 << 2)) : (1 | (0 << 1) | (1 << 2) | (1 << 3));
}

// Steps per launch at most: the surface PAR of every stage clock travels in
// the kernel's arguments.
constexpr int WAVE_MAX_STEPS = 16;

template <typename FT>
struct WaveArgs {
    StepArgs<FT> a;
    int nsteps;                         // steps of this launch
    int lpc, cpw;                       // lanes per column, columns per wave
    unsigned ncol;                      // Nx Ny
    FT PAR0s[WAVE_MAX_STEPS][3];        // surface PAR at the stage clocks (no surface array)
    float rk_c[2];                      // FP32: Δt (γ1 + ζ2), Δt (γ2 + ζ3)
    // FP32: log2 of the bands' (R_chl / r)^e times the chlorophyll attenuation
    // (in powers of 2), on a uniform grid times Δz / 2
    float cr, cb;
    const FastParams<FT>* fpar;         // FP64: the transitions' constants in device memory
    int uniform;                        // uniform grid, constant sinking speeds (k_top_steps, the hook)
    int scale;                          // negative scaling at the start of every stage (2: of every cell)
    int sed;                            // InstantRemineralisation sediment under the column
    int scheme;                         // the sinking face value
    // the top cell is stepped by k_top_steps (scaling with the CO2 flux): its
    // P and sinking tracers at each stage, [(step 3 + stage) 3 + q][ncol]
    const FT* toprec;
};

// Value of lane r+1 (lane 63: 0).
template <typename T>
__device__ __forceinline__ T lane_shl1(T x)
{
    return dpp<0x130, 0xf, true>(x);
}

// x with the bits of a lane mask (0 or ~0) applied.
__device__ __forceinline__ float lane_and(float x, int m)
{
    return __builtin_bit_cast(float, __builtin_bit_cast(int, x) & m);
}
__device__ __forceinline__ double lane_and(double x, int m)
{
    const unsigned long long b = __builtin_bit_cast(unsigned long long, x);
    const unsigned long long mm = ((unsigned long long)(unsigned)m << 32) | (unsigned)m;
    return __builtin_bit_cast(double, b & mm);
}

// The lane masks of the prefix sum over columns of lpc lanes: whether the
// source lane of each step belongs to the lane's own column.
// SEG = 16, 32 or 64: columns of exactly that many lanes, whose boundaries the
// row shifts and broadcasts respect by themselves; 0: any lpc, masked.
struct ColumnMasks {
    int m1, m2, m4, m8, mA, mB;
};
template <int SEG>
__device__ __forceinline__ ColumnMasks column_masks(int lane, int r)
{
    ColumnMasks c;
    c.m1 = r >= 1 ? -1 : 0;
    c.m2 = r >= 2 ? -1 : 0;
    c.m4 = r >= 4 ? -1 : 0;
    c.m8 = r >= 8 ? -1 : 0;
    // row_bcast:15 gives rows 1 and 3 the last lane of the row before
    c.mA = ((lane & 16) && r > (lane & 15)) ? -1 : 0;
    // row_bcast:31 gives rows 2 and 3 lane 31
    c.mB = ((lane & 32) && r > lane - 32) ? -1 : 0;
    // (opaque: the compiler keeps the masks in registers, one v_and with the
    // lane shift folded in per use, instead of a move and a select)
    asm volatile("" : "+v"(c.m1), "+v"(c.m2), "+v"(c.m4), "+v"(c.m8), "+v"(c.mA), "+v"(c.mB));
    return c;
}

// The value of the lane above in the column (0 for the top lane).
template <int SEG, typename T>
__device__ __forceinline__ T lane_above(T x, const ColumnMasks& c)
{
    if constexpr (SEG == 16) return dpp<0x111, 0xf, true>(x);
    else if constexpr (SEG == 64) return lane_shr1(x);
    else return lane_and(lane_shr1(x), c.m1);
}

// The sum over the column's lanes from the top to this one.
template <int SEG, typename T>
__device__ __forceinline__ T column_prefix(T x, const ColumnMasks& c)
{
    if constexpr (SEG != 0) {
        return seg_prefix<SEG>(x);
    } else {
        x = x + lane_and(dpp<0x111, 0xf, true>(x), c.m1);
        x = x + lane_and(dpp<0x112, 0xf, true>(x), c.m2);
        x = x + lane_and(dpp<0x114, 0xf, true>(x), c.m4);
        x = x + lane_and(dpp<0x118, 0xf, true>(x), c.m8);
        x = x + lane_and(dpp<0x142, 0xf, true>(x), c.mA);
        x = x + lane_and(dpp<0x143, 0xf, true>(x), c.mB);
        return x;
    }
}

// A sinking tracer's value at the bottom face of the cell of level k, for
// flow from above (w <= 0): sink_face with one quotient per weight.
template <typename FT>
__device__ __forceinline__ FT wave_weno5(FT cm2, FT cm1, FT c0, FT cp1, FT cp2)
{
    if constexpr (sizeof(FT) == 8) {
        return weno5_from_above(cm2, cm1, c0, cp1, cp2);
    } else {
        const float e = 1e-8f;
        const float q0 = fmaf(2.0f, cp2, fmaf(-7.0f, cp1, 11.0f * c0));
        const float q1 = fmaf(5.0f, c0, fmaf(2.0f, cm1, -cp1));
        const float q2 = fmaf(2.0f, c0, fmaf(5.0f, cm1, -cm2));
        const float s0 = cp2 - 2.0f * cp1 + c0, t0 = cp2 - 4.0f * cp1 + 3.0f * c0;
        const float s1 = cp1 - 2.0f * c0 + cm1, t1 = cp1 - cm1;
        const float s2 = c0 - 2.0f * cm1 + cm2, t2 = 3.0f * c0 - 4.0f * cm1 + cm2;
        const float b0 = fmaf(13.0f / 12, s0 * s0, 0.25f * (t0 * t0));
        const float b1 = fmaf(13.0f / 12, s1 * s1, 0.25f * (t1 * t1));
        const float b2 = fmaf(13.0f / 12, s2 * s2, 0.25f * (t2 * t2));
        const float tau = fabsf(b0 - b2);
        const float r0 = m_div(tau, b0 + e), r1 = m_div(tau, b1 + e), r2 = m_div(tau, b2 + e);
        const float a0 = fmaf(0.1f * r0, r0, 0.1f), a1 = fmaf(0.6f * r1, r1, 0.6f), a2 = fmaf(0.3f * r2, r2, 0.3f);
        return m_div(fmaf(a0, q0, fmaf(a1, q1, a2 * q2)), 6.0f * (a0 + a1 + a2));
    }
}
template <typename FT>
__device__ __forceinline__ FT wave_weno3(FT cm1, FT c0, FT cp1)
{
    if constexpr (sizeof(FT) == 8) {
        return weno3_from_above(cm1, c0, cp1);
    } else {
        const float e = 1e-8f;
        const float d0 = c0 - cp1, d1 = cm1 - c0;
        const float b0 = d0 * d0, b1 = d1 * d1, tau = fabsf(b0 - b1);
        const float r0 = m_div(tau, b0 + e), r1 = m_div(tau, b1 + e);
        const float a0 = fmaf((1.0f / 3) * r0, r0, 1.0f / 3), a1 = fmaf((2.0f / 3) * r1, r1, 2.0f / 3);
        return m_div(fmaf(a0, 3.0f * c0 - cp1, a1 * (c0 + cm1)), 2.0f * (a0 + a1));
    }
}

// The constants of the transitions, from the arguments (scalar registers) or
// (SHARED) from their copy in LDS, a broadcast read each.
template <bool SHARED, typename FT>
__device__ __forceinline__ const FastParams<FT>& transition_params(const WaveArgs<FT>& w, const FT* lds)
{
    if constexpr (!SHARED) return w.a.f;
    using Shared = const __attribute__((address_space(3))) FastParams<FT>*;
    unsigned p = (unsigned)(unsigned long long)(Shared)(const void*)lds;
    asm volatile("" : "+v"(p));          // a new address to the compiler: no value is kept over it
    return *(const FastParams<FT>*)(Shared)(unsigned long long)p;
}

// MODE: TILE_STEP or TILE_TENDENCY.  UNI: uniform grid with
// constant sinking speeds (FP32 folds the half cell into the attenuation).
// GEN (step): the negative scaling, the sediment and the recorded top cell,
// chosen at run time.  WIN: the centred and WENO face values.
template <int MODEL, int CARB, typename FT, int MODE, bool UNI, int L, bool GEN, bool WIN, int FM, int SEG>
__device__ __forceinline__ void column_wave(const WaveArgs<FT>& w, FT* lds)
{
    using TR = ModelTraits<MODEL, CARB>;
    constexpr int NT = TR::NT;
    constexpr int RO = TR::RO_IDX;
    constexpr int S0 = TR::SINK0, S1 = TR::SINK1, PI = TR::P_IDX;
    constexpr bool F32 = sizeof(FT) == 4;
    constexpr bool STEP = MODE == TILE_STEP;
    constexpr int OX = NT - 1;          // the O₂ tracer (CARB & 2)
    // FP32 without the scaling: the pending sum E of the Runge-Kutta
    // increments instead of the increment and the last tendency
    constexpr bool PEND = F32 && STEP && !GEN;
    // FP64, one level per lane: the transitions' 30 constants take more scalar
    // registers than there are, and kept through the loop they are moved from
    // vector lanes (180 of 1000 vector instructions of a stage); with two
    // levels the vector registers have no room for the reads
    constexpr bool SHARED = !F32 && L == 1;
    const StepArgs<FT>& a = w.a;

    const int tid = threadIdx.x, T = blockDim.x;
    const int lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lpc = SEG ? SEG : w.lpc, cpw = SEG ? 64 / (SEG ? SEG : 1) : w.cpw;
    const int C = (T >> 6) * cpw;       // columns of the workgroup
    const int Nz = a.Nz;
    const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);

    // the lane's column and levels
    const int seg = lane / lpc;
    const int r = lane - seg * lpc;
    const unsigned q = tile * (unsigned)C + (unsigned)(wv * cpw + seg);
    const bool col_ok = seg < cpw && q < w.ncol;
    const unsigned qc = col_ok ? q : 0u;
    auto has = [&](int m) -> bool { return col_ok && r * L + m < Nz; };
    const ColumnMasks cm = column_masks<SEG>(lane, r);

    // stage in: thread (column tc, level tl + u LPP) of the workgroup's tile
    const int LPP = T / C;
    const int tc = tid % C, tl = tid / C;
    const unsigned qio = tile * (unsigned)C + (unsigned)tc;
    const bool io_ok = tl < LPP && qio < w.ncol;
    const unsigned io_base = a.base0 + (io_ok ? qio % (unsigned)a.Nx + a.sx * (qio / (unsigned)a.Nx) : 0u);
    const int io_slot0 = (tc / cpw) * (64 * L) + (tc % cpw) * lpc;
    auto io_slot = [&](int k) -> int {
        const int jt = Nz - 1 - k;
        return io_slot0 + (jt % L) * 64 + jt / L;
    };
    auto reads = [&](int n) -> bool {
        if (MODE == TILE_TENDENCY && CARB != 0 && n >= 7 && MODEL == OBME_LOBSTER)
            return (CARB & 2) != 0 && n == OX && a.o2_on;
        if (MODE == TILE_TENDENCY && MODEL == OBME_NPZD && (CARB & 2) != 0 && n == OX) return false;
        return true;
    };
    const int TL = T * L;
    {
        FT stg[L][NT];
#pragma unroll
        for (int u = 0; u < L; u++) {
            const int k = tl + u * LPP;
            const bool ok = io_ok && k < Nz;
            const unsigned off = (io_base + (ok ? a.sxy * (unsigned)k : 0u)) * (unsigned)sizeof(FT);
#pragma unroll
            for (int n = 0; n < NT; n++) stg[u][n] = (ok && reads(n)) ? gload(a.tr[n], off) : FT(1);
        }
#pragma unroll
        for (int u = 0; u < L; u++) {
            const int k = tl + u * LPP;
            if (io_ok && k < Nz) {
                const int sl = io_slot(k);
#pragma unroll
                for (int n = 0; n < NT; n++)
                    if (reads(n)) lds[n * TL + sl] = stg[u][n];
            }
        }
    }
    if constexpr (SHARED) {
        constexpr int NP = (int)(sizeof(FastParams<FT>) / sizeof(FT));
        for (int n = tid; n < NP; n += T) lds[(NT + 1) * TL + n] = reinterpret_cast<const FT*>(w.fpar)[n];
    }
    __syncthreads();
    const int own = wv * (64 * L) + lane;     // the slot of level m: own + 64 m
    // a lane without a cell computes on ones and stores nothing
    FT U[NT][L];
#pragma unroll
    for (int n = 0; n < NT; n++)
#pragma unroll
        for (int m = 0; m < L; m++) U[n][m] = (has(m) && reads(n)) ? lds[n * TL + own + 64 * m] : FT(1);

    // the levels' geometry: the light left by the water alone (both bands),
    // the half cells, the face velocities of the sinking
    FT wr[L], wb[L], cw[L], dn[L], idz[L], whi[L][2], wlo[L][2];
    FT Lt[L];
    int lk[L];
#pragma unroll
    for (int m = 0; m < L; m++) {
        int k = Nz - 1 - (r * L + m);
        k = (k < 0 || !col_ok) ? 0 : k;
        lk[m] = k;
        wr[m] = a.lev[LEV_WR * Nz + k];
        wb[m] = a.lev[LEV_WB * Nz + k];
        if constexpr (UNI) {
            cw[m] = dn[m] = FT(1);
            idz[m] = a.invdz_u;
            whi[m][0] = wlo[m][0] = a.w0_u;
            whi[m][1] = wlo[m][1] = a.w1_u;
        } else {
            dn[m] = a.lev[LEV_DN * Nz + k];
            cw[m] = dn[m] + (k > 0 ? a.lev[LEV_UP * Nz + k - 1] : FT(0));
            idz[m] = a.lev[LEV_INVDZ * Nz + k];
            wlo[m][0] = a.wsink[k];
            whi[m][0] = a.wsink[k + 1];
            wlo[m][1] = a.wsink[(Nz + 1) + k];
            whi[m][1] = a.wsink[(Nz + 1) + k + 1];
        }
        Lt[m] = FT(1);
        if constexpr (MODEL == OBME_NPZD) {
            // Q10^(T/10): T is fixed
            if (fm_q10<FM>(a.f)) Lt[m] = q10_factor<FM>(a.f, U[3][m]);
        }
    }
    const bool top = r == 0;            // the column's top level is level 0 of its first lane
    FT PAR0col = FT(0);
    if (a.surface_mode == OBME_SURFACE_ARRAY) PAR0col = a.surf[qc];
    // LOBSTER's O2 exchange at the top cell
    FT o2k = FT(0), o2air = FT(0);
    if constexpr ((CARB & 2) != 0) {
        if (a.o2_on && top) {
            o2k = (FT)a.o2c[2 * qc];
            o2air = (FT)a.o2c[2 * qc + 1];
        }
    }
    // FP32 with the CO2 exchange: the top-cell Alk's residual
    float resid = 0.0f;
    if constexpr (F32 && STEP && (CARB & 1)) {
        if (a.topres && top && col_ok) resid = a.topres[w.ncol + qc];
    }
    // the sediment of the column, held by the lane of its bottom cell
    const int mb = (Nz - 1) % L;
    bool sed = false;
    double sed_u = 0.0, sed_ge = 0.0, sed_gm = 0.0;
    if constexpr (GEN) {
        sed = w.sed && col_ok && r == (Nz - 1) / L;
        if (sed) {
            sed_u = a.storage ? a.storage[qc] : 0.0;
            sed_gm = a.sed_ab2 ? a.sedG[w.ncol + qc] : 0.0;
        }
    }
    FT trec[3] = {FT(0), FT(0), FT(0)};
    auto load_toprec = [&](int n) {
        if (top && col_ok) {
#pragma unroll
            for (int c = 0; c < 3; c++) trec[c] = w.toprec[(size_t)(n * 3 + c) * w.ncol + qc];
        }
    };
    if constexpr (GEN) {
        if (w.toprec) load_toprec(0);
    }

    const double g1 = 8.0 / 15.0, g2 = 5.0 / 12.0, g3 = 3.0 / 4.0, z2 = -17.0 / 60.0, z3 = -5.0 / 12.0;
    FT X[NT][L];                                     // the stage's input
    FT D[PEND || !F32 ? 1 : NT][L], Gm[PEND ? 1 : NT][L], E[PEND ? NT : 1][L];
    FT PARv[L];

    // one stage from the input I (the first stage's is U where nothing alters
    // it); leaves the next stage's input in X, and after the last the new
    // state in U
    auto stage = [&](auto st_c, int sn, FT (&I)[NT][L]) {
        constexpr int st = decltype(st_c)::value;
        FT PAR0 = PAR0col;
        if (a.surface_mode != OBME_SURFACE_ARRAY) PAR0 = w.PAR0s[sn][st];

        if constexpr (GEN) {
            if (w.scale) {
                // ScaleNegativeTracers, where a member is negative or not
                // finite: elsewhere t = p and it is the identity up to
                // rounding; the scaled value is the new U with no increment
                unsigned members = 0;
#pragma unroll 1
                for (int g = 0; g < a.ns.n_groups; g++) members |= a.ns.mask[g];
#pragma unroll
                for (int m = 0; m < L; m++) {
                    FT x[NT];
                    bool need = !F32 && w.scale == 2;
#pragma unroll
                    for (int n = 0; n < NT; n++) {
                        x[n] = I[n][m];
                        if (members & (1u << n)) need = need || !(x[n] >= FT(0)) || __builtin_isinf(x[n]);
                    }
                    if (need) {
                        scale_negatives_cell<NT>(a.ns, x);
#pragma unroll
                        for (int n = 0; n < NT; n++)
                            if (members & (1u << n)) {
                                I[n][m] = x[n];
                                U[n][m] = x[n];
                                if constexpr (F32) D[n][m] = FT(0);
                            }
                    }
                }
            }
            if (w.toprec) {
                // the top cell as k_top_steps stepped it
                if (top) {
                    I[PI][0] = trec[0];
                    I[S0][0] = trec[1];
                    I[S1][0] = trec[2];
                }
                if (sn * 3 + st + 1 < 3 * w.nsteps) load_toprec(sn * 3 + st + 1);
            }
        }

        // ---- TwoBand PAR (Light/2band.jl:18-32)
        if constexpr (F32 && !STEP) {
            // the hook's PAR is a result: its sums go in FP64, as in k_light, and
            // the attenuations stay out of the powers' constants (64 levels of P
            // about 0.1: rms error 3.8e-7, summed as the step's 1.2e-6; a step's
            // tracers are no nearer the FP64 ones for it)
            FT pr[L], pb[L];
            double above[2][L], whole[2][L], Ir = 0.0, Ib = 0.0;
#pragma unroll
            for (int m = 0; m < L; m++) {
                chlorophyll_powers(a, I[PI][m], pr[m], pb[m]);
                above[0][m] = a.light[LIGHT_ABOVE_R * Nz + lk[m]];
                above[1][m] = a.light[LIGHT_ABOVE_B * Nz + lk[m]];
                whole[0][m] = a.light[LIGHT_WHOLE_R * Nz + lk[m]];
                whole[1][m] = a.light[LIGHT_WHOLE_B * Nz + lk[m]];
                Ir = fma(whole[0][m], (double)pr[m], Ir);
                Ib = fma(whole[1][m], (double)pb[m], Ib);
            }
            Ir = lane_above<SEG>(column_prefix<SEG>(Ir, cm), cm);
            Ib = lane_above<SEG>(column_prefix<SEG>(Ib, cm), cm);
#pragma unroll
            for (int m = 0; m < L; m++) {
                const float Jr = (float)fma(above[0][m], (double)pr[m], Ir), Jb = (float)fma(above[1][m], (double)pb[m], Ib);
                PARv[m] = PAR0 * fmaf(wr[m], m_exp2(-Jr), wb[m] * m_exp2(-Jb));
                Ir = fma(whole[0][m], (double)pr[m], Ir);
                Ib = fma(whole[1][m], (double)pb[m], Ib);
            }
        } else {
            FT pr[L], pb[L];
#pragma unroll
            for (int m = 0; m < L; m++) {
                if constexpr (F32) {
                    // the attenuation (and, on a uniform grid, the half cell) is
                    // part of the power's constant
                    const float lg = m_log2(I[PI][m]);
                    pr[m] = m_exp2(fmaf(a.er, lg, w.cr));
                    pb[m] = m_exp2(fmaf(a.eb, lg, w.cb));
                } else {
                    pow_pair<false>(I[PI][m] * a.Rr, a.er, a.eb, pr[m], pb[m]);
                }
            }
            // the integral to level j: with c = the half cells either side of the
            // levels above, Σ c p over them, plus the half cell down to j (uniform:
            // in half cells, 2 Σ p + p_j); one level per lane takes it from the
            // inclusive sum
            FT totr = FT(0), totb = FT(0);
#pragma unroll
            for (int m = 0; m < L; m++) {
                const FT cr_ = UNI ? pr[m] : cw[m] * pr[m], cb_ = UNI ? pb[m] : cw[m] * pb[m];
                totr = m == 0 ? cr_ : totr + cr_;
                totb = m == 0 ? cb_ : totb + cb_;
            }
            FT runr = column_prefix<SEG>(totr, cm), runb = column_prefix<SEG>(totb, cm);
            if constexpr (L > 1) {
                runr = lane_above<SEG>(runr, cm);
                runb = lane_above<SEG>(runb, cm);
            }
#pragma unroll
            for (int m = 0; m < L; m++) {
                FT Ir, Ib;
                if constexpr (L == 1) {
                    Ir = UNI ? fma(FT(2), runr, -pr[0]) : fma(dn[0] - cw[0], pr[0], runr);
                    Ib = UNI ? fma(FT(2), runb, -pb[0]) : fma(dn[0] - cw[0], pb[0], runb);
                } else {
                    Ir = UNI ? fma(FT(2), runr, pr[m]) : fma(dn[m], pr[m], runr);
                    Ib = UNI ? fma(FT(2), runb, pb[m]) : fma(dn[m], pb[m], runb);
                    runr = UNI ? runr + pr[m] : fma(cw[m], pr[m], runr);
                    runb = UNI ? runb + pb[m] : fma(cw[m], pb[m], runb);
                }
                if constexpr (F32) {
                    PARv[m] = PAR0 * fmaf(wr[m], m_exp2(-Ir), wb[m] * m_exp2(-Ib));
                } else {
                    const FT h = UNI ? a.dz_u * FT(0.5) : FT(1);
                    PARv[m] = PAR0 * (wr[m] * m_exp(-(a.xr * h) * Ir) + wb[m] * m_exp(-(a.xb * h) * Ib));
                }
            }
        }

        // ---- sinking: the values above (and for WIN below) of the two tracers
        FT fx[2][L], fxu[2][L];         // the face value below each cell, and of the face above
        if constexpr (WIN) {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const int n = s == 0 ? S0 : S1;
                FT c[L + 4];            // levels j - 2 .. j + L + 1 of the lane, from above to below
#pragma unroll
                for (int m = 0; m < L; m++) c[m + 2] = I[n][m];
                c[1] = lane_shr1(I[n][L - 1]);
                c[0] = L >= 2 ? lane_shr1(I[n][L >= 2 ? L - 2 : 0]) : lane_shr1(c[1]);
                c[L + 2] = lane_shl1(I[n][0]);
                c[L + 3] = L >= 2 ? lane_shl1(I[n][L >= 2 ? 1 : 0]) : lane_shl1(c[L + 2]);
#pragma unroll
                for (int m = 0; m < L; m++) {
                    const int k = lk[m];
                    const FT cp2 = c[m], cp1 = c[m + 1], c0 = c[m + 2], cm1 = c[m + 3], cm2 = c[m + 4];
                    FT f = c0;
                    if (w.scheme == OBME_CENTERED2) {
                        f = k > 0 ? (cm1 + c0) / FT(2) : c0;
                    } else {
                        if (k >= 3 && k <= Nz - 3) f = wave_weno5(cm2, cm1, c0, cp1, cp2);
                        else if (k > 1 && (k == 2 || k == Nz - 2) && k < Nz - 1) f = wave_weno3(cm1, c0, cp1);
                    }
                    fx[s][m] = f;
                }
                const FT fu = lane_above<SEG>(fx[s][L - 1], cm);
#pragma unroll
                for (int m = 0; m < L; m++) fxu[s][m] = m == 0 ? fu : fx[s][m > 0 ? m - 1 : 0];
            }
        } else {
#pragma unroll
            for (int s = 0; s < 2; s++) {
                const int n = s == 0 ? S0 : S1;
                const FT xu = lane_above<SEG>(I[n][L - 1], cm);
#pragma unroll
                for (int m = 0; m < L; m++) {
                    fx[s][m] = I[n][m];
                    fxu[s][m] = m == 0 ? xu : I[n][m > 0 ? m - 1 : 0];
                }
            }
        }

        // ---- the sediment at the bottom cell (as in column_lane)
        FT cpl = FT(0);
        if constexpr (GEN) {
            if (sed) {
                FT x0 = I[S0][0], x1 = I[S1][0];
#pragma unroll
                for (int m = 1; m < L; m++)
                    if (m == mb) {
                        x0 = I[S0][m];
                        x1 = I[S1][m];
                    }
                const bool second = F32 && sediment_second<CARB>(w.scale != 0, st);
                const FT f = sediment_flux(a, x0, x1, second);
                const FT e = sediment_burial(a, f);
                cpl = ((FT(1) - e) * f) / a.sed_dz0;
                const double ge = (double)(e * f);
                const bool init = a.sed_init && sn == 0;
                if (st == 0) {
                    if (!init) sed_u = sediment_step(a, 0, sed_u, ge, a.sed_ab2 && sn == 0, sed_gm);
                } else {
                    if (st == 1 && init) sed_u = sediment_step(a, 0, sed_u, ge, 0, 0.0);
                    sed_u = sediment_step(a, st, sed_u, ge, 0, 0.0);
                }
                sed_ge = ge;
            }
        }

#pragma unroll
        for (int m = 0; m < L; m++) {
            // ---- the transitions
            const FastParams<FT>& f = transition_params<SHARED>(w, lds + (NT + 1) * TL);
            FT Gv[NT];
            {
                FT v[NT];
#pragma unroll
                for (int n = 0; n < NT; n++) v[n] = (CARB != 0 && n >= 7) ? FT(0) : I[n][m];
                if constexpr (MODEL == OBME_NPZD) {
                    npzd_fast<FM>(f, v[0], v[1], v[2], v[4], PARv[m], Lt[m], Gv[0], Gv[1], Gv[2], Gv[4],
                                  (CARB & 2) ? &Gv[OX] : nullptr);
                    Gv[3] = FT(0);
                } else if constexpr (F32 && GEN) {
                    if (w.sed) lobster_sediment<CARB, FM>(a.fs, v, PARv[m], Gv);
                    else lobster_fast<CARB, FM>(f, v, PARv[m], Gv);
                } else {
                    lobster_fast<CARB, FM>(f, v, PARv[m], Gv);
                }
            }
            // ---- minus the drift flux divergence
            if constexpr (F32 && UNI && !WIN) {
                Gv[S0] = fmaf(-a.wi0, fxu[0][m] - fx[0][m], Gv[S0]);
                Gv[S1] = fmaf(-a.wi1, fxu[1][m] - fx[1][m], Gv[S1]);
            } else if (F32 && !STEP && !WIN && w.uniform) {
                // (the hook has one kernel for every grid: with constant speeds
                // the difference first, which the flux of either face would
                // round away)
                Gv[S0] = fma((FT)-a.wi0, fxu[0][m] - fx[0][m], Gv[S0]);
                Gv[S1] = fma((FT)-a.wi1, fxu[1][m] - fx[1][m], Gv[S1]);
            } else {
                // (no flux through the surface)
                const FT h0 = (top && m == 0) ? FT(0) : whi[m][0] * fxu[0][m];
                const FT h1 = (top && m == 0) ? FT(0) : whi[m][1] * fxu[1][m];
                Gv[S0] = Gv[S0] - (h0 - wlo[m][0] * fx[0][m]) * idz[m];
                Gv[S1] = Gv[S1] - (h1 - wlo[m][1] * fx[1][m]) * idz[m];
            }
            if constexpr ((CARB & 2) != 0) {
                if (a.o2_on && top && m == 0) Gv[OX] = Gv[OX] - o2k * (I[OX][0] - o2air);
            }
            if constexpr (GEN) {
                if (sed && m == mb) {
#pragma unroll
                    for (int n = 0; n < NT; n++)
                        if (n == a.sed_recv) Gv[n] = Gv[n] + cpl;
                }
            }
            if constexpr (MODE == TILE_TENDENCY) {
#pragma unroll
                for (int n = 0; n < NT; n++) U[n][m] = Gv[n];
            } else {
                if constexpr (CARB & 1) {
                    // the surface kernel's record: DIC transition without the flux, Alk at the stage start
                    if (m == 0 && a.co2_on && top && col_ok) {
                        FT* rec = a.srec + (size_t)(sn * SURF_REC) * w.ncol + qc;
                        rec[(size_t)st * w.ncol] = Gv[7];
                        rec[(size_t)(3 + st) * w.ncol] = (st == 0 && F32) ? I[8][0] + (FT)resid : I[8][0];
                    }
                }
                // ---- the substep
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    if (n == RO) continue;
                    if constexpr (PEND) {
                        // U + Δt (γ1 G1), U + Δt ((γ1 + ζ2) G1 + γ2 G2), and the
                        // step's sum: E carries the part of the earlier stages
                        const float R0 = ((CARB & 1) && n == 8 && m == 0) ? resid : 0.0f;
                        if constexpr (st == 0) {
                            const bool res = (CARB & 1) && n == 8 && m == 0;
                            X[n][m] = res ? U[n][m] + fmaf(a.rk_a[0], Gv[n], R0) : fmaf(a.rk_a[0], Gv[n], U[n][m]);
                            E[n][m] = res ? fmaf(w.rk_c[0], Gv[n], R0) : w.rk_c[0] * Gv[n];
                        } else if constexpr (st == 1) {
                            X[n][m] = U[n][m] + fmaf(a.rk_a[1], Gv[n], E[n][m]);
                            E[n][m] = fmaf(w.rk_c[1], Gv[n], E[n][m]);
                        } else {
                            E[n][m] = fmaf(a.rk_a[2], Gv[n], E[n][m]);
                            if ((CARB & 1) && n == 8 && m == 0) {
                                // U + E = s + e exactly (TwoSum): s stored, e to the next step
                                const float u = U[n][m], d = E[n][m], sum = u + d, dv = sum - u;
                                if (a.topres && top) resid = (u - (sum - dv)) + (d - dv);
                                U[n][m] = sum;
                            } else {
                                U[n][m] = U[n][m] + E[n][m];
                            }
                        }
                    } else if constexpr (F32) {
                        if (st == 0) D[n][m] = fmaf(a.rk_a[0], Gv[n], D[n][m]);
                        else D[n][m] = fmaf(a.rk_a[st], Gv[n], fmaf(a.rk_b[st], Gm[n][m], D[n][m]));
                        Gm[n][m] = Gv[n];
                        if constexpr (st < 2) {
                            X[n][m] = U[n][m] + D[n][m];
                        } else if ((CARB & 1) && n == 8 && m == 0) {
                            const float u = U[n][m], d = D[n][m], sum = u + d, dv = sum - u;
                            if (a.topres && top) resid = (u - (sum - dv)) + (d - dv);
                            U[n][m] = sum;
                        } else {
                            U[n][m] = U[n][m] + D[n][m];
                        }
                    } else {
                        const double gs = (st == 1) ? g2 : g3;
                        const double zs = (st == 1) ? z2 : z3;
                        U[n][m] += (st == 0) ? (a.dtf * g1) * Gv[n] : a.dtf * (gs * Gv[n] + zs * Gm[n][m]);
                        Gm[n][m] = Gv[n];
                    }
                }
            }
        }
    };

    if constexpr (!STEP) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int m = 0; m < L; m++) X[n][m] = U[n][m];
        stage(std::integral_constant<int, 0>{}, 0, X);
    } else {
#pragma unroll 1
        for (int sn = 0; sn < w.nsteps; sn++) {
            if constexpr (!PEND) {
#pragma unroll
                for (int n = 0; n < NT; n++)
#pragma unroll
                    for (int m = 0; m < L; m++) {
                        if constexpr (F32) D[n][m] = FT(0);
                        Gm[n][m] = FT(0);
                    }
                // the top-cell Alk includes its residual from the first stage on
                if constexpr (F32 && (CARB & 1)) D[8][0] = resid;
            }
            // FP64 (and the scaling) alter the state in place
            stage(std::integral_constant<int, 0>{}, sn, U);
            if constexpr (F32) {
                stage(std::integral_constant<int, 1>{}, sn, X);
                stage(std::integral_constant<int, 2>{}, sn, X);
            } else {
                stage(std::integral_constant<int, 1>{}, sn, U);
                stage(std::integral_constant<int, 2>{}, sn, U);
            }
        }
        if constexpr (F32 && (CARB & 1)) {
            if (a.topres && top && col_ok) a.topres[w.ncol + qc] = resid;
        }
        if constexpr (GEN) {
            if (sed) {
                FT x0 = U[S0][0], x1 = U[S1][0];
#pragma unroll
                for (int m = 1; m < L; m++)
                    if (m == mb) {
                        x0 = U[S0][m];
                        x1 = U[S1][m];
                    }
                const FT f = sediment_flux(a, x0, x1, false);
                if (a.storage) a.storage[qc] = sed_u;
                a.sedG[qc] = (double)(sediment_burial(a, f) * f);
                a.sedG[w.ncol + qc] = sed_ge;
            }
        }
    }

    // stage out: each lane into its own slots, then runs of C values per level
    __syncthreads();
#pragma unroll
    for (int m = 0; m < L; m++) {
#pragma unroll
        for (int n = 0; n < NT; n++)
            if (n != RO) lds[n * TL + own + 64 * m] = U[n][m];
        if constexpr (!STEP) lds[NT * TL + own + 64 * m] = PARv[m];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < L; u++) {
        const int k = tl + u * LPP;
        if (!(io_ok && k < Nz)) continue;
        const unsigned off = (io_base + a.sxy * (unsigned)k) * (unsigned)sizeof(FT);
        const int sl = io_slot(k);
        const bool ktop = k == Nz - 1;
        if constexpr (MODE == TILE_TENDENCY) {
            FT g0[NT];
#pragma unroll
            for (int n = 0; n < NT; n++)
                if (n != RO) g0[n] = gload(a.G[n], off);
#pragma unroll
            for (int n = 0; n < NT; n++)
                if (n != RO) gstore(a.G[n], off, g0[n] + lds[n * TL + sl]);
            if (a.PAR) gstore(a.PAR, off, lds[NT * TL + sl]);
        } else {
            if (GEN && w.toprec && ktop) continue;      // k_top_steps wrote it
#pragma unroll
            for (int n = 0; n < NT; n++) {
                if (n == RO) continue;
                if ((CARB & 1) && n == 7 && ktop && a.co2_on) continue;   // the surface kernel writes it
                gstore(a.tr[n], off, lds[n * TL + sl]);
            }
        }
    }
}

// The top cell of every column through the steps of a launch, with the
// negative scaling and the CO2 flux: the scaled top-cell DIC feeds back into
// the cell's other tracers, so the flux is solved between the stages.  One
// thread per column; nothing flows into the top cell from below, so it is
// stepped ahead of the column, and column_wave takes its P and its sinking
// tracers from the record.  The solve (FP64 Newton, latency-bound) thereby
// stays out of the column's kernel, where one lane per column would run it
// for the whole wave.
template <int CARB, typename FT, int FM>
__device__ __forceinline__ void top_steps(const WaveArgs<FT>& w, FT* rec)
{
    using TR = ModelTraits<OBME_LOBSTER, CARB>;
    constexpr int NT = TR::NT, S0 = TR::SINK0, S1 = TR::SINK1, PI = TR::P_IDX;
    constexpr bool F32 = sizeof(FT) == 4;
    const StepArgs<FT>& a = w.a;
    const unsigned q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= w.ncol) return;
    const int Nz = a.Nz, k = Nz - 1;
    const unsigned cell = a.base0 + q % (unsigned)a.Nx + a.sx * (q / (unsigned)a.Nx) + a.sxy * (unsigned)k;
    FT U[NT], D[NT], Gm[NT], X[NT];
#pragma unroll
    for (int n = 0; n < NT; n++) U[n] = a.tr[n][cell];
    const FT wr = a.lev[LEV_WR * Nz + k], wb = a.lev[LEV_WB * Nz + k];
    const FT dn = a.lev[LEV_DN * Nz + k], idz = a.lev[LEV_INVDZ * Nz + k];
    const FT wlo0 = a.wsink[k], wlo1 = a.wsink[(Nz + 1) + k];
    const double T = a.T3 ? (double)a.T3[cell] : (a.Tprof ? a.Tprof[k] : a.Tconst);
    const double S = a.S3 ? (double)a.S3[cell] : (a.Sprof ? a.Sprof[k] : a.Sconst);
    SurfaceCarbon sc;
    surface_carbon_setup(a.co2, T, S, a.co2.wind_speed, sc);
    double H = a.Hprev ? a.Hprev[q] : 0.0;
    FT o2k = FT(0), o2air = FT(0);
    if constexpr ((CARB & 2) != 0) {
        if (a.o2_on) {
            o2k = (FT)a.o2c[2 * q];
            o2air = (FT)a.o2c[2 * q + 1];
        }
    }
    unsigned members = 0;
#pragma unroll 1
    for (int g = 0; g < a.ns.n_groups; g++) members |= a.ns.mask[g];
    const double g1 = 8.0 / 15.0, g2 = 5.0 / 12.0, g3 = 3.0 / 4.0, z2 = -17.0 / 60.0, z3 = -5.0 / 12.0;
#pragma unroll 1
    for (int sn = 0; sn < w.nsteps; sn++) {
#pragma unroll
        for (int n = 0; n < NT; n++) {
            X[n] = U[n];
            D[n] = Gm[n] = FT(0);
        }
#pragma unroll 1
        for (int st = 0; st < 3; st++) {
            FT PAR0 = a.surface_mode == OBME_SURFACE_ARRAY ? a.surf[q] : w.PAR0s[sn][st];
            bool need = !F32 && w.scale == 2;
            FT x[NT];
#pragma unroll
            for (int n = 0; n < NT; n++) {
                x[n] = X[n];
                if (members & (1u << n)) need = need || !(x[n] >= FT(0)) || __builtin_isinf(x[n]);
            }
            if (need) {
                scale_negatives_cell<NT>(a.ns, x);
#pragma unroll
                for (int n = 0; n < NT; n++)
                    if (members & (1u << n)) {
                        X[n] = U[n] = x[n];
                        D[n] = FT(0);
                    }
            }
            const size_t at = (size_t)((sn * 3 + st) * 3) * w.ncol + q;
            rec[at] = X[PI];
            rec[at + w.ncol] = X[S0];
            rec[at + 2 * (size_t)w.ncol] = X[S1];
            int ev = 0;
            const double F = surface_flux_warm(sc, a.solver, (double)X[7], (double)X[8], a.co2.air_concentration, H, ev,
                                               F32 ? FP32_NEWTON_TOL : FP64_NEWTON_TOL);
            FT pr, pb, PAR;
            if constexpr (F32) {
                const float lg = m_log2(X[PI]);
                pr = m_exp2(fmaf(a.er, lg, w.cr));
                pb = m_exp2(fmaf(a.eb, lg, w.cb));
                const float h = w.uniform ? 1.0f : (float)dn;   // (a uniform grid's half cell is in cr, cb)
                PAR = PAR0 * fmaf(wr, m_exp2(-(h * pr)), wb * m_exp2(-(h * pb)));
            } else {
                pow_pair<false>(X[PI] * a.Rr, a.er, a.eb, pr, pb);
                PAR = PAR0 * (wr * m_exp(-a.xr * (dn * pr)) + wb * m_exp(-a.xb * (dn * pb)));
            }
            FT Gv[NT], v[NT];
#pragma unroll
            for (int n = 0; n < NT; n++) v[n] = n >= 7 ? FT(0) : X[n];
            if constexpr (F32) {
                if (w.sed) lobster_sediment<CARB, FM>(a.fs, v, PAR, Gv);
                else lobster_fast<CARB, FM>(a.f, v, PAR, Gv);
            } else {
                lobster_fast<CARB, FM>(a.f, v, PAR, Gv);
            }
            if (F32 && w.uniform) {
                Gv[S0] = fma((FT)-a.wi0, FT(0) - X[S0], Gv[S0]);
                Gv[S1] = fma((FT)-a.wi1, FT(0) - X[S1], Gv[S1]);
            } else {
                Gv[S0] = Gv[S0] - (FT(0) - wlo0 * X[S0]) * idz;
                Gv[S1] = Gv[S1] - (FT(0) - wlo1 * X[S1]) * idz;
            }
            Gv[7] = Gv[7] - (FT)F * a.invdz_top;
            if constexpr ((CARB & 2) != 0) {
                if (a.o2_on) Gv[NT - 1] = Gv[NT - 1] - o2k * (X[NT - 1] - o2air);
            }
#pragma unroll
            for (int n = 0; n < NT; n++) {
                if constexpr (F32) {
                    D[n] = fmaf(a.rk_a[st], Gv[n], fmaf(a.rk_b[st], Gm[n], D[n]));
                    X[n] = U[n] + D[n];
                } else {
                    const double gs = (st == 1) ? g2 : g3, zs = (st == 1) ? z2 : z3;
                    U[n] += (st == 0) ? (a.dtf * g1) * Gv[n] : a.dtf * (gs * Gv[n] + zs * Gm[n]);
                    X[n] = U[n];
                }
                Gm[n] = Gv[n];
            }
        }
#pragma unroll
        for (int n = 0; n < NT; n++) U[n] = X[n];
    }
#pragma unroll
    for (int n = 0; n < NT; n++) a.tr[n][cell] = U[n];
    if (a.Hprev) a.Hprev[q] = H;
}

// The column sweep's workgroups: at most eight waves.
constexpr int SWEEP_MAX_THREADS = 512;
template <typename FT>
using LaneKernel = void (*)(StepArgs<FT>);
// The sweep kernel of a launch (obme_sweep.hip, one translation unit per model).
template <int MODEL, int CARB, typename FT>
LaneKernel<FT> lane_kernel(int mode, bool uniform, bool whole, bool forms, int scheme, int extra);

template <typename FT>
using WaveKernel = void (*)(WaveArgs<FT>);

// The levels per lane that the kernels are compiled for (0: none left).
template <typename FT>
constexpr int wave_levels(int i)
{
    constexpr int f32[] = {1, 2, 4, 0}, f64[] = {1, 2, 0, 0};
    return sizeof(FT) == 4 ? f32[i] : f64[i];
}
// Threads of a workgroup at most.
constexpr int WAVE_MAX_THREADS = 512;

// The kernel of a model (obme_wave.hip, one translation unit per model); null
// where none is compiled.
template <int MODEL, int CARB, typename FT>
WaveKernel<FT> wave_kernel(int mode, bool uniform, int levels, int lpc, bool general, bool win);
template <int CARB, typename FT>
void (*top_kernel())(WaveArgs<FT>, FT*);

}  // namespace obme
