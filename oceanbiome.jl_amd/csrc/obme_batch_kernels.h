// obme_batch_kernels.h — the batched ensemble of independent NPZD water
// columns: ragged depths, per-column parameters and surface PAR, every
// column advanced many RK3 steps with its state held in registers.
//
// Reference semantics: one NPZD column per entry, the column stepper of the
// fused sweep (TwoBand PAR, Light/2band.jl:1-33; upwind sinking with an open
// bottom, Utils/sinking_velocity_fields.jl:10-35; NPZD transitions,
// NutrientsPlanktonDetritus/*.jl; the RK3 substep, BoxModel/timesteppers.jl:79-92),
// with the column's parameters in place of the model defaults.
//
// FP32-mixed: the state is U plus an increment D.  Within a step D gathers
// the stage increments (stage inputs U + D); at the end of the step U + D is
// split exactly (TwoSum) into its rounding s and the residual, U = s and D =
// the residual, so no step's increment is lost to the rounding of U: the
// state is carried to about twice FP32's precision for as long as it stays
// in registers.  A call split over several launches hands the residual to
// the next launch through a residual array; the stored state is rounded
// once, at the end of the call.
//
// Layout: tracer n (N, P, Z, D) is one packed array; column c occupies
// [offsets[c], offsets[c+1]) with k = 0 at the bottom.  Lane r of a column
// holds the L levels counted from the top, j = r*L + m (k = Nz_c - 1 - j).
// Cell centres depend only on j: zc = -(j + 1/2) dz.  A column takes
// ceil(Nz_c / L) lanes and a wave as many columns as fit into its 64 lanes,
// of every class with the same L (the host sorts columns into classes by
// depth); the sums down a column are masked to its lanes.  FP32 with a
// sediment is a kernel of its own (batch_ragged_sediment): the sediment's
// storage is FP64, and a sum down a column in another order moves it.
#pragma once

#include "obme_wave_kernels.h"

namespace obme {

// Column constants beyond the NPZD parameters.
struct BatchColumn {
    double PAR0;         // surface PAR (constant)
    double wP, wD;       // face velocities (<= 0) of P and D
    double Lt;           // Q10^(T/10) at the ensemble's temperature
};

template <typename FT>
struct BatchArgs {
    FT* U[4];                       // N, P, Z, D packed arrays
    FT* C[4];                       // FP32: the residuals of U, packed alike (launch to launch)
    int c_in, c_out;                // FP32: start from the stored residuals; store them at the end
    const int* offsets;             // [n_columns + 1]
    const int* cols;                // each lane's column (or -1)
    const FastParams<FT>* fpar;     // per-column derived constants
    const SedimentParams* fsed;     // FP32 with a sediment: these instead, for its transitions
    const BatchColumn* bcol;        // per-column constants
    int nsteps;
    FT dtf, dz, invdz;
    float rk_a[3], rk_b[3];         // FP32: Δt γ, Δt ζ per stage
    // TwoBand coefficients: FP64 reference form and FP32 log2-scaled form
    double kr, kb, xr, xb, er, eb, Rr;
    float kr2, kb2, er_f, eb_f, cr, cb, xr2h, xb2h;
    // InstantRemineralisation sediment under every column (storage
    // null: the coupling alone, the storage not advanced).  The flux through
    // the bottom face f = sedP (-wP) P + sedD (-wD) D
    // of the bottom cell, burial e = a + b (f / (k + f))^2, the receiver's
    // coupled tendency (1 - e) f / dz; after each stage's substep the storage
    // steps by the stage Δt with the tendency e f of the stage's start
    // (update_state.jl:6-17; instant_remineralisation.jl:101-123).
    double* storage;                // [n_columns] or null
    double* sedGm;                  // [n_columns] G⁻: the tendency of the sediment's last step
    int sed_init;                   // the sediment's first step ever is this launch's first step
    int sed_ab2;                    // this launch's first sediment step is a QuasiAdamsBashforth2 step
    int sed_recv;                   // receiver: 0 N, 1 P, 2 Z, 3 D
    double sed_dt[3];               // Δt γ1, Δt (γ2 + ζ2), Δt (γ3 + ζ3)
    double sed_cn, sed_cm;          // 3/2 + χ, 1/2 + χ
    FT sed_a, sed_b, sed_k;         // burial efficiency constants
    FT sedP, sedD;                  // 1 where P / D is one of the sinking tracers, else 0
};

constexpr int RAGGED_WAVES = 4;   // waves per workgroup

// The lane's place in its column: from the last lane at or before it whose
// predecessor has another (a lane without a column stands alone).
__device__ __forceinline__ int column_lane(int lane, int at)
{
    const int before = __shfl_up(at, 1, 64);   // (by every lane)
    const unsigned long long starts = __ballot(lane == 0 || at < 0 || before != at);
    return lane - (63 - __clzll((long long)(starts & (~0ull >> (63 - lane)))));
}

// The sum over the column's lanes from the top to this one, rounded as
// seg_prefix rounds it in a segment of its own: steps of 1, 2, 4 and 8 lanes
// within the column's groups of 16, then the group before, then the second
// group's last lane.  (column_prefix groups by the wave's rows of 16: its last
// bits depend on where the packing puts a column.)
struct FixedPrefix {
    bool b1, b2, b4, b8, odd, far, any_odd, any_far;
    int lane4, before4, l31;
    __device__ __forceinline__ FixedPrefix(int lane, int r)
    {
        const int g = r & 15;
        b1 = g >= 1;
        b2 = g >= 2;
        b4 = g >= 4;
        b8 = g >= 8;
        odd = (r & 16) != 0;
        far = r >= 32;
        any_odd = __any(odd);
        any_far = __any(far);
        lane4 = lane * 4;
        before4 = (lane - g - 1) * 4;
        l31 = (lane - r + 31) * 4;
    }
    __device__ __forceinline__ static float from(int lane4, float x)
    {
        return __int_as_float(__builtin_amdgcn_ds_bpermute(lane4, __float_as_int(x)));
    }
    __device__ __forceinline__ float operator()(float x) const
    {
        float y = lane_shr1(x);
        x = x + (b1 ? y : 0.0f);
        y = lane_shr1(lane_shr1(x));
        x = x + (b2 ? y : 0.0f);
        y = from(lane4 - 16, x);
        x = x + (b4 ? y : 0.0f);
        y = from(lane4 - 32, x);
        x = x + (b8 ? y : 0.0f);
        if (any_odd) {
            y = from(before4, x);
            x = x + (odd ? y : 0.0f);
        }
        if (any_far) {
            y = from(l31, x);
            x = x + (far ? y : 0.0f);
        }
        return x;
    }
};

// The same sums where every column starts at a row of 16 lanes (and a column of
// three or four rows at row 0): the wave's rows are the column's groups.
struct RowPrefix {
    int mA, mB;
    __device__ __forceinline__ RowPrefix(int lane, int r)
    {
        // (a column of two rows may start at row 2, one of three at row 0 only)
        mA = (r & 16) ? -1 : 0;
        mB = r >= 32 ? -1 : 0;
    }
    __device__ __forceinline__ float operator()(float x) const
    {
        x = seg_prefix<16>(x);
        x = x + lane_and(dpp<0x142, 0xf, true>(x), mA);
        x = x + lane_and(dpp<0x143, 0xf, true>(x), mB);
        return x;
    }
};

// FP32 with a sediment, in the ragged packing (ROWS: in whole rows of lanes).
// What bounds it is what bounds batch_ragged, and with a wave or two per SIMD
// the sums' latency.  In segments of 32 and 64 lanes per class, a launch each:
// 8192 columns of 16 to 128 levels, 50 steps, 463 us; this 340 (307 of 34 to
// 79 levels, 20 steps: 92.8 and 46).  FM: the default formulations compiled
// in, or < 0 (fm_light): they are read per lane, and each choice is a branch
// over the lanes (478 against 463 us), with the same roundings.
template <int L, int FM, bool ROWS>
__device__ __forceinline__ void batch_ragged_sediment(const BatchArgs<float>& a)
{
    const int lane = threadIdx.x & 63;
    const int at = a.cols[blockIdx.x * blockDim.x + threadIdx.x];
    const int col = at;
    const int r = column_lane(lane, at);
    const int off = (col >= 0) ? a.offsets[col] : 0;
    const int Nzc = (col >= 0) ? a.offsets[col + 1] - off : 0;
    const std::conditional_t<ROWS, RowPrefix, FixedPrefix> prefix(lane, r);
    // level m of this lane: j = r*L + m from the top, k = Nzc-1-j
    auto has = [&](int m) -> bool { return r * L + m < Nzc; };
    auto idx = [&](int m) -> int { return off + Nzc - 1 - (r * L + m); };

    float U[4][L], D[4][L], Gm[4][L];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int m = 0; m < L; m++) {
            U[n][m] = has(m) ? a.U[n][idx(m)] : 0.0f;
            Gm[n][m] = 0.0f;
            D[n][m] = (a.c_in && has(m)) ? a.C[n][idx(m)] : 0.0f;
        }
    auto val = [&](int n, int m) -> float { return U[n][m] + D[n][m]; };

    // column constants (every lane of a column reads the same entry)
    const int cc = (col >= 0) ? col : 0;
    const BatchColumn bc = a.bcol[cc];
    const float PAR0 = (float)bc.PAR0;
    const float Lt = (float)bc.Lt;
    const float wP = (float)bc.wP, wD = (float)bc.wD;
    const SedimentParams fp = a.fsed[cc];
    const float wiP = (float)(bc.wP / (double)a.dz), wiD = (float)(bc.wD / (double)a.dz);

    // the sediment of this column, held by the lane of its bottom cell
    // (j = Nzc - 1: lane rb, level mb)
    const int jb = Nzc - 1;
    const bool sed = col >= 0 && r == jb / L;
    const int mb = jb % L;
    // the storage and the last tendency in LDS (not held in registers
    // through the launch)
    __shared__ double s_sed[2][RAGGED_WAVES * 64];
    const int seg = threadIdx.x;
    if (sed) {
        s_sed[0][seg] = a.storage ? a.storage[col] : 0.0;
        s_sed[1][seg] = (a.storage && a.sed_ab2) ? a.sedGm[col] : 0.0;
    }

    // water terms of the own levels
    float ezr[L], ezb[L];
#pragma unroll
    for (int m = 0; m < L; m++) {
        const float zc = -((float)(r * L + m) + 0.5f) * a.dz;
        ezr[m] = a.kr2 * zc;
        ezb[m] = a.kb2 * zc;
    }

#pragma unroll 1
    for (int s = 0; s < a.nsteps; s++) {
#pragma unroll 1
        for (int st = 0; st < 3; st++) {
            // chlorophyll terms and the light integral (as in the sweep)
            float pr[L], pb[L];
#pragma unroll
            for (int m = 0; m < L; m++) {
                const float lg = m_log2(val(1, m));
                pr[m] = m_exp2(fmaf(a.er_f, lg, a.cr));
                pb[m] = m_exp2(fmaf(a.eb_f, lg, a.cb));
            }
            const float pr_up = lane_shr1(pr[L - 1]);
            const float pb_up = lane_shr1(pb[L - 1]);
            const float cP_up = lane_shr1(val(1, L - 1));
            const float cD_up = lane_shr1(val(3, L - 1));
            float incr[L], incb[L];
            float totr = 0.0f, totb = 0.0f;
#pragma unroll
            for (int m = 0; m < L; m++) {
                const bool top = (m == 0) && (r == 0);
                const float prn = (m == 0) ? pr_up : pr[m > 0 ? m - 1 : 0];
                const float pbn = (m == 0) ? pb_up : pb[m > 0 ? m - 1 : 0];
                const float ir = top ? pr[m] : prn + pr[m];
                const float ib = top ? pb[m] : pbn + pb[m];
                incr[m] = has(m) ? ir : 0.0f;
                incb[m] = has(m) ? ib : 0.0f;
                totr = totr + incr[m];
                totb = totb + incb[m];
            }
            float runr = lane_shr1(prefix(totr));
            float runb = lane_shr1(prefix(totb));
            if (r == 0) {
                runr = 0.0f;
                runb = 0.0f;
            }
            float PARv[L];
#pragma unroll
            for (int m = 0; m < L; m++) {
                runr = runr + incr[m];
                runb = runb + incb[m];
                PARv[m] = (PAR0 * 0.5f) * (m_exp2(fmaf(-a.xr2h, runr, ezr[m])) +
                                           m_exp2(fmaf(-a.xb2h, runb, ezb[m])));
            }
            // the sediment: the bottom cell's flux and burial, the
            // receiver's coupled tendency, the sediment step
            float cpl = 0.0f;
            if (sed) {
                float Pb = val(1, 0), Db = val(3, 0);
#pragma unroll
                for (int m = 1; m < L; m++)
                    if (m == mb) {
                        Pb = val(1, m);
                        Db = val(3, m);
                    }
                const float f = a.sedP * (-wP) * Pb + a.sedD * (-wD) * Db;
                // the hardware reciprocal (1 ulp) and 1/Δz
                const float qf = f * __builtin_amdgcn_rcpf(a.sed_k + f);
                const float e = a.sed_a + a.sed_b * (qf * qf);
                cpl = ((1.0f - e) * f) * a.invdz;
                const double ge = (double)(e * f);
                const bool init = a.sed_init && s == 0;
                if (st == 0) {
                    if (!init) {
                        const bool ab2 = a.sed_ab2 && s == 0;
                        s_sed[0][seg] += a.sed_dt[0] * (ab2 ? a.sed_cn * ge - a.sed_cm * s_sed[1][seg] : ge);
                    }
                } else {
                    if (st == 1 && init) s_sed[0][seg] += a.sed_dt[0] * ge;
                    s_sed[0][seg] += a.sed_dt[st] * ge;
                }
                s_sed[1][seg] = ge;
            }
            // tendencies bottom-up within the lane, sinking, RK3 substep
#pragma unroll
            for (int m = L - 1; m >= 0; m--) {
                const bool top = (m == 0) && (r == 0);
                const float N = val(0, m), P = val(1, m), Z = val(2, m), Dd = val(3, m);
                float G[4];
                npzd_sediment<FM>(fp, N, P, Z, Dd, PARv[m], Lt, G[0], G[1], G[2], G[3]);
                const float cPn = (m == 0) ? cP_up : val(1, m > 0 ? m - 1 : 0);
                const float cDn = (m == 0) ? cD_up : val(3, m > 0 ? m - 1 : 0);
                G[1] = fmaf(-wiP, (top ? 0.0f : cPn) - P, G[1]);
                G[3] = fmaf(-wiD, (top ? 0.0f : cDn) - Dd, G[3]);
                if (sed && m == mb) {
#pragma unroll
                    for (int n = 0; n < 4; n++)
                        if (n == a.sed_recv) G[n] = G[n] + cpl;
                }
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    const float A = (st == 0) ? a.rk_a[0] : (st == 1 ? a.rk_a[1] : a.rk_a[2]);
                    const float B = (st == 0) ? a.rk_b[0] : (st == 1 ? a.rk_b[1] : a.rk_b[2]);
                    D[n][m] = fmaf(A, G[n], fmaf(B, Gm[n][m], D[n][m]));
                    Gm[n][m] = G[n];
                }
            }
        }
        // U + D = s + e exactly (TwoSum): U = s, and e carries on
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int m = 0; m < L; m++) {
                const float u = U[n][m], d = D[n][m];
                const float sum = u + d;
                const float dv = sum - u;
                D[n][m] = (u - (sum - dv)) + (d - dv);
                U[n][m] = sum;
            }
    }
    if (sed && a.storage) {
        a.storage[col] = s_sed[0][seg];
        a.sedGm[col] = s_sed[1][seg];
    }
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int m = 0; m < L; m++)
            if (has(m)) {
                a.U[n][idx(m)] = U[n][m];
                if (a.c_out) a.C[n][idx(m)] = D[n][m];
            }
}

// The ragged packing: the lane's column from the host's table.
// What bounds it is the instructions of the transitions (four waves per SIMD,
// nothing read or written between the first step and the last), so lanes
// without a level are time lost: segments of 32 and 64 lanes held 72 % levels
// where columns have 16 to 128, in two launches of one wave's length each
// (8192 such columns, 50 steps in FP32: 404 us; this 269).  FM: the
// default formulations compiled in, or < 0 (fm_light).
template <typename FT, int L, int FM, bool SED>
__device__ __forceinline__ void batch_ragged(const BatchArgs<FT>& a)
{
    constexpr bool F32 = sizeof(FT) == 4;
    static_assert(!(F32 && SED), "FP32 with a sediment: batch_ragged_sediment");
    const int lane = threadIdx.x & 63;
    const int at = a.cols[blockIdx.x * blockDim.x + threadIdx.x];
    const bool ok = at >= 0;
    const int col = ok ? at : 0;
    const int r = column_lane(lane, at);
    const int off = a.offsets[col];
    const int Nzc = ok ? a.offsets[col + 1] - off : 0;
    auto has = [&](int m) -> bool { return r * L + m < Nzc; };
    auto idx = [&](int m) -> int { return off + Nzc - 1 - (r * L + m); };
    const ColumnMasks cm = column_masks<0>(lane, r);

    // (a lane's levels below the bottom hold 1: they feed no other lane or
    // level, and their powers are ordinary ones)
    FT U[4][L], D[F32 ? 4 : 1][L], Gm[4][L];
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int m = 0; m < L; m++) {
            U[n][m] = has(m) ? a.U[n][idx(m)] : FT(1);
            if constexpr (F32) D[n][m] = (a.c_in && has(m)) ? a.C[n][idx(m)] : FT(0);
        }
    const BatchColumn bc = a.bcol[col];
    const FT Lt = (FT)bc.Lt;
    const FT wiP = (FT)(bc.wP / (double)a.dz), wiD = (FT)(bc.wD / (double)a.dz);
    const FastParams<FT> fp = a.fpar[col];

    // the sediment of the column, held by the lane of its bottom cell
    const int jb = Nzc - 1, mb = jb % L;
    const bool sed = SED && ok && r == jb / L;
    double sed_u = 0.0, sed_ge = 0.0;
    if (sed) {
        sed_u = a.storage ? a.storage[col] : 0.0;
        sed_ge = (a.storage && a.sed_ab2) ? a.sedGm[col] : 0.0;
    }

    // the surface light left by the water alone at the own levels, halved
    FT wr[L], wb[L];
#pragma unroll
    for (int m = 0; m < L; m++) {
        const double zc = -((double)(r * L + m) + 0.5) * (double)a.dz, h = 0.5 * (ok ? bc.PAR0 : 0.0);
        wr[m] = (FT)(h * exp(a.kr * zc));
        wb[m] = (FT)(h * exp(a.kb * zc));
    }
    const double g2 = 5.0 / 12.0, g3 = 3.0 / 4.0, z2 = -17.0 / 60.0, z3 = -5.0 / 12.0;
    const FT hr = F32 ? (FT)a.xr2h : (FT)(a.xr * (0.5 * (double)a.dz));
    const FT hb = F32 ? (FT)a.xb2h : (FT)(a.xb * (0.5 * (double)a.dz));

#pragma unroll 1
    for (int s = 0; s < a.nsteps; s++) {
        auto stage = [&](auto st_c) {
            constexpr int st = decltype(st_c)::value;
            FT X[4][L];
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int m = 0; m < L; m++) {
                    if constexpr (F32) X[n][m] = U[n][m] + D[n][m];
                    else X[n][m] = U[n][m];
                }
            // the light: the integral to level j is, in half cells, twice the
            // sum over the levels above and the level's own
            FT pr[L], pb[L];
            FT totr = FT(0), totb = FT(0);
#pragma unroll
            for (int m = 0; m < L; m++) {
                if constexpr (F32) {
                    const float lg = m_log2(X[1][m]);
                    pr[m] = m_exp2(fmaf(a.er_f, lg, a.cr));
                    pb[m] = m_exp2(fmaf(a.eb_f, lg, a.cb));
                } else {
                    pow_pair<FM < 0>(X[1][m] * a.Rr, a.er, a.eb, pr[m], pb[m]);
                }
                totr = m == 0 ? pr[m] : totr + pr[m];
                totb = m == 0 ? pb[m] : totb + pb[m];
            }
            FT runr = lane_above<0>(column_prefix<0>(totr, cm), cm);
            FT runb = lane_above<0>(column_prefix<0>(totb, cm), cm);
            const FT cP_up = lane_above<0>(X[1][L - 1], cm), cD_up = lane_above<0>(X[3][L - 1], cm);
            FT PARv[L];
#pragma unroll
            for (int m = 0; m < L; m++) {
                const FT Ir = fma(FT(2), runr, pr[m]), Ib = fma(FT(2), runb, pb[m]);
                runr = runr + pr[m];
                runb = runb + pb[m];
                if constexpr (F32) PARv[m] = fma(wr[m], m_exp2(-hr * Ir), wb[m] * m_exp2(-hb * Ib));
                else PARv[m] = wr[m] * m_exp(-hr * Ir) + wb[m] * m_exp(-hb * Ib);
            }
            // the sediment: the bottom cell's flux and burial, the receiver's
            // coupled tendency, the sediment step
            FT cpl = FT(0);
            if constexpr (SED) {
                if (sed) {
                    FT Pb = X[1][0], Db = X[3][0];
#pragma unroll
                    for (int m = 1; m < L; m++)
                        if (m == mb) {
                            Pb = X[1][m];
                            Db = X[3][m];
                        }
                    const FT f = a.sedP * (-bc.wP) * Pb + a.sedD * (-bc.wD) * Db;
                    const FT qf = f / (a.sed_k + f);
                    const FT e = a.sed_a + a.sed_b * (qf * qf);
                    cpl = ((FT(1) - e) * f) / a.dz;
                    const double ge = (double)(e * f);
                    const bool init = a.sed_init && s == 0;
                    if (st == 0) {
                        if (!init)
                            sed_u += a.sed_dt[0] * (a.sed_ab2 && s == 0 ? a.sed_cn * ge - a.sed_cm * sed_ge : ge);
                    } else {
                        if (st == 1 && init) sed_u += a.sed_dt[0] * ge;
                        sed_u += a.sed_dt[st] * ge;
                    }
                    sed_ge = ge;
                }
            }
            // tendencies, sinking, RK3 substep
#pragma unroll
            for (int m = 0; m < L; m++) {
                FT G[4];
                npzd_fast<FM>(fp, X[0][m], X[1][m], X[2][m], X[3][m], PARv[m], Lt, G[0], G[1], G[2], G[3]);
                // (the lane above the top one gives 0)
                const FT cPn = m == 0 ? cP_up : X[1][m > 0 ? m - 1 : 0];
                const FT cDn = m == 0 ? cD_up : X[3][m > 0 ? m - 1 : 0];
                G[1] = fma(-wiP, cPn - X[1][m], G[1]);
                G[3] = fma(-wiD, cDn - X[3][m], G[3]);
                if constexpr (SED) {
                    if (sed && m == mb) {
#pragma unroll
                        for (int n = 0; n < 4; n++)
                            if (n == a.sed_recv) G[n] = G[n] + cpl;
                    }
                }
#pragma unroll
                for (int n = 0; n < 4; n++) {
                    if constexpr (F32) {
                        if constexpr (st == 0) D[n][m] = fmaf(a.rk_a[0], G[n], D[n][m]);
                        else D[n][m] = fmaf(a.rk_a[st], G[n], fmaf(a.rk_b[st], Gm[n][m], D[n][m]));
                    } else {
                        if constexpr (st == 0) U[n][m] += (a.dtf * (8.0 / 15.0)) * G[n];
                        else U[n][m] += a.dtf * ((st == 1 ? g2 : g3) * G[n] + (st == 1 ? z2 : z3) * Gm[n][m]);
                    }
                    Gm[n][m] = G[n];
                }
            }
        };
        stage(std::integral_constant<int, 0>{});
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        if constexpr (F32) {
            // U + D = s + e exactly (TwoSum): U = s, and e carries on
#pragma unroll
            for (int n = 0; n < 4; n++)
#pragma unroll
                for (int m = 0; m < L; m++) {
                    const float u = U[n][m], d = D[n][m];
                    const float sum = u + d;
                    const float dv = sum - u;
                    D[n][m] = (u - (sum - dv)) + (d - dv);
                    U[n][m] = sum;
                }
        }
    }
    if constexpr (SED) {
        if (sed && a.storage) {
            a.storage[col] = sed_u;
            a.sedGm[col] = sed_ge;
        }
    }
#pragma unroll
    for (int n = 0; n < 4; n++)
#pragma unroll
        for (int m = 0; m < L; m++)
            if (has(m)) {
                a.U[n][idx(m)] = U[n][m];
                if constexpr (F32) {
                    if (a.c_out) a.C[n][idx(m)] = D[n][m];
                }
            }
}

}  // namespace obme
