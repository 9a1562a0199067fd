// obme_sweep.hip — the column sweep's kernels (obme_npd_kernels.h) for one
// model (OBME_TU_MODEL, OBME_TU_CARB), compiled once per model.
#include "obme_wave_kernels.h"

namespace obme {

// The sweep: lane per water column, workgroups of blockDim.x = 64 NW
// consecutive columns (obme_npd_kernels.h).  FP32 is held to 128
// VGPRs (4 waves per SIMD, the occupancy at which the 512x512 grid's 4096
// waves fill the chip once).
template <int MODEL, int CARB, typename FT, int MODE, bool UNIFORM, int FM = -1, int EXTRA = 0, bool MASKX = true,
          int SCHEME = OBME_UPWIND1>
__global__ void __launch_bounds__(SWEEP_MAX_THREADS, (sizeof(FT) == 4 && (EXTRA & 2) == 0) ? 4 : 1)
k_column_lane(StepArgs<FT> a)
{
    column_lane<MODEL, CARB, FT, MODE, UNIFORM, FM, EXTRA, MASKX, true, SCHEME>(a, (int)blockDim.x);
}

// The kernel of a launch: mode, uniform grid, whole workgroups (stores without
// a mask), the model's default formulations (compiled in, FP32), the
// sinking scheme and the fused step's extra work.
template <int MODEL, int CARB, typename FT>
LaneKernel<FT> lane_kernel(int mode, bool uniform, bool whole, bool forms, int scheme, int extra)
{
    constexpr int FM = default_fm<MODEL>();
    if (mode == TILE_STAGE) {
        // centred / WENO sinking, one stage per launch (the general-grid form)
        return scheme == OBME_WENO5 ? k_column_lane<MODEL, CARB, FT, TILE_STAGE, false, -1, 0, true, OBME_WENO5>
                                    : k_column_lane<MODEL, CARB, FT, TILE_STAGE, false, -1, 0, true, OBME_CENTERED2>;
    }
    if (mode == TILE_PAR) {
        if (whole && uniform) return k_column_lane<MODEL, CARB, FT, TILE_PAR, true, -1, 0, false>;
        return uniform ? k_column_lane<MODEL, CARB, FT, TILE_PAR, true>
                       : k_column_lane<MODEL, CARB, FT, TILE_PAR, false>;
    }
    if (mode == TILE_TENDENCY) {
        if (scheme == OBME_WENO5) return k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, false, -1, 0, true, OBME_WENO5>;
        if (scheme == OBME_CENTERED2)
            return k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, false, -1, 0, true, OBME_CENTERED2>;
        if (whole && uniform && forms) return k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, true, FM, 0, false>;
        if (forms)
            return uniform ? k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, true, FM>
                           : k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, false, FM>;
        return uniform ? k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, true>
                       : k_column_lane<MODEL, CARB, FT, TILE_TENDENCY, false>;
    }
#define OBME_EXTRA_KERNEL(E)                                                              \
    (uniform ? k_column_lane<MODEL, CARB, FT, TILE_STEP, true, -1, E>                     \
             : k_column_lane<MODEL, CARB, FT, TILE_STEP, false, -1, E>)
    if (extra == 1) return OBME_EXTRA_KERNEL(1);
    if (extra == 4) return OBME_EXTRA_KERNEL(4);
    if (extra == 5) return OBME_EXTRA_KERNEL(5);
    if constexpr ((CARB & 1) != 0) {
        if (extra == 3) return OBME_EXTRA_KERNEL(3);
        if (extra == 7) return OBME_EXTRA_KERNEL(7);
    }
#undef OBME_EXTRA_KERNEL
    if (forms && whole)
        return uniform ? k_column_lane<MODEL, CARB, FT, TILE_STEP, true, FM, 0, false>
                       : k_column_lane<MODEL, CARB, FT, TILE_STEP, false, FM, 0, false>;
    if (forms)
        return uniform ? k_column_lane<MODEL, CARB, FT, TILE_STEP, true, FM>
                       : k_column_lane<MODEL, CARB, FT, TILE_STEP, false, FM>;
    return uniform ? k_column_lane<MODEL, CARB, FT, TILE_STEP, true> : k_column_lane<MODEL, CARB, FT, TILE_STEP, false>;
}
template LaneKernel<float> lane_kernel<OBME_TU_MODEL, OBME_TU_CARB, float>(int, bool, bool, bool, int, int);
template LaneKernel<double> lane_kernel<OBME_TU_MODEL, OBME_TU_CARB, double>(int, bool, bool, bool, int, int);

}  // namespace obme
