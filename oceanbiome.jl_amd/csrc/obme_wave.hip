// obme_wave.hip — the kernels of obme_wave_kernels.h for one model
// (OBME_TU_MODEL, OBME_TU_CARB), compiled once per model.
#include "obme_wave_kernels.h"

namespace obme {

// FP32: held to 128 VGPRs (4 waves per SIMD) up to two levels per lane.
template <int MODEL, int CARB, typename FT, int MODE, bool UNI, int L, bool GEN, bool WIN, int FM, int SEG = 0>
__global__ void __launch_bounds__(WAVE_MAX_THREADS, sizeof(FT) == 4 && L < 4 ? 4 : 2) k_column_wave(WaveArgs<FT> w)
{
    extern __shared__ __align__(16) unsigned char smem[];
    column_wave<MODEL, CARB, FT, MODE, UNI, L, GEN, WIN, FM, SEG>(w, reinterpret_cast<FT*>(smem));
}

template <int CARB, typename FT, int FM>
__global__ void __launch_bounds__(64) k_top_steps(WaveArgs<FT> w, FT* rec)
{
    top_steps<CARB, FT, FM>(w, rec);
}

template <int MODEL, int CARB, typename FT, int L>
static WaveKernel<FT> wave_kernel_levels(int mode, bool uniform, int lpc, bool general, bool win)
{
    constexpr int FM = default_fm<MODEL>();
    // 64 levels (FP32 with more than one level per lane: wave_shape has one for
    // them on any number of columns)
    if constexpr (sizeof(FT) == 8 || L == 1) {
        constexpr int SEG = 64 / L;
        if (mode == TILE_STEP && !general && !win && uniform && lpc == SEG)
            return k_column_wave<MODEL, CARB, FT, TILE_STEP, true, L, false, false, FM, SEG>;
    }
    if (mode == TILE_STEP && !general && !win)
        return uniform ? k_column_wave<MODEL, CARB, FT, TILE_STEP, true, L, false, false, FM>
                       : k_column_wave<MODEL, CARB, FT, TILE_STEP, false, L, false, false, FM>;
    if constexpr (L <= 2) {
        if (mode == TILE_STEP && general && !win)
            return uniform ? k_column_wave<MODEL, CARB, FT, TILE_STEP, true, L, true, false, FM>
                           : k_column_wave<MODEL, CARB, FT, TILE_STEP, false, L, true, false, FM>;
        if (mode == TILE_STEP && !general && win)
            return k_column_wave<MODEL, CARB, FT, TILE_STEP, false, L, false, true, FM>;
        if (mode == TILE_TENDENCY)
            return win ? k_column_wave<MODEL, CARB, FT, TILE_TENDENCY, false, L, false, true, FM>
                       : k_column_wave<MODEL, CARB, FT, TILE_TENDENCY, false, L, false, false, FM>;
    }
    return nullptr;
}

template <int MODEL, int CARB, typename FT>
WaveKernel<FT> wave_kernel(int mode, bool uniform, int levels, int lpc, bool general, bool win)
{
    if (levels == 1) return wave_kernel_levels<MODEL, CARB, FT, 1>(mode, uniform, lpc, general, win);
    if (levels == 2) return wave_kernel_levels<MODEL, CARB, FT, 2>(mode, uniform, lpc, general, win);
    if constexpr (sizeof(FT) == 4)
        if (levels == 4) return wave_kernel_levels<MODEL, CARB, FT, 4>(mode, uniform, lpc, general, win);
    return nullptr;
}
template WaveKernel<float> wave_kernel<OBME_TU_MODEL, OBME_TU_CARB, float>(int, bool, int, int, bool, bool);
template WaveKernel<double> wave_kernel<OBME_TU_MODEL, OBME_TU_CARB, double>(int, bool, int, int, bool, bool);

#if OBME_TU_MODEL == 2 && (OBME_TU_CARB & 1)
template <int CARB, typename FT>
void (*top_kernel())(WaveArgs<FT>, FT*)
{
    return k_top_steps<CARB, FT, default_fm<OBME_LOBSTER>()>;
}
template void (*top_kernel<OBME_TU_CARB, float>())(WaveArgs<float>, float*);
template void (*top_kernel<OBME_TU_CARB, double>())(WaveArgs<double>, double*);
#endif

}  // namespace obme
