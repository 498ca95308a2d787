// mm_stage.hip -- the stage kernel's instantiations and launches (mm_stage.h)
// for one precision (MM_STAGE_T) and physics class (MM_STAGE_EN, MM_STAGE_STT,
// MM_STAGE_GEN, MM_STAGE_P1S); the Makefile builds one object per class.
#include "mm_stage.h"

template <typename T, bool EN, bool STT, int GEN, bool P1S> void stage_run(const StageArgs<T> &a)
{
    mm_with_len(a.len, a.generic, [&](auto lc) {
        hipLaunchKernelGGL((k_stage<T, EN, decltype(lc)::value, STT, GEN, P1S>), dim3(a.grid), dim3(a.threads), a.lds,
                           a.s, a.sys, a.rec, a.ctl, a.S1, a.p, a.Hx, a.Hp, a.rpw, a.demag, a.epart, a.Hdem);
    });
    MM_HIP(hipGetLastError());
}
template void stage_run<MM_STAGE_T, MM_STAGE_EN, MM_STAGE_STT, MM_STAGE_GEN, MM_STAGE_P1S>(
    const StageArgs<MM_STAGE_T> &);

#if !MM_STAGE_EN
#if !MM_STAGE_P1S
template <typename T, bool STT, int GEN> int stage_blocks_per_cu(int len, bool generic, int threads, size_t lds)
{
    int nb = 0;
    mm_with_len(len, generic, [&](auto lc) {
        MM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &nb, reinterpret_cast<const void *>(k_stage<T, false, decltype(lc)::value, STT, GEN, false>), threads, lds));
    });
    return nb;
}
template int stage_blocks_per_cu<MM_STAGE_T, MM_STAGE_STT, MM_STAGE_GEN>(int, bool, int, size_t);
#endif

template <typename T, bool STT, int GEN, bool P1S> void stage_run_batch(const BatchPass &bp, hipStream_t s, int st)
{
    if (bp.compiled)
        hipLaunchKernelGGL((kb_stage<T, MM_LC_ANY, STT, GEN, P1S>), dim3(bp.ntiles), dim3(bp.threads), bp.lds, s,
                           (const BStageDesc<T> *)bp.desc, (const int *)bp.tsys, st);
    else
        hipLaunchKernelGGL((kb_stage<T, 0, STT, GEN, P1S>), dim3(bp.ntiles), dim3(bp.threads), bp.lds, s,
                           (const BStageDesc<T> *)bp.desc, (const int *)bp.tsys, st);
    MM_HIP(hipGetLastError());
}
template void stage_run_batch<MM_STAGE_T, MM_STAGE_STT, MM_STAGE_GEN, MM_STAGE_P1S>(const BatchPass &, hipStream_t, int);
#endif
