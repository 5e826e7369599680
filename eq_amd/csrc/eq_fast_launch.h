// eq_fast_launch.h -- launches of the transform kernels, for the translation
// units that instantiate them.
#pragma once

#include "eq_fast.h"

namespace eqk {

// (a launch within 64 KiB needs no leave)
template <typename T, bool GEN>
int fast_allow_lds(const FastSolver* F)
{
    int rc = EQ_OK;
    for (const FastClass& c : F->classes)
        if (c.lds > 64 * 1024) by_threads(c.threads, [&](auto t) {
            constexpr int NT = std::min(1024, decltype(t)::value), V = decltype(t)::value / NT * kFastValues;
            for (const void* k : {(const void*)k_fast_forward<T, NT, V, GEN>, (const void*)k_fast_backward<T, NT, V, GEN>})
                if (hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kFastLds) != hipSuccess)
                    rc = set_error(EQ_ERR_HIP, "hipFuncSetAttribute");
        });
    return rc;
}

template <typename T, bool GEN>
void fast_forward(eq_batch* b, int k, bool start)
{
    FastSolver* F = b->fast;
    for (const FastClass& c : F->classes)
        by_threads(c.threads, [&](auto t) {
            constexpr int NT = std::min(1024, decltype(t)::value), V = decltype(t)::value / NT * kFastValues;
            launch(b, EQ_KERNEL_STENCIL64, c.nodes * (16.0 + sizeof(T)), k_fast_forward<T, NT, V, GEN>,
                   dim3(grid8(c.njobs)), dim3(NT), c.lds, b->stream, (const FastJob*)F->d_jobs + c.job0, c.njobs,
                   (const LevelProb*)b->levels[0].d_probs, (const FastProb*)F->d_probs, (const FastRows*)F->d_rows,
                   (const FastPlan*)F->d_plans, (const Cx<T>*)F->d_tables, (const double*)b->u, (const double*)b->xprev,
                   (const double*)F->d_stiff, F->stiff_stride, (T*)b->z, F->d_partial, b->d_state, k, start ? 1 : 0);
        });
}

template <typename T, bool GEN>
void fast_backward(eq_batch* b, int k)
{
    FastSolver* F = b->fast;
    for (const FastClass& c : F->classes)
        by_threads(c.threads, [&](auto t) {
            constexpr int NT = std::min(1024, decltype(t)::value), V = decltype(t)::value / NT * kFastValues;
            launch(b, EQ_KERNEL_CG_UPDATE, c.nodes * ((GEN ? 32.0 : 16.0) + sizeof(T)), k_fast_backward<T, NT, V, GEN>,
                   dim3(grid8(c.njobs)), dim3(NT), c.lds, b->stream, (const FastJob*)F->d_jobs + c.job0, c.njobs,
                   (const LevelProb*)b->levels[0].d_probs, (const FastProb*)F->d_probs, (const FastPlan*)F->d_plans,
                   (const Cx<T>*)F->d_tables, (const T*)b->z, b->xprev, (const CgState*)b->d_state, b->q,
                   (const double2*)F->d_cheb, F->d_partial, k);
        });
}

} // namespace eqk
