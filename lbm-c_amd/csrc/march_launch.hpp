// Launcher of the D3Q15 march kernels (march_kernel.hpp), one translation
// unit per storage format (march_<storage>.hip).
#pragma once

#include "dispatch.hpp"
#include "march_kernel.hpp"

namespace lbmc {

template <class St, bool GUO, bool SMAG, int CLS, bool REUSE = false>
static hipError_t launch_march_one(const StepArgs<typename St::C> &a, const MarchPass &p, hipStream_t s)
{
    constexpr int T = march_threads((int)sizeof(typename St::S));
    hipLaunchKernelGGL((march_kernel<D3Q15, St, 0, GUO, SMAG, false, CLS, T, REUSE>), dim3(8 * p.per_xcd), dim3(T), 0, s, a,
                       p);
    return hipGetLastError();
}

template <class St, int CLS>
static hipError_t launch_march_cls(const KernelKey &k, const StepArgs<typename St::C> &a, const MarchPass &p,
                                   hipStream_t s)
{
    if constexpr (sizeof(typename St::C) == 4)
        if (k.closure)
            return k.guo ? launch_march_one<St, true, true, CLS, true>(a, p, s)
                         : launch_march_one<St, false, true, CLS, true>(a, p, s);
    if (k.guo)
        return k.smag ? launch_march_one<St, true, true, CLS>(a, p, s) : launch_march_one<St, true, false, CLS>(a, p, s);
    return k.smag ? launch_march_one<St, false, true, CLS>(a, p, s) : launch_march_one<St, false, false, CLS>(a, p, s);
}

template <class St>
static hipError_t launch_march_st(const KernelKey &k, const StepArgs<typename St::C> &a, const MarchPass &p,
                                  hipStream_t s)
{
    if (k.family != 0) return hipErrorInvalidValue;
    return p.cls == MARCH_FLUID ? launch_march_cls<St, MARCH_FLUID>(k, a, p, s)
                                : launch_march_cls<St, MARCH_SOLID>(k, a, p, s);
}

}  // namespace lbmc
