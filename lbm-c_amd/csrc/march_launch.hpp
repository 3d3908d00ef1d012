// Launcher of the D3Q15 march kernels (march_kernel.hpp), one translation
// unit per storage format (march_<storage>.hip).
#pragma once

#include "dispatch.hpp"
#include "march_kernel.hpp"

namespace lbmc {

template <class St, int FAM, int FORCE, bool SMAG, bool MFIX, int CLS, bool REUSE = false>
static hipError_t launch_march_one(const StepArgs<typename St::C> &a, const MarchPass &p, hipStream_t s)
{
    constexpr int T = march_threads((int)sizeof(typename St::S));
    hipLaunchKernelGGL((march_kernel<D3Q15, St, FAM, FORCE, SMAG, MFIX, CLS, T, REUSE>), dim3(8 * p.per_xcd), dim3(T),
                       0, s, a, p);
    return hipGetLastError();
}

template <class St, int FORCE, int CLS>
static hipError_t launch_march_force(const KernelKey &k, const StepArgs<typename St::C> &a, const MarchPass &p,
                                     hipStream_t s)
{
    if constexpr (sizeof(typename St::C) == 4)
        if (k.closure) return launch_march_one<St, 0, FORCE, true, false, CLS, true>(a, p, s);
    if (k.family != 0) {
        if (!k.mfix) return launch_march_one<St, 1, FORCE, false, false, CLS>(a, p, s);
        if constexpr (march_takes((int)sizeof(typename St::S), true, true, FORCE != MARCH_NO_FORCE))
            return launch_march_one<St, 1, FORCE, false, true, CLS>(a, p, s);
        else return hipErrorInvalidValue;
    }
    return k.smag ? launch_march_one<St, 0, FORCE, true, false, CLS>(a, p, s)
                  : launch_march_one<St, 0, FORCE, false, false, CLS>(a, p, s);
}

template <class St, int CLS>
static hipError_t launch_march_cls(const KernelKey &k, const StepArgs<typename St::C> &a, const MarchPass &p,
                                   hipStream_t s)
{
    if (!k.guo) return launch_march_force<St, MARCH_NO_FORCE, CLS>(k, a, p, s);
    return a.force[0] ? launch_march_force<St, MARCH_NODE_FORCE, CLS>(k, a, p, s)
                      : launch_march_force<St, MARCH_UNIFORM_FORCE, CLS>(k, a, p, s);
}

template <class St>
static hipError_t launch_march_st(const KernelKey &k, const StepArgs<typename St::C> &a, const MarchPass &p,
                                  hipStream_t s)
{
    return p.cls == MARCH_FLUID ? launch_march_cls<St, MARCH_FLUID>(k, a, p, s)
                                : launch_march_cls<St, MARCH_SOLID>(k, a, p, s);
}

}  // namespace lbmc
