// Launcher of the D2Q9 tile kernels (tile_kernel.hpp), one translation unit
// per storage format (tile_<storage>.hip).
#pragma once

#include "dispatch.hpp"
#include "tile_kernel.hpp"

namespace lbmc {

template <class St, int FAM, bool GUO, bool SMAG, int T, int NPT>
static void launch_tile_size(const StepArgs<typename St::C> &a, const TilePass &p, int tiles, hipStream_t s)
{
    hipLaunchKernelGGL((tile_kernel<D2Q9, St, FAM, GUO, SMAG, T, NPT>), dim3(tiles), dim3(T), 0, s, a, p);
}

template <class St, int FAM, bool GUO, bool SMAG>
static hipError_t launch_tile_one(int size, const StepArgs<typename St::C> &a, const TilePass &p, int tiles,
                                  hipStream_t s)
{
    constexpr int slot = (int)sizeof(typename St::S);
    if (size == 0)
        launch_tile_size<St, FAM, GUO, SMAG, tile_capacity(0, slot).threads, tile_capacity(0, slot).per_thread>(
            a, p, tiles, s);
    else if (size == 1)
        launch_tile_size<St, FAM, GUO, SMAG, tile_capacity(1, slot).threads, tile_capacity(1, slot).per_thread>(
            a, p, tiles, s);
    else
        launch_tile_size<St, FAM, GUO, SMAG, tile_capacity(2, slot).threads, tile_capacity(2, slot).per_thread>(
            a, p, tiles, s);
    return hipGetLastError();
}

template <class St>
static hipError_t launch_tile_st(const KernelKey &k, int size, const StepArgs<typename St::C> &a, const TilePass &p,
                                 int tiles, hipStream_t s)
{
    if (k.family == 0) {
        if (k.guo)
            return k.smag ? launch_tile_one<St, 0, true, true>(size, a, p, tiles, s)
                          : launch_tile_one<St, 0, true, false>(size, a, p, tiles, s);
        return k.smag ? launch_tile_one<St, 0, false, true>(size, a, p, tiles, s)
                      : launch_tile_one<St, 0, false, false>(size, a, p, tiles, s);
    }
    return k.guo ? launch_tile_one<St, 1, true, false>(size, a, p, tiles, s)
                 : launch_tile_one<St, 1, false, false>(size, a, p, tiles, s);
}

}  // namespace lbmc
