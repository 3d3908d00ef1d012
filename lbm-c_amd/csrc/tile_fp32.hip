// D2Q9 tile kernels with StFP32 population storage.
#include "tile_launch.hpp"

namespace lbmc {

hipError_t launch_tile_fp32(const KernelKey &k, int size, const StepArgs<float> &a, const TilePass &p, int tiles,
                          hipStream_t s)
{
    return launch_tile_st<StFP32>(k, size, a, p, tiles, s);
}

}  // namespace lbmc
