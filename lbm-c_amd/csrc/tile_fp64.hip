// D2Q9 tile kernels with StFP64 population storage.
#include "tile_launch.hpp"

namespace lbmc {

hipError_t launch_tile_fp64(const KernelKey &k, int size, const StepArgs<double> &a, const TilePass &p, int tiles,
                          hipStream_t s)
{
    return launch_tile_st<StFP64>(k, size, a, p, tiles, s);
}

}  // namespace lbmc
