// D2Q9 tile kernels with StBF16S population storage.
#include "tile_launch.hpp"

namespace lbmc {

hipError_t launch_tile_bf16s(const KernelKey &k, int size, const StepArgs<float> &a, const TilePass &p, int tiles,
                          hipStream_t s)
{
    return launch_tile_st<StBF16S>(k, size, a, p, tiles, s);
}

}  // namespace lbmc
