// Passes over batches with FP64 population storage (built with contraction
// off, like step_fp64.hip, so members round like the reference).
#include "batch_tile_kernel.hpp"
#include "dispatch.hpp"

namespace lbmc {

hipError_t launch_batch_tiles_fp64(const void *members, const int2 *tiles, int ntiles, const BatchPass &bp,
                                   hipStream_t s)
{
    return launch_batch_tiles<StFP64>(members, tiles, ntiles, bp, s);
}

}  // namespace lbmc
