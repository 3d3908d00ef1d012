// Passes over batches with FP32 population storage, and their evaluating calls.
#include "batch_tile_kernel.hpp"
#include "dispatch.hpp"

namespace lbmc {

hipError_t launch_batch_tiles_fp32(const void *members, const int2 *tiles, int ntiles, const BatchPass &bp,
                                   hipStream_t s)
{
    return launch_batch_tiles<StFP32>(members, tiles, ntiles, bp, s);
}

hipError_t launch_batch_call_fp32(const void *members, const int2 *chunks, int nchunks, int grid, int sub,
                                  const void *mlp, bool record, bool fp16, const BatchPass &bp, hipStream_t s)
{
    auto go = [&](auto rec, auto h) {
        hipLaunchKernelGGL((batch_call_kernel<StFP32, decltype(rec)::value, decltype(h)::value>), dim3(grid),
                           dim3(kBlock), 0, s, (const BatchTileMember<float> *)members, chunks, nchunks, sub, mlp, bp);
        return hipGetLastError();
    };
    if (record) return fp16 ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    return fp16 ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
}

}  // namespace lbmc
