// D3Q15 march kernels with StFP32 population storage.
#include "march_launch.hpp"

namespace lbmc {

hipError_t launch_march_fp32(const KernelKey &k, const StepArgs<float> &a, const MarchPass &p, hipStream_t s)
{
    return launch_march_st<StFP32>(k, a, p, s);
}

}  // namespace lbmc
