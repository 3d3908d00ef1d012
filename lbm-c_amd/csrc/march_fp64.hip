// D3Q15 march kernels with StFP64 population storage.
#include "march_launch.hpp"

namespace lbmc {

hipError_t launch_march_fp64(const KernelKey &k, const StepArgs<double> &a, const MarchPass &p, hipStream_t s)
{
    return launch_march_st<StFP64>(k, a, p, s);
}

}  // namespace lbmc
