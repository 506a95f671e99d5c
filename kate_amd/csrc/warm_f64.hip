// warm_f64.hip -- instantiates the passes of small states (plan fetched ahead) for complex128.
#include "kernels_dev.hpp"
#include "kernels_inst.hpp"

namespace kate {

int launch_warm_f64(int tile_bits, void* state, const PassArgs& pa, const DevPlan& dp, void* stream)
{
    return warm_r<double>(tile_bits, state, pa, dp, (hipStream_t)stream);
}

}  // namespace kate
