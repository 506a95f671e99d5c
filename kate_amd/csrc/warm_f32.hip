// warm_f32.hip -- instantiates the passes of small states (plan fetched ahead) for complex64.
#include "kernels_dev.hpp"
#include "kernels_inst.hpp"

namespace kate {

int launch_warm_f32(int tile_bits, void* state, const PassArgs& pa, const DevPlan& dp, void* stream)
{
    return warm_r<float>(tile_bits, state, pa, dp, (hipStream_t)stream);
}

}  // namespace kate
