// stream_f32.hip -- instantiates k_stream for complex64 states.
#include "kernels_dev.hpp"
#include "kernels_inst.hpp"

namespace kate {

int launch_stream_f32(int tile_bits, void* state, const PassArgs& pa, const DevPlan& dp, void* stream)
{
    return stream_r<float, false>(tile_bits, state, pa, dp, (hipStream_t)stream);
}

}  // namespace kate
