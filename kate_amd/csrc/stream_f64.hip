// stream_f64.hip -- instantiates k_stream for complex128 states.
#include "kernels_dev.hpp"
#include "kernels_inst.hpp"

namespace kate {

int launch_stream_f64(int tile_bits, void* state, const PassArgs& pa, const DevPlan& dp, void* stream)
{
    return stream_r<double, false>(tile_bits, state, pa, dp, (hipStream_t)stream);
}

}  // namespace kate
