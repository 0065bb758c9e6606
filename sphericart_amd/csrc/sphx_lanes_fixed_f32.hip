// gradients_fixed_kernel in float: a translation unit of its own, so that the kernels of the library compile side by side.
#include "sphx_lanes_fixed_kernel.hpp"

namespace sphx {

template hipError_t dispatch_gradients_fixed<float>(const Launch&, bool, const float*, float*, float*, hipStream_t);
template hipError_t upload_channel_tables<float>(const HostTables&);

} // namespace sphx
