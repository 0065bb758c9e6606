// values_fixed_kernel in float: a translation unit of its own, so that the kernels of the library compile side by side.
#include "sphx_values_fixed_kernel.hpp"

namespace sphx {

template hipError_t dispatch_values_fixed<float>(const Launch&, bool, const float*, float*, hipStream_t);
template hipError_t upload_value_channel_tables<float>(const HostTables&);

} // namespace sphx
