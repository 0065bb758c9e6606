// hessians_fixed_kernel in float: a translation unit of its own, so that the kernels of the library compile side by side.
#include "sphx_hessians_fixed_kernel.hpp"

namespace sphx {

template hipError_t dispatch_hessians_fixed<float>(const Launch&, bool, const float*, float*, float*, float*, hipStream_t);
template hipError_t upload_hessian_channel_tables<float>(const HostTables&);

} // namespace sphx
