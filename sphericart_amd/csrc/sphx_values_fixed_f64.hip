// values_fixed_kernel in double: a translation unit of its own, so that the kernels of the library compile side by side.
#include "sphx_values_fixed_kernel.hpp"

namespace sphx {

template hipError_t dispatch_values_fixed<double>(const Launch&, bool, const double*, double*, hipStream_t);
template hipError_t upload_value_channel_tables<double>(const HostTables&);

} // namespace sphx
