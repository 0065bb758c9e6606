// Column kernels with l_max a compile-time number, a translation unit of their own.
#include "sphx_columns_fixed.hpp"

namespace sphx {

SPHX_INSTANTIATE_FIXED_COLUMNS(double, COLUMNS_VJP);

} // namespace sphx
