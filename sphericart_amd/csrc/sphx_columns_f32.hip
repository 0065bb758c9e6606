// The column kernels in float: a translation unit of its own, so that the kernels of the library compile side by side.
#include "sphx_columns_dispatch.hpp"

namespace sphx {

template hipError_t dispatch_columns<float>(ColumnsKind, const ColumnsLaunch&, bool, const float*, const float*, const float*, float*,
                                          float*, hipStream_t);
template hipError_t upload_column_tables<float>(const HostTables&);

} // namespace sphx
