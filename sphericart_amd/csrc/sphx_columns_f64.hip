// The column kernels in double: a translation unit of its own, so that the kernels of the library compile side by side.
#include "sphx_columns_dispatch.hpp"

namespace sphx {

template hipError_t dispatch_columns<double>(ColumnsKind, const ColumnsLaunch&, bool, const double*, const double*, const double*, double*,
                                          double*, hipStream_t);
template hipError_t upload_column_tables<double>(const HostTables&);

} // namespace sphx
