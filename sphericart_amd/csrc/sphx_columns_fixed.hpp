// The column kernels with l_max a compile-time number: their launches, as templates over the arithmetic type and the
// kind of product; the sphx_columns_fixed_*.hip instantiate them, one of each a translation unit.
#ifndef SPHX_COLUMNS_FIXED_HPP
#define SPHX_COLUMNS_FIXED_HPP

#include "sphx_columns_dispatch.hpp"

namespace sphx {

template <typename T, int KIND>
hipError_t dispatch_columns_fixed(const ColumnsLaunch& l, bool normalized, const T* xyz, const T* sph_grad, const T* upstream,
                                  T* xyz_grad, T* sph_grad_grad, hipStream_t s) {
    hipError_t status = hipErrorInvalidValue; // (what fixed_columns() or fixed_columns_on() do not name)
    each_of(std::make_integer_sequence<int, fixed_columns_last(KIND) - fixed_columns_first(KIND) + 1>{}, [&](auto i) {
        constexpr int L = fixed_columns_first(KIND) + decltype(i)::value;
        if (l.g.l_max != L) return;
        if constexpr (KIND == COLUMNS_ROWS) {
            status = normalized ? launch_columns(column_rows_kernel<T, true, L>, l, s, xyz, sph_grad, upstream, xyz_grad)
                                : launch_columns(column_rows_kernel<T, false, L>, l, s, xyz, sph_grad, upstream, xyz_grad);
        } else {
            constexpr bool SECOND = KIND == COLUMNS_VJP_BACKWARD;
            auto go = [&](auto kernel) { status = launch_columns(kernel, l, s, xyz, sph_grad, upstream, xyz_grad, sph_grad_grad); };
            if (l.groups == 2) {
                if (normalized) go(columns_kernel<T, true, SECOND, 2, false, L>);
                else go(columns_kernel<T, false, SECOND, 2, false, L>);
            } else if constexpr (fixed_columns_on(KIND, sizeof(T), L, 1)) {
                if (normalized) go(columns_kernel<T, true, SECOND, 1, false, L>);
                else go(columns_kernel<T, false, SECOND, 1, false, L>);
            }
        }
    });
    return status;
}

template <typename T, int KIND> hipError_t upload_fixed_columns(const HostTables& t) { return fill_column_table<T>(t); }

#define SPHX_INSTANTIATE_FIXED_COLUMNS(T, KIND)                                                                      \
    template hipError_t dispatch_columns_fixed<T, KIND>(const ColumnsLaunch&, bool, const T*, const T*, const T*, T*, T*, \
                                                        hipStream_t);                                                \
    template hipError_t upload_fixed_columns<T, KIND>(const HostTables&)

} // namespace sphx

#endif
