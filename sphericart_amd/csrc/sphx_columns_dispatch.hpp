// The launches of columns_kernel and column_rows_kernel, as templates over the arithmetic type; sphx_columns_f32.hip
// and sphx_columns_f64.hip instantiate them.
#ifndef SPHX_COLUMNS_DISPATCH_HPP
#define SPHX_COLUMNS_DISPATCH_HPP

#include "sphx_columns_kernel.hpp"
#include "sphx_runtime.hpp"

namespace sphx {

template <typename Kernel, typename... Args>
static hipError_t launch_columns(Kernel kernel, const ColumnsLaunch& l, hipStream_t stream, Args... args) {
    if (l.lds_bytes > 64u * 1024u) {
        unsigned unused = 0;
        const hipError_t e = kernel_facts(reinterpret_cast<const void*>(kernel), l.threads, l.lds_bytes, &unused);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(kernel, dim3(l.workgroups), dim3(l.threads), l.lds_bytes, stream, l.g, args...);
    return hipGetLastError();
}

template <typename T>
hipError_t dispatch_columns(ColumnsKind kind, const ColumnsLaunch& l, bool normalized, const T* xyz, const T* sph_grad,
                            const T* upstream, T* xyz_grad, T* sph_grad_grad, hipStream_t s) {
    if (l.fixed && l.g.accumulate == 0) {
        auto go = [&](auto dispatch) { return dispatch(l, normalized, xyz, sph_grad, upstream, xyz_grad, sph_grad_grad, s); };
        if (kind == COLUMNS_VJP) return go(dispatch_columns_fixed<T, COLUMNS_VJP>);
        if (kind == COLUMNS_VJP_BACKWARD) return go(dispatch_columns_fixed<T, COLUMNS_VJP_BACKWARD>);
        return go(dispatch_columns_fixed<T, COLUMNS_ROWS>);
    }
    if (kind == COLUMNS_ROWS) {
        return normalized ? launch_columns(column_rows_kernel<T, true>, l, s, xyz, sph_grad, upstream, xyz_grad)
                          : launch_columns(column_rows_kernel<T, false>, l, s, xyz, sph_grad, upstream, xyz_grad);
    }
    auto go = [&](auto kernel) { return launch_columns(kernel, l, s, xyz, sph_grad, upstream, xyz_grad, sph_grad_grad); };
    auto by_lanes = [&](auto second, auto add) {
        constexpr bool SECOND = decltype(second)::value, ADD = decltype(add)::value;
        if (l.groups == 2) {
            return normalized ? go(columns_kernel<T, true, SECOND, 2, ADD>) : go(columns_kernel<T, false, SECOND, 2, ADD>);
        }
        return normalized ? go(columns_kernel<T, true, SECOND, 1, ADD>) : go(columns_kernel<T, false, SECOND, 1, ADD>);
    };
    if (kind == COLUMNS_VJP_BACKWARD) return by_lanes(std::true_type{}, std::false_type{});
    return l.g.accumulate != 0 ? by_lanes(std::false_type{}, std::true_type{}) : by_lanes(std::false_type{}, std::false_type{});
}

// (every translation unit has its own copy of the table: internal linkage here as well)
template <typename T> static hipError_t fill_column_table(const HostTables& t) {
    if constexpr (sizeof(T) == 4) {
        const std::vector<float> table = column_table_of<float>(t.f32.data());
        return hipMemcpyToSymbol(HIP_SYMBOL(kColumns32), table.data(), table.size() * sizeof(float));
    } else {
        const std::vector<double> table = column_table_of<double>(t.f64.data());
        return hipMemcpyToSymbol(HIP_SYMBOL(kColumns64), table.data(), table.size() * sizeof(double));
    }
}

template <typename T> hipError_t upload_column_tables(const HostTables& t) { return fill_column_table<T>(t); }

} // namespace sphx

#endif
