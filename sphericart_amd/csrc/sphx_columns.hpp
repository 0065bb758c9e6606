// The launches of columns_kernel and column_rows_kernel: their geometry (host and device) and what plans them.
#ifndef SPHX_COLUMNS_HPP
#define SPHX_COLUMNS_HPP

#include <cstddef>
#include <vector>

namespace sphx {

// The columns' table holds l <= kColumnsLMax: in float32 the iterates of the forward kernels' recursion start to leave
// the range of the type at l = 28, in float64 the rows of 32 points no longer fit LDS from l_max = 25 on.
constexpr int kColumnsLMax = 27;
constexpr int kColumnEntries = (kColumnsLMax + 1) * (kColumnsLMax + 2) / 2;
// numbers per entry (l, m): the factors of e_n and g_n, those of the sums A, B, C, then E, G, K
constexpr int kColumnEntry = 8;
// column m lists l = m .. kColumnsLMax one after the other
constexpr int column_start(int m) { return m * (kColumnsLMax + 1) - m * (m - 1) / 2; }

// threads of the largest workgroup
constexpr unsigned kColumnsThreads = 512;

struct Columns {
    unsigned long long n_samples;
    unsigned n_tiles, tiles_per_xcd;
    int l_max;
    unsigned ny;             // (l_max + 1)^2
    unsigned pad;            // elements left free after every staged row
    unsigned off_rows;       // column_rows_kernel: where the rows of the values' weights start
    unsigned off_sums;       // the sums of the waves beyond the first (0: where the rows were)
    unsigned accumulate;     // add to the output instead of overwriting it
    unsigned magic_ny, magic_vectors, magic_vectors3; // magic_of(ny), (ny in 16-byte vectors), (3 ny in vectors)
};

struct ColumnsLaunch {
    Columns g;
    unsigned workgroups, threads, lds_bytes;
    int groups; // lanes per point (columns_kernel: 1 or 2)
};

enum ColumnsKind {
    COLUMNS_VJP = 0,      // xyz_grad from sph_grad
    COLUMNS_VJP_BACKWARD, // its derivatives
    COLUMNS_ROWS          // xyz_grad from sph_grad and dsph_grad
};

// Whether the kernels take this shape, and how. Plain host arithmetic, a few dozen instructions.
bool plan_columns(ColumnsKind kind, size_t n_samples, int l_max, size_t elem, int lds_limit, int cus, ColumnsLaunch* out);

// Whether columns_kernel takes the vector-Jacobian product of this shape, for which the older kernels have `other`; then
// `out` is its plan.
struct VjpPlan;
bool vjp_by_columns(size_t n_samples, int l_max, size_t elem, int lds_limit, int cus, const VjpPlan& other, ColumnsLaunch* out);

// The table described above, in the arithmetic of T, made from the prefactors F of sphx_tables.hpp.
template <typename T> std::vector<T> column_table_of(const T* F);

} // namespace sphx

#endif
