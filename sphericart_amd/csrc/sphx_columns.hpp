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
// numbers per entry (l, m): the factor of e_n and those of the sums A, B, C, then the factor of g_n and those of E, G, K
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
    bool fixed; // the kernel that has l_max for a constant (not where the product is added to the output)
};

enum ColumnsKind {
    COLUMNS_VJP = 0,      // xyz_grad from sph_grad
    COLUMNS_VJP_BACKWARD, // its derivatives
    COLUMNS_ROWS          // xyz_grad from sph_grad and dsph_grad
};

// elements left free after every staged row: rows an odd number of elements apart start on different banks (a row of one
// vector stays as it is: the division by its length that places the pads has no multiplier)
constexpr unsigned columns_pad(size_t elem, unsigned ny) { return ny % 2 == 0 && ny > 16u / elem ? 1u : 0u; }
// Points per tile of columns_kernel in large calls, 64 while three such tiles fit a CU, else 32, and how many fit then
// (derivatives of the product, 200 000 points at l_max = 12: 56.6 against 55.0 us in float32 where 43 KB still fit three
// times, 128 against 111 in float64 where 86 KB do not; the product, 100 000 at l_max = 16 in float64: 73 against 63)
constexpr unsigned kColumnsLds = 160u * 1024u;
constexpr unsigned columns_row_bytes(size_t elem, int l_max) {
    const unsigned ny = static_cast<unsigned>((l_max + 1) * (l_max + 1));
    return (ny + columns_pad(elem, ny)) * static_cast<unsigned>(elem);
}
constexpr unsigned columns_tile(size_t elem, int l_max) { return 64u * columns_row_bytes(elem, l_max) <= kColumnsLds / 3u ? 64u : 32u; }
constexpr unsigned columns_resident(size_t elem, int l_max) {
    return kColumnsLds / (columns_tile(elem, l_max) * columns_row_bytes(elem, l_max));
}
// What has a kernel with l_max for a constant: the l_max of the products that are asked for most (the code of a kernel, and
// the time it takes to compile, grow with l_max^2), on the lanes per point that large and small calls are planned with.
constexpr int fixed_columns_first(int kind) { return kind == COLUMNS_VJP ? 7 : 1; }
constexpr int fixed_columns_last(int kind) { return kind == COLUMNS_VJP ? 20 : 12; }
constexpr bool fixed_columns(int kind, int l_max) {
    return l_max >= fixed_columns_first(kind) && l_max <= fixed_columns_last(kind);
}
constexpr bool fixed_columns_on(int kind, size_t elem, int l_max, int groups) {
    return kind == COLUMNS_ROWS || groups == 2 || columns_tile(elem, l_max) == 64u;
}
// Waves of a workgroup of the kernels that have l_max for a constant, in large calls. us with 1 / 2 / 4 / 8: the product,
// 400 000 points, float32 l_max = 8 31.8 24.9 22.5 22.2, 14 105 76 68 80, 17 235 140 101 108, 20 (two on a CU) 375 223
// 147 133; float64 12 180 126 106 115, 14 (two) 313 200 152 144. Its derivatives, float32 3 10.5 12.5 13.2 -, 5 26.0 23.6
// 22.7 25.2, 8 61 50 44 46; float64 2 17.1 18.1 17.0 -, 4 35.7 32.9 32.5 55.5, 8 128 96 88 122. The rows, float32 3 24.0
// 28.0 40.2 -, 6 82 68 76 129, 8 148 114 106 157; float64 4 81 88 107 -, 6 173 137 152 334, 9 400 278 236 440.
constexpr int fixed_column_waves(int kind, size_t elem, int l_max) {
    if (kind == COLUMNS_VJP) return columns_resident(elem, l_max) >= 3u ? 4 : 8;
    if (kind == COLUMNS_ROWS) return l_max < 5 ? 1 : (l_max < 8 ? 2 : 4);
    const int first = elem == 4 ? 4 : 3;
    return l_max < first ? 1 : (l_max == first ? 2 : 4);
}
// 16-byte vectors per lane of a tile with so many elements, and how many of them are under way at a time: all, or equal
// parts of at most 12
constexpr unsigned column_rounds(int kind, size_t elem, int l_max, unsigned elements) {
    const unsigned lanes = 64u * static_cast<unsigned>(fixed_column_waves(kind, elem, l_max));
    const unsigned all = (elements / (16u / static_cast<unsigned>(elem)) + lanes - 1u) / lanes, blocks = (all + 11u) / 12u;
    return (all + blocks - 1u) / blocks;
}

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
