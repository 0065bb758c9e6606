// Host side of columns_kernel and column_rows_kernel: their constants and the geometry of a launch.
#include "sphx_columns.hpp"

#include <cstring>

#include "sphx_geometry.hpp"
#include "sphx_plan.hpp"

namespace sphx {

// Q_l^m at the pole is (-1)^m (l+m)! / (2^m m! (l-m)!), zero for m > l; e_n and g_n (sphx_columns_kernel.hpp) are
// there -(n-1)/(2m+2) and (n-2)(n-3)/((2m+2)(2m+4)), n = l - m. In float32 the prefactors F are used as they are in the
// tables of the forward kernels, their underflow from l = 19 on included, so that both describe the same functions.
template <typename T> std::vector<T> column_table_of(const T* F) {
    auto pole = [](int l, int m) -> long double {
        if (m > l || l < 0) return 0.0L;
        long double q = (m & 1) ? -1.0L : 1.0L;
        for (int k = l - m + 1; k <= l + m; ++k) q *= k;
        for (int k = 1; k <= m; ++k) q /= 2 * k;
        return q;
    };
    std::vector<T> table(static_cast<size_t>(kColumnEntries) * kColumnEntry);
    for (int m = 0; m <= kColumnsLMax; ++m) {
        for (int l = m; l <= kColumnsLMax; ++l) {
            T* t = table.data() + static_cast<size_t>(column_start(m) + l - m) * kColumnEntry;
            const int n = l - m;
            const long double f = F[l * (l + 1) / 2 + m], lm = l + m, w = 2 * m + 2;
            t[0] = n < 2 ? T(0) : static_cast<T>((n - 1) / lm);
            t[4] = n < 3 ? T(0) : static_cast<T>((n - 2) / lm);
            t[1] = static_cast<T>(f * pole(l, m));
            t[2] = n < 2 ? T(0) : static_cast<T>(-f * pole(l - 1, m + 1) * w / (n - 1));
            t[3] = static_cast<T>(f * lm * pole(l - 1, m));
            t[5] = n < 4 ? T(0) : static_cast<T>(f * pole(l - 2, m + 2) * w * (w + 2) / ((n - 2) * (n - 3)));
            t[6] = n < 3 ? T(0) : static_cast<T>(-f * lm * pole(l - 2, m + 1) * w / (n - 2));
            t[7] = static_cast<T>(f * lm * (lm - 1) * pole(l - 2, m));
        }
    }
    return table;
}
template std::vector<float> column_table_of<float>(const float*);
template std::vector<double> column_table_of<double>(const double*);

bool plan_columns(ColumnsKind kind, size_t n_samples, int l_max, size_t elem, int lds_limit, int cus, ColumnsLaunch* out) {
    if (l_max < 0 || l_max > kColumnsLMax) return false;
    const unsigned ny = static_cast<unsigned>((l_max + 1) * (l_max + 1)), e = static_cast<unsigned>(elem);
    const unsigned vec = 16u / e, pad = columns_pad(elem, ny);
    const unsigned limit = static_cast<unsigned>(lds_limit);
    auto rounded = [&](unsigned n) { return (n + vec - 1u) / vec * vec; };
    // The sums of the waves beyond the first (3 or 6 numbers per lane, 7 per point): where dw waits in the rows for its
    // flush they have a place of their own, else that of the rows, which are no longer needed then.
    const unsigned sums = kind == COLUMNS_ROWS ? 7u * 16u : (kind == COLUMNS_VJP ? 3u : 6u) * 64u;
    const bool apart = kind == COLUMNS_VJP_BACKWARD;

    int waves = 1;
    unsigned tile = 0, rows = 0, off_rows = 0;
    auto lay_out = [&](unsigned t, int w) {
        tile = t;
        waves = w;
        off_rows = kind == COLUMNS_ROWS ? rounded(t * (3u * ny + pad)) : 0u;
        rows = off_rows + rounded(t * (ny + pad));
        const unsigned all = static_cast<unsigned>(w - 1) * sums;
        return (apart ? rows + all : (rows > all ? rows : all)) * e;
    };
    const int forced_waves = switch_or(SW_COLUMNS_WAVES, 0), forced_tile = switch_or(SW_COLUMNS_TILE, 0);
    unsigned bytes = 0;
    const int most = l_max + 1 < 8 ? l_max + 1 : 8;
    // Waves per workgroup: enough workgroups fit a CU for one to compute while another one loads, and more waves than
    // that make a tile wait for its sums. Derivatives of the product, 1M points, l_max = 1, 3, 6 in float32, us with
    // 1 / 2 / 4 / 8 waves: 13.4 15.2 - -, 29.2 28.8 35.0 -, 86.0 74.8 66.2 86.2; 400 000 at l_max = 8 71 58 50 51;
    // float64 alike. A tile of 16 points (rows): l_max = 3, 6, 9, 12, 37 51 - -, 66 56 75 146, 98 68 59 98, 179 110 81
    // 87. Too few tiles for the CUs: as many waves as there are columns, up to eight (1 000 points at l_max = 6: 8.1 us
    // with one, 4.7 with eight).
    const size_t cu = static_cast<size_t>(cus > 0 ? cus : 1);
    if (kind == COLUMNS_ROWS) {
        waves = fixed_column_waves(kind, elem, l_max);
        if ((n_samples + 15) / 16 <= cu) waves = most;
        if (forced_waves > 0) waves = forced_waves < most ? forced_waves : most;
        bytes = lay_out(16u, waves);
    } else {
        tile = columns_tile(elem, l_max);
        const unsigned resident = columns_resident(elem, l_max);
        // four waves while many workgroups share a CU, eight below (the product, us with 4 / 8: float32 l_max = 8 27.5
        // 34.4, 10 37.1 33.1, 20 55.4 46.6; float64 l_max = 7 76 84, 8 55 48, 10 69 74, 13 93 85). The derivatives in
        // float64 need so many registers that eight waves would fill a CU: four unless the workgroup is alone (l_max =
        // 8: 95 143).
        waves = resident >= (e == 4 ? 6u : 4u) || (kind == COLUMNS_VJP_BACKWARD && e == 8 && resident > 1) ? 4 : 8;
        if (l_max < 6) waves = l_max < 3 ? 1 : 2;
        if (fixed_columns(kind, l_max)) waves = fixed_column_waves(kind, elem, l_max);
        if ((n_samples + 63) / 64 <= cu) {
            tile = 32u;
            waves = most;
        }
        if (forced_waves > 0) waves = forced_waves < most ? forced_waves : most;
        if (forced_tile == 32 || forced_tile == 64) tile = static_cast<unsigned>(forced_tile);
        bytes = lay_out(tile, waves);
        if (bytes > limit && tile == 64u) bytes = lay_out(32u, waves);
    }
    while (bytes > limit && waves > 1) bytes = lay_out(tile, waves / 2); // (the largest rows leave no room for many sums)
    if (bytes > limit) return false;
    // A launch holds fewer than 2^32 threads: fewer waves, where those of one wave are too many as well another path
    // (5.4e8 points at l_max = 10 in float32, 1.07e9 with arrays: 270 and 43 GB of them)
    const size_t tiles = (n_samples + tile - 1) / tile;
    auto too_many = [&]() { return (tiles + 7) / 8 * 8 > 0xffffffffull / (64u * static_cast<unsigned>(waves)); };
    while (too_many() && waves > 1) bytes = lay_out(tile, waves / 2);
    if (too_many()) return false;

    std::memset(&out->g, 0, sizeof(out->g));
    out->g.n_samples = n_samples;
    out->g.n_tiles = static_cast<unsigned>(tiles);
    out->g.tiles_per_xcd = (out->g.n_tiles + 7u) / 8u;
    out->g.l_max = l_max;
    out->g.ny = ny;
    out->g.pad = pad;
    out->g.off_rows = off_rows;
    out->g.off_sums = apart ? rows : 0u;
    out->g.magic_ny = magic_of(ny);
    out->g.magic_vectors = magic_of(ny / vec ? ny / vec : 1u);
    out->g.magic_vectors3 = magic_of(3u * ny / vec ? 3u * ny / vec : 1u);
    out->workgroups = out->g.tiles_per_xcd * 8u;
    out->threads = 64u * static_cast<unsigned>(waves);
    out->lds_bytes = bytes;
    out->groups = kind == COLUMNS_ROWS ? 4 : static_cast<int>(64u / tile);
    out->fixed = fixed_columns(kind, l_max) && fixed_columns_on(kind, elem, l_max, out->groups);
    return true;
}

// Up to l_max = 6 the sum runs over the closed forms in index order (number for number what contracting the gradients
// gives). Beyond, columns_kernel is ahead of the kernels that form every entry, but where the lane kernel's tiles are
// larger and so many points take it fewer rounds on the CUs: one instead of two, or, where a tile of columns_kernel leaves
// room for nothing else on a CU (float64 from l_max = 17, float32 from 25) and a few rounds follow one another, up to
// three for four. us, columns / lanes, rounds: float64 l_max = 17, 9 000 points 14.8 10.1 (2, 1), 17 000 27.1 23.0 (3, 2),
// 25 900 35.3 33.7 (4, 3), 41 100 50.3 45.7 (6, 4), as against 15 000 20.4 22.4 (2, 2), 38 000 42.6 45.1 (5, 4), 200 000 205 215; float32 20,
// 17 600 16.4 14.2 (2, 1), 19 000 18.0 20.9 (2, 2); 26, 9 000 18.5 13.6 (2, 1), 41 100 64 60 (6, 4).
bool vjp_by_columns(size_t n_samples, int l_max, size_t elem, int lds_limit, int cus, const VjpPlan& other, ColumnsLaunch* out) {
    if (l_max <= 6 || switch_or(SW_VJP_LANES, 1) == 0) return false;
    if (!plan_columns(COLUMNS_VJP, n_samples, l_max, elem, lds_limit, cus, out)) return false;
    if (!other.use_lanes) return true;
    auto resident = [&](unsigned bytes, unsigned threads) { // workgroups on a CU (LDS is handed out in pieces of 1 280 bytes)
        const unsigned by_lds = static_cast<unsigned>(lds_limit) / ((bytes + 1279u) / 1280u * 1280u), by_waves = 2048u / threads;
        return by_lds < by_waves ? (by_lds > 0 ? by_lds : 1u) : by_waves;
    };
    auto rounds = [&](unsigned tiles, unsigned at_once) { return (tiles + at_once - 1u) / at_once; };
    const unsigned units = static_cast<unsigned>(cus > 0 ? cus : 1);
    const unsigned beside = resident(out->lds_bytes, out->threads);
    const unsigned columns = rounds(out->g.n_tiles, units * beside);
    const unsigned lanes = rounds(other.lanes.g.n_tiles, units * resident(other.lanes.lds_bytes, other.lanes.threads));
    return !(beside == 1 ? lanes <= 4 && 10u * columns > 13u * lanes : columns == 2 && lanes == 1);
}

} // namespace sphx
