// What the planner and gradients_fixed_kernel both need to know: which l_max it exists for, how a workgroup's work is cut
// into units and dealt to its waves, how the rows lie in LDS. Plain C++.
#ifndef SPHX_LANES_FIXED_HPP
#define SPHX_LANES_FIXED_HPP

#include <cstddef>

namespace sphx {

// l_max of the kernels
constexpr int kGradientsFixedFirst = 7;
constexpr int gradients_fixed_last(size_t elem) { return elem == 4 ? 30 : 24; }
constexpr bool gradients_fixed(size_t elem, int l_max) {
    return l_max >= kGradientsFixedFirst && l_max <= gradients_fixed_last(elem);
}
// (beyond, only the form with eight waves is of use)
constexpr int gradients_fixed_last_sixteen(size_t elem) { return elem == 4 ? 16 : 11; }
constexpr unsigned kGradientsFixedPoints = 32; // the most points of a tile: two lanes each

// elements left free after the rows of a point (ny of the values, 3 ny of the gradients): where ny is even, a multiple of
// four, rows 8 bytes further apart start on 32 different pairs of banks and can still be read 8 bytes at a time
constexpr unsigned gradients_fixed_pad(size_t elem, unsigned ny) { return ny % 2u == 0u ? 8u / static_cast<unsigned>(elem) : 0u; }

// The units of a tile's work: the closed forms of l <= 6 in eight slices, then the channels from l_max down, each whole or in
// two parts, the upper half of its m and the lower one, which runs the recursions bare down to where it begins.
constexpr int kClosedSlices = 8;
constexpr int gradients_fixed_parts(int l_max, int waves) { return l_max <= 11 || waves > 8 ? 2 : 1; }
constexpr int gradients_fixed_units(int l_max, int waves) { return kClosedSlices + (l_max - 6) * gradients_fixed_parts(l_max, waves); }
struct ChannelPart {
    int l, m_top, m_bottom;
};
constexpr ChannelPart channel_part(int l_max, int waves, int unit) {
    const int parts = gradients_fixed_parts(l_max, waves), i = unit - kClosedSlices, l = l_max - i / parts;
    if (parts == 1) return {l, l, 0};
    return i % 2 == 0 ? ChannelPart{l, l, l / 2} : ChannelPart{l, l / 2 - 1, 0};
}
// instructions of a unit, roughly
constexpr int unit_cost(bool normalized, int l_max, int waves, int unit) {
    if (unit < kClosedSlices) return normalized ? 190 : 110;
    const ChannelPart c = channel_part(l_max, waves, unit);
    return (normalized ? 44 : 30) * (c.m_top - c.m_bottom + 1) + 8 * (c.l - c.m_top) + 20;
}

// Which units each of `waves` waves takes, one bit each: the longest unit left to the wave with the least so far.
constexpr int kFixedMostWaves = 16;
struct UnitMasks {
    unsigned long long of[kFixedMostWaves];
};
constexpr UnitMasks deal_units(bool normalized, int l_max, int waves) {
    UnitMasks masks{};
    int load[kFixedMostWaves] = {};
    bool taken[64] = {};
    const int units = gradients_fixed_units(l_max, waves);
    for (int round = 0; round < units; ++round) {
        int longest = -1;
        for (int u = 0; u < units; ++u) {
            if (!taken[u] && (longest < 0 || unit_cost(normalized, l_max, waves, u) > unit_cost(normalized, l_max, waves, longest))) longest = u;
        }
        int least = 0;
        for (int w = 1; w < waves; ++w) {
            if (load[w] < load[least]) least = w;
        }
        taken[longest] = true;
        load[least] += unit_cost(normalized, l_max, waves, longest);
        masks.of[least] |= 1ull << longest;
    }
    return masks;
}

// ---- values ------------------------------------------------------------------------------------------------------
constexpr int values_fixed_last(size_t elem) { return elem == 4 ? 32 : 28; }
constexpr bool values_fixed(size_t elem, int l_max) { return l_max >= kGradientsFixedFirst && l_max <= values_fixed_last(elem); }
// units: two slices of the closed forms, then the channels from l_max down; a wave that has any of those makes c_m, s_m and
// 2(m+1)z first
constexpr int kValueSlices = 2;
constexpr int value_unit_cost(int l_max, int unit) { return unit < kValueSlices ? 90 : 9 * (l_max - (unit - kValueSlices) + 1); }
constexpr UnitMasks deal_value_units(int l_max, int waves) {
    UnitMasks masks{};
    int load[kFixedMostWaves] = {};
    const int units = kValueSlices + l_max - 6;
    for (int i = 0; i < units; ++i) {
        const int u = (i + kValueSlices) % units; // the channels, longest first, then the slices
        int least = 0, least_load = 1 << 30;
        for (int w = 0; w < waves; ++w) {
            const int with = load[w] + (u >= kValueSlices && load[w] == 0 ? 7 * l_max : 0);
            if (with < least_load) {
                least = w;
                least_load = with;
            }
        }
        masks.of[least] |= 1ull << u;
        load[least] = least_load + value_unit_cost(l_max, u);
    }
    return masks;
}

// ---- second derivatives --------------------------------------------------------------------------------------
constexpr int kHessiansFixedFirst = 2;
// (normalised in float64 the entries outgrow the 128 registers that sixteen waves on a CU leave a lane: 4 spilled at l_max = 6,
// 8 at 7, where the kernel is still ahead)
constexpr int kHessiansFixedLast = 13;
constexpr int hessians_fixed_last(size_t elem, bool normalized) { return elem == 4 ? kHessiansFixedLast : (normalized ? 7 : 10); }
constexpr bool hessians_fixed(size_t elem, int l_max, bool normalized) {
    return l_max >= kHessiansFixedFirst && l_max <= hessians_fixed_last(elem, normalized);
}

// The units: l <= 1 in closed form, then the channels l = l_max .. 2, each in equal parts of at most `longest` entries m
// (an entry is a hundred operations and more, the bare steps down to where a part begins twelve each).
constexpr int hessians_fixed_longest(int l_max, int waves) {
    const int entries = (l_max + 1) * (l_max + 2) / 2 - 3, longest = (2 * entries + 3 * waves - 1) / (3 * waves);
    return longest < 2 ? 2 : longest;
}
constexpr int channel_parts(int l_max, int waves, int l) {
    const int longest = hessians_fixed_longest(l_max, waves);
    return (l + longest) / longest;
}
constexpr int hessians_fixed_units(int l_max, int waves) {
    int units = 1;
    for (int l = 2; l <= l_max; ++l) units += channel_parts(l_max, waves, l);
    return units;
}
constexpr ChannelPart hessian_part(int l_max, int waves, int unit) {
    int i = unit - 1;
    for (int l = l_max; l >= 2; --l) {
        const int parts = channel_parts(l_max, waves, l);
        if (i < parts) return {l, l - i * (l + 1) / parts, l + 1 - (i + 1) * (l + 1) / parts};
        i -= parts;
    }
    return {0, 0, 0};
}
constexpr int hessian_unit_cost(bool normalized, int l_max, int waves, int unit) {
    if (unit == 0) return normalized ? 260 : 60;
    const ChannelPart c = hessian_part(l_max, waves, unit);
    return (normalized ? 170 : 65) * (c.m_top - c.m_bottom + 1) + 12 * (c.l - c.m_top) + 20;
}
constexpr UnitMasks deal_hessian_units(bool normalized, int l_max, int waves) {
    UnitMasks masks{};
    int load[kFixedMostWaves] = {};
    bool taken[32] = {};
    const int units = hessians_fixed_units(l_max, waves);
    for (int round = 0; round < units; ++round) {
        int longest = -1;
        for (int u = 0; u < units; ++u) {
            if (!taken[u] && (longest < 0 || hessian_unit_cost(normalized, l_max, waves, u) > hessian_unit_cost(normalized, l_max, waves, longest))) longest = u;
        }
        int least = 0;
        for (int w = 1; w < waves; ++w) {
            if (load[w] < load[least]) least = w;
        }
        taken[longest] = true;
        load[least] += hessian_unit_cost(normalized, l_max, waves, longest);
        masks.of[least] |= 1ull << longest;
    }
    return masks;
}

} // namespace sphx

#endif
