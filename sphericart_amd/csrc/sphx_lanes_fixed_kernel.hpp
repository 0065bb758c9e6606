// gradients_fixed_kernel: values and gradients just above the closed forms, l_max a compile-time number.
#ifndef SPHX_LANES_FIXED_KERNEL_HPP
#define SPHX_LANES_FIXED_KERNEL_HPP

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

#include "sphx_lane_kernels.hpp"
#include "sphx_lanes_fixed.hpp"
#include "sphx_runtime.hpp"

namespace sphx {

// ---------------------------------------------------------------------------
// Two lanes per point, up to 32 points per workgroup: one lane for the entries (l, +m) and one for (l, -m), which share the
// recursions and little else. The work of a tile is cut into units, eight slices of the closed forms of l <= 6 and the l
// channels above, whole or in two halves of their m; which wave takes which is settled at compile time, longest first. No
// wave waits for another before the rows are complete.
//
// With l_max a constant everything around the arithmetic goes: c_m, s_m and 2(m+1)z of all m stay in registers, the
// constants of an entry come as one scalar load, several entries ahead, the places of its four numbers in the rows are
// offsets in the instructions, and no loop, job table or iterate in LDS is left. gradients_lanes_kernel waited at every step of
// a channel for a scalar load and an LDS read, recursion_kernel stores nothing while it works out its entries. The vector
// instructions are about as many as there, the recursions being run by +m and -m, those to LDS and to the scalar unit fewer
// (SQ counters, 400 000 points of l_max = 10 in float32, recursion_kernel / here: vector 57e6 63e6, scalar 25e6 20e6, LDS 7.7e6
// 4.7e6, bank conflicts 7.9e6 0 cycles): the gain is that workgroups are small and many, so one computes while another
// stores, and that they are dispatched in the order of the addresses they write: 1.2 GB leave at 5.9-6.5 TB/s in a loop where
// persistent workgroups reached 5.3-5.9 (behind another kernel: sphx_plan_shapes.hpp). us, normalised, before and after: float32 l_max = 7 3 000 points 6.0 4.3, 50 000 16.3 11.7, 1.2 GB 209 186; 9
// 20 000 14.0 7.7, 750 000 208 188; 12 15 000 17.2 9.6, 444 000 210 188; float64 8 10 000 points 9.0 7.6, 463 000 207 193;
// 9 20 000 24.6 15.0; 13 191 000 232 203. At larger l_max a tile holds few points and half of the lanes are idle (float32 from
// l_max = 20, float64 from 16 with more than one tile per CU): there it is ahead only while the call is latency, float32 22
// 2 500 13.2 9.0, 14 000 32.9 31.3, solid 20 000 40.9 34.4, 28 2 000 14.5 12.1; float64 17 200
// 32.4 8.4, 4 000 22.3 18.1, 23 200 55.8 13.1.
//
// Same operations in the same order as the reference (templates_core.hpp:122-426, through finish()), hence the same numbers.
// LDS: the value rows, then (g.off_dsph) the gradient rows, in HBM layout, an even row length padded by 8 bytes.
// ---------------------------------------------------------------------------

// Per entry (l, m), l >= 7, four numbers side by side, one scalar load: the constants of the recursions of Q_l and Q_{l-1}
// at m, F_l^m, F_l^m (l + m).
constexpr int kChannelEntry = 4;
constexpr int channel_start(int l) { return l * (l + 1) / 2 - 28; } // (28 entries of l <= 6 are not listed)
static __constant__ float kChannels32[kChannelEntry * channel_start(gradients_fixed_last(4) + 1)];
static __constant__ double kChannels64[kChannelEntry * channel_start(gradients_fixed_last(8) + 1)];
template <typename T> __device__ __forceinline__ const T* channel_table();
template <> __device__ __forceinline__ const float* channel_table<float>() { return kChannels32; }
template <> __device__ __forceinline__ const double* channel_table<double>() { return kChannels64; }

template <int... I, typename F> __host__ __device__ __forceinline__ void for_each_number(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}

// The rows of `points` points, ROW elements each and PAD elements apart, to one run in HBM.
template <typename T, unsigned ROW, unsigned PAD>
__device__ __forceinline__ void flush_fixed_rows(const T* staged, T* dst, unsigned points, unsigned tid, unsigned threads) {
    using V = typename Pack<T>::type;
    constexpr unsigned W = Pack<T>::width;
    const unsigned len = points * ROW;
    if constexpr (PAD == 0) {
        copy_out<T, SPHX_STREAMING_STORES, false, 1, true>(staged, dst, len, ROW, 0, 0, tid, threads);
    } else if ((reinterpret_cast<uintptr_t>(dst) & 15u) == 0) {
        typedef T Half __attribute__((ext_vector_type(8 / sizeof(T))));
        V* out = reinterpret_cast<V*>(dst);
        const unsigned nvec = len / W; // (a row is a whole number of vectors)
        for (unsigned v = tid; v < nvec; v += threads) {
            const Half* from = reinterpret_cast<const Half*>(staged + v * W + PAD * (v / (ROW / W)));
            const Half a = from[0], b = from[1];
            V both;
#pragma unroll
            for (unsigned e = 0; e < W / 2; ++e) {
                both[e] = a[e];
                both[W / 2 + e] = b[e];
            }
            emit<T, SPHX_STREAMING_STORES>(both, out + v);
        }
    } else {
        for (unsigned e = tid; e < len; e += threads) dst[e] = staged[e + PAD * (e / ROW)];
    }
}

template <typename T, bool NORM, int L, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void gradients_fixed_kernel(Tiling g, const T* __restrict__ xyz, T* __restrict__ sph,
                                                                               T* __restrict__ dsph) {
    constexpr unsigned NY = (L + 1) * (L + 1), PAD = gradients_fixed_pad(sizeof(T), NY);
    constexpr unsigned S_STRIDE = NY + PAD, D_STRIDE = 3 * NY + PAD;
    constexpr int UNITS = gradients_fixed_units(L, WAVES);
    T* lds = reinterpret_cast<T*>(lds_raw);
    const unsigned tid = threadIdx.x;
    const unsigned lane = tid & 63u;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr unsigned threads = 64 * WAVES;
    const unsigned group = (blockIdx.x & 7u) * g.tiles_per_xcd + (blockIdx.x >> 3);
    if (group >= g.n_tiles) return;
    const unsigned tile = static_cast<unsigned>(g.tile);
    const unsigned long long first = static_cast<unsigned long long>(group) * tile;
    const unsigned long long left = g.n_samples - first;
    const unsigned valid = left < tile ? static_cast<unsigned>(left) : tile;

    const unsigned point = lane & (kGradientsFixedPoints - 1u);
    const bool minus = lane >= kGradientsFixedPoints;
    static constexpr UnitMasks kMasks = deal_units(NORM, L, WAVES);
    const unsigned long long mine = kMasks.of[wave];
    T* row_s = lds + point * S_STRIDE;
    T* row_d = lds + g.off_dsph + point * D_STRIDE;
    if (point < valid) {
        const Point<T> p = load_point<T, NORM>(xyz + (first + point) * 3);
        if (!minus) {
            Rows<T> rows;
            rows.ny = static_cast<int>(NY);
            rows.sph = row_s;
            rows.dsph = row_d;
            rows.ddsph = nullptr;
            closed_form_slices<T, NORM, 6>(p, rows, [&](unsigned j) -> bool { return ((mine >> j) & 1u) != 0; });
        }
        if (mine >> kClosedSlices) {
            // c_m, s_m of the point: u the lane's own (c for +m, s for -m), w the other one with its sign in d/dy
            T u[L + 1], w[L + 1];
            {
                T cm = 1.0, sm = 0.0;
#pragma unroll
                for (int m = 0; m <= L; ++m) {
                    if (m > 0) {
                        const T cn = cm * p.x - sm * p.y;
                        const T sn = cm * p.y + sm * p.x;
                        cm = cn;
                        sm = sn;
                    }
                    u[m] = minus ? sm : cm;
                    w[m] = minus ? cm : -sm;
                }
            }
            T tz[L];
            {
                const T twoz = p.z + p.z;
                T t = twoz;
#pragma unroll
                for (int m = 0; m < L; ++m) {
                    tz[m] = t;
                    t = t + twoz;
                }
            }
            const T rxy = p.x2 + p.y2;
            const T zero = static_cast<T>(0.0);
            const int step = minus ? -1 : 1;
            for_each_number(std::make_integer_sequence<int, UNITS - kClosedSlices>{}, [&](auto unit) {
                constexpr int U = kClosedSlices + decltype(unit)::value;
                constexpr ChannelPart C = channel_part(L, WAVES, U);
                constexpr int l = C.l;
                if (!((mine >> U) & 1u)) return;
                const T* k = channel_table<T>() + channel_start(l) * kChannelEntry;
                T* at_s = row_s + l * (l + 1) + step * C.m_top;
                T* at_d = row_d + l * (l + 1) + step * C.m_top;
                T a2 = k[l * kChannelEntry];           // Q_l^l
                T a1 = -p.z * a2;                      // Q_l^{l-1}
                T b2 = 0;                              // the Q_{l-1} sequence: 0 at m = l,
                T b1 = k[(l - 1) * kChannelEntry + 1]; // Q_{l-1}^{l-1} at m = l - 1
                auto stage_at = [&](T v, T gx, T gy, T gz) {
                    Entry<T> e;
                    e.v = v;
                    e.gx = gx;
                    e.gy = gy;
                    e.gz = gz;
                    e.hxx = e.hxy = e.hxz = e.hyy = e.hyz = e.hzz = zero;
                    e = finish<T, 1, NORM>(p, e);
                    at_s[0] = e.v;
                    at_d[0] = e.gx;
                    at_d[NY] = e.gy;
                    at_d[2 * NY] = e.gz;
                };
                for_each_number(std::make_integer_sequence<int, l - C.m_bottom + 1>{}, [&](auto down) {
                    constexpr int m = l - decltype(down)::value;
                    const T* km = k + m * kChannelEntry;
                    if constexpr (m == l) {
                        // templates_core.hpp:122-152
                        if constexpr (m <= C.m_top) {
                            auto pq = a2 * km[2];
                            const T v = pq * u[m];
                            pq *= l;
                            stage_at(v, pq * u[m - 1], pq * w[m - 1], zero);
                        }
                    } else if constexpr (m == l - 1) {
                        // :154-198
                        if constexpr (m <= C.m_top) {
                            auto pq = a1 * km[2];
                            const T v = pq * u[m];
                            pq *= (l - 1);
                            stage_at(v, pq * u[m - 1], pq * w[m - 1], (km[3] * b1) * u[m]);
                        }
                    } else {
                        const T a0 = km[0] * (tz[m] * a1 + rxy * a2);
                        const T b0 = km[1] * (tz[m] * b1 + rxy * b2);
                        if constexpr (m <= C.m_top && m > 0) {
                            // :201-294
                            auto pq = a0 * km[2];
                            const T v = pq * u[m];
                            pq *= m;
                            auto pdq = km[2] * b1;
                            auto pdqx = pdq * p.x;
                            auto pdqy = pdq * p.y;
                            auto pdz = km[3] * b0;
                            stage_at(v, (pdqx * u[m] + pq * u[m - 1]), (pdqy * u[m] + pq * w[m - 1]), pdz * u[m]);
                        } else if constexpr (m == 0) {
                            // :392-426
                            if (!minus) stage_at(a0 * km[2], km[2] * p.x * b1, km[2] * p.y * b1, km[3] * b0);
                        }
                        a2 = a1;
                        a1 = a0;
                        b2 = b1;
                        b1 = b0;
                    }
                    if constexpr (m <= C.m_top) {
                        at_s -= step;
                        at_d -= step;
                    }
                });
            });
        }
    }
    __syncthreads(); // the rows
    flush_fixed_rows<T, NY, PAD>(lds, sph + first * NY, valid, tid, threads);
    flush_fixed_rows<T, 3 * NY, PAD>(lds + g.off_dsph, dsph + first * 3 * NY, valid, tid, threads);
}

template <typename T> static hipError_t fill_channel_table(const HostTables& t) {
    constexpr int last = gradients_fixed_last(sizeof(T));
    const T* F;
    if constexpr (sizeof(T) == 4) F = t.f32.data();
    else F = t.f64.data();
    const T* Q = F + kTableEntries;
    T table[kChannelEntry * channel_start(last + 1)];
    for (int l = kGradientsFixedFirst; l <= last; ++l) {
        for (int m = 0; m <= l; ++m) {
            const int at = l * (l + 1) / 2 + m;
            T* k = table + (channel_start(l) + m) * kChannelEntry;
            k[0] = Q[at];
            k[1] = Q[at - l]; // (m = l: not used)
            k[2] = F[at];
            k[3] = F[at] * static_cast<T>(l + m); // rounded as in pkm * (l + m) * ..
        }
    }
    if constexpr (sizeof(T) == 4) return hipMemcpyToSymbol(HIP_SYMBOL(kChannels32), table, sizeof(table));
    else return hipMemcpyToSymbol(HIP_SYMBOL(kChannels64), table, sizeof(table));
}

template <typename T, bool NORM>
static hipError_t launch_gradients_fixed(const Launch& l, const T* xyz, T* sph, T* dsph, hipStream_t stream) {
    hipError_t status = hipErrorInvalidValue; // (what gradients_fixed() does not name)
    if (l.threads != 512u && l.threads != 1024u) return status; // never planned
    for_each_number(std::make_integer_sequence<int, gradients_fixed_last(sizeof(T)) - kGradientsFixedFirst + 1>{}, [&](auto i) {
        constexpr int L = kGradientsFixedFirst + decltype(i)::value;
        if (l.g.l_max != L) return;
        auto kernel = gradients_fixed_kernel<T, NORM, L, 8>;
        if constexpr (L <= gradients_fixed_last_sixteen(sizeof(T))) {
            if (l.threads == 1024u) kernel = gradients_fixed_kernel<T, NORM, L, 16>;
        } else if (l.threads != 512u) {
            return; // never planned
        }
        if (l.lds_bytes > 64u * 1024u) {
            unsigned unused = 0;
            status = kernel_facts(reinterpret_cast<const void*>(kernel), l.threads, l.lds_bytes, &unused);
            if (status != hipSuccess) return;
        }
        hipLaunchKernelGGL(kernel, dim3(l.workgroups), dim3(l.threads), l.lds_bytes, stream, l.g, xyz, sph, dsph);
        status = hipGetLastError();
    });
    return status;
}

template <typename T>
hipError_t dispatch_gradients_fixed(const Launch& l, bool normalized, const T* xyz, T* sph, T* dsph, hipStream_t stream) {
    return normalized ? launch_gradients_fixed<T, true>(l, xyz, sph, dsph, stream)
                      : launch_gradients_fixed<T, false>(l, xyz, sph, dsph, stream);
}
template <typename T> hipError_t upload_channel_tables(const HostTables& t) { return fill_channel_table<T>(t); }

} // namespace sphx

#endif
