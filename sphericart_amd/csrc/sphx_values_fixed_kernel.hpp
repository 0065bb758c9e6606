// values_fixed_kernel: values beyond the closed forms, l_max a compile-time number.
#ifndef SPHX_VALUES_FIXED_KERNEL_HPP
#define SPHX_VALUES_FIXED_KERNEL_HPP

#include "sphx_lanes_fixed_kernel.hpp"

namespace sphx {

// ---------------------------------------------------------------------------
// gradients_fixed_kernel with values only: two lanes per point (+m and -m), up to 32 points per workgroup, whole channels
// l > 6 and two slices of the closed forms dealt to the waves at compile time. c_m, s_m, 2(m+1)z and the constants of an entry
// come from registers and scalar loads where values_kernel reads them from LDS or from a lane at every step, behind a barrier
// that waits for one wave to make the tables, and pairs_kernel's one workgroup per CU stores in turn with its recursions. Half
// of the recursions are done twice (by +m and -m), and that is still a fraction of the time its row takes to HBM (SQ counters,
// values_kernel / here, e6: 500 000 points of l_max = 12 in float32, two channels, vector 18 27, scalar 11 8, LDS 3.5 1.7; of
// 22, one channel, 83 96, 78 19, 16 8): tiles are small, so that some workgroups store while others compute, and no smaller, since c_m and 2(m+1)z of all m are made anew by every
// wave. us, normalised, before and after: float32 l_max = 12 30 000 points 7.0
// 5.7; 18 3 000 5.6 4.0; 22 30 000 17.4 13.7, 500 000 171 163; 28 30 000 40.4 21.3, 1.2 GB 251 198; 32 12 000 17.0 13.7, 1.2 GB
// 227 190; float64 7 100 000 16.0 10.2; 13 1.2 GB 223 191; 23 100 000 110 81, 1.2 GB 272 189; 28 1.2 GB 227 203.
//
// Same operations in the same order as the reference (templates_core.hpp:122-123,155,202-204,393), hence the same numbers.
// LDS: the value rows in HBM layout, an even row length padded by 8 bytes.
// ---------------------------------------------------------------------------

// Per entry (l, m), l >= 7, two numbers side by side: the constant of the recursion of Q_l at m and F_l^m.
static __constant__ float kValueChannels32[2 * channel_start(values_fixed_last(4) + 1)];
static __constant__ double kValueChannels64[2 * channel_start(values_fixed_last(8) + 1)];
template <typename T> __device__ __forceinline__ const T* value_channel_table();
template <> __device__ __forceinline__ const float* value_channel_table<float>() { return kValueChannels32; }
template <> __device__ __forceinline__ const double* value_channel_table<double>() { return kValueChannels64; }

template <typename T, bool NORM, int L, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void values_fixed_kernel(Tiling g, const T* __restrict__ xyz, T* __restrict__ sph) {
    constexpr unsigned NY = (L + 1) * (L + 1), PAD = gradients_fixed_pad(sizeof(T), NY), STRIDE = NY + PAD;
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
    static constexpr UnitMasks kMasks = deal_value_units(L, WAVES);
    const unsigned mine = static_cast<unsigned>(kMasks.of[wave]);
    T* row = lds + point * STRIDE;
    if (point < valid) {
        const Point<T> p = load_point<T, NORM>(xyz + (first + point) * 3);
        if ((mine & 3u) != 0 && !minus) {
            Rows<T> rows;
            rows.ny = static_cast<int>(NY);
            rows.sph = row;
            rows.dsph = rows.ddsph = nullptr;
            if (mine & 1u) closed_form_job<T, 0, NORM, 6, 0, 25>(p, rows);
            if (mine & 2u) closed_form_job<T, 0, NORM, 6, 25, 49>(p, rows);
        }
        if (mine >> kValueSlices) {
            T u[L + 1]; // c_m (+m) or s_m (-m)
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
            const int step = minus ? -1 : 1;
            for_each_number(std::make_integer_sequence<int, L - 6>{}, [&](auto unit) {
                constexpr int U = kValueSlices + decltype(unit)::value, l = L - decltype(unit)::value;
                if (!((mine >> U) & 1u)) return;
                const T* k = value_channel_table<T>() + channel_start(l) * 2;
                T* at = row + l * (l + 1) + step * l;
                T a2 = k[l * 2]; // Q_l^l
                T a1 = -p.z * a2; // Q_l^{l-1}
                for_each_number(std::make_integer_sequence<int, l + 1>{}, [&](auto down) {
                    constexpr int m = l - decltype(down)::value;
                    const T* km = k + m * 2;
                    if constexpr (m == l) {
                        at[0] = a2 * km[1] * u[m];
                    } else if constexpr (m == l - 1) {
                        at[0] = a1 * km[1] * u[m];
                    } else {
                        const T a0 = km[0] * (tz[m] * a1 + rxy * a2);
                        if constexpr (m > 0) {
                            at[0] = a0 * km[1] * u[m];
                        } else {
                            if (!minus) at[0] = a0 * km[1];
                        }
                        a2 = a1;
                        a1 = a0;
                    }
                    at -= step;
                });
            });
        }
    }
    __syncthreads(); // the rows
    flush_fixed_rows<T, NY, PAD>(lds, sph + first * NY, valid, tid, threads);
}

template <typename T> static hipError_t fill_value_channel_table(const HostTables& t) {
    constexpr int last = values_fixed_last(sizeof(T));
    const T* F;
    if constexpr (sizeof(T) == 4) F = t.f32.data();
    else F = t.f64.data();
    const T* Q = F + kTableEntries;
    T table[2 * channel_start(last + 1)];
    for (int l = kGradientsFixedFirst; l <= last; ++l) {
        for (int m = 0; m <= l; ++m) {
            const int at = l * (l + 1) / 2 + m;
            table[(channel_start(l) + m) * 2] = Q[at];
            table[(channel_start(l) + m) * 2 + 1] = F[at];
        }
    }
    if constexpr (sizeof(T) == 4) return hipMemcpyToSymbol(HIP_SYMBOL(kValueChannels32), table, sizeof(table));
    else return hipMemcpyToSymbol(HIP_SYMBOL(kValueChannels64), table, sizeof(table));
}

template <typename T, bool NORM>
static hipError_t launch_values_fixed(const Launch& l, const T* xyz, T* sph, hipStream_t stream) {
    hipError_t status = hipErrorInvalidValue; // (what values_fixed() does not name)
    if (l.threads != 512u && l.threads != 256u) return status; // never planned
    for_each_number(std::make_integer_sequence<int, values_fixed_last(sizeof(T)) - kGradientsFixedFirst + 1>{}, [&](auto i) {
        constexpr int L = kGradientsFixedFirst + decltype(i)::value;
        if (l.g.l_max != L) return;
        auto kernel = l.threads == 512u ? values_fixed_kernel<T, NORM, L, 8> : values_fixed_kernel<T, NORM, L, 4>;
        if (l.lds_bytes > 64u * 1024u) {
            unsigned unused = 0;
            status = kernel_facts(reinterpret_cast<const void*>(kernel), l.threads, l.lds_bytes, &unused);
            if (status != hipSuccess) return;
        }
        hipLaunchKernelGGL(kernel, dim3(l.workgroups), dim3(l.threads), l.lds_bytes, stream, l.g, xyz, sph);
        status = hipGetLastError();
    });
    return status;
}

template <typename T> hipError_t dispatch_values_fixed(const Launch& l, bool normalized, const T* xyz, T* sph, hipStream_t stream) {
    return normalized ? launch_values_fixed<T, true>(l, xyz, sph, stream) : launch_values_fixed<T, false>(l, xyz, sph, stream);
}
template <typename T> hipError_t upload_value_channel_tables(const HostTables& t) { return fill_value_channel_table<T>(t); }

} // namespace sphx

#endif
