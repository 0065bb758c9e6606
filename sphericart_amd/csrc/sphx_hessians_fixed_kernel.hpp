// hessians_fixed_kernel: values, gradients and second derivatives at small l_max, l_max a compile-time number.
#ifndef SPHX_HESSIANS_FIXED_KERNEL_HPP
#define SPHX_HESSIANS_FIXED_KERNEL_HPP

#include "sphx_lanes_fixed_kernel.hpp"

namespace sphx {

// ---------------------------------------------------------------------------
// gradients_fixed_kernel with second derivatives: two lanes per point (+m and -m), up to 32 points per workgroup, the channels
// l = 2 .. l_max in parts of a few entries m dealt to the waves at compile time, the three recursions of a channel in
// registers. An entry is entry_job_from (sphx_device.hpp) with l and m literals. recursion_kernel's one workgroup per CU
// stores nothing while it computes; here two to five workgroups per CU do both. What the entries issue to the vector units is
// about the same (SQ counters, recursion_kernel / here, e6: float32 normalised l_max = 5, 500 000 points, vector 80 80, scalar
// 32 23, LDS 7.8 4.0; 7, 300 000, 98 108, 33 13, 9.3 5.7; solid 5, 300 000, 29 21, 21 14, 4.5 2.4; float64 6, 100 000, 30 36, 10
// 7.5, 2.9 2.1): look-up and addresses are gone, the recursions are run by both sides of an entry. Normalised in float64 at
// l_max = 6, 7 and solid at 10 2 to 8 vector registers are spilled to scratch (128 per lane). us, before and after: float32 normalised l_max =
// 3 30 000 points 9.3 6.2, 1.2 GB 291 189; 5 2 000 9.9 4.3, 30 000 17.1 12.5, 300 000 108 102; 7 30 000 33 21, 1.2 GB 243
// 210; float64 4 30 000 26.7 17.2, 1.2 GB 237 199; 6 30 000 44 30, 1.2 GB 255 207; solid 8 30 000 59 49, 1.2 GB 223 201.
// From l_max = 11 in float32 (one workgroup per CU holds the rows) 2 500 12.2 9.5, solid 10 000 24.2 17.0, 1.2 GB 209 190;
// beyond 13, and in float64 beyond 10, level or behind.
//
// Same operations in the same order as the reference, hence the same numbers. LDS: the rows of the three arrays.
// ---------------------------------------------------------------------------

// Per entry (l, m), l >= 2, four numbers side by side, one scalar load: the constants of the three recursions at m (or the
// value one of them starts with) and F_l^m.
constexpr int kHessianEntry = 4;
constexpr int hessian_channel_start(int l) { return l * (l + 1) / 2 - 3; }
static __constant__ float kHessianChannels32[kHessianEntry * hessian_channel_start(kHessiansFixedLast + 1)];
static __constant__ double kHessianChannels64[kHessianEntry * hessian_channel_start(kHessiansFixedLast + 1)];
template <typename T> __device__ __forceinline__ const T* hessian_channel_table();
template <> __device__ __forceinline__ const float* hessian_channel_table<float>() { return kHessianChannels32; }
template <> __device__ __forceinline__ const double* hessian_channel_table<double>() { return kHessianChannels64; }

// The inputs of entry_job_from (sphx_device.hpp) in registers, for the side of the lane: u stands for c (+m) or s (-m), w for
// -s or c, and the entry is asked for as one with +m.
template <typename T> struct SideWindow {
    T pk_, u_[3], w_[3]; // at m - 2, m - 1, m
    T A_[2], B_[2], C_[3];
    __device__ __forceinline__ T pk() const { return pk_; }
    __device__ __forceinline__ T c(int d) const { return u_[2 + d]; }
    __device__ __forceinline__ T s(int d) const { return -w_[2 + d]; }
    __device__ __forceinline__ T A(int d) const { return A_[d]; }
    __device__ __forceinline__ T B(int d) const { return B_[d]; }
    __device__ __forceinline__ T C(int d) const { return C_[d]; }
};

template <typename T, bool NORM, int L, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 4) void hessians_fixed_kernel(Tiling g, const T* __restrict__ xyz, T* __restrict__ sph,
                                                                    T* __restrict__ dsph, T* __restrict__ ddsph) {
    constexpr unsigned NY = (L + 1) * (L + 1), PAD = gradients_fixed_pad(sizeof(T), NY);
    constexpr int UNITS = hessians_fixed_units(L, WAVES);
    static_assert(UNITS <= 32, "a bit per unit");
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
    static constexpr UnitMasks kMasks = deal_hessian_units(NORM, L, WAVES);
    const unsigned mine = kMasks.of[wave];
    Rows<T> rows;
    rows.ny = static_cast<int>(NY);
    rows.sph = lds + point * (NY + PAD);
    rows.dsph = lds + g.off_dsph + point * (3 * NY + PAD);
    rows.ddsph = lds + g.off_ddsph + point * (9 * NY + PAD);
    if (point < valid) {
        const Point<T> p = load_point<T, NORM>(xyz + (first + point) * 3);
        if ((mine & 1u) != 0 && !minus) closed_form_job<T, 2, NORM, 1>(p, rows);
        if (mine >> 1) {
            // c_m, s_m of the point: u the lane's own (c for +m, s for -m), w the other one with its sign in d/dy
            T u[L + 1], w[L + 1], tz[L];
            {
                T cm = 1.0, sm = 0.0;
                const T twoz = p.z + p.z;
                T t = twoz;
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
                    if (m < L) tz[m] = t;
                    t = t + twoz;
                }
            }
            const T rxy = p.x2 + p.y2;
            for_each_number(std::make_integer_sequence<int, UNITS - 1>{}, [&](auto unit) {
                constexpr int U = 1 + decltype(unit)::value;
                constexpr ChannelPart PART = hessian_part(L, WAVES, U);
                constexpr int l = PART.l;
                if (!((mine >> U) & 1u)) return;
                const T* k = hessian_channel_table<T>() + hessian_channel_start(l) * kHessianEntry;
                // the iterates at m, m + 1, m + 2 of the three recursions (sequence_job)
                T A0 = 0, A1 = 0, A2 = 0, B0 = 0, B1 = 0, B2 = 0, C0 = 0, C1 = 0, C2 = 0;
                for_each_number(std::make_integer_sequence<int, l - PART.m_bottom + 1>{}, [&](auto down) {
                    constexpr int m = l - decltype(down)::value;
                    const T* km = k + m * kHessianEntry;
                    A2 = A1;
                    A1 = A0;
                    B2 = B1;
                    B1 = B0;
                    C2 = C1;
                    C1 = C0;
                    if constexpr (m == l) {
                        A0 = km[0];
                        B0 = 0;
                        C0 = 0;
                    } else if constexpr (m == l - 1) {
                        A0 = -p.z * A1;
                        B0 = km[1];
                        C0 = 0;
                    } else {
                        A0 = km[0] * (tz[m] * A1 + rxy * A2);
                        B0 = km[1] * (tz[m] * B1 + rxy * B2);
                        if constexpr (m == l - 2) C0 = km[2];
                        else C0 = km[2] * (tz[m] * C1 + rxy * C2);
                    }
                    if constexpr (m <= PART.m_top) {
                        SideWindow<T> in;
                        in.pk_ = km[3];
#pragma unroll
                        for (int d = 0; d < 3; ++d) {
                            constexpr int base = m - 2;
                            in.u_[d] = base + d >= 0 ? u[base + d >= 0 ? base + d : 0] : T(0);
                            in.w_[d] = base + d >= 0 ? w[base + d >= 0 ? base + d : 0] : T(0);
                        }
                        in.A_[0] = A0;
                        in.A_[1] = A1;
                        in.B_[0] = B0;
                        in.B_[1] = B1;
                        in.C_[0] = C0;
                        in.C_[1] = C1;
                        in.C_[2] = C2;
                        Rows<T> at = rows;
                        const int back = minus ? -2 * m : 0;
                        at.sph += back;
                        at.dsph += back;
                        at.ddsph += back;
                        if (m > 0 || !minus) entry_job_from<T, 2, NORM, true>(l, m, l * (l + 1) / 2, 0, p, in, at);
                    }
                });
            });
        }
    }
    __syncthreads(); // the rows
    flush_fixed_rows<T, NY, PAD>(lds, sph + first * NY, valid, tid, threads);
    flush_fixed_rows<T, 3 * NY, PAD>(lds + g.off_dsph, dsph + first * 3 * NY, valid, tid, threads);
    flush_fixed_rows<T, 9 * NY, PAD>(lds + g.off_ddsph, ddsph + first * 9 * NY, valid, tid, threads);
}

template <typename T> static hipError_t fill_hessian_channel_table(const HostTables& t) {
    constexpr int last = kHessiansFixedLast;
    const T* F;
    if constexpr (sizeof(T) == 4) F = t.f32.data();
    else F = t.f64.data();
    const T* Q = F + kTableEntries;
    T table[kHessianEntry * hessian_channel_start(last + 1)];
    for (int l = kHessiansFixedFirst; l <= last; ++l) {
        for (int m = 0; m <= l; ++m) {
            T* k = table + (hessian_channel_start(l) + m) * kHessianEntry;
            k[0] = Q[l * (l + 1) / 2 + m];                         // m = l: Q_l^l
            k[1] = m < l ? Q[l * (l - 1) / 2 + m] : T(0);          // m = l - 1: Q_{l-1}^{l-1}
            k[2] = m < l - 1 ? Q[(l - 1) * (l - 2) / 2 + m] : T(0); // m = l - 2: Q_{l-2}^{l-2}
            k[3] = F[l * (l + 1) / 2 + m];
        }
    }
    if constexpr (sizeof(T) == 4) return hipMemcpyToSymbol(HIP_SYMBOL(kHessianChannels32), table, sizeof(table));
    else return hipMemcpyToSymbol(HIP_SYMBOL(kHessianChannels64), table, sizeof(table));
}

template <typename T, bool NORM>
static hipError_t launch_hessians_fixed(const Launch& l, const T* xyz, T* sph, T* dsph, T* ddsph, hipStream_t stream) {
    hipError_t status = hipErrorInvalidValue; // (what hessians_fixed() does not name)
    if (l.threads != 512u && l.threads != 1024u) return status; // never planned
    for_each_number(std::make_integer_sequence<int, hessians_fixed_last(sizeof(T), NORM) - kHessiansFixedFirst + 1>{}, [&](auto i) {
        constexpr int L = kHessiansFixedFirst + decltype(i)::value;
        if (l.g.l_max != L) return;
        auto kernel = l.threads == 512u ? hessians_fixed_kernel<T, NORM, L, 8> : hessians_fixed_kernel<T, NORM, L, 16>;
        if (l.lds_bytes > 64u * 1024u) {
            unsigned unused = 0;
            status = kernel_facts(reinterpret_cast<const void*>(kernel), l.threads, l.lds_bytes, &unused);
            if (status != hipSuccess) return;
        }
        hipLaunchKernelGGL(kernel, dim3(l.workgroups), dim3(l.threads), l.lds_bytes, stream, l.g, xyz, sph, dsph, ddsph);
        status = hipGetLastError();
    });
    return status;
}

template <typename T>
hipError_t dispatch_hessians_fixed(const Launch& l, bool normalized, const T* xyz, T* sph, T* dsph, T* ddsph, hipStream_t stream) {
    return normalized ? launch_hessians_fixed<T, true>(l, xyz, sph, dsph, ddsph, stream)
                      : launch_hessians_fixed<T, false>(l, xyz, sph, dsph, ddsph, stream);
}
template <typename T> hipError_t upload_hessian_channel_tables(const HostTables& t) { return fill_hessian_channel_table<T>(t); }

} // namespace sphx

#endif
