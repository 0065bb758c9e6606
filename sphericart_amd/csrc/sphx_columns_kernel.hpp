// Products with the derivatives of the harmonics, summed column by column: columns_kernel (the vector-Jacobian
// product, and its own derivatives) and column_rows_kernel (the product with gradient and second-derivative arrays).
#ifndef SPHX_COLUMNS_KERNEL_HPP
#define SPHX_COLUMNS_KERNEL_HPP

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "sphx_columns.hpp"
#include "sphx_tiling.hpp"

namespace sphx {

// ---------------------------------------------------------------------------
// The entries (l, +m) and (l, -m) of a point are Q_l^m c_m and Q_l^m s_m times a prefactor F_l^m, and every
// derivative of Q is another Q (sphericart/include/templates_core.hpp:129-133, 219-235, 323-387):
//
//   d/dx Q_l^m = x Q_{l-1}^{m+1}     d/dy Q_l^m = y Q_{l-1}^{m+1}     d/dz Q_l^m = (l+m) Q_{l-1}^m
//
// A sum over all entries with weights w therefore splits, at fixed m, into a few sums over l that do not involve
// x, y, c or s,
//
//   A = sum_l w F Q_l^m        B = sum_l w F Q_{l-1}^{m+1}        C = sum_l w F (l+m) Q_{l-1}^m          (gradients)
//   E = sum_l w F Q_{l-2}^{m+2}  G = sum_l w F (l+m) Q_{l-2}^{m+1}  K = sum_l w F (l+m)(l+m-1) Q_{l-2}^m  (second)
//
// and what depends on x, y, c_m, s_m is applied once per m ("column") instead of once per entry: six (gradients) or
// twelve (second derivatives) multiply-adds per pair of entries instead of 30 or 250 operations. The chain rule of
// the normalised harmonics is linear too and is applied once per point. Second derivatives never exist as numbers.
//
// Q runs upward in l at fixed m. With q_n the iterate at l = m + n over its value at the pole (x = y = 0, z = 1) and
// rho^2 = x^2 + y^2, the recursion of the Gegenbauer polynomials reads
//
//   e_n = (n-1)/(n+2m) (z e_{n-1} - q_{n-2})     q_n = z q_{n-1} + rho^2 e_n     g_n = (n-2)/(n+2m) (z g_{n-1} - e_{n-2})
//
// and e_n, g_n are, but for factors, the neighbouring columns Q_{l-1}^{m+1} and Q_{l-2}^{m+2} that the sums ask for
// anyway: four or six operations per step for all of them, and no weight is read a second time from LDS. Near the axis
// a recursion in z alone has a double root and collects its roundings l^2 times over; rho^2 is a factor of its own
// here, as in the recursion in m of the forward kernels. Error against float64 over that of the float32 arrays
// contracted in float32, root mean square over 1 500 points, normalised, l_max = 8-17: the vector-Jacobian product
// 0.69-0.83 within a tenth of a radian of the axis and 0.79-0.93 anywhere, the second-order products 0.71-0.92 and
// 0.80-0.96 (q_l = z q_{l-1} + b r^2 q_{l-2} with r^2 = 1: 1.4-2.8 and 0.96-1.23). The values at the pole are folded
// into the prefactors on the host (sphx_columns.cpp): |q| <= 1 on the unit sphere. m is the same for all lanes of a
// wave, so the table comes from the scalar unit.
//
// The products are sums in another order than the entries' own, with fused multiply-adds: they agree with the
// contraction of the derivative arrays to rounding.
//
// LMAX > 0: kernels for one l_max each (fixed_columns(), sphx_columns.hpp), the same operations in the same order within a
// wave; where the columns are dealt to another number of waves than in the general kernel (the product in float32 at l_max =
// 10, its derivatives at 3), the waves' sums are as many fewer or more, added in that other order: rounding of the same width.
// What the general kernel is bound by is the issue of instructions and, in small calls, the wait at every step: per step it
// loads the entry's factors through the scalar unit and the weights from LDS, which share a counter, and waits for both. With
// l_max a constant a column is one run of instructions, the loads of several steps ahead, the offsets of the weights part of
// the instructions, and the rows come into LDS without a branch between the loads (SQ counters, general / fixed, e6: the
// product, 400 003 points, float32 l_max = 8, vector 8.6 6.3, scalar 8.5 2.3; 100 000 points at 17, 10.0 8.4, 8.5 1.4). The
// derivatives of the product in float64 at l_max = 11 and 12 on two lanes per point spill 2-9 vector registers. us, general and fixed: the product, 400 000 points, float32
// l_max = 8 27.3 22.5 (floor 20.2), 12 56 43 (41), 17 134 101 (77), float64 8 50 42 (40), 12 130 106 (81), 20 000 points
// at 14 in float32 8.8 5.1; its derivatives, float32 8 51.6 43.9 (39.7), float64 10 169 147 (116); the rows, float32 8 144
// 108 (77), float64 9 295 236 (177), 20 000 points 22.9 18.2.
// ---------------------------------------------------------------------------

__device__ __forceinline__ float fma_of(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fma_of(double a, double b, double c) { return __builtin_fma(a, b, c); }

template <typename T> __device__ __forceinline__ const T* column_table();
static __constant__ float kColumns32[kColumnEntries * kColumnEntry];
static __constant__ double kColumns64[kColumnEntries * kColumnEntry];
template <> __device__ __forceinline__ const float* column_table<float>() { return kColumns32; }
template <> __device__ __forceinline__ const double* column_table<double>() { return kColumns64; }

// Walks l = m .. L of column m and hands visit(step, l, FA, FB, FC, FE, FG, FK) the products of the prefactors with
// the six Q above. `step` is l - m as a compile-time number while that is below 5 and 5 from there on: what is zero
// or one by construction in the first steps takes no instruction (FB is meaningful from step 2 on, FC 1, FE 4, FG 3,
// FK 2). rho2 = x^2 + y^2.
template <int... I, typename F> __host__ __device__ __forceinline__ void each_of(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}

// LMAX > 0: m and L = LMAX are compile-time numbers (m an integral_constant), and the column is one run of
// instructions without a branch.
template <typename T, bool SECOND, int LMAX, typename M, typename Visit>
__device__ __forceinline__ void walk_column(M m, int L, T z, T rho2, Visit&& visit) {
    const T* t = column_table<T>() + column_start(m) * kColumnEntry;
    T q1 = 0, q2 = 0, e1 = 0, e2 = 0, g1 = 0;
    auto one = [&](auto step, auto l) {
        constexpr int S = decltype(step)::value;
        const T* k = t;
        t += kColumnEntry;
        T q = 1, e = 0, g = 0;
        if constexpr (S == 2) e = -k[0];
        else if constexpr (S >= 3) e = k[0] * fma_of(z, e1, -q2);
        if constexpr (SECOND) {
            if constexpr (S == 4) g = -k[4] * e2;
            else if constexpr (S >= 5) g = k[4] * fma_of(z, g1, -e2);
        }
        if constexpr (S == 1) q = z;
        else if constexpr (S >= 2) q = fma_of(rho2, e, z * q1);
        T fa = k[1], fb = 0, fc = 0, fe = 0, fg = 0, fk = 0;
        if constexpr (S >= 1) fa *= q;
        if constexpr (S >= 1) fc = k[3];
        if constexpr (S >= 2) fc *= q1;
        if constexpr (S >= 2) fb = k[2] * e;
        if constexpr (SECOND) {
            if constexpr (S >= 2) fk = k[7];
            if constexpr (S >= 3) fk *= q2;
            if constexpr (S >= 3) fg = k[6] * e1;
            if constexpr (S >= 4) fe = k[5] * g;
        }
        visit(step, l, fa, fb, fc, fe, fg, fk);
        q2 = q1;
        q1 = q;
        e2 = e1;
        e1 = e;
        g1 = g;
    };
    using std::integral_constant;
    if constexpr (LMAX > 0) {
        each_of(std::make_integer_sequence<int, LMAX - M::value + 1>{}, [&](auto n) {
            constexpr int N = decltype(n)::value;
            one(integral_constant<int, (N < 5 ? N : 5)>{}, integral_constant<int, M::value + N>{});
        });
        return;
    }
    one(integral_constant<int, 0>{}, static_cast<int>(m));
    if (m + 1 > L) return;
    one(integral_constant<int, 1>{}, m + 1);
    if (m + 2 > L) return;
    one(integral_constant<int, 2>{}, m + 2);
    if (m + 3 > L) return;
    one(integral_constant<int, 3>{}, m + 3);
    if (m + 4 > L) return;
    one(integral_constant<int, 4>{}, m + 4);
#pragma unroll 2
    for (int l = m + 5; l <= L; ++l) one(integral_constant<int, 5>{}, l);
}

// The sums of one column and one side (entries (l, +m) or (l, -m)).
template <typename T> struct ColumnSums {
    T A = 0, B = 0, C = 0, E = 0, G = 0, K = 0;

    template <int S, bool SECOND>
    __device__ __forceinline__ void add(T w, T fa, T fb, T fc, T fe, T fg, T fk) {
        A = fma_of(w, fa, A);
        if constexpr (S >= 2) B = fma_of(w, fb, B);
        if constexpr (S >= 1) C = fma_of(w, fc, C);
        if constexpr (SECOND) {
            if constexpr (S >= 4) E = fma_of(w, fe, E);
            if constexpr (S >= 3) G = fma_of(w, fg, G);
            if constexpr (S >= 2) K = fma_of(w, fk, K);
        }
    }
};

// c_m, s_m of a lane's point, walked upward in m; kept with their two predecessors.
template <typename T> struct Azimuth {
    T c = 1, s = 0, c1 = 0, s1 = 0, c2 = 0, s2 = 0;
    __device__ __forceinline__ void next(T x, T y) {
        c2 = c1;
        s2 = s1;
        c1 = c;
        s1 = s;
        const T cn = fma_of(c1, x, -(s1 * y));
        s = fma_of(c1, y, s1 * x);
        c = cn;
    }
};

// What the columns of a point add up to, with x and y still factored out. u stands for c_m (entries +m) or s_m (-m),
// u1 for c_{m-1} or s_{m-1}, w1 for -s_{m-1} or c_{m-1}, and so on one order down.
template <typename T, bool SECOND> struct PointSums {
    T Bu = 0, Cu = 0, A1 = 0, Aw = 0;
    T B1 = 0, Bw = 0, C1 = 0, Cw = 0, A2 = 0, Aw2 = 0, Eu = 0, Gu = 0, Ku = 0;

    __device__ __forceinline__ void add(const ColumnSums<T>& k, T fm, T u, T u1, T w1, T u2, T w2) {
        const T p1 = fm * u1, q1 = fm * w1;
        Bu = fma_of(k.B, u, Bu);
        Cu = fma_of(k.C, u, Cu);
        A1 = fma_of(k.A, p1, A1);
        Aw = fma_of(k.A, q1, Aw);
        if constexpr (SECOND) {
            const T fmm = fm * (fm - 1);
            B1 = fma_of(k.B, p1, B1);
            Bw = fma_of(k.B, q1, Bw);
            C1 = fma_of(k.C, p1, C1);
            Cw = fma_of(k.C, q1, Cw);
            A2 = fma_of(k.A, fmm * u2, A2);
            Aw2 = fma_of(k.A, fmm * w2, Aw2);
            Eu = fma_of(k.E, u, Eu);
            Gu = fma_of(k.G, u, Gu);
            Ku = fma_of(k.K, u, Ku);
        }
    }
    __device__ __forceinline__ void add_plus(const ColumnSums<T>& k, T fm, const Azimuth<T>& z) {
        add(k, fm, z.c, z.c1, -z.s1, z.c2, -z.s2);
    }
    __device__ __forceinline__ void add_minus(const ColumnSums<T>& k, T fm, const Azimuth<T>& z) {
        add(k, fm, z.s, z.s1, z.c1, z.s2, z.c2);
    }
    __device__ __forceinline__ T gx(T x) const { return fma_of(x, Bu, A1); }
    __device__ __forceinline__ T gy(T y) const { return fma_of(y, Bu, Aw); }
    __device__ __forceinline__ T gz() const { return Cu; }
    __device__ __forceinline__ T xx(T x) const { return fma_of(x, fma_of(x, Eu, 2 * B1), Bu + A2); }
    __device__ __forceinline__ T yy(T y) const { return fma_of(y, fma_of(y, Eu, 2 * Bw), Bu - A2); }
    __device__ __forceinline__ T xy(T x, T y) const { return fma_of(y, fma_of(x, Eu, B1), fma_of(x, Bw, Aw2)); }
    __device__ __forceinline__ T xz(T x) const { return fma_of(x, Gu, C1); }
    __device__ __forceinline__ T yz(T y) const { return fma_of(y, Gu, Cw); }
    __device__ __forceinline__ T zz() const { return Ku; }
};

// ---------------------------------------------------------------------------
// One entry at a time, for points whose sums are not finite: an infinite weight (or one so large that a sum over a
// column overflows) makes the sums of its column infinite, and what is then multiplied by s_0 = 0 or projected on the
// tangent plane a NaN in all components. Entry by entry such a point gets what contracting the arrays gives: an infinite
// number where the entry's derivative is not zero, and a NaN where it is. The test costs a call 0.05 to 0.1 us (the product
// in small calls 1-2 %; with the entries' part in front of the stores, or with the registers it would like, 3-4 %).
// ---------------------------------------------------------------------------
template <typename T, bool NORM, bool SECOND> struct EntryDerivatives {
    T d[3];    // gradient
    T h[3][3]; // second derivatives

    // (the chain rule of the normalised harmonics, templates.hpp:572-613, product by product as the arrays have it)
    __device__ __forceinline__ EntryDerivatives(const PointSums<T, SECOND>& one, const Point<T>& p) {
        d[0] = one.gx(p.x);
        d[1] = one.gy(p.y);
        d[2] = one.gz();
        if constexpr (SECOND) {
            h[0][0] = one.xx(p.x);
            h[1][1] = one.yy(p.y);
            h[2][2] = one.zz();
            h[0][1] = h[1][0] = one.xy(p.x, p.y);
            h[0][2] = h[2][0] = one.xz(p.x);
            h[1][2] = h[2][1] = one.yz(p.y);
        }
        if constexpr (NORM) {
            const T n[3] = {p.x, p.y, p.z};
            const T along = d[0] * n[0] + d[1] * n[1] + d[2] * n[2];
            if constexpr (SECOND) {
                T hn[3];
#pragma unroll
                for (int a = 0; a < 3; ++a) hn[a] = n[0] * h[a][0] + n[1] * h[a][1] + n[2] * h[a][2];
                const T nhn = n[0] * hn[0] + n[1] * hn[1] + n[2] * hn[2];
                const T irsq = p.ir * p.ir;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
#pragma unroll
                    for (int b = a; b < 3; ++b) {
                        const T both = n[a] * n[b];
                        T of = h[a][b] - n[a] * (hn[b] + d[b]) - n[b] * (hn[a] + d[a]) + both * (3 * along + nhn);
                        if (a == b) of -= along;
                        h[a][b] = h[b][a] = of * irsq;
                    }
                }
            }
#pragma unroll
            for (int a = 0; a < 3; ++a) d[a] = (d[a] - n[a] * along) * p.ir;
        }
    }
};

// visit(k, derivatives) for all entries k = l (l + 1) +- m.
template <typename T, bool NORM, bool SECOND, typename Visit>
__device__ __forceinline__ void each_entry(int L, Point<T> p, Visit&& visit) {
    const T rho2 = p.x2 + p.y2;
    Azimuth<T> azimuth;
#pragma unroll 1
    for (int m = 0; m <= L; ++m) {
        if (m > 0) azimuth.next(p.x, p.y);
        const T* k = column_table<T>() + column_start(m) * kColumnEntry;
        T q1 = 0, q2 = 0, e1 = 0, e2 = 0, g1 = 0;
#pragma unroll 1
        for (int l = m; l <= L; ++l, k += kColumnEntry) { // (the table has zeros where walk_column takes steps apart)
            const T e = k[0] * fma_of(p.z, e1, -q2);
            const T g = k[4] * fma_of(p.z, g1, -e2);
            const T q = l == m ? T(1) : fma_of(rho2, e, p.z * q1);
            ColumnSums<T> sums;
            sums.A = k[1] * q;
            sums.B = k[2] * e;
            sums.C = k[3] * q1;
            if constexpr (SECOND) {
                sums.E = k[5] * g;
                sums.G = k[6] * e1;
                sums.K = k[7] * q2;
            }
#pragma unroll 1
            for (int side = 0; side < (m > 0 ? 2 : 1); ++side) {
                // (keeps the products of the coordinates from being formed ahead of the loops: 28 registers in float64)
                asm volatile("" : "+v"(p.x), "+v"(p.y), "+v"(p.z), "+v"(p.ir));
                PointSums<T, SECOND> one;
                if (side == 0) one.add_plus(sums, static_cast<T>(m), azimuth);
                else one.add_minus(sums, static_cast<T>(m), azimuth);
                visit(l * (l + 1) + (side == 0 ? m : -m), EntryDerivatives<T, NORM, SECOND>(one, p));
            }
            q2 = q1;
            q1 = q;
            e2 = e1;
            e1 = e;
            g1 = g;
        }
    }
}

// an infinity or a NaN among three numbers: three comparisons
__device__ __forceinline__ bool lost_one(float a, float b, float c) {
    return __builtin_amdgcn_classf(a, 0x207) | __builtin_amdgcn_classf(b, 0x207) | __builtin_amdgcn_classf(c, 0x207);
}
__device__ __forceinline__ bool lost_one(double a, double b, double c) {
    return __builtin_amdgcn_class(a, 0x207) | __builtin_amdgcn_class(b, 0x207) | __builtin_amdgcn_class(c, 0x207);
}
template <typename T> __device__ __forceinline__ bool is_number(const Point<T>& p) { // (at the origin every entry is a NaN)
    return p.x == p.x && p.y == p.y && p.z == p.z;
}

// Column after column to wave after wave, the direction changing every time round: the longest columns come first.
struct Deal {
    unsigned waves, at = 0;
    bool down = false;
    __device__ __forceinline__ explicit Deal(unsigned n) : waves(n) {}
    __device__ __forceinline__ bool next(unsigned wave) {
        const unsigned owner = down ? waves - 1u - at : at;
        if (++at == waves) {
            at = 0;
            down = !down;
        }
        return owner == wave;
    }
};

// The same deal as a bit per column.
__device__ __forceinline__ unsigned columns_of(unsigned wave, unsigned waves, int l_max) {
    const unsigned period = 2u * waves, both = (1u << wave) | (1u << (period - 1u - wave));
    unsigned mine = 0;
    for (unsigned at = 0; at <= static_cast<unsigned>(l_max); at += period) mine |= both << at;
    return mine;
}

// `len` consecutive elements of HBM, rows of `row` elements, to LDS with the rows `row + pad` apart. pad is 0 or, for
// even rows (a multiple of 16 bytes then), 1, so that the rows of the points start on different banks. `magic` =
// magic_of(row in 16-byte vectors). Many 16-byte loads in flight per lane: a tile is read once, and its latency is
// most of what a workgroup would otherwise wait for.
template <typename T>
__device__ __forceinline__ void rows_to_lds(const T* __restrict__ run, T* staged, unsigned len, unsigned row, unsigned pad,
                                            unsigned magic, unsigned tid, unsigned threads) {
    using V = typename Pack<T>::type;
    constexpr unsigned W = Pack<T>::width;
    if ((reinterpret_cast<uintptr_t>(run) & 15u) != 0) {
        for (unsigned e = tid; e < len; e += threads) staged[e + pad * (e / row)] = run[e];
        return;
    }
    const V* in = reinterpret_cast<const V*>(run);
    const unsigned nvec = len / W;
    auto put = [&](unsigned at, V v) {
        if (pad == 0) {
            reinterpret_cast<V*>(staged)[at] = v;
        } else {
            T* to = staged + at * W + __umulhi(at, magic);
#pragma unroll
            for (unsigned e = 0; e < W; ++e) to[e] = v[e];
        }
    };
    constexpr unsigned DEPTH = 8;
    unsigned v = tid;
    for (; v + (DEPTH - 1) * threads < nvec; v += DEPTH * threads) {
        V hold[DEPTH];
#pragma unroll
        for (unsigned u = 0; u < DEPTH; ++u) hold[u] = in[v + u * threads];
#pragma unroll
        for (unsigned u = 0; u < DEPTH; ++u) put(v + u * threads, hold[u]);
    }
    {
        // the rest, fewer than DEPTH vectors per lane: all of them in flight as well
        V hold[DEPTH];
#pragma unroll
        for (unsigned u = 0; u < DEPTH; ++u) {
            if (v + u * threads < nvec) hold[u] = in[v + u * threads];
        }
#pragma unroll
        for (unsigned u = 0; u < DEPTH; ++u) {
            if (v + u * threads < nvec) put(v + u * threads, hold[u]);
        }
    }
    for (unsigned e = nvec * W + tid; e < len; e += threads) staged[e + pad * (e / row)] = run[e]; // pad == 0 here
}

// The same with the rows' length and pad compile-time numbers and without a branch between the loads: issue() sends the
// loads of ROUNDS vectors per lane, put() stores them, then the next ROUNDS. A lane that has run out of vectors loads and
// stores the last one once more.
template <typename T, unsigned ROW, unsigned PAD, unsigned ROUNDS> struct FixedRows {
    using V = typename Pack<T>::type;
    static constexpr unsigned W = Pack<T>::width;
    static_assert(ROW >= W && (PAD == 0 || ROW % W == 0), "padded rows are whole vectors");
    const T* __restrict__ run;
    T* staged;
    unsigned len, threads, last, at;
    bool vectors;
    V hold[ROUNDS];
    __device__ __forceinline__ FixedRows(const T* run_, T* staged_, unsigned points, unsigned tid, unsigned threads_)
        : run(run_), staged(staged_), len(points * ROW), threads(threads_), last(points * ROW / W - 1u), at(tid),
          vectors((reinterpret_cast<uintptr_t>(run_) & 15u) == 0) {}
    __device__ __forceinline__ unsigned clamped(unsigned u) const {
        const unsigned v = at + u * threads;
        return v < last ? v : last;
    }
    __device__ __forceinline__ void issue() {
        if (!vectors) return;
#pragma unroll
        for (unsigned u = 0; u < ROUNDS; ++u) hold[u] = reinterpret_cast<const V*>(run)[clamped(u)];
    }
    __device__ __forceinline__ void put() {
        if (!vectors) return;
#pragma unroll
        for (unsigned u = 0; u < ROUNDS; ++u) {
            const unsigned v = clamped(u);
            if constexpr (PAD == 0) {
                reinterpret_cast<V*>(staged)[v] = hold[u];
            } else {
                T* to = staged + v * W + PAD * (v / (ROW / W));
#pragma unroll
                for (unsigned e = 0; e < W; ++e) to[e] = hold[u][e];
            }
        }
        at += ROUNDS * threads;
    }
    // what the first issue() and put() have left
    __device__ __forceinline__ void rest(unsigned tid) {
        if (!vectors) {
            for (unsigned e = tid; e < len; e += threads) staged[e + PAD * (e / ROW)] = run[e];
            return;
        }
        while (at - tid <= last) { // (the same for all lanes)
            issue();
            put();
        }
        for (unsigned e = (last + 1u) * W + tid; e < len; e += threads) staged[e] = run[e]; // PAD == 0 here
    }
};

// Waves per SIMD that the registers are to allow: what the sums need by themselves. (The compiler allots registers for
// the whole kernel, and the entry by entry part, which hardly ever runs, would take a wave from each.)
template <typename T, bool NORM, bool SECOND, int GROUPS, int LMAX> constexpr int columns_residence() {
    if (LMAX > 0) return sizeof(T) == 4 ? (SECOND ? 5 : 6) : (SECOND ? 3 : 4); // (a column's loads are under way together)
    if (sizeof(T) == 8 && SECOND) return NORM ? 3 : 4;
    return SECOND && NORM && GROUPS == 2 ? 6 : 7;
}

// ---------------------------------------------------------------------------
// columns_kernel: one point per lane (GROUPS == 1, 64 points per workgroup) or per pair of lanes (GROUPS == 2, 32
// points, one lane for the entries +m and one for -m). The tile's rows of weights pass through LDS, read from HBM with
// consecutive lanes at consecutive addresses; the columns m are dealt to the waves, longest first in both
// directions, and every wave walks c_m, s_m along for itself.
//
// SECOND == false: the vector-Jacobian product  out[i][a] (+)= sum_k dsph[i][a][k] w[i][k].
// SECOND == true: its derivatives, for a backward pass through it with the upstream gradient `grad` [n][3]:
//   out[i][b]  = sum_a grad[i][a] sum_k w[i][k] d^2 sph[i][k] / dx_a dx_b
//   dw[i][k]   = sum_a grad[i][a] dsph[i][a][k]
// dw replaces w in LDS entry by entry and leaves as one contiguous run.
//
// With n = x/r, P = 1 - n n^T, h = sum w grad R(n) and H = sum w hess R(n) of the polynomials R the chain rule
// (sphericart/include/templates.hpp:572-613) summed over the entries and applied to g reads
//   out = (P (H g' - a h) - t g' - n (h . g')) / r^2,   g' = P g, a = n . g, t = n . h,
// and dw = (g' / r) . grad R.
// ---------------------------------------------------------------------------
template <typename T, bool NORM, bool SECOND, int GROUPS, bool ADD, int LMAX = 0>
__global__ __launch_bounds__(kColumnsThreads, (columns_residence<T, NORM, SECOND, GROUPS, LMAX>())) void columns_kernel(Columns g, const T* __restrict__ xyz, const T* __restrict__ weights,
                                                     const T* __restrict__ grad, T* __restrict__ out,
                                                     T* __restrict__ dw) {
    constexpr unsigned TILE = 64 / GROUPS;
    T* lds = reinterpret_cast<T*>(lds_raw);
    const unsigned tid = threadIdx.x;
    const unsigned lane = tid & 63u;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6); // the same for all lanes: scalar
    const unsigned threads = blockDim.x;
    const unsigned waves = threads >> 6;
    const int L = LMAX > 0 ? LMAX : g.l_max;
    const unsigned ny = LMAX > 0 ? (LMAX + 1) * (LMAX + 1) : g.ny;
    const unsigned pad = LMAX > 0 ? columns_pad(sizeof(T), ny) : g.pad, stride = ny + pad;
    // consecutive workgroups go to the XCDs in turn: one contiguous stretch of tiles for each
    const unsigned group = (blockIdx.x & 7u) * g.tiles_per_xcd + (blockIdx.x >> 3);
    if (group >= g.n_tiles) return;
    const unsigned long long first = static_cast<unsigned long long>(group) * TILE;
    const unsigned long long left = g.n_samples - first;
    const unsigned valid = left < TILE ? static_cast<unsigned>(left) : TILE;
    const unsigned point = lane & (TILE - 1u);
    const bool minus = GROUPS == 2 && lane >= TILE;

    // lanes past the last point compute on the first one's coordinates and write nothing
    const unsigned mine = point < valid ? point : 0u;
    xyz += first * 3;
    out += first * 3;
    if constexpr (SECOND) grad += first * 3;
    Point<T> p;
    if constexpr (LMAX > 0) {
        constexpr unsigned ROW = (LMAX + 1) * (LMAX + 1);
        constexpr int KIND = SECOND ? COLUMNS_VJP_BACKWARD : COLUMNS_VJP;
        // (all loads of the tile under way before the first is waited for)
        const T raw[3] = {xyz[mine * 3u], xyz[mine * 3u + 1u], xyz[mine * 3u + 2u]};
        FixedRows<T, ROW, columns_pad(sizeof(T), ROW), column_rounds(KIND, sizeof(T), LMAX, TILE * ROW)> rows(
            weights + first * ny, lds, valid, tid, threads);
        rows.issue();
        p = load_point<T, NORM>(raw);
        rows.put();
        rows.rest(tid);
    } else {
        rows_to_lds<T>(weights + first * ny, lds, valid * ny, ny, g.pad, g.magic_vectors, tid, threads);
        p = load_point<T, NORM>(xyz + mine * 3u);
    }
    T gx = 0, gy = 0, gz = 0, along = 0;
    bool lost_grad = false; // any of the tile's
    if constexpr (SECOND) {
        gx = grad[mine * 3u];
        gy = grad[mine * 3u + 1u];
        gz = grad[mine * 3u + 2u];
        lost_grad = __any(lost_one(gx, gy, gz));
        if constexpr (NORM) {
            along = fma_of(gx, p.x, fma_of(gy, p.y, gz * p.z));
            gx = fma_of(-along, p.x, gx);
            gy = fma_of(-along, p.y, gy);
            gz = fma_of(-along, p.z, gz);
        }
    }
    const T rho2 = p.x2 + p.y2;
    // the direction of dw, the chain rule's 1/r included
    const T scale = NORM ? p.ir : T(1);
    const T dx = gx * scale, dy = gy * scale, dz = gz * scale;
    const T radial = fma_of(dx, p.x, dy * p.y);
    __syncthreads(); // weights

    PointSums<T, SECOND> sums;
    Azimuth<T> azimuth;
    T* row = lds + point * stride;
    auto column = [&](auto m) {
        const T fm = static_cast<T>(static_cast<int>(m));
        if constexpr (GROUPS == 1) {
            ColumnSums<T> plus, neg;
            T along_plus = 0, along_minus = 0;
            if constexpr (SECOND) {
                along_plus = fm * fma_of(dx, azimuth.c1, -(dy * azimuth.s1));
                along_minus = fm * fma_of(dx, azimuth.s1, dy * azimuth.c1);
            }
            walk_column<T, SECOND, LMAX>(m, L, p.z, rho2, [&](auto step, auto l, T fa, T fb, T fc, T fe, T fg, T fk) {
                constexpr int S = decltype(step)::value;
                T* mid = row + l * (l + 1);
                const T wp = mid[m], wn = mid[-m];
                plus.template add<S, SECOND>(wp, fa, fb, fc, fe, fg, fk);
                neg.template add<S, SECOND>(wn, fa, fb, fc, fe, fg, fk);
                if constexpr (SECOND) {
                    T q = 0;
                    if constexpr (S >= 1) q = dz * fc;
                    if constexpr (S >= 2) q = fma_of(radial, fb, q);
                    // (m = 0: both are the same entry, the second store is the one that counts)
                    mid[-m] = fma_of(q, azimuth.s, fa * along_minus);
                    mid[m] = fma_of(q, azimuth.c, fa * along_plus);
                }
            });
            sums.add_plus(plus, fm, azimuth);
            sums.add_minus(neg, fm, azimuth);
        } else {
            const T u = minus ? azimuth.s : azimuth.c;
            const T u1 = minus ? azimuth.s1 : azimuth.c1, w1 = minus ? azimuth.c1 : -azimuth.s1;
            const T u2 = minus ? azimuth.s2 : azimuth.c2, w2 = minus ? azimuth.c2 : -azimuth.s2;
            ColumnSums<T> k;
            const T along_u = SECOND ? fm * fma_of(dx, u1, dy * w1) : T(0);
            const bool writes = m > 0 || !minus; // (m = 0 is one entry)
            T* at = row + (minus ? -m : m);
            walk_column<T, SECOND, LMAX>(m, L, p.z, rho2, [&](auto step, auto l, T fa, T fb, T fc, T fe, T fg, T fk) {
                constexpr int S = decltype(step)::value;
                T* here = at + l * (l + 1);
                k.template add<S, SECOND>(*here, fa, fb, fc, fe, fg, fk);
                if constexpr (SECOND) {
                    T q = 0;
                    if constexpr (S >= 1) q = dz * fc;
                    if constexpr (S >= 2) q = fma_of(radial, fb, q);
                    if (writes) *here = fma_of(q, u, fa * along_u);
                }
            });
            sums.add(k, fm, u, u1, w1, u2, w2);
        }
    };
    if constexpr (LMAX > 0) {
        const unsigned mine = columns_of(wave, waves, LMAX);
        each_of(std::make_integer_sequence<int, LMAX + 1>{}, [&](auto m) {
            if constexpr (m.value > 0) azimuth.next(p.x, p.y);
            if ((mine >> m.value) & 1u) column(m);
        });
    } else {
        Deal deal(waves);
        for (int m = 0; m <= L; ++m) {
            if (m > 0) azimuth.next(p.x, p.y);
            if (deal.next(wave)) column(m);
        }
    }

    // h, and H g': the two lanes of a point, then the waves, are added up
    constexpr unsigned NS = SECOND ? 6 : 3;
    T total[NS];
    total[0] = sums.gx(p.x);
    total[1] = sums.gy(p.y);
    total[2] = sums.gz();
    if constexpr (SECOND) {
        const T hxy = sums.xy(p.x, p.y), hxz = sums.xz(p.x), hyz = sums.yz(p.y);
        total[3] = fma_of(sums.xx(p.x), gx, fma_of(hxy, gy, hxz * gz));
        total[4] = fma_of(hxy, gx, fma_of(sums.yy(p.y), gy, hyz * gz));
        total[5] = fma_of(hxz, gx, fma_of(hyz, gy, sums.zz() * gz));
    }
    if constexpr (GROUPS == 2) {
#pragma unroll
        for (unsigned i = 0; i < NS; ++i) total[i] += __shfl_xor(total[i], 32);
    }
    T* partial = lds + g.off_sums;
    bool lost = false;
    if (!SECOND && waves > 1) __syncthreads(); // the sums take the place of the weights
    if (wave != 0) {
#pragma unroll
        for (unsigned i = 0; i < NS; ++i) partial[((wave - 1u) * NS + i) * 64u + lane] = total[i];
    }
    if (waves > 1 || SECOND) __syncthreads(); // the waves' sums, and every entry of dw
    if (wave == 0) {
        for (unsigned w = 0; w + 1 < waves; ++w) {
#pragma unroll
            for (unsigned i = 0; i < NS; ++i) total[i] += partial[(w * NS + i) * 64u + lane];
        }
        T ox = total[0], oy = total[1], oz = total[2];
        if constexpr (SECOND) {
            ox = total[3];
            oy = total[4];
            oz = total[5];
        }
        if constexpr (NORM) {
            const T hx = total[0], hy = total[1], hz = total[2];
            if constexpr (SECOND) {
                ox = fma_of(-along, hx, ox);
                oy = fma_of(-along, hy, oy);
                oz = fma_of(-along, hz, oz);
            }
            const T inward = fma_of(ox, p.x, fma_of(oy, p.y, oz * p.z));
            ox = fma_of(-inward, p.x, ox);
            oy = fma_of(-inward, p.y, oy);
            oz = fma_of(-inward, p.z, oz);
            if constexpr (SECOND) {
                const T t = fma_of(hx, p.x, fma_of(hy, p.y, hz * p.z));
                const T hg = fma_of(hx, gx, fma_of(hy, gy, hz * gz));
                ox = fma_of(-t, gx, fma_of(-hg, p.x, ox)) * p.ir;
                oy = fma_of(-t, gy, fma_of(-hg, p.y, oy)) * p.ir;
                oz = fma_of(-t, gz, fma_of(-hg, p.z, oz)) * p.ir;
            }
            ox *= p.ir;
            oy *= p.ir;
            oz *= p.ir;
        }
        if (point < valid && !minus) {
            T* to = out + mine * 3u;
            lost = lost_one(ox, oy, oz);
            if constexpr (ADD) {
                if (!lost) { // (lost: added below, to what is there)
                    to[0] += ox;
                    to[1] += oy;
                    to[2] += oz;
                }
            } else {
                to[0] = ox;
                to[1] = oy;
                to[2] = oz;
            }
        }
    }
    if constexpr (SECOND) {
        if (pad == 0) {
            copy_out<T, SPHX_STREAMING_STORES, false>(lds, dw + first * ny, valid * ny, ny, 0, 0, tid, threads);
        } else {
            copy_out<T, SPHX_STREAMING_STORES, true>(lds, dw + first * ny, valid * ny, ny, pad, g.magic_ny, tid, threads);
        }
    }
    if constexpr (SECOND) {
        // (the same in all waves, each of which has all points of the tile: dw is written once more, after the flush)
        if (__builtin_expect(lost_grad, 0)) {
            __threadfence();
            __syncthreads();
        }
    }
    if (__builtin_expect(lost, 0)) {
        const Point<T> q = load_point<T, NORM>(xyz + mine * 3u);
        const T* w = weights + (first + mine) * ny;
        const T* u = SECOND ? grad + mine * 3u : nullptr;
        volatile T* to = out + mine * 3u; // (summed in memory: registers here would be paid for by every call)
        if (!ADD || !is_number(q)) {     // (at the origin every entry is a NaN)
            to[0] = is_number(q) ? T(0) : q.x;
            to[1] = is_number(q) ? T(0) : q.y;
            to[2] = is_number(q) ? T(0) : q.z;
        }
        if (is_number(q)) {
            each_entry<T, NORM, SECOND>(L, q, [&](int k, const EntryDerivatives<T, NORM, SECOND>& of) {
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    if constexpr (SECOND) {
                        to[b] = to[b] + (of.h[0][b] * (u[0] * w[k]) + of.h[1][b] * (u[1] * w[k]) + of.h[2][b] * (u[2] * w[k]));
                    } else {
                        to[b] = to[b] + of.d[b] * w[k];
                    }
                }
                if constexpr (SECOND) {
                    if (lost_one(u[0], u[1], u[2])) dw[(first + mine) * ny + k] = u[0] * of.d[0] + u[1] * of.d[1] + u[2] * of.d[2];
                }
            });
        }
    }
}

// ---------------------------------------------------------------------------
// column_rows_kernel: the backward pass from values and gradients,
//
//   out[i][b] = sum_k w[i][k] dsph[i][b][k] + sum_a sum_k v[i][a][k] ddsph[i][a][b][k],
//
// w (may be null) the upstream gradient of the values, v [n][3][ny] that of the gradients. Four rows of weights per
// point fill LDS four times as fast, so a point has four lanes and a tile 16 points: a lane takes one side (+m or -m)
// and two of the four sets of weights, (x, y) or (z, values), and all lanes run the same instructions.
//
// Normalised: with s = n . v_k per entry, p = v_k - n s and the polynomials' d = grad R_k, H = hess R_k, the chain rule
// summed over the entries is
//   out = (P sum_k (H p + (w r - s) d) - sum_k (n . d) p - n sum_k d . p) / r^2,
// and n . d = l R_k (R_k is homogeneous of degree l): the sets are p_x, p_y, p_z and w r - s, and one more sum per set,
// of l w F Q, serves the second term.
// ---------------------------------------------------------------------------
template <typename T, bool NORM, int LMAX = 0>
__global__ __launch_bounds__(kColumnsThreads) void column_rows_kernel(Columns g, const T* __restrict__ xyz, const T* __restrict__ w,
                                                         const T* __restrict__ v, T* __restrict__ out) {
    constexpr unsigned TILE = 16;
    T* lds = reinterpret_cast<T*>(lds_raw);
    const unsigned tid = threadIdx.x;
    const unsigned lane = tid & 63u;
    const unsigned wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned threads = blockDim.x;
    const unsigned waves = threads >> 6;
    const int L = LMAX > 0 ? LMAX : g.l_max;
    const unsigned ny = LMAX > 0 ? (LMAX + 1) * (LMAX + 1) : g.ny;
    const unsigned pad = LMAX > 0 ? columns_pad(sizeof(T), ny) : g.pad, w_stride = ny + pad, v_stride = 3u * ny + pad;
    const unsigned group = (blockIdx.x & 7u) * g.tiles_per_xcd + (blockIdx.x >> 3);
    if (group >= g.n_tiles) return;
    const unsigned long long first = static_cast<unsigned long long>(group) * TILE;
    const unsigned long long left = g.n_samples - first;
    const unsigned valid = left < TILE ? static_cast<unsigned>(left) : TILE;
    const unsigned point = lane & (TILE - 1u);
    const bool minus = (lane & 16u) != 0;
    const bool second_half = lane >= 32u; // the sets z and values
    const bool have_w = w != nullptr;

    T* w_rows = lds + g.off_rows;
    const unsigned mine = point < valid ? point : 0u;
    xyz += first * 3;
    out += first * 3;
    Point<T> p;
    auto no_weights = [&]() {
        for (unsigned e = tid; e < TILE * w_stride; e += threads) w_rows[e] = 0;
    };
    if constexpr (LMAX > 0) {
        constexpr unsigned ROW = (LMAX + 1) * (LMAX + 1), PAD = columns_pad(sizeof(T), ROW);
        const T raw[3] = {xyz[mine * 3u], xyz[mine * 3u + 1u], xyz[mine * 3u + 2u]};
        FixedRows<T, 3u * ROW, PAD, column_rounds(COLUMNS_ROWS, sizeof(T), LMAX, TILE * 3u * ROW)> three(
            v + first * 3u * ny, lds, valid, tid, threads);
        FixedRows<T, ROW, PAD, column_rounds(COLUMNS_ROWS, sizeof(T), LMAX, TILE * ROW)> one(
            have_w ? w + first * ny : three.run, w_rows, valid, tid, threads);
        three.issue();
        one.issue(); // (without weights a part of v once more, thrown away: no branch among the loads)
        p = load_point<T, NORM>(raw);
        three.put();
        if (have_w) {
            one.put();
            one.rest(tid);
        } else {
            no_weights();
        }
        three.rest(tid);
    } else {
        rows_to_lds<T>(v + first * 3u * ny, lds, valid * 3u * ny, 3u * ny, g.pad, g.magic_vectors3, tid, threads);
        if (have_w) {
            rows_to_lds<T>(w + first * ny, w_rows, valid * ny, ny, g.pad, g.magic_vectors, tid, threads);
        } else {
            no_weights();
        }
        p = load_point<T, NORM>(xyz + mine * 3u);
    }
    const T rho2 = p.x2 + p.y2;
    // set 0 = v_a - n_a s with a = x or z; set 1 = v_y - y s or w r - s
    const T n0 = second_half ? p.z : p.x, n1 = second_half ? T(1) : p.y;
    const T scale1 = second_half && NORM ? 1 / p.ir : T(1);
    __syncthreads();

    PointSums<T, true> sums0, sums1;
    T euler0 = 0, euler1 = 0; // sum of l times the set's values
    Azimuth<T> azimuth;
    const T* v_row = lds + point * v_stride;
    const T* w_row = w_rows + point * w_stride;
    auto column = [&](auto m) {
        const T fm = static_cast<T>(static_cast<int>(m));
        // (m = 0 is one entry: it has s_0 = 0 and m = 0 for factors on the minus side)
        const T u = minus ? azimuth.s : azimuth.c;
        const T u1 = minus ? azimuth.s1 : azimuth.c1, w1 = minus ? azimuth.c1 : -azimuth.s1;
        const T u2 = minus ? azimuth.s2 : azimuth.c2, w2 = minus ? azimuth.c2 : -azimuth.s2;
        const int side = minus ? -static_cast<int>(m) : static_cast<int>(m);
        const T* v_at = v_row + side;
        const T* w_at = w_row + side;
        const T* at0 = v_at + (second_half ? 2u * ny : 0u);
        const T* at1 = second_half ? w_at : v_at + ny;
        ColumnSums<T> k0, k1;
        T le0 = 0, le1 = 0;
        walk_column<T, true, LMAX>(m, L, p.z, rho2, [&](auto step, auto l, T fa, T fb, T fc, T fe, T fg, T fk) {
            constexpr int S = decltype(step)::value;
            const int at = l * (l + 1);
            T set0, set1;
            if constexpr (NORM) {
                const T vx = v_at[at], vy = v_at[at + ny], vz = v_at[at + 2u * ny];
                const T s = fma_of(vx, p.x, fma_of(vy, p.y, vz * p.z));
                const T wk = w_at[at];
                set0 = fma_of(-n0, s, second_half ? vz : vx);
                set1 = fma_of(-n1, s, (second_half ? wk : vy) * scale1);
                const T lfa = fa * static_cast<T>(l);
                le0 = fma_of(set0, lfa, le0);
                le1 = fma_of(set1, lfa, le1);
            } else {
                set0 = at0[at];
                set1 = at1[at];
            }
            k0.template add<S, true>(set0, fa, fb, fc, fe, fg, fk);
            k1.template add<S, true>(set1, fa, fb, fc, fe, fg, fk);
        });
        sums0.add(k0, fm, u, u1, w1, u2, w2);
        sums1.add(k1, fm, u, u1, w1, u2, w2);
        if constexpr (NORM) {
            euler0 = fma_of(le0, u, euler0);
            euler1 = fma_of(le1, u, euler1);
        }
    };
    if constexpr (LMAX > 0) {
        const unsigned mine = columns_of(wave, waves, LMAX);
        each_of(std::make_integer_sequence<int, LMAX + 1>{}, [&](auto m) {
            if constexpr (m.value > 0) azimuth.next(p.x, p.y);
            if ((mine >> m.value) & 1u) column(m);
        });
    } else {
        Deal deal(waves);
        for (int m = 0; m <= L; ++m) {
            if (m > 0) azimuth.next(p.x, p.y);
            if (deal.next(wave)) column(m);
        }
    }

    constexpr unsigned NS = NORM ? 7 : 3;
    T total[NS];
    if (!second_half) {
        const T xy0 = sums0.xy(p.x, p.y), xy1 = sums1.xy(p.x, p.y);
        total[0] = sums0.xx(p.x) + xy1;
        total[1] = xy0 + sums1.yy(p.y);
        total[2] = sums0.xz(p.x) + sums1.yz(p.y);
        if constexpr (NORM) {
            total[3] = sums0.gx(p.x) + sums1.gy(p.y);
            total[4] = euler0;
            total[5] = euler1;
            total[6] = 0;
        }
    } else {
        total[0] = sums0.xz(p.x) + sums1.gx(p.x);
        total[1] = sums0.yz(p.y) + sums1.gy(p.y);
        total[2] = sums0.zz() + sums1.gz();
        if constexpr (NORM) {
            total[3] = sums0.gz();
            total[4] = 0;
            total[5] = 0;
            total[6] = euler0;
        }
    }
#pragma unroll
    for (unsigned i = 0; i < NS; ++i) {
        total[i] += __shfl_xor(total[i], 16);
        total[i] += __shfl_xor(total[i], 32);
    }
    T* partial = lds + g.off_sums;
    if (waves > 1) __syncthreads(); // the sums take the place of the weights
    if (wave != 0 && lane < TILE) {
#pragma unroll
        for (unsigned i = 0; i < NS; ++i) partial[((wave - 1u) * NS + i) * TILE + lane] = total[i];
    }
    if (waves > 1) __syncthreads();
    if (wave == 0 && lane < valid) {
        for (unsigned q = 0; q + 1 < waves; ++q) {
#pragma unroll
            for (unsigned i = 0; i < NS; ++i) total[i] += partial[(q * NS + i) * TILE + lane];
        }
        T ox = total[0], oy = total[1], oz = total[2];
        if constexpr (NORM) {
            const T inward = fma_of(ox, p.x, fma_of(oy, p.y, fma_of(oz, p.z, total[3])));
            const T irsq = p.ir * p.ir;
            ox = (fma_of(-inward, p.x, ox) - total[4]) * irsq;
            oy = (fma_of(-inward, p.y, oy) - total[5]) * irsq;
            oz = (fma_of(-inward, p.z, oz) - total[6]) * irsq;
        }
        T* to = out + mine * 3u;
        to[0] = ox;
        to[1] = oy;
        to[2] = oz;
        if (__builtin_expect(lost_one(ox, oy, oz), 0)) {
            const Point<T> q = load_point<T, NORM>(xyz + mine * 3u);
            if (!is_number(q)) return; // (at the origin every entry is a NaN)
            const T* v_of = v + (first + mine) * 3u * ny;
            const T* w_of = w + (first + mine) * ny;
            volatile T* sum = to; // (as above)
            sum[0] = 0;
            sum[1] = 0;
            sum[2] = 0;
            each_entry<T, NORM, true>(L, q, [&](int k, const EntryDerivatives<T, NORM, true>& of) {
                const T vx = v_of[k], vy = v_of[k + ny], vz = v_of[k + 2u * ny];
#pragma unroll
                for (int b = 0; b < 3; ++b) {
                    T add = of.h[0][b] * vx + of.h[1][b] * vy + of.h[2][b] * vz;
                    if (have_w) add += of.d[b] * w_of[k];
                    sum[b] = sum[b] + add;
                }
            });
        }
    }
}

} // namespace sphx

#endif
