// matrix.hpp -- device code shared by the kernels that run on the matrix cores: the 16x16x4 products and
// the places of their operands, spherical harmonics with literal constants, and spline rows.
//
// Operands of a 16x16x4 product on a wave: lane (i = lane % 16, g = lane / 16) holds A[i][g] and
// B[g][i], and of the result the column i and the rows mm_row(g, r), r = 0..3.  The result of one
// product is therefore the B operand of another whose step r contracts over the rows
// {mm_row(0, r), ..., mm_row(3, r)}: no data moves between lanes.
#pragma once

#include <hip/hip_runtime.h>

#include "device.hpp"
#include "kernels.hpp"

namespace magace {

template <typename T> struct Mm;
template <> struct Mm<float> {
    typedef float V __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ V mul(float a, float b, V c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    __host__ __device__ static constexpr int row(int g, int r) { return 4 * g + r; }
};
template <> struct Mm<double> {
    typedef double V __attribute__((ext_vector_type(4)));
    __device__ static __forceinline__ V mul(double a, double b, V c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __host__ __device__ static constexpr int row(int g, int r) { return g + 4 * r; }
};

// ---------------------------------------------------------------- spherical harmonics
constexpr double const_sqrt(double x) {
    double y = x > 1.0 ? x : 1.0;
    for (int i = 0; i < 64; ++i) y = 0.5 * (y + x / y);
    return y;
}
// recursion constants (src/spherical.F90:18-49) as a table that the unrolled loops read at constant places
struct LegTable {
    double a[7][7] = {}, b[7][7] = {}, c[7] = {}, d[7] = {};
    constexpr LegTable() {
        for (int l = 1; l <= 6; ++l) {
            const double ll = (double)l * l, l2 = (double)(l - 1) * (l - 1);
            for (int m = 0; m <= l - 2; ++m) {
                const double mm = (double)m * m;
                a[l][m] = const_sqrt((4.0 * ll - 1.0) / (ll - mm));
                b[l][m] = -const_sqrt((l2 - mm) / (4.0 * l2 - 1.0));
            }
            c[l] = -const_sqrt(1.0 + 0.5 / l);
            d[l] = const_sqrt(2.0 * (l - 1) + 3.0);
        }
    }
};
__device__ constexpr LegTable kLeg;

// Y_lm of (x, y, z), m >= 0 and l <= lmax <= L, order by order: put(l(l+1)/2 + m, P, dP, phase, phase of
// m - 1, m) with Y = P phase and dP = dP/dz (src/spherical.F90:55-155); one m at a time, so that only two
// Legendre values live
template <typename T, int L, typename F>
__device__ __forceinline__ void harmonics(T x, T y, T z, int lmax, F&& put) {
    static_assert(L <= 6, "the constants reach l = 6");
    cplx<T> ph = {1, 0}, ph1 = {1, 0};
    T pmm = (T)1;
#pragma unroll
    for (int m = 0; m <= L; ++m) {
        if (m > 0) {
            pmm *= (T)kLeg.c[m];
            ph1 = ph;
            ph = cmul(ph, cplx<T>{x, y});
        }
        if (m > lmax) continue;
        T p2 = pmm, d2 = (T)0, p1 = (T)0, d1 = (T)0;
        put(m * (m + 1) / 2 + m, pmm, (T)0, ph, ph1, m);
#pragma unroll
        for (int l = m + 1; l <= L; ++l) {
            if (l > lmax) continue;
            T p, d;
            if (l == m + 1) {
                d = (T)kLeg.d[l] * pmm;
                p = d * z;
            } else {
                const T a = (T)kLeg.a[l][m], b = (T)kLeg.b[l][m];
                p = a * fma(z, p1, b * p2);
                d = a * (p1 + fma(z, d1, b * d2));
                p2 = p1;
                d2 = d1;
            }
            p1 = p;
            d1 = d;
            put(l * (l + 1) / 2 + m, p, d, ph, ph1, m);
        }
    }
}

// ---------------------------------------------------------------- spline rows
// Row number and fraction of a distance or moment (src/radial.F90:68-84, 126-158); row < 0: every function
// is 0 (kRowZero: beyond the table) or, for moments below the first node, 1 (kRowOne).  A value that is not a number
// is in no row: it takes the error's side of every comparison.
constexpr int kRowZero = -1, kRowOne = -2;
template <typename T>
__device__ __forceinline__ int atomic_index(const DevParams<T>& P, double r, T& w, int* err) {
    const double x = r * P.rs_a, fl = floor(x);
    w = (T)(x - fl);
    if (!(fl > 0.0)) {
        atomicOr(err, kErrSmallDistance);
        return kRowZero;
    }
    return fl >= (double)P.nlut ? kRowZero : (int)fl - 1;
}
template <typename T>
__device__ __forceinline__ int magnetic_index(const DevParams<T>& P, double mu, T& w, int* err) {
    const double x = mu * P.rs_m, fl = floor(x);
    w = (T)(x - fl);
    if (!(fl >= 0.0 && fl <= (double)P.nlut)) {
        atomicOr(err, kErrMomentRange);
        return kRowZero;
    }
    return fl == 0.0 ? kRowOne : (int)fl - 1;
}

template <typename T> struct Coef {  // one function of a row
    T c[4];
};
__device__ __forceinline__ Coef<float> coef_at(const float* __restrict__ p) {
    const float4 v = *(const float4*)p;
    return {{v.x, v.y, v.z, v.w}};
}
__device__ __forceinline__ Coef<double> coef_at(const double* __restrict__ p) {
    const double2 a = *(const double2*)p, b = *(const double2*)(p + 2);
    return {{a.x, a.y, b.x, b.y}};
}
template <typename T> __device__ __forceinline__ T coef_value(const Coef<T>& k, T w) {
    return fma(w, fma(w, fma(w, k.c[3], k.c[2]), k.c[1]), k.c[0]);
}
template <typename T> __device__ __forceinline__ T coef_slope(const Coef<T>& k, T w, T rs) {
    return fma(w, fma(w, (T)3 * k.c[3], (T)2 * k.c[2]), k.c[1]) * rs;
}

}  // namespace magace
