// kernels.hpp -- device code shared by the kernel files: complex arithmetic, aligned LDS reads
// by byte address, and the energy of one atom from its density.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "device.hpp"

namespace magace {

template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ __forceinline__ void cfma(cplx<T>& acc, cplx<T> a, cplx<T> b) {
    acc.re = fma(a.re, b.re, fma(-a.im, b.im, acc.re));
    acc.im = fma(a.re, b.im, fma(a.im, b.re, acc.im));
}
template <typename T>
__device__ __forceinline__ T re_mul(cplx<T> a, cplx<T> b) {  // Re(a*b)
    return fma(a.re, b.re, -a.im * b.im);
}
template <typename T>
__device__ __forceinline__ cplx<T> cconj_sign(cplx<T> a, int m) {  // (-1)^m conj(a)
    return (m & 1) ? cplx<T>{-a.re, a.im} : cplx<T>{a.re, -a.im};
}

// embedding F(rho) and F'(rho) (src/forces.F90:1134-1233, nfemb 0..2)
__device__ inline void embed(int nfemb, double rho, double wpre, double mexp, double& F, double& dF) {
    if (nfemb == 0) { F = rho; dF = 1.0; return; }
    const double w = 10.0, eps = 1e-10;
    const double s = nfemb == 2 ? 1.0 + rho : rho;
    if (fabs(s) > eps) {
        double y1 = w * s * s;
        const double g = y1 > 30.0 ? 0.0 : exp(-y1);
        const double omg = 1.0 - g, a = fabs(s), sg = s >= 0.0 ? 1.0 : -1.0;
        y1 = pow(omg * a, mexp);
        const double y2 = mexp * g * a;
        F = nfemb == 2 ? wpre * (sg * (y1 + y2) - 1.0) : wpre * sg * (y1 + y2);
        const double dg = -2.0 * w * s * g, da = sg;
        const double dy = fabs(y1) < eps ? 0.0 : mexp * y1 / (omg * a);
        dF = wpre * sg * (dy * (-dg * a + omg * da) + mexp * (dg * a + g * da));
    } else {
        F = nfemb == 2 ? wpre * mexp * (s - 1.0) : wpre * mexp * rho;
        dF = wpre * mexp;
    }
}

// An aligned vector at LDS byte address `off`. The adjoint kernels declare no static LDS (the
// host checks this before launching them), so their dynamic LDS, and with it Z' at its start,
// begins at address 0: a record's byte offset into Z' is the address itself, and reading it
// this way saves the add of the dynamic base, which the compiler resolves only after
// instruction selection and so cannot fold away.
template <typename E, int N>
__device__ __forceinline__ E __attribute__((ext_vector_type(N))) lds_at(uint32_t off) {
    typedef E V __attribute__((ext_vector_type(N)));
    return *(const __attribute__((address_space(3))) V*)(size_t)off;
}
__device__ __forceinline__ float4 lds_f4(uint32_t off) {
    const auto v = lds_at<float, 4>(off);
    return make_float4(v.x, v.y, v.z, v.w);
}
// one complex entry of Z' at a byte offset, as a single aligned vector read
template <typename T> __device__ __forceinline__ cplx<T> lds_cplx(uint32_t off) {
    const auto v = lds_at<T, 2>(off);
    return {v.x, v.y};
}

// E_i = f_in(e_hc) sum_d F(rho_d) + e_hc (src/forces.F90:1066-1128) for nd densities whose
// B parts sum to tots[d]; writes eout, dE_i/drho_d = fc F'(rho_d) (also into scale[d]), the
// e_hc factor and rho
template <typename T>
__device__ inline void atom_energy(const DevParams<T>& P, int nd, int atom, const double* tots, double e,
                                   const double* r1, double* __restrict__ eout, double* __restrict__ dEout,
                                   double* __restrict__ edfout, double* __restrict__ rho_out, double* scale) {
    // e = e_hc of the atom, r1[d] its B1 parts of rho (loaded by the caller ahead of time)
    double Fs = 0.0, dF[2] = {0.0, 0.0};
    for (int d = 0; d < nd; ++d) {
        const double r = tots[d] + r1[d];
        rho_out[(size_t)atom * nd + d] = r;
        double F;
        embed(P.nfemb, r, P.p1[d][0], P.p1[d][1], F, dF[d]);
        Fs += F;
    }
    const double elow = P.ecut - P.decut;
    double fc = 1.0, dfc = 0.0;
    if (e >= P.ecut) { fc = 0.0; dfc = 0.0; }
    else if (e > elow) {
        const double pi = 3.14159265358979323846;
        fc = 0.5 * (1.0 + cos(pi * (e - elow) / P.decut));
        dfc = -0.5 * sin(pi * (e - elow) / P.decut) * pi / P.decut;
    }
    eout[atom] = fc * Fs + e;
    for (int d = 0; d < nd; ++d) {
        dEout[(size_t)atom * nd + d] = fc * dF[d];
        scale[d] = fc * dF[d];
    }
    edfout[atom] = dfc * Fs + 1.0;
}

// ---------------------------------------------------------------- lanes
// sums of a and b over the two halves of the wave, a's in the lower half and b's in the upper; the same over
// pairs of 16 lanes
__device__ __forceinline__ float fold32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float fold16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double fold32(double a, double b) {
    const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}
__device__ __forceinline__ double fold16(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
    return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
}

}  // namespace magace
