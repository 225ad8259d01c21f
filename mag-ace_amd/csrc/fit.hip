// fit.hip -- the sums over atoms of monomials and their derivatives that the gradient in the coefficients is made of.
//
// With a monomial P_t = X_p X_q (nodes.cpp, FitPlan) an atom's part of M_t is
//   Re(alpha P_t + beta D_u P_t) = Re((alpha X_p + beta D_u X_p) X_q + beta X_p D_u X_q),
// four real products: U.re X.re - U.im X.im + V.re X'.re - V.im X'.im.  A tile of sixteen p by sixteen q is therefore
// one 16x16x4 matrix product an atom, and the atoms follow one another in its sums.
//
// One thread a monomial read four entries and their derivatives and made nine complex products, an atom at a time
// with its loads in the open; here a step of 62000 atoms of the lmax-4 header (3636 monomials, 89 tiles with a sixth of
// their entries in use, two groups) takes 444 us where it took 2074.  What bounds it: the loads of Z, one atom ahead
// with two workgroups a compute unit (4.6 TB/s), then LDS (a quarter of the time).  Registers decide: spilled
// ones are read back behind the loads that run ahead and wait for them (700 to 990 us), so a thread has two entries and two
// nodes of a group and no loop behind them, and a wave six tiles.
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "kernels.hpp"
#include "magace.hpp"
#include "matrix.hpp"

namespace magace {

namespace {

typedef double Pair2 __attribute__((ext_vector_type(2)));
struct FitSlot {  // a value and its derivative; of a node p: (U.re, -U.im), (V.re, -V.im)
    Pair2 v, d;
};
__device__ __forceinline__ Pair2 mul2(Pair2 a, Pair2 b) {
    Pair2 r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}
__device__ __forceinline__ FitSlot product(const FitSlot& a, const FitSlot& b) {
    return {mul2(a.v, b.v), mul2(a.d, b.v) + mul2(a.v, b.d)};
}

}  // namespace

// Workgroup: a group of tiles (x), `chunk` atoms (y), a density (z); TW tiles a wave, of which those that a group does
// not have repeat its first one and are not added.  An atom's entries are loaded while the one before is summed.
template <int TW>
__global__ void __launch_bounds__(64 * kFitWaves) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_fit_accum(FitTab F, int nz, int nterms, int nd, const cplx<double>* __restrict__ Z, const cplx<double>* __restrict__ Zdot,
            const double* __restrict__ alpha, const double* __restrict__ beta, int natom, int chunk, double* __restrict__ M) {
    typedef Mm<double>::V V;
    constexpr int NT = 64 * kFitWaves, U = kFitEntries / NT, UN = kFitNodes / NT;  // entries and nodes of a thread
    static_assert(U == 2 && UN == 2, "both are written out below");
    extern __shared__ __align__(16) unsigned char smem[];
    // values, and their derivatives at a fixed distance: a slot of either is 16 bytes, of which 16 lanes read 16
    // consecutive ones without bank conflicts (with both in one slot of 32 bytes half of the LDS cycles were conflicts)
    Pair2* s = (Pair2*)smem;
    auto get = [&](uint32_t i) { return FitSlot{s[i], s[i + kFitSlots]}; };
    auto set = [&](uint32_t i, const FitSlot& x) { s[i] = x.v, s[i + kFitSlots] = x.d; };
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, d = blockIdx.z;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int* __restrict__ h = F.head + kFitHead * blockIdx.x;
    const unsigned short* __restrict__ entry = F.entry + h[0];
    const int ne = h[1], ny = h[3], np = h[5], nn = h[6], tile0 = h[7], tiles = h[8];
    const int sn = ne + 1 + ny;  // first node
    const int a0 = blockIdx.y * chunk, a1 = min(natom, a0 + chunk);

    V acc[TW];
    uint32_t place[TW];  // this lane's operands, in doubles
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        const int i = wave + kFitWaves * t;
        acc[t] = (V)0.0;
        place[t] = 2 * F.place[(size_t)(tile0 + (i < tiles ? i : 0)) * 64 + lane] + 0x10001u * ((g & 1) + (g >> 1) * 2 * kFitSlots);
    }
    auto load = [&](int a, uint32_t e) {  // a ZLayout::half entry
        const size_t x = (size_t)a * nz + (e & 0xfff);
        const cplx<double> z = Z[x], y = Zdot[x];
        return FitSlot{{z.re, z.im}, {y.re, y.im}};
    };
    auto put = [&](int i, FitSlot v, uint32_t e) {
        const double re = e >> 14 & 1 ? -1.0 : 1.0, im = e >> 15 & 1 ? -1.0 : 1.0;
        v.v.x *= re, v.d.x *= re, v.v.y *= im, v.d.y *= im;
        set(i, v);
    };
    uint32_t e[U], pair[UN];
    FitSlot next[U];
#pragma unroll
    for (int u = 0; u < UN; ++u) pair[u] = F.node[h[4] + min(u * NT + tid, nn - 1)];
    const uint32_t prod = ny > 0 ? F.prod[h[2] + min(tid, ny - 1)] : 0u;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        e[u] = entry[min(u * NT + tid, ne - 1)];
        next[u] = load(a0, e[u]);
    }
    if (tid == 0) set(ne, {{1.0, 0.0}, {0.0, 0.0}});
    double al1 = alpha[(size_t)a0 * nd + d], be1 = beta[(size_t)a0 * nd + d];
    for (int a = a0; a < a1; ++a) {
        const int an = min(a + 1, a1 - 1);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u * NT + tid < ne) put(u * NT + tid, next[u], e[u]);
            next[u] = load(an, e[u]);
        }
        const double al = al1, be = be1;
        al1 = alpha[(size_t)an * nd + d], be1 = beta[(size_t)an * nd + d];
        __syncthreads();
        if (ny > 0) {
            if (tid < ny) set(ne + 1 + tid, product(get(prod & 0xffff), get(prod >> 16)));
            __syncthreads();
        }
        auto node_at = [&](int i, const FitSlot& p) {
            FitSlot x = p;
            if (i < np) {
                const Pair2 w = al * x.v + be * x.d, v = be * x.v;
                x.v.x = w.x, x.v.y = -w.y, x.d.x = v.x, x.d.y = -v.y;
            }
            if (i < nn) set(sn + i, x);
        };
        {
            const FitSlot x = product(get(pair[0] & 0xffff), get(pair[0] >> 16));
            node_at(tid, x);
        }
        if (NT < nn) {
            const FitSlot x = product(get(pair[1] & 0xffff), get(pair[1] >> 16));
            node_at(NT + tid, x);
        }
        __syncthreads();
        const double* sd = (const double*)smem;
#pragma unroll
        for (int t = 0; t < TW; ++t)
            acc[t] = Mm<double>::mul(sd[place[t] & 0xffff], sd[place[t] >> 16], acc[t]);
    }
#pragma unroll
    for (int t = 0; t < TW; ++t) {
        const int i = wave + kFitWaves * t;
        if (i < tiles) {
            const int4 m = F.t[(size_t)(tile0 + i) * 64 + lane];
            const int r[4] = {m.x, m.y, m.z, m.w};
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (r[u] >= 0) atomicAdd(&M[(size_t)d * nterms + (r[u] >> 1)], r[u] & 1 ? -acc[t][u] : acc[t][u]);
        }
    }
}

namespace {

template <int TW, typename... A>
hipError_t launch_accum(dim3 grid, size_t lds, hipStream_t s, A... a) {
    int dev = 0, most = 0;
    hipError_t e;
    if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
    if ((e = hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) != hipSuccess) return e;
    if (lds > (size_t)most) return hipErrorInvalidValue;
    if ((e = hipFuncSetAttribute((const void*)k_fit_accum<TW>, hipFuncAttributeMaxDynamicSharedMemorySize, most)) != hipSuccess)
        return e;
    hipLaunchKernelGGL(k_fit_accum<TW>, grid, dim3(64 * kFitWaves), lds, s, a...);
    return hipGetLastError();
}

}  // namespace

hipError_t fit_accumulate(const FitTab& F, int nz, int nterms, int nd, int natom, const void* Z, const void* Zdot,
                          const double* alpha, const double* beta, double* M, hipStream_t s) {
    if (natom <= 0 || F.groups <= 0) return hipSuccess;
    // about four workgroups a compute unit; at least four atoms each, so that the additions to M stay few
    const long long per = ((long long)natom * F.groups * nd + 1023) / 1024;
    const int chunk = (int)(per < 4 ? 4 : per);
    const dim3 grid((unsigned)F.groups, (unsigned)((natom + chunk - 1) / chunk), (unsigned)nd);
    auto go = [&](auto k) {
        return k(grid, ((size_t)kFitSlots + F.slots) * sizeof(Pair2), s, F, nz, nterms, nd, (const cplx<double>*)Z,
                 (const cplx<double>*)Zdot, alpha, beta, natom, chunk, M);
    };
    static_assert(kFitTiles == 6, "an instance for every number of tiles");
#define MAGACE_ACCUM(TW) launch_accum<TW, FitTab, int, int, int, const cplx<double>*, const cplx<double>*, const double*, const double*, int, int, double*>
    return go(F.most <= 3 ? MAGACE_ACCUM(3) : F.most <= 5 ? MAGACE_ACCUM(5) : MAGACE_ACCUM(6));
#undef MAGACE_ACCUM
}

}  // namespace magace
