// device.hip -- HIP kernels (gfx950) for the magnetic-ACE energy / force / torque path.
//
// One evaluation (the work of libace's acelib_, src/ace.F90:280-286) is three launches:
//
//   density    (prepA, src/a_basis.F90:59-359) k_density_mm (density.hip), for the accumulation recipe k_density
//              (here): one workgroup per atom writes Z = [A | A2 | A0], the core sum and the B1 part of rho.
//              k_density stages pair radial functions and Y_lm of the bond and of the neighbour moment in LDS
//              for a chunk of neighbours; threads then own (lm, n-block) columns of A and
//              (l'm', n-block) columns of A2 and accumulate in registers.
//   adjoint    (prepB + forceweights, src/b_basis.F90:62-307, src/forces.F90:84-349) k_adjoint_nodes (adjoint.hip)
//              for one density and body orders up to 4; otherwise, and for the accumulation recipe, k_adjoint and
//              k_adjoint_pair (here): one workgroup per atom, or two atoms in FP32.  Z and dZ in LDS; each thread
//              sums chunks of gradient records w*Z[a]Z[b]Z[c] per target (the transposed
//              monomial table), partial sums meet in a fixed order (no atomics); then rho,
//              E_i, dE/drho and the scaled gradient W = dE/dZ are written.
//   forces     (forcecompute + torquecompute, src/forces.F90:418-623, 688-961) k_forces_mm (forces.hip): nothing per
//              pair is stored between launches; F_p = dE_i/du_p, T_p = dE_i/dm_j and T0_i = dE_i/dm_i are
//              contractions of W with the pair's derivatives.
//
// T = double (FP64 path) or float (mixed path: FP32 splines, Y_lm, A, B products; FP64 for
// rho, the energy and all outputs).
#include <hip/hip_runtime.h>

#include <cmath>

#include "device.hpp"
#include "kernels.hpp"

namespace magace {

constexpr int kLmaxC = 12;
constexpr int kLhC = (kLmaxC + 1) * (kLmaxC + 2) / 2;

// Legendre recursion coefficients of k_density (src/spherical.F90:18-49): a_lm, b_lm (m <= l-2), c_l, d_l
__constant__ float c_alm[kLhC], c_blm[kLhC], c_cl[kLmaxC + 1], c_dl[kLmaxC + 1];

hipError_t upload_legendre_constants() {
    float a[kLhC] = {0}, b[kLhC] = {0}, c[kLmaxC + 1] = {0}, d[kLmaxC + 1] = {0};
    for (int l = 1; l <= kLmaxC; ++l) {
        const double lsq = (double)(l * l), l1 = 4.0 * lsq - 1.0, l2 = lsq - 2.0 * l + 1.0;
        for (int m = 0; m <= l - 2; ++m) {
            const double msq = (double)(m * m);
            const int k = l * (l + 1) / 2 + m;
            a[k] = (float)std::sqrt(l1 / (lsq - msq));
            b[k] = (float)-std::sqrt((l2 - msq) / (4.0 * l2 - 1.0));
        }
        c[l] = (float)-std::sqrt(1.0 + 0.5 / (double)l);
        d[l] = (float)std::sqrt(2.0 * (double)(l - 1) + 3.0);
    }
    hipError_t e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_alm), a, sizeof a))) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_blm), b, sizeof b))) return e;
    if ((e = hipMemcpyToSymbol(HIP_SYMBOL(c_cl), c, sizeof c))) return e;
    return hipMemcpyToSymbol(HIP_SYMBOL(c_dl), d, sizeof d);
}

// ---------------------------------------------------------------- small helpers
// Kahan step: s += x, with c holding minus the part of the running sum that s has lost
// (the compensated sum is s - c)
template <typename T>
__device__ __forceinline__ void kahan_add(T& s, T& c, T x) {
    const T y = x - c;
    const T t = s + y;
    c = (t - s) - y;
    s = t;
}

// cubic Hermite row entry: value and derivative (d/dr) at fractional position w
template <typename T>
__device__ __forceinline__ void horner(const T* __restrict__ c, T w, T rs, T& v, T& dv) {
    const T c0 = c[0], c1 = c[1], c2 = c[2], c3 = c[3];
    v = fma(w, fma(w, fma(w, c3, c2), c1), c0);
    dv = fma(w, fma(w, (T)3 * c3, (T)2 * c2), c1) * rs;
}

// The four coefficients of one spline function as one 16-byte load (rows and functions are 16-byte aligned)
__device__ __forceinline__ void load_coef(const float* __restrict__ p, float (&c)[4]) {
    const float4 v = *(const float4*)p;
    c[0] = v.x; c[1] = v.y; c[2] = v.z; c[3] = v.w;
}

// Values of the spline functions koff + k, k0 <= k < k1, of one table row at fraction w
// (horner's value, in the same operation order), with the coefficient loads of eight functions issued together
// so that one trip to L2 serves them all instead of one; dflt for every function when the row is absent.
// put(k, v) stores each.  `safe` is any readable coefficient address, read in place of the row's where a
// function is past k1 or the row is absent.
template <typename F>
__device__ __forceinline__ void spline_values(const float* __restrict__ row, const float* __restrict__ safe, float w,
                                              int k0, int k1, int koff, float dflt, F&& put) {
    constexpr int B = 8;
    for (int k = k0; k < k1; k += B) {
        float c[B][4];
#pragma unroll
        for (int u = 0; u < B; ++u) load_coef(row && k + u < k1 ? row + 4 * (koff + k + u) : safe, c[u]);
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (k + u < k1) put(k + u, row ? fma(w, fma(w, fma(w, c[u][3], c[u][2]), c[u][1]), c[u][0]) : dflt);
    }
}

// Spline row and fraction for the atomic table (src/radial.F90:68-84).
// Returns nullptr when the pair is beyond the table (all functions zero).  A distance or moment that is
// not a number is an error too: its row number would be -1, in front of the table.
template <typename T>
__device__ __forceinline__ const T* atomic_row(const DevParams<T>& P, double r, T& w, int* err) {
    const double x = r * P.rs_a;
    const double fl = floor(x);
    if (!(fl > 0.0)) { atomicOr(err, kErrSmallDistance); return nullptr; }
    if (fl >= (double)P.nlut) return nullptr;
    const int nl = (int)fl;
    w = (T)(x - fl);
    return P.lut_a + (size_t)(nl - 1) * P.stride_a;
}
// magnetic table (src/radial.F90:126-158): nl == 0 -> every function is 1, derivative 0
// (returned as row == nullptr with unit == true)
template <typename T>
__device__ __forceinline__ const T* magnetic_row(const DevParams<T>& P, double mu, T& w, bool& unit,
                                                 int* err) {
    unit = false;
    const double x = mu * P.rs_m;
    const double fl = floor(x);
    if (!(fl >= 0.0 && fl <= (double)P.nlut)) { atomicOr(err, kErrMomentRange); return nullptr; }
    if (fl == 0.0) { unit = true; return nullptr; }
    w = (T)(x - fl);
    return P.lut_m + (size_t)((int)fl - 1) * P.stride_m;
}

// Normalised associated Legendre functions P[lh] for l <= L, m <= l
// (src/spherical.F90:55-155); lh = l(l+1)/2 + m.  Y_lm(x,y,z) = P[lh] (x+iy)^m.
template <int L>
__device__ __forceinline__ void legendre(float z, float* P) {
    P[0] = 1.0f;
    if (L == 0) return;
    const float sq3 = (float)1.73205080756887719318, sq3o2 = (float)1.22474487139158894067;
    P[1] = sq3 * z;
    P[2] = -sq3o2;
#pragma unroll
    for (int l = 2; l <= L; ++l) {
#pragma unroll
        for (int m = 0; m <= l - 2; ++m) {
            const int k = l * (l + 1) / 2 + m, k1 = (l - 1) * l / 2 + m, k2 = (l - 2) * (l - 1) / 2 + m;
            P[k] = c_alm[k] * fma(z, P[k1], c_blm[k] * P[k2]);
        }
        const int kp = (l - 1) * l / 2 + (l - 1);
        const float t = c_dl[l] * P[kp];
        P[l * (l + 1) / 2 + l - 1] = t * z;
        P[l * (l + 1) / 2 + l] = c_cl[l] * P[kp];
    }
}

// half set of Y_lm (m >= 0) written to out[lh]
template <int L>
__device__ __forceinline__ void ylm_half(float x, float y, float z, int lmax, cplx<float>* out) {
    float P[(L + 1) * (L + 2) / 2];
    legendre<L>(z, P);
    cplx<float> ph = {1, 0};
    const cplx<float> e = {x, y};
#pragma unroll
    for (int m = 0; m <= L; ++m) {
#pragma unroll
        for (int l = m; l <= L; ++l) {
            if (l <= lmax) {
                const int k = l * (l + 1) / 2 + m;
                out[k] = {P[k] * ph.re, P[k] * ph.im};
            }
        }
        ph = cmul(ph, e);
    }
}

template <typename T>
__device__ __forceinline__ cplx<T> yfull(const cplx<T>* half, int l, int m) {
    const cplx<T> v = half[l * (l + 1) / 2 + (m < 0 ? -m : m)];
    return m < 0 ? cconj_sign(v, -m) : v;
}

// ============================================================================ k_density
// Shapes: NB n-block of A columns, NM3X max magnetic columns of A, NB2 n-block of A2,
// NR2X max magnetic radial index of A2.
// FP32 sums with Kahan compensation (the accumulation recipe): 153 to 156 registers in shape class 0, three waves
// per SIMD; 239 to 256 in the others, two.
// Stores of the m >= 0 density tasks: A[n][l,m][q] for the task's radial block, A2[n][n'][l',m'], in the
// places of ZLayout::half.
template <typename T, int NB, int NM3X, int NACC, int NQ>
__device__ __forceinline__ void store_a_half(const DevParams<T>& P, const cplx<T> (&acc)[NACC][NQ], int n0, int lh,
                                             cplx<T>* __restrict__ Z) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int n = n0 + b;
        if (n < P.nr3a)
#pragma unroll
            for (int q = 0; q < NM3X; ++q)
                if (q < P.nm3) Z[(n * P.lha + lh) * P.nm3 + q] = acc[b][q];
    }
}
template <typename T, int NB2, int NR2X, int NACC, int NQ>
__device__ __forceinline__ void store_a2_half(const DevParams<T>& P, const cplx<T> (&acc)[NACC][NQ], int n0, int lh,
                                              cplx<T>* __restrict__ Z) {
#pragma unroll
    for (int b = 0; b < NB2; ++b) {
        const int n = n0 + b;
        if (n < P.nb_a)
#pragma unroll
            for (int q = 0; q < NR2X; ++q)
                if (q < P.nr2m) Z[P.hA2 + (n * P.nr2m + q) * P.lhm + lh] = acc[b][q];
    }
}

// The density of the accumulation recipe (MAGACE_MIXED_ACC): A and A2 summed over the neighbours with
// Kahan compensation, which the matrix cores of density.hip cannot do.
template <typename T, int L, int CH, int NB, int NM3X, int NB2, int NR2X, bool SPLIT, bool TASKSPLIT>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(L == 6 && NM3X <= 4 ? 3 : 2, 8))) k_density(DevParams<T> P, const int* __restrict__ off,
                                                const double* __restrict__ dlist,
                                                const double* __restrict__ elist,
                                                const double* __restrict__ dmomi,
                                                const double* __restrict__ emomi,
                                                const double* __restrict__ dmom,
                                                const double* __restrict__ emom,
                                                cplx<T>* __restrict__ Zout, double* __restrict__ ehc_out,
                                                double* __restrict__ rho1_out, int* err) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int atom = blockIdx.x;
    const int tid = threadIdx.x, nthr = blockDim.x;
    const int nfa = P.nr3a * (P.l3a + 1), nfm = P.nr2m * (P.l2m + 1);
    // LDS carve-up (sizes mirror density_lds_bytes on the host).  The per-pair rows have odd
    // lengths (one entry of padding where the count is even), so that the staging threads,
    // which write the rows of consecutive pairs at once, fall in distinct banks
    const int sYs = P.lha | 1, sYms = P.lhm | 1, sHs = P.nm3 | 1, sRs = nfa | 1, sGs = P.nb_a | 1, sMs = nfm | 1;
    cplx<T>* sY = (cplx<T>*)smem;                        // [CH][sYs]
    cplx<T>* sYm = sY + CH * sYs;                         // [CH][sYms]
    cplx<T>* sH = sYm + CH * sYms;                        // [CH][sHs]
    cplx<T>* sYc = sH + CH * sHs;                         // [lhm] central moment
    T* sR = (T*)(sYc + P.lhm);                            // [CH][sRs]  R_{l,n}
    T* sG = sR + CH * sRs;                                // [CH][sGs]
    T* sM = sG + CH * sGs;                                // [CH][sMs]  M_{l',n'}
    T* sCr = sM + CH * sMs;                               // [CH]
    T* sMc = sCr + CH;                                    // [nfm + nb_m] central M and g^m
    double* sEhc = (double*)(((uintptr_t)(sMc + nfm + P.nb_m) + 15) & ~(uintptr_t)15);

    const int p0 = off[atom], nn = off[atom + 1] - p0;
    Zout += (size_t)atom * P.nz;

    // central-atom magnetic functions: A0 and B1 (src/a_basis.F90:69-106, b_basis.F90:62-83),
    // one spline function per thread and the moment's Y_lm on the last wave, so that the block
    // does not wait for one thread to evaluate them all
    for (int k = tid; k < P.nb_m + nfm; k += nthr) {
        T w;
        bool unit;
        const T* row = magnetic_row(P, dmomi[atom], w, unit, err);
        T v = unit ? (T)1 : (T)0, dv;
        if (row) horner(row + 4 * k, w, (T)P.rs_m, v, dv);
        if (k < P.nb_m)
            sMc[nfm + k] = v;
        else
            sMc[k - P.nb_m] = v;
    }
    if (tid == nthr - 64) {
        ylm_half<L>((T)emomi[3 * atom], (T)emomi[3 * atom + 1], (T)emomi[3 * atom + 2], P.l2m, sYc);
        *sEhc = 0.0;
    }
    __syncthreads();
    if (tid == 0) {  // B1 part of rho, in the order of the sum over k
        double rho1[2] = {0.0, 0.0};
        for (int k = 0; k < P.nb_m; ++k) {
            const double v = (double)sMc[nfm + k];
            rho1[0] += P.c1[0][k] * (v - 1.0);
            rho1[1] += P.c1[1][k] * (v - 1.0);
        }
        for (int d = 0; d < P.nd; ++d) rho1_out[(size_t)atom * P.nd + d] = rho1[d];
    }
    for (int t = tid; t < P.nr2m * P.lhm; t += nthr) {
        const int np = t / P.lhm, lh = t % P.lhm;
        int l = 0;
        while ((l + 1) * (l + 2) / 2 <= lh) ++l;
        const cplx<T> y = sYc[lh];
        const T mv = sMc[l * P.nr2m + np];
        Zout[P.hA0 + t] = {mv * y.re, mv * y.im};
    }

    // Tasks cover m >= 0 only (P.lha and P.lhm entries per radial block): since R, M and g are
    // real and Y_{l,-m} = (-1)^m conj(Y_lm),
    //   A[n][l,-m][n',l',-m'] = (-1)^(m+m') conj(A[n][l,m][n',l',m'])  and
    //   A2[n][n'][l',-m'] = (-1)^m' conj(A2[n][n'][l',m']),
    // which are not stored.
    const int nblkA = (P.nr3a + NB - 1) / NB, nblkA2 = (P.nb_a + NB2 - 1) / NB2;
    const int nTA = P.lha * nblkA, nTA2 = P.lhm * nblkA2;
    // TASKSPLIT: when the A and A2 column tasks leave threads idle, each A task's neighbours
    // are split over SA threads (neighbour j on part j mod SA); the parts meet in LDS at the
    // end, in the staging area, which is free by then.  SA is P.sa when that is set (a tuned
    // choice), otherwise the largest that fits (at most 4), and 1 when that is below 3 (the
    // extra barrier and scratch traffic of SA = 2 cost more than it gained with all-m tasks).
    int SA = 1;
    if constexpr (TASKSPLIT) if (nTA + nTA2 <= nthr) {
        SA = min(P.sa > 0 ? P.sa : 4, (nthr - nTA2) / max(nTA, 1));
        const size_t room = (size_t)((const char*)sEhc - (const char*)smem);
        while (SA > 1 && (size_t)(SA - 1) * nTA * NB * NM3X * sizeof(cplx<T>) > room) --SA;
        if (P.sa <= 0 && SA < 3) SA = 1;
    }
    // A2 tasks start at a wave boundary when that still fits in one round: a wave holding both
    // kinds would run both loops one after the other
    const int nAt = (TASKSPLIT ? SA : 1) * nTA;
    const int a2base = ((nAt + 63) & ~63) + nTA2 <= nthr ? (nAt + 63) & ~63 : nAt;
    for (int round = 0; round * nthr < a2base + nTA2; ++round) {
        const int task = round * nthr + tid;
        cplx<T> acc[NB > NB2 ? NB : NB2][NM3X > NR2X ? NM3X : NR2X];
#pragma unroll
        for (int a = 0; a < (NB > NB2 ? NB : NB2); ++a)
#pragma unroll
            for (int b = 0; b < (NM3X > NR2X ? NM3X : NR2X); ++b) acc[a][b] = {0, 0};
        constexpr int kCa = NB > NB2 ? NB : NB2, kCq = NM3X > NR2X ? NM3X : NR2X;
        cplx<T> cmp[kCa][kCq];
#pragma unroll
        for (int a = 0; a < kCa; ++a)
#pragma unroll
            for (int b = 0; b < kCq; ++b) cmp[a][b] = {0, 0};
        // decode task
        // only light headers split tasks; the others keep a compile-time SA = 1
        constexpr bool kSplit = TASKSPLIT;
        const int sa = kSplit ? SA : 1;
        const bool isA = task < sa * nTA, isA2 = task >= a2base && task < a2base + nTA2;
        const int ta = kSplit && isA ? task % nTA : task, part = kSplit && isA ? task / nTA : 0;
        int lh = 0, l = 0, n0 = 0;
        if (isA) { lh = ta % P.lha; n0 = (ta / P.lha) * NB; }
        if (isA2) { lh = (task - a2base) % P.lhm; n0 = ((task - a2base) / P.lhm) * NB2; }
        while ((l + 1) * (l + 2) / 2 <= lh) ++l;

        for (int c0 = 0; c0 < nn; c0 += CH) {
            const int nj = nn - c0 < CH ? nn - c0 : CH;
            __syncthreads();
            if constexpr (SPLIT) {
                // staging of pair c0 + j, spread over the block: thread tid works on pair
                // j = tid % CH in role tid / CH.  Roles 0 and 1, which share a wave: the bond's
                // Y_lm and the core term, and the magnetic side (Y_l'm' of the neighbour moment,
                // the M and the products H_q the A columns need), through one Y_lm call for both;
                // roles 2..nsplit + 1: a share of the radial functions g_n, R_{l,n} and, after
                // them, of the magnetic functions M_{l',n'}
                const int j = tid % CH, role = tid / CH, nsplit = nthr / CH - 2;
                const bool live = j < nj;
                const int p = p0 + c0 + (live ? j : 0);
                if (role <= 1) {
                    const bool bond = role == 0;
                    if (live) {
                        T w = 0;
                        bool unit = false;
                        const T* row = bond ? atomic_row(P, dlist[p], w, err) : magnetic_row(P, dmom[p], w, unit, err);
                        if (bond) {
                            T cr = 0, dcr;
                            if (row) horner(row + 4 * (P.nb_a + nfa), w, (T)P.rs_a, cr, dcr);
                            sCr[j] = cr;
                        }
                        const double* v3 = bond ? elist : emom;
                        cplx<T>* yo = bond ? sY + j * sYs : sYm + j * sYms;
                        // the moment's M coefficients for H (four-column class: l' <= 1, one n'),
                        // loaded before the Y_lm so that their trip overlaps it
                        constexpr bool kMh = NM3X == 4 && sizeof(T) == 4;
                        T cmh[kMh ? 2 : 1][4];
                        if constexpr (kMh)
#pragma unroll
                            for (int lp = 0; lp < 2; ++lp)
                                load_coef(!bond && row && lp <= P.l3m ? row + 4 * (P.nb_m + lp * P.nr2m) : P.lut_m, cmh[lp]);
                        ylm_half<L>((T)v3[3 * p], (T)v3[3 * p + 1], (T)v3[3 * p + 2], bond ? P.l3a : P.l2m, yo);
                        if (!bond) {
                            // H_q = M_{l',n'} Y_{l'm'} for the magnetic columns of A (l' <= l3m,
                            // q = n' lsm3 + l'^2 + l' + m'); the few M it needs are evaluated
                            // here rather than waiting for the spline roles
                            for (int np = 0; np * P.lsm3 < P.nm3; ++np)
                                for (int lp = 0; lp <= P.l3m; ++lp) {
                                    T mv = unit ? (T)1 : (T)0, dv;
                                    if (kMh && np == 0 && lp < 2) {
                                        if (row) horner(cmh[kMh && lp < 2 ? lp : 0], w, (T)P.rs_m, mv, dv);
                                    } else if (row) {
                                        horner(row + 4 * (P.nb_m + lp * P.nr2m + np), w, (T)P.rs_m, mv, dv);
                                    }
                                    for (int mp = -lp; mp <= lp; ++mp) {
                                        const int q = np * P.lsm3 + lp * lp + lp + mp;
                                        const cplx<T> y = yfull(yo, lp, mp);
                                        sH[j * sHs + q] = {mv * y.re, mv * y.im};
                                    }
                                }
                        }
                    } else if (bond) {
                        sCr[j] = 0;
                    }
                } else {
                    // a share of the pair's radial functions g_n, R_{l,n} and, after them, of
                    // its magnetic functions M_{l',n'}
                    if (live) {
                        const int nf = P.nb_a + nfa, per = (nf + nfm + nsplit - 1) / nsplit;
                        const int k0 = (role - 2) * per, k1 = min(nf + nfm, k0 + per);
                        if (k0 < nf) {
                            T w = 0;
                            const T* row = atomic_row(P, dlist[p], w, err);
                            spline_values(row, P.lut_a, w, k0, min(k1, nf), 0, (T)0, [&](int k, T v) {
                                if (k < P.nb_a)
                                    sG[j * sGs + k] = v;
                                else
                                    sR[j * sRs + (k - P.nb_a)] = v;
                            });
                        }
                        if (k1 > nf) {
                            T w = 0;
                            bool unit;
                            const T* row = magnetic_row(P, dmom[p], w, unit, err);
                            spline_values(row, P.lut_m, w, max(k0, nf), k1, P.nb_m - nf, unit ? (T)1 : (T)0,
                                             [&](int k, T v) { sM[j * sMs + (k - nf)] = v; });
                        }
                    }
                }
            } else {
                // one thread per pair and side: atomic side (threads 0..CH-1), magnetic
                // side (CH..2CH-1)
                if (tid < CH) {  // atomic side of pair c0+tid
                    const int j = tid;
                    if (j < nj) {
                        const int p = p0 + c0 + j;
                        T w = 0;
                        const T* row = atomic_row(P, dlist[p], w, err);
                        spline_values(row, P.lut_a, w, 0, P.nb_a + nfa, 0, (T)0, [&](int k, T v) {
                            if (k < P.nb_a)
                                sG[j * sGs + k] = v;
                            else
                                sR[j * sRs + (k - P.nb_a)] = v;
                        });
                        T cr = 0, dcr;
                        if (row) horner(row + 4 * (P.nb_a + nfa), w, (T)P.rs_a, cr, dcr);
                        sCr[j] = cr;
                        ylm_half<L>((T)elist[3 * p], (T)elist[3 * p + 1], (T)elist[3 * p + 2], P.l3a,
                                       sY + j * sYs);
                    } else {
                        sCr[j] = 0;
                    }
                } else if (tid < 2 * CH) {  // magnetic side of pair c0+j
                    const int j = tid - CH;
                    if (j < nj) {
                        const int p = p0 + c0 + j;
                        T w = 0;
                        bool unit;
                        const T* row = magnetic_row(P, dmom[p], w, unit, err);
                        spline_values(row, P.lut_m, w, 0, nfm, P.nb_m, unit ? (T)1 : (T)0,
                                         [&](int k, T v) { sM[j * sMs + k] = v; });
                        cplx<T>* yh = sYm + j * sYms;
                        ylm_half<L>((T)emom[3 * p], (T)emom[3 * p + 1], (T)emom[3 * p + 2], P.l2m, yh);
                        // H_q = M_{l',n'} Y_{l'm'} for the magnetic columns of A (l' <= l3m)
                        for (int q = 0; q < P.nm3; ++q) {
                            const int np = q / P.lsm3, lmp = q % P.lsm3;
                            int lp = 0;
                            while ((lp + 1) * (lp + 1) <= lmp) ++lp;
                            const int mp = lmp - lp * lp - lp;
                            const cplx<T> y = yfull(yh, lp, mp);
                            const T mv = sM[j * sMs + lp * P.nr2m + np];
                            sH[j * sHs + q] = {mv * y.re, mv * y.im};
                        }
                    }
                }
            }
            __syncthreads();
            if (round == 0 && tid == 0) {
                double s = 0.0;
                for (int j = 0; j < nj; ++j) s += (double)sCr[j];
                *sEhc += s;
            }
            if (isA) {
                // A[n][lm][q] += R_{l,n} Y_lm H_q   (src/a_basis.F90:248-291).  Columns past nm3
                // and radial indices past nr3a are read without a test: those reads stay inside
                // the staging area, and their sums land in slots that are never stored.
                for (int j = part; j < nj; j += sa) {
                    // the pair's Y, H and R reads issued together (R read after the products
                    // Y H had waited for LDS a second time); the wide classes keep the later
                    // reads, as they would spill
                    const cplx<T> y = sY[j * sYs + lh];
                    cplx<T> h[NM3X];
#pragma unroll
                    for (int q = 0; q < NM3X; ++q) h[q] = sH[j * sHs + q];
                    const T* rr = sR + j * sRs + l * P.nr3a + n0;
                    constexpr bool kEarly = NM3X <= 4;
                    T rv[kEarly ? NB : 1];
                    if constexpr (kEarly)
#pragma unroll
                        for (int b = 0; b < NB; ++b) rv[b] = rr[b];
                    // Y H_q once per pair and column, then two real FMAs per radial index
                    cplx<T> yh[NM3X];
#pragma unroll
                    for (int q = 0; q < NM3X; ++q) yh[q] = cmul(y, h[q]);
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        const T r = kEarly ? rv[kEarly ? b : 0] : rr[b];
#pragma unroll
                        for (int q = 0; q < NM3X; ++q) {
                            kahan_add(acc[b][q].re, cmp[b][q].re, r * yh[q].re);
                            kahan_add(acc[b][q].im, cmp[b][q].im, r * yh[q].im);
                        }
                    }
                }
            } else if (isA2) {
                // A2[n][n'][l'm'] += g_n M_{l',n'} Y_{l'm'}   (src/a_basis.F90:193-201); unused
                // slots as above
                for (int j = 0; j < nj; ++j) {
                    // the pair's g reads issued with its Y and M reads, as in the A loop
                    const cplx<T> y = sYm[j * sYms + lh];
                    const T* mr = sM + j * sMs + l * P.nr2m;
                    const T* gr = sG + j * sGs + n0;
                    constexpr bool kEarly = NM3X <= 4;
                    T gv[kEarly ? NB2 : 1];
                    if constexpr (kEarly)
#pragma unroll
                        for (int b = 0; b < NB2; ++b) gv[b] = gr[b];
                    cplx<T> my[NR2X];
#pragma unroll
                    for (int q = 0; q < NR2X; ++q) my[q] = {mr[q] * y.re, mr[q] * y.im};
#pragma unroll
                    for (int b = 0; b < NB2; ++b) {
                        const T g = kEarly ? gv[kEarly ? b : 0] : gr[b];
#pragma unroll
                        for (int q = 0; q < NR2X; ++q) {
                            kahan_add(acc[b][q].re, cmp[b][q].re, g * my[q].re);
                            kahan_add(acc[b][q].im, cmp[b][q].im, g * my[q].im);
                        }
                    }
                }
            }
        }
        // the compensated sums
#pragma unroll
        for (int a = 0; a < kCa; ++a)
#pragma unroll
            for (int b = 0; b < kCq; ++b) {
                acc[a][b].re -= cmp[a][b].re;
                acc[a][b].im -= cmp[a][b].im;
            }
        if (kSplit && sa > 1) {  // one round only: every thread of the block reaches these barriers
            cplx<T>* scr = (cplx<T>*)smem;  // [SA - 1][nTA][NB][NM3X]
            __syncthreads();
            if (isA && part > 0)
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int q = 0; q < NM3X; ++q) scr[(((part - 1) * nTA + ta) * NB + b) * NM3X + q] = acc[b][q];
            __syncthreads();
            if (isA && part == 0)
                for (int h = 1; h < sa; ++h)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int q = 0; q < NM3X; ++q) {
                            const cplx<T> v = scr[(((h - 1) * nTA + ta) * NB + b) * NM3X + q];
                            acc[b][q].re += v.re;
                            acc[b][q].im += v.im;
                        }
        }
        if (isA && part == 0) {
            store_a_half<T, NB, NM3X>(P, acc, n0, lh, Zout);
        } else if (isA2) {
            store_a2_half<T, NB2, NR2X>(P, acc, n0, lh, Zout);
        }
    }
    __syncthreads();
    if (tid == 0) ehc_out[atom] = *sEhc;
}

size_t density_lds_bytes(const DevParams<double>& Pd, int CH, size_t tsize) {
    const int nfa = Pd.nr3a * (Pd.l3a + 1), nfm = Pd.nr2m * (Pd.l2m + 1);
    size_t cb = 2 * tsize;
    // per-pair rows padded to odd lengths (k_density)
    size_t n = cb * ((size_t)CH * (Pd.lha | 1) + (size_t)CH * (Pd.lhm | 1) + (size_t)CH * (Pd.nm3 | 1) + Pd.lhm) +
               tsize * ((size_t)CH * (nfa | 1) + (size_t)CH * (Pd.nb_a | 1) + (size_t)CH * (nfm | 1) + CH + nfm + Pd.nb_m);
    return ((n + 15) & ~(size_t)15) + 16;
}

// ============================================================================ k_adjoint
// entry of the full feature vector from its place in memory (ZLayout::half)
template <typename T>
__device__ __forceinline__ cplx<T> full_entry(const cplx<T>* __restrict__ Z, uint32_t e) {
    const cplx<T> v = Z[e & 0xfff];
    return {e >> 14 & 1 ? -v.re : v.re, e >> 15 & 1 ? -v.im : v.im};
}

template <typename T> __device__ __forceinline__ T rec_weight(uint4 r);
template <> __device__ __forceinline__ double rec_weight<double>(uint4 r) {
    return __hiloint2double((int)r.w, (int)r.z);
}
template <> __device__ __forceinline__ float rec_weight<float>(uint4 r) { return __uint_as_float(r.z); }

template <typename T>
__device__ __forceinline__ double block_sum(double v, double* red) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    if (ln == 0) red[wv] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int i = 0; i < (int)(blockDim.x >> 6); ++i) s += red[i];
    return s;  // valid on thread 0
}

__device__ __forceinline__ float4 vadd(float4 a, float4 b) {
    return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w);
}
template <typename T>
__device__ __forceinline__ cplx<T> vadd(cplx<T> a, cplx<T> b) {
    return {a.re + b.re, a.im + b.im};
}

// The adjoint's partial sums of one atom (or atom pair), part[slot], added up per target in a
// fixed order.  First pass: a thread sums one group of <= kCombGroup consecutive slots of a
// target, its loads issued together, into sW[x] when the group is the target's only one and
// into the group's first slot otherwise.  Second pass: a thread sums the group results of one
// target with several groups.  Two round trips to L2 instead of one per slot.
// cb, cb2: this thread's first descriptors (comb[tid], comb2[tid]), loaded ahead by the caller.
template <typename P_t, typename V>
__device__ __forceinline__ void combine_partials(const P_t& P, V* __restrict__ part, V* __restrict__ sW, int2 cb,
                                                 int2 cb2) {
    const int nthr = (int)blockDim.x, tid = (int)threadIdx.x;
    for (int k = tid; k < P.ncomb; k += nthr) {
        const int2 e = k == tid ? cb : P.comb[k];
        const int x = e.y & 0xfff, n = (e.y >> 12) & 15;
        V v[kCombGroup];
#pragma unroll
        for (int u = 0; u < kCombGroup; ++u)
            if (u < n) v[u] = part[e.x + u];
        V sum = v[0];
#pragma unroll
        for (int u = 1; u < kCombGroup; ++u)
            if (u < n) sum = vadd(sum, v[u]);
        if ((e.y >> 16) & 1)
            sW[x] = sum;
        else
            part[e.x] = sum;
    }
    __syncthreads();
    for (int k = tid; k < P.ncomb2; k += nthr) {
        const int2 e = k == tid ? cb2 : P.comb2[k];
        const int x = e.y & 0xfff, ng = e.y >> 12;
        V sum = part[e.x];
        for (int g0 = 1; g0 < ng; g0 += kCombGroup) {
            V v[kCombGroup];
#pragma unroll
            for (int u = 0; u < kCombGroup; ++u)
                if (g0 + u < ng) v[u] = part[e.x + (g0 + u) * kCombGroup];
#pragma unroll
            for (int u = 0; u < kCombGroup; ++u)
                if (g0 + u < ng) sum = vadd(sum, v[u]);
        }
        sW[x] = sum;
    }
}

// ND2: two densities (rho_d = sum_k c_{k,d} B_k, E = fc sum_d F(rho_d) + e_hc,
// src/forces.F90:976-1089): a second weight per record, a second gradient array in LDS
// ACC (FP32 only, MAGACE_MIXED_ACC): rho = sum of the A0 targets' gradient records summed in
// FP64 (double-float record weights: the FP32 weight in z plus its low part in w); in every
// round where some lane of the wave has an A0 target, the whole wave accumulates in FP64
template <typename T, bool ND2, bool ACC>
__global__ void __launch_bounds__(kAdjointThreads) k_adjoint(DevParams<T> P, int atom_base,
                                                const cplx<T>* __restrict__ Zin,
                                                cplx<T>* __restrict__ Wout, cplx<T>* __restrict__ Wd,
                                                char* __restrict__ Pt,
                                                const double* __restrict__ ehc,
                                                const double* __restrict__ rho1,
                                                double* __restrict__ eout, double* __restrict__ dEout,
                                                double* __restrict__ edfout, double* __restrict__ rho_out) {
    extern __shared__ __align__(16) unsigned char smem[];
    // extended vector Z' = [Z | 1 | Y] (nzx entries; Y: products for body orders 5, 6)
    cplx<T>* sZ = (cplx<T>*)smem;           // [nzx], sZ[nz] = 1
    cplx<T>* sW = sZ + P.nzx;               // [nzx]
    cplx<T>* sW2 = sW + P.nzx;              // [nzx] (ND2 only)
    double* red = (double*)(sW + (ND2 ? 2 : 1) * P.nzx);
    // the energy's scale factors after the two block sums; in dynamic LDS, so that it starts at
    // address 0 and the records' offsets address sZ without an add
    double* s_scale = red + 2 * (kAdjointThreads / 64);
    const int atom = blockIdx.x, tid = threadIdx.x;
    Zin += (size_t)atom * P.nz;
    {
        // Z' from Z, with all of a thread's loads issued before the stores
        constexpr int U = 8;  // covers nzx <= 8 * kAdjointThreads = 4096 in one pass
        static_assert(U * kAdjointThreads >= 4096, "one pass over the largest feature vector");
        cplx<T> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int x = tid + u * kAdjointThreads;
            v[u] = x < P.nz ? full_entry(Zin, P.zmap[x]) : cplx<T>{0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int x = tid + u * kAdjointThreads;
            if (x < P.nz) sZ[x] = v[u];
            if (x < P.nzx) {
                sW[x] = {0, 0};
                if (ND2) sW2[x] = {0, 0};
            }
        }
    }
    // what the tail needs from global memory, loaded now so that its latency passes during the
    // record walk: the fold words of this thread's entries, its first combine descriptors and
    // (thread 0) the atom's e_hc and B1 part of rho
    constexpr int kFold = 8;  // nz <= 8 * kAdjointThreads
    uint32_t fw[kFold];
#pragma unroll
    for (int u = 0; u < kFold; ++u) {
        const int x = tid + u * kAdjointThreads;
        fw[u] = x < P.nz ? P.fold[x] : 0u;
    }
    const int2 cb = tid < P.ncomb ? P.comb[tid] : make_int2(0, 0);
    const int2 cb2 = tid < P.ncomb2 ? P.comb2[tid] : make_int2(0, 0);
    double e_hc = 0.0, r1v[2] = {0.0, 0.0};
    if (tid == 0) {
        e_hc = ehc[atom];
        r1v[0] = rho1[(size_t)atom * P.nd];
        if (ND2) r1v[1] = rho1[(size_t)atom * P.nd + 1];
    }
    if (tid == 0) sZ[P.nz] = {1, 0};
    __syncthreads();
    if (P.ny > 0) {
        for (int i = tid; i < P.ny; i += blockDim.x) {
            const int2 pr = P.ypair[i];
            sZ[P.nz + 1 + i] = cmul(sZ[pr.x], sZ[pr.y]);
        }
        __syncthreads();
    }
    // Gather form of the gradient: a thread sums one chunk of contributions
    // w * Z[a] Z[b] Z[c] to a single target x in registers (four 16-byte records per step,
    // loads issued together; the 64 lanes of a wave read consecutive records).  Thread t
    // takes chunks t + kAdjointThreads j; the chunk -> thread mapping must match the record
    // layout built by build_terms.  While the thread's next chunk (round j + 1) has the same
    // target the sum stays in registers; at the end of such a run it is stored: into sW[x]
    // when the chunk is its target's only one, otherwise into the run's slot of the atom's
    // partial sums in global memory, which the pass after the walk adds up per target in slot
    // order.  No atomics: the evaluation is bitwise repeatable.  The walk starts at round rot,
    // a function of the atom's index in the whole system, so that the blocks of an XCD stream
    // different parts of the record table at any moment instead of all reading the same L2
    // lines; a run that crosses from round rot - 1 into round rot is met in two parts, and the
    // first part's sum is held in registers until the walk ends with the second.
    cplx<T>* part = (cplx<T>*)(Pt + (size_t)atom * partials_bytes(P.nslot, P.nd));
    cplx<T>* part2 = part + P.nslot;
    const int nthr = (int)blockDim.x;
    const int nj = (P.nchunks + nthr - 1) / nthr;
    const int rot = nj > 0 ? (int)((unsigned)(atom_base + atom) % (unsigned)nj) : 0;
    cplx<T> acc = {0, 0}, acc2 = {0, 0}, head = {0, 0}, head2 = {0, 0};
    cplx<double> acd = {0, 0}, acd2 = {0, 0};  // ACC: the run's FP64 rounds
    double rho = 0.0, rho2 = 0.0;              // ACC: summed at the flushes
    int j = rot;
    int2 ch = tid + j * nthr < P.nchunks ? P.chunks[tid + j * nthr] : make_int2(0, 0);
    bool split = false;
    if (rot > 0 && tid + rot * nthr < P.nchunks) split = ((P.chunks[tid + (rot - 1) * nthr].y ^ ch.y) & 0xfff) == 0;
    bool hold = split;
    for (int j0 = 0; j0 < nj; ++j0) {
        const int c = tid + j * nthr;
        const int jn = j + 1 < nj ? j + 1 : 0;
        const int cn = tid + jn * nthr;
        const bool has_next = j0 + 1 < nj && cn < P.nchunks;
        const int2 chn = has_next ? P.chunks[cn] : make_int2(0, 0);
        if (c < P.nchunks) {
            const int x = ch.y & 0xfff, cnt = (ch.y >> 12) & 63;
            const bool sole = (ch.y >> 18) & 1;  // the target's only chunk
            // records of this lane, stride 64; FP32 without the recipe reads the table whose
            // offsets need no unpacking
            constexpr bool kU = sizeof(T) == 4 && !ACC;
            const uint4* __restrict__ rec = (kU ? P.crecu : P.crec) + ch.x;
            const T* __restrict__ w2p = ND2 ? P.cw2 + ch.x : nullptr;
            const double* __restrict__ w2d = ND2 && ACC ? P.cw2d + ch.x : nullptr;
            if (ACC && __any(x >= P.oA0 && x < P.nz)) {
                for (int k = 0; k < cnt; k += 4) {
                    uint4 r[4];
                    double w2[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        r[u] = rec[(size_t)(k + u) * 64];
                        if (ND2) w2[u] = w2d[(size_t)(k + u) * 64];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const double w = (double)__uint_as_float(r[u].z) + (double)__uint_as_float(r[u].w);
                        const cplx<T> pr = cmul(cmul(lds_cplx<T>(r[u].x & 0xffff), lds_cplx<T>(r[u].x >> 16)),
                                                lds_cplx<T>(r[u].y));
                        acd.re = fma(w, (double)pr.re, acd.re);
                        acd.im = fma(w, (double)pr.im, acd.im);
                        if (ND2) {
                            acd2.re = fma(w2[u], (double)pr.re, acd2.re);
                            acd2.im = fma(w2[u], (double)pr.im, acd2.im);
                        }
                    }
                }
            } else
            for (int k = 0; k < cnt; k += 4) {
                uint4 r[4];
                T w2[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    r[u] = rec[(size_t)(k + u) * 64];
                    if (ND2) w2[u] = w2p[(size_t)(k + u) * 64];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const T w = kU ? (T)__uint_as_float(r[u].w) : rec_weight<T>(r[u]);
                    // records hold byte offsets into sZ, which starts at LDS address 0
                    const cplx<T> za = lds_cplx<T>(kU ? r[u].x : r[u].x & 0xffff);
                    const cplx<T> zb = lds_cplx<T>(kU ? r[u].y : r[u].x >> 16);
                    const cplx<T> zc = lds_cplx<T>(kU ? r[u].z : r[u].y);
                    const cplx<T> pr = cmul(cmul(za, zb), zc);
                    acc.re = fma(w, pr.re, acc.re);
                    acc.im = fma(w, pr.im, acc.im);
                    if (ND2) {
                        acc2.re = fma(w2[u], pr.re, acc2.re);
                        acc2.im = fma(w2[u], pr.im, acc2.im);
                    }
                }
            }
            if (!(jn == j + 1 && has_next && ((chn.y ^ ch.y) & 0xfff) == 0)) {
                if constexpr (ACC) {  // the run's FP64 and FP32 rounds; rho of an A0 target in FP64
                    const cplx<double> t = {acd.re + (double)acc.re, acd.im + (double)acc.im};
                    const cplx<double> t2 = {acd2.re + (double)acc2.re, acd2.im + (double)acc2.im};
                    if (x >= P.oA0 && x < P.nz) {
                        const cplx<T> z = sZ[x];
                        rho += (double)z.re * t.re - (double)z.im * t.im;
                        if (ND2) rho2 += (double)z.re * t2.re - (double)z.im * t2.im;
                    }
                    acc = {(T)t.re, (T)t.im};
                    acc2 = {(T)t2.re, (T)t2.im};
                    acd = {0, 0};
                    acd2 = {0, 0};
                }
                if (hold) {  // first part of the run split by the start of the walk
                    head = acc;
                    head2 = acc2;
                    hold = false;
                } else {
                    if (split && j0 + 1 == nj) {  // its second part: the whole run
                        acc.re += head.re;
                        acc.im += head.im;
                        acc2.re += head2.re;
                        acc2.im += head2.im;
                    }
                    if (sole) {
                        sW[x] = acc;
                        if (ND2) sW2[x] = acc2;
                    } else {
                        const int slot = (int)((unsigned)ch.y >> 19);
                        part[slot] = acc;
                        if (ND2) part2[slot] = acc2;
                    }
                }
                acc = {0, 0};
                acc2 = {0, 0};
            }
        }
        ch = chn;
        j = jn;
    }
    __syncthreads();  // every run stored: sole targets in sW, the others in their slots
    combine_partials(P, part, sW, cb, cb2);
    if (ND2) {
        __syncthreads();
        combine_partials(P, part2, sW2, cb, cb2);
    }
    __syncthreads();
    // products Y: dRho/dZ[x] += dRho/dY Z[other] for the Y entries that hold Z[x], one thread
    // per target in a fixed order (the targets read only Y entries, and write only their own)
    if (P.nyt > 0) {
        for (int k = tid; k < P.nyt; k += nthr) {
            const int2 e = P.yft[k];
            const int x = e.y & 0xfff, n = e.y >> 12;
            cplx<T> w = sW[x], w2 = ND2 ? sW2[x] : cplx<T>{0, 0};
            for (int u = 0; u < n; ++u) {
                const int2 t = P.yfe[e.x + u];
                cfma(w, sW[t.x], sZ[t.y]);
                if (ND2) cfma(w2, sW2[t.x], sZ[t.y]);
            }
            sW[x] = w;
            if (ND2) sW2[x] = w2;
        }
        __syncthreads();
    }
    // rho = Re sum over A0 targets of Z[x] dRho/dZ[x] (every monomial has exactly one A0
    // factor), summed in FP64 in a fixed order (with ACC: already summed at the flushes)
    if constexpr (!ACC)
        for (int x = P.oA0 + tid; x < P.nz; x += nthr) {
            rho += (double)re_mul(sZ[x], sW[x]);
            if (ND2) rho2 += (double)re_mul(sZ[x], sW2[x]);
        }
    const double tot = block_sum<T>(rho, red);
    double tot2 = 0.0;
    if (ND2) {
        __syncthreads();
        tot2 = block_sum<T>(rho2, red + kAdjointThreads / 64);
    }
    if (tid == 0) {
        const double tots[2] = {tot, tot2};
        atom_energy<T>(P, ND2 ? 2 : 1, atom, tots, e_hc, r1v, eout, dEout, edfout, rho_out, s_scale);
    }
    __syncthreads();
    // W_eff on representatives of conjugate pairs: since Z_xbar = s conj(Z_x),
    // Re(W_x dZ_x + W_xbar dZ_xbar) = Re((W_x + s conj(W_xbar)) dZ_x); zero elsewhere
    // (the reference's half-range loops with factor 2, src/forces.F90:460-614)
    // With ND2 and Wd set (fitting), each density's folded gradient dRho_d/dZ is also written,
    // unscaled: Wd[atom][d][x]
    const T sc = (T)s_scale[0], sc2 = ND2 ? (T)s_scale[1] : (T)0;
    Wout += (size_t)atom * P.nz;
    cplx<T>* wd = ND2 && Wd ? Wd + (size_t)atom * 2 * P.nz : nullptr;
#pragma unroll
    for (int u = 0; u < kFold; ++u) {
        const int x = tid + u * kAdjointThreads;
        if (x >= P.nz) break;
        const uint32_t f = fw[u];
        cplx<T> w = {0, 0}, w2 = {0, 0};
        if (f & (1u << 17)) {
            w = sW[x];
            if (ND2) w2 = sW2[x];
            if (!(f & (1u << 18))) {
                const cplx<T> b = sW[f & 0xffff];
                const T s = (f & (1u << 16)) ? (T)-1 : (T)1;
                w.re += s * b.re;
                w.im -= s * b.im;
                if (ND2) {
                    const cplx<T> b2 = sW2[f & 0xffff];
                    w2.re += s * b2.re;
                    w2.im -= s * b2.im;
                }
            }
        }
        if (!(f & (1u << 19))) continue;  // not stored
        const int h = P.zmap[x];
        Wout[h] = ND2 ? cplx<T>{sc * w.re + sc2 * w2.re, sc * w.im + sc2 * w2.im} : cplx<T>{sc * w.re, sc * w.im};
        if (wd) {
            wd[h] = w;
            wd[P.nz + h] = w2;
        }
    }
}

// Two atoms per block (FP32, one density): the atoms' Z and W are interleaved in LDS
// (float4 = Z0.re, Z0.im, Z1.re, Z1.im), so one 16-byte read fetches a factor for both, and
// each record (byte offsets of 16-byte entries, FP32 weight) is loaded and decoded once for
// both atoms.  Same chunk walk, carry, sole stores and rotation as k_adjoint; an odd last
// atom is paired with itself and its second copy is not written.
template <bool ACC>
__global__ void __launch_bounds__(kAdjointThreads) k_adjoint_pair(DevParams<float> P, int atom_base,
                                                     const uint4* __restrict__ crec16,
                                                     const cplx<float>* __restrict__ Zin,
                                                     cplx<float>* __restrict__ Wout, char* __restrict__ Pt,
                                                     const double* __restrict__ ehc,
                                                     const double* __restrict__ rho1, double* __restrict__ eout,
                                                     double* __restrict__ dEout, double* __restrict__ edfout,
                                                     double* __restrict__ rho_out, int natom) {
    using T = float;
    extern __shared__ __align__(16) unsigned char smem[];
    float4* sZ = (float4*)smem;                  // [nzx] (Z' of k_adjoint), sZ[nz] = (1, 0, 1, 0)
    float4* sW = sZ + P.nzx;                     // [nzx]
    double* red = (double*)(sW + P.nzx);         // [2 * waves]: one sum per atom and wave
    double* s_scale = red + 2 * (kAdjointThreads / 64);  // dynamic LDS, as in k_adjoint
    const int a0 = 2 * (int)blockIdx.x, tid = threadIdx.x;
    const bool two = a0 + 1 < natom;
    const cplx<T>* Z0 = Zin + (size_t)a0 * P.nz;
    const cplx<T>* Z1 = two ? Z0 + P.nz : Z0;
    {
        // Z' of both atoms, with all of a thread's loads issued before the stores
        constexpr int U = 8;  // covers nzx <= 8 * kAdjointThreads = 4096 in one pass
        cplx<T> a[U], b[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int x = tid + u * kAdjointThreads;
            const uint32_t e = x < P.nz ? P.zmap[x] : 0u;
            a[u] = x < P.nz ? full_entry(Z0, e) : cplx<T>{0, 0};
            b[u] = x < P.nz ? full_entry(Z1, e) : cplx<T>{0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int x = tid + u * kAdjointThreads;
            if (x < P.nz) sZ[x] = make_float4(a[u].re, a[u].im, b[u].re, b[u].im);
            if (x < P.nzx) sW[x] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    }
    // the tail's inputs from global memory, loaded now (as in k_adjoint); the two atoms'
    // energies are evaluated by threads 0 and 64 (two waves) at the same time
    constexpr int kFold = 8;
    uint32_t fw[kFold];
#pragma unroll
    for (int u = 0; u < kFold; ++u) {
        const int x = tid + u * kAdjointThreads;
        fw[u] = x < P.nz ? P.fold[x] : 0u;
    }
    const int2 cb = tid < P.ncomb ? P.comb[tid] : make_int2(0, 0);
    const int2 cb2 = tid < P.ncomb2 ? P.comb2[tid] : make_int2(0, 0);
    const int eatom = tid == 0 ? a0 : tid == 64 && two ? a0 + 1 : -1;  // the atom whose energy this thread evaluates
    double e_hc = 0.0, r1v = 0.0;
    if (eatom >= 0) {
        e_hc = ehc[eatom];
        r1v = rho1[eatom];
    }
    if (tid == 0) sZ[P.nz] = make_float4(1.f, 0.f, 1.f, 0.f);
    __syncthreads();
    if (P.ny > 0) {
        for (int i = tid; i < P.ny; i += blockDim.x) {
            const int2 pr = P.ypair[i];
            const float4 a = sZ[pr.x], b = sZ[pr.y];
            const cplx<T> y0 = cmul(cplx<T>{a.x, a.y}, cplx<T>{b.x, b.y});
            const cplx<T> y1 = cmul(cplx<T>{a.z, a.w}, cplx<T>{b.z, b.w});
            sZ[P.nz + 1 + i] = make_float4(y0.re, y0.im, y1.re, y1.im);
        }
        __syncthreads();
    }
    // the walk, runs, slots and rotation of k_adjoint; a slot holds both atoms' sums
    float4* part = (float4*)(Pt + (size_t)blockIdx.x * partials_bytes(P.nslot, 1));
    const int nthr = (int)blockDim.x;
    const int nj = (P.nchunks + nthr - 1) / nthr;
    const int rot = nj > 0 ? (int)((unsigned)((atom_base >> 1) + (int)blockIdx.x) % (unsigned)nj) : 0;
    cplx<T> acc0 = {0, 0}, acc1 = {0, 0}, head0 = {0, 0}, head1 = {0, 0};
    cplx<double> acd0 = {0, 0}, acd1 = {0, 0};  // ACC: the run's FP64 rounds (k_adjoint's ACC)
    double rho0 = 0.0, rho1s = 0.0;             // ACC: summed at the flushes
    int j = rot;
    int2 ch = tid + j * nthr < P.nchunks ? P.chunks[tid + j * nthr] : make_int2(0, 0);
    bool split = false;
    if (rot > 0 && tid + rot * nthr < P.nchunks) split = ((P.chunks[tid + (rot - 1) * nthr].y ^ ch.y) & 0xfff) == 0;
    bool hold = split;
    for (int j0 = 0; j0 < nj; ++j0) {
        const int c = tid + j * nthr;
        const int jn = j + 1 < nj ? j + 1 : 0;
        const int cn = tid + jn * nthr;
        const bool has_next = j0 + 1 < nj && cn < P.nchunks;
        const int2 chn = has_next ? P.chunks[cn] : make_int2(0, 0);
        if (c < P.nchunks) {
            const int x = ch.y & 0xfff, cnt = (ch.y >> 12) & 63;
            const bool sole = (ch.y >> 18) & 1;
            const uint4* __restrict__ rec = crec16 + ch.x;
            if (ACC && __any(x >= P.oA0 && x < P.nz)) {
                for (int k = 0; k < cnt; k += 4) {
                    uint4 r[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) r[u] = rec[(size_t)(k + u) * 64];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        const double w = (double)__uint_as_float(r[u].z) + (double)__uint_as_float(r[u].w);
                        const float4 za = lds_f4(r[u].x & 0xffff);
                        const float4 zbv = lds_f4(r[u].x >> 16);
                        const float4 zc = lds_f4(r[u].y);
                        const cplx<T> p0 = cmul(cmul(cplx<T>{za.x, za.y}, cplx<T>{zbv.x, zbv.y}), cplx<T>{zc.x, zc.y});
                        const cplx<T> p1 = cmul(cmul(cplx<T>{za.z, za.w}, cplx<T>{zbv.z, zbv.w}), cplx<T>{zc.z, zc.w});
                        acd0.re = fma(w, (double)p0.re, acd0.re);
                        acd0.im = fma(w, (double)p0.im, acd0.im);
                        acd1.re = fma(w, (double)p1.re, acd1.re);
                        acd1.im = fma(w, (double)p1.im, acd1.im);
                    }
                }
            } else
            for (int k = 0; k < cnt; k += 4) {
                uint4 r[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) r[u] = rec[(size_t)(k + u) * 64];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    // without the recipe the table's offsets need no unpacking (crec16u)
                    const T w = __uint_as_float(ACC ? r[u].z : r[u].w);
                    const float4 za = lds_f4(ACC ? r[u].x & 0xffff : r[u].x);
                    const float4 zbv = lds_f4(ACC ? r[u].x >> 16 : r[u].y);
                    const float4 zc = lds_f4(ACC ? r[u].y : r[u].z);
                    const cplx<T> p0 = cmul(cmul(cplx<T>{za.x, za.y}, cplx<T>{zbv.x, zbv.y}), cplx<T>{zc.x, zc.y});
                    const cplx<T> p1 = cmul(cmul(cplx<T>{za.z, za.w}, cplx<T>{zbv.z, zbv.w}), cplx<T>{zc.z, zc.w});
                    acc0.re = fma(w, p0.re, acc0.re);
                    acc0.im = fma(w, p0.im, acc0.im);
                    acc1.re = fma(w, p1.re, acc1.re);
                    acc1.im = fma(w, p1.im, acc1.im);
                }
            }
            if (!(jn == j + 1 && has_next && ((chn.y ^ ch.y) & 0xfff) == 0)) {
                if constexpr (ACC) {
                    const cplx<double> t0 = {acd0.re + (double)acc0.re, acd0.im + (double)acc0.im};
                    const cplx<double> t1 = {acd1.re + (double)acc1.re, acd1.im + (double)acc1.im};
                    if (x >= P.oA0 && x < P.nz) {
                        const float4 z = sZ[x];
                        rho0 += (double)z.x * t0.re - (double)z.y * t0.im;
                        rho1s += (double)z.z * t1.re - (double)z.w * t1.im;
                    }
                    acc0 = {(T)t0.re, (T)t0.im};
                    acc1 = {(T)t1.re, (T)t1.im};
                    acd0 = {0, 0};
                    acd1 = {0, 0};
                }
                if (hold) {
                    head0 = acc0;
                    head1 = acc1;
                    hold = false;
                } else {
                    if (split && j0 + 1 == nj) {
                        acc0.re += head0.re;
                        acc0.im += head0.im;
                        acc1.re += head1.re;
                        acc1.im += head1.im;
                    }
                    const float4 v = make_float4(acc0.re, acc0.im, acc1.re, acc1.im);
                    if (sole)
                        sW[x] = v;
                    else
                        part[(unsigned)ch.y >> 19] = v;
                }
                acc0 = {0, 0};
                acc1 = {0, 0};
            }
        }
        ch = chn;
        j = jn;
    }
    __syncthreads();
    combine_partials(P, part, sW, cb, cb2);
    __syncthreads();
    if (P.nyt > 0) {  // products Y, as in k_adjoint
        for (int k = tid; k < P.nyt; k += nthr) {
            const int2 e = P.yft[k];
            const int x = e.y & 0xfff, n = e.y >> 12;
            float4 w = sW[x];
            for (int u = 0; u < n; ++u) {
                const int2 t = P.yfe[e.x + u];
                const float4 g = sW[t.x], z = sZ[t.y];
                cplx<T> w0 = {w.x, w.y}, w1 = {w.z, w.w};
                cfma(w0, cplx<T>{g.x, g.y}, cplx<T>{z.x, z.y});
                cfma(w1, cplx<T>{g.z, g.w}, cplx<T>{z.z, z.w});
                w = make_float4(w0.re, w0.im, w1.re, w1.im);
            }
            sW[x] = w;
        }
        __syncthreads();
    }
    if constexpr (!ACC)
        for (int x = P.oA0 + tid; x < P.nz; x += nthr) {
            const float4 z = sZ[x], w = sW[x];
            rho0 += (double)re_mul(cplx<T>{z.x, z.y}, cplx<T>{w.x, w.y});
            rho1s += (double)re_mul(cplx<T>{z.z, z.w}, cplx<T>{w.z, w.w});
        }
    const double tot0 = block_sum<T>(rho0, red);
    __syncthreads();
    double tot1 = block_sum<T>(rho1s, red + kAdjointThreads / 64);  // valid on thread 0
    if (tid == 64) {  // the second atom's sum, from the same partials in the same order
        tot1 = 0.0;
        for (int i = 0; i < kAdjointThreads / 64; ++i) tot1 += red[kAdjointThreads / 64 + i];
    }
    if (eatom >= 0) {
        double sc[1];
        const double t[1] = {eatom == a0 ? tot0 : tot1};
        atom_energy<T>(P, 1, eatom, t, e_hc, &r1v, eout, dEout, edfout, rho_out, sc);
        s_scale[eatom - a0] = sc[0];
    }
    __syncthreads();
    // W_eff on representatives of conjugate pairs, as in k_adjoint
    const T sc0 = (T)s_scale[0], sc1 = two ? (T)s_scale[1] : (T)0;
    cplx<T>* W0 = Wout + (size_t)a0 * P.nz;
    cplx<T>* W1 = W0 + P.nz;
#pragma unroll
    for (int u = 0; u < kFold; ++u) {
        const int x = tid + u * kAdjointThreads;
        if (x >= P.nz) break;
        const uint32_t f = fw[u];
        float4 w = make_float4(0.f, 0.f, 0.f, 0.f);
        if (f & (1u << 17)) {
            w = sW[x];
            if (!(f & (1u << 18))) {
                const float4 b = sW[f & 0xffff];
                const T sg = (f & (1u << 16)) ? (T)-1 : (T)1;
                w.x += sg * b.x;
                w.y -= sg * b.y;
                w.z += sg * b.z;
                w.w -= sg * b.w;
            }
        }
        if (!(f & (1u << 19))) continue;  // not stored
        const int h = P.zmap[x];
        W0[h] = cplx<T>{sc0 * w.x, sc0 * w.y};
        if (two) W1[h] = cplx<T>{sc1 * w.z, sc1 * w.w};
    }
}

// ============================================================================ fitting
// Gradient of L = sum_s gE_s E_s + sum_j gF_j . F_j with respect to the expansion
// coefficients (the contraction of src/forces.F90:93-141 run backwards): with
// E_i = fc(e_hc) F(rho_i) + e_hc and rho_i = sum_k c_k B_k,i,
//   dL/dc_k = sum_i [alpha_i B_k,i + beta_i D_u B_k,i],  u = gF (a displacement field),
//   alpha_i = gE_s(i) fc F' - fc F'' D_u rho_i - F' D_u fc,   beta_i = -fc F'
// (F_j = -dE/dx_j, so sum_j gF_j . dF_j/dc = -D_u dE/dc).  B_k = Re sum_t u_{k,t} P_t with
// P_t = prod Z[idx_t]; D_u P_t follows from Zdot = D_u Z, the forward-mode derivative of the
// density along u.  FP64 only.

// F, F' and F'' of the embedding (src/forces.F90:1134-1233)
__device__ inline void embed2(int nfemb, double rho, double wpre, double mexp, double& F, double& dF,
                              double& d2F) {
    embed(nfemb, rho, wpre, mexp, F, dF);
    d2F = 0.0;
    if (nfemb == 0) return;
    const double w = 10.0, eps = 1e-10;
    const double s = nfemb == 2 ? 1.0 + rho : rho;
    if (!(fabs(s) > eps)) return;
    const double a = fabs(s), sg = s >= 0.0 ? 1.0 : -1.0;
    const double y0 = w * s * s;
    const double g = y0 > 30.0 ? 0.0 : exp(-y0);
    const double g1 = -2.0 * w * s * g, g2 = -2.0 * w * g + 4.0 * w * w * s * s * g;
    const double q = (1.0 - g) * a, q1 = -g1 * a + (1.0 - g) * sg, q2 = -g2 * a - 2.0 * g1 * sg;
    double y1pp = 0.0;
    if (q > 0.0) y1pp = mexp * (mexp - 1.0) * pow(q, mexp - 2.0) * q1 * q1 + mexp * pow(q, mexp - 1.0) * q2;
    const double y2pp = mexp * (g2 * a + 2.0 * g1 * sg);
    d2F = wpre * sg * (y1pp + y2pp);
}

__device__ inline void inner_cutoff(double e, double ecut, double decut, double& fc, double& dfc) {
    const double elow = ecut - decut;
    fc = 1.0;
    dfc = 0.0;
    if (e >= ecut) {
        fc = 0.0;
    } else if (e > elow) {
        const double pi = 3.14159265358979323846;
        fc = 0.5 * (1.0 + cos(pi * (e - elow) / decut));
        dfc = -0.5 * sin(pi * (e - elow) / decut) * pi / decut;
    }
}

// alpha_{i,d}, beta_{i,d} (one block per atom), the factors of B_{k,i} and D_u B_{k,i} in
// dL/dc_{k,d} for L = sum_s gE_s E_s - D_u E:
//   alpha = gE fc F'_d - fc F''_d D_u rho_d - F'_d dfc D_u e_hc,  beta = -fc F'_d.
// D_u rho_d = Re sum_x G_x Zdot_x over the representatives of conjugate pairs, G = drho_d/dZ
// folded (the conjugate symmetry of Zdot allows it): with one density G = W, or W / (fc F') where
// the adjoint scaled it, with two the adjoint's per-density output Wd[atom][d].
template <int ND>
__global__ void __launch_bounds__(256) k_fit_atom(DevParams<double> P, bool scaled, const cplx<double>* __restrict__ W,
                                                 const cplx<double>* __restrict__ Zdot,
                                                 const double* __restrict__ rho, const double* __restrict__ ehc,
                                                 const double* __restrict__ ehc_dot,
                                                 const int* __restrict__ atom_struct,
                                                 const double* __restrict__ gE, double* __restrict__ alpha,
                                                 double* __restrict__ beta) {
    __shared__ double red[8];
    const int atom = blockIdx.x;
    double tot[ND];
    const cplx<double>* zd = Zdot + (size_t)atom * P.nz;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        const cplx<double>* w = W + ((size_t)atom * ND + d) * P.nz;
        double s = 0.0;
        for (int x = threadIdx.x; x < P.nzh; x += blockDim.x) s += re_mul(w[x], zd[x]);
        tot[d] = block_sum<double>(s, red);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        double fc, dfc;
        inner_cutoff(ehc[atom], P.ecut, P.decut, fc, dfc);
        const double g = atom_struct ? gE[atom_struct[atom]] : 0.0;
#pragma unroll
        for (int d = 0; d < ND; ++d) {
            double F, dF, d2F;
            embed2(P.nfemb, rho[(size_t)atom * ND + d], P.p1[d][0], P.p1[d][1], F, dF, d2F);
            const double sc = fc * dF;
            const double rho_dot = ND == 2 || !scaled ? tot[d] : (sc != 0.0 ? tot[d] / sc : 0.0);
            alpha[(size_t)atom * ND + d] = g * fc * dF - fc * d2F * rho_dot - dF * dfc * ehc_dot[atom];
            beta[(size_t)atom * ND + d] = -fc * dF;
        }
    }
}

// gradient of the B1 coefficients: grad[d * nb_m + n] = sum_i alpha_{i,d} (g^m_n(mu_i) - 1)
__global__ void k_fit_b1(DevParams<double> P, int natom, int nd, const double* __restrict__ dmomi,
                         const double* __restrict__ alpha, double* __restrict__ grad, int* err) {
    const int atom = blockIdx.x * blockDim.x + threadIdx.x;
    if (atom >= natom) return;
    double w;
    bool unit;
    const double* row = magnetic_row(P, dmomi[atom], w, unit, err);
    for (int n = 0; n < P.nb_m; ++n) {
        double v = unit ? 1.0 : 0.0, dv;
        if (row) horner(row + 4 * n, w, P.rs_m, v, dv);
        for (int d = 0; d < nd; ++d) atomicAdd(&grad[d * P.nb_m + n], alpha[(size_t)atom * nd + d] * (v - 1.0));
    }
}

// gradient of the coefficients of orders 2..6: function k of the concatenated list (nb.n[0]
// functions of order 2, ..., nb.n[4] of order 6), density d: sum_t u_{k,t} M_{t,d}, stored at
// grad[nd * (functions of lower orders) + d * nb.n[o] + j] (the file's order: per body order,
// density-major); grid.y = density
struct OrderCounts {
    int n[5];
};
__global__ void k_fit_grad(int nterms, OrderCounts nb, const int* __restrict__ ptr, const int* __restrict__ tt,
                           const double* __restrict__ uu, const double* __restrict__ M, double* __restrict__ grad) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x, d = blockIdx.y, nd = gridDim.y;
    int lower = 0, o = 0;
    while (o < 5 && k >= lower + nb.n[o]) lower += nb.n[o++];
    if (o == 5) return;
    const double* Md = M + (size_t)d * nterms;
    double s = 0.0;
    for (int e = ptr[k]; e < ptr[k + 1]; ++e) s += uu[e] * Md[tt[e]];
    grad[nd * lower + d * nb.n[o] + (k - lower)] = s;
}

// per-atom forces f_i = -sum_p F_p (own pairs) + sum_{p: j(p) = i} F_p, and per-structure
// energies (atomics; outputs zeroed by the caller)
// Sixteen lanes an atom, kAsmAtoms atoms a workgroup.  The neighbours' parts meet in LDS, in a window of kAsmWindow
// atoms about the workgroup's own (a structure of up to 768 atoms lies in it, and the near planes of a larger one), and
// the window's sums then go to memory; neighbours outside it are added there directly.  62000
// atoms of 57 neighbours: 430 us with every addition in memory, 74 us.
constexpr int kAsmAtoms = 256, kAsmWindow = 1792, kAsmThreads = 1024;
__global__ void __launch_bounds__(kAsmThreads) k_fit_assemble(int natom, const int* __restrict__ off,
                                                      const int* __restrict__ nlist, const double* __restrict__ flist,
                                                      const double* __restrict__ eout,
                                                      const int* __restrict__ atom_struct, double* __restrict__ f,
                                                      double* __restrict__ estruct) {
    constexpr int kRow = 16;
    __shared__ double win[3 * kAsmWindow];
    const int lane = threadIdx.x % kRow;
    const int a0 = blockIdx.x * kAsmAtoms, lo = a0 - (kAsmWindow - kAsmAtoms) / 2;
    for (int x = threadIdx.x; x < 3 * kAsmWindow; x += kAsmThreads) win[x] = 0.0;
    __syncthreads();
    for (int i = a0 + (int)threadIdx.x / kRow; i < min(natom, a0 + kAsmAtoms); i += kAsmThreads / kRow) {
        double s[3] = {0, 0, 0};
        const int end = off[i + 1];
        for (int p = off[i] + lane; p < end; p += kRow) {
            const int j = nlist[p];
            const bool in = j >= lo && j < lo + kAsmWindow;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const double a = flist[3 * (size_t)p + k];
                s[k] -= a;
                if (in)
                    atomicAdd(&win[3 * (j - lo) + k], a);
                else
                    atomicAdd(&f[3 * (size_t)j + k], a);
            }
        }
#pragma unroll
        for (int o = kRow / 2; o > 0; o >>= 1)
#pragma unroll
            for (int k = 0; k < 3; ++k) s[k] += __shfl_xor(s[k], o, kRow);
        if (lane < 3) atomicAdd(&win[3 * (i - lo) + lane], lane == 0 ? s[0] : lane == 1 ? s[1] : s[2]);
        if (lane == 0 && estruct) atomicAdd(&estruct[atom_struct[i]], eout[i]);
    }
    __syncthreads();
    for (int x = threadIdx.x; x < 3 * kAsmWindow; x += kAsmThreads)
        if (win[x] != 0.0) atomicAdd(&f[3 * (long long)lo + x], win[x]);  // only atoms that exist have sums
}

__global__ void k_fill_double(double* __restrict__ p, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

hipError_t fit_backward(const DevParams<double>& P, bool scaled, int natom, const int* off, const int* nlist,
                        const double* du, const double* dlist, const double* elist, const double* dmomi,
                        const double* dmom, const double* emom, const int* atom_struct, const double* gE,
                        Buffers& B, FitBuffers& F, int nterms, const int* nbo5, double* grad, hipStream_t s) {
    if (natom <= 0) return hipSuccess;
    const int nd = P.nd == 2 ? 2 : 1;
    if (nd == 2 && !B.Wd) return hipErrorInvalidValue;
    OrderCounts nbo;
    int nb234 = 0;
    for (int o = 0; o < 5; ++o) nb234 += (nbo.n[o] = nbo5[o]);
    hipError_t e = run_density_jvp(P, natom, off, nlist, du, dlist, elist, dmom, emom, F.Zdot, F.ehc_dot, B.err, s);
    if (e != hipSuccess) return e;
    if (nd == 2)
        hipLaunchKernelGGL(k_fit_atom<2>, dim3(natom), dim3(256), 0, s, P, scaled, (const cplx<double>*)B.Wd,
                           (const cplx<double>*)F.Zdot, B.rho, B.ehc, F.ehc_dot, atom_struct, gE, F.alpha, F.beta);
    else
        hipLaunchKernelGGL(k_fit_atom<1>, dim3(natom), dim3(256), 0, s, P, scaled, (const cplx<double>*)B.W,
                           (const cplx<double>*)F.Zdot, B.rho, B.ehc, F.ehc_dot, atom_struct, gE, F.alpha, F.beta);
    const size_t nM = (size_t)nterms * nd;
    hipLaunchKernelGGL(k_fill_double, dim3((unsigned)((nM + 255) / 256)), dim3(256), 0, s, F.M, nM);
    const size_t ng = ((size_t)P.nb_m + nb234) * nd;
    hipLaunchKernelGGL(k_fill_double, dim3((unsigned)((ng + 255) / 256)), dim3(256), 0, s, grad, ng);
    if ((e = fit_accumulate(F.plan, P.nz, nterms, nd, natom, B.Z, F.Zdot, F.alpha, F.beta, F.M, s)) != hipSuccess) return e;
    hipLaunchKernelGGL(k_fit_b1, dim3((natom + 255) / 256), dim3(256), 0, s, P, natom, nd, dmomi, F.alpha, grad,
                       B.err);
    if (nb234 > 0)
        hipLaunchKernelGGL(k_fit_grad, dim3((nb234 + 255) / 256, nd), dim3(256), 0, s, nterms, nbo, F.ub_ptr, F.ub_t,
                           F.ub_u, F.M, grad + (size_t)nd * P.nb_m);
    return hipGetLastError();
}

hipError_t fit_assemble(int natom, const int* off, const int* nlist, const double* flist, const double* eout,
                        const int* atom_struct, int nstruc, double* f, double* estruct, hipStream_t s) {
    const size_t nf = 3 * (size_t)natom;
    if (nf) hipLaunchKernelGGL(k_fill_double, dim3((unsigned)((nf + 255) / 256)), dim3(256), 0, s, f, nf);
    if (estruct && nstruc > 0)
        hipLaunchKernelGGL(k_fill_double, dim3((unsigned)((nstruc + 255) / 256)), dim3(256), 0, s, estruct,
                           (size_t)nstruc);
    if (natom > 0)
        hipLaunchKernelGGL(k_fit_assemble, dim3((unsigned)((natom + kAsmAtoms - 1) / kAsmAtoms)), dim3(kAsmThreads), 0, s, natom,
                           off, nlist, flist, eout, atom_struct, f, estruct);
    return hipGetLastError();
}

// ============================================================================ launch
__global__ void k_clear_flags(int* p) { *p = 0; }

// n slots of 16 bytes; then *flag_out = *flag, or *flag = 0 where there is no flag_out
__global__ void __launch_bounds__(256) k_copy_slots(const uint4* __restrict__ src, uint4* __restrict__ dst, int n, int* flag,
                                                    int* flag_out) {
    constexpr int U = 4;  // in flight a thread: a trip to host memory takes microseconds
    const int i0 = blockIdx.x * (U * 256) + threadIdx.x;
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = src[min(i0 + 256 * u, n - 1)];
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (i0 + 256 * u < n) dst[i0 + 256 * u] = v[u];
    if (i0 == 0) {
        if (flag_out)
            *flag_out = *flag;
        else
            *flag = 0;
    }
}

hipError_t copy_slots(const void* src, void* dst, size_t n, int* flag, int* flag_out, hipStream_t s) {
    if (n == 0 || n > (size_t)1 << 24) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_copy_slots, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, (const uint4*)src, (uint4*)dst,
                       (int)n, flag, flag_out);
    return hipGetLastError();
}

hipError_t clear_flags(int* p, hipStream_t s) {
    // a kernel rather than hipMemsetAsync, so that the evaluation can be captured in a graph
    hipLaunchKernelGGL(k_clear_flags, dim3(1), dim3(1), 0, s, p);
    return hipGetLastError();
}

// shape classes: 0 = small magnetic A block (nm3 <= 4, nr2m <= 2, nb_a <= 10, nr3a <= 8, l <= 6)
//                1 = wide magnetic A block  (nm3 <= 27, nr2m <= 5, nb_a <= 16, nr3a <= 4, l <= 2)
//                2 = medium magnetic A block at l <= 6 (nm3 <= 9, nr2m <= 5, nb_a <= 16, nr3a <= 8)
int supported_nm3_class(int nm3, int nr2m, int nb_a, int l3a, int l2m, int nr3a) {
    if (nb_a > 16) return -1;
    if (nm3 <= 4 && nr2m <= 2 && l3a <= 6 && l2m <= 6 && nr3a <= 8 && nb_a <= 10) return 0;
    if (nm3 <= 27 && nr2m <= 5 && l3a <= 2 && l2m <= 2 && nr3a <= 4) return 1;
    if (nm3 <= 9 && nr2m <= 5 && l3a <= 6 && l2m <= 6 && nr3a <= 8) return 2;
    return -1;
}

template <typename T, int L, int CH, bool SPLIT, bool TASKSPLIT, int NB, int NM3X, int NB2, int NR2X, int NRAX, int NBAX,
          bool ACC>
static hipError_t run_class(const DevParams<T>& P, const NodeTab<T>& N, int natom, int atom_base, const int* off, const double* dlist,
                            const double* elist, const double* dmomi, const double* emomi,
                            const double* dmom, const double* emom, double* eout, double* flist,
                            double* tlist, double* tlist0, Buffers& B, hipStream_t s, hipEvent_t* ev) {
    DevParams<double> Pd;  // only the dims are used for LDS sizing
    Pd.nr3a = P.nr3a; Pd.l3a = P.l3a; Pd.nr2m = P.nr2m; Pd.l2m = P.l2m; Pd.lha = P.lha;
    Pd.lhm = P.lhm; Pd.nm3 = P.nm3; Pd.nb_a = P.nb_a; Pd.nb_m = P.nb_m;
    const size_t lds1 = density_lds_bytes(Pd, CH, sizeof(T));
    static_assert(!ACC || sizeof(T) == 4, "the accumulation recipe belongs to the FP32 kernels");
    // the accumulation recipe's density; the others run on the matrix cores (density.hip)
    const void* k1 = nullptr;
    if constexpr (ACC) k1 = (const void*)k_density<T, L, CH, NB, NM3X, NB2, NR2X, SPLIT, TASKSPLIT>;
    const bool nd2 = P.nd == 2;
    hipError_t e = hipSuccess;
    // the dynamic-LDS limit is raised once per kernel instantiation (to the workgroup
    // maximum), so that evaluations can be captured into graphs without further API calls.
    // limit[]: 0 density, 1 adjoint, 2 adjoint with two densities, 3 two-atom adjoint
    static bool attributes_set = false;
    static size_t limit[4] = {0, 0, 0, 0};
    if (!attributes_set) {
        int dev = 0, maxsh = 0;
        if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
        if ((e = hipDeviceGetAttribute(&maxsh, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) != hipSuccess)
            return e;
        const void* ks[4] = {k1, (const void*)k_adjoint<T, false, ACC>, (const void*)k_adjoint<T, true, ACC>, nullptr};
        if constexpr (sizeof(T) == 4) ks[3] = (const void*)k_adjoint_pair<ACC>;
        for (int i = 0; i < 4; ++i) {
            if (!ks[i]) continue;
            hipFuncAttributes fa;
            if ((e = hipFuncGetAttributes(&fa, ks[i])) != hipSuccess) return e;
            // the adjoints address their dynamic LDS from 0 (lds_at)
            if (i >= 1 && i <= 3 && fa.sharedSizeBytes != 0) return hipErrorInvalidKernelFile;
            limit[i] = (size_t)maxsh > fa.sharedSizeBytes ? (size_t)maxsh - fa.sharedSizeBytes : 0;
            if ((e = hipFuncSetAttribute(ks[i], hipFuncAttributeMaxDynamicSharedMemorySize, (int)limit[i])) !=
                hipSuccess)
                return e;
        }
        attributes_set = true;
    }
    // FP32 with one density: two atoms per adjoint block (their Z and W interleaved in LDS)
    const bool pair = sizeof(T) == 4 && !nd2 && P.crec16 != nullptr;
    const size_t lds2p = 2 * (size_t)P.nzx * 16 + (2 * (kAdjointThreads / 64) + 2) * sizeof(double);
    const size_t lds2 =
        (nd2 ? 3 : 2) * (size_t)P.nzx * sizeof(cplx<T>) + (2 * (kAdjointThreads / 64) + 2) * sizeof(double);
    // the node plan where the potential has one; the accumulation recipe keeps the record walk, whose
    // FP64 sums over monomial products it is defined by
    const bool nodes = N.nw > 0 && !ACC;
    if (!nodes && pair && lds2p > limit[3]) return hipErrorInvalidValue;
    if ((ACC && lds1 > limit[0]) || (!nodes && lds2 > limit[nd2 ? 2 : 1]))
        return hipErrorInvalidValue;
    if (ev) (void)hipEventRecord(ev[0], s);
    if constexpr (ACC) {
        hipLaunchKernelGGL((k_density<T, L, CH, NB, NM3X, NB2, NR2X, SPLIT, TASKSPLIT>), dim3(natom), dim3(256), lds1, s, P,
                           off, dlist, elist, dmomi, emomi, dmom, emom, (cplx<T>*)B.Z, B.ehc, B.rho1, B.err);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    } else if ((e = run_density<T>(P, natom, off, dlist, elist, dmomi, emomi, dmom, emom, B, s)) != hipSuccess) {
        return e;
    }
    if (ev) (void)hipEventRecord(ev[1], s);
    if (nodes && (e = run_adjoint_nodes<T>(P, N, natom, B, eout, s)) != hipSuccess) return e;
    if constexpr (sizeof(T) == 4) {
        if (!nodes && pair)
            hipLaunchKernelGGL(k_adjoint_pair<ACC>, dim3((natom + 1) / 2), dim3(kAdjointThreads), lds2p, s, P, atom_base,
                               ACC ? P.crec16 : P.crec16u, (const cplx<T>*)B.Z, (cplx<T>*)B.W, (char*)B.Pt, B.ehc, B.rho1, eout, B.dE,
                               B.edf, B.rho, natom);
    }
    if (nodes || pair) {
    } else if (nd2)
        hipLaunchKernelGGL((k_adjoint<T, true, ACC>), dim3(natom), dim3(kAdjointThreads), lds2, s, P, atom_base,
                           (const cplx<T>*)B.Z, (cplx<T>*)B.W, (cplx<T>*)B.Wd, (char*)B.Pt, B.ehc, B.rho1, eout,
                           B.dE, B.edf, B.rho);
    else
        hipLaunchKernelGGL((k_adjoint<T, false, ACC>), dim3(natom), dim3(kAdjointThreads), lds2, s, P, atom_base,
                           (const cplx<T>*)B.Z, (cplx<T>*)B.W, (cplx<T>*)nullptr, (char*)B.Pt, B.ehc, B.rho1, eout,
                           B.dE, B.edf, B.rho);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (ev) (void)hipEventRecord(ev[2], s);
    if (B.forces && (e = run_forces<T>(P, natom, off, dlist, elist, dmomi, emomi, dmom, emom, B, !nodes, flist, tlist, tlist0, s)) !=
        hipSuccess)
        return e;
    if (ev) (void)hipEventRecord(ev[3], s);
    return hipGetLastError();
}

template <typename T>
hipError_t Launch<T>::run(const DevParams<T>& P, const NodeTab<T>& N, int natom, int atom_base, const int* off, const double* dlist,
                          const double* elist, const double* dmomi, const double* emomi,
                          const double* dmom, const double* emom, double* eout, double* flist,
                          double* tlist, double* tlist0, Buffers& B, hipStream_t s, int cls,
                          hipEvent_t* ev, int dvar, bool acc) {
    if (natom <= 0) return hipSuccess;
    // Density staging: with many radial functions per pair (lmax-6 headers) or in FP64 the
    // per-pair staging is spread over the whole block, 32 neighbours per round; light FP32
    // headers stage 64 neighbours per round, one thread per pair and side (measured on the
    // 16000-atom workload: lmax 6 0.91 vs 1.07 ms, lmax 4 0.80 vs 0.60 ms).  Light headers
    // also split their A-column tasks over idle threads (lmax 4: FP32 0.61 -> 0.52 ms, FP64
    // 0.93 -> 0.81 ms; with lmax 6 the runtime split costs FP64 3%).
    const bool heavy = P.nb_a + P.nr3a * (P.l3a + 1) >= 40;
#define MAGACE_RUN_ACC(CH, SPLIT, TS, ACC)                                                                     \
    (cls == 0   ? run_class<T, 6, CH, SPLIT, TS, 4, 4, 4, 2, 8, 10, ACC>(P, N, natom, atom_base, off, dlist, elist,      \
                                                                         dmomi, emomi, dmom, emom, eout, flist,      \
                                                                         tlist, tlist0, B, s, ev)                    \
     : cls == 1 ? run_class<T, 2, CH, SPLIT, TS, 1, 27, 2, 5, 4, 16, ACC>(P, N, natom, atom_base, off, dlist, elist,     \
                                                                          dmomi, emomi, dmom, emom, eout, flist,     \
                                                                          tlist, tlist0, B, s, ev)                   \
                : run_class<T, 6, CH, SPLIT, TS, 4, 9, 4, 5, 8, 16, ACC>(P, N, natom, atom_base, off, dlist, elist,      \
                                                                         dmomi, emomi, dmom, emom, eout, flist,      \
                                                                         tlist, tlist0, B, s, ev))
    if constexpr (sizeof(T) == 4) {
        if (acc) {
            // the accumulation recipe's density staging: a variant chosen by the tuner (kDensityVariants)
            // replaces the rule
            if (dvar < 0) dvar = heavy ? 0 : 2;
            if (dvar == 0) return MAGACE_RUN_ACC(32, true, false, true);
            if (dvar == 1) return MAGACE_RUN_ACC(32, true, true, true);
            return MAGACE_RUN_ACC(64, false, true, true);
        }
    }
    return MAGACE_RUN_ACC(32, true, false, false);
#undef MAGACE_RUN_ACC
}

template struct Launch<double>;
template struct Launch<float>;

}  // namespace magace
