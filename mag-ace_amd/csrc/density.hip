// density.hip -- A, A2, A0 of every atom on the matrix cores, and their derivative along a displacement.
//
// k_density_mm does the work of prepA (src/a_basis.F90:59-359).  With R_{l,n} = sum_k C_{nlk} g_k the sums
// over neighbours are taken for the base functions first,
//   B[k][lm,q] = sum_j g_k(j) Y_lm(j) H_q(j),   A[n][lm][q] = sum_k C_{nlk} B[k][lm,q],
//   A2[k][n'][l'm'] = sum_j g_k(j) M_{l',n'}(j) Y_l'm'(j),
// which is one product G^T F of the pairs' base functions (at most 16 rows) with all columns, and a small
// one with C whose B operand is the first one's result as it lies in the registers.  Only the g_k (10 for
// the lmax-6 header) are looked up for a pair, in a table of their own that stays in L2, where the 49
// R_{l,n} had to come from a table six times as large.  Where the C cancel, or where there are no more R than g, A is
// summed over radial factors h_f in place of the g_k (RadialFactors), A = U B, and both are looked up.
//
// Measured against the kernel that staged all R_{l,n} and summed on the vector units (us): 16000 atoms
// lmax 6 mixed 403 -> 248, FP64 735 -> 470; 27648 atoms lmax 4 mixed 494 -> 268, FP64 855 -> 474; 4394 atoms
// of the example potential's shape, with its factors, 161 -> 75 and 338 -> 132 (through the g 78 and 110); 128 atoms
// lmax 4 FP64 24.4 -> 12.4.  Of the 248 the matrix cores issue for 90 and the vector units for 107: the phases of a
// workgroup do not overlap, and a compute unit holds four workgroups (two in FP64).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"
#include "matrix.hpp"

namespace magace {

namespace {

constexpr int kPairs = 60;  // pairs of a round: 15 steps of four; lane 60 of the staging is the central atom

// pairs summed before they join the atom's sum: one chain of all 57 would round 57 times at the size of
// the whole sum (FP32 errors of E and of the forces against 64 bits, lmax-4 header: 60 pairs a chain
// 5.4e-7 and 3.5e-7, 20 pairs 3.2e-7 and 2.5e-7, and shorter chains less)
template <typename T> constexpr int kChain = sizeof(T) == 4 ? 12 : kPairs;
template <typename T> constexpr int kRound = sizeof(T) == 4 ? 12 : 4;  // pairs of an unrolled turn; divides kPairs

constexpr int kG = 17;  // row of a pair's base functions: 16, and one for the banks
// the same where radial factors of A's own come before them (the 16 rows of a product's operand may reach into what
// lies behind: their results are not used)
template <bool SEP> __host__ __device__ constexpr int functions_row(int og, int nb) {
    return !SEP || og + nb < kG ? kG : (og + nb) | 1;
}

// Harmonics in a pair's row of Y or Y'.  In FP32 those of the instance's lmax, so that the rows' addresses are known
// when it is compiled; in FP64 the longer rows of headers below it cost a workgroup of a compute unit (4394 atoms
// of the example potential's shape 111 -> 128 us).
template <typename T, int L> __host__ __device__ constexpr int harmonics_row(int n) {
    return sizeof(T) == 4 ? (L + 1) * (L + 2) / 2 : n;
}

struct DensityLds {  // strides and offsets (in T) of the staging arrays
    int sY, sYm, sH, sM, sG;      // row lengths: Y, Y' and H in complex entries, M and the functions in values; odd
    int oYm, oH, oG, oM, oYd, oGd, size;
    // lha, lhm: harmonics_row; row: functions_row
    __host__ __device__ constexpr DensityLds(int lha, int lhm, int nm3, int nfm, bool jvp, int row = kG)
        : sY(lha | 1), sYm(lhm | 1), sH(nm3 | 1), sM(nfm | 1), sG(row), oYm(0), oH(0), oG(0), oM(0), oYd(0), oGd(0), size(0) {
        oYm = 2 * kPairs * sY;
        oH = oYm + 2 * (kPairs + 1) * sYm;
        oG = (oH + 2 * kPairs * sH + 3) & ~3;
        oM = oG + sG * kPairs + (sG > kG ? 16 : 0);  // 16: the last row's operands end here
        oYd = (oM + (kPairs + 1) * sM + 3) & ~3;
        oGd = oYd + (jvp ? 2 * kPairs * sY : 0);
        size = oGd + (jvp ? oM - oG : 0);
    }
};

// harmonics() without a branch on l where the header has all of the instance's, in FP32 up to l = 4 always (rows have
// room for them).  The conditions of the other case are not to be kept across the rounds: 40 to 77 scalars of masks,
// spilled to vector registers, were up to a third of the staging's instructions.  27648 atoms lmax 4: mixed 295 -> 287
// us, FP64 480 -> 470 us; 16000 atoms lmax 6 FP64 484 -> 465 us.  FP32 at l = 6 spills with the long straight code (267
// us) and keeps its branches (264 us, 265 before).
template <typename T, int L, typename F>
__device__ __forceinline__ void row_of_harmonics(T x, T y, T z, int lmax, F&& put) {
    if (sizeof(T) == 4 && L <= 4) lmax = L;
    if (lmax == L && !(sizeof(T) == 4 && L > 4)) {
        harmonics<T, L>(x, y, z, L, put);
    } else {
        asm volatile("" : "+s"(lmax));
        harmonics<T, L>(x, y, z, lmax, put);
    }
}

// functions first .. first + nf - 1 of a row: value(k, coefficients), some more than once
template <typename T, typename F>
__device__ __forceinline__ void spline_row(const T* __restrict__ row, int first, int nf, F&& value) {
    constexpr int U = 4;
    row += 4 * first;
    for (int k0 = 0; k0 < nf; k0 += U) {
        Coef<T> n[U];
#pragma unroll
        for (int u = 0; u < U; ++u) n[u] = coef_at(row + 4 * min(k0 + u, nf - 1));
#pragma unroll
        for (int u = 0; u < U; ++u) value(min(k0 + u, nf - 1), n[u]);
    }
}

}  // namespace

// One workgroup of four waves an atom, rounds of up to kPairs pairs.  Staging, a wave each: Y_lm of the
// bonds and the core term; Y_l'm' of the moments and H_q = M_{l',n'} Y_l'm'; the g_k; the M_{l',n'}.  Then
// wave w takes the column tiles w, w + 4, ... (16 columns of A or A2, real and imaginary parts: two
// products a step of four pairs).  TA, T2: tiles of A and of A2 of a wave at most.  JVP: the derivative of A and A2 along
// the pairs' displacements u_i - u_j (k_density_jvp's work in a fit) in place of the values.  SEP: radial factors of
// A's own before the base functions (DevParams::og).
// Waves per SIMD: what the LDS of the usual headers lets in.  Under that bound the FP32 instances of two and one tiles
// spill six registers (95 MB of writes at 16000 atoms of lmax 6, half as much again as Z), those of four and three tiles, which
// class-2 headers with many magnetic radial functions run, 37 to 51, and 94 to 205 in FP64.
template <typename T, int L, int TA, int T2, bool JVP, bool SEP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TA > 2 ? 2 : sizeof(T) == 4 ? 4 : L <= 4 ? 3 : 2, 8)))
k_density_mm(DevParams<T> P, const int* __restrict__ off,
                                                    const double* __restrict__ dlist, const double* __restrict__ elist,
                                                    const double* __restrict__ dmomi, const double* __restrict__ emomi,
                                                    const double* __restrict__ dmom, const double* __restrict__ emom,
                                                    const int* __restrict__ nlist, const double* __restrict__ du,
                                                    cplx<T>* __restrict__ Zout, double* __restrict__ ehc_out,
                                                    double* __restrict__ rho1_out, int* err) {
    typedef typename Mm<T>::V V;
    extern __shared__ __align__(16) unsigned char smem[];
    const int atom = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nfm = P.nr2m * (P.l2m + 1);
    const int SY = harmonics_row<T, L>(P.lha) | 1, SYM = harmonics_row<T, L>(P.lhm) | 1;  // DensityLds::sY and sYm
    const int og = SEP ? P.og : 0, SG = functions_row<SEP>(og, P.nb_a);
    const DensityLds D(harmonics_row<T, L>(P.lha), harmonics_row<T, L>(P.lhm), P.nm3, nfm, JVP, SG);
    T* lds = (T*)smem;
    cplx<T>*sY = (cplx<T>*)lds, *sYm = (cplx<T>*)(lds + D.oYm), *sH = (cplx<T>*)(lds + D.oH);
    T *sG = lds + D.oG, *sM = lds + D.oM;
    cplx<T>* sYd = (cplx<T>*)(lds + D.oYd);
    T* sGd = lds + D.oGd;
    const int p0 = off[atom], nn = off[atom + 1] - p0;
    Zout += (size_t)atom * P.nz;

    // this lane's columns (P.cols): wave w has the tiles w, w + 4, ... of those of A followed by those of A2.  There may
    // be none of either: a potential of pair functions has A2 only, one of the moments' functions alone neither.
    const int nA = P.lha * P.nm3, nA2 = P.nr2m * P.lhm;
    const int tA = (nA + 15) >> 4, tAll = tA + ((nA2 + 15) >> 4);
    const int ci = lane & 15, g = lane >> 4;
    const int na = (tA - wave + 3) >> 2, n2 = ((tAll - wave + 3) >> 2) - na;
    V ar[TA], ai[TA], a2r[T2], a2i[T2];
    uint32_t ca[TA], c2[T2];
#pragma unroll
    for (int t = 0; t < TA; ++t) {
        ar[t] = (V)(T)0;
        ai[t] = (V)(T)0;
        ca[t] = tA > 0 ? P.cols[min(wave + 4 * t, tA - 1) * 16 + ci] : 0u;
    }
#pragma unroll
    for (int t = 0; t < T2; ++t) {
        a2r[t] = (V)(T)0;
        a2i[t] = (V)(T)0;
        c2[t] = tAll > 0 ? P.cols[min(wave + 4 * (na + t), tAll - 1) * 16 + ci] : 0u;
    }
    // what lies behind a pair's functions stays zero
    for (int i = tid; i < D.oM - D.oG; i += 256) {
        sG[i] = (T)0;
        if (JVP) sGd[i] = (T)0;
    }
    double ux = 0, uy = 0, uz = 0;
    if constexpr (JVP) {
        ux = du[3 * (size_t)atom];
        uy = du[3 * (size_t)atom + 1];
        uz = du[3 * (size_t)atom + 2];
    }
    double core = 0.0;
    for (int c0 = 0; c0 == 0 || c0 < nn; c0 += kPairs) {
        // whole chains of pairs; those past the end have g = 0
        const int nj = min(nn - c0, kPairs), nr = (nj + kRound<T> - 1) / kRound<T> * kRound<T>;
        const bool live = lane < nj, centre = !JVP && lane == kPairs && c0 == 0;
        const size_t p = (size_t)p0 + c0 + (live ? lane : 0);
        __syncthreads();
        if (wave == 0) {
            if (lane < nr) {
                T w = 0;
                const int row = live ? atomic_index(P, dlist[p], w, err) : kRowZero;
                const T x = live ? (T)elist[3 * p] : (T)0, y = live ? (T)elist[3 * p + 1] : (T)0,
                        z = live ? (T)elist[3 * p + 2] : (T)1;
                const Coef<T> cc = coef_at(P.lut_g + (size_t)(row < 0 ? 0 : row) * P.stride_g + 4 * (og + P.nb_a));
                if constexpr (!JVP) {
                    row_of_harmonics<T, L>(x, y, z, P.l3a, [&](int k, T pl, T, cplx<T> ph, cplx<T>, int) {
                        sY[lane * SY + k] = {pl * ph.re, pl * ph.im};
                    });
                    core += row < 0 ? 0.0 : (double)coef_value(cc, w);
                } else {
                    T dx = 0, dy = 0, dz = 0;
                    if (live) {
                        const size_t jn = 3 * (size_t)nlist[p];
                        dx = ux - du[jn];
                        dy = uy - du[jn + 1];
                        dz = uz - du[jn + 2];
                    }
                    const T rdot = x * dx + y * dy + z * dz;
                    const T invr = live ? (T)(1.0 / dlist[p]) : (T)0;
                    // the displacement's part across the bond, over r: D_u Y = grad Y . t
                    const T tx = (dx - rdot * x) * invr, ty = (dy - rdot * y) * invr, tz = (dz - rdot * z) * invr;
                    row_of_harmonics<T, L>(x, y, z, P.l3a, [&](int k, T pl, T dpl, cplx<T> ph, cplx<T> ph1, int m) {
                        sY[lane * SY + k] = {pl * ph.re, pl * ph.im};
                        // Y = P(z) (x + iy)^m
                        const T a = dpl * tz, b = (T)m * pl;
                        const cplx<T> e = cmul(ph1, cplx<T>{tx, ty});
                        sYd[lane * SY + k] = {fma(a, ph.re, b * e.re), fma(a, ph.im, b * e.im)};
                    });
                    core += row < 0 ? 0.0 : (double)(coef_slope(cc, w, (T)P.rs_a) * rdot);
                }
            }
        } else if (wave == 1) {
            if (lane < nr || centre) {
                const bool any = live || centre;
                T w = 0;
                const int row = live ? magnetic_index(P, dmom[p], w, err) : kRowZero;
                const double* v = centre ? emomi + 3 * (size_t)atom : emom + 3 * p;
                const T x = any ? (T)v[0] : (T)0, y = any ? (T)v[1] : (T)0, z = any ? (T)v[2] : (T)1;
                const T* mrow = P.lut_m + (size_t)(row < 0 ? 0 : row) * P.stride_m + 4 * P.nb_m;
                // the first M of H, so that their trip to memory passes during the Y_l'm'
                constexpr int U = 2;
                Coef<T> cm[U];
#pragma unroll
                for (int u = 0; u < U; ++u) cm[u] = coef_at(mrow + 4 * (u <= P.l3m ? u * P.nr2m : 0));
                row_of_harmonics<T, L>(x, y, z, P.l2m, [&](int k, T pl, T, cplx<T> ph, cplx<T>, int) {
                    sYm[lane * SYM + k] = {pl * ph.re, pl * ph.im};
                });
                if (lane < nr)
                    for (int np = 0; np * P.lsm3 < P.nm3; ++np)
                        for (int lp = 0; lp <= P.l3m; ++lp) {
                            Coef<T> c;
                            if (np > 0 || lp >= U)
                                c = coef_at(mrow + 4 * (lp * P.nr2m + np));
                            else
#pragma unroll
                                for (int u = 0; u < 4; ++u) c.c[u] = lp ? cm[1].c[u] : cm[0].c[u];
                            const T mv = row == kRowOne ? (T)1 : row < 0 ? (T)0 : coef_value(c, w);
                            for (int mp = -lp; mp <= lp; ++mp) {
                                const cplx<T> h = sYm[lane * SYM + lp * (lp + 1) / 2 + (mp < 0 ? -mp : mp)];
                                const cplx<T> yv = mp < 0 ? cconj_sign(h, -mp) : h;
                                sH[lane * D.sH + np * P.lsm3 + lp * lp + lp + mp] = {mv * yv.re, mv * yv.im};
                            }
                        }
            }
        } else if (wave == 2) {
            T w = 0;
            const int row = live ? atomic_index(P, dlist[p], w, err) : kRowZero;
            T rdot = 0;
            if constexpr (JVP) {
                if (live) {
                    const size_t jn = 3 * (size_t)nlist[p];
                    rdot = elist[3 * p] * (ux - du[jn]) + elist[3 * p + 1] * (uy - du[jn + 1]) +
                           elist[3 * p + 2] * (uz - du[jn + 2]);
                }
            }
            if (lane < nr)
                spline_row<T>(P.lut_g + (size_t)(row < 0 ? 0 : row) * P.stride_g, 0, og + P.nb_a,
                              [&](int k, const Coef<T>& c) {
                                  sG[lane * SG + k] = row < 0 ? (T)0 : coef_value(c, w);
                                  // g'_k (u_i - u_j) . e
                                  if constexpr (JVP)
                                      sGd[lane * SG + k] = row < 0 ? (T)0 : coef_slope(c, w, (T)P.rs_a) * rdot;
                              });
        } else {
            T w = 0;
            const int row = centre ? magnetic_index(P, dmomi[atom], w, err)
                                   : live ? magnetic_index(P, dmom[p], w, err) : kRowZero;
            const bool first = !JVP && c0 == 0;
            if (nfm > 0 && (lane < nr || centre))
                spline_row<T>(P.lut_m + (size_t)(row < 0 ? 0 : row) * P.stride_m, P.nb_m, nfm,
                              [&](int k, const Coef<T>& c) {
                                  sM[lane * D.sM + k] = row == kRowOne ? (T)1 : row < 0 ? (T)0 : coef_value(c, w);
                              });
            if (first) {
                // B1 part of rho (b_basis.F90:62-83): lane k has g^m_k of the central moment
                const int rc = __shfl(row, kPairs, 64);
                const T wc = __shfl(w, kPairs, 64);
                double b0 = 0.0, b1 = 0.0;
                if (lane < P.nb_m) {
                    const Coef<T> c = coef_at(P.lut_m + (size_t)(rc < 0 ? 0 : rc) * P.stride_m + 4 * lane);
                    const double v = (double)(rc == kRowOne ? (T)1 : rc < 0 ? (T)0 : coef_value(c, wc)) - 1.0;
                    b0 = P.c1[0][lane] * v;
                    b1 = P.c1[1][lane] * v;
                }
                double s0 = 0.0, s1 = 0.0;
                for (int k = 0; k < P.nb_m; ++k) {  // in the order of the functions
                    s0 += __shfl(b0, k, 64);
                    s1 += __shfl(b1, k, 64);
                }
                if (lane < P.nd) rho1_out[(size_t)atom * P.nd + lane] = lane ? s1 : s0;
            }
        }
        __syncthreads();
        if (c0 == 0) {
            // A0 (src/a_basis.F90:90-106); it does not depend on positions
            for (int t = tid; t < nA2; t += 256) {
                cplx<T> z = {0, 0};
                if constexpr (!JVP) {
                    const uint32_t d = P.cols[tA * 16 + t];
                    const cplx<T> h = sYm[kPairs * SYM + (d & 0xff)];
                    const T mv = sM[kPairs * D.sM + (d >> 8 & 0xff)];
                    z = {mv * h.re, mv * h.im};
                }
                Zout[P.hA0 + t] = z;
            }
        }
        // NA tiles of A and N2 of A2
        auto products = [&](auto NA_, auto N2_) {
            constexpr int NA = NA_, N2 = N2_;
            constexpr bool kPart = kChain<T> < kPairs;  // the sums of kChain pairs join the atom's
            int iy[TA], ih[TA], iy2[T2], im[T2];
#pragma unroll
            for (int t = 0; t < NA; ++t) {
                iy[t] = g * SY + (ca[t] & 0xff);
                ih[t] = g * D.sH + (ca[t] >> 8 & 0xff);
            }
#pragma unroll
            for (int t = 0; t < N2; ++t) {
                iy2[t] = g * SYM + (c2[t] & 0xff);
                im[t] = g * D.sM + (c2[t] >> 8 & 0xff);
            }
            int ig = g * SG + ci;
            for (int s0 = 0; s0 < nr; s0 += kRound<T>) {
                V br[TA], bi[TA], b2r[T2], b2i[T2];
#pragma unroll
                for (int t = 0; t < NA; ++t) {
                    br[t] = kPart ? (V)(T)0 : ar[t];
                    bi[t] = kPart ? (V)(T)0 : ai[t];
                }
#pragma unroll
                for (int t = 0; t < N2; ++t) {
                    b2r[t] = kPart ? (V)(T)0 : a2r[t];
                    b2i[t] = kPart ? (V)(T)0 : a2i[t];
                }
#pragma unroll
                for (int s = 0; s < kRound<T>; s += 4) {
                    // the step's operands of every tile first, so that one trip to LDS serves them all
                    const T a = sG[ig + s * SG];
                    const T a2 = SEP && N2 > 0 ? sG[ig + s * SG + og] : a;
                    T ad = 0, ad2 = 0;
                    if constexpr (JVP) {
                        ad = sGd[ig + s * SG];
                        ad2 = SEP && N2 > 0 ? sGd[ig + s * SG + og] : ad;
                    }
                    cplx<T> y[TA], h[TA], yd[JVP ? TA : 1], y2[T2];
                    T m2[T2];
#pragma unroll
                    for (int t = 0; t < NA; ++t) {
                        y[t] = sY[iy[t] + s * SY];
                        h[t] = sH[ih[t]];
                        ih[t] += 4 * D.sH;
                        if constexpr (JVP) yd[JVP ? t : 0] = sYd[iy[t] + s * SY];
                    }
#pragma unroll
                    for (int t = 0; t < N2; ++t) {
                        y2[t] = sYm[iy2[t] + s * SYM];
                        m2[t] = sM[im[t]];
                        im[t] += 4 * D.sM;
                    }
#pragma unroll
                    for (int t = 0; t < NA; ++t) {
                        const cplx<T> v = cmul(y[t], h[t]);
                        br[t] = Mm<T>::mul(JVP ? ad : a, v.re, br[t]);
                        bi[t] = Mm<T>::mul(JVP ? ad : a, v.im, bi[t]);
                        if constexpr (JVP) {
                            const cplx<T> vd = cmul(yd[JVP ? t : 0], h[t]);
                            br[t] = Mm<T>::mul(a, vd.re, br[t]);
                            bi[t] = Mm<T>::mul(a, vd.im, bi[t]);
                        }
                    }
#pragma unroll
                    for (int t = 0; t < N2; ++t) {
                        b2r[t] = Mm<T>::mul(JVP ? ad2 : a2, m2[t] * y2[t].re, b2r[t]);
                        b2i[t] = Mm<T>::mul(JVP ? ad2 : a2, m2[t] * y2[t].im, b2i[t]);
                    }
                }
                ig += kRound<T> * SG;
#pragma unroll
                for (int t = 0; t < NA; ++t) {
                    ar[t] = kPart ? ar[t] + br[t] : br[t];
                    ai[t] = kPart ? ai[t] + bi[t] : bi[t];
                    iy[t] += kRound<T> * SY;
                }
#pragma unroll
                for (int t = 0; t < N2; ++t) {
                    a2r[t] = kPart ? a2r[t] + b2r[t] : b2r[t];
                    a2i[t] = kPart ? a2i[t] + b2i[t] : b2i[t];
                    iy2[t] += kRound<T> * SYM;
                }
            }
        };
        // The loops have no branch on a wave's tiles: a tile that it does not have repeats the last one and is not
        // stored.
        using std::integral_constant;
        if (na >= TA) {
            if (n2 >= T2)
                products(integral_constant<int, TA>(), integral_constant<int, T2>());
            else
                products(integral_constant<int, TA>(), integral_constant<int, T2 - 1>());
        } else {
            if (n2 >= T2)
                products(integral_constant<int, TA - 1>(), integral_constant<int, T2>());
            else
                products(integral_constant<int, TA - 1>(), integral_constant<int, T2 - 1>());
        }
    }
#pragma unroll
    for (int t = 0; t < TA; ++t)
        if (t < na) {
            // A = U B for each l that the tile's columns have
            const int l = ca[t] >> 16 & 15;
            const int l0 = __builtin_amdgcn_readlane(l, 0), l1 = __builtin_amdgcn_readlane(l, 15);
            V zr = (V)(T)0, zi = (V)(T)0;
            T k[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) k[r] = P.cperm[(size_t)l0 * 256 + 64 * r + lane];
            for (int ll = l0; ll <= l1; ++ll) {
                V br = (V)(T)0, bi = (V)(T)0;
                T kn[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) kn[r] = P.cperm[(size_t)min(ll + 1, l1) * 256 + 64 * r + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    br = Mm<T>::mul(k[r], ar[t][r], br);
                    bi = Mm<T>::mul(k[r], ai[t][r], bi);
                    k[r] = kn[r];
                }
                if (l == ll) {
                    zr = br;
                    zi = bi;
                }
            }
            const int c = (wave + 4 * t) * 16 + ci;
            if (c < nA)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int n = Mm<T>::row(g, r);
                    if (n < P.nr3a) Zout[n * nA + c] = {zr[r], zi[r]};
                }
        }
#pragma unroll
    for (int t = 0; t < T2; ++t) {
        const int c = (wave + 4 * (na + t) - tA) * 16 + ci;
        if (t < n2 && c < nA2)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = Mm<T>::row(g, r);
                if (k < P.nb_a) Zout[P.hA2 + k * nA2 + c] = {a2r[t][r], a2i[t][r]};
            }
    }
    if (wave == 0) {
        for (int o = 32; o > 0; o >>= 1) core += __shfl_xor(core, o, 64);
        if (lane == 0) ehc_out[atom] = core;
    }
}

namespace {

template <typename T, int L, int TA, int T2, bool JVP, bool SEP>
hipError_t launch_density(const DevParams<T>& P, int natom, const int* off, const double* dlist, const double* elist,
                          const double* dmomi, const double* emomi, const double* dmom, const double* emom,
                          const int* nlist, const double* du, void* Z, double* ehc, double* rho1, int* err,
                          hipStream_t s) {
    auto k = k_density_mm<T, L, TA, T2, JVP, SEP>;
    const size_t lds = (size_t)DensityLds(harmonics_row<T, L>(P.lha), harmonics_row<T, L>(P.lhm), P.nm3,
                                         P.nr2m * (P.l2m + 1), JVP, functions_row<SEP>(P.og, P.nb_a)).size * sizeof(T);
    static bool set = false;
    static size_t limit = 0;
    hipError_t e;
    if (!set) {
        int dev = 0, most = 0;
        if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
        if ((e = hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) != hipSuccess) return e;
        if ((e = hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, most)) != hipSuccess)
            return e;
        limit = (size_t)most;
        set = true;
    }
    if (lds > limit) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k, dim3(natom), dim3(256), lds, s, P, off, dlist, elist, dmomi, emomi, dmom, emom, nlist, du,
                       (cplx<T>*)Z, ehc, rho1, err);
    return hipGetLastError();
}

template <typename T, int L, bool JVP, bool SEP, typename... A>
hipError_t by_tiles(const DevParams<T>& P, A... a) {
    const int tA = (P.lha * P.nm3 + 15) >> 4, tAll = tA + ((P.nr2m * P.lhm + 15) >> 4);
    int ta = 0, t2 = 0;
    for (int w = 0; w < 4; ++w) {
        const int na = (tA - w + 3) >> 2;
        ta = ta > na ? ta : na;
        const int n2 = ((tAll - w + 3) >> 2) - na;
        t2 = t2 > n2 ? t2 : n2;
    }
    if (ta <= 1 && t2 <= 1) return launch_density<T, L, 1, 1, JVP, SEP>(P, a...);
    if (ta <= 2 && t2 <= 1) return launch_density<T, L, 2, 1, JVP, SEP>(P, a...);
    if (ta <= 4 && t2 <= 1) return launch_density<T, L, 4, 1, JVP, SEP>(P, a...);
    if (ta <= 4 && t2 <= 3) return launch_density<T, L, 4, 3, JVP, SEP>(P, a...);
    return hipErrorInvalidValue;  // no header of the supported classes has more
}

}  // namespace

template <typename T>
hipError_t run_density(const DevParams<T>& P, int natom, const int* off, const double* dlist, const double* elist,
                       const double* dmomi, const double* emomi, const double* dmom, const double* emom,
                       const Buffers& B, hipStream_t s) {
    const int l = P.l3a > P.l2m ? P.l3a : P.l2m;
    const int* no_list = nullptr;
    const double* no_u = nullptr;
    auto go = [&](auto sep) {
        constexpr bool SEP = decltype(sep)::value;
        if (l <= 2) return by_tiles<T, 2, false, SEP>(P, natom, off, dlist, elist, dmomi, emomi, dmom, emom, no_list, no_u, B.Z, B.ehc, B.rho1, B.err, s);
        if (l <= 4) return by_tiles<T, 4, false, SEP>(P, natom, off, dlist, elist, dmomi, emomi, dmom, emom, no_list, no_u, B.Z, B.ehc, B.rho1, B.err, s);
        return by_tiles<T, 6, false, SEP>(P, natom, off, dlist, elist, dmomi, emomi, dmom, emom, no_list, no_u, B.Z, B.ehc, B.rho1, B.err, s);
    };
    return P.og > 0 ? go(std::true_type()) : go(std::false_type());
}

hipError_t run_density_jvp(const DevParams<double>& P, int natom, const int* off, const int* nlist, const double* du,
                           const double* dlist, const double* elist, const double* dmom, const double* emom, void* Zdot,
                           double* ehc_dot, int* err, hipStream_t s) {
    const int l = P.l3a > P.l2m ? P.l3a : P.l2m;
    const double* none = nullptr;
    double* no_rho = nullptr;
    auto go = [&](auto sep) {
        constexpr bool SEP = decltype(sep)::value;
        if (l <= 2) return by_tiles<double, 2, true, SEP>(P, natom, off, dlist, elist, none, none, dmom, emom, nlist, du, Zdot, ehc_dot, no_rho, err, s);
        if (l <= 4) return by_tiles<double, 4, true, SEP>(P, natom, off, dlist, elist, none, none, dmom, emom, nlist, du, Zdot, ehc_dot, no_rho, err, s);
        return by_tiles<double, 6, true, SEP>(P, natom, off, dlist, elist, none, none, dmom, emom, nlist, du, Zdot, ehc_dot, no_rho, err, s);
    };
    return P.og > 0 ? go(std::true_type()) : go(std::false_type());
}

template hipError_t run_density<double>(const DevParams<double>&, int, const int*, const double*, const double*,
                                        const double*, const double*, const double*, const double*, const Buffers&,
                                        hipStream_t);
template hipError_t run_density<float>(const DevParams<float>&, int, const int*, const double*, const double*,
                                       const double*, const double*, const double*, const double*, const Buffers&,
                                       hipStream_t);

}  // namespace magace
