// forces.hip -- pair forces, pair torques and self torques on the matrix cores.
//
// k_forces_mm does the work of forcecompute and torquecompute (src/forces.F90:418-623, 688-961).  With
// V[k][lm,q] = sum_n C_{nlk} W[n][lm][q] once an atom, the pair's weights are
//   P[lm,q] = sum_k g_k V[k][lm,q],  Q[lm,q] = sum_k g'_k V[k][lm,q]
// (and the same of A2's W2[k][n'][l'm']), matrix products over at most 16 base functions, or for A over its radial
// factors h_f with V[f] = sum_n U_{nlf} W[n] (RadialFactors).  The columns q of a
// pair +m', -m' enter as the real and the imaginary part h of H_{m'} = M Y_{m'} (V of the two columns added and
// subtracted), which halves the work behind the products:
//   S = sum_q P h,  dE/dY = S;   dE/dr = Re sum Q h Y;   u_q = dE/dh_q = Re sum_lm P Y.
// Of a product's result lane (j, g), j the pair and g = 0..3, holds four rows of group g.  Each group walks
// through harmonics of its own (ForceStep): the orders m are spread over the groups (28 harmonics of l <= 6 are
// four walks of seven, U is their sum), or, where there are many columns q, every group takes all harmonics
// with four columns of its own.  So neither harmonics nor weights pass through LDS.  A wave holds 16
// pairs; waves meet only for V.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.hpp"
#include "kernels.hpp"
#include "matrix.hpp"

namespace magace {

namespace {

// one step of a walk through the harmonics: p_l = a z p_{l-1} + b p_{l-2} + c, a = b = 0 at the first l of an
// order m and all three 0 where a group's walk has ended
template <typename T>
struct alignas(16) ForceStep {
    T a, b, c;
    int lm;  // l | m << 8 | first l of its order << 16 | harmonic << 17; offset of M_l. << 18
    __device__ __forceinline__ int l() const { return lm & 0xff; }
    __device__ __forceinline__ int m() const { return lm >> 8 & 0xff; }
};

template <typename T>
struct Walk {
    T p = 0, d = 0, p1 = 0, d1 = 0, m = 0;
    cplx<T> ph = {0, 0}, ph1 = {0, 0};
    // e: powers of x + iy of the lane's pair; first: some group is at the first l of an order
    __device__ __forceinline__ void step(const ForceStep<T>& s, T z, const cplx<T>* e, bool first) {
        if (first) {
            const int o = s.m();
            const cplx<T> a = e[o], b = e[o > 0 ? o - 1 : 0];
            const bool on = s.lm >> 16 & 1;
            ph.re = on ? a.re : ph.re, ph.im = on ? a.im : ph.im;
            ph1.re = on ? b.re : ph1.re, ph1.im = on ? b.im : ph1.im;
            m = on ? (T)o : m;
        }
        const T az = s.a * z, q = p, e1 = d;
        p = fma(az, q, fma(s.b, p1, s.c));
        d = fma(s.a, q, fma(az, e1, s.b * d1));
        p1 = q;
        d1 = e1;
    }
    // G += Re(S grad Y) of the extension P(z) (x + iy)^m, before the projection on the tangent plane
    __device__ __forceinline__ void gradient(T Sr, T Si, T& gx, T& gy, T& gz) const {
        const T mp = m * p;
        gx = fma(mp, Sr * ph1.re - Si * ph1.im, gx);
        gy = fma(-mp, Sr * ph1.im + Si * ph1.re, gy);
        gz = fma(d, Sr * ph.re - Si * ph.im, gz);
    }
    __device__ __forceinline__ cplx<T> value() const { return {p * ph.re, p * ph.im}; }
};

// orders the wave's LDS accesses of its lanes to each other
__device__ __forceinline__ void wave_order() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// powers 0..6 of x + iy of the wave's 16 pairs, lane (j, g) those of g and g + 4
constexpr int kPowers = 7;
template <typename T>
__device__ __forceinline__ void put_powers(cplx<T>* e, int g, T x, T y) {
    const cplx<T> e1 = {x, y}, e2 = cmul(e1, e1), e4 = cmul(e2, e2);
    cplx<T> a = {g & 1 ? x : (T)1, g & 1 ? y : (T)0};
    const cplx<T> b = cmul(a, e2);
    a.re = g & 2 ? b.re : a.re;
    a.im = g & 2 ? b.im : a.im;
    e[g] = a;
    if (g < 3) e[g + 4] = cmul(a, e4);
}

// lane group g: the sum of u[g] over the four groups
template <typename T>
__device__ __forceinline__ T fold_groups(const T (&u)[4]) {
    return fold16(fold32(u[0], u[2]), fold32(u[1], u[3]));
}

struct ForceLds {  // offsets in T
    // rows of n complex values that 16 lanes read at different banks (64 of four bytes)
    __host__ __device__ static int spread(int n, size_t t) { return t == 8 ? n | 1 : n % 4 ? n : n + 1; }
    int tiles, rounds, nqp, oStep, oWave, oM, oP, oE, wave, size;
    __host__ __device__ ForceLds(int na, int nk, int ta, int nq4, int tm, int steps, bool qsplit, int nfm, int waves, size_t t) {
        rounds = qsplit ? (nq4 + 3) >> 2 : nq4;
        nqp = 4 * (qsplit ? 4 * rounds : nq4);  // columns q with their padding
        tiles = rounds * ta + tm;
        oStep = 2 * (rounds * ta * na + tm * nk) * 64;  // operands of V, complex
        oWave = oStep + steps * 4;              // a ForceStep is four T
        // of a wave: h, then u [16][nqp], (M, M') [16][spread(nfm)], powers, then results [16][kPowers], directions [16][8]
        oM = 16 * nqp;
        oP = oM + 2 * 16 * spread(nfm, t);
        oE = oP + 2 * 16 * kPowers;
        wave = oE + 16 * 8;
        size = oWave + waves * wave;
    }
};

}  // namespace

// Workgroup: one atom, up to four waves of 16 pairs (fewer where their LDS does not fit).  NK: steps of four base
// functions; NA: of four radial factors of A.  SEP: these are functions of their own (DevParams::og).
//
// Bound by issue: at 16000 atoms of lmax 6 a wave has 1670 vector instructions and 132 products of 32 cycles
// (FP32; 64 in FP64), about 11000 cycles of a SIMD, which measures 280 us (FP64 622 us).  One lane a pair, with W
// in LDS and sums over n, columns and the harmonics in vector instructions, took 449 us (1093 us); at lmax 4
// and 27648 atoms 419 -> 316 us (901 -> 587 us), with 27 magnetic columns and 4394 atoms 213 -> 103 us (454 ->
// 193 us; 130 and 320 with A's sixteen base functions in place of its eight factors), at 128 atoms of lmax 4 in FP64,
// where a wave's length counts, 36 -> 15 us.  Five waves a SIMD in
// FP32 need at most 96 registers and 32000 bytes of LDS a workgroup, which the layout below keeps at lmax 6;
// loading the pairs' inputs before V is made costs the fifth wave and was slower (323 us).  The 96 registers are not
// quite enough: with three steps of base functions two are spilled (34 MB of writes at 16000 atoms), with four three, and
// up to fourteen with factors.
template <typename T, int NK, int NA, bool SEP>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 5 : 2, sizeof(T) == 4 ? 5 : 3)))
k_forces_mm(DevParams<T> P, const int* __restrict__ off, const double* __restrict__ dlist,
            const double* __restrict__ elist, const double* __restrict__ dmomi, const double* __restrict__ emomi,
            const double* __restrict__ dmom, const double* __restrict__ emom, const cplx<T>* __restrict__ Win, bool scaled,
            const double* __restrict__ dEin, const double* __restrict__ edfin, double* __restrict__ flist,
            double* __restrict__ tlist, double* __restrict__ tlist0, int* err) {
    typedef typename Mm<T>::V V;
    static_assert(sizeof(ForceStep<T>) == 4 * sizeof(T), "ForceLds counts a step as four values");
    extern __shared__ __align__(16) unsigned char smem[];
    const int atom = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ji = lane & 15, g = lane >> 4;
    const int nthr = blockDim.x, nw = nthr >> 6;
    const int nfm = P.nr2m * (P.l2m + 1), sMs = ForceLds::spread(nfm, sizeof(T));
    const int tm = (P.stm * P.nr2m + 3) >> 2, steps = 4 * (P.sta + P.stm);
    const int og = SEP ? P.og : 0, nf = SEP ? P.nf : P.nb_a;
    const ForceLds D(NA, NK, P.sta, (P.nm3 + 3) >> 2, tm, steps, P.qsplit, nfm, nw, sizeof(T));
    T* lds = (T*)smem;
    cplx<T>* sV = (cplx<T>*)lds;
    ForceStep<T>* sStep = (ForceStep<T>*)(lds + D.oStep);
    T* mine = lds + D.oWave + wave * D.wave;
    T* sH = mine + ji * D.nqp;
    cplx<T>* sM = (cplx<T>*)(mine + D.oM) + ji * sMs;  // (M, M')
    cplx<T>* sP = (cplx<T>*)(mine + D.oP) + ji * kPowers;
    T* sE = mine + D.oE;  // per pair: e, 1/r, s, 1/mu
    T* sR = mine + D.oP;  // the sums over its harmonics
    const cplx<T>* __restrict__ W = Win + (size_t)atom * P.nz;
    const T sc = scaled ? (T)1 : (T)dEin[atom];
    const int p0 = off[atom], nn = off[atom + 1] - p0;
    const int nA = P.lha * P.nm3, nA2 = P.nr2m * P.lhm;

    const T rsa = (T)P.rs_a, rsm = (T)P.rs_m;
    if (wave == nw - 1) {
        for (int i = lane; i < steps; i += 64) {
            const double* s = P.steps + 4 * i;
            sStep[i] = {(T)s[0], (T)s[1], (T)s[2], (int)s[3]};
        }
        // self torque dE_i/dm_i (src/forces.F90:712-749): lane (n', step, g) of the moments' walks, and the B1
        // functions.  The last wave has the fewest rows of V and the fewest pairs.
        const double mu_d = dmomi[atom];
        const T sx = (T)emomi[3 * (size_t)atom], sy = (T)emomi[3 * (size_t)atom + 1], sz = (T)emomi[3 * (size_t)atom + 2];
        const double dE0 = dEin[(size_t)atom * P.nd], dE1 = P.nd > 1 ? dEin[(size_t)atom * P.nd + 1] : 0.0;
        T wm = 0;
        const int rowm = magnetic_index(P, mu_d, wm, err);
        const T* __restrict__ ma = P.lut_m + (size_t)(rowm < 0 ? 0 : rowm) * P.stride_m;
        T tr = 0, tx = 0, ty = 0, tz = 0;
        if (lane < P.nb_m && rowm >= 0) {
            // B1: dE/dg^m_n = dE/drho c1_n
            const Coef<T> c = coef_at(ma + 4 * lane);
            tr = (T)(dE0 * P.c1[0][lane] + dE1 * P.c1[1][lane]) * coef_slope(c, wm, rsm);
        }
        put_powers(sP, g, sx, sy);
        wave_order();
        // 16 (step, n') at a time, of each the four harmonics of the groups
        for (int s0 = 0; s0 < P.stm * P.nr2m; s0 += 16) {
            const int own = (s0 + ji) / P.nr2m, np = (s0 + ji) - own * P.nr2m;
            const ForceStep<T> so = sStep[4 * (P.sta + (own < P.stm ? own : 0)) + g];
            const bool on = own < P.stm && (so.lm >> 17 & 1);
            const int l = so.l();
            const Coef<T> c = coef_at(ma + 4 * (P.nb_m + l * P.nr2m + np));
            const cplx<T> w = W[P.hA0 + np * P.lhm + l * (l + 1) / 2 + so.m()];
            Walk<T> k, h;
            for (int t = 0; t < P.stm; ++t) {
                k.step(sStep[4 * (P.sta + t) + g], sz, sP, P.firstm >> t & 1);
                if (t == own) h = k;
            }
            const T v = !on ? (T)0 : rowm == kRowOne ? (T)1 : rowm < 0 ? (T)0 : coef_value(c, wm);
            const T dv = !on || rowm < 0 ? (T)0 : coef_slope(c, wm, rsm);
            if (on) {
                tr = fma(dv * sc, re_mul(w, h.value()), tr);
                h.gradient(sc * v * w.re, sc * v * w.im, tx, ty, tz);
            }
        }
        const T a[4] = {tr, tx, ty, tz};
        T sum = fold_groups(a);  // of 16 lanes each
#pragma unroll
        for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
        tr = __shfl(sum, 0, 64), tx = __shfl(sum, 16, 64), ty = __shfl(sum, 32, 64), tz = __shfl(sum, 48, 64);
        const T invmu = (T)(1.0 / mu_d), gs = tx * sx + ty * sy + tz * sz;
        if (lane < 3) {
            const T s = lane == 0 ? sx : lane == 1 ? sy : sz, t = lane == 0 ? tx : lane == 1 ? ty : tz;
            tlist0[3 * (size_t)atom + lane] = (double)fma(tr, s, invmu * (t - gs * s));
        }
    }
    // V: a thread has one row of a tile with all base functions
    for (int x = tid; x < D.tiles * 16; x += nthr) {
        const uint2 vc = P.vcol[x];
        T re[4 * NK], im[4 * NK];
#pragma unroll
        for (int u = 0; u < 4 * NK; ++u) re[u] = im[u] = (T)0;
        if (vc.x != ~0u) {
            const int c = vc.x & 0xffff;
            if (vc.x >> 24 & 1) {
#pragma unroll
                for (int u = 0; u < 4 * NK; ++u) {
                    const cplx<T> w = W[P.hA2 + (u < P.nb_a ? u : 0) * nA2 + c];
                    re[u] = u < P.nb_a ? sc * w.re : (T)0;
                    im[u] = u < P.nb_a ? sc * w.im : (T)0;
                }
            } else {
                // the sum (cosine) or i times the difference (sine) of a pair of columns +m', -m'
                const T* __restrict__ cn = P.crow + (size_t)(vc.x >> 16 & 0xff) * 8 * 16;
                const T sb = vc.x >> 25 & 1 ? (vc.x >> 27 & 1 ? -sc : sc) : (T)0;
                const int cb = vc.x >> 25 & 1 ? (int)vc.y : c;
                const bool sine = vc.x >> 26 & 1;
                // NB of n at a time, all their loads before the first use (the coefficients past nr3a are 0).  With
                // 4 the FP32 kernel had room for 4 waves on a SIMD instead of 5: 305 instead of 294 us at
                // 16000 atoms, lmax 6; in FP64, with room for 3 either way, 2 took 634 instead of 622 us.
                constexpr int NB = sizeof(T) == 4 ? 2 : 4;
                for (int n0 = 0; n0 < P.nr3a; n0 += NB) {
                    cplx<T> w[NB], wb[NB];
                    Coef<T> k[NB][NA];
#pragma unroll
                    for (int n = 0; n < NB; ++n) {
                        const int o = (n0 + n < P.nr3a ? n0 + n : 0) * nA;
                        w[n] = W[o + c];
                        wb[n] = W[o + cb];
#pragma unroll
                        for (int s = 0; s < NA; ++s) k[n][s] = coef_at(cn + 16 * (n0 + n) + 4 * s);
                    }
#pragma unroll
                    for (int n = 0; n < NB; ++n) {
                        const T ar = fma(sb, wb[n].re, sc * w[n].re), ai = fma(sb, wb[n].im, sc * w[n].im);
                        const T wr = sine ? -ai : ar, wi = sine ? ar : ai;
#pragma unroll
                        for (int u = 0; u < 4 * NA; ++u) {
                            re[u] = fma(k[n][u / 4].c[u % 4], wr, re[u]);
                            im[u] = fma(k[n][u / 4].c[u % 4], wi, im[u]);
                        }
                    }
                }
            }
        }
        const int tile = x >> 4, tb = D.rounds * P.sta;
        cplx<T>* o = sV + (tile < tb ? tile * NA : tb * NA + (tile - tb) * NK) * 64 + (x & 15);
#pragma unroll
        for (int u = 0; u < 4 * NK; ++u)
            if (NA == NK || u < 4 * NA || tile >= tb) o[16 * u] = {re[u], im[u]};
    }
    __syncthreads();

    const T edf = (T)edfin[atom];
    for (int c0 = 16 * wave; c0 < nn; c0 += 16 * nw) {
        const bool live = c0 + ji < nn;
        const size_t p = (size_t)p0 + c0 + (live ? ji : 0);
        const double r_d = dlist[p], mu_d = dmom[p];
        const T ex = (T)elist[3 * p], ey = (T)elist[3 * p + 1], ez = (T)elist[3 * p + 2];
        const T sx = (T)emom[3 * p], sy = (T)emom[3 * p + 1], sz = (T)emom[3 * p + 2];
        T wa = 0, wm = 0;
        const int rowa = live ? atomic_index(P, r_d, wa, err) : kRowZero;
        // a pair beyond the atomic table does not look at its moment
        const int rowm = rowa >= 0 ? magnetic_index(P, mu_d, wm, err) : kRowZero;
        put_powers(sP, g, sx, sy);
        if (g < 2) {
            // 1/r 0: no pair
            const T inv = (T)(1.0 / (g ? mu_d : r_d));
            T* o = sE + 8 * ji + 4 * g;
            o[0] = g ? sx : ex, o[1] = g ? sy : ey, o[2] = g ? sz : ez, o[3] = rowa >= 0 ? inv : (T)0;
        }
        // radial factors, and with SEP later the base functions (n of them from function `first` on): lane group g has
        // k = 4 s + g
        T gv[NK], gd[NK];
        T fr = 0;  // dE/dr
        const T* __restrict__ ga = P.lut_g + (size_t)(rowa < 0 ? 0 : rowa) * P.stride_g;
        auto functions = [&](auto steps, int first, int n) {
            constexpr int N = decltype(steps)::value;
            Coef<T> c[N];
#pragma unroll
            for (int s = 0; s < N; ++s) c[s] = coef_at(ga + 4 * (first + (4 * s + g < n ? 4 * s + g : 0)));
#pragma unroll
            for (int s = 0; s < N; ++s) {
                const bool on = rowa >= 0 && 4 * s + g < n;
                gv[s] = on ? coef_value(c[s], wa) : (T)0;
                gd[s] = on ? coef_slope(c[s], wa, rsa) : (T)0;
            }
        };
        {
            const Coef<T> cc = coef_at(ga + 4 * (og + P.nb_a));
            functions(std::integral_constant<int, NA>(), 0, nf);
            if (g == 0 && rowa >= 0) fr = edf * coef_slope(cc, wa, rsa);  // core term
        }
        // M and M' of the pair, spread over its four lanes
        {
            const T* __restrict__ ma = P.lut_m + (size_t)(rowm < 0 ? 0 : rowm) * P.stride_m + 4 * P.nb_m;
            constexpr int U = 4;
            for (int k0 = g; k0 < nfm; k0 += 4 * U) {
                Coef<T> c[U];
#pragma unroll
                for (int u = 0; u < U; ++u) c[u] = coef_at(ma + 4 * (k0 + 4 * u < nfm ? k0 + 4 * u : 0));
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (k0 + 4 * u < nfm)
                        sM[k0 + 4 * u] = {rowm == kRowOne ? (T)1 : rowm < 0 ? (T)0 : coef_value(c[u], wm),
                                          rowm < 0 ? (T)0 : coef_slope(c[u], wm, rsm)};
            }
        }
        // h_q: M_{l',n'} Re Y_l'm' at column m', M_{l',n'} Im Y_l'm' at -m'; each lane of the pair the orders of its
        // walk
        for (int q = P.nm3 + g; q < D.nqp; q += 4) sH[q] = (T)0;
        wave_order();
        {
            Walk<T> k;
            for (int t = 0; t < P.sth; ++t) {
                const ForceStep<T> st = sStep[4 * (P.sta + t) + g];
                k.step(st, sz, sP, P.firstm >> t & 1);
                const int l = st.l(), m = st.m();
                if ((st.lm >> 17 & 1) && l <= P.l3m) {
                    const cplx<T> y = k.value();
                    for (int np = 0; np < P.nr3m; ++np) {
                        const T mv = sM[l * P.nr2m + np].re;
                        T* h = sH + np * P.lsm3 + l * l + l;
                        h[m] = mv * y.re;
                        if (m > 0) h[-m] = mv * y.im;
                    }
                }
            }
        }
        wave_order();
        put_powers(sP, g, ex, ey);
        wave_order();
        // ---- bonds
        T gx = 0, gy = 0, gz = 0;
        for (int rd = 0; rd < D.rounds; ++rd) {
            const int q0 = 4 * (P.qsplit ? 4 * rd + g : rd);
            T h[4], u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                h[r] = sH[q0 + r];
                u[r] = 0;
            }
            const cplx<T>* __restrict__ v = sV + (size_t)rd * P.sta * NA * 64 + lane;
            Walk<T> k;
            for (int t = 0; t < P.sta; ++t, v += NA * 64) {
                const ForceStep<T> st = sStep[4 * t + g];
                V pr = (V)(T)0, pi = (V)(T)0, qr = (V)(T)0, qi = (V)(T)0;
#pragma unroll
                for (int s = 0; s < NA; ++s) {
                    const cplx<T> a = v[64 * s];
                    pr = Mm<T>::mul(a.re, gv[s], pr);
                    pi = Mm<T>::mul(a.im, gv[s], pi);
                    qr = Mm<T>::mul(a.re, gd[s], qr);
                    qi = Mm<T>::mul(a.im, gd[s], qi);
                }
                k.step(st, ez, sP, P.firsta >> t & 1);
                const cplx<T> y = k.value();
                T Sr = 0, Si = 0, Rr = 0, Ri = 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    Sr = fma(pr[r], h[r], Sr);
                    Si = fma(pi[r], h[r], Si);
                    Rr = fma(qr[r], h[r], Rr);
                    Ri = fma(qi[r], h[r], Ri);
                    u[r] = fma(-pi[r], y.im, fma(pr[r], y.re, u[r]));
                }
                fr = fma(-Ri, y.im, fma(Rr, y.re, fr));
                k.gradient(Sr, Si, gx, gy, gz);
            }
            if (P.qsplit) {
#pragma unroll
                for (int r = 0; r < 4; ++r) sH[q0 + r] = u[r];
            } else {
                sH[q0 + g] = fold_groups(u);  // the four walks together
            }
        }
        if constexpr (SEP) functions(std::integral_constant<int, NK>(), og, P.nb_a);
        wave_order();
        put_powers(sP, g, sx, sy);
        wave_order();
        // ---- moments: four (step, n') a tile
        T tr = 0, tx = 0, ty = 0, tz = 0;
        {
            const cplx<T>* __restrict__ v = sV + (size_t)D.rounds * P.sta * NA * 64 + lane;
            Walk<T> k;
            ForceStep<T> st = {};
            T Sr = 0, Si = 0, S1r = 0, S1i = 0, Rr = 0, Ri = 0;  // sums over n' of M X, M' X, M Q
            int np = 0, t = 0;
            for (int tile = 0; tile < tm; ++tile, v += NK * 64) {
                V pr = (V)(T)0, pi = (V)(T)0, qr = (V)(T)0, qi = (V)(T)0;
#pragma unroll
                for (int s = 0; s < NK; ++s) {
                    const cplx<T> a = v[64 * s];
                    pr = Mm<T>::mul(a.re, gv[s], pr);
                    pi = Mm<T>::mul(a.im, gv[s], pi);
                    qr = Mm<T>::mul(a.re, gd[s], qr);
                    qi = Mm<T>::mul(a.im, gd[s], qi);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (t < P.stm) {
                        if (np == 0) {
                            st = sStep[4 * (P.sta + t) + g];
                            k.step(st, sz, sP, P.firstm >> t & 1);
                            Sr = Si = S1r = S1i = Rr = Ri = (T)0;
                        }
                        const cplx<T> mv = sM[(st.lm >> 18) + np];
                        T xr = pr[r], xi = pi[r];
                        if (np < P.nr3m && t < P.sth) {
                            // dE/dH of the column of A
                            const int l = st.l(), m = st.m();
                            const bool on = l <= P.l3m;
                            const T* a = sH + (on ? np * P.lsm3 + l * l + l : 0);
                            xr += on ? a[m] : (T)0;
                            xi -= on && m > 0 ? a[-m] : (T)0;
                        }
                        Sr = fma(mv.re, xr, Sr);
                        Si = fma(mv.re, xi, Si);
                        S1r = fma(mv.im, xr, S1r);
                        S1i = fma(mv.im, xi, S1i);
                        Rr = fma(mv.re, qr[r], Rr);
                        Ri = fma(mv.re, qi[r], Ri);
                        if (++np == P.nr2m) {
                            const cplx<T> y = k.value();
                            fr = fma(-Ri, y.im, fma(Rr, y.re, fr));
                            tr = fma(-S1i, y.im, fma(S1r, y.re, tr));
                            k.gradient(Sr, Si, tx, ty, tz);
                            np = 0;
                            ++t;
                        }
                    }
                }
            }
        }
        // the four walks of a pair together
        {
            const T a[4] = {fr, gx, gy, gz}, b[4] = {tr, tx, ty, tz};
            const T ra = fold_groups(a), rb = fold_groups(b);
            wave_order();
            sR[8 * ji + g] = ra;
            sR[8 * ji + 4 + g] = rb;
        }
        wave_order();
        // dE/dr e + (G - (G.e) e) / r, and the same of the moment; lane i has value i of the 16 pairs' 48, so that a
        // store covers whole lines, also where the results lie in host memory
        if (lane < 3 * min(16, nn - c0)) {
            const int j = lane / 3, x = lane - 3 * j;
            const T* e = sE + 8 * j;
            const T* v = sR + 8 * j;
            const bool pair = e[3] != (T)0;
            const T ge = v[1] * e[0] + v[2] * e[1] + v[3] * e[2], gs = v[5] * e[4] + v[6] * e[5] + v[7] * e[6];
            const size_t o = 3 * ((size_t)p0 + c0) + lane;
            flist[o] = pair ? (double)fma(v[0], e[x], e[3] * (v[1 + x] - ge * e[x])) : 0.0;
            tlist[o] = pair ? (double)fma(v[4], e[4 + x], e[7] * (v[5 + x] - gs * e[4 + x])) : 0.0;
        }
        wave_order();
    }
}

namespace {

template <typename T, int NK, int NA, bool SEP>
hipError_t launch_forces(const DevParams<T>& P, int natom, const int* off, const double* dlist, const double* elist,
                         const double* dmomi, const double* emomi, const double* dmom, const double* emom,
                         const Buffers& B, bool scaled, double* flist, double* tlist, double* tlist0, hipStream_t s) {
    auto k = k_forces_mm<T, NK, NA, SEP>;
    int waves = 4;
    auto bytes = [&] {
        return (size_t)ForceLds(NA, NK, P.sta, (P.nm3 + 3) >> 2, (P.stm * P.nr2m + 3) >> 2, 4 * (P.sta + P.stm), P.qsplit,
                                P.nr2m * (P.l2m + 1), waves, sizeof(T)).size * sizeof(T);
    };
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
    while (waves > 1 && bytes() > limit) waves >>= 1;
    const size_t lds = bytes();
    if (lds > limit) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k, dim3(natom), dim3(64 * waves), lds, s, P, off, dlist, elist, dmomi, emomi, dmom, emom,
                       (const cplx<T>*)B.W, scaled, B.dE, B.edf, flist, tlist, tlist0, B.err);
    return hipGetLastError();
}

}  // namespace

template <typename T>
hipError_t run_forces(const DevParams<T>& P, int natom, const int* off, const double* dlist, const double* elist,
                      const double* dmomi, const double* emomi, const double* dmom, const double* emom, const Buffers& B,
                      bool scaled, double* flist, double* tlist, double* tlist0, hipStream_t s) {
    auto go = [&](auto k) { return k(P, natom, off, dlist, elist, dmomi, emomi, dmom, emom, B, scaled, flist, tlist, tlist0, s); };
    if (P.og > 0) {
        if (P.nb_a <= 4) return go(launch_forces<T, 1, 1, true>);
        if (P.nb_a <= 8) return go(launch_forces<T, 2, 2, true>);
        if (P.nb_a <= 12) return P.nf <= 8 ? go(launch_forces<T, 3, 2, true>) : go(launch_forces<T, 3, 3, true>);
        return P.nf <= 8 ? go(launch_forces<T, 4, 2, true>) : go(launch_forces<T, 4, 4, true>);
    }
    if (P.nb_a <= 4) return go(launch_forces<T, 1, 1, false>);
    if (P.nb_a <= 8) return go(launch_forces<T, 2, 2, false>);
    if (P.nb_a <= 12) return go(launch_forces<T, 3, 3, false>);
    return go(launch_forces<T, 4, 4, false>);
}

template hipError_t run_forces<double>(const DevParams<double>&, int, const int*, const double*, const double*,
                                       const double*, const double*, const double*, const double*, const Buffers&, bool,
                                       double*, double*, double*, hipStream_t);
template hipError_t run_forces<float>(const DevParams<float>&, int, const int*, const double*, const double*,
                                      const double*, const double*, const double*, const double*, const Buffers&, bool,
                                      double*, double*, double*, hipStream_t);

}  // namespace magace
