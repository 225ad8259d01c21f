// adjoint.hip -- dRho/dZ and the energy of every atom from the node plan (nodes.cpp).
//
// k_adjoint_nodes does the work of prepB + forceweights (src/b_basis.F90:62-307,
// src/forces.F90:84-349) for one density and body orders 2 to 4: with the pair products X_p
// (A0 entry times A entry) and X_q (A times A) it forms G_p = sum w X_q and G_q = sum w X_p, a
// sparse matrix with constant weights times the atoms' products, and takes the gradient in the
// entries of Z from G times the other factor.  One workgroup holds two atoms in FP32 (an LDS slot
// is 16 bytes: both atoms' complex values) and one in FP64.
//
// The sparse product works on blocks of four rows that share most of their columns: a column is
// read from LDS once for four rows (fill 0.87 for the lmax-6 header), a lane holds one block (or
// a 2^s-th of its columns), and the tables stream from L2 once per workgroup.
//
// Measured on 16000 atoms of the lmax-6 header against the walk over three-factor gradient records
// (k_adjoint, k_adjoint_pair): mixed 786 -> 388 us, FP64 1566 -> 893 us; 4394 atoms of the example
// potential's shape 214 -> 97 us and 369 -> 230 us; 27648 atoms of the lmax-4 header 346 -> 205 us
// and 621 -> 414 us.  What bounds it: in FP32 the vector units, 63% busy, and the latency between the phases; in
// FP64 (40%) also the tables' way from L2 (0.83 MB a workgroup, 15 TB/s together; 0.44 MB in FP32).
#include <hip/hip_runtime.h>

#include "device.hpp"
#include "kernels.hpp"

namespace magace {

namespace {

template <typename T> struct Slot {  // one LDS slot: 16 bytes
    typedef T V __attribute__((ext_vector_type(16 / sizeof(T))));
};
template <typename T> __device__ __forceinline__ typename Slot<T>::V slot_get(uint32_t off) {
    return lds_at<T, 16 / sizeof(T)>(off);
}
template <typename T> __device__ __forceinline__ void slot_put(uint32_t off, typename Slot<T>::V v) {
    typedef typename Slot<T>::V V;
    *(__attribute__((address_space(3))) V*)(size_t)off = v;
}
__device__ __forceinline__ Slot<float>::V slot_mul(Slot<float>::V a, Slot<float>::V b) {
    Slot<float>::V r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    r.z = a.z * b.z - a.w * b.w;
    r.w = a.z * b.w + a.w * b.z;
    return r;
}
__device__ __forceinline__ Slot<double>::V slot_mul(Slot<double>::V a, Slot<double>::V b) {
    Slot<double>::V r;
    r.x = a.x * b.x - a.y * b.y;
    r.y = a.x * b.y + a.y * b.x;
    return r;
}
// the sign bits of a gradient record: real part (bit 30), imaginary part (bit 31)
__device__ __forceinline__ float flip(float v, uint32_t mask) { return __uint_as_float(__float_as_uint(v) ^ mask); }
__device__ __forceinline__ double flip(double v, uint32_t mask) {
    return __hiloint2double((int)((uint32_t)__double2hiint(v) ^ mask), __double2loint(v));
}
__device__ __forceinline__ Slot<float>::V slot_flip(Slot<float>::V v, uint32_t re, uint32_t im) {
    Slot<float>::V r;
    r.x = flip(v.x, re), r.y = flip(v.y, im), r.z = flip(v.z, re), r.w = flip(v.w, im);
    return r;
}
__device__ __forceinline__ Slot<double>::V slot_flip(Slot<double>::V v, uint32_t re, uint32_t im) {
    Slot<double>::V r;
    r.x = flip(v.x, re), r.y = flip(v.y, im);
    return r;
}
// +-1 with the sign of bit 31
__device__ __forceinline__ float unit(uint32_t b, float) { return __uint_as_float((b & 0x80000000u) | 0x3f800000u); }
__device__ __forceinline__ double unit(uint32_t b, double) {
    return __hiloint2double((int)((b & 0x80000000u) | 0x3ff00000u), 0);
}
// s + t with the signs of a gradient record
template <typename V> __device__ __forceinline__ V slot_add(V s, V t, uint32_t rec) {
    const auto re = unit(rec << 1, s[0]), im = unit(rec, s[0]);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(V) / sizeof(s[0])); ++i) s[i] = fma(i & 1 ? im : re, t[i], s[i]);
    return s;
}
// sums over the 2^s lanes of a block, every lane with the result: rows of 16 by the vector units' lane
// permutations (7 - i and 15 - i do for i + 4 and i + 8, as 4 and 8 lanes hold one value by then), where shuffles
// through LDS had been half of its instructions at lmax 4
template <int CTRL> __device__ __forceinline__ float lane_mov(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xf, 0xf, true));
}
template <int CTRL> __device__ __forceinline__ double lane_mov(double v) {
    return __hiloint2double(__builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true));
}
template <typename F> __device__ __forceinline__ void sum_lanes(int s, F&& each) {
    // each(f): v = f(v) for all values
    if (s < 1) return;
    each([](auto x) { return x + lane_mov<0xb1>(x); });  // quads 1 0 3 2
    if (s < 2) return;
    each([](auto x) { return x + lane_mov<0x4e>(x); });  // quads 2 3 0 1
    if (s < 3) return;
    each([](auto x) { return x + lane_mov<0x141>(x); });  // 7 - i
    if (s < 4) return;
    each([](auto x) { return x + lane_mov<0x140>(x); });  // 15 - i
    if (s < 5) return;
    each([](auto x) { return fold16(x, x); });
    if (s < 6) return;
    each([](auto x) { return fold32(x, x); });
}
template <int N, typename V> __device__ __forceinline__ void sum_slots(int s, V (&v)[N]) {
    sum_lanes(s, [&](auto f) {
#pragma unroll
        for (int r = 0; r < N; ++r)
#pragma unroll
            for (int i = 0; i < (int)(sizeof(V) / sizeof(v[r][0])); ++i) v[r][i] = f(v[r][i]);
    });
}

// A lane's records, read four steps ahead of their use: the tasks of a wave are one stream in memory,
// so the ring runs on from task to task and across the barriers between the phases.  A task's steps
// are a multiple of four, so that the ring's registers keep their places (moving a loaded value would
// wait for it).
template <typename T>
struct Ring {
    static_assert(kNodeQuantumDev == 4, "a turn of the ring is four steps");
    typedef typename NodeTab<T>::W4 W4;
    const uint2* __restrict__ col;
    const W4* __restrict__ w;
    uint2 c;
    W4 wt[4];
    __device__ __forceinline__ void start(const NodeTab<T>& N, int step, int lane) {
        col = N.col + (size_t)(step >> 2) * 64 + lane;
        w = N.w + (size_t)step * 64 + lane;
        c = col[0];
#pragma unroll
        for (int u = 0; u < 4; ++u) wt[u] = w[u * 64];
    }
};

// four rows' sums over the columns of one task; every lane of a block ends with the block's sums
template <typename T>
__device__ __forceinline__ void side_task(Ring<T>& R, int steps, int s, typename Slot<T>::V (&acc)[4]) {
    typedef typename Slot<T>::V V;
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = (V)(T)0;
    for (int k = 0; k < steps; k += 4) {
        const V x[4] = {slot_get<T>((R.c.x & 0xffff) << 4), slot_get<T>((R.c.x >> 16) << 4),
                        slot_get<T>((R.c.y & 0xffff) << 4), slot_get<T>((R.c.y >> 16) << 4)};
        R.col += 64;
        R.w += 256;
        R.c = R.col[0];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] = R.wt[u].v[r] * x[u] + acc[r];
            R.wt[u] = R.w[u * 64];
        }
    }
    sum_slots(s, acc);
}

}  // namespace

// NT threads, 64 a wave of the plan.
// Phases, a barrier between them: entries of Z to LDS; pair products; G_p (in registers); G_q, which
// replaces X_q; G_p in place of X_p, and rho = Re sum X_p G_p on the way; the gradient.  Each phase
// issues the first table loads of the next before the barrier.
template <typename T, int NT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4, 8)))
k_adjoint_nodes(DevParams<T> P, NodeTab<T> N, const cplx<T>* __restrict__ Zin, cplx<T>* __restrict__ Wout,
                const double* __restrict__ ehc, const double* __restrict__ rho1, double* __restrict__ eout,
                double* __restrict__ dEout, double* __restrict__ edfout, double* __restrict__ rho_out, int natom) {
    typedef typename Slot<T>::V V;
    constexpr int NA = sizeof(T) == 4 ? 2 : 1;  // atoms of a workgroup
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int a0 = NA * (int)blockIdx.x;
    const bool two = NA == 2 && a0 + 1 < natom;
    double* red = (double*)(smem + (size_t)N.nslots * 16);  // [NA][NT / 64]
    const cplx<T>* __restrict__ Z0 = Zin + (size_t)a0 * P.nz;
    const cplx<T>* __restrict__ Z1 = two ? Z0 + P.nz : Z0;  // an odd last atom is paired with itself
    auto load = [&](uint32_t e) {  // a ZLayout::half entry
        V v;
        const uint32_t x = e & 0xfff;
        const cplx<T> a = Z0[x];
        v[0] = a.re, v[1] = a.im;
        if constexpr (NA == 2) {
            const cplx<T> b = Z1[x];
            v[2] = b.re, v[3] = b.im;
        }
        return slot_flip(v, (e << 17) & 0x80000000u, (e << 16) & 0x80000000u);
    };
    // the atoms' e_hc and B1 part of rho, read ahead by the threads that evaluate their energies
    const int eatom = tid == NT - 64 ? a0 : NA == 2 && tid == NT - 63 && two ? a0 + 1 : -1;
    double e_hc = 0.0, r1v = 0.0;
    if (eatom >= 0) {
        e_hc = ehc[eatom];
        r1v = rho1[eatom];
    }
    // the headers of the wave's tasks, one a lane
    const int4 head = N.head[wave * 64 + lane];
    auto head_of = [&](int t) {
        return make_int3(__builtin_amdgcn_readlane(head.x, t), __builtin_amdgcn_readlane(head.y, t),
                         __builtin_amdgcn_readlane(head.z, t));
    };
    // Entries of Z, four in flight a thread, and the sums over A2 entries, eight lanes an A0 entry: all places are
    // loaded before the first entry, so that the phase is two trips to memory.
    constexpr int UZ = 4, KD = 2;
    {
        uint32_t cz[UZ], dx[KD];
        T dw[KD];
        V v[UZ], dv[KD];
        const int di = tid >> 3;
#pragma unroll
        for (int u = 0; u < UZ; ++u) cz[u] = N.core_z[u * NT + tid < N.slot_one ? u * NT + tid : 0];
        auto places = [&](int i, int k0) {
#pragma unroll
            for (int k = 0; k < KD; ++k) {
                const bool on = i < N.nd && k0 + k < N.kd;
                const int r = on ? ((k0 + k) * N.nd + i) * 8 + (tid & 7) : 0;
                dx[k] = N.nd > 0 ? N.d_x[r] : 0u;
                dw[k] = on ? N.d_w[r] : (T)0;
            }
        };
        places(di, 0);
#pragma unroll
        for (int u = 0; u < UZ; ++u) v[u] = load(cz[u]);
#pragma unroll
        for (int k = 0; k < KD; ++k) dv[k] = load(dx[k]);
#pragma unroll
        for (int u = 0; u < UZ; ++u)
            if (u * NT + tid < N.slot_one) slot_put<T>(16 * (u * NT + tid), v[u]);
        for (int i = UZ * NT + tid; i < N.slot_one; i += NT) slot_put<T>(16 * i, load(N.core_z[i]));
        if (tid < 2) {
            V o = (V)(T)0;
            if (tid == 0) {
                o[0] = (T)1;
                if constexpr (NA == 2) o[2] = (T)1;
            }
            slot_put<T>(16 * (N.slot_one + tid), o);
        }
        for (int i = di; i < N.nd; i += NT / 8) {
            V s[1] = {(V)(T)0};
            if (i != di) places(i, 0);
            for (int k0 = 0; k0 < N.kd; k0 += KD) {
                if (k0 > 0 || i != di)
#pragma unroll
                    for (int k = 0; k < KD; ++k) dv[k] = load(dx[k]);
                T w[KD];
#pragma unroll
                for (int k = 0; k < KD; ++k) w[k] = dw[k];
                if (k0 + KD < N.kd) places(i, k0 + KD);
#pragma unroll
                for (int k = 0; k < KD; ++k) s[0] = w[k] * dv[k] + s[0];
            }
            sum_slots(3, s);
            if ((tid & 7) == 0) slot_put<T>(16 * (N.d_slot[i] & 0xffff), s[0]);
        }
    }
    const int3 cnt = head_of(62), first = head_of(63);
    const int npt = cnt.x, nqt = cnt.y, ngt = cnt.z;
    Ring<T> R;
    R.start(N, first.x, lane);
    constexpr int U = 4;  // node indices in flight
    uint32_t ab[U];
#pragma unroll
    for (int u = 0; u < U; ++u) ab[u] = u * NT + tid < N.npair ? N.pair[u * NT + tid] : 0u;
    constexpr int K2 = 2;  // an A2 entry's terms read ahead
    uint32_t a2c[K2];
    T a2w[K2];
#pragma unroll
    for (int k = 0; k < K2; ++k) {
        const bool on = tid < N.na2 && k < N.k2;
        a2c[k] = on ? N.a2_c[k * N.na2 + tid] : 0u;
        a2w[k] = on ? N.a2_w[k * N.na2 + tid] : (T)0;
    }
    const int a2x = tid < N.na2 ? N.a2_x[tid] : 0;
    __syncthreads();
    cplx<T>* __restrict__ W0 = Wout + (size_t)a0 * P.nz;
    auto store = [&](int x, V v) {
        W0[x] = {v[0], v[1]};
        if constexpr (NA == 2)
            if (two) W0[P.nz + x] = {v[2], v[3]};
    };
    // A2 entries need the A0 entries only
    auto a2_term = [&](V s, uint32_t c, T w) {
        return w * slot_flip(slot_get<T>((c & 0x3fff) << 4), 0u, c & 0x80000000u) + s;
    };
    for (int i = tid; i < N.na2; i += NT) {
        V s = (V)(T)0;
        if (i == tid) {
#pragma unroll
            for (int k = 0; k < K2; ++k)
                if (k < N.k2) s = a2_term(s, a2c[k], a2w[k]);
        }
        for (int k0 = i == tid ? K2 : 0; k0 < N.k2; k0 += 4) {
            uint32_t c[4];
            T w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int r = (k0 + k < N.k2 ? k0 + k : k0) * N.na2 + i;
                c[k] = N.a2_c[r];
                w[k] = k0 + k < N.k2 ? N.a2_w[r] : (T)0;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) s = a2_term(s, c[k], w[k]);
        }
        store(i == tid ? a2x : (int)N.a2_x[i], s);
    }
    for (int i0 = 0; i0 < N.npair; i0 += U * NT) {
        uint32_t nb[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + (U + u) * NT + tid;
            nb[u] = i < N.npair ? N.pair[i] : 0u;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * NT + tid;
            if (i < N.npair)
                slot_put<T>(16 * (N.first_node + i),
                            slot_mul(slot_get<T>((ab[u] & 0xffff) << 4), slot_get<T>((ab[u] >> 16) << 4)));
            ab[u] = nb[u];
        }
    }
    __syncthreads();
    V gp[kNodeTasksDev][4];
    ushort4 prow[kNodeTasksDev];
#pragma unroll
    for (int t = 0; t < kNodeTasksDev; ++t)
        if (t < npt) {
            const int3 h = head_of(t);
            prow[t] = N.row[h.z + (lane >> h.y)];
            side_task<T>(R, h.x, h.y, gp[t]);
        }
    __syncthreads();
    for (int t = npt; t < npt + nqt; ++t) {
        const int3 h = head_of(t);
        const ushort4 row = N.row[h.z + (lane >> h.y)];
        V g[4];
        side_task<T>(R, h.x, h.y, g);
        if ((lane & ((1 << h.y) - 1)) == 0) {
            const unsigned short rs[4] = {row.x, row.y, row.z, row.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (rs[r] == 0xffff) continue;
                if (rs[r] & 0x4000)  // a single entry: its sum waits in its row of W
                    store(rs[r] & 0xfff, g[r]);
                else
                    slot_put<T>(16 * rs[r], g[r]);
            }
        }
    }
    constexpr int DG = kNodeQuantumGDev / 2;  // pairs of gradient records read ahead
    const uint2* __restrict__ rec = N.g_rec + (size_t)(first.y >> 1) * 64 + lane;
    uint2 gn[DG];
#pragma unroll
    for (int u = 0; u < DG; ++u) gn[u] = rec[u * 64];
    __syncthreads();
    double rho[NA];
#pragma unroll
    for (int a = 0; a < NA; ++a) rho[a] = 0.0;
    auto tally = [&](V x, V g) {
#pragma unroll
        for (int a = 0; a < NA; ++a) rho[a] += (double)fma(x[2 * a], g[2 * a], -x[2 * a + 1] * g[2 * a + 1]);
    };
#pragma unroll
    for (int t = 0; t < kNodeTasksDev; ++t)
        if (t < npt) {
            const int3 h = head_of(t);
            if ((lane & ((1 << h.y) - 1)) == 0) {
                const unsigned short rs[4] = {prow[t].x, prow[t].y, prow[t].z, prow[t].w};
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (rs[r] != 0xffff) {
                        tally(slot_get<T>(16 * rs[r]), gp[t][r]);
                        slot_put<T>(16 * rs[r], gp[t][r]);
                    }
            }
        }
    for (int i = tid; i < N.nd; i += NT) {
        const uint32_t s = N.d_slot[i];
        tally(slot_get<T>((s >> 16) << 4), slot_get<T>((s & 0xffff) << 4));
    }
#pragma unroll
    for (int a = 0; a < NA; ++a) {
        sum_lanes(6, [&](auto f) { rho[a] = f(rho[a]); });
        if (lane == 0) red[a * (NT / 64) + wave] = rho[a];
    }
    __syncthreads();
    // the gradient of the stored entries (0 where the conjugate partner stands for the pair)
    auto fetch = [&](int x) {
        V v;
        const cplx<T> a = W0[x];
        v[0] = a.re, v[1] = a.im;
        if constexpr (NA == 2) {
            const cplx<T> b = W0[two ? P.nz + x : x];
            v[2] = b.re, v[3] = b.im;
        }
        return v;
    };
    for (int t = npt + nqt; t < npt + nqt + ngt; ++t) {
        const int3 h = head_of(t);
        const bool lead = (lane & ((1 << h.y) - 1)) == 0;
        const uint32_t row = lead ? N.g_row[h.z + (lane >> h.y)] : 0x80000000u;
        const int x = row & 0xfff, xb = row >> 12 & 0xfff;
        V s[1] = {(V)(T)0}, own = (V)(T)0, part = (V)(T)0;
        if (row & (1u << 24)) own = fetch(x);
        if (row & (1u << 25)) part = fetch(xb);
        for (int k = 0; k < h.x; k += 2 * DG) {
#pragma unroll
            for (int u = 0; u < DG; ++u) {
                const uint2 r = gn[u];
                gn[u] = rec[(DG + u) * 64];
                const V t0 = slot_mul(slot_get<T>((r.x & 0x3fff) << 4), slot_get<T>((r.x >> 12) & 0x3fff0));
                const V t1 = slot_mul(slot_get<T>((r.y & 0x3fff) << 4), slot_get<T>((r.y >> 12) & 0x3fff0));
                s[0] = slot_add(s[0], t0, r.x);
                s[0] = slot_add(s[0], t1, r.y);
            }
            rec += 64 * DG;
        }
        sum_slots(h.y, s);
        if (!(row >> 31)) {
            // the conjugate partner's single sum enters as s conj(G)
            const uint32_t minus = row & (1u << 26) ? 0x80000000u : 0u;
            store(x, s[0] + own + slot_flip(part, minus, minus ^ 0x80000000u));
        }
    }
    if (eatom >= 0) {
        double tot = 0.0, sc[1];
        for (int w = 0; w < NT / 64; ++w) tot += red[(eatom - a0) * (NT / 64) + w];
        const double t[1] = {tot};
        atom_energy<T>(P, 1, eatom, t, e_hc, &r1v, eout, dEout, edfout, rho_out, sc);
    }
}

__global__ void k_node_weights(int n, const int* __restrict__ t, const double* __restrict__ w,
                               double* __restrict__ w64, float* __restrict__ w32) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double v = t[i] < 0 ? 0.0 : (t[i] & 1) ? -w[t[i] >> 1] : w[t[i] >> 1];
    w64[i] = v;
    w32[i] = (float)v;
}

hipError_t fill_node_weights(const NodeWeights& n, const double* w, hipStream_t s) {
    if (n.n > 0)
        hipLaunchKernelGGL(k_node_weights, dim3((n.n + 255) / 256), dim3(256), 0, s, n.n, n.t, w, n.w64, n.w32);
    return hipGetLastError();
}

template <typename T>
hipError_t run_adjoint_nodes(const DevParams<T>& P, const NodeTab<T>& N, int natom, const Buffers& B, double* eout,
                             hipStream_t s) {
    constexpr int NA = sizeof(T) == 4 ? 2 : 1;
    const size_t lds = (size_t)N.nslots * 16 + (size_t)2 * 16 * sizeof(double);
    static bool set = false;
    hipError_t e;
    if (!set) {
        int dev = 0, most = 0;
        if ((e = hipGetDevice(&dev)) != hipSuccess) return e;
        if ((e = hipDeviceGetAttribute(&most, hipDeviceAttributeMaxSharedMemoryPerBlock, dev)) != hipSuccess) return e;
        for (const void* k : {(const void*)k_adjoint_nodes<T, 256>, (const void*)k_adjoint_nodes<T, 512>,
                              (const void*)k_adjoint_nodes<T, 1024>}) {
            hipFuncAttributes fa;
            if ((e = hipFuncGetAttributes(&fa, k)) != hipSuccess) return e;
            if (fa.sharedSizeBytes != 0) return hipErrorInvalidKernelFile;  // slots are addressed from 0
            if ((e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, most)) != hipSuccess) return e;
        }
        set = true;
    }
    const dim3 grid((unsigned)((natom + NA - 1) / NA));
    auto k = N.nw == 4 ? k_adjoint_nodes<T, 256> : N.nw == 8 ? k_adjoint_nodes<T, 512> : k_adjoint_nodes<T, 1024>;
    hipLaunchKernelGGL(k, grid, dim3(64 * N.nw), lds, s, P, N, (const cplx<T>*)B.Z, (cplx<T>*)B.W, B.ehc, B.rho1, eout,
                       B.dE, B.edf, B.rho, natom);
    return hipGetLastError();
}

template hipError_t run_adjoint_nodes<double>(const DevParams<double>&, const NodeTab<double>&, int, const Buffers&,
                                              double*, hipStream_t);
template hipError_t run_adjoint_nodes<float>(const DevParams<float>&, const NodeTab<float>&, int, const Buffers&,
                                             double*, hipStream_t);

}  // namespace magace
