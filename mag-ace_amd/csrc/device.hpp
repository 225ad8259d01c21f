// device.hpp -- device-side parameter block and launch interface of the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace magace {

template <typename T>
struct cplx {
    T re, im;
};

// threads of an adjoint workgroup; chunk c of the gradient records runs on thread
// c % kAdjointThreads, and the chunk order built with the records assumes this count
constexpr int kAdjointThreads = 512;
// slots per group of the adjoint's first combine pass (TermList::kGroup)
constexpr int kCombGroup = 8;

// Everything a kernel needs about the potential, passed by value as a kernel argument.
template <typename T>
struct DevParams {
    const T* lut_a = nullptr;  // atomic spline rows [nlut][stride_a]
    const T* lut_m = nullptr;  // magnetic spline rows [nlut][stride_m]
    // rows of the radial factors h_1..h_nf (RadialFactors), the base functions g_1..g_nb and the core term
    // [nlut][stride_g]; the g begin at function og.  og = 0: the factors are the g, nf = nb_a.
    const T* lut_g = nullptr;
    int nf = 0, og = 0;
    const T* cperm = nullptr;  // coefficients of the factors in R_{l,n} as A operands, [l3a + 1][4][64] (density.hip)
    // columns of the density's products, 16 a tile: of A (Y entry | q << 8 | l << 16), then of A2 (Y' entry | M
    // entry << 8)
    const uint32_t* cols = nullptr;
    // forces (forces.hip): walks through the harmonics, four lane groups a step, of the bonds (sta steps; all
    // groups the same if qsplit, each with columns q of its own) and of the moments (stm, of which the first
    // sth meet l' <= l3m): a, b, c, l | m << 8 | first of its order << 16 | harmonic << 17 |
    // l nr2m << 18, firsta and firstm the steps that are some group's first of an order; rows of the tiles of
    // V: column of A | l << 16 | it and y are a pair +m', -m' << 25 | its sine << 26 | its odd m' << 27, column of
    // A2 | 1 << 24, or ~0; coefficients of the factors [l3a + 1][8][16]
    const double* steps = nullptr;
    const uint2* vcol = nullptr;
    const T* crow = nullptr;
    int sta = 0, stm = 0, sth = 0;
    uint32_t firsta = 0, firstm = 0;
    bool qsplit = false;
    // places of Z and W in memory (ZLayout::half): offsets of A2 and A0, entries, and the place of every
    // full index
    int hA2 = 0, hA0 = 0, nzh = 0;
    const unsigned short* zmap = nullptr;
    int stride_a = 0, stride_m = 0, stride_g = 0, nlut = 0;
    double rs_a = 0, rs_m = 0;  // nlut / cutoff (index arithmetic stays FP64)
    int nb_a = 0, nb_m = 0, nr2m = 0, l2m = 0, nr3a = 0, nr3m = 0, l3a = 0, l3m = 0;
    int lsa = 0, lsm = 0, lsm3 = 0, nm3 = 0, oA2 = 0, oA0 = 0, nz = 0;
    int lha = 0, lhm = 0;  // (l+1)(l+2)/2 for l3a, l2m
    int sa = 0;                 // k_density: neighbour split of the A tasks (0 = automatic)
    // gradient contributions, one 16-byte record each: x = a | b << 16, y = c as byte offsets
    // of the factors in the adjoint's LDS copy of Z (index * sizeof(cplx<T>)), (z, w) = weight
    // (FP64 bits as lo/hi words, or FP32 bits in z)
    const uint4* crec = nullptr;
    const uint4* crec16 = nullptr;   // FP32 only: the records with offsets of 16-byte entries (two
                                     // atoms' Z interleaved, k_adjoint_pair)
    // FP32 without the accumulation recipe: the same records with the three offsets in x, y, z
    // as they are (no unpacking) and the FP32 weight in w; 8-byte entries (crecu) and 16-byte
    // entries (crec16u, k_adjoint_pair)
    const uint4* crecu = nullptr;
    const uint4* crec16u = nullptr;
    const int2* chunks = nullptr;    // (start, target | count << 12 | sole << 18 | slot << 19), count = its
                                     // group's length; chunk c runs on thread c % kAdjointThreads
    // partial-sum combine (TermList::comb, comb2): groups of <= kCombGroup slots
    // (first slot, target | slots << 12 | only group << 16) and targets with several groups
    // (first slot, target | groups << 12)
    const int2* comb = nullptr;
    const int2* comb2 = nullptr;
    int ncomb = 0, ncomb2 = 0, nslot = 0;  // groups, such targets, partial-sum slots per atom and density
    const uint32_t* fold = nullptr;  // conjugate-pair folding of W (see TermList::fold)
    // products Y_i = Z[a] Z[b] at index nz + 1 + i (body orders 5, 6; TermList::ypair), and the
    // way of their gradient back to Z: per target (first term, target | terms << 12), per term
    // (index of Y, the other factor)
    const int2* ypair = nullptr;
    const int2* yft = nullptr;
    const int2* yfe = nullptr;
    int ny = 0, nyt = 0, nzx = 0;  // products, targets with product terms, nz + 1 + ny
    int nchunks = 0;
    int nfemb = 0;
    int nd = 1;                  // densities (1 or 2)
    const T* cw2 = nullptr;      // record weights of density 2 (same order as crec)
    const double* cw2d = nullptr;  // the same in FP64 (FP32 kernels' accumulation recipe)
    double p1[2][2] = {{1, 1}, {1, 1}};  // per density: embedding prefactor, exponent
    double ecut = 0, decut = 1;
    double c1[2][32] = {{0}};    // per density: coefficients of B1_n = g^m_n(mu_i) - 1
};

// Error bits raised by kernels (reported by the host API).
enum : int {
    kErrSmallDistance = 1,   // r < rcut/nlut ("Encountered very small distance.")
    kErrMomentRange = 2,     // |m| outside [0, rcut_magnetic*(1+1/nlut)) (reference reads out of bounds)
    kErrTooManyNeighbors = 4,
};

struct Buffers {
    void* Z = nullptr;       // [natom][nz] complex, in the places of ZLayout::half
    void* W = nullptr;       // [natom][nz] complex, likewise
    double* ehc = nullptr;   // core sum
    double* rho1 = nullptr;  // B1 part of rho, [natom][nd]
    double* dE = nullptr;    // fcut * F'(rho), [natom][nd]
    double* edf = nullptr;   // d f_in/d e_hc * F + 1
    double* rho = nullptr;   // rho_i (including the B1 part), [natom][nd]
    void* Pt = nullptr;      // adjoint partial sums, [natom][nd][nslot] x 16 bytes (partials_bytes)
    void* Wd = nullptr;      // fitting with two densities: [natom][2][nz] per-density dRho/dZ (FP64),
                             // written by the adjoint when set
    int* err = nullptr;
    size_t cap_atoms = 0;
    bool forces = true;      // false: a fit's gradient is to follow, which needs Z and W only
};

// bytes of Buffers::Pt per atom
__host__ __device__ inline size_t partials_bytes(int nslot, int nd) { return (size_t)nslot * 16 * (size_t)nd; }

// tasks of a wave whose sums wait in registers (kNodeTasks of the plan)
constexpr int kNodeTasksDev = 2;
// steps of a task come in multiples of these: the sparse product's and the gradient's (NodePlan)
constexpr int kNodeQuantumDev = 4, kNodeQuantumGDev = 4;
// The node plan of the adjoint on the device (NodePlan; adjoint.hip).  nw = 0: there is none for this
// potential, and k_adjoint walks the gradient records.
template <typename T>
struct NodeTab {
    struct W4 {
        T v[4];
    };
    int nw = 0, slot_one = 0, first_node = 0, npair = 0, nslots = 0, na2 = 0, k2 = 0, nd = 0, kd = 0;
    const unsigned short* core_z = nullptr;
    const uint32_t* pair = nullptr;
    const int4* head = nullptr;    // [waves][64]
    const ushort4* row = nullptr;
    const uint2* col = nullptr;    // LDS slots of four steps of a lane
    const W4* w = nullptr;
    const uint32_t* g_row = nullptr;
    const uint2* g_rec = nullptr;  // two steps of a lane
    const unsigned short* a2_x = nullptr;
    const uint32_t* a2_c = nullptr;
    const T* a2_w = nullptr;
    const uint32_t* d_slot = nullptr;
    const int* d_x = nullptr;
    const T* d_w = nullptr;
};
// weights of a plan's records in both precisions, from the monomials' (t: monomial * 2 + (1: minus), -1: 0)
struct NodeWeights {
    int n = 0;
    const int* t = nullptr;
    double* w64 = nullptr;
    float* w32 = nullptr;
};
hipError_t fill_node_weights(const NodeWeights& n, const double* w, hipStream_t s);
// energies and the unscaled gradient dRho/dZ of the representatives (B.W; the entries between them are
// not written), from B.Z
template <typename T>
hipError_t run_adjoint_nodes(const DevParams<T>& P, const NodeTab<T>& N, int natom, const Buffers& B, double* eout,
                             hipStream_t s);

// atom_base: the index of the launch's first atom in the whole system (even), which fixes the
// adjoint's walk per atom, so that results do not depend on how the atoms are split into
// launches
// Density staging variants (Launch::run's dvar; -1 = the built-in rule): 0 = 32 neighbours per
// round, each pair's staging spread over 8 threads, no neighbour split of the A tasks; 1 = the
// same with the split (DevParams::sa); 2 = 64 neighbours per round, one thread per pair and
// side, with the split.
constexpr int kDensityVariants = 3;

template <typename T>
struct Launch {
    static hipError_t run(const DevParams<T>& P, const NodeTab<T>& N, int natom, int atom_base, const int* offsets,
                          const double* dlist, const double* elist, const double* dmomi,
                          const double* emomi, const double* dmom, const double* emom, double* eout,
                          double* flist, double* tlist, double* tlist0, Buffers& B, hipStream_t s,
                          int nm3_class, hipEvent_t* ev, int dvar = -1, bool acc = false);
};

// FitPlan on the device (fit.hip)
struct FitTab {
    int groups = 0, slots = 0, most = 0;  // most: tiles of a wave
    const int* head = nullptr;
    const unsigned short* entry = nullptr;
    const uint32_t *prod = nullptr, *node = nullptr, *place = nullptr;
    const int4* t = nullptr;
};
// M[d][t] += sum_i alpha_{i,d} Re P_{t,i} + beta_{i,d} Re D_u P_{t,i}
hipError_t fit_accumulate(const FitTab& F, int nz, int nterms, int nd, int natom, const void* Z, const void* Zdot,
                          const double* alpha, const double* beta, double* M, hipStream_t s);

// fitting (FP64): forward-mode density, per-atom adjoint scalars, monomial accumulation
struct FitBuffers {
    void* Zdot = nullptr;        // [natom][nz] complex
    double* ehc_dot = nullptr;   // [natom]
    double* alpha = nullptr;     // [natom][nd]
    double* beta = nullptr;      // [natom][nd]
    double* M = nullptr;         // [nd][nterms], real parts
    void* Wd = nullptr;          // [natom][2][nz] complex: per-density dRho/dZ (two densities)
    FitTab plan;                 // its arrays belong to the context
    int *ub_ptr = nullptr, *ub_t = nullptr;
    double* ub_u = nullptr;
    size_t cap_atoms = 0;
};
hipError_t fit_backward(const DevParams<double>& P, bool scaled, int natom, const int* off, const int* nlist,
                        const double* du, const double* dlist, const double* elist, const double* dmomi,
                        const double* dmom, const double* emom, const int* atom_struct, const double* gE,
                        Buffers& B, FitBuffers& F, int nterms, const int* nbo5, double* grad, hipStream_t s);
hipError_t fit_assemble(int natom, const int* off, const int* nlist, const double* flist, const double* eout,
                        const int* atom_struct, int nstruc, double* f, double* estruct, hipStream_t s);

// Z, e_hc and the B1 part of rho (density.hip)
template <typename T>
hipError_t run_density(const DevParams<T>& P, int natom, const int* off, const double* dlist, const double* elist,
                       const double* dmomi, const double* emomi, const double* dmom, const double* emom,
                       const Buffers& B, hipStream_t s);
// their derivative along the displacements du of the atoms (fitting)
hipError_t run_density_jvp(const DevParams<double>& P, int natom, const int* off, const int* nlist, const double* du,
                           const double* dlist, const double* elist, const double* dmom, const double* emom, void* Zdot,
                           double* ehc_dot, int* err, hipStream_t s);
// pair forces, pair torques and self torques from B.W; scaled: W holds dE/dZ, else dRho/dZ (forces.hip)
template <typename T>
hipError_t run_forces(const DevParams<T>& P, int natom, const int* off, const double* dlist, const double* elist,
                      const double* dmomi, const double* emomi, const double* dmom, const double* emom, const Buffers& B,
                      bool scaled, double* flist, double* tlist, double* tlist0, hipStream_t s);
hipError_t upload_legendre_constants();
hipError_t clear_flags(int* p, hipStream_t s);
// n >= 1 slots of 16 bytes between device memory and pinned host memory; with flag_out its copy of *flag, without it
// *flag is cleared
hipError_t copy_slots(const void* src, void* dst, size_t n, int* flag, int* flag_out, hipStream_t s);
int supported_nm3_class(int nm3, int nr2m, int nb_a, int l3a, int l2m, int nr3a);

}  // namespace magace
