// magace.hpp -- host-side model of a magnetic-ACE potential for the MI355X evaluator.
//
// Scope: the per-atom energy / force / magnetic-gradient path of libace
// (src/ace.F90:79-321 -> prepA, prepB, forceweights, forcecompute, torquecompute),
// single element, body order <= 6, ndensity 1 or 2.  The host side parses the potential file,
// enumerates the basis, builds Clebsch-Gordan couplings and FP64 spline tables, and
// compiles everything into flat tables the HIP kernels consume.
#pragma once

#include <array>
#include <cstdint>
#include <string>
#include <vector>

namespace magace {

// Potential-file header (src/util.F90:603-653).
struct Header {
    int nb_a = 0, nb_m = 0, nr2_m = 0, l2m = 0;   // "nradbase l2max"
    int nr3_a = 0, nr3_m = 0, l3a = 0, l3m = 0;   // "nradial3 l3max"
    int nr4_a = 0, nr4_m = 0, l4a = 0, l4m = 0;   // "nradial4 l4max"
    int nr5_a = 0, nr5_m = 0, l5a = 0, l5m = 0;
    int nr6_a = 0, nr6_m = 0, l6a = 0, l6m = 0;
    int ndensity = 1, npot = 0, nfemb = 0, radtype_a = 3, radtype_m = 7;
    double lambda_a = 0, lambda_m = 0, cut_a = 0, cut_m = 0, dcut_a = 0, dcut_m = 0;
    double ecut = 0, decut = 0;
};

// Enumerated basis: index tuples with the column meaning of b1index/b2index/b3index/b4index.
struct Basis {
    std::vector<std::array<int, 1>> b1;   // n0'
    std::vector<std::array<int, 4>> b2;   // n0' n1' n1 l
    std::vector<std::array<int, 9>> b3;   // n1 n2 n0' n1' n2' l1 l0' l1' l2'
    std::vector<std::array<int, 15>> b4;  // n1 n2 n3 n0'..n3' l1 l2 l3 l0'..l3' L01'
    // n1..n4 n0'..n4' l1..l4 l0'..l4' L12 L01' L23' (b5index)
    std::vector<std::array<int, 21>> b5;
    // n1..n5 n0'..n5' l1..l5 l0'..l5' L12 L34 L01' L23' L45' (b6index)
    std::vector<std::array<int, 27>> b6;
    // non-empty when the reference's enumeration pairs atomic and magnetic couplings of
    // different counts (it then fills the missing side with zero indices and reads outside
    // its arrays): the reason such a header is refused
    std::string undefined;
};

struct Potential {
    Header h;
    Basis basis;
    // expansion coefficients, one per B function and density: c[d * nvar + k]
    std::vector<double> c1, c2, c3, c4, c5, c6;
    std::vector<double> crad_a;          // [nr3_a][l3a+1][nb_a]
    std::vector<double> crad_m;          // [nr2_m][l2m+1][nb_m]
    double p1[2][2] = {{1.0, 1.0}, {1.0, 1.0}};  // per density: embedding prefactor, exponent
    double core[2] = {3.0, 3.0};         // core repulsion prefactor / exponent
    double rcut = 0, rcut_m = 0;         // global cutoffs from acelibini_
    std::string element = "Fe", xc = "pbe";
    double smear = 0.0;
    std::vector<std::string> header_lines;  // the 14 header lines as read
};

// Per-atom complex feature vector Z = [A | A2 | A0] (all m, m' stored).
// A covers the magnetic l' <= l3max_magnetic and nradial3_magnetic radial functions, as the
// reference's A does (src/a_basis.F90:61,248-251,346: entries of higher l' stay zero, so
// higher-order functions with such a factor vanish and are left out of the term list).
struct ZLayout {
    int lsa = 0, lsm = 0, lsm3 = 0;  // (l3a+1)^2, (l2m+1)^2, (lAm+1)^2
    int lAm = 0;                     // magnetic l' range of A (l3max_magnetic)
    int nm3 = 0;                     // nr3_m * lsm3 (magnetic columns of A)
    int oA = 0, oA2 = 0, oA0 = 0, nz = 0;
    int a(int n, int l, int m, int np, int lp, int mp) const {
        return oA + (n * lsa + l * l + l + m) * nm3 + np * lsm3 + lp * lp + lp + mp;
    }
    int a2(int n, int np, int lp, int mp) const { return oA2 + (n * nr2m_ + np) * lsm + lp * lp + lp + mp; }
    int a0(int np, int lp, int mp) const { return oA0 + np * lsm + lp * lp + lp + mp; }
    int nr2m_ = 0;
    // Z and W in device memory hold the entries of m >= 0 (A) and m' >= 0 (A2, A0) only, the others being
    // conjugates: [A: n][l, m >= 0][q] at 0, [A2: n][n'][l', m' >= 0] at hA2, [A0: n'][l', m' >= 0] at hA0, nh
    // in all.  half[x] of a full index: its place | real part negative << 14 | imaginary part negative
    // << 15 (an entry with `stored` has neither flag).
    int hA2 = 0, hA0 = 0, nh = 0;
    std::vector<uint16_t> half;
    std::vector<char> stored;
};

// rho = Re sum_t w_t prod_{s<4} Z[i_ts] with Z[nz] == 1 padding lower-degree terms.
// The gradient is stored transposed ("gather" form): for every target x of Z, the list of
// contributions w_t * prod_{s' != s} Z[i_ts'] of the monomials containing x, split into
// chunks of at most kChunk contributions.  rho = Re sum_{x in A0} Z[x] dRho/dZ[x], because
// every monomial has exactly one A0 factor.
struct TermList {
    static constexpr int kChunk = 32;
    static constexpr int kLanes = 512;  // threads per adjoint workgroup the chunk order is built for
    std::vector<uint16_t> idx;   // 4 per term (slot 0 = A0 factor)
    std::vector<double> w;       // merged weights, density-major: w[d * nterms + t]
    std::vector<uint16_t> cidx;  // 4 per contribution: the three other factors + padding
    std::vector<double> cw;      // weight per contribution, density-major (d * ncontrib + r)
    std::vector<int32_t> chunks; // 2 per chunk: first record, target | (count << 12) | (sole << 18)
                                 // | (slot << 19), count = the length of its group of 64 chunks
                                 // (padded with zero weights), sole = the target's only chunk,
                                 // slot = the partial-sum slot of its run (below); records of a
                                 // chunk are 64 apart (wave-interleaved layout)
    // Runs: chunk c runs on lane c % kLanes in round c / kLanes; a run is a maximal sequence of
    // a lane's chunks in consecutive rounds with one target.  The adjoint flushes one sum per
    // run: a sole chunk's sum is its target's gradient and is stored; the other runs store
    // their sums into slots, numbered so that a target's slots are consecutive.  Two passes
    // then add them up in a fixed order (the evaluation is bitwise repeatable): the first sums
    // groups of up to kGroup consecutive slots of a target (loads issued together) and writes
    // the result into the group's first slot, or straight into the gradient when the target has
    // one group; the second sums the group results of targets with several groups.
    // comb: 2 per group: first slot, target | (slots << 12) | (the target's only group << 16);
    // comb2: 2 per target with several groups: first slot, target | (groups << 12).
    static constexpr int kGroup = 8;
    std::vector<int32_t> comb, comb2;
    int nslot = 0;
    // folding of the gradient onto representatives of conjugate pairs (x, xbar):
    // partner | sign << 16 (1 = odd m+m') | representative << 17 | self-conjugate << 18 | stored << 19
    // (ZLayout::half); representatives are the stored entries, of A's m = 0 those of m' >= 0 only
    std::vector<uint32_t> fold;
    // Products of two A entries for monomials of five or six factors (body orders 5 and 6):
    // entry i is Y_i = Z[a] Z[b] at index nz + 1 + i of the extended vector Z' = [Z | 1 | Y],
    // so that every monomial has at most four factors of Z' (a five-factor monomial
    // z0 z1 z2 z3 z4 is z0 z1 z2 Y(z3 z4), a six-factor one z0 z1 Y(z2 z3) Y(z4 z5)).
    // ypair: 2 per entry (a, b).  The gradient of a Y entry goes back to its factors after the
    // record walk: yft holds 2 per Z target with such terms (first entry, target | count << 12),
    // yfe 2 per term (Z' index of Y, the other factor): dRho/dZ[x] += dRho/dY Z[other].
    int ny = 0;
    std::vector<int32_t> ypair, yft, yfe;
    int nzx() const { return nzx_; }
    int nzx_ = 0;                // nz + 1 + ny
    // coefficient structure: B function k (orders 2..6 in file order) -> monomials,
    // rho = sum_k c_k B_k with B_k = Re sum_t u_{k,t} prod Z[idx_t]; CSR by k and by t
    std::vector<int32_t> ub_ptr, ub_t;
    std::vector<double> ub_u;
    std::vector<int32_t> ut_ptr, ut_k;
    std::vector<double> ut_u;
    std::vector<int32_t> rec_t;  // monomial of each gradient record (-1: padding)
    int n2 = 0, n3 = 0, n4 = 0, n5 = 0, n6 = 0;  // raw (before merging) m-combination counts per order
    int raw = 0;
    int nd = 1;                  // densities
    size_t nterms() const { return idx.size() / 4; }
    size_t ncontrib() const { return rec_t.size(); }
};

// The adjoint's plan (nodes.cpp): the monomials as products of two nodes, p = A0 entry times A
// entry and q = product of two A entries or one A entry, rho = Re sum w X_p X_q.  A workgroup keeps
// the entries it needs in LDS slots: the core [the A and A0 entries in use | 1 | 0], the pair
// products [p | q] and the sums over A2 entries.  The work is cut into tasks of one wave each,
// assigned to the waves of a workgroup at build time (head); records are stored step by step,
// 64 lanes after one another.
constexpr size_t kNodeLdsTail = 384;          // sums and scalars behind the slots
constexpr size_t kNodeLdsMost = 160 * 1024;
constexpr int kNodeSingle = 0x4000;           // NodePlan::row: a single entry, its place in the row of W below
constexpr uint32_t kNodeOwn = 1u << 24, kNodeConj = 1u << 25, kNodeMinus = 1u << 26, kNodeNone = 1u << 31;
constexpr int kNodeQuantum = 4, kNodeQuantumG = 4;  // a task's steps are a multiple of these (product, gradient)
constexpr int kNodeAhead = 16;                // steps that the kernel reads ahead
constexpr int kNodeTasks = 2;                 // p tasks of a wave at most (their sums wait in registers)
struct NodePlan {
    bool ok = false;
    int nw = 8;                      // waves of a workgroup
    int slot_one = 0, slot_zero = 0, first_node = 0, np = 0, nq = 0, nslots = 0;
    std::vector<uint16_t> core_z;    // Z entry of core slot i (ZLayout::half)
    std::vector<uint32_t> pair;      // nodes: slots of the two factors
    // [waves][64][4]: headers of a wave's tasks (steps, multiples of four; log2 of the lanes per block; first row), p
    // tasks, then q tasks, then gradient tasks; entry 62: their numbers, entry 63: first steps of the
    // wave's two record streams, which run through its tasks in order
    std::vector<int32_t> head;
    // G_p = sum w X_q, G_q (and single entries) = sum w X_p
    std::vector<uint16_t> row;       // 4 per block: LDS slots of its rows, kNodeSingle | place in W, or 0xffff: none
    std::vector<uint16_t> col;       // per step and lane: LDS slot of the column's entry
    std::vector<int32_t> t;          // 4 per step and lane: monomial * 2 + (1: minus), -1: weight 0
    // gradient of the representatives: per step and lane G slot | slot of the other factor << 16 | real
    // part negative << 30 | imaginary part negative << 31; rows: place in W | place of the conjugate
    // partner's single G << 12 | kNodeOwn (the entry's own single G, which waits in its place, is added),
    // kNodeConj (the partner's, conjugated, with kNodeMinus negated)
    std::vector<uint32_t> g_row;
    std::vector<uint32_t> g_rec;
    // two-factor monomials A0 A2: per A2 representative k2 records (A0 slot | conjugate << 31), one
    // array after another; per A0 entry its A2 entries
    int k2 = 0;
    std::vector<uint16_t> a2_x;
    std::vector<uint32_t> a2_c;
    std::vector<int32_t> a2_t;
    std::vector<uint32_t> d_slot;    // G slot | slot of the A0 entry << 16
    int kd = 0;
    std::vector<int32_t> d_x, d_t;   // [kd][A0 entries][8]: A2 entry (ZLayout::half), monomial * 2 or -1
};

// The plan of the gradient in the coefficients (nodes.cpp, fit.hip): tiles of 16 pair products p (A0 entry times another
// factor) by 16 pair products q, in groups that a workgroup has in LDS slots [entries of Z | 1 | products Y | p | q].
constexpr int kFitWaves = 8, kFitTiles = 6;  // waves of a workgroup, tiles of a wave at most
constexpr int kFitSlots = 2400;              // slots of a group (32 bytes each) unless one tile needs more
constexpr int kFitEntries = 1024, kFitNodes = 1024, kFitProducts = 512;  // of a group at most (two, two and one a thread)
constexpr int kFitHead = 12;
struct FitPlan {
    int groups = 0, slots = 0, tiles = 0;  // slots and tiles: of the largest group
    // [groups][kFitHead]: first and number of the group's entries, of its products Y, first of its nodes, number of
    // nodes p, of all nodes, first and number of its tiles
    std::vector<int32_t> head;
    std::vector<uint16_t> entry;   // ZLayout::half
    std::vector<uint32_t> prod, node;  // slots of the two factors
    std::vector<uint32_t> place;   // [tiles][64]: slots of node p and node q of row and column lane % 16
    std::vector<int32_t> t;        // [tiles][64][4]: monomial * 2 + (1: minus) of a lane's results, -1: none
};

// Spline tables in node-major layout: row n holds [4 coeffs] for every function family.
struct Splines {
    int nlut = 10000;                    // src/radial.F90:43
    int nfa = 0, nfm = 0;                // functions per atomic / magnetic row
    int atomic_stride = 0, magnetic_stride = 0;  // doubles per row
    double rs_a = 0, rs_m = 0;           // nlut / cutoff
    // atomic row: [g_1..g_nb_a | R_{l,n} (l major, n minor) | core], each 4 coefficients
    std::vector<double> atomic;
    // magnetic row: [g^m_1..g^m_nb_m | M_{l',n'} (l' major)], each 4 coefficients
    std::vector<double> magnetic;
};

// The atomic radial functions R_{l,n} = sum_k C_{nlk} g_k as sums over at most nb_a factors h, R_{l,n} = sum_f U_{nlf}
// h_f.  The C of a fitted potential cancel (sum |C g| is 21 times |R| in the example
// potential, hundreds of times in a fit to narrow functions), so that g and C rounded to 32 bits lose what the sum in 64
// bits behind a table of R keeps.  Where there are no more R than g the factors are the R themselves, in FP64
// too, whose results then are those of the table of R (example potential, pair forces: 5e-15 from the reference and 5e-12
// through g, which is what the reference's rounded table differs from its own g by).  Otherwise, in FP32, U
// has orthonormal columns over the R, each scaled by its size (a QR decomposition of C), so that no term of
// the sum is larger than the R together.  Relative rms errors of R in 32 bits (U and h rounded, sum in FP32):
// table of R 3.6e-8; through g, random C 1.1e-7 to 2.0e-7, fits 1.2e-5 to 4.5e-5; through h 0.8e-7 to 0.9e-7 for
// either.
//
// The factors stand beside the g, which A2 needs, and their lookups take 2 to 5% of an evaluation.  With more R than g
// they are left out (nf = 0: the factors are the g) while the root mean square over the R of |terms C g| / |R| is at
// most kFactorLine.  Errors of energies, forces, torques and self torques against 64 bits, 128 atoms, table of R /
// through g / factors in 1e-7: lmax 4 at 2.4 2.3 2.5 2.9 2.3 / 2.0 2.2 2.2 1.8 / 2.0 2.3 2.2 2.1, at 4.3 3.1 2.5 2.6
// 3.3 / 3.2 3.3 2.6 3.6 / 2.0 2.2 2.0 2.2; lmax 6 at 3.0 14.9 7.5 6.7 11.4 / 10.7 6.7 5.3 9.3 / 9.5 6.7 5.4 8.6, at 4.2
// 4.1 4.1 3.6 4.4 / 3.8 4.5 3.1 4.2 / 2.4 3.7 2.7 3.0; a fit to narrow functions at lmax 6, 2.8 6.4 7.1 3.1 / 350 310
// 360 320 / 2.3 5.3 5.7 2.3.  With no more R than g they always pay: example potential's shape at 2.8, 1.8 4.4 4.0 6.8 /
// 2.1 7.9 7.3 16.9 / 0.9 1.8 1.6 1.8.
constexpr double kFactorLine = 3.0;
struct RadialFactors {
    int nf = 0;
    bool own = false;           // the factors are the R themselves
    std::vector<double> u;      // [nr3_a][l3a + 1][nf]
    std::vector<double> table;  // [nlut][nf][4], as Splines::atomic
};

struct Model {
    Potential pot;
    ZLayout z;
    TermList terms;
    NodePlan nodes;
    Splines spl;
    RadialFactors factors;
};

// api.cpp: the library's last-error state (magace_last_error / magace_error_string)
void report_error(int code, const std::string& msg);
void reset_error();
// api.cpp: a counter that changes whenever state baked into a captured evaluation changes
// (a new or finalised potential, reallocated per-atom buffers, the precision mode, new
// coefficients); a graph captured at one value must not be replayed at another
unsigned long long context_generation();
// api.cpp: uploads the potential's tables and sizes the per-atom buffers for natom atoms
// (no evaluation), so that a following capture records no allocation; MAGACE_ERR_STATE
// without a potential
int context_prepare(int natom);
// noalloc.hip: the fixed device scratch of magace_compute_device_noalloc
int scratch_setup();                 // looks up the scratch address on the current device
void* scratch_device_ptr(int dev);   // nullptr until scratch_setup ran on that device
size_t scratch_bytes();
// potential.cpp
bool parse_potential(const std::string& path, const std::string& element, int xc, double smear,
                     Potential& pot, std::string& err);
// writes the potential with its current parameters in the file format it was read from
// (record order of src/util.F90:1110-1362: par, core, rad_atomic, rad_magnetic, clu 1..4)
bool write_potential(const std::string& path, const Potential& pot, std::string& err);
// basis.cpp
bool check_header(const Header& h, std::string& err);
Basis enumerate_basis(const Header& h);
double clebsch_gordan(int j1, int j2, int J, int m1, int m2, int M);
ZLayout make_layout(const Header& h);
TermList build_terms(const Potential& pot, const ZLayout& z);
// nodes.cpp: the adjoint's plan; not ok for monomials of other forms (body orders 5, 6), two densities,
// or more than entry_limit LDS slots
NodePlan build_nodes(const ZLayout& z, const TermList& T, int entry_limit);
FitPlan build_fit_plan(const ZLayout& z, const TermList& T);
// row of a 16x16x4 product's result in register r of lane group g, by the size of a value (matrix.hpp)
inline int matrix_row(size_t bytes, int g, int r) { return bytes == 4 ? 4 * g + r : g + 4 * r; }
// splines.cpp
void radial_basis(int radtype, double lambda, int nb, double cut, double dcut, double r,
                  double* g, double* dg);
void core_repulsion(double r, double pre, double lambda, double cut, double& cr, double& dcr);
Splines build_splines(const Potential& pot);
RadialFactors radial_factors(const Potential& pot, const Splines& S);

}  // namespace magace
