// nodes.cpp -- the adjoint's evaluation plan: the monomials of rho as products of two nodes.
//
// rho = Re sum_t w_t A0 A A A (and A0 A A, A0 A2) is written as rho = Re sum_e w_e X_p X_q with
// p a product of an A0 entry and an A entry and q a product of two A entries (or one A entry for
// the three-factor monomials).  Then
//   G_p = sum_q w X_q,  G_q = sum_p w X_p            (a sparse matrix, real weights)
//   dRho/dZ[a] = sum over the nodes that hold a of G Z[other factor],
// which costs two real-by-complex products per monomial where differentiating each factor on its
// own costs four products of three: the lmax-6 header's 31 272 monomials need 59 884 weights and
// 3 398 pair products in place of 116 695 three-factor records.
#include <algorithm>
#include <cstdint>
#include <map>
#include <queue>
#include <unordered_map>

#include "magace.hpp"

namespace magace {

namespace {

using Pair = std::pair<int, int>;  // two Z indices, ascending

struct Conj {
    const std::vector<uint32_t>& fold;
    int one;
    int partner(int x) const { return x == one ? one : (int)(fold[x] & 0xffff); }
    int sign(int x) const { return x != one && (fold[x] >> 16 & 1) ? -1 : 1; }
};

Pair ordered(int a, int b) { return a < b ? Pair(a, b) : Pair(b, a); }

// Greedy cover: every item picks one of its options; options that cover most of what is left go
// first (`bonus` options, which exist anyway, before all others).
std::vector<int> cover(const std::vector<std::vector<int>>& options, int nopt, const std::vector<char>& bonus) {
    std::vector<std::vector<int>> by(nopt);
    for (size_t t = 0; t < options.size(); ++t)
        for (size_t k = 0; k < options[t].size(); ++k) {
            const int o = options[t][k];
            if (by[o].empty() || by[o].back() != (int)t) by[o].push_back((int)t);
        }
    std::vector<int> pick(options.size(), -1);
    const long big = (long)options.size() + 1;
    std::priority_queue<std::pair<long, int>> q;  // ties: the largest index
    for (int o = 0; o < nopt; ++o)
        if (!by[o].empty()) q.emplace((long)by[o].size() + (bonus[o] ? big : 0), o);
    while (!q.empty()) {
        const auto top = q.top();
        q.pop();
        const int o = top.second;
        long left = 0;
        for (int t : by[o]) left += pick[t] < 0;
        if (!left) continue;
        if (left + (bonus[o] ? big : 0) != top.first) {
            q.emplace(left + (bonus[o] ? big : 0), o);
            continue;
        }
        for (int t : by[o])
            if (pick[t] < 0) pick[t] = o;
    }
    return pick;
}

struct Entry {
    int col;  // LDS slot
    int t;    // monomial * 2 + (1 if the weight enters with a minus)
};
struct Row {
    int slot;                  // where G goes
    std::vector<Entry> e;
};

// rows -> blocks of up to G rows with as many common columns as possible
template <int G> struct BlockOf {
    std::array<int, G> slot;
    std::vector<int> col;
    std::vector<std::array<int, G>> t;  // monomial * 2 + minus, -1: none
};
using Block = BlockOf<4>;

template <int G> std::vector<BlockOf<G>> make_blocks(const std::vector<Row>& rows, int nslots) {
    const int n = (int)rows.size();
    std::vector<std::vector<int>> inv(nslots);
    for (int r = 0; r < n; ++r)
        for (const Entry& e : rows[r].e) inv[e.col].push_back(r);
    std::vector<int> order(n);
    for (int i = 0; i < n; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return rows[a].e.size() > rows[b].e.size(); });
    std::vector<char> used(n, 0);
    std::vector<int> common(n, 0), touched, at(nslots, -1);
    std::vector<BlockOf<G>> out;
    std::array<int, G> none;
    none.fill(-1);
    for (int seed : order) {
        if (used[seed]) continue;
        BlockOf<G> b;
        b.slot = none;
        std::vector<int> cols;
        int g = 0;
        auto take = [&](int r) {
            used[r] = 1;
            b.slot[g] = rows[r].slot;
            for (const Entry& e : rows[r].e) {
                if (at[e.col] < 0) {
                    at[e.col] = (int)cols.size();
                    cols.push_back(e.col);
                    b.t.push_back(none);
                    for (int k : inv[e.col])
                        if (!used[k]) {
                            if (common[k]++ == 0) touched.push_back(k);
                        }
                }
                b.t[at[e.col]][g] = e.t;
            }
            ++g;
        };
        take(seed);
        while (g < G) {
            int best = -1;
            double score = 0;
            for (int k : touched) {
                if (used[k]) continue;
                const double c = common[k], add = (double)rows[k].e.size() - c, miss = (double)cols.size() - c;
                const double s = c - add - 0.5 * miss;
                if (best < 0 || s > score || (s == score && k < best)) {
                    best = k;
                    score = s;
                }
            }
            if (best < 0) break;
            take(best);
        }
        for (int k : touched) common[k] = 0;
        touched.clear();
        for (int c : cols) at[c] = -1;
        b.col = std::move(cols);
        out.push_back(std::move(b));
    }
    return out;
}

int round_up(int n, int q) { return std::max(q, (n + q - 1) / q * q); }

struct Unit {  // a row (or block of rows) for the scheduler: len records on 2^s lanes
    int id, len, s, per;
};

// Splits every unit over 2^s lanes so that a lane holds at most `target` records, packs units of
// one split into wave tasks of 64 lanes and the tasks onto nw waves, the longest first.  Returns
// the load of the fullest wave; tasks[w] = the wave's tasks, each a list of unit ids.
struct Sched {
    std::vector<std::vector<std::vector<Unit>>> waves;
    double worst = 0;
    size_t most = 0;  // tasks of the wave that has most
};
Sched schedule(const std::vector<int>& len, int target, int nw, double c0, double c1, int quantum) {
    std::vector<Unit> u;
    for (size_t i = 0; i < len.size(); ++i) {
        int s = 0;
        while (s < 6 && ((len[i] + (1 << s) - 1) >> s) > target) ++s;
        u.push_back({(int)i, len[i], s, (len[i] + (1 << s) - 1) >> s});
    }
    std::stable_sort(u.begin(), u.end(), [](const Unit& a, const Unit& b) { return a.s != b.s ? a.s > b.s : a.per > b.per; });
    std::vector<std::pair<double, std::vector<Unit>>> tasks;
    for (size_t i = 0; i < u.size();) {
        const int s = u[i].s;
        std::vector<Unit> t;
        const int per = round_up(u[i].per, quantum);
        while (i < u.size() && u[i].s == s && (int)t.size() < (64 >> s)) t.push_back(u[i++]);
        tasks.emplace_back(c0 + 6.0 * s + c1 * per, std::move(t));
    }
    std::stable_sort(tasks.begin(), tasks.end(), [](const auto& a, const auto& b) { return a.first > b.first; });
    Sched S;
    S.waves.resize(nw);
    std::vector<double> load(nw, 0.0);
    for (auto& t : tasks) {
        int w = 0;
        for (int k = 1; k < nw; ++k)
            if (load[k] < load[w] || (load[k] == load[w] && S.waves[k].size() < S.waves[w].size())) w = k;
        load[w] += t.first;
        S.waves[w].push_back(std::move(t.second));
    }
    for (int w = 0; w < nw; ++w) {
        S.worst = std::max(S.worst, load[w]);
        S.most = std::max(S.most, S.waves[w].size());
    }
    return S;
}

Sched best_schedule(const std::vector<int>& len, int nw, double c0, double c1, int quantum, size_t most) {
    Sched best;
    bool have = false;
    for (int target : {2, 4, 6, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48, 64, 96, 128, 256, 512, 4096}) {
        Sched s = schedule(len, target, nw, c0, c1, quantum);
        if (s.most > most) continue;
        if (!have || s.worst < best.worst) {
            best = std::move(s);
            have = true;
        }
    }
    if (!have) best.waves.clear();
    return best;
}

// the 16-lane group of a 16-byte LDS read that a lane belongs to on gfx950 (two per half wave:
// quads of lanes whose number has an even, and an odd, count of set bits)
int lds_group(int lane) {
    const int q = (lane >> 2) & 7;
    return ((lane >> 5) << 1) | ((q ^ (q >> 1) ^ (q >> 2)) & 1);
}

// Order of the lanes' records over the steps of one task so that the slots that a 16-lane group
// reads in one step fall in distinct classes slot mod 16 (the banks of a 16-byte read); lanes that
// read one slot share it.  slots(i): the LDS slots that record i reads.
template <typename F>
void spread_banks(std::vector<std::vector<int>>& lanes, int steps, F&& slots) {
    std::vector<std::vector<int>> out(lanes.size());
    for (int k = 0; k < steps; ++k) {
        std::vector<int> seen[4][2];
        int load[4][2][16] = {};
        for (size_t L = 0; L < lanes.size(); ++L) {
            auto& rem = lanes[L];
            if (rem.empty()) continue;
            const int g = lds_group((int)L);
            int best = 0, cost = 1 << 30;
            for (size_t i = 0; i < rem.size() && cost > 0; ++i) {
                const auto sl = slots(rem[i]);
                int c = 0;
                for (int f = 0; f < 2; ++f)
                    if (sl[f] >= 0 && std::find(seen[g][f].begin(), seen[g][f].end(), sl[f]) == seen[g][f].end())
                        c += load[g][f][sl[f] & 15];
                if (c < cost) {
                    cost = c;
                    best = (int)i;
                }
            }
            const auto sl = slots(rem[best]);
            for (int f = 0; f < 2; ++f)
                if (sl[f] >= 0 && std::find(seen[g][f].begin(), seen[g][f].end(), sl[f]) == seen[g][f].end()) {
                    seen[g][f].push_back(sl[f]);
                    ++load[g][f][sl[f] & 15];
                }
            out[L].push_back(rem[best]);
            rem.erase(rem.begin() + best);
        }
    }
    lanes = std::move(out);
}

// one side of the sparse product as tasks of the waves
struct Side {
    std::vector<Block> blocks;
    Sched sc;
};
bool cut_side(const std::vector<Row>& rows, int nslots, int nw, size_t most, Side& S) {
    S.blocks = make_blocks<4>(rows, nslots);
    std::vector<int> len;
    for (const Block& b : S.blocks) len.push_back((int)b.col.size());
    S.sc = best_schedule(len, nw, 40.0, 22.0, kNodeQuantum, most);
    return !S.sc.waves.empty();
}

// appends a task's records to the plan's stream; its header
std::array<int32_t, 3> emit_task(NodePlan& N, const Side& S, const std::vector<Unit>& t) {
    const int s = t[0].s, steps = round_up(t[0].per, kNodeQuantum);
    const std::array<int32_t, 3> head{steps, s, (int32_t)(N.row.size() / 4)};
    for (int g = 0; g < (64 >> s); ++g)
        for (int r = 0; r < 4; ++r)
            N.row.push_back((uint16_t)(g < (int)t.size() && S.blocks[t[g].id].slot[r] >= 0 ? S.blocks[t[g].id].slot[r] : 0xffff));
    std::vector<std::vector<int>> lanes(64);
    std::vector<std::pair<const Block*, int>> recs;
    for (size_t g = 0; g < t.size(); ++g)
        for (int i = 0; i < t[g].len; ++i) {
            lanes[(g << s) + (i & ((1 << s) - 1))].push_back((int)recs.size());
            recs.emplace_back(&S.blocks[t[g].id], i);
        }
    spread_banks(lanes, steps, [&](int i) { return std::array<int, 2>{recs[i].first->col[recs[i].second], -1}; });
    for (int k = 0; k < steps; ++k)
        for (int L = 0; L < 64; ++L) {
            const bool have = k < (int)lanes[L].size();
            const auto* r = have ? &recs[lanes[L][k]] : nullptr;
            N.col.push_back((uint16_t)(have ? r->first->col[r->second] : N.slot_zero));
            for (int g = 0; g < 4; ++g) N.t.push_back(have ? r->first->t[r->second][g] : -1);
        }
    return head;
}

}  // namespace

NodePlan build_nodes(const ZLayout& z, const TermList& T, int entry_limit) {
    NodePlan N;
    const int one = z.nz;
    if (T.ny > 0 || T.nd != 1) return N;
    const Conj cj{T.fold, one};
    const size_t nt = T.nterms();
    if (nt == 0) return N;  // the atoms' own moments alone: nothing to plan, and no entry of Z
    struct Mono {
        int a0, f[3], n;  // factors past n: none
    };
    std::vector<Mono> mono(nt);
    for (size_t t = 0; t < nt; ++t) {
        Mono m{T.idx[4 * t], {one, one, one}, 0};
        for (int k = 1; k < 4; ++k)
            if (T.idx[4 * t + k] != one) m.f[m.n++] = T.idx[4 * t + k];
        const bool a2 = m.n == 1 && m.f[0] >= z.oA2 && m.f[0] < z.oA0;
        bool a = m.n >= 2;
        for (int k = 0; k < m.n && a; ++k) a = m.f[k] < z.oA2;
        if (!(a2 || a) || m.a0 < z.oA0) return N;  // not of the forms A0 A2, A0 A A, A0 A A A
        mono[t] = m;
    }
    // a monomial may be replaced by its conjugate, Re P = s Re P', which makes pairs coincide
    auto canon = [&](int a, int b) { return std::min(ordered(a, b), ordered(cj.partner(a), cj.partner(b))); };
    // q of the four-factor monomials: which two of the three A factors
    std::map<Pair, int> qid;
    std::vector<std::vector<int>> options;
    std::vector<int> item;
    std::vector<Pair> qpair;
    auto id_of = [](std::map<Pair, int>& m, std::vector<Pair>& v, Pair p) {
        auto it = m.emplace(p, (int)v.size());
        if (it.second) v.push_back(p);
        return it.first->second;
    };
    static const int rest3[3][3] = {{0, 1, 2}, {0, 2, 1}, {1, 2, 0}};
    for (size_t t = 0; t < nt; ++t)
        if (mono[t].n == 3) {
            std::vector<int> o;
            for (const auto& r : rest3) o.push_back(id_of(qid, qpair, canon(mono[t].f[r[0]], mono[t].f[r[1]])));
            options.push_back(o);
            item.push_back((int)t);
        }
    std::vector<int> pick = cover(options, (int)qpair.size(), std::vector<char>(qpair.size(), 0));
    // nodes in the order of their first use: p = (A0 entry, A entry), q = (A entry, A entry)
    std::map<Pair, int> pnode, qnode;
    std::vector<Pair> P, Q;
    struct Edge {
        int p, q, single, t;  // q < 0: the single A entry `single`; t = monomial * 2 + minus
    };
    std::vector<Edge> edges;
    for (size_t i = 0; i < item.size(); ++i) {
        const Mono& m = mono[item[i]];
        const Pair qp = qpair[pick[i]];
        for (const auto& r : rest3) {
            const int x = m.f[r[0]], y = m.f[r[1]];
            int c = m.a0, k = m.f[r[2]], minus = 0;
            if (canon(x, y) != qp) continue;
            if (ordered(x, y) != qp) {
                minus = cj.sign(c) * cj.sign(k) * cj.sign(x) * cj.sign(y) < 0;
                c = cj.partner(c);
                k = cj.partner(k);
            }
            edges.push_back({id_of(pnode, P, Pair(c, k)), id_of(qnode, Q, qp), -1, 2 * item[i] + minus});
            break;
        }
    }
    // three factors: p = (A0, one A entry), the other A entry stands alone
    std::map<Pair, int> oid;
    std::vector<Pair> opair;
    options.clear();
    item.clear();
    auto canon_p = [&](int c, int a) { return std::min(Pair(c, a), Pair(cj.partner(c), cj.partner(a))); };
    for (size_t t = 0; t < nt; ++t)
        if (mono[t].n == 2) {
            std::vector<int> o;
            for (int k = 0; k < 2; ++k) {
                // an orientation that exists already is taken as it is
                const Pair a(mono[t].a0, mono[t].f[k]), b(cj.partner(a.first), cj.partner(a.second));
                const Pair c = pnode.count(a) ? a : pnode.count(b) ? b : canon_p(a.first, a.second);
                o.push_back(id_of(oid, opair, c));
            }
            options.push_back(o);
            item.push_back((int)t);
        }
    std::vector<char> bonus(opair.size());
    for (size_t i = 0; i < opair.size(); ++i) bonus[i] = pnode.count(opair[i]) != 0;
    pick = cover(options, (int)opair.size(), bonus);
    std::map<int, Row> single;  // A entries that stand alone: their G passes through W in memory
    for (size_t i = 0; i < item.size(); ++i) {
        const Mono& m = mono[item[i]];
        const Pair pp = opair[pick[i]];
        for (int k = 0; k < 2; ++k) {
            int c = m.a0, a = m.f[k], b = m.f[1 - k], minus = 0;
            if (Pair(c, a) != pp) {
                if (Pair(cj.partner(c), cj.partner(a)) != pp) continue;
                minus = cj.sign(c) * cj.sign(a) * cj.sign(b) < 0;
                b = cj.partner(b);
            }
            single[b];
            edges.push_back({id_of(pnode, P, pp), -1, b, 2 * item[i] + minus});
            break;
        }
    }
    // where a single entry's sum waits: a representative's in its place in W, the others' behind the stored
    // entries (a row of W has room for all nz)
    std::map<int, int> wait;
    int behind = z.nh;
    for (auto& s : single) {
        wait[s.first] = T.fold[s.first] >> 17 & 1 ? z.half[s.first] : behind++;
        s.second.slot = kNodeSingle | wait[s.first];
    }
    if (behind > z.nz) return N;
    // core slots: the A and A0 entries that the plan reads, then 1 and 0
    std::vector<char> used(z.nz, 0);
    for (const Pair& p : P) used[p.first] = used[p.second] = 1;
    for (const Pair& p : Q) used[p.first] = used[p.second] = 1;
    for (const auto& s : single) used[s.first] = 1;
    for (const Mono& m : mono)
        if (m.n == 1) used[m.a0] = 1;
    std::vector<int> slot(z.nz + 1, -1);
    for (int x = 0; x < z.nz; ++x)
        if (used[x]) {
            slot[x] = (int)N.core_z.size();
            N.core_z.push_back(z.half[x]);
        }
    N.slot_one = (int)N.core_z.size();
    N.slot_zero = N.slot_one + 1;
    N.first_node = N.slot_one + 2;
    N.np = (int)P.size();
    N.nq = (int)Q.size();
    int next = N.first_node + N.np + N.nq;
    // A0 entries with two-factor monomials: sum_x w A2[x], one G slot each
    std::map<int, std::vector<std::pair<int, int>>> dcol;  // A0 entry -> (A2 entry, monomial)
    for (size_t t = 0; t < nt; ++t)
        if (mono[t].n == 1) dcol[mono[t].a0].emplace_back(mono[t].f[0], (int)t);
    std::map<int, int> dslot;
    for (const auto& d : dcol) {
        dslot[d.first] = next;
        N.d_slot.push_back((uint32_t)next++ | (uint32_t)slot[d.first] << 16);
        N.kd = std::max(N.kd, (int)(d.second.size() + 7) / 8);
    }
    // eight lanes an A0 entry, kd records a lane
    for (int k = 0; k < N.kd; ++k)
        for (const auto& d : dcol)
            for (size_t i = 8 * (size_t)k; i < 8 * (size_t)k + 8; ++i) {
                const bool have = i < d.second.size();
                N.d_x.push_back(z.half[have ? d.second[i].first : z.oA0]);
                N.d_t.push_back(have ? 2 * d.second[i].second : -1);
            }
    N.nslots = next;
    if (next > entry_limit || next > 0x3fff) return N;
    auto pslot = [&](int i) { return N.first_node + i; };
    auto qslot = [&](int i) { return N.first_node + N.np + i; };
    for (const Pair& p : P) N.pair.push_back((uint32_t)slot[p.first] | (uint32_t)slot[p.second] << 16);
    for (const Pair& p : Q) N.pair.push_back((uint32_t)slot[p.first] | (uint32_t)slot[p.second] << 16);
    // both sides of the sparse product
    std::vector<Row> prow(N.np), qrow(N.nq);
    for (int i = 0; i < N.np; ++i) prow[i].slot = pslot(i);
    for (int i = 0; i < N.nq; ++i) qrow[i].slot = qslot(i);
    for (const Edge& e : edges) {
        prow[e.p].e.push_back({e.q >= 0 ? qslot(e.q) : slot[e.single], e.t});
        (e.q >= 0 ? qrow[e.q] : single[e.single]).e.push_back({pslot(e.p), e.t});
    }
    for (const auto& s : single) qrow.push_back(s.second);
    // waves of a workgroup: a CU holds sixteen (128 registers a lane); four workgroups of four where their
    // slots fit in its LDS, else two of eight or one of sixteen.  Two waves a workgroup were faster for
    // many atoms of small plans and slower for few (lmax-4 header, two / four / eight waves: 27648 atoms
    // mixed 278 / 312 / 409 us, 2000 atoms 31 / 28 / 37 us, 128 atoms FP64 18.1 / 13.6 / 13.0 us), and
    // a plan per system size would make an atom's sums depend on the launch that it is in.
    const size_t lds = (size_t)next * 16 + kNodeLdsTail;
    const int fit = (int)(kNodeLdsMost / lds);
    N.nw = fit >= 4 ? 4 : fit >= 2 ? 8 : 16;
    Side ps, qs;
    while (!cut_side(prow, next, N.nw, kNodeTasks, ps)) {
        if (N.nw == 16) return N;
        N.nw *= 2;
    }
    if (!cut_side(qrow, next, N.nw, 1u << 20, qs)) return N;
    // per wave 64 headers of four words: its tasks p, q, gradient (steps, log2 of the lanes per block,
    // first row), then their numbers and the starts of its two record streams
    N.head.assign((size_t)N.nw * 256, 0);
    std::vector<int> nt_of(N.nw, 0);
    auto add_task = [&](int w, const std::array<int32_t, 3>& h) {
        if (nt_of[w] >= 62) return false;
        std::copy(h.begin(), h.end(), N.head.begin() + (size_t)w * 256 + 4 * nt_of[w]++);
        return true;
    };
    for (int w = 0; w < N.nw; ++w) {
        int32_t* tail = &N.head[(size_t)w * 256 + 4 * 62];
        tail[0] = (int32_t)ps.sc.waves[w].size();
        tail[1] = (int32_t)qs.sc.waves[w].size();
        tail[4] = (int32_t)(N.col.size() / 64);
        for (const auto& t : ps.sc.waves[w])
            if (!add_task(w, emit_task(N, ps, t))) return N;
        for (const auto& t : qs.sc.waves[w])
            if (!add_task(w, emit_task(N, qs, t))) return N;
    }
    // gradient of the representatives of conjugate pairs, W_x = g_x + s conj(g_xbar)
    // (TermList::fold), g_x = sum over the nodes that hold x of G Z[other], the single entry's G
    std::vector<std::vector<std::pair<int, int>>> g(z.nz);  // (G slot, slot of the other factor)
    for (int i = 0; i < N.np + N.nq; ++i) {
        const Pair& p = i < N.np ? P[i] : Q[i - N.np];
        g[p.first].emplace_back(N.first_node + i, slot[p.second]);
        g[p.second].emplace_back(N.first_node + i, slot[p.first]);
    }
    for (const auto& d : dslot) g[d.first].emplace_back(d.second, N.slot_one);
    std::vector<std::vector<uint32_t>> lists;
    std::vector<uint32_t> target;  // NodePlan::g_row
    for (int x = 0; x < z.nz; ++x) {
        if (x >= z.oA2 && x < z.oA0) continue;
        if (!z.stored[x]) continue;
        const bool rep = T.fold[x] >> 17 & 1;  // the others (m = 0, m' < 0) are written as zeros
        std::vector<uint32_t> l;
        if (rep)
            for (const auto& e : g[x]) l.push_back((uint32_t)e.first | (uint32_t)e.second << 16);
        if (rep && !(T.fold[x] >> 18 & 1)) {
            const int xb = cj.partner(x), s = cj.sign(x);
            // s conj(G Z): the real part times s, the imaginary part times -s
            for (const auto& e : g[xb])
                l.push_back((uint32_t)e.first | (uint32_t)e.second << 16 | (s < 0 ? 1u << 30 : 0u) | (s < 0 ? 0u : 1u << 31));
        }
        const int xb = cj.partner(x);
        uint32_t row = z.half[x];
        if (rep && single.count(x)) row |= kNodeOwn;
        if (rep && !(T.fold[x] >> 18 & 1) && single.count(xb))
            row |= kNodeConj | (uint32_t)wait[xb] << 12 | (cj.sign(x) < 0 ? kNodeMinus : 0u);
        lists.push_back(std::move(l));
        target.push_back(row);
    }
    std::vector<int> len;
    for (const auto& l : lists) len.push_back((int)l.size());
    const Sched sc = best_schedule(len, N.nw, 40.0, 34.0, kNodeQuantumG, 1u << 20);
    for (int w = 0; w < N.nw; ++w) {
        int32_t* tail = &N.head[(size_t)w * 256 + 4 * 62];
        tail[2] = (int32_t)sc.waves[w].size();
        tail[5] = (int32_t)(N.g_rec.size() / 64);
        for (const auto& t : sc.waves[w]) {
            const int s = t[0].s, steps = round_up(t[0].per, kNodeQuantumG);
            if (!add_task(w, {steps, s, (int32_t)N.g_row.size()})) return N;
            for (int k = 0; k < (64 >> s); ++k)
                N.g_row.push_back(k < (int)t.size() ? target[t[k].id] : kNodeNone);
            std::vector<std::vector<int>> lanes(64);
            std::vector<uint32_t> recs;
            for (size_t k = 0; k < t.size(); ++k)
                for (int i = 0; i < t[k].len; ++i) {
                    lanes[(k << s) + (i & ((1 << s) - 1))].push_back((int)recs.size());
                    recs.push_back(lists[t[k].id][i]);
                }
            spread_banks(lanes, steps, [&](int i) {
                const int zo = (int)(recs[i] >> 16 & 0x3fff);
                return std::array<int, 2>{(int)(recs[i] & 0x3fff), zo == N.slot_one ? -1 : zo};
            });
            for (int k = 0; k < steps; ++k)
                for (int L = 0; L < 64; ++L)
                    N.g_rec.push_back(k < (int)lanes[L].size() ? recs[lanes[L][k]]
                                                               : (uint32_t)N.slot_zero | (uint32_t)N.slot_one << 16);
        }
    }
    // the kernel reads ahead of the last task
    for (int k = 0; k < kNodeAhead * 64; ++k) {
        N.col.push_back((uint16_t)N.slot_zero);
        N.t.insert(N.t.end(), 4, -1);
        N.g_rec.push_back((uint32_t)N.slot_zero | (uint32_t)N.slot_one << 16);
    }
    // A2 entries: W_x = sum_c w A0[c] (plus the conjugate partner's, as above)
    std::vector<std::vector<std::pair<int, int>>> acol(z.nz);  // A2 entry -> (A0 entry, monomial)
    for (const auto& d : dcol)
        for (const auto& e : d.second) acol[e.first].emplace_back(d.first, e.second);
    std::vector<std::vector<std::pair<uint32_t, int>>> al;
    size_t k2 = 0;
    for (int x = z.oA2; x < z.oA0; ++x) {
        if (!z.stored[x]) continue;
        std::vector<std::pair<uint32_t, int>> l;
        for (const auto& e : acol[x]) l.emplace_back((uint32_t)slot[e.first], 2 * e.second);
        if (!(T.fold[x] >> 18 & 1)) {
            const int xb = cj.partner(x), s = cj.sign(x);
            for (const auto& e : acol[xb]) l.emplace_back((uint32_t)slot[e.first] | 1u << 31, 2 * e.second + (s < 0));
        }
        k2 = std::max(k2, l.size());
        al.push_back(std::move(l));
        N.a2_x.push_back(z.half[x]);
    }
    N.k2 = (int)k2;
    for (size_t k = 0; k < k2; ++k)
        for (const auto& l : al) {
            N.a2_c.push_back(k < l.size() ? l[k].first : (uint32_t)N.slot_zero);
            N.a2_t.push_back(k < l.size() ? l[k].second : -1);
        }
    N.ok = true;
    return N;
}

// The gradient in the coefficients is a sum over atoms of products X_p X_q of pair products, with p of an A0 entry and
// another factor and q of the other two.  Rows p that share columns q are taken sixteen at a time, and their
// columns sixteen at a time, so that a tile of 256 products is a matrix product over the atoms (FitPlan).
FitPlan build_fit_plan(const ZLayout& z, const TermList& T) {
    FitPlan F;
    const int one = z.nz;
    const Conj cj{T.fold, one};
    const size_t nt = T.nterms();
    auto product = [&](int x) { return x > one; };  // an entry Y, whose conjugate is not at hand
    auto partner = [&](Pair p) { return ordered(cj.partner(p.first), cj.partner(p.second)); };
    auto canon = [&](Pair p) { return product(p.first) || product(p.second) ? p : std::min(p, partner(p)); };
    auto id_of = [](std::map<Pair, int>& m, std::vector<Pair>& v, Pair p) {
        auto it = m.emplace(p, (int)v.size());
        if (it.second) v.push_back(p);
        return it.first->second;
    };
    // which two of the three factors behind A0 make q: monomials of three factors leave one alone
    static const int rest3[3][3] = {{0, 1, 2}, {0, 2, 1}, {1, 2, 0}};
    std::map<Pair, int> qid;
    std::vector<Pair> qpair;
    std::vector<std::vector<int>> options(nt);
    for (size_t t = 0; t < nt; ++t) {
        const uint16_t* f = &T.idx[4 * t + 1];
        for (const auto& r : rest3) {
            const Pair q = ordered(f[r[0]], f[r[1]]);
            if (q != Pair(one, one)) options[t].push_back(id_of(qid, qpair, canon(q)));
        }
    }
    const std::vector<int> pick = cover(options, (int)qpair.size(), std::vector<char>(qpair.size(), 0));
    std::map<Pair, int> pid;
    std::vector<Pair> P;
    std::vector<Row> rows;
    for (size_t t = 0; t < nt; ++t) {
        const uint16_t* f = &T.idx[4 * t + 1];
        for (const auto& r : rest3) {
            const int x = f[r[0]], y = f[r[1]];
            if (ordered(x, y) == Pair(one, one) || pick[t] != qid[canon(ordered(x, y))]) continue;
            int c = T.idx[4 * t], k = f[r[2]], minus = 0;
            // Re P = s Re P' of the conjugate monomial (an entry Y beside a pair that is not its own conjugate
            // keeps the monomial as it is: its q then has a column of its own)
            Pair q = ordered(x, y);
            if (q != canon(q) && !product(k)) {
                minus = cj.sign(c) * cj.sign(k) * cj.sign(x) * cj.sign(y) < 0;
                c = cj.partner(c);
                k = cj.partner(k);
                q = canon(q);
            }
            const int p = id_of(pid, P, Pair(c, k)), qi = id_of(qid, qpair, q);
            if (p == (int)rows.size()) rows.push_back({p, {}});
            rows[p].e.push_back({qi, (int)(2 * t) + minus});
            break;
        }
    }
    // two monomials never share both nodes
    const std::vector<BlockOf<16>> blocks = make_blocks<16>(rows, (int)qpair.size());
    struct Tile {
        const BlockOf<16>* b;
        size_t c0;
    };
    std::vector<Tile> tiles;
    for (const auto& b : blocks)
        for (size_t c = 0; c < b.col.size(); c += 16) tiles.push_back({&b, c});
    const size_t most = (size_t)kFitWaves * kFitTiles, want = std::max<size_t>(1, (tiles.size() + most - 1) / most);
    const size_t per = (tiles.size() + want - 1) / want;
    // a group of tiles with the entries and nodes that it needs
    for (size_t i = 0; i < tiles.size();) {
        std::map<int, int> entry;                  // Z entry -> slot; entries Y behind them
        std::vector<int> entries, prods;
        std::map<int, int> prow, pcol;             // node -> number
        std::vector<int> nrow, ncol;
        auto add_entry = [&](int x) {
            if (x == one || entry.count(x)) return;
            if (product(x)) {
                for (int k = 0; k < 2; ++k) {
                    const int a = T.ypair[2 * (x - one - 1) + k];
                    if (!entry.count(a)) entry[a] = 0, entries.push_back(a);
                }
                entry[x] = 0;
                prods.push_back(x);
            } else {
                entry[x] = 0;
                entries.push_back(x);
            }
        };
        const size_t i0 = i;
        while (i < tiles.size() && i - i0 < per) {
            const auto e0 = entry;
            const auto r0 = prow, c0 = pcol;
            const size_t ne = entries.size(), ny = prods.size(), nr = nrow.size(), nc = ncol.size();
            const Tile& t = tiles[i];
            for (int r : t.b->slot)
                if (r >= 0 && !prow.count(r)) {
                    prow[r] = (int)nrow.size();
                    nrow.push_back(r);
                    add_entry(P[r].first);
                    add_entry(P[r].second);
                }
            for (size_t c = t.c0; c < std::min(t.c0 + 16, t.b->col.size()); ++c) {
                const int q = t.b->col[c];
                if (pcol.count(q)) continue;
                pcol[q] = (int)ncol.size();
                ncol.push_back(q);
                add_entry(qpair[q].first);
                add_entry(qpair[q].second);
            }
            const int ge = (int)entries.size(), gy = (int)prods.size(), gn = (int)(nrow.size() + ncol.size());
            if (i > i0 && (ge > kFitEntries || gy > kFitProducts || gn > kFitNodes || ge + 1 + gy + gn > kFitSlots)) {
                entry = e0, prow = r0, pcol = c0;
                entries.resize(ne), prods.resize(ny), nrow.resize(nr), ncol.resize(nc);
                break;
            }
            ++i;
        }
        // in the order of their places, so that neighbouring lanes load neighbouring entries
        std::sort(entries.begin(), entries.end(), [&](int a, int b) {
            return std::make_pair(z.half[a] & 0xfff, a) < std::make_pair(z.half[b] & 0xfff, b);
        });
        for (size_t k = 0; k < entries.size(); ++k) entry[entries[k]] = (int)k;
        const int so = (int)entries.size();  // the slot of 1
        for (size_t k = 0; k < prods.size(); ++k) entry[prods[k]] = so + 1 + (int)k;
        entry[one] = so;
        const int n0 = so + 1 + (int)prods.size(), nn = (int)(nrow.size() + ncol.size());
        for (int v : {(int)F.entry.size(), so, (int)F.prod.size(), (int)prods.size(), (int)F.node.size(),
                      (int)nrow.size(), nn, (int)(F.place.size() / 64), (int)(i - i0)})
            F.head.push_back(v);
        F.head.resize(F.head.size() + kFitHead - 9, 0);
        for (int x : entries) F.entry.push_back(z.half[x]);
        auto slots = [&](Pair p) { return (uint32_t)entry[p.first] | (uint32_t)entry[p.second] << 16; };
        for (int x : prods) F.prod.push_back(slots({T.ypair[2 * (x - one - 1)], T.ypair[2 * (x - one - 1) + 1]}));
        for (int r : nrow) F.node.push_back(slots(P[r]));
        for (int q : ncol) F.node.push_back(slots(qpair[q]));
        for (size_t k = i0; k < i; ++k) {
            const Tile& t = tiles[k];
            auto row = [&](int r) { return t.b->slot[r]; };
            auto col = [&](int c) { return t.c0 + c < t.b->col.size() ? t.b->col[t.c0 + c] : -1; };
            for (int lane = 0; lane < 64; ++lane) {
                const int r = row(lane & 15), q = col(lane & 15);  // none: any node
                F.place.push_back((uint32_t)(n0 + (r < 0 ? 0 : prow[r])) |
                                  (uint32_t)(n0 + (int)nrow.size() + (q < 0 ? 0 : pcol[q])) << 16);
                for (int u = 0; u < 4; ++u)
                    F.t.push_back(q < 0 ? -1 : t.b->t[t.c0 + (lane & 15)][matrix_row(8, lane >> 4, u)]);
            }
        }
        F.slots = std::max(F.slots, n0 + nn);
        F.tiles = std::max(F.tiles, (int)(i - i0));
        ++F.groups;
    }
    return F;
}

}  // namespace magace
