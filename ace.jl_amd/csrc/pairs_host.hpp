// Host-side (CPU) compiler of the pair programs: the site energy of an
// Invariant basis as a quadratic form in the products of two pooled values,
// for the kernel k_pairs (ace_pairs.hip).
//
// Monomials of more than four factors (correlation order 5 to 7) are first
// brought to four: products of two pooled values that occur in many of them
// become values of their own, rows behind the pooled ones (greedily, the product
// that shortens most monomials next; order 5 of degree 10: 38 rows for 7,128
// monomials of five factors).  G of such a row u = X_s X_t is passed on in the
// end: G[s] += G_u X_t, G[t] += G_u X_s.
//
// Every monomial of the energy polynomial E = c0 + Re sum c prod X_f (X_f =
// A+[k] or its conjugate; the reference's sum over AA functions,
// evaluator.jl:121-147, mirror images merged) is split into two halves, p and
// q, of at most two factors; absent factors are the constant 1, a row of its
// own behind the pooled values.  Halves are kept up to conjugation with total
// m >= 0, so a monomial is Re(x_p conj(x_q)) for m > 0.  The split with the
// largest |m| is taken: the halves of m = 0 are then products of two real
// values (a monomial with any m != 0 factor has a split with |m| > 0), and one
// real coefficient serves the real and the imaginary part alike:
//   E = c0 + sum_{p, q} C_pq (re_p re_q + im_p im_q).
// Its derivative h_p = sum_q S_pq x_q (S = C + C^T) costs each monomial one
// multiply-add per half, and gives every G[k] at once: x_p = X_a X_d, so h_p
// X_d adds to G[a] and h_p X_a to G[d]; the energy is half of sum_p h_p . x_p.
//
// Rows p of equal (m, parity of l) are packed into panels of up to 8 whose
// columns q overlap; a panel's columns are records that share one factor.  The
// panels are scheduled in rounds, one panel per wave.  The waves of a round
// add to G in turns (sub-phases), such that the panels of one turn have no
// target in common: G is summed in a fixed order, by LDS additions of one wave at a
// time per target.
#pragma once

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <unordered_map>
#include <vector>

#include "pack_host.hpp"

namespace acehost {

constexpr int PAIR_ROWS = 8;     // rows per panel
constexpr int PAIR_WAVES = 16;   // waves per workgroup
constexpr int PAIR_SEQ = 1 + PAIR_WAVES;  // words of a round: turns, panels [wave]
constexpr int PAIR_HDR = 4 + 2 * PAIR_ROWS;  // header words of a panel (the fourth is not used)
constexpr int PAIR_MAXP = 8;     // workgroups a tile's rounds can be split over (and one more for tail tiles)
// Words of a record of nq columns: the shared factor, nq factors.
constexpr int pair_rec_words(int nq) { return 1 + nq; }
// Vector instructions of a record: the shared factor and its sign, per column
// two addresses, two products and 8 multiply-adds.
constexpr int pair_rec_cost(int nq) { return 6 + 12 * nq; }

constexpr uint32_t PAIR_BACK_IN = 1, PAIR_BACK_OUT = 2;

// One mode's program.  Panel words: [records of 4 | of 2 << 10 | of 1 << 20
// columns, rows | turn << 8, first coefficient, 0], then per
// row the LDS offsets of its two factors (bit 0 of the second: the second
// factor is conjugated), then the records: LDS offset of the shared factor (bit 0:
// conjugated), the offsets of the other factors.  Coefficients of a panel's
// records in the same order: [column][row].
struct PairProgram {
    std::vector<uint32_t> words;
    std::vector<double> coef;
    std::vector<int32_t> panel;  // [round][wave] first word of the panel, -1: none
    std::vector<int32_t> turns;  // [round] sub-phases in which the panels add to G
    std::vector<double> cost;    // [round] clocks of a workgroup, estimated
    // term c[leaf] * scale of coef[at]
    struct Term {
        uint32_t at;
        int32_t leaf;
        float scale;
    };
    std::vector<Term> terms;
    // products of their own: [row] LDS offsets of the two factors (bit 0 of the
    // second: conjugated); and per pooled value k those it is a factor of:
    // back_ptr[npool + 1], then [offset of the product's row, offset of the
    // other factor | PAIR_BACK_IN: conjugated | PAIR_BACK_OUT: the sum is]
    std::vector<uint32_t> virt, back;
    std::vector<int32_t> back_ptr;
    // the rounds of each of P workgroups: at seq_ptr[P][part] their count, then
    // the rounds (PAIR_SEQ words each), one unused round behind the last
    std::vector<int32_t> seq_ptr[PAIR_MAXP + 2], seq[PAIR_MAXP + 2];
    std::vector<double> part_cost;  // [P] the longest part's cost
    int nrounds() const { return (int)turns.size(); }
};

// The monomials of the energy polynomial: factors (device ids) and leaf index.
struct PairMono {
    int n;
    uint16_t f[7];
    int32_t leaf;
};

// The split of every monomial into two halves, as rows of a sparse symmetric
// matrix per class (m, parity of l).
struct PairForm {
    struct Half {
        uint16_t a, d;  // x = A[a] * (conj ? conj(A[d]) : A[d]); ONE = npool, rows of virt behind it
        bool conj;
    };
    struct Entry {
        int32_t p, q, leaf;
    };
    std::vector<Half> virt;    // products that are values of their own
    std::vector<Half> halves;
    std::vector<int> cls;      // class of every half
    std::vector<Entry> entries;
    int ncls = 0;
};

// max_rows: pooled values and products of their own that the kernel has room for.
inline std::string pair_form(const PackCopy& pc, const std::vector<int32_t>& pool, int max_rows, PairForm& out) {
    const int npool = (int)pool.size() / 4, ONE = npool;
    out = PairForm();
    // |m|, degree and parity of l of every row
    std::vector<int> rm, rdeg, rpar;
    for (int k = 0; k < npool; ++k) {
        rm.push_back(pool[4 * (size_t)k + 3]);
        rdeg.push_back(pool[4 * (size_t)k + 1] - 1 + pool[4 * (size_t)k + 2]);
        rpar.push_back(pool[4 * (size_t)k + 2] & 1);
    }
    rm.push_back(0);
    rdeg.push_back(0);
    rpar.push_back(0);
    auto m_of = [&](uint32_t f) { return (f & 0x8000) ? -rm[f & 0x7fff] : rm[f & 0x7fff]; };
    auto deg = [&](uint32_t f) { return rdeg[f & 0x7fff]; };
    auto par = [&](uint32_t f) { return rpar[f & 0x7fff]; };
    auto cj = [&](uint32_t f) { return m_of(f) == 0 ? f & 0x7fffu : f ^ 0x8000u; };
    // a product up to conjugation, m >= 0, the conjugated factor (if any) second
    auto half_key = [&](uint32_t f, uint32_t g) -> uint32_t {
        if (m_of(f) + m_of(g) < 0) {
            f = cj(f);
            g = cj(g);
        }
        const bool fc = (f & 0x8000) != 0, gc = (g & 0x8000) != 0;
        if ((fc && !gc) || (fc == gc && f > g)) std::swap(f, g);
        return f << 16 | g;
    };
    // one real coefficient serves both parts: not for m = 0 products of complex factors
    auto usable = [&](uint32_t f, uint32_t g) { return m_of(f) + m_of(g) != 0 || (m_of(f) == 0 && m_of(g) == 0); };
    std::vector<PairMono> monos;
    for (int t = 0; t < pc.ntasks; ++t) {
        if (pc.tasks[5 * (size_t)t + 2] >= 0) continue;  // gradient tasks
        if (pc.task_term_ptr[t + 1] != pc.task_term_ptr[t]) return "energy task with constant terms";
        for (int r = pc.tasks[5 * (size_t)t]; r < pc.tasks[5 * (size_t)t + 1]; ++r) {
            const int32_t* run = pc.runs.data() + (size_t)ACE_RUN_W * r;
            if (run[0] > 6) return "correlation order above 7";  // the last two of 8 factors may be X and its conjugate
            for (int i = 0; i < run[2]; ++i) {
                PairMono m;
                m.n = run[0] + 1;
                for (int q = 0; q < run[0]; ++q) m.f[q] = (uint16_t)run[4 + q];
                m.f[run[0]] = (uint16_t)pc.leaf_fid[(size_t)run[3] + i];
                m.leaf = run[3] + i;
                monos.push_back(m);
            }
        }
    }
    // products of their own until no monomial has more than four factors
    for (;;) {
        std::unordered_map<uint32_t, int> count;
        for (const PairMono& m : monos) {
            if (m.n <= 4) continue;
            uint32_t seen[21];
            int ns = 0;
            for (int i = 0; i < m.n; ++i)
                for (int j = i + 1; j < m.n; ++j) {
                    if ((m.f[i] & 0x7fff) > ONE || (m.f[j] & 0x7fff) > ONE || !usable(m.f[i], m.f[j])) continue;
                    const uint32_t k = half_key(m.f[i], m.f[j]);
                    if (std::find(seen, seen + ns, k) == seen + ns) seen[ns++] = k;
                }
            if (ns == 0) return "monomial without a product to replace";
            for (int i = 0; i < ns; ++i) ++count[seen[i]];
        }
        if (count.empty()) break;
        if (npool + (int)out.virt.size() >= max_rows) return "too many products";
        uint32_t key = 0;
        int most = 0;
        for (const auto& kv : count)
            if (kv.second > most || (kv.second == most && kv.first < key)) {
                key = kv.first;
                most = kv.second;
            }
        const uint32_t f = key >> 16, g = key & 0xffffu, u = (uint32_t)rm.size();
        out.virt.push_back({(uint16_t)(f & 0x7fff), (uint16_t)(g & 0x7fff), (g & 0x8000) != 0});
        rm.push_back(m_of(f) + m_of(g));
        rdeg.push_back(deg(f) + deg(g));
        rpar.push_back((par(f) + par(g)) & 1);
        for (PairMono& m : monos)
            for (int i = 0; i < m.n && m.n > 4; ++i)
                for (int j = i + 1; j < m.n && m.n > 4; ++j) {
                    const uint32_t a = m.f[i], b = m.f[j];
                    if ((int)(a & 0x7fff) > ONE || (int)(b & 0x7fff) > ONE || !usable(a, b) || half_key(a, b) != key) continue;
                    m.f[i] = (uint16_t)(m_of(a) + m_of(b) < 0 ? u | 0x8000u : u);
                    m.f[j] = m.f[m.n - 1];
                    --m.n;
                    j = i;  // the rest against the new factor: it is passed over
                }
    }
    for (PairMono& m : monos)
        for (int q = m.n; q < 4; ++q) m.f[q] = (uint16_t)ONE;
    std::unordered_map<uint32_t, int32_t> ids;
    std::map<std::pair<int, int>, int> classes;
    auto half = [&](uint32_t f, uint32_t g) -> int32_t {
        const int M = std::abs(m_of(f) + m_of(g));
        if (!usable(f, g)) return -1;
        const uint32_t key = half_key(f, g);
        f = key >> 16;
        g = key & 0xffffu;
        auto it = ids.find(key);
        if (it != ids.end()) return it->second;
        const std::pair<int, int> c(M, (par(f) + par(g)) & 1);
        const int ci = classes.emplace(c, (int)classes.size()).first->second;
        const int32_t id = (int32_t)out.halves.size();
        out.halves.push_back({(uint16_t)(f & 0x7fff), (uint16_t)(g & 0x7fff), (g & 0x8000) != 0});
        out.cls.push_back(ci);
        ids.emplace(key, id);
        return id;
    };
    for (const PairMono& m : monos) {
        // the three splits of four factors; shorter monomials are padded with
        // the constant and keep one factor per half where they can
        // (largest |m|, then halves of equal degree, then the smallest factors,
        // so that the same halves recur)
        uint32_t ha[2] = {0, 0}, hb[2] = {0, 0};
        std::tuple<int, int, uint32_t, uint32_t> best;
        const int nsplit = m.n <= 2 ? 1 : 3;
        for (int s = 0; s < nsplit; ++s) {
            // n <= 2: (f0, 1)(f1, 1); n = 3: one factor alone, two together
            uint32_t a[2], b[2];
            if (m.n <= 2) {
                a[0] = m.f[0], a[1] = ONE, b[0] = m.f[1], b[1] = ONE;
            } else if (m.n == 3) {
                a[0] = m.f[s], a[1] = ONE, b[0] = m.f[(s + 1) % 3], b[1] = m.f[(s + 2) % 3];
            } else {
                a[0] = m.f[0], a[1] = m.f[1 + s], b[0] = m.f[1 + (s + 1) % 3], b[1] = m.f[1 + (s + 2) % 3];
            }
            const int M = std::abs(m_of(a[0]) + m_of(a[1]));
            const int dd = m.n == 3 ? 0 : std::abs(deg(a[0]) + deg(a[1]) - deg(b[0]) - deg(b[1]));
            const uint32_t ka = half_key(a[0], a[1]), kb = half_key(b[0], b[1]);
            const std::tuple<int, int, uint32_t, uint32_t> k(-M, dd, std::min(ka, kb), std::max(ka, kb));
            if (s == 0 || k < best) {
                best = k;
                std::copy(a, a + 2, ha);
                std::copy(b, b + 2, hb);
            }
        }
        const int32_t p = half(ha[0], ha[1]), q = half(hb[0], hb[1]);
        if (p < 0 || q < 0 || out.cls[(size_t)p] != out.cls[(size_t)q]) return "monomial without a pair split";
        out.entries.push_back({p, q, m.leaf});
    }
    out.ncls = (int)classes.size();
    return "";
}

// The program of one mode: forces (symmetric rows, G and energy) or energy
// only (every monomial in one row; no turns).  row_bytes: LDS bytes between
// pooled values.  cap: columns per panel above which it is cut.
inline std::string pair_program(const PairForm& pf, bool forces, int row_bytes, int npool, int cap, PairProgram& out) {
    out = PairProgram();
    const int nh = (int)pf.halves.size();
    {
        std::vector<std::vector<uint32_t>> back((size_t)npool);
        for (size_t i = 0; i < pf.virt.size(); ++i) {
            const PairForm::Half& v = pf.virt[i];
            const uint32_t u = ((uint32_t)npool + 1 + (uint32_t)i) * row_bytes, oa = (uint32_t)v.a * row_bytes,
                           od = (uint32_t)v.d * row_bytes;
            out.virt.push_back(oa);
            out.virt.push_back(od | (v.conj ? 1u : 0u));
            back[v.a].push_back(u);
            back[v.a].push_back(od | (v.conj ? PAIR_BACK_IN : 0u));
            back[v.d].push_back(u);
            back[v.d].push_back(oa | (v.conj ? PAIR_BACK_OUT : 0u));
        }
        out.back_ptr.push_back(0);
        for (const auto& b : back) {
            out.back.insert(out.back.end(), b.begin(), b.end());
            out.back_ptr.push_back((int32_t)out.back.size() / 2);
        }
    }
    struct Cell {
        int32_t q;
        std::vector<std::pair<int32_t, float>> terms;
    };
    // rows: cells sorted by column
    std::vector<std::map<int32_t, std::vector<std::pair<int32_t, float>>>> rows((size_t)nh);
    if (forces) {
        for (const auto& e : pf.entries) {
            if (e.p == e.q) {
                rows[(size_t)e.p][e.q].push_back({e.leaf, 2.0f});
            } else {
                rows[(size_t)e.p][e.q].push_back({e.leaf, 1.0f});
                rows[(size_t)e.q][e.p].push_back({e.leaf, 1.0f});
            }
        }
    } else {
        // each monomial goes to the half with more monomials (fewer, longer rows)
        std::vector<int> use((size_t)nh, 0);
        for (const auto& e : pf.entries) {
            ++use[(size_t)e.p];
            ++use[(size_t)e.q];
        }
        for (const auto& e : pf.entries) {
            const bool to_p = use[(size_t)e.p] != use[(size_t)e.q] ? use[(size_t)e.p] > use[(size_t)e.q] : e.p < e.q;
            rows[(size_t)(to_p ? e.p : e.q)][to_p ? e.q : e.p].push_back({e.leaf, 1.0f});
        }
    }
    struct Panel {
        std::vector<int32_t> rows, cols;
        double cost = 0;
        std::vector<int32_t> targets;
        int nrec[3] = {0, 0, 0};
        struct Rec {
            int nq;
            uint32_t shared;     // pooled index | conj << 16
            int32_t q[4];
            uint16_t other[4];
        };
        std::vector<Rec> recs;
    };
    std::vector<Panel> panels;
    const int nw = (nh + 63) / 64;
    std::vector<uint64_t> bits((size_t)nh * nw, 0);
    for (int p = 0; p < nh; ++p)
        for (const auto& c : rows[(size_t)p]) bits[(size_t)p * nw + c.first / 64] |= 1ull << (c.first % 64);
    for (int c = 0; c < pf.ncls; ++c) {
        std::vector<int32_t> left;
        for (int p = 0; p < nh; ++p)
            if (pf.cls[(size_t)p] == c && !rows[(size_t)p].empty()) left.push_back(p);
        std::stable_sort(left.begin(), left.end(),
                         [&](int x, int y) { return rows[(size_t)x].size() > rows[(size_t)y].size(); });
        while (!left.empty()) {
            Panel pn;
            pn.rows.push_back(left.front());
            left.erase(left.begin());
            std::vector<uint64_t> u(bits.begin() + (size_t)pn.rows[0] * nw, bits.begin() + (size_t)(pn.rows[0] + 1) * nw);
            while ((int)pn.rows.size() < PAIR_ROWS && !left.empty()) {
                int best = -1, score = 0;
                for (size_t i = 0; i < left.size(); ++i) {
                    const uint64_t* b = &bits[(size_t)left[i] * nw];
                    int in = 0, add = 0;
                    for (int w = 0; w < nw; ++w) {
                        in += __builtin_popcountll(b[w] & u[(size_t)w]);
                        add += __builtin_popcountll(b[w] & ~u[(size_t)w]);
                    }
                    const auto& h = pf.halves[(size_t)left[i]];
                    int same = 0;
                    for (int32_t r : pn.rows) {
                        const auto& g = pf.halves[(size_t)r];
                        same |= (g.a == h.a || g.d == h.a ? 1 : 0) | (g.a == h.d || g.d == h.d ? 2 : 0);
                    }
                    // shared columns, few new ones, and (fewer turns) shared targets
                    const int sc = 2 * in - add + 3 * ((same & 1) + (same >> 1));
                    if (best < 0 || sc > score) {
                        best = (int)i;
                        score = sc;
                    }
                }
                const int32_t p = left[(size_t)best];
                left.erase(left.begin() + best);
                pn.rows.push_back(p);
                for (int w = 0; w < nw; ++w) u[(size_t)w] |= bits[(size_t)p * nw + w];
            }
            std::vector<int32_t> cols;
            for (int q = 0; q < nh; ++q)
                if (u[(size_t)(q / 64)] >> (q % 64) & 1) cols.push_back(q);
            // long panels are cut into equal pieces by columns (sorted by factor)
            std::stable_sort(cols.begin(), cols.end(), [&](int x, int y) {
                return std::make_tuple(pf.halves[(size_t)x].conj, pf.halves[(size_t)x].a, pf.halves[(size_t)x].d) <
                       std::make_tuple(pf.halves[(size_t)y].conj, pf.halves[(size_t)y].a, pf.halves[(size_t)y].d);
            });
            const int n = (int)cols.size(), pieces = std::max(1, (n + cap - 1) / cap);
            for (int i = 0; i < pieces; ++i) {
                Panel pp;
                pp.cols.assign(cols.begin() + (size_t)n * i / pieces, cols.begin() + (size_t)n * (i + 1) / pieces);
                for (int32_t r : pn.rows) {
                    bool any = false;
                    for (int32_t q : pp.cols) any = any || rows[(size_t)r].count(q);
                    if (any) pp.rows.push_back(r);
                }
                if (!pp.rows.empty()) panels.push_back(std::move(pp));
            }
        }
    }
    // records: columns that share a factor, four, two or one at a time
    for (Panel& pn : panels) {
        std::map<uint32_t, std::vector<int32_t>> by;  // shared factor -> columns
        std::vector<char> done(pn.cols.size(), 0);
        std::unordered_map<int32_t, size_t> at;
        for (size_t i = 0; i < pn.cols.size(); ++i) at[pn.cols[i]] = i;
        auto keys = [&](int32_t q, uint32_t k[2]) {
            const auto& h = pf.halves[(size_t)q];
            if (h.conj) {
                k[0] = (uint32_t)h.d | 1u << 16;  // the conjugated factor is the shared one
                return 1;
            }
            k[0] = h.a;
            k[1] = h.d;
            return h.a == h.d ? 1 : 2;
        };
        for (int32_t q : pn.cols) {
            uint32_t k[2];
            const int n = keys(q, k);
            for (int i = 0; i < n; ++i) by[k[i]].push_back(q);
        }
        for (int need = 4; need >= 1; need /= 2) {
            for (;;) {
                uint32_t bk = 0;
                size_t bn = 0;
                for (auto& kv : by) {
                    auto& v = kv.second;
                    v.erase(std::remove_if(v.begin(), v.end(), [&](int32_t q) { return done[at[q]] != 0; }), v.end());
                    if (v.size() > bn) {
                        bn = v.size();
                        bk = kv.first;
                    }
                }
                if (bn < (size_t)need) break;
                const std::vector<int32_t> v = by[bk];
                const size_t take = bn / need * need;
                for (size_t i = 0; i < take; i += need) {
                    Panel::Rec r;
                    r.nq = need;
                    r.shared = bk;
                    for (int j = 0; j < need; ++j) {
                        const int32_t q = v[i + j];
                        const auto& h = pf.halves[(size_t)q];
                        r.q[j] = q;
                        r.other[j] = h.conj ? h.a : (h.a == (bk & 0xffff) ? h.d : h.a);
                        done[at[q]] = 1;
                    }
                    pn.recs.push_back(r);
                    ++pn.nrec[need == 4 ? 0 : need == 2 ? 1 : 2];
                }
            }
        }
        // vector instructions: the records, and per row the products of the scatter
        pn.cost = 20.0 + (forces ? 18.0 : 8.0) * pn.rows.size();
        for (const auto& r : pn.recs) pn.cost += pair_rec_cost(r.nq);
        for (int32_t p : pn.rows)
            for (int k : {(int)pf.halves[(size_t)p].a, (int)pf.halves[(size_t)p].d})
                if (k != npool) pn.targets.push_back(k);
        std::sort(pn.targets.begin(), pn.targets.end());
        pn.targets.erase(std::unique(pn.targets.begin(), pn.targets.end()), pn.targets.end());
    }
    std::stable_sort(panels.begin(), panels.end(), [](const Panel& x, const Panel& y) { return x.cost > y.cost; });
    // rounds of PAIR_WAVES panels of similar cost; with forces, turns of four
    // panels (one per SIMD: waves 4 s .. 4 s + 3) without a common target
    std::vector<char> used(panels.size(), 0);
    size_t first = 0;
    auto disjoint = [&](const Panel& x, const std::vector<char>& hit) {
        if (!forces) return true;
        for (int k : x.targets)
            if (hit[(size_t)k]) return false;
        return true;
    };
    constexpr int NP = PAIR_WAVES;
    constexpr size_t WINDOW = 6 * PAIR_WAVES;
    constexpr int TURNS = 6;  // turns a round is given before it gets more
    while (first < panels.size()) {
        std::vector<std::pair<int, int>> got;  // panel, turn
        std::vector<std::vector<char>> hit;    // [turn][target]
        std::vector<int> load;
        auto place = [&](size_t i, int most) {
            int t = -1;
            for (size_t k = 0; k < hit.size(); ++k)
                if (disjoint(panels[i], hit[k]) && (t < 0 || load[k] < load[(size_t)t])) t = (int)k;
            if ((int)hit.size() < most && (t < 0 || load[(size_t)t] >= NP / TURNS)) {
                t = (int)hit.size();
                hit.emplace_back((size_t)npool + 1 + pf.virt.size(), (char)0);
                load.push_back(0);
            }
            if (t < 0) return;
            for (int k : panels[i].targets) hit[(size_t)t][(size_t)k] = 1;
            ++load[(size_t)t];
            used[i] = 1;
            got.push_back({(int)i, t});
        };
        for (int most = TURNS; (int)got.size() < NP && most <= NP; ++most) {
            size_t seen = 0;
            for (size_t i = first; i < panels.size() && seen < WINDOW && (int)got.size() < NP; ++i) {
                if (used[i]) continue;
                ++seen;
                place(i, forces ? most : 1);
            }
        }
        while (first < panels.size() && used[first]) ++first;
        const int nt = (int)hit.size();
        // waves w, w + 4, .. share a SIMD: equal sums
        int slots[NP], turn_of[NP];
        std::fill(slots, slots + NP, -1);
        {
            std::stable_sort(got.begin(), got.end(), [&](const auto& x, const auto& y) {
                return panels[(size_t)x.first].cost > panels[(size_t)y.first].cost;
            });
            double simd[4] = {0, 0, 0, 0};
            for (const auto& x : got) {
                int b = -1;
                for (int w = 0; w < NP; ++w)
                    if (slots[w] < 0 && (b < 0 || simd[w & 3] < simd[b & 3])) b = w;
                slots[b] = x.first;
                turn_of[b] = x.second;
                simd[b & 3] += panels[(size_t)x.first].cost;
            }
        }
        double simd[4] = {0, 0, 0, 0};
        for (int w = 0; w < NP; ++w) {
            if (slots[w] < 0) {
                out.panel.push_back(-1);
                continue;
            }
            const Panel& pn = panels[(size_t)slots[w]];
            simd[w & 3] += pn.cost;
            out.panel.push_back((int32_t)out.words.size());
            std::vector<uint32_t> hd(PAIR_HDR, 0);
            hd[0] = (uint32_t)pn.nrec[0] | (uint32_t)pn.nrec[1] << 10 | (uint32_t)pn.nrec[2] << 20;
            hd[1] = (uint32_t)pn.rows.size() | (uint32_t)turn_of[w] << 8;
            hd[2] = (uint32_t)out.coef.size();
            for (int r = 0; r < PAIR_ROWS; ++r) {
                // absent rows: the constant's (their h is zero)
                const PairForm::Half h = r < (int)pn.rows.size() ? pf.halves[(size_t)pn.rows[(size_t)r]]
                                                                 : PairForm::Half{(uint16_t)npool, (uint16_t)npool, false};
                hd[4 + 2 * r] = (uint32_t)h.a * row_bytes;
                hd[5 + 2 * r] = (uint32_t)h.d * row_bytes | (h.conj ? 1u : 0u);
            }
            out.words.insert(out.words.end(), hd.begin(), hd.end());
            for (int need = 4; need >= 1; need /= 2)
                for (const auto& rc : pn.recs) {
                    if (rc.nq != need) continue;
                    out.words.push_back((rc.shared & 0xffff) * row_bytes | (rc.shared >> 16));
                    for (int j = 0; j < need; ++j) out.words.push_back((uint32_t)rc.other[j] * row_bytes);
                    for (int j = 0; j < need; ++j)
                        for (int r = 0; r < PAIR_ROWS; ++r) {
                            const uint32_t at = (uint32_t)out.coef.size();
                            out.coef.push_back(0.0);
                            if (r >= (int)pn.rows.size()) continue;
                            const auto& row = rows[(size_t)pn.rows[(size_t)r]];
                            const auto it = row.find(rc.q[j]);
                            if (it != row.end())
                                for (const auto& t : it->second) out.terms.push_back({at, t.first, t.second});
                        }
                }
        }
        out.turns.push_back(forces ? nt : 0);
        // measured: an FP64 wave instruction takes 4.6 clocks of its SIMD (a probe;
        // 5.9 of the nominal clock with the whole chip at work), an
        // LDS atomic 9.3 of the CU, a turn's barrier about 150
        out.cost.push_back(4.6 * *std::max_element(simd, simd + 4) + (forces ? 150.0 * nt : 0.0));
    }
    // the rounds of P workgroups: longest first to the least loaded
    const int nr = out.nrounds();
    out.part_cost.assign(PAIR_MAXP + 2, 0.0);
    for (int P = 1; P <= PAIR_MAXP + 1; ++P) {
        std::vector<std::vector<int>> lists((size_t)P);
        std::vector<double> load((size_t)P, 0.0);
        std::vector<int> order((size_t)nr);
        for (int i = 0; i < nr; ++i) order[(size_t)i] = i;
        std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return out.cost[(size_t)x] > out.cost[(size_t)y]; });
        for (int i : order) {
            const size_t w = (size_t)(std::min_element(load.begin(), load.end()) - load.begin());
            lists[w].push_back(i);
            load[w] += out.cost[(size_t)i];
        }
        for (auto& l : lists) {
            std::sort(l.begin(), l.end());
            std::vector<int32_t>& sq = out.seq[P];
            out.seq_ptr[P].push_back((int32_t)sq.size());
            sq.push_back((int32_t)l.size());
            for (int rd : l) {
                sq.push_back(out.turns[(size_t)rd]);
                sq.insert(sq.end(), out.panel.begin() + (size_t)NP * rd, out.panel.begin() + (size_t)NP * (rd + 1));
            }
            sq.insert(sq.end(), PAIR_SEQ, -1);
        }
        out.part_cost[(size_t)P] = *std::max_element(load.begin(), load.end());
    }
    // slack behind the last record (the kernel reads one record ahead)
    out.words.resize(out.words.size() + 16, 0u);
    out.coef.resize(out.coef.size() + 64, 0.0);
    return "";
}

// What k_pairs executes per environment with `parts` workgroups per tile, as its
// code has it: FP64 vector operations and bytes that loads take from LDS (the
// atomic additions to G are neither).  A lane has half an environment.  Order 4,
// degree 12, whole tiles: 337,926 operations; the counter
// SQ_INSTS_VALU_FLOPS_FP64 gives 337,984.
struct DagWork {
    double flops = 0, lds = 0;
};
inline DagWork pair_work(const PairProgram& pp, bool forces, double parts) {
    DagWork w;
    for (int32_t at : pp.panel) {
        if (at < 0) continue;
        const uint32_t cnt = pp.words[(size_t)at];
        for (int k = 0; k < 3; ++k) {
            const int nq = k == 0 ? 4 : k == 1 ? 2 : 1;
            const double n = cnt >> (10 * k) & (k < 2 ? 1023u : 4095u);
            // per column a multiplication and a multiply-add, then one multiply-add per row
            w.flops += n * nq * (3.0 + 2.0 * PAIR_ROWS);
            w.lds += n * (16.0 + 16.0 * nq);
        }
        // per row: both products, and the energy
        w.flops += PAIR_ROWS * (forces ? 8.0 : 5.0);
        w.lds += PAIR_ROWS * 32.0;
    }
    const double nvirt = (double)pp.virt.size() / 2, nback = (double)pp.back.size() / 2;
    const double npool = (double)pp.back_ptr.size() - 1;
    w.flops += parts * (nvirt * 3.0 + (forces ? nback * 4.0 : 0.0));
    w.lds += parts * (nvirt * 32.0 + (forces ? nback * 32.0 + npool * 8.0 : 0.0));
    w.flops *= 2.0;
    w.lds *= 2.0;
    return w;
}

// The program's coefficients from those of the leaves.
inline void pair_coefs(PairProgram& pp, const std::vector<double>& leaf) {
    std::fill(pp.coef.begin(), pp.coef.end(), 0.0);
    for (const auto& t : pp.terms) pp.coef[t.at] += (double)t.scale * leaf[(size_t)t.leaf];
}

}  // namespace acehost
