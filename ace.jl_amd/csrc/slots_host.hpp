// Host-side (CPU) compiler of the slot programs: the class-split polynomials
// of an EuclideanVector basis of correlation order <= 3 for the kernel k_slots
// (ace_slots.hip).
//
// A G slot (pooled value k, class c) is a polynomial of the products of at most
// two pooled values (or conjugates) with complex coefficients, G = sum C y.
// Slots whose products overlap are packed into panels of up to SLOT_ROWS, whose
// columns are the union of their products: a product is formed once and
// multiplied into every slot of the panel.  A panel's columns come in steps of
// four (two for each half-wave, two of a half-wave's read at a time), ordered by
// the order of the monomials they come from: with the class value
//   Q_c = sum_k A[k] sum_o G_o[k, c] / o
// (Euler's identity for the part G_o that monomials of order o leave), the
// energy falls off the same sums.  Long panels are cut into pieces, each a slot
// of its own for the force kernel to add up.  The energies' program has one
// slot per (factor, class): every monomial is X_f times a product, f its factor
// of the highest degree, so that the products are few and shared.
#pragma once

#include <algorithm>
#include <cstdint>
#include <map>
#include <string>
#include <vector>

#include "pack_host.hpp"

namespace acehost {

constexpr int SLOT_ROWS = 4;      // slots per panel
constexpr int SLOT_WAVES = 16;    // waves per workgroup
constexpr int SLOT_MAXP = 16;     // workgroups a tile is split over, at most
constexpr int SLOT_COLS = 512;    // columns of a piece, at most
constexpr int SLOT_HDR = 4 + 3 * SLOT_ROWS;
constexpr int SLOT_MAX_POOL = 319;  // a tile's A+ and the constant: 160 KB

struct SlotProgram {
    // per piece: first step, steps of order 1, 2, 3, then per row: slot (-1:
    // none), the slot's factor (code), its class
    std::vector<uint32_t> hdr;
    // per step: [half-wave][column][factor] half the LDS offset of the factor | 1 << 31: conjugated
    std::vector<uint32_t> codes;
    std::vector<double> coef;  // per step: [half-wave][column][row][re, im]
    struct Term {
        uint32_t at;
        int32_t leaf;  // leaf, or ~task of a constant
    };
    std::vector<Term> terms;
    int nslots = 0;
    std::vector<int32_t> slot_k, slot_cls;             // forces: pooled value and class of a slot
    std::vector<int32_t> list_ptr[SLOT_MAXP + 1], list[SLOT_MAXP + 1];  // [P] pieces of [part][wave]
    double load[SLOT_MAXP + 1] = {0};                  // [P] clocks of the longest part
    int pieces() const { return (int)hdr.size() / SLOT_HDR; }
};

// Clocks of a SIMD per step: 2 columns of 2 products and 16 multiply-adds per row
// of 4.6 clocks (a probe; 5.9 with the whole chip at work), and the addresses and signs; of a piece besides; a step's
// latency in a wave that has its SIMD to itself.
constexpr double SLOT_STEP = 2 * (4 * SLOT_ROWS + 5) * 4.6 + 80, SLOT_PIECE = 600, SLOT_LATENCY = 500;

// gslot_ptr/list: slots per pooled value; cls: class per slot (both of the pack).
inline std::string slot_program(const PackCopy& pc, const std::vector<int32_t>& pool, const std::vector<int32_t>& gslot_ptr,
                                const std::vector<int32_t>& gslot_list, const std::vector<int32_t>& gslot_cls, bool forces,
                                SlotProgram& out) {
    out = SlotProgram();
    const int npool = (int)pool.size() / 4, ONE = npool;
    if (npool > SLOT_MAX_POOL) return "too many pooled values";
    auto m_of = [&](uint32_t f) {
        const int k = (int)(f & 0x7fff), m = k == ONE ? 0 : pool[4 * (size_t)k + 3];
        return (f & 0x8000) ? -m : m;
    };
    auto l_of = [&](uint32_t f) { return (int)(f & 0x7fff) == ONE ? 0 : pool[4 * (size_t)(f & 0x7fff) + 2]; };
    auto deg = [&](uint32_t f) { return (int)(f & 0x7fff) == ONE ? -1 : pool[4 * (size_t)(f & 0x7fff) + 1] - 1 + l_of(f); };
    struct Col {
        uint32_t f, g;  // factors, f <= g
        int order;
        bool operator<(const Col& o) const {
            return order != o.order ? order < o.order : f != o.f ? f < o.f : g < o.g;
        }
    };
    struct Slot {
        int32_t k = 0, cls = 0;
        uint32_t factor = 0;
        std::map<Col, std::vector<int32_t>> cols;  // leaves
    };
    std::vector<Slot> slots;
    // pooled value of each slot of the pack
    std::vector<int32_t> k_of(gslot_cls.size(), -1);
    for (int k = 0; k < npool; ++k)
        for (int i = gslot_ptr[(size_t)k]; i < gslot_ptr[(size_t)k + 1]; ++i) k_of[(size_t)gslot_list[(size_t)i]] = k;
    std::map<std::pair<uint32_t, int>, size_t> where;  // (factor, class) -> slot
    auto slot_at = [&](uint32_t f, int cls) -> Slot& {
        const auto it = where.emplace(std::make_pair(f, cls), slots.size());
        if (it.second) {
            slots.push_back(Slot());
            slots.back().k = (int32_t)(f & 0x7fff);
            slots.back().cls = cls;
            slots.back().factor = f;
        }
        return slots[it.first->second];
    };
    for (int t = 0; t < pc.ntasks; ++t) {
        const int o = pc.tasks[5 * (size_t)t + 2];
        if ((o >= 0) != forces) continue;
        if (o >= 0 && k_of[(size_t)o] < 0) return "slot without a pooled value";
        if (pc.task_term_ptr[t + 1] != pc.task_term_ptr[t]) {
            if (o < 0) return "energy task with constant terms";
            slot_at((uint32_t)k_of[(size_t)o], gslot_cls[(size_t)o]).cols[Col{(uint32_t)ONE, (uint32_t)ONE, 1}].push_back(~t);
        }
        for (int r = pc.tasks[5 * (size_t)t]; r < pc.tasks[5 * (size_t)t + 1]; ++r) {
            const int32_t* run = pc.runs.data() + (size_t)ACE_RUN_W * r;
            if (run[0] > (forces ? 1 : 2)) return "correlation order above 3";
            for (int i = 0; i < run[2]; ++i) {
                const int32_t leaf = run[3] + i;
                uint32_t f[3] = {(uint32_t)ONE, (uint32_t)ONE, (uint32_t)ONE};
                for (int q = 0; q < run[0]; ++q) f[q] = (uint32_t)run[4 + q];
                f[run[0]] = (uint32_t)pc.leaf_fid[(size_t)leaf];
                int n = run[0] + 1;
                if (forces) {
                    ++n;  // and the slot's own
                } else {
                    int best = 0;
                    for (int q = 1; q < n; ++q)
                        if (deg(f[q]) > deg(f[best]) || (deg(f[q]) == deg(f[best]) && f[q] > f[best])) best = q;
                    std::swap(f[best], f[2]);
                }
                Slot& s = forces ? slot_at((uint32_t)k_of[(size_t)o], gslot_cls[(size_t)o]) : slot_at(f[2], -1 - o);
                s.cols[Col{std::min(f[0], f[1]), std::max(f[0], f[1]), n}].push_back(leaf);
            }
        }
    }
    if (slots.empty()) return "no monomials";
    // panels: within slots of equal total m and parity of l of their products,
    // the longest slot left and those that add the fewest columns
    struct Panel {
        std::vector<size_t> rows;
        std::vector<Col> cols;
    };
    std::vector<Panel> panels;
    std::map<std::pair<int, int>, std::vector<size_t>> groups;
    for (size_t i = 0; i < slots.size(); ++i) {
        const Col& c = slots[i].cols.rbegin()->first;
        groups[{m_of(c.f) + m_of(c.g), (l_of(c.f) + l_of(c.g)) & 1}].push_back(i);
    }
    for (auto& gr : groups) {
        std::vector<size_t> left = gr.second;
        std::stable_sort(left.begin(), left.end(), [&](size_t a, size_t b) { return slots[a].cols.size() > slots[b].cols.size(); });
        // columns of the group, numbered
        std::map<Col, int> id;
        for (size_t i : left)
            for (const auto& c : slots[i].cols) id.emplace(c.first, 0);
        int n = 0;
        std::vector<Col> cols;
        for (auto& c : id) {
            c.second = n++;
            cols.push_back(c.first);
        }
        const size_t nw = ((size_t)n + 63) / 64;
        std::vector<uint64_t> bits(left.size() * nw, 0);
        std::map<size_t, size_t> at;
        for (size_t i = 0; i < left.size(); ++i) {
            at[left[i]] = i;
            for (const auto& c : slots[left[i]].cols) {
                const int q = id[c.first];
                bits[i * nw + (size_t)q / 64] |= 1ull << (q % 64);
            }
        }
        while (!left.empty()) {
            Panel pn;
            std::vector<uint64_t> u(nw, 0);
            while ((int)pn.rows.size() < SLOT_ROWS && !left.empty()) {
                size_t best = 0;
                long score = 0;
                for (size_t i = 0; i < left.size() && (i == 0 || !pn.rows.empty()); ++i) {
                    const uint64_t* b = &bits[at[left[i]] * nw];
                    long add = 0, miss = 0;
                    for (size_t w = 0; w < nw; ++w) {
                        add += __builtin_popcountll(b[w] & ~u[w]);
                        miss += __builtin_popcountll(u[w] & ~b[w]);
                    }
                    const long sc = SLOT_ROWS * add + miss;
                    if (i == 0 || sc < score) {
                        best = i;
                        score = sc;
                    }
                }
                const uint64_t* b = &bits[at[left[best]] * nw];
                for (size_t w = 0; w < nw; ++w) u[w] |= b[w];
                pn.rows.push_back(left[best]);
                left.erase(left.begin() + (long)best);
            }
            for (int q = 0; q < n; ++q)
                if (u[(size_t)q / 64] >> (q % 64) & 1) pn.cols.push_back(cols[(size_t)q]);
            panels.push_back(std::move(pn));
        }
    }
    // pieces: equal shares of a panel's columns, each order in whole steps
    std::vector<double> cost;
    std::vector<int> steps;
    for (const Panel& pn : panels) {
        const int n = (int)pn.cols.size(), pieces = (n + SLOT_COLS - 1) / SLOT_COLS;
        for (int p = 0; p < pieces; ++p) {
            const int c0 = (int)((int64_t)n * p / pieces), c1 = (int)((int64_t)n * (p + 1) / pieces);
            uint32_t hd[SLOT_HDR];
            hd[0] = (uint32_t)(out.codes.size() / 8);
            int at = c0, total = 0;
            for (int o = 1; o <= 3; ++o) {
                const int b = at;
                while (at < c1 && pn.cols[(size_t)at].order == o) ++at;
                const int ns = (at - b + 3) / 4;
                hd[o] = (uint32_t)ns;
                total += ns;
                for (int i = 0; i < 4 * ns; ++i) {
                    const bool in = b + i < at;
                    const Col c = in ? pn.cols[(size_t)(b + i)] : Col{(uint32_t)ONE, (uint32_t)ONE, o};
                    for (uint32_t f : {c.f, c.g}) out.codes.push_back((f & 0x7fffu) * 256u | (f & 0x8000u) << 16);
                    for (int r = 0; r < SLOT_ROWS; ++r) {
                        const uint32_t ca = (uint32_t)out.coef.size();
                        out.coef.push_back(0.0);
                        out.coef.push_back(0.0);
                        if (!in || r >= (int)pn.rows.size()) continue;
                        const auto& sc = slots[pn.rows[(size_t)r]].cols;
                        const auto it = sc.find(c);
                        if (it != sc.end())
                            for (int32_t l : it->second) out.terms.push_back({ca, l});
                    }
                }
            }
            for (int r = 0; r < SLOT_ROWS; ++r) {
                const bool in = r < (int)pn.rows.size();
                const Slot* s = in ? &slots[pn.rows[(size_t)r]] : nullptr;
                hd[4 + r] = in ? (uint32_t)out.nslots : ~0u;
                hd[4 + SLOT_ROWS + r] = in ? (s->factor & 0x7fffu) * 256u | (s->factor & 0x8000u) << 16 : 0u;
                hd[4 + 2 * SLOT_ROWS + r] = in ? (uint32_t)s->cls : 0u;
                if (!in) continue;
                ++out.nslots;
                out.slot_k.push_back(s->k);
                out.slot_cls.push_back(s->cls);
            }
            out.hdr.insert(out.hdr.end(), hd, hd + SLOT_HDR);
            cost.push_back(SLOT_PIECE + SLOT_STEP * total);
            steps.push_back(total);
        }
    }
    // pieces of [part][wave]: the longest first to the least loaded SIMD (waves
    // w, w + 4, .. of a workgroup share one), there to the least loaded wave
    std::vector<int> order(cost.size());
    for (size_t i = 0; i < order.size(); ++i) order[i] = (int)i;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cost[(size_t)x] > cost[(size_t)y]; });
    for (int P = 1; P <= SLOT_MAXP; ++P) {
        std::vector<double> simd((size_t)P * 4, 0.0), wave((size_t)P * SLOT_WAVES, 0.0), lat((size_t)P * SLOT_WAVES, 0.0);
        std::vector<std::vector<int32_t>> of((size_t)P * SLOT_WAVES);
        for (int i : order) {
            const size_t s = (size_t)(std::min_element(simd.begin(), simd.end()) - simd.begin());
            size_t best = 0;
            for (size_t j = 0; j < 4; ++j) {
                const size_t w = s / 4 * SLOT_WAVES + s % 4 + 4 * j;
                if (j == 0 || wave[w] < wave[best]) best = w;
            }
            simd[s] += cost[(size_t)i];
            wave[best] += cost[(size_t)i];
            lat[best] += SLOT_LATENCY * steps[(size_t)i];
            of[best].push_back(i);
        }
        out.list_ptr[P].push_back(0);
        for (const auto& l : of) {
            out.list[P].insert(out.list[P].end(), l.begin(), l.end());
            out.list_ptr[P].push_back((int32_t)out.list[P].size());
        }
        out.load[P] = std::max(*std::max_element(simd.begin(), simd.end()), *std::max_element(lat.begin(), lat.end()));
    }
    // slack for reading two steps ahead
    out.codes.resize(out.codes.size() + 3 * 8, 0u);
    out.coef.resize(out.coef.size() + 3 * 8 * SLOT_ROWS, 0.0);
    return "";
}

// Workgroups per tile, P of the first tiles and P_hi of the last nhi ones:
// per_cu workgroups share a compute unit, each staging its tile and doing the
// longest part.  The tiles that would leave a last round nearly empty are split
// further to fill one, or all tiles alike (16,385 environments, 220 pooled
// values: the last of 513 tiles over 16 workgroups 0.61 ms, all over 6 0.66).
struct SlotShape {
    int P = 1, P_hi = 1;
    int64_t nhi = 0;
};
inline SlotShape slot_shape(const SlotProgram& sp, int64_t ntile, int ncu, int per_cu) {
    const int64_t slots = (int64_t)ncu * per_cu;
    // the last round's workgroups have a compute unit each if they are few
    auto clocks = [&](int P, int64_t n) { return (n <= ncu ? 1 : per_cu) * sp.load[P] + 6000.0; };
    SlotShape best;
    double tb = 1e300;
    auto consider = [&](double t, int P, int P_hi, int64_t nhi) {
        if (t >= tb * 0.995) return;
        tb = t;
        best.P = P;
        best.P_hi = P_hi;
        best.nhi = nhi;
    };
    for (int P = 1; P <= SLOT_MAXP; ++P) {
        const int64_t full = ntile * P / slots, rest = ntile * P - full * slots;
        const double whole = (double)full * clocks(P, slots);
        consider(whole + (rest ? clocks(P, rest) : 0.0), P, P, 0);
        // the remaining tiles in a round of their own, which starts late (a
        // workgroup of any length takes some 12,000 clocks to get going)
        const int64_t left = ntile - full * slots / P;
        if (full == 0 || left == 0 || left > slots) continue;
        const int hi = (int)std::min<int64_t>(SLOT_MAXP, slots / left);
        if (hi > P) consider(whole + clocks(hi, left * hi) + 12000.0, P, hi, left);
    }
    return best;
}

// What k_slots executes per environment, as its code has it: FP64 vector
// operations and bytes that loads take from LDS.  Two lanes have an environment.
struct SlotWork {
    double flops = 0, lds = 0;
};
inline SlotWork slot_work(const SlotProgram& sp, bool forces) {
    SlotWork w;
    for (int p = 0; p < sp.pieces(); ++p) {
        const uint32_t* hd = sp.hdr.data() + (size_t)SLOT_HDR * p;
        // a step: two products of two values, four multiply-adds per row and product
        w.flops += (double)(hd[1] + hd[2] + hd[3]) * (2.0 * 6.0 + 2.0 * 8.0 * SLOT_ROWS);
        w.lds += (double)(hd[1] + hd[2] + hd[3]) * 4.0 * 16.0;
        if (forces) w.flops += 3.0 * 4.0 * SLOT_ROWS;
        for (int r = 0; r < SLOT_ROWS; ++r) {
            if (hd[4 + r] == ~0u) continue;
            w.flops += 6.0 + 2.0 + (forces ? 1.0 : 0.0);  // the slot's share of Q, the half-waves' sum
            w.lds += 16.0;
        }
    }
    w.flops *= 2.0;
    w.lds *= 2.0;
    return w;
}

// The program's coefficients from those of the leaves and the tasks' constants
// (complex numbers).
inline void slot_coefs(SlotProgram& sp, const Coeffs& cf) {
    std::fill(sp.coef.begin(), sp.coef.end(), 0.0);
    for (const auto& t : sp.terms)
        for (int q = 0; q < 2; ++q)
            sp.coef[t.at + q] += t.leaf >= 0 ? cf.leaf[2 * (size_t)t.leaf + q] : cf.task[2 * (size_t)~t.leaf + q];
}

}  // namespace acehost
