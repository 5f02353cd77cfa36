// Host-side (CPU) layout of the basis-value kernel's records (k_Bv,
// ace_basis.hip): B = A2B AA and its directional derivative for Invariant
// bases of correlation order <= 4 (symmbasis.jl:248-264, evaluator.jl:225-240).
//
// A basis function is B_b = Re sum_z v_z prod X_f (X_f = A+[k] or its
// conjugate).  Nonzeros of one row whose monomials are equal or mirror images
// (every factor conjugated) have the same real part, so they merge into one
// record with the sum of their values; the m < 0 factor signs go into the
// value.  A row's records of one order are a segment; the two half-waves of
// the kernel take the records of a segment alternately, and an odd last record
// is given to both with half its value each (exact in binary).
#pragma once

#include <algorithm>
#include <cstdint>
#include <map>
#include <vector>

#include "pack_host.hpp"

namespace acehost {

constexpr int BV_UNITS = 768;  // equal shares of the segments: 16 waves x up to 48 workgroups per tile
constexpr int BV_WAVES = 16;

// Factors: pooled index (9 bits) | 0x8000: conjugated; the first one never is.
struct BvRec {
    uint16_t f[4];
    double c;
};
static_assert(sizeof(BvRec) == 16, "BvRec is one 16-byte load");

struct BvProgram {
    std::vector<BvRec> rec;      // pairs of records; one unused pair behind the last (read ahead)
    std::vector<int32_t> seg;    // [segment] row | 1 << 31: the row ends here, pairs of records | order << 28
    std::vector<int32_t> unit;   // [BV_UNITS + 1] first segment, first pair
    double iter = 0, cost = 0;   // pairs of records, and clocks of a compute unit per tile, estimated
};

// Clocks of a compute unit per pair of records of an order (LDS reads and
// vector instructions of one wave), and per segment (its header, the sum over
// the half-waves, the store).
inline double bv_pair_cost(int order) { return 2.0 + 7.0 * order; }
constexpr double BV_SEG_COST = 40.0;

inline bool bv_usable(const ace_pack* pk) {
    return pk->prop == ACE_PROP_INVARIANT && pk->maxorder <= 4 && pk->npool <= 320;
}

inline BvProgram bv_program(const ace_pack* pk) {
    BvProgram p;
    struct Key {
        int n;
        uint16_t f[4];
        bool operator<(const Key& o) const {
            if (n != o.n) return n < o.n;
            return std::lexicographical_compare(f, f + 4, o.f, o.f + 4);
        }
    };
    auto real = [&](uint16_t f) { return pk->pool[4 * (f & 0x7fff) + 3] == 0; };
    // complex factors first, by pooled index, plain before conjugated
    auto sorted = [&](Key k) {
        std::sort(k.f, k.f + k.n, [&](uint16_t a, uint16_t b) {
            if (real(a) != real(b)) return !real(a);
            return (a & 0x7fff) != (b & 0x7fff) ? (a & 0x7fff) < (b & 0x7fff) : a < b;
        });
        return k;
    };
    std::vector<double> at;  // cost before each segment
    std::vector<int32_t> pair0;
    for (int b = 0; b < pk->nB; ++b) {
        std::map<Key, double> row;
        for (int z = pk->a2b_rowptr[b]; z < pk->a2b_rowptr[b + 1]; ++z) {
            const int col = pk->a2b_cols[z];
            Key k{pk->orders[col], {0, 0, 0, 0}}, m = k;
            double v = pk->a2b_vals[z];
            for (int q = 0; q < k.n; ++q) {
                const int iA = pk->iAA2iA[(size_t)col * pk->maxorder + q];
                const int f = pk->aspec_fid[iA];
                v *= pk->aspec_sgn[iA];
                k.f[q] = (uint16_t)(real((uint16_t)f) ? f & 0x7fff : f);
                m.f[q] = (uint16_t)(real((uint16_t)f) ? f & 0x7fff : f ^ 0x8000);
            }
            k = sorted(k);
            m = sorted(m);
            // the image whose first factor is plain; the smaller one if both are
            const bool kc = k.n > 0 && (k.f[0] & 0x8000), mc = m.n > 0 && (m.f[0] & 0x8000);
            if (kc || (!mc && m < k)) k = m;
            row[k] += v;
        }
        // the map is ordered by order first: one segment per order
        for (int o = 0; o <= 4; ++o) {
            std::vector<BvRec> r;
            for (auto& [k, v] : row)
                if (k.n == o) r.push_back(BvRec{{k.f[0], k.f[1], k.f[2], k.f[3]}, v});
            const bool last = row.empty() || row.rbegin()->first.n <= o;
            if (r.empty() && !(row.empty() && o == 0)) continue;
            if (r.size() & 1) {
                r.back().c *= 0.5;
                r.push_back(r.back());
            }
            at.push_back(p.cost);
            pair0.push_back((int32_t)(p.rec.size() / 2));
            p.seg.push_back((int32_t)((uint32_t)b | (last ? 1u << 31 : 0u)));
            p.seg.push_back((int32_t)(r.size() / 2) | (o << 28));
            p.rec.insert(p.rec.end(), r.begin(), r.end());
            p.cost += BV_SEG_COST + (double)(r.size() / 2) * bv_pair_cost(o);
            if (last) break;
        }
    }
    const int nseg = (int)at.size();
    pair0.push_back((int32_t)(p.rec.size() / 2));
    p.iter = (double)pair0.back();
    // unit u: the segments whose cost begins in its share, cut between rows only
    int s = 0;
    for (int u = 0; u <= BV_UNITS; ++u) {
        const double from = p.cost * u / BV_UNITS;
        while (s < nseg && (u == BV_UNITS || at[(size_t)s] < from || (s > 0 && p.seg[2 * (size_t)(s - 1)] >= 0))) ++s;
        p.unit.push_back(s);
        p.unit.push_back(pair0[(size_t)s]);
    }
    p.rec.push_back(BvRec{{0, 0, 0, 0}, 0.0});
    p.rec.push_back(BvRec{{0, 0, 0, 0}, 0.0});
    return p;
}

// Workgroups per tile (a divisor of 48) for a number of tiles: rounds of
// workgroups over the compute units, each staging the tile and doing its share
// of a tile's `cost` clocks.  `resident` workgroups share a compute unit; a
// wave's iteration takes 700 clocks at least (record load, LDS reads, the
// products' chain), however few waves there are.
inline int bv_chunks(double iter, double cost, int64_t tiles, int ncu, int resident, double tile_bytes) {
    static const int div[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 48};
    const double work = std::max(resident * cost, 700.0 * iter / BV_WAVES);
    const double stage = 3000.0 + resident * tile_bytes / 24.0;
    int best = 1;
    double tb = 1e300;
    for (int c : div) {
        const double rounds = (double)((tiles * c + (int64_t)ncu * resident - 1) / ((int64_t)ncu * resident));
        const double t = rounds * (stage + work / c);
        if (t < tb * 0.999) {
            tb = t;
            best = c;
        }
    }
    return best;
}

}  // namespace acehost
