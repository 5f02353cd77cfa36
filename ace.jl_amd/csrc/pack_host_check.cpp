// CPU test shim over pack_host.hpp and compile_host.hpp: the host-side pack
// logic and the program compiler of libacehip.so built without HIP (tests
// build it with the address sanitizer, and plain for the larger bases).
#include <algorithm>
#include <complex>
#include <cstring>
#include <map>
#include <set>

#include "basis_host.hpp"
#include "compile_host.hpp"
#include "grow_buf.hpp"
#include "nbrlist_host.hpp"
#include "pack_host.hpp"
#include "pairs_host.hpp"
#include "slots_host.hpp"
#include "tail_host.hpp"

extern "C" int acehost_validate(const ace_pack* pk, char* msg, int len) {
    std::string e = acehost::validate_pack(pk);
    if (e.empty()) {
        std::vector<acehost::WaveTable> wt;
        e = acehost::wave_tables(pk, wt);
    }
    if (msg && len > 0) {
        std::strncpy(msg, e.c_str(), (size_t)len - 1);
        msg[len - 1] = 0;
    }
    return e.empty() ? 0 : -1;
}

extern "C" int acehost_coeffs(const ace_pack* pk, const double* c, double* leaf, double* task, double* e0) {
    if (!acehost::validate_pack(pk).empty()) return -1;
    acehost::PackCopy p = acehost::copy_pack(pk);
    acehost::Coeffs cf = acehost::coefficients(p, c);
    std::memcpy(leaf, cf.leaf.data(), cf.leaf.size() * sizeof(double));
    std::memcpy(task, cf.task.data(), cf.task.size() * sizeof(double));
    std::memcpy(e0, cf.e0, 6 * sizeof(double));
    return 0;
}

extern "C" int acehost_lookup(const ace_pack* pk, short* kidx, int* a4) {
    if (!acehost::validate_pack(pk).empty()) return -1;
    std::vector<int16_t> kx = acehost::pool_lookup(pk);
    std::memcpy(kidx, kx.data(), kx.size() * sizeof(int16_t));
    std::vector<int32_t> a = acehost::aspec_rows(pk);
    std::memcpy(a4, a.data(), a.size() * sizeof(int32_t));
    return 0;
}

// A pair program run on the CPU as k_pairs runs it, on pooled values A[npool]
// (re, im) and parameters c: the energy, and with forces G[npool].  Returns 0,
// 1 when the basis has no pair form, -1 on a rejected table or two panels of
// one turn with a common target.
extern "C" int acehost_pairs(const ace_pack* pk, const double* c, int forces, int parts, const double* A, double* E,
                             double* G) {
    if (!acehost::validate_pack(pk).empty()) return -1;
    const acehost::PackCopy pc = acehost::copy_pack(pk);
    const int np = pk->npool, rb = forces ? 1024 : 512;
    acehost::PairForm pf;
    acehost::PairProgram pp;
    if (!acehost::pair_form(pc, std::vector<int32_t>(pk->pool, pk->pool + 4 * (size_t)np), 159, pf).empty()) return 1;
    if (!acehost::pair_program(pf, forces != 0, rb, np, 96, pp).empty()) return -1;
    const acehost::Coeffs cf = acehost::coefficients(pc, c);
    acehost::pair_coefs(pp, cf.leaf);
    typedef std::complex<double> C;
    const int nrow = np + 1 + (int)pf.virt.size();
    std::vector<C> row;
    auto val = [&](uint32_t w) {
        const C a = row[(w & ~1u) / rb];
        return w & 1u ? std::conj(a) : a;
    };
    for (int k = 0; k < np; ++k) row.push_back(C(A[2 * k], A[2 * k + 1]));
    row.push_back(1.0);
    for (size_t i = 0; i < pf.virt.size(); ++i) row.push_back(val(pp.virt[2 * i]) * val(pp.virt[2 * i + 1]));
    std::vector<C> g((size_t)nrow, 0.0);
    double e = 0.0;
    for (int part = 0; part < parts; ++part) {
        const int32_t* sq = pp.seq[parts].data() + pp.seq_ptr[parts][(size_t)part];
        const int nround = *sq++;
        for (int r = 0; r < nround; ++r, sq += acehost::PAIR_SEQ) {
            std::map<int, std::set<int>> hit;
            for (int w = 0; w < acehost::PAIR_WAVES; ++w) {
                if (sq[1 + w] < 0) continue;
                const uint32_t* hd = pp.words.data() + sq[1 + w];
                const double* co = pp.coef.data() + hd[2];
                const uint32_t* q = hd + acehost::PAIR_HDR;
                C h[acehost::PAIR_ROWS] = {};
                const int n[3] = {(int)(hd[0] & 1023u), (int)(hd[0] >> 10 & 1023u), (int)(hd[0] >> 20)};
                for (int kind = 0; kind < 3; ++kind)
                    for (int i = 0, nq = 4 >> kind; i < n[kind]; ++i, q += acehost::pair_rec_words(nq))
                        for (int j = 0; j < nq; ++j)
                            for (C& hr : h) hr += *co++ * val(q[0]) * val(q[1 + j]);
                std::set<int> mine;
                for (int s = 0; s < acehost::PAIR_ROWS; ++s) {
                    const uint32_t wa = hd[4 + 2 * s], wd = hd[5 + 2 * s];
                    const int ka = (int)wa / rb, kd = (int)(wd & ~1u) / rb;
                    const C gp = std::conj(h[s]), t2 = gp * val(wa);
                    e += (gp * val(wa) * val(wd)).real();
                    g[(size_t)ka] += gp * val(wd);
                    g[(size_t)kd] += wd & 1u ? std::conj(t2) : t2;
                    if (ka != np) mine.insert(ka);
                    if (kd != np) mine.insert(kd);
                }
                if (!forces) continue;
                const int turn = (int)(hd[1] >> 8);
                if (turn >= sq[0]) return -1;
                for (int k : mine)
                    if (!hit[turn].insert(k).second) return -1;
            }
        }
    }
    *E = cf.e0[0] + (forces ? 0.5 : 1.0) * e;
    for (int k = 0; k < np; ++k)
        for (int i = pp.back_ptr[(size_t)k]; i < pp.back_ptr[(size_t)k + 1]; ++i) {
            const uint32_t o = pp.back[2 * (size_t)i + 1];
            const C x = row[(o & ~3u) / rb], t = g[pp.back[2 * (size_t)i] / rb] * (o & acehost::PAIR_BACK_IN ? std::conj(x) : x);
            g[(size_t)k] += o & acehost::PAIR_BACK_OUT ? std::conj(t) : t;
        }
    for (int k = 0; forces && k < np; ++k) {
        G[2 * k] = g[(size_t)k].real();
        G[2 * k + 1] = g[(size_t)k].imag();
    }
    return 0;
}

// Lane sets of the pooling kernel: writes 64 kp slots, returns 1 when the
// sets fit 64 lanes, else 0.
extern "C" int acehost_pool_sets(const int32_t* pool, int npool, int kp, int32_t* slot) {
    std::vector<int32_t> v;
    if (!acehost::pool_lane_sets(pool, npool, kp, v)) return 0;
    std::memcpy(slot, v.data(), v.size() * sizeof(int32_t));
    return 1;
}

// Neighbour-list binning (nbrlist_host.hpp).  bin_start must hold
// 2 * natoms + 66 entries (the bin count never exceeds 2 natoms + 64).
extern "C" int acehost_nbr_grid(int64_t natoms, const double* pos, const double* cell, const int32_t* pbc,
                                double rcut, int* nb, int* R, int32_t* bin, int32_t* bin_start, int32_t* bin_atoms,
                                int32_t* wrap, double* pw, char* msg, int len) {
    acehost::NbrGrid g;
    std::string e = acehost::nbr_grid(natoms, pos, cell, pbc, rcut, g);
    if (msg && len > 0) {
        std::strncpy(msg, e.c_str(), (size_t)len - 1);
        msg[len - 1] = 0;
    }
    if (!e.empty()) return -1;
    for (int d = 0; d < 3; ++d) {
        nb[d] = g.nb[d];
        R[d] = g.R[d];
    }
    std::memcpy(bin, g.bin.data(), g.bin.size() * sizeof(int32_t));
    std::memcpy(bin_start, g.bin_start.data(), g.bin_start.size() * sizeof(int32_t));
    std::memcpy(bin_atoms, g.bin_atoms.data(), g.bin_atoms.size() * sizeof(int32_t));
    std::memcpy(wrap, g.wrap.data(), g.wrap.size() * sizeof(int32_t));
    std::memcpy(pw, g.p.data(), g.p.size() * sizeof(double));
    return 0;
}

// The program compiler (compile_host.hpp): compiles an ace_jl_basis, keeps the
// tables, and hands out any of them by name for comparison with the Python
// host's pack.  acehost_compiled_array returns the element count (copying
// into out when it is not null) or -1 for an unknown name.
extern "C" void* acehost_compile(const ace_jl_basis* b, char* msg, int len) {
    auto* ps = new acehost::PackStore();
    std::string e = acehost::compile_jl(b, *ps);
    if (e.empty()) {
        const ace_pack pk = ps->view();
        e = acehost::validate_pack(&pk);
    }
    if (msg && len > 0) {
        std::strncpy(msg, e.c_str(), (size_t)len - 1);
        msg[len - 1] = 0;
    }
    if (!e.empty()) {
        delete ps;
        return nullptr;
    }
    return ps;
}

extern "C" void acehost_compiled_free(void* p) { delete static_cast<acehost::PackStore*>(p); }

extern "C" int64_t acehost_compiled_array(void* p, const char* name, void* out) {
    const auto* ps = static_cast<const acehost::PackStore*>(p);
    auto put = [&](const auto& v) -> int64_t {
        if (out && !v.empty()) std::memcpy(out, v.data(), v.size() * sizeof(v[0]));
        return (int64_t)v.size();
    };
    const std::string n(name);
#define ACE_ARR(F) \
    if (n == #F) return put(ps->F);
    ACE_ARR(rA) ACE_ARR(rB) ACE_ARR(rC) ACE_ARR(pool) ACE_ARR(aspec_fid) ACE_ARR(aspec_sgn) ACE_ARR(orders)
    ACE_ARR(iAA2iA) ACE_ARR(a2b_rowptr) ACE_ARR(a2b_cols) ACE_ARR(a2b_vals) ACE_ARR(runs) ACE_ARR(leaf_fid)
    ACE_ARR(leaf_term_ptr) ACE_ARR(tasks) ACE_ARR(task_term_ptr) ACE_ARR(term_row) ACE_ARR(term_scale)
    ACE_ARR(term_conj) ACE_ARR(gslot_ptr) ACE_ARR(gslot_list) ACE_ARR(gslot_class) ACE_ARR(rec_hdr) ACE_ARR(rec_leaf) ACE_ARR(feat_rows)
    ACE_ARR(feat_ptr) ACE_ARR(feat_f) ACE_ARR(feat_coef) ACE_ARR(fgrad_ptr) ACE_ARR(fgrad_feat) ACE_ARR(fgrad_f)
    ACE_ARR(fgrad_coef) ACE_ARR(wave_cfg_W) ACE_ARR(wave_task_ptr) ACE_ARR(wave_task_list) ACE_ARR(wave_etask_ptr)
    ACE_ARR(wave_etask_list)
#undef ACE_ARR
    return -1;
}

// The basis-value records run on the CPU as k_Bv runs them on pooled values
// A[npool] and directions W[npool] (re, im): B[nB] and its derivative D[nB],
// with nchunk workgroups a tile.  Returns 0, 1 when the basis has no such
// records, -1 when a row is not written exactly once or a unit's records are
// not where it begins.
extern "C" int acehost_bv(const ace_pack* pk, int nchunk, const double* A, const double* W, double* B, double* D) {
    if (!acehost::validate_pack(pk).empty()) return -1;
    if (!acehost::bv_usable(pk)) return 1;
    const acehost::BvProgram p = acehost::bv_program(pk);
    typedef std::complex<double> C;
    auto val = [](const double* x, uint16_t f) {
        const C a(x[2 * (f & 0x1ff)], x[2 * (f & 0x1ff) + 1]);
        return f & 0x8000 ? std::conj(a) : a;
    };
    std::vector<int> seen((size_t)pk->nB, 0);
    const int uw = acehost::BV_UNITS / acehost::BV_WAVES / nchunk;
    for (int w = 0; w < nchunk * acehost::BV_WAVES; ++w) {
        const int32_t* u = p.unit.data() + 2 * (size_t)w * uw;
        int pair = u[1];
        double b = 0.0, d = 0.0;
        for (int g = u[0]; g < u[2 * uw]; ++g) {
            const int row = p.seg[2 * (size_t)g], n = p.seg[2 * (size_t)g + 1] & 0xfffffff, o = p.seg[2 * (size_t)g + 1] >> 28;
            for (int i = 0; i < 2 * n; ++i) {
                const acehost::BvRec& r = p.rec[2 * (size_t)pair + i];
                if (o > 0 && (r.f[0] & 0x8000)) return -1;
                C x = 1.0, dx = 0.0;
                for (int q = 0; q < o; ++q) {
                    dx = dx * val(A, r.f[q]) + x * val(W, r.f[q]);
                    x *= val(A, r.f[q]);
                }
                b += r.c * x.real();
                d += r.c * dx.real();
            }
            pair += n;
            if (row < 0) {
                seen[(size_t)(row & 0x7fffffff)] += 1;
                B[row & 0x7fffffff] = b;
                D[row & 0x7fffffff] = d;
                b = d = 0.0;
            }
        }
        if (pair != u[2 * uw + 1] || 2 * (size_t)pair + 2 > p.rec.size()) return -1;
    }
    for (int n : seen)
        if (n != 1) return -1;
    return 0;
}

// A slot program run on the CPU as k_slots runs it, on pooled values A[npool]
// (re, im) and parameters c, with P workgroups: the class values Q[3], and with
// forces G[npool][3 classes].  Returns 0, 1 when the basis has no slot form,
// -1 on a rejected table or when a piece is not run exactly once.
extern "C" int acehost_slots(const ace_pack* pk, const double* c, int forces, int P, const double* A, double* Q, double* G) {
    if (!acehost::validate_pack(pk).empty()) return -1;
    if (!pk->classed) return 1;
    const acehost::PackCopy pc = acehost::copy_pack(pk);
    acehost::SlotProgram sp;
    const std::vector<int32_t> ptr(pk->gslot_ptr, pk->gslot_ptr + pk->npool + 1);
    if (!acehost::slot_program(pc, std::vector<int32_t>(pk->pool, pk->pool + 4 * (size_t)pk->npool), ptr,
                               std::vector<int32_t>(pk->gslot_list, pk->gslot_list + ptr.back()),
                               std::vector<int32_t>(pk->gslot_class, pk->gslot_class + pk->ngslots), forces != 0, sp)
             .empty())
        return 1;
    acehost::slot_coefs(sp, acehost::coefficients(pc, c));
    typedef std::complex<double> C;
    constexpr int R = acehost::SLOT_ROWS;
    auto val = [&](uint32_t w) {
        const int k = (int)((w & 0x7fffffffu) / 256);
        const C a = k == pk->npool ? C(1.0) : C(A[2 * k], A[2 * k + 1]);
        return w >> 31 ? std::conj(a) : a;
    };
    std::vector<C> q(3, 0.0), g((size_t)pk->npool * 3, 0.0);
    std::vector<int> seen((size_t)sp.pieces(), 0);
    for (int w = 0; w < P * acehost::SLOT_WAVES; ++w)
        for (int i = sp.list_ptr[P][(size_t)w]; i < sp.list_ptr[P][(size_t)w + 1]; ++i) {
            const int piece = sp.list[P][(size_t)i];
            ++seen[(size_t)piece];
            const uint32_t* hd = sp.hdr.data() + (size_t)acehost::SLOT_HDR * piece;
            C acc[R] = {}, wt[R] = {};
            size_t col = 4 * (size_t)hd[0];
            for (int o = 1; o <= 3; ++o) {
                for (uint32_t n = 0; n < 4 * hd[o]; ++n, ++col) {
                    const C y = val(sp.codes[2 * col]) * val(sp.codes[2 * col + 1]);
                    for (int r = 0; r < R; ++r)
                        acc[r] += C(sp.coef[2 * (R * col + r)], sp.coef[2 * (R * col + r) + 1]) * y;
                }
                for (int r = 0; r < R; ++r) wt[r] += acc[r] * (o == 1 ? 0.5 : o == 2 ? 1.0 / 6.0 : 1.0 / 3.0);
            }
            for (int r = 0; r < R; ++r) {
                if (hd[4 + r] == ~0u) continue;
                const uint32_t cls = hd[4 + 2 * R + r];
                q[cls] += val(hd[4 + R + r]) * (forces ? wt[r] : acc[r]);
                if (forces) g[(size_t)sp.slot_k[hd[4 + r]] * 3 + (size_t)sp.slot_cls[hd[4 + r]]] += acc[r];
            }
        }
    for (int n : seen)
        if (n != 1) return -1;
    for (int i = 0; i < 3; ++i) {
        Q[2 * i] = q[(size_t)i].real();
        Q[2 * i + 1] = q[(size_t)i].imag();
    }
    for (size_t i = 0; forces && i < g.size(); ++i) {
        G[2 * i] = g[i].real();
        G[2 * i + 1] = g[i].imag();
    }
    return 0;
}

// The class vectors u[3][3] (re, im) of a class-split pack and the constant
// term e0[3], for checks against the polynomials.
extern "C" int acehost_class(const ace_pack* pk, const double* c, double* u, double* e0) {
    if (!acehost::validate_pack(pk).empty() || !pk->classed) return -1;
    const acehost::PackCopy pc = acehost::copy_pack(pk);
    const acehost::Coeffs cf = acehost::coefficients(pc, c);
    for (int i = 0; i < 3; ++i)
        for (int q = 0; q < 6; ++q) u[6 * i + q] = pc.cv.u[i][q];
    for (int q = 0; q < 3; ++q) e0[q] = cf.e0[2 * q];
    return 0;
}

// Calls of sizes[n], those with captured[i] set recorded in a graph: how many
// of the blocks that the graphs point to are live after the last call, of how
// many graphs; *blocks the blocks alive then, *left those alive once the
// buffer is gone.
namespace {
struct CheckMemory {
    static std::set<void*>& live() {
        static std::set<void*> s;
        return s;
    }
    static int alloc(void** p, size_t bytes) {
        live().insert(*p = new char[bytes]);
        return 0;
    }
    static void release(void* p) {
        live().erase(p);
        delete[] static_cast<char*>(p);
    }
};
}  // namespace
extern "C" int acehost_grow_buf(const int64_t* sizes, const int32_t* captured, int n, int* graphs, int* blocks,
                                int* left) {
    int ok = 0;
    {
        acehost::GrowBuf<double, CheckMemory> buf;
        std::vector<void*> used;
        for (int i = 0; i < n; ++i) {
            if (buf.ensure((size_t)sizes[i], captured[i] != 0)) return -1;
            if (captured[i]) used.push_back(buf.p);
        }
        for (void* p : used) ok += CheckMemory::live().count(p) ? 1 : 0;
        *graphs = (int)used.size();
        *blocks = (int)CheckMemory::live().size();
    }
    *left = (int)CheckMemory::live().size();
    return ok;
}

extern "C" int64_t acehost_choose_tail(int64_t ntile, int P, int ncu, double d, double dh) {
    return acehost::choose_tail(ntile, P, ncu, d, dh);
}

// What the pair kernel (classed packs: the slot kernel) executes per
// environment: FP64 operations, LDS bytes; and the columns of all panels, the
// panels, the rows of all panels (slots: steps, pieces, rows).
extern "C" int acehost_dag_work(const ace_pack* pk, int forces, double* out) {
    if (!acehost::validate_pack(pk).empty()) return -1;
    const acehost::PackCopy pc = acehost::copy_pack(pk);
    const int np = pk->npool;
    const std::vector<int32_t> pool(pk->pool, pk->pool + 4 * (size_t)np);
    if (pk->classed) {
        acehost::SlotProgram sp;
        if (!acehost::slot_program(pc, pool, std::vector<int32_t>(pk->gslot_ptr, pk->gslot_ptr + np + 1),
                                   std::vector<int32_t>(pk->gslot_list, pk->gslot_list + pk->gslot_ptr[np]),
                                   std::vector<int32_t>(pk->gslot_class, pk->gslot_class + pk->ngslots), forces != 0, sp)
                 .empty())
            return 1;
        const acehost::SlotWork w = acehost::slot_work(sp, forces != 0);
        out[0] = w.flops;
        out[1] = w.lds;
        out[2] = (double)(sp.codes.size() / 8 - 3);
        out[3] = sp.pieces();
        out[4] = forces ? sp.nslots : 0;
        return 0;
    }
    acehost::PairForm pf;
    acehost::PairProgram pp;
    if (!acehost::pair_form(pc, pool, 159, pf).empty() ||
        !acehost::pair_program(pf, forces != 0, forces ? 1024 : 512, np, 96, pp).empty())
        return 1;
    const acehost::DagWork w = acehost::pair_work(pp, forces != 0, 1.0);
    out[0] = w.flops;
    out[1] = w.lds;
    out[2] = (double)(pp.coef.size() - 64) / acehost::PAIR_ROWS;
    out[3] = (double)std::count_if(pp.panel.begin(), pp.panel.end(), [](int32_t p) { return p >= 0; });
    out[4] = (double)pf.virt.size();
    return 0;
}
