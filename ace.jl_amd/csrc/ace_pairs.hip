// libacehip.so, pair kernel: site energies and the adjoint G of Invariant
// bases of correlation order 3 to 7 (evaluator.jl:121-185 restated on A+) as a
// quadratic form in the products of two pooled values; the programs are
// compiled by pairs_host.hpp, whose head states the form.
#include "ace_common.hpp"

namespace {

struct PairArgs {
    const uint32_t* words;
    const double* coef;
    const int32_t* seq;  // the parts of the first ntile_lo tiles: their rounds
    const int32_t* seq_hi;  // and those of the tail tiles, parts + 1 workgroups each
    int32_t seq_ptr[acehost::PAIR_MAXP + 1], seq_ptr_hi[acehost::PAIR_MAXP + 1];
    // products that are values of their own, and what they pass on
    const uint32_t* virt;
    const uint32_t* back;
    const int32_t* back_ptr;
    int npool, nvirt;
    int parts;
    int64_t ntile_lo;
};

// Program words are read through the constant address space: wave-uniform
// addresses, so LDS offsets arrive as scalar operands.
typedef const __attribute__((address_space(4))) uint32_t PairWord;
typedef const __attribute__((address_space(4))) int32_t PairInt;

__device__ __forceinline__ double xor_hi(double v, uint32_t m) {
    return __hiloint2double(__double2hiint(v) ^ (int)m, __double2loint(v));
}

// The value of the pair's even (re) or odd (im) lane in both lanes, or the
// other lane's value.
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
constexpr int DPP_RE = 0xA0, DPP_IM = 0xF5, DPP_SWAP = 0xB1;  // quad_perm 0,0,2,2 / 1,1,3,3 / 1,0,3,2

// h[row] += coefficient[row] x0 + coefficient[8 + row] x1, the coefficients in
// lanes 0..15 of every row of 16 lanes (c holds one each): a multiply-add takes
// its coefficient by a DPP row broadcast, so 16 of them cost one vector load
// and no scalar registers.  (Read as scalars, the coefficients were bound by
// the scalar cache's misses: k_pairs 2.33 ms at 100,000 order-4 environments,
// 1.41 ms with every scalar load a hit.)  The s_nop keeps two wait states
// between a vector write of c and the DPP reads.
__device__ __forceinline__ void fmac16(double (&h)[acehost::PAIR_ROWS], double c, double x0, double x1) {
    static_assert(acehost::PAIR_ROWS == 8, "16 coefficients are two columns");
#define ACE_B(N, X) "v_fmac_f64_dpp %" #N ", %8, %" #X " row_newbcast:"
#define ACE_E " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" ACE_B(0, 9) "0" ACE_E ACE_B(1, 9) "1" ACE_E ACE_B(2, 9) "2" ACE_E ACE_B(3, 9) "3" ACE_E
            ACE_B(4, 9) "4" ACE_E ACE_B(5, 9) "5" ACE_E ACE_B(6, 9) "6" ACE_E ACE_B(7, 9) "7" ACE_E
                ACE_B(0, 10) "8" ACE_E ACE_B(1, 10) "9" ACE_E ACE_B(2, 10) "10" ACE_E ACE_B(3, 10) "11" ACE_E
                    ACE_B(4, 10) "12" ACE_E ACE_B(5, 10) "13" ACE_E ACE_B(6, 10) "14" ACE_E ACE_B(7, 10) "15" ACE_E
        : "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "+v"(h[4]), "+v"(h[5]), "+v"(h[6]), "+v"(h[7])
        : "v"(c), "v"(x0), "v"(x1));
}
__device__ __forceinline__ void fmac8(double (&h)[acehost::PAIR_ROWS], double c, double x0) {
    asm("s_nop 1\n\t" ACE_B(0, 9) "0" ACE_E ACE_B(1, 9) "1" ACE_E ACE_B(2, 9) "2" ACE_E ACE_B(3, 9) "3" ACE_E
            ACE_B(4, 9) "4" ACE_E ACE_B(5, 9) "5" ACE_E ACE_B(6, 9) "6" ACE_E ACE_B(7, 9) "7" ACE_E
        : "+v"(h[0]), "+v"(h[1]), "+v"(h[2]), "+v"(h[3]), "+v"(h[4]), "+v"(h[5]), "+v"(h[6]), "+v"(h[7])
        : "v"(c), "v"(x0));
#undef ACE_B
#undef ACE_E
}

// n records of NQ columns: x = X_shared A_other (own part of the complex
// product), h[row] += C[row][column] x.  cp: this lane's coefficient.  The
// next record's words and coefficients are loaded while this one is used (one
// record past the last is read and dropped).
template <int NQ>
__device__ __forceinline__ void pair_records(const char* a16, const char* own, const char* oth, uint32_t mim,
                                             PairWord*& w, const double*& cp, int n,
                                             double (&h)[acehost::PAIR_ROWS]) {
    constexpr int R = acehost::PAIR_ROWS, RW = acehost::pair_rec_words(NQ), NC = (NQ + 1) / 2;
    uint32_t o[RW];
    double c[NC];
#pragma unroll
    for (int q = 0; q < RW; ++q) o[q] = w[q];
#pragma unroll
    for (int q = 0; q < NC; ++q) c[q] = cp[2 * R * q];
    for (int i = 0; i < n; ++i) {
        w += RW;
        cp += R * NQ;
        uint32_t on[RW];
        double cn[NC];
#pragma unroll
        for (int q = 0; q < RW; ++q) on[q] = w[q];
#pragma unroll
        for (int q = 0; q < NC; ++q) cn[q] = cp[2 * R * q];
        // bit 0: the shared factor is conjugated.  re lanes: ar dr -+ ai di,
        // im lanes: ar di +- ai dr
        const double2 a = *reinterpret_cast<const double2*>(a16 + (o[0] & ~1u));
        const double ai = xor_hi(a.y, mim ^ (~o[0] << 31));
        double x[NQ];
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            x[q] = fma(ai, *reinterpret_cast<const double*>(oth + o[1 + q]),
                       a.x * *reinterpret_cast<const double*>(own + o[1 + q]));
        if (NQ == 1) {
            fmac8(h, c[0], x[0]);
        } else {
#pragma unroll
            for (int q = 0; q < NQ; q += 2) fmac16(h, c[q / 2], x[q], x[q + (NQ > 1)]);
        }
#pragma unroll
        for (int q = 0; q < RW; ++q) o[q] = on[q];
#pragma unroll
        for (int q = 0; q < NC; ++q) c[q] = cn[q];
    }
}

// A panel's contributions to G, kept until its turn.
struct PairSums {
    double t1[acehost::PAIR_ROWS], t2[acehost::PAIR_ROWS];
    uint32_t rw[2 * acehost::PAIR_ROWS];  // the rows' factors
    int turn;
};

// k_pairs: a workgroup of 16 waves holds 32 environments; lane = 2 (environment)
// + (0: real, 1: imaginary part), since every coefficient multiplies both parts
// alike.  LDS: A+ as [k][64 doubles], with forces each row followed by the 64
// of G[k] (one workgroup per CU at config sizes; 159 pooled values at most).
// Per round each wave evaluates one panel of up to 8 rows: the products x_q of
// its columns, h_p += S_pq x_q, then h_p X_d and h_p X_a per row, kept in
// registers until the panel's turn adds them to G.  Panels of one turn share no
// target and turns are separated by barriers, so each G[k] is summed in a
// fixed order.
//
// What bounds it: FP64 vector issue and the rounds' barriers.  Order 4, degree
// 12, Lmax 6 (139 pooled values, 3235 functions): 148,000 vector instructions
// per tile, 0.87 ms for 100,000 environments at full issue; measured 1.50 ms
// (the segment kernel's 677,000 per 64 environments and 2.6 times the LDS
// reads: 2.89 ms), of which 0.21 ms are the turns' LDS atomics, 0.1 ms loading
// A+ and storing G.  Energies alone need no turns: 0.51 ms (0.79 ms).  Columns
// per panel and rows per panel: 8 rows keep 64 % of the coefficients nonzero;
// 16 rows 47 %, more multiply-adds on zeros than products saved.
// Order 5, degree 10, Lmax 4 (84 pooled values and 38 products of their own):
// 0.394 ms for 30,000 environments; with each monomial's five factors
// multiplied out in the segment kernel, 0.973 ms.
template <bool FORCES>
__global__ __launch_bounds__(1024) void k_pairs(PairArgs a, int64_t nenv, const double* __restrict__ Aplus,
                                                int64_t estride, double* __restrict__ E_out,
                                                double* __restrict__ Gbuf, const double* __restrict__ e0p) {
    constexpr int R = acehost::PAIR_ROWS, NW = acehost::PAIR_WAVES;
    constexpr int RB = FORCES ? 1024 : 512;  // LDS bytes per pooled value
    extern __shared__ char lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t blo = a.ntile_lo * a.parts;
    const bool tail = (int64_t)blockIdx.x >= blo;
    const int P = tail ? a.parts + 1 : a.parts;
    const int64_t bt = tail ? (int64_t)blockIdx.x - blo : xcd_env(blockIdx.x, blo);
    const int64_t tile = (tail ? a.ntile_lo : 0) + bt / P;
    const int part = (int)(bt % P);
    const int64_t env0 = tile * 32;
    const bool valid = env0 + (lane >> 1) < nenv;
    char* const own = lds + 8 * lane;
    for (int k = wave; k < a.npool; k += NW) {
        *reinterpret_cast<double*>(own + k * RB) =
            valid ? __builtin_nontemporal_load(Aplus + 2 * ((int64_t)k * estride + env0) + lane) : 0.0;
        if (FORCES) *reinterpret_cast<double*>(own + k * RB + 512) = 0.0;
    }
    if (wave == 0) *reinterpret_cast<double*>(own + a.npool * RB) = (lane & 1) ? 0.0 : 1.0;  // the constant
    __syncthreads();

    const char* const a16 = lds + 16 * (lane >> 1);
    const char* const oth = lds + 8 * (lane ^ 1);
    const uint32_t mim = (uint32_t)lane << 31;  // sign bit in imaginary lanes
    // own part of (x.x + i x.y) X, X the value at o or its conjugate (cj: sign
    // bit set): re x.x X.re - x.y X.im, im x.x X.im + x.y X.re
    auto times = [&](double2 x, uint32_t o, uint32_t cj) {
        return fma(xor_hi(x.y, mim ^ 0x80000000u ^ (cj & ~mim)), *reinterpret_cast<const double*>(oth + o),
                   xor_hi(x.x, cj & mim) * *reinterpret_cast<const double*>(own + o));
    };
    if (a.nvirt > 0) {
        PairWord* const vw = (PairWord*)(uintptr_t)a.virt;
        for (int i = wave; i < a.nvirt; i += NW) {
            const uint32_t oa = vw[2 * i], od = vw[2 * i + 1];
            char* const to = own + (a.npool + 1 + i) * RB;
            *reinterpret_cast<double*>(to) = times(*reinterpret_cast<const double2*>(a16 + oa), od & ~1u, od << 31);
            if (FORCES) *reinterpret_cast<double*>(to + 512) = 0.0;
        }
        __syncthreads();
    }
    double e = 0.0;
    // one panel: h_p of its rows, then h_p X_d and h_p X_a per row (forces), and
    // its energy
    auto evaluate = [&](int po, PairSums& ps) {
        ps.turn = -1;
        if (po < 0) return;
        PairWord* const hd = (PairWord*)(uintptr_t)(a.words + po);
        const uint32_t cnt = hd[0];
        ps.turn = (int)(hd[1] >> 8);
        double h[R];
#pragma unroll
        for (int r = 0; r < R; ++r) h[r] = 0.0;
        PairWord* w = hd + acehost::PAIR_HDR;
        const double* cp = a.coef + hd[2] + (lane & 15);
        pair_records<4>(a16, own, oth, mim, w, cp, (int)(cnt & 1023u), h);
        pair_records<2>(a16, own, oth, mim, w, cp, (int)(cnt >> 10 & 1023u), h);
        pair_records<1>(a16, own, oth, mim, w, cp, (int)(cnt >> 20), h);
#pragma unroll
        for (int r = 0; r < 2 * R; ++r) ps.rw[r] = hd[4 + r];
        if (FORCES) {
            // g = hr - i hi; t1 = g X_d for G[a], t2 = g A_a for G[d],
            // conjugated where X_d is (cj); e = Re(g X_d A_a) over the pair
            double ao[R], ax[R], dow[R], dx[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t oa = ps.rw[2 * r], od = ps.rw[2 * r + 1] & ~1u;
                ao[r] = *reinterpret_cast<const double*>(own + oa);
                ax[r] = *reinterpret_cast<const double*>(oth + oa);
                dow[r] = *reinterpret_cast<const double*>(own + od);
                dx[r] = *reinterpret_cast<const double*>(oth + od);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t cj = ps.rw[2 * r + 1] << 31;
                const double hr = dpp<DPP_RE>(h[r]), hi = xor_hi(dpp<DPP_IM>(h[r]), mim);
                ps.t1[r] = xor_hi(fma(xor_hi(hi, cj), dx[r], hr * dow[r]), cj & mim);
                ps.t2[r] = xor_hi(fma(hi, ax[r], hr * ao[r]), cj & mim);
                e = fma(ps.t1[r], ao[r], e);
            }
        } else {
            // e = hr re(x) + hi im(x)
            double2 av[R];
            double dow[R], dx[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const uint32_t od = ps.rw[2 * r + 1] & ~1u;
                av[r] = *reinterpret_cast<const double2*>(a16 + ps.rw[2 * r]);
                dow[r] = *reinterpret_cast<const double*>(own + od);
                dx[r] = *reinterpret_cast<const double*>(oth + od);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                // d conjugated: re ar dr + ai di, im ai dr - ar di
                const uint32_t cj = ps.rw[2 * r + 1] << 31;
                const double ar = xor_hi(av[r].x, cj & mim);
                const double ai = xor_hi(av[r].y, cj ? 0u : mim ^ 0x80000000u);
                e = fma(h[r], fma(ai, dx[r], ar * dow[r]), e);
            }
        }
    };
    // a panel's sums into G (the constant's row takes what nobody reads, so
    // that no row needs a branch)
    auto scatter = [&](PairSums& ps) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            __hip_atomic_fetch_add(reinterpret_cast<double*>(own + ps.rw[2 * r] + 512), ps.t1[r], __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
            __hip_atomic_fetch_add(reinterpret_cast<double*>(own + (ps.rw[2 * r + 1] & ~1u) + 512), ps.t2[r],
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    };
    // the part's rounds; the next round's panels are looked up ahead
    PairInt* ps = (PairInt*)(uintptr_t)(tail ? a.seq_hi : a.seq) + (tail ? a.seq_ptr_hi : a.seq_ptr)[part];
    const int nround = ps[0];
    ++ps;
    int po = ps[1 + wave], nt = ps[0];
    for (int ri = 0; ri < nround; ++ri) {
        ps += acehost::PAIR_SEQ;
        const int ntn = ps[0], pn = ps[1 + wave];
        PairSums sums;
        evaluate(po, sums);
        if (FORCES) {
            // the panel's turn: nt barriers in all, its sums after turn + 1 of them
            const int pre = sums.turn >= 0 ? sums.turn + 1 : nt;
            for (int s = 0; s < pre; ++s) __syncthreads();
            if (sums.turn >= 0) scatter(sums);
            for (int s = pre; s < nt; ++s) __syncthreads();
        }
        nt = ntn;
        po = pn;
    }
    __syncthreads();
    if (FORCES) {
        PairInt* const bp = (PairInt*)(uintptr_t)a.back_ptr;
        PairWord* const bw = (PairWord*)(uintptr_t)a.back;
        for (int k = wave; k < a.npool; k += NW) {
            double g = *reinterpret_cast<const double*>(own + k * RB + 512);
            if (a.nvirt > 0)
                for (int i = bp[k]; i < bp[k + 1]; ++i) {
                    const uint32_t o = bw[2 * i + 1];
                    const double2 gu = *reinterpret_cast<const double2*>(a16 + bw[2 * i] + 512);
                    const double t = times(gu, o & ~3u, (o & acehost::PAIR_BACK_IN) << 31);
                    g += xor_hi(t, (o & acehost::PAIR_BACK_OUT ? 0x80000000u : 0u) & mim);
                }
            if (valid)
                __builtin_nontemporal_store(g, Gbuf + 2 * (((int64_t)part * a.npool + k) * estride + env0) + lane);
        }
        if (a.nvirt > 0) __syncthreads();  // the A+ rows are read above and reused below
    }
    // energy: the waves' sums over the A+ rows, which nothing reads any more
    if (FORCES) e = xor_hi(e, mim);
    e += dpp<DPP_SWAP>(e);
    *reinterpret_cast<double*>(own + wave * RB) = e;
    __syncthreads();
    if (wave == 0 && valid && !(lane & 1) && E_out) {
        double s = 0.0;
        for (int w = 0; w < NW; ++w) s += *reinterpret_cast<const double*>(own + w * RB);
        if (FORCES) s *= 0.5;
        const int64_t env = env0 + (lane >> 1);
        if (a.parts > 1)
            E_out[(int64_t)part * estride + env] = s;  // this part's share, summed by k_esum
        else
            E_out[env] = *e0p + s;
    }
}

}  // namespace

// LDS bytes of a workgroup: the pooled values, the constant and the products
// of their own, at least one row per wave for the energy sums.
static size_t pair_lds(int npool, int nvirt, bool forces) {
    return (size_t)std::max(npool + 1 + nvirt, acehost::PAIR_WAVES) * (forces ? 1024 : 512);
}

int pairs_create(ace_ctx* ctx, const std::vector<int32_t>& pool) {
    ctx->pairs_ok = false;
    if (ctx->prop != ACE_PROP_INVARIANT || ctx->maxorder < 3 || ctx->npool > PAIR_MAX_POOL ||
        ctx->ngslots < ctx->npool)
        return 0;
    acehost::PairForm pf;
    if (!acehost::pair_form(ctx->host, pool, PAIR_MAX_POOL, pf).empty() || pf.entries.empty()) return 0;  // other kernels take it
    for (int m = 0; m < 2; ++m) {
        PairDev& d = ctx->pairs[m];
        const std::string err = acehost::pair_program(pf, m == 0, m == 0 ? 1024 : 512, ctx->npool, PAIR_CAP, d.host);
        if (!err.empty()) return set_err(err);
        if (d.words.upload(d.host.words.data(), d.host.words.size()) ||
            d.virt.upload(d.host.virt.data(), d.host.virt.size()) ||
            d.back.upload(d.host.back.data(), d.host.back.size()) ||
            d.back_ptr.upload(d.host.back_ptr.data(), d.host.back_ptr.size()))
            return -1;
        for (int P = 1; P <= acehost::PAIR_MAXP + 1; ++P)
            if (d.seq[P].upload(d.host.seq[P].data(), d.host.seq[P].size())) return -1;
    }
    ctx->pairs_ok = true;
    return 0;
}

int pairs_set_coeffs(ace_ctx* ctx, const std::vector<double>& leaf) {
    for (PairDev& d : ctx->pairs) {
        acehost::pair_coefs(d.host, leaf);
        if (d.coef.upload(d.host.coef.data(), d.host.coef.size())) return -1;
    }
    return 0;
}

int launch_pairs(ace_ctx* ctx, hipStream_t st, int64_t nenv, int64_t estride, bool forces, int P, int64_t nhi,
                 const Workspace& ws, double* E_out) {
    const PairDev& d = ctx->pairs[forces ? 0 : 1];
    const int64_t ntile = (nenv + 31) / 32, nblk = (ntile - nhi) * P + nhi * (P + 1);
    if (P < 1 || P > acehost::PAIR_MAXP || nblk >= ((int64_t)1 << 31)) return set_err("pair kernel: bad launch");
    PairArgs a;
    a.words = d.words.p;
    a.coef = d.coef.p;
    a.seq = d.seq[P].p;
    a.seq_hi = d.seq[P + 1].p;
    for (int q = 0; q < P; ++q) a.seq_ptr[q] = d.host.seq_ptr[P][(size_t)q];
    for (int q = 0; q < P + 1; ++q) a.seq_ptr_hi[q] = d.host.seq_ptr[P + 1][(size_t)q];
    a.virt = d.virt.p;
    a.back = d.back.p;
    a.back_ptr = d.back_ptr.p;
    a.npool = ctx->npool;
    a.nvirt = (int)d.host.virt.size() / 2;
    a.parts = P;
    a.ntile_lo = ntile - nhi;
    const size_t lds = pair_lds(ctx->npool, a.nvirt, forces);
    auto go = [&](auto kern) {
        if (set_func_lds((const void*)kern, lds)) return -1;
        hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(64 * acehost::PAIR_WAVES), lds, st, a, nenv,
                           reinterpret_cast<const double*>(ws.Aplus), estride, E_out,
                           reinterpret_cast<double*>(ws.Gbuf), ctx->e0v.p);
        HIP_TRY(hipGetLastError());
        return 0;
    };
    return forces ? go(k_pairs<true>) : go(k_pairs<false>);
}
