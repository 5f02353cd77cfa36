// libacehip.so, slot kernel: class values Q_c and the adjoint G of class-split
// EuclideanVector bases of correlation order <= 3 (evaluator.jl:121-185 on A+);
// the programs are compiled by slots_host.hpp, whose head states the form.
#include "ace_common.hpp"

namespace {

constexpr int SR = acehost::SLOT_ROWS, SNW = acehost::SLOT_WAVES;

struct SlotArgs {
    const uint32_t* hdr;
    const uint4* codes;
    const double* coef;
    // pieces of the first ntile_lo tiles' workgroups, parts of them a tile, and of
    // the others', parts_hi a tile
    const int32_t *list_ptr, *list, *list_ptr_hi, *list_hi;
    int npool, parts, parts_hi;
    int64_t ntile_lo;
};

typedef const __attribute__((address_space(4))) uint32_t SlotWord;
typedef const __attribute__((address_space(4))) int32_t SlotInt;

// acc[row] += C[row] y for one column, y = yr + i yi, ni = -yi: lanes 8 B .. 8 B + 7
// of every row of 16 lanes hold the column's coefficients (row, re / im) in c.
// The s_nop keeps two wait states between a vector write of c and the DPP reads.
template <int B>
__device__ __forceinline__ void slot_fmac(double (&ar)[SR], double (&ai)[SR], double c, double yr, double yi, double ni) {
    static_assert(SR == 4, "8 coefficients per column");
#define ACE_S(D, X, N) "v_fmac_f64_dpp %" #D ", %8, %" #X " row_newbcast:%c" #N " row_mask:0xf bank_mask:0xf\n\t"
    asm("s_nop 1\n\t" ACE_S(0, 9, 12) ACE_S(4, 10, 12) ACE_S(1, 9, 14) ACE_S(5, 10, 14) ACE_S(2, 9, 16) ACE_S(6, 10, 16)
            ACE_S(3, 9, 18) ACE_S(7, 10, 18) ACE_S(0, 11, 13) ACE_S(4, 9, 13) ACE_S(1, 11, 15) ACE_S(5, 9, 15)
                ACE_S(2, 11, 17) ACE_S(6, 9, 17) ACE_S(3, 11, 19) ACE_S(7, 9, 19)
        : "+v"(ar[0]), "+v"(ar[1]), "+v"(ar[2]), "+v"(ar[3]), "+v"(ai[0]), "+v"(ai[1]), "+v"(ai[2]), "+v"(ai[3])
        : "v"(c), "v"(yr), "v"(yi), "v"(ni), "i"(8 * B), "i"(8 * B + 1), "i"(8 * B + 2), "i"(8 * B + 3),
          "i"(8 * B + 4), "i"(8 * B + 5), "i"(8 * B + 6), "i"(8 * B + 7));
#undef ACE_S
}

__device__ __forceinline__ double slot_xor(double v, uint32_t m) {
    return __hiloint2double(__double2hiint(v) ^ (int)m, __double2loint(v));
}

// A + i B of both half-waves: re in lanes 0-31, im in lanes 32-63.
__device__ __forceinline__ double slot_halves(double a, double b) {
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a), (unsigned)__double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a), (unsigned)__double2hiint(b), false, false);
    return __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
}

// k_slots: a workgroup of 16 waves holds A+ of 32 environments in LDS; lane =
// environment, the half-waves take different columns of a piece.  Per step a
// half-wave forms two products of two pooled values and multiplies them into
// the piece's 4 slots, whose sums stay in registers; each slot belongs to one
// wave, so G is stored straight from them, without LDS sums or barriers.
// Bound by FP64 vector issue: 4 multiply-adds per complex coefficient (the
// basis functions' phases are arbitrary), 90 % of them nonzero with 4 slots
// per panel (8: 70 %, fewer products but as many clocks).  Two species, order 3,
// degree 10 (220 pooled values, 5,408 functions): 7,700 steps of some 250 clocks
// of a SIMD per tile, 0.20 ms at full issue; measured 0.27 ms per tile and
// compute unit, 0.283 ms for 8,192 environments against the segment kernel's
// 0.611 (all factors multiplied out per slot, two leaves at a time), 64
// environments 0.046 against 0.186; energies alone 0.112 against 0.207.
template <bool FORCES>
__global__ __launch_bounds__(64 * SNW) void k_slots(SlotArgs a, int64_t nenv, const double2* __restrict__ Aplus,
                                                    int64_t estride, double* __restrict__ Epart,
                                                    double* __restrict__ Gbuf) {
    extern __shared__ double2 tilebuf[];
    const int lane = threadIdx.x & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int64_t blo = a.ntile_lo * a.parts;
    const bool tail = (int64_t)blockIdx.x >= blo;
    const int P = tail ? a.parts_hi : a.parts;
    const int64_t bt = tail ? (int64_t)blockIdx.x - blo : xcd_env(blockIdx.x, blo);
    const int64_t env0 = ((tail ? a.ntile_lo : 0) + bt / P) * 32;
    const int part = (int)(bt % P);
    for (int i = threadIdx.x; i < a.npool * 32; i += 64 * SNW) {
        const int64_t env = env0 + i % 32;
        tilebuf[i] = env < nenv ? Aplus[(int64_t)(i / 32) * estride + env] : make_double2(0.0, 0.0);
    }
    if (threadIdx.x < 32) tilebuf[a.npool * 32 + threadIdx.x] = make_double2(1.0, 0.0);  // the constant
    __syncthreads();
    const int64_t env = env0 + (lane & 31);
    const bool valid = env < nenv;
    // a factor: half its row's offset, and the conjugation in the sign bit, so
    // that one shift-and-add is its address
    typedef double LdsPair __attribute__((ext_vector_type(2)));
    typedef const __attribute__((address_space(3))) LdsPair LdsValue;
    const uint32_t e16 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)tilebuf + (uint32_t)(lane & 31) * 16;
    auto value = [&](uint32_t code) {
        const LdsPair v = *(LdsValue*)(uintptr_t)((code << 1) + e16);
        return make_double2(v.x, slot_xor(v.y, code & 0x80000000u));
    };
    double qr[3] = {0.0, 0.0, 0.0}, qi[3] = {0.0, 0.0, 0.0};  // this lane's share of Q_c
    SlotInt* const lp = (SlotInt*)(uintptr_t)((tail ? a.list_ptr_hi : a.list_ptr) + part * SNW + wave);
    SlotInt* const list = (SlotInt*)(uintptr_t)(tail ? a.list_hi : a.list);
    const int l1 = lp[1];
    for (int li = lp[0]; li < l1; ++li) {
        SlotWord* const hd = (SlotWord*)(uintptr_t)a.hdr + (int64_t)list[li] * acehost::SLOT_HDR;
        const uint4* code = a.codes + 2 * (int64_t)hd[0] + half;
        const double* co = a.coef + 8 * SR * (int64_t)hd[0] + 4 * SR * half + (lane & 15);
        double ar[SR] = {0.0, 0.0, 0.0, 0.0}, ai[SR] = {0.0, 0.0, 0.0, 0.0};
        double wr[SR] = {0.0, 0.0, 0.0, 0.0}, wi[SR] = {0.0, 0.0, 0.0, 0.0};
        // steps are read two ahead, over the orders' ends
        uint4 ka = code[0], kb = code[2];
        double ca = co[0], cb = co[8 * SR];
        auto step = [&](const uint4& k, double c) {
            const double2 f0 = value(k.x), g0 = value(k.y), f1 = value(k.z), g1 = value(k.w);
            const double2 y0 = cmul(f0, g0), y1 = cmul(f1, g1);
            slot_fmac<0>(ar, ai, c, y0.x, y0.y, -y0.y);
            slot_fmac<1>(ar, ai, c, y1.x, y1.y, -y1.y);
        };
#pragma unroll
        for (int o = 0; o < 3; ++o) {
            const int n = (int)hd[1 + o];
            for (int s = 0; s + 1 < n; s += 2) {
                step(ka, ca);
                code += 4;
                co += 16 * SR;
                ka = code[0];
                ca = co[0];
                step(kb, cb);
                kb = code[2];
                cb = co[8 * SR];
            }
            if (n & 1) {
                step(ka, ca);
                code += 2;
                co += 8 * SR;
                ka = kb;
                ca = cb;
                kb = code[2];
                cb = co[8 * SR];
            }
            if (FORCES) {
                // sum_o G_o / o: 1/2, 1/6, 1/3 of the sums up to order 1, 2, 3
                const double t = o == 0 ? 0.5 : o == 1 ? 1.0 / 6.0 : 1.0 / 3.0;
#pragma unroll
                for (int r = 0; r < SR; ++r) {
                    wr[r] = fma(t, ar[r], wr[r]);
                    wi[r] = fma(t, ai[r], wi[r]);
                }
            }
        }
#pragma unroll
        for (int r = 0; r < SR; ++r) {
            const uint32_t slot = hd[4 + r];
            if (slot == ~0u) continue;
            const double2 x = value(hd[4 + SR + r]);
            const double vr = FORCES ? wr[r] : ar[r], vi = FORCES ? wi[r] : ai[r];
            const double er = x.x * vr - x.y * vi, ei = x.x * vi + x.y * vr;
            const uint32_t cls = hd[4 + 2 * SR + r];
#pragma unroll
            for (int q = 0; q < 3; ++q)
                if (cls == (uint32_t)q) {
                    qr[q] += er;
                    qi[q] += ei;
                }
            if (FORCES) {
                const double g = slot_halves(ar[r], ai[r]);
                if (valid) __builtin_nontemporal_store(g, Gbuf + 2 * ((int64_t)slot * estride + env) + half);
            }
        }
    }
    // the waves' class values over the tile, which nothing reads any more
    __syncthreads();
    double* red = reinterpret_cast<double*>(tilebuf);  // [wave][class][re / im][32]
#pragma unroll
    for (int q = 0; q < 3; ++q) red[((wave * 3 + q) * 2 + half) * 32 + (lane & 31)] = slot_halves(qr[q], qi[q]);
    __syncthreads();
    const int q = threadIdx.x / 32;
    if (q < 6 && env0 + threadIdx.x % 32 < nenv) {
        double s = 0.0;
        for (int w = 0; w < SNW; ++w) s += red[(w * 6 + q) * 32 + threadIdx.x % 32];
        Epart[((int64_t)part * 6 + q) * estride + env0 + threadIdx.x % 32] = s;
    }
}

}  // namespace

int slots_create(ace_ctx* ctx, const ace_pack* pk) {
    ctx->slots_ok = false;
    if (!ctx->classed || ctx->maxorder > 3 || ctx->npool > acehost::SLOT_MAX_POOL) return 0;
    const std::vector<int32_t> pool(pk->pool, pk->pool + 4 * (size_t)pk->npool),
        ptr(pk->gslot_ptr, pk->gslot_ptr + pk->npool + 1), list(pk->gslot_list, pk->gslot_list + ptr.back()),
        cls(pk->gslot_class, pk->gslot_class + pk->ngslots);
    for (int m = 0; m < 2; ++m) {
        SlotDev& d = ctx->slots[m];
        if (!acehost::slot_program(ctx->host, pool, ptr, list, cls, m == 0, d.host).empty()) return 0;  // other kernels take it
        if (d.hdr.upload(d.host.hdr.data(), d.host.hdr.size()) || d.codes.upload(d.host.codes.data(), d.host.codes.size()))
            return -1;
        for (int P = 1; P <= acehost::SLOT_MAXP; ++P)
            if (d.list_ptr[P].upload(d.host.list_ptr[P].data(), d.host.list_ptr[P].size()) ||
                d.list[P].upload(d.host.list[P].data(), d.host.list[P].size()))
                return -1;
    }
    // the force kernel's table: the slots of each pooled value
    const acehost::SlotProgram& sp = ctx->slots[0].host;
    std::vector<int32_t> gp(1, 0), gl;
    for (int k = 0; k < ctx->npool; ++k) {
        for (int s = 0; s < sp.nslots; ++s)
            if (sp.slot_k[(size_t)s] == k) gl.push_back(s);
        gp.push_back((int32_t)gl.size());
    }
    if (ctx->slot_ptr.upload(gp.data(), gp.size()) || ctx->slot_list.upload(gl.data(), gl.size()) ||
        ctx->slot_cls.upload(sp.slot_cls.data(), sp.slot_cls.size()))
        return -1;
    ctx->slots_ok = true;
    return 0;
}

int slots_set_coeffs(ace_ctx* ctx, const acehost::Coeffs& cf) {
    for (SlotDev& d : ctx->slots) {
        acehost::slot_coefs(d.host, cf);
        if (d.coef.upload(d.host.coef.data(), d.host.coef.size())) return -1;
    }
    return 0;
}

static size_t slot_lds(int npool) {
    return std::max((size_t)(npool + 1) * 32 * sizeof(double2), (size_t)SNW * 6 * 32 * sizeof(double));
}

acehost::SlotShape slot_shape(const ace_ctx* ctx, int64_t nenv, bool forces) {
    const int per_cu = 2 * slot_lds(ctx->npool) <= 160 * 1024 ? 2 : 1;
    return acehost::slot_shape(ctx->slots[forces ? 0 : 1].host, (nenv + 31) / 32, ctx->ncu, per_cu);
}

int launch_slots(ace_ctx* ctx, hipStream_t st, int64_t nenv, int64_t estride, bool forces, const acehost::SlotShape& sh,
                 const Workspace& ws) {
    const SlotDev& d = ctx->slots[forces ? 0 : 1];
    const int64_t ntile = (nenv + 31) / 32, nblk = (ntile - sh.nhi) * sh.P + sh.nhi * sh.P_hi;
    if (sh.P < 1 || sh.P > sh.P_hi || sh.P_hi > acehost::SLOT_MAXP || sh.nhi < 0 || sh.nhi > ntile || nblk >= ((int64_t)1 << 31)) return set_err("slot kernel: bad launch");
    SlotArgs a;
    a.hdr = d.hdr.p;
    a.codes = reinterpret_cast<const uint4*>(d.codes.p);
    a.coef = d.coef.p;
    a.list_ptr = d.list_ptr[sh.P].p;
    a.list = d.list[sh.P].p;
    a.list_ptr_hi = d.list_ptr[sh.P_hi].p;
    a.list_hi = d.list[sh.P_hi].p;
    a.npool = ctx->npool;
    a.parts = sh.P;
    a.parts_hi = sh.P_hi;
    a.ntile_lo = ntile - sh.nhi;
    const size_t lds = slot_lds(ctx->npool);
    auto go = [&](auto kern) {
        if (set_func_lds((const void*)kern, lds)) return -1;
        hipLaunchKernelGGL(kern, dim3((unsigned)nblk), dim3(64 * SNW), lds, st, a, nenv, (const double2*)ws.Aplus,
                           estride, ws.Epart, reinterpret_cast<double*>(ws.Gbuf));
        HIP_TRY(hipGetLastError());
        return 0;
    };
    return forces ? go(k_slots<true>) : go(k_slots<false>);
}
