// libacehip.so, basis level: Product1pBasis A (product_1pbasis.jl:123-134),
// PIBasis AA (pibasis.jl:265-275), SymmetricBasis B = A2B AA
// (symmbasis.jl:248-315) and their derivatives dB (pibasis.jl:338-432,
// symmbasis.jl:322-336), and adjoint_EVAL_D (evaluator.jl:204-244): the calls
// behind grad_params and the least-squares design matrices.
#include "ace_common.hpp"

// ---------------------------------------------------------------------------
// basis level: A (full), AA, B, dB

__global__ void k_expandA(int64_t nenv, int nA, const int32_t* __restrict__ fid,
                          const double* __restrict__ sgn, const double2* __restrict__ Aplus,
                          int64_t estride, double2* __restrict__ A_out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nenv * nA) return;
    const int64_t env = i / nA;
    const int iA = (int)(i % nA);
    const int f = fid[iA];
    double2 v = Aplus[(int64_t)(f & 0x7fff) * estride + env];
    if (f & ACE_CONJ) v.y = -v.y;
    v.x *= sgn[iA];
    v.y *= sgn[iA];
    A_out[i] = v;
}

// AA[env][iAA] = prod_t A[iAA2iA[iAA][t]], left to right (pibasis.jl:265-275)
__global__ void k_AA(int64_t nenv, int nA, int nAA, int maxord, const int32_t* __restrict__ orders,
                     const int32_t* __restrict__ iAA2iA, const double2* __restrict__ A,
                     double2* __restrict__ AA) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nenv * nAA) return;
    const int64_t env = i / nAA;
    const int r = (int)(i % nAA);
    const double2* Ae = A + env * nA;
    double2 aa = make_double2(1.0, 0.0);
    const int o = orders[r];
    for (int t = 0; t < o; ++t) aa = cmul(aa, Ae[iAA2iA[r * maxord + t]]);
    AA[i] = aa;
}

// B[env][b][p] = Re sum_{nz in row b} val * AA
template <int PROP>
__global__ void k_B(int64_t nenv, int nB, int nAA, const int32_t* __restrict__ rowptr,
                    const int32_t* __restrict__ cols, const double* __restrict__ vals,
                    const double2* __restrict__ AA, double* __restrict__ B) {
    constexpr int NC = PROP == 0 ? 1 : 3;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nenv * nB) return;
    const int64_t env = i / nB;
    const int b = (int)(i % nB);
    double s[NC];
#pragma unroll
    for (int p = 0; p < NC; ++p) s[p] = 0.0;
    for (int z = rowptr[b]; z < rowptr[b + 1]; ++z) {
        const double2 a = AA[env * nAA + cols[z]];
        if (PROP == 0) {
            s[0] += vals[z] * a.x;  // isrealAA: AA = real(prod A)
        } else {
#pragma unroll
            for (int p = 0; p < NC; ++p) s[p] += vals[6 * z + 2 * p] * a.x - vals[6 * z + 2 * p + 1] * a.y;
        }
    }
#pragma unroll
    for (int p = 0; p < NC; ++p) B[i * NC + p] = s[p];
}

// per-neighbour 1p gradients dphi[j][iA][3] (complex), product_1pbasis.jl:169-221:
// a thread per neighbour, blockIdx.y a share of `per` functions.  A thread's
// functions follow one another, so a small batch is bound by that chain and is split
// further: 4,536 neighbours, 139 functions 99 us in 71 waves, 25 in 1,278.
template <int L>
__global__ __launch_bounds__(64) void k_dphi(RadialParams rp, int64_t nnbr,
                                             const double* __restrict__ xyz,
                                             const int8_t* __restrict__ species,
                                             const int32_t* __restrict__ aspec4, int nA, int per,
                                             double2* __restrict__ dphi) {
    constexpr int NP = (L + 1) * (L + 2) / 2;
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nnbr) return;
    const double x = xyz[j], y = xyz[nnbr + j], z = xyz[2 * nnbr + j];
    const int mu = species ? (int)species[j] : -1;
    Sph S = cart2spher(x, y, z);
    double t, dtdr;
    transform_ed(rp, S.r, t, dtdr);
    double R[ACE_NRMAX], dR[ACE_NRMAX];
    R[0] = rp.A[0] * fcut(rp, t);
    dR[0] = rp.A[0] * fcut_d(rp, t);
    for (int n = 1; n < rp.nr && n < ACE_NRMAX; ++n) {
        const double al = rp.A[n] * t + rp.B[n];
        if (n == 1) {
            R[1] = al * R[0];
            dR[1] = al * dR[0] + rp.A[1] * R[0];
        } else {
            R[n] = al * R[n - 1] + rp.C[n] * R[n - 2];
            dR[n] = al * dR[n - 1] + rp.C[n] * dR[n - 2] + rp.A[n] * R[n - 1];
        }
    }
    double P[NP], dP[NP];
    alp_eval_ed<L>(rp, S, P, dP);
    const double rinv = 1.0 / (S.r + 2.220446049250313e-16);
    const double rh[3] = {x / S.r, y / S.r, z / S.r};
    const int i1 = min(nA, ((int)blockIdx.y + 1) * per);
    for (int iA = blockIdx.y * per; iA < i1; ++iA) {
        const int amu = aspec4[4 * iA], n = aspec4[4 * iA + 1] - 1, l = aspec4[4 * iA + 2],
                  mm = aspec4[4 * iA + 3];
        double2* out = dphi + (j * nA + iA) * 3;
        if (amu >= 0 && amu != mu) {
            for (int d = 0; d < 3; ++d) out[d] = make_double2(0.0, 0.0);
            continue;
        }
        const int m = mm < 0 ? -mm : mm;
        // e^{i m phi}/sqrt2
        double epr = 0.7071067811865475, epi = 0.0;
        for (int q = 0; q < m; ++q) {
            const double a = epr * S.cphi - epi * S.sphi;
            const double b = epr * S.sphi + epi * S.cphi;
            epr = a;
            epi = b;
        }
        double pds = 0.0, dpt = 0.0;
        for (int ll = 0; ll <= L; ++ll)
            for (int q = 0; q <= ll; ++q)
                if (ll == l && q == m) {
                    pds = P[idxp(ll, q)];
                    dpt = dP[idxp(ll, q)];
                }
        double Yr, Yi, fpr, fpi, ftr, fti;
        if (m == 0) {
            Yr = pds * 0.7071067811865475;
            Yi = 0.0;
            fpr = fpi = 0.0;
            ftr = dpt * 0.7071067811865475;
            fti = 0.0;
        } else {
            Yr = epr * pds * S.sth;
            Yi = epi * pds * S.sth;
            fpr = -m * epi * pds;
            fpi = m * epr * pds;
            ftr = epr * dpt;
            fti = epi * dpt;
        }
        if (mm < 0) {  // Y_l^-m = (-1)^m conj(Y_l^m), same for the gradient
            const double s = (m & 1) ? -1.0 : 1.0;
            Yr *= s;
            Yi *= -s;
            fpr *= s;
            fpi *= -s;
            ftr *= s;
            fti *= -s;
        }
        const double dYr[3] = {(-S.sphi * fpr + S.cphi * S.cth * ftr) * rinv,
                               (S.cphi * fpr + S.sphi * S.cth * ftr) * rinv,
                               (-S.sth * ftr) * rinv};
        const double dYi[3] = {(-S.sphi * fpi + S.cphi * S.cth * fti) * rinv,
                               (S.cphi * fpi + S.sphi * S.cth * fti) * rinv,
                               (-S.sth * fti) * rinv};
        const double Rv = R[n], dRv = dR[n] * dtdr;
        for (int d = 0; d < 3; ++d)
            out[d] = make_double2(dRv * rh[d] * Yr + Rv * dYr[d], dRv * rh[d] * Yi + Rv * dYi[d]);
    }
}


// dAAw[env][iAA] = sum_t dAw_t prod_{s != t} A_s by a left-to-right dual
// product (p, dp) <- (p a, dp a + p da) (evaluator.jl:225-235).
__global__ void k_AAdir(int64_t nenv, int nA, int nAA, int maxord, const int32_t* __restrict__ orders,
                        const int32_t* __restrict__ iAA2iA, const double2* __restrict__ A,
                        const double2* __restrict__ dA, double2* __restrict__ dAA) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nenv * nAA) return;
    const int64_t env = i / nAA;
    const int r = (int)(i % nAA);
    const double2* Ae = A + env * nA;
    const double2* dAe = dA + env * nA;
    double2 p = make_double2(1.0, 0.0), dp = make_double2(0.0, 0.0);
    const int o = orders[r];
    for (int t = 0; t < o; ++t) {
        const int v = iAA2iA[r * maxord + t];
        const double2 a = Ae[v], da = dAe[v];
        const double2 x = cmul(dp, a), y = cmul(p, da);
        dp = make_double2(x.x + y.x, x.y + y.y);
        p = cmul(p, a);
    }
    dAA[i] = dp;
}



// Factor f of the staged tile, conjugated when f carries ACE_CONJ (the sign
// bit of the imaginary part flipped without a branch).
__device__ __forceinline__ double2 conj_if(double2 v, uint32_t sign) {
    return make_double2(v.x, __hiloint2double(__double2hiint(v.y) ^ (int)sign, __double2loint(v.y)));
}

template <int ENVS>
__device__ __forceinline__ double2 bt_factor(const double2* As, int f, int e) {
    return conj_if(As[(f & 0x7fff) * ENVS + e], (uint32_t)(f & ACE_CONJ) << 16);
}

// The records [za, zb) of one row whose AA columns have order O: each
// recomputes its product left to right from the staged tile, straight-line
// code, four records per iteration so that their scalar loads and LDS reads
// overlap.
template <int O, int ENVS>
__device__ __forceinline__ void bt_order(int za, int zb, const BtRec* __restrict__ recs,
                                         const double* __restrict__ vals, const double2* As, int e, double* s) {
#pragma unroll(4)
    for (int z = za; z < zb; ++z) {
        const BtRec r = recs[z];
        double2 p = make_double2(1.0, 0.0);
#pragma unroll
        for (int q = 0; q < O; ++q) p = cmul(p, bt_factor<ENVS>(As, r.f[q], e));
        const double sg = r.sgn;
#pragma unroll
        for (int q = 0; q < 3; ++q) s[q] += sg * (vals[6 * r.z + 2 * q] * p.x - vals[6 * r.z + 2 * q + 1] * p.y);
    }
}

// k_Bt: EuclideanVector basis values B = A2B . AA (pibasis.jl:265-275,
// symmbasis.jl:248-264) for a tile of ENVS environments, without
// materialising AA.  The pooled A+ tile is staged in LDS; every A2B nonzero
// (one BtRec, read with scalar loads) recomputes its AA product from it.  A
// row's nonzeros are ordered by the order of their AA column (rowo: where each
// order starts), one straight-line loop per order.  A workgroup is (tile,
// chunk of rows); each wave takes rpw consecutive rows (with ENVS = 32 the two
// half-waves take alternate rows).  Workgroups of one tile are consecutive on
// one XCD so the staged tile is read from that XCD's L2.
constexpr int BT_NW = 16;  // waves per k_Bt workgroup

template <int ENVS>
__global__ __launch_bounds__(64 * BT_NW) void k_Bt(int64_t nenv, int npool, int nB, int nchunk, int rpw,
                                            const int32_t* __restrict__ rowo, const BtRec* __restrict__ recs,
                                            const double* __restrict__ vals, const double2* __restrict__ Aplus,
                                            int64_t estride, double* __restrict__ out) {
    extern __shared__ double2 tilebuf[];
    double2* As = tilebuf;
    const int64_t ntile = (nenv + ENVS - 1) / ENVS;
    const int64_t lin = xcd_env(blockIdx.x, ntile * nchunk);
    const int64_t t = lin / nchunk;
    const int chunk = (int)(lin % nchunk);
    const int64_t e0 = t * ENVS;
    for (int i = threadIdx.x; i < npool * ENVS; i += 64 * BT_NW) {
        const int k = i / ENVS;
        const int64_t env = e0 + (i % ENVS);
        double2 v = make_double2(0.0, 0.0);
        if (env < nenv) v = Aplus[(int64_t)k * estride + env];
        As[i] = v;
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int e = lane % ENVS;
    const int half = ENVS == 32 ? (lane >> 5) : 0;
    const int64_t env = e0 + e;
    const int b0 = (chunk * BT_NW + wave) * rpw;
    const int b1 = min(b0 + rpw, nB);
    for (int b = b0 + half; b < b1; b += (ENVS == 32 ? 2 : 1)) {
        double s[3] = {0.0, 0.0, 0.0};
        const int32_t* ro = rowo + (int64_t)b * BT_ROWO;
        bt_order<0, ENVS>(ro[0], ro[1], recs, vals, As, e, s);
        bt_order<1, ENVS>(ro[1], ro[2], recs, vals, As, e, s);
        bt_order<2, ENVS>(ro[2], ro[3], recs, vals, As, e, s);
        bt_order<3, ENVS>(ro[3], ro[4], recs, vals, As, e, s);
        bt_order<4, ENVS>(ro[4], ro[5], recs, vals, As, e, s);
        if (env < nenv) {
#pragma unroll
            for (int q = 0; q < 3; ++q) out[(env * nB + b) * 3 + q] = s[q];
        }
    }
}

// n pairs of records of order O from r on (lanes 0-31 the first of a pair,
// lanes 32-63 the second).  `next` is the record read ahead: the stream runs on
// over the segments of a wave, so a record is in flight while one is used.
template <int O, bool DIR>
__device__ __forceinline__ void bv_run(int n, const uint4*& r, uint4& next, const char* tile, uint32_t e16, double& s) {
    constexpr int SH = DIR ? 10 : 9;  // a pooled value's row: 32 x A+, and 32 x dA+w
    for (int i = 0; i < n; ++i) {
        const uint4 q = next;
        r += 2;
        next = *r;
        const double c = __hiloint2double((int)q.w, (int)q.z);
        if (O == 0) {
            if (!DIR) s += c;
            continue;
        }
        double2 a[4], d[4];
#pragma unroll
        for (int t = 0; t < O; ++t) {
            const uint32_t w = t < 2 ? q.x : q.y;
            const char* at = tile + ((((t & 1 ? w >> 16 : w) & 0x1ffu) << SH) | e16);
            const uint32_t sign = (t & 1 ? w : w << 16) & 0x80000000u;
            a[t] = *reinterpret_cast<const double2*>(at);
            if (DIR) d[t] = *reinterpret_cast<const double2*>(at + 512);
            if (t > 0) {
                a[t] = conj_if(a[t], sign);
                if (DIR) d[t] = conj_if(d[t], sign);
            }
        }
        // products and their derivatives of the first two and the other factors
        double2 p = a[0], dp = d[0], u, du;
        if (O == 2) {
            u = a[1];
            if (DIR) du = d[1];
        } else if (O >= 3) {
            if (DIR) {
                const double2 x = cmul(d[0], a[1]), y = cmul(a[0], d[1]);
                dp = make_double2(x.x + y.x, x.y + y.y);
            }
            p = cmul(a[0], a[1]);
            u = a[2];
            if (DIR) du = d[2];
            if (O == 4) {
                if (DIR) {
                    const double2 x = cmul(d[2], a[3]), y = cmul(a[2], d[3]);
                    du = make_double2(x.x + y.x, x.y + y.y);
                }
                u = cmul(a[2], a[3]);
            }
        }
        if (O == 1)
            s += c * (DIR ? dp.x : p.x);
        else if (DIR)
            s += c * ((dp.x * u.x - dp.y * u.y) + (p.x * du.x - p.y * du.y));
        else
            s += c * (p.x * u.x - p.y * u.y);
    }
}

// k_Bv: Invariant basis values B = A2B . AA (DIR = false; pibasis.jl:265-275,
// symmbasis.jl:248-264) or their directional derivative A2B . dAA along
// per-neighbour weights (DIR = true; evaluator.jl:225-240), records and their
// order as basis_host.hpp lays them out.  Tiles of 32 environments staged in
// LDS (A+, with DIR dA+w beside it); lane = environment, the half-waves take
// alternate records.  Bound by the LDS reads (16 B per factor and environment,
// twice that with DIR), with the vector unit close behind, provided that the
// records arrive in time: they are vector loads, one record ahead.  Scalar
// loads, each waited for before its product's LDS reads, left a wave 0.75 us
// per record.  Rows are shared out by cost over the waves of nchunk
// workgroups per tile (bv_chunks), so that a batch of a few tiles still fills the chip.
// Measured with 3,235 functions of 139 pooled values, pooling included: 2,003
// environments 438 -> 112 us for values and 903 -> 210 us for derivatives, 108
// environments 317 -> 45 us, 20,000 environments 2.77 -> 0.88 ms and 6.17 ->
// 1.61 ms (one scalar-loaded record per A2B nonzero, 12 workgroups per tile of
// 64); with 97 functions of order 3, where pooling dominates, 20,000
// environments 66 -> 63 and 185 -> 151 us.
// Two rows are finished at a time: one swap of half-waves and one add sum
// both, and lanes 0-31 store the first, lanes 32-63 the second.
template <bool DIR>
__global__ __launch_bounds__(64 * acehost::BV_WAVES) void k_Bv(int64_t nenv, int npool, int nB, int nchunk,
                                                               const int2* __restrict__ seg,
                                                               const int2* __restrict__ unit,
                                                               const uint4* __restrict__ recs,
                                                               const double2* __restrict__ Aplus,
                                                               const double2* __restrict__ Wplus, int64_t estride,
                                                               double* __restrict__ out) {
    extern __shared__ double2 tilebuf[];
    const int64_t ntile = (nenv + 31) / 32;
    const int64_t lin = xcd_env(blockIdx.x, ntile * nchunk);
    const int64_t e0 = lin / nchunk * 32;
    const int chunk = (int)(lin % nchunk);
    for (int i = threadIdx.x; i < npool * 32; i += 64 * acehost::BV_WAVES) {
        const int k = i / 32;
        const int64_t env = e0 + i % 32;
        double2 v = make_double2(0.0, 0.0), w = make_double2(0.0, 0.0);
        if (env < nenv) {
            v = Aplus[(int64_t)k * estride + env];
            if (DIR) w = Wplus[(int64_t)k * estride + env];
        }
        double2* to = tilebuf + (DIR ? k * 64 : k * 32) + i % 32;
        to[0] = v;
        if (DIR) to[32] = w;
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63, half = lane >> 5;
    const int64_t env = e0 + (lane & 31);
    const char* tile = reinterpret_cast<const char*>(tilebuf);
    const uint32_t e16 = (uint32_t)(lane & 31) * 16;
    constexpr int UW = acehost::BV_UNITS / acehost::BV_WAVES;  // shares of a wave if one workgroup does a tile
    const int u = (chunk * acehost::BV_WAVES + wave) * (UW / nchunk);
    const int2 from = unit[u];
    const int s1 = unit[u + UW / nchunk].x;
    const uint4* r = recs + 2 * (int64_t)from.y + half;
    uint4 next = *r;
    int2 head = make_int2(0, 0);
    double s = 0.0, first = 0.0;
    int bfirst = -1;
    auto finish = [&](double x, double y, int bx, int by, bool both) {
        const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(x), (unsigned)__double2loint(y), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(x), (unsigned)__double2hiint(y), false, false);
        const double v = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
        if (env < nenv && (both || half == 0)) out[env * nB + (half ? by : bx)] = v;
    };
    for (int g = from.x; g < s1; ++g) {
        const int i = (g - from.x) & 63;
        if (i == 0) head = seg[min(g + lane, s1 - 1)];
        const int row = __builtin_amdgcn_readlane(head.x, i), nw = __builtin_amdgcn_readlane(head.y, i);
        const int n = nw & 0xfffffff;
        switch (nw >> 28) {
            case 4: bv_run<4, DIR>(n, r, next, tile, e16, s); break;
            case 3: bv_run<3, DIR>(n, r, next, tile, e16, s); break;
            case 2: bv_run<2, DIR>(n, r, next, tile, e16, s); break;
            case 1: bv_run<1, DIR>(n, r, next, tile, e16, s); break;
            default: bv_run<0, DIR>(n, r, next, tile, e16, s);
        }
        if (row < 0) {
            const int b = row & 0x7fffffff;
            if (bfirst < 0) {
                first = s;
                bfirst = b;
            } else {
                finish(first, s, bfirst, b, true);
                bfirst = -1;
            }
            s = 0.0;
        }
    }
    if (bfirst >= 0) finish(first, 0.0, bfirst, bfirst, false);
}

// dAA[j][iAA][3] = sum_a (prod_{t != a} A_t) dphi[j][v_a]  (pibasis.jl:402-432)
__global__ void k_dAA(int64_t nnbr, int nA, int nAA, int maxord, const int32_t* __restrict__ nbr_env,
                      const int32_t* __restrict__ orders, const int32_t* __restrict__ iAA2iA,
                      const double2* __restrict__ A, const double2* __restrict__ dphi,
                      double2* __restrict__ dAA) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnbr * nAA) return;
    const int64_t j = i / nAA;
    const int r = (int)(i % nAA);
    const int64_t env = nbr_env[j];
    const double2* Ae = A + env * nA;
    const int o = orders[r];
    double2 g[3] = {make_double2(0.0, 0.0), make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
    for (int a = 0; a < o; ++a) {
        double2 w = make_double2(1.0, 0.0);
        for (int t = 0; t < o; ++t)
            if (t != a) w = cmul(w, Ae[iAA2iA[r * maxord + t]]);
        const double2* dp = dphi + (j * nA + iAA2iA[r * maxord + a]) * 3;
        for (int d = 0; d < 3; ++d) {
            const double2 v = cmul(w, dp[d]);
            g[d].x += v.x;
            g[d].y += v.y;
        }
    }
    for (int d = 0; d < 3; ++d) dAA[(i * 3) + d] = g[d];
}

template <int PROP>
__global__ void k_dB(int64_t nnbr, int nB, int nAA, const int32_t* __restrict__ rowptr,
                     const int32_t* __restrict__ cols, const double* __restrict__ vals,
                     const double2* __restrict__ dAA, double* __restrict__ dB) {
    constexpr int NC = PROP == 0 ? 1 : 3;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nnbr * nB) return;
    const int64_t j = i / nB;
    const int b = (int)(i % nB);
    double s[NC][3];
#pragma unroll
    for (int p = 0; p < NC; ++p) s[p][0] = s[p][1] = s[p][2] = 0.0;
    for (int z = rowptr[b]; z < rowptr[b + 1]; ++z) {
        const double2* g = dAA + ((j * nAA) + cols[z]) * 3;
        for (int d = 0; d < 3; ++d) {
            if (PROP == 0) {
                s[0][d] += vals[z] * g[d].x;
            } else {
#pragma unroll
                for (int p = 0; p < NC; ++p)
                    s[p][d] += vals[6 * z + 2 * p] * g[d].x - vals[6 * z + 2 * p + 1] * g[d].y;
            }
        }
    }
#pragma unroll
    for (int p = 0; p < NC; ++p)
        for (int d = 0; d < 3; ++d) dB[(i * NC + p) * 3 + d] = s[p][d];
}

// k_dBw: per-neighbour basis gradients through per-environment adjoint
// weights (symmbasis.jl:322-336 with pibasis.jl:402-432 reorganised).
// dB[j][b] = Re sum_k W+[b][k] dphi+[j][k], where W+ collects, for every A2B
// entry z of row b and factor t of its AA column, the A2B value times the
// product of the other factors (prefix and suffix products) times the
// factors' signs, conjugated for conjugated (m < 0) factors, in the slot of
// the factor's pooled function.  One workgroup per (environment, chunk of up
// to 256 basis functions); thread = basis function.  W+ of the chunk lives in
// LDS, [slot][lane] per wave; the neighbours' pooled gradients dphi+ [npool][3]
// are staged DB_NJ at a time (as many as DB_STAGE double2 hold), the next stage
// loaded into registers while the current one is used.  Bound by the LDS reads of
// the gradients, three of 16 bytes per slot at each lane's own k (bank
// conflicts): 108 environments of 42 neighbours, 3,235 functions 481 -> 436 us
// with merged entries, functions ordered by loop length and stages that are
// really in flight (97 functions, with all launches 142 -> 101 us).  The weights are built once per
// workgroup, so a (environment, chunk) pair costs O(A2B entries x order) for
// the weights and O(neighbours x slots) for the gradients, instead of the
// dAA[neighbour][AA function] the materialising path writes.
struct DbArgs {
    const int4* wave;         // [nchunk][4]: first position, functions, first slot, first entry
    const int32_t* fn;        // [position] basis function
    const int2* cnt;          // [position] slots, entries
    const int32_t* chunk_s;   // [nchunk + 1]
    const int32_t* slot_k;
    const uint4* ztab;        // [entry][MO / 4]: factor and slot codes
    const double* vals;       // [entry] or [entry][6]
    int npool, nB;
};

constexpr int DB_NJ = DB_NJ_MAX;  // neighbours per stage (at most)
constexpr int DB_STAGE = 2048;    // double2 per stage (8 per thread)

// A barrier for LDS data alone: __syncthreads also waits for the workgroup's
// global loads and stores, here the next stage on its way in and the gradients
// on theirs out, once per neighbour.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

template <int PROP, int MO, int NPF>
__global__ __launch_bounds__(256) void k_dBw(DbArgs a, int64_t nenv, const int32_t* __restrict__ off,
                                             const double2* __restrict__ Aplus, int64_t estride,
                                             const double2* __restrict__ dphi, double* __restrict__ dB) {
    constexpr int NC = PROP == 0 ? 1 : 3;
    extern __shared__ double2 sm[];
    const int64_t env = blockIdx.x;
    const int c = blockIdx.y;
    const int tid = threadIdx.x;
    const int s0 = a.chunk_s[c], ns = a.chunk_s[c + 1] - s0;
    const int nq = 3 * a.npool;                           // double2 per neighbour
    const int njs = max(1, min(DB_NJ, DB_STAGE / nq));     // neighbours per stage
    double2* As = sm;                       // [npool]
    double2* dp = As + a.npool;             // [njs][npool][3]
    double2* W = dp + (size_t)njs * nq;     // [ns][NC]
    int* sk = reinterpret_cast<int*>(W + (size_t)ns * NC);  // [ns]
    for (int k = tid; k < a.npool; k += 256) As[k] = Aplus[(int64_t)k * estride + env];
    for (int q = tid; q < ns; q += 256) {
        sk[q] = a.slot_k[s0 + q];
#pragma unroll
        for (int p = 0; p < NC; ++p) W[q * NC + p] = make_double2(0.0, 0.0);
    }
    __syncthreads();
    const int4 wv = a.wave[4 * c + (tid >> 6)];
    const int lane = tid & 63, lanes = wv.y;
    const bool active = lane < lanes;
    const int2 n = active ? a.cnt[wv.x + lane] : make_int2(0, 0);
    const int b = active ? a.fn[wv.x + lane] : 0;
    const int sb = wv.z + lane;  // slot q of this function: sb + q lanes
    const int nsb = n.x;
    for (int z = 0; z < n.y; ++z) {
        const size_t e = (size_t)wv.w + (size_t)z * lanes + lane;
        uint32_t code[MO];
#pragma unroll
        for (int h = 0; h < MO / 4; ++h) {
            const uint4 w4 = a.ztab[e * (MO / 4) + h];
            code[4 * h] = w4.x;
            code[4 * h + 1] = w4.y;
            code[4 * h + 2] = w4.z;
            code[4 * h + 3] = w4.w;
        }
        double2 f[MO];
#pragma unroll
        for (int q = 0; q < MO; ++q) {
            f[q] = make_double2(1.0, 0.0);
            if (code[q] & (1u << 13)) {
                f[q] = As[code[q] & 0x3ffu];
                if (code[q] & 0x8000u) f[q].y = -f[q].y;
            }
        }
        double2 pre[MO];
        pre[0] = make_double2(1.0, 0.0);
#pragma unroll
        for (int q = 1; q < MO; ++q) pre[q] = cmul(pre[q - 1], f[q - 1]);
        double2 suf = make_double2(1.0, 0.0);
#pragma unroll
        for (int t = MO - 1; t >= 0; --t) {
            if (code[t] & (1u << 13)) {
                const double2 P = cmul(pre[t], suf);
                const uint32_t sc = code[t] >> 16;
                const bool cj = (sc & 0x8000u) != 0;
                double2* w = W + (size_t)(sb + (int)(sc & 0x7fffu) * lanes) * NC;
#pragma unroll
                for (int p = 0; p < NC; ++p) {
                    double2 v;
                    if (PROP == 0) {
                        const double cv = a.vals[e];
                        v = make_double2(cv * P.x, cv * P.y);
                    } else {
                        const double2 cv = make_double2(a.vals[6 * e + 2 * p], a.vals[6 * e + 2 * p + 1]);
                        v = cmul(cv, P);
                    }
                    w[p].x += v.x;
                    w[p].y += cj ? -v.y : v.y;
                }
                suf = cmul(suf, f[t]);
            }
        }
    }
    __syncthreads();
    const int j0 = off[env], j1 = off[env + 1];
    // stages of njs neighbours: their dphi+ rows are consecutive in memory, NPF
    // values per thread (unconditional loads: a branch around each made the
    // thread wait for it, and for the stores before it, at once)
    double2 pf[NPF];
    auto fetch = [&](int jb) {
        const int last = min(njs, j1 - jb) * nq - 1;
        const double2* src = dphi + (int64_t)jb * nq;
#pragma unroll
        for (int r = 0; r < NPF; ++r) pf[r] = src[min(tid + 256 * r, last)];
    };
    if (j0 < j1) fetch(j0);
    for (int jb = j0; jb < j1; jb += njs) {
        const int nj = min(njs, j1 - jb);
#pragma unroll
        for (int r = 0; r < NPF; ++r) {
            const int q = tid + 256 * r;
            if (q < nj * nq) dp[q] = pf[r];
        }
        lds_barrier();
        if (jb + njs < j1) fetch(jb + njs);  // in flight while this stage is used
        if (active) {
            for (int jj = 0; jj < nj; ++jj) {
                const double2* d = dp + (size_t)jj * nq;
                double acc[NC][3];
#pragma unroll
                for (int p = 0; p < NC; ++p) acc[p][0] = acc[p][1] = acc[p][2] = 0.0;
                for (int q = 0; q < nsb; ++q) {
                    const int k = sk[sb + q * lanes];
                    const double2 x0 = d[3 * k], x1 = d[3 * k + 1], x2 = d[3 * k + 2];
#pragma unroll
                    for (int p = 0; p < NC; ++p) {
                        const double2 w = W[(size_t)(sb + q * lanes) * NC + p];
                        acc[p][0] += w.x * x0.x - w.y * x0.y;
                        acc[p][1] += w.x * x1.x - w.y * x1.y;
                        acc[p][2] += w.x * x2.x - w.y * x2.y;
                    }
                }
                double* out = dB + ((int64_t)(jb + jj) * a.nB + b) * NC * 3;
#pragma unroll
                for (int p = 0; p < NC; ++p) {
                    out[3 * p] = acc[p][0];
                    out[3 * p + 1] = acc[p][1];
                    out[3 * p + 2] = acc[p][2];
                }
            }
        }
        lds_barrier();
    }
}

__global__ void k_nbr_env(int64_t nenv, const int32_t* __restrict__ off, int32_t* __restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= nenv) return;
    for (int j = off[e]; j < off[e + 1]; ++j) out[j] = (int32_t)e;
}

// ---- basis level

static int basis_A_internal(ace_ctx* ctx, int64_t nenv, const int32_t* off, const double* xyz,
                            const int8_t* species, int64_t nnbr, hipStream_t st) {
    const int64_t estride = ((nenv + 63) / 64) * 64;
    if (ctx->Aplus.ensure((size_t)ctx->npool * estride, ctx->capturing)) return -1;
    if (ctx->Afull.ensure((size_t)nenv * ctx->nA, ctx->capturing)) return -1;
    if (launch_pool_any(ctx, st, nenv, off, xyz, nnbr, species, estride, ctx_buffers(ctx), false)) return -1;
    const int64_t n = nenv * ctx->nA;
    hipLaunchKernelGGL(k_expandA, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nenv, ctx->nA,
                       ctx->aspec_fid.p, ctx->aspec_sgn.p, ctx->Aplus.p, estride, ctx->Afull.p);
    HIP_TRY(hipGetLastError());
    return 0;
}

extern "C" int ace_basis_A(ace_ctx* ctx, int64_t nenv, const int32_t* off, const double* xyz,
                           const int8_t* species, double* A_out, void* stream) {
    int64_t nnbr = 0;
    if (check_common(ctx, nenv, off, xyz, species, &nnbr, stream)) return -1;
    if (nenv == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    if (basis_A_internal(ctx, nenv, off, xyz, species, nnbr, st)) return -1;
    HIP_TRY(hipMemcpyAsync(A_out, ctx->Afull.p, sizeof(double2) * nenv * ctx->nA,
                           hipMemcpyDeviceToDevice, st));
    return 0;
}

static int basis_AA_internal(ace_ctx* ctx, int64_t nenv, hipStream_t st) {
    if (ctx->AA.ensure((size_t)nenv * ctx->nAA, ctx->capturing)) return -1;
    const int64_t n = nenv * ctx->nAA;
    hipLaunchKernelGGL(k_AA, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nenv, ctx->nA, ctx->nAA,
                       ctx->maxorder, ctx->orders.p, ctx->iAA2iA.p, ctx->Afull.p, ctx->AA.p);
    HIP_TRY(hipGetLastError());
    return 0;
}

__global__ void k_realpart(int64_t n, const double2* __restrict__ in, double* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = in[i].x;
}

extern "C" int ace_basis_AA(ace_ctx* ctx, int64_t nenv, const int32_t* off, const double* xyz,
                            const int8_t* species, double* AA_out, void* stream) {
    int64_t nnbr = 0;
    if (check_common(ctx, nenv, off, xyz, species, &nnbr, stream)) return -1;
    if (nenv == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    if (basis_A_internal(ctx, nenv, off, xyz, species, nnbr, st)) return -1;
    if (basis_AA_internal(ctx, nenv, st)) return -1;
    const int64_t n = nenv * ctx->nAA;
    if (ctx->prop == ACE_PROP_INVARIANT) {
        hipLaunchKernelGGL(k_realpart, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, ctx->AA.p, AA_out);
    } else {
        HIP_TRY(hipMemcpyAsync(AA_out, ctx->AA.p, sizeof(double2) * n, hipMemcpyDeviceToDevice, st));
    }
    HIP_TRY(hipGetLastError());
    return 0;
}

// Whether the fused kernels (k_Bv, k_Bt) take this basis: four factors per
// record, and the staged tile of 32 environments fits LDS (A+ alone up to 320
// pooled values, A+ and dA+w up to 160).
static bool bt_fits(const ace_ctx* ctx, bool dir) {
    return ctx->maxorder <= 4 && (size_t)ctx->npool * 32 * sizeof(double2) * (dir ? 2 : 1) <= 160 * 1024;
}

template <int ENVS>
static int launch_bt_shape(ace_ctx* ctx, hipStream_t st, int64_t nenv, int64_t estride, double* out) {
    const size_t lds = (size_t)ctx->npool * ENVS * sizeof(double2);
    constexpr int NW = BT_NW;
    const int rpw = std::max(1, (ctx->nB + NW * 12 - 1) / (NW * 12));
    const int nchunk = (ctx->nB + NW * rpw - 1) / (NW * rpw);
    const int64_t nblk = (nenv + ENVS - 1) / ENVS * nchunk;
    if (nblk >= ((int64_t)1 << 31)) return set_err("batch too large for one launch");
    set_func_lds((const void*)k_Bt<ENVS>, lds);
    hipLaunchKernelGGL(k_Bt<ENVS>, dim3((unsigned)nblk), dim3(64 * NW), lds, st, nenv, ctx->npool, ctx->nB, nchunk,
                       rpw, ctx->bt_rowo.p, ctx->bt_rec.p, ctx->vals.p, ctx->Aplus.p, estride, out);
    HIP_TRY(hipGetLastError());
    return 0;
}

template <bool DIR>
static int launch_bv(ace_ctx* ctx, hipStream_t st, int64_t nenv, int64_t estride, double* out) {
    if (ctx->nB == 0) return 0;
    const int64_t tiles = (nenv + 31) / 32;
    const size_t lds = (size_t)ctx->npool * 32 * sizeof(double2) * (DIR ? 2 : 1);
    const int resident = 2 * lds <= 160 * 1024 ? 2 : 1;  // 16 waves each
    const int nchunk = acehost::bv_chunks(ctx->bv_iter, ctx->bv_cost * (DIR ? 1.8 : 1.0), tiles, ctx->ncu, resident, (double)lds);
    if (tiles * nchunk >= ((int64_t)1 << 31)) return set_err("batch too large for one launch");
    set_func_lds((const void*)k_Bv<DIR>, lds);
    hipLaunchKernelGGL(k_Bv<DIR>, dim3((unsigned)(tiles * nchunk)), dim3(64 * acehost::BV_WAVES), lds, st, nenv,
                       ctx->npool, ctx->nB, nchunk, reinterpret_cast<const int2*>(ctx->bv_seg.p),
                       reinterpret_cast<const int2*>(ctx->bv_unit.p), reinterpret_cast<const uint4*>(ctx->bv_rec.p),
                       ctx->Aplus.p, DIR ? ctx->Wplus.p : nullptr, estride, out);
    HIP_TRY(hipGetLastError());
    return 0;
}

template <bool DIR>
static int launch_bt(ace_ctx* ctx, hipStream_t st, int64_t nenv, int64_t estride, double* out) {
    if (!bt_fits(ctx, DIR)) return set_err("pooled tile does not fit LDS");
    if (ctx->prop == ACE_PROP_INVARIANT) return launch_bv<DIR>(ctx, st, nenv, estride, out);
    if (DIR) return set_err("directional basis derivative: Invariant bases only");
    return (size_t)ctx->npool * 64 * sizeof(double2) <= 160 * 1024 ? launch_bt_shape<64>(ctx, st, nenv, estride, out)
                                                                   : launch_bt_shape<32>(ctx, st, nenv, estride, out);
}

extern "C" int ace_basis_B(ace_ctx* ctx, int64_t nenv, const int32_t* off, const double* xyz,
                           const int8_t* species, double* B_out, void* stream) {
    int64_t nnbr = 0;
    if (check_common(ctx, nenv, off, xyz, species, &nnbr, stream)) return -1;
    if (nenv == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    {
        const int64_t estride = ((nenv + 63) / 64) * 64;
        if (bt_fits(ctx, false)) {
            if (ctx->Aplus.ensure((size_t)ctx->npool * estride, ctx->capturing)) return -1;
            if (launch_pool_any(ctx, st, nenv, off, xyz, nnbr, species, estride, ctx_buffers(ctx), false)) return -1;
            return launch_bt<false>(ctx, st, nenv, estride, B_out);
        }
    }
    if (basis_A_internal(ctx, nenv, off, xyz, species, nnbr, st)) return -1;
    if (basis_AA_internal(ctx, nenv, st)) return -1;
    const int64_t n = nenv * ctx->nB;
    if (ctx->prop == ACE_PROP_INVARIANT)
        hipLaunchKernelGGL(k_B<0>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nenv, ctx->nB, ctx->nAA,
                           ctx->rowptr.p, ctx->cols.p, ctx->vals.p, ctx->AA.p, B_out);
    else
        hipLaunchKernelGGL(k_B<1>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nenv, ctx->nB, ctx->nAA,
                           ctx->rowptr.p, ctx->cols.p, ctx->vals.p, ctx->AA.p, B_out);
    HIP_TRY(hipGetLastError());
    return 0;
}

// rows: (mu, n, l, m) of each function, all of them (aspec4) or the pooled ones
template <int L>
static void launch_dphi(ace_ctx* ctx, hipStream_t st, int64_t nnbr, const double* xyz, const int8_t* species,
                        const int32_t* rows, int n) {
    const int64_t nblk = (nnbr + 63) / 64;
    // shares of eight functions or more, while there are fewer than eight waves per compute unit
    const int64_t want = std::max<int64_t>(1, std::min<int64_t>((n + 7) / 8, 8 * ctx->ncu / nblk));
    const int per = (int)((n + want - 1) / want);
    hipLaunchKernelGGL(k_dphi<L>, dim3((unsigned)nblk, (unsigned)((n + per - 1) / per)), dim3(64), 0, st,
                       radial_params(ctx), nnbr, xyz, ctx->nspecies > 0 ? species : nullptr, rows, n,
                       per, ctx->dphi.p);
}

// Basis gradients through per-environment adjoint weights (k_dBw): 0, or 1
// when the tables do not fit the kernel's LDS (the caller then runs the
// materialising path).
static int basis_dB_weights(ace_ctx* ctx, hipStream_t st, int64_t nenv, const int32_t* off, const double* xyz,
                            const int8_t* species, int64_t nnbr, double* dB_out) {
    if (!ctx->db_usable) return 1;
    const int NC = ctx->prop == ACE_PROP_INVARIANT ? 1 : 3;
    const size_t fixed = db_fixed_lds(ctx->npool);
    const size_t per_slot = (size_t)NC * sizeof(double2) + sizeof(int32_t);
    if (!ctx->db_ready) {
        acehost::DbTables& t = ctx->db_host;
        // no empty uploads (a basis without A2B entries)
        if (t.slot_k.empty()) t.slot_k.push_back(0);
        if (t.ztab.size() < 4) t.ztab.resize(4, 0u);
        if (t.vals.empty()) t.vals.push_back(0.0);
        if (ctx->db_wave.upload(t.wave.data(), t.wave.size()) || ctx->db_fn.upload(t.fn.data(), t.fn.size()) ||
            ctx->db_cnt.upload(t.cnt.data(), t.cnt.size()) ||
            ctx->db_chunk_s.upload(t.chunk_s.data(), t.chunk_s.size()) ||
            ctx->db_slot_k.upload(t.slot_k.data(), t.slot_k.size()) ||
            ctx->db_ztab.upload(t.ztab.data(), t.ztab.size()) || ctx->db_vals.upload(t.vals.data(), t.vals.size()))
            return -1;
        ctx->db_nchunk = t.nchunk();
        ctx->db_max_slots = t.max_chunk_slots;
        ctx->db_ready = true;
    }
    const int64_t estride = ((nenv + 63) / 64) * 64;
    if (ctx->Aplus.ensure((size_t)ctx->npool * estride, ctx->capturing) ||
        ctx->dphi.ensure((size_t)nnbr * ctx->npool * 3, ctx->capturing))
        return -1;
    if (launch_pool_any(ctx, st, nenv, off, xyz, nnbr, species, estride, ctx_buffers(ctx), false)) return -1;
    // the pooled (m >= 0) functions: pool rows are (mu, n, l, m) like aspec rows
    DISPATCH_L(ctx->L, launch_dphi, ctx, st, nnbr, xyz, species, ctx->pool.p, ctx->npool);
    HIP_TRY(hipGetLastError());
    DbArgs a;
    a.wave = reinterpret_cast<const int4*>(ctx->db_wave.p);
    a.fn = ctx->db_fn.p;
    a.cnt = reinterpret_cast<const int2*>(ctx->db_cnt.p);
    a.chunk_s = ctx->db_chunk_s.p;
    a.slot_k = ctx->db_slot_k.p;
    a.ztab = reinterpret_cast<const uint4*>(ctx->db_ztab.p);
    a.vals = ctx->db_vals.p;
    a.npool = ctx->npool;
    a.nB = ctx->nB;
    if (ctx->db_nchunk == 0) return 0;  // no basis functions
    const size_t lds = fixed + (size_t)ctx->db_max_slots * per_slot;
    const dim3 grid((unsigned)nenv, (unsigned)ctx->db_nchunk);
    auto go = [&](auto kern) {
        set_func_lds((const void*)kern, lds);
        hipLaunchKernelGGL(kern, grid, dim3(256), lds, st, a, nenv, off, ctx->Aplus.p, estride, ctx->dphi.p, dB_out);
    };
    const bool wide = ctx->db_host.zw == 8;
    // values per thread of a stage
    const int nq = 3 * ctx->npool, npf = (std::max(1, std::min(DB_NJ, DB_STAGE / nq)) * nq + 255) / 256;
    auto stage = [&](auto n) {
        constexpr int N = decltype(n)::value;
        if (ctx->prop == ACE_PROP_INVARIANT)
            wide ? go(k_dBw<0, 8, N>) : go(k_dBw<0, 4, N>);
        else
            wide ? go(k_dBw<1, 8, N>) : go(k_dBw<1, 4, N>);
    };
    if (npf <= 1)
        stage(std::integral_constant<int, 1>());
    else if (npf <= 2)
        stage(std::integral_constant<int, 2>());
    else if (npf <= 4)
        stage(std::integral_constant<int, 4>());
    else
        stage(std::integral_constant<int, DB_STAGE / 256>());
    HIP_TRY(hipGetLastError());
    return 0;
}

extern "C" int ace_basis_dB(ace_ctx* ctx, int64_t nenv, const int32_t* off, const double* xyz,
                            const int8_t* species, double* dB_out, void* stream) {
    int64_t nnbr = 0;
    if (check_common(ctx, nenv, off, xyz, species, &nnbr, stream)) return -1;
    if (nenv == 0 || nnbr == 0) return 0;
    hipStream_t st = (hipStream_t)stream;
    const int rc = basis_dB_weights(ctx, st, nenv, off, xyz, species, nnbr, dB_out);
    if (rc <= 0) return rc;
    // bases whose tables exceed the weight kernel's LDS: dAA per neighbour
    if (basis_A_internal(ctx, nenv, off, xyz, species, nnbr, st)) return -1;
    if (ctx->nbr_env.ensure(nnbr, ctx->capturing) || ctx->dphi.ensure((size_t)nnbr * ctx->nA * 3, ctx->capturing) ||
        ctx->dAA.ensure((size_t)nnbr * ctx->nAA * 3, ctx->capturing))
        return -1;
    hipLaunchKernelGGL(k_nbr_env, dim3((unsigned)((nenv + 255) / 256)), dim3(256), 0, st, nenv, off,
                       ctx->nbr_env.p);
    DISPATCH_L(ctx->L, launch_dphi, ctx, st, nnbr, xyz, species, ctx->aspec4.p, ctx->nA);
    HIP_TRY(hipGetLastError());
    const int64_t n1 = nnbr * ctx->nAA;
    hipLaunchKernelGGL(k_dAA, dim3((unsigned)((n1 + 255) / 256)), dim3(256), 0, st, nnbr, ctx->nA, ctx->nAA,
                       ctx->maxorder, ctx->nbr_env.p, ctx->orders.p, ctx->iAA2iA.p, ctx->Afull.p,
                       ctx->dphi.p, ctx->dAA.p);
    const int64_t n2 = nnbr * ctx->nB;
    if (ctx->prop == ACE_PROP_INVARIANT)
        hipLaunchKernelGGL(k_dB<0>, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, nnbr, ctx->nB,
                           ctx->nAA, ctx->rowptr.p, ctx->cols.p, ctx->vals.p, ctx->dAA.p, dB_out);
    else
        hipLaunchKernelGGL(k_dB<1>, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, nnbr, ctx->nB,
                           ctx->nAA, ctx->rowptr.p, ctx->cols.p, ctx->vals.p, ctx->dAA.p, dB_out);
    HIP_TRY(hipGetLastError());
    return 0;
}

extern "C" int ace_adjoint_EVAL_D(ace_ctx* ctx, int64_t nenv, const int32_t* off, const double* xyz,
                                  const int8_t* species, const double* w, double* dB_out, void* stream) {
    int64_t nnbr = 0;
    if (check_common(ctx, nenv, off, xyz, species, &nnbr, stream)) return -1;
    if (ctx->prop != ACE_PROP_INVARIANT) return set_err("ace_adjoint_EVAL_D: Invariant bases only");
    if (nenv == 0) return 0;
    if (!dB_out || (nnbr > 0 && !w)) return set_err("ace_adjoint_EVAL_D: null argument");
    hipStream_t st = (hipStream_t)stream;
    const int64_t estride = ((nenv + 63) / 64) * 64;
    if (bt_fits(ctx, true)) {
        if (ctx->Aplus.ensure((size_t)ctx->npool * estride, ctx->capturing) ||
            ctx->Wplus.ensure((size_t)ctx->npool * estride, ctx->capturing))
            return -1;
        if (launch_pool_any(ctx, st, nenv, off, xyz, nnbr, species, estride, ctx_buffers(ctx), false) ||
            launch_poolw_any(ctx, st, nenv, off, xyz, w, nnbr, species, estride))
            return -1;
        return launch_bt<true>(ctx, st, nenv, estride, dB_out);
    }
    if (basis_A_internal(ctx, nenv, off, xyz, species, nnbr, st)) return -1;
    if (ctx->Wplus.ensure((size_t)ctx->npool * estride, ctx->capturing) ||
        ctx->Wfull.ensure((size_t)nenv * ctx->nA, ctx->capturing) ||
        ctx->AA.ensure((size_t)nenv * ctx->nAA, ctx->capturing))
        return -1;
    if (launch_poolw_any(ctx, st, nenv, off, xyz, w, nnbr, species, estride)) return -1;
    const int64_t n = nenv * ctx->nA;
    hipLaunchKernelGGL(k_expandA, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, nenv, ctx->nA,
                       ctx->aspec_fid.p, ctx->aspec_sgn.p, ctx->Wplus.p, estride, ctx->Wfull.p);
    const int64_t n1 = nenv * ctx->nAA;
    hipLaunchKernelGGL(k_AAdir, dim3((unsigned)((n1 + 255) / 256)), dim3(256), 0, st, nenv, ctx->nA, ctx->nAA,
                       ctx->maxorder, ctx->orders.p, ctx->iAA2iA.p, ctx->Afull.p, ctx->Wfull.p, ctx->AA.p);
    const int64_t n2 = nenv * ctx->nB;
    hipLaunchKernelGGL(k_B<0>, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, nenv, ctx->nB, ctx->nAA,
                       ctx->rowptr.p, ctx->cols.p, ctx->vals.p, ctx->AA.p, dB_out);
    HIP_TRY(hipGetLastError());
    return 0;
}

// out[c] = sum_r w[r] B[r][c]: rows in shares of `per`, a thread per column, then
// the shares in order.  Bound by reading B once: 2,003 x 3,235, 52 MB, 10 us
// and the shares 3 (as a matrix product of one row, from a library, 65).
__global__ __launch_bounds__(256) void k_wrows(int64_t nrow, int64_t ncol, int per, const double* __restrict__ w,
                                               const double* __restrict__ B, double* __restrict__ part) {
    const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t r0 = (int64_t)blockIdx.y * per, r1 = min(r0 + per, nrow);
    if (c >= ncol) return;
    double s = 0.0;
#pragma unroll 8
    for (int64_t r = r0; r < r1; ++r) s = fma(w[r], B[r * ncol + c], s);
    part[(int64_t)blockIdx.y * ncol + c] = s;
}

__global__ __launch_bounds__(256) void k_wshares(int nshare, int64_t ncol, const double* __restrict__ part,
                                                 double* __restrict__ out) {
    __shared__ double red[4][64];
    const int l = threadIdx.x & 63, q = threadIdx.x >> 6;
    const int64_t c = (int64_t)blockIdx.x * 64 + l;
    double s = 0.0;
    if (c < ncol) {
#pragma unroll 8
        for (int i = q; i < nshare; i += 4) s += part[(int64_t)i * ncol + c];
    }
    red[q][l] = s;
    __syncthreads();
    if (q == 0 && c < ncol) out[c] = (red[0][l] + red[1][l]) + (red[2][l] + red[3][l]);
}

extern "C" int ace_weighted_rows(ace_ctx* ctx, int64_t nrow, int64_t ncol, const double* w, const double* B,
                                 double* out, void* stream) {
    if (!ctx) return set_err("null context");
    if (nrow < 0 || ncol < 0) return set_err("ace_weighted_rows: negative size");
    if (ncol == 0) return 0;
    if (!out || (nrow > 0 && (!w || !B))) return set_err("ace_weighted_rows: null argument");
    HIP_TRY(hipSetDevice(ctx->device));
    const int64_t gx = (ncol + 255) / 256;
    if (gx >= ((int64_t)1 << 31)) return set_err("ace_weighted_rows: too many columns");
    // eight workgroups per compute unit, eight rows each at least
    const int64_t want = std::max<int64_t>(1, std::min((int64_t)8 * ctx->ncu / gx, (nrow + 7) / 8));
    const int64_t per = std::max<int64_t>(1, (nrow + want - 1) / want);
    const int nshare = (int)((nrow + per - 1) / per);
    if (per >= ((int64_t)1 << 31)) return set_err("ace_weighted_rows: too many rows");
    hipStream_t st = (hipStream_t)stream;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    HIP_TRY(hipStreamIsCapturing(st, &cap));
    ctx->capturing = cap != hipStreamCaptureStatusNone;
    if (ctx->wrows.ensure((size_t)std::max(1, nshare) * ncol, ctx->capturing)) return -1;
    if (nshare > 0)
        hipLaunchKernelGGL(k_wrows, dim3((unsigned)gx, (unsigned)nshare), dim3(256), 0, st, nrow, ncol, (int)per, w, B,
                           ctx->wrows.p);
    hipLaunchKernelGGL(k_wshares, dim3((unsigned)((ncol + 63) / 64)), dim3(256), 0, st, nshare, ncol,
                       (const double*)ctx->wrows.p, out);
    HIP_TRY(hipGetLastError());
    return 0;
}
