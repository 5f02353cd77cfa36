// Environment extraction and force assembly on either side of the basis
// evaluation (the atoms-level callers of ACE.jl: src/testing/testlsq.jl:
// 27-35,42-69 call energy(V, at) / forces(V, at) on whole configurations).
//
//   ace_nbrlist_build   cell-list neighbour search with periodic images:
//                       host bins the atoms (nbrlist_host.hpp), the device
//                       counts and fills every atom's environment (relative
//                       positions, neighbour index, image shift, species)
//                       and the reverse index of each pair.
//   ace_nbrlist_update  recomputes the relative positions of an existing
//                       list from new positions (a list built with a skin
//                       stays valid for several MD steps); stream-ordered,
//                       no host synchronization.
//   ace_nbrlist_forces_multi  the same for many fields at once, e.g. the
//                       per-basis-function forces of least-squares fitting.
//   ace_nbrlist_forces  F_k = -dE/dx_k from the per-neighbour gradients
//                       g_m = +dE_i/dr_m (the ACE.jl grad_config sign) and
//                       the virial W = -sum_m g_m r_m^T, deterministically
//                       (a gather over each atom's own entries, no atomics).
//
// Entry m of atom i is the pair (i -> j, S') with r_m = (x_j - x_i) + S' . cell.
// E = sum_i E_i(r_m : m in N(i)), so
//   dE/dx_k = sum_{m : j(m) = k} g_m - sum_{m in N(k)} g_m
//           = sum_{m in N(k)} (g_rev(m) - g_m),
// where rev(m) is the entry (j -> i, -S') of the symmetric list.

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include <hipcub/hipcub.hpp>

#include "../../include/acehip.h"
#include "host_util.hpp"
#include "nbrlist_host.hpp"

// No multiply-add contraction in this file: the search evaluates every pair
// in both orientations and in two passes, and the decisions must agree
// exactly (the negated operands of the reverse pair round identically only
// when the same separately rounded operations are used).
#pragma clang fp contract(off)

struct NbrArgs {
    double cell[9];
    double rc2;
    int nb[3], R[3], pbc[3];
    int natoms;
    const int32_t* bin;        // [natoms]
    const int32_t* bin_start;  // [nbins + 1]
    const int32_t* bin_atoms;  // [natoms]
    // in bin order: wrapped positions, positions, wrap counts, [3][natoms] each
    const double* sp;
    const double* sx;
    const int32_t* sw;
};

__device__ __forceinline__ int floordiv(int z, int n) { return z >= 0 ? z / n : -((n - 1 - z) / n); }

// Shift vector S0 a + S1 b + S2 c and the squared distance.
__device__ __forceinline__ void shift_vec(const double* cell, int s0, int s1, int s2, double& vx, double& vy,
                                          double& vz) {
    const double a = s0, b = s1, c = s2;
    vx = (a * cell[0] + b * cell[3]) + c * cell[6];
    vy = (a * cell[1] + b * cell[4]) + c * cell[7];
    vz = (a * cell[2] + b * cell[5]) + c * cell[8];
}

__device__ __forceinline__ double norm2(double x, double y, double z) { return (x * x + y * y) + z * z; }

// Workgroups go to the 8 XCDs in turn: workgroup b of n takes share w(b), so that
// each XCD, with an L2 of its own, has a run of neighbouring atoms.
__device__ __forceinline__ int xcd_share(int b, int n) {
    const int x = b & 7, q = n >> 3, r = n & 7;
    return x * q + min(x, r) + (b >> 3);
}

// Workgroups of 256 threads, `first` on, in launches of fewer than 2^32 threads
// each (what a launch takes): launch(first, workgroups).
template <typename F>
void in_launches(int64_t nwg, F launch) {
    constexpr int64_t most = ((int64_t)1 << 24) - 1;
    for (int64_t w = 0; w < nwg; w += most) launch((int)w, dim3((unsigned)std::min(most, nwg - w)));
}

// The atoms' data in bin order, so that the search reads a row of bins as one
// stretch of memory.
__global__ __launch_bounds__(256) void k_nbr_gather(int n, const int32_t* __restrict__ bin_atoms,
                                                    const double* __restrict__ pw, const double* __restrict__ pos,
                                                    const int32_t* __restrict__ wrap, double* __restrict__ sp,
                                                    double* __restrict__ sx, int32_t* __restrict__ sw) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t >= n) return;
    const int i = bin_atoms[t];
    for (int d = 0; d < 3; ++d) {
        sp[d * (int64_t)n + t] = pw[d * (int64_t)n + i];
        sx[d * (int64_t)n + t] = pos[d * (int64_t)n + i];
        sw[d * (int64_t)n + t] = wrap[d * (int64_t)n + i];
    }
}

// One wave per atom, atoms taken in bin order.  FILL = false counts, FILL =
// true writes the entries in the same order: bins (z, y, x ascending, images
// included), atoms of a bin ascending.  The bins of a row (z, y) that lie in one
// image along x are one stretch of the sorted atoms: a segment.  Lane s of a group of
// 64 segments looks up segment s (its atoms and its shift); the wave then goes
// through the non-empty ones, 64 atoms at a time, the next atoms loaded before
// the present ones are tested.  Hits go to a ring in LDS in order, and leave it 64
// at a time, one lane per entry, so that the stores of the fill are whole lines.
// 55,296 atoms of 54 neighbours: count 170 -> 69 us, fill 468 -> 96 us against one
// thread per atom, whose lanes diverged at every hit and stored 4 or 8 bytes
// to a line of their own.
template <bool FILL>
__global__ __launch_bounds__(256) void k_nbr_search(NbrArgs a, int first, int32_t* __restrict__ cnt,
                                                    const int32_t* __restrict__ off, int64_t nnbr,
                                                    int32_t* __restrict__ env_off, int32_t* __restrict__ nbr_j,
                                                    int32_t* __restrict__ shift, double* __restrict__ xyz,
                                                    const int8_t* __restrict__ zat, int8_t* __restrict__ znbr,
                                                    int32_t* __restrict__ flag) {
    __shared__ int2 ring[4][FILL ? 128 : 1];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int64_t tw = ((int64_t)first + xcd_share(blockIdx.x, gridDim.x)) * 4 + wave;
    const int t = (int)tw;
    if (tw >= a.natoms) return;  // whole waves; the kernel has no barrier
    const int64_t n = a.natoms;
    const int i = a.bin_atoms[t];
    // positions that are refused may all lie in one bin
    if (!FILL && (*flag & 12)) {
        if (lane == 0) cnt[i] = 0;
        return;
    }
    const int b = a.bin[i];
    const int bx = b % a.nb[0], by = (b / a.nb[0]) % a.nb[1], bz = b / (a.nb[0] * a.nb[1]);
    const double pix = a.sp[t], piy = a.sp[n + t], piz = a.sp[2 * n + t];
    int64_t m = 0, mend = 0;
    int wi0 = 0, wi1 = 0, wi2 = 0;
    double xix = 0, xiy = 0, xiz = 0;
    int2* pend = ring[wave];
    int head = 0, held = 0;
    if (FILL) {
        m = off[i];
        mend = off[i + 1];
        if (lane == 0) env_off[i] = (int32_t)m;
        if (lane == 0 && i == a.natoms - 1) env_off[a.natoms] = (int32_t)mend;
        wi0 = a.sw[t];
        wi1 = a.sw[n + t];
        wi2 = a.sw[2 * n + t];
        xix = a.sx[t];
        xiy = a.sx[n + t];
        xiz = a.sx[2 * n + t];
    }
    // the first k entries of the ring
    auto flush = [&](int k) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < k && m + lane < mend) {
            const int2 h = pend[(head + lane) & 127];
            const int j = a.bin_atoms[h.x];
            const int s0 = ((h.y & 255) - 128) - a.sw[h.x] + wi0;
            const int s1 = ((h.y >> 8 & 255) - 128) - a.sw[n + h.x] + wi1;
            const int s2 = ((h.y >> 16 & 255) - 128) - a.sw[2 * n + h.x] + wi2;
            double ux, uy, uz;
            shift_vec(a.cell, s0, s1, s2, ux, uy, uz);
            const int64_t e = m + lane;
            nbr_j[e] = j;
            shift[e] = s0;
            shift[nnbr + e] = s1;
            shift[2 * nnbr + e] = s2;
            xyz[e] = (a.sx[h.x] - xix) + ux;
            xyz[nnbr + e] = (a.sx[n + h.x] - xiy) + uy;
            xyz[2 * nnbr + e] = (a.sx[2 * n + h.x] - xiz) + uz;
            if (znbr) znbr[e] = zat[j];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        m += k;
        head += k;
        held -= k;
    };
    const int xlo = bx - a.R[0], xhi = bx + a.R[0];
    const int S00 = a.pbc[0] ? floordiv(xlo, a.nb[0]) : 0;
    const int nsx = a.pbc[0] ? floordiv(xhi, a.nb[0]) - S00 + 1 : 1;
    const int ny = 2 * a.R[1] + 1, nseg = (2 * a.R[2] + 1) * ny * nsx;
    int c = 0;
    for (int base = 0; base < nseg; base += 64) {
        // lane: segment base + lane
        int sq0 = 0, sq1 = 0, scode = 0;
        double svx = 0, svy = 0, svz = 0;
        if (base + lane < nseg) {
            const int g = base + lane, row = g / nsx;
            int z = bz + row / ny - a.R[2], y = by + row % ny - a.R[1], S1 = 0, S2 = 0;
            const int S0 = S00 + g % nsx;
            bool in = true;
            if (a.pbc[2]) {
                S2 = floordiv(z, a.nb[2]);
                z -= S2 * a.nb[2];
            } else {
                in = z >= 0 && z < a.nb[2];
            }
            if (a.pbc[1]) {
                S1 = floordiv(y, a.nb[1]);
                y -= S1 * a.nb[1];
            } else {
                in = in && y >= 0 && y < a.nb[1];
            }
            const int xa = max(xlo - S0 * a.nb[0], 0), xb = min(xhi - S0 * a.nb[0], a.nb[0] - 1);
            if (in && xa <= xb) {
                const int row0 = (z * a.nb[1] + y) * a.nb[0];
                sq0 = a.bin_start[row0 + xa];
                sq1 = a.bin_start[row0 + xb + 1];
                shift_vec(a.cell, S0, S1, S2, svx, svy, svz);
                scode = (S0 + 128) | (S1 + 128) << 8 | (S2 + 128) << 16;
            }
        }
        uint64_t left = __ballot(sq1 > sq0);
        int q = 0, q1 = 0, code = 0;
        double vx = 0, vy = 0, vz = 0, nx = 0, ny_ = 0, nz = 0;
        // the next 64 atoms: of this segment, else of the next one
        auto advance = [&]() {
            q += 64;
            if (q >= q1) {
                if (!left) return false;
                const int l = __ffsll((unsigned long long)left) - 1;
                left &= left - 1;
                q = __builtin_amdgcn_readlane(sq0, l);
                q1 = __builtin_amdgcn_readlane(sq1, l);
                code = __builtin_amdgcn_readlane(scode, l);
                auto bcast = [&](double v) {
                    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                                            __builtin_amdgcn_readlane(__double2loint(v), l));
                };
                vx = bcast(svx);
                vy = bcast(svy);
                vz = bcast(svz);
            }
            const int64_t p = min(q + lane, q1 - 1);
            nx = a.sp[p];
            ny_ = a.sp[n + p];
            nz = a.sp[2 * n + p];
            return true;
        };
        bool more = advance();
        while (more) {
            const double ex = (nx - pix) + vx, ey = (ny_ - piy) + vy, ez = (nz - piz) + vz;
            const int qq = q + lane, code0 = code;
            const bool self = code == (128 | 128 << 8 | 128 << 16) && qq == t;
            const bool hit = qq < q1 && !self && norm2(ex, ey, ez) < a.rc2;
            more = advance();
            const uint64_t hm = __ballot(hit);
            const int k = __popcll((unsigned long long)hm);
            if (FILL) {
                const int at = __builtin_amdgcn_mbcnt_hi((uint32_t)(hm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hm, 0));
                if (hit) pend[(head + held + at) & 127] = make_int2(qq, code0);
                held += k;
                if (held >= 64) flush(64);
            } else {
                c += k;
            }
        }
    }
    if (!FILL && lane == 0) cnt[i] = c;
    if (FILL) {
        flush(held);
        if (m != mend && lane == 0) atomicOr(flag, 1);
    }
}

// Offsets of the counts: every block of SCAN_CH counts first sums them, then
// adds the sums before it to its own prefix sums.  64-bit sums; the last block's
// end is the number of entries.
constexpr int SCAN_CH = 2048;

__global__ __launch_bounds__(256) void k_nbr_scan_sum(int n, const int32_t* __restrict__ cnt, int64_t* __restrict__ bsum) {
    __shared__ int64_t red[256];
    int64_t s = 0;
    for (int q = 0; q < SCAN_CH / 256; ++q) {
        const int64_t i = (int64_t)blockIdx.x * SCAN_CH + q * 256 + threadIdx.x;
        if (i < n) s += cnt[i];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) bsum[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(256) void k_nbr_scan(int n, const int32_t* __restrict__ cnt,
                                                  const int64_t* __restrict__ bsum, int32_t* __restrict__ off,
                                                  int64_t* __restrict__ total) {
    __shared__ int64_t red[256];
    const int tid = threadIdx.x;
    int64_t s = 0;
    for (int b = tid; b < (int)blockIdx.x; b += 256) s += bsum[b];
    red[tid] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h) red[tid] += red[tid + h];
        __syncthreads();
    }
    const int64_t before = red[0];
    __syncthreads();
    // a thread's counts are consecutive
    const int64_t i0 = (int64_t)blockIdx.x * SCAN_CH + tid * (SCAN_CH / 256);
    int32_t v[SCAN_CH / 256];
    int64_t mine = 0;
    for (int q = 0; q < SCAN_CH / 256; ++q) {
        v[q] = i0 + q < n ? cnt[i0 + q] : 0;
        mine += v[q];
    }
    red[tid] = mine;
    __syncthreads();
    for (int h = 1; h < 256; h <<= 1) {
        const int64_t x = tid >= h ? red[tid - h] : 0;
        __syncthreads();
        red[tid] += x;
        __syncthreads();
    }
    int64_t at = before + red[tid] - mine;
    for (int q = 0; q < SCAN_CH / 256; ++q) {
        if (i0 + q < n) off[i0 + q] = (int32_t)at;
        at += v[q];
        if (i0 + q == n - 1) {
            off[n] = (int32_t)at;
            *total = at;
        }
    }
}

// rev[m] = index of (j -> i, -S') in the list of j; flag bit 2 if absent.
// One wave per atom i, atoms taken in bin order so that the lists of
// neighbouring j are shared in cache.  64 entries are looked up at a time (a lane
// each: j, -S', the ends of j's list).  Their lists are searched for i four at
// a time, 16 lanes on a list, all loads independent; lane e keeps the first
// match of entry e.  Then all 64 matches are checked against the shift at once, and only
// an entry whose first match is another image of i (cells below twice the
// reach) is searched again with its shift, by the whole wave.  Bound by the latency of
// those loads: checking every match where it was found took 214 us for 55,296
// atoms of 54 neighbours, this 143; one thread per entry, with a search for its
// atom and a scan of the list one entry after the other, 422.
__global__ __launch_bounds__(256) void k_nbr_rev(int natoms, int first, const int32_t* __restrict__ atoms,
                                                 const int32_t* __restrict__ off, const int32_t* __restrict__ nbr_j,
                                                 const int32_t* __restrict__ shift, int64_t nnbr,
                                                 int32_t* __restrict__ rev, int32_t* __restrict__ flag) {
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int lane = threadIdx.x & 63;
    const int64_t t = ((int64_t)first + xcd_share(blockIdx.x, gridDim.x)) * 4 + wave;
    if (t >= natoms) return;
    const int i = atoms[t];
    // entries are counted without a sign: a list may end at 2^31 - 1, and the
    // steps of 64 and the lanes past its end go beyond
    const uint32_t m0 = off[i], m1 = off[i + 1];
    const int sub = lane & 15;
    for (uint32_t mb = m0; mb < m1; mb += 64) {
        const int cnt = (int)min(64u, m1 - mb);
        const bool mine = lane < cnt;
        uint32_t qa = 0, qb = 0;
        int s0 = 0, s1 = 0, s2 = 0;
        if (mine) {
            const int64_t m = (int64_t)mb + lane;
            const int j = nbr_j[m];
            s0 = -shift[m];
            s1 = -shift[nnbr + m];
            s2 = -shift[2 * nnbr + m];
            qa = off[j];
            qb = off[j + 1];
        }
        int found = -1;
#pragma unroll 2
        for (int e = 0; e < cnt; e += 4) {
            const int src = e + (lane >> 4);  // lanes past the last entry search an empty list
            const uint32_t q0 = __shfl(qa, src), q1 = __shfl(qb, src);
            for (uint32_t p = 0; __any(q0 + p < q1); p += 64) {
                bool is[4];
#pragma unroll
                for (int h = 0; h < 4; ++h) {
                    const uint32_t q = q0 + p + 16 * h + sub;
                    is[h] = q < q1 && nbr_j[q] == i;
                }
                uint64_t hits[4];
#pragma unroll
                for (int h = 0; h < 4; ++h) hits[h] = __ballot(is[h]);
                // lane e + g takes the result of list g
                const int g = lane - e;
                if ((unsigned)g < 4u && found < 0) {
#pragma unroll
                    for (int h = 3; h >= 0; --h) {
                        const uint32_t f = (uint32_t)(hits[h] >> (16 * g)) & 0xffffu;
                        if (f) found = (int)(qa + p + 16 * h + __ffs((int)f) - 1);
                    }
                }
            }
        }
        const int64_t f = max(found, 0);
        const bool ok = !mine || (found >= 0 && shift[f] == s0 && shift[nnbr + f] == s1 && shift[2 * nnbr + f] == s2);
        for (uint64_t bad = __ballot(!ok); bad; bad &= bad - 1) {
            const int l = __ffsll((unsigned long long)bad) - 1;
            const uint32_t q1 = __builtin_amdgcn_readlane(qb, l);
            const int t0 = __builtin_amdgcn_readlane(s0, l), t1 = __builtin_amdgcn_readlane(s1, l),
                      t2 = __builtin_amdgcn_readlane(s2, l);
            int at = -1;
            for (uint32_t q = __builtin_amdgcn_readlane(qa, l); q < q1 && at < 0; q += 64) {
                const uint32_t p = q + lane;
                const bool is = p < q1 && nbr_j[p] == i && shift[p] == t0 && shift[nnbr + p] == t1 &&
                                shift[2 * nnbr + p] == t2;
                const uint64_t hit = __ballot(is);
                if (hit) at = (int)(q + __ffsll((unsigned long long)hit) - 1);
            }
            if (lane == l) found = at;
        }
        if (mine) rev[(int64_t)mb + lane] = found;
        if (__any(mine && found < 0) && lane == 0) atomicOr(flag, 2);
    }
}

// New relative positions of the entries: 16 lanes per atom.
__global__ __launch_bounds__(256) void k_nbr_update(int natoms, int first, NbrArgs a, const double* __restrict__ pos,
                                                    const int32_t* __restrict__ off, const int32_t* __restrict__ nbr_j,
                                                    const int32_t* __restrict__ shift, int64_t nnbr,
                                                    double* __restrict__ xyz) {
    const int64_t n = natoms;
    const int64_t i = ((int64_t)first + blockIdx.x) * 16 + (threadIdx.x >> 4);
    if (i >= n) return;
    // entries outside the offsets belong to the first and the last atom
    const int64_t m0 = i == 0 ? 0 : max(off[i], 0), m1 = i == n - 1 ? nnbr : min((int64_t)off[i + 1], nnbr);
    const double xi = pos[i], yi = pos[n + i], zi = pos[2 * n + i];
    for (int64_t m = m0 + (threadIdx.x & 15); m < m1; m += 16) {
        const int j = nbr_j[m];
        double ux, uy, uz;
        shift_vec(a.cell, shift[m], shift[nnbr + m], shift[2 * nnbr + m], ux, uy, uz);
        xyz[m] = (pos[j] - xi) + ux;
        xyz[nnbr + m] = (pos[n + j] - yi) + uy;
        xyz[2 * nnbr + m] = (pos[2 * n + j] - zi) + uz;
    }
}

// F_k = sum_{m in N(k)} (g_m - g_rev(m)): 16 lanes per atom take its entries in
// turn, four at a time so that their gathers are in flight together, and are
// summed by a fixed tree.  A workgroup takes `per` groups of 16 atoms, the
// workgroups of one XCD neighbouring ones.  Virial partials -g_m r_m^T stay in
// registers to the end and are reduced over the workgroup in a fixed order.
// Bound by the gathers of g at rev(m), 24 bytes to lines of their own: 55,296 atoms
// of 54 neighbours, 92 -> 54 us, 256 atoms 36 -> 8 us, against 64 atoms per
// workgroup staged in LDS, one thread of which then added up each atom.
constexpr int FA_ATOMS = 16;
constexpr int FA_BLOCKS = 2048;  // workgroups at most

__global__ __launch_bounds__(256) void k_nbr_forces(int natoms, int per, const int32_t* __restrict__ off,
                                                    const int32_t* __restrict__ rev, int64_t nnbr,
                                                    const double* __restrict__ g, const double* __restrict__ xyz,
                                                    double* __restrict__ F, double* __restrict__ vpart) {
    __shared__ double red[9][256];
    const int tid = threadIdx.x, sub = tid & 15;
    const int64_t n = natoms;
    const int64_t g0 = (int64_t)xcd_share(blockIdx.x, gridDim.x) * per;
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t q = g0; q < g0 + per; ++q) {
        const int64_t k = q * FA_ATOMS + (tid >> 4);
        // unsigned, as in k_nbr_rev
        const uint32_t m0 = k < n ? max(off[k], 0) : 0, m1 = k < n ? max(off[k + 1], 0) : 0;
        double f[3] = {0, 0, 0};
        for (uint32_t mb = m0 + sub; mb < m1; mb += 64) {
            int r[4];
            double gm[4][3], gr[4][3], x[4][3];
#pragma unroll
            for (int h = 0; h < 4; ++h) r[h] = mb + 16 * h < m1 ? rev[mb + 16 * h] : -1;
#pragma unroll
            for (int h = 0; h < 4; ++h)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    gm[h][d] = gr[h][d] = x[h][d] = 0.0;
                    if (r[h] >= 0) {
                        gm[h][d] = g[d * nnbr + mb + 16 * h];
                        gr[h][d] = g[d * nnbr + r[h]];
                        if (vpart) x[h][d] = xyz[d * nnbr + mb + 16 * h];
                    }
                }
#pragma unroll
            for (int h = 0; h < 4; ++h)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    f[d] += gm[h][d] - gr[h][d];
#pragma unroll
                    for (int c = 0; c < 3; ++c) v[3 * d + c] -= gm[h][d] * x[h][c];
                }
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
#pragma unroll
            for (int h = 8; h > 0; h >>= 1) f[d] += __shfl_xor(f[d], h);
        }
        if (k < n && sub < 3) F[sub * n + k] = sub == 0 ? f[0] : sub == 1 ? f[1] : f[2];
    }
    if (!vpart) return;  // uniform over the block
    for (int c = 0; c < 9; ++c) red[c][tid] = v[c];
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (tid < s)
            for (int c = 0; c < 9; ++c) red[c][tid] += red[c][tid + s];
        __syncthreads();
    }
    if (tid < 9) vpart[(int64_t)blockIdx.x * 9 + tid] = red[tid][0];
}

// F[k][v][d] = sum_{m in N(k)} (g[m][v][d] - g[rev(m)][v][d]) for nvec
// fields at once (per-basis-function forces): thread per (atom, field),
// consecutive threads read consecutive fields of one entry.
__global__ __launch_bounds__(256) void k_nbr_forces_multi(int natoms, const int32_t* __restrict__ off,
                                                          const int32_t* __restrict__ rev, int64_t nvec,
                                                          const double* __restrict__ g, double* __restrict__ F) {
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (int64_t)natoms * nvec) return;
    const int k = (int)(t / nvec);
    const int64_t v = t - (int64_t)k * nvec;
    double fx = 0, fy = 0, fz = 0;
    const int m1 = off[k + 1];
    for (int m = off[k]; m < m1; ++m) {
        const double* a = g + ((int64_t)m * nvec + v) * 3;
        const double* b = g + ((int64_t)rev[m] * nvec + v) * 3;
        fx += a[0] - b[0];
        fy += a[1] - b[1];
        fz += a[2] - b[2];
    }
    double* o = F + t * 3;
    o[0] = fx;
    o[1] = fy;
    o[2] = fz;
}

// W[c] = sum over blocks of vpart[b][c] in a fixed order: 64 lanes per
// component take every 64th block, then a tree over the lanes.
__global__ __launch_bounds__(576) void k_nbr_vsum(int nblk, const double* __restrict__ vpart,
                                                  double* __restrict__ W) {
    __shared__ double part[9][64];
    const int c = threadIdx.x >> 6, l = threadIdx.x & 63;
    double s = 0.0;
    for (int b = l; b < nblk; b += 64) s += vpart[(int64_t)b * 9 + c];
    part[c][l] = s;
    __syncthreads();
    for (int h = 32; h > 0; h >>= 1) {
        if (l < h) part[c][l] += part[c][l + h];
        __syncthreads();
    }
    if (l == 0) W[c] = part[c][0];
}

__global__ void k_nbr_zero(int32_t* p, int n) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) p[t] = 0;
}

// ---------------------------------------------------------------------------
// binning on the device (the operations of nbrlist_host.hpp: nbr_frac,
// nbr_bin1, wrapped positions), so that the bins match the host's exactly

struct NbrFracArgs {
    double cell[9], inv[9];
    int pbc[3];
    int natoms;
};

// Wrapped fractional coordinates sf[3][n], wrap counts, wrapped positions
// pw[3][n], and per-block minima / maxima of sf (bmm[block][6]).  flag bit 4:
// a non-finite position; bit 8: a wrap beyond 1e6 cells.
__global__ __launch_bounds__(256) void k_nbr_frac(NbrFracArgs a, const double* __restrict__ pos,
                                                  double* __restrict__ sf, int32_t* __restrict__ wrap,
                                                  double* __restrict__ pw, double* __restrict__ bmm,
                                                  int32_t* __restrict__ flag) {
    __shared__ double red[6][256];
    const int n = a.natoms;
    const int i = blockIdx.x * 256 + threadIdx.x;
    double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
    if (i < n) {
        const double x = pos[i], y = pos[n + i], z = pos[2 * n + i];
        int w[3] = {0, 0, 0};
        if (!isfinite(x) || !isfinite(y) || !isfinite(z)) atomicOr(flag, 4);
        for (int d = 0; d < 3; ++d) {
            double sv = x * a.inv[d] + y * a.inv[3 + d] + z * a.inv[6 + d];
            if (a.pbc[d]) {
                const double f = floor(sv);
                if (!(fabs(f) <= 1e6)) {
                    atomicOr(flag, 8);
                } else {
                    w[d] = (int)f;
                }
                sv -= f;
                if (sv >= 1.0) sv = 0.0;
            }
            sf[d * n + i] = sv;
            wrap[d * n + i] = w[d];
            lo[d] = sv;
            hi[d] = sv;
        }
        for (int q = 0; q < 3; ++q)
            pw[q * n + i] = pos[q * n + i] - ((double)w[0] * a.cell[q] + (double)w[1] * a.cell[3 + q] +
                                              (double)w[2] * a.cell[6 + q]);
    }
    for (int d = 0; d < 3; ++d) {
        red[d][threadIdx.x] = lo[d];
        red[3 + d][threadIdx.x] = hi[d];
    }
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            for (int d = 0; d < 3; ++d) {
                red[d][threadIdx.x] = fmin(red[d][threadIdx.x], red[d][threadIdx.x + h]);
                red[3 + d][threadIdx.x] = fmax(red[3 + d][threadIdx.x], red[3 + d][threadIdx.x + h]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 6) bmm[(int64_t)blockIdx.x * 6 + threadIdx.x] = red[threadIdx.x][0];
}

// mm[0..2] = minima, mm[3..5] = maxima over the blocks (one block).
__global__ __launch_bounds__(256) void k_nbr_minmax(int nblk, const double* __restrict__ bmm, double* __restrict__ mm) {
    __shared__ double red[6][256];
    double v[6] = {1e300, 1e300, 1e300, -1e300, -1e300, -1e300};
    for (int b = threadIdx.x; b < nblk; b += 256)
        for (int c = 0; c < 6; ++c) v[c] = c < 3 ? fmin(v[c], bmm[(int64_t)b * 6 + c]) : fmax(v[c], bmm[(int64_t)b * 6 + c]);
    for (int c = 0; c < 6; ++c) red[c][threadIdx.x] = v[c];
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h)
            for (int c = 0; c < 6; ++c)
                red[c][threadIdx.x] = c < 3 ? fmin(red[c][threadIdx.x], red[c][threadIdx.x + h])
                                            : fmax(red[c][threadIdx.x], red[c][threadIdx.x + h]);
        __syncthreads();
    }
    if (threadIdx.x < 6) mm[threadIdx.x] = red[threadIdx.x][0];
}

struct NbrBinArgs {
    int nb[3];
    double s0[3], w[3];
    int natoms;
};

__device__ __forceinline__ int bin1(const NbrBinArgs& g, double s, int d) {
    const int v = (int)floor((s - g.s0[d]) / g.w[d]);
    return min(max(v, 0), g.nb[d] - 1);
}

// bin[i] and the sort values (atom index)
__global__ __launch_bounds__(256) void k_nbr_bin(NbrBinArgs g, const double* __restrict__ sf,
                                                 int32_t* __restrict__ bin, int32_t* __restrict__ idx) {
    const int n = g.natoms;
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    bin[i] = (bin1(g, sf[2 * n + i], 2) * g.nb[1] + bin1(g, sf[n + i], 1)) * g.nb[0] + bin1(g, sf[i], 0);
    idx[i] = i;
}

// bin_start[b] = first position of bin b in the sorted keys (b <= nbins)
__global__ __launch_bounds__(256) void k_nbr_binstart(int nbins, int n, const int32_t* __restrict__ keys,
                                                      int32_t* __restrict__ bin_start) {
    const int b = blockIdx.x * 256 + threadIdx.x;
    if (b > nbins) return;
    int lo = 0, hi = n;  // first q with keys[q] >= b
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (keys[mid] < b) lo = mid + 1;
        else hi = mid;
    }
    bin_start[b] = lo;
}

// ---------------------------------------------------------------------------
// host side

struct ace_nbrlist {
    int device = 0;
    acehost::NbrGrid g;  // grid parameters (nb, R, s0, w) of the last build
    int natoms = 0;
    // read back after a build's stages: [0..5] extents, [6] flags, [7] entries
    struct Mail {
        double mm[6];
        int64_t flag, total;
    };
    Mail* mail = nullptr;  // pinned host memory
    DevBuf<Mail> dmail;
    DevBuf<double> pw, vpart, sf, bmm, sp, sx;
    DevBuf<int32_t> wrap, bin, bin_start, bin_atoms, cnt, keys, idx, sw, off;
    DevBuf<int64_t> bsum;
    DevBuf<char> sort_tmp;
};

static NbrArgs grid_args(ace_nbrlist* nl, const double* cell) {
    NbrArgs a{};
    for (int q = 0; q < 9; ++q) a.cell[q] = cell[q];
    const acehost::NbrGrid& g = nl->g;
    a.rc2 = g.rcut * g.rcut;
    for (int d = 0; d < 3; ++d) {
        a.nb[d] = g.nb[d];
        a.R[d] = g.R[d];
        a.pbc[d] = g.pbc[d];
    }
    a.natoms = nl->natoms;
    a.bin = nl->bin.p;
    a.bin_start = nl->bin_start.p;
    a.bin_atoms = nl->bin_atoms.p;
    a.sp = nl->sp.p;
    a.sx = nl->sx.p;
    a.sw = nl->sw.p;
    return a;
}

extern "C" int ace_nbrlist_create(int device, ace_nbrlist** out) {
    if (!out) return set_err("ace_nbrlist_create: null argument");
    *out = nullptr;
    int ndev = 0;
    HIP_TRY(hipGetDeviceCount(&ndev));
    if (device < 0 || device >= ndev) return set_err("ace_nbrlist_create: device index out of range");
    HIP_TRY(hipSetDevice(device));
    ace_nbrlist* nl = new ace_nbrlist();
    nl->device = device;
    if (hipHostMalloc((void**)&nl->mail, sizeof(ace_nbrlist::Mail), hipHostMallocDefault) != hipSuccess) {
        delete nl;
        return set_err("ace_nbrlist_create: pinned host allocation failed");
    }
    *out = nl;
    return 0;
}

extern "C" void ace_nbrlist_destroy(ace_nbrlist* nl) {
    if (!nl) return;
    (void)hipSetDevice(nl->device);
    (void)hipHostFree(nl->mail);
    delete nl;
}

extern "C" int ace_nbrlist_build(ace_nbrlist* nl, int64_t natoms, const double* pos, const double* cell,
                                 const int32_t* pbc, double rcut, const int8_t* atom_species, int64_t capacity,
                                 int32_t* env_offsets, int32_t* nbr_j, int32_t* shift, double* xyz, int32_t* rev,
                                 int8_t* nbr_species, int64_t* nnbr_out, void* stream) {
    if (!nl || !cell || !pbc || !env_offsets || !nnbr_out) return set_err("ace_nbrlist_build: null argument");
    if (natoms < 0 || natoms >= ((int64_t)1 << 31) - 1) return set_err("ace_nbrlist_build: natoms out of range");
    if (natoms > 0 && !pos) return set_err("ace_nbrlist_build: null positions");
    if (capacity < 0) return set_err("ace_nbrlist_build: capacity < 0");
    if (capacity > 0 && (!nbr_j || !shift || !xyz)) return set_err("ace_nbrlist_build: null neighbour arrays");
    if (nbr_species && !atom_species) return set_err("ace_nbrlist_build: nbr_species needs atom_species");
    *nnbr_out = 0;
    HIP_TRY(hipSetDevice(nl->device));
    hipStream_t st = (hipStream_t)stream;
    const int n = (int)natoms;
    acehost::NbrGeom geo;
    const std::string gerr = acehost::nbr_setup(cell, pbc, rcut, geo);
    if (!gerr.empty()) return set_err("ace_nbrlist_build: " + gerr);
    nl->natoms = n;
    if (n == 0) {
        hipLaunchKernelGGL(k_nbr_zero, dim3(1), dim3(64), 0, st, env_offsets, 1);
        HIP_TRY(hipGetLastError());
        HIP_TRY(hipStreamSynchronize(st));
        return 0;
    }
    const unsigned nblk = (unsigned)((n + 255) / 256), nscan = (unsigned)((n + SCAN_CH - 1) / SCAN_CH);
    if (nl->pw.ensure(3 * (size_t)n) || nl->wrap.ensure(3 * (size_t)n) || nl->sf.ensure(3 * (size_t)n) ||
        nl->bin.ensure(n) || nl->idx.ensure(n) || nl->keys.ensure(n) || nl->bin_atoms.ensure(n) ||
        nl->cnt.ensure(n) || nl->dmail.ensure(1) || nl->bmm.ensure((size_t)nblk * 6) || nl->sp.ensure(3 * (size_t)n) ||
        nl->sx.ensure(3 * (size_t)n) || nl->sw.ensure(3 * (size_t)n) || nl->off.ensure((size_t)n + 1) ||
        nl->bsum.ensure(nscan))
        return -1;
    int32_t* flag = reinterpret_cast<int32_t*>(&nl->dmail.p->flag);
    // the flags and numbers of the stages so far, in host memory
    auto read_back = [&]() -> int {
        HIP_TRY(hipMemcpyAsync(nl->mail, nl->dmail.p, sizeof(ace_nbrlist::Mail), hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        if (nl->mail->flag & 4) return set_err("ace_nbrlist_build: positions must be finite");
        if (nl->mail->flag & 8) return set_err("ace_nbrlist_build: positions too far outside the cell");
        return 0;
    };
    // wrap and bin on the device: fractional coordinates, extents (for open axes)
    NbrFracArgs fa{};
    for (int q = 0; q < 9; ++q) {
        fa.cell[q] = geo.cell[q];
        fa.inv[q] = geo.inv[q];
    }
    for (int d = 0; d < 3; ++d) fa.pbc[d] = geo.pbc[d];
    fa.natoms = n;
    hipLaunchKernelGGL(k_nbr_zero, dim3(1), dim3(64), 0, st, flag, (int)(2 * sizeof(int64_t) / sizeof(int32_t)));
    hipLaunchKernelGGL(k_nbr_frac, dim3(nblk), dim3(256), 0, st, fa, pos, nl->sf.p, nl->wrap.p, nl->pw.p, nl->bmm.p,
                       flag);
    HIP_TRY(hipGetLastError());
    // The bins of a cell that is periodic along all axes do not depend on the
    // positions: only open axes wait for their extents here.  Positions found
    // invalid above are wrapped to some bin and not searched; the next read back
    // refuses them.
    const bool open = !(geo.pbc[0] && geo.pbc[1] && geo.pbc[2]);
    if (open) {
        hipLaunchKernelGGL(k_nbr_minmax, dim3(1), dim3(256), 0, st, (int)nblk, (const double*)nl->bmm.p,
                           nl->dmail.p->mm);
        HIP_TRY(hipGetLastError());
        if (read_back()) return -1;
    }
    acehost::NbrGrid& g = nl->g;
    const std::string perr = acehost::nbr_params(geo, natoms, nl->mail->mm, nl->mail->mm + 3, g);
    if (!perr.empty()) return set_err("ace_nbrlist_build: " + perr);
    const int nbins = g.nbins();
    if (nl->bin_start.ensure((size_t)nbins + 1)) return -1;
    NbrBinArgs ba{};
    for (int d = 0; d < 3; ++d) {
        ba.nb[d] = g.nb[d];
        ba.s0[d] = g.s0[d];
        ba.w[d] = g.w[d];
    }
    ba.natoms = n;
    hipLaunchKernelGGL(k_nbr_bin, dim3(nblk), dim3(256), 0, st, ba, (const double*)nl->sf.p, nl->bin.p, nl->idx.p);
    HIP_TRY(hipGetLastError());
    // stable sort of the atoms by bin (ascending atom index within a bin)
    int end_bit = 1;
    while (end_bit < 31 && (1 << end_bit) < nbins) ++end_bit;
    size_t tmp_bytes = 0;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, nl->bin.p, nl->keys.p, nl->idx.p,
                                               nl->bin_atoms.p, n, 0, end_bit, st));
    if (nl->sort_tmp.ensure(std::max<size_t>(tmp_bytes, 1))) return -1;
    HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nl->sort_tmp.p, tmp_bytes, nl->bin.p, nl->keys.p, nl->idx.p,
                                               nl->bin_atoms.p, n, 0, end_bit, st));
    hipLaunchKernelGGL(k_nbr_binstart, dim3((unsigned)((nbins + 1 + 255) / 256)), dim3(256), 0, st, nbins, n,
                       (const int32_t*)nl->keys.p, nl->bin_start.p);
    HIP_TRY(hipGetLastError());
    hipLaunchKernelGGL(k_nbr_gather, dim3(nblk), dim3(256), 0, st, n, (const int32_t*)nl->bin_atoms.p,
                       (const double*)nl->pw.p, pos, (const int32_t*)nl->wrap.p, nl->sp.p, nl->sx.p, nl->sw.p);
    const NbrArgs a = grid_args(nl, cell);
    const int64_t nwg = ((int64_t)n + 3) / 4;
    in_launches(nwg, [&](int first, dim3 grid) {
        hipLaunchKernelGGL(k_nbr_search<false>, grid, dim3(256), 0, st, a, first, nl->cnt.p, nullptr, (int64_t)0,
                           nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, flag);
    });
    hipLaunchKernelGGL(k_nbr_scan_sum, dim3(nscan), dim3(256), 0, st, n, (const int32_t*)nl->cnt.p, nl->bsum.p);
    hipLaunchKernelGGL(k_nbr_scan, dim3(nscan), dim3(256), 0, st, n, (const int32_t*)nl->cnt.p,
                       (const int64_t*)nl->bsum.p, nl->off.p, &nl->dmail.p->total);
    HIP_TRY(hipGetLastError());
    if (read_back()) return -1;
    const int64_t total = nl->mail->total;
    if (total >= ((int64_t)1 << 31)) return set_err("ace_nbrlist_build: more than 2^31 - 1 neighbour entries");
    *nnbr_out = total;
    if (total > capacity) {
        set_err("ace_nbrlist_build: capacity " + std::to_string(capacity) + " < " + std::to_string(total) +
                " neighbour entries (*nnbr_out holds the size needed)");
        return ACE_ERR_CAPACITY;
    }
    in_launches(nwg, [&](int first, dim3 grid) {
        hipLaunchKernelGGL(k_nbr_search<true>, grid, dim3(256), 0, st, a, first, nullptr, (const int32_t*)nl->off.p,
                           total, env_offsets, nbr_j, shift, xyz, atom_species, nbr_species, flag);
    });
    HIP_TRY(hipGetLastError());
    if (rev && total > 0) {
        in_launches(nwg, [&](int first, dim3 grid) {
            hipLaunchKernelGGL(k_nbr_rev, grid, dim3(256), 0, st, n, first, (const int32_t*)nl->bin_atoms.p,
                               (const int32_t*)nl->off.p, (const int32_t*)nbr_j, (const int32_t*)shift, total, rev,
                               flag);
        });
        HIP_TRY(hipGetLastError());
    }
    if (read_back()) return -1;
    if (nl->mail->flag & 1) return set_err("ace_nbrlist_build: fill pass disagrees with the count pass");
    if (nl->mail->flag & 2) return set_err("ace_nbrlist_build: neighbour list not symmetric (reverse entry missing)");
    return 0;
}

extern "C" int ace_nbrlist_update(ace_nbrlist* nl, int64_t natoms, const double* pos, const double* cell,
                                  int64_t nnbr, const int32_t* env_offsets, const int32_t* nbr_j,
                                  const int32_t* shift, double* xyz, void* stream) {
    if (!nl || !cell) return set_err("ace_nbrlist_update: null argument");
    if (natoms < 0 || natoms >= ((int64_t)1 << 31) - 1 || nnbr < 0 || nnbr >= ((int64_t)1 << 31))
        return set_err("ace_nbrlist_update: size out of range");
    if (nnbr == 0) return 0;
    if (!pos || !env_offsets || !nbr_j || !shift || !xyz || natoms == 0)
        return set_err("ace_nbrlist_update: null argument");
    HIP_TRY(hipSetDevice(nl->device));
    NbrArgs a{};
    for (int q = 0; q < 9; ++q) a.cell[q] = cell[q];
    in_launches((natoms + 15) / 16, [&](int first, dim3 grid) {
        hipLaunchKernelGGL(k_nbr_update, grid, dim3(256), 0, (hipStream_t)stream, (int)natoms, first, a, pos,
                           env_offsets, nbr_j, shift, nnbr, xyz);
    });
    HIP_TRY(hipGetLastError());
    return 0;
}

extern "C" int ace_nbrlist_forces(ace_nbrlist* nl, int64_t natoms, const int32_t* env_offsets, const int32_t* rev,
                                  int64_t nnbr, const double* xyz, const double* dE_dr, double* F, double* virial,
                                  void* stream) {
    if (!nl) return set_err("ace_nbrlist_forces: null argument");
    if (natoms < 0 || natoms >= ((int64_t)1 << 31) - 1 || nnbr < 0 || nnbr >= ((int64_t)1 << 31))
        return set_err("ace_nbrlist_forces: size out of range");
    if (natoms > 0 && (!env_offsets || !F)) return set_err("ace_nbrlist_forces: null argument");
    if (nnbr > 0 && (!rev || !dE_dr)) return set_err("ace_nbrlist_forces: null argument");
    if (virial && nnbr > 0 && !xyz) return set_err("ace_nbrlist_forces: the virial needs xyz");
    HIP_TRY(hipSetDevice(nl->device));
    hipStream_t st = (hipStream_t)stream;
    const int n = (int)natoms;
    if (n == 0) {
        if (virial) hipLaunchKernelGGL(k_nbr_vsum, dim3(1), dim3(576), 0, st, 0, (const double*)nullptr, virial);
        HIP_TRY(hipGetLastError());
        return 0;
    }
    const int64_t ngrp = ((int64_t)n + FA_ATOMS - 1) / FA_ATOMS;
    const int per = (int)((ngrp + FA_BLOCKS - 1) / FA_BLOCKS);
    const int nblk = (int)((ngrp + per - 1) / per);
    if (virial) {
        // a graph keeps its block: fewer atoms may take more workgroups (32,768
        // 2,048, 40,000 1,250)
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        HIP_TRY(hipStreamIsCapturing(st, &cap));
        if (nl->vpart.ensure((size_t)nblk * 9, cap != hipStreamCaptureStatusNone)) return -1;
    }
    hipLaunchKernelGGL(k_nbr_forces, dim3((unsigned)nblk), dim3(256), 0, st, n, per, env_offsets, rev, nnbr, dE_dr, xyz, F,
                       virial ? nl->vpart.p : nullptr);
    HIP_TRY(hipGetLastError());
    if (virial) {
        hipLaunchKernelGGL(k_nbr_vsum, dim3(1), dim3(576), 0, st, nblk, (const double*)nl->vpart.p, virial);
        HIP_TRY(hipGetLastError());
    }
    return 0;
}

extern "C" int ace_nbrlist_forces_multi(ace_nbrlist* nl, int64_t natoms, const int32_t* env_offsets,
                                        const int32_t* rev, int64_t nnbr, int64_t nvec, const double* g, double* F,
                                        void* stream) {
    if (!nl) return set_err("ace_nbrlist_forces_multi: null argument");
    if (natoms < 0 || natoms >= ((int64_t)1 << 31) - 1 || nnbr < 0 || nnbr >= ((int64_t)1 << 31) || nvec < 0)
        return set_err("ace_nbrlist_forces_multi: size out of range");
    const int64_t n = natoms * nvec;
    if (n == 0) return 0;
    if (!env_offsets || !F || (nnbr > 0 && (!rev || !g))) return set_err("ace_nbrlist_forces_multi: null argument");
    HIP_TRY(hipSetDevice(nl->device));
    hipLaunchKernelGGL(k_nbr_forces_multi, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (int)natoms, env_offsets, rev, nvec, g, F);
    HIP_TRY(hipGetLastError());
    return 0;
}
