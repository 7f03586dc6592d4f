// Force kernels of the DMD force field (ForceField_DMD_I::force_calc,
// src/ff_dmd_I.cpp:88-450, and energy_calc, :454-668).
//
// The reference scatters every half-list pair into both ends (E[j] +=,
// f[j] -=).  Here one wavefront owns one site and never writes another
// site's row; what a pair owes its partner goes to a per-pair share slot at
// the pair's position in the partner's reverse list:
//   pass 1   the site's list entries inside the quadrature cut are staged in
//            LDS; lanes (pair, type pair, part) evaluate the Gauss-Hermite
//            averaged density and pair terms, the site's own density sums
//            stay in registers, the partner's density share (nt doubles)
//            goes to its share slot, and the r- and alpha-derivatives go to
//            the pair's derivative record (PairRec);
//   embed    a lane group per site adds the density shares of the sites that
//            list it (reverse CSR, ascending pair index), then F(rho_bar), F',
//            the per-site energy terms and the alpha entropic force;
//   pass 2   half a wavefront per site, one lane per pair: the lane combines the
//            pair's derivative record with F' of both ends into the site's force
//            row and the partner's force share (3 + nt doubles);
//   gather   a lane group per site adds its force shares (reverse CSR).
// No floating-point atomics: every sum has a fixed order, so results are
// bitwise reproducible run to run.  Energy and virial partials are written per
// wavefront and reduced in two fixed-shape stages.
//
// Q is the arithmetic of the quadrature (double, or float for the mixed
// mode whose point sums run in FP32 with FP32 accumulation); site-level sums,
// F(rho_bar), energies and forces are FP64 in both.
#pragma once
#include "dmd_common.hpp"

// The force kernels do not need the reference's bitwise operation order (the
// bar is 1e-12 relative), so a*b+c may fuse into FMA here; the geometry
// kernels, which must reproduce the reference's list bit for bit, are
// compiled before this region with contraction off.
#pragma clang fp contract(fast)

namespace mappdmd {

constexpr int kBlock = 256;
constexpr int kQuadRow = 8;  // rho c0..c3, r*phi c0..c3 of one ordered type pair
// The quadrature table is bin-major, quad[m][tp][kQuadRow]: the rows of all
// type pairs at one grid row are adjacent, so the type pairs of a pair that
// evaluate at the same distance (the middle node of an odd rule, t = r) share
// cache lines.  Type pair tp starts at quad + tp * kQuadRow; consecutive rows
// of one type pair are quad_stride(nt) elements apart.
__host__ __device__ constexpr int quad_stride(int nt) { return nt * nt * kQuadRow; }

__host__ __device__ constexpr int type2rho(int nt, int i, int j) { return j * nt + i; }
__host__ __device__ constexpr int type2phi(int i, int j) {
    return i < j ? (j + 1) * j / 2 + i : (i + 1) * i / 2 + j;
}

template <typename T>
__device__ __forceinline__ T horner3(const T* c, T p) {
    return fma(fma(fma(c[3], p, c[2]), p, c[1]), p, c[0]);
}

// classical EAM values for alpha >= alpha_max (src/ff_dmd_I.cpp:261-310), FP64
__device__ __forceinline__ void classical_pair(const FFParams<double>& P, double rsq, double r_inv,
                                               const double* __restrict__ rho7, const double* __restrict__ phi7,
                                               bool want_phi, double* g, double* f) {
    double r = sqrt(rsq);
    double p = r * P.dr_inv;
    int m = (int)p;
    m = m < P.nr - 2 ? m : P.nr - 2;
    p -= m;
    p = p < 1.0 ? p : 1.0;
    double p2 = p * p, p3 = p2 * p;
    if (want_phi) {
        const double* c = phi7 + (size_t)m * 7;
        double z2p = c[6] * p2 + c[5] * p + c[4];
        double z2 = c[3] * p3 + c[2] * p2 + c[1] * p + c[0];
        f[0] = z2 * r_inv;
        f[2] = 0.0;
        f[1] = (z2p - z2 * r_inv) * r_inv;
    }
    const double* c = rho7 + (size_t)m * 7;
    g[0] = c[3] * p3 + c[2] * p2 + c[1] * p + c[0];
    g[2] = 0.0;
    g[1] = c[6] * p2 + c[5] * p + c[4];
}

__device__ __forceinline__ double calc_ent(double x) {
    if (x < 1.0e-8 || 0.99999999 < x) return 0.0;
    return x * log(x) + (1 - x) * log(1 - x);
}

// F(rho_bar), F', F'' by the quartic spline with linear extrapolation above
// rho_max (src/ff_dmd_I.cpp:322-341, :2484-2491)
__device__ __forceinline__ void embed_F(const FFParams<double>& P, const double* __restrict__ F9, int type,
                                        double e, double* Fv, double* dF, double* ddF) {
    double p = e * P.drho_inv;
    int m = (int)p;
    m = m < P.nr - 2 ? m : P.nr - 2;
    m = m < 0 ? 0 : m;  // negative density: outside the reference's defined range
    p -= m;
    p = p < 1.0 ? p : 1.0;
    double p2 = p * p, p3 = p2 * p, p4 = p3 * p;
    const double* c = F9 + ((size_t)type * (P.nrho + 1) + m) * 9;
    double t0 = c[4] * p4 + c[3] * p3 + c[2] * p2 + c[1] * p + c[0];
    double t1 = c[8] * p3 + c[7] * p2 + c[6] * p + c[5];
    if (e > P.rho_max) t0 += t1 * (e - P.rho_max);
    *Fv = t0;
    *dF = t1;
    if (ddF) *ddF = (3.0 * c[8] * p2 + c[7] * p + c[6]) * P.drho_inv;
}

// XCD-aware block order: consecutive atoms (spatial neighbours) land on the
// same XCD, whose L2 then holds their shared neighbour rows.  Dispatch places
// block b on XCD b % 8.
__device__ __forceinline__ int xcd_block(int nblocks) {
    const int b = blockIdx.x;
    const int per = (nblocks + 7) / 8;
    const int xcd = b & 7, k = b >> 3;
    const int full = nblocks - 8 * (per - 1);  // XCDs that receive 'per' blocks
    int start = xcd < full ? xcd * per : full * per + (xcd - full) * (per - 1);
    return start + k;
}

struct PairBufs {
    const int* off;    // half list
    const int2* nlrp;  // {partner, its position in the partner's reverse list or -1}
    const int* roff;   // reverse list: the owners of the pairs that list a site
};

// Which half-list entries lay inside the quadrature cut at the last pass 1: the
// top bit of the partner index in the packed list {partner, reverse position},
// read with the entry at no extra cost, and the top bit of the owner's index in
// the partner's reverse list, by which the force gather knows the shares that
// count.  Both are written only when an entry enters or leaves the cut.  The
// density share of an entry outside reads zero in the embedding: it is cleared
// when the list is built and again only when the entry leaves (the embedding
// reading the owners too took 0.29 ms in place of 0.21 at 1,048,576 sites).
constexpr int kInsideBit = (int)0x80000000u;
__device__ __forceinline__ int list_partner(int2 e) { return e.x & 0x7fffffff; }
struct CutState {
    int2* nlrp;
    int* rowner;
    // entry pc of owner i (as read: e, partner jc) is inside the cut now or not: record a
    // change; on leaving, clear the density share of an owned partner
    template <int NT>
    __device__ __forceinline__ void update(int pc, int2 e, bool in, int i, int jc, int natms, double* pairE) const {
        const bool was = (e.x & kInsideBit) != 0;
        if (was != in) {
            nlrp[pc].x = in ? (jc | kInsideBit) : jc;
            if (jc < natms) {
                rowner[e.y] = in ? (i | kInsideBit) : i;
                if (!in) {
#pragma unroll
                    for (int t = 0; t < NT; ++t) pairE[(size_t)e.y * NT + t] = 0.0;
                }
            }
        }
    }
};

// Force share of a pair, kLen doubles at the pair's position in the partner's reverse
// list: {S, alpha forces of the partner's types}, the force on the owner being
// S (x_owner - x_partner); padded to whole 16-byte pieces (two types: one 32-byte
// sector, where the three components and two alpha forces took two writes of 32 and
// 8 bytes).
template <int NT>
struct ForceShare {
    static constexpr int kLen = (1 + NT + 1) / 2 * 2;
};

// ---------------------------------------------------------------- lane exchanges
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    int lo = __double2loint(v), hi = __double2hiint(v);
    lo = __builtin_amdgcn_update_dpp(0, lo, CTRL, 0xF, 0xF, false);
    hi = __builtin_amdgcn_update_dpp(0, hi, CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
constexpr int kDppXor1 = 0xB1;       // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;       // quad_perm [2,3,0,1]
constexpr int kDppRowRor8 = 0x128;   // row_ror:8 (rotate by 8 lanes within a row of 16)
constexpr int kDppRowRor4 = 0x124;   // row_ror:4
constexpr int kDppRowRor12 = 0x12C;  // row_ror:12: lane l reads lane (l + 4) mod 16 of its row

// v summed with the same lane of the paired row (rows 0+1, 2+3: permlane16
// swap) or of the other half of the wavefront (permlane32 swap); both lanes of
// a pair add in the same order, so they hold the same bits
template <bool HALVES>
__device__ __forceinline__ double row_pair_sum(double v) {
    const int lo = __double2loint(v), hi = __double2hiint(v);
    const auto a = HALVES ? __builtin_amdgcn_permlane32_swap(lo, lo, false, false)
                          : __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto b = HALVES ? __builtin_amdgcn_permlane32_swap(hi, hi, false, false)
                          : __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __hiloint2double(b[0], a[0]) + __hiloint2double(b[1], a[1]);
}

// which branch of the reference applies to the pair width alpha = 1/ia:
// 1 quadrature (alpha_min < alpha < alpha_max), 2 classical (alpha >= alpha_max),
// 0 nothing.  ia = 1/alpha_i + 1/alpha_j equals the reference's
// alpha_i alpha_j / (alpha_i + alpha_j) to within two ulp; within 1e-12 of a
// bound the reference's own expression decides.
__device__ __forceinline__ int alpha_branch(const FFParams<double>& P, double ia, double ai, double aj) {
    const double lo = P.inv_amax, hi = P.inv_amin;
    if (fabs(ia - hi) <= 1e-12 * hi || fabs(ia - lo) <= 1e-12 * lo) {
        const double a = (ai * aj) / (ai + aj);
        return (P.alpha_min < a && a < P.alpha_max) ? 1 : (P.alpha_max <= a ? 2 : 0);
    }
    return (ia > lo && ia < hi) ? 1 : (ia <= lo ? 2 : 0);
}

// Gauss-Hermite average with sqrt(alpha) = asq and 1/alpha = ia given
// (src/ff_dmd_I.cpp:180-242); no divisions and no branches: a point outside
// the window (xi_k <= lower or xi_k >= upper) or a rule beyond the cutoff
// (lower >= xi_max) contributes zero, its row index being clamped in range.
// g, f = {value, d/dr, d/dalpha}; returns whether the rule is inside.
template <typename Q, int NQ, bool DERIV>
__device__ __forceinline__ bool gh_avg(const FFParams<Q>& P, Q r, Q r_inv, Q asq, Q ia, const Q* __restrict__ tab,
                                       int stride, Q* g, Q* f) {
    const int nq = NQ > 0 ? NQ : P.no_i;
    const Q inv = ia * asq;
    const Q upper = (r + P.rc) * asq;
    const Q lower = (r - P.rc) * asq;
    const bool rule = lower < P.xi[nq - 1];
    Q g0 = 0, g1 = 0, g2 = 0, f0 = 0, f1 = 0, f2 = 0;
#pragma unroll
    for (int k = 0; k < (NQ > 0 ? NQ : kMaxPoints); ++k) {
        if (NQ == 0 && k >= nq) break;
        const Q xk = P.xi[k];
        const bool inside = rule && xk > lower && xk < upper;
        const Q t = r - xk * inv;
        Q p = fabs(t) * P.dr_inv;
        int m = (int)p;
        m = m < P.nr - 2 ? m : P.nr - 2;
        m = m > 0 ? m : 0;
        p -= (Q)m;
        p = p < Q(1) ? p : Q(1);
        const Q* row = tab + (size_t)m * stride;
        Q rv = horner3(row, p) * t;
        Q pv = horner3(row + 4, p);
        pv = t < Q(0) ? -pv : pv;
        rv = inside ? rv : Q(0);
        pv = inside ? pv : Q(0);
        g0 += P.w0[k] * rv;
        f0 += P.w0[k] * pv;
        if (DERIV) {
            g1 += P.w1[k] * rv;
            g2 += P.w2[k] * rv;
            f1 += P.w1[k] * pv;
            f2 += P.w2[k] * pv;
        }
    }
    const Q sc = Q(kPiInSq) * r_inv;
    g0 *= sc;
    f0 *= sc;
    g[0] = g0;
    f[0] = f0;
    if (DERIV) {
        g1 *= sc;
        g2 *= sc;
        f1 *= sc;
        f2 *= sc;
        g[1] = -g0 * r_inv - Q(2) * asq * g1;
        g[2] = (Q(0.5) * g0 - g2) * ia;
        f[1] = -f0 * r_inv - Q(2) * asq * f1;
        f[2] = (Q(0.5) * f0 - f2) * ia;
    }
    return rule;
}

// per (site, type) record {alpha, c, 1/alpha, dE}, ghosts included
__global__ void k_pack_atoms(const double* __restrict__ alpha, const double* __restrict__ conc, long n,
                             double4* __restrict__ rec) {
    long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k < n) {
        const double a = alpha[k];
        rec[k] = make_double4(a, conc[k], 1.0 / a, 0.0);
    }
}

// sum over the wavefront, the same value in every lane: a DPP rotation tree
// inside each row of 16 lanes, then the four row sums in a fixed order
__device__ __forceinline__ double read_lane(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_f64<kDppRowRor8>(v);
    v += dpp_f64<kDppRowRor4>(v);
    v += dpp_f64<kDppXor2>(v);
    v += dpp_f64<kDppXor1>(v);
    return (read_lane(v, 0) + read_lane(v, 16)) + (read_lane(v, 32) + read_lane(v, 48));
}

// deterministic per-block sum of NV wave partials (lane 0 of each wave holds them)
template <int NV, int MAXW = kBlock / 64>
__device__ __forceinline__ void block_store_waves(const double* v, double* __restrict__ out) {
    __shared__ double sh[MAXW][NV];  // blockDim.x <= 64 * MAXW
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, nw = blockDim.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) sh[w][k] = v[k];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            double s = 0.0;
            for (int q = 0; q < nw; ++q) s += sh[q][k];
            out[(size_t)blockIdx.x * NV + k] = s;
        }
    }
}

// deterministic sum of NV doubles over a block of kBlock threads: a fixed tree in each
// wavefront, then the wavefronts in order; thread k writes out[blockIdx.x*NV + k]
template <int NV>
__device__ __forceinline__ void block_sum_store(const double* v, double* __restrict__ out) {
    __shared__ double sh[kBlock / 64][NV];
    const int w = threadIdx.x >> 6;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double t = wave_sum(v[k]);
        if ((threadIdx.x & 63) == 0) sh[w][k] = t;
    }
    __syncthreads();
    if (threadIdx.x < NV) {
        double t = 0.0;
#pragma unroll
        for (int q = 0; q < kBlock / 64; ++q) t += sh[q][threadIdx.x];
        out[(size_t)blockIdx.x * NV + threadIdx.x] = t;
    }
}

// Per-wavefront partials without a block barrier: lane 0 of wavefront w of
// block b stores the wave's NV totals at out[(b * waves per block + w) * NV].
// A wave that finishes early leaves at once instead of holding its slot until
// the block's slowest wave reaches a barrier.
template <int NV>
__device__ __forceinline__ void wave_store(const double* v, double* __restrict__ out) {
    if ((threadIdx.x & 63) == 0) {
        const size_t w = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
#pragma unroll
        for (int k = 0; k < NV; ++k) out[w * NV + k] = v[k];
    }
}

// Sites of one group of LANES consecutive lanes (a wavefront, or half of one).
// Dispatch places block b on XCD b % 8; the sites are split into 8 contiguous
// ranges, one per XCD, so spatial neighbours share an L2, and the groups of an
// XCD stride through its range.  With one group per site (the default grid)
// each group takes one site; a smaller grid makes the launch persistent.
// Every group of a block runs the same number of iterations or fewer; kernels
// that synchronise a block inside the loop must not use it.
template <int LANES = 64>
struct SiteLoop {
    int first, end, stride;
    // wpb: wavefronts per block (an argument, because reading blockDim is a load)
    __device__ __forceinline__ SiteLoop(int n, int wpb) {
        const int gpb = wpb * (64 / LANES), g = threadIdx.x / LANES;
        const int nb = gridDim.x, b = blockIdx.x;
        if (nb >= 8) {
            const int x = b & 7, lb = b >> 3;
            const int nbx = (nb - x + 7) >> 3;
            first = (int)((long long)n * x / 8) + lb * gpb + g;
            end = (int)((long long)n * (x + 1) / 8);
            stride = nbx * gpb;
        } else {
            first = b * gpb + g;
            end = n;
            stride = nb * gpb;
        }
    }
};

// Pairs inside the cut, packed.  Each lane holds one list entry of a 64-entry
// chunk and whether it lies inside the cut; pack_dest gives the lane the entry
// moves to (inside entries to their rank in list order, the others after
// them), and packed() moves any per-entry value there through ds_permute, so
// lane l < count then holds the l-th inside entry's values.
__device__ __forceinline__ int pack_dest(bool in, int* count) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(in);
    const int cnt = __popcll(m);
    const int lane = threadIdx.x & 63;
    const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
    *count = cnt;
    return in ? rank : cnt + (lane - rank);
}
__device__ __forceinline__ int packed(int dest, int v) { return __builtin_amdgcn_ds_permute(dest << 2, v); }
__device__ __forceinline__ int pack_in_range(int p, bool in, int* out) {
    int cnt;
    *out = packed(pack_dest(in, &cnt), p);
    return cnt;
}

// ---------------------------------------------------------------- pass 1
// Wave per site, PARTS lanes per ordered type pair: lane l = k*LPP + q*PARTS + part.
// A spline row of one type pair holds rho c0..c3 and r*phi c0..c3.
// PARTS = 4: the four part lanes load one quarter each (16 bytes in FP64), so
// each table row costs one cache-line access; each evaluates half of a cubic
// (c_lo + c_hi p) and one DPP exchange joins the halves (val = h0 + p^2 h1) in
// lane part 0 (rho) and lane part 2 (phi).
// PARTS = 2: part 0 loads the rho half of the row and evaluates its cubic,
// part 1 the phi half: twice the pairs per wavefront iteration and half the
// lanes repeating the point set-up, for one more cache-line access per row in
// FP64 (in FP32 a half row is one 16-byte load).
// PARTS = 1: one lane loads the whole row and evaluates both cubics.
// Every variant evaluates a cubic as (c0 + c1 p) + p^2 (c2 + c3 p), so the
// results do not depend on the variant.
// The rho and phi lanes then carry the weighted Gauss-Hermite sums of their
// function.
//
// The derivative records stream out with nontemporal stores (whole lines, read
// back only after the whole pass, so they are kept from displacing the spline
// tables in L2); the partner shares, 16 bytes at scattered reverse positions,
// use ordinary stores so that L2 merges them into lines before they leave.
//
// ENERGY_ONLY restates energy_calc's triangle (jtype starts at itype, so phi
// only for itype == jtype; src/ff_dmd_I.cpp:508).  The partner's density share
// goes to pairE in reverse-list order (nlrp[].y), so the embedding reads it
// contiguously.  Unless ENERGY_ONLY, the rho lane stores {drho/dr, drho/dalpha}
// and the phi lane {dphi/dr, dphi/dalpha} in the pair's record (PairRec; the
// reference's per-pair caches, src/ff_dmd_I.cpp:227-242, restricted to what the
// back-pass reads), for the site's pairs inside the quadrature cut, whose number
// goes to info with the site's list offset.  The phi lanes of the type pairs it < jt
// have no value of their own: the back-pass takes their phi from the transposed pair.
//
// Lanes of pass 1.  In general lane l works on pair slot k = l / kLPP and, within it,
// on part prt of type pair q: lane k*kLPP + q*PARTS + prt.
// Three types with two lanes per type pair have their own map: of the 18 lanes of
// a pair 3 would do nothing (the phi of it < jt), and 3 pairs fill 54 lanes.  With
// the 6 type pairs it >= jt as (rho, phi) lanes, then the 3 densities it < jt, a pair
// takes 15 lanes, 4 pairs fill 60, and the last 4 lanes write the 4 partners: pass 1
// at 114,840 sites 0.77 -> 0.64 ms.
template <int NT, int PARTS = 4>
struct Pass1Map {
    static constexpr bool kCompact = NT == 3 && PARTS == 2;
    static constexpr int kLPP = kCompact ? 15 : NT * NT * PARTS;
    static constexpr int kPPW = 64 / kLPP;
    int k, it, jt, prt;
    bool on;  // the lane evaluates
    __device__ __forceinline__ explicit Pass1Map(int lane) {
        k = lane / kLPP;
        on = k < kPPW;
        const int l = lane % kLPP;
        if constexpr (kCompact) {
            if (!on) k = lane - kLPP * kPPW;  // the lane that writes slot k's partner
            const int c = l < 12 ? l / 2 : 0;
            prt = l < 12 ? l % 2 : 0;
            it = c >= 3 ? 2 : (c >= 1 ? 1 : 0);
            jt = c - it * (it + 1) / 2;
            if (l >= 12) {
                it = l == 14 ? 1 : 0;
                jt = l == 12 ? 1 : 2;
            }
        } else {
            const int q = l / PARTS;
            prt = l % PARTS;
            it = q / NT;
            jt = q % NT;
        }
    }
    // lane of the density of type pair (a, b) within a pair's lanes
    __device__ static int rho_at(int a, int b) {
        if constexpr (kCompact) return a >= b ? a * (a + 1) + 2 * b : (a == 0 ? 11 + b : 14);
        else return (a * NT + b) * PARTS;
    }
};

// The records of the pairs of a site inside the cut, what pass 1 leaves for
// pass 2.  A record has kComps components of two values of the quadrature type:
// {drho/dr, drho/dalpha} of every ordered type pair q = it*NT + jt, then
// {dphi/dr, dphi/dalpha} of the type pairs it >= jt only (the back-pass uses the
// phi of (it, jt) for it >= jt on both (it, jt) and (jt, it), as
// ForceField_DMD_I::force_calc reads one phi cache slot for both orders,
// src/ff_dmd_I.cpp:244-248, :376), then {partner, reverse position or -1 for a
// ghost partner} as two ints.  The k-th inside pair of site i is pair k % kG of
// the site's group k / kG; a group holds its kG pairs component by component, so
// a component of a group is one run: pass 1's lanes (pair, type pair) write it
// whole, and pass 2's lanes (one pair each) read 16-byte pieces of the same runs
// instead of 16-byte pieces 112 bytes apart.  A run is 64 bytes, or what one round
// of pass 1 fills (two lanes per type pair) where that is less: runs of 64 bytes
// that two or four rounds wrote in parts, past L2, cost four types more than the
// rest gained -- 131,072 sites, 3 points, FP64 2.15 ms (1.89 with a record in one
// piece) and FP32 2.01 (1.64); runs of 32 and 16 bytes, two pairs, 1.69 and 1.22.
// Site i's groups start at off[i] / kG + i, which leaves room for every listed
// pair in whole groups.
template <int NT, typename Q>
struct PairRec {
    static constexpr int kRun = 64 / (2 * (int)sizeof(Q)), kRound = Pass1Map<NT, 2>::kPPW;
    static constexpr int kG = kRun < kRound ? kRun : kRound;
    static constexpr int kComps = NT * NT + NT * (NT + 1) / 2 + 1;
    __host__ __device__ static constexpr int rho(int q) { return q; }
    __host__ __device__ static constexpr int phi(int it, int jt) { return NT * NT + type2phi(it, jt); }
    static constexpr int kIdx = kComps - 1;
    // groups to hold npairs listed pairs of natms sites
    __host__ __device__ static size_t groups(long npairs, long natms) { return (size_t)(npairs / kG + natms + 1); }
    // first element ({value, value}) of site i's records
    __device__ static size_t first(int off_i, int i) { return ((size_t)(off_i / kG) + (size_t)i) * (kG * kComps); }
    // element of component c of the site's pair k, relative to first()
    __device__ static int elem(int k, int c) { return (k / kG) * (kG * kComps) + c * kG + k % kG; }
};

template <typename Q>
struct Vec2;
template <>
struct Vec2<double> {
    using T = double2;
    // two ints in the bits of one component
    static __device__ __forceinline__ double2 ints(int a, int b) { return make_double2(__hiloint2double(b, a), 0.0); }
    static __device__ __forceinline__ int2 ints(double2 v) { return make_int2(__double2loint(v.x), __double2hiint(v.x)); }
};
template <>
struct Vec2<float> {
    using T = float2;
    static __device__ __forceinline__ float2 ints(int a, int b) { return make_float2(__int_as_float(a), __int_as_float(b)); }
    static __device__ __forceinline__ int2 ints(float2 v) { return make_int2(__float_as_int(v.x), __float_as_int(v.y)); }
};
// streaming store of one component (whole lines, read back only after the pass)
template <typename Q2>
__device__ __forceinline__ void store_comp(Q2* p, Q2 v) {
    __builtin_nontemporal_store(v.x, &p->x);
    __builtin_nontemporal_store(v.y, &p->y);
}

template <typename Q>
__device__ __forceinline__ Q dpp_xor1_q(Q v);
template <>
__device__ __forceinline__ double dpp_xor1_q<double>(double v) {
    return dpp_f64<kDppXor1>(v);
}
template <>
__device__ __forceinline__ float dpp_xor1_q<float>(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kDppXor1, 0xF, 0xF, false));
}


// Per-wavefront LDS stage of pass 1 (dynamic shared memory, kBytes per wavefront):
// for the inside entries of the current chunk, in rank order, {r^2, 1/r},
// {1/alpha, c} of the partner per type, and {partner, reverse position or -1}.
template <int NT>
struct Pass1Stage {
    static constexpr int kBytes = 64 * (16 + 16 * NT + 8);
    double2* geo;
    double2* typ;
    int2* idx;
    __device__ __forceinline__ explicit Pass1Stage(int wave) {
        extern __shared__ __attribute__((aligned(32))) unsigned char pass1_lds[];
        unsigned char* base = pass1_lds + (size_t)wave * kBytes;
        geo = reinterpret_cast<double2*>(base);
        typ = geo + 64;
        idx = reinterpret_cast<int2*>(typ + 64 * NT);
    }
};

// Quadrature-table rows through buffer loads: each point costs a 32-bit byte
// offset (one multiply-add) instead of a 64-bit address, and the resource's
// size bounds every access.
template <typename Q2>
struct RowLoad;
template <>
struct RowLoad<double2> {
    static __device__ __forceinline__ double2 get(__amdgpu_buffer_rsrc_t r, int off) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
        return make_double2(__hiloint2double((int)v[1], (int)v[0]), __hiloint2double((int)v[3], (int)v[2]));
    }
};
template <>
struct RowLoad<float2> {
    static __device__ __forceinline__ float2 get(__amdgpu_buffer_rsrc_t r, int off) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
        return make_float2(__int_as_float((int)v[0]), __int_as_float((int)v[1]));
    }
};
// raw buffer (stride 0, 32-bit data format) over n bytes
__device__ __forceinline__ __amdgpu_buffer_rsrc_t raw_rsrc(const void* p, int nbytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, nbytes, 0x00020000);
}

constexpr int kNoRow = 0x60000000;  // a row offset beyond any table (its reads give 0)

// 1/x by the hardware estimate and two Newton steps (x normal and positive here)
__device__ __forceinline__ double rcp_nr(double x) {
    double y = __builtin_amdgcn_rcp(x);
    y = y * (2.0 - x * y);
    return y * (2.0 - x * y);
}
// 1/sqrt(x) by the hardware estimate and one third-order step: the arithmetic of
// rsqrt() without its test for zero and infinity
__device__ __forceinline__ double rsqrt_nr(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = 1.0 - (x * y) * y;
    return y + (y * e) * (0.5 + 0.375 * e);
}

// What the lane's cubic is multiplied by at u = r - xi/sqrt(alpha): u for the
// density (rho lane: keep = ~0, unit = 0), the sign of u for the pair term
// (keep = the sign bit, unit = the bits of 1) -- the odd extensions u rho(|u|)
// and sgn(u) r*phi(|u|), without a comparison or a select.
template <typename Q>
struct OddFactor;
template <>
struct OddFactor<double> {
    int lo, hi, unit;
    __device__ __forceinline__ explicit OddFactor(bool rho)
        : lo(rho ? -1 : 0), hi(rho ? -1 : kInsideBit), unit(rho ? 0 : 0x3FF00000) {}
    __device__ __forceinline__ double operator()(double u) const {
        return __hiloint2double((__double2hiint(u) & hi) | unit, __double2loint(u) & lo);
    }
};
template <>
struct OddFactor<float> {
    int hi, unit;
    __device__ __forceinline__ explicit OddFactor(bool rho) : hi(rho ? -1 : kInsideBit), unit(rho ? 0 : 0x3F800000) {}
    __device__ __forceinline__ float operator()(float u) const { return __int_as_float((__float_as_int(u) & hi) | unit); }
};

// Points of a rule whose rows are requested together: all of a rule with a kernel of its
// own (3 and 5 points), else two at a time in a loop (a rule of an odd number of points has
// its last with one of zero weight).  With a general rule unrolled over kMaxPoints the rows,
// points and values lay in scratch memory: force_calc of 55,296 sites of two types, FP64, 7
// and 14 points 2.60 and 7.82 ms, the site table of c_d_calc 1.43 and 3.46; so 0.40 and
// 0.66, 0.39 and 0.60.
template <int NQ>
constexpr int kRowPoints = NQ > 0 ? NQ : 2;
static_assert(kMaxPoints % 2 == 0, "the last pair of a general rule lies in the arrays");

// The weighted sums of a Gauss-Hermite rule over x[k] = g(r - xi[k]/sqrt(alpha)):
// s[0] = sum w0 x, s[1] = sum w1 x, s[2] = sum w2 x with w1 = w0 xi, w2 = w0 xi^2.
// The nodes come in pairs -xi, xi of equal weight (exactly, in the tables in
// use) around a middle node 0, so a pair costs two additions and three
// multiply-adds instead of six.  A general rule adds its points k0, k0 + 1.
template <typename Q, int NQ, bool DERIV>
__device__ __forceinline__ void gh_sums(const FFParams<Q>& P, int k0, const Q* x, Q* s) {
    if constexpr (NQ > 0) {
        Q a0 = 0, a1 = 0, a2 = 0;
        if constexpr (NQ % 2) a0 = P.w0[NQ / 2] * x[NQ / 2];
#pragma unroll
        for (int k = NQ / 2 + NQ % 2; k < NQ; ++k) {
            const Q e = x[k] + x[NQ - 1 - k];
            a0 += P.w0[k] * e;
            if (DERIV) {
                a1 += P.w1[k] * (x[k] - x[NQ - 1 - k]);
                a2 += P.w2[k] * e;
            }
        }
        s[0] = a0;
        s[1] = a1;
        s[2] = a2;
    } else {
#pragma unroll
        for (int k = 0; k < kRowPoints<NQ>; ++k) {
            s[0] += P.w0[k0 + k] * x[k];
            if (DERIV) {
                s[1] += P.w1[k0 + k] * x[k];
                s[2] += P.w2[k0 + k] * x[k];
            }
        }
    }
}
// f(k0) for the first point of every set of kRowPoints
template <int NQ, typename F>
__device__ __forceinline__ void for_points(int no_i, F&& f) {
    if constexpr (NQ > 0) f(0);
    else
        for (int k0 = 0; k0 < no_i; k0 += kRowPoints<NQ>) f(k0);
}

// ENERGY_ONLY: the loop of ForceField_DMD_I::energy_calc (src/ff_dmd_I.cpp:454-668),
// type pairs jt >= it only (:508) unless FULL, which sums every ordered pair so the
// energy equals force_calc's.
//
// What bounds it: about 1,000 cycles of a CU's vector ALUs, of its address unit
// (the 64-byte spline rows) and of its L1-to-L2 path per site, and the latency of
// the rows between them.  So the loop over the pairs is straight-line code: every
// lane evaluates (a lane past the last pair repeats it with zero weight), a point
// beyond the cutoff reads the table's zero row nr - 1 (u < rc exactly when
// u/dr < nr - 1, so this is the reference's window test, src/ff_dmd_I.cpp:196-204),
// 1/r is formed once per list entry when it is staged, and the pair widths
// outside the quadrature regime, if a chunk has any, are told before and put
// right behind uniform branches: 2.90 -> 2.68 ms at 1,048,576 sites of two types, 3-point rule,
// FP64, with 14% more bytes of records.  Of the 2.68 ms, 0.5 go with the record
// stores, 0.24 with the scattered density shares and 0.2 with the rows' L1 misses.
// Loads of the next round ahead of a round's stores (128 registers) took 2.73 ms,
// rows read by four lanes as whole 64-byte segments (a quarter fewer cache accesses,
// a fifth more vector instructions) 2.80, ordinary stores of the records 3.16.
template <int NT, typename Q, int NQ, bool ENERGY_ONLY, bool FULL = false, int PARTS = 4>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4))) void k_pass1(
    FFParams<double> P, FFParams<Q> PQ, const double4* __restrict__ pos, const double4* __restrict__ arec,
    const int* __restrict__ off, const int2* nlrp, const Q* __restrict__ quad, const double* __restrict__ rho7,
    const double* __restrict__ phi7, double* __restrict__ Eown, double* __restrict__ pairE,
    typename Vec2<Q>::T* __restrict__ deriv, int2* __restrict__ info, double* __restrict__ part, CutState C, int wpb) {
    static_assert(PARTS == 1 || PARTS == 2 || PARTS == 4, "one, two or four lanes per (pair, type pair)");
    using Q2 = typename Vec2<Q>::T;
    using R = PairRec<NT, Q>;
    using Map = Pass1Map<NT, PARTS>;
    constexpr int LPP = Map::kLPP, PPW = Map::kPPW;
    const int lane = threadIdx.x & 63;
    const Map map(lane);
    const int k = map.k, prt = map.prt, it = map.it, jt = map.jt, q = it * NT + jt;
    const bool on = map.on && (!ENERGY_ONLY || FULL || jt >= it);
    // four parts: quarters of the row, rho in parts 0/1 and phi in 2/3 (results in 0 and 2);
    // two parts: part 0 the rho cubic, part 1 the phi cubic; one part: both
    const bool rho_lane = prt == 0, phi_lane = prt == PARTS / 2;
    const bool want_phi = it >= jt;
    const bool live = on && (PARTS == 1 || prt < PARTS / 2 || want_phi);
    // a phi lane whose phi is not kept reads its type pair's rho row instead (the same cache line)
    const int half = PARTS == 1 ? 0 : (prt >= PARTS / 2 && !want_phi ? prt - PARTS / 2 : prt) * (8 / PARTS);
    // energy_calc: the lanes without a part in it (three of eight with two types) read beyond
    // the buffer, which fetches nothing; 131,072 sites, 5 points, FP32 sums: 0.33 -> 0.29 ms
    const int tab_off = ENERGY_ONLY && !live ? kNoRow : (q * kQuadRow + half) * (int)sizeof(Q);
    const __amdgpu_buffer_rsrc_t qrs = raw_rsrc(quad, P.nr * quad_stride(NT) * (int)sizeof(Q));
    const OddFactor<Q> odd(prt < (PARTS + 1) / 2);
    // the lane's record component; the partner goes out on a lane whose phi is not kept
    // (type pair (0, NT-1)), on a spare lane, or with one type on the phi lane too
    const bool ix = Map::kCompact ? !map.on : NT > 1 && phi_lane && PARTS > 1 && q == NT - 1;
    const int comp = (ix ? R::kIdx : (rho_lane ? R::rho(q) : R::phi(it, jt))) * R::kG;
    const bool keeps = ix || (map.on && (rho_lane || (phi_lane && want_phi)));
    double en = 0.0, npair = 0.0;  // energy, pairs inside the quadrature cut (this lane's share)
    const Pass1Stage<NT> st(threadIdx.x >> 6);
    const SiteLoop<> sl(P.natms, wpb);
    for (int i0 = sl.first; i0 < sl.end; i0 += sl.stride) {
        const int i = __builtin_amdgcn_readfirstlane(i0);
        const int p0 = off[i], p1 = off[i + 1];
        const double4 xi = pos[i];
        const double4 ra = arec[(size_t)i * NT + it];
        const double ai = ra.x, iai = ra.z, ci = ra.y, ci_jt = arec[(size_t)i * NT + jt].y;
        double ia_min = arec[(size_t)i * NT].z, ia_max = ia_min;
#pragma unroll
        for (int t = 1; t < NT; ++t) {
            const double v = arec[(size_t)i * NT + t].z;
            ia_min = v < ia_min ? v : ia_min;
            ia_max = v > ia_max ? v : ia_max;
        }
        // weights of the lane's value: the partner's c for a rho lane, the pair energy's
        // c c + c c for a phi lane (src/ff_dmd_I.cpp:244-255)
        const double xw = it != jt ? P.xw : 1.0;
        const double wr = on && rho_lane ? 1.0 : 0.0;
        const double wa = on && phi_lane && want_phi ? xw * ci : 0.0;
        const double wb = on && phi_lane && want_phi ? xw * ci_jt : 0.0;
        Q2* const rec = deriv + R::first(p0, i);
        double Ei = 0.0, ep = 0.0;  // sums of the rho and of the phi lanes (one register unless PARTS == 1)
        int done = 0;  // inside entries of the earlier chunks: the pair's rank among the site's
        for (int chunk = p0; chunk < p1; chunk += 64) {
            // one list entry per lane: the cut state of each entry is kept current
            // (CutState); each entry inside the cut is staged in LDS at its rank
            // among the inside entries, with its partner's inverse width and
            // concentration of every type, read from HBM once per entry
            int cnt;
            bool regular = true;  // every pair width surely in the quadrature regime
            {
                const int pc = chunk + lane;
                bool in = false;
                int jc = 0, rp = 0;
                double r2 = 1.0;
                if (pc < p1) {
                    const int2 e = nlrp[pc];
                    jc = list_partner(e);
                    rp = e.y;  // meaningful for owned partners only
                    const double4 xj = pos[jc];
                    const double dx0 = xi.x - xj.x, dx1 = xi.y - xj.y, dx2 = xi.z - xj.z;
                    {
#pragma clang fp contract(off)
                        r2 = dx0 * dx0 + dx1 * dx1 + dx2 * dx2;
                    }
                    in = r2 < P.cut_sq_mod;
                    C.update<NT>(pc, e, in, i, jc, P.natms, pairE);
                }
                const int dest = pack_dest(in, &cnt);
                if (in) {
                    double2 ac[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t)
                        ac[t] = *reinterpret_cast<const double2*>(arec + (size_t)jc * NT + t);
                    st.geo[dest] = make_double2(r2, rsqrt_nr(r2));
                    st.idx[dest] = make_int2(jc, jc < P.natms ? rp : -1);
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const double iaj = rcp_nr(ac[t].x);
                        regular = regular && iaj + ia_min > P.ia_quad_lo && iaj + ia_max < P.ia_quad_hi;
                        st.typ[dest * NT + t] = make_double2(iaj, ac[t].y);
                    }
                }
                regular = __builtin_amdgcn_ballot_w64(!regular) == 0;
                __builtin_amdgcn_wave_barrier();
            }
            // whole groups of records are written (whole cache lines), also past the last pair
            const int kept = chunk + 64 < p1 ? cnt : (done + cnt + R::kG - 1) / R::kG * R::kG - done;
            for (int base = 0; base < cnt; base += PPW) {
                const int slot = base + k, s = slot < cnt ? slot : cnt - 1;
                const bool valid = slot < cnt && map.on;
                const int2 e = st.idx[s];
                const double2 geo = st.geo[s];
                const double2 tj = st.typ[s * NT + jt];
                const double cj = tj.y, cj_it = st.typ[s * NT + it].y;
                const double r_inv = geo.y, r = geo.x * r_inv;
                const double ia = iai + tj.x, asq = rsqrt_nr(ia);
                // v1: the lane's function (rho on the rho lane, phi on the phi lane) or,
                // with one lane per pair, rho; v2: phi with one lane per pair.
                // Each holds value, d/dr, d/dalpha.
                double v1[3] = {0.0, 0.0, 0.0}, v2[3] = {0.0, 0.0, 0.0};
                // pair widths outside the quadrature regime, or within rounding of its bounds; a
                // round without a lane that needs the quadrature goes past it (131,072 sites of
                // two types, every pair classical: force_calc 0.80 -> 0.69 ms, energy_calc 0.37
                // -> 0.28, for 0.3% of force_calc where every pair has its rule)
                int br = 1;
                bool some = true;
                if (!regular) {
                    if (live) br = alpha_branch(P, ia, ai, arec[(size_t)e.x * NT + jt].x);
                    some = __builtin_amdgcn_ballot_w64(live && br == 1) != 0;
                }
                if (some) {
                    const Q rq = (Q)r, iq = (Q)ia, aq = (Q)asq, inv = iq * aq;
                    // the rows of a set of points are requested before any is used, so their
                    // latencies overlap
                    constexpr int KP = kRowPoints<NQ>;
                    constexpr int NV = PARTS == 4 ? 1 : (PARTS == 2 ? 2 : 4);
                    Q sx[3] = {0, 0, 0}, sy[3] = {0, 0, 0};
                    for_points<NQ>(PQ.no_i, [&](int k0) {
                        Q2 rowv[KP][NV];
                        Q ppv[KP], uv[KP];
#pragma unroll
                        for (int kp = 0; kp < KP; ++kp) {
                            const Q u = rq - PQ.xi[k0 + kp] * inv;
                            int m = (int)(fabs(u) * PQ.dr_inv);
                            m = m < P.nr - 1 ? m : P.nr - 1;  // the zero row beyond the cutoff
                            uv[kp] = u;
                            ppv[kp] = fabs(u) * PQ.dr_inv - (Q)m;
                            const int row = tab_off + m * (quad_stride(NT) * (int)sizeof(Q));
#pragma unroll
                            for (int v = 0; v < NV; ++v)  // one lane per pair: the phi half only where it >= jt
                                rowv[kp][v] = PARTS != 1 || v < 2 || want_phi
                                                  ? RowLoad<Q2>::get(qrs, row + v * (int)sizeof(Q2))
                                                  : Q2{Q(0), Q(0)};
                        }
                        // keep the requests ahead of the arithmetic where the rows fit the
                        // register budget of four waves per SIMD (at most 24 registers)
                        if constexpr (KP * NV * sizeof(Q2) <= 96) __builtin_amdgcn_sched_barrier(0);
                        Q x[KP], y[KP];
#pragma unroll
                        for (int kp = 0; kp < KP; ++kp) {
                            const Q pp = ppv[kp], p2 = pp * pp;
                            if constexpr (PARTS == 4) {
                                const Q2 c = rowv[kp][0];
                                const Q h = c.x + c.y * pp;
                                x[kp] = (h + p2 * dpp_xor1_q<Q>(h)) * odd(uv[kp]);
                            } else {
                                const Q2 a0 = rowv[kp][0], a1 = rowv[kp][1];
                                x[kp] = ((a0.x + a0.y * pp) + p2 * (a1.x + a1.y * pp)) * odd(uv[kp]);
                                if constexpr (PARTS == 1) {
                                    const Q2 b0 = rowv[kp][2], b1 = rowv[kp][3];
                                    y[kp] = ((b0.x + b0.y * pp) + p2 * (b1.x + b1.y * pp)) * OddFactor<Q>(false)(uv[kp]);
                                }
                            }
                        }
                        gh_sums<Q, NQ, !ENERGY_ONLY>(PQ, k0, x, sx);
                        if constexpr (PARTS == 1) gh_sums<Q, NQ, !ENERGY_ONLY>(PQ, k0, y, sy);
                    });
                    const Q sc = Q(kPiInSq) * (Q)r_inv;
                    auto close = [&](const Q* sum, double* v) {
                        const Q v0 = sum[0] * sc;
                        v[0] = (double)v0;
                        if (!ENERGY_ONLY) {
                            v[1] = (double)(-v0 * (Q)r_inv - Q(2) * aq * (sum[1] * sc));
                            v[2] = (double)((Q(0.5) * v0 - sum[2] * sc) * iq);
                        }
                    };
                    close(sx, v1);
                    if constexpr (PARTS == 1) close(sy, v2);
                }
                if (!regular) {
                    if (br != 1) {
                        double g[3] = {0.0, 0.0, 0.0}, f[3] = {0.0, 0.0, 0.0};
                        if (br == 2 && geo.x < P.cut_sq)
                            classical_pair(P, geo.x, r_inv, rho7 + (size_t)type2rho(NT, it, jt) * P.nr * 7,
                                           phi7 + (size_t)type2phi(it, jt) * P.nr * 7, true, g, f);
#pragma unroll
                        for (int c = 0; c < 3; ++c) {
                            v1[c] = PARTS == 1 || rho_lane ? g[c] : f[c];
                            v2[c] = f[c];
                        }
                    }
                }
                // the site's density (rho lanes) and the pair energy (phi lanes)
                const double hw = valid ? (e.y >= 0 ? 0.5 : 0.25) : 0.0;
                const double we = (cj * wa + cj_it * wb) * hw;
                const double wE = valid ? cj * wr : 0.0;
                if constexpr (PARTS == 1) {
                    Ei += v1[0] * wE;
                    if (want_phi) ep += v2[0] * we;
                } else {
                    if (live) Ei += v1[0] * (rho_lane ? wE : we);
                }
                double ej = on && rho_lane ? v1[0] * ci : 0.0;
                if (!ENERGY_ONLY && slot < kept) {
                    Q2* d = rec + R::elem(done + slot, 0);
                    if constexpr (PARTS == 1) {
                        if (keeps) {
                            store_comp(d + comp, Q2{(Q)v1[1], (Q)v1[2]});
                            if (want_phi) store_comp(d + R::phi(it, jt) * R::kG, Q2{(Q)v2[1], (Q)v2[2]});
                            if (NT == 1 || q == NT - 1) store_comp(d + R::kIdx * R::kG, Vec2<Q>::ints(e.x, e.y));
                        }
                    } else {
                        const Q2 v = ix ? Vec2<Q>::ints(e.x, e.y) : Q2{(Q)v1[1], (Q)v1[2]};
                        if (keeps) store_comp(d + comp, v);
                        if (NT == 1 && phi_lane) store_comp(d + R::kIdx * R::kG, Vec2<Q>::ints(e.x, e.y));
                    }
                }
                // sum over it: the (0, jt) and (1, jt) lanes of a pair are NT * PARTS apart
                if constexpr (NT == 2 && PARTS == 4) ej += dpp_f64<kDppRowRor8>(ej);
                if constexpr (NT == 2 && PARTS == 2) ej += dpp_f64<kDppRowRor12>(ej);  // lane l + 4 for l % 8 < 4
                if constexpr (NT == 2 && PARTS == 1) ej += __shfl_xor(ej, 2, 64);
                if constexpr (NT > 2) {  // the rho lanes (0..NT-1, jt) of the pair, in a fixed order
                    double sum = 0.0;
#pragma unroll
                    for (int t = 0; t < NT; ++t) sum += __shfl(ej, k * LPP + Map::rho_at(t, jt), 64);
                    ej = sum;
                }
                // an ordinary store: the 16-byte shares land scattered, and L2 merges them into lines
                if (valid && rho_lane && it == 0 && e.y >= 0) pairE[(size_t)e.y * NT + jt] = ej;
            }
            done += cnt;
        }
        if (lane == 0) {
            npair += (double)done;  // the site's pairs inside the cut
            if (!ENERGY_ONLY) info[i] = make_int2(p0, done);
        }
        if constexpr (NT == 2 && PARTS == 2) {
            // the pair slots of a wavefront are 8 lanes apart; then the jt lanes are
            // joined: lanes 0 and 4 hold the densities of type 0 and 1, lanes 1 and 5
            // the energies of (0, *) and (1, *)
            double e = Ei;
            e += dpp_f64<kDppRowRor8>(e);
            e = row_pair_sum<false>(e);
            e = row_pair_sum<true>(e);
            e += dpp_f64<kDppXor2>(e);
            if ((lane & ~4) == 0) Eown[(size_t)i * NT + (lane >> 2)] = e;
            if ((lane & ~4) == 1) en += e;
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const double sum = wave_sum(rho_lane && it == t ? Ei : 0.0);
                if (lane == 0) Eown[(size_t)i * NT + t] = sum;
            }
            en += PARTS == 1 ? ep : (phi_lane ? Ei : 0.0);
        }
    }
    double acc[2] = {0.0, npair};  // npair: lane 0 only
    if constexpr (NT == 2 && PARTS == 2) acc[0] = read_lane(en, 1) + read_lane(en, 5);
    else acc[0] = wave_sum(en);
    wave_store<2>(acc, part);
}

// ---------------------------------------------------------------- lane groups
// G consecutive lanes per site (a DPP row for G = 16, a quad for G = 4);
// blocks are remapped so that each XCD takes a contiguous range of sites.
template <int G>
struct SiteGroup {
    int site, l;
    __device__ __forceinline__ SiteGroup() {
        const int b = xcd_block(gridDim.x);
        site = (b * kBlock + (int)threadIdx.x) / G;
        l = threadIdx.x & (G - 1);
    }
};

// sum over the G lanes of a group (fixed tree; every lane of the group gets it)
template <int G>
__device__ __forceinline__ double group_sum(double v) {
    static_assert(G == 16 || G == 4, "lane groups of 4 or 16");
    if constexpr (G == 16) {
        v += dpp_f64<kDppRowRor8>(v);
        v += dpp_f64<kDppRowRor4>(v);
    }
    v += dpp_f64<kDppXor2>(v);
    v += dpp_f64<kDppXor1>(v);
    return v;
}

// value v[t] of the lane whose group index is t (t < N)
template <int N>
__device__ __forceinline__ double pick(const double* v, int t) {
    double r = v[0];
#pragma unroll
    for (int x = 1; x < N; ++x)
        if (t == x) r = v[x];
    return r;
}

constexpr int kGatherG = 16;  // lanes per site of the reverse-CSR gathers
constexpr int kEmbedG = 4;    // lanes per site of the embedding (its per-site arithmetic runs on NT lanes of each group)

// ---------------------------------------------------------------- embed
// rho_bar = own share + partner shares (kEmbedG lanes per site over the site's
// contiguous reverse range); F, F', energy terms, alpha entropic force
template <int NT, bool ENERGY_ONLY>
__global__ __launch_bounds__(kBlock) void k_embed(FFParams<double> P, const double* __restrict__ alpha,
                                                  const double* __restrict__ conc, const int* __restrict__ roff,
                                                  const double* __restrict__ Eown,
                                                  const double* __restrict__ pairE,
                                                  const double* __restrict__ F9, double* __restrict__ E,
                                                  double* __restrict__ dE, double* __restrict__ fa,
                                                  double4* __restrict__ arec, double* __restrict__ part) {
    const SiteGroup<kEmbedG> g;
    const int i = g.site;
    double acc[1] = {0.0};
    if (i < P.natms) {
        double e[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) e[t] = 0.0;
        const int q1 = roff[i + 1];
        for (int q = roff[i] + g.l; q < q1; q += kEmbedG) {
#pragma unroll
            for (int t = 0; t < NT; ++t) e[t] += pairE[(size_t)q * NT + t];
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) e[t] = group_sum<kEmbedG>(e[t]);
        if (g.l < NT) {
            const int t = g.l;
            const size_t k = (size_t)i * NT + t;
            const double et = Eown[k] + pick<NT>(e, t);
            double Fv, dF;
            embed_F(P, F9, t, et, &Fv, &dF, nullptr);
            const double c = conc[k];
            const double a = alpha[k];
            E[k] = Fv;
            if (!ENERGY_ONLY) {
                dE[k] = dF;
                arec[k].w = dF;
                fa[k] = -(1.5 * P.kbT * c / a);
            }
            acc[0] += c * Fv;
            acc[0] += P.kbT * calc_ent(c);
            acc[0] += 1.5 * P.kbT * c * log(a) + c * P.c0[t];
        }
    }
    acc[0] = wave_sum(acc[0]);
    wave_store<1>(acc, part);
}

// ---------------------------------------------------------------- pass 2
// Two values summed over pairs of lanes: even lanes get the pair's sum of a, odd
// lanes the pair's sum of b (XOR1), or lanes with bit 1 clear / set (XOR2).
template <int CTRL>
__device__ __forceinline__ double fold2(double a, double b) {
    const bool hi = threadIdx.x & (CTRL == kDppXor1 ? 1 : 2);
    return (hi ? b : a) + dpp_f64<CTRL>(hi ? a : b);
}
// Sums over 32 lanes (half a wavefront), the value of lane l % 4 in each lane
// (fixed tree: lane pairs, quads, the four quads of a row, the two rows).
__device__ __forceinline__ double half_sums(double quad) {
    quad += dpp_f64<kDppRowRor4>(quad);
    quad += dpp_f64<kDppRowRor8>(quad);
    return row_pair_sum<false>(quad);
}
__device__ __forceinline__ double quad4(double a, double b, double c, double d) {
    return fold2<kDppXor2>(fold2<kDppXor1>(a, b), fold2<kDppXor1>(c, d));
}

constexpr int kPass2Lanes = 32;  // lanes per site

// src/ff_dmd_I.cpp:357-436: fpair/apair of each ordered type pair from the
// records of pass 1 (slot type2rho[jt][it], i.e. the transposed type pair's
// values, pairs with dE_i; phi for it < jt is the phi of (jt, it), as in the
// reference's shared COMP slot).  No table lookups.
//
// One lane per pair: it reads the pair's whole record (16-byte pieces of 64-byte
// runs, PairRec), the partner's position and {alpha, c, F'} of every type, and
// sums over the type pairs in registers, so nothing is exchanged between lanes
// but the site's sums at the end; the record names the partner, so no list entry
// is read and nothing is packed.  Half a wavefront per site, since a site of a
// close-packed crystal has about 27 pairs inside the cut.  With a lane per (pair,
// type pair) and the pairs packed through ds_permute this pass took 1.69 ms at
// 1,048,576 sites of two types (572 vector instructions per site, 15 memory
// instructions per site) and now takes 1.36 ms (FP32 records 1.57 -> 1.07).  Its
// bound is the bytes: without the records it takes 1.10 ms, without the shares'
// scattered writes 0.99 ms.  Shares at the pair's own list position, written in
// whole lines and read scattered by the gather, took 1.25 ms here and 0.51 ms
// there in place of 0.37.
template <int NT, typename Q>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(NT <= 2 ? 4 : (NT == 3 ? 3 : 2)))) void k_pass2(
    int natms, const double4* __restrict__ pos, const double4* __restrict__ arec, const int2* __restrict__ info,
    const typename Vec2<Q>::T* __restrict__ deriv, double* __restrict__ fown, double* __restrict__ share,
    double* __restrict__ part, int wpb) {
    using R = PairRec<NT, Q>;
    using Q2 = typename Vec2<Q>::T;
    constexpr int XD = 3 + NT, NPHI = NT * (NT + 1) / 2;
    const int l = threadIdx.x % kPass2Lanes;
    const bool odd = l & 1;
    double vir[6] = {0, 0, 0, 0, 0, 0};
    const SiteLoop<kPass2Lanes> sl(natms, wpb);
    for (int i = sl.first; i < sl.end; i += sl.stride) {
        const int2 in = info[i];  // list offset, pairs inside the cut
        const double4 xi = pos[i];
        double ai[NT], ci[NT], dEi[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const double4 ra = arec[(size_t)i * NT + t];
            ai[t] = ra.x;
            ci[t] = ra.y;
            dEi[t] = ra.w;
        }
        const int cnt = in.y;
        const Q2* const rec = deriv + R::first(in.x, i);
        double f[3] = {0.0, 0.0, 0.0}, fa[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) fa[t] = 0.0;
        for (int base = 0; base < cnt; base += kPass2Lanes) {
            // lanes past the last pair repeat it with zero weight and store nothing
            const bool valid = base + l < cnt;
            const Q2* const d = rec + R::elem(valid ? base + l : cnt - 1, 0);
            const int2 e = Vec2<Q>::ints(d[R::kIdx * R::kG]);
            const int j = e.x, rp = valid ? e.y : -1;
            Q2 g[NT * NT], ph[NPHI];
#pragma unroll
            for (int q = 0; q < NT * NT; ++q) g[q] = d[R::rho(q) * R::kG];
#pragma unroll
            for (int q = 0; q < NPHI; ++q) ph[q] = d[(NT * NT + q) * R::kG];
            const double4 xj = pos[j];
            double aj[NT], cj[NT], dEj[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const double4 rj = arec[(size_t)j * NT + t];
                aj[t] = rj.x;
                cj[t] = valid ? rj.y : 0.0;
                dEj[t] = rj.w;
            }
            const double dx0 = xi.x - xj.x, dx1 = xi.y - xj.y, dx2 = xi.z - xj.z;
            double rsq;
            {
#pragma clang fp contract(off)
                rsq = dx0 * dx0 + dx1 * dx1 + dx2 * dx2;
            }
            double S = 0.0, aJ[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) aJ[t] = 0.0;
#pragma unroll
            for (int it = 0; it < NT; ++it)
#pragma unroll
                for (int jt = 0; jt < NT; ++jt) {
                    const Q2 gq = g[it * NT + jt], gT = g[jt * NT + it], pq = ph[type2phi(it, jt)];
                    const double cc = ci[it] * cj[jt];
                    // 1/(alpha_i + alpha_j)
                    const double as = ai[it] + aj[jt];
                    double is = __builtin_amdgcn_rcp(as);
                    is = is * (2.0 - as * is);
                    is = is * (2.0 - as * is);
                    S += ((double)gT.x * dEi[it] + (double)gq.x * dEj[jt] + (double)pq.x) * cc;
                    const double ap = ((double)gT.y * dEi[it] + (double)gq.y * dEj[jt] + (double)pq.y) * cc * (is * is);
                    fa[it] -= ap * (aj[jt] * aj[jt]);
                    aJ[jt] -= ap * (ai[it] * ai[it]);
                }
            S *= -rsqrt(rsq);
            const double h0 = dx0 * S, h1 = dx1 * S, h2 = dx2 * S;
            f[0] += h0;
            f[1] += h1;
            f[2] += h2;
            const double wf = rp >= 0 ? 1.0 : 0.5;  // an owned partner, or half of a pair seen from both ends
            vir[0] -= wf * (h0 * dx0);
            vir[1] -= wf * (h1 * dx1);
            vir[2] -= wf * (h2 * dx2);
            vir[3] -= wf * (h1 * dx2);
            vir[4] -= wf * (h2 * dx0);
            vir[5] -= wf * (h0 * dx1);
            // the partner's share (ForceShare)
            double out[ForceShare<NT>::kLen] = {S};
#pragma unroll
            for (int t = 0; t < NT; ++t) out[1 + t] = aJ[t];
            if constexpr (ForceShare<NT>::kLen == 4) {
                // the two lanes of a pair of lanes write the 16-byte halves of one share
                // together, first the even lane's pair, then the odd lane's: one 32-byte write
                const double r0 = dpp_f64<kDppXor1>(odd ? out[0] : out[2]), r1 = dpp_f64<kDppXor1>(odd ? out[1] : out[3]);
                const int rpx = __builtin_amdgcn_update_dpp(0, rp, kDppXor1, 0xF, 0xF, false);
                const int rpe = odd ? rpx : rp, rpo = odd ? rp : rpx;
                if (rpe >= 0)
                    reinterpret_cast<double2*>(share + (size_t)rpe * 4)[odd] = make_double2(odd ? r0 : out[0], odd ? r1 : out[1]);
                if (rpo >= 0)
                    reinterpret_cast<double2*>(share + (size_t)rpo * 4)[odd] = make_double2(odd ? out[2] : r0, odd ? out[3] : r1);
            } else if (rp >= 0) {
                double2* const d2 = reinterpret_cast<double2*>(share + (size_t)rp * ForceShare<NT>::kLen);
#pragma unroll
                for (int t = 0; t < ForceShare<NT>::kLen / 2; ++t) d2[t] = make_double2(out[2 * t], out[2 * t + 1]);
            }
        }
        double* const fo = fown + (size_t)i * XD;
        const double s = half_sums(quad4(f[0], f[1], f[2], fa[0]));
        if (l < 4) fo[l] = s;
        if constexpr (NT > 1) {
            const double sx = half_sums(quad4(fa[1], NT > 2 ? fa[NT > 2 ? 2 : 0] : 0.0, NT > 3 ? fa[NT > 3 ? 3 : 0] : 0.0, 0.0));
            if (l < NT - 1) fo[4 + l] = sx;
        }
    }
    const double v03 = row_pair_sum<true>(half_sums(quad4(vir[0], vir[1], vir[2], vir[3])));
    const double v45 = row_pair_sum<true>(half_sums(quad4(vir[4], vir[5], 0.0, 0.0)));
    const int lane = threadIdx.x & 63;
    const size_t w = (size_t)blockIdx.x * wpb + (threadIdx.x >> 6);
    if (lane < 4) part[w * 6 + lane] = v03;
    if (lane < 2) part[w * 6 + 4 + lane] = v45;
}

// ---------------------------------------------------------------- force gather
template <int NT>
__global__ __launch_bounds__(kBlock) void k_fgather(int natms, const double4* __restrict__ pos,
                                                    const int* __restrict__ roff, const int* __restrict__ rowner,
                                                    const double* __restrict__ fown,
                                                    const double* __restrict__ share,
                                                    const double* __restrict__ fa, double* __restrict__ f) {
    constexpr int XD = 3 + NT;
    const SiteGroup<kGatherG> g;
    const int i = g.site;
    if (i >= natms) return;
    double acc[XD];
#pragma unroll
    for (int k = 0; k < XD; ++k) acc[k] = 0.0;
    const double4 xi = pos[i];
    const int q1 = roff[i + 1];
    for (int q = roff[i] + g.l; q < q1; q += kGatherG) {
        const int o = rowner[q];
        if (o < 0) {  // inside the cut
            const double2* const d2 = reinterpret_cast<const double2*>(share + (size_t)q * ForceShare<NT>::kLen);
            double v[ForceShare<NT>::kLen];
#pragma unroll
            for (int t = 0; t < ForceShare<NT>::kLen / 2; ++t) {
                const double2 w = d2[t];
                v[2 * t] = w.x;
                v[2 * t + 1] = w.y;
            }
            const double4 xo = pos[o & ~kInsideBit];
            acc[0] -= (xo.x - xi.x) * v[0];
            acc[1] -= (xo.y - xi.y) * v[0];
            acc[2] -= (xo.z - xi.z) * v[0];
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[3 + t] += v[1 + t];
        }
    }
#pragma unroll
    for (int k = 0; k < XD; ++k) acc[k] = group_sum<kGatherG>(acc[k]);
    if (g.l < XD) {
        const int k = g.l;
        double v = fown[(size_t)i * XD + k];
        if (k >= 3) v += fa[(size_t)i * NT + k - 3];
        f[(size_t)i * XD + k] = v + pick<XD>(acc, k);
    }
}

// Two-stage deterministic sums of up to kMaxSegs arrays of partials (at most 8
// values each) in one pair of launches.  Stage 1: segment s takes the blocks
// [first[s], first[s] + nb[s]), each of which sums a contiguous range of kReduceChunk
// partials; stage 2: block s sums the segment's stage-1 results.  Both in fixed trees.
// A chunk is two partials per thread: with 4,096 (sixteen loads in a row) stage 1 took
// 16 us on the 8,000 partials of a 4,000-site system, with a barrier per tree level and
// value; at 1,048,576 sites (1.8 million partials) 25 us.
constexpr int kMaxSegs = 4;
constexpr long kReduceChunk = 2 * kBlock;
struct ReduceSegs {
    const double* part[kMaxSegs];
    long nparts[kMaxSegs];
    int nv[kMaxSegs], stride[kMaxSegs], out_off[kMaxSegs], first[kMaxSegs], nb[kMaxSegs];
    int nseg;
};
// sums of 8 values over the block, in thread 0..7 (fixed tree)
__device__ __forceinline__ double block_sum8(const double* s, int nv) {
    __shared__ double sh[kBlock / 64][8];
    for (int k = 0; k < nv; ++k) {
        const double t = wave_sum(s[k]);
        if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6][k] = t;
    }
    __syncthreads();
    double t = 0.0;
    if ((int)threadIdx.x < nv)
        for (int q = 0; q < kBlock / 64; ++q) t += sh[q][threadIdx.x];
    return t;
}
__global__ __launch_bounds__(kBlock) void k_reduce_segs1(ReduceSegs R, double* __restrict__ stage) {
    int sg = 0;
    while (sg + 1 < R.nseg && (int)blockIdx.x >= R.first[sg + 1]) ++sg;
    const long lo = (long)(blockIdx.x - R.first[sg]) * kReduceChunk;
    long hi = lo + kReduceChunk;
    hi = hi < R.nparts[sg] ? hi : R.nparts[sg];
    const double* part = R.part[sg];
    const int nv = R.nv[sg], stride = R.stride[sg];
    // every value of a partial in one sweep (they share its cache line), then one tree per value
    double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (long b = lo + threadIdx.x; b < hi; b += kBlock) {
        const double* pb = part + (size_t)b * stride;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k < nv) s[k] += pb[k];
    }
    const double t = block_sum8(s, nv);
    if ((int)threadIdx.x < nv) stage[(size_t)blockIdx.x * 8 + threadIdx.x] = t;
}
__global__ __launch_bounds__(kBlock) void k_reduce_segs2(ReduceSegs R, const double* __restrict__ stage,
                                                         double* __restrict__ out) {
    const int sg = blockIdx.x, nv = R.nv[sg];
    double s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int b = threadIdx.x; b < R.nb[sg]; b += kBlock) {
        const double* pb = stage + (size_t)(R.first[sg] + b) * 8;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            if (k < nv) s[k] += pb[k];
    }
    const double t = block_sum8(s, nv);
    if ((int)threadIdx.x < nv) out[R.out_off[sg] + threadIdx.x] = t;
}

// smallest and largest of n pairs {smallest, largest} (one block)
__global__ __launch_bounds__(kBlock) void k_fold_minmax(const double* __restrict__ part, int n,
                                                        double* __restrict__ out) {
    __shared__ double mn[kBlock], mx[kBlock];
    double lo = INFINITY, hi = -INFINITY;
    for (int b = threadIdx.x; b < n; b += kBlock) {
        lo = fmin(lo, part[2 * b]);
        hi = fmax(hi, part[2 * b + 1]);
    }
    mn[threadIdx.x] = lo;
    mx[threadIdx.x] = hi;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) {
            mn[threadIdx.x] = fmin(mn[threadIdx.x], mn[threadIdx.x + w]);
            mx[threadIdx.x] = fmax(mx[threadIdx.x], mx[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = mn[0];
        out[1] = mx[0];
    }
}

}  // namespace mappdmd

#pragma clang fp contract(off)
