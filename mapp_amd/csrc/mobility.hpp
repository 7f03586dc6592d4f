// Concentration-rate kernels of the DMD force field, gather form:
//   create_2nd_neigh_lst   src/ff_dmd_I.cpp:2138-2217
//   c_d_calc  DMD_I / DMD_II / DMD   src/ff_dmd_I.cpp:2241-2398, src/ff_dmd_II.cpp:2186-2337, src/ff_dmd.cpp:2241-2398
//   calc_g    DMD_I / DMD_II / DMD   src/ff_dmd_I.cpp:2402-2674, src/ff_dmd_II.cpp:2341-2630, src/ff_dmd.cpp:2402-2671
// The reference sweeps the half list and scatters every pair term into both
// ends.  Here each site gathers the terms of all its pairs and never writes
// another site's row, so there are no atomics and every sum has a fixed
// order.
//
// Pair values.  rho_bar (every ordered type pair) and phi_bar depend on
// positions and widths only; the reference caches them in force_calc.  Here
// k_table_values evaluates them with the same quadrature as force_calc into the
// site table: for each owned site, the entries of its own half-list row that can
// have a value (table_pair), then the entries of the lower-index sites that list it
// (ascending owner), each holding the partner index and the pair's
// nt^2 + nt(nt+1)/2 values in the owner's orientation.  The other pairs add
// nothing to any sum and are left out.  Seen from site i with
// type m and a partner k of type b, each sweep's term is the same expression
// whichever end owns the pair (slot(b, m) for the density, slot(m, b) for the
// chemical potential and the last g sweep), so one loop covers both.
//
// Sweeps run G = 16 lanes per site: the lanes stride through the site's
// entries (coalesced: consecutive lanes read consecutive entries), then a
// fixed DPP rotation tree sums the lane partials.  The 2nd list (rates) runs
// 4 lanes per site over its own table, where the entry's sign tells which end
// owns the pair, since the rate terms are antisymmetric in the two ends.
// The index quirk of the chemical-potential sweep (dE[jatm+jtype],
// dE[iatm+itype] instead of [atom*nt+type]) is kept.
#pragma once
#include "force.hpp"

#pragma clang fp contract(fast)

namespace mappdmd {

// ---------------------------------------------------------------- site table
constexpr int kTableG = 16;  // lanes per site over the pair table
constexpr int kList2G = 4;   // lanes per site over the 2nd list

struct SiteTable {
    const int* off;     // [natms + 1] entries of site i: off[i] .. off[i+1]
    const int* idx;     // partner
    const double* rho;  // [entry][nt*nt] rho_bar, slot type2rho of the owner's (it, jt)
    const double* phi;  // [entry][nt(nt+1)/2] phi_bar
};

// |x_i - x_j|^2 as force_calc forms it (the same bits from either end)
__device__ __forceinline__ double pair_rsq(double4 xi, double4 xj) {
    const double dx0 = xi.x - xj.x, dx1 = xi.y - xj.y, dx2 = xi.z - xj.z;
    double rsq;
    {
#pragma clang fp contract(off)
        rsq = dx0 * dx0 + dx1 * dx1 + dx2 * dx2;
    }
    return rsq;
}

// {x, y, z, largest 1/alpha} per site, ghosts included, for table_pair (infinite for a
// width that is no number)
template <int NT>
__global__ void k_table_pack(const double4* __restrict__ pos, const double* __restrict__ alpha, int n,
                             double4* __restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 p = pos[i];
    p.w = 1.0 / alpha[(size_t)i * NT];
#pragma unroll
    for (int t = 1; t < NT; ++t) {
        const double v = 1.0 / alpha[(size_t)i * NT + t];
        if (!(v <= p.w)) p.w = v;
    }
    if (!(p.w == p.w)) p.w = INFINITY;
    rec[i] = p;
}
// Whether the pair can have a value: inside the quadrature cut, and its rule's nearest
// point r - xi_max/sqrt(alpha), at the widths of the two sites, not beyond rc (by more than
// the rounding of FP32 sums).  alpha_min sets the cut and may lie far below the widths in
// use: with 5 points, alpha_min = 1 and widths of 60 to 120, more than half of the pairs
// inside the cut have none.  256,000 sites so: c_d_calc after a move 2.82 ms and calc_g 1.59
// with every pair inside the cut in the table, 1.63 and 0.69 with these; with alpha_min =
// 25 the records cost 0.01 ms of 1.24.  The same bits from either end and in every kernel.
__device__ __forceinline__ bool table_pair(const FFParams<double>& P, double4 xi, double4 xj, double* rsq) {
#pragma clang fp contract(off)
    *rsq = pair_rsq(xi, xj);
    const double reach = P.rc + P.xi[P.no_i - 1] * sqrt(xi.w + xj.w);
    return *rsq < P.cut_sq_mod && !(*rsq > reach * reach * (1.0 + 4e-6));
}

// rank of this lane's flag among the set flags of lower lanes of its 16-lane group,
// and the number of set flags in the group
__device__ __forceinline__ int group_rank16(bool flag, int l, int* total) {
    const unsigned long long m = __builtin_amdgcn_ballot_w64(flag);
    const int gbase = (threadIdx.x & 63) & ~15;
    const unsigned bits = (unsigned)((m >> gbase) & 0xFFFFull);
    *total = __popc(bits);
    return __popc(bits & ((1u << l) - 1u));
}

// Entries per site: the pairs of the own row (own[i]) and of the reverse list that can have
// a value (table_pair), and for each reverse entry its rank among those
// (16 lanes per site, strided over both ranges).
__global__ __launch_bounds__(kBlock) void k_table_count(FFParams<double> P, PairBufs L, const int* __restrict__ rowner,
                                                        const double4* __restrict__ rec, int* __restrict__ own,
                                                        int* __restrict__ cnt, int* __restrict__ rrank) {
    const SiteGroup<kTableG> g;
    const int i = g.site;
    if (i >= P.natms) return;
    const double4 xi = rec[i];
    int c = 0, r = 0;
    double rsq;
    for (int p = L.off[i] + g.l; p < L.off[i + 1]; p += kTableG)
        c += table_pair(P, xi, rec[list_partner(L.nlrp[p])], &rsq) ? 1 : 0;
    const int q1 = L.roff[i + 1];
    for (int b = L.roff[i]; b < q1; b += kTableG) {
        const int q = b + g.l;
        const bool in = q < q1 && table_pair(P, xi, rec[rowner[q < q1 ? q : b] & ~kInsideBit], &rsq);
        int tot;
        const int rk = group_rank16(in, g.l, &tot);
        if (in) rrank[q] = r + rk;
        r += tot;
    }
    const double sc = group_sum<kTableG>((double)c);
    if (g.l == 0) {
        own[i] = (int)sc;
        cnt[i] = (int)sc + r;
    }
}

// The table: rho_bar of every ordered type pair and phi_bar for it >= jt of the pairs
// that can have a value, written from the pair's owner to both ends' rows; zeros where the
// reference computes nothing (alpha out of range, or the whole rule of a type pair beyond
// rc).  A site's row holds its own pairs in list order, then those of its reverse list
// in that order (rrank, k_table_count).  One wavefront per site and two lanes per
// (pair, type pair), the lanes and the arithmetic of pass 1 (k_pass1) without the
// derivatives.  Bound by the stores: the partner's entries are 8-byte words of rows
// that 50 other waves fill.  At 442,368 sites of two types 1.26 ms, with 0.18 for the
// count; one thread per listed pair, values kept in list order, counted and copied to
// both rows took 1.04 + 0.47 + 1.33 ms, and own rows here with the partner's rows
// copied by a second kernel 0.84 + 0.12 + 0.61.
template <int NT>
struct TableStage {
    static constexpr int kBytes = 64 * (16 + 8 * NT + 8);
    double2* geo;  // {r^2, 1/r}
    double* typ;   // 1/alpha of the partner per type
    int2* idx;     // {partner, the pair's entry in the partner's row or -1 for a ghost}
    __device__ __forceinline__ explicit TableStage(int wave) {
        extern __shared__ __attribute__((aligned(32))) unsigned char table_lds[];
        unsigned char* base = table_lds + (size_t)wave * kBytes;
        geo = reinterpret_cast<double2*>(base);
        typ = reinterpret_cast<double*>(geo + 64);
        idx = reinterpret_cast<int2*>(typ + 64 * NT);
    }
};
template <int NT, typename Q, int NQ>
__global__ __launch_bounds__(kBlock) void k_table_values(FFParams<double> P, FFParams<Q> PQ,
                                                         const double4* __restrict__ rec,
                                                         const double* __restrict__ alpha,
                                                         const int* __restrict__ off, const int2* __restrict__ nlrp,
                                                         const Q* __restrict__ quad, const double* __restrict__ rho7,
                                                         const double* __restrict__ phi7,
                                                         const int* __restrict__ toff, const int* __restrict__ own,
                                                         const int* __restrict__ rrank, int* __restrict__ tidx,
                                                         double* __restrict__ trho,
                                                         double* __restrict__ tphi) {
    using Q2 = typename Vec2<Q>::T;
    using Map = Pass1Map<NT, 2>;
    constexpr int NPHI = NT * (NT + 1) / 2;
    constexpr int KP = kRowPoints<NQ>;
    const int lane = threadIdx.x & 63;
    const Map map(lane);
    const int k = map.k, prt = map.prt, it = map.it, jt = map.jt;
    const bool rho_lane = prt == 0, keeps = map.on && (rho_lane || it >= jt);
    const int tab_off = ((it * NT + jt) * kQuadRow + (rho_lane || it < jt ? 0 : 4)) * (int)sizeof(Q);
    const __amdgpu_buffer_rsrc_t qrs = raw_rsrc(quad, P.nr * quad_stride(NT) * (int)sizeof(Q));
    const OddFactor<Q> odd(rho_lane);
    const TableStage<NT> st(threadIdx.x >> 6);
    const SiteLoop<> sl(P.natms, kBlock / 64);
    for (int i0 = sl.first; i0 < sl.end; i0 += sl.stride) {
        const int i = __builtin_amdgcn_readfirstlane(i0);
        const int p0 = off[i], p1 = off[i + 1];
        const double4 xi = rec[i];
        const double ai = alpha[(size_t)i * NT + it], iai = rcp_nr(ai);
        double ia_min = rcp_nr(alpha[(size_t)i * NT]), ia_max = ia_min;
#pragma unroll
        for (int t = 1; t < NT; ++t) {
            const double v = rcp_nr(alpha[(size_t)i * NT + t]);
            ia_min = v < ia_min ? v : ia_min;
            ia_max = v > ia_max ? v : ia_max;
        }
        size_t at = (size_t)toff[i];
        for (int chunk = p0; chunk < p1; chunk += 64) {
            int cnt;
            bool regular = true;  // every pair width surely in the quadrature regime
            {
                const int pc = chunk + lane;
                bool in = false;
                int jc = 0, qc = -1;
                double r2 = 1.0;
                if (pc < p1) {
                    const int2 e = nlrp[pc];
                    jc = e.x & ~kInsideBit;
                    qc = e.y;
                    in = table_pair(P, xi, rec[jc], &r2);
                }
                const int dest = pack_dest(in, &cnt);
                if (in) {
                    double a[NT];
#pragma unroll
                    for (int t = 0; t < NT; ++t) a[t] = alpha[(size_t)jc * NT + t];
                    const int there = qc >= 0 ? toff[jc] + own[jc] + rrank[qc] : -1;
                    tidx[at + dest] = jc;
                    if (there >= 0) tidx[there] = i;
                    st.geo[dest] = make_double2(r2, rsqrt_nr(r2));
                    st.idx[dest] = make_int2(jc, there);
#pragma unroll
                    for (int t = 0; t < NT; ++t) {
                        const double iaj = rcp_nr(a[t]);
                        regular = regular && iaj + ia_min > P.ia_quad_lo && iaj + ia_max < P.ia_quad_hi;
                        st.typ[dest * NT + t] = iaj;
                    }
                }
                regular = __builtin_amdgcn_ballot_w64(!regular) == 0;
                __builtin_amdgcn_wave_barrier();
            }
            for (int base = 0; base < cnt; base += Map::kPPW) {
                const int slot = base + k, s = slot < cnt ? slot : cnt - 1;
                const double2 geo = st.geo[s];
                const double r_inv = geo.y, r = geo.x * r_inv;
                const double ia = iai + st.typ[s * NT + jt], asq = rsqrt_nr(ia);
                const Q rq = (Q)r, inv = (Q)ia * (Q)asq;
                Q sum[3] = {0, 0, 0};
                for_points<NQ>(PQ.no_i, [&](int k0) {
                    Q2 lo[KP], hi[KP];
                    Q ppv[KP];
#pragma unroll
                    for (int kp = 0; kp < KP; ++kp) {
                        const Q u = rq - PQ.xi[k0 + kp] * inv;
                        int m = (int)(fabs(u) * PQ.dr_inv);
                        m = m < P.nr - 1 ? m : P.nr - 1;  // the zero row beyond the cutoff
                        ppv[kp] = fabs(u) * PQ.dr_inv - (Q)m;
                        const int row = tab_off + m * (quad_stride(NT) * (int)sizeof(Q));
                        lo[kp] = RowLoad<Q2>::get(qrs, row);
                        hi[kp] = RowLoad<Q2>::get(qrs, row + (int)sizeof(Q2));
                    }
                    if constexpr (KP * 2 * sizeof(Q2) <= 96) __builtin_amdgcn_sched_barrier(0);
                    Q x[KP];
#pragma unroll
                    for (int kp = 0; kp < KP; ++kp) {
                        const Q u = rq - PQ.xi[k0 + kp] * inv, pp = ppv[kp], p2 = pp * pp;
                        x[kp] = ((lo[kp].x + lo[kp].y * pp) + p2 * (hi[kp].x + hi[kp].y * pp)) * odd(u);
                    }
                    gh_sums<Q, NQ, false>(PQ, k0, x, sum);
                });
                double v = (double)(sum[0] * (Q(kPiInSq) * (Q)r_inv));
                if (!regular && keeps) {
                    const int br = alpha_branch(P, ia, ai, alpha[(size_t)st.idx[s].x * NT + jt]);
                    if (br != 1) {
                        double gv[3] = {0.0, 0.0, 0.0}, fv[3] = {0.0, 0.0, 0.0};
                        if (br == 2 && geo.x < P.cut_sq)
                            classical_pair(P, geo.x, r_inv, rho7 + (size_t)type2rho(NT, it, jt) * P.nr * 7,
                                           phi7 + (size_t)type2phi(it, jt) * P.nr * 7, true, gv, fv);
                        v = rho_lane ? gv[0] : fv[0];
                    }
                }
                if (keeps && slot < cnt) {
                    const int there = st.idx[s].y;
                    double* const row = rho_lane ? trho + type2rho(NT, it, jt) : tphi + type2phi(it, jt);
                    const int len = rho_lane ? NT * NT : NPHI;
                    row[(at + slot) * len] = v;
                    if (there >= 0) row[(size_t)there * len] = v;
                }
            }
            __builtin_amdgcn_wave_barrier();
            at += cnt;
        }
    }
}

// The vectors that one sweep hands to the next (n, s, t, v, F'') are read where their site
// is owned, through the ghost's owner, so that no copy to the ghosts stands between two
// sweeps; c and dE (whose element the quirk picks by the ghost's own index) lie at the
// ghosts too.  A copy takes the stream about 4 us, six of them stood in a calc_g whose
// sweeps take 8 to 14 us each on a batch of six cells of 6^3 to 12^3.
struct Owner {
    const int* owner;  // owner[g] of ghost natms + g
    int natms;
    __device__ __forceinline__ int operator()(int k) const { return k < natms ? k : owner[k - natms]; }
};

// E = sum c rho_bar; n = E = F(E), dE = F', ddE = F''
// (first sweep of c_d_calc, src/ff_dmd_I.cpp:2269-2312, and calc_g, :2447-2493).
// Site i of type m, partner k of type b: E[i][m] += c[k][b] rho[slot(b, m)]
// (own row :2285-2286 and the partner end :2287, with the reference's slot).
template <int NT>
__global__ __launch_bounds__(kBlock) void k_density_table(FFParams<double> P, const double* __restrict__ conc,
                                                          SiteTable T, const double* __restrict__ F9,
                                                          double* __restrict__ E, double* __restrict__ n,
                                                          double* __restrict__ dE, double* __restrict__ ddE) {
    const SiteGroup<kTableG> g;
    const int i = g.site;
    if (i >= P.natms) return;
    double e[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) e[t] = 0.0;
    for (int q = T.off[i] + g.l; q < T.off[i + 1]; q += kTableG) {
        const int k = T.idx[q];
        double r[NT * NT], c[NT];
#pragma unroll
        for (int x = 0; x < NT * NT; ++x) r[x] = T.rho[(size_t)q * NT * NT + x];
#pragma unroll
        for (int b = 0; b < NT; ++b) c[b] = conc[(size_t)k * NT + b];
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int b = 0; b < NT; ++b) e[m] += c[b] * r[type2rho(NT, b, m)];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) e[t] = group_sum<kTableG>(e[t]);
    if (g.l < NT) {
        double et = e[0];
#pragma unroll
        for (int t = 1; t < NT; ++t)
            if (g.l == t) et = e[t];
        double Fv, dF, ddF;
        embed_F(P, F9, g.l, et, &Fv, &dF, &ddF);
        const size_t k = (size_t)i * NT + g.l;
        E[k] = Fv;
        n[k] = Fv;
        dE[k] = dF;
        if (ddE) ddE[k] = ddF;
    }
}

// n += sum c (rho dE[flat jatm+jtype] + phi), then the closing terms:
// CLOSE 0: c_d_calc DMD / DMD_I   n = (n + c_0 + 1.5 kT log a) * beta
// CLOSE 1: c_d_calc DMD_II        n =  n + c_0 + 1.5 kT log a
// CLOSE 2: calc_g   DMD / DMD_I   n = (n + c_0) * beta + 1.5 log a
// CLOSE 3: calc_g   DMD_II        n = (n + c_0) + 1.5 kT log a
// Site i of type m, partner k of type b: c[k][b] (rho[slot(m, b)] dE[q(k, b)] + phi[(m, b)])
// (src/ff_dmd_I.cpp:2336-2339 at both ends).
template <int NT, int CLOSE>
__global__ __launch_bounds__(kBlock) void k_chem_pot(FFParams<double> P, const double* __restrict__ alpha,
                                                     const double* __restrict__ conc, SiteTable T,
                                                     const double* __restrict__ dE, const int* __restrict__ qidx,
                                                     double* __restrict__ n) {
    // qidx[j*NT + t] is the element that the reference's dE[jatm + jtype] reads for
    // site j (jatm + t within the site's own cell numbering: j + t for one cell)
    constexpr int NPHI = NT * (NT + 1) / 2;
    const SiteGroup<kTableG> g;
    const int i = g.site;
    if (i >= P.natms) return;
    double acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = 0.0;
    for (int q = T.off[i] + g.l; q < T.off[i + 1]; q += kTableG) {
        const int k = T.idx[q];
        double r[NT * NT], f[NPHI], cd[NT];
#pragma unroll
        for (int x = 0; x < NT * NT; ++x) r[x] = T.rho[(size_t)q * NT * NT + x];
#pragma unroll
        for (int x = 0; x < NPHI; ++x) f[x] = T.phi[(size_t)q * NPHI + x];
#pragma unroll
        for (int b = 0; b < NT; ++b) cd[b] = dE[qidx[(size_t)k * NT + b]];
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int b = 0; b < NT; ++b)
                acc[m] += conc[(size_t)k * NT + b] * (r[type2rho(NT, m, b)] * cd[b] + f[type2phi(m, b)]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = group_sum<kTableG>(acc[t]);
    if (g.l < NT) {
        const int t = g.l;
        double v = acc[0];
#pragma unroll
        for (int x = 1; x < NT; ++x)
            if (t == x) v = acc[x];
        const size_t k = (size_t)i * NT + t;
        v += n[k];
        const double la = log(alpha[k]);
        if (CLOSE == 0) {
            v += P.c0[t] + 1.5 * P.kbT * la;
            v *= P.beta;
        } else if (CLOSE == 1) {
            v += P.c0[t] + 1.5 * P.kbT * la;
        } else if (CLOSE == 2) {
            v += P.c0[t];
            v *= P.beta;
            v += 1.5 * la;
        } else {
            v += P.c0[t];
            v += 1.5 * P.kbT * la;
        }
        n[k] = v;
    }
}

// exchange term of a 2nd-list pair (i, j) for type t, in the reference's roles
// VAR 0 = DMD, 1 = DMD_I, 2 = DMD_II.  Returns the c_d_calc s_ij.
template <int VAR>
__device__ __forceinline__ double rate_sij(const FFParams<double>& P, double ni, double nj, double ci, double cj) {
    if (VAR == 2) {
        const double mt = ni > nj ? ni + 0.5 : nj + 0.5;
        const double efi = exp(P.beta * (ni - mt));
        const double efj = exp(P.beta * (nj - mt));
        const double tmpi = ci * (1.0 - cj);
        const double tmpj = cj * (1.0 - ci);
        return tmpj * efj - tmpi * efi;
    }
    const double Mat = VAR == 0 ? 5.2 * P.beta : 0.4 * P.beta;
    double t0, t1;
    if (VAR == 1) {
        t0 = exp(0.5 * (ni - nj) + Mat);
        t1 = exp(0.5 * (nj - ni) + Mat);
    } else {
        t0 = exp(ni + Mat);
        t1 = exp(nj + Mat);
    }
    return ((1.0 - ci) * cj * t1 - (1.0 - cj) * ci * t0);
}

// c_d over the 2nd list; an entry e >= 0 is the own-row partner j (pair (i, j)),
// e < 0 the owner ~e of the pair (~e, i)
template <int NT, int VAR>
__global__ __launch_bounds__(kBlock) void k_c_d(FFParams<double> P, Owner at, const double* __restrict__ conc,
                                                const int* __restrict__ foff, const int* __restrict__ fidx,
                                                const double* __restrict__ n, double* __restrict__ c_d) {
    const SiteGroup<kList2G> g;
    const int i = g.site;
    if (i >= P.natms) return;
    double acc[NT], ni[NT], ci[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        acc[t] = 0.0;
        ni[t] = n[(size_t)i * NT + t];
        ci[t] = conc[(size_t)i * NT + t];
    }
    for (int q = foff[i] + g.l; q < foff[i + 1]; q += kList2G) {
        const int e = fidx[q];
        const bool own = e >= 0;
        const int k = own ? e : ~e, ko = at(k);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const double nk = n[(size_t)ko * NT + t], ck = conc[(size_t)k * NT + t];
            const double sij = own ? rate_sij<VAR>(P, ni[t], nk, ci[t], ck) : rate_sij<VAR>(P, nk, ni[t], ck, ci[t]);
            acc[t] += own ? sij : -sij;
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = group_sum<kList2G>(acc[t]);
    if (g.l == 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) c_d[(size_t)i * NT + t] = acc[t];
    }
}

// calc_g residual s = 2(c + a) - 2 alpha (rate sums) (and c_d for DMD_II); partial sums of s^2
template <int NT, int VAR>
__global__ __launch_bounds__(kBlock) void k_calc_g_s(FFParams<double> P, Owner at, double alpha_t,
                                                     const double* __restrict__ conc, const double* __restrict__ a,
                                                     const int* __restrict__ foff, const int* __restrict__ fidx,
                                                     const double* __restrict__ n, double* __restrict__ s,
                                                     double* __restrict__ c_d, double* __restrict__ part) {
    const SiteGroup<kList2G> g;
    const int i = g.site;
    double sq = 0.0;
    if (i < P.natms) {
        double acc[NT], ni[NT], ci[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            acc[t] = 0.0;
            ni[t] = n[(size_t)i * NT + t];
            ci[t] = conc[(size_t)i * NT + t];
        }
        for (int q = foff[i] + g.l; q < foff[i + 1]; q += kList2G) {
            const int e = fidx[q];
            const bool own = e >= 0;
            const int k = own ? e : ~e, ko = at(k);
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const double nk = n[(size_t)ko * NT + t], ck = conc[(size_t)k * NT + t];
                const double sij =
                    own ? rate_sij<VAR>(P, ni[t], nk, ci[t], ck) : rate_sij<VAR>(P, nk, ni[t], ck, ci[t]);
                acc[t] += own ? sij : -sij;
            }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[t] = group_sum<kList2G>(acc[t]);
        if (g.l == 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const size_t k = (size_t)i * NT + t;
                const double sv = 2.0 * (ci[t] + a[k]) - 2.0 * alpha_t * acc[t];
                s[k] = sv;
                if (VAR == 2) c_d[k] = acc[t];
                sq += sv * sv;
            }
        }
    }
    double v[1] = {sq};
    block_sum_store<1>(v, part);
}

// pair terms of the t / g sweep for the pair (I, J) of type t in the reference's
// roles; returns contributions to (t_I, g_I) and (t_J, g_J)
template <int VAR>
__device__ __forceinline__ void tg_pair(const FFParams<double>& P, double alpha_t, double nI, double nJ, double cI,
                                        double cJ, double sI, double sJ, double* tI, double* gI, double* tJ,
                                        double* gJ) {
    if (VAR == 2) {
        const double s_ij = sI - sJ;
        const double mt = nI > nJ ? nI + 0.5 : nJ + 0.5;
        const double efi = exp(P.beta * (nI - mt));
        const double efj = exp(P.beta * (nJ - mt));
        const double tmpi = cI * (1.0 - cJ);
        const double tmpj = cJ * (1.0 - cI);
        const double dij = nI > nJ ? 1.0 : 0.0, dji = nJ > nI ? 1.0 : 0.0;
        double ti = tmpi * efi + dij * (tmpj * efj - tmpi * efi);
        ti *= s_ij;
        double tj = tmpj * efj + dji * (tmpi * efi - tmpj * efj);
        tj *= s_ij;
        *tI = ti;
        *gI = -(alpha_t * ((1.0 - cJ) * efi + cJ * efj) * s_ij);
        *tJ = -tj;
        *gJ = alpha_t * ((1.0 - cI) * efj + cI * efi) * s_ij;
        return;
    }
    const double Mat = VAR == 0 ? 5.2 * P.beta : 0.4 * P.beta;
    double t0, t1;
    if (VAR == 1) {
        t0 = exp(0.5 * (nI - nJ) + Mat);
        t1 = exp(0.5 * (nJ - nI) + Mat);
        t0 *= (sI - sJ);
        t1 *= (sI - sJ);
        const double t_ij = 0.5 * (cI * (1.0 - cJ) * t0 + cJ * (1.0 - cI) * t1);
        *tI = t_ij;
        *tJ = -t_ij;
    } else {
        t0 = (sI - sJ) * exp(Mat + nI);
        t1 = (sI - sJ) * exp(Mat + nJ);
        *tI = cI * t0 * (1.0 - cJ);
        *tJ = -(cJ * t1 * (1.0 - cI));
    }
    *gI = -(alpha_t * (t0 * (1.0 - cJ) + t1 * cJ));
    *gJ = alpha_t * (t1 * (1.0 - cI) + cI * t0);
}

// t and the first g term over the 2nd list (src/ff_dmd_I.cpp:2576-2606)
template <int NT, int VAR>
__global__ __launch_bounds__(kBlock) void k_calc_g_t(FFParams<double> P, Owner at, double alpha_t,
                                                     const double* __restrict__ conc, const int* __restrict__ foff,
                                                     const int* __restrict__ fidx, const double* __restrict__ n,
                                                     const double* __restrict__ s, double* __restrict__ t,
                                                     double* __restrict__ g) {
    const SiteGroup<kList2G> grp;
    const int i = grp.site;
    if (i >= P.natms) return;
    double tv[NT], gv[NT], ni[NT], ci[NT], si[NT];
#pragma unroll
    for (int ty = 0; ty < NT; ++ty) {
        const size_t k = (size_t)i * NT + ty;
        tv[ty] = 0.0;
        gv[ty] = 0.0;
        ni[ty] = n[k];
        ci[ty] = conc[k];
        si[ty] = s[k];
    }
    for (int q = foff[i] + grp.l; q < foff[i + 1]; q += kList2G) {
        const int e = fidx[q];
        const bool own = e >= 0;
        const int k = own ? e : ~e, ko = at(k);
#pragma unroll
        for (int ty = 0; ty < NT; ++ty) {
            const size_t kk = (size_t)ko * NT + ty;
            const double nk = n[kk], ck = conc[(size_t)k * NT + ty], sk = s[kk];
            double tI, gI, tJ, gJ;
            if (own) {
                tg_pair<VAR>(P, alpha_t, ni[ty], nk, ci[ty], ck, si[ty], sk, &tI, &gI, &tJ, &gJ);
                tv[ty] += tI;
                gv[ty] += gI;
            } else {
                tg_pair<VAR>(P, alpha_t, nk, ni[ty], ck, ci[ty], sk, si[ty], &tI, &gI, &tJ, &gJ);
                tv[ty] += tJ;
                gv[ty] += gJ;
            }
        }
    }
#pragma unroll
    for (int ty = 0; ty < NT; ++ty) {
        tv[ty] = group_sum<kList2G>(tv[ty]);
        gv[ty] = group_sum<kList2G>(gv[ty]);
    }
    if (grp.l == 0) {
#pragma unroll
        for (int ty = 0; ty < NT; ++ty) {
            const size_t k = (size_t)i * NT + ty;
            t[k] = tv[ty];
            g[k] = gv[ty] - si[ty];
        }
    }
}

// v and the next g term over the pair table (src/ff_dmd_I.cpp:2610-2642).
// Site i of type m, partner k of type b:
//   v[i][m] += rho[slot(b, m)] t[k][b]
//   g[i][m] += alpha beta (phi[(m, b)] + rho[slot(b, m)] dE[i][m] + rho[slot(m, b)] dE[k][b]) t[k][b]
template <int NT>
__global__ __launch_bounds__(kBlock) void k_calc_g_v(FFParams<double> P, Owner at, double alpha_t, SiteTable T,
                                                     const double* __restrict__ dE, const double* __restrict__ t,
                                                     double* __restrict__ v, double* __restrict__ g) {
    constexpr int NPHI = NT * (NT + 1) / 2;
    const SiteGroup<kTableG> grp;
    const int i = grp.site;
    if (i >= P.natms) return;
    const double ba = P.beta * alpha_t;
    double vv[NT], gg[NT], dEi[NT];
#pragma unroll
    for (int ty = 0; ty < NT; ++ty) {
        vv[ty] = 0.0;
        gg[ty] = 0.0;
        dEi[ty] = dE[(size_t)i * NT + ty];
    }
    for (int q = T.off[i] + grp.l; q < T.off[i + 1]; q += kTableG) {
        const int k = T.idx[q], ko = at(k);
        double r[NT * NT], f[NPHI], tk[NT], dk[NT];
#pragma unroll
        for (int x = 0; x < NT * NT; ++x) r[x] = T.rho[(size_t)q * NT * NT + x];
#pragma unroll
        for (int x = 0; x < NPHI; ++x) f[x] = T.phi[(size_t)q * NPHI + x];
#pragma unroll
        for (int b = 0; b < NT; ++b) {
            tk[b] = t[(size_t)ko * NT + b];
            dk[b] = dE[(size_t)k * NT + b];
        }
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int b = 0; b < NT; ++b) {
                const double rbm = r[type2rho(NT, b, m)];
                const double tmp0 = (f[type2phi(m, b)] + rbm * dEi[m] + r[type2rho(NT, m, b)] * dk[b]) * ba;
                vv[m] += rbm * tk[b];
                gg[m] += tmp0 * tk[b];
            }
    }
#pragma unroll
    for (int ty = 0; ty < NT; ++ty) {
        vv[ty] = group_sum<kTableG>(vv[ty]);
        gg[ty] = group_sum<kTableG>(gg[ty]);
    }
    if (grp.l == 0) {
#pragma unroll
        for (int ty = 0; ty < NT; ++ty) {
            const size_t k = (size_t)i * NT + ty;
            v[k] = vv[ty];
            g[k] += gg[ty];
        }
    }
}

// last g term: alpha beta rho ddE c v (src/ff_dmd_I.cpp:2647-2671).
// Site i of type m, partner k of type b: alpha beta rho[slot(m, b)] ddE[k][b] c[k][b] v[k][b]
template <int NT>
__global__ __launch_bounds__(kBlock) void k_calc_g_w(FFParams<double> P, Owner at, double alpha_t,
                                                     const double* __restrict__ conc, SiteTable T,
                                                     const double* __restrict__ ddE, const double* __restrict__ v,
                                                     double* __restrict__ g) {
    const SiteGroup<kTableG> grp;
    const int i = grp.site;
    if (i >= P.natms) return;
    const double ab = alpha_t * P.beta;
    double gg[NT];
#pragma unroll
    for (int ty = 0; ty < NT; ++ty) gg[ty] = 0.0;
    for (int q = T.off[i] + grp.l; q < T.off[i + 1]; q += kTableG) {
        const int k = T.idx[q], ko = at(k);
        double r[NT * NT], w[NT];
#pragma unroll
        for (int x = 0; x < NT * NT; ++x) r[x] = T.rho[(size_t)q * NT * NT + x];
#pragma unroll
        for (int b = 0; b < NT; ++b) {
            const size_t kk = (size_t)ko * NT + b;
            w[b] = ddE[kk] * conc[(size_t)k * NT + b] * v[kk];
        }
#pragma unroll
        for (int m = 0; m < NT; ++m)
#pragma unroll
            for (int b = 0; b < NT; ++b) gg[m] += ab * r[type2rho(NT, m, b)] * w[b];
    }
#pragma unroll
    for (int ty = 0; ty < NT; ++ty) gg[ty] = group_sum<kTableG>(gg[ty]);
    if (grp.l == 0) {
#pragma unroll
        for (int ty = 0; ty < NT; ++ty) g[(size_t)i * NT + ty] += gg[ty];
    }
}

}  // namespace mappdmd

#pragma clang fp contract(off)
