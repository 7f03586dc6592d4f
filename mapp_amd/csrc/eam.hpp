// MD-mode potentials of the reference on the DMD context's geometry (same
// ghosts, half list and reverse CSR; a group of kEamG = 16 lanes per site, each
// lane a stride of the site's list, summed in a fixed tree; partner shares through
// pair buffers in reverse-CSR order, no floating-point atomics):
//   plain EAM   ForceField_eam::force_calc / energy_calc, src/ff_eam.cpp:44-356
//               (F the cubic rows of ForceField_eam::interpolate, 7 coefficients;
//               rho and r*phi the rows of the DMD tables; Horner as the reference)
//   LJ          ForceField_lj::force_calc / energy_calc, src/ff_lj.cpp:160-341
//   FS          ForceField_fs::force_calc / energy_calc, src/ff_fs.cpp:379-686
// Types are carried in the per-site concentration column.  FS keeps the
// reference's factors: rho_i stores -A/sqrt(rho) after the embedding and the
// pair records hold -(t1 + 1.5 t2 dr) dr / r, so the density force of a pair is
// the reference's drhoi_dr*rho[i] + drhoj_dr*rho[j].
#pragma once
#include "force.hpp"

#pragma clang fp contract(fast)

namespace mappdmd {

struct EamBufs {
    const double* rows;  // [nr][nt*nt][kEamRow]: per row and ordered type pair (i, j) the cubic
                         // coefficients of j's density at i, i's density at j and r phi
    const double* F7;    // [nt][nrho+1][7]
    int nt;
};
// A pair reads 96 consecutive bytes of one 128-byte line; from the three tables of 7
// coefficients it read 168 bytes of three or more (the derivative's coefficients are
// those of the value times 1, 2, 3 and 1/dr).
constexpr int kEamRow = 16;

// FSM is FS with the cutoff tests on squares (rsq < cut^2, src/ff_fsm.cpp:424,
// :463, :518); its one-sweep density force (:466-476) is the same sum as FS's
// two factors (-A/sqrt(rho) kept per site) in another rounding order
enum { kModelEam = 0, kModelLj = 1, kModelFs = 2, kModelFsm = 3 };

// 16 lanes (one DPP row) per site in every pass: each lane takes every 16th
// list entry, the group sums per-site values in a fixed tree
constexpr int kEamG = 16;
// rounds of a list whose loads are issued together, before the first of their stores
// (a load waits for the stores issued before it)
constexpr int kEamR = 3;

// {x, y, z, type} per site: a pair's partner comes with one 32-byte read
__global__ void k_eam_pack(const double4* __restrict__ pos, const double* __restrict__ type, int n,
                           double4* __restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 p = pos[i];
    p.w = type[i];
    rec[i] = p;
}
// dF of the ghosts into rec[].w (pass 2 needs no types)
__global__ void k_eam_ghost_dF(double4* __restrict__ rec, int natms, int nghost, const int* __restrict__ owner) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g < nghost) rec[natms + g].w = rec[owner[g]].w;
}

// the row of a pair at distance^2 rsq (any value: the last row beyond the table)
struct EamLine {
    double c[12], r_inv, p;
    __device__ __forceinline__ void load(const FFParams<double>& P, const EamBufs& T, int it, int jt, double rsq) {
        r_inv = rsqrt_nr(rsq);
        p = rsq * r_inv * P.dr_inv;
        int m = (int)p;
        m = m < P.nr - 2 ? m : P.nr - 2;
        m = m > 0 ? m : 0;
        p -= m;
        p = p < 1.0 ? p : 1.0;
        const double2* row =
            reinterpret_cast<const double2*>(T.rows + ((size_t)m * (T.nt * T.nt) + it * T.nt + jt) * kEamRow);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            const double2 v = row[k];
            c[2 * k] = v.x;
            c[2 * k + 1] = v.y;
        }
    }
    __device__ __forceinline__ double value(int f) const {
        return ((c[4 * f + 3] * p + c[4 * f + 2]) * p + c[4 * f + 1]) * p + c[4 * f];
    }
    __device__ __forceinline__ double slope(int f, double dr_inv) const {
        return ((3.0 * c[4 * f + 3] * p + 2.0 * c[4 * f + 2]) * p + c[4 * f + 1]) * dr_inv;
    }
};

// one pair (i of type it, j of type jt at distance^2 rsq) of a model:
// density shares rho_i (at i) and rho_j (at j), pair energy, pair force
// coefficient fpair (force on i = fpair * dx) and the density records
// {drho_i, drho_j} of pass 2; returns false when the pair contributes nothing
template <int MODEL, bool ENERGY_ONLY>
__device__ __forceinline__ bool md_pair(const EamLine& row,
                                        const FFParams<double>& P, const EamBufs& T, const MdParams& M, int it,
                                        int jt, double rsq, double* rho_i, double* rho_j, double* phi,
                                        double* fpair, double2* dr) {
    *rho_i = *rho_j = *phi = *fpair = 0.0;
    *dr = make_double2(0.0, 0.0);
    if constexpr (MODEL == kModelEam) {
        if (!(rsq < P.cut_sq)) return false;
        const double r_inv = row.r_inv;
        *rho_i = row.value(0);
        *rho_j = row.value(1);
        *phi = row.value(2) * r_inv;
        if (!ENERGY_ONLY) {
            const double dphi_dr = row.slope(2, P.dr_inv) * r_inv - *phi * r_inv;
            *fpair = -dphi_dr * r_inv;
            *dr = make_double2(-row.slope(0, P.dr_inv) * r_inv, -row.slope(1, P.dr_inv) * r_inv);
        }
        return true;
    } else if constexpr (MODEL == kModelLj) {
        const int c = md_comp(it, jt);
        if (!M.chk[c] || !(rsq < M.cut_sq[c])) return false;
        const double sig = M.sig[c], eps = M.eps[c];
        const double sig2 = sig * sig / rsq;
        const double sig6 = sig2 * sig2 * sig2;
        const double sig12 = sig6 * sig6;
        *phi = 4.0 * eps * (sig12 - sig6) + M.offset[c];
        if (!ENERGY_ONLY) *fpair = 24.0 * eps * (2.0 * sig12 - sig6) / rsq;
        return true;
    } else {
        const int c = md_comp(it, jt);
        if (!M.chk[c] || !(rsq < M.cut_sq[c])) return false;
        const double r = sqrt(rsq);
        const double r_inv = 1.0 / r;
        constexpr bool kSq = MODEL == kModelFsm;
        if (kSq ? rsq < M.cut_sq_rho[c] : r < M.cut_rho[c]) {
            const double d = r - M.cut_rho[c];
            *rho_i = d * d * (M.t1[jt][it] + M.t2[jt][it] * d);
            *rho_j = d * d * (M.t1[it][jt] + M.t2[it][jt] * d);
            if (!ENERGY_ONLY)
                *dr = make_double2(-r_inv * d * (M.t1[jt][it] + 1.5 * M.t2[jt][it] * d),
                                   -r_inv * d * (M.t1[it][jt] + 1.5 * M.t2[it][jt] * d));
        }
        if (kSq ? rsq < M.cut_sq_phi[c] : r < M.cut_phi[c]) {
            const double d = r - M.cut_phi[c];
            const double k1 = M.k1[c], k2 = M.k2[c], k3 = M.k3[c];
            *phi = d * d * (k1 + k2 * r + k3 * rsq);
            if (!ENERGY_ONLY) {
                double pc = 2.0 * d * (k1 + k2 * r + k3 * rsq) + d * d * (k2 + 2.0 * k3 * r);
                pc *= -r_inv;
                *fpair = pc;
            }
        }
        return true;
    }
}


// Sums and records of a pair list go through three passes.  The force on i from a pair
// is S (x_i - x_j), S = fpair + F'_i drho_i + F'_j drho_j: pass 1 keeps fpair, drho_i and
// drho_j per pair (component by component, so that a round stores whole lines) and gives
// the partner its density share; pass 2 forms S, the own force and the virial, and
// leaves S at the pair's place in the partner's reverse list; the gather adds S
// (x_owner - x_i) over that list.  The first version summed pair and embedding forces
// separately, with a 24-byte share to the partner from each pass.  LJ has no densities:
// pass 1 does the work of pass 2.
struct EamPairs {
    double *f, *di, *dj;  // per pair: fpair, drho_i, drho_j
    double *rho, *S;      // per reverse-list entry: the partner's density share; S
};

// the pair's part of the force and the virial
struct ForceSums {
    double f[3] = {0.0, 0.0, 0.0}, v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    __device__ __forceinline__ void add(double S, double w, double dx0, double dx1, double dx2) {
        const double s0 = S * dx0, s1 = S * dx1, s2 = S * dx2;
        f[0] += s0;
        f[1] += s1;
        f[2] += s2;
        v[0] -= w * s0 * dx0;
        v[1] -= w * s1 * dx1;
        v[2] -= w * s2 * dx2;
        v[3] -= w * s1 * dx2;
        v[4] -= w * s2 * dx0;
        v[5] -= w * s0 * dx1;
    }
    // sums of the group, stored by its first lane
    __device__ __forceinline__ void store(int l, double* fown) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double a = group_sum<kEamG>(f[k]);
            if (l == 0) fown[k] = a;
        }
    }
};

// Pass 1 is bound by the gathers of positions and table rows (L2; TA 86% busy).  At 1,048,576 sites
// of two EAM types (41 million list entries): 0.74 ms, pass 2 0.41 and the gather 0.18;
// with rows of 7 coefficients, one entry at a time and both shares as vectors they took
// 1.27, 0.65 and 0.28.  kEamR = 2 gives 0.76, 0.45, 0.21; 4 gives 0.77, 0.46, 0.20.
template <int MODEL, bool ENERGY_ONLY>
__global__ __launch_bounds__(kBlock) void k_eam_pass1(FFParams<double> P, EamBufs T, MdParams M,
                                                      const double4* __restrict__ rec, PairBufs L, EamPairs O,
                                                      double* __restrict__ rho_own, double* __restrict__ fown,
                                                      double* __restrict__ part) {
    constexpr bool kForce = MODEL == kModelLj && !ENERGY_ONLY;
    const SiteGroup<kEamG> g;
    const int i = g.site;
    double acc[kForce ? 7 : 1] = {};
    if (i < P.natms) {
        const double4 xi = rec[i];
        const int it = (int)xi.w;
        double rho = 0.0;
        ForceSums F;
        const int p1 = L.off[i + 1];
        for (int p0 = L.off[i] + g.l; p0 < p1; p0 += kEamG * kEamR) {
            int2 e[kEamR];
            double dx0[kEamR], dx1[kEamR], dx2[kEamR], rsq[kEamR], rho_j[kEamR], pf[kEamR];
            double2 dr[kEamR];
            int jt[kEamR];
            EamLine row[kEamR];
#pragma unroll
            for (int r = 0; r < kEamR; ++r) {
                const int p = p0 + r * kEamG;
                e[r] = L.nlrp[p < p1 ? p : p1 - 1];
            }
#pragma unroll
            for (int r = 0; r < kEamR; ++r) {
                const double4 xj = rec[e[r].x];
                dx0[r] = xi.x - xj.x;
                dx1[r] = xi.y - xj.y;
                dx2[r] = xi.z - xj.z;
                jt[r] = (int)xj.w;
                {
#pragma clang fp contract(off)
                    rsq[r] = dx0[r] * dx0[r] + dx1[r] * dx1[r] + dx2[r] * dx2[r];
                }
                if constexpr (MODEL == kModelEam) row[r].load(P, T, it, jt[r], rsq[r]);
            }
#pragma unroll
            for (int r = 0; r < kEamR; ++r) {
                const bool listed = p0 + r * kEamG < p1, owned = e[r].y >= 0;
                double rho_i, phi;
                rho_j[r] = pf[r] = 0.0;
                dr[r] = make_double2(0.0, 0.0);
                if (listed && md_pair<MODEL, ENERGY_ONLY>(row[r], P, T, M, it, jt[r], rsq[r], &rho_i, &rho_j[r], &phi,
                                                          &pf[r], &dr[r])) {
                    const double w = owned ? 1.0 : 0.5;
                    rho += rho_i;
                    acc[0] += w * phi;
                    if constexpr (kForce) F.add(pf[r], w, dx0[r], dx1[r], dx2[r]);
                }
            }
#pragma unroll
            for (int r = 0; r < kEamR; ++r) {
                const int p = p0 + r * kEamG;
                if (p >= p1) continue;
                if (!ENERGY_ONLY && MODEL != kModelLj) {
                    O.f[p] = pf[r];
                    O.di[p] = dr[r].x;
                    O.dj[p] = dr[r].y;
                }
                if (e[r].y >= 0) {
                    if (MODEL != kModelLj) O.rho[e[r].y] = rho_j[r];
                    if (kForce) O.S[e[r].y] = pf[r];
                }
            }
        }
        rho = group_sum<kEamG>(rho);
        if (g.l == 0) rho_own[i] = rho;
        if constexpr (kForce) {
            F.store(g.l, fown + (size_t)i * 3);
#pragma unroll
            for (int k = 0; k < 6; ++k) acc[1 + k] = F.v[k];
        }
    }
    block_sum_store<kForce ? 7 : 1>(acc, part);
}

// rho_i = own + partner shares; EAM: F(rho) (cubic rows, linear above
// rho_max), F' kept; FS: -A sqrt(rho), and -A/sqrt(rho) kept
// (src/ff_fs.cpp:524-526)
template <int MODEL, bool ENERGY_ONLY>
__global__ __launch_bounds__(kBlock) void k_eam_embed(FFParams<double> P, EamBufs T, MdParams M,
                                                      const double* __restrict__ type, PairBufs L,
                                                      const double* __restrict__ rho_own,
                                                      const double* __restrict__ pairE, double* __restrict__ rho,
                                                      double* __restrict__ dF, double4* __restrict__ rec,
                                                      double* __restrict__ part) {
    const SiteGroup<kEamG> g;
    const int i = g.site;
    double acc[1] = {0.0};
    if (i < P.natms) {
        double part_r = 0.0;
        const int q1 = L.roff[i + 1];
        for (int q0 = L.roff[i] + g.l; q0 < q1; q0 += kEamG * kEamR) {
            double v[kEamR];
#pragma unroll
            for (int r = 0; r < kEamR; ++r) v[r] = q0 + r * kEamG < q1 ? pairE[q0 + r * kEamG] : 0.0;
#pragma unroll
            for (int r = 0; r < kEamR; ++r) part_r += v[r];
        }
        double r = rho_own[i] + group_sum<kEamG>(part_r);
        const int it = (int)type[i];
        if (g.l != 0) {
            // one lane per site evaluates the embedding
        } else if constexpr (MODEL == kModelFs || MODEL == kModelFsm) {
            const double sq = sqrt(r);
            acc[0] = -(M.A[it] * sq);
            rho[i] = r;
            if (!ENERGY_ONLY) dF[i] = rec[i].w = -M.A[it] / sq;
        } else {
            double pp = r * P.drho_inv;
            int m = (int)pp;
            m = m < P.nr - 2 ? m : P.nr - 2;
            m = m > 0 ? m : 0;
            pp -= m;
            pp = pp < 1.0 ? pp : 1.0;
            const double* c = T.F7 + ((size_t)it * (P.nrho + 1) + m) * 7;
            const double d = (c[6] * pp + c[5]) * pp + c[4];
            double Fv = ((c[3] * pp + c[2]) * pp + c[1]) * pp + c[0];
            if (r > P.rho_max) Fv += d * (r - P.rho_max);
            acc[0] = Fv;
            rho[i] = r;
            if (!ENERGY_ONLY) dF[i] = rec[i].w = d;
        }
    }
    block_sum_store<1>(acc, part);
}

// rec = {x, y, z, F'}
__global__ __launch_bounds__(kBlock) void k_eam_pass2(FFParams<double> P, const double4* __restrict__ rec, PairBufs L,
                                                      EamPairs O, double* __restrict__ fown,
                                                      double* __restrict__ part) {
    const SiteGroup<kEamG> g;
    const int i = g.site;
    ForceSums F;
    if (i < P.natms) {
        const double4 xi = rec[i];
        const int p1 = L.off[i + 1];
        for (int p0 = L.off[i] + g.l; p0 < p1; p0 += kEamG * kEamR) {
            int2 e[kEamR];
            double S[kEamR], di[kEamR], dj[kEamR];
            double4 xj[kEamR];
#pragma unroll
            for (int r = 0; r < kEamR; ++r) {
                const int p = p0 + r * kEamG < p1 ? p0 + r * kEamG : p1 - 1;
                e[r] = L.nlrp[p];
                S[r] = O.f[p];
                di[r] = O.di[p];
                dj[r] = O.dj[p];
            }
#pragma unroll
            for (int r = 0; r < kEamR; ++r) xj[r] = rec[e[r].x];
#pragma unroll
            for (int r = 0; r < kEamR; ++r) {
                // pairs outside the cutoff have zero records; F' of a site without density
                // may be infinite (FS), and counts only where there is a slope
                if (di[r] != 0.0 || dj[r] != 0.0) S[r] += xi.w * di[r] + xj[r].w * dj[r];
                const bool on = p0 + r * kEamG < p1 && S[r] != 0.0;
                if (on) F.add(S[r], e[r].y >= 0 ? 1.0 : 0.5, xi.x - xj[r].x, xi.y - xj[r].y, xi.z - xj[r].z);
            }
#pragma unroll
            for (int r = 0; r < kEamR; ++r)
                if (p0 + r * kEamG < p1 && e[r].y >= 0) O.S[e[r].y] = S[r];
        }
        F.store(g.l, fown + (size_t)i * 3);
    }
    block_sum_store<6>(F.v, part);
}

// f = own sum + the shares of the pairs that list the site
__global__ __launch_bounds__(kBlock) void k_eam_gather(int natms, PairBufs L, const int* __restrict__ rowner,
                                                       const double4* __restrict__ rec, const double* __restrict__ S,
                                                       const double* __restrict__ fown, double* __restrict__ f) {
    const SiteGroup<kEamG> g;
    const int i = g.site;
    if (i >= natms) return;
    const double4 xi = rec[i];
    double a[3] = {0.0, 0.0, 0.0};
    const int q1 = L.roff[i + 1];
    for (int q0 = L.roff[i] + g.l; q0 < q1; q0 += kEamG * kEamR) {
        int o[kEamR];
        double s[kEamR];
        double4 xo[kEamR];
#pragma unroll
        for (int r = 0; r < kEamR; ++r) {
            const int q = q0 + r * kEamG < q1 ? q0 + r * kEamG : q1 - 1;
            o[r] = rowner[q];
            s[r] = S[q];
        }
#pragma unroll
        for (int r = 0; r < kEamR; ++r) xo[r] = rec[o[r]];
#pragma unroll
        for (int r = 0; r < kEamR; ++r) {
            if (q0 + r * kEamG >= q1 || s[r] == 0.0) continue;
            a[0] += s[r] * (xi.x - xo[r].x);
            a[1] += s[r] * (xi.y - xo[r].y);
            a[2] += s[r] * (xi.z - xo[r].z);
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double v = group_sum<kEamG>(a[k]);
        if (g.l == 0) f[(size_t)i * 3 + k] = fown[(size_t)i * 3 + k] + v;
    }
}

}  // namespace mappdmd

#pragma clang fp contract(off)
