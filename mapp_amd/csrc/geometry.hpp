// Geometry kernels: periodic ghosts in reduced coordinates, cell binning and
// the half neighbor list, restating the single-rank reference algorithms
//   Atoms::set_ph / ph_setup / ph_xchng   src/atoms.cpp:249-372, :464-497
//   Atoms::update (x and plain vectors)   src/atoms.cpp:1088-1220
//   Atoms::update_0 / x2s / s2x           src/atoms.cpp:1780-1941
//   Neighbor::create_bin_list / find_bin_no / bin_atoms_s / s2bin / create_list
//                                         src/neighbor.cpp:137-525
// The library is compiled with -ffp-contract=off, so the s->x transform and
// the squared distances are the same separately rounded binary64 operations
// as the reference's; the list is therefore bit-identical, including order.
#pragma once
#include "dmd_common.hpp"

namespace mappdmd {

constexpr int kScanThreads = 256;
constexpr int kScanItems = 4;
constexpr int kScanTile = kScanThreads * kScanItems;

__device__ __forceinline__ double& comp3(double4& p, int d) {
    return d == 0 ? p.x : (d == 1 ? p.y : p.z);
}
__device__ __forceinline__ double comp3c(const double4& p, int d) {
    return d == 0 ? p.x : (d == 1 ? p.y : p.z);
}

// ---- exclusive scan over non-negative ints: tiles, the tile sums in one block,
// the sums added.  The total is kept in 64 bits (offsets are int: a total of 2^31 or
// more is refused by the caller) and written to host memory with the last launch. ----
__global__ __launch_bounds__(kScanThreads) void k_scan_tile(const int* __restrict__ in, int* __restrict__ out,
                                                            unsigned long long* __restrict__ sums, long n) {
    __shared__ unsigned long long sh[kScanThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const long base = (long)blockIdx.x * kScanTile + (long)tid * kScanItems;
    int v[kScanItems];
    unsigned long long tsum = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        long idx = base + k;
        v[k] = idx < n ? in[idx] : 0;
        tsum += (unsigned)v[k];
    }
    unsigned long long incl = tsum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const unsigned long long t = __shfl_up(incl, d, 64);
        if (lane >= d) incl += t;
    }
    if (lane == 63) sh[w] = incl;
    __syncthreads();
    unsigned long long before = 0, all = 0;
#pragma unroll
    for (int q = 0; q < kScanThreads / 64; ++q) {
        if (q < w) before += sh[q];
        all += sh[q];
    }
    int excl = (int)(before + incl - tsum);
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        long idx = base + k;
        if (idx < n) out[idx] = excl;
        excl += v[k];
    }
    if (tid == 0) sums[blockIdx.x] = all;
}

constexpr int kScanSumThreads = 1024;
// exclusive scan of the nb tile sums in place by one block; the total to *total
__global__ __launch_bounds__(kScanSumThreads) void k_scan_sums(unsigned long long* __restrict__ sums, int nb,
                                                               unsigned long long* __restrict__ total) {
    __shared__ unsigned long long sh[kScanSumThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    unsigned long long carry = 0;
    for (int base = 0; base < nb; base += kScanSumThreads) {
        const unsigned long long v = base + tid < nb ? sums[base + tid] : 0;
        unsigned long long incl = v;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const unsigned long long t = __shfl_up(incl, d, 64);
            if (lane >= d) incl += t;
        }
        if (lane == 63) sh[w] = incl;
        __syncthreads();
        unsigned long long before = 0, all = 0;
#pragma unroll
        for (int q = 0; q < kScanSumThreads / 64; ++q) {
            if (q < w) before += sh[q];
            all += sh[q];
        }
        if (base + tid < nb) sums[base + tid] = carry + before + incl - v;
        carry += all;
        __syncthreads();
    }
    if (tid == 0) *total = carry;
}

// adds the tile sums; *end (optional) = the total; host[0] = the total and, with
// mid >= 0, host[1] = out[mid]; *aux (optional) to *host_aux
__global__ __launch_bounds__(kScanThreads) void k_scan_add(int* __restrict__ out,
                                                           const unsigned long long* __restrict__ add, long n,
                                                           const unsigned long long* __restrict__ total,
                                                           int* __restrict__ end, long mid, unsigned long long* host,
                                                           const int* __restrict__ aux, int* host_aux) {
    const long base = (long)blockIdx.x * kScanTile + (long)threadIdx.x * kScanItems;
    const int a = (int)add[blockIdx.x];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        long idx = base + k;
        if (idx < n) {
            const int v = out[idx] + a;
            out[idx] = v;
            if (idx == mid) host[1] = (unsigned long long)v;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (end) *end = (int)*total;
        host[0] = *total;
        if (aux) *host_aux = *aux;
    }
}

// ---- ghosts ----------------------------------------------------------------
// flag[i] = 1 when atom i lies within the ghost shell of the low face of dimension idim
// (s <= thr_lo), flag[n + i] that of the high face (thr_hi <= s)
__global__ void k_ghost_flag(const double4* __restrict__ pos, int n, int idim, double thr_lo, double thr_hi,
                             int* __restrict__ flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double s = comp3c(pos[i], idim);
    flag[i] = s <= thr_lo ? 1 : 0;
    flag[(long)n + i] = thr_hi <= s ? 1 : 0;
}

// copies flagged atoms to ghost rows n + offs[...], shifted by +1 (low face) or -1 in s
template <int NT>
__global__ void k_ghost_emit(double4* __restrict__ pos, double* __restrict__ alpha, double* __restrict__ conc, int n,
                             int idim, const int* __restrict__ flag, const int* __restrict__ offs, int natms,
                             int* __restrict__ ghost_src, int* __restrict__ ghost_owner) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
        const long e = (long)dir * n + i;
        if (!flag[e]) continue;
        const int g = n + offs[e];
        double4 p = pos[i];
        if (dir == 0) comp3(p, idim) += 1.0;
        else comp3(p, idim) -= 1.0;
        pos[g] = p;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            alpha[(long)g * NT + t] = alpha[(long)i * NT + t];
            conc[(long)g * NT + t] = conc[(long)i * NT + t];
        }
        ghost_src[g - natms] = i;
        ghost_owner[g - natms] = i < natms ? i : ghost_owner[i - natms];
    }
}

// Atoms::update of x between rebuilds: ghost = source +- H[idim][0..idim], its source
// itself a ghost of an earlier swap or owned.  One thread per ghost walks back to the
// owned site (at most one swap per dimension) and applies the shifts in the swaps' order,
// the additions of six launches, one per swap, that took 2.8 us each (this one 4.2 at
// 32,000 sites).
struct GhostSwaps {
    int end[6];  // ghosts up to the end of each swap: low and high face of each dimension
    double H[3][3];
};
template <int NT>
__global__ void k_ghost_update_x(double4* __restrict__ pos, double* __restrict__ alpha, int natms, int nghost,
                                 const int* __restrict__ ghost_src, GhostSwaps W) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nghost) return;
    int swap[3], n = 0, src = natms + g;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (src < natms) break;
        const int e = src - natms;
        int w = 0;
#pragma unroll
        for (int q = 0; q < 5; ++q) w += e >= W.end[q] ? 1 : 0;
        swap[k] = w;
        n = k + 1;
        src = ghost_src[e];
    }
    double4 p = pos[src];
#pragma unroll
    for (int k = 2; k >= 0; --k) {
        if (k >= n) continue;
        const int d = swap[k] >> 1;
        const double sgn = swap[k] & 1 ? -1.0 : 1.0;
        p.x += sgn * W.H[d][0];
        if (d >= 1) p.y += sgn * W.H[d][1];
        if (d >= 2) p.z += sgn * W.H[d][2];
    }
    pos[natms + g] = p;
#pragma unroll
    for (int t = 0; t < NT; ++t) alpha[(long)(natms + g) * NT + t] = alpha[(long)src * NT + t];
}

// forward copy of a per-atom vector to its ghosts (Atoms::update of E, dE, n ...)
template <typename T>
__global__ void k_ghost_copy(T* __restrict__ v, int d, int natms, int nghost, const int* __restrict__ owner) {
    int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= nghost) return;
    int o = owner[g];
    for (int k = 0; k < d; ++k) v[(long)(natms + g) * d + k] = v[(long)o * d + k];
}

// ---- box transforms --------------------------------------------------------
// Atoms::s2x: x_j = s_j H_jj + sum_{k>j} H_kj s_k (lower-triangular H)
__device__ __forceinline__ double4 s2x(double4 s, const BoxParams& bp) {
    double x0 = s.x * bp.H[0][0];
    x0 += bp.H[1][0] * s.y;
    x0 += bp.H[2][0] * s.z;
    double x1 = s.y * bp.H[1][1];
    x1 += bp.H[2][1] * s.z;
    const double x2 = s.z * bp.H[2][2];
    return make_double4(x0, x1, x2, 0.0);
}

// Atoms::x2s with the wrap into [0,1)
__global__ void k_x2s(double4* __restrict__ pos, int n, BoxParams bp) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double4 x = pos[i];
    double s0 = x.x * bp.B[0][0];
    s0 += bp.B[1][0] * x.y;
    s0 += bp.B[2][0] * x.z;
    double s1 = x.y * bp.B[1][1];
    s1 += bp.B[2][1] * x.z;
    double s2 = x.z * bp.B[2][2];
    double s[3] = {s0, s1, s2};
    for (int j = 0; j < 3; ++j) {
        // bounded loops: a site more than 64 boxes away is an input error
        for (int it = 0; it < 64 && s[j] < 0.0; ++it) s[j]++;
        for (int it = 0; it < 64 && s[j] >= 1.0; ++it) s[j]--;
    }
    pos[i] = make_double4(s[0], s[1], s[2], 0.0);
}

// ---- cell binning (reduced coordinates) -----------------------------------
// slot[i] = the arrival number of atom i in its bin (arbitrary: atomics); the atoms are
// [first, n).  bin_cnt[bp.tot_bin] += the bins that were empty (the owned sites come first,
// so after their launch it is the number of bins with an owned site).
__global__ __launch_bounds__(256) void k_s2bin(const double4* __restrict__ pos, int first, int n, BoxParams bp,
                                               int* __restrict__ bin_of, int* __restrict__ bin_cnt,
                                               int* __restrict__ slot) {
    const int i = first + blockIdx.x * blockDim.x + threadIdx.x;
    int opened = 0;
    if (i < n) {
        double4 s = pos[i];
        int no = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            int t = (int)((comp3c(s, d) + bp.cut_ph_s[d] - 0.0) / bp.bin_size[d]);
            t = t < 0 ? 0 : (t > bp.grid[d] - 1 ? bp.grid[d] - 1 : t);  // in range for valid input
            no += t * bp.denom[d];
        }
        bin_of[i] = no;
        const int at = atomicAdd(&bin_cnt[no], 1);
        slot[i] = at;
        opened = at == 0 ? 1 : 0;
    }
    const int total = __syncthreads_count(opened);
    if (threadIdx.x == 0 && total) atomicAdd(&bin_cnt[bp.tot_bin], total);
}

__global__ void k_bin_fill(const int* __restrict__ bin_of, int n, const int* __restrict__ bin_start,
                           const int* __restrict__ slot, int* __restrict__ bin_atoms) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    bin_atoms[bin_start[bin_of[i]] + slot[i]] = i;
}

// Atom indices in ascending order inside every bin, as the reference's linked bins
// built by pushing atoms from the highest index down (src/neighbor.cpp:428-434), and
// the end of Neighbor::bin_atoms_s, s2x of every atom.  One thread per atom: atom x of
// bin s goes to bin_start[s] + r, r = the number of the bin's atoms below x; its
// position (w: its type, with a cutoff per type pair) is also kept in that order, where
// the list kernel reads consecutive candidates from consecutive addresses.
__global__ void k_bin_place(const int* __restrict__ v, int n, const int* __restrict__ bin_of,
                            const int* __restrict__ bin_start, BoxParams bp, const double* __restrict__ type,
                            double4* __restrict__ pos, int* __restrict__ bin_atoms, double4* __restrict__ bin_pos) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= n) return;
    const int x = v[q];
    const int s = bin_of[x];
    const int lo = bin_start[s], hi = bin_start[s + 1];
    int r = 0;
    for (int t = lo; t < hi; ++t) r += v[t] < x ? 1 : 0;
    double4 p = s2x(pos[x], bp);
    pos[x] = p;
    if (bp.pairwise) p.w = type[x];
    bin_atoms[lo + r] = x;
    bin_pos[lo + r] = p;
}

// ---- half neighbor list ----------------------------------------------------
// stencil order of find_bin_no: offset of dimension 0 outermost, 2 innermost;
// inside a bin ascending index; j > i (every j != i with bp.full, the full list
// of src/neighbor.cpp:240-284); rsq = ((d0*d0) + d1*d1) + d2*d2 < cut.
// One wavefront per group of kBinSites sites of one bin: lane s < 27 takes stencil bin s
// (s = 9(a+1) + 3(b+1) + c+1 for offsets a, b, c), a prefix sum of the bin sizes
// concatenates the 27 bins in stencil order, and 64 consecutive candidates, read once,
// are tested per round against each site of the group; ballot ranks write the accepted
// ones in candidate order, which is the list order of a single thread walking the
// stencil.
//
// The same tests give a site's reverse list: the owners of pairs with site i are the
// accepted j < i (the stencil and the distance are the same from either end).  The
// count launch keeps each round's accept bits, kMaskWords rounds of them, and the fill
// launch tests again only what lies beyond; the owners come out in stencil order and
// are sorted by k_sort_owners.
//
// Bound by the vector instructions of the tests and, at the start of a wavefront, by
// the chain of loads that finds the candidates.  At 293,000 sites (16 to a bin, 430
// candidates each) the count takes 0.15 ms, the fill 0.17 and the sort 0.09; one
// wavefront per site, both launches testing, took 0.33 + 0.36 for the half list alone,
// and the reverse list made from it by atomics, a sort and four passes over the pairs
// 0.74 where the sort and k_pair_links take 0.24.  Groups of 8 or 16 sites are slower
// (0.20 and 0.50: fewer wavefronts, more registers).
//
// A box that is mostly empty has more bins than sites, and a block for each costs 0.2 us
// per 1,000 empty bins in either launch, up to the launch limit of 2^24 blocks of this
// size.  So where there are more than kFewBins bins, and more than a quarter of the sites
// (a filled box has some 16 sites to a bin), the launch goes over the list of the bins
// that hold an owned site, which five small launches make.  864 sites in a box of 500 A
// (730,000 bins), rebuild with the host's part: 478 -> 212 us; in one of 1,000 A (5.6
// million bins) 2,534 -> 264 us.
constexpr long kFewBins = 65536;
constexpr int kBinSites = 4;
constexpr int kBinWaves = 4;  // wavefronts per block; those of a bin's blocks take its groups in turn
// Blocks per bin for a mean of `sites` owned sites to an occupied bin: one for each
// kBinShare, the sites that a block's wavefronts take in one turn, so that a crowded bin (a
// long cutoff, a compressed box) is not left to four wavefronts.  Rebuild with the host's
// part, one block per bin -> this: 4,000 LJ sites with a cutoff of 12 A (150 to a bin) 1.72
// -> 0.62 ms, 32,000 with 16 A (348) 11.8 -> 4.3, 4,000 sites in a box of 9 A (500) 39.1 ->
// 4.0; a cluster of 4,000 with 16 A in a box of 20 cutoffs 3.21 -> 0.99 (the mean over the
// occupied bins, not over the box, counts).
constexpr int kBinShare = 16;
inline int bin_blocks(double sites) {
    const double b = sites / kBinShare;
    return b < 1.0 ? 1 : (b > 256.0 ? 256 : (int)b);
}
constexpr int kMaskWords = 16;
// what one lane of a wavefront left in LDS is there for the others (no instruction: LDS
// accesses of a wavefront are in order, so only the compiler has to keep theirs)
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// set bits of m below this lane
__device__ __forceinline__ int lane_rank(unsigned long long m) {
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
}
__device__ __forceinline__ unsigned long long read_lane_u64(unsigned long long v, int l) {
    const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)v, l);
    const unsigned hi = __builtin_amdgcn_readlane((int)(unsigned)(v >> 32), l);
    return (unsigned long long)hi << 32 | lo;
}
struct HalfLists {
    unsigned long long* mask;  // [natms][kMaskWords] accept bits
    int *cnt, *rcnt;           // count: entries of the site's own and reverse lists
    const int *off, *roff;     // fill: their offsets
    int *nl, *rlist;           // fill: partners in list order; owners in stencil order
};
// flag[b] = 1 for a bin with an owned site (owned sites come first in a bin)
__global__ void k_bin_owned(const int* __restrict__ bin_start, const int* __restrict__ bin_atoms, int tot_bin,
                            int natms, int* __restrict__ flag) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= tot_bin) return;
    const int k = bin_start[b];
    flag[b] = k < bin_start[b + 1] && bin_atoms[k] < natms ? 1 : 0;
}
__global__ void k_bin_list(const int* __restrict__ flag, const int* __restrict__ offs, int tot_bin,
                           int* __restrict__ bins) {
    const int b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b < tot_bin && flag[b]) bins[offs[b]] = b;
}
// bins: the bins with an owned site, nbin of them; null: every bin.
// PAIRWISE: a cutoff per type pair (bp.cut_sk_sq_tp), the type in bin_pos[].w
template <bool FILL, bool PAIRWISE>
__global__ __launch_bounds__(64 * kBinWaves) void k_half_list(int natms, const int* __restrict__ bins, int nbin,
                                                              const int* __restrict__ bin_start,
                                                              const int* __restrict__ bin_atoms,
                                                              const double4* __restrict__ bin_pos, BoxParams bp,
                                                              HalfLists L) {
    __shared__ unsigned long long ends_lds[kBinWaves][64];
    __shared__ int2 bin_lds[kBinWaves][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int at = blockIdx.z * gridDim.x + blockIdx.x;
    if (at >= nbin) return;  // the whole block
    const int bin = bins ? bins[at] : at;
    const int k1 = bin_start[bin + 1];
    int k0 = bin_start[bin] + (blockIdx.y * kBinWaves + wave) * kBinSites;
    // owned sites come first in a bin
    if (k0 >= k1 || bin_atoms[k0] >= natms) return;  // the whole wavefront
    int tmp = bin;
    int loc[3];
    for (int d = 2; d > -1; --d) {
        loc[d] = tmp / bp.denom[d];
        tmp -= loc[d] * bp.denom[d];
    }
    int bstart = 0, bsize = 0;
    if (lane < 27) {
        const int t0 = loc[0] + lane / 9 - 1, t1 = loc[1] + (lane / 3) % 3 - 1, t2 = loc[2] + lane % 3 - 1;
        if (t0 >= 0 && t0 < bp.grid[0] && t1 >= 0 && t1 < bp.grid[1] && t2 >= 0 && t2 < bp.grid[2]) {
            const int no = t0 * bp.denom[0] + t1 * bp.denom[1] + t2 * bp.denom[2];
            bstart = bin_start[no];
            bsize = bin_start[no + 1] - bstart;
        }
    }
    // the occupied bins packed into the low lanes, so that their last candidates are distinct
    const unsigned long long occ = __ballot(bsize > 0);
    const int nocc = __popcll(occ);
    if (bsize > 0) bin_lds[wave][lane_rank(occ)] = make_int2(bstart, bsize);
    wave_lds_sync();
    bstart = bsize = 0;
    if (lane < nocc) {
        const int2 e = bin_lds[wave][lane];
        bstart = e.x;
        bsize = e.y;
    }
    int incl = bsize;  // inclusive prefix over the bins
    for (int d = 1; d < 32; d <<= 1) {
        const int v = __shfl_up(incl, d, 64);
        if (lane >= d) incl += v;
    }
    const int to_bin = bstart - (incl - bsize);  // candidate number -> place in the bins
    const int total = __builtin_amdgcn_readlane(incl, 31);
    for (; k0 < k1; k0 += gridDim.y * kBinWaves * kBinSites) {
        int site[kBinSites], w[kBinSites], wr[kBinSites];
        double4 xi[kBinSites];
        unsigned long long keep[kBinSites];
#pragma unroll
        for (int u = 0; u < kBinSites; ++u) {
            const int k = k0 + u < k1 ? k0 + u : k1 - 1;
            const int i = bin_atoms[k];
            site[u] = k0 + u < k1 && i < natms ? i : -1;
            xi[u] = bin_pos[k];
            // in vector registers: as scalars the group does not fit, and each use pays a move
            if (!FILL) asm("" : "+v"(xi[u].x), "+v"(xi[u].y), "+v"(xi[u].z));
            w[u] = wr[u] = 0;
            keep[u] = 0;
            if (FILL && site[u] >= 0) {
                w[u] = L.off[i];
                wr[u] = L.roff[i];
                if (lane < kMaskWords && lane * 64 < total) keep[u] = L.mask[(size_t)i * kMaskWords + lane];
            }
        }
        if (site[0] < 0) break;
        unsigned long long ends = 0;  // lane r: which candidates of the 64 rounds' round r are the last of their bin
        int nb = 0;                   // bins that end before this round
        for (int base = 0, round = 0; base < total; base += 64, ++round) {
            if ((round & 63) == 0) {
                wave_lds_sync();
                ends_lds[wave][lane] = 0;
                wave_lds_sync();
                const int e = incl - 1 - base;
                if (lane < nocc && e >= 0 && e < 4096) atomicOr(&ends_lds[wave][e >> 6], 1ull << (e & 63));
                wave_lds_sync();
                ends = ends_lds[wave][lane];
            }
            const unsigned long long last = read_lane_u64(ends, round & 63);
            const int s = nb + lane_rank(last);  // bin of candidate base + lane
            nb += __popcll(last);
            const int q = base + lane;
            const int k = __shfl(to_bin, s, 64) + q;
            const bool kept = FILL && round < kMaskWords;
            const unsigned long long valid = __builtin_amdgcn_ballot_w64(q < total);
            int j = 0;
            double4 xj{};
            if (q < total) {
                j = bin_atoms[k];
                if (!kept) xj = bin_pos[k];
            }
#pragma unroll
            for (int u = 0; u < kBinSites; ++u) {
                const int i = site[u];
                if (i < 0) continue;
                unsigned long long near;
                if (kept) {
                    near = read_lane_u64(keep[u], round);
                } else {
                    double d0 = xi[u].x - xj.x, d1 = xi[u].y - xj.y, d2 = xi[u].z - xj.z;
                    double rsq = 0.0;
                    rsq += d0 * d0;
                    rsq += d1 * d1;
                    rsq += d2 * d2;
                    const double cut =
                        PAIRWISE ? bp.cut_sk_sq_tp[md_comp((int)xi[u].w, (int)xj.w)] : bp.cut_sk_sq;
                    near = __builtin_amdgcn_ballot_w64(rsq < cut) & valid;
                }
                // j == i is neither
                const unsigned long long above = __builtin_amdgcn_ballot_w64(j > i) & near;
                const unsigned long long below = __builtin_amdgcn_ballot_w64(j < i) & near;
                const unsigned long long own = bp.full ? above | below : above, rv = bp.full ? 0 : below;
                if constexpr (FILL) {
                    if (own >> lane & 1) L.nl[w[u] + lane_rank(own)] = j;
                    if (rv >> lane & 1) L.rlist[wr[u] + lane_rank(rv)] = j;
                } else if (lane == round) {
                    keep[u] = own | rv;
                }
                w[u] += __popcll(own);
                wr[u] += __popcll(rv);
            }
        }
        if constexpr (!FILL) {
#pragma unroll
            for (int u = 0; u < kBinSites; ++u) {
                const int i = site[u];
                if (i < 0) continue;
                if (lane < kMaskWords && lane * 64 < total) L.mask[(size_t)i * kMaskWords + lane] = keep[u];
                if (lane == 0) {
                    L.cnt[i] = w[u];
                    L.rcnt[i] = wr[u];
                }
            }
        }
    }
}

// the owners of a site's reverse list in ascending order: ranked 64 at a time against
// each other (they are distinct), one wavefront per site
__global__ __launch_bounds__(256) void k_sort_owners(int natms, const int* __restrict__ roff,
                                                     const int* __restrict__ tmp, int* __restrict__ rowner) {
    const int lane = threadIdx.x & 63;
    const long site = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (site >= natms) return;  // the whole wavefront
    const int i = __builtin_amdgcn_readfirstlane((int)site);
    const int q0 = roff[i], q1 = roff[i + 1];
    for (int a = q0; a < q1; a += 64) {
        const int x = a + lane < q1 ? tmp[a + lane] : 0x7FFFFFFF;
        int r = 0;
        for (int b = q0; b < q1; b += 64) {
            const int y = b == a ? x : (b + lane < q1 ? tmp[b + lane] : 0x7FFFFFFF);
            const int ny = q1 - b < 64 ? q1 - b : 64;
            for (int l = 0; l < ny; l += 8) {  // those beyond ny rank below nothing
#pragma unroll
                for (int d = 0; d < 8; ++d) r += __builtin_amdgcn_readlane(y, l + d) < x ? 1 : 0;
            }
        }
        if (a + lane < q1) rowner[q0 + r] = x;
    }
}

// per half-list entry {partner, its position in the partner's reverse list or -1 for a
// ghost}: the owner's place among the partner's ascending owners, by bisection.  kLinkG
// lanes per site.  Every entry starts outside the quadrature cut.
constexpr int kLinkG = 32;
__global__ void k_pair_links(const int* __restrict__ off, const int* __restrict__ nl, int natms,
                             const int* __restrict__ roff, const int* __restrict__ rowner,
                             int2* __restrict__ nlrp) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = (int)(t / kLinkG), l = (int)(t % kLinkG);
    if (i >= natms) return;
    for (int p = off[i] + l; p < off[i + 1]; p += kLinkG) {
        const int j = nl[p];
        int q = -1;
        if (j < natms) {
            int lo = roff[j], hi = roff[j + 1];
            while (lo < hi) {
                const int mid = lo + (hi - lo) / 2;
                if (rowner[mid] < i) lo = mid + 1;
                else hi = mid;
            }
            q = lo;
        }
        nlrp[p] = make_int2(j, q);
    }
}

// Both ends of the 2nd list (create_2nd_neigh_lst: the half-list pairs with
// rsq < rsq_crd) per site: own pairs in list order as the partner (also nl2, the list
// itself), then the owners of the pairs that list the site, ascending, as ~owner.  One
// wavefront per site, 64 entries per round, ballot ranks keep the order.  cnt / tot:
// the own pairs and both ends, crd = both ends.
template <bool FILL>
__global__ __launch_bounds__(256) void k_list2(const double4* __restrict__ pos, int natms,
                                               const int* __restrict__ off, const int* __restrict__ nl,
                                               const int* __restrict__ roff, const int* __restrict__ rowner,
                                               double rsq_crd, int* __restrict__ cnt_or_off,
                                               int* __restrict__ tot_or_off, int* __restrict__ crd,
                                               int* __restrict__ nl2, int* __restrict__ fidx) {
    const int lane = threadIdx.x & 63;
    const long site = ((long)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    if (site >= natms) return;  // the whole wavefront
    const int i = (int)site;
    const double4 xi = pos[i];
    int w = FILL ? cnt_or_off[i] : 0, f = FILL ? tot_or_off[i] : 0;
#pragma unroll
    for (int end = 0; end < 2; ++end) {
        const int* const list = end ? rowner : nl;
        const int p1 = end ? roff[i + 1] : off[i + 1];
        for (int p0 = end ? roff[i] : off[i]; p0 < p1; p0 += 64) {
            const int p = p0 + lane;
            bool take = false;
            int j = 0;
            if (p < p1) {
                j = list[p] & 0x7FFFFFFF;  // owners carry a flag in the top bit
                const double4 xj = pos[j];
                double d0 = xi.x - xj.x, d1 = xi.y - xj.y, d2 = xi.z - xj.z;
                double rsq = d0 * d0 + d1 * d1 + d2 * d2;
                take = rsq < rsq_crd;
            }
            const unsigned long long m = __ballot(take);
            if (FILL && take) {
                const int r = lane_rank(m);
                fidx[f + r] = end ? ~j : j;
                if (!end) nl2[w + r] = j;
            }
            f += __popcll(m);
            if (!end) w += __popcll(m);
        }
    }
    if (!FILL && lane == 0) {
        cnt_or_off[i] = w;
        tot_or_off[i] = f;
        crd[i] = f;
    }
}

// Atoms::update_0 skin test: any owned site moved more than skin since the build
__global__ void k_skin_check(const double4* __restrict__ pos, const double4* __restrict__ x0, int natms,
                             double sq_skin, int* __restrict__ flag) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= natms) return;
    double4 a = pos[i], b = x0[i];
    double d0 = a.x - b.x, d1 = a.y - b.y, d2 = a.z - b.z;
    double sq = 0.0;
    sq += d0 * d0;
    sq += d1 * d1;
    sq += d2 * d2;
    // flag lies in host memory and starts at zero; one store per wavefront with a moved site
    const unsigned long long m = __builtin_amdgcn_ballot_w64(sq > sq_skin);
    if (m && (int)(threadIdx.x & 63) == __ffsll((long long)m) - 1) *flag = 1;
}

}  // namespace mappdmd
