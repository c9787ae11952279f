// neighbor.hip -- periodic cell-list neighbour build with image vectors.
//
// Replaces NeighborList::build / verlet::List::build (src/struc absent; the
// contract comes from the call sites src/nnp/nnpce.cpp:282,
// src/nnp/nnp.cpp:343-348, 389-395, 478-482 and README.md:39): for every atom
// i, every periodic image (j, n) with 0 < |r_i - r_j - R n| < rc, in the
// canonical order j ascending then n lexicographic, plus the reverse-slot map
// (i -> j, n) <-> (j -> i, -n) that the atomic-free force reduction needs.
//
// Layout: positions FP64 [N][3]; per structure R^-1 and a bin grid in
// fractional coordinates (nb_a = floor(w_a / rc) bins along lattice direction
// a, w_a the perpendicular width), so that the search box is +-k_a bins with
// k_a = ceil(rc nb_a / w_a); a wavefront per centre atom walks the flattened
// candidate set of its search box (lanes over candidates, not over bins),
// applies the exact FP64 inclusion test in the same operation order as the
// oracle and compacts accepted keys (j << 30 | packed n) through a ballot; the
// staged search meets its candidates in the list's order, the wide one sorts
// every row with a bitonic network.  Integer work; the roofline is
// HBM/latency (positions in, 16 B + 13 B per pair out).
#include <atomic>
#include <chrono>

#include "common.h"
#include "pairvec_dev.h"

#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <tuple>

namespace ann {

constexpr int kMaxImages = 1024;   // bin images searched per atom

// per structure grid: nb[3] bins, search half-width k[3] in bins, bin count
// and offset; the staged search groups sb^3 bins into one block (super-bins:
// nsb[3], offset sboff)
struct CellInfo {
    int nb[3], k[3], nbins, boff;
    int sb, nsb[3], sboff;
    int single;               // every perpendicular width is at least 2 rc: no partner has two images in a row
};

__global__ void k_struc_of(const int* __restrict__ off, int nstruc, int* __restrict__ sof) {
    const int s = blockIdx.x;
    if (s >= nstruc) return;
    for (int i = off[s] + threadIdx.x; i < off[s + 1]; i += blockDim.x) sof[i] = s;
}

// bin of atom i from its fractional coordinates; writes the atom's integer
// shift (the lattice vector that wraps it into the cell)
// A position whose fractional coordinate is not finite (or beyond 1e8 cells)
// is binned as if at the origin and reported through flag bit 16: the build
// stays in bounds and ann_neighbors returns an argument error.
__device__ __forceinline__ int bin_atom(int i, const double* __restrict__ pos, const int* __restrict__ sof,
                                        const CellInfo* __restrict__ ci, const double* __restrict__ rinv,
                                        int* __restrict__ shift, int* __restrict__ flag) {
    const int s = sof[i];
    const CellInfo c = ci[s];
    const double* Ri = rinv + 9 * s;
    int b[3];
    for (int a = 0; a < 3; ++a) {
        double f = Ri[3 * a] * pos[3 * i] + Ri[3 * a + 1] * pos[3 * i + 1] + Ri[3 * a + 2] * pos[3 * i + 2];
        if (!(fabs(f) < 1e8)) {
            f = 0.0;
            if (flag) atomicOr(flag, 16);
        }
        const double fl = floor(f);
        shift[3 * i + a] = (int)fl;
        int bb = (int)floor((f - fl) * c.nb[a]);
        b[a] = bb < 0 ? 0 : (bb >= c.nb[a] ? c.nb[a] - 1 : bb);
    }
    return c.boff + (b[0] * c.nb[1] + b[1]) * c.nb[2] + b[2];
}

__device__ __forceinline__ double4 bin_record(int i, const double* __restrict__ pos, const int* __restrict__ shift) {
    const uint64_t js = ((uint64_t)(uint32_t)i << 32) | pack_img(shift[3 * i], shift[3 * i + 1], shift[3 * i + 2]);
    return make_double4(pos[3 * i], pos[3 * i + 1], pos[3 * i + 2], __longlong_as_double((long long)js));
}

// Binning.  The bin counts are zero on entry: k_fill_bins takes every count
// back to zero.
__global__ void k_bin(int N, const double* __restrict__ pos, const int* __restrict__ sof,
                      const CellInfo* __restrict__ ci, const double* __restrict__ rinv,
                      int* __restrict__ bin_of, int* __restrict__ shift, int* __restrict__ bin_cnt,
                      int* __restrict__ flag) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int g = bin_atom(i, pos, sof, ci, rinv, shift, flag);
    bin_of[i] = g;
    atomicAdd(&bin_cnt[g], 1);
}

// Atoms in bin order: index, and a 32-byte record (x, y, z, atom | shift)
// that the staged search copies with one load per candidate.  The slot is
// taken by counting the bin's count down, so every count is zero again when
// the kernel ends.
__global__ void k_fill_bins(int N, const int* __restrict__ bin_of, const int* __restrict__ bin_start,
                            int* __restrict__ bin_cnt, int* __restrict__ bin_atoms,
                            const double* __restrict__ pos, const int* __restrict__ shift,
                            double4* __restrict__ rec) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const int g = bin_of[i];
    const int p = atomicSub(&bin_cnt[g], 1) - 1;
    const int slot = bin_start[g] + p;
    bin_atoms[slot] = i;
    rec[slot] = bin_record(i, pos, shift);
}

// Binning, bin offsets and bin order of one structure in one block: atoms and bins
// are numbered structure by structure, so a structure's bins start at its first
// atom and no sum over structures is needed.  Counts live in LDS; the slot an atom
// takes from its bin's count is its place in the bin.  Replaces binning, scan and
// fill (three launches) in batches of such structures: E+F of one water box 82.4 ->
// 76.4 us, of 64 boxes 185 -> 173 us, energies of 512 Li/P/S cells 496 -> 464 us
// (with the two-barrier scan of the row offsets).
// T threads take structures of up to 4 T atoms and bins.  Blocks of one wavefront
// where structures are many (kSBinMany on) and small, else blocks of eight: us, eight
// wavefronts / one, 500 structures of 192 atoms 8.3 / 11.1, 1,500 14.1 / 14.1, 3,000
// 21.9 / 19.1; of four atoms 1,500 8.9 / 6.7, 20,000 62 / 17.
constexpr int kSBinThreads = 512;
constexpr int kSBinIt = 4;
// largest structure (atoms, bins) of this path; at the limit, whole builds with three
// launches / one: one structure of 2,000 atoms 39.3 / 38.3, 50 of them 276 / 268
constexpr int kSBinAtoms = kSBinIt * kSBinThreads;
constexpr int kSBinMany = 1536;

template <int T>
__global__ __launch_bounds__(T) void k_bin_struc(
    int nstruc, const int* __restrict__ aoff, const double* __restrict__ pos, const int* __restrict__ sof,
    const CellInfo* __restrict__ ci, const double* __restrict__ rinv, int* __restrict__ bin_of, int* __restrict__ shift,
    int* __restrict__ bin_start, int* __restrict__ bin_atoms, double4* __restrict__ rec, int* __restrict__ flag) {
    __shared__ int cnt[kSBinIt * T];
    __shared__ int wsum[T / kWave];
    const int s = blockIdx.x, t = threadIdx.x, lane = t % kWave, w = t / kWave;
    const int a0 = aoff[s], n = aoff[s + 1] - a0, nb = ci[s].nbins, boff = ci[s].boff;
    for (int q = t; q < kSBinIt * T; q += T) cnt[q] = 0;
    __syncthreads();
    int g[kSBinIt], slot[kSBinIt];
#pragma unroll
    for (int r = 0; r < kSBinIt; ++r) {
        const int a = t + r * T;
        g[r] = -1;
        slot[r] = 0;
        if (a < n) {
            const int b = bin_atom(a0 + a, pos, sof, ci, rinv, shift, flag);
            bin_of[a0 + a] = b;
            g[r] = b - boff;
            slot[r] = atomicAdd(&cnt[g[r]], 1);
        }
    }
    __syncthreads();
    // exclusive scan of the counts, kSBinIt consecutive bins per thread
    int v[kSBinIt], sum = 0;
#pragma unroll
    for (int r = 0; r < kSBinIt; ++r) {
        v[r] = cnt[kSBinIt * t + r];
        sum += v[r];
    }
    int inc = sum;
#pragma unroll
    for (int o = 1; o < kWave; o <<= 1) {
        const int u = __shfl_up(inc, o);
        if (lane >= o) inc += u;
    }
    if (lane == kWave - 1) wsum[w] = inc;
    __syncthreads();
    int run = inc - sum;
#pragma unroll
    for (int k = 0; k < T / kWave; ++k) run += k < w ? wsum[k] : 0;
#pragma unroll
    for (int r = 0; r < kSBinIt; ++r) {
        const int q = kSBinIt * t + r;
        cnt[q] = run;
        if (q < nb) bin_start[boff + q] = a0 + run;
        run += v[r];
    }
    if (s == nstruc - 1 && t == 0) bin_start[boff + nb] = a0 + n;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSBinIt; ++r)
        if (g[r] >= 0) {
            const int i = a0 + t + r * T, at = a0 + cnt[g[r]] + slot[r];
            bin_atoms[at] = i;
            rec[at] = bin_record(i, pos, shift);
        }
}

__device__ __forceinline__ int floordiv(int a, int b) { return a >= 0 ? a / b : -((-a + b - 1) / b); }

// one wavefront (block of 64) per centre atom
__global__ __launch_bounds__(64) void k_search(
    int N, const double* __restrict__ pos, const int* __restrict__ sof, const CellInfo* __restrict__ ci,
    const double* __restrict__ cells, const int* __restrict__ bin_of, const int* __restrict__ shift,
    const int* __restrict__ bin_start, const int* __restrict__ bin_atoms, double rc2,
    uint64_t* __restrict__ keys_out, int* __restrict__ cnt_out, int* __restrict__ flag,
    const int* __restrict__ bin_only) {
    __shared__ int im_bin[kMaxImages];
    __shared__ int im_m[kMaxImages];     // packed m
    __shared__ int im_pre[kMaxImages + 1];
    __shared__ uint64_t keys[kMaxNeigh];
    __shared__ int s_total, s_cnt;
    const int i = blockIdx.x;
    const int lane = threadIdx.x;
    if (i >= N) return;
    if (bin_only && !bin_only[bin_of[i]]) return;     // handled by the staged search
    const int s = sof[i];
    const CellInfo c = ci[s];
    const double* R = cells + 9 * s;
    const int gi = bin_of[i] - c.boff;
    const int b0 = gi / (c.nb[1] * c.nb[2]), b1 = (gi / c.nb[2]) % c.nb[1], b2 = gi % c.nb[2];
    const int e0 = 2 * c.k[0] + 1, e1 = 2 * c.k[1] + 1, e2 = 2 * c.k[2] + 1;
    const int nimg = e0 * e1 * e2;
    if (nimg > kMaxImages) {
        if (lane == 0) { atomicOr(flag, 2); cnt_out[i] = 0; }
        return;
    }
    // bin images of the search box: (wrapped bin, image shift) and candidate counts
    for (int t = lane; t < nimg; t += kWave) {
        const int u0 = b0 - c.k[0] + t / (e1 * e2);
        const int u1 = b1 - c.k[1] + (t / e2) % e1;
        const int u2 = b2 - c.k[2] + t % e2;
        const int m0 = floordiv(u0, c.nb[0]), m1 = floordiv(u1, c.nb[1]), m2 = floordiv(u2, c.nb[2]);
        const int g = c.boff + ((u0 - m0 * c.nb[0]) * c.nb[1] + (u1 - m1 * c.nb[1])) * c.nb[2] + (u2 - m2 * c.nb[2]);
        im_bin[t] = g;
        im_m[t] = (int)pack_img(m0, m1, m2);
        im_pre[t + 1] = bin_start[g + 1] - bin_start[g];
    }
    __syncthreads();
    if (lane == 0) {
        im_pre[0] = 0;
        for (int t = 0; t < nimg; ++t) im_pre[t + 1] += im_pre[t];
        s_total = im_pre[nimg];
        s_cnt = 0;
    }
    __syncthreads();
    const int total = s_total;
    const int si0 = shift[3 * i], si1 = shift[3 * i + 1], si2 = shift[3 * i + 2];
    int count = 0;  // uniform running count
    for (int base = 0; base < total; base += kWave) {
        const int cidx = base + lane;
        bool ok = false;
        uint64_t key = 0;
        if (cidx < total) {
            int lo = 0, hi = nimg;  // largest t with im_pre[t] <= cidx
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (im_pre[mid] <= cidx) lo = mid; else hi = mid;
            }
            const int j = bin_atoms[bin_start[im_bin[lo]] + (cidx - im_pre[lo])];
            int m0, m1, m2;
            unpack_img((uint32_t)im_m[lo], m0, m1, m2);
            const int n0 = si0 - shift[3 * j] + m0;
            const int n1 = si1 - shift[3 * j + 1] + m1;
            const int n2 = si2 - shift[3 * j + 2] + m2;
            double x, y, z, d2;
            pair_vec(pos, i, j, R, n0, n1, n2, x, y, z, d2);
            ok = d2 > 0.0 && d2 < rc2 && !(j == i && n0 == 0 && n1 == 0 && n2 == 0);
            key = ((uint64_t)j << 30) | (uint64_t)pack_img(n0, n1, n2);
        }
        const uint64_t mask = __ballot(ok);
        const int before = __popcll(mask & ((1ull << lane) - 1ull));
        if (ok && count + before < kMaxNeigh) keys[count + before] = key;
        count += __popcll(mask);
    }
    const int n = count < kMaxNeigh ? count : kMaxNeigh;
    if (count > kMaxNeigh && lane == 0) atomicOr(flag, 1);
    int np2 = 1;
    while (np2 < n) np2 <<= 1;
    for (int t = n + lane; t < np2; t += kWave) keys[t] = ~0ull;
    __syncthreads();
    for (int k = 2; k <= np2; k <<= 1) {
        for (int jj = k >> 1; jj > 0; jj >>= 1) {
            for (int t = lane; t < np2; t += kWave) {
                const int p = t ^ jj;
                if (p > t) {
                    const uint64_t a = keys[t], b = keys[p];
                    const bool up = (t & k) == 0;
                    if ((a > b) == up) { keys[t] = b; keys[p] = a; }
                }
            }
            __syncthreads();
        }
    }
    uint64_t* dst = keys_out + (size_t)i * kMaxNeigh;
    for (int t = lane; t < n; t += kWave) dst[t] = keys[t];
    if (lane == 0) { cnt_out[i] = n; atomicMax(flag + 1, count); }
}

// Staged search, one block per bin or super-bin: the candidates of the search
// box (every atom of the (2k+1)^3 bin images with its image offset) are copied to
// LDS with one 32-byte load each, in the list's canonical order (atom index, then
// image), and each wavefront then tests one centre atom against all of them: the
// accepted keys (j << 30 | packed image) leave the ballots in order and go
// straight to the centre's row.  One sort of the box replaces a sort of every row,
// which was two thirds of the instructions per centre.
// The sort is a counting sort by bucket of the atom index (one atom per bucket up
// to kBuckets atoms in the box's index range, else 2^sh neighbouring indices; few
// atoms, which then have many images each, take several buckets per atom), then each
// candidate's rank among its bucket's few members; a block that meets a wide index
// range still sorts, with longer buckets.
// Boxes with more than kStageCap candidates or kStageImages images are flagged: the
// bins of a super-bin are searched one by one by the SPLIT instance (one block per
// marked bin), bins that do not fit either are left to k_search.  Each block writes
// the overflow mark (0 or 1) of each of its centre bins exactly once per build, so
// the marks need no clearing between builds.
// 470 vector instructions per atom on 64 water boxes (counters), issued 39 % of the
// time: latency of the staging's phases, then issue.  Against one sort per row, us:
// 1,048,576 atoms (rc 6.5, super-bins now within the capacity) 5767 -> 1540, 273,561
// atoms 621 -> 256, 87,912 Li/P/S atoms 213 -> 146, 12,288 atoms 39.5 -> 25.2, 192
// atoms 28.6 -> 11.4.
constexpr int kStageCap = 1280;
constexpr int kStageImages = 216;
constexpr int kStageThreads = 512;
constexpr int kBuckets = 1024;
constexpr int kOvfBin = 8, kOvfSuper = 32;                  // build flags: a bin's or a super-bin's box did not fit
constexpr int kStageWaves = kStageThreads / kWave;
constexpr int kStageIt = (kStageCap + kStageThreads - 1) / kStageThreads;
constexpr int kImageBits = 8;
static_assert(kStageImages <= 1 << kImageBits, "image numbers in kImageBits");
static_assert(kBuckets == 2 * kStageThreads, "the bucket scan gives every thread two buckets");

// the image and wrapped index of unwrapped bin u (|u| is a few cells at most)
__device__ __forceinline__ int wrap_bin(int u, int nb, int& m) {
    m = 0;
    while (u < 0) { u += nb; --m; }
    while (u >= nb) { u -= nb; ++m; }
    return u;
}

template <bool SPLIT>
__global__ __launch_bounds__(kStageThreads) void k_search_bins(
    const CellInfo* __restrict__ ci, const double* __restrict__ cells, const int* __restrict__ bin_struc,
    const int* __restrict__ bin_start, const double4* __restrict__ rec, const double* __restrict__ pos, double rc2,
    uint64_t* __restrict__ keys_out, int* __restrict__ cnt_out, int* __restrict__ flag, int* __restrict__ bin_ovf,
    const int* __restrict__ bin_atoms, const int* __restrict__ sof, const int* __restrict__ bin_of, int first) {
    __shared__ int im_first[kStageImages];
    __shared__ int im_m[kStageImages];
    __shared__ int im_pre[kStageImages + 1];
    __shared__ signed char im_cen[kStageImages];            // centre bin of the image, or -1
    __shared__ float4 cf[kStageCap];                        // FP32 image position x_j + R (m - shift_j), sorted
    __shared__ uint64_t ckey[kStageCap];                    // j << 30 | packed (image - shift_j), sorted
    __shared__ int bucket[kBuckets + 1];
    __shared__ uint16_t cen_rank[kStageCap];                // sorted place of each centre
    __shared__ int cen_bin[8], cen_pre[9], wsum[kStageWaves];
    __shared__ int s_total, s_max, s_xmax, s_jmin, s_jmax;
    uint64_t* sk = reinterpret_cast<uint64_t*>(cf);         // (j << 32 | image number) by bucket, until the ranks are known
    int g = first + xcd_block(blockIdx.x, gridDim.x);
    const int t = threadIdx.x, lane = t % kWave, wave = t / kWave;
    if (SPLIT && bin_of) {                                  // one block per atom in bin order: the first of each bin
        const int slot = g;
        g = bin_of[bin_atoms[slot]];
        if (bin_start[g] != slot) return;
    }
    if (SPLIT && (!bin_ovf[g] || bin_start[g] == bin_start[g + 1])) return;
    const int s = SPLIT ? sof[bin_atoms[bin_start[g]]] : bin_struc[g];   // structure of this bin or super-bin
    const CellInfo c = ci[s];
    if (SPLIT && c.sb == 1) return;                         // a single bin's box did not fit: left to k_search
    const double* R = cells + 9 * s;
    const int gi = SPLIT ? g - c.boff : g - c.sboff, sb = SPLIT ? 1 : c.sb;
    const int w1 = SPLIT ? c.nb[1] : c.nsb[1], w2 = SPLIT ? c.nb[2] : c.nsb[2];
    const int B0 = gi / (w1 * w2), B1 = (gi / w2) % w1, B2 = gi % w2;
    const int lo0 = sb * B0, lo1 = sb * B1, lo2 = sb * B2;
    const int n0b = min(sb, c.nb[0] - lo0), n1b = min(sb, c.nb[1] - lo1), n2b = min(sb, c.nb[2] - lo2);
    const int ncb = n0b * n1b * n2b;
    const int e0 = n0b + 2 * c.k[0], e1 = n1b + 2 * c.k[1], e2 = n2b + 2 * c.k[2];
    const int nimg = e0 * e1 * e2;
    for (int q = t; q <= kBuckets; q += kStageThreads) bucket[q] = 0;
    if (wave == kStageWaves - 1) {
        // centre bins of the super-bin and their atom ranges (at most eight)
        int n = 0;
        if (lane < ncb) {
            const int d0 = lane / (n1b * n2b), d1 = (lane / n2b) % n1b, d2 = lane % n2b;
            const int bg = c.boff + ((lo0 + d0) * c.nb[1] + (lo1 + d1)) * c.nb[2] + (lo2 + d2);
            cen_bin[lane] = bg;
            n = bin_start[bg + 1] - bin_start[bg];
        }
        int inc = n;
#pragma unroll
        for (int o = 1; o < 8; o <<= 1) {
            const int u = __shfl_up(inc, o);
            if (lane >= o) inc += u;
        }
        if (lane < ncb) cen_pre[lane + 1] = inc;
        if (lane == 0) {
            cen_pre[0] = 0;
            s_max = 0;
            s_xmax = 0;
            s_jmin = INT32_MAX;
            s_jmax = -1;
        }
    }
    if (nimg > kStageImages) {
        __syncthreads();
        if (t < ncb) bin_ovf[cen_bin[t]] = 1;
        if (t == 0) atomicOr(flag, sb > 1 ? kOvfSuper : kOvfBin);
        return;
    }
    if (t < nimg) {
        const int x0 = t / (e1 * e2), x1 = (t / e2) % e1, x2 = t % e2;
        int m0, m1, m2;
        const int w0 = wrap_bin(lo0 - c.k[0] + x0, c.nb[0], m0), w1 = wrap_bin(lo1 - c.k[1] + x1, c.nb[1], m1),
                  w2 = wrap_bin(lo2 - c.k[2] + x2, c.nb[2], m2);
        const int gg = c.boff + (w0 * c.nb[1] + w1) * c.nb[2] + w2;
        const int f = bin_start[gg];
        im_first[t] = f;
        im_m[t] = (int)pack_img(m0, m1, m2);
        im_pre[t + 1] = bin_start[gg + 1] - f;
        const int d0 = x0 - c.k[0], d1 = x1 - c.k[1], d2 = x2 - c.k[2];
        const bool in = d0 >= 0 && d0 < n0b && d1 >= 0 && d1 < n1b && d2 >= 0 && d2 < n2b;
        im_cen[t] = (signed char)(in ? (d0 * n1b + d1) * n2b + d2 : -1);
    }
    __syncthreads();
    if (t < kWave) {   // inclusive scan of the image counts by the first wavefront
        int carry = 0;
        for (int q0 = 0; q0 < nimg; q0 += kWave) {
            const int q = q0 + lane;
            int v = q < nimg ? im_pre[q + 1] : 0;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const int u = __shfl_up(v, o);
                if (lane >= o) v += u;
            }
            if (q < nimg) im_pre[q + 1] = v + carry;
            carry += __shfl(v, kWave - 1);
        }
        if (lane == 0) { im_pre[0] = 0; s_total = carry; }
    }
    __syncthreads();
    const int total = s_total;
    const int ncen = cen_pre[ncb];
    if (ncen == 0) {                                        // no centres in this super-bin
        if (t < ncb) bin_ovf[cen_bin[t]] = 0;
        return;
    }
    if (total > kStageCap) {
        if (t < ncb) bin_ovf[cen_bin[t]] = 1;
        if (t == 0) atomicOr(flag, sb > 1 ? kOvfSuper : kOvfBin);
        return;
    }
    {
        // every thread resolves all its candidates first, then issues their loads together
        int src[kStageIt], iq[kStageIt];
#pragma unroll
        for (int r = 0; r < kStageIt; ++r) {
            const int q = t + r * kStageThreads;
            src[r] = -1;
            iq[r] = 0;
            if (q < total) {
                int lo = 0, hi = nimg;
                while (hi - lo > 1) {
                    const int mid = (lo + hi) >> 1;
                    if (im_pre[mid] <= q) lo = mid; else hi = mid;
                }
                src[r] = im_first[lo] + (q - im_pre[lo]);
                iq[r] = lo;
            }
        }
        double4 r4[kStageIt];
#pragma unroll
        for (int r = 0; r < kStageIt; ++r)
            if (src[r] >= 0) r4[r] = rec[src[r]];
        float x[kStageIt], y[kStageIt], z[kStageIt], xm = 0.0f;
        uint64_t jd[kStageIt];
        int jlo = INT32_MAX, jhi = -1;
#pragma unroll
        for (int r = 0; r < kStageIt; ++r) {
            if (src[r] < 0) continue;
            const uint64_t js = (uint64_t)__double_as_longlong(r4[r].w);
            int m0, m1, m2, s0, s1, s2;
            unpack_img((uint32_t)im_m[iq[r]], m0, m1, m2);
            unpack_img((uint32_t)(js & 0xffffffffu), s0, s1, s2);
            const double d0 = m0 - s0, d1 = m1 - s1, d2 = m2 - s2;
            x[r] = (float)(r4[r].x + (R[0] * d0 + R[1] * d1 + R[2] * d2));
            y[r] = (float)(r4[r].y + (R[3] * d0 + R[4] * d1 + R[5] * d2));
            z[r] = (float)(r4[r].z + (R[6] * d0 + R[7] * d1 + R[8] * d2));
            xm = fmaxf(xm, fmaxf(fabsf(x[r]), fmaxf(fabsf(y[r]), fabsf(z[r]))));
            jd[r] = (js & 0xffffffff00000000ull) | (uint64_t)pack_img(m0 - s0, m1 - s1, m2 - s2);
            const int j = (int)(js >> 32);
            jlo = min(jlo, j);
            jhi = max(jhi, j);
        }
        int xi = __float_as_int(xm);                        // non-negative floats order as integers
#pragma unroll
        for (int o = kWave / 2; o > 0; o >>= 1) {
            xi = max(xi, __shfl_xor(xi, o));
            jlo = min(jlo, __shfl_xor(jlo, o));
            jhi = max(jhi, __shfl_xor(jhi, o));
        }
        if (lane == 0) {
            atomicMax(&s_xmax, xi);
            atomicMin(&s_jmin, jlo);
            atomicMax(&s_jmax, jhi);
        }
        __syncthreads();
        // buckets of 2^sh atom indices, or 2^ib buckets per index split by image number
        const int jmin = s_jmin, range = s_jmax - jmin;
        int sh = 0, ib = 0;
        while ((range >> sh) >= kBuckets) ++sh;
        while (ib < kImageBits && ((range + 1) << (ib + 1)) <= kBuckets) ++ib;
        int bk[kStageIt], slot[kStageIt];
#pragma unroll
        for (int r = 0; r < kStageIt; ++r) {
            bk[r] = 0;
            slot[r] = 0;
            if (src[r] < 0) continue;
            bk[r] = (((int)(jd[r] >> 32) - jmin) >> sh) << ib | iq[r] >> (kImageBits - ib);
            slot[r] = atomicAdd(&bucket[bk[r]], 1);
        }
        __syncthreads();
        {
            const int v0 = bucket[2 * t], v1 = bucket[2 * t + 1];
            int inc = v0 + v1;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const int u = __shfl_up(inc, o);
                if (lane >= o) inc += u;
            }
            if (lane == kWave - 1) wsum[wave] = inc;
            __syncthreads();
            int before = inc - v0 - v1;
#pragma unroll
            for (int w = 0; w < kStageWaves; ++w) before += w < wave ? wsum[w] : 0;
            bucket[2 * t] = before;
            bucket[2 * t + 1] = before + v0;
            if (t == 0) bucket[kBuckets] = total;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kStageIt; ++r)
            if (src[r] >= 0) sk[bucket[bk[r]] + slot[r]] = (jd[r] & 0xffffffff00000000ull) | (uint64_t)iq[r];
        __syncthreads();
        int rank[kStageIt];
#pragma unroll
        for (int r = 0; r < kStageIt; ++r) {
            rank[r] = 0;
            if (src[r] < 0) continue;
            const int b0 = bucket[bk[r]], b1 = bucket[bk[r] + 1];
            const uint64_t me = (jd[r] & 0xffffffff00000000ull) | (uint64_t)iq[r];
            rank[r] = b0;
            for (int k = b0; k < b1; ++k) rank[r] += sk[k] < me ? 1 : 0;
        }
        __syncthreads();                                    // cf takes the place of sk
#pragma unroll
        for (int r = 0; r < kStageIt; ++r) {
            if (src[r] < 0) continue;
            cf[rank[r]] = make_float4(x[r], y[r], z[r], 0.0f);
            ckey[rank[r]] = ((jd[r] >> 32) << 30) | (jd[r] & 0x3fffffffu);
            const int cb = im_cen[iq[r]];
            // a centre is the zero image of its own bin, where (image - shift) = -shift
            if (cb >= 0) cen_rank[cen_pre[cb] + (t + r * kStageThreads - im_pre[iq[r]])] = (uint16_t)rank[r];
        }
    }
    // the last chunk of 64 is filled up with NaN places: no comparison accepts their
    // distance, also where a non-finite position has made the band infinite
    if (t < kWave && t >= (total & (kWave - 1)) && (total & (kWave - 1)))
        cf[total / kWave * kWave + t] = make_float4(__int_as_float(0x7fc00000), 0.f, 0.f, 0.f);
    __syncthreads();
    // FP32 pre-test.  With u = 2^-24 and every FP32 coordinate within
    // X = max |x| of its FP64 value to u X, the FP32 squared distance of a
    // pair within 1.1 rc is within  e = 2 sqrt3 rc D + 3 D^2 + 4 u rc^2,
    // D = 2 u X + 1.2 u rc, of the FP64 value.  Four times e is the band:
    // below rc^2 - band a pair is in, above rc^2 + band out, and the exact
    // FP64 test of the oracle decides inside the band and near zero.
    const double rc = sqrt(rc2), uu = 5.9604644775390625e-08;
    const double D = 2.0 * uu * (double)__int_as_float(s_xmax) + 1.2 * uu * rc;
    const float band = (float)(4.0 * (3.4641016151377544 * rc * D + 3.0 * D * D + 4.0 * uu * rc2) + 2.0 * uu * rc2);
    const float rc2f = (float)rc2, lo_thr = rc2f - band, hi_thr = rc2f + band;
    int wmax = 0;          // largest neighbour count of this wavefront's centres
    for (int cq = wave; cq < ncen; cq += kStageWaves) {
        const int qc = cen_rank[cq];
        const float4 xi = cf[qc];
        const uint64_t ki = ckey[qc];
        const int i = __builtin_amdgcn_readfirstlane((int)(ki >> 30));
        // the centre's packed image is -shift_i: taking it off a candidate's key
        // leaves (j << 30 | packed n).  Fields wrap one by one: shifts beyond +-511
        // (a structure far from its cell) must not reach the index in the high bits
        const uint32_t si = (uint32_t)__builtin_amdgcn_readfirstlane((int)(ki & 0x3fffffffu));
        uint64_t* dst = keys_out + (size_t)i * kMaxNeigh;
        int count = 0;
        for (int base = 0; base < total; base += kWave) {
            const int q = base + lane;
            const float4 xq = cf[q];
            const float dx = xi.x - xq.x, dy = xi.y - xq.y, dz = xi.z - xq.z;
            const float d2f = fmaf(dz, dz, fmaf(dy, dy, dx * dx));
            const bool near = d2f <= hi_thr && q != qc;
            bool ok = near && d2f < lo_thr && d2f > band;
            const uint64_t mnear = __ballot(near);
            if (mnear == 0) continue;
            const uint64_t kq = near ? ckey[q] : 0ull;
            const uint64_t key = (kq & 0xffffffff00000000ull) | img_minus((uint32_t)kq, si);
            uint64_t mask = __ballot(ok);
            if (mask != mnear) {
                if (near && !ok) {
                    int n0, n1, n2;
                    unpack_img((uint32_t)(key & 0x3fffffffu), n0, n1, n2);
                    double px, py, pz, d2;
                    pair_vec(pos, i, (int)(key >> 30), R, n0, n1, n2, px, py, pz, d2);
                    ok = d2 > 0.0 && d2 < rc2;
                }
                mask = __ballot(ok);
            }
            const int at = count + __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
            if (ok && at < kMaxNeigh) dst[at] = key;
            count += __popcll(mask);
        }
        if (count > kMaxNeigh && lane == 0) atomicOr(flag, 1);
        if (lane == 0) cnt_out[i] = min(count, kMaxNeigh);
        wmax = max(wmax, count);
    }
    // one global atomic per block (a contended atomic per atom serialises the kernel)
    if (lane == 0) atomicMax(&s_max, wmax);
    __syncthreads();
    if (t == 0) atomicMax(flag + 1, s_max);
    if (t < ncb) bin_ovf[cen_bin[t]] = 0;
}

// CSR fill: index, packed image, neighbour species and FP32 pair geometry.
// TAB: also the row's rank table, one 8-byte word per 32 atoms of the structure:
// which of them the row holds (low half) and how many entries come before them
// (high half), from which k_rev_table reads any partner's place in the row.
// Against a binary search of the partner's row per pair (k_rev), us, tables and
// reverse slots together: 273,561 atoms 286 + 406 -> 289 + 179, 12,288 atoms 14.1 +
// 19.7 -> 16.4 + 9.3, 87,912 Li/P/S atoms (several images per partner) 44 + 53 ->
// 50 + 44, 2,048 atoms 10.6 + 15.8 -> 10.7 + 7.3.
constexpr int kTabAtoms = 2048;              // largest structure with rank tables
constexpr int kTabWords = kTabAtoms / 32;
constexpr int kCompactThreads = 128;

template <bool TAB>
__global__ __launch_bounds__(kCompactThreads) void k_compact(
    int N, const double* __restrict__ pos, const int* __restrict__ sof, const double* __restrict__ cells,
    const int* __restrict__ species, const uint64_t* __restrict__ keys, const int* __restrict__ off,
    int* __restrict__ idx, uint32_t* __restrict__ img, int* __restrict__ rev, float4* __restrict__ geo,
    uint8_t* __restrict__ nsp, const int* __restrict__ order, int cap, const int* __restrict__ aoff, int tabw,
    uint64_t* __restrict__ tab) {
    __shared__ unsigned mask[TAB ? kTabWords : 1];
    __shared__ int ent[TAB ? kTabWords : 1];
    // centres in bin order: the blocks of one XCD cover one region of space,
    // so the partners they read stay in that XCD's L2
    const int b = xcd_block(blockIdx.x, gridDim.x);
    if (b >= N || off[N] > cap) return;     // a list that does not fit is compacted again after growing
    const int i = order[b];
    const int o = off[i], n = off[i + 1] - o, s = sof[i];
    const double* R = cells + 9 * s;
    const int a0 = TAB ? aoff[s] : 0;
    if (TAB) {
        if (threadIdx.x < kTabWords) {
            mask[threadIdx.x] = 0;
            ent[threadIdx.x] = 0;
        }
        __syncthreads();
    }
    for (int t = threadIdx.x; t < n; t += kCompactThreads) {
        const uint64_t key = keys[(size_t)i * kMaxNeigh + t];
        const int j = (int)(key >> 30);
        const uint32_t p = (uint32_t)(key & 0x3fffffffu);
        if (TAB) {
            atomicOr(&mask[(j - a0) >> 5], 1u << ((j - a0) & 31));
            atomicAdd(&ent[(j - a0) >> 5], 1);
        }
        int n0, n1, n2;
        unpack_img(p, n0, n1, n2);
        double x, y, z, d2;
        pair_vec(pos, i, j, R, n0, n1, n2, x, y, z, d2);
        idx[o + t] = j;
        img[o + t] = p;
        if (!TAB) rev[o + t] = o + t;
        geo[o + t] = make_float4((float)x, (float)y, (float)z, (float)sqrt(d2));
        nsp[o + t] = (uint8_t)species[j];
    }
    if (TAB) {
        __syncthreads();
        const int w = threadIdx.x;
        if (w < kWave) {
            const int v = ent[w];            // kTabWords is the wavefront's width
            int inc = v;
#pragma unroll
            for (int q = 1; q < kWave; q <<= 1) {
                const int u = __shfl_up(inc, q);
                if (w >= q) inc += u;
            }
            if (w < tabw) tab[(size_t)i * tabw + w] = ((uint64_t)(uint32_t)(inc - v) << 32) | mask[w];
        }
    }
}
static_assert(kTabWords == kWave, "one lane per word of the rank table");

// Reverse slots from the rank tables: the place of centre i in partner j's row is
// the entries before i's word plus the set bits below i.  Where a partner can
// appear with several images the bits undercount, and the row is walked on from
// there to the entry (j -> i, -n).
__global__ __launch_bounds__(256) void k_rev_table(int N, const int* __restrict__ idx, const uint32_t* __restrict__ img,
                                                   const int* __restrict__ off, int* __restrict__ rev,
                                                   int* __restrict__ flag, int cap, const int* __restrict__ sof,
                                                   const int* __restrict__ aoff, const CellInfo* __restrict__ ci, int tabw,
                                                   const uint64_t* __restrict__ tab) {
    const int i = xcd_block(blockIdx.x, gridDim.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (i >= N || off[N] > cap) return;
    const int o = off[i], n = off[i + 1] - o, s = sof[i], r = i - aoff[s];
    const int w = r >> 5;
    const unsigned below = (1u << (r & 31)) - 1u;
    const bool single = ci[s].single != 0;
    for (int t = threadIdx.x % kWave; t < n; t += kWave) {
        const int j = idx[o + t];
        const uint64_t e = tab[(size_t)j * tabw + w];
        const int oj = off[j];
        int at = oj + (int)(e >> 32) + __popc((unsigned)e & below);
        if (!single) {
            const int end = off[j + 1];
            int n0, n1, n2;
            unpack_img(img[o + t], n0, n1, n2);
            const uint32_t want = pack_img(-n0, -n1, -n2);
            while (at < end && (idx[at] < i || (idx[at] == i && img[at] < want))) ++at;
            if (at >= end || idx[at] != i || img[at] != want) {   // impossible for the symmetric FP64 test
                atomicOr(flag, 4);
                at = o + t;
            }
        } else if (!((unsigned)e >> (r & 31) & 1u)) {
            atomicOr(flag, 4);
            at = o + t;
        }
        rev[o + t] = at;
    }
}

// Reverse slots.  rev is an involution, so each pair is resolved once, from its
// upper slot (partner index above the centre's, or the same atom with the
// larger packed image): a binary search in the partner's CSR run, which is
// sorted by (partner index, packed image) like the keys, on the 4-byte partner
// indices, then a scan over the few images of the same partner; the result
// is written to both slots.  k_compact has set every slot to itself before,
// so a slot without a partner (an asymmetric list, impossible for the
// symmetric FP64 test) stays in range; the missing upper match is flagged.
__global__ void k_rev(int N, const int* __restrict__ idx, const uint32_t* __restrict__ img,
                      const int* __restrict__ off, int* __restrict__ rev, int* __restrict__ flag,
                      const int* __restrict__ order, int cap) {
    // one wavefront per centre, the centres of a workgroup consecutive in bin
    // order (see k_compact): their partner rows overlap, so the searches of a
    // workgroup share the lines they bring into its CU's cache
    const int b = xcd_block(blockIdx.x, gridDim.x) * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (b >= N || off[N] > cap) return;
    const int i = order[b];
    const int o = off[i], n = off[i + 1] - o;
    for (int t = threadIdx.x % kWave; t < n; t += kWave) {
        const int j = idx[o + t];
        const uint32_t p = img[o + t];
        int n0, n1, n2;
        unpack_img(p, n0, n1, n2);
        const uint32_t want = pack_img(-n0, -n1, -n2);
        if (j < i || (j == i && p < want)) continue;       // lower slot: written by its partner
        const int b0 = off[j], e = off[j + 1];
        int lo = b0, hi = e;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (idx[mid] < i) lo = mid + 1; else hi = mid;
        }
        while (lo < e && idx[lo] == i && img[lo] < want) ++lo;
        if (lo < e && idx[lo] == i && img[lo] == want) {
            rev[o + t] = lo;
            rev[lo] = o + t;
        } else {
            atomicOr(flag, 4);
        }
    }
}

static void inv3(const double* R, double* Ri) {
    const double a = R[0], b = R[1], c = R[2], d = R[3], e = R[4], f = R[5], g = R[6], h = R[7], i = R[8];
    const double A = e * i - f * h, B = -(d * i - f * g), C = d * h - e * g;
    const double id = 1.0 / (a * A + b * B + c * C);
    Ri[0] = A * id; Ri[1] = -(b * i - c * h) * id; Ri[2] = (b * f - c * e) * id;
    Ri[3] = B * id; Ri[4] = (a * i - c * g) * id;  Ri[5] = -(a * f - c * d) * id;
    Ri[6] = C * id; Ri[7] = -(a * h - b * g) * id; Ri[8] = (a * e - b * d) * id;
}

template <typename T>
static hipError_t grow(T*& p, int64_t& cap, int64_t want) {
    if (want <= cap && p) return hipSuccess;
    if (p) { hipError_t e = hipFree(p); if (e != hipSuccess) return e; p = nullptr; }
    int64_t c = std::max<int64_t>(want, 1);
    c += c / 4;
    hipError_t e = hipMalloc((void**)&p, sizeof(T) * c);
    if (e == hipSuccess) cap = c;
    return e;
}

// Small exclusive scans in one workgroup: every wavefront takes one contiguous
// range with all of its values in registers (IT vectors of four per lane), the
// wavefront totals meet in LDS, and each wavefront scans its own range: two
// barriers, and the host-visible words written by the same kernel.
constexpr int kScanThreads = 1024;
constexpr int kScanMax = 1 << 16;

__device__ __forceinline__ void store_host(int* rb, int q, int v) {
    __hip_atomic_store(rb + q, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Exclusive scan of n values by one workgroup of kScanThreads threads; returns
// the sum of all n values to every thread.  n <= IT * 4 * kScanThreads; in and out
// are 16-byte aligned.
template <int IT>
__device__ int scan_block(const int* __restrict__ in, int* __restrict__ out, int n) {
    constexpr int NWV = kScanThreads / kWave;
    __shared__ int wsum[NWV];
    const int lane = threadIdx.x % kWave, w = threadIdx.x / kWave;
    const int first = w * IT * 4 * kWave + 4 * lane;        // element of vector k: first + 256 k
    int4 v[IT];
    int sum = 0;
#pragma unroll
    for (int k = 0; k < IT; ++k) {
        const int e = first + 4 * kWave * k;
        if (e + 3 < n) v[k] = *reinterpret_cast<const int4*>(in + e);
        else v[k] = make_int4(e < n ? in[e] : 0, e + 1 < n ? in[e + 1] : 0, e + 2 < n ? in[e + 2] : 0, 0);
        sum += v[k].x + v[k].y + v[k].z + v[k].w;
    }
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    if (lane == 0) wsum[w] = sum;
    __syncthreads();
    int run = 0, all = 0;
#pragma unroll
    for (int k = 0; k < NWV; ++k) {
        run += k < w ? wsum[k] : 0;
        all += wsum[k];
    }
#pragma unroll
    for (int k = 0; k < IT; ++k) {
        const int e = first + 4 * kWave * k;
        const int own = v[k].x + v[k].y + v[k].z + v[k].w;
        int inc = own;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int u = __shfl_up(inc, o);
            if (lane >= o) inc += u;
        }
        const int4 x = make_int4(run + inc - own, run + inc - own + v[k].x, run + inc - own + v[k].x + v[k].y,
                                 run + inc - v[k].w);
        if (e + 3 < n) *reinterpret_cast<int4*>(out + e) = x;
        else {
            if (e < n) out[e] = x.x;
            if (e + 1 < n) out[e + 1] = x.y;
            if (e + 2 < n) out[e + 2] = x.z;
        }
        run += __shfl(inc, kWave - 1);
    }
    return all;
}

// One-workgroup scan; with rb, the flags, the last element's exclusive prefix
// and then seq go to the pinned host words, and the first nclear flags are
// cleared once read (the next build starts from zero without a clear launch).
template <int IT>
__global__ __launch_bounds__(kScanThreads) void k_scan_small(const int* __restrict__ in, int* __restrict__ out, int n,
                                                             int* __restrict__ flags, int nflags, int nclear, int* rb,
                                                             int seq) {
    const int tot = scan_block<IT>(in, out, n);
    if (rb && threadIdx.x == kScanThreads - 1) {
        for (int q = 0; q < nflags; ++q) store_host(rb, q, flags[q]);
        for (int q = 0; q < nclear; ++q) flags[q] = 0;
        store_host(rb, nflags, n > 0 ? tot - in[n - 1] : 0);
        __threadfence_system();
        store_host(rb, nflags + 1, seq);            // the words above are complete
    }
}

// flags and one more word (the total) to the host words, then the marker
__global__ void k_readback_build(int* flags, int nflags, const int* total, int* rb, int seq, int nclear) {
    const int t = threadIdx.x;
    if (t < nflags) store_host(rb, t, flags[t]);
    if (t == nflags) store_host(rb, t, *total);
    if (t < nclear) flags[t] = 0;                   // cleared once read
    __threadfence_system();
    __syncthreads();
    if (t == 0) store_host(rb, nflags + 1, seq);
}

__global__ void k_readback(int* src, int n, int* rb, int seq, int nclear) {
    const int t = threadIdx.x;
    if (t < n) store_host(rb, t, src[t]);
    if (t < nclear) src[t] = 0;                     // cleared once read
    __threadfence_system();
    __syncthreads();
    if (seq && t == 0) {
        store_host(rb, n, seq);
        __threadfence_system();
    }
}

hipError_t readback(const int* src, int n, int* rb, hipStream_t st) {
    k_readback<<<1, 64, 0, st>>>(const_cast<int*>(src), n, rb, 0, 0);
    return hipGetLastError();
}

hipError_t exclusive_scan(const int* in, int* out, int n, hipStream_t st, int* flags, int nflags, int* rb, int seq,
                          int nclear) {
    if (n <= kScanMax) {
        const int it = (n + 4 * kScanThreads - 1) / (4 * kScanThreads);   // vectors of four per thread
        (it <= 1 ? k_scan_small<1> : it <= 2 ? k_scan_small<2> : it <= 4 ? k_scan_small<4> : it <= 8 ? k_scan_small<8>
                                                                             : k_scan_small<16>)
            <<<1, kScanThreads, 0, st>>>(in, out, n, flags, nflags, nclear, rb, seq);
        return hipGetLastError();
    }
    size_t bytes = 0;
    hipError_t e = hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, in, out, n, st);
    if (e != hipSuccess) return e;
    static thread_local void* tmp = nullptr;
    static thread_local size_t tmp_cap = 0;
    if (bytes > tmp_cap) {
        if (tmp) hipFree(tmp);
        e = hipMalloc(&tmp, bytes);
        if (e != hipSuccess) { tmp = nullptr; tmp_cap = 0; return e; }
        tmp_cap = bytes;
    }
    if ((e = hipcub::DeviceScan::ExclusiveSum(tmp, bytes, in, out, n, st)) != hipSuccess) return e;
    if (rb) {
        k_readback_build<<<1, kWave, 0, st>>>(flags, nflags, out + n - 1, rb, seq, nclear);
        e = hipGetLastError();
    }
    return e;
}

#define HIPCHK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) return e_; } while (0)

// Bin grid of every structure for cutoff rc: computed on the host from the
// cells once per batch and cutoff (the cells are read at the first build after
// ann_set_batch), then kept on the device.
static hipError_t grid_setup(ann_ctx* ctx, double rc) {
    if (ctx->grid_valid && ctx->grid_rc == rc) return hipSuccess;
    const int S = ctx->nstruc;
    hipStream_t st = ctx->stream;
    // the cells: the host copy given with the batch, else read from the device
    std::vector<double> cells;
    if (ctx->h_cells_valid) {
        cells = ctx->h_cells;
    } else {
        cells.resize(9 * (size_t)S);
        HIPCHK(hipMemcpyAsync(cells.data(), ctx->d_cells, sizeof(double) * 9 * S, hipMemcpyDeviceToHost, st));
        HIPCHK(hipStreamSynchronize(st));
    }
    std::vector<CellInfo> info(S);
    std::vector<double> rinv(9 * (size_t)S);
    std::vector<int> bin_struc;
    int nbins = 0;
    for (int s = 0; s < S; ++s) {
        inv3(&cells[9 * s], &rinv[9 * s]);
        CellInfo& c = info[s];
        for (int a = 0; a < 3; ++a) {
            // bins at least rc/2 wide, so that the search box is +-2 bins
            const double* r = &rinv[9 * s + 3 * a];
            const double w = 1.0 / std::sqrt(r[0] * r[0] + r[1] * r[1] + r[2] * r[2]);
            c.nb[a] = std::max(1, (int)std::floor(2.0 * w / rc * (1.0 - 1e-12)));
            c.nb[a] = std::min(c.nb[a], 256);
            c.k[a] = (int)std::ceil(rc * c.nb[a] / w * (1.0 + 1e-12));
            c.single = (a == 0 || c.single) && w >= 2.0 * rc * (1.0 + 1e-9);
        }
        c.nbins = c.nb[0] * c.nb[1] * c.nb[2];
        c.boff = nbins;
        nbins += c.nbins;
    }
    // 2x2x2 bins per staged block share one box of candidates; with few bins one
    // bin per block spreads the centres over the chip instead (192 atoms in 64 bins:
    // 12.0 us against 21.8 in super-bins; 2,048 bins and more lose by it, 12,288
    // atoms 64.5 against 29.2)
    const bool few = nbins <= 2 * ctx->num_cu;
    // rank tables pay in structures of 64 atoms or more (below, rows are short and the
    // table is one more thing to write) whose rows rarely hold several images of a
    // partner (the images that the table's bits leave out are walked one by one): the
    // cutoff sphere at most 0.85 of the cell.  Fill and reverse slots together, us,
    // search / tables: 20,000 structures of 4 atoms 69 / 81, 4,096 of 16 65 / 71, 1,024
    // sparse ones of 64 67.5 / 67.5, 512 of 200 198 / 121; dense cells by sphere / cell:
    // 2.9 150 / 371, 1.4 136 / 184, 0.93 107 / 113, 0.80 125 / 115, 0.70 144 / 134
    double tab_pairs = 0.0, all_pairs = 0.0;                // in proportion to the pairs expected
    for (int s = 0; s < S; ++s) {
        CellInfo& c = info[s];
        const double* r = &cells[9 * s];
        const double vol = std::fabs(r[0] * (r[4] * r[8] - r[5] * r[7]) - r[1] * (r[3] * r[8] - r[5] * r[6]) +
                                     r[2] * (r[3] * r[7] - r[4] * r[6]));
        const int n = ctx->atom_off[s + 1] - ctx->atom_off[s];
        all_pairs += (double)n * n / vol;
        if (n >= 64 && 4.18879 * rc * rc * rc <= 0.85 * vol) tab_pairs += (double)n * n / vol;
        // when the enlarged search box still fits
        const double per_bin = (double)n / c.nbins;
        const double box2 = (double)(std::min(2, c.nb[0]) + 2 * c.k[0]) * (std::min(2, c.nb[1]) + 2 * c.k[1]) *
                            (std::min(2, c.nb[2]) + 2 * c.k[2]);
        c.sb = (ctx->tune_sb != 1 && !few && box2 * per_bin <= 0.8 * kStageCap && box2 <= kStageImages) ? 2 : 1;
        for (int a = 0; a < 3; ++a) c.nsb[a] = (c.nb[a] + c.sb - 1) / c.sb;
        const int nsbins = c.nsb[0] * c.nsb[1] * c.nsb[2];
        c.sboff = (int)bin_struc.size();
        bin_struc.insert(bin_struc.end(), nsbins, s);       // structure of each super-bin
    }
    if (S > ctx->struc_cap || !ctx->d_cellinfo) {
        if (ctx->d_cellinfo) { hipFree(ctx->d_cellinfo); hipFree(ctx->d_cellmat); }
        HIPCHK(hipMalloc(&ctx->d_cellinfo, sizeof(CellInfo) * S));
        HIPCHK(hipMalloc(&ctx->d_cellmat, sizeof(double) * 9 * S));
        ctx->struc_cap = S;
    }
    if (nbins + 1 > ctx->bin_cap) {
        if (ctx->d_bin_cnt) { hipFree(ctx->d_bin_cnt); hipFree(ctx->d_bin_start); hipFree(ctx->d_bin_struc); }
        // counts and overflow marks share one allocation; the counts are
        // cleared before the first build and return to zero by the end of
        // every build
        HIPCHK(hipMalloc(&ctx->d_bin_cnt, sizeof(int) * 3 * (nbins + 1)));
        HIPCHK(hipMalloc(&ctx->d_bin_start, sizeof(int) * (nbins + 1)));
        HIPCHK(hipMalloc(&ctx->d_bin_struc, sizeof(int) * (nbins + 1)));
        ctx->bin_cap = nbins + 1;
        ctx->nb_dirty = true;
    }
    ctx->d_bin_ovf = ctx->d_bin_cnt + 2 * (size_t)ctx->bin_cap;
    HIPCHK(staged_upload(ctx, kStCellInfo, ctx->d_cellinfo, info.data(), sizeof(CellInfo) * S));
    HIPCHK(staged_upload(ctx, kStRinv, ctx->d_cellmat, rinv.data(), sizeof(double) * 9 * S));
    HIPCHK(staged_upload(ctx, kStBinStruc, ctx->d_bin_struc, bin_struc.data(), sizeof(int) * bin_struc.size()));
    ctx->grid_valid = true;
    ctx->grid_rc = rc;
    ctx->grid_nbins = nbins;
    ctx->grid_tab = 2.0 * tab_pairs >= all_pairs;           // most pairs are in such structures
    ctx->grid_maxbins = 0;
    for (const CellInfo& c : info) ctx->grid_maxbins = std::max(ctx->grid_maxbins, c.nbins);
    ctx->grid_nsb = (int)bin_struc.size();
    return hipSuccess;
}

// Wait until the pinned word slot holds seq (written last by the readback of a
// kernel on the stream), polling instead of synchronising the stream so that
// work queued behind that kernel keeps the device busy meanwhile.
static hipError_t wait_marker(ann_ctx* ctx, int slot, int seq) {
    volatile const int* w = ctx->h_rb + slot;
    // The stream is queried only when the marker is late (2 ms, then every
    // millisecond): queried every 256 polls, the queries while the build's
    // kernels ran left a 5.6 us idle gap before the next kernel on the stream
    // (1.0 us without them).
    auto next = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
    for (long it = 0;; ++it) {
        if (*w == seq) break;
        if ((it & 255) == 255 && std::chrono::steady_clock::now() >= next) {
            const hipError_t e = hipStreamQuery(ctx->stream);
            if (e == hipSuccess) {                   // stream drained: the marker must be there
                if (*w == seq) break;
                return hipErrorUnknown;
            }
            if (e != hipErrorNotReady) return e;
            next = std::chrono::steady_clock::now() + std::chrono::milliseconds(1);
        }
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return hipSuccess;
}

static void launch_compact(ann_ctx* ctx, int cap) {
    const int N = ctx->natoms;
    hipStream_t st = ctx->stream;
    NList& nl = ctx->nl;
    // rank tables where every structure fits one (8 bytes per 32 atoms and row) and
    // they pay (grid_setup); else the partners' rows are searched
    const bool tab = ctx->tab_words > 0;
    {
        Launch L(ctx, "nb_compact");
        (tab ? k_compact<true> : k_compact<false>)<<<N, kCompactThreads, 0, st>>>(
            N, ctx->d_pos, ctx->d_struc_of, ctx->d_cells, ctx->d_species, ctx->d_keys, nl.off, nl.idx, nl.img, nl.rev,
            nl.geo, nl.nsp, ctx->d_bin_atoms, cap, ctx->d_atom_off, ctx->tab_words, ctx->d_tab);
    }
    // a missing reverse slot (impossible for the symmetric FP64 test) is
    // reported by the next synchronising call (ann_nlist_size, next build)
    Launch L(ctx, "nb_rev");
    constexpr int kRevRows = 4;                 // centres (wavefronts) per workgroup
    if (tab)
        k_rev_table<<<(N + kRevRows - 1) / kRevRows, kRevRows * kWave, 0, st>>>(
            N, nl.idx, nl.img, nl.off, nl.rev, ctx->d_flag + 2, cap, ctx->d_struc_of, ctx->d_atom_off,
            reinterpret_cast<const CellInfo*>(ctx->d_cellinfo), ctx->tab_words, ctx->d_tab);
    else
        k_rev<<<(N + kRevRows - 1) / kRevRows, kRevRows * kWave, 0, st>>>(N, nl.idx, nl.img, nl.off, nl.rev,
                                                                          ctx->d_flag + 2, ctx->d_bin_atoms, cap);
}

hipError_t neighbors_build(ann_ctx* ctx, double rc) {
    const int N = ctx->natoms;
    hipStream_t st = ctx->stream;
    HIPCHK(grid_setup(ctx, rc));
    const int nbins = ctx->grid_nbins;
    int64_t kc = ctx->keys_cap;
    HIPCHK(grow(ctx->d_keys, kc, (int64_t)N * kMaxNeigh));
    ctx->keys_cap = kc;
    ctx->tab_words = 0;
    int most = 0;                               // atoms of the largest structure
    for (int s = 0; s < ctx->nstruc; ++s) most = std::max(most, ctx->atom_off[s + 1] - ctx->atom_off[s]);
    if (most <= kTabAtoms && ctx->grid_tab) {
        ctx->tab_words = (most + 31) / 32;
        HIPCHK(grow(ctx->d_tab, ctx->tab_cap, (int64_t)N * ctx->tab_words));
    }
    int64_t rcap = ctx->binrec_cap;
    HIPCHK(grow(ctx->d_binrec, rcap, (int64_t)N));
    ctx->binrec_cap = rcap;
    const CellInfo* dci = reinterpret_cast<const CellInfo*>(ctx->d_cellinfo);
    // The bin counts and flag[0..1] are zero at the start of a build without a
    // clear launch: the fill counts every bin back down and the readback scan
    // clears the flags it reports (flag[2], the reverse-slot error, stays set
    // until reported).  New bin arrays, or a build that stopped part-way
    // (nb_dirty), are cleared here first.
    if (ctx->nb_dirty) {
        HIPCHK(hipMemsetAsync(ctx->d_bin_cnt, 0, sizeof(int) * (size_t)ctx->bin_cap, st));
        HIPCHK(hipMemsetAsync(ctx->d_flag, 0, sizeof(int) * 2, st));
    }
    ctx->nb_dirty = true;
    {
        if (most <= kSBinAtoms && ctx->grid_maxbins <= kSBinAtoms) {
            // one launch instead of three where every structure fits a block
            Launch L(ctx, "nb_bin");
            const bool wave = ctx->nstruc >= kSBinMany && std::max(most, ctx->grid_maxbins) <= kSBinIt * kWave;
            (wave ? k_bin_struc<kWave> : k_bin_struc<kSBinThreads>)<<<ctx->nstruc, wave ? kWave : kSBinThreads, 0, st>>>(
                ctx->nstruc, ctx->d_atom_off, ctx->d_pos, ctx->d_struc_of, dci, ctx->d_cellmat, ctx->d_bin_of, ctx->d_shift,
                ctx->d_bin_start, ctx->d_bin_atoms, ctx->d_binrec, ctx->d_flag);
        } else {
        {
            Launch L(ctx, "nb_bin");
            k_bin<<<(N + 255) / 256, 256, 0, st>>>(N, ctx->d_pos, ctx->d_struc_of, dci, ctx->d_cellmat,
                                                  ctx->d_bin_of, ctx->d_shift, ctx->d_bin_cnt, ctx->d_flag);
        }
        HIPCHK(hipGetLastError());
        HIPCHK(exclusive_scan(ctx->d_bin_cnt, ctx->d_bin_start, nbins + 1, st));
        k_fill_bins<<<(N + 255) / 256, 256, 0, st>>>(N, ctx->d_bin_of, ctx->d_bin_start, ctx->d_bin_cnt,
                                                    ctx->d_bin_atoms, ctx->d_pos, ctx->d_shift, ctx->d_binrec);
        }
        HIPCHK(hipGetLastError());
    }
    {
        Launch L(ctx, "nb_search");
        k_search_bins<false><<<ctx->grid_nsb, kStageThreads, 0, st>>>(dci, ctx->d_cells, ctx->d_bin_struc, ctx->d_bin_start,
                                                      ctx->d_binrec, ctx->d_pos, rc * rc, ctx->d_keys, ctx->d_cnt,
                                                      ctx->d_flag, ctx->d_bin_ovf, nullptr, nullptr, nullptr, 0);
    }
    // Super-bins are chosen on a structure's mean density; where its dense part (a
    // slab, a droplet) does not fit them, their bins are searched one by one.  A
    // context that met this in its last build launches that pass at once instead of
    // after the wait.  Whole builds, us, against leaving such bins to k_search: 4,212
    // atoms 153 -> 86, 33,696 atoms 504 -> 218, 57,132 atoms 1746 -> 632 (a loop over
    // the bins inside the block that found them costs every search registers: 1,048,576
    // uniform atoms 1.57 -> 2.66 ms).
    auto search_split = [&]() {
        Launch L(ctx, "nb_search_split");
        // a block per bin, or per atom where most bins are empty; a launch holds 2^32 threads
        const bool atoms = N < nbins;
        const int blocks = atoms ? N : nbins, most_blocks = 1 << 22;
        for (int b = 0; b < blocks; b += most_blocks)
            k_search_bins<true><<<std::min(blocks - b, most_blocks), kStageThreads, 0, st>>>(
                dci, ctx->d_cells, ctx->d_bin_struc, ctx->d_bin_start, ctx->d_binrec, ctx->d_pos, rc * rc, ctx->d_keys,
                ctx->d_cnt, ctx->d_flag, ctx->d_bin_ovf, ctx->d_bin_atoms, ctx->d_struc_of,
                atoms ? ctx->d_bin_of : nullptr, b);
    };
    const bool ahead = ctx->nb_split;
    if (ahead) search_split();
    HIPCHK(hipGetLastError());
    NList& nl = ctx->nl;
    // Offsets, then flags, pair count and a completion marker to pinned host
    // words -- the build's one wait.  While the host waits, the compaction runs
    // speculatively into the current list arrays; it does nothing if the list
    // does not fit, and is repeated after growing them.
    int seq = ++ctx->rb_seq;
    HIPCHK(exclusive_scan(ctx->d_cnt, ctx->nl.off, N + 1, st, ctx->d_flag, 4, ctx->d_rb, seq, 2));
    ctx->nb_dirty = false;
    const int spec_cap = (int)std::min<int64_t>(nl.cap, INT32_MAX);
    if (spec_cap > 0) launch_compact(ctx, spec_cap);
    HIPCHK(hipGetLastError());
    HIPCHK(wait_marker(ctx, 5, seq));
    volatile const int* rb = ctx->h_rb;
    int flags[4] = {rb[0], rb[1], rb[2], rb[3]};
    int total = rb[4];
    if (flags[2]) {
        // reported once: the flag of the list that lacked a reverse slot is cleared
        HIPCHK(hipMemsetAsync(ctx->d_flag + 2, 0, sizeof(int), st));
        ctx->nb_status = ANN_ERR_HIP;
        set_error("the previous neighbour list was not symmetric (reverse slot missing)");
        return hipErrorInvalidValue;
    }
    ctx->nb_split = flags[0] & kOvfSuper;
    const bool behind = ctx->nb_split && !ahead;
    // Rows that the search left out or cut short have no reverse slots: what the
    // compaction beside this wait found missing there is no fault of a list
    auto forget_rev = [&]() {
        return spec_cap > 0 ? hipMemsetAsync(ctx->d_flag + 2, 0, sizeof(int), st) : hipSuccess;
    };
    if (behind || (flags[0] & ~kOvfSuper)) HIPCHK(forget_rev());
    if (behind || (flags[0] & kOvfBin)) {
        ctx->nb_dirty = true;
        if (behind) search_split();
        // bins with a search box too large to stage: one wavefront per centre atom
        {
            Launch L(ctx, "nb_search_wide");
            k_search<<<N, 64, 0, st>>>(N, ctx->d_pos, ctx->d_struc_of, dci, ctx->d_cells, ctx->d_bin_of,
                                       ctx->d_shift, ctx->d_bin_start, ctx->d_bin_atoms, rc * rc, ctx->d_keys,
                                       ctx->d_cnt, ctx->d_flag, ctx->d_bin_ovf);
        }
        HIPCHK(hipGetLastError());
        seq = ++ctx->rb_seq;
        HIPCHK(exclusive_scan(ctx->d_cnt, ctx->nl.off, N + 1, st, ctx->d_flag, 4, ctx->d_rb, seq, 2));
        ctx->nb_dirty = false;
        if (spec_cap > 0) launch_compact(ctx, spec_cap);
        HIPCHK(hipGetLastError());
        HIPCHK(wait_marker(ctx, 5, seq));
        // the first pass's flags were cleared when read: merge both passes
        flags[0] |= rb[0];
        flags[1] = std::max(flags[1], (int)rb[1]);
        total = rb[4];
        if (flags[0] & ~(kOvfBin | kOvfSuper)) HIPCHK(forget_rev());
    }
    if (flags[0] & 16) {
        ctx->nb_status = ANN_ERR_ARG;
        set_error("an atom position is not finite (or lies beyond 1e8 cells)");
        return hipErrorInvalidValue;
    }
    if (flags[0] & 2) {
        ctx->nb_status = ANN_ERR_UNSUPPORTED;
        set_error("neighbour search box exceeds the image limit (cell far narrower than rc)");
        return hipErrorInvalidValue;
    }
    if (flags[0] & 1) {
        ctx->nb_status = ANN_ERR_CAPACITY;
        set_error("an atom has " + std::to_string(flags[1]) + " neighbours; capacity is " + std::to_string(kMaxNeigh));
        return hipErrorInvalidValue;
    }
    nl.npairs = total;
    nl.maxn = flags[1];
    if (spec_cap > 0 && total <= spec_cap) return hipSuccess;     // the speculative compaction stands
    if (spec_cap > 0) HIPCHK(hipStreamSynchronize(st));            // its kernels still hold the old arrays
    int64_t c1 = nl.cap, c2 = nl.cap, c3 = nl.cap, c4 = nl.cap, c5 = nl.cap;
    HIPCHK(grow(nl.idx, c1, total));
    HIPCHK(grow(nl.img, c2, total));
    HIPCHK(grow(nl.rev, c3, total));
    HIPCHK(grow(nl.geo, c4, total));
    HIPCHK(grow(nl.nsp, c5, total));
    nl.cap = std::min(std::min(c1, c2), std::min(std::min(c3, c4), c5));
    launch_compact(ctx, (int)std::min<int64_t>(nl.cap, INT32_MAX));
    return hipGetLastError();
}

// ---- a neighbour list supplied by the caller ----

__global__ void k_neigh_species(int64_t P, const int* __restrict__ idx, const int* __restrict__ species,
                                uint8_t* __restrict__ nsp) {
    const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (s < P) nsp[s] = (uint8_t)species[idx[s]];
}

// Reverse slots of a list whose rows have any order: a lane per entry walks the
// partner's whole row and counts the entries (j -> i, -n).  Exactly one for every
// entry of the list means that it is symmetric and holds nothing twice; anything
// else raises the flag.  Entries times row length loads (1,536 atoms with 91
// partners: 13 M, about 0.1 ms) against sorting the list on the host (17 ms).
__global__ __launch_bounds__(256) void k_rev_scan(int N, const int* __restrict__ off, const int* __restrict__ idx,
                                                  const uint32_t* __restrict__ img, int* __restrict__ rev,
                                                  int* __restrict__ flag) {
    const int i = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    if (i >= N) return;
    for (int s = off[i] + threadIdx.x % kWave; s < off[i + 1]; s += kWave) {
        const int j = idx[s];
        int n0, n1, n2;
        unpack_img(img[s], n0, n1, n2);
        const uint32_t want = pack_img(-n0, -n1, -n2);
        int found = 0, at = s;
        const int e = off[j + 1];
#pragma unroll 8
        for (int q = off[j]; q < e; ++q) {
            const bool hit = idx[q] == i && img[q] == want;
            found += hit ? 1 : 0;
            at = hit ? q : at;
        }
        rev[s] = at;
        if (found != 1) atomicOr(flag, 1);
    }
}

// The fault of a list that k_rev_scan refused, found on the host by sorting it
static int list_fault(const int* off, const int* idx, const uint32_t* pimg, int N) {
    const int64_t P = off[N];
    std::vector<int> owner(std::max<int64_t>(P, 1));
    for (int i = 0; i < N; ++i)
        for (int q = off[i]; q < off[i + 1]; ++q) owner[q] = i;
    std::vector<int64_t> order(P);
    for (int64_t q = 0; q < P; ++q) order[q] = q;
    auto key = [&](int64_t q) { return std::make_tuple(owner[q], idx[q], pimg[q]); };
    std::sort(order.begin(), order.end(), [&](int64_t x, int64_t y) { return key(x) < key(y); });
    for (int64_t q = 1; q < P; ++q)
        if (key(order[q]) == key(order[q - 1]))
            return fail(ANN_ERR_ARG, "neighbour list: atom " + std::to_string(owner[order[q]]) + " lists partner " +
                                         std::to_string(idx[order[q]]) + " twice with the same image");
    for (int64_t q = 0; q < P; ++q) {
        int n0, n1, n2;
        unpack_img(pimg[q], n0, n1, n2);
        const auto want = std::make_tuple(idx[q], owner[q], pack_img(-n0, -n1, -n2));
        auto it = std::lower_bound(order.begin(), order.end(), want,
                                   [&](int64_t x, const std::tuple<int, int, uint32_t>& w) { return key(x) < w; });
        if (it == order.end() || key(*it) != want)
            return fail(ANN_ERR_ARG, "neighbour list is not symmetric: entry " + std::to_string(q) + " (atom " +
                                         std::to_string(owner[q]) + " -> " + std::to_string(idx[q]) +
                                         ") has no reverse entry");
    }
    return fail(ANN_ERR_HIP, "neighbour list: reverse slots not found");
}

// Host CSR (off [N+1], idx [P], img [P][3]) of the current batch into the
// context's list: packed images, reverse slots found by walking the partners'
// rows, neighbour species and pair geometry on the device.  Returns an ANN status.
int set_neighbors_host(ann_ctx* ctx, const int* off, const int* idx, const int* img, double rc) {
    const int N = ctx->natoms;
    if (off[0] != 0) return fail(ANN_ERR_ARG, "neighbour list: off[0] must be 0");
    int maxn = 0;
    for (int i = 0; i < N; ++i) {
        if (off[i + 1] < off[i]) return fail(ANN_ERR_ARG, "neighbour list: offsets must not decrease");
        maxn = std::max(maxn, off[i + 1] - off[i]);
    }
    if (maxn > kMaxNeigh)
        return fail(ANN_ERR_CAPACITY, "an atom has " + std::to_string(maxn) + " neighbours; capacity is " +
                                          std::to_string(kMaxNeigh));
    const int64_t P = off[N];
    std::vector<uint32_t> pimg(std::max<int64_t>(P, 1));
    int s = 0;
    for (int i = 0; i < N; ++i) {
        while (ctx->atom_off[s + 1] <= i) ++s;
        for (int q = off[i]; q < off[i + 1]; ++q) {
            const int j = idx[q];
            if (j < ctx->atom_off[s] || j >= ctx->atom_off[s + 1])
                return fail(ANN_ERR_ARG, "neighbour list: partner outside the centre's structure");
            for (int x = 0; x < 3; ++x)
                if (img[3 * (int64_t)q + x] < -511 || img[3 * (int64_t)q + x] > 511)
                    return fail(ANN_ERR_UNSUPPORTED, "neighbour list: image vector beyond +-511 cells");
            pimg[q] = pack_img(img[3 * (int64_t)q], img[3 * (int64_t)q + 1], img[3 * (int64_t)q + 2]);
            if (j == i && pimg[q] == pack_img(0, 0, 0))
                return fail(ANN_ERR_ARG, "neighbour list: atom " + std::to_string(i) + " lists itself in its own cell");
        }
    }
    NList& nl = ctx->nl;
    hipStream_t st = ctx->stream;
    int64_t c1 = nl.cap, c2 = nl.cap, c3 = nl.cap, c4 = nl.cap, c5 = nl.cap;
    if (P > nl.cap) {
        ANN_HIP(hipStreamSynchronize(st));
        ANN_HIP(grow(nl.idx, c1, P));
        ANN_HIP(grow(nl.img, c2, P));
        ANN_HIP(grow(nl.rev, c3, P));
        ANN_HIP(grow(nl.geo, c4, P));
        ANN_HIP(grow(nl.nsp, c5, P));
        nl.cap = std::min(std::min(c1, c2), std::min(std::min(c3, c4), c5));
    }
    ANN_HIP(hipMemcpyAsync(nl.off, off, sizeof(int) * (N + 1), hipMemcpyHostToDevice, st));
    if (P > 0) {
        ANN_HIP(hipMemcpyAsync(nl.idx, idx, sizeof(int) * P, hipMemcpyHostToDevice, st));
        ANN_HIP(hipMemcpyAsync(nl.img, pimg.data(), sizeof(uint32_t) * P, hipMemcpyHostToDevice, st));
        k_rev_scan<<<(N + 3) / 4, 256, 0, st>>>(N, nl.off, nl.idx, nl.img, nl.rev, ctx->d_flag + 3);
        ANN_HIP(hipGetLastError());
        k_neigh_species<<<(unsigned)((P + 255) / 256), 256, 0, st>>>(P, nl.idx, ctx->d_species, nl.nsp);
        ANN_HIP(hipGetLastError());
    }
    nl.npairs = P;
    nl.maxn = maxn;
    ANN_HIP(refresh_geometry(ctx));
    // the refusal flag to the host words, cleared once read
    k_readback<<<1, kWave, 0, st>>>(ctx->d_flag + 3, 1, ctx->d_rb + 9, 0, 1);
    ANN_HIP(hipGetLastError());
    ANN_HIP(hipStreamSynchronize(st));       // the host vectors go out of scope
    (void)rc;
    if (((volatile const int*)ctx->h_rb)[9]) return list_fault(off, idx, pimg.data(), N);
    return ANN_OK;
}

// Pair geometry of every slot from the current positions and the list's image
// vectors (verlet-list reuse between rebuilds, the geometry of
// NNP::symm(..., verlet::List) src/nnp/nnp.cpp:389-395): same FP64 operation
// order as the build, so an unchanged position set reproduces the build's
// geometry bit for bit.  One wavefront per atom, lanes over its slots.
__global__ __launch_bounds__(256) void k_geom(int N, const double* __restrict__ pos, const int* __restrict__ sof,
                                              const double* __restrict__ cells, const int* __restrict__ off,
                                              const int* __restrict__ idx, const uint32_t* __restrict__ img,
                                              float4* __restrict__ geo) {
    const int i = blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (i >= N) return;
    const double* R = cells + 9 * sof[i];
    for (int s = off[i] + lane; s < off[i + 1]; s += kWave) {
        int n0, n1, n2;
        unpack_img(img[s], n0, n1, n2);
        double x, y, z, d2;
        pair_vec(pos, i, idx[s], R, n0, n1, n2, x, y, z, d2);
        geo[s] = make_float4((float)x, (float)y, (float)z, (float)sqrt(d2));
    }
}

hipError_t refresh_geometry(ann_ctx* ctx) {
    const int N = ctx->natoms;
    if (N == 0) return hipSuccess;
    Launch L(ctx, "nb_geometry");
    k_geom<<<(N + 3) / 4, 256, 0, ctx->stream>>>(N, ctx->d_pos, ctx->d_struc_of, ctx->d_cells, ctx->nl.off,
                                                 ctx->nl.idx, ctx->nl.img, ctx->nl.geo);
    return hipGetLastError();
}

// Positions back into the cell, x <- R (f - floor f) with f = R^-1 x
// (Cell::returnToCell, src/format/xyz_struc.cpp:176-181).
__global__ void k_wrap(int N, double* __restrict__ pos, const int* __restrict__ sof,
                       const double* __restrict__ cells) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= N) return;
    const double* R = cells + 9 * sof[i];
    const double a = R[0], b = R[1], c = R[2], d = R[3], e = R[4], f = R[5], g = R[6], h = R[7], k = R[8];
    const double A = e * k - f * h, B = -(d * k - f * g), C = d * h - e * g;
    const double id = 1.0 / (a * A + b * B + c * C);
    const double Ri[9] = {A * id, -(b * k - c * h) * id, (b * f - c * e) * id,
                          B * id, (a * k - c * g) * id,  -(a * f - c * d) * id,
                          C * id, -(a * h - b * g) * id, (a * e - b * d) * id};
    const double x[3] = {pos[3 * i], pos[3 * i + 1], pos[3 * i + 2]};
    double fr[3];
    for (int q = 0; q < 3; ++q) {
        const double t = Ri[3 * q] * x[0] + Ri[3 * q + 1] * x[1] + Ri[3 * q + 2] * x[2];
        fr[q] = t - floor(t);
    }
    for (int q = 0; q < 3; ++q) pos[3 * i + q] = R[3 * q] * fr[0] + R[3 * q + 1] * fr[1] + R[3 * q + 2] * fr[2];
}

hipError_t wrap_positions(ann_ctx* ctx, double* pos) {
    const int N = ctx->natoms;
    if (N == 0) return hipSuccess;
    k_wrap<<<(N + 255) / 256, 256, 0, ctx->stream>>>(N, pos, ctx->d_struc_of, ctx->d_cells);
    return hipGetLastError();
}

hipError_t struc_index(ann_ctx* ctx) {
    k_struc_of<<<ctx->nstruc, 256, 0, ctx->stream>>>(ctx->d_atom_off, ctx->nstruc, ctx->d_struc_of);
    return hipGetLastError();
}

}  // namespace ann
