// symm.hip -- symmetry functions G (NNP::symm), the force adjoint
// P[s] = dE_i/dr_ij (NNP::force / NNP::compute) and the forward-mode basis
// tangent used by the force-loss weight gradient.
//
// Reference loops: src/nnp/nnp.cpp:333-375 (symm), 461-520 and 601-665
// (force/compute; angular assembly :503-516), basis functions
// src/nnp/basis_radial.cpp:263-376 and src/nnp/basis_angular.cpp:371-563.
//
// Two forms, one wavefront (block of 64) per centre atom in both:
//
//  PLAIN (reference-shaped): neighbours in canonical order in LDS; lane j
//    loops k > j exactly like the reference (triangular, unbalanced),
//    evaluates every angular function of the triplet from scratch (cutoffs,
//    exp and pow per function), accumulates G in lane-private LDS columns and
//    scatters the k-side of the force through LDS atomics.
//
//  FAST: neighbours regrouped by species in LDS so that every (species j,
//    species k) block of the angular basis is a rectangle (j, k in different
//    species) or a triangle (same species) of index space; the exponential of
//    the GAUSS family factorises over the pair, exp(-(rij^2+rik^2)/eta^2) =
//    E(rij) E(rik), so E*fc is computed once per neighbour and per distinct
//    width; blocks whose functions form a {width} x {(lambda,zeta)} grid run a
//    kernel specialised on the grid shape with integer powers by repeated
//    squaring and register accumulators.
//      forward: unordered pairs flattened over the 64 lanes (triangle folded
//        into an n x (n-1)/2 rectangle), wave-reduced per block;
//      adjoint / tangent: skewed schedule, lane = owner j, partner
//        k = (j + t) mod n at step t, so that lanes of one instruction touch
//        distinct partners; each unordered triplet is evaluated once and its
//        two slot contributions are accumulated in registers (owner) and LDS
//        (partner) -- no global atomics, deterministic.
//  Both are FP32 VALU-bound (the roofline that prices them is the FP32 peak).
#include <algorithm>
#include <vector>

#include "basis_dev.h"
#include "harm_dev.h"
#include "net_dev.h"

namespace ann {

struct SymmArgs {
    const DevModel* dm;
    const float* rad_rs;
    const float* rad_eta;
    const float* ang_eta;
    const float* ang_zeta;
    const float* ang_lam;
    int N, ldg, maxn;
    int smem_wave;            // bytes of dynamic LDS per wavefront (moment kernels: one atom per wavefront)
    const int* species;
    const int* off;
    const float4* geo;
    const uint8_t* nsp;
    const int* nidx;
    float* G;
    const float* dEdG;
    float* P;
    const float* u;
    float* v;
    float* Tout;              // moment form, G: store each atom's moments T here (or null)
    const float* Tin;         // moment form, adjoint and tangent: moments of the same geometry (or null: recompute)
    int rad_gauss;            // every radial block is GAUSSIAN
    int nrad, nrs;            // widest radial block; its row stride in the adjoint's tables (odd)
    int grows;                // function rows in LDS at a time (G, stored-moment tangent, recomputing adjoint)
    int atomsK;               // atoms per wavefront of G and of the stored-moment adjoint
    // fused E+F (mode 3): the network's parameter tables and inputs, the atom energies
    const float* wchunk;      // forward weight rows, biases, output neuron (net_dev.h layout)
    const float* wtrans;      // transposed weight rows (backward)
    const float* inpw;
    const float* inpb;
    float* Eatom;
    // persistent dispatch of the moment kernels (or null): per XCD a queue of
    // (first atom, atom count) items, its counter at queue[32 q]
    int* queue;
    const int2* items;
    const int* qoff;          // [kXcds + 1] item ranges of the queues
};

// Sum N per-lane values over the 64 lanes with a transposing butterfly: at
// each halving step a lane keeps half of its values and receives the partner's
// copy of that half (N - 1 exchanges instead of 6N), then the lanes that hold
// the same value index finish with plain butterflies.  Afterwards lane l holds
// the total of value index vidx(l); returns it.
template <int N>
__device__ __forceinline__ float wave_sum_multi(float (&v)[N], int& idx) {
    const int lane = threadIdx.x % kWave;
    int base = 0;
#pragma unroll
    for (int h = N / 2, bit = 32; h >= 1; h >>= 1, bit >>= 1) {
        const bool upper = (lane & bit) != 0;
        // bitwise blend of two statically indexed registers: a conditional
        // choice between v[q] and v[q + h] is otherwise rewritten by the
        // compiler into a runtime-indexed register access (a compare/select
        // chain over all N registers)
        const unsigned m = upper ? 0xffffffffu : 0u;
#pragma unroll
        for (int q = 0; q < h; ++q) {
            const unsigned lo = __float_as_uint(v[q]), hi = __float_as_uint(v[q + h]);
            const float send = __uint_as_float((lo & m) | (hi & ~m));
            const float keep = __uint_as_float((hi & m) | (lo & ~m));
            v[q] = keep + __shfl_xor(send, bit);
        }
        if (upper) base += h;
    }
    float s = v[0];
    constexpr int steps = (N >= 64) ? 0 : 6 - __builtin_ctz(N);
    int bit = 1;
#pragma unroll
    for (int q = 0; q < steps; ++q, bit <<= 1) s += __shfl_xor(s, bit);
    idx = base;
    return s;
}

// LDS ordering between the lanes of one wavefront (each wavefront of a
// moment-kernel block owns its own LDS slice, so no block barrier is needed)
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// =========================================================== PLAIN form ====

// mode 0: G, 1: adjoint P, 2: tangent v
template <int MODE>
__global__ __launch_bounds__(64) void k_plain(SymmArgs A) {
    extern __shared__ float smem[];
    const int i = blockIdx.x, lane = threadIdx.x;
    if (i >= A.N) return;
    const DevModel& M = *A.dm;
    const int a = A.species[i], o = A.off[i], n = A.off[i + 1] - o;
    const int S = M.S, NP = M.NP, ldg = A.ldg, maxn = A.maxn;
    float4* sg = reinterpret_cast<float4*>(smem);          // (x, y, z, r) canonical order
    float* sfc = reinterpret_cast<float*>(sg + maxn);
    float* sgc = sfc + maxn;
    int* ssp = reinterpret_cast<int*>(sgc + maxn);
    float* rest = reinterpret_cast<float*>(ssp + maxn);
    constexpr int LP = 65;                                  // padded lane stride
    for (int t = lane; t < n; t += kWave) {
        const float4 gq = A.geo[o + t];
        sg[t] = gq;
        float f, g;
        cutoff_fg(M.cutoff, M.rc, M.rci, M.pirc, gq.w, f, g);
        sfc[t] = f;
        sgc[t] = g;
        ssp[t] = A.nsp[o + t];
    }
    float* acc = rest;                                      // [ldg][LP]   (modes 0, 2)
    float* sd = rest;                                       // [ldg]       (mode 1)
    float* sP = rest + ldg;                                 // [maxn][3]   (mode 1)
    float4* st = reinterpret_cast<float4*>(rest + ldg * LP);  // [maxn] (tx,ty,tz, r^.t) (mode 2)
    if (MODE == 1) {
        for (int m = lane; m < ldg; m += kWave) sd[m] = A.dEdG[(size_t)i * ldg + m];
        for (int t = lane; t < 3 * n; t += kWave) sP[t] = 0.0f;
    } else {
        for (int m = 0; m < ldg; ++m) acc[m * LP + lane] = 0.0f;
    }
    if (MODE == 2) {
        for (int t = lane; t < n; t += kWave) {
            const int j = A.nidx[o + t];
            const float tx = A.u[3 * i] - A.u[3 * j], ty = A.u[3 * i + 1] - A.u[3 * j + 1],
                        tz = A.u[3 * i + 2] - A.u[3 * j + 2];
            const float4 gq = sg[t];
            st[t] = make_float4(tx, ty, tz, (gq.x * tx + gq.y * ty + gq.z * tz) / gq.w);
        }
    }
    __syncthreads();
    // radial
    for (int j = lane; j < n; j += kWave) {
        const RadBlock rb = M.rad[a * S + ssp[j]];
        const float r = sg[j].w;
        float amp = 0.0f;
        for (int m = 0; m < rb.n; ++m) {
            float v, d;
            radial_fd(rb.name, A.rad_eta[rb.par + m], A.rad_rs[rb.par + m], r, sfc[j], sgc[j], v, d);
            if (MODE == 0) acc[(rb.goff + m) * LP + lane] += v;
            if (MODE == 1) amp += sd[rb.goff + m] * d;
            if (MODE == 2) acc[(rb.goff + m) * LP + lane] += d * st[j].w;
        }
        if (MODE == 1) {
            const float4 gq = sg[j];
            atomicAdd(&sP[3 * j], amp * gq.x / r);
            atomicAdd(&sP[3 * j + 1], amp * gq.y / r);
            atomicAdd(&sP[3 * j + 2], amp * gq.z / r);
        }
    }
    // angular: lane j, partners k > j (reference loop order)
    for (int j = lane; j < n; j += kWave) {
        const float4 gj = sg[j];
        const float rj = gj.w;
        float pjx = 0, pjy = 0, pjz = 0;
        for (int k = j + 1; k < n; ++k) {
            const float4 gk = sg[k];
            const float rk = gk.w;
            // cutoffs recomputed per triplet, as BasisA::symm/force do
            float fj, gcj, fk, gck;
            cutoff_fg(M.cutoff, M.rc, M.rci, M.pirc, rj, fj, gcj);
            cutoff_fg(M.cutoff, M.rc, M.rci, M.pirc, rk, fk, gck);
            const float c = (gj.x * gk.x + gj.y * gk.y + gj.z * gk.z) / (rj * rk);
            const AngBlock& ab = M.ang[a * NP + pair_idx(ssp[j], ssp[k])];
            float sA = 0, sBj = 0, sBk = 0;
            for (int m = 0; m < ab.n; ++m) {
                const float eta = A.ang_eta[ab.par + m];
                float G, dc, d0, d1;
                angular_fd(ab.name, 1.0f / (eta * eta), A.ang_zeta[ab.par + m], 0.5f * A.ang_lam[ab.par + m],
                           rj, rk, c, fj, fk, gcj, gck, G, dc, d0, d1);
                if (MODE == 0) acc[(ab.goff + m) * LP + lane] += G;
                if (MODE == 1) {
                    const float de = sd[ab.goff + m];
                    sA += de * dc;
                    sBj += de * d0;
                    sBk += de * d1;
                }
                if (MODE == 2) {
                    const float4 tj = st[j], tk = st[k];
                    const float cdot = ((gk.x * tj.x + gk.y * tj.y + gk.z * tj.z) / rk - c * tj.w) / rj +
                                       ((gj.x * tk.x + gj.y * tk.y + gj.z * tk.z) / rj - c * tk.w) / rk;
                    acc[(ab.goff + m) * LP + lane] += dc * cdot + d0 * tj.w + d1 * tk.w;
                }
            }
            if (MODE == 1) {
                const float hjx = gj.x / rj, hjy = gj.y / rj, hjz = gj.z / rj;
                const float hkx = gk.x / rk, hky = gk.y / rk, hkz = gk.z / rk;
                pjx += sA * (hkx - c * hjx) / rj + sBj * hjx;
                pjy += sA * (hky - c * hjy) / rj + sBj * hjy;
                pjz += sA * (hkz - c * hjz) / rj + sBj * hjz;
                atomicAdd(&sP[3 * k], sA * (hjx - c * hkx) / rk + sBk * hkx);
                atomicAdd(&sP[3 * k + 1], sA * (hjy - c * hky) / rk + sBk * hky);
                atomicAdd(&sP[3 * k + 2], sA * (hjz - c * hkz) / rk + sBk * hkz);
            }
        }
        if (MODE == 1) {
            atomicAdd(&sP[3 * j], pjx);
            atomicAdd(&sP[3 * j + 1], pjy);
            atomicAdd(&sP[3 * j + 2], pjz);
        }
    }
    __syncthreads();
    if (MODE == 1) {
        for (int t = lane; t < 3 * n; t += kWave) A.P[3 * (size_t)o + t] = sP[t];
    } else {
        float* out = (MODE == 0 ? A.G : A.v) + (size_t)i * ldg;
        for (int m = lane; m < ldg; m += kWave) {
            float s = 0.0f;
            for (int l = 0; l < kWave; ++l) s += acc[m * LP + l];
            out[m] = s;
        }
    }
}

// ============================================================ FAST form ====

constexpr int kFastU = 4;   // distinct angular widths per centre species in the fast form

struct FastSmem {
    float4* g;      // [maxn] (hx, hy, hz, 1/r), species-sorted
    float4* ef;     // [maxn] exp(-r^2 ieta2_u) fc for u = 0..3
    float4* efd;    // [maxn] d/dr of ef
    float2* fg;     // [maxn] cutoff and its derivative
    float* r;       // [maxn]
    int* canon;     // [maxn] canonical slot of each sorted entry
    int* seg;       // [kMaxSpecies + 1]
    float* extra;   // kernel specific
};

__device__ __forceinline__ float f4get(const float4& v, int u) {
    return u == 0 ? v.x : (u == 1 ? v.y : (u == 2 ? v.z : v.w));
}

// w^e for a wave-uniform integer e >= 0 (common exponents unrolled)
__device__ __forceinline__ float ipow(float w, int e) {
    switch (e) {
        case 0: return 1.0f;
        case 1: return w;
        case 2: return w * w;
        case 3: return w * w * w;
        case 4: { const float q = w * w; return q * q; }
        case 7: { const float q = w * w, q4 = q * q; return q4 * q * w; }
        case 8: { const float q = w * w, q4 = q * q; return q4 * q4; }
        default: {
            float r = 1.0f, b = w;
            for (int x = e; x; x >>= 1) {
                if (x & 1) r *= b;
                b *= b;
            }
            return r;
        }
    }
}

// w^(zeta-1) for integer (zi >= 1) or general zeta (zi < 0)
__device__ __forceinline__ float pow_m1(float w, int zi, float zeta) {
    if (zi >= 1) return ipow(w, zi - 1);
    return w > 0.0f ? exp2f((zeta - 1.0f) * __log2f(w)) : 0.0f;
}

// Regroup the neighbours of atom i by species (stable) and precompute the
// per-neighbour factors; seg[] gives the species segments.  Entries beyond the
// cutoff (a list built with rc + skin) are dropped here; their adjoint slots
// are written as zero when zero_P is set.  Returns the number kept.
__device__ __forceinline__ int fast_load(const SymmArgs& A, const DevModel& M, int i, int a, int o, int n, FastSmem& sm,
                         bool need_deriv, bool zero_P, float4* tv = nullptr) {
    const int lane = threadIdx.x % kWave, S = M.S, U = M.nunion[a];
    const float rc = M.rc;
    int cnt[kMaxSpecies];
#pragma unroll
    for (int b = 0; b < kMaxSpecies; ++b) cnt[b] = 0;
    // the first two rows of 64 neighbours stay in registers for the second pass
    float4 g0 = make_float4(0.f, 0.f, 0.f, 0.f), g1 = g0;
    int p0 = -1, p1 = -1, j0 = 0, j1 = 0;
    for (int q = 0; q < n; q += kWave) {
        const int t = q + lane;
        float4 gq = make_float4(0.f, 0.f, 0.f, 0.f);
        int raw = -1, jr = 0;
        if (t < n) {
            gq = A.geo[o + t];
            raw = (int)A.nsp[o + t];
            if (tv) jr = A.nidx[o + t];
        }
        if (q == 0) { g0 = gq; p0 = raw; j0 = jr; }
        if (q == kWave) { g1 = gq; p1 = raw; j1 = jr; }
        const int sp = (t < n && gq.w <= rc) ? raw : -1;
#pragma unroll
        for (int b = 0; b < kMaxSpecies; ++b)
            if (b < S) cnt[b] += __popcll(__ballot(sp == b));
    }
    int base[kMaxSpecies];
    int acc = 0;
#pragma unroll
    for (int b = 0; b < kMaxSpecies; ++b) {
        base[b] = acc;
        if (b < S) acc += cnt[b];
    }
#pragma unroll
    for (int b = 0; b < kMaxSpecies; ++b)
        if (b < S && lane == b) sm.seg[b] = base[b];
    if (lane == S) sm.seg[S] = acc;
    float ie[kFastU];
#pragma unroll
    for (int u = 0; u < kFastU; ++u) ie[u] = u < U ? M.uieta2[a][u] : 0.0f;
    const uint64_t lt = (1ull << lane) - 1ull;
    // tangent: the centre's displacement (the same for every lane)
    float uix = 0.f, uiy = 0.f, uiz = 0.f;
    if (tv) {
        uix = A.u[3 * i];
        uiy = A.u[3 * i + 1];
        uiz = A.u[3 * i + 2];
    }
    for (int q = 0; q < n; q += kWave) {
        const int t = q + lane;
        float4 gq;
        int raw, jr;
        if (q == 0) { gq = g0; raw = p0; jr = j0; }
        else if (q == kWave) { gq = g1; raw = p1; jr = j1; }
        else {
            gq = t < n ? A.geo[o + t] : make_float4(0.f, 0.f, 0.f, 0.f);
            raw = t < n ? (int)A.nsp[o + t] : -1;
            jr = (tv && t < n) ? A.nidx[o + t] : 0;
        }
        const bool keep = t < n && gq.w <= rc;
        const int sp = keep ? raw : -1;
        if (zero_P && t < n && !keep) {
            A.P[3 * ((size_t)o + t)] = 0.0f;
            A.P[3 * ((size_t)o + t) + 1] = 0.0f;
            A.P[3 * ((size_t)o + t) + 2] = 0.0f;
        }
        int pos = 0;
#pragma unroll
        for (int b = 0; b < kMaxSpecies; ++b) {
            if (b < S) {
                const uint64_t mk = __ballot(sp == b);
                if (sp == b) pos = base[b] + __popcll(mk & lt);
                base[b] += __popcll(mk);
            }
        }
        if (keep) {
            const float r = gq.w, ir = __builtin_amdgcn_rcpf(r);   // 1 ulp
            sm.g[pos] = make_float4(gq.x * ir, gq.y * ir, gq.z * ir, ir);
            if (tv) {
                // tangent direction t = u_i - u_j and its projection on the unit vector
                const float tx = uix - A.u[3 * jr], ty = uiy - A.u[3 * jr + 1], tz = uiz - A.u[3 * jr + 2];
                tv[pos] = make_float4(tx, ty, tz, (gq.x * ir) * tx + (gq.y * ir) * ty + (gq.z * ir) * tz);
            }
            sm.r[pos] = r;
            if (sm.canon) sm.canon[pos] = t;                     // slot map (kernels that need it)
            float f, gcut;
            cutoff_fg(M.cutoff, M.rc, M.rci, M.pirc, r, f, gcut);
            sm.fg[pos] = make_float2(f, gcut);
            float e[kFastU], d[kFastU];
#pragma unroll
            for (int u = 0; u < kFastU; ++u) {
                const float x = u < U ? __expf(-ie[u] * r * r) : 0.0f;
                e[u] = x * f;
                d[u] = x * (-2.0f * r * ie[u] * f + gcut);
            }
            sm.ef[pos] = make_float4(e[0], e[1], e[2], e[3]);
            if (need_deriv) sm.efd[pos] = make_float4(d[0], d[1], d[2], d[3]);
        }
    }
    return acc;
}

// Distance factor of width g for a pair of legs j, k: GAUSS blocks multiply the
// per-neighbour factors e_g(r) = exp(-r^2/eta^2) fc(r) (and their r-derivatives)
// computed once per neighbour; the other families depend on r_j^2 + r_k^2
// through a factor that does not separate, evaluated here per pair:
// D = fr(r_j^2 + r_k^2) fc_j fc_k, dD/dr_j = (2 r_j fr' fc_j + fr fc'_j) fc_k.
template <bool GS, int NG>
__device__ __forceinline__ void pair_factors(const AngBlock& B, const float* uie, const int (&gu)[NG], const FastSmem& sm,
                                             int jj, int kk, bool deriv, float (&D)[NG], float (&Dj)[NG],
                                             float (&Dk)[NG]) {
    if (GS) {
        const float4 ej4 = sm.ef[jj], ek4 = sm.ef[kk];
        float4 dj4 = make_float4(0.f, 0.f, 0.f, 0.f), dk4 = dj4;
        if (deriv) { dj4 = sm.efd[jj]; dk4 = sm.efd[kk]; }
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            const float ej = f4get(ej4, g), ek = f4get(ek4, g);
            D[g] = ej * ek;
            Dj[g] = deriv ? f4get(dj4, g) * ek : 0.0f;
            Dk[g] = deriv ? ej * f4get(dk4, g) : 0.0f;
        }
    } else {
        const float rj = sm.r[jj], rk = sm.r[kk];
        const float2 fj = sm.fg[jj], fk = sm.fg[kk];
        const float r2s = rj * rj + rk * rk, ff = fj.x * fk.x;
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            float fr, dfr;
            ang_radial(B.name, uie[gu[g]], r2s, fr, dfr);
            D[g] = fr * ff;
            Dj[g] = deriv ? (2.0f * rj * dfr * fj.x + fr * fj.y) * fk.x : 0.0f;
            Dk[g] = deriv ? (2.0f * rk * dfr * fk.x + fr * fk.y) * fj.x : 0.0f;
        }
    }
}

// ---- forward / tangent over one grid block (unordered pairs, flattened) ----
template <int NG, int NK, int MODE, bool GS>
__device__ __forceinline__ void fast_block_flat(const AngBlock& B, const float* uie, const FastSmem& sm, int sb, int nb,
                                                int sc, int nc, bool tri, const float4* tv, float* out) {
    const int lane = threadIdx.x % kWave;
    float lamh[NK], zeta[NK];
    int zi[NK], gu[NG];
#pragma unroll
    for (int k = 0; k < NK; ++k) { lamh[k] = B.lamh[k]; zeta[k] = B.zeta[k]; zi[k] = B.zint[k]; }
#pragma unroll
    for (int g = 0; g < NG; ++g) gu[g] = B.gu[g];
    float acc[NG][NK];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int k = 0; k < NK; ++k) acc[g][k] = 0.0f;
    const int h = tri ? (nb - 1) / 2 : 0;
    const int cols = tri ? h : nc;
    const int main_total = tri ? nb * h : nb * nc;
    const int total = tri ? nb * (nb - 1) / 2 : nb * nc;
    int j = 0, t = 0;
    if (cols > 0) { j = lane / cols; t = lane % cols; }
    const int dj = cols > 0 ? kWave / cols : 0, dt = cols > 0 ? kWave % cols : 0;
    for (int tau = lane; tau < total; tau += kWave) {
        int jj, kk;
        if (tau < main_total) {
            jj = j;
            kk = tri ? j + 1 + t : t;
            if (tri && kk >= nb) kk -= nb;
        } else {
            jj = tau - main_total;
            kk = jj + (nb >> 1);
        }
        jj += sb;
        kk += sc;
        const float4 gj = sm.g[jj], gk = sm.g[kk];
        const float c = gj.x * gk.x + gj.y * gk.y + gj.z * gk.z;
        float Dg[NG], Dj[NG], Dk[NG];
        pair_factors<GS, NG>(B, uie, gu, sm, jj, kk, MODE != 0, Dg, Dj, Dk);
        if (MODE == 0) {
            float p[NK];
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const float cw = fabsf(0.5f + lamh[k] * c);
                p[k] = zi[k] >= 0 ? ipow(cw, zi[k]) : pow_m1(cw, -1, zeta[k]) * cw;
            }
#pragma unroll
            for (int g = 0; g < NG; ++g) {
#pragma unroll
                for (int k = 0; k < NK; ++k) acc[g][k] += p[k] * Dg[g];
            }
        } else {
            const float4 tj = tv[jj], tk = tv[kk];
            const float cdot = ((gk.x * tj.x + gk.y * tj.y + gk.z * tj.z) - c * tj.w) * gj.w +
                               ((gj.x * tk.x + gj.y * tk.y + gj.z * tk.z) - c * tk.w) * gk.w;
            float p[NK], dp[NK];
#pragma unroll
            for (int k = 0; k < NK; ++k) {
                const float cw = fabsf(0.5f + lamh[k] * c);
                const float w1 = pow_m1(cw, zi[k], zeta[k]);
                p[k] = w1 * cw;
                dp[k] = zeta[k] * lamh[k] * w1;
            }
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const float rdot = Dj[g] * tj.w + Dk[g] * tk.w;
                const float D = Dg[g] * cdot;
#pragma unroll
                for (int k = 0; k < NK; ++k) acc[g][k] += dp[k] * D + p[k] * rdot;
            }
        }
        t += dt;
        j += dj;
        if (t >= cols) { t -= cols; j += 1; }
    }
    float flat[NG * NK];
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
        for (int k = 0; k < NK; ++k) flat[g * NK + k] = acc[g][k];
    if constexpr ((NG * NK & (NG * NK - 1)) == 0) {
        int idx;
        const float s = wave_sum_multi<NG * NK>(flat, idx);
        constexpr int lpv = kWave / (NG * NK);   // lanes holding each value
        if ((lane & (lpv - 1)) == 0 && lane < kWave) out[B.goff + B.outm[idx]] = s;
    } else {
#pragma unroll
        for (int q = 0; q < NG * NK; ++q) {
            const float s = wave_sum(flat[q]);
            if (lane == 0) out[B.goff + B.outm[q]] = s;
        }
    }
}

// ---- adjoint over one grid block: skewed owner/partner schedule ----
template <int NG, int NK, bool GS>
__device__ __forceinline__ void fast_block_adj(const AngBlock& B, const float* uie, const FastSmem& sm, int sb, int nb,
                                               int sc, int nc, bool tri, const float* sd, float* sP) {
    const int lane = threadIdx.x % kWave;
    float lamh[NK], zeta[NK], dl[NG][NK];
    int zi[NK], gu[NG];
#pragma unroll
    for (int k = 0; k < NK; ++k) { lamh[k] = B.lamh[k]; zeta[k] = B.zeta[k]; zi[k] = B.zint[k]; }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
        gu[g] = B.gu[g];
#pragma unroll
        for (int k = 0; k < NK; ++k) dl[g][k] = sd[B.goff + B.outm[g * NK + k]];
    }
    // owners: the smaller segment (triangle: all items)
    int so = sb, no = nb, spp = sc, np = nc;
    if (!tri && nb > nc) { so = sc; no = nc; spp = sb; np = nb; }
    const int Q = tri ? 1 : np / no;
    const int items = no * Q;
    const int h = tri ? (no - 1) / 2 : 0;
    for (int r0 = 0; r0 < items; r0 += kWave) {
        const int id = r0 + lane;
        const bool act = id < items;
        const int j = act ? id % no : 0;
        const int q = act ? id / no : 0;
        const int J = so + j;
        const float4 gj = sm.g[J];
        float ej[NG], edj[NG];                  // GAUSS: the owner's per-neighbour factors, loaded once
        if constexpr (GS) {
            const float4 ej4 = sm.ef[J], dj4 = sm.efd[J];
#pragma unroll
            for (int g = 0; g < NG; ++g) { ej[g] = f4get(ej4, g); edj[g] = f4get(dj4, g); }
        }
        float px = 0.0f, py = 0.0f, pz = 0.0f;
        int len, koff;
        if (tri) {
            len = h + ((no & 1) == 0 && j < (no >> 1) ? 1 : 0);
            koff = j + 1;
        } else {
            len = (q < Q - 1) ? no : np - (Q - 1) * no;
            koff = j + q * no;
        }
        const int lmax = tri ? h + ((no & 1) == 0 ? 1 : 0) : (np - (Q - 1) * no);
        for (int t = 0; t < lmax; ++t) {
            if (act && t < len) {
                int k = koff + t;
                if (k >= np) k -= np;
                const int K = spp + k;
                const float4 gk = sm.g[K];
                const float c = gj.x * gk.x + gj.y * gk.y + gj.z * gk.z;
                float Dg[NG], Dj[NG], Dk[NG];
                if constexpr (GS) {
                    const float4 ek4 = sm.ef[K], dk4 = sm.efd[K];
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        const float ek = f4get(ek4, g);
                        Dg[g] = ej[g] * ek;
                        Dj[g] = edj[g] * ek;
                        Dk[g] = ej[g] * f4get(dk4, g);
                    }
                } else {
                    pair_factors<GS, NG>(B, uie, gu, sm, J, K, true, Dg, Dj, Dk);
                }
                float p[NK], dp[NK];
#pragma unroll
                for (int kk = 0; kk < NK; ++kk) {
                    const float cw = fabsf(0.5f + lamh[kk] * c);
                    const float w1 = pow_m1(cw, zi[kk], zeta[kk]);
                    p[kk] = w1 * cw;
                    dp[kk] = zeta[kk] * lamh[kk] * w1;
                }
                float Ac = 0.0f, Bj = 0.0f, Bk = 0.0f;
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    float Sg = 0.0f, Tg = 0.0f;
#pragma unroll
                    for (int kk = 0; kk < NK; ++kk) {
                        Sg += dl[g][kk] * p[kk];
                        Tg += dl[g][kk] * dp[kk];
                    }
                    Ac += Tg * Dg[g];
                    Bj += Sg * Dj[g];
                    Bk += Sg * Dk[g];
                }
                const float aj = Ac * gj.w, ak = Ac * gk.w;
                px += aj * (gk.x - c * gj.x) + Bj * gj.x;
                py += aj * (gk.y - c * gj.y) + Bj * gj.y;
                pz += aj * (gk.z - c * gj.z) + Bj * gj.z;
                atomicAdd(&sP[3 * K], ak * (gj.x - c * gk.x) + Bk * gk.x);
                atomicAdd(&sP[3 * K + 1], ak * (gj.y - c * gk.y) + Bk * gk.y);
                atomicAdd(&sP[3 * K + 2], ak * (gj.z - c * gk.z) + Bk * gk.z);
            }
        }
        if (act) {
            atomicAdd(&sP[3 * J], px);
            atomicAdd(&sP[3 * J + 1], py);
            atomicAdd(&sP[3 * J + 2], pz);
        }
    }
}

#define ANN_SHAPES(X) X(1, 8) X(4, 4) X(3, 4) X(2, 4) X(1, 4) X(1, 2) X(1, 1) X(2, 2) X(4, 2) X(3, 2)

// shapes with a compiled fast kernel
__host__ __device__ inline bool fast_shape_ok(int ng, int nk) {
#define X(G, K) if (ng == G && nk == K) return true;
    ANN_SHAPES(X)
#undef X
    return false;
}

// radial part, lane over the neighbours of one species segment, 16 functions at a time
// GAUSSIAN radial functions of one (centre, neighbour species) block, CH per
// pass with widths and centres in registers.  Adjoint: per neighbour,
// d/dr [e fc] = e (gc - 2 eta x fc) weighted by dE/dG, split into two running
// sums; G / tangent: lanes over the neighbours, one transposing reduction.
template <int MODE, int CH>
__device__ __forceinline__ void radial_gauss(const SymmArgs& A, const RadBlock& rb, const FastSmem& sm, int s0, int s1,
                                             const float4* tv, const float* sd, float* sP, float* out) {
    const int lane = threadIdx.x % kWave;
    for (int m0 = 0; m0 < rb.n; m0 += CH) {
        float eta[CH], rs[CH], gs[CH];
#pragma unroll
        for (int m = 0; m < CH; ++m) {
            const bool in = m0 + m < rb.n;
            eta[m] = in ? A.rad_eta[rb.par + m0 + m] : 0.0f;
            rs[m] = in ? A.rad_rs[rb.par + m0 + m] : 0.0f;
            gs[m] = (MODE == 1 && in) ? sd[rb.goff + m0 + m] : 0.0f;
        }
        if (MODE == 1) {
            for (int J = s0 + lane; J < s1; J += kWave) {
                const float r = sm.r[J];
                const float2 fg = sm.fg[J];
                float se = 0.0f, sx = 0.0f;
#pragma unroll
                for (int m = 0; m < CH; ++m) {
                    const float x = eta[m] * (r - rs[m]), ge = gs[m] * __expf(-x * x);
                    se += ge;
                    sx += ge * eta[m] * x;
                }
                const float amp = se * fg.y - 2.0f * fg.x * sx;
                const float4 gj = sm.g[J];
                sP[3 * J] += amp * gj.x;
                sP[3 * J + 1] += amp * gj.y;
                sP[3 * J + 2] += amp * gj.z;
            }
            continue;
        }
        float acc[CH];
#pragma unroll
        for (int m = 0; m < CH; ++m) acc[m] = 0.0f;
        for (int J = s0 + lane; J < s1; J += kWave) {
            const float r = sm.r[J];
            const float w = MODE == 2 ? tv[J].w : 0.0f;
            const float2 fg = sm.fg[J];
            const float fc = fg.x, gc = fg.y;
#pragma unroll
            for (int m = 0; m < CH; ++m) {
                const float x = eta[m] * (r - rs[m]), e = __expf(-x * x);
                acc[m] += MODE == 0 ? e * fc : e * (gc - 2.0f * eta[m] * x * fc) * w;
            }
        }
        int idx;
        const float sum = wave_sum_multi<CH>(acc, idx);
        if ((lane & (kWave / CH - 1)) == 0 && m0 + idx < rb.n) out[rb.goff + m0 + idx] = sum;
    }
}

// GAUSSIAN block of at most 16 functions (G and tangent): lanes over
// (neighbour, function) pairs, W = 8 or 16 functions per lane group and 64 / W
// neighbours per pass, so every lane evaluates one exponential per pass and the
// sum over neighbours is log2(64 / W) butterflies.  Against W exponentials per
// lane on a partly idle wavefront and a W-value transposing reduction it wins
// up to about 32 passes (water: 60 neighbours of one species, 15 passes).
template <int MODE>
__device__ __forceinline__ void radial_gauss_pairs(const SymmArgs& A, const RadBlock& rb, const FastSmem& sm, int s0, int s1,
                                                   int W, const float4* tv, float* out) {
    const int lane = threadIdx.x % kWave;
    const int m = lane & (W - 1), nj = kWave / W;
    const bool in = m < rb.n;
    const float eta = in ? A.rad_eta[rb.par + m] : 0.0f;
    const float rs = in ? A.rad_rs[rb.par + m] : 0.0f;
    float acc = 0.0f;
    for (int J = s0 + lane / W; J < s1; J += nj) {
        const float r = sm.r[J];
        const float2 fg = sm.fg[J];
        const float x = eta * (r - rs), e = __expf(-x * x);
        acc += MODE == 0 ? e * fg.x : e * (fg.y - 2.0f * eta * x * fg.x) * tv[J].w;
    }
    for (int bit = W; bit < kWave; bit <<= 1) acc += __shfl_xor(acc, bit);
    if (lane < W && in) out[rb.goff + m] = acc;
}

// passes of the pair form above which the lane-over-neighbour form is used
constexpr int kPairPasses = 32;

// the moment kernels index block widths by union width: both bounds must agree
static_assert(kMaxUnionEta == kGridG, "union widths and block widths share one index");

template <int MODE>
__device__ __forceinline__ void fast_radial(const SymmArgs& A, const DevModel& M, int a, const FastSmem& sm, const float4* tv,
                            const float* sd, float* sP, float* out) {
    const int lane = threadIdx.x % kWave, S = M.S;
    for (int b = 0; b < S; ++b) {
        const RadBlock rb = M.rad[a * S + b];
        if (rb.n == 0) continue;
        const int s0 = sm.seg[b], s1 = sm.seg[b + 1];
        if (rb.name == RAD_GAUSSIAN && MODE != 1 && rb.n <= 16) {
            const int W = rb.n <= 8 ? 8 : 16;
            if ((s1 - s0) * W <= kPairPasses * kWave) {
                radial_gauss_pairs<MODE>(A, rb, sm, s0, s1, W, tv, out);
                continue;
            }
        }
        if (rb.name == RAD_GAUSSIAN) {
            // eight per pass for blocks of at most eight functions, else sixteen
            // (the tangent keeps sixteen: a second copy raises its register count)
            if (MODE != 2 && rb.n <= 8) radial_gauss<MODE, 8>(A, rb, sm, s0, s1, tv, sd, sP, out);
            else radial_gauss<MODE, 16>(A, rb, sm, s0, s1, tv, sd, sP, out);
            continue;
        }
        if (MODE == 1) {
            for (int J = s0 + lane; J < s1; J += kWave) {
                const float4 gj = sm.g[J];
                const float2 fg = sm.fg[J];
                const float fc = fg.x, gc = fg.y;
                float amp = 0.0f;
                for (int m = 0; m < rb.n; ++m) {
                    float v, d;
                    radial_fd(rb.name, A.rad_eta[rb.par + m], A.rad_rs[rb.par + m], sm.r[J], fc, gc, v, d);
                    amp += sd[rb.goff + m] * d;
                }
                sP[3 * J] += amp * gj.x;
                sP[3 * J + 1] += amp * gj.y;
                sP[3 * J + 2] += amp * gj.z;
            }
            continue;
        }
        // other families: one function at a time, plain wave sums
        for (int m = 0; m < rb.n; ++m) {
            float acc = 0.0f;
            for (int J = s0 + lane; J < s1; J += kWave) {
                const float r = sm.r[J];
                const float2 fg = sm.fg[J];
                const float fc = fg.x, gc = fg.y;
                float v, d;
                radial_fd(rb.name, A.rad_eta[rb.par + m], A.rad_rs[rb.par + m], r, fc, gc, v, d);
                acc += MODE == 0 ? v : d * tv[J].w;
            }
            acc = wave_sum(acc);
            if (lane == 0) out[rb.goff + m] = acc;
        }
    }
}

// mode 0: G, 1: adjoint P, 2: tangent v; every angular block has the grid shape NG x NK
template <int MODE, int NG, int NK>
__global__ __launch_bounds__(64) void k_fast(SymmArgs A) {
    extern __shared__ float4 smem4[];
    const int i = blockIdx.x, lane = threadIdx.x;
    if (i >= A.N) return;
    const DevModel& M = *A.dm;
    const int a = A.species[i], o = A.off[i];
    int n = A.off[i + 1] - o;
    const int S = M.S, NP = M.NP, ldg = A.ldg, maxn = A.maxn;
    FastSmem sm;
    sm.g = smem4;
    sm.ef = sm.g + maxn;
    sm.efd = sm.ef + maxn;
    float4* tv = sm.efd + (MODE == 0 ? 0 : maxn);                // [maxn] (mode 2)
    sm.fg = reinterpret_cast<float2*>(tv + (MODE == 2 ? maxn : 0));
    sm.r = reinterpret_cast<float*>(sm.fg + maxn);
    sm.canon = reinterpret_cast<int*>(sm.r + maxn);
    sm.seg = sm.canon + maxn;
    sm.extra = reinterpret_cast<float*>(sm.seg + 16);
    float* rowbuf = sm.extra;                                   // [ldg] output row (modes 0, 2) / dE/dG (mode 1)
    float* sP = sm.extra + ldg;                                 // [maxn][3] (mode 1)
    n = fast_load(A, M, i, a, o, n, sm, MODE != 0, MODE == 1);   // n: neighbours within rc
    if (MODE == 1) {
        for (int m = lane; m < ldg; m += kWave) rowbuf[m] = A.dEdG[(size_t)i * ldg + m];
        for (int t = lane; t < 3 * n; t += kWave) sP[t] = 0.0f;
    } else {
        for (int m = lane; m < ldg; m += kWave) rowbuf[m] = 0.0f;
    }
    __syncthreads();
    if (MODE == 2) {
        // per neighbour tangent t_j = u_i - u_j and r^_j . t_j, species-sorted
        for (int J = lane; J < n; J += kWave) {
            const int j = A.nidx[o + sm.canon[J]];
            const float tx = A.u[3 * i] - A.u[3 * j], ty = A.u[3 * i + 1] - A.u[3 * j + 1],
                        tz = A.u[3 * i + 2] - A.u[3 * j + 2];
            const float4 gq = sm.g[J];
            tv[J] = make_float4(tx, ty, tz, gq.x * tx + gq.y * ty + gq.z * tz);
        }
        __syncthreads();
    }
    fast_radial<MODE>(A, M, a, sm, tv, rowbuf, sP, rowbuf);
    __syncthreads();
    for (int b = 0; b < S; ++b) {
        for (int c = b; c < S; ++c) {
            const AngBlock& B = M.ang[a * NP + pair_idx(b, c)];
            if (B.n == 0) continue;
            const int sb = sm.seg[b], nb = sm.seg[b + 1] - sb;
            const int sc = sm.seg[c], nc = sm.seg[c + 1] - sc;
            const bool tri = (b == c);
            if (tri ? nb < 2 : (nb == 0 || nc == 0)) continue;
            const float* uie = M.uieta2[a];
            if (B.name == ANG_GAUSS) {
                if (MODE == 1) fast_block_adj<NG, NK, true>(B, uie, sm, sb, nb, sc, nc, tri, rowbuf, sP);
                else fast_block_flat<NG, NK, MODE == 0 ? 0 : 1, true>(B, uie, sm, sb, nb, sc, nc, tri, tv, rowbuf);
            } else {
                if (MODE == 1) fast_block_adj<NG, NK, false>(B, uie, sm, sb, nb, sc, nc, tri, rowbuf, sP);
                else fast_block_flat<NG, NK, MODE == 0 ? 0 : 1, false>(B, uie, sm, sb, nb, sc, nc, tri, tv, rowbuf);
            }
            __syncthreads();
        }
    }
    if (MODE == 1) {
        for (int J = lane; J < n; J += kWave) {
            const int t = sm.canon[J];
            A.P[3 * ((size_t)o + t)] = sP[3 * J];
            A.P[3 * ((size_t)o + t) + 1] = sP[3 * J + 1];
            A.P[3 * ((size_t)o + t) + 2] = sP[3 * J + 2];
        }
    } else {
        float* out = (MODE == 0 ? A.G : A.v) + (size_t)i * ldg;
        for (int m = lane; m < ldg; m += kWave) out[m] = rowbuf[m];
    }
}

// =========================================================== MOMENT form ====
//
// For GAUSS angular blocks with integer zeta <= 5 the triplet sum factorises
// exactly.  With e_u(r) = exp(-r^2/eta_u^2) fc(r) and c = r^_j . r^_k,
//   (1/2 + lambda c / 2)^zeta = sum_l a_l P_l(c),
//   P_l(c) = sum_m Y_lm(r^_j) Y_lm(r^_k)                 (harm_dev.h)
// so a block (species b, species c, width u) needs only the per-species
// moments T_b[u][lm] = sum_{j in b} e_u(r_j) Y_lm(r^_j) and
// D_b[u] = sum_{j in b} e_u(r_j)^2:
//   A_l = sum_m T_b T_c                                  (b != c)
//   A_l = (sum_m T_b T_b - D_b) / 2                      (b == c: pairs j < k)
//   G(u, lambda, zeta) = sum_l a_l A_l.
// Work per atom is O(n M) with M = (Z+1)^2 functions instead of O(n^2)
// triplets.  The adjoint differentiates the same chain: dE/dT_b from the block
// contractions, then per neighbour the function sum_lm dE/dT_b[u][lm] Y_lm(r^)
// and its gradient.  The tangent (force-loss second backward) is the
// forward-mode derivative.
// The kernels issue vector instructions most of the time, so the number of
// functions is what counts: the harmonics are the (Z+1)^2 independent functions
// among the (Z+1)(Z+2)(Z+3)/6 monomials of the unit vector's components (25
// against 35 at zeta 4, 36 against 56 at zeta 5).  Their recurrences round more
// often than products of powers: in an FP32 emulation with exact widths one
// angular input rounds 1.3 (zeta 2) to 2.0 times (zeta 5) as much as from
// monomials.  With the exponentials of the widths the inputs' errors against
// FP64, harmonics to monomials, are 1.09 (zeta 1) and 0.73 (zeta 4) on water, 0.98
// and 0.91 (zeta 1, 2) on Li/P/S, 1.00, 1.01 and 0.91 (zeta 1, 2, 5) on argon.
// Monomials against
// harmonics, MI355X: E+F of 32 preconditioned water boxes (FP64 moments) 265 ->
// 216 us, 512 uneven water cells 4.18 -> 3.94 ms, five MD steps of 1 M atoms
// 103.0 -> 97.2 ms, 64 water boxes and Li/P/S training unchanged.

// moment_atom's chunk of function rows (adjoint: set by the host, 64 or 32; fused:
// 32; tangent: every neighbour at once while a row is short, up to degree 2, else 32), and the
// floats of the region that holds them (it also holds the cutoff pairs, two
// floats per neighbour, before the rows are needed).  Mode 1 here is the adjoint
// that recomputes the moments: it serves calls whose geometry no G call has seen.
constexpr int kPwRows = 64;
// adjoint: dE/dT entries per lane held in registers while they replace the moments
constexpr int kUbRegs = 8;
__host__ __device__ inline int pw_chunk(int mode, int maxn, int pws, int grows) {
    return mode == 2 && pws <= 32 ? maxn : (mode == 1 ? grows : kPwRows / 2);
}
__host__ __device__ inline int pw_floats(int mode, int maxn, int pws, int grows) {
    const int rows = pw_chunk(mode, maxn, pws, grows);
    if (mode == 3) {                                // fused: also the adjoint vectors and network vectors
        const int m = rows * pws > 3 * maxn ? rows * pws : 3 * maxn;
        return m > 3 * kVecMaxWidth ? m : 3 * kVecMaxWidth;
    }
    return rows * pws > 2 * maxn ? rows * pws : 2 * maxn;
}

__device__ __forceinline__ int pair_of(int b, int c) { return b <= c ? c * (c + 1) / 2 + b : b * (b + 1) / 2 + c; }

// groups of lanes sharing a reduction of n outputs (n <= 16: four groups of
// 16 lanes, <= 32: two of 32, else one of 64)
__device__ __forceinline__ int lane_groups(int n) { return n <= 16 ? 4 : (n <= 32 ? 2 : 1); }

// The atom's network on its own wavefront (fused E+F; ANN::fpbp + DODZ::grad,
// src/ml/nn.cpp:1367-1389, 1801-1830): rowbuf holds the G row on entry and
// dE/dG on exit (zero past the species' inputs); the atom energy goes to
// A.Eatom.  Lanes over a layer's outputs, its reduction split over up to four
// lane groups joined by butterflies; the layer's inputs are broadcast LDS
// reads, the weights coalesced reads of the row tables (forward: rows of W,
// backward: rows of W^T, net_dev.h layout).  nb: [3][kVecMaxWidth] LDS floats.
__device__ __forceinline__ void fused_net(const SymmArgs& A, const NetDesc& D, int i, float* rowbuf, float* nb) {
    const int lane = threadIdx.x % kWave;
    const int L = D.nlayer, nin = D.nin, ldg = A.ldg;
    const float* iw = A.inpw + D.inoff;
    const float* ib = A.inpb + D.inoff;
    for (int k = lane; k < nin; k += kWave) rowbuf[k] = iw[k] * (rowbuf[k] + ib[k]);
    wave_sync();
    const float* x = rowbuf;
    int ni = nin;
    float sp[kMaxLayers - 1];                               // sigma' of the lane's neuron per hidden layer
#pragma unroll
    for (int l = 0; l < kMaxLayers - 1; ++l) sp[l] = 0.0f;
#pragma unroll
    for (int l = 0; l < kMaxLayers - 1; ++l) {
        if (l >= L - 1) break;
        const int no = D.nodes[l], ps = D.wcs[l];
        const float* W = A.wchunk + D.wcf[l];
        const float* b = A.wchunk + D.wcb[l];
        const int G = lane_groups(no), gw = kWave / G;
        const int j = lane % gw, grp = lane / gw, jj = min(j, no - 1);
        const int kper = (ni + G - 1) / G, k0 = grp * kper, k1 = min(ni, k0 + kper);
        float acc = 0.0f;
#pragma unroll 4
        for (int k = k0; k < k1; ++k) acc += W[k * ps + jj] * x[k];
        for (int m = gw; m < kWave; m <<= 1) acc += __shfl_xor(acc, m);
        float z[1] = {acc + b[jj]}, av[1], dv[1], d2[1];
        act_many<false, 1>(D.neuron, D.c, z, av, dv, d2);
        sp[l] = dv[0];
        float* h = nb + (l & 1) * kVecMaxWidth;
        if (grp == 0 && j < no) h[j] = av[0];
        wave_sync();
        x = h;
        ni = no;
    }
    // linear output neuron
    const float* WL = A.wchunk + D.wco;                     // weights, then (at a multiple of 4) the bias
    float part = 0.0f;
    for (int m = lane; m < ni; m += kWave) part += WL[m] * x[m];
    part = wave_sum(part);
    if (lane == 0) A.Eatom[i] = D.outb + D.outw * (WL[vec_pad4(ni)] + part);
    wave_sync();                                            // every lane is done with x
    if (L == 1) {
        for (int k = lane; k < ldg; k += kWave) rowbuf[k] = k < nin ? D.outw * WL[k] * iw[k] : 0.0f;
        wave_sync();
        return;
    }
    // g of the last hidden layer (its lanes hold sigma' for neuron lane % gw)
    float* dc = nb + 2 * kVecMaxWidth;
    float* dn = nb;
    {
        const int G = lane_groups(ni), gw = kWave / G, j = lane % gw;
        float spl = 0.0f;
#pragma unroll
        for (int q = 0; q < kMaxLayers - 1; ++q)
            if (q == L - 2) spl = sp[q];
        if (lane < gw && j < ni) dc[j] = D.outw * WL[j] * spl;
    }
    wave_sync();
    // hidden layers: g_{l-1}[k] = sigma'_{l-1}[k] sum_j W_l[k][j] g_l[j], lanes over k
#pragma unroll
    for (int l = kMaxLayers - 2; l >= 1; --l) {
        if (l > L - 2) continue;
        const int no = D.nodes[l], nil = D.nodes[l - 1], pst = D.wts[l];
        const float* WT = A.wtrans + D.wtf[l];
        const int G = lane_groups(nil), gw = kWave / G;
        const int k = lane % gw, grp = lane / gw, kk = min(k, nil - 1);
        const int jper = (no + G - 1) / G, j0 = grp * jper, j1 = min(no, j0 + jper);
        float acc = 0.0f;
#pragma unroll 4
        for (int j = j0; j < j1; ++j) acc += WT[j * pst + kk] * dc[j];
        for (int m = gw; m < kWave; m <<= 1) acc += __shfl_xor(acc, m);
        if (grp == 0 && k < nil) dn[k] = acc * sp[l - 1];
        wave_sync();
        float* t = dc;
        dc = dn;
        dn = t;
    }
    // input layer: dE/dG[k] = inpw[k] sum_j W_0[k][j] g_0[j], blocks of up to 64 inputs
    {
        const int no = D.nodes[0], pst = D.wts[0];
        const float* WT = A.wtrans + D.wtf[0];
        for (int kb = 0; kb < nin; kb += kWave) {
            const int nk = min(kWave, nin - kb);
            const int G = lane_groups(nk), gw = kWave / G;
            const int k = kb + lane % gw, grp = lane / gw, kk = min(k, nin - 1);
            const int jper = (no + G - 1) / G, j0 = grp * jper, j1 = min(no, j0 + jper);
            float acc = 0.0f;
#pragma unroll 4
            for (int j = j0; j < j1; ++j) acc += WT[j * pst + kk] * dc[j];
            for (int m = gw; m < kWave; m <<= 1) acc += __shfl_xor(acc, m);
            if (grp == 0 && lane % gw < nk) rowbuf[k] = acc * iw[k];
        }
        for (int k = nin + lane; k < ldg; k += kWave) rowbuf[k] = 0.0f;
        wave_sync();
    }
}

// One wavefront per atom with its own LDS slice (smem4); no block barriers, so
// the waves of a workgroup are independent.
template <int MODE, int Z>
__device__ __forceinline__ void moment_atom(const SymmArgs& A, const int i, float4* smem4) {
    static_assert(MODE >= 1 && MODE <= 3, "adjoint, tangent, fused");
    constexpr int NM = nharm(Z);
    constexpr int ZP = Z + 1;
    constexpr int PWS = (NM * (MODE == 2 ? 2 : 1)) | 1;      // function values per neighbour, odd stride
    constexpr int U4 = kMaxUnionEta;
    constexpr int NW = NM <= 4 ? 4 : (NM <= 16 ? 16 : (NM <= 32 ? 32 : kWave));   // lanes of one group
    constexpr int NG = kWave / NW;                           // lane groups over the neighbours
    constexpr bool FUSED = MODE == 3;                        // G, network and adjoint of the atom
    constexpr bool ADJ = MODE == 1 || FUSED;                 // per-slot adjoint vectors written
    constexpr int GM = FUSED ? 0 : MODE;                     // mode of the basis phase
    const int lane = threadIdx.x % kWave;
    const DevModel& Mo = *A.dm;
    const int a = A.species[i], o = A.off[i];
    int n = A.off[i + 1] - o;
    const int S = Mo.S, NP = Mo.NP, ldg = A.ldg, maxn = A.maxn;
    FastSmem sm;
    sm.g = smem4;
    sm.ef = sm.g + maxn;
    sm.efd = sm.ef + maxn;
    float4* tv = sm.efd + maxn;
    sm.r = reinterpret_cast<float*>(tv + (MODE == 2 ? maxn : 0));
    int* const after_r = reinterpret_cast<int*>(sm.r + maxn);
    sm.canon = ADJ ? after_r : nullptr;                         // the adjoint's slot map
    sm.seg = after_r + (ADJ ? maxn : 0);
    sm.extra = reinterpret_cast<float*>(sm.seg + 16);
    float* rowbuf = sm.extra;                                   // [ldg]
    // [maxn][3] adjoint vectors (mode 1; fused: they share the power rows'
    // region, whose rows are dead once the moments are summed)
    float* sP = rowbuf + ldg + (FUSED ? 2 * maxn : 0);
    const int TS = S * U4 * NM;                                 // moments per atom
    float* fgr = rowbuf + ldg;                                  // fused: [maxn] cutoff pairs of their own
    float* pw = FUSED ? sP : sP + (MODE == 1 ? 3 * maxn : 0);  // [pw_chunk][PWS] (one chunk of neighbours)
    float* T = pw + pw_floats(MODE, maxn, PWS, A.grows);      // [S][U4][NM]
    float* dT = T + S * U4 * NM;                                // [S][U4][NM] (mode 2)
    float* D = dT + (MODE == 2 ? S * U4 * NM : 0);              // [S][U4]
    float* dD = D + S * U4;                                     // [S][U4] (mode 2: dD, mode 1: dE/dD)
    float* Am = dD + S * U4;                                    // [NP][U4][ZP]
    // adjoint: dE/dT overwrites the moments when it fits a few registers per lane
    const bool ub_in_T = S * NM * U4 <= kUbRegs * kWave;
    float* Ub = ub_in_T ? T : Am + NP * U4 * ZP;               // [S][NM][U4] (mode 1)
    float* nb = pw;                                             // fused: [3][kVecMaxWidth] network vectors (function rows' region)
    // cutoffs live in the power rows until the radial part is done (fused: the
    // adjoint's radial part runs after the moments, so they have their own rows)
    sm.fg = reinterpret_cast<float2*>(FUSED ? fgr : pw);

    n = fast_load(A, Mo, i, a, o, n, sm, true, ADJ, MODE == 2 ? tv : nullptr);
    if (MODE == 1) {
        for (int m = lane; m < ldg; m += kWave) rowbuf[m] = A.dEdG[(size_t)i * ldg + m];
        for (int t = lane; t < 3 * n; t += kWave) sP[t] = 0.0f;
    } else {
        for (int m = lane; m < ldg; m += kWave) rowbuf[m] = 0.0f;
    }
    wave_sync();
    fast_radial<GM>(A, Mo, a, sm, tv, rowbuf, sP, rowbuf);
    wave_sync();
    // function values of the unit vector (and, for the tangent, their derivatives
    // along the projected direction (t - r^ (r^.t)) / r) of neighbours c0 .. c1-1,
    // at most pw_chunk, into the chunk rows (the moment loop below walks each
    // species segment in such chunks, so for the adjoint the rows take a
    // fixed slice of LDS instead of one row per neighbour)
    auto function_rows = [&](int c0, int c1) {
        for (int J = c0 + lane; J < c1; J += kWave) {
            const float4 gq = sm.g[J];
            float* row = pw + (size_t)(J - c0) * PWS;
            float C[ZP], Sn[ZP], q[qidx(Z, Z) + 1], y[NM];
            harm_factors<Z, float>(gq.x, gq.y, gq.z, C, Sn, q);
            harm_values<Z, float>(C, Sn, q, y);
#pragma unroll
            for (int f = 0; f < NM; ++f) row[f] = y[f];
            if (MODE == 2) {
                const float4 t4 = tv[J];
                harm_along<Z, float>(C, Sn, q, (t4.x - gq.x * t4.w) * gq.w, (t4.y - gq.y * t4.w) * gq.w,
                                     (t4.z - gq.z * t4.w) * gq.w, y);
#pragma unroll
                for (int f = 0; f < NM; ++f) row[NM + f] = y[f];
            }
        }
    };
    wave_sync();
    // moments T_b[u][f]: lane = (function, group); groups stride the neighbours
    {
        const int al = lane % NW, grp = lane / NW;
        const bool act = al < NM;
        for (int b = 0; b < S; ++b) {
            const int s0 = sm.seg[b], s1 = sm.seg[b + 1];
            float acc[U4], dacc[U4];
#pragma unroll
            for (int u = 0; u < U4; ++u) { acc[u] = 0.0f; dacc[u] = 0.0f; }
            // one neighbour of the segment: T[u][f] += e_u(r) Y_f(r^)
            auto step = [&](const float* row, int J) {
                const float yv = row[al];
                const float4 e4 = sm.ef[J];
                acc[0] += e4.x * yv; acc[1] += e4.y * yv; acc[2] += e4.z * yv; acc[3] += e4.w * yv;
                if (MODE == 2) {
                    const float dy = row[NM + al];
                    const float4 f4 = sm.efd[J];
                    const float wm = tv[J].w * yv;
                    dacc[0] += f4.x * wm + e4.x * dy;
                    dacc[1] += f4.y * wm + e4.y * dy;
                    dacc[2] += f4.z * wm + e4.z * dy;
                    dacc[3] += f4.w * wm + e4.w * dy;
                }
            };
            const int chunk = pw_chunk(MODE, maxn, PWS, A.grows);
            for (int c0 = s0; c0 < s1; c0 += chunk) {
                const int c1 = min(c0 + chunk, s1);
                wave_sync();                                    // the previous chunk's rows are read
                function_rows(c0, c1);
                wave_sync();
                if (act) {
                    int J = c0 + grp;
                    // four neighbours per trip: their rows sit at fixed offsets
                    // from one address, so the loads use immediate offsets and overlap
                    for (; J + 3 * NG < c1; J += 4 * NG) {
                        const float* row = pw + (size_t)(J - c0) * PWS;
                        step(row, J);
                        step(row + NG * PWS, J + NG);
                        step(row + 2 * NG * PWS, J + 2 * NG);
                        step(row + 3 * NG * PWS, J + 3 * NG);
                    }
                    for (; J < c1; J += NG) step(pw + (size_t)(J - c0) * PWS, J);
                }
            }
            // butterflies over the groups, whose width is a power of two
#pragma unroll
            for (int bit = NW; bit < kWave; bit <<= 1)
#pragma unroll
                for (int u = 0; u < U4; ++u) {
                    acc[u] += __shfl_xor(acc[u], bit);
                    if (MODE == 2) dacc[u] += __shfl_xor(dacc[u], bit);
                }
            if (lane < NM) {
#pragma unroll
                for (int u = 0; u < U4; ++u) {
                    T[(b * U4 + u) * NM + al] = acc[u];
                    if (MODE == 2) dT[(b * U4 + u) * NM + al] = dacc[u];
                }
            }
        }
        // diagonal sums D_b[u] (mode 2 also their tangent): lanes over the
        // segment, one transposing reduction of the four widths
        if (MODE != 1) {
            for (int b = 0; b < S; ++b) {
                float d4[U4], t4[U4];
#pragma unroll
                for (int u = 0; u < U4; ++u) { d4[u] = 0.0f; t4[u] = 0.0f; }
                for (int J = sm.seg[b] + lane; J < sm.seg[b + 1]; J += kWave) {
                    const float4 e4 = sm.ef[J];
                    d4[0] += e4.x * e4.x; d4[1] += e4.y * e4.y; d4[2] += e4.z * e4.z; d4[3] += e4.w * e4.w;
                    if (MODE == 2) {
                        const float4 f4 = sm.efd[J];
                        const float w2 = 2.0f * tv[J].w;
                        t4[0] += w2 * e4.x * f4.x; t4[1] += w2 * e4.y * f4.y;
                        t4[2] += w2 * e4.z * f4.z; t4[3] += w2 * e4.w * f4.w;
                    }
                }
                int idx;
                const float sd = wave_sum_multi<U4>(d4, idx);
                if ((lane & (kWave / U4 - 1)) == 0) D[b * U4 + idx] = sd;
                if (MODE == 2) {
                    const float st = wave_sum_multi<U4>(t4, idx);
                    if ((lane & (kWave / U4 - 1)) == 0) dD[b * U4 + idx] = st;
                }
            }
        }
    }
    wave_sync();
    // block contractions (modes 2, 3) or their adjoint seeds (mode 1; mode 3
    // after its network)
    auto adjoint_seeds = [&]() {
        // lanes over (pair, width, power) of every block at once; each lane loads
        // all of its output indices and coefficients before using any, so the
        // block descriptors cost a few rounds of memory latency, not one per term
        for (int it = lane; it < NP * U4 * ZP; it += kWave) {
            const int p = it / (U4 * ZP), u = (it / ZP) % U4, m = it % ZP;
            const AngBlock& B = Mo.ang[a * NP + p];
            const int nk = min(max(B.nk, 0), kGridK), goff = B.goff;
            const bool use = B.n > 0 && u < B.ng;
            // u * nk + k < kGridG * kGridK for every k < kGridK (u < kGridG, nk <= kGridK):
            // entries past nk are read but not used
            int om[kGridK];
            float mc[kGridK];
#pragma unroll
            for (int k = 0; k < kGridK; ++k) {
                om[k] = B.outm[u * nk + k];
                mc[k] = B.lcoef[k][m];
            }
            float s = 0.0f;
            if (use) {
#pragma unroll
                for (int k = 0; k < kGridK; ++k)
                    if (k < nk) s += rowbuf[goff + om[k]] * mc[k];
            }
            Am[it] = s;
        }
    };
    if (MODE == 1) adjoint_seeds();
    for (int it = lane; MODE != 1 && it < NP * U4 * ZP; it += kWave) {
        const int p = it / (U4 * ZP), u = (it / ZP) % U4, m = it % ZP;
        int c = 0;
        while ((c + 1) * (c + 2) / 2 <= p) ++c;
        const int b = p - c * (c + 1) / 2;
        float s = 0.0f;
        {
            const float* Tb = T + (b * U4 + u) * NM;
            const float* Tc = T + (c * U4 + u) * NM;
            const float* dTb = dT + (b * U4 + u) * NM;
            const float* dTc = dT + (c * U4 + u) * NM;
            // degree m has 2m + 1 functions; every lane runs the length of the
            // highest degree with the surplus terms weighted 0, so all loads are
            // issued before the first product instead of one dependent round per
            // function
            constexpr int QD = 2 * Z + 1;
            const int q0 = m * m, q1 = q0 + 2 * m + 1;
#pragma unroll
            for (int j = 0; j < QD; ++j) {
                const int q = min(q0 + j, NM - 1);
                const float w = q0 + j < q1 ? 1.0f : 0.0f;
                s += GM == 0 ? (w * Tb[q]) * Tc[q] : w * (dTb[q] * Tc[q] + Tb[q] * dTc[q]);
            }
            if (b == c) s = 0.5f * (s - (GM == 0 ? D[b * U4 + u] : dD[b * U4 + u]));
        }
        Am[it] = s;
    }
    wave_sync();
    if (MODE != 1) {
        // lanes over (pair, width, combination) of every block at once, loads
        // issued before the guards that use them
        for (int it = lane; it < NP * kGridG * kGridK; it += kWave) {
            const int p = it / (kGridG * kGridK), g = (it / kGridK) % kGridG, k = it % kGridK;
            const AngBlock& B = Mo.ang[a * NP + p];
            const int nk = min(max(B.nk, 0), kGridK), goff = B.goff;
            const bool use = B.n > 0 && g < B.ng && k < nk;
            const int om = B.outm[g * nk + k];   // < kGridG * kGridK; used only when use
            float mc[ZP];
#pragma unroll
            for (int m = 0; m < ZP; ++m) mc[m] = B.lcoef[k][m];
            if (use) {
                float v = 0.0f;
#pragma unroll
                for (int m = 0; m < ZP; ++m) v += mc[m] * Am[(p * U4 + g) * ZP + m];
                rowbuf[goff + om] = v;
            }
        }
        wave_sync();
        if (!FUSED) {
            float* out = A.v + (size_t)i * ldg;
            for (int m = lane; m < ldg; m += kWave) out[m] = rowbuf[m];
            return;
        }
    }
    if (FUSED) {
        // the atom's G row in rowbuf: its energy and dE/dG (in place), then the
        // radial adjoint and the angular seeds as the adjoint kernel forms them
        fused_net(A, Mo.net[a], i, rowbuf, nb);
        for (int t = lane; t < 3 * n; t += kWave) sP[t] = 0.0f;
        wave_sync();
        fast_radial<1>(A, Mo, a, sm, tv, rowbuf, sP, rowbuf);
        wave_sync();
        adjoint_seeds();
        wave_sync();
    }
    // adjoint: dE/dT_b[alpha][u] and dE/dD_b[u]
    auto dEdT = [&](int it) {
        const int b = it / (NM * U4), al = (it / U4) % NM, u = it % U4;
        int m = 0;   // degree of function al
#pragma unroll
        for (int mm = 1; mm <= Z; ++mm) m += al >= mm * mm ? 1 : 0;
        float s = 0.0f;
        for (int c = 0; c < S; ++c) s += Am[(pair_of(b, c) * U4 + u) * ZP + m] * T[(c * U4 + u) * NM + al];
        return s;
    };
    if (ub_in_T) {
        // every lane's entries in registers, then written over the moments
        float ub[kUbRegs];
#pragma unroll
        for (int h = 0; h < kUbRegs; ++h) {
            const int it = lane + h * kWave;
            ub[h] = it < S * NM * U4 ? dEdT(it) : 0.0f;
        }
        wave_sync();
#pragma unroll
        for (int h = 0; h < kUbRegs; ++h) {
            const int it = lane + h * kWave;
            if (it < S * NM * U4) Ub[it] = ub[h];
        }
    } else {
        for (int it = lane; it < S * NM * U4; it += kWave) Ub[it] = dEdT(it);
    }
    if (lane < S * U4) {
        const int b = lane / U4, u = lane % U4;
        float s = 0.0f;
        for (int m = 0; m < ZP; ++m) s += Am[(pair_of(b, b) * U4 + u) * ZP + m];
        dD[lane] = -0.5f * s;
    }
    wave_sync();
    // per neighbour: the radial and angular derivatives of sum_u e_u sum_f dE/dT[f][u] Y_f
    for (int J = lane; J < n; J += kWave) {
        int b = 0;
        while (b + 1 < S && J >= sm.seg[b + 1]) ++b;
        const float4 gq = sm.g[J];
        const float4 e4 = sm.ef[J], f4 = sm.efd[J];
        float Qd, g0, g1, g2;
        harm_adjoint<Z>(gq.x, gq.y, gq.z, e4, f4, reinterpret_cast<const float4*>(Ub + b * NM * U4), Qd, g0, g1, g2);
        const float dd = 2.0f * (dD[b * U4] * e4.x * f4.x + dD[b * U4 + 1] * e4.y * f4.y +
                                 dD[b * U4 + 2] * e4.z * f4.z + dD[b * U4 + 3] * e4.w * f4.w);
        const float rg = gq.x * g0 + gq.y * g1 + gq.z * g2;
        const float radial = Qd + dd;
        sP[3 * J] += radial * gq.x + (g0 - gq.x * rg) * gq.w;
        sP[3 * J + 1] += radial * gq.y + (g1 - gq.y * rg) * gq.w;
        sP[3 * J + 2] += radial * gq.z + (g2 - gq.z * rg) * gq.w;
    }
    wave_sync();
    for (int J = lane; J < n; J += kWave) {
        const int t = sm.canon[J];
        A.P[3 * ((size_t)o + t)] = sP[3 * J];
        A.P[3 * ((size_t)o + t) + 1] = sP[3 * J + 1];
        A.P[3 * ((size_t)o + t) + 2] = sP[3 * J + 2];
    }
}

// Adjoint with stored moments.  One wavefront serves K consecutive atoms; its
// lanes run over the atoms' list entries in list order, which are contiguous,
// so every entry's vector stays in registers from the load to the store: no
// regrouping by species and no LDS row per neighbour.  What differs between
// entries (centre and neighbour species) is an LDS table per (atom, species):
// the radial functions with their dE/dG and the moment adjoints dE/dT.
//   1. dE/dG rows and moments of the K atoms into LDS;
//   2. per block, width and degree, A = sum over functions of dE/dG times the
//      Legendre coefficient; dE/dT[b][f] = sum_c A(b, c) T[c][f];
//   3. lanes over entries: cutoff, radial sum, harm_adjoint, store.
// The entries of two atoms fill the 64 lanes better than one atom's (water: 85
// entries take two passes, 170 take three); K comes from the batch
// (adj_atoms).  LDS does not depend on the widest row, so the registers
// alone set the number of resident wavefronts, also for lists with a skin.
// Bound by vector issue: 1,410 vector instructions per atom (water, two atoms per
// wavefront, counters) of which the vector units are busy 74 % of the time, LDS
// waits below 1 %.  Measured against the form with one LDS row per neighbour:
// 1,048,576 atoms, list with a skin, 8.57 -> 3.03 ms; 273,561 atoms 1285 -> 555 us;
// 12,288 atoms 54 -> 35 us; Li/P/S, 21,872 atoms, 67 -> 35 us.
constexpr int kAdjAtoms = 2;

// float4 entries of the wavefront's LDS slice (layout at the top of adjoint_wave)
__host__ __device__ inline int adj_units(int K, int Z, int S, int NP, int nrs, int ldg) {
    const int NM = nharm(Z), U4 = kMaxUnionEta;
    return K * S * (NM | 1) + K * S * nrs + K * S + K * S * NM + K * (ldg / 4) + (K * NP * U4 * (Z + 1) + 3) / 4;
}

template <int Z>
__device__ __forceinline__ void adjoint_wave(const SymmArgs& A, const int i0, const int K, float4* smem4) {
    constexpr int NM = nharm(Z), NS = NM | 1, ZP = Z + 1, U4 = kMaxUnionEta;
    const int lane = threadIdx.x % kWave;
    const DevModel& Mo = *A.dm;
    const int S = Mo.S, NP = Mo.NP, ldg = A.ldg, nrs = A.nrs;
    float4* W = smem4;                                          // [K][S][NS] dE/dT, widths in the components
    float4* R = W + K * S * NS;                                 // [K][S][nrs] radial: eta, rs, dE/dG, dE/dG eta
    float4* dD = R + K * S * nrs;                               // [K][S] dE/dD
    float* T = reinterpret_cast<float*>(dD + K * S);            // [K][S][NM][U4]
    float* row = T + K * S * U4 * NM;                           // [K][ldg]
    float* Am = row + K * ldg;                                  // [K][NP][U4][ZP]
    int o[kAdjAtoms + 1], sp[kAdjAtoms];
#pragma unroll
    for (int q = 0; q <= kAdjAtoms; ++q) o[q] = A.off[i0 + min(q, K)];
#pragma unroll
    for (int q = 0; q < kAdjAtoms; ++q) sp[q] = A.species[i0 + min(q, K - 1)];
    const int s_end = o[kAdjAtoms];
    // the first entries' loads are in flight while the tables are built
    int s = o[0] + lane;
    float4 gn = make_float4(0.f, 0.f, 0.f, 0.f);
    int bn = 0;
    if (s < s_end) {
        gn = A.geo[s];
        bn = A.nsp[s];
    }
    {
        const float4* gT = reinterpret_cast<const float4*>(A.Tin + (size_t)i0 * S * U4 * NM);
        float4* lT = reinterpret_cast<float4*>(T);
        for (int x = lane; x < K * S * NM; x += kWave) lT[x] = gT[x];
        // the caller's rows: no alignment beyond a float's
        for (int x = lane; x < K * ldg; x += kWave) row[x] = A.dEdG[(size_t)i0 * ldg + x];
    }
    wave_sync();
    auto spec = [&](int q) {                                    // species of atom q, without a register array index
        int a = sp[0];
#pragma unroll
        for (int k = 1; k < kAdjAtoms; ++k)
            if (q == k) a = sp[k];
        return a;
    };
    // radial tables (functions past a block's own carry dE/dG = 0)
    for (int x = lane; x < K * S * nrs; x += kWave) {
        const int m = x % nrs, b = (x / nrs) % S, q = x / (nrs * S);
        const RadBlock rb = Mo.rad[spec(q) * S + b];
        float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < rb.n) {
            const float e = A.rad_eta[rb.par + m], g = row[q * ldg + rb.goff + m];
            t = make_float4(e, A.rad_rs[rb.par + m], g, g * e);
        }
        R[x] = t;
    }
    // angular seeds: lanes over (atom, pair, width, degree); every descriptor load
    // of a lane is issued before the first use
    for (int x = lane; x < K * NP * U4 * ZP; x += kWave) {
        const int l = x % ZP, u = (x / ZP) % U4, p = (x / (ZP * U4)) % NP, q = x / (ZP * U4 * NP);
        const AngBlock& B = Mo.ang[spec(q) * NP + p];
        const int nk = min(max(B.nk, 0), kGridK), goff = B.goff;
        const bool use = B.n > 0 && u < B.ng;
        int om[kGridK];
        float lc[kGridK];
#pragma unroll
        for (int k = 0; k < kGridK; ++k) {
            om[k] = B.outm[u * nk + k];                         // past nk: read, not used
            lc[k] = B.lcoef[k][l];
        }
        float v = 0.0f;
        if (use) {
#pragma unroll
            for (int k = 0; k < kGridK; ++k)
                if (k < nk) v += row[q * ldg + goff + om[k]] * lc[k];
        }
        Am[x] = v;
    }
    wave_sync();
    // dE/dT and dE/dD: lanes over (atom, species, function, width)
    for (int x = lane; x < K * S * NM * U4; x += kWave) {
        const int u = x % U4, f = (x / U4) % NM, b = (x / (U4 * NM)) % S, q = x / (U4 * NM * S);
        int l = 0;                                              // degree of function f
#pragma unroll
        for (int d = 1; d <= Z; ++d) l += f >= d * d ? 1 : 0;
        const float* Aq = Am + q * NP * U4 * ZP + u * ZP + l;
        const float* Tq = T + (q * S * NM + f) * U4 + u;
        float v = 0.0f;
        for (int c = 0; c < S; ++c) v += Aq[pair_of(b, c) * U4 * ZP] * Tq[c * U4 * NM];
        reinterpret_cast<float*>(W)[((q * S + b) * NS + f) * U4 + u] = v;
    }
    for (int x = lane; x < K * S * U4; x += kWave) {
        const int u = x % U4, b = (x / U4) % S, q = x / (U4 * S);
        const float* Aq = Am + q * NP * U4 * ZP + (pair_of(b, b) * U4 + u) * ZP;
        float v = 0.0f;
#pragma unroll
        for (int l = 0; l < ZP; ++l) v += Aq[l];
        reinterpret_cast<float*>(dD)[x] = -0.5f * v;
    }
    wave_sync();
    const float rc = Mo.rc, rci = Mo.rci, pirc = Mo.pirc;
    const int cut = Mo.cutoff;
    // 1/eta^2 of the atoms' widths (0 past them: their dE/dT is 0), in scalars: a lane
    // picks its atom's by a select instead of four loads per pass
    float ke[kAdjAtoms][U4];
#pragma unroll
    for (int q = 0; q < kAdjAtoms; ++q)
#pragma unroll
        for (int u = 0; u < U4; ++u) ke[q][u] = Mo.uieta2[sp[q]][u];
    for (; s < s_end; s += kWave) {
        const float4 gq = gn;
        const int b = bn;
        if (s + kWave < s_end) {
            gn = A.geo[s + kWave];
            bn = A.nsp[s + kWave];
        }
        int q = 0, a = sp[0];
#pragma unroll
        for (int k = 1; k < kAdjAtoms; ++k)
            if (s >= o[k]) { q = k; a = sp[k]; }
        float px = 0.0f, py = 0.0f, pz = 0.0f;
        if (gq.w <= rc) {                                       // entries beyond the cutoff (skin lists) get zero
            const float r = gq.w, ir = __builtin_amdgcn_rcpf(r);   // 1 ulp
            const float hx = gq.x * ir, hy = gq.y * ir, hz = gq.z * ir;
            float fc, gc;
            cutoff_fg(cut, rc, rci, pirc, r, fc, gc);
            const int qb = q * S + b;
            const float4* Rq = R + qb * nrs;
            float amp;
            if (A.rad_gauss) {
                // d/dr [e fc] = e (gc - 2 eta^2 (r - rs) fc)
                float se = 0.0f, sx = 0.0f;
#pragma unroll 4
                for (int m = 0; m < A.nrad; ++m) {
                    const float4 t = Rq[m];
                    const float x = t.x * (r - t.y), e = __expf(-x * x);
                    se += t.z * e;
                    sx += t.w * (x * e);
                }
                amp = se * gc - 2.0f * fc * sx;
            } else {
                const RadBlock rb = Mo.rad[a * S + b];
                amp = 0.0f;
                for (int m = 0; m < rb.n; ++m) {
                    const float4 t = Rq[m];
                    float v, d;
                    radial_fd(rb.name, t.x, t.y, r, fc, gc, v, d);
                    amp += t.z * d;
                }
            }
            float e[U4], d[U4];
#pragma unroll
            for (int u = 0; u < U4; ++u) {
                float k = ke[0][u];
#pragma unroll
                for (int x = 1; x < kAdjAtoms; ++x) k = q == x ? ke[x][u] : k;
                const float x = __expf(-k * r * r);
                e[u] = x * fc;
                d[u] = x * (-2.0f * r * k * fc + gc);
            }
            const float4 e4 = make_float4(e[0], e[1], e[2], e[3]), d4 = make_float4(d[0], d[1], d[2], d[3]);
            float rad, g0, g1, g2;
            harm_adjoint<Z>(hx, hy, hz, e4, d4, W + qb * NS, rad, g0, g1, g2);
            const float4 D = dD[qb];
            rad += amp + 2.0f * (D.x * e4.x * d4.x + D.y * e4.y * d4.y + D.z * e4.z * d4.z + D.w * e4.w * d4.w);
            const float rg = hx * g0 + hy * g1 + hz * g2;
            px = rad * hx + (g0 - hx * rg) * ir;
            py = rad * hy + (g1 - hy * rg) * ir;
            pz = rad * hz + (g2 - hz * rg) * ir;
        }
        A.P[3 * (size_t)s] = px;
        A.P[3 * (size_t)s + 1] = py;
        A.P[3 * (size_t)s + 2] = pz;
    }
}

// Grid dispatch of the stored-moment adjoint: every wavefront of a block takes
// A.atomsK consecutive atoms on its own LDS slice.
template <int Z>
__global__ __launch_bounds__(256) void k_adjoint(SymmArgs A) {
    extern __shared__ float4 smem_all[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i0 = (xcd_block(blockIdx.x, gridDim.x) * (blockDim.x / kWave) + wave) * A.atomsK;
    if (i0 >= A.N) return;
    adjoint_wave<Z>(A, i0, min(A.atomsK, A.N - i0), smem_all + (size_t)wave * (A.smem_wave / 16));
}

// G in the moment form.  One wavefront serves one atom and walks its list
// entries 64 at a time: each lane forms its entry's cutoff, width factors and
// harmonics in registers, and the entries of the pass get LDS places ordered by
// neighbour species, found with ballots; entries beyond the cutoff (skin lists)
// get none.  Then lanes over functions sum each species' run: moments
// T_b[u][f] = sum e_u Y_f with the four widths in registers (lanes NM .. NM + 3
// read e_u in place of a function, which gives D_b[u] = sum e_u^2), radial
// functions with lanes over (entry, function).  Every sum stays
// in registers until the row ends, for three species or for all eight.  LDS holds
// one pass, not one row per neighbour, so it does not grow with the widest row.
// 1,356 vector instructions per water atom (counters), issued 59 % of the time with
// 78 % of the lanes, LDS waits 6 %: bound by issue and by the chain of a pass's
// phases.  Against the form that regroups the whole row by species in LDS first
// (one row of 36 bytes per neighbour), us: 1,048,576 atoms with a skin 5119 ->
// 4037, 273,561 atoms 820 -> 737, 12,288 atoms 47.4 -> 43.5, 87,912 Li/P/S atoms
// 200 -> 153, 5.5 k 27.0 -> 18.1.  Two atoms per wavefront: 923 on the 273,561
// atoms, sums added up in LDS after every run: 829.  More species, 100,000 atoms, us,
// whole row regrouped / sums in LDS / in registers: four (degree 4) 557 / 534 / 481,
// five (degree 2) 402 / 440 / 387, eight (degree 2) 767 / 847 / 743; tangent with
// stored moments, LDS / registers: 1073 / 997, 653 / 624, 1212 / 1094 (its eight-species
// instances at one wavefront per SIMD less, or their sums spill: 1061, 688, 1219).
constexpr int kGRegSpecies = 3;         // species with their sums in registers
constexpr int kGRegMany = kMaxSpecies;  // of the instances for more species

template <int Z>
struct GShape {
    static constexpr int NM = nharm(Z), NX = NM + kMaxUnionEta;
    static constexpr int NW = NX <= 8 ? 8 : (NX <= 16 ? 16 : (NX <= 32 ? 32 : kWave));   // lanes of one group
    static constexpr int NG = kWave / NW;
};

// float4 entries of the wavefront's LDS slice (layout at the top of g_atom)
__host__ inline int g_units(bool tan, int Z, int S, int NP, int nrad, int ldg, int rows) {
    const int NM = nharm(Z), NX = NM + kMaxUnionEta, NR = (tan ? 2 * NX : NX) | 1, t = tan ? 2 : 1;
    return t * kWave + t * S * NM + S + t * kWave / 2 + (S * nrad + 1) / 2 + rows * NR / 4 + ldg / 4 +
           (NP * kMaxUnionEta * (Z + 1) + 3) / 4;
}

// TAN: the tangent v = dG/dr . u along the atoms' displacements u, with the
// moments T that the G kernel stored: the runs then sum
// dT_b[u][f] = sum (w de_u/dr Y_f + e_u dY_f), w = r^ . (u_i - u_j), and the
// contraction is its product rule.  Against the form that regroups the row in LDS
// and sums the moments again, Li/P/S: 21,872 atoms 89 -> 62 us (rows 24 / 32 / 48 /
// 64 at a time: 64.5 / 67.3 / 70.2 / 85.5), 5.5 k 32 -> 24 us.
template <int Z, int SR, bool TAN>
__device__ __forceinline__ void g_atom(const SymmArgs& A, const int i, float4* smem4) {
    constexpr int NM = GShape<Z>::NM, NX = GShape<Z>::NX, NW = GShape<Z>::NW, NG = GShape<Z>::NG;
    constexpr int NR = (TAN ? 2 * NX : NX) | 1;                 // functions and e_u (TAN: then their derivatives), odd
    constexpr int ZP = Z + 1, U4 = kMaxUnionEta;
    const int lane = threadIdx.x % kWave;
    const DevModel& Mo = *A.dm;
    const int S = Mo.S, NP = Mo.NP, ldg = A.ldg, nrad = A.nrad;
    const int nrow = A.grows;                                   // function rows in LDS at a time (a multiple of 4)
    float4* ef = smem4;                                         // [64] width factors of the pass
    float4* fw = ef + (TAN ? kWave : 0);                        // [64] TAN: w de_u/dr
    float4* T = fw + kWave;                                     // [S][NM] sums (moments or dT), widths in the components
    float4* D = T + S * NM;                                     // [S]
    float4* Ts = D + S;                                         // [S][NM] TAN: stored moments
    float2* rf = reinterpret_cast<float2*>(Ts + (TAN ? S * NM : 0));   // [64] distance, cutoff (TAN: also its derivative, w)
    float2* par = rf + (TAN ? 2 : 1) * kWave;                   // [S][nrad] radial eta, rs
    float* rows = reinterpret_cast<float*>(par + ((S * nrad + 1) & ~1));   // [nrow][NR] functions, then e_u
    float* row = rows + nrow * NR;                              // [ldg]
    float* Am = row + ldg;                                      // [NP][U4][ZP]
    const int o0 = A.off[i], o1 = A.off[i + 1], a = A.species[i];
    float4 gn = make_float4(0.f, 0.f, 0.f, 0.f);
    int bn = 0, jn = 0;
    if (o0 + lane < o1) {
        gn = A.geo[o0 + lane];
        bn = A.nsp[o0 + lane];
        if (TAN) jn = A.nidx[o0 + lane];
    }
    float uix = 0.f, uiy = 0.f, uiz = 0.f;
    if (TAN) {
        uix = A.u[3 * (size_t)i];
        uiy = A.u[3 * (size_t)i + 1];
        uiz = A.u[3 * (size_t)i + 2];
        const float4* gT = reinterpret_cast<const float4*>(A.Tin) + (size_t)i * S * NM;
        for (int x = lane; x < S * NM; x += kWave) Ts[x] = gT[x];
    }
    for (int x = lane; x < ldg; x += kWave) row[x] = 0.0f;
    for (int x = lane; x < S * nrad; x += kWave) {
        const int m = x % nrad, b = x / nrad;
        const RadBlock rb = Mo.rad[a * S + b];
        float2 t = make_float2(0.f, 0.f);
        if (m < rb.n) t = make_float2(A.rad_eta[rb.par + m], A.rad_rs[rb.par + m]);
        par[x] = t;
    }
    const float rc = Mo.rc;
    const int al = lane % NW, grp = lane / NW;
    float mom[SR][U4], rad[SR];
#pragma unroll
    for (int b = 0; b < SR; ++b) {
        rad[b] = 0.0f;
#pragma unroll
        for (int u = 0; u < U4; ++u) mom[b][u] = 0.0f;
    }
    // the groups of lanes meet, then the sums of species b go to LDS
    auto put_moments = [&](int b, float (&acc)[U4]) {
#pragma unroll
        for (int bit = NW; bit < kWave; bit <<= 1)
#pragma unroll
            for (int u = 0; u < U4; ++u) acc[u] += __shfl_xor(acc[u], bit);
        if (lane < NM) {
            T[b * NM + lane] = make_float4(acc[0], acc[1], acc[2], acc[3]);
        } else if (lane < NX) {                                 // lane NM + u: sum of e_u e_u
            const int u = lane - NM;
            reinterpret_cast<float*>(D + b)[u] = u == 0 ? acc[0] : (u == 1 ? acc[1] : (u == 2 ? acc[2] : acc[3]));
        }
    };
    auto put_radial = [&](const RadBlock& rb, float acc) {
        const int W = rb.n <= 8 ? 8 : (rb.n <= 16 ? 16 : 32);
        for (int bit = W; bit < kWave; bit <<= 1) acc += __shfl_xor(acc, bit);
        if (lane < rb.n) row[rb.goff + lane] += acc;
    };
    for (int base = o0; base < o1; base += kWave) {
        const int s = base + lane;
        const float4 gq = gn;
        const bool keep = s < o1 && gq.w <= rc;
        const int key = keep ? bn : -1;
        float tx = 0.f, ty = 0.f, tz = 0.f;
        if (TAN && keep) {
            tx = uix - A.u[3 * (size_t)jn];
            ty = uiy - A.u[3 * (size_t)jn + 1];
            tz = uiz - A.u[3 * (size_t)jn + 2];
        }
        if (s + kWave < o1) {
            gn = A.geo[s + kWave];
            bn = A.nsp[s + kWave];
            if (TAN) jn = A.nidx[s + kWave];
        }
        int pos = 0, cnt = 0;
        for (int b = 0; b < S; ++b) {
            const uint64_t m = __ballot(key == b);
            if (key == b) pos = cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            cnt += __popcll(m);
        }
        float y[NM], e[U4], dy[TAN ? NM : 1], d[U4];
        wave_sync();                                            // the previous pass's LDS reads are done
        if (keep) {
            const float r = gq.w, ir = __builtin_amdgcn_rcpf(r);   // 1 ulp
            const float hx = gq.x * ir, hy = gq.y * ir, hz = gq.z * ir;
            float C[ZP], Sn[ZP], ql[qidx(Z, Z) + 1];
            harm_factors<Z, float>(hx, hy, hz, C, Sn, ql);
            harm_values<Z, float>(C, Sn, ql, y);
            float w = 0.0f;
            if constexpr (TAN) {
                w = hx * tx + hy * ty + hz * tz;
                harm_along<Z, float>(C, Sn, ql, (tx - hx * w) * ir, (ty - hy * w) * ir, (tz - hz * w) * ir, dy);
            }
            float fc, gc;
            cutoff_fg(Mo.cutoff, Mo.rc, Mo.rci, Mo.pirc, r, fc, gc);
#pragma unroll
            for (int u = 0; u < U4; ++u) {
                const float k = Mo.uieta2[a][u], x = u < Mo.nunion[a] ? __expf(-k * r * r) : 0.0f;
                e[u] = x * fc;
                d[u] = x * (-2.0f * r * k * fc + gc) * w;       // TAN
            }
            ef[pos] = make_float4(e[0], e[1], e[2], e[3]);
            if constexpr (TAN) {
                fw[pos] = make_float4(d[0], d[1], d[2], d[3]);
                rf[2 * pos] = make_float2(r, fc);
                rf[2 * pos + 1] = make_float2(gc, w);
            } else {
                rf[pos] = make_float2(r, fc);
            }
        }
        // moments: rows of up to nrow entries at a time
        for (int c0 = 0; c0 < cnt; c0 += nrow) {
            if (c0 > 0) wave_sync();                            // the previous rows are read
            if (keep && pos >= c0 && pos < c0 + nrow) {
                float* w = rows + (pos - c0) * NR;
#pragma unroll
                for (int f = 0; f < NM; ++f) w[f] = y[f];
#pragma unroll
                for (int u = 0; u < U4; ++u) w[NM + u] = e[u];
                if constexpr (TAN) {
#pragma unroll
                    for (int f = 0; f < NM; ++f) w[NX + f] = dy[f];
#pragma unroll
                    for (int u = 0; u < U4; ++u) w[NX + NM + u] = d[u];
                }
            }
            wave_sync();
            auto run = [&](int j0, int j1, float (&acc)[U4]) {
                auto step = [&](const float* w, int J) {
                    const float v = w[al];
                    const float4 e4 = ef[J];
                    if constexpr (TAN) {
                        const float dv = w[NX + al];
                        const float4 f4 = fw[J];
                        acc[0] += f4.x * v + e4.x * dv; acc[1] += f4.y * v + e4.y * dv;
                        acc[2] += f4.z * v + e4.z * dv; acc[3] += f4.w * v + e4.w * dv;
                    } else {
                        acc[0] += e4.x * v; acc[1] += e4.y * v; acc[2] += e4.z * v; acc[3] += e4.w * v;
                    }
                };
                if (al < NX) {
                    int J = j0 + grp;
                    // four entries per trip: rows at fixed offsets from one address
                    for (; J + 3 * NG < j1; J += 4 * NG) {
                        const float* w = rows + (J - c0) * NR;
                        step(w, J);
                        step(w + NG * NR, J + NG);
                        step(w + 2 * NG * NR, J + 2 * NG);
                        step(w + 3 * NG * NR, J + 3 * NG);
                    }
                    for (; J < j1; J += NG) step(rows + (J - c0) * NR, J);
                }
            };
            int s0 = 0;
#pragma unroll
            for (int b = 0; b < SR; ++b) {
                if (SR > kGRegSpecies && b >= S) break;
                const int n = __popcll(__ballot(key == b));
                run(max(s0, c0), min(s0 + n, c0 + nrow), mom[b]);
                s0 += n;
            }
        }
        // radial: lanes over (entry, function) of every species' run
        auto radial = [&](int b, const RadBlock& rb, int j0, int j1) {
            const int sh = rb.n <= 8 ? 3 : (rb.n <= 16 ? 4 : 5), nj = kWave >> sh;
            const int m = lane & ((1 << sh) - 1);
            const float2 t = m < rb.n ? par[b * nrad + m] : make_float2(0.f, 0.f);
            float acc = 0.0f;
            if (A.rad_gauss) {
#pragma unroll 4
                for (int J = j0 + (lane >> sh); J < j1; J += nj) {
                    const float2 v = rf[TAN ? 2 * J : J];
                    const float x = t.x * (v.x - t.y), ex = __expf(-x * x);
                    if constexpr (TAN) {
                        const float2 gw = rf[2 * J + 1];
                        acc += ex * (gw.x - 2.0f * (t.x * x) * v.y) * gw.y;
                    } else {
                        acc += ex * v.y;
                    }
                }
            } else {
                for (int J = j0 + (lane >> sh); J < j1; J += nj) {
                    const float2 v = rf[TAN ? 2 * J : J];
                    const float2 gw = TAN ? rf[2 * J + 1] : make_float2(0.f, 0.f);
                    float g, dr;
                    radial_fd(rb.name, t.x, t.y, v.x, v.y, gw.x, g, dr);
                    acc += TAN ? dr * gw.y : g;
                }
            }
            return acc;
        };
        int s0 = 0;
#pragma unroll
        for (int b = 0; b < SR; ++b) {
            if (SR > kGRegSpecies && b >= S) break;
            const int n = __popcll(__ballot(key == b));
            if (n > 0) rad[b] += radial(b, Mo.rad[a * S + b], s0, s0 + n);
            s0 += n;
        }
    }
    wave_sync();
#pragma unroll
    for (int b = 0; b < SR; ++b)
        if (b < S) {
            put_moments(b, mom[b]);
            put_radial(Mo.rad[a * S + b], rad[b]);
        }
    wave_sync();
    if (!TAN && A.Tout) {
        float4* out = reinterpret_cast<float4*>(A.Tout) + (size_t)i * S * NM;
        for (int x = lane; x < S * NM; x += kWave) out[x] = T[x];
    }
    // block contractions: lanes over (pair, width, degree); a degree has 2m + 1
    // functions, every lane runs the length of the highest with the surplus terms
    // weighted 0, so that the loads issue together
    for (int x = lane; x < NP * U4 * ZP; x += kWave) {
        const int m = x % ZP, u = (x / ZP) % U4, p = x / (ZP * U4);
        int c = 0;
        while ((c + 1) * (c + 2) / 2 <= p) ++c;
        const int b = p - c * (c + 1) / 2;
        const float* Tb = reinterpret_cast<const float*>(T + b * NM) + u;
        const float* Tc = reinterpret_cast<const float*>(T + c * NM) + u;
        float v = 0.0f;
#pragma unroll
        for (int j = 0; j < 2 * Z + 1; ++j) {
            const int f = min(m * m + j, NM - 1);
            const float w = j <= 2 * m ? 1.0f : 0.0f;
            if constexpr (TAN) {
                const float* Sb = reinterpret_cast<const float*>(Ts + b * NM) + u;
                const float* Sc = reinterpret_cast<const float*>(Ts + c * NM) + u;
                v += w * (Tb[U4 * f] * Sc[U4 * f] + Sb[U4 * f] * Tc[U4 * f]);
            } else {
                v += (w * Tb[U4 * f]) * Tc[U4 * f];
            }
        }
        if (b == c) v = 0.5f * (v - reinterpret_cast<const float*>(D + b)[u]);
        Am[x] = v;
    }
    wave_sync();
    // outputs: lanes over (pair, width, combination), loads before the guards that use them
    for (int x = lane; x < NP * kGridG * kGridK; x += kWave) {
        const int k = x % kGridK, g = (x / kGridK) % kGridG, p = x / (kGridK * kGridG);
        const AngBlock& B = Mo.ang[a * NP + p];
        const int nk = min(max(B.nk, 0), kGridK), goff = B.goff;
        const bool use = B.n > 0 && g < B.ng && k < nk;
        const int om = B.outm[g * nk + k];                      // < kGridG * kGridK; used only when use
        float lc[ZP];
#pragma unroll
        for (int l = 0; l < ZP; ++l) lc[l] = B.lcoef[k][l];
        if (use) {
            const float* Aq = Am + (p * U4 + g) * ZP;
            float v = 0.0f;
#pragma unroll
            for (int l = 0; l < ZP; ++l) v += lc[l] * Aq[l];
            row[goff + om] = v;
        }
    }
    wave_sync();
    float* out = TAN ? A.v : A.G;
    for (int x = lane; x < ldg; x += kWave) out[(size_t)i * ldg + x] = row[x];
}

// Grid dispatch: a block holds blockDim.x / 64 atoms (the "atoms per
// workgroup" tuning).
template <int MODE, int Z>
__global__ __launch_bounds__(256) void k_moment(SymmArgs A) {
    extern __shared__ float4 smem_all[];
    const int wave = threadIdx.x / kWave;
    const int i = blockIdx.x * (blockDim.x / kWave) + wave;
    if (i >= A.N) return;
    moment_atom<MODE, Z>(A, i, smem_all + (size_t)wave * (A.smem_wave / 16));
}

// G and the tangent with stored moments: one atom per wavefront
template <int Z, int SR, bool TAN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(
    (Z <= 2 ? 5 : 4) - (TAN && SR > kGRegSpecies && Z != 3 ? 1 : 0)))) void k_moment_g(SymmArgs A) {
    extern __shared__ float4 smem_all[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int i = xcd_block(blockIdx.x, gridDim.x) * (blockDim.x / kWave) + wave;
    if (i >= A.N) return;
    g_atom<Z, SR, TAN>(A, i, smem_all + (size_t)wave * (A.smem_wave / 16));
}

constexpr int kModeAdjT = 4, kModeTanT = 5;                     // the stored-moment adjoint and tangent

// Persistent dispatch (a separate kernel, so that the grid kernel keeps its
// own register allocation): a grid sized to the resident capacity, every
// wavefront pulls (first atom, count) items off the queue of its XCD (blocks
// go to XCD blockIdx.x % 8) until the queue is empty; the items of a batch
// run largest structure first.
template <int MODE, int Z, int SR = 0>
__global__ __launch_bounds__(256) void k_moment_queue(SymmArgs A) {
    extern __shared__ float4 smem_all[];
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    float4* smem4 = smem_all + (size_t)wave * (A.smem_wave / 16);
    const int q = blockIdx.x % kXcds;
    const int beg = A.qoff[q], cnt = A.qoff[q + 1] - beg;
    int* ctr = A.queue + 32 * q;
    int k = 0;
    if (lane == 0) k = atomicAdd(ctr, 1);
    k = __shfl(k, 0);
    while (k < cnt) {
        // the next item is claimed before this one runs: the atomic's round
        // trip overlaps the item's own loads
        int nk = 0;
        if (lane == 0) nk = atomicAdd(ctr, 1);
        const int2 it = A.items[beg + k];
        const int ib = __builtin_amdgcn_readfirstlane(it.x), ie = ib + __builtin_amdgcn_readfirstlane(it.y);
        for (int a = ib; a < ie; a += A.atomsK) {
            if constexpr (MODE == 0) g_atom<Z, SR, false>(A, a, smem4);
            else if constexpr (MODE == kModeTanT) g_atom<Z, SR, true>(A, a, smem4);
            else if constexpr (MODE == kModeAdjT) adjoint_wave<Z>(A, a, min(A.atomsK, ie - a), smem4);
            else moment_atom<MODE, Z>(A, a, smem4);
            wave_sync();                                        // the next atoms reuse the LDS slice
        }
        k = __shfl(nk, 0);
    }
}

__global__ void k_queue_reset(int* __restrict__ queue) {
    if (threadIdx.x < kXcds) queue[32 * threadIdx.x] = 0;
}

// LDS bytes of one wavefront of moment_atom<mode> (the layout at its top)
static size_t moment_smem(const SymmArgs& A, int mode, int Z, int S, int NP) {
    const int NM = nharm(Z), ZP = Z + 1, U4 = kMaxUnionEta;
    const bool adj = mode == 1 || mode == 3;
    const int PWS = (NM * (mode == 2 ? 2 : 1)) | 1;
    size_t b = 16 * (size_t)A.maxn * (3 + (mode == 2 ? 1 : 0));
    b += 4 * (adj ? 2 : 1) * (size_t)A.maxn + 4 * 16;                              // r, canon (adjoint), seg
    size_t f = (size_t)A.ldg + (mode == 1 ? 3 * (size_t)A.maxn : 0) + (mode == 3 ? 2 * (size_t)A.maxn : 0) +
               (size_t)pw_floats(mode, A.maxn, PWS, A.grows);
    f += (size_t)S * U4 * NM * (mode == 2 ? 2 : 1) + 2 * (size_t)S * U4 + (size_t)NP * U4 * ZP;
    f += (adj && S * NM * U4 > kUbRegs * kWave ? (size_t)S * NM * U4 : 0);         // dE/dT beside the moments
    return b + 4 * f;
}

// ================================================================ host ====

// Work items of the persistent dispatch: every structure cut into ranges of
// up to kItemAtoms atoms (fewer when the batch would leave resident
// wavefronts without items: about four items per wavefront the chip holds),
// structures in decreasing size, items dealt round robin to the XCD queues so
// that each queue gets an equal share of every size.
constexpr int kItemAtoms = 8;

hipError_t build_items(ann_ctx* ctx) {
    const int S = ctx->nstruc;
    hipError_t e;
    if (!ctx->d_queue) {
        if ((e = hipMalloc(&ctx->d_queue, sizeof(int) * 32 * kXcds)) != hipSuccess) return e;
        if ((e = hipMalloc(&ctx->d_qoff, sizeof(int) * (kXcds + 1))) != hipSuccess) return e;
    }
    const int resident = std::max(1, ctx->num_cu) * 32;            // wavefronts per CU the kernels can hold
    const int len = std::max(1, std::min(kItemAtoms, ctx->atom_off[S] / (4 * resident)));
    std::vector<int> order(S);
    for (int s = 0; s < S; ++s) order[s] = s;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
        return ctx->atom_off[a + 1] - ctx->atom_off[a] > ctx->atom_off[b + 1] - ctx->atom_off[b];
    });
    std::vector<int2> all;
    for (int s : order)
        for (int a = ctx->atom_off[s]; a < ctx->atom_off[s + 1]; a += len)
            all.push_back(make_int2(a, std::min(len, ctx->atom_off[s + 1] - a)));
    std::vector<int2> items;
    items.reserve(all.size());
    std::vector<int> qoff(kXcds + 1, 0);
    for (int q = 0; q < kXcds; ++q) {
        qoff[q] = (int)items.size();
        for (size_t k = q; k < all.size(); k += kXcds) items.push_back(all[k]);
    }
    qoff[kXcds] = (int)items.size();
    if ((int)items.size() > ctx->items_cap) {
        if (ctx->d_items && (e = hipFree(ctx->d_items)) != hipSuccess) return e;
        ctx->d_items = nullptr;
        ctx->items_cap = 0;
        if ((e = hipMalloc(&ctx->d_items, sizeof(int2) * items.size())) != hipSuccess) return e;
        ctx->items_cap = (int)items.size();
    }
    if ((e = staged_upload(ctx, kStItems, ctx->d_items, items.data(), sizeof(int2) * items.size())) != hipSuccess)
        return e;
    if ((e = staged_upload(ctx, kStQoff, ctx->d_qoff, qoff.data(), sizeof(int) * (kXcds + 1))) != hipSuccess)
        return e;
    ctx->items_valid = true;
    return hipSuccess;
}

// Work items of the current batch, built on the first persistent dispatch
// after ann_set_batch (host set-up and uploads, so callers that capture a
// graph build them before the capture).
hipError_t ensure_items(ann_ctx* ctx) {
    if (ctx->items_valid) return hipSuccess;
    if (ctx->capturing) return hipErrorStreamCaptureUnsupported;
    return build_items(ctx);
}

static SymmArgs make_args(ann_ctx* ctx) {
    SymmArgs A{};
    A.dm = ctx->dm;
    A.rad_rs = ctx->da.rad_rs;
    A.rad_eta = ctx->da.rad_eta;
    A.ang_eta = ctx->da.ang_eta;
    A.ang_zeta = ctx->da.ang_zeta;
    A.ang_lam = ctx->da.ang_lam;
    A.N = ctx->natoms;
    A.ldg = ctx->ldg;
    A.maxn = (std::max(ctx->nl.maxn, 1) + 3) / 4 * 4;   // keeps every LDS array 16-byte aligned
    A.species = ctx->d_species;
    A.off = ctx->nl.off;
    A.geo = ctx->nl.geo;
    A.nsp = ctx->nl.nsp;
    A.nidx = ctx->nl.idx;
    A.rad_gauss = ctx->hm.rad_gauss;
    A.nrad = ctx->hm.nrad;
    A.nrs = A.nrad | 1;
    A.atomsK = 1;
    return A;
}

// Atoms per wavefront of the stored-moment adjoint.  A row of n entries takes
// ceil(n / 64) passes, two rows together often one less; but two atoms' tables
// are built one after the other, and half the wavefronts must still fill the
// chip.  Measured (us, one / two atoms): 1,048,576 atoms 3349 / 3035, 273,561 atoms
// 650 / 556, Li/P/S 21,872 atoms 40.5 / 35.3, 12,288 atoms 38.8 / 36.2, 5.5 k 14.8 /
// 15.8, 2,048 atoms 16.4 / 23.9, 192 atoms 11.9 / 15.9; argon, 4,096 atoms of 18
// entries, 13.3 / 11.7 (both rows in one pass).  Three (an earlier form, two / three
// 576 / 649 on 273,561 atoms) make more lanes of an instruction read different LDS
// rows.
static int adj_atoms(const ann_ctx* ctx) {
    const int64_t N = ctx->natoms;
    const bool one_pass = 2 * ctx->nl.npairs <= (int64_t)kWave * 7 / 8 * N;
    return N >= 8192 || (N >= 4096 && one_pass) ? 2 : 1;
}

static size_t plain_smem(const SymmArgs& A, int mode) {
    size_t b = (size_t)A.maxn * (16 + 4 + 4 + 4);
    if (mode == 1) b += 4 * ((size_t)A.ldg + 3 * A.maxn);
    else b += 4 * (size_t)A.ldg * 65;
    if (mode == 2) b += 16 * (size_t)A.maxn;
    return b;
}

static size_t fast_smem(const SymmArgs& A, int mode) {
    size_t b = 16 * (size_t)A.maxn * (2 + (mode == 0 ? 0 : 1) + (mode == 2 ? 1 : 0));   // g, ef, efd, tv
    b += 8 * (size_t)A.maxn + 4 * 2 * (size_t)A.maxn + 4 * 16;                         // fg, r, canon, seg
    b += 4 * (size_t)A.ldg;
    if (mode == 1) b += 12 * (size_t)A.maxn;
    return b;
}

using MomentKernel = void (*)(SymmArgs);
template <int MODE, int Z>
static MomentKernel pick_kernel(bool queued, int S) {
    if constexpr (MODE == 0 || MODE == kModeTanT) {
        constexpr bool tan = MODE == kModeTanT;
        if (S <= kGRegSpecies) return queued ? k_moment_queue<MODE, Z, kGRegSpecies> : k_moment_g<Z, kGRegSpecies, tan>;
        return queued ? k_moment_queue<MODE, Z, kGRegMany> : k_moment_g<Z, kGRegMany, tan>;
    } else if constexpr (MODE == kModeAdjT) {
        return queued ? k_moment_queue<MODE, Z> : k_adjoint<Z>;
    } else {
        return queued ? k_moment_queue<MODE, Z> : k_moment<MODE, Z>;
    }
}
template <int MODE>
static MomentKernel moment_kernel(int z, bool queued, int S) {
    switch (z) {
        case 1: return pick_kernel<MODE, 1>(queued, S);
        case 2: return pick_kernel<MODE, 2>(queued, S);
        case 3: return pick_kernel<MODE, 3>(queued, S);
        case 4: return pick_kernel<MODE, 4>(queued, S);
        default: return pick_kernel<MODE, 5>(queued, S);
    }
}

template <int MODE>
static hipError_t run(ann_ctx* ctx, int form, SymmArgs A) {
    if (A.N == 0) return hipSuccess;
    const DevModel& M = ctx->hm;
    const bool fast = form != ANN_FORM_PLAIN && M.all_grid && M.fast_ng > 0;
    const bool moment = fast && form == ANN_FORM_FAST && M.moment_z > 0 && ctx->tune_angular == 0;
    const char* names[3][3] = {{"symm_fwd_plain", "symm_bwd_plain", "symm_tan_plain"},
                               {"symm_fwd_fast", "symm_bwd_fast", "symm_tan_fast"},
                               {"symm_fwd_mom", "symm_bwd_mom", "symm_tan_mom"}};
    Launch L(ctx, names[moment ? 2 : (fast ? 1 : 0)][MODE]);
    if (moment) {
        // the moment store holds work_atoms rows: it is used only when the batch
        // fits (a forward call on a grown batch before any fused call skips it)
        const bool tfits = ctx->d_T && ctx->work_atoms >= A.N;
        if (MODE == 0 && tfits) A.Tout = ctx->d_T;
        if (MODE != 0 && tfits && ctx->T_gen == ctx->geo_gen) A.Tin = ctx->d_T;
        const bool adjT = MODE == 1 && A.Tin, tanT = MODE == 2 && A.Tin;
        size_t sw = 0;
        if (adjT) {
            A.atomsK = adj_atoms(ctx);
            if (adj_units(A.atomsK, M.moment_z, M.S, M.NP, A.nrs, A.ldg) > 1024) A.atomsK = 1;   // above 16 KiB
            sw = 16 * (size_t)adj_units(A.atomsK, M.moment_z, M.S, M.NP, A.nrs, A.ldg);
        } else if (MODE == 0 || tanT) {
            // a pass's 64 rows at once where rows are short (G up to degree 2) or where the
            // chip holds every wavefront's slice all the same, else 32 (measured, 32 / 64
            // rows: 273,561 water atoms 735 / 1010 us, 12,288 43.8 / 53.3, 2,048 20.0 / 18.7,
            // 87,912 Li/P/S atoms of degree 2 157 / 152)
            auto units = [&](int rows) { return g_units(tanT, M.moment_z, M.S, M.NP, A.nrad, A.ldg, rows); };
            const bool fits = (int64_t)A.N <= (int64_t)ctx->num_cu * ((160 << 10) / (16 * units(kWave)));
            A.grows = (MODE == 0 && M.moment_z <= 2) || fits ? kWave : (tanT && M.moment_z <= 2 ? 24 : kWave / 2);
            A.grows = std::min(A.grows, A.maxn);                // no more than the widest row has (a multiple of 4)
            sw = 16 * (size_t)units(A.grows);
        } else {
            // the adjoint that sums the moments: 64 function rows at a time where the chip
            // holds every wavefront's slice all the same or rows are short, else 32 (us, 64 /
            // 32: 12,288 atoms of one species and degree 4 70 / 56, of two 80 / 65, of three 100
            // / 78; 512 atoms 13.9 / 14.6; degree 5 98 / 98)
            A.grows = kPwRows;
            sw = (moment_smem(A, MODE, M.moment_z, M.S, M.NP) + 15) / 16 * 16;
            if (MODE == 1 && M.moment_z >= 4 && (int64_t)A.N > (int64_t)ctx->num_cu * (int64_t)((160 << 10) / sw)) {
                A.grows = kPwRows / 2;
                sw = (moment_smem(A, MODE, M.moment_z, M.S, M.NP) + 15) / 16 * 16;
            }
        }
        int apb = ctx->tune_apb[MODE];
        while (apb > 1 && sw * apb > 65536) apb /= 2;          // dynamic LDS of one workgroup
        A.smem_wave = (int)sw;
        const int per = apb * A.atomsK;                          // atoms of one workgroup
        unsigned grid = (unsigned)((A.N + per - 1) / per), block = 64u * apb;
        const size_t sm = sw * apb;
        const bool queued = ctx->tune_queue == 1;
        if (queued) {
            const hipError_t ei = ensure_items(ctx);
            if (ei != hipSuccess) return ei;
        }
        MomentKernel kern = adjT   ? moment_kernel<kModeAdjT>(M.moment_z, queued, M.S)
                            : tanT ? moment_kernel<kModeTanT>(M.moment_z, queued, M.S)
                                   : moment_kernel<MODE>(M.moment_z, queued, M.S);
        if (queued) {
            // persistent: enough workgroups for the most wavefronts a CU can hold
            // (32); those that find no room start later, find the queues empty
            // and exit.  A multiple of the XCD count, so every queue has workers.
            const unsigned cap = (unsigned)std::max(1, ctx->num_cu) * (32u / (unsigned)apb);
            grid = std::min(grid, cap);
            grid = std::max(kXcds, (int)((grid + kXcds - 1) / kXcds * kXcds));
            A.queue = ctx->d_queue;
            A.items = ctx->d_items;
            A.qoff = ctx->d_qoff;
            k_queue_reset<<<1, 64, 0, ctx->stream>>>(ctx->d_queue);
        }
        kern<<<grid, block, sm, ctx->stream>>>(A);
        if (MODE == 0) ctx->T_gen = A.Tout ? ctx->geo_gen : ~0ull;
        return hipGetLastError();
    }
    if (fast) {
        const size_t sm = fast_smem(A, MODE);
#define X(G, K)                                                                \
        if (M.fast_ng == G && M.fast_nk == K) {                                \
            k_fast<MODE, G, K><<<A.N, 64, sm, ctx->stream>>>(A);               \
            return hipGetLastError();                                          \
        }
        ANN_SHAPES(X)
#undef X
        return hipErrorInvalidValue;
    }
    const size_t sm = plain_smem(A, MODE);
    k_plain<MODE><<<A.N, 64, sm, ctx->stream>>>(A);
    return hipGetLastError();
}

hipError_t symm_fwd(ann_ctx* ctx, int form, float* G) {
    SymmArgs A = make_args(ctx);
    A.G = G;
    return run<0>(ctx, form, A);
}

hipError_t symm_bwd(ann_ctx* ctx, int form, const float* dEdG, float* P) {
    SymmArgs A = make_args(ctx);
    A.dEdG = dEdG;
    A.P = P;
    return run<1>(ctx, form, A);
}

// Fused E+F: G, the network and the force adjoint of each atom in one
// moment-form kernel (moment_atom<3>), for FAST in the moment form with FP32
// inputs and networks of at most 128 inputs and 64 neurons per layer.
bool fused_supported(const ann_ctx* ctx, int form) {
    const DevModel& M = ctx->hm;
    if (form != ANN_FORM_FAST || !M.all_grid || M.fast_ng <= 0 || M.moment_z <= 0 || ctx->tune_angular != 0 ||
        ctx->npre != 0 || ctx->natoms == 0)
        return false;
    for (int a = 0; a < M.S; ++a) {
        const NetDesc& D = M.net[a];
        if (D.nin > 2 * kWave) return false;
        for (int l = 0; l < D.nlayer - 1; ++l)
            if (D.nodes[l] > kVecMaxWidth) return false;
    }
    const SymmArgs A = make_args(const_cast<ann_ctx*>(ctx));   // reads only
    return moment_smem(A, 3, M.moment_z, M.S, M.NP) <= 65536;
}

hipError_t symm_fused(ann_ctx* ctx, const float* inpb, float* Eatom, float* P) {
    SymmArgs A = make_args(ctx);
    if (A.N == 0) return hipSuccess;
    hipError_t e;
    if (!ctx->wchunk_valid && (e = chunk_weights(ctx)) != hipSuccess) return e;
    A.P = P;
    A.Eatom = Eatom;
    A.wchunk = ctx->d_wchunk;
    A.wtrans = ctx->d_wtrans;
    A.inpw = ctx->da.inpw;
    A.inpb = inpb;
    const DevModel& M = ctx->hm;
    Launch L(ctx, "ef_fused");
    const size_t sw = (moment_smem(A, 3, M.moment_z, M.S, M.NP) + 15) / 16 * 16;
    int apb = ctx->tune_apb[1];                             // the adjoint's atoms per workgroup
    while (apb > 1 && sw * apb > 65536) apb /= 2;
    A.smem_wave = (int)sw;
    const unsigned grid = (unsigned)((A.N + apb - 1) / apb), block = 64u * apb;
    void (*kern)(SymmArgs) = M.moment_z == 1 ? k_moment<3, 1> : M.moment_z == 2 ? k_moment<3, 2>
                             : M.moment_z == 3 ? k_moment<3, 3> : M.moment_z == 4 ? k_moment<3, 4>
                             : k_moment<3, 5>;
    kern<<<grid, block, sw * apb, ctx->stream>>>(A);
    ctx->T_gen = ~0ull;                                     // no stored moments
    return hipGetLastError();
}

hipError_t symm_tangent(ann_ctx* ctx, int form, const float* u, float* v) {
    SymmArgs A = make_args(ctx);
    A.u = u;
    A.v = v;
    return run<2>(ctx, form, A);
}

bool fast_shape_supported(int ng, int nk) { return fast_shape_ok(ng, nk); }

}  // namespace ann
