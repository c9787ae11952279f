// net_mfma.hip -- per-species networks as batched GEMMs on the matrix cores.
//
// Same mathematics as ANN::fpbp + DODZ::grad (src/ml/nn.cpp:1367-1389,
// 1801-1830).  Atoms are grouped by species (a species-sorted permutation of
// the batch) into tiles of 16 rows; four or eight wavefronts share a tile and run every
// layer as 16 x N x K products on the matrix cores (BF16 operands split into
// three terms, FP32 accumulation; Operands below):
//   forward:  Z_l = A_{l-1} W_l^T (+ b_l), activation on the accumulator;
//   backward: g_{L-1} = outw W_L^T . sigma'_{L-1}, g_{l-1} = (g_l W_l) . sigma'_{l-1},
//             dE/dG = (g_0 W_0) . inpw.
// Activations move between the accumulator layout and the operand layout
// through LDS; the weights come as operand tables split once per parameter
// update (k_wtables).
#include <type_traits>

#include "net_dev.h"

namespace ann {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

hipError_t species_perm(ann_ctx* ctx);

constexpr int kTile = 16;
constexpr int kMaxK = 128;     // padded input width supported (n_in <= 128)

struct MfmaArgs {
    const DevModel* dm;
    const float* W;
    const float* inpw;
    const float* inpb;
    int ldg;
    const int* perm;       // species-sorted atom order
    const int2* tiles;     // (species, start in perm); count from the species end
    const int* spend;      // end of each species block in perm
    int ntiles;
    const float* G;
    float* Eatom;
    float* dEdG;
    const uint4* wtab;     // BF16x3 operand tables of the hidden-layer weights
};

// acc += X (16 x K, rows = atoms, from LDS) * B (K x 16 columns of one tile)
// on v_mfma_f32_16x16x32_bf16.  BF16 carries 8
// mantissa bits, so both operands are split into three BF16 terms
// x = x0 + x1 + x2 (x0 = bf16(x), x1 = bf16(x - x0), x2 = bf16(x - x0 - x1)) and
// the six products with i + j <= 2 are accumulated in FP32: truncation
// ~2^-24 relative, the FP32 level the 1e-5 force bar needs.
// Lane l supplies row l % 16 of X and column l % 16 of B for k block
// 8 (l / 16) .. +7 and receives D rows 4 (l / 16) .. +3 of column l % 16.
__device__ __forceinline__ void split3(float x, __bf16& a, __bf16& b, __bf16& c) {
    a = (__bf16)x;
    const float r1 = x - (float)a;
    b = (__bf16)r1;
    c = (__bf16)(r1 - (float)b);
}

__device__ __forceinline__ bf16x8 as_bf16x8(uint4 u) {
    bf16x8 v;
    __builtin_memcpy(&v, &u, sizeof(v));
    return v;
}

// The right operands come pre-split from a table (k_wtables): for k block kk
// and column tile ct, the three BF16 terms of lane l are the 16-byte entries
// ((kk * nt + ct) * 3 + p) * 64 + l, p = 0, 1, 2.  The left operands are split
// once, by the thread that writes them, into three BF16 planes of the tile.
constexpr int kPlaneK = kMaxK + 8;          // row stride of a plane: 16-byte rows, all banks in a 16-row read
typedef __bf16 PlaneRow[kPlaneK];

// The operands of one of NW wavefronts (column tile ct belongs to wavefront ct % NW)
// of a product with NH own column tiles and up to KB k blocks.  Loaded a phase ahead, so that the loads' latency runs beside the phase
// before (they depend on nothing but the tile's species).
template <int NH, int KB, int NW>
struct Operands {
    uint4 w[NH][KB][3];
    __device__ __forceinline__ void load(const uint4* __restrict__ tab, int K, int ncol, int wv) {
        const int lane = threadIdx.x % kWave, nt = (ncol + 15) / 16, nkb = (K + 31) / 32;
#pragma unroll
        for (int h = 0; h < NH; ++h)
#pragma unroll
            for (int kk = 0; kk < KB; ++kk) {
                const int ct = h * NW + wv;
                if (ct < nt && kk < nkb) {
                    const uint4* e = tab + (size_t)((kk * nt + ct) * 3) * kWave + lane;
#pragma unroll
                    for (int p = 0; p < 3; ++p) w[h][kk][p] = e[p * kWave];
                }
            }
    }
    // acc[h] += X (16 x K planes) * (own column tile h)
    __device__ __forceinline__ void mul(const PlaneRow* X0, const PlaneRow* X1, const PlaneRow* X2, int K, int ncol,
                                        int wv, f32x4 (&acc)[NH]) const {
        const int lane = threadIdx.x % kWave, row = lane % 16, kb = 8 * (lane / 16);
        const int nt = (ncol + 15) / 16, nkb = (K + 31) / 32;
        if (wv >= nt) return;
#pragma unroll
        for (int kk = 0; kk < KB; ++kk) {
            if (kk >= nkb) break;
            const bf16x8 a0 = *reinterpret_cast<const bf16x8*>(&X0[row][32 * kk + kb]);
            const bf16x8 a1 = *reinterpret_cast<const bf16x8*>(&X1[row][32 * kk + kb]);
            const bf16x8 a2 = *reinterpret_cast<const bf16x8*>(&X2[row][32 * kk + kb]);
#pragma unroll
            for (int h = 0; h < NH; ++h) {
                if (h * NW + wv >= nt) break;
                const bf16x8 b0 = as_bf16x8(w[h][kk][0]), b1 = as_bf16x8(w[h][kk][1]), b2 = as_bf16x8(w[h][kk][2]);
                f32x4 c = acc[h];
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a2, b0, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b2, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b0, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b1, c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, c, 0, 0, 0);
                acc[h] = c;
            }
        }
    }
};

// The weight tables, all read from the FP32 weights W and rewritten after
// every parameter update, in one launch (grid row = role and segment):
//  * matrix-core operand tables of every hidden layer, segment (species,
//    layer, direction): direction 0 holds W_l as the right operand of the
//    forward product (K = inputs, columns = neurons), direction 1 holds W_l^T
//    for the backward product (K = neurons, columns = inputs); one thread per
//    16-byte entry; tick (the Adam step counter) is advanced by one thread;
//  * the vector-ALU network's table of each species: the hidden layers' weight
//    rows, their biases and the output neuron's weights and bias, one thread
//    per float including the padding (written as zero);
//  * its transposed weight rows W_l^T[j][k], segment (species, layer).
struct WTabArgs {
    const DevModel* dm;
    const float* W;
    uint4* split;       // null: the operand tables are not rewritten
    float* chunk;
    float* trans;
    int* tick;
    int ys, yc;         // grid rows of the operand tables and of the species tables
};

__device__ __forceinline__ void wsplit_entry(const DevModel* __restrict__ dm, const float* __restrict__ W,
                                             uint4* __restrict__ tab, int seg, int e) {
    const int a = seg / (2 * kMaxLayers), l = (seg / 2) % kMaxLayers, dir = seg % 2;
    if (a >= dm->S) return;
    const NetDesc& D = dm->net[a];
    if (l >= D.nlayer - 1) return;
    const int ni = l == 0 ? D.nin : D.nodes[l - 1], no = D.nodes[l];
    const int K = dir == 0 ? ni : no, ncol = dir == 0 ? no : ni;
    const int nt = (ncol + 15) / 16;
    if (e >= (K + 31) / 32 * nt * 3 * kWave) return;
    const int lane = e % kWave, p = (e / kWave) % 3, ct = (e / (3 * kWave)) % nt, kk = e / (3 * kWave * nt);
    const int col = ct * 16 + lane % 16, kb = kk * 32 + 8 * (lane / 16);
    const float* Wl = W + D.woff[l];
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int k = kb + j;
        const float x = (k < K && col < ncol) ? (dir == 0 ? Wl[k * no + col] : Wl[col * no + k]) : 0.0f;
        __bf16 x0, x1, x2;
        split3(x, x0, x1, x2);
        v[j] = p == 0 ? x0 : (p == 1 ? x1 : x2);
    }
    uint4 u;
    __builtin_memcpy(&u, &v, sizeof(u));
    tab[(dir == 0 ? D.wsf[l] : D.wsb[l]) + e] = u;
}

__device__ __forceinline__ void wchunk_entry(const DevModel* __restrict__ dm, const float* __restrict__ W,
                                             float* __restrict__ tab, int a, int x) {
    if (a >= dm->S) return;
    const NetDesc& D = dm->net[a];
    const int e = D.wc0 + x;
    if (e >= D.wc0 + D.wcn) return;
    const int L = D.nlayer;
    float v = 0.0f;
    if (e >= D.wco) {                                       // output neuron
        const int nlast = L > 1 ? D.nodes[L - 2] : D.nin, m = e - D.wco;
        if (m < nlast) v = W[D.woff[L - 1] + m];
        else if (m == vec_pad4(nlast)) v = W[D.boff[L - 1]];
    } else if (L > 1 && e >= D.wcb[0]) {                    // hidden-layer biases
        int l = 0;
        while (l + 1 < L - 1 && e >= D.wcb[l + 1]) ++l;
        const int j = e - D.wcb[l];
        if (j < D.nodes[l]) v = W[D.boff[l] + j];
    } else {                                                // weight rows
        int l = 0;
        while (l + 1 < L - 1 && e >= D.wcf[l + 1]) ++l;
        const int ni = l == 0 ? D.nin : D.nodes[l - 1], no = D.nodes[l];
        const int r = e - D.wcf[l], k = r / D.wcs[l], j = r % D.wcs[l];
        if (k < ni && j < no) v = W[D.woff[l] + k * no + j];
    }
    tab[e] = v;
}

__device__ __forceinline__ void wtrans_entry(const DevModel* __restrict__ dm, const float* __restrict__ W,
                                             float* __restrict__ tab, int seg, int e) {
    const int a = seg / kMaxLayers, l = seg % kMaxLayers;
    if (a >= dm->S) return;
    const NetDesc& D = dm->net[a];
    if (l >= D.nlayer - 1) return;
    const int ni = l == 0 ? D.nin : D.nodes[l - 1], no = D.nodes[l], ps = D.wts[l];
    if (e >= vec_pad4(no * ps)) return;
    const int j = e / ps, k = e % ps;
    tab[D.wtf[l] + e] = (j < no && k < ni) ? W[D.woff[l] + k * no + j] : 0.0f;
}

__global__ __launch_bounds__(256) void k_wtables(WTabArgs A) {
    const int e = blockIdx.x * blockDim.x + threadIdx.x;
    int y = blockIdx.y;
    if (A.tick && y == 0 && e == 0) *A.tick += 1;
    if (y < A.ys) { wsplit_entry(A.dm, A.W, A.split, y, e); return; }
    y -= A.ys;
    if (y < A.yc) { wchunk_entry(A.dm, A.W, A.chunk, y, e); return; }
    wtrans_entry(A.dm, A.W, A.trans, y - A.yc, e);
}

// All weight tables after a change of the FP32 weights (split: the matrix-core
// operand tables too); tick as in k_wtables.
hipError_t weight_tables(ann_ctx* ctx, int* tick, bool split) {
    const DevModel& M = ctx->hm;
    const int S = std::max(M.S, 1);
    int most = std::max(ctx->wchunk_max, 1);
    for (int a = 0; a < M.S; ++a)
        for (int l = 0; l < M.net[a].nlayer - 1; ++l) {
            const int ni = l == 0 ? M.net[a].nin : M.net[a].nodes[l - 1], no = M.net[a].nodes[l];
            if (split) {
                most = std::max(most, (ni + 31) / 32 * ((no + 15) / 16) * 3 * kWave);
                most = std::max(most, (no + 31) / 32 * ((ni + 15) / 16) * 3 * kWave);
            }
            most = std::max(most, vec_pad4(no * M.net[a].wts[l]));
        }
    WTabArgs A{ctx->dm, ctx->da.W, split ? ctx->d_wsplit : nullptr, ctx->d_wchunk, ctx->d_wtrans, tick,
               split ? S * 2 * kMaxLayers : 0, S};
    dim3 grid((most + 255) / 256, A.ys + A.yc + S * kMaxLayers);
    k_wtables<<<grid, 256, 0, ctx->stream>>>(A);
    const hipError_t e = hipGetLastError();
    if (e == hipSuccess) {
        if (split) ctx->wsplit_valid = true;
        ctx->wchunk_valid = true;
    }
    return e;
}

hipError_t split_weights(ann_ctx* ctx, int* tick) {
    // the vector-ALU network's tables follow every change of the weights (a
    // graph that captures a parameter update rebuilds them on every replay)
    return weight_tables(ctx, tick, true);
}

// NW wavefronts per 16-atom single-species tile, the column tiles of every
// product dealt round.  A batch of small structures has fewer tiles than the chip
// has SIMDs and a tile is a chain of short products, so latency is what counts:
// every product's weight operands are loaded a phase ahead, the inputs come
// straight into the split planes, and the output neuron and the first gradient
// share a phase.
// NT: column tiles of 16 of the widest hidden layer (4 up to 64 neurons, 8 up
// to 128), so narrow networks keep their registers and LDS.  Four wavefronts for 4
// column tiles, eight for 8: each then holds one tile's operands.  With two tiles'
// on four wavefronts 316 registers left one wavefront per SIMD; 128-128-1, us, before
// the loads ahead / four wavefronts / eight: 256 atoms 38 / 17 / 14.6, 6,144 atoms 41 /
// 32 / 20, 102,400 atoms 286 / 362 / 186; 128-1: 150 / 232 / 113.
// Against two wavefronts per tile that split the left operand at every product and
// loaded each operand where it was used, us: 192 atoms 22.6 -> 12.1, 2,048 atoms 22
// -> 12.4, 12,288 atoms 28.8 -> 17.3, 273,561 atoms 308 -> 248 (water 80-32-32-1),
// 21,872 Li/P/S atoms (96-48-48-1) 35.4 -> 25.6.
template <int NT, int NW>
__global__ __launch_bounds__(NW * kWave) void k_net_mfma(MfmaArgs A) {
    constexpr int W = 16 * NT;                  // widest hidden layer of this instance
    constexpr int NH = NT / NW;          // own column tiles of a hidden layer
    constexpr int NB = kMaxK / 16 / NW;  // own column tiles of the input side
    constexpr int KH = W / 32;                  // k blocks of a hidden layer
    constexpr int kThreads = NW * kWave;
    __shared__ __align__(16) PlaneRow X0[kTile], X1[kTile], X2[kTile];   // left operand, split
    __shared__ float act[kTile][W + 1];         // activations of the last hidden layer
    __shared__ float sdz[kMaxLayers - 1][kTile][W + 1];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid % kWave;
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int2 tl = A.tiles[t];
    const int a = tl.x;
    const int nrow = min(kTile, A.spend[a] - tl.y);
    const NetDesc& D = A.dm->net[a];
    const int L = D.nlayer, nin = D.nin;
    const float* iw = A.inpw + D.inoff;
    const float* ib = A.inpb + D.inoff;
    Operands<NH, kMaxK / 32, NW> wf;
    if (L > 1) wf.load(A.wtab + D.wsf[0], nin, D.nodes[0], wv);
    // a value and its right neighbour, split, into the planes
    auto put2 = [&](int r, int k, float x, float y) {
        __bf16 p[3], q[3];
        split3(x, p[0], p[1], p[2]);
        split3(y, q[0], q[1], q[2]);
        X0[r][k] = p[0]; X0[r][k + 1] = q[0];
        X1[r][k] = p[1]; X1[r][k + 1] = q[1];
        X2[r][k] = p[2]; X2[r][k + 1] = q[2];
    };
    auto put1 = [&](int r, int k, float x) {
        __bf16 p, q, u;
        split3(x, p, q, u);
        X0[r][k] = p;
        X1[r][k] = q;
        X2[r][k] = u;
    };
    // scaled input s = inpw (G + inpb): a wavefront takes every NW-th row, lanes two inputs each
    {
        const int k = 2 * lane;
        const bool in0 = k < nin, in1 = k + 1 < nin;
        const float w0 = in0 ? iw[k] : 0.0f, w1 = in1 ? iw[k + 1] : 0.0f;
        const float b0 = in0 ? ib[k] : 0.0f, b1 = in1 ? ib[k + 1] : 0.0f;
        float g0[kTile / NW], g1[kTile / NW];
#pragma unroll
        for (int q = 0; q < kTile / NW; ++q) {
            const int r = wv + q * NW;
            const float* G = A.G + (size_t)A.perm[tl.y + min(r, nrow - 1)] * A.ldg;
            g0[q] = in0 ? G[k] : 0.0f;
            g1[q] = in1 ? G[k + 1] : 0.0f;
        }
#pragma unroll
        for (int q = 0; q < kTile / NW; ++q) {
            const int r = wv + q * NW;
            const float x = r < nrow ? w0 * (g0[q] + b0) : 0.0f, y = r < nrow ? w1 * (g1[q] + b1) : 0.0f;
            put2(r, k, x, y);                               // zero past the inputs, up to kMaxK
        }
    }
    const int col = lane % 16, rb = 4 * (lane / 16);
    // thread (row, slot) of the phases that run over a row's neurons
    constexpr int SL = kThreads / kTile;
    const int orow = tid / SL, osl = tid % SL;
    const float* WL = A.W + D.woff[L - 1];
    if (L == 1) {
        // no hidden layer: the output neuron reads the scaled inputs
        float z = 0.0f;
        if (orow < nrow) {
            const float* G = A.G + (size_t)A.perm[tl.y + orow] * A.ldg;
            for (int m = osl; m < nin; m += SL) z += WL[m] * (iw[m] * (G[m] + ib[m]));
        }
#pragma unroll
        for (int o = SL / 2; o > 0; o >>= 1) z += __shfl_xor(z, o);
        if (orow < nrow && osl == 0) A.Eatom[A.perm[tl.y + orow]] = D.outb + D.outw * (A.W[D.boff[0]] + z);
        if (!A.dEdG) return;
        for (int q = tid; q < kTile * A.ldg; q += kThreads) {
            const int r = q / A.ldg, m = q % A.ldg;
            if (r < nrow) A.dEdG[(size_t)A.perm[tl.y + r] * A.ldg + m] = m < nin ? D.outw * WL[m] * iw[m] : 0.0f;
        }
        return;
    }
    int ni = nin;
    for (int l = 0; l < L - 1; ++l) {
        const int no = D.nodes[l];
        const float* bl = A.W + D.boff[l];
        float bias[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const int n = (h * NW + wv) * 16 + col;
            bias[h] = n < no ? bl[n] : 0.0f;
        }
        __syncthreads();                                    // the planes are written
        f32x4 acc[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        wf.mul(X0, X1, X2, ni, no, wv, acc);
        if (l + 1 < L - 1) wf.load(A.wtab + D.wsf[l + 1], no, D.nodes[l + 1], wv);
        __syncthreads();                                    // the planes are read
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const int n = (h * NW + wv) * 16 + col;
            float av[4] = {0.f, 0.f, 0.f, 0.f}, dv[4] = {0.f, 0.f, 0.f, 0.f}, d2[4];
            if ((h * NW + wv) * 16 < no) {
                float z[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) z[i] = acc[h][i] + bias[h];
                act_many<false, 4>(D.neuron, D.c, z, av, dv, d2);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float x = n < no ? av[i] : 0.0f;
                put1(rb + i, n, x);                         // zero past the neurons, up to W
                act[rb + i][n] = x;
                sdz[l][rb + i][n] = n < no ? dv[i] : 0.0f;
            }
        }
        ni = no;
    }
    using OpHidden = Operands<NH, KH, NW>;
    using OpInput = Operands<NB, KH, NW>;
    OpHidden wbh;                                           // backward through hidden layers
    OpInput wbi;                                            // and through the input layer
    // where the shapes agree they share registers: one is loaded when the other is used up
    OpInput& wb0 = [&]() -> OpInput& {
        if constexpr (std::is_same_v<OpHidden, OpInput>) return wbh;
        else return wbi;
    }();
    const bool grad = A.dEdG != nullptr;
    if (grad) {
        if (L > 2) wbh.load(A.wtab + D.wsb[L - 2], ni, D.nodes[L - 3], wv);
        else wb0.load(A.wtab + D.wsb[0], ni, nin, wv);
    }
    __syncthreads();
    // linear output neuron, and g_{L-1} = outw W_L . sigma'_{L-1} into the planes
    {
        if (grad)
            for (int m = osl; m < W; m += SL) put1(orow, m, m < ni ? D.outw * WL[m] * sdz[L - 2][orow][m] : 0.0f);
        // one lane per atom, terms in order: atoms in like environments round alike, so
        // the order of this sum shows in a structure's energy
        if (tid < nrow) {
            float z = A.W[D.boff[L - 1]];
            for (int m = 0; m < ni; ++m) z += WL[m] * act[tid][m];
            A.Eatom[A.perm[tl.y + tid]] = D.outb + D.outw * z;
        }
    }
    if (!grad) return;
    for (int l = L - 2; l >= 1; --l) {
        const int no = D.nodes[l], nprev = D.nodes[l - 1];
        __syncthreads();
        f32x4 acc[NH];
#pragma unroll
        for (int h = 0; h < NH; ++h) acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        wbh.mul(X0, X1, X2, no, nprev, wv, acc);
        if (l > 1) wbh.load(A.wtab + D.wsb[l - 1], nprev, D.nodes[l - 2], wv);
        else wb0.load(A.wtab + D.wsb[0], nprev, nin, wv);
        __syncthreads();
#pragma unroll
        for (int h = 0; h < NH; ++h) {
            const int m = (h * NW + wv) * 16 + col;
#pragma unroll
            for (int i = 0; i < 4; ++i) put1(rb + i, m, m < nprev ? acc[h][i] * sdz[l - 1][rb + i][m] : 0.0f);
        }
    }
    {
        float iwm[NB];
#pragma unroll
        for (int h = 0; h < NB; ++h) {
            const int m = (h * NW + wv) * 16 + col;
            iwm[h] = m < nin ? iw[m] : 0.0f;
        }
        __syncthreads();
        f32x4 acc[NB];
#pragma unroll
        for (int h = 0; h < NB; ++h) acc[h] = f32x4{0.f, 0.f, 0.f, 0.f};
        wb0.mul(X0, X1, X2, D.nodes[0], nin, wv, acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = rb + i;
            if (r >= nrow) continue;
            float* out = A.dEdG + (size_t)A.perm[tl.y + r] * A.ldg;
#pragma unroll
            for (int h = 0; h < NB; ++h) {
                const int m = (h * NW + wv) * 16 + col;
                if (m < A.ldg) out[m] = m < nin ? acc[h][i] * iwm[h] : 0.0f;
            }
        }
    }
}

hipError_t net_fwd_mfma(ann_ctx* ctx, const float* G, float* Eatom, float* dEdG, const float* inpb) {
    hipError_t e = species_perm(ctx);
    if (e != hipSuccess) return e;
    MfmaArgs A{};
    A.dm = ctx->dm;
    A.W = ctx->da.W;
    A.inpw = ctx->da.inpw;
    A.inpb = inpb;
    A.ldg = ctx->ldg;
    A.perm = ctx->d_perm;
    A.tiles = reinterpret_cast<const int2*>(ctx->d_tiles);
    A.spend = ctx->d_spend_end;
    A.ntiles = ctx->ntiles;
    A.G = G;
    A.Eatom = Eatom;
    A.dEdG = dEdG;
    A.wtab = ctx->d_wsplit;
    if (A.ntiles == 0) return hipSuccess;
    if (!ctx->wsplit_valid && (e = split_weights(ctx, nullptr)) != hipSuccess) return e;
    int wmax = 1;
    for (int a = 0; a < ctx->hm.S; ++a)
        for (int l = 0; l < ctx->hm.net[a].nlayer - 1; ++l) wmax = std::max(wmax, ctx->hm.net[a].nodes[l]);
    Launch L(ctx, "net_mfma");
    if (wmax <= 64) k_net_mfma<4, 4><<<A.ntiles, 4 * kWave, 0, ctx->stream>>>(A);
    else k_net_mfma<8, 8><<<A.ntiles, 8 * kWave, 0, ctx->stream>>>(A);
    return hipGetLastError();
}

bool mfma_net_supported(const DevModel& M) {
    for (int a = 0; a < M.S; ++a) {
        if (M.net[a].nin > kMaxK) return false;
        for (int l = 0; l < M.net[a].nlayer; ++l)
            if (M.net[a].nodes[l] > kMaxWidth) return false;
    }
    return true;
}

}  // namespace ann
