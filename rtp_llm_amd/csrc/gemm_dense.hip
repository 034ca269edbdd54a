// Dense linear layers on weights kept in checkpoint layout: y[M, N] = x[M, K] . W[N, K]^T with W row-major [out, in].
//
// Both operands are contiguous along K, which is the layout v_mfma_f32_16x16x32_bf16 wants for its A and B fragments (8 consecutive k per
// lane), so no weight image is built: a model whose layers have many small, differently shaped projections (recurrent gates, low-rank
// decays, shared-KV attention) loads its tensors as they are.  Three kernels, all with fp32 accumulation and an fp32 epilogue:
//   * tile kernels, bf16: block tiles of 64 x 128 up to 256 x 256, both operands through LDS by DMA, MFMA 16x16x32; one that stages 64 x 128 through registers
//     for operands without 16-byte alignment;
//   * tile kernel, fp32:  64 x 64 block tile, 4 x 4 register micro-tiles, true fp32 FMAs (no reduced-precision matrix mode);
//   * skinny kernel, bf16, 2 <= M <= 16: one block per 8 weight rows, its waves split K, both operands through LDS in runs of 1 KB a row;
//   * row kernel (M = 1; fp32 up to M = 16): a wave per output column streams its weight row once, 16-byte loads, wave reduction at the end.
//   * grouped forms of these kernels (per-head or per-branch weights over column slices; rows sorted by expert with a gather and a tile
//     list; the few rows of a decode step, each with its own expert's weight): mi355_dense_grouped.
// Epilogues: bias, gated activation act(gate) * up (weight rows grouped [32 gate | 32 up], so one lane holds both; also the clamped form
// min(g, L) sigmoid(1.702 min(g, L)) (clamp(u, -L, L) + 1)), an activation of the plain output (also the square of relu), tanh soft cap.
// Output is fp32 or the activation type.  A result row depends only on its own input row: the k order of the accumulation is fixed by
// the kernel, never by M or by the row's place in the batch.
#include "common.h"
#include "hybrid_recur.h"
#include "../../include/mi355_hybrid.h"

// The tile shape of a bf16 call of M x N x K through `groups` weights (64-row tiles of sorted rows in `row_tiles`, 0: all M rows through each): 0 64x64, 1 64x128 in three stages,
// 2 64x128 in two, 3 128x128, 4 256x256.  The one with the least expected time, us per 32 columns of k: a constant and the blocks per CU times what one costs a busy CU (256 x 256:
// whole rounds count half, one block fills a CU; 64x128 in three stages: two blocks fill one).  Measured at M = 70..8192, N = 16..32000, K = 16..5632: within 10 % of the fastest.
// Grouped rows come in tiles of 64.
extern "C" int mi355_dense_tile_shape(int32_t M, int32_t N, int32_t K, int32_t groups, int32_t row_tiles) {
    auto share = [&](int bm, int bn) { return (double)((N + bn - 1) / bn) * (row_tiles ? row_tiles : (M + bm - 1) / bm) * groups / 256.0; };
    const double sa = share(256, 256), sb = share(128, 128), sc = share(64, 128), se = share(64, 64), k = K / 32.0;
    const double ta = row_tiles ? 1e30 : k * fmax(0.65, 0.475 * (sa + ceil(sa))) + 12.0, tb = row_tiles ? 1e30 : k * fmax(0.34, 0.255 * sb + 0.13) + 5.0;
    const double tc = k * fmax(0.27, 0.15 * sc + 0.09) + 4.0, td = k * (sc <= 2.0 ? 0.18 + 0.06 * sc : 0.15 * sc + 0.22) + 4.0;
    const double te = k * fmax(0.125, 0.105 * se + 0.02) + 4.0, t = fmin(fmin(ta, tb), fmin(tc, fmin(td, te)));
    return t == te ? 0 : t == td ? 1 : t == tc ? 2 : t == tb ? 3 : 4;
}

namespace {

constexpr int DN_ACT_NONE = 0, DN_ACT_RELU = 1, DN_ACT_SILU = 2, DN_ACT_GELU_TANH = 3, DN_ACT_TANH = 4, DN_ACT_SWIGLU_CLAMP = 5, DN_ACT_RELU2 = 6;

struct DenseParams {
    const void* x; const void* w; const void* bias; void* y;
    int M, N, K, ldx, ldy;
    int gated;       // 0: N outputs; 1: rows of w are [32 gate | 32 up] groups, N / 2 outputs
    int act;         // DN_ACT_* applied to the gate
    float act_param; // DN_ACT_SWIGLU_CLAMP: the limit of the gate (from above) and of the up value (both sides)
    int out_f32;
    float softcap;   // > 0: y = cap * tanh(y / cap)
    int vec;         // 16-byte loads allowed (alignment and K % 8 == 0 checked on the host)
    int yvec;        // four consecutive outputs of a row that start at a multiple of four may be stored together (ldy % 4 == 0, y aligned)
    // groups (tile kernels, blockIdx.z): group g multiplies its rows by the weight w + g * ws (bias + g * N) and writes columns ys * g + ...
    // of y; it reads x from column xs * g on.  Its rows are all M rows, or rows offs[g] .. offs[g + 1] - 1 of a list sorted by group, whose
    // entry r reads x row gather[r] (identity without gather) and writes y row r.  tiles (with offs): {count, (group, first row) x count}, the
    // 64-row tiles that hold rows; the row tile indexes this list instead of (blockIdx.z, row tile), so no block is spent on a tile without rows.
    int G;
    long long xs, ws, ys;
    const int32_t* offs; const int32_t* gather; const int32_t* tiles;
    // y[row, col] is multiplied by sigmoid(egate[row * ldg + goff + col]) before it is stored (fp32 pre-activations; null: no gate)
    const float* egate; int ldg, goff;
    // a weight that a later launch streams (its lines of 128 bytes): blocks past the list of tiles read one word of each
    const char* ahead = nullptr; uint32_t ahead_lines = 0;
    int streamed = 0;    // MI355_DENSE_STREAMED (host only)
};

// The chip deals consecutive blocks to its eight XCDs in turn, each with an L2 of its own.  The (column tile, row tile) pair of a block is chosen such
// that an XCD walks a contiguous run of tiles in an order of bands of DN_BAND row tiles, column by column: its blocks share the band's rows of x and read
// every weight column of the run once.
constexpr int DN_XCD = 8, DN_BAND = 16;
template <int BAND>
__device__ __forceinline__ void dn_block_tile(int gx, int gy, int& bx, int& by) {
    const int nb = gx * gy, id = blockIdx.y * gridDim.x + blockIdx.x;
    if (id >= nb) { bx = 0; by = gy; return; }               // a block past the list of tiles
    const int k = id % DN_XCD, j = k * (nb / DN_XCD) + min(k, nb % DN_XCD) + id / DN_XCD;
    const int band = j / (gx * BAND), rest = j - band * gx * BAND, h = min(BAND, gy - band * BAND);
    bx = rest / h; by = band * BAND + rest % h;
}

// the block's column tile, first row and end of the rows of its tile in its group, and the group's operand bases
struct DnGroup { int bx, m0, rend; long long xo, wo, yo; int bo; };
template <int BAND = DN_BAND>
__device__ __forceinline__ DnGroup dn_group(const DenseParams& p, int tile_rows) {
    int g = blockIdx.z, by;
    DnGroup r;
    dn_block_tile<BAND>(gridDim.x, p.tiles ? p.tiles[0] : gridDim.y, r.bx, by);
    if (p.tiles) {
        if (by >= p.tiles[0]) { r.m0 = r.rend = 0; return r; }
        g = p.tiles[1 + 2 * by]; r.m0 = p.tiles[2 + 2 * by]; r.rend = p.offs[g + 1];
    } else {
        r.m0 = (p.offs ? p.offs[g] : 0) + by * tile_rows; r.rend = p.offs ? p.offs[g + 1] : p.M;
    }
    r.xo = p.xs * g; r.wo = p.ws * g; r.yo = p.ys * g; r.bo = g * p.N;
    return r;
}

// A block past the list of tiles (of one group only in z): its share of the lines of p.ahead, four loads at a time.  The list is bounded by rows / 64 + groups tiles, so about half
// as many rows of blocks as there are groups are left over, and they run while the launch multiplies and HBM is idle: 16 experts 1024 -> 704 -> 1024 over 6148 rows, the second linear
// 31.6 -> 24.2 us, the first no slower.  They are dealt last, and of few experts there may be one row of them or none, so a thread reads DN_AHEAD_ROUNDS times four lines and no more: shared
// out over however many blocks are left, one row of 16 read 3 MB a CU behind a finished product (64 experts of 384, 364 pairs: sort and linears 49.7 us without, 66.7 so, 51.2 so bounded).
constexpr int DN_AHEAD_ROUNDS = 4;
__device__ __forceinline__ void dn_read_ahead(const DenseParams& p) {
    const uint32_t used = gridDim.x * (uint32_t)p.tiles[0], n = (gridDim.x * gridDim.y - used) * blockDim.x;
    uint32_t i = (blockIdx.y * gridDim.x + blockIdx.x - used) * blockDim.x + threadIdx.x;
#pragma unroll 1
    for (int r = 0; r < DN_AHEAD_ROUNDS && i < p.ahead_lines; ++r, i += 4 * n) {
        uint32_t v[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = i + k * n < p.ahead_lines ? *(const uint32_t*)(p.ahead + (size_t)(i + k * n) * 128) : 0u;
#pragma unroll
        for (int k = 0; k < 4; ++k) asm volatile("" :: "v"(v[k]));
    }
}

__device__ __forceinline__ float dn_act(float g, int act) {
    if (act == DN_ACT_RELU) return g > 0.f ? g : 0.f;
    if (act == DN_ACT_SILU) return g / (1.f + __expf(-g));
    if (act == DN_ACT_GELU_TANH) return 0.5f * g * (1.f + tanhf(0.7978845608028654f * (g + 0.044715f * g * g * g)));
    if (act == DN_ACT_TANH) return tanhf(g);
    if (act == DN_ACT_RELU2) { const float r = g > 0.f ? g : 0.f; return r * r; }
    return g;
}

// act(gate) * up of a gated pair.  DN_ACT_SWIGLU_CLAMP: g' = min(g, L), u' = clamp(u, -L, L), g' sigmoid(1.702 g') (u' + 1).
__device__ __forceinline__ float dn_gated(float g, float u, int act, float lim) {
    if (act == DN_ACT_SWIGLU_CLAMP) {
        g = fminf(g, lim); u = fminf(fmaxf(u, -lim), lim);
        return g / (1.f + expf(-1.702f * g)) * (u + 1.f);
    }
    return dn_act(g, act) * u;
}

template <typename T> __device__ __forceinline__ float dn_ld(const T* p) { return (float)*p; }

template <typename T>
__device__ __forceinline__ void dn_store(const DenseParams& p, int row, int col, float v) {
    if (p.softcap > 0.f) v = p.softcap * tanhf(v / p.softcap);
    if (p.egate) v *= 1.f / (1.f + expf(-p.egate[(size_t)row * p.ldg + p.goff + col]));
    if (p.out_f32) ((float*)p.y)[(size_t)row * p.ldy + col] = v;
    else           ((T*)p.y)[(size_t)row * p.ldy + col] = (T)v;
}

// four consecutive outputs of one row (cnt of them exist)
__device__ __forceinline__ void dn_store4(const DenseParams& p, int row, int col, f32x4 v, int cnt) {
    if (p.softcap > 0.f) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = p.softcap * tanhf(v[e] / p.softcap);
    }
    if (p.egate) {
#pragma unroll
        for (int e = 0; e < 4; ++e) if (e < cnt) v[e] *= 1.f / (1.f + expf(-p.egate[(size_t)row * p.ldg + p.goff + col + e]));
    }
    const size_t at = (size_t)row * p.ldy + col;
    if (p.out_f32) {
        float* y = (float*)p.y + at;
        if (cnt == 4 && p.yvec && !(col & 3)) *(f32x4*)y = v;
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (e < cnt) y[e] = v[e];
        }
    } else {
        bf16* y = (bf16*)p.y + at;
        if (cnt == 4 && p.yvec && !(col & 3)) { u32x2 o = {act_pack<true>(v[0], v[1]), act_pack<true>(v[2], v[3])}; *(u32x2*)y = o; }
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (e < cnt) y[e] = (bf16)v[e];
        }
    }
}

// ------------------------------------------------------------------------------------------------ bf16 tile kernel
constexpr int TB_M = 64, TB_N = 128, TB_K = 64, TB_LD = TB_K + 8;   // LDS row stride in elements (144 bytes: 16-byte aligned)

__device__ __forceinline__ u32x4 dn_chunk_bf16(const bf16* base, int row, int rows, int k, int K, int ld, int vec) {
    u32x4 z = {0u, 0u, 0u, 0u};
    if (row >= rows || k >= K) return z;     // row 0x7fffffff: no row
    const bf16* p = base + (size_t)row * ld + k;
    if (vec) return *(const u32x4*)p;
    uint16_t e[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) e[i] = (k + i < K) ? __builtin_bit_cast(uint16_t, p[i]) : (uint16_t)0;
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (uint32_t)e[2 * i] | ((uint32_t)e[2 * i + 1] << 16);
    return r;
}

__global__ __launch_bounds__(256) void dense_tile_bf16_kernel(DenseParams p) {
    __shared__ __attribute__((aligned(16))) bf16 As[TB_M * TB_LD];
    __shared__ __attribute__((aligned(16))) bf16 Bs[TB_N * TB_LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;                       // wave tile: rows wm*32.., cols wn*64..
    const DnGroup gr = dn_group(p, TB_M);
    const int m0 = gr.m0, n0 = gr.bx * TB_N;
    if (m0 >= gr.rend) return;
    const bf16* X = (const bf16*)p.x + gr.xo;
    const bf16* W = (const bf16*)p.w + gr.wo;
    const bf16* Bi = p.bias ? (const bf16*)p.bias + gr.bo : nullptr;
    int arow[2];                                                   // x rows this thread stages (past the group's end: none)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int r = m0 + ((tid + i * 256) >> 3);
        arow[i] = r < gr.rend ? (p.gather ? p.gather[r] : r) : 0x7fffffff;
    }
    f32x4 acc[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // staging: chunk c of 8 elements; A has 64 x 8 chunks (2 per thread), B 128 x 8 (4 per thread)
    u32x4 ra[2], rb[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 2; ++i) { const int c = tid + i * 256; ra[i] = dn_chunk_bf16(X, arow[i], 0x7fffffff, k0 + (c & 7) * 8, p.K, p.ldx, p.vec); }
#pragma unroll
        for (int i = 0; i < 4; ++i) { const int c = tid + i * 256; rb[i] = dn_chunk_bf16(W, n0 + (c >> 3), p.N, k0 + (c & 7) * 8, p.K, p.K, p.vec); }
    };
    fetch(0);
    for (int k0 = 0; k0 < p.K; k0 += TB_K) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 2; ++i) { const int c = tid + i * 256; *(u32x4*)&As[(c >> 3) * TB_LD + (c & 7) * 8] = ra[i]; }
#pragma unroll
        for (int i = 0; i < 4; ++i) { const int c = tid + i * 256; *(u32x4*)&Bs[(c >> 3) * TB_LD + (c & 7) * 8] = rb[i]; }
        __syncthreads();
        if (k0 + TB_K < p.K) fetch(k0 + TB_K);
#pragma unroll
        for (int ks = 0; ks < TB_K; ks += 32) {
            const int kk = ks + (lane >> 4) * 8, r = lane & 15;
            bf16x8 a[2], b[4];
#pragma unroll
            for (int i = 0; i < 2; ++i) a[i] = *(const bf16x8*)&As[(wm * 32 + i * 16 + r) * TB_LD + kk];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *(const bf16x8*)&Bs[(wn * 64 + j * 16 + r) * TB_LD + kk];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
        }
    }
    // C fragment: lane holds column (lane & 15), rows 4 * (lane >> 4) + e
    const int cl = lane & 15, rq = (lane >> 4) * 4;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = m0 + wm * 32 + i * 16 + rq + e;
            if (row >= gr.rend) continue;
            if (p.gated) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int ng = n0 + wn * 64 + j * 16 + cl;         // weight row of the gate; its up row is ng + 32
                    if (ng + 32 >= p.N) continue;
                    float g = acc[i][j][e], u = acc[i][j + 2][e];
                    if (Bi) { g += dn_ld(Bi + ng); u += dn_ld(Bi + ng + 32); }
                    dn_store<bf16>(p, row, (int)gr.yo + (ng >> 6) * 32 + (ng & 31), dn_gated(g, u, p.act, p.act_param));
                }
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int n = n0 + wn * 64 + j * 16 + cl;
                    if (n >= p.N) continue;
                    float v = acc[i][j][e];
                    if (Bi) v += dn_ld(Bi + n);
                    dn_store<bf16>(p, row, (int)gr.yo + n, dn_act(v, p.act));
                }
            }
        }
}

// ------------------------------------------------------------------------------------------------ bf16 tile kernel, LDS-DMA staging
// BM rows of x by BN rows of w per block, K in tiles of BK; waves of WM x WN outputs.  Both operands go to LDS by `global_load_lds_dwordx4` (no staging registers, no
// ds_write) into NS stages, one barrier per tile.  An LDS row is the BK * 2 bytes of a K tile; its 16-byte pieces are permuted by the row (applied to the source
// address, which the DMA leaves free per lane), so that the 16-row fragment reads hit every bank once.  w is the MFMA's first operand: a lane ends with four
// consecutive outputs of one row.  The sums run over k in steps of 32 like the other tile kernel's: same bits.
// BK = 64: NS = 2, two blocks or more per CU hide each other's waits; NS = 3 and 4 where few blocks have to keep the loads in flight alone.  BK = 32: a wave reads the
// fragments of tile t + 1 between the products of tile t.
// Time in us of 256x256 (BK 32, NS 4) / 128x128 (NS 2) / 64x128 (NS 2) / 64x128 (NS 3) / 64x64 (NS 4) tiles and of the 64x128 kernel that stages through registers;
// weights not in L2, as in a model:
//   M x N x K       8192x2048x2048 62 / 71 / 82 / 86 / 112, 118    6148x1408x1024 gated 33 / 31 / 29 / 32 / 37, 43     768x11264x2048 gated 50 / 52 / 49 / 53 / 61, 73
//                   1537x2176x1024 30 / 15 / 14 / 13 /  17,  25    1537x1024x1024       29 / 15 / 13 / 11 / 10, 21     768x2048x5632       109 / 57 / 52 / 36 / 34, 77
//                   1537x3072x1024 30 / 20 / 18 / 21 /  22,  30    1537x1024x2816       60 / 32 / 29 / 21 / 20, 45      70x2048x2048        42 / 23 / 20 / 16 / 12, 32
template <int BM, int BN, int WM, int WN, int BK, int NS>
__global__ __launch_bounds__(64 * (BM / WM) * (BN / WN), 2) void dense_dma_bf16_kernel(DenseParams p) {
    constexpr int NWM = BM / WM, NWN = BN / WN, NW = NWM * NWN, MI = WM / 16, NJ = WN / 16;
    constexpr bool AHEAD = BK == 32;                                          // fragments of tile t + 1 are read while tile t is multiplied
    constexpr int RB = BK * 2, PPR = BK / 8, RPL = 64 / PPR;                  // bytes and 16-byte pieces of a row, rows per wave load
    constexpr int STAGE = (BM + BN) * RB, ULD = (BM + BN) / (RPL * NW), ULA = BM / (RPL * NW);   // loads per wave and tile; the first ULA are rows of x
    static_assert((AHEAD ? NS >= 3 : BK == 64) && BM % (RPL * NW) == 0 && BN % (RPL * NW) == 0, "whole wave loads per operand");
    constexpr int PH = MI >= 4 && NS * STAGE >= NW * 16384 ? 4 : MI >= 2 ? 2 : 1;   // 16-row blocks of results that pass through LDS together
    static_assert(WN == 64 && NS * STAGE >= NW * PH * 4096, "a wave's output columns; room for its results");
    __shared__ __attribute__((aligned(1024))) char smem[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % NWM, wn = wave / NWM;
    const DnGroup gr = dn_group<1024 / BM>(p, BM);
    const int m0 = gr.m0, n0 = gr.bx * BN;
    if (m0 >= gr.rend) {
        if (p.ahead_lines) dn_read_ahead(p);
        return;
    }
    const bf16* X = (const bf16*)p.x + gr.xo + (p.gather ? 0 : (size_t)m0 * p.ldx);
    const bf16* W = (const bf16*)p.w + gr.wo + (size_t)n0 * p.K;
    // lane l of a wave load owns row (l >> 3) of its eight, LDS piece l & 7 = source piece (l & 7) ^ (row & 7); rows past the end repeat the last one
    auto swizzle = [](int row) { return BK == 64 ? row & 7 : (row >> 1) & 3; };
    const int lr = lane / PPR, piece = (lane % PPR) ^ swizzle(lr);
    uint32_t voff[ULD];
    int xrow[ULA];
#pragma unroll
    for (int u = 0; u < ULD; ++u) {
        const int r = ((u < ULA ? u : u - ULA) * NW + wave) * RPL + lr;
        if (u < ULA) {
            const int m = min(m0 + r, gr.rend - 1);
            xrow[u] = p.gather ? p.gather[m] : m - m0;
            voff[u] = (uint32_t)xrow[u] * (uint32_t)p.ldx * 2u + piece * 16u;
        } else {
            voff[u] = (uint32_t)min(r, p.N - 1 - n0) * (uint32_t)p.K * 2u + piece * 16u;
        }
    }
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem);
    auto issue1 = [&](int buf, int kt, int u) {
        dma16(lds0 + buf * STAGE + (u < ULA ? 0 : BM * RB) + ((u < ULA ? u : u - ULA) * NW + wave) * 1024, voff[u], u < ULA ? X + kt * BK : W + kt * BK);
    };
    auto issue = [&](int buf, int kt) {
#pragma unroll
        for (int u = 0; u < ULD; ++u) issue1(buf, kt, u);
    };
    f32x4 acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int fr = lane & 15, q = lane >> 4;
    struct Frags { bf16x8 w[NJ], x[MI]; };
    auto load = [&](Frags& f, int buf, int ks) {
        const int foff = (((ks * 4 + q) ^ swizzle(fr)) << 4) + fr * RB;
        const char* xs = smem + buf * STAGE + wm * WM * RB + foff;
        const char* ws = smem + buf * STAGE + (BM + wn * WN) * RB + foff;
#pragma unroll
        for (int j = 0; j < NJ; ++j) f.w[j] = *(const bf16x8*)(ws + j * 16 * RB);
#pragma unroll
        for (int i = 0; i < MI; ++i) f.x[i] = *(const bf16x8*)(xs + i * 16 * RB);
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[j], f.x[i], acc[i][j], 0, 0, 0);
    };
    const int nk = p.K / BK;
    Frags fa, fb;
#pragma unroll
    for (int t = 0; t < NS - 1; ++t) if (t < nk) issue(t, t);
    if constexpr (!AHEAD) {
        int at = 0;
        for (int kt = 0; kt < nk; ++kt) {
            // this wave's part of tile kt is in LDS, its reads of tile kt - 1 are done
            if (NS == 2 || kt + NS - 2 >= nk) wait_vm<0>(); else wait_vm<ULD * (NS - 2)>();
            __builtin_amdgcn_s_barrier();
            if (kt + NS - 1 < nk) issue(at == 0 ? NS - 1 : at - 1, kt + NS - 1);
#pragma unroll
            for (int ks = 0; ks < BK / 32; ++ks) { load(fa, at, ks); multiply(fa); }
            at = at + 1 == NS ? 0 : at + 1;
        }
    } else {
        if (nk > 0) {
            if (nk >= NS - 1) wait_vm<ULD * (NS - 2)>(); else wait_vm<0>();
            __builtin_amdgcn_s_barrier();
            load(fa, 0, 0);
        }
        int next = 1, ahead = NS - 1, kt = 0;                               // stages of tile kt + 1 and of tile kt + NS - 1
        // IN_FLIGHT: tile kt + 1 is in LDS once at most that many of the wave's loads are left; its reads of tile kt are done by then, so behind the barrier
        // tile kt + NS - 1 may go over tile kt - 1
        auto advance = [&](Frags& nxt, auto in_flight, bool more) {
            wait_vm<decltype(in_flight)::value>();
            __builtin_amdgcn_s_barrier();
            if (more) issue(ahead, kt + NS - 1);
            load(nxt, next, 0);
            next = next + 1 == NS ? 0 : next + 1;
            ahead = ahead + 1 == NS ? 0 : ahead + 1;
        };
        constexpr std::integral_constant<int, ULD * (NS - 3)> steady{};
        // One tile in ULD parts: a load of tile kt + NS - 1, its share of the reads of tile kt + 1, its share of tile kt's products, and nothing across a part's end.  Asked for at once behind the
        // barrier, the block's 32 loads of 16 cycles each stood in front of every wave's products: 1720 cycles a tile instead of the 1024 of the products.
        constexpr int RP = (MI + NJ + ULD - 1) / ULD, MP = MI / ULD;
        static_assert(!AHEAD || MI % ULD == 0, "whole rows of products a part");
        auto tile = [&](const Frags& cur, Frags& nxt) {
            wait_vm<decltype(steady)::value>();
            __builtin_amdgcn_s_barrier();
            const int foff = ((q ^ swizzle(fr)) << 4) + fr * RB;
            const char* xs = smem + next * STAGE + wm * WM * RB + foff;
            const char* ws = smem + next * STAGE + (BM + wn * WN) * RB + foff;
#pragma unroll
            for (int u = 0; u < ULD; ++u) {
                issue1(ahead, kt + NS - 1, u);
#pragma unroll
                for (int g = u * RP; g < (u + 1) * RP && g < MI + NJ; ++g) {
                    if (g < NJ) nxt.w[g] = *(const bf16x8*)(ws + g * 16 * RB);
                    else        nxt.x[g - NJ] = *(const bf16x8*)(xs + (g - NJ) * 16 * RB);
                }
#pragma unroll
                for (int i = u * MP; i < (u + 1) * MP; ++i)
#pragma unroll
                    for (int j = 0; j < NJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.w[j], cur.x[i], acc[i][j], 0, 0, 0);
#pragma unroll
                for (int g = 0; g < RP; ++g) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, MP * NJ / RP, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x008, MP * NJ, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
            next = next + 1 == NS ? 0 : next + 1;
            ahead = ahead + 1 == NS ? 0 : ahead + 1;
            ++kt;
        };
        while (kt + NS < nk) {                                              // no conditions inside: the compiler's own waits stay as late as they can be
            tile(fa, fb);
            tile(fb, fa);
        }
        for (; kt < nk; ++kt) {
            if (kt + 1 < nk) {
                if (kt + NS - 1 < nk) advance(fb, steady, true); else advance(fb, std::integral_constant<int, 0>{}, false);
            }
            multiply(fa);
            if (kt + 1 < nk) fa = fb;
        }
    }
    if (p.K % BK) {                                                         // the last K % BK columns: through registers, zeros behind them
        __syncthreads();
#pragma unroll
        for (int u = 0; u < ULD; ++u) {
            u32x4 v = {0u, 0u, 0u, 0u};
            const char* src = (const char*)(u < ULA ? X : W) + voff[u] + (size_t)nk * RB;
            if (nk * BK + piece * 8 < p.K) v = *(const u32x4*)src;
            *(u32x4*)(smem + (u < ULA ? 0 : BM * RB) + ((u < ULA ? u : u - ULA) * NW + wave) * 1024 + lane * 16) = v;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < BK / 32; ++ks) { load(fa, 0, ks); multiply(fa); }
    }
    // Results through LDS, up to 64 rows of a wave's 64 columns at a time: a lane holds four outputs (4 q + e of 16) of row fr, and reads back four consecutive ones of a
    // row that its 15 neighbours continue -- whole 256-byte runs per store, and ONE copy of the epilogue's code (unrolled over the 32 fragments it did not fit the
    // instruction cache: 46 of the 93 us of an 8192 x 2048 x 2048 product).  16-byte pieces permuted by the row.
    const bf16* Bi = p.bias ? (const bf16*)p.bias + gr.bo : nullptr;
    char* mine = smem + wave * (PH * 4096);
    const int nc = n0 + wn * WN;                                            // the wave's first weight row
    // What most calls ask for has code of its own: the choice among activations, caps, gates and output types a value took 1400 cycles a trip of the general loops (8192 x 11264 x 2048
    // gated: 11 of a block's 67 us, 3.6 now; all of it 359 / 325 us, 1537 x 1408 x 1024 gated 14.2 / 11.8, 456 x 11264 x 2048 gated 41.3 / 39.1, 1537 x 2176 x 1024 15.3 / 14.5).
    const bool lean = p.softcap <= 0.f && p.yvec && p.N % 4 == 0;
    const bool lean_gated = lean && p.gated && !p.egate && !Bi && !p.out_f32 && (p.act == DN_ACT_RELU || p.act == DN_ACT_SILU) && p.ldy % 8 == 0 && (uintptr_t)p.y % 16 == 0 && gr.yo % 8 == 0;
    const bool lean_plain = lean && !p.gated && !p.egate && p.out_f32 && p.act == DN_ACT_NONE && gr.yo % 4 == 0;
    const bool lean_scaled = lean && !p.gated && p.egate && !Bi && !p.out_f32 && p.act == DN_ACT_NONE && gr.yo % 4 == 0 && p.ldg % 4 == 0 && p.goff % 4 == 0 && (uintptr_t)p.egate % 16 == 0;
    __syncthreads();
#pragma unroll
    for (int i0 = 0; i0 < MI; i0 += PH) {
#pragma unroll
        for (int i = 0; i < PH; ++i)
#pragma unroll
            for (int j = 0; j < NJ; ++j) *(f32x4*)(mine + (i * 16 + fr) * 256 + (((j * 4 + q) ^ fr) << 4)) = acc[i0 + i][j];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                  // the wave's own stores, read by its other lanes
        const int r0 = m0 + wm * WM + i0 * 16, rows = min(PH * 16, gr.rend - r0);
        if (lean_gated) {                                                   // 8 channels a lane, 4 lanes a row: 16 bytes a store
            const int c8 = lane & 3, c = nc + c8 * 8;
            bf16* y = (bf16*)p.y + (size_t)(r0 + (lane >> 2)) * p.ldy + (int)gr.yo + (nc >> 1) + c8 * 8;
            auto out = [&](auto gate) {
#pragma unroll
                for (int k = 0; k < PH; ++k) {
                    const int r = k * 16 + (lane >> 2);
                    const char* at = mine + r * 256;
                    f32x4 g[2], u[2];
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        g[h] = *(const f32x4*)(at + (((2 * c8 + h) ^ (r & 15)) << 4));
                        u[h] = *(const f32x4*)(at + (((2 * c8 + h + 8) ^ (r & 15)) << 4));
                    }
                    u32x4 o;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = gate(g[h][e]) * u[h][e];
                        o[2 * h] = act_pack<true>(v[0], v[1]); o[2 * h + 1] = act_pack<true>(v[2], v[3]);
                    }
                    if (r < rows && c < p.N) *(u32x4*)(y + (size_t)(k * 16) * p.ldy) = o;
                }
            };
            if (p.act == DN_ACT_SILU) out([](float g) { return dn_act(g, DN_ACT_SILU); }); else out([](float g) { return dn_act(g, DN_ACT_RELU); });
        } else if (lean_plain) {
            const int c4 = lane & 15, n = nc + c4 * 4;
            f32x4 bias = {0.f, 0.f, 0.f, 0.f};
            if (Bi && n < p.N) {
#pragma unroll
                for (int e = 0; e < 4; ++e) bias[e] = dn_ld(Bi + n + e);
            }
            float* y = (float*)p.y + (size_t)(r0 + (lane >> 4)) * p.ldy + (int)gr.yo + n;
#pragma unroll 4
            for (int k = 0; k < PH * 4; ++k) {
                const int r = k * 4 + (lane >> 4);
                f32x4 v = *(const f32x4*)(mine + r * 256 + ((c4 ^ (r & 15)) << 4));
                if (Bi) v += bias;
                if (r < rows && n < p.N) *(f32x4*)(y + (size_t)(k * 4) * p.ldy) = v;
            }
        } else if (lean_scaled) {
            const int c4 = lane & 15, n = nc + c4 * 4;
            const size_t row = r0 + (lane >> 4);
            const float* z = p.egate + row * p.ldg + p.goff + (int)gr.yo + n;
            bf16* y = (bf16*)p.y + row * p.ldy + (int)gr.yo + n;
            constexpr int U = 4;                                            // rows whose gates are asked for together
#pragma unroll 1
            for (int k0 = 0; k0 < PH * 4; k0 += U) {
                f32x4 zv[U];
#pragma unroll
                for (int k = 0; k < U; ++k)
                    if ((k0 + k) * 4 + (lane >> 4) < rows && n < p.N) zv[k] = *(const f32x4*)(z + (size_t)((k0 + k) * 4) * p.ldg);
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const int r = (k0 + k) * 4 + (lane >> 4);
                    f32x4 v = *(const f32x4*)(mine + r * 256 + ((c4 ^ (r & 15)) << 4));
                    if (r >= rows || n >= p.N) continue;
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] *= 1.f / (1.f + expf(-zv[k][e]));
                    *(u32x2*)(y + (size_t)((k0 + k) * 4) * p.ldy) = u32x2{act_pack<true>(v[0], v[1]), act_pack<true>(v[2], v[3])};
                }
            }
        } else if (p.gated) {
            const int c4 = lane & 7;                                        // channels 4 c4 .. of the wave's 32
            if (nc + c4 * 4 + 32 < p.N)
#pragma unroll 1
                for (int r = lane >> 3; r < rows; r += 8) {
                    f32x4 g = *(const f32x4*)(mine + r * 256 + ((c4 ^ (r & 15)) << 4)), u = *(const f32x4*)(mine + r * 256 + (((c4 + 8) ^ (r & 15)) << 4)), v;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (Bi) { g[e] += dn_ld(Bi + nc + c4 * 4 + e); u[e] += dn_ld(Bi + nc + 32 + c4 * 4 + e); }
                        v[e] = dn_gated(g[e], u[e], p.act, p.act_param);
                    }
                    dn_store4(p, r0 + r, (int)gr.yo + (nc >> 1) + c4 * 4, v, 4);
                }
        } else {
            const int c4 = lane & 15, n = nc + c4 * 4, cnt = min(4, p.N - n);
            f32x4 bias = {0.f, 0.f, 0.f, 0.f};
            if (Bi) {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (e < cnt) bias[e] = dn_ld(Bi + n + e);
            }
            if (cnt > 0)
#pragma unroll 1
                for (int r = lane >> 4; r < rows; r += 4) {
                    f32x4 v = *(const f32x4*)(mine + r * 256 + ((c4 ^ (r & 15)) << 4));
                    if (Bi) v += bias;
                    if (p.act != DN_ACT_NONE) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = dn_act(v[e], p.act);
                    }
                    dn_store4(p, r0 + r, (int)gr.yo + n, v, cnt);
                }
        }
        if (i0 + PH < MI) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read before the next rows overwrite them
    }
}

// ------------------------------------------------------------------------------------------------ fp32 tile kernel
constexpr int TF_M = 64, TF_N = 64, TF_K = 16, TF_LD = 68;

__device__ __forceinline__ f32x4 dn_chunk_f32(const float* base, int row, int rows, int k, int K, int ld, int vec) {
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    if (row >= rows || k >= K) return r;
    const float* p = base + (size_t)row * ld + k;
    if (vec) return *(const f32x4*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = (k + i < K) ? p[i] : 0.f;
    return r;
}

__global__ __launch_bounds__(256) void dense_tile_f32_kernel(DenseParams p) {
    __shared__ __attribute__((aligned(16))) float As[TF_K * TF_LD];   // [k][m]
    __shared__ __attribute__((aligned(16))) float Bs[TF_K * TF_LD];   // [k][n]
    const int tid = threadIdx.x, ty = tid >> 4, tx = tid & 15;
    const DnGroup gr = dn_group(p, TF_M);
    const int m0 = gr.m0, n0 = gr.bx * TF_N;
    if (m0 >= gr.rend) return;
    const float* X = (const float*)p.x + gr.xo;
    const float* W = (const float*)p.w + gr.wo;
    const float* Bi = p.bias ? (const float*)p.bias + gr.bo : nullptr;
    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;
    const int lr = tid >> 2, lk = (tid & 3) * 4;          // staging: row lr, k offset lk
    const int arow = m0 + lr < gr.rend ? (p.gather ? p.gather[m0 + lr] : m0 + lr) : 0x7fffffff;
    f32x4 ra = dn_chunk_f32(X, arow, 0x7fffffff, lk, p.K, p.ldx, p.vec);
    f32x4 rb = dn_chunk_f32(W, n0 + lr, p.N, lk, p.K, p.K, p.vec);
    for (int k0 = 0; k0 < p.K; k0 += TF_K) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) { As[(lk + i) * TF_LD + lr] = ra[i]; Bs[(lk + i) * TF_LD + lr] = rb[i]; }
        __syncthreads();
        if (k0 + TF_K < p.K) {
            ra = dn_chunk_f32(X, arow, 0x7fffffff, k0 + TF_K + lk, p.K, p.ldx, p.vec);
            rb = dn_chunk_f32(W, n0 + lr, p.N, k0 + TF_K + lk, p.K, p.K, p.vec);
        }
#pragma unroll
        for (int k = 0; k < TF_K; ++k) {
            const f32x4 a = *(const f32x4*)&As[k * TF_LD + ty * 4];
            const float b0 = Bs[k * TF_LD + 2 * tx], b1 = Bs[k * TF_LD + 2 * tx + 1];
            const float b2 = Bs[k * TF_LD + 32 + 2 * tx], b3 = Bs[k * TF_LD + 32 + 2 * tx + 1];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                acc[i][0] = __builtin_fmaf(a[i], b0, acc[i][0]); acc[i][1] = __builtin_fmaf(a[i], b1, acc[i][1]);
                acc[i][2] = __builtin_fmaf(a[i], b2, acc[i][2]); acc[i][3] = __builtin_fmaf(a[i], b3, acc[i][3]);
            }
        }
    }
    // thread columns: {2 tx, 2 tx + 1} of the first 32 and the same of the second 32 (gate / up of one channel under `gated`)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = m0 + ty * 4 + i;
        if (row >= gr.rend) continue;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + 2 * tx + j;
            if (p.gated) {
                if (n + 32 >= p.N) continue;
                float g = acc[i][j], u = acc[i][j + 2];
                if (Bi) { g += Bi[n]; u += Bi[n + 32]; }
                dn_store<float>(p, row, (int)gr.yo + (n >> 6) * 32 + (n & 31), dn_gated(g, u, p.act, p.act_param));
            } else {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int nn = n + 32 * h;
                    if (nn >= p.N) continue;
                    float v = acc[i][j + 2 * h];
                    if (Bi) v += Bi[nn];
                    dn_store<float>(p, row, (int)gr.yo + nn, dn_act(v, p.act));
                }
            }
        }
    }
}

// ------------------------------------------------------------------------------------------------ row kernel (small M)
template <typename T> struct DnVec;
template <> struct DnVec<bf16> {
    static constexpr int W = 8;
    static __device__ __forceinline__ void load(const bf16* p, int n, int vec, float (&o)[8]) {
        if (vec && n >= 8) { act_unpack8<true>(*(const u32x4*)p, o); return; }
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = i < n ? (float)p[i] : 0.f;
    }
};
template <> struct DnVec<float> {
    static constexpr int W = 8;
    static __device__ __forceinline__ void load(const float* p, int n, int vec, float (&o)[8]) {
        if (vec && n >= 8) {
            const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) { o[i] = a[i]; o[4 + i] = b[i]; }
            return;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) o[i] = i < n ? p[i] : 0.f;
    }
};

__device__ __forceinline__ float dn_wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// One wave per NC outputs: plain columns, or under GATED channels (a gate row and an up row each).  MR rows of x per pass: every 16-byte
// piece of x is loaded once per wave and meets NC (2 NC) weight pieces, so the wave streams its weight rows with few loads of x between.
template <typename T, int MR, int NC, bool GATED>
__global__ __launch_bounds__(256) void dense_rows_kernel(DenseParams p, int mbase) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int o0 = (blockIdx.x * 4 + wave) * NC, grp = blockIdx.y;     // grp: group of a column-sliced launch (0 otherwise)
    const int nout = GATED ? p.N / 2 : p.N;
    if (o0 >= nout) return;
    const T* X = (const T*)p.x + p.xs * grp;
    const T* W0[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int o = min(o0 + c, nout - 1);                       // a column past the end repeats the last one and is not stored
        W0[c] = (const T*)p.w + p.ws * grp + (size_t)(GATED ? (o >> 5) * 64 + (o & 31) : o) * p.K;
    }
    const T* Bi = p.bias ? (const T*)p.bias + (size_t)grp * p.N : nullptr;
    const int rows = min(MR, p.M - mbase);
    float a0[MR][NC], a1[GATED ? MR : 1][NC];
#pragma unroll
    for (int m = 0; m < MR; ++m)
#pragma unroll
        for (int c = 0; c < NC; ++c) { a0[m][c] = 0.f; if (GATED) a1[m][c] = 0.f; }
    for (int k = lane * 8; k < p.K; k += 64 * 8) {
        float w0[NC][8], w1[GATED ? NC : 1][8], xv[8];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            DnVec<T>::load(W0[c] + k, p.K - k, p.vec, w0[c]);
            if (GATED) DnVec<T>::load(W0[c] + (size_t)32 * p.K + k, p.K - k, p.vec, w1[c]);
        }
#pragma unroll
        for (int m = 0; m < MR; ++m) {
            if (m >= rows) break;
            DnVec<T>::load(X + (size_t)(mbase + m) * p.ldx + k, p.K - k, p.vec, xv);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
#pragma unroll
                for (int i = 0; i < 8; ++i) a0[m][c] = __builtin_fmaf(xv[i], w0[c][i], a0[m][c]);
                if (GATED) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) a1[m][c] = __builtin_fmaf(xv[i], w1[c][i], a1[m][c]);
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MR; ++m) {
        if (m >= rows) break;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float g = dn_wave_sum(a0[m][c]);
            float u = GATED ? dn_wave_sum(a1[m][c]) : 0.f;
            const int o = o0 + c;
            if (lane != 0 || o >= nout) continue;
            const int n0 = GATED ? (o >> 5) * 64 + (o & 31) : o;
            if (Bi) { g += dn_ld(Bi + n0); if (GATED) u += dn_ld(Bi + n0 + 32); }
            dn_store<T>(p, mbase + m, (int)(p.ys * grp) + o, GATED ? dn_gated(g, u, p.act, p.act_param) : dn_act(g, p.act));
        }
    }
}

// The same for a few rows that each belong to a group of their own (the experts of a decode step): blockIdx.y is the sorted row, its group is
// found in offs, a wave streams the weight row(s) of NC outputs of that group's weight once.
template <typename T, int NC, bool GATED>
__global__ __launch_bounds__(256) void dense_rows_grouped_kernel(DenseParams p) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int o0 = (blockIdx.x * 4 + wave) * NC, r = blockIdx.y;
    const int nout = GATED ? p.N / 2 : p.N;
    if (o0 >= nout || r >= p.offs[p.G]) return;
    int g = 0;
    while (g + 1 < p.G && p.offs[g + 1] <= r) ++g;
    const T* X = (const T*)p.x + (size_t)(p.gather ? p.gather[r] : r) * p.ldx + p.xs * g;
    const T* W0[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int o = min(o0 + c, nout - 1);
        W0[c] = (const T*)p.w + p.ws * g + (size_t)(GATED ? (o >> 5) * 64 + (o & 31) : o) * p.K;
    }
    float a0[NC], a1[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) a0[c] = a1[c] = 0.f;
    for (int k = lane * 8; k < p.K; k += 64 * 8) {
        float w0[NC][8], w1[GATED ? NC : 1][8], xv[8];
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            DnVec<T>::load(W0[c] + k, p.K - k, p.vec, w0[c]);
            if (GATED) DnVec<T>::load(W0[c] + (size_t)32 * p.K + k, p.K - k, p.vec, w1[c]);
        }
        DnVec<T>::load(X + k, p.K - k, p.vec, xv);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int i = 0; i < 8; ++i) a0[c] = __builtin_fmaf(xv[i], w0[c][i], a0[c]);
            if (GATED) {
#pragma unroll
                for (int i = 0; i < 8; ++i) a1[c] = __builtin_fmaf(xv[i], w1[c][i], a1[c]);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        float gsum = dn_wave_sum(a0[c]);
        const float u = GATED ? dn_wave_sum(a1[c]) : 0.f;
        const int o = o0 + c;
        if (lane != 0 || o >= nout) continue;
        dn_store<T>(p, r, (int)(p.ys * g) + o, GATED ? dn_gated(gsum, u, p.act, p.act_param) : dn_act(gsum, p.act));
    }
}

// The bf16 tile launch of p: gy64 row tiles of 64 rows (blockIdx.y) when the rows are grouped, groups in z.
void launch_tiles_bf16(const DenseParams& p, int gy64, int gz, hipStream_t st) {
    const bool dma = p.vec && (!p.gather || (uint64_t)p.M * p.ldx * 2 < 0xFFFFFFFFull) && (uint64_t)p.ldx * 512 < 0xFFFFFFFFull && (uint64_t)p.K * 512 < 0xFFFFFFFFull;
    if (!dma) {                                                             // unaligned operands, K % 8 != 0, 32-bit offsets that do not reach
        hipLaunchKernelGGL(dense_tile_bf16_kernel, dim3((p.N + TB_N - 1) / TB_N, gy64, gz), dim3(256), 0, st, p);
        return;
    }
    const int shape = mi355_dense_tile_shape(p.M, p.N, p.K, gz, p.offs ? gy64 : 0);
    const int gn = (p.N + 127) / 128;
    if (shape == 0)      hipLaunchKernelGGL((dense_dma_bf16_kernel<64, 64, 16, 64, 64, 4>), dim3((p.N + 63) / 64, gy64, gz), dim3(256), 0, st, p);
    else if (shape == 1) hipLaunchKernelGGL((dense_dma_bf16_kernel<64, 128, 32, 64, 64, 3>), dim3(gn, gy64, gz), dim3(256), 0, st, p);
    else if (shape == 2) hipLaunchKernelGGL((dense_dma_bf16_kernel<64, 128, 32, 64, 64, 2>), dim3(gn, gy64, gz), dim3(256), 0, st, p);
    else if (shape == 3) hipLaunchKernelGGL((dense_dma_bf16_kernel<128, 128, 32, 64, 64, 2>), dim3(gn, (p.M + 127) / 128, gz), dim3(512), 0, st, p);
    else                 hipLaunchKernelGGL((dense_dma_bf16_kernel<256, 256, 128, 64, 32, 4>), dim3((p.N + 255) / 256, (p.M + 255) / 256, gz), dim3(512), 0, st, p);
}

template <typename T, bool GATED>
void launch_rows(const DenseParams& p, hipStream_t st) {
    const int nout = GATED ? p.N / 2 : p.N;
    for (int mb = 0; mb < p.M; mb += 16) {
        const int r = p.M - mb;
        // few rows: one output per wave keeps the most waves streaming; more rows: several outputs per wave share the loads of x
        if (r <= 2)      hipLaunchKernelGGL((dense_rows_kernel<T, 2, 1, GATED>), dim3((nout + 3) / 4, p.G), dim3(256), 0, st, p, mb);
        else if (r <= 4) hipLaunchKernelGGL((dense_rows_kernel<T, 4, 2, GATED>), dim3((nout + 7) / 8, p.G), dim3(256), 0, st, p, mb);
        else if (r <= 8) hipLaunchKernelGGL((dense_rows_kernel<T, 8, GATED ? 2 : 4, GATED>), dim3((nout + (GATED ? 7 : 15)) / (GATED ? 8 : 16), p.G), dim3(256), 0, st, p, mb);
        else             hipLaunchKernelGGL((dense_rows_kernel<T, 16, GATED ? 2 : 4, GATED>), dim3((nout + (GATED ? 7 : 15)) / (GATED ? 8 : 16), p.G), dim3(256), 0, st, p, mb);
    }
}

// ------------------------------------------------------------------------------------------------ skinny kernel (bf16, M <= 16)
// One block of four waves per 8 weight rows: 8 outputs, or the gate and up rows of 4 channels.  What bounds it is how the weight comes out of memory: 8 rows of a row-major weight
// lie side by side, and read as MFMA fragments (16 rows by 64 bytes a wave load) they came at 3.2 TB/s however the steps were ordered.  Here every wave load is one
// row's run of 1 KB, by DMA into LDS, three stages of 512 columns; the rows of x beside them the same way, so that nothing but the fragments passes through registers.  8 weight rows a
// block and 48 KB (M <= 8): three blocks a compute unit, 96 KB of loads in flight.  More rows a block and more waves are slower; which stages
// pay is in skinny_stage, which shapes are better off without LDS in skinny_short.
// Weights from memory, M = 8, us before / now: 17408 x 2048 22.4 / 14.4, 32000 x 2048 35.1 / 24.3, 4096 x 2048 7.5 / 5.2, 2048 x 5632 13.6 / 6.5, 2048 x 2048 5.4 / 3.6.
// Sums: k in steps of 32, step s into chain s mod skinny_chains (4 or 8), the chains added in order: bits that depend on N, K and G only.
// 16-byte pieces are permuted by the row (applied to the source address), so that the 8 or 16 rows of a fragment read hit different banks.
constexpr int SK_RB = 8;
template <int XR_, int KC_, int NS_> struct SkinnyForm {                      // rows of x that are staged (M <= XR), columns of a stage, stages
    static constexpr int XR = XR_, KC = KC_, NS = NS_, STAGE = (SK_RB + XR) * KC * 2, BYTES = NS * STAGE;
};

// The weight rows bx * 8 .. of group grp.  NCH: chains.  NT: the weight is not kept in the caches.  Whole block of 256.
template <class F, int NCH, bool NT>
__device__ __forceinline__ void dense_skinny_tile(const DenseParams& p, int bx, int grp, char* smem) {
    constexpr int XR = F::XR, KC = F::KC, NS = F::NS, STAGE = F::STAGE, RB = KC * 2, NW = 4, PPR = KC / 8;   // PPR: 16-byte pieces of a row
    constexpr int LW = SK_RB * PPR / (64 * NW), LX = XR * PPR / (64 * NW), LD = LW + LX;                                   // loads per wave and stage
    static_assert((NCH == 4 || NCH == 8) && LX * 64 * NW == XR * PPR, "a wave adds one or two chains; whole wave loads");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem);
    const int no = p.gated ? SK_RB / 2 : SK_RB, nout = p.gated ? p.N / 2 : p.N, o0 = bx * no;   // the block's outputs
    const bf16* X = (const bf16*)p.x + p.xs * grp;
    // gated: rows 0 to 3 are the gates of channels o0 .., 4 to 7 their up rows, 32 further on; a row past the end repeats the last one and is not stored
    const int first = p.gated ? (o0 >> 5) * 64 + (o0 & 31) : o0;
    const bf16* W = (const bf16*)p.w + p.ws * grp + (size_t)first * p.K;
    uint32_t row[LD], pc[LD];                                              // byte offset of the lane's row, its piece of it
#pragma unroll
    for (int u = 0; u < LD; ++u) {
        const int at = ((u < LW ? u : u - LW) * NW + wave) * 64 + lane, r = at / PPR;
        if (u < LW) row[u] = (uint32_t)(p.gated ? (r & 3) + (r >> 2) * 32 : min(r, nout - 1 - o0)) * (uint32_t)p.K * 2u;
        else        row[u] = (uint32_t)min(r, p.M - 1) * (uint32_t)p.ldx * 2u;
        pc[u] = (at % PPR) ^ (r & 15);
    }
    auto issue = [&](int buf, int c) {
        const uint32_t last = (uint32_t)min(KC, p.K - c * KC) / 8 - 1;  // pieces past the end of K repeat the last one
#pragma unroll
        for (int u = 0; u < LD; ++u) {
            const uint32_t to = lds0 + buf * STAGE + (u < LW ? 0 : SK_RB * RB) + ((u < LW ? u : u - LW) * NW + wave) * 1024, from = row[u] + min(pc[u], last) * 16u;
            if (u < LW && NT) dma16_nt(to, from, W + c * KC);
            else              dma16(to, from, (u < LW ? W : X) + c * KC);
        }
    };
    const int nc = (p.K + KC - 1) / KC, fr = lane & 15, q = lane >> 4, wr = fr & (SK_RB - 1), xr = fr & (XR - 1);
    f32x4 acc[NCH / 4];
#pragma unroll
    for (int i = 0; i < NCH / 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NS - 1; ++c) if (c < nc) issue(c, c);
    int at = 0;
    for (int c = 0; c < nc; ++c) {
        if (c + NS - 2 < nc) wait_vm<LD * (NS - 2)>(); else wait_vm<0>();    // this wave's part of the columns is in LDS, its reads of the stage before are done
        __builtin_amdgcn_s_barrier();
        if (c + NS - 1 < nc) issue(at == 0 ? NS - 1 : at - 1, c + NS - 1);
        const char* wb = smem + at * STAGE + wr * RB;
        const char* xb = smem + at * STAGE + (SK_RB + xr) * RB;
        auto step = [&](int s, bool tail) {                                   // the wave's step s of the stage
            const int piece = (s * NW + wave) * 4 + q;
            bf16x8 b = *(const bf16x8*)(wb + ((piece ^ wr) << 4)), a = *(const bf16x8*)(xb + ((piece ^ xr) << 4));
            if (tail && c * KC + piece * 8 >= p.K) { a = bf16x8{}; b = bf16x8{}; }
            acc[NCH == 8 ? s & 1 : 0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc[NCH == 8 ? s & 1 : 0], 0, 0, 0);
        };
        if ((c + 1) * KC <= p.K) {
#pragma unroll
            for (int s = 0; s < KC / 32 / NW; ++s) step(s, false);
        } else {
#pragma unroll
            for (int s = 0; s < KC / 32 / NW; ++s) if (c * KC + (s * NW + wave) * 32 < p.K) step(s, true);
        }
        at = at + 1 == NS ? 0 : at + 1;
    }
    // the chains meet in a stage that no wave reads any more: not the last one's, and behind its barrier all others are done with
    f32x4* red = (f32x4*)(smem + (at + 1 == NS ? 0 : at + 1) * STAGE);
    static_assert(NCH * 64 * 16 <= STAGE && NS >= 3, "room for the chains beside the stage that is still read");
#pragma unroll
    for (int i = 0; i < NCH / 4; ++i) red[(i * 4 + wave) * 64 + lane] = acc[i];
    __syncthreads();
    // C fragment: lane holds weight row (lane & 15), rows 4 * (lane >> 4) + e of x; wave e takes the rows of its e
    if (fr >= no || o0 + fr >= nout) return;
    const int m = q * 4 + wave, oc = o0 + fr;
    if (m >= p.M) return;
    const float* mine = (const float*)(red + lane) + wave;
    float g = mine[0], v = p.gated ? mine[16] : 0.f;                          // the up row's lane is four on
#pragma unroll
    for (int i = 1; i < NCH; ++i) {
        g += mine[i * 256];
        if (p.gated) v += mine[i * 256 + 16];
    }
    if (p.bias) { const bf16* Bi = (const bf16*)p.bias + (size_t)grp * p.N + first + fr; g += dn_ld(Bi); if (p.gated) v += dn_ld(Bi + 32); }
    dn_store<bf16>(p, m, (int)(p.ys * grp) + oc, p.gated ? dn_gated(g, v, p.act, p.act_param) : dn_act(g, p.act));
}

template <class F, int NCH, bool NT>
__global__ __launch_bounds__(256) void dense_skinny_bf16_kernel(DenseParams p) {
    __shared__ __attribute__((aligned(1024))) char smem[F::BYTES];
    dense_skinny_tile<F, NCH, NT>(p, blockIdx.x, blockIdx.y, smem);
}

// Two of them in one launch, the second's blocks behind the first's: a launch of few rows costs 2 to 3 us whatever it reads, and the weights of the two keep each other's compute
// units busy.  Chains as in a launch of its own, so that the bits are the same.
template <class F, bool NT>
__global__ __launch_bounds__(256) void dense_skinny_pair_kernel(DenseParams p0, DenseParams p1, int blocks0, int chains0, int chains1) {
    __shared__ __attribute__((aligned(1024))) char smem[F::BYTES];
    const int b = blockIdx.x;
    if (b < blocks0) {
        if (chains0 == 8) dense_skinny_tile<F, 8, NT>(p0, b, 0, smem); else dense_skinny_tile<F, 4, NT>(p0, b, 0, smem);
    } else {
        if (chains1 == 8) dense_skinny_tile<F, 8, NT>(p1, b - blocks0, 0, smem); else dense_skinny_tile<F, 4, NT>(p1, b - blocks0, 0, smem);
    }
}

// A linear and the recurrence of the same decode step, which need nothing of each other: the recurrence is 128 blocks (16 heads of 8 sequences) in a chain of four trips to memory, 8.5 us, and
// the linear's blocks stream their weights meanwhile.  The recurrence's blocks come first, so that none of them waits for a unit.  A layer of width 2048 with 8 rows: both input linears 16.4 us and
// the recurrence 8.5 before, now the mixer's own 8.2 and this launch 13.5 (11264 x 2048); a prompt pass and 12 steps of 2 / 4 / 8 / 16 sequences, us before / now: width 1024, 8 layers 3483 / 3274,
// 3529 / 3335, 3691 / 3450, 4066 / 3727; width 2048, 16 layers 9389 / 8927, 9650 / 9175, 10456 / 9998, 12044 / 11845.
template <class F, int RPT, bool NT>
__global__ __launch_bounds__(256) void hy_recur_linear_kernel(RecurStep r, DenseParams p, int nseq, int chains) {
    __shared__ __attribute__((aligned(1024))) char smem[F::BYTES];
    static_assert(sizeof(RecurLds) <= F::BYTES, "the recurrence's arrays lie where the stages do");
    const int heads = nseq * r.H, b = blockIdx.x;
    if (b < heads) hy_recur_step<bf16, RPT>(r, b % nseq, b / nseq, *(RecurLds*)smem);
    else if (chains == 8) dense_skinny_tile<F, 8, NT>(p, b - heads, 0, smem);
    else                  dense_skinny_tile<F, 4, NT>(p, b - heads, 0, smem);
}

// Where that costs more than it gains (skinny_short): fragments straight from memory, the same sums.  16 outputs a block, a wave for each of the NW chains, U steps of it in flight.
// HALF (M <= 8): 8 outputs a block and half the waves, each with two chains: rows 0 to 7 of the first operand are x in the steps of chain w, rows 8 to 15 x in those of chain w + NW / 2, the second
// operand likewise; of the 16 x 16 sums the two 8 x 8 blocks on the diagonal are the two chains, the rest is not used.
template <int NW> struct SkinnySums { f32x4 at[NW][2][64]; };
template <bool GATED, int NW, int U, bool HALF>
__device__ __forceinline__ void dense_skinny_short_tile(const DenseParams& p, int bx, int grp, SkinnySums<NW>& red) {
    constexpr int NO = HALF ? 8 : 16, WAVES = HALF ? NW / 2 : NW;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nout = GATED ? p.N / 2 : p.N;
    const int r = lane & (NO - 1), kq = (lane >> 4) * 8 + (HALF && (lane & 8) ? WAVES * 32 : 0), o = min(bx * NO + r, nout - 1), n = GATED ? (o >> 5) * 64 + (o & 31) : o;
    const bf16* wg = (const bf16*)p.w + p.ws * grp + (size_t)n * p.K + kq;
    const bf16* wu = wg + (size_t)32 * p.K;
    const bf16* xr = (const bf16*)p.x + p.xs * grp + (size_t)min(r, p.M - 1) * p.ldx + kq;
    f32x4 ag = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
    const bf16x8 zero = {};
    for (int k0 = wave * 32; k0 < p.K; k0 += U * NW * 32) {
        bf16x8 a[U], b[U], c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * NW * 32;
            const bool ok = k + kq < p.K;
            a[u] = ok ? *(const bf16x8*)(xr + k) : zero;
            b[u] = ok ? *(const bf16x8*)(wg + k) : zero;
            if (GATED) c[u] = ok ? *(const bf16x8*)(wu + k) : zero;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            ag = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], b[u], ag, 0, 0, 0);
            if (GATED) au = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u], c[u], au, 0, 0, 0);
        }
    }
    red.at[wave][0][lane] = ag;
    if (GATED) red.at[wave][1][lane] = au;
    __syncthreads();
    if (wave != 0) return;
    for (int w = 1; w < WAVES; ++w) {
        ag += red.at[w][0][lane];
        if (GATED) au += red.at[w][1][lane];
    }
    if constexpr (HALF) {                                                     // the other chains' sum of (output, row) lies at (output + 8, row + 8), 40 lanes on
        if ((lane & 8) || lane >= 32) return;
        for (int w = 0; w < WAVES; ++w) {
            ag += red.at[w][0][lane + 40];
            if (GATED) au += red.at[w][1][lane + 40];
        }
    }
    if (bx * NO + r >= nout) return;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int row = (lane >> 4) * 4 + e;
        if (row >= p.M) continue;
        float g = ag[e], u = au[e];
        if (p.bias) { const bf16* Bi = (const bf16*)p.bias + (size_t)grp * p.N; g += dn_ld(Bi + n); if (GATED) u += dn_ld(Bi + n + 32); }
        dn_store<bf16>(p, row, (int)(p.ys * grp) + bx * NO + r, GATED ? dn_gated(g, u, p.act, p.act_param) : dn_act(g, p.act));
    }
}
template <bool GATED, int NW, int U, bool HALF>
__global__ __launch_bounds__(64 * (HALF ? NW / 2 : NW)) void dense_skinny_short_kernel(DenseParams p) {
    __shared__ SkinnySums<NW> red;
    dense_skinny_short_tile<GATED, NW, U, HALF>(p, blockIdx.x, blockIdx.y, red);
}
template <bool GATED0, bool GATED1, int NW, int U, bool HALF>
__global__ __launch_bounds__(64 * (HALF ? NW / 2 : NW)) void dense_skinny_short_pair_kernel(DenseParams p0, DenseParams p1, int blocks0) {
    __shared__ SkinnySums<NW> red;
    if ((int)blockIdx.x < blocks0) dense_skinny_short_tile<GATED0, NW, U, HALF>(p0, blockIdx.x, 0, red);
    else                           dense_skinny_short_tile<GATED1, NW, U, HALF>(p1, blockIdx.x - blocks0, 0, red);
}
// The columns of a stage of the DMA form for M rows of K columns (the shorter of two) in so many blocks.  512 of them, three stages, except:
//   256, four stages, and so more blocks a compute unit, for short K, of which a stage of 512 would be mostly empty; where many blocks would load a tenth more columns than there are with 512 (a stage's
//   loads past K cost what the others do); and for 9 to 16 rows in more than 256 blocks of K below 2048, or 1024 of any (32000 x 2048 26.2 us; 2048 x 5632, 256 blocks, 7.8 against 7.2; steps of 9 and
//   16 rows at width 2048 7535 and 8170 us with 256 from 257 blocks on, 7475 and 8080 with 512 there; of 12 rows at width 1024 6065 / 6120);
//   1024, three stages, half the barriers, for up to 8 rows where no compute unit has a second block to hide them and the last stage is not mostly empty.  Time over that of 512, K that fills both: up
//   to 192 blocks 0.93 to 0.95 (2 rows), 0.95 to 0.98 (3 and 4), 0.98 to 0.99 (5 to 8); 193 to 256 0.97 to 1.00; 257 to 320 1.04 to 1.23; 9 to 16 rows 1.00 to 1.03.
int skinny_stage(int M, int K, long long blocks) {
    auto padded = [&](int kc) { return ((long long)K + kc - 1) / kc * kc; };
    if (K < 1024 || (blocks > 256 && (padded(512) * 10 > padded(256) * 11 || (M > 8 && (K < 2048 || blocks >= 1024))))) return 256;
    return M <= 8 && blocks <= 256 && padded(1024) * 10 <= padded(512) * 12 ? 1024 : 512;
}
bool skinny_fills(int K, int stage) { return ((long long)K + stage - 1) / stage * stage * 20 < 21ll * K; }      // less than a twentieth loaded for nothing

// Which linears of M rows, K columns and so many weight rows are better off without LDS: they have no stages to fill, but their wave loads are 8 or 16 rows by 64 bytes, which the weights' stream of
// long K pays for, and of gated weights half as many blocks read twice as much each.  So up to 8 rows HALF serves K of 1024 and more that does not fill the DMA form's stages (fills), up to a length that
// falls with the rows, and at 2 rows, of which the stages hold copies, any K so short; gated weights only from 2048 rows on (128 blocks); 16 outputs a block serve many outputs of short K.
// Time without LDS / with, means over random calls, each behind a launch that writes its x, as a step has them: 5 to 8 rows, K 1024 to 1279 that fills / does not, 512 to 4096 weight rows 1.04 to 1.09 / 0.96 to
// 1.03, gated below 2048 1.08 to 1.15 / 1.03 to 1.06, gated 2048 to 4096 1.02 to 1.04 / 0.93 to 0.99; K 2048 to 2303 1.06 to 1.24; 2 rows, K 1024 to 2047 0.87 to 1.00, gated of K over 1536 below 2048 rows 1.04 to
// 1.17; K below 512, over 8192 rows 0.78 to 0.92.  (Timed back to back with x in the caches the form without LDS looked 5 to 15 % better: by lines from such times 1408 gated x 1024 took 5.6 us in a
// step of 8 rows and 4880 x 1024 6.7, through LDS 4.7 and 5.7.)
// K below 1024 through fewer outputs goes through LDS although HALF is 0.87 to 1.02 of it alone: in a step the stages' code is at hand from the launches around.  Eight layers of experts with such linears (704
// and 64 columns), eight prompts and seven steps 6400 / 6300 us, two prompts 5520 / 5460.
//   9 to 16 rows, us: 11 x 1024 x 47616 gated 29.1 / - / 24.5, 10 x 1024 x 22784 gated 16.4 / - / 13.1; 12 x 1808 x 8128, just two blocks of 16 a compute unit, 11.8 / - / 10.6; past the lines
//   11 x 1728 x 10368 gated 13.0 / - / 14.0, 16 x 1864 x 8256 gated 13.5 / - / 16.4, 12 x 1832 x 4224 8.3 / - / 9.5.
// 1986 times of 993 random calls of 2 to 8 rows that the lines were not fitted to, from memory and from the memory-side cache: 1.018 of the fastest form's, at worst 1.18; 0.958 of the time of the kernels
// before the DMA form, 297 more than 3 % behind it, most of them of K below 1024.
int skinny_short(int M, int K, long long weight_rows, bool gated, bool fills) {           // outputs a block; 0: through LDS
    if (M > 8) return weight_rows >= 6144 && (K <= 1152 || (K <= 1856 && (weight_rows <= 8192 || weight_rows >= 12288))) ? 16 : 0;
    if (weight_rows < (K < 512 ? 8192 : K < 1024 ? 4096 : gated ? 2048 : 0)) return 0;
    if (fills && M > 2 && weight_rows < (K < 1024 ? 8192 : 12288)) return 0;
    if (K <= 1152 && weight_rows >= (K < 512 ? 8192 : K < 1024 ? 6144 : 12288)) return 16;
    return K <= (M <= 2 ? 2304 : M <= 4 ? 2048 : 1792) && weight_rows < 12288 ? 8 : 0;
}
int skinny_short_blocks(const DenseParams& p, int outputs) { return ((p.gated ? p.N / 2 : p.N) + outputs - 1) / outputs; }
// launch(chains, steps in flight, half) with the instance for as many outputs a block
template <class L>
void skinny_short_form(int outputs, bool eight, L&& launch) {
    const std::integral_constant<int, 4> four{};
    const std::integral_constant<int, 8> eights{};
    if (outputs == 16) { if (eight) launch(eights, four, std::false_type{}); else launch(four, four, std::false_type{}); }
    else               { if (eight) launch(eights, eights, std::true_type{}); else launch(four, eights, std::true_type{}); }
}

// The partial sums that K is split into (part of a result's bits): eight, four of many outputs or short K.
int skinny_chains(const DenseParams& p) { return (((p.gated ? p.N / 2 : p.N) + 15) / 16) * p.G >= 1024 || p.K < 1024 ? 4 : 8; }
int skinny_blocks(const DenseParams& p) { return (p.N + SK_RB - 1) / SK_RB; }

// A weight that the 256 MB memory-side cache does not hold from one step to the next is read past the caches where a launch reads 24 MB or more.  Only the caller knows: the same weight in a
// small model, or under a draft's head, comes from that cache.  40 random weights of 24 to 130 MB, time with / without the hint: 0.97 (0.91 to 1.01) in a footprint of 1 GB, 0.96 in 400 MB,
// 1.12 (0.99 to 1.37) in 256 MB, 1.10 in 128 MB.  17408 x 2048 from memory 15.5 / 14.4 us, 32000 x 2048 26.5 / 24.3; eight prompts and eight steps of a 16-layer model of width 2048 8920 / 8400 us.
// What a marked weight displaces counts too: a head of 64 MB read past the caches leaves them to the layers (eight layers, 247 MB a step, eight prompts and seven steps 2690 -> 2622 us, the head itself
// 16.4 -> 17.7), so up to 8 rows such a launch goes through LDS, which has the hint.
bool skinny_nt(bool streamed, size_t weights) { return streamed && weights * 2 >= (size_t)24 << 20; }

// launch(form) with the form of skinny_stage columns.  As few rows of x staged as there are: they come from the L2, but pass through the same loads as the weights (32000 x 2048 with 4 / 8 / 16:
// 21.2 / 24.3 / 28.6 us).
template <class L>
void skinny_form(int M, int stage, L&& launch) {
    auto rows = [&](auto kc, auto ns) {
        constexpr int KC = decltype(kc)::value, NS = decltype(ns)::value;
        if (M > 8) launch(SkinnyForm<16, KC < 1024 ? KC : 512, NS>{});                       // no stage of 1024 there
        else if (M > 4 || KC < 512) launch(SkinnyForm<8, KC, NS>{});
        else if constexpr (KC >= 512) launch(SkinnyForm<4, KC, NS>{});
    };
    if (stage == 256)       rows(std::integral_constant<int, 256>{}, std::integral_constant<int, 4>{});
    else if (stage == 1024) rows(std::integral_constant<int, 1024>{}, std::integral_constant<int, 3>{});
    else                    rows(std::integral_constant<int, 512>{}, std::integral_constant<int, 3>{});
}
// The DMA form adds 32-bit byte offsets to the first row of x and of a block's weight rows.  Rows of x further apart than that reaches (15 steps of 143 million elements: the last tokens of eight
// sequences of 131072 x 2048) go in launches of fewer rows, the same bits; a K that the 35 rows between a gate and the last up row of a block do not reach has no such form.
constexpr long long SK_REACH = 0xFFFFFFFFll - 2 * 1024;                        // in front of a stage's columns
bool skinny_weight_reach(int K) { return 35ll * K * 2 <= SK_REACH; }
int skinny_rows_reach(int ldx) { return (int)(SK_REACH / (2ll * ldx)) + 1; }
// M of 2 to 16, p.vec, skinny_weight_reach
void launch_skinny(const DenseParams& p, hipStream_t st) {
    const int reach = skinny_rows_reach(p.ldx);
    if (p.M > reach) {
        for (int m = 0; m < p.M; m += reach) {
            DenseParams q = p;
            q.M = p.M - m < reach ? p.M - m : reach;
            q.x = (const bf16*)p.x + (size_t)m * p.ldx;
            q.y = (char*)p.y + (size_t)m * p.ldy * (p.out_f32 ? 4 : 2);
            if (p.egate) q.egate = p.egate + (size_t)m * p.ldg;
            launch_skinny(q, st);
        }
        return;
    }
    const bool eight = skinny_chains(p) == 8;
    const int stage = skinny_stage(p.M, p.K, (long long)skinny_blocks(p) * p.G);
    const bool nt = skinny_nt(p.streamed, (size_t)p.N * p.K * p.G);
    if (const int out = nt && p.M <= 8 ? 0 : skinny_short(p.M, p.K, (long long)p.N * p.G, p.gated, skinny_fills(p.K, stage))) {
        skinny_short_form(out, eight, [&](auto nw, auto u, auto half) {
            constexpr int NW = decltype(nw)::value, U = decltype(u)::value;
            constexpr bool H = decltype(half)::value;
            const dim3 grid(skinny_short_blocks(p, out), p.G), block(64 * (H ? NW / 2 : NW));
            if (p.gated) hipLaunchKernelGGL((dense_skinny_short_kernel<true, NW, U, H>), grid, block, 0, st, p); else hipLaunchKernelGGL((dense_skinny_short_kernel<false, NW, U, H>), grid, block, 0, st, p);
        });
        return;
    }
    const dim3 grid(skinny_blocks(p), p.G), block(256);
    skinny_form(p.M, stage, [&](auto f) {
        using F = decltype(f);
        if (eight) { if (nt) hipLaunchKernelGGL((dense_skinny_bf16_kernel<F, 8, true>), grid, block, 0, st, p); else hipLaunchKernelGGL((dense_skinny_bf16_kernel<F, 8, false>), grid, block, 0, st, p); }
        else       { if (nt) hipLaunchKernelGGL((dense_skinny_bf16_kernel<F, 4, true>), grid, block, 0, st, p); else hipLaunchKernelGGL((dense_skinny_bf16_kernel<F, 4, false>), grid, block, 0, st, p); }
    });
}
void launch_skinny_pair(const DenseParams (&p)[2], hipStream_t st) {
    const int chains = skinny_chains(p[0]), M = p[0].M > p[1].M ? p[0].M : p[1].M, b0 = skinny_blocks(p[0]), b1 = skinny_blocks(p[1]);
    const int stage = skinny_stage(M, p[0].K < p[1].K ? p[0].K : p[1].K, (long long)b0 + b1);
    const bool nt = skinny_nt(p[0].streamed && p[1].streamed, (size_t)p[0].N * p[0].K + (size_t)p[1].N * p[1].K);
    // two launches' weights keep the stages full: by the lines of 3 rows at least (2 rows, K 1024 through 832 to 960 blocks: 5.3 to 5.9 us through LDS, 6.8 to 7.1 without)
    const int out = (nt && M <= 8) || skinny_chains(p[1]) != chains ? 0 : skinny_short(M < 3 ? 3 : M, p[0].K > p[1].K ? p[0].K : p[1].K, (long long)p[0].N + p[1].N, p[0].gated || p[1].gated,
                                                                     skinny_fills(p[0].K, stage) && skinny_fills(p[1].K, stage));
    if (out) {
        const int s0 = skinny_short_blocks(p[0], out);
        const dim3 grid(s0 + skinny_short_blocks(p[1], out));
        skinny_short_form(out, chains == 8, [&](auto nw, auto u, auto half) {
            constexpr int NW = decltype(nw)::value, U = decltype(u)::value;
            constexpr bool H = decltype(half)::value;
            const dim3 block(64 * (H ? NW / 2 : NW));
            if (p[0].gated) { if (p[1].gated) hipLaunchKernelGGL((dense_skinny_short_pair_kernel<true, true, NW, U, H>), grid, block, 0, st, p[0], p[1], s0); else hipLaunchKernelGGL((dense_skinny_short_pair_kernel<true, false, NW, U, H>), grid, block, 0, st, p[0], p[1], s0); }
            else            { if (p[1].gated) hipLaunchKernelGGL((dense_skinny_short_pair_kernel<false, true, NW, U, H>), grid, block, 0, st, p[0], p[1], s0); else hipLaunchKernelGGL((dense_skinny_short_pair_kernel<false, false, NW, U, H>), grid, block, 0, st, p[0], p[1], s0); }
        });
        return;
    }
    const int c0 = skinny_chains(p[0]), c1 = skinny_chains(p[1]);
    skinny_form(M, stage, [&](auto f) {
        using F = decltype(f);
        if (nt) hipLaunchKernelGGL((dense_skinny_pair_kernel<F, true>), dim3(b0 + b1), dim3(256), 0, st, p[0], p[1], b0, c0, c1);
        else    hipLaunchKernelGGL((dense_skinny_pair_kernel<F, false>), dim3(b0 + b1), dim3(256), 0, st, p[0], p[1], b0, c0, c1);
    });
}

// The parameters of a linear of 2 to 16 bf16 rows from a caller's arguments; MI355_ERR_UNSUPPORTED where the kernels that share a launch do not take it.
int few_rows_params(mi355_dense_args_t d, const char* who, DenseParams& q) {
    const int streamed = (d.gated & MI355_DENSE_STREAMED) != 0; d.gated &= ~MI355_DENSE_STREAMED;
    MI355_CHECK_ARG(d.x && d.w && d.y && d.M > 0 && d.N > 0 && d.K > 0 && d.ldx >= d.K && (!d.gated || d.N % 64 == 0) && d.ldy >= (d.gated ? d.N / 2 : d.N) && d.act >= 0 &&
                        d.act <= DN_ACT_RELU2 && (d.act != DN_ACT_SWIGLU_CLAMP || (d.gated && d.act_param > 0.f)),
                    "%s: M=%d N=%d K=%d ldx=%d ldy=%d gated=%d act=%d", who, d.M, d.N, d.K, d.ldx, d.ldy, d.gated, d.act);
    if (d.M < 2 || d.M > 16 || d.K % 8 || d.ldx % 8 || (uintptr_t)d.x % 16 || (uintptr_t)d.w % 16 || !skinny_weight_reach(d.K) || d.M > skinny_rows_reach(d.ldx)) return MI355_ERR_UNSUPPORTED;
    q.x = d.x; q.w = d.w; q.bias = d.bias; q.y = d.y; q.M = d.M; q.N = d.N; q.K = d.K; q.ldx = d.ldx; q.ldy = d.ldy;
    q.gated = d.gated; q.streamed = streamed; q.act = d.act; q.act_param = d.act_param; q.out_f32 = d.out_f32; q.softcap = 0.f; q.vec = 1;
    q.yvec = (d.ldy % 4 == 0) && ((uintptr_t)d.y % (d.out_f32 ? 16 : 8) == 0);
    q.G = 1; q.xs = q.ws = q.ys = 0; q.offs = nullptr; q.gather = nullptr; q.tiles = nullptr; q.egate = nullptr; q.ldg = q.goff = 0;
    return MI355_OK;
}

// Where a recurrence takes a linear along: up to 8 key rows a thread (registers: three blocks a compute unit are left), and a linear that goes through LDS, by the lines of 3 rows at least as in a pair.
bool recur_linear_fits(int dim, int vdim, int M, int N, int K, bool gated, bool streamed) {
    const int blocks = (N + SK_RB - 1) / SK_RB;
    return hy_recur_rows(dim, vdim) <= 8 && ((skinny_nt(streamed, (size_t)N * K) && M <= 8) || !skinny_short(M < 3 ? 3 : M, K, N, gated, skinny_fills(K, skinny_stage(M, K, blocks))));
}
void launch_recur_linear(const RecurStep& r, int nseq, const DenseParams& p, hipStream_t st) {
    const dim3 grid(nseq * r.H + skinny_blocks(p));
    const int chains = skinny_chains(p);
    const bool nt = skinny_nt(p.streamed, (size_t)p.N * p.K);
    skinny_form(p.M, skinny_stage(p.M, p.K, skinny_blocks(p)), [&](auto f) {
        using F = decltype(f);
        if (nt) hipLaunchKernelGGL((hy_recur_linear_kernel<F, 8, true>), grid, dim3(256), 0, st, r, p, nseq, chains);
        else    hipLaunchKernelGGL((hy_recur_linear_kernel<F, 8, false>), grid, dim3(256), 0, st, r, p, nseq, chains);
    });
}

} // namespace

// x [M, K] (row stride ldx) and w [N, K] of act_dtype (MI355_ACT_BF16 or MI355_ACT_F32); bias [N] of act_dtype or null;
// y [M, N or N / 2] fp32 (out_f32) or act_dtype, row stride ldy.  gated: the N weight rows are groups of 64 = 32 gate rows followed by
// the 32 up rows of the same channels (N % 64 == 0); y[m, c] = act(gate_c) * up_c.  act: 0 none, 1 relu, 2 silu, 3 gelu (tanh form), 4 tanh (on the gate,
// or on the plain output), 6 the square of relu.  softcap > 0: y <- softcap * tanh(y / softcap).
extern "C" int mi355_dense_linear(const void* x, int32_t ldx, int32_t M, const void* w, int32_t N, int32_t K, const void* bias,
                                  void* y, int32_t ldy, int32_t out_f32, int32_t gated, int32_t act, float softcap,
                                  int32_t act_dtype, mi355_stream_t stream) {
    return mi355_dense_linear_ex(x, ldx, M, w, N, K, bias, y, ldy, out_f32, gated, act, 0.f, softcap, act_dtype, stream);
}

// The same with a parameter for the activation.  act 5 (gated only): with L = act_param > 0, g' = min(gate, L), u' = clamp(up, -L, L) and
// y = g' sigmoid(1.702 g') (u' + 1).
extern "C" int mi355_dense_linear_ex(const void* x, int32_t ldx, int32_t M, const void* w, int32_t N, int32_t K, const void* bias,
                                     void* y, int32_t ldy, int32_t out_f32, int32_t gated, int32_t act, float act_param, float softcap,
                                     int32_t act_dtype, mi355_stream_t stream) {
    const int streamed = (gated & MI355_DENSE_STREAMED) != 0; gated &= ~MI355_DENSE_STREAMED;
    MI355_CHECK_ARG(x && w && y && M > 0 && N > 0 && K > 0 && ldx >= K, "dense_linear: M=%d N=%d K=%d ldx=%d", M, N, K, ldx);
    MI355_CHECK_ARG(act_dtype == MI355_ACT_BF16 || act_dtype == MI355_ACT_F32, "dense_linear: act_dtype=%d (bf16 or fp32)", act_dtype);
    MI355_CHECK_ARG(!gated || N % 64 == 0, "dense_linear: gated needs N %% 64 == 0 (N=%d)", N);
    MI355_CHECK_ARG(act >= 0 && act <= DN_ACT_RELU2 && (act != DN_ACT_SWIGLU_CLAMP || (gated && act_param > 0.f)), "dense_linear: act=%d (gated=%d, parameter %g)", act, gated, (double)act_param);
    MI355_CHECK_ARG(ldy >= (gated ? N / 2 : N), "dense_linear: ldy=%d", ldy);
    const bool bf = act_dtype == MI355_ACT_BF16;
    const size_t es = bf ? 2 : 4;
    DenseParams p;
    p.x = x; p.w = w; p.bias = bias; p.y = y; p.M = M; p.N = N; p.K = K; p.ldx = ldx; p.ldy = ldy;
    p.gated = gated; p.streamed = streamed; p.act = act; p.act_param = act_param; p.out_f32 = bf ? out_f32 : 1; p.softcap = softcap;
    p.vec = (K % 8 == 0) && (ldx % 8 == 0) && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0);
    p.yvec = (ldy % 4 == 0) && ((uintptr_t)y % (p.out_f32 ? 16 : 8) == 0);
    p.G = 1; p.xs = p.ws = p.ys = 0; p.offs = nullptr; p.gather = nullptr; p.tiles = nullptr; p.egate = nullptr; p.ldg = p.goff = 0;
    (void)es;
    hipStream_t st = (hipStream_t)stream;
    if (bf && M > 1 && M <= 16 && p.vec && skinny_weight_reach(K)) {
        launch_skinny(p, st);
        MI355_CHECK_LAUNCH("dense_skinny_bf16_kernel");
        return MI355_OK;
    }
    if (M <= 16) {
        if (bf) { if (gated) launch_rows<bf16, true>(p, st); else launch_rows<bf16, false>(p, st); }
        else    { if (gated) launch_rows<float, true>(p, st); else launch_rows<float, false>(p, st); }
        MI355_CHECK_LAUNCH("dense_rows_kernel");
        return MI355_OK;
    }
    if (bf) {
        launch_tiles_bf16(p, (M + TB_M - 1) / TB_M, 1, st);
        MI355_CHECK_LAUNCH("dense bf16 tile kernel");
    } else {
        const dim3 grid((N + TF_N - 1) / TF_N, (M + TF_M - 1) / TF_M);
        hipLaunchKernelGGL(dense_tile_f32_kernel, grid, dim3(256), 0, st, p);
        MI355_CHECK_LAUNCH("dense_tile_f32_kernel");
    }
    return MI355_OK;
}

// Two linears of bf16 rows in one launch, arguments as in mi355_dense_linear_ex each (M of 2 to 16 rows, whole 16-byte pieces, rows within reach of 32-bit offsets): the results are those of two calls, bit for bit.
// MI355_ERR_UNSUPPORTED: other forms, which take two calls.
extern "C" int mi355_dense_linear_pair(const mi355_dense_args_t* a, mi355_stream_t stream) {
    MI355_CHECK_ARG(a, "dense_linear_pair: null arguments");
    DenseParams p[2];
    for (int i = 0; i < 2; ++i)
        if (int e = few_rows_params(a[i], "dense_linear_pair", p[i])) return e;
    hipStream_t st = (hipStream_t)stream;
    launch_skinny_pair(p, st);
    MI355_CHECK_LAUNCH("dense_skinny_pair_kernel");
    return MI355_OK;
}

// Whether mi355_hy_recur_step_beside takes aligned operands of these sizes.  Host only.
extern "C" int mi355_hy_recur_step_beside_fits(int32_t dim, int32_t vdim, int32_t M, int32_t N, int32_t K, int32_t gated) {
    return mi355_hy_recur_step_fits(dim, vdim) && M >= 2 && M <= 16 && N > 0 && K > 0 && K % 8 == 0 && skinny_weight_reach(K) &&
           recur_linear_fits(dim, vdim, M, N, K, gated & ~MI355_DENSE_STREAMED, (gated & MI355_DENSE_STREAMED) != 0);
}

// mi355_hy_recur_step (bf16) and a linear that neither reads nor writes anything of it, in one launch: the same bits as the two calls.
extern "C" int mi355_hy_recur_step_beside(const mi355_recur_args_t* a, const mi355_dense_args_t* lin, mi355_stream_t stream) {
    MI355_CHECK_ARG(a && lin, "hy_recur_step_beside: null arguments");
    const RecurStep r{a->proj, a->ld, a->qo, a->ko, a->vo, a->go, a->ao, a->rank, a->w2, a->b2, a->z, a->ldz, a->lower, a->fbias, a->tau, a->qscale, a->mode, a->H, a->dim, a->vdim, a->row_start,
                      a->slot, a->first_pos, a->state, a->w, a->w_heads, a->eps, a->out};
    if (int e = hy_recur_check(r, a->nseq)) return e;
    DenseParams p;
    if (int e = few_rows_params(*lin, "hy_recur_step_beside", p)) return e;
    if (!recur_linear_fits(r.dim, r.vdim, p.M, p.N, p.K, p.gated, p.streamed)) return MI355_ERR_UNSUPPORTED;
    launch_recur_linear(r, a->nseq, p, (hipStream_t)stream);
    MI355_CHECK_LAUNCH("hy_recur_linear_kernel");
    return MI355_OK;
}

// The same product for G groups in one launch: group g uses the weight w + g * N * K ([G, N, K] contiguous) and
// bias + g * N, reads x from column xs * g on and writes y from column ys * g on.  offs null: every group takes all M rows (per-head
// projections: xs, ys = the head's column step).  offs [G + 1] (device): M rows are sorted by group, group g owns rows offs[g] .. offs[g + 1] - 1;
// sorted row r reads x row gather[r] (device, or null for r itself) and writes y row r (experts of a mixture: xs = ys = 0).  A row's result
// depends on its own input and its group's weight only.  tiles (device, with offs; null: every group is given ceil(M / 64) row tiles, most of
// them empty): {n, (group, first row) x n}, the 64-row tiles that hold rows, at most max_tiles of them (mi355_hy_moe_align writes the list).
// egate (fp32 [M, ldg], or null): y[m, c] is multiplied by sigmoid(egate[m, goff + c]), c counted over the whole output row.
extern "C" int mi355_dense_grouped(const void* x, int32_t ldx, int32_t M, const void* w, int32_t N, int32_t K, const void* bias, void* y,
                                   int32_t ldy, int32_t out_f32, int32_t gated, int32_t act, int32_t act_dtype, int32_t G, int64_t xs,
                                   int64_t ys, const int32_t* offs, const int32_t* gather, const int32_t* tiles, int32_t max_tiles,
                                   const float* egate, int32_t ldg, int32_t goff, mi355_stream_t stream) {
    return mi355_dense_grouped_ex(x, ldx, M, w, N, K, bias, y, ldy, out_f32, gated, act, 0.f, act_dtype, G, xs, ys, offs, gather, tiles, max_tiles, egate, ldg,
                                  goff, stream);
}

// The same with the activation's parameter (act 5 as in mi355_dense_linear_ex).
extern "C" int mi355_dense_grouped_ex(const void* x, int32_t ldx, int32_t M, const void* w, int32_t N, int32_t K, const void* bias, void* y,
                                      int32_t ldy, int32_t out_f32, int32_t gated, int32_t act, float act_param, int32_t act_dtype, int32_t G,
                                      int64_t xs, int64_t ys, const int32_t* offs, const int32_t* gather, const int32_t* tiles, int32_t max_tiles,
                                      const float* egate, int32_t ldg, int32_t goff, mi355_stream_t stream) {
    return mi355_dense_grouped_ahead(x, ldx, M, w, N, K, bias, y, ldy, out_f32, gated, act, act_param, act_dtype, G, xs, ys, offs, gather, tiles, max_tiles, egate, ldg, goff,
                                     nullptr, 0, stream);
}

// The same, and a weight that a later launch streams (ahead_bytes of ahead; at most 48 MB of it, and 2 KB a thread): read by blocks past the list of tiles.
extern "C" int mi355_dense_grouped_ahead(const void* x, int32_t ldx, int32_t M, const void* w, int32_t N, int32_t K, const void* bias, void* y,
                                         int32_t ldy, int32_t out_f32, int32_t gated, int32_t act, float act_param, int32_t act_dtype, int32_t G,
                                         int64_t xs, int64_t ys, const int32_t* offs, const int32_t* gather, const int32_t* tiles, int32_t max_tiles,
                                         const float* egate, int32_t ldg, int32_t goff, const void* ahead, int64_t ahead_bytes, mi355_stream_t stream) {
    const int streamed = (gated & MI355_DENSE_STREAMED) != 0; gated &= ~MI355_DENSE_STREAMED;
    MI355_CHECK_ARG(x && w && y && M > 0 && N > 0 && K > 0 && G > 0 && xs >= 0 && ys >= 0, "dense_grouped: M=%d N=%d K=%d G=%d", M, N, K, G);
    MI355_CHECK_ARG(ldx >= xs * (G - 1) + K, "dense_grouped: ldx=%d for %d groups of K=%d at step %lld", ldx, G, K, (long long)xs);
    MI355_CHECK_ARG(act_dtype == MI355_ACT_BF16 || act_dtype == MI355_ACT_F32, "dense_grouped: act_dtype=%d (bf16 or fp32)", act_dtype);
    MI355_CHECK_ARG(!gated || N % 64 == 0, "dense_grouped: gated needs N %% 64 == 0 (N=%d)", N);
    MI355_CHECK_ARG(act >= 0 && act <= DN_ACT_RELU2 && (act != DN_ACT_SWIGLU_CLAMP || (gated && act_param > 0.f)), "dense_grouped: act=%d (gated=%d, parameter %g)", act, gated, (double)act_param);
    MI355_CHECK_ARG(ldy >= ys * (G - 1) + (gated ? N / 2 : N), "dense_grouped: ldy=%d", ldy);
    MI355_CHECK_ARG(G <= 65535 && (!gather || offs) && (!tiles || (offs && max_tiles > 0)), "dense_grouped: G=%d, gather and tiles need offs", G);
    const bool bf = act_dtype == MI355_ACT_BF16;
    DenseParams p;
    p.x = x; p.w = w; p.bias = bias; p.y = y; p.M = M; p.N = N; p.K = K; p.ldx = ldx; p.ldy = ldy;
    p.gated = gated; p.streamed = streamed; p.act = act; p.act_param = act_param; p.out_f32 = bf ? out_f32 : 1; p.softcap = 0.f;
    p.vec = (K % 8 == 0) && (ldx % 8 == 0) && (xs % 8 == 0) && ((uintptr_t)x % 16 == 0) && ((uintptr_t)w % 16 == 0);
    p.yvec = (ldy % 4 == 0) && ((uintptr_t)y % (p.out_f32 ? 16 : 8) == 0);
    p.G = G; p.xs = xs; p.ws = (long long)N * K; p.ys = ys; p.offs = offs; p.gather = gather; p.tiles = tiles;
    p.egate = egate; p.ldg = ldg; p.goff = goff;
    if (ahead && tiles && ahead_bytes > 0) { p.ahead = (const char*)ahead; p.ahead_lines = (uint32_t)((ahead_bytes < (int64_t)48 << 20 ? ahead_bytes : (int64_t)48 << 20) / 128); }
    MI355_CHECK_ARG(!egate || (goff >= 0 && ldg >= goff + (offs ? 0 : ys * (G - 1)) + (gated ? N / 2 : N)), "dense_grouped: gate row stride %d", ldg);
    static_assert(TB_M == 64 && TF_M == 64, "the tile list is made of 64-row tiles");
    hipStream_t st = (hipStream_t)stream;
    const int gy = tiles ? max_tiles : (M + 63) / 64, gz = tiles ? 1 : G;
    if (offs && M <= 16 && !bias) {            // a decode step's few rows: each streams its own group's weight
        const int nout = gated ? N / 2 : N, nc = gated ? 1 : 2;
        const dim3 grid((nout + 4 * nc - 1) / (4 * nc), M);
        if (bf) { if (gated) hipLaunchKernelGGL((dense_rows_grouped_kernel<bf16, 1, true>), grid, dim3(256), 0, st, p);
                  else       hipLaunchKernelGGL((dense_rows_grouped_kernel<bf16, 2, false>), grid, dim3(256), 0, st, p); }
        else    { if (gated) hipLaunchKernelGGL((dense_rows_grouped_kernel<float, 1, true>), grid, dim3(256), 0, st, p);
                  else       hipLaunchKernelGGL((dense_rows_grouped_kernel<float, 2, false>), grid, dim3(256), 0, st, p); }
        MI355_CHECK_LAUNCH("dense_rows_grouped_kernel");
        return MI355_OK;
    }
    if (!offs && M <= 16) {                    // a decode step's rows through every group: the kernels of the plain linear, groups in the grid
        if (bf && M > 1 && p.vec && skinny_weight_reach(K)) {
            launch_skinny(p, st);
            MI355_CHECK_LAUNCH("dense_skinny_bf16_kernel");
            return MI355_OK;
        }
        if (bf) { if (gated) launch_rows<bf16, true>(p, st); else launch_rows<bf16, false>(p, st); }
        else    { if (gated) launch_rows<float, true>(p, st); else launch_rows<float, false>(p, st); }
        MI355_CHECK_LAUNCH("dense_rows_kernel");
        return MI355_OK;
    }
    if (bf) {
        launch_tiles_bf16(p, gy, gz, st);
        MI355_CHECK_LAUNCH("dense bf16 tile kernel");
    } else {
        const dim3 grid((N + TF_N - 1) / TF_N, gy, gz);
        hipLaunchKernelGGL(dense_tile_f32_kernel, grid, dim3(256), 0, st, p);
        MI355_CHECK_LAUNCH("dense_tile_f32_kernel");
    }
    return MI355_OK;
}
