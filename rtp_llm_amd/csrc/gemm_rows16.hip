// Linears of up to 8 rows through 16-bit weights, hidden size at most 1024, with the whole layer's elementwise work fused in, gfx950: a step of a small model is a chain of short launches.
//
// A 0.5B model in fp16 reads 30 MB a layer, 6 us of memory, in launches of 2.5 to 7.5 us; two of eight were RMSNorms, one RoPE and the cache write, and three handed fp32 slabs of split K
// to them.  Taken where gate_up is one slice of at most eight chunks of 128, so hidden sizes up to 1024, and the other linears' slices are at most three chunks.  Here a block owns one to three 16-column tiles and all of K, its waves are the tiles' K slices (slice s of a tile is what split s of the staged kernel of gemm.hip was: the same
// chunks in the same order, each slice's sum by one wave, the slices added in order), and
//   NORM   the input rows are normalised on load: every block rebuilds the rows' sums of squares, lane by lane as add_rmsnorm_kernel adds them, while its weights are on their way;
//   ROPE   bias + rotation + Q + 16-bit cache write in the epilogue, the tile pair (d, d + hd / 2) of one head a block;     SLAB  fp32 sums, for the cache writer that quantises;
//   RESID  h' = h + y;     SILU  silu(gate) * up of interleaved columns.
// Five launches a layer in place of eight (six with an 8-bit cache), every bit as before.  A step of the 0.5B model, one row: 762 -> 618 us.
#include "gemm_fullk.h"

namespace {

enum { R16_ROPE = 0, R16_SLAB = 1, R16_RESID = 2, R16_SILU = 3 };

struct Rows16Params {
    const f16*  x;          // [M][K]; under NORM the rows before the norm
    const void* qw;
    int         M, K, N, N_pad, NT, KC;
    int         slices, cps, tw;      // K slices of cps chunks; tiles a block
    int         units;                // blocks of whole tiles (PARTS = 2: twice as many blocks)
    uint32_t    x_bytes;
    const f16*  gamma;
    float       eps;
    const f16*  res_in;     // RESID
    f16*        res_out;
    f16*        y;          // SILU [M][N / 2]
    float*      slab;       // SLAB [M][N_pad]
    const f16*  bias;       // ROPE
    RopeEpi     r;
};

// Every block normalises all rows, which costs more than the launches it saves from some 12 rows on: a step of the 0.5B model, the staged launches / these, us: 1 row 762 / 618, 4 (8-bit cache)
// 867 / 778, 8 889 / 806; 12 825 / 817, 16 903 / 940, 16 (8-bit cache) 916 / 1009.
constexpr int kRows16 = 8;
constexpr int kHidden = 1024;                        // columns of the residual rows
constexpr int kNormJobs = 2;                         // (row, 64 lanes of 8 columns) pairs a wave adds up at most

// D: chunks a slice has at most (SILU: 3 or 8; 3 in the others); all of them are asked for at once.  What a block waits for is the number of its vector-memory instructions as much as their bytes (a wave load of 16 bytes a
// lane is 16 cycles of a compute unit's address path whatever its lanes ask for), so none is half empty:
// PARTS 2 (RESID; ROPE and SLAB of up to 128 blocks): a block owns eight of its tiles' sixteen columns (block b: half b & 1); a wave load is two k-steps of them, lanes jj < 8 the even one, and the odd one is turned by eight lanes
//   into the product's first rows.  Twice the blocks where whole tiles leave more than half of the chip without one (down_proj of the 0.5B model, 56 tiles: 6.4 us whole).
// XL (RESID): activation loads a chunk.  1 (M <= 4): lane jj row jj % 4 of k-step jj / 4; 2 (M <= 8): row jj % 8, k-steps 2 l + jj / 8.
template <bool BF, int EPI, int D, int PARTS, int XL = 1>
__global__ __launch_bounds__(D <= 3 ? 1024 : 512) void gemm_rows16_kernel(const Rows16Params p) {
    constexpr bool NORM = EPI != R16_RESID;
    constexpr uint32_t FLAGS = 0x00020000u, OOBX = 0x80000000u;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
    const int jj = lane & 15, q = lane >> 4;
    const int pieces = p.K >> 3, njob = (pieces + 63) >> 6;          // 16-byte pieces of a row; jobs a row
    u32x4* xs  = reinterpret_cast<u32x4*>(smem);                     // NORM: [M][pieces], pieces permuted by the row
    float* ssq = reinterpret_cast<float*>(smem + (NORM ? (size_t)p.M * p.K * 2 : 0));   // [M][8]
    f32x4* red = reinterpret_cast<f32x4*>(smem + (NORM ? (size_t)p.M * p.K * 2 + 512 : 0));   // [K waves][64]

    const int kwaves = p.slices * p.tw, t = wave / p.slices, sl = wave - t * p.slices;
    const int unit = PARTS == 2 ? blockIdx.x >> 1 : blockIdx.x;
    constexpr int cols = 16 / PARTS;
    const int col0 = PARTS == 2 ? (blockIdx.x & 1) * 8 : 0;
    int tile0, tstep = 1;
    if constexpr (EPI == R16_ROPE) { const int hh = p.r.hd >> 5; tile0 = (unit / hh) * 2 * hh + unit % hh; tstep = hh; }
    else tile0 = unit * p.tw;

    // ---- the norm's share of this wave
    u32x4 hv[kNormJobs], gv[kNormJobs];
    const int job0 = wave == waves - 1 ? waves - 1 : waves - 2 - wave;   // the last wave last: ROPE's chain of position, block and rotation row is its own
    if constexpr (NORM) {
#pragma unroll
        for (int u = 0; u < kNormJobs; ++u) {
            const int j = job0 + u * waves, row = j / njob, vi = (j - row * njob) * 64 + lane;
            const bool ok = row < p.M && vi < pieces;
            hv[u] = gv[u] = u32x4{0u, 0u, 0u, 0u};
            if (ok) {
                hv[u] = *reinterpret_cast<const u32x4*>(p.x + (size_t)row * p.K + vi * 8);
                gv[u] = *reinterpret_cast<const u32x4*>(p.gamma + vi * 8);
            }
        }
    }
    // ---- operands of the epilogue: wave e finishes tile e (ROPE: the last wave finishes the pair)
    const bool epi = EPI == R16_ROPE ? wave == waves - 1 : wave < p.tw;
    u32x2 pre0 = {0u, 0u}, pre1 = {0u, 0u};
    int   pre_pos = 0, pre_blk = 0;
    f32x4 cs01 = {0.f, 0.f, 0.f, 0.f}, cs23 = cs01;
    const int etile = tile0 + (EPI == R16_ROPE ? 0 : wave), n0 = etile * 16 + col0 + q * 4;
    const bool mine = epi && jj < p.M && q * 4 < cols;                // a part's columns are the first rows of the product, and again the others
    if (mine) {
        if constexpr (EPI == R16_RESID) { if (n0 < p.N) pre0 = *reinterpret_cast<const u32x2*>(p.res_in + (size_t)jj * p.N + n0); }
        if constexpr (EPI == R16_ROPE) {
            const RopeEpi& R = p.r;
            const int half = R.hd >> 1, d0 = n0 % R.hd;
            if (p.bias) { pre0 = *reinterpret_cast<const u32x2*>(p.bias + n0); pre1 = *reinterpret_cast<const u32x2*>(p.bias + n0 + half); }
            pre_pos = R.positions[jj];
            const int pos = min(max(pre_pos, 0), min(R.max_pos, R.max_blocks * R.page) - 1);
            pre_blk = R.block_table[(size_t)(jj / R.q_len) * R.max_blocks + pos / R.page];
            const float* cs = R.cos_sin + ((size_t)pos * half + d0) * 2;
            cs01 = *reinterpret_cast<const f32x4*>(cs); cs23 = *reinterpret_cast<const f32x4*>(cs + 4);
        }
    }
    // ---- the slice's weights, all of them (without the norm its activations in front)
    const int tile = tile0 + t * tstep, c0 = sl * p.cps;
    const int n_ch = wave < kwaves && tile < p.NT ? max(0, min(p.cps, p.KC - c0)) : 0;
    constexpr int RPL = 4 * XL, SPL = 4 / XL, LW = 4 / PARTS;         // rows and k-steps of an activation load; weight loads a chunk
    u32x4 xr[NORM ? 1 : D][NORM ? 1 : XL], wr[D][LW];
    if constexpr (!NORM) {
        __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, p.x_bytes, FLAGS);
        const int row = jj % RPL;
        const uint32_t xv = row < p.M ? (uint32_t)((row * p.K + c0 * 128 + (jj / RPL) * 32 + q * 8) * 2) : OOBX;
#pragma unroll
        for (int c = 0; c < D; ++c)
#pragma unroll
            for (int l = 0; l < XL; ++l) xr[c][l] = bload128<0>(rx, c < n_ch ? xv : OOBX, (uint32_t)c * 256u + l * SPL * 64u);
    }
    __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)((const char*)p.qw + ((size_t)tile * p.KC + c0) * 4096), 0, n_ch * 4096, FLAGS);
    const uint32_t wv = PARTS == 2 ? (uint32_t)((jj >> 3) * 64 + q * 16 + col0 + (jj & 7)) * 16u : lane * 16u;
#pragma unroll
    for (int c = 0; c < D; ++c)                                       // chunks past the slice: past the descriptor, zeros without traffic
#pragma unroll
        for (int l = 0; l < LW; ++l) wr[c][l] = bload128<2 /*nt*/>(rw, wv, (uint32_t)(c * 4 + l * PARTS) * 1024u);

    if constexpr (NORM) {
#pragma unroll
        for (int u = 0; u < kNormJobs; ++u) {
            const int j = job0 + u * waves, row = j / njob;
            if (row >= p.M) break;
            float v[8], ss = 0.f;
            act_unpack8<BF>(hv[u], v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[e] * v[e];
            ss = wave_sum(ss);
            if (lane == 0) ssq[row * 8 + (j - row * njob)] = ss;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kNormJobs; ++u) {
            const int j = job0 + u * waves, row = j / njob, vi = (j - row * njob) * 64 + lane;
            if (row >= p.M) break;
            float tot = 0.f;
            for (int i = 0; i < njob; ++i) tot += ssq[row * 8 + i];
            const float rs = rsqrtf(tot / (float)p.K + p.eps);
            float v[8], g[8], o[8];
            act_unpack8<BF>(hv[u], v);
            act_unpack8<BF>(gv[u], g);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = g[e] * act_round<BF>(v[e] * rs);
            if (vi < pieces) xs[row * pieces + (vi ^ (row & 15))] = act_pack8<BF>(o);
        }
        __syncthreads();
    }
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const int xrow = min(jj, p.M - 1);                                // a column of the product past the rows is not stored
    const u32x4* xl = xs + xrow * pieces;
#pragma unroll
    for (int c = 0; c < D; ++c)
        if (c < n_ch) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                u32x4 a = wr[c][s / PARTS], b;
                if (PARTS == 2 && (s & 1)) {                          // lanes jj < 8 take jj + 8
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)a[e], 0x128, 0xF, 0xF, true);
                }
                if constexpr (NORM) b = xl[((c0 + c) * 16 + s * 4 + q) ^ (xrow & 15)];
                else {
                    b = xr[c][s / SPL];
                    switch (s % SPL * RPL) {                          // lanes jj < RPL take jj + RPL (s % SPL): row_shl
                    case 4: for (int e = 0; e < 4; ++e) b[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b[e], 0x104, 0xF, 0xF, true); break;
                    case 8: for (int e = 0; e < 4; ++e) b[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b[e], 0x108, 0xF, 0xF, true); break;
                    case 12: for (int e = 0; e < 4; ++e) b[e] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)b[e], 0x10C, 0xF, 0xF, true); break;
                    default: break;
                    }
                }
                acc = mfma_act<BF>(a, b, acc);
            }
        }
    if constexpr (EPI != R16_SILU) {
        if (wave < kwaves) red[wave * 64 + lane] = acc;
        __syncthreads();
    }
    if (!mine) return;
    auto sum = [&](int tt) {                                          // the slices of tile tt, in order, as the slabs were added
        f32x4 v = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < p.slices; s0 += 4) {
            f32x4 a[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) a[u] = red[(tt * p.slices + min(s0 + u, p.slices - 1)) * 64 + lane];
#pragma unroll
            for (int u = 0; u < 4; ++u) if (s0 + u < p.slices) v += a[u];
        }
        return v;
    };
    if constexpr (EPI == R16_ROPE) {
        const RopeEpi& R = p.r;
        const f32x4 v0 = sum(0), v1 = sum(1);
        const int h = n0 / R.hd, d0 = n0 - h * R.hd;
        const float b0[4] = {act_lo<BF>(pre0[0]), act_hi<BF>(pre0[0]), act_lo<BF>(pre0[1]), act_hi<BF>(pre0[1])};
        const float b1[4] = {act_lo<BF>(pre1[0]), act_hi<BF>(pre1[0]), act_lo<BF>(pre1[1]), act_hi<BF>(pre1[1])};
        float x0[4], x1[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) { x0[e] = act_round<BF>(v0[e] + b0[e]); x1[e] = act_round<BF>(v1[e] + b1[e]); }   // the linear's output is a 16-bit tensor
        rope_rows_out(R, jj, h, d0, x0, x1, pre_pos, pre_blk, [&](f32x4& lo, f32x4& hi) { lo = cs01; hi = cs23; }, [](float x) { return act_round<BF>(x); },
                      [](float x, float y) { return act_pack<BF>(x, y); });
    } else {
        if (n0 >= p.N) return;
        if constexpr (EPI == R16_SLAB) {
            *reinterpret_cast<f32x4*>(p.slab + (size_t)jj * p.N_pad + n0) = sum(wave);
        } else if constexpr (EPI == R16_RESID) {
            const f32x4 v = sum(wave);
            const float r[4] = {act_lo<BF>(pre0[0]), act_hi<BF>(pre0[0]), act_lo<BF>(pre0[1]), act_hi<BF>(pre0[1])};
            float o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = act_round<BF>(v[e]) + r[e];
            *reinterpret_cast<u32x2*>(p.res_out + (size_t)jj * p.N + n0) = u32x2{act_pack<BF>(o[0], o[1]), act_pack<BF>(o[2], o[3])};
        } else {
            *reinterpret_cast<uint32_t*>(p.y + (size_t)jj * (p.N / 2) + (n0 >> 1)) = silu_pair<BF>(acc);   // one slice (checked on the host), this wave's
        }
    }
}

// The launch's shape, or false: M rows, the splits that the staged kernel would take (mi355_gemm_plan: shapes without k-groups), no slice of more chunks than a form has (gate_up's one slice
// bounds the hidden size), few enough columns for the grid.
bool rows16_shape(int M, const mi355_weight_t* w, int epi, int max_splits, Rows16Params& p, int& waves, size_t& lds) {
    if (!w || !w->qweight || w->wbits != 16 || M < 1 || M > kRows16 || w->K % 128 != 0 || w->K_pad != w->K || w->N % 16 != 0 || w->N_pad != w->N) return false;
    if (epi == R16_RESID ? w->N > kHidden : w->K > kHidden) return false;
    int cfg = 0, cps = 0;
    const int slices = mi355_gemm_plan(M, w, max_splits, &cfg, &cps);
    if (cfg != 5 || cps > (epi == R16_SILU ? 8 : 3) || (epi == R16_SILU && slices != 1)) return false;
    p.M = M; p.K = w->K; p.N = w->N; p.N_pad = w->N_pad; p.NT = w->N_pad / 16; p.KC = w->K_pad / 128; p.qw = w->qweight;
    p.slices = slices; p.cps = cps; p.x_bytes = (uint32_t)((size_t)M * w->K * 2);
    // one round of blocks over the chip where a block has room for the tiles (RESID: K is deep, a tile a block); the cache writer's pair
    p.tw = epi == R16_ROPE ? 2 : epi == R16_SILU ? cdiv(p.NT, 256) : 1;
    p.units = epi == R16_ROPE ? p.NT / 2 : cdiv(p.NT, p.tw);
    const int kw = slices * p.tw;
    waves = epi == R16_RESID || kw > 8 ? kw : 8;                      // under the norm at least 8: eight rows of 1024 are kNormJobs jobs a wave
    lds = epi == R16_SILU ? 0 : (size_t)kw * 1024;
    if (epi != R16_RESID) lds += (size_t)M * w->K * 2 + 512;
    return waves <= (cps <= 3 ? 16 : 8);
}

template <bool BF, int EPI, int D, int PARTS, int XL = 1>
void launch_rows16_t(const Rows16Params& p, int waves, size_t lds, hipStream_t st) {
    hipLaunchKernelGGL((gemm_rows16_kernel<BF, EPI, D, PARTS, XL>), dim3(p.units * PARTS), dim3(64 * waves), lds, st, p);
}
template <bool BF, int EPI>
void launch_rows16_bf(const Rows16Params& p, int waves, size_t lds, hipStream_t st) {
    if constexpr (EPI == R16_RESID) { if (p.M <= 4) launch_rows16_t<BF, EPI, 3, 2, 1>(p, waves, lds, st); else launch_rows16_t<BF, EPI, 3, 2, 2>(p, waves, lds, st); }
    else if constexpr (EPI == R16_SILU) { if (p.cps <= 3) launch_rows16_t<BF, EPI, 3, 1>(p, waves, lds, st); else launch_rows16_t<BF, EPI, 8, 1>(p, waves, lds, st); }
    else { if (p.units <= 128) launch_rows16_t<BF, EPI, 3, 2>(p, waves, lds, st); else launch_rows16_t<BF, EPI, 3, 1>(p, waves, lds, st); }
}
template <int EPI>
int launch_rows16(const Rows16Params& p, bool bf, int waves, size_t lds, hipStream_t st) {
    if (bf) launch_rows16_bf<true, EPI>(p, waves, lds, st); else launch_rows16_bf<false, EPI>(p, waves, lds, st);
    MI355_CHECK_LAUNCH("gemm_rows16_kernel");
    return MI355_OK;
}

} // namespace

// Does a layer of these linears run on these launches at M rows (all four, or none)?
extern "C" int mi355_rows16_ok(int M, const mi355_weight_t* qkv, const mi355_weight_t* o, const mi355_weight_t* gate_up, const mi355_weight_t* down, int quantised_cache, int max_splits) {
    Rows16Params p{};
    int waves; size_t lds;
    return rows16_shape(M, qkv, quantised_cache ? R16_SLAB : R16_ROPE, max_splits, p, waves, lds) && rows16_shape(M, o, R16_RESID, max_splits, p, waves, lds) &&
           rows16_shape(M, gate_up, R16_SILU, 1, p, waves, lds) && rows16_shape(M, down, R16_RESID, max_splits, p, waves, lds);
}

// h [M][K]: the residual rows.  kv with a 16-bit cache: bias, RoPE, Q and the cache write; kv null: fp32 sums in slab [M][N_pad].
extern "C" int mi355_rows16_norm_qkv(const void* h, int M, const mi355_weight_t* w, const void* norm_weight, float eps, const void* bias, const float* cos_sin, int max_pos,
                                     const int32_t* positions, const int32_t* block_table, int max_blocks_per_seq, int q_len, int nh, const mi355_kv_layer_t* kv, void* q_out,
                                     int32_t* oob_count, float* slab, int max_splits, mi355_stream_t stream) {
    Rows16Params p{};
    int waves; size_t lds;
    MI355_CHECK_ARG(h && norm_weight && (kv ? cos_sin && positions && block_table && q_out && q_len >= 1 : slab != nullptr), "rows16_norm_qkv: bad args");
    if (!rows16_shape(M, w, kv ? R16_ROPE : R16_SLAB, max_splits, p, waves, lds)) return MI355_ERR_UNSUPPORTED;
    p.x = (const f16*)h; p.gamma = (const f16*)norm_weight; p.eps = eps; p.bias = (const f16*)bias; p.slab = slab;
    const bool bf = w->act_dtype == MI355_ACT_BF16;
    if (!kv) return launch_rows16<R16_SLAB>(p, bf, waves, lds, (hipStream_t)stream);
    if (kv->kv_dtype != (bf ? MI355_KV_BF16 : MI355_KV_FP16) || (kv->hd != 64 && kv->hd != 128) || w->N != (nh + 2 * kv->nkv) * kv->hd) return MI355_ERR_UNSUPPORTED;
    p.r = RopeEpi{cos_sin, positions, block_table, max_blocks_per_seq, nh, kv->nkv, kv->hd, kv->page, max_pos, kv->num_blocks, q_len, oob_count, kv->kv_base, (f16*)q_out};
    return launch_rows16<R16_ROPE>(p, bf, waves, lds, (hipStream_t)stream);
}

// h <- h + x W [M][N]
extern "C" int mi355_rows16_residual(const void* x, int M, const mi355_weight_t* w, void* h, int max_splits, mi355_stream_t stream) {
    Rows16Params p{};
    int waves; size_t lds;
    MI355_CHECK_ARG(x && h, "rows16_residual: bad args");
    if (!rows16_shape(M, w, R16_RESID, max_splits, p, waves, lds)) return MI355_ERR_UNSUPPORTED;
    p.x = (const f16*)x; p.res_in = (const f16*)h; p.res_out = (f16*)h;
    return launch_rows16<R16_RESID>(p, w->act_dtype == MI355_ACT_BF16, waves, lds, (hipStream_t)stream);
}

// y [M][N / 2] = silu(gate) * up of RMSNorm(h) W
extern "C" int mi355_rows16_norm_silu(const void* h, int M, const mi355_weight_t* w, const void* norm_weight, float eps, void* y, mi355_stream_t stream) {
    Rows16Params p{};
    int waves; size_t lds;
    MI355_CHECK_ARG(h && norm_weight && y, "rows16_norm_silu: bad args");
    if (!rows16_shape(M, w, R16_SILU, 1, p, waves, lds)) return MI355_ERR_UNSUPPORTED;
    p.x = (const f16*)h; p.gamma = (const f16*)norm_weight; p.eps = eps; p.y = (f16*)y;
    return launch_rows16<R16_SILU>(p, w->act_dtype == MI355_ACT_BF16, waves, lds, (hipStream_t)stream);
}
