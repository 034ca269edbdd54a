// (split-K reduce +) bias + RoPE + Q-extract + paged KV-cache write for decode, gfx950.
//
// Replaces FusedRopeKVCacheDecodeOp::forward (rtp_llm/models_py/bindings/rocm/
// FusedRopeKVCacheOp.cc:519-646 -> add_fusedQKV_bias_transpose_decode_kernel,
// rocm/kernels/fused_rope_kvcache_kernel.cu:1297-1466) and re-instates the INT8
// KV branch the reference removed: per-(token, kv-head) fp32 scale
// = max|x|/127, round-to-nearest-even + saturate (rocm_utils/_cast_to_int8.h:5-24), bytes stored as code + 128,
// scale plane [block][K|V][nkv][page] (kv_cache_utils.h:265-271).
//
// One wave per (token, head): lane i owns the NeoX pair (i, i + hd/2)
// (rotary_position_embedding.h:278-321,444-449: x' = cos*x - sin*y, y' = cos*y + sin*x
// in fp32, one rounding to fp16).  Launch-bound by nature (T*(nh+2nkv) waves).
#include "common.h"

namespace {

struct RopeParams {
    const f16*     qkv;
    const float*   partials;
    int            nsplit, ld;
    const f16*     bias;
    const float*   cos_sin;
    const int32_t* positions;
    const int32_t* block_table;
    int            max_blocks, T, nh, nkv, hd, page, max_pos, num_blocks, q_len;
    const int32_t* row_seq;   // non-null: the sequence of every row (t / q_len otherwise)
    int32_t*       oob_count;
    void*          kv_base;
    float*         scale_base;
    int            kv_int8;
    f16*           q_out;
};

// BF: qkv / bias / q_out and a 16-bit cache are bf16 (kv_dtype MI355_KV_BF16); the INT8 cache is quantised from the same fp32 values either way
template <bool BF>
__global__ __launch_bounds__(256) void rope_kv_write_kernel(const RopeParams p) {
    using raw16 = uint16_t;
    const int t    = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int h    = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int nheads = p.nh + 2 * p.nkv;
    if (h >= nheads) return;
    const int half = p.hd >> 1;
    const bool act = lane < half;
    const int col0 = h * p.hd + lane, col1 = col0 + half;

    // Everything is requested before the first wait (round 2 walked 8 dependent round trips: 4 slabs, 3 tail slabs one by
    // one, bias, position, rotation row, block id): the position and the block id are wave-uniform (scalar loads), the
    // slabs of a column are up to 16 independent loads, the rotation row follows the position.
    const int pos_in = p.positions[t];
    const int pos_lim = min(p.max_pos, p.max_blocks * p.page);
    const int pos = min(max(pos_in, 0), pos_lim - 1);       // clamped: the rotation table and the block table stay in range
    const bool is_v = h >= p.nh + p.nkv;
    const int blk = (h >= p.nh) ? p.block_table[(size_t)(p.row_seq ? p.row_seq[t] : t / p.q_len) * p.max_blocks + pos / p.page] : 0;
    float2 cs = {1.f, 0.f};
    if (!is_v && act) cs = *reinterpret_cast<const float2*>(p.cos_sin + ((size_t)pos * half + lane) * 2);
    float x0 = 0.f, x1 = 0.f;
    if (act) {
        float bh0 = 0.f, bh1 = 0.f;
        const raw16* bias = reinterpret_cast<const raw16*>(p.bias);
        if (p.partials) {
            const size_t sstride = (size_t)p.T * p.ld;
            const float* src = p.partials + (size_t)t * p.ld;
            for (int s0 = 0; s0 < p.nsplit; s0 += 8) {      // 8 slabs (16 loads) in flight per round trip, summed in index order
                float a[8], b[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {               // slabs past the end: re-read the last one, add zero
                    const int su = min(s0 + u, p.nsplit - 1);
                    a[u] = src[su * sstride + col0]; b[u] = src[su * sstride + col1];
                }
                if (s0 == 0 && p.bias) { bh0 = act_from_bits<BF>(bias[col0]); bh1 = act_from_bits<BF>(bias[col1]); }   // behind the slabs in the (in-order) queue
#pragma unroll
                for (int u = 0; u < 8; ++u) { const bool ok = s0 + u < p.nsplit; x0 += ok ? a[u] : 0.f; x1 += ok ? b[u] : 0.f; }
            }
        } else {
            const raw16* qkv = reinterpret_cast<const raw16*>(p.qkv);
            const raw16 q0 = qkv[(size_t)t * p.ld + col0], q1 = qkv[(size_t)t * p.ld + col1];
            if (p.bias) { bh0 = act_from_bits<BF>(bias[col0]); bh1 = act_from_bits<BF>(bias[col1]); }
            x0 = act_from_bits<BF>(q0); x1 = act_from_bits<BF>(q1);
        }
        x0 += bh0; x1 += bh1;
        // the QKV linear's output is a 16-bit tensor in the reference
        x0 = act_round<BF>(x0); x1 = act_round<BF>(x1);
    }
    if (!is_v && act) {
        const float r0 = cs.x * x0 - cs.y * x1;
        const float r1 = cs.x * x1 + cs.y * x0;
        x0 = act_round<BF>(r0); x1 = act_round<BF>(r1);
    }
    if (h < p.nh) {
        if (act) {
            raw16* dst = reinterpret_cast<raw16*>(p.q_out) + ((size_t)t * p.nh + h) * p.hd;
            dst[lane] = act_to_bits<BF>(x0); dst[lane + half] = act_to_bits<BF>(x1);
        }
        return;
    }
    // ---- K / V into the paged cache
    const int kh  = is_v ? h - p.nh - p.nkv : h - p.nh;
    if (pos_in < 0) return;                                  // padding row of a multi-row step: nothing to store
    if (pos != pos_in || blk < 0 || blk >= p.num_blocks) {   // stale position / block id: never write somebody else's page
        if (h == p.nh && lane == 0 && p.oob_count) atomicAdd(p.oob_count, 1);
        return;
    }
    const int tok = pos % p.page;
    const size_t head_elems = (size_t)p.page * p.hd;
    const size_t blk_base   = ((size_t)blk * 2 + (is_v ? 1 : 0)) * p.nkv + kh; // in units of heads
    int s0, s1; // element offsets inside this head's [page*hd] region
    if (!is_v) { s0 = tok * p.hd + lane; s1 = s0 + half; }
    else       { s0 = lane * p.page + tok; s1 = (lane + half) * p.page + tok; }
    if (!p.kv_int8) {
        if (act) {
            raw16* dst = (raw16*)p.kv_base + blk_base * head_elems;
            dst[s0] = act_to_bits<BF>(x0); dst[s1] = act_to_bits<BF>(x1);
        }
    } else {
        float amax = act ? fmaxf(fabsf(x0), fabsf(x1)) : 0.f;
        amax = wave_max(amax);
        const float scale = amax > 0.f ? amax / 127.f : 1.f;
        if (act) {
            int8_t* dst = (int8_t*)p.kv_base + blk_base * head_elems;
            const float q0 = fminf(fmaxf(rintf(x0 / scale), -128.f), 127.f);
            const float q1 = fminf(fmaxf(rintf(x1 / scale), -128.f), 127.f);
            // stored offset-binary (code + 128): the attention kernel widens bytes under an fp16 exponent, which wants
            // unsigned bytes -- flipping the top bit here (2 lanes x 1 op per token) saves it 2 VALU per 8 bytes there
            dst[s0] = (int8_t)((int)q0 ^ 0x80); dst[s1] = (int8_t)((int)q1 ^ 0x80);
        }
        if (lane == 0) p.scale_base[blk_base * p.page + tok] = scale;
    }
}

// The same for the rows of prompts (16-bit tensors and cache): a block takes 16 rows of 4 query or key heads, a thread 8 pairs of a row at a time in 16-byte loads and stores, or 16 rows of a value head,
// whose columns lie token by token in a page: through LDS, so that a store's lanes are 16 tokens of a column.  By a wave per row and head a value went out as 64 lines of 2 bytes, and the lines of
// consecutive rows from eight L2s.  us by waves / here: 28 over 4 heads of 128, 4096 rows 31.7 / 15.9
// (4.7 TB/s), 1055 10.5 / 6.6, 265 4.5 / 4.2; 14 over 2 of 64, 4096 15.7 / 6.1, 512 4.1 / 3.2; 32 over 32 of 64, 1055 25.8 / 8.6, 64 3.8 / 3.0.
constexpr int RP_ROWS = 16, RP_HEADS = 4;
template <bool BF, int HD>
__global__ __launch_bounds__(256) void rope_kv_prompt_kernel(const RopeParams p) {
    constexpr int half = HD / 2, P = half / 8, LD = HD + 2;                  // 16-byte pieces of a half, a row of values in LDS
    __shared__ uint32_t vs[RP_ROWS * LD / 2];
    const int t0 = blockIdx.x * RP_ROWS, nrot = p.nh + p.nkv, chunks = (nrot + RP_HEADS - 1) / RP_HEADS;
    const int pos_lim = min(p.max_pos, p.max_blocks * p.page);
    const uint16_t* qkv = reinterpret_cast<const uint16_t*>(p.qkv);
    const uint16_t* bias = reinterpret_cast<const uint16_t*>(p.bias);
    auto load8 = [&](int t, int col, float (&x)[8]) {                        // a row's 8 columns with their bias, rounded
        const u32x4 v = *reinterpret_cast<const u32x4*>(qkv + (size_t)t * p.ld + col);
        u32x4 b = {0, 0, 0, 0};
        if (bias) b = *reinterpret_cast<const u32x4*>(bias + col);
#pragma unroll
        for (int i = 0; i < 4; ++i) { x[2 * i] = act_round<BF>(act_lo<BF>(v[i]) + act_lo<BF>(b[i])); x[2 * i + 1] = act_round<BF>(act_hi<BF>(v[i]) + act_hi<BF>(b[i])); }
    };
    auto place = [&](int t, int pos_in, int pos, size_t heads, uint16_t*& dst, int& tok) -> int {     // the page of a row (heads: units of heads behind a block's first): 0 none, -1 out of range
        if (pos_in < 0) return 0;
        const int blk = p.block_table[(size_t)(p.row_seq ? p.row_seq[t] : t / p.q_len) * p.max_blocks + pos / p.page];
        if (pos != pos_in || blk < 0 || blk >= p.num_blocks) return -1;
        tok = pos % p.page;
        dst = (uint16_t*)p.kv_base + ((size_t)blk * 2 * p.nkv + heads) * p.page * HD;
        return 1;
    };
    if ((int)blockIdx.y < chunks) {
#pragma unroll
        for (int i = 0; i < RP_ROWS * RP_HEADS * P / 256; ++i) {
            const int item = i * 256 + (int)threadIdx.x, c = item % P * 8, h = blockIdx.y * RP_HEADS + item / P % RP_HEADS, t = t0 + item / (P * RP_HEADS);
            if (h >= nrot || t >= p.T) continue;
            const int pos_in = p.positions[t], pos = min(max(pos_in, 0), pos_lim - 1);
            float x0[8], x1[8];
            load8(t, h * HD + c, x0); load8(t, h * HD + half + c, x1);
            const float4* rot = reinterpret_cast<const float4*>(p.cos_sin + ((size_t)pos * half + c) * 2);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float4 cs = rot[k];
                const float a0 = x0[2 * k], b0 = x1[2 * k], a1 = x0[2 * k + 1], b1 = x1[2 * k + 1];
                x0[2 * k] = cs.x * a0 - cs.y * b0; x1[2 * k] = cs.x * b0 + cs.y * a0;
                x0[2 * k + 1] = cs.z * a1 - cs.w * b1; x1[2 * k + 1] = cs.z * b1 + cs.w * a1;
            }
            u32x4 y0, y1;
#pragma unroll
            for (int k = 0; k < 4; ++k) { y0[k] = act_pack<BF>(x0[2 * k], x0[2 * k + 1]); y1[k] = act_pack<BF>(x1[2 * k], x1[2 * k + 1]); }
            uint16_t* dst;
            if (h < p.nh) dst = reinterpret_cast<uint16_t*>(p.q_out) + ((size_t)t * p.nh + h) * HD + c;
            else {
                int tok = 0;
                const int at = place(t, pos_in, pos, h - p.nh, dst, tok);
                if (at < 0 && h == p.nh && c == 0 && p.oob_count) atomicAdd(p.oob_count, 1);
                if (at <= 0) continue;
                dst += tok * HD + c;
            }
            *reinterpret_cast<u32x4*>(dst) = y0;
            *reinterpret_cast<u32x4*>(dst + half) = y1;
        }
        return;
    }
    const int kh = (int)blockIdx.y - chunks;
    for (int item = threadIdx.x; item < RP_ROWS * HD / 8; item += 256) {
        const int r = item / (HD / 8), c = item % (HD / 8) * 8;
        if (t0 + r >= p.T) continue;
        float x[8];
        load8(t0 + r, (nrot + kh) * HD + c, x);
#pragma unroll
        for (int k = 0; k < 4; ++k) vs[(r * LD + c) / 2 + k] = act_pack<BF>(x[2 * k], x[2 * k + 1]);
    }
    __syncthreads();
    const int r = threadIdx.x % RP_ROWS, t = t0 + r;
    if (t >= p.T) return;
    const int pos_in = p.positions[t];
    uint16_t* dst;
    int tok = 0;
    if (place(t, pos_in, min(max(pos_in, 0), pos_lim - 1), p.nkv + kh, dst, tok) <= 0) return;
    for (int d = threadIdx.x / RP_ROWS; d < HD; d += 256 / RP_ROWS) dst[(size_t)d * p.page + tok] = reinterpret_cast<const uint16_t*>(vs)[r * LD + d];
}

} // namespace

extern "C" int mi355_rope_kv_write(const void* qkv_f16, const float* partials, int32_t nsplit, int32_t ld,
                                   const void* qkv_bias, const float* cos_sin, int32_t rope_dim, int32_t max_pos,
                                   const int32_t* positions, const int32_t* block_table, int32_t max_blocks_per_seq,
                                   int32_t T, int32_t nh, const mi355_kv_layer_t* kv, void* q_out, int32_t* oob_count,
                                   mi355_stream_t stream) {
    return mi355_rope_kv_write_rows(qkv_f16, partials, nsplit, ld, qkv_bias, cos_sin, rope_dim, max_pos, positions, block_table,
                                    max_blocks_per_seq, T, 1, nh, kv, q_out, oob_count, stream);
}

extern "C" int mi355_rope_kv_write_rows(const void* qkv_f16, const float* partials, int32_t nsplit, int32_t ld,
                                        const void* qkv_bias, const float* cos_sin, int32_t rope_dim, int32_t max_pos,
                                        const int32_t* positions, const int32_t* block_table, int32_t max_blocks_per_seq,
                                        int32_t T, int32_t q_len, int32_t nh, const mi355_kv_layer_t* kv, void* q_out,
                                        int32_t* oob_count, mi355_stream_t stream) {
    return mi355_rope_kv_write_rows_ragged(qkv_f16, partials, nsplit, ld, qkv_bias, cos_sin, rope_dim, max_pos, positions, nullptr, block_table,
                                           max_blocks_per_seq, T, q_len, nh, kv, q_out, oob_count, stream);
}

// row_seq non-null (device, [T]): the sequence of every row; q_len is 1 then
extern "C" int mi355_rope_kv_write_rows_ragged(const void* qkv_f16, const float* partials, int32_t nsplit, int32_t ld,
                                               const void* qkv_bias, const float* cos_sin, int32_t rope_dim, int32_t max_pos,
                                               const int32_t* positions, const int32_t* row_seq, const int32_t* block_table, int32_t max_blocks_per_seq,
                                               int32_t T, int32_t q_len, int32_t nh, const mi355_kv_layer_t* kv, void* q_out,
                                               int32_t* oob_count, mi355_stream_t stream) {
    MI355_CHECK_ARG(q_len >= 1 && T % q_len == 0, "rope_kv_write: T=%d must be a multiple of q_len=%d", T, q_len);
    MI355_CHECK_ARG((qkv_f16 != nullptr) != (partials != nullptr), "rope_kv_write: exactly one of qkv_f16 / partials");
    MI355_CHECK_ARG(kv && kv->kv_base && cos_sin && positions && block_table && q_out, "rope_kv_write: null pointer");
    MI355_CHECK_ARG(kv->hd == 64 || kv->hd == 128, "rope_kv_write: hd=%d (64 or 128)", kv->hd);
    MI355_CHECK_ARG(rope_dim == kv->hd, "rope_kv_write: rope_dim=%d must equal hd=%d", rope_dim, kv->hd);
    MI355_CHECK_ARG(kv->page > 0 && T > 0 && nh > 0 && kv->nkv > 0 && max_pos > 0 && max_blocks_per_seq > 0 && kv->num_blocks > 0,
                    "rope_kv_write: bad dims");
    MI355_CHECK_ARG(kv->kv_dtype == MI355_KV_FP16 || kv->kv_dtype == MI355_KV_BF16 || (kv->kv_dtype == MI355_KV_INT8 && kv->scale_base),
                    "rope_kv_write: int8 cache needs scale_base");
    const bool bf = kv->act_dtype == MI355_ACT_BF16;
    MI355_CHECK_ARG((kv->act_dtype == MI355_ACT_F16 || bf) && (kv->kv_dtype == MI355_KV_INT8 || bf == (kv->kv_dtype == MI355_KV_BF16)),
                    "rope_kv_write: act_dtype=%d with kv_dtype=%d (a 16-bit cache has the dtype of the activations)", kv->act_dtype, kv->kv_dtype);
    const int nheads = nh + 2 * kv->nkv;
    MI355_CHECK_ARG(ld >= nheads * kv->hd, "rope_kv_write: ld=%d", ld);
    RopeParams p;
    p.qkv = (const f16*)qkv_f16; p.partials = partials; p.nsplit = nsplit; p.ld = ld; p.bias = (const f16*)qkv_bias;
    p.cos_sin = cos_sin; p.positions = positions; p.block_table = block_table; p.max_blocks = max_blocks_per_seq;
    p.T = T; p.nh = nh; p.nkv = kv->nkv; p.hd = kv->hd; p.page = kv->page; p.kv_base = kv->kv_base;
    p.max_pos = max_pos; p.num_blocks = kv->num_blocks; p.oob_count = oob_count; p.q_len = q_len; p.row_seq = row_seq;
    p.scale_base = kv->scale_base; p.kv_int8 = kv->kv_dtype == MI355_KV_INT8; p.q_out = (f16*)q_out;
    const uintptr_t at = (uintptr_t)qkv_f16 | (uintptr_t)qkv_bias | (uintptr_t)cos_sin | (uintptr_t)q_out | (uintptr_t)kv->kv_base;
    // Few waves: a block's two trips of 16 bytes a thread take longer than one wave's single one.  28 over 4 heads of 128, us by waves / by blocks: 64 rows 3.2 / 3.9, 192 3.9 / 4.1, 265 4.5 / 4.2; 5 over 1, 512
    // rows 3.4 / 4.4, 1055 4.4 / 4.3.  Heads of 64 (one trip): 64 rows 2.9 / 2.9, 192 3.2 / 3.2.
    if (T >= 64 && (kv->hd == 64 || (long)T * nheads >= 7400) && qkv_f16 && !p.kv_int8 && at % 16 == 0 && ld % 8 == 0) {
        const dim3 grid(cdiv(T, RP_ROWS), cdiv(nh + kv->nkv, RP_HEADS) + kv->nkv);
        hipStream_t st = (hipStream_t)stream;
        if (kv->hd == 128) { if (bf) hipLaunchKernelGGL((rope_kv_prompt_kernel<true, 128>), grid, dim3(256), 0, st, p);
                             else    hipLaunchKernelGGL((rope_kv_prompt_kernel<false, 128>), grid, dim3(256), 0, st, p); }
        else               { if (bf) hipLaunchKernelGGL((rope_kv_prompt_kernel<true, 64>), grid, dim3(256), 0, st, p);
                             else    hipLaunchKernelGGL((rope_kv_prompt_kernel<false, 64>), grid, dim3(256), 0, st, p); }
        MI355_CHECK_LAUNCH("rope_kv_prompt_kernel");
        return MI355_OK;
    }
    if (bf)
        hipLaunchKernelGGL(rope_kv_write_kernel<true>, dim3(T, cdiv(nheads, 4)), dim3(256), 0, (hipStream_t)stream, p);
    else
        hipLaunchKernelGGL(rope_kv_write_kernel<false>, dim3(T, cdiv(nheads, 4)), dim3(256), 0, (hipStream_t)stream, p);
    MI355_CHECK_LAUNCH("rope_kv_write_kernel");
    return MI355_OK;
}
