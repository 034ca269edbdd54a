// Parameter block, epilogue kinds and the per-wave stamps shared by the full-K launches: gemm_fullk.hip (<= 16 rows and the
// generic shapes) and gemm_fullk64.hip (1-64 rows, W4 group-wise).
#pragma once
#include "gemm_common.h"

namespace {

struct RopeEpi {
    const float*   cos_sin;
    const int32_t* positions;
    const int32_t* block_table;
    int            max_blocks, nh, nkv, hd, page, max_pos, num_blocks, q_len;
    int32_t*       oob_count;
    void*          kv_base;
    f16*           q_out;
};
// What a lane of a linear with the rotation and the 16-bit cache write inside does with its columns: x0 = dims d0..d0+3 of head h of row m, x1 = the same of the head's upper half, with the bias and
// rounded to the activation type; rot gives {cos, sin} of dims d0, d0+1 and d0+2, d0+3 (asked for where the head is rotated); pos_in and blk are the row's position and the block that its table has
// at the clamped position.  round and pack: the activation type's.  Rows of a negative position are padding and write no cache; a position past the pages or the rotations and a block id outside the
// cache are refused and counted once a row, by the lane of the first K head's first dims: never somebody else's page.
template <class Rot, class Round, class Pack>
__device__ __forceinline__ void rope_rows_out(const RopeEpi& R, int m, int h, int d0, float (&x0)[4], float (&x1)[4], int pos_in, int blk, Rot rot, Round round, Pack pack) {
    const int half = R.hd >> 1, pos = min(max(pos_in, 0), min(R.max_pos, R.max_blocks * R.page) - 1);
    const bool is_v = h >= R.nh + R.nkv;
    if (!is_v) {
        f32x4 cs01, cs23;
        rot(cs01, cs23);
        const float c[4] = {cs01[0], cs01[2], cs23[0], cs23[2]}, s[4] = {cs01[1], cs01[3], cs23[1], cs23[3]};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float r0 = c[e] * x0[e] - s[e] * x1[e];
            const float r1 = c[e] * x1[e] + s[e] * x0[e];
            x0[e] = round(r0); x1[e] = round(r1);
        }
    }
    const u32x2 o0 = {pack(x0[0], x0[1]), pack(x0[2], x0[3])}, o1 = {pack(x1[0], x1[1]), pack(x1[2], x1[3])};
    if (h < R.nh) {
        f16* dst = R.q_out + ((size_t)m * R.nh + h) * R.hd + d0;
        *reinterpret_cast<u32x2*>(dst) = o0;
        *reinterpret_cast<u32x2*>(dst + half) = o1;
        return;
    }
    if (pos_in < 0) return;
    if (pos != pos_in || blk < 0 || blk >= R.num_blocks) {
        if (h == R.nh && d0 == 0 && R.oob_count) atomicAdd(R.oob_count, 1);
        return;
    }
    const int kh = is_v ? h - R.nh - R.nkv : h - R.nh, tok = pos % R.page;
    uint16_t* dst = (uint16_t*)R.kv_base + (((size_t)blk * 2 + (is_v ? 1 : 0)) * R.nkv + kh) * ((size_t)R.page * R.hd);
    if (!is_v) {
        *reinterpret_cast<u32x2*>(dst + tok * R.hd + d0) = o0;
        *reinterpret_cast<u32x2*>(dst + tok * R.hd + d0 + half) = o1;
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dst[(d0 + e) * R.page + tok]        = (uint16_t)(o0[e >> 1] >> (16 * (e & 1)));
            dst[(d0 + e + half) * R.page + tok] = (uint16_t)(o1[e >> 1] >> (16 * (e & 1)));
        }
    }
}
struct FullKParams {
    GemmParams g;
    const f16* res_in;
    f16*       res_out;
    RopeEpi    r;
    // NORM: x is the un-normed residual row h; the kernel applies RMSNorm on the fly, x_n = gamma * fp16(h * rs), with
    // rs = rsqrt(sum_k h^2 / K + eps) rebuilt from the per-tile partial sums the producing launch left in ssq_in
    const float* ssq_in;     // [rows][ssq_ld], ssq_ld >= ssq_tiles: sum over the 16 columns of tile t of h[row]^2
    int          ssq_tiles, ssq_ld;
    const f16*   gamma;
    float        eps;
    float*       ssq_out;    // FK_RESID: the same partial sums of the rows this launch produces ([M][ssq_ld]), or null
    int          ilv;        // K slices of the waves interleaved chunk by chunk (see the kernel)
    // FK_RESID of gemm_fullk64.hip, deferred RMSNorm of the rows it produces: besides h' it stores g = fp16(gamma 2^-e h') as an
    // activation image for the next GEMM, which multiplies its accumulators by rsqrt(mean h'^2 + eps) 2^e (from ssq_out)
    f16*         xg_img;     // image of g ([M][N]), or null
    const f16*   xg_gamma;   // norm weight [N]
    float        xg_scale;   // 2^-e with e >= log2(max |gamma|): |g| <= |h'|, no overflow whatever the residual stream holds
    int          rowsplit;   // gemm_fullk64.hip: two blocks per tile pair, 32 rows each (block b: pair b / 2, row blocks 2 (b & 1) .. + 1)
    int          bf16;       // gemm_fullk64.hip: bias / residual / norm weight / q / KV cache are bf16 (the activation image and the MFMAs stay fp16)
    // FK_PUB (gemm_fullk64.hip, tensor parallelism; round 6): y = 16-bit(xW + bias) goes straight into THIS RANK'S REGISTERED ALL-REDUCE BUFFER
    // (csrc/allreduce.hip), in the slot and parity the next fused all-reduce launch of that context reads -- a row-parallel shard (O / down) then needs
    // neither split-K slabs nor the fold + publish stage in front of the flag exchange (mi355_allreduce_fused_published_dt).  Row m of a <= 64-row
    // call lives in slot m (one row per block), parity (epoch[m] + 1) & 1 of the context's device-resident call counters.
    const uint32_t* pub_epoch;
    void*           pub_data;
    uint32_t        pub_bytes, pub_parity_elems, pub_slot_elems;
    int             pub_plain;  // 1: plain stores (full-fence hand-over: the all-reduce launch's system-scope release fence publishes them); 0: write-through (sc0 sc1)
#ifdef MI355_FULLK_STAMPS   // tuning build with MI355_EXTRA_CFLAGS=-DMI355_FULLK_STAMPS only: the stamp stores change the schedule
    unsigned long long* stamps;   // tools/fullk_stamps.py: wall_clock64 per wave at entry / requests out (+ 1 / rms there) / first chunk done / loop done / slices met / exit
#endif
};
#ifdef MI355_FULLK_STAMPS
#define FK_STAMP(i) do { if (fp.stamps && lane == 0) fp.stamps[((size_t)blockIdx.x * 16 + wave) * 6 + (i)] = wall_clock64(); } while (0)
#else
#define FK_STAMP(i) do { } while (0)
#endif
enum { FK_PLAIN = 0, FK_RESID = 1, FK_ROPE = 2, FK_PUB = 3 };

} // namespace
