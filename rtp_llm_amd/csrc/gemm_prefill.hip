// GEMM on the packed weight images for large M (prefill chunks, more than 64 rows), gfx950.
//
// Same contract and weight image as gemm.hip (reference slot: LinearBase.forward,
// rtp_llm/models_py/modules/factory/linear/linear_base.py:75-85; the reference notes that weight-only quantisation "may
// cause performance degradation for long sequences during the Prefill phase", docs/backend/quantization.md:3 -- the
// decode kernels of this library would re-read every weight once per 64 rows).  Here the problem is compute-shaped:
//   * block = 8 waves; a wave owns 1, 2 or 4 adjacent 16-column weight tiles and all rows of the block's tile (32, 64 or 128);
//   * per 128-k chunk a wave dequantises its tiles' A-fragments ONCE (operand side) and uses each for every row block: at 128 rows 64 v_mfma_f32_16x16x32 per
//     104 dequant VALU, so the matrix pipe, not the VALU, sets the pace; the second wave of each SIMD dequantises while the first one multiplies;
//   * the activation chunk (128 rows x 128 k = 32 KiB) goes to LDS by DMA while the chunk before it is multiplied, row by row with the 16-byte pieces of a row swizzled
//     by the row (conflict-free ds_read_b128); two buffers, one barrier a chunk.  Through registers, as before, the chunk cost 16 of them, and with them the reach of the
//     fragment reads: 3 fragments are now read ahead of their products.  Both sides in turn on one machine: fp16 W4 37888 x 3584 and 3584 x 18944 at 4096 rows 6 and 7 % faster (at the rate
//     of a large dense product on the 224 of 256 CUs that have a block), the same in 8 bits at 1055 rows 8 and 1 %, bf16 W16 9728 x 896 at 512 rows 12 %.  Times move by 5 to 8 % between machines
//     and with the operands' values (power); those of the present loops are at WHOLE below;
//   * weights stream from HBM/L2 once per row tile (an XCD's blocks walk a column tile's row tiles together and meet in its L2: prefill_tile),
//     through a 2-deep register ring (128 x 512: half a chunk at a time, see WHOLE), buffer range checks instead of tail branches.
#include <type_traits>
#include "gemm_common.h"

namespace {

// the epilogue of gemm_store for bf16 tensors: bias, one rounding, SiLU-gate on the rounded pair
__device__ __forceinline__ void store_bf16(const GemmParams& p, f32x4 v, int m, int n0) {
    if (n0 >= p.N) return;
    if (p.bias) {
        const u32x2 b = *reinterpret_cast<const u32x2*>(p.bias + n0);
        v[0] += act_lo<true>(b[0]); v[1] += act_hi<true>(b[0]); v[2] += act_lo<true>(b[1]); v[3] += act_hi<true>(b[1]);
    }
    if (p.mode == MODE_SILU) {
        float o[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const float g = act_round<true>(v[2 * t]), u = act_round<true>(v[2 * t + 1]);
            o[t] = (g / (1.f + __expf(-g))) * u;
        }
        *reinterpret_cast<uint32_t*>((f16*)p.y + (size_t)m * p.ldy + (n0 >> 1)) = act_pack<true>(o[0], o[1]);
    } else {
        u32x2 o;
        o[0] = act_pack<true>(v[0], v[1]); o[1] = act_pack<true>(v[2], v[3]);
        *reinterpret_cast<u32x2*>((f16*)p.y + (size_t)m * p.ldy + n0) = o;
    }
}

// The stores of tiles two or four weight tiles wide to rows on 16 bytes: the finished values pass through LDS, so that a store writes 16 bytes a lane and whole runs of a row (128 bytes of it where
// a wave has 64 columns, 64 of gated ones).  From the accumulators a store was 16 rows by 32 bytes, of gated pairs 16 by 16, with a choice of mode, bias and image in front of each: us a block, before /
// now: 128 x 512 gated 10.7 / 5.2 (divisions), plain 7.6 / 3.0, 128 x 256 4.4 / 1.9, 64 x 256 2.2 / 1.3.  us a call: fp16 W4 at 4096 rows 37888 x 3584 gated 925 / 888, 3584 x 3584 97 / 90, 8 bits
// at 1055 rows 37888 x 3584 gated 270 / 256.
__device__ __forceinline__ bool lean_store(const GemmParams& p) {
    const bool silu = p.mode == MODE_SILU;
    return !p.y_img && (silu || p.mode == MODE_F16) && p.ldy % 8 == 0 && (uintptr_t)p.y % 16 == 0 && p.N % (silu ? 16 : 8) == 0;
}
// acc of a wave: row m0 + 16 mb + (lane & 15), columns n0 + 16 t + 4 (lane >> 4) + r, times the column's scale.  mine: the wave's 1 KB of LDS per 16 rows.  The arithmetic of gemm_store and store_bf16.
template <bool BF, int MB, int TPW, bool SILU>
__device__ __forceinline__ void store_rows(const GemmParams& p, const f32x4 (&acc)[TPW][MB], const f32x4 (&sc)[TPW], char* mine, int m0, int n0, int lane) {
    constexpr int RB = SILU ? TPW * 16 : TPW * 32, P = RB / 16;              // bytes and 16-byte pieces of a row of the wave's results
    constexpr int PH = MB * 1024 / (RB * 16) < MB ? MB * 1024 / (RB * 16) : MB;   // 16-row blocks that fit the wave's LDS together
    const int jj = lane & 15, q = lane >> 4;
    auto place = [](int row, int piece) { return row * RB + ((piece ^ (P == 8 ? row & 7 : P == 4 ? (row >> 1) & 3 : (row >> 2) & 1)) << 4); };
    f32x4 bias[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        bias[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int n = n0 + t * 16 + q * 4;
        if (p.bias && n < p.N) {
            const u32x2 b = *reinterpret_cast<const u32x2*>(p.bias + n);
            bias[t] = f32x4{act_lo<BF>(b[0]), act_hi<BF>(b[0]), act_lo<BF>(b[1]), act_hi<BF>(b[1])};
        }
    }
#pragma unroll
    for (int p0 = 0; p0 < MB; p0 += PH) {
#pragma unroll
        for (int mb = p0; mb < p0 + PH; ++mb)
#pragma unroll
            for (int t = 0; t < TPW; ++t) {
                f32x4 v = acc[t][mb] * sc[t];
                if (p.bias) v += bias[t];
                const int row = (mb - p0) * 16 + jj;
                if constexpr (SILU) {
                    float o[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const float g = act_round<BF>(v[2 * e]), u = act_round<BF>(v[2 * e + 1]);
                        o[e] = (g / (1.f + __expf(-g))) * u;
                    }
                    *(uint32_t*)(mine + place(row, t) + q * 4) = act_pack<BF>(o[0], o[1]);
                } else *(u32x2*)(mine + place(row, t * 2 + (q >> 1)) + (q & 1) * 8) = u32x2{act_pack<BF>(v[0], v[1]), act_pack<BF>(v[2], v[3])};
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                  // the wave's own, read by its other lanes
        const int r0 = lane / P, piece = lane % P, col = (SILU ? n0 >> 1 : n0) + piece * 8, m = m0 + p0 * 16 + r0;
        f16* y = (f16*)p.y + (size_t)m * p.ldy + col;
        const bool ok = col < (SILU ? p.N >> 1 : p.N);
#pragma unroll
        for (int k = 0; k < PH * 16 * P / 64; ++k) {
            const u32x4 v = *(const u32x4*)(mine + place(k * (64 / P) + r0, piece));
            if (ok && m + k * (64 / P) < p.M) *(u32x4*)(y + (size_t)(k * (64 / P)) * p.ldy) = v;
        }
        if (p0 + PH < MB) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
}

// The chip deals consecutive blocks to its eight XCDs in turn, each with an L2 of its own.  Dealt row by row, the 32 blocks of an XCD read 32 column tiles of the weights
// and hardly share one: at 128 x 512 tiles 2 MB of 8-bit codes per XCD and 128-k chunk from the Infinity Cache, 5.7 TB/s over the chip.  So an XCD takes a contiguous run
// of tiles in an order of bands of up to PF_BAND row tiles, column by column: per chunk 4 column tiles and 8 row tiles, a quarter of the bytes.  Column counts that eight
// divides stay in rows: there an XCD has its columns to itself anyway, and their weights stay in its L2 from one row tile to the next (72 columns 1.6 % faster so, 32
// columns 2 to 3 %).  us in rows / in bands: 8 bits 37888 x 3584 at 1055 rows 300 / 266, W4 at 4096 rows 1005 / 985, W16 11008 x 4096 at 2667 rows 418 / 315, 896 x 4864 at
// 1753 rows 42 / 36; 110 random calls 0.97 of the time in rows; bands of 6, 8 and 12 alike, 24 1 % slower.  Tiles that stay in rows are the launch's own blocks: the divisions that
// find a tile stand in front of a block's first load, 0.9 us of 15.  In bands except where K is short (up to 8 whole chunks of
// 128) for more than 192 rows, a column tile's weights are below 128 KB and x below 4 MB: a band's blocks of an XCD all wait for the same strip of weights, and the launch is over before reading it
// once pays.  565 random calls of 65 to 4096 rows, band / rows: 422 in bands 0.958 (39 above 1.03, at worst 1.11), 143 in rows 1.031
// (0.96 to 1.13; W4 896 x 896 at 292 rows 5.2 / 5.9 us, 8 bits 5.2 / 5.6).
constexpr int PF_XCD = 8, PF_BAND = 8;
bool prefill_short(const GemmParams& p, int wbits, int tile_cols) {
    return p.K % 128 == 0 && p.K <= 1024 && p.M > 192 && (uint64_t)p.KC * 16 * tile_cols * wbits < 128 << 10 && (uint64_t)p.M * p.K * 2 < 4 << 20;
}
int prefill_band(int rows, int cols) {                        // 0: in rows; else the height of all bands but the last
    const int bands = (rows + PF_BAND - 1) / PF_BAND;
    return cols % PF_XCD == 0 ? 0 : (rows + bands - 1) / bands;
}
__host__ __device__ __forceinline__ void prefill_tile(int id, int rows, int cols, int band, int& bx, int& by) {
    const int nb = rows * cols, k = id % PF_XCD, j = k * (nb / PF_XCD) + (k < nb % PF_XCD ? k : nb % PF_XCD) + id / PF_XCD;
    const int r0 = band >= rows ? 0 : j / (band * cols) * band, i = j - r0 * cols, h = band < rows - r0 ? band : rows - r0;
    bx = i / h; by = r0 + i % h;
}

// One block = 8 waves: NWN = 8 / KS of them side by side along N, KS of them along K (slice ks takes the chunks c with c % KS == ks; the slices' sums meet in
// LDS at the end).  TPW = weight tiles per wave, MB = 16-row blocks of the tile, so the tile is 16 MB rows x 16 TPW NWN columns.
//   TPW = 4, MB = 8 (128 x 512, one block per CU): one B-fragment read from LDS feeds four MFMAs.  At TPW = 2 (128 x 256, two blocks per CU) the 8 waves of a
//   block pull 256 KiB of fragments per 128-k chunk through the CU's LDS port for 512 MFMAs -- 2048 cycles of each, neither hidden behind the other.
//   MB = 4 and the K-sliced forms are for grids that would leave most CUs without a block (narrow outputs, short prompts): see pick_shape.
// BF: bf16 activations.  16-bit weights are the MFMA operand as they are; a 4-bit code enters it as the exact integer u - z and the group's scale multiplies the
// group's fp32 sums (a bf16 product s (u - z) would round the weight to 8 bits); an 8-bit code as the exact u - 128, its column scale on the finished sums.
// WHOLE: K is a multiple of 128 and x lies on 16 bytes, so that every chunk comes by DMA and the loop has no branch.  With the branches of the general loop the
// compiler's count of loads in flight, taken over all paths, made the products wait for the DMA of the chunk after (37 to 42 % of the waves' time at 128 x 512 went into
// waits), and the first three fragment reads of a chunk waited one by one.  In front of the last chunk of a straight loop lies one DMA too many (K sliced: left out);
// it reads a chunk again that is there, and is waited for.
// us general / WHOLE, same bits, one shape, both with the stores from the accumulators: 8 bits 37888 x 3584 at 1055 rows 279 / 263 (128 x 512), 3584 x 18944 155 / 136
// (64 x 256); fp16 W4 37888 x 3584 at 4096 rows 1060 / 1004 (power), 3584 x 3584 at 512 rows 36 / 32 (64 x 256), 26.6 / 22.7 (64 x 128); bf16 W4 37888 x 3584 at 4096 rows
// 1257 / 1091 (128 x 256); W16 896 x 4864 at 777 rows 21.3 / 19.1 (64 x 64), 9728 x 896 39 / 34 (32 x 64).  Whole calls of the present code, plain, us: 8 bits 235 and 134,
// fp16 W4 845 (two shapes) and 21.4, bf16 W4 1068, W16 16.5; fp16 W4 at 4096 rows 1305 TFLOP/s over the four linears of a 7B layer, 1639 on zeros.
// The 128 x 512 form has 128 registers of sums and none for two chunks of weights: it holds one chunk's, each half loaded again as soon as its last operand is formed
// (a little more than half a chunk, 1.4 us, ahead of its use; the other row tiles of the XCD's band have most of them in L2).  230 and 236 registers; a ring of two spills.
template <int WBITS, int TPW, int MB, int AHEAD>
__device__ __forceinline__ void pace(int i0, int n) {         // the order of fragment reads, products and operand arithmetic of fragments i0 .. i0 + n - 1 of a chunk
#pragma unroll
    for (int i = i0; i < i0 + n; ++i) {
        if (i + AHEAD < 4 * MB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if constexpr (WBITS != 16) __builtin_amdgcn_sched_group_barrier(0x002, (14 + MB - 1) / MB, 0);
        }
    }
}
// Waves a SIMD that the registers have to leave room for.  The general loop of 4-bit weights in groups of 64 and 128: 8 for 32 x 64 (64 registers, four blocks a CU; left alone the compiler takes
// 62 to 67), 6 for bf16 in 64 x 128 (80, three blocks; it takes 77 and 90).  bf16 9728 x 896 in groups of 64 at 395 rows 22.6 -> 20.0 us, fp16 1408 x 256 at 362 rows 4.6 -> 3.9.
constexpr int prefill_waves(int wbits, int gs, bool bf, int mb, int tpw, int ks, bool whole) {
    if (wbits == 4 && gs != 1 && !whole && mb == 2 && ks == 2) return 8;
    if (wbits == 4 && gs != 1 && !whole && bf && mb == 4 && tpw == 1 && ks == 1) return 6;
    return tpw * mb <= 16 && wbits != 16 && !(bf && wbits == 4) ? 2 : 1;
}
// xmem: the block's LDS, 8 MB KS KB; the block's tile: rows from m0 on, weight tiles from nt_block on
template <int WBITS, int GS, bool BF, int MB, int TPW, int KS, bool WHOLE>
__device__ __forceinline__ void prefill_block(const GemmParams& p, u32x4* xmem, const int m0, const int nt_block) {
    constexpr int NWN = 8 / KS;                               // waves side by side
    constexpr int LPC  = WBITS / 4;
    constexpr int NSUB = (GS > 0) ? 4 / GS : 1;
    constexpr int SPG  = 4 / NSUB;
    constexpr bool GROUPED = GS > 0;
    constexpr bool CSCALE = BF && GROUPED;                    // the group's scale on the accumulator side
    constexpr int XSLOTS = 256 * MB;                          // 16-byte pieces of an x chunk tile
    constexpr int UPT = XSLOTS / (64 * NWN);                  // staging loads per wave
    constexpr bool HALVES = WHOLE && TPW == 4;                // the weights of half a chunk in registers, not of two chunks
    constexpr int WLD = TPW * ((HALVES ? 2 : LPC) + (GS > 0 ? NSUB : 0));     // weight loads per wave and chunk
    static_assert(!HALVES || (WBITS != 16 && !CSCALE && NSUB == 1 && KS == 1), "one scale a chunk");
    u32x4 (*xs)[2][XSLOTS] = (u32x4(*)[2][XSLOTS])xmem;
    static_assert(KS == 1 || (size_t)(KS - 1) * NWN * TPW * MB * 1024 <= sizeof(u32x4) * 2 * KS * XSLOTS, "the slices' sums meet in the x buffers");

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ks = wave / NWN;
    const int jj = lane & 15, q = lane >> 4;
    const int nt_base = nt_block + wave % NWN * TPW;
    const int KC = p.KC;

    constexpr uint32_t FLAGS = 0x00020000u;
    __amdgpu_buffer_rsrc_t rw[TPW], rm[TPW];
    bool tile_ok[TPW];
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        const int nt = nt_base + t;
        tile_ok[t] = nt < p.NT;
        const char* wb = (const char*)p.qw + (size_t)nt * KC * (LPC * 1024);
        rw[t] = __builtin_amdgcn_make_buffer_rsrc((void*)wb, 0, tile_ok[t] ? KC * LPC * 1024 : 0, FLAGS);
        const char* mb = (const char*)p.meta + (size_t)nt * 16 * 4;
        const int mbytes = GROUPED ? ((KC * NSUB - 1) * p.N_pad + 16) * 4 : 64;
        rm[t] = __builtin_amdgcn_make_buffer_rsrc((void*)mb, 0, tile_ok[t] && WBITS != 16 ? mbytes : 0, FLAGS);
    }
    __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, p.x_bytes, FLAGS);

    // x staging: load u of a wave covers 64 pieces of 16 bytes = 4 rows of the chunk; piece pp of row j lies at j * 16 + (pp ^ (j & 15))
    uint32_t xoff[UPT];
#pragma unroll
    for (int u = 0; u < UPT; ++u) {
        const int pi = (u * NWN + wave % NWN) * 64 + lane, j = pi >> 4, pp = (pi & 15) ^ (j & 15);
        xoff[u] = (uint32_t)(((size_t)min(m0 + j, p.M - 1) * p.K + pp * 8) * 2);      // rows past M repeat the last one: their sums are never stored
    }
    if constexpr (HALVES) {                                   // load u starts 32 u rows further down, at most at the last row: two registers for all
        const int j = wave * 4 + (lane >> 4), pp = (lane & 15) ^ (j & 15);
        xoff[0] = (uint32_t)(m0 + j) * (uint32_t)p.K * 2u + pp * 16u;
        xoff[1] = (uint32_t)(p.M - 1) * (uint32_t)p.K * 2u + pp * 16u;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)&xs[ks][0][0];
    const bool dma = WHOLE || ((uintptr_t)p.x % 16 == 0 && p.K % 8 == 0);
    auto load_x = [&](int c, int buf) __attribute__((always_inline)) {
        if constexpr (HALVES) {
            asm volatile("" : "+v"(xoff[0]));                 // the sums are formed here, not kept through the loop
#pragma unroll
            for (int u = 0; u < UPT; ++u)
                dma16(lds0 + (buf * XSLOTS + (u * NWN + wave % NWN) * 64) * 16, min(xoff[0] + (uint32_t)u * 64u * (uint32_t)p.K, xoff[1]), (const char*)p.x + (size_t)c * 256);
        } else if (WHOLE || (dma && c * 128 + 128 <= p.K)) {
#pragma unroll
            for (int u = 0; u < UPT; ++u)
                dma16(lds0 + (buf * XSLOTS + (u * NWN + wave % NWN) * 64) * 16, xoff[u], (const char*)p.x + (size_t)c * 256);
        } else {                                              // the last chunk of a K that is no multiple of 128 (columns past K are zero), a tensor off 16 bytes
#pragma unroll
            for (int u = 0; u < UPT; ++u) {
                const int pi = (u * NWN + wave % NWN) * 64 + lane, pp = (pi & 15) ^ (pi >> 4 & 15);
                xs[ks][buf][pi] = bload128<0>(rx, c * 128 + pp * 8 < p.K ? xoff[u] : 0x80000000u, (uint32_t)c * 256u);
            }
        }
    };

    const uint32_t lane16 = lane * 16u, jj4 = jj * 4u;
    u32x4    wr[2][TPW][LPC];                                 // HALVES: wr[0][t][h] (8 bits) or the half-filled wr[0][t][0] (4 bits) are the chunk at work
    uint32_t mr[2][TPW][NSUB];
    auto load_half = [&](int h, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            if constexpr (WBITS == 8) wr[0][t][h % LPC] = bload128<0>(rw[t], lane16, (uint32_t)(c * LPC + h) * 1024u);
            else {
                const u32x2 v = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rw[t], lane16 + h * 8, (uint32_t)c * 1024u, 0));
                wr[0][t][0][2 * h] = v[0]; wr[0][t][0][2 * h + 1] = v[1];
            }
        }
    };
    auto load_meta = [&](int d, int c) __attribute__((always_inline)) {
        if (GROUPED) {
#pragma unroll
            for (int t = 0; t < TPW; ++t) mr[d][t][0] = __builtin_amdgcn_raw_buffer_load_b32(rm[t], jj4, (uint32_t)c * (uint32_t)p.N_pad * 4u, 0);
        }
    };
    auto load_w = [&](int d, int c) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
#pragma unroll
            for (int lp = 0; lp < LPC; ++lp) wr[d][t][lp] = bload128<0>(rw[t], lane16, (uint32_t)(c * LPC + lp) * 1024u);
            if (GROUPED) {
#pragma unroll
                for (int gi = 0; gi < NSUB; ++gi)
                    mr[d][t][gi] = __builtin_amdgcn_raw_buffer_load_b32(rm[t], jj4, (uint32_t)(c * NSUB + gi) * (uint32_t)p.N_pad * 4u, 0);
            }
        }
    };
    uint32_t mch[TPW];
    if (!GROUPED && WBITS != 16) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) mch[t] = __builtin_amdgcn_raw_buffer_load_b32(rm[t], jj4, 0, 0);
    }

    f32x4 acc[TPW][MB];
#pragma unroll
    for (int t = 0; t < TPW; ++t)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[t][mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const W4Consts w4c = w4_consts();
    const f16x2 c960 = {(f16)960.f, (f16)960.f};

    load_x(WHOLE ? min(ks, KC - 1) : ks, 0);
    if constexpr (HALVES) {
        load_half(0, 0); load_half(1, 0); load_meta(0, 0);
    } else {
        load_w(0, ks);
        load_w(1, ks + KS);
    }

    auto dq = [&](int d, int t, int s) __attribute__((always_inline)) -> u32x4 {
        if constexpr (WBITS == 16) return wr[d][t][s];
        const uint32_t m = GROUPED ? mr[d][t][s / SPG] : mch[t];
        f16x2 zn, sc;
        if constexpr (HALVES) {      // halves that the packed operations pick themselves: eight registers less
            zn = (f16x2){as_h2(m)[0], as_h2(m)[0]}; sc = (f16x2){as_h2(m)[1], as_h2(m)[1]};
        } else {
            zn = as_h2(__builtin_amdgcn_perm(m, m, 0x05040504u)); sc = as_h2(__builtin_amdgcn_perm(m, m, 0x07060706u));
        }
        if constexpr (BF) {          // small integers: exact in fp16, in fp32 and in bf16 (the high half of the fp32)
            f16x8 v;
            if constexpr (WBITS == 4) {
                const f16x2 one = {(f16)1.f, (f16)1.f};
                v = dequant_w4_vc(wr[d][t][0][s], zn, zn + c960, one, w4c);
            } else {
                const u32x4 w = wr[d][t][(s >> 1) % LPC];
                v = dequant_w8<false>(w[(s & 1) * 2], w[(s & 1) * 2 + 1], zn, sc);
            }
            u32x4 r;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                r[i] = __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, (float)v[2 * i + 1]), __builtin_bit_cast(uint32_t, (float)v[2 * i]), 0x07060302u);
            return r;
        } else {
            const int r = HALVES ? 0 : d;
            if constexpr (WBITS == 4) return __builtin_bit_cast(u32x4, dequant_w4_vc(wr[r][t][0][s], zn, zn + c960, sc, w4c));
            const u32x4 w = wr[r][t][(s >> 1) % LPC];   // per-channel int8: exact (u - z) operand, the column scale is applied in fp32 in the epilogue
            return __builtin_bit_cast(u32x4, dequant_w8<GROUPED>(w[(s & 1) * 2], w[(s & 1) * 2 + 1], zn, sc));
        }
    };
    uint32_t fo[4];                                           // HALVES: this lane's first fragment of each k-step in the buffer at work
#pragma unroll
    for (int s = 0; s < 4; ++s) fo[s] = lds0 + (jj * 16 + ((s * 4 + q) ^ jj)) * 16;
    auto frag = [&](int buf, int s, int mb) __attribute__((always_inline)) {
        if constexpr (HALVES) return *(const __attribute__((address_space(3))) u32x4*)(fo[s] + mb * 4096);
        else return xs[ks][buf][mb * 256 + jj * 16 + ((s * 4 + q) ^ jj)];
    };
    u32x4 an[TPW];                                            // operands of the next k-step (a chunk starts with those the one before left)
    auto next = [&](int d, int s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) an[t] = dq(d, t, s);
    };
    auto compute = [&](int c, int d, int buf) __attribute__((always_inline)) {
        if constexpr (CSCALE) {              // a group's sums on accumulators of their own, scaled as they join the tile's
#pragma unroll
            for (int gi = 0; gi < NSUB; ++gi) {
                f32x4 ag[TPW][MB];
#pragma unroll
                for (int ss = 0; ss < SPG; ++ss) {
                    u32x4 a[TPW];
#pragma unroll
                    for (int t = 0; t < TPW; ++t) a[t] = dq(d, t, gi * SPG + ss);
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        const u32x4 b = frag(buf, gi * SPG + ss, mb);
#pragma unroll
                        for (int t = 0; t < TPW; ++t) ag[t][mb] = mfma_act<BF>(a[t], b, ss ? ag[t][mb] : (f32x4){0.f, 0.f, 0.f, 0.f});
                    }
                }
#pragma unroll
                for (int t = 0; t < TPW; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {   // this lane's rows of the sums are columns 4 q + r: their scales sit in lanes 4 q + r
                        const float sc = (float)as_h2((uint32_t)__builtin_amdgcn_ds_bpermute((q * 4 + r) * 4, (int)mr[d][t][gi]))[1];
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb) acc[t][mb][r] = __builtin_fmaf(sc, ag[t][mb][r], acc[t][mb][r]);
                    }
            }
        } else {
            // Fragment i + AHEAD is read while fragment i is multiplied, the next k-step's operands are formed between the products: left to itself the compiler
            // reads two fragments, waits for them and multiplies (one LDS latency per 8 products and wave)
            constexpr int AHEAD = WBITS == 8 && TPW == 4 && !HALVES ? 1 : 3, N = 4 * MB;
            u32x4 b[AHEAD + 1];
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) b[i] = frag(buf, i / MB, i % MB);
            if (WHOLE) __builtin_amdgcn_sched_barrier(0);
            else       __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                u32x4 a[TPW];
#pragma unroll
                for (int t = 0; t < TPW; ++t) a[t] = an[t];
                next(s == 3 ? d ^ 1 : d, (s + 1) & 3);
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) {
                    const int i = s * MB + mb;
                    if (i + AHEAD < N) b[(i + AHEAD) % (AHEAD + 1)] = frag(buf, (i + AHEAD) / MB, (i + AHEAD) % MB);
#pragma unroll
                    for (int t = 0; t < TPW; ++t) acc[t][mb] = mfma_act<BF>(a[t], b[i % (AHEAD + 1)], acc[t][mb]);
                }
                if constexpr (HALVES) {
                    pace<WBITS, TPW, MB, AHEAD>(s * MB, MB);
                    __builtin_amdgcn_sched_barrier(0);
                    if (s == 0) { load_half(0, c + 1); load_meta(d ^ 1, c + 1); }
                    if (s == 2) load_half(1, c + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (!HALVES) pace<WBITS, TPW, MB, AHEAD>(0, N);
        }
    };

    // Chunk c lies in buffer and ring d.  One barrier: behind it every wave's part of chunk c is in LDS and chunk c - KS is done with, so that the DMA of chunk c + KS may
    // go over it.  At most the weights of chunk c + KS are younger than the DMA of chunk c; in front of a last chunk nothing is (its loads of weights past the end are
    // unused, and the compiler leaves them out).
    const std::true_type more{};                     // WHOLE: a chunk follows, or is loaded all the same
    const std::false_type last{};
    auto chunk = [&](int c, int d, int buf, auto follows) __attribute__((always_inline)) {
        if (WHOLE && !decltype(follows)::value) wait_vm<0>();
        else wait_vm<WLD>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (WHOLE) {
            if (decltype(follows)::value) load_x(min(c + KS, KC - 1), buf ^ 1);
        } else if (c + KS < KC) load_x(c + KS, buf ^ 1);
        if ((WHOLE && KS == 1) || c < KC) compute(c, d, buf);    // slices past the end have nothing left
        if (!HALVES) load_w(d, c + 2 * KS);
        if (WHOLE) __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (!CSCALE) next(0, 0);
    if constexpr (HALVES) {
        for (int c = 0; c < KC; ++c) {
            chunk(c, 0, c & 1, more);
#pragma unroll
            for (int t = 0; t < TPW; ++t) mr[0][t][0] = mr[1][t][0];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                fo[s] += c & 1 ? -XSLOTS * 16 : XSLOTS * 16;
                asm volatile("" : "+v"(fo[s]));
            }
        }
        wait_vm<0>();
    } else if constexpr (WHOLE) {
        int c = ks, left = (KC + KS - 1) / KS;       // the same number of rounds for every slice
        for (; left > (KS > 1 ? 2 : 1); left -= 2, c += 2 * KS) {
            chunk(c, 0, 0, more);
            chunk(c + KS, 1, 1, more);
        }
        if (KS > 1 && left == 2) {
            chunk(c, 0, 0, more);
            chunk(c + KS, 1, 1, last);
        } else if (left) chunk(c, 0, 0, last);
        wait_vm<0>();
    } else {
        for (int c = ks; c - ks < KC; c += 2 * KS) { // the same number of rounds for every slice
            chunk(c, 0, 0, last);
            if (c - ks + KS < KC) chunk(c + KS, 1, 1, last);
        }
    }
    if constexpr (KS > 1) __syncthreads();

    if constexpr (KS > 1) {                          // the slices' sums, in slice order
        f32x4* red = (f32x4*)&xs[0][0][0];
        const int wn = wave % NWN;
        if (ks > 0) {
#pragma unroll
            for (int t = 0; t < TPW; ++t)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) red[((((ks - 1) * NWN + wn) * TPW + t) * MB + mb) * 64 + lane] = acc[t][mb];
        }
        __syncthreads();
        if (ks > 0) return;
#pragma unroll
        for (int k = 1; k < KS; ++k)
#pragma unroll
            for (int t = 0; t < TPW; ++t)
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[t][mb] += red[((((k - 1) * NWN + wn) * TPW + t) * MB + mb) * 64 + lane];
    }

    f32x4 scales[TPW];                               // of 8 bits a column
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        scales[t] = (f32x4){1.f, 1.f, 1.f, 1.f};
        if (!GROUPED && WBITS != 16) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t m = __builtin_amdgcn_raw_buffer_load_b32(rm[t], (uint32_t)(q * 4 + r) * 4u, 0, 0);
                scales[t][r] = (float)as_h2(m)[1];
            }
        }
    }
    if constexpr (KS == 1 && TPW >= 2 && !(TPW == 4 && GS == 1)) {           // 128 x 512 in groups of 32 has no registers left for it
        if (lean_store(p)) {                         // the x buffers hold nothing any more: no DMA is left, and behind the barrier no reader
            __syncthreads();
            char* mine = (char*)&xs[0][0][0] + wave * (MB * 1024);
            if (p.mode == MODE_SILU) store_rows<BF, MB, TPW, true>(p, acc, scales, mine, m0, nt_base * 16, lane);
            else                     store_rows<BF, MB, TPW, false>(p, acc, scales, mine, m0, nt_base * 16, lane);
            return;
        }
    }

    // ---- epilogue: lane holds, for row m0 + mb*16 + jj, the 4 consecutive columns 16 nt + 4q + r
#pragma unroll
    for (int t = 0; t < TPW; ++t) {
        if (!tile_ok[t]) continue;
        const int n0 = (nt_base + t) * 16 + q * 4;
        const f32x4 sc = scales[t];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int m = m0 + mb * 16 + jj;
            if (m >= p.M) continue;
            if constexpr (BF) store_bf16(p, acc[t][mb] * sc, m, n0);
            else              gemm_store(p, acc[t][mb] * sc, m, n0, 0);
        }
    }
}

template <int WBITS, int GS, bool BF, int MB, int TPW, int KS, bool WHOLE>
__global__ __launch_bounds__(512, prefill_waves(WBITS, GS, BF, MB, TPW, KS, WHOLE)) void gemm_prefill_kernel(const GemmParams p, const int band) {
    __shared__ u32x4 xs[KS * 512 * MB];
    int bx = blockIdx.x, by = blockIdx.y;
    if (band) prefill_tile(by * (int)gridDim.x + bx, gridDim.y, gridDim.x, band, bx, by);
    prefill_block<WBITS, GS, BF, MB, TPW, KS, WHOLE>(p, xs, by * 16 * MB, bx * (8 / KS * TPW));
}
// Two shapes in one launch (pick_rest): blocks of 16 MB rows for the first `cols` column tiles, whole rounds of them over the chip, and smaller ones for the columns behind.  Blocks start in order, so
// the small ones run where the large ones are done first.  In a launch of their own they waited for the last of them: fp16 W4 at 4096 rows, us one shape / two launches / one, the same bits:
// 37888 x 3584 gated 902 / 885 / 868, 4608 x 3584 138 / 126 / 114.
template <int WBITS, int GS, bool BF, int MB, int TPW, int MB2, int TPW2>
__global__ __launch_bounds__(512, prefill_waves(WBITS, GS, BF, MB, TPW, 1, true)) void gemm_prefill_rest_kernel(const GemmParams p, const int cols, const int band, const int band2) {
    static_assert(MB2 <= MB && TPW2 <= TPW, "the rest's blocks are smaller");
    __shared__ u32x4 xs[512 * MB];
    const int rows = (p.M + 16 * MB - 1) / (16 * MB), n = rows * cols, id = blockIdx.x;
    int bx, by;
    if (id < n) {
        bx = id % cols; by = id / cols;
        if (band) prefill_tile(id, rows, cols, band, bx, by);
        prefill_block<WBITS, GS, BF, MB, TPW, 1, true>(p, xs, by * 16 * MB, bx * 8 * TPW);
    } else {
        const int rows2 = (p.M + 16 * MB2 - 1) / (16 * MB2), cols2 = (p.NT - cols * 8 * TPW + 8 * TPW2 - 1) / (8 * TPW2);
        bx = (id - n) % cols2; by = (id - n) / cols2;
        if (band2) prefill_tile(id - n, rows2, cols2, band2, bx, by);
        prefill_block<WBITS, GS, BF, MB2, TPW2, 1, true>(p, xs, by * 16 * MB2, (cols * TPW + bx * TPW2) * 8);
    }
}

// Block shapes: {row blocks, weight tiles per wave, K slices}.
struct PrefillShape { int mb, tpw, ks; };
constexpr PrefillShape kPrefillShapes[] = {{8, 4, 1}, {8, 2, 1}, {4, 2, 1}, {4, 1, 1}, {4, 1, 2}, {2, 1, 2}, {2, 1, 4}};
constexpr int kPrefillShapeCount = sizeof(kPrefillShapes) / sizeof(kPrefillShapes[0]);

// The shape of a call: a time model in us.  A round of a block (KS chunks of 128 k) takes `lat` alone on its CU -- loads, LDS, barrier -- and `sat` of a CU whose
// share of the grid keeps it busy; the share counts half as the exact quotient and half as the whole blocks of the fullest CU.  Fitted (random operands, one MI355X) per
// operand class over M = 70..4096 at the Qwen2-0.5B and 7B projections to the loop with branches and tiles in rows, whose pick was within 8 % of the fastest shape; it now decides whether K is
// sliced and by how many, and what other paths are compared with (kUnslicedCost has the present loops).  Examples of that loop, us at 128x512 / 128x256 / 64x256 /
// 64x128 / 64x64 / 32x64 / 32x32 tiles: fp16 W4 37888 x 3584 at M = 4096 1002 / 1057 / 1144 / 1244 / 1503 / 1806 / 2516, bf16 W4 3584 x 18944 at M = 128 - / 309 / 223 / 144 / 81 /
// 64 / 50; W16 9728 x 896 at M = 512 - / 22 / 23 / 18 / 18 / 23 / 33; bf16 W4 37888 x 3584 at M = 512 - / 192 / 180 / 188 / 222 / 263 / 363.
struct PrefillCost { double lat, sat; };
constexpr PrefillCost kPrefillCost[3][kPrefillShapeCount] = {
    {{2.82, 3.58}, {1.59, 2.02}, {1.12, 1.14}, {0.69, 0.613}, {0.75, 0.708}, {0.53, 0.439}, {0.61, 0.585}},     // codes on the operand side
    {{1e9, 1e9},   {2.16, 2.45}, {1.52, 1.32}, {0.94, 0.708}, {0.98, 0.856}, {0.72, 0.507}, {0.69, 0.708}},      // bf16 under group scales: two sets of accumulators
    {{1e9, 1e9},   {1.41, 2.82}, {0.92, 1.84}, {0.49, 0.856}, {0.49, 0.779}, {0.45, 0.532}, {0.37, 0.742}},     // 16-bit weights
};
// Does shape I run the loop without branches (WHOLE) where x allows it?  gs: 4, 2, 1 for groups of 128, 64, 32.  Not 128 x 512 under groups of 32 or 64 (two or four scales a chunk and tile have
// no registers left), 64 x 256 in groups of 32 and the 64-row forms of bf16 W4 (held in one piece the compiler takes more than 128 or 80 registers for them and a block less fits a CU:
// 37888 x 3584 at 4096 rows 1293 -> 1485 us), bf16 W4 in groups of 32 (198 random calls 1.04 of the general loop's time), nor 4-bit weights under sliced K (8 or 16 products and 56 operand
// instructions a wave and chunk: 2 % either way, 3584 x 18944 at 104 rows 59 -> 60 to 62 us).  The others take 0.85 to 1.00 of it, mean over about 200 calls each.
constexpr bool prefill_straight(int I, int wbits, int gs, bool bf) {
    if (wbits != 4) return true;
    if (kPrefillShapes[I].ks > 1 || (bf && (kPrefillShapes[I].mb == 4 || gs == 1))) return false;
    return I == 0 ? gs == 4 : I == 2 ? gs != 1 : true;
}
// The same for the shapes that do not slice K, fitted to the present loops, per operand class: where K or x leaves every shape the general loop (first row) and where each has the loop it can
// have (second).  `base` us a launch beside its chunks: 12 for a block of 128 x 512, 5 for 64 x 128; one round of blocks takes `lat` a chunk, however few they are.  These shapes choose among each
// other only: whether K is sliced stays with the table above, so that a call's sums keep their order.  Fitted to times and picks of 81 to 139 random calls of M = 65..4096 a row, weights from
// memory: the pick takes 1.0003 to 1.0035 of the fastest shape's time on average; 412 other calls 1.004, at worst 1.13.  With 2.5 us for every shape and one row for both loops and all groups it
// took 1.004 to 1.033, at worst 1.31 (16-bit weights, 37888 x 3584 at 1825 rows 590 us where 128 x 256 takes 462).
constexpr int kWholeShapes = 4;
struct UnslicedCost { double base, lat, sat; };
constexpr UnslicedCost kUnslicedCost[9][2][kWholeShapes] = {
    {{{15.0, 2.40, 3.401}, {7.7, 1.60, 1.940}, {5.9, 1.09, 1.054}, {5.6, 0.50, 0.568}},
     {{12.4, 2.20, 3.414}, {8.7, 1.30, 1.830}, {5.6, 1.02, 1.022}, {5.1, 0.49, 0.559}}},     // fp16 W4, groups of 128
    {{{15.3, 2.59, 3.572}, {10.7, 1.43, 1.992}, {6.8, 1.08, 1.091}, {6.1, 0.49, 0.588}},
     {{13.3, 2.65, 3.565}, {9.3, 1.24, 1.924}, {6.2, 0.97, 1.038}, {5.6, 0.42, 0.570}}},     // of 64
    {{{12.4, 2.63, 3.678}, {8.2, 1.56, 2.079}, {6.3, 1.17, 1.132}, {5.3, 0.77, 0.623}},
     {{12.7, 2.61, 3.630}, {8.5, 1.29, 2.047}, {8.0, 1.03, 1.108}, {4.6, 0.62, 0.602}}},     // of 32
    {{{0, 1e9, 1e9}, {7.4, 2.00, 2.525}, {6.1, 1.48, 1.296}, {6.4, 0.30, 0.695}},
     {{0, 1e9, 1e9}, {8.1, 1.65, 2.237}, {7.2, 1.45, 1.285}, {5.7, 0.34, 0.703}}},     // bf16 W4, groups of 128
    {{{0, 1e9, 1e9}, {7.9, 2.30, 2.799}, {6.8, 1.72, 1.509}, {5.2, 1.05, 0.792}},
     {{0, 1e9, 1e9}, {9.2, 2.17, 2.636}, {6.1, 1.78, 1.526}, {5.7, 1.57, 0.776}}},     // of 64
    {{{0, 1e9, 1e9}, {7.9, 2.89, 3.573}, {5.7, 2.09, 2.402}, {7.1, 0.34, 0.981}},
     {{0, 1e9, 1e9}, {7.6, 2.90, 3.575}, {5.5, 2.08, 2.410}, {7.0, 0.57, 0.980}}},     // of 32
    {{{11.3, 2.70, 3.396}, {7.1, 1.55, 1.897}, {6.1, 1.01, 0.978}, {5.5, 0.62, 0.524}},
     {{11.7, 2.35, 2.964}, {7.0, 1.33, 1.697}, {6.5, 0.91, 0.869}, {5.0, 0.57, 0.520}}},     // fp16 8 bits
    {{{0, 1e9, 1e9}, {7.7, 1.75, 2.238}, {6.6, 1.23, 1.192}, {5.7, 0.79, 0.634}},
     {{0, 1e9, 1e9}, {8.0, 1.48, 2.055}, {6.3, 1.16, 1.152}, {5.7, 0.49, 0.611}}},     // bf16 8 bits
    {{{0, 1e9, 1e9}, {7.2, 1.54, 2.097}, {6.0, 1.17, 1.163}, {6.0, 0.45, 0.649}},
     {{0, 1e9, 1e9}, {6.8, 1.39, 1.920}, {6.5, 0.79, 1.164}, {4.8, 0.47, 0.685}}},     // 16-bit weights
};
// the share of a busy CU that a launch gives the fullest one, and how many rounds of blocks that is at least
struct PrefillShare { double share; bool round; };
PrefillShare prefill_share(const PrefillShape& s, int M, int NT) {
    const double full = (double)cdiv(NT, 8 / s.ks * s.tpw) * cdiv(M, 16 * s.mb) / 256.0, whole = (double)(long)(full + 0.9999);
    return {0.5 * (full + whole), whole <= 1.0};
}
const UnslicedCost* unsliced_cost(bool bf, int wbits, int group_size, bool whole) {
    return kUnslicedCost[wbits == 16 ? 8 : wbits == 8 ? (bf ? 7 : 6) : (bf ? 3 : 0) + (group_size == 128 ? 0 : group_size == 64 ? 1 : 2)][whole];
}
double unsliced_us(const UnslicedCost* own, int i, int M, int NT, int KC) {
    const PrefillShare sh = prefill_share(kPrefillShapes[i], M, NT);
    const double share = sh.round ? 0.0 : own[i].sat * sh.share;
    return own[i].base + KC * (share > own[i].lat ? share : own[i].lat);
}
int pick_shape(int M, int NT, int KC, bool bf, int wbits, int group_size, bool whole, double* t_best) {
    const int first = (bf || wbits == 16) ? 1 : 0;
    const PrefillCost* cost = kPrefillCost[wbits == 16 ? 2 : (bf && wbits == 4) ? 1 : 0];
    int best = 1;
    *t_best = 1e30;
    for (int i = first; i < kPrefillShapeCount; ++i) {
        const double share = cost[i].sat * prefill_share(kPrefillShapes[i], M, NT).share;
        const double t = cdiv(KC, kPrefillShapes[i].ks) * (share > cost[i].lat ? share : cost[i].lat) + 2.5;
        if (t < *t_best) { *t_best = t; best = i; }
    }
    if (best >= kWholeShapes) return best;
    const UnslicedCost* own = unsliced_cost(bf, wbits, group_size, whole);
    double least = 1e30;
    for (int i = first; i < kWholeShapes; ++i) {
        const double t = unsliced_us(own, i, M, NT, KC);
        if (t < least) { least = t; best = i; }
    }
    return best;
}
// Two shapes in one launch: a last round of blocks that is nearly empty costs most of a full one (37888 x 3584 at 4096 rows has 9.25 rounds of 128 x 512).  The first shape takes the columns that fill
// whole rounds, a smaller one, a block to a CU like it, the rest, where the model expects 2.5 % of it.  Of codes (4 bits: groups of 128), where K is not sliced and runs the loop without branches.
// 660 random calls (130 to 135 a class) that could: mean share of the time with one shape, over all of them, fp16 W4 0.971 (best choice of each 0.956), fp16 8 bits 0.972 (0.962), bf16 W4 0.982 (0.974), bf16 8
// bits 0.973 (0.967); 11 above 1.02, at worst 1.05.  16-bit weights 0.996, at worst 1.17: one shape.  us one shape / two: fp16 W4 37888 x 3584 gated at 4096 rows 902 / 868 (128 x 512 and 64 x 256),
// 2667 625 / 577 (and 64 x 128), 1825 442 / 415 (and 128 x 256), 4608 x 3584 at 4096 138 / 114; fp16 8 bits the same at 4096 845 / 822 and 123 / 105; bf16 W4 4608 x 3584 at 4096 161 / 137
// (128 x 256 and 64 x 128), 37888 x 3584 at 1055 331 / 306.
// Under bf16 W4 the rest's 64 x 128 blocks run the loop without branches, which a call of that shape alone does not (prefill_straight), while the table's row for it is the general loop's.  It decides as
// well as one of their own: 152 random calls that could take two, of 400 to 9000 rows, 0.977 of the time with one shape (best choice of each 0.971; 41 take two, none of them slower), with the row
// fitted to their times (0.48 and 0.74) 0.979.
struct PrefillRest { int shape, rest, cols; };               // cols 0: one shape
PrefillRest pick_rest(int best, int M, int NT, int KC, bool bf, int wbits, int group_size, bool whole) {
    PrefillRest pick{best, 0, 0};
    if (!whole || best >= kWholeShapes || wbits == 16 || (wbits == 4 && group_size != 128)) return pick;
    const UnslicedCost* own = unsliced_cost(bf, wbits, group_size, true);
    double least = 0.975 * unsliced_us(own, best, M, NT, KC);
    for (int i = bf ? 1 : 0; i < 2; ++i) {
        const int rows = cdiv(M, 128), tiles = 8 * kPrefillShapes[i].tpw, rounds = rows * cdiv(NT, tiles) / 256, cols = rounds * 256 / rows;
        if (cols == 0 || cols * tiles >= NT) continue;
        for (int r = i == 0 ? 1 : 3; r < kWholeShapes; ++r) {
            const int blocks = cdiv(M, 16 * kPrefillShapes[r].mb) * cdiv(NT - cols * tiles, 8 * kPrefillShapes[r].tpw);
            // a full round takes what the chip's throughput asks for, the last as much less as it is empty, at least 0.8 of a block alone
            const int n = cdiv(blocks, 256);
            const double full = own[r].lat > own[r].sat ? own[r].lat : own[r].sat, alone = 0.8 * own[r].lat;
            const double t = own[i].base + KC * own[i].sat * rows * cols / 256.0 + n + KC * ((n - 1) * full + alone + (full - alone) * (blocks / 256.0 - (n - 1)));
            if (t < least) { least = t; pick = {i, r, cols}; }
        }
    }
    return pick;
}
// K below 2^23: the 128 x 512 form's row offsets are formed past the last row, in 32 bits.
bool prefill_whole(const void* x, int K) { return (uintptr_t)x % 16 == 0 && K % 128 == 0 && K < 1 << 23; }

template <int WBITS, int GS, bool BF, int I>
void launch_shape_t(const GemmParams& p, hipStream_t st) {
    constexpr PrefillShape s = kPrefillShapes[I];
    const dim3 grid(cdiv(p.NT, 8 / s.ks * s.tpw), cdiv(p.M, 16 * s.mb));
    const int band = prefill_short(p, WBITS, 8 / s.ks * s.tpw * 16) ? 0 : prefill_band(grid.y, grid.x);
    if constexpr (prefill_straight(I, WBITS, GS, BF)) {
        if (prefill_whole(p.x, p.K)) {
            hipLaunchKernelGGL((gemm_prefill_kernel<WBITS, GS, BF, s.mb, s.tpw, s.ks, true>), grid, dim3(512), 0, st, p, band);
            return;
        }
    }
    hipLaunchKernelGGL((gemm_prefill_kernel<WBITS, GS, BF, s.mb, s.tpw, s.ks, false>), grid, dim3(512), 0, st, p, band);
}
template <int WBITS, int GS, bool BF, int I, int J>
void launch_rest_t(int cols, const GemmParams& p, hipStream_t st) {
    constexpr PrefillShape s = kPrefillShapes[I], r = kPrefillShapes[J];
    const int rows = cdiv(p.M, 16 * s.mb), rows2 = cdiv(p.M, 16 * r.mb), cols2 = cdiv(p.NT - cols * 8 * s.tpw, 8 * r.tpw);
    hipLaunchKernelGGL((gemm_prefill_rest_kernel<WBITS, GS, BF, s.mb, s.tpw, r.mb, r.tpw>), dim3(rows * cols + rows2 * cols2), dim3(512), 0, st, p, cols,
                       prefill_short(p, WBITS, s.tpw * 128) ? 0 : prefill_band(rows, cols), prefill_short(p, WBITS, r.tpw * 128) ? 0 : prefill_band(rows2, cols2));
}
template <int WBITS, int GS, bool BF>
int launch_shape(const PrefillRest& pick, const GemmParams& p, hipStream_t st) {
    if constexpr (WBITS == 8 || (WBITS == 4 && GS == 4)) {
        if (pick.cols) {
            switch (pick.shape * 4 + pick.rest) {
                case 1: if constexpr (!BF) { launch_rest_t<WBITS, GS, BF, 0, 1>(pick.cols, p, st); break; } return MI355_ERR_UNSUPPORTED;
                case 2: if constexpr (!BF) { launch_rest_t<WBITS, GS, BF, 0, 2>(pick.cols, p, st); break; } return MI355_ERR_UNSUPPORTED;
                case 3: if constexpr (!BF) { launch_rest_t<WBITS, GS, BF, 0, 3>(pick.cols, p, st); break; } return MI355_ERR_UNSUPPORTED;
                case 7: launch_rest_t<WBITS, GS, BF, 1, 3>(pick.cols, p, st); break;
                default: return MI355_ERR_UNSUPPORTED;
            }
            MI355_CHECK_LAUNCH("gemm_prefill_rest_kernel");
            return MI355_OK;
        }
    }
    switch (pick.shape) {
        case 0: if constexpr (!BF && WBITS != 16) { launch_shape_t<WBITS, GS, BF, 0>(p, st); break; } return MI355_ERR_UNSUPPORTED;
        case 1: launch_shape_t<WBITS, GS, BF, 1>(p, st); break;
        case 2: launch_shape_t<WBITS, GS, BF, 2>(p, st); break;
        case 3: launch_shape_t<WBITS, GS, BF, 3>(p, st); break;
        case 4: launch_shape_t<WBITS, GS, BF, 4>(p, st); break;
        case 5: launch_shape_t<WBITS, GS, BF, 5>(p, st); break;
        case 6: launch_shape_t<WBITS, GS, BF, 6>(p, st); break;
        default: return MI355_ERR_UNSUPPORTED;
    }
    MI355_CHECK_LAUNCH("gemm_prefill_kernel");
    return MI355_OK;
}

} // namespace

// The tile that block id of a rows x cols grid of tiles takes where bands are worth it: column tile in the low half, row tile in the high half (for the tests: every tile once).
extern "C" int64_t mi355_gemm_prefill_tile(int32_t id, int32_t rows, int32_t cols) {
    int bx = id % cols, by = id / cols;
    if (const int band = prefill_band(rows, cols)) prefill_tile(id, rows, cols, band, bx, by);
    return (int64_t)by << 32 | bx;
}

// The block shape of a call that runs one (mi355_gemm_prefill_rest 0; else the one that the two were compared with), by its place in kPrefillShapes: NT = N_pad / 16, KC = K_pad / 128.  4-bit weights in groups of 128, x on 16 bytes, K a multiple of 128.
extern "C" int mi355_gemm_prefill_shape(int32_t M, int32_t NT, int32_t KC, int32_t bf16, int32_t wbits) {
    return mi355_gemm_prefill_form(M, NT, KC, bf16, wbits, 128, 1) & 15;
}
// The same for any call (whole: x on 16 bytes and K a multiple of 128), plus 16 where it runs the loop without branches.
extern "C" int mi355_gemm_prefill_form(int32_t M, int32_t NT, int32_t KC, int32_t bf16, int32_t wbits, int32_t group_size, int32_t whole) {
    double t;
    const int s = pick_shape(M, NT, KC, bf16 != 0, wbits, group_size, whole != 0, &t);
    return s + (whole && prefill_straight(s, wbits, group_size / 32, bf16 != 0) ? 16 : 0);
}

// Whether such a call runs two shapes in one launch: 0, or the first shape's place + 4 times the rest's + 16 times the first's column tiles.
extern "C" int mi355_gemm_prefill_rest(int32_t M, int32_t NT, int32_t KC, int32_t bf16, int32_t wbits, int32_t group_size, int32_t whole) {
    double t;
    const int s = pick_shape(M, NT, KC, bf16 != 0, wbits, group_size, whole != 0, &t);
    const PrefillRest r = pick_rest(s, M, NT, KC, bf16 != 0, wbits, group_size, whole != 0);
    return r.cols ? r.shape + 4 * r.rest + 16 * r.cols : 0;
}

// Direct-mode launch (fused epilogue in p.mode).  MI355_ERR_UNSUPPORTED: shape / format not covered, caller falls back.
// t_limit: the caller's estimate (us) for its other path; a launch expected to take longer is not made (MI355_ERR_UNSUPPORTED).
extern "C" int mi355_gemm_prefill(const void* gp, int wbits, int group_size, double t_limit, mi355_stream_t stream) {
    const GemmParams& g = *reinterpret_cast<const GemmParams*>(gp);
    if (g.M <= 64 || g.mode == MODE_PARTIAL || g.mode == MODE_F32) return MI355_ERR_UNSUPPORTED;
    if ((uint64_t)g.M * g.K * 2 >= 0x7FFFFFF0ull) return MI355_ERR_UNSUPPORTED;       // x image must stay below the OOB offset
    hipStream_t st = (hipStream_t)stream;
    const bool bf = g.bf16 != 0;
    double t;
    const bool whole = prefill_whole(g.x, g.K);
    const int one = pick_shape(g.M, g.NT, g.KC, bf, wbits, group_size, whole, &t);
    if (t > t_limit) return MI355_ERR_UNSUPPORTED;
    const PrefillRest s = pick_rest(one, g.M, g.NT, g.KC, bf, wbits, group_size, whole);
    if (wbits == 16) return bf ? launch_shape<16, 0, true>(s, g, st) : launch_shape<16, 0, false>(s, g, st);
    if (wbits == 8 && group_size == 0) return bf ? launch_shape<8, 0, true>(s, g, st) : launch_shape<8, 0, false>(s, g, st);
    if (wbits == 4) {
        if (group_size == 128) return bf ? launch_shape<4, 4, true>(s, g, st) : launch_shape<4, 4, false>(s, g, st);
        if (group_size == 64) return bf ? launch_shape<4, 2, true>(s, g, st) : launch_shape<4, 2, false>(s, g, st);
        if (group_size == 32) return bf ? launch_shape<4, 1, true>(s, g, st) : launch_shape<4, 1, false>(s, g, st);
    }
    return MI355_ERR_UNSUPPORTED;
}
