// What a decode step's linear recurrence is made of, for the two places that run it: a launch of its own (hybrid_ops.hip) and the blocks beside a linear of the same step (gemm_dense.hip).
#pragma once
#include "common.h"
#include "../../include/mi355_hybrid.h"

namespace {

template <typename T> __device__ __forceinline__ void hy_load8(const T* p, float (&o)[8]);
template <> __device__ __forceinline__ void hy_load8<bf16>(const bf16* p, float (&o)[8]) { act_unpack8<true>(*(const u32x4*)p, o); }
template <> __device__ __forceinline__ void hy_load8<float>(const float* p, float (&o)[8]) {
    const f32x4 a = *(const f32x4*)p, b = *(const f32x4*)(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { o[i] = a[i]; o[4 + i] = b[i]; }
}

__device__ __forceinline__ float hy_wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ float hy_sigmoid(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float hy_silu(float z) { return z / (1.f + expf(-z)); }

enum { SCAN_HGRN2 = 0, SCAN_GLA = 1, SCAN_FIXED = 2, SCAN_FIXED_SILU = 3 };

struct RecurStep {
    const float* proj; int ld, qo, ko, vo, go, ao, rank;
    const void* w2; const void* b2;
    const float* z; int ldz;
    const void* lower; const void* fbias;
    float tau, qscale;
    int mode, H, dim, vdim;
    const int32_t* row_start; const int32_t* slot; const int32_t* first_pos;
    float* state;
    const void* w; int w_heads;
    float eps;
    void* out;
};
struct __attribute__((aligned(16))) RecurLds { float part[1024], q[256], k[256], a[256], red[8]; };      // part first: it is read in fours

// Host: what every launch of it asks of its arguments.
inline int hy_recur_check(const RecurStep& p, int nseq) {
    MI355_CHECK_ARG(p.proj && p.row_start && p.slot && p.first_pos && p.state && p.out && nseq > 0 && p.H > 0 && p.dim > 0 && p.vdim > 0, "hy_recur_step: bad argument");
    MI355_CHECK_ARG(p.mode == SCAN_HGRN2 ? (p.lower && p.fbias) : (p.mode == SCAN_FIXED || p.mode == SCAN_FIXED_SILU) ? p.lower != nullptr
                                                          : (p.mode == SCAN_GLA && p.tau > 0.f && (p.ao >= 0 ? (p.w2 && p.rank > 0 && p.rank <= 64) : p.z != nullptr)),
                    "hy_recur_step: mode %d lacks its gate inputs", p.mode);
    if (!mi355_hy_recur_step_fits(p.dim, p.vdim) || (uintptr_t)p.state % 16) {
        mi355_set_error("hy_recur_step: heads of %d x %d", p.dim, p.vdim);
        return MI355_ERR_UNSUPPORTED;
    }
    return MI355_OK;
}
inline int hy_recur_rows(int dim, int vdim) { const int KG = 256 / (vdim / 4); return (dim + KG - 1) / KG; }       // key rows a thread holds

template <typename T, int RPT>
__device__ __forceinline__ void hy_recur_step(const RecurStep& p, int sq, int h, RecurLds& lds) {
    float *q_s = lds.q, *k_s = lds.k, *a_s = lds.a, *red = lds.red, *part = lds.part;
    const int tid = threadIdx.x, CG = p.vdim >> 2, KG = 256 / CG, cg = tid % CG, kg = tid / CG;
    const int r0 = p.row_start[sq], r1 = p.row_start[sq + 1];
    const bool on = kg < KG;
    float* st = p.state + ((size_t)p.slot[sq] * p.H + h) * p.dim * p.vdim + cg * 4;
    f32x4 s[RPT];
    const bool fresh = p.first_pos[sq] == 0;
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
        const int d = kg + j * KG;
        s[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (on && !fresh && d < p.dim) s[j] = *(const f32x4*)(st + (size_t)d * p.vdim);
    }
    const int hd = h * p.dim + min(tid, p.dim - 1), hv = h * p.vdim + min(tid, p.vdim - 1);
    const float norm = p.w ? (float)((const T*)p.w)[p.w_heads ? hv : min(tid, p.vdim - 1)] : 1.f;
    const bool low = p.mode == SCAN_GLA && p.ao >= 0;
    for (int t = r0; t < r1; ++t) {
        // everything the token needs is asked for at once: a later load is another trip to memory in a launch of a few microseconds
        const float* row = p.proj + (size_t)t * p.ld;
        float qv = row[p.qo + hd], kv = row[p.ko + hd], av = 0.f, zz = 0.f, lr = 0.f;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = row[p.vo + h * p.vdim + cg * 4 + e];
        const float gz = p.go >= 0 ? row[p.go + hv] : 0.f;
        if (low) {
            lr = (float)(T)row[p.ao + min(tid & 63, p.rank - 1)];
            zz = p.b2 ? (float)((const T*)p.b2)[hd] : 0.f;
            const T* w2 = (const T*)p.w2 + (size_t)hd * p.rank;
            float dot = 0.f;
            if (p.rank % 8 == 0 && (uintptr_t)p.w2 % 32 == 0)
                for (int j = 0; j < p.rank; j += 8) {
                    float w8[8];
                    hy_load8<T>(w2 + j, w8);
#pragma unroll
                    for (int e = 0; e < 8; ++e) dot = __builtin_fmaf(w8[e], __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lr), j + e)), dot);
                }
            else
                for (int j = 0; j < p.rank; ++j)
                    dot = __builtin_fmaf((float)w2[j], __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lr), j)), dot);
            zz += dot;
        } else if (p.mode == SCAN_GLA) zz = p.z[(size_t)t * p.ldz + hd];
        if (p.mode == SCAN_HGRN2) {
            const float lw = (float)((const T*)p.lower)[hd], f = lw + (1.f - lw) * hy_sigmoid(kv + (float)((const T*)p.fbias)[hd]);
            qv = hy_silu(qv); av = f; kv = 1.f - f;
        } else if (p.mode == SCAN_GLA) {
            qv *= p.qscale;
            av = expf((fminf(zz, 0.f) - log1pf(expf(-fabsf(zz)))) / p.tau);
        } else {
            if (p.mode == SCAN_FIXED_SILU) {
                qv = hy_silu(qv); kv = hy_silu(kv);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = hy_silu(v[e]);
            }
            av = ((const float*)p.lower)[h];
        }
        if (tid < p.dim) { q_s[tid] = qv; k_s[tid] = kv; a_s[tid] = av; }
        __syncthreads();
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        if (on) {
#pragma unroll
            for (int j = 0; j < RPT; ++j) {
                const int d = kg + j * KG;
                if (d >= p.dim) continue;
                const float a = a_s[d], k = k_s[d], q = q_s[d];
#pragma unroll
                for (int e = 0; e < 4; ++e) { s[j][e] = __builtin_fmaf(a, s[j][e], k * v[e]); o[e] = __builtin_fmaf(s[j][e], q, o[e]); }
            }
            *(f32x4*)(part + (kg * CG + cg) * 4) = o;
        }
        __syncthreads();
        float y = 0.f;
        if (tid < p.vdim)
            for (int g = 0; g < KG; ++g) y += part[g * p.vdim + tid];
        const float ss = hy_wave_sum(y * y);
        if ((tid & 63) == 0) red[(t & 1) * 4 + (tid >> 6)] = ss;
        __syncthreads();
        if (tid < p.vdim) {
            const float* rd = red + (t & 1) * 4;
            y *= 1.f / sqrtf(((rd[0] + rd[1]) + (rd[2] + rd[3])) / (float)p.vdim + p.eps);
            if (p.w) y *= norm;
            if (p.go >= 0) y *= hy_silu(gz);
            ((T*)p.out)[((size_t)t * p.H + h) * p.vdim + tid] = (T)y;
        }
    }
    if (r0 < r1) {
#pragma unroll
        for (int j = 0; j < RPT; ++j) {
            const int d = kg + j * KG;
            if (on && d < p.dim) *(f32x4*)(st + (size_t)d * p.vdim) = s[j];
        }
    }
}

} // namespace
