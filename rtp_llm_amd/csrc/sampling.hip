// Sampler kernels on fp32 logit rows, gfx950: the speculative-decoding verify step (row softmax, chain rejection sampling) and
// the non-greedy branch of the sampler (temperature + repetition / presence / frequency penalties, top-k / top-p filter,
// inverse-CDF draw: bindings/core/CudaSampleOp.cc:632-786, common/kernels/sampling_penalty_kernels.cu:26-180).
//
// Replaces rejection_sampling_kernel / invokeRejectionSampling
// (rtp_llm/models_py/bindings/rocm/speculative_sampling/sampling.cu:306-530, called from
// cpp/normal_engine/speculative/SpeculativeSampler.cc:214 and MtpExecutor.cc:1405).  Argument meaning, output
// padding (-1) and the accepted-count convention (accepted drafts + 1) follow the reference; the residual draw is
// "first index whose inclusive prefix sum of relu(q - p) exceeds u * sum" with the prefix taken in index order.
// One 1024-thread block per row: the accept chain is serial in one lane (gamma <= 16 dependent reads), the residual
// draw is two passes over the vocabulary row (sum, then locate), each thread owning a contiguous segment so that the
// block-level prefix over threads is the prefix over indices.
#include <math.h>
#include <string.h>
#include <type_traits>

#include "common.h"

namespace {

constexpr int kThreads = 1024;
constexpr int kMostSplits = 16;              // blocks of a row at most, in the launches that split rows

__device__ __forceinline__ float block_sum(float v, float* s_red) {
    v = wave_sum(v);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) s_red[wave] = v;
    __syncthreads();
    float t = (threadIdx.x < kThreads / 64) ? s_red[threadIdx.x] : 0.f;
    if (wave == 0) {
        t = wave_sum(t);
        if (lane == 0) s_red[0] = t;
    }
    __syncthreads();
    const float r = s_red[0];
    __syncthreads();
    return r;
}

// Inverse-CDF draw from the unnormalised non-negative weights f(0..V-1): the first index j with f(j) > 0 whose inclusive
// prefix sum, taken in index order, exceeds u01 * sum (V - 1 when rounding leaves none: sampling.cu:418).  Thread tx owns
// the contiguous segment [lo, hi) (a multiple of 4 long: segments start on 16-byte boundaries of an aligned row), so the block-level
// prefix over threads is the prefix over indices.  Result in *s_found (valid for every thread after the call); returns sum.
__device__ __forceinline__ int draw_segment(int V) { return (((V + kThreads - 1) / kThreads) + 3) & ~3; }

template <class F>
__device__ __forceinline__ float block_draw(F&& f, int V, float u01, float* s_red, float* s_scan, int* s_found) {
    const int tx = threadIdx.x;
    const int seg = draw_segment(V);
    const int lo = min(V, tx * seg), hi = min(V, lo + seg);
    float local = 0.f;
#pragma unroll 4
    for (int j = lo; j < hi; ++j) local += f(j);
    const float total = block_sum(local, s_red);
    const float u = u01 * total;
    // inclusive prefix over threads (Hillis-Steele in LDS; 1024 entries)
    s_scan[tx] = local;
    if (tx == 0) *s_found = V - 1;
    __syncthreads();
    for (int off = 1; off < kThreads; off <<= 1) {
        const float add = (tx >= off) ? s_scan[tx - off] : 0.f;
        __syncthreads();
        s_scan[tx] += add;
        __syncthreads();
    }
    const float incl = s_scan[tx], excl = incl - local;
    if (local > 0.f && excl <= u && incl > u) {   // the prefix crosses u inside this segment (at most one thread)
        float c = excl;
        int found = -1, last_pos = -1;              // the rescan rounds differently from the scanned prefix: if c never exceeds u here,
        for (int j = lo; j < hi; ++j) {             // fall back to the LAST index of the segment with weight > 0 -- never to a token the
            const float r = f(j);                   // filter / ban / residual removed (weight 0)
            c += r;
            if (r > 0.f) { last_pos = j; if (c > u) { found = j; break; } }
        }
        *s_found = found >= 0 ? found : last_pos;   // local > 0: the segment holds at least one positive weight
    }
    __syncthreads();
    return total;
}

// One pass over a row of V floats by the whole block: g(value) for every element, 16-byte loads with four in flight per thread
// when the row allows (a scalar loop waits a full L2 round trip per element: 60 us per pass over a 152064-wide row instead of 4).
template <class G>
__device__ __forceinline__ void row_pass(const float* __restrict__ q, int V, bool vec, G&& g) {
    const int tx = threadIdx.x;
    int done = 0;
    if (vec) {
        const f32x4* q4 = reinterpret_cast<const f32x4*>(q);
        const int V4 = V >> 2;
#pragma unroll 4
        for (int j = tx; j < V4; j += kThreads) {
            const f32x4 v = q4[j];
            g(v[0]); g(v[1]); g(v[2]); g(v[3]);
        }
        done = V4 << 2;
    }
    for (int j = done + tx; j < V; j += kThreads) g(q[j]);
}

struct RejectParams {
    const float*   draft_probs;
    const int32_t* draft_ids;
    const float*   uniform;
    const float*   target_probs;
    const int32_t* target_ids;
    int            target_stride;
    int32_t*       out_ids;
    int32_t*       out_accepted;
    const uint8_t* do_sample;
    int            B, gamma, V, point_mass;
};

__global__ __launch_bounds__(kThreads) void rejection_sample_kernel(const RejectParams p) {
    const int row = blockIdx.x, tx = threadIdx.x;
    const int G = p.gamma, G1 = p.gamma + 1;
    __shared__ int   s_pos, s_skip;
    __shared__ float s_red[kThreads / 64];
    __shared__ float s_scan[kThreads];
    __shared__ int   s_found;

    if (tx == 0) { // accept chain (sampling.cu:336-379)
        const bool sample = p.do_sample[row] != 0;
        bool fallback = false;
        int pos = G;
        for (int i = 0; i < G; ++i) {
            const int d = p.draft_ids[row * G + i];
            const int t = p.target_ids[(size_t)(row * G1 + i) * p.target_stride + p.target_stride - 1];
            const float q = p.target_probs[(size_t)(row * G1 + i) * p.V + d];
            const float pr = p.point_mass ? 1.0f : p.draft_probs[(size_t)(row * G + i) * p.V + d];
            const float u = p.uniform[row * G1 + i];
            const bool accept = sample ? (u * pr < q) : (t == d);
            if (accept) {
                p.out_ids[row * G1 + i] = d;
            } else {
                pos = i;
                if (!sample) {
                    p.out_ids[row * G1 + i] = t;
                    for (int n = i + 1; n < G1; ++n) p.out_ids[row * G1 + n] = -1;
                    fallback = true;
                }
                break;
            }
        }
        p.out_accepted[row] = pos + 1;
        if (pos == G) p.out_ids[row * G1 + pos] = p.target_ids[(size_t)(row * G1 + pos) * p.target_stride + p.target_stride - 1];
        s_pos = pos;
        s_skip = (fallback || pos == G) ? 1 : 0;
    }
    __syncthreads();
    if (s_skip) return;
    const int pos = s_pos;

    // residual distribution relu(q - p) of position pos; thread tx owns indices [lo, hi)
    const float* q = p.target_probs + (size_t)(row * G1 + pos) * p.V;
    const float* dp = p.point_mass ? nullptr : p.draft_probs + (size_t)(row * G + pos) * p.V;
    const int dtok = p.draft_ids[row * G + pos];
    auto resid = [&](int j) {
        const float pv = dp ? dp[j] : (j == dtok ? 1.0f : 0.0f);
        return fmaxf(q[j] - pv, 0.f);
    };
    block_draw(resid, p.V, p.uniform[row * G1 + min(pos + 1, G)], s_red, s_scan, &s_found);
    if (tx == 0) {
        p.out_ids[row * G1 + pos] = s_found;
        for (int n = pos + 1; n < G1; ++n) p.out_ids[row * G1 + n] = -1;
    }
}

// probs[r, :] = softmax(logits[r, :] / temperature), fp32 (the sampler's distribution; SpeculativeSampler.cc feeds
// rejection sampling with these rows)
// WIDE: rows of both on 16 bytes, no remainder
template <bool WIDE>
__global__ __launch_bounds__(kThreads) void softmax_rows_kernel(const float* logits, int V, int ld, float inv_temp, float* probs) {
    __shared__ float s_red[kThreads / 64];
    const float* x = logits + (size_t)blockIdx.x * ld;
    float* y = probs + (size_t)blockIdx.x * V;
    const bool vec = WIDE || ((ld & 3) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0);
    float m = -3.0e38f;
    row_pass(x, V, vec, [&](float v) { m = fmaxf(m, v); });
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) s_red[threadIdx.x >> 6] = m;
    __syncthreads();
    m = s_red[0];
    for (int w = 1; w < kThreads / 64; ++w) m = fmaxf(m, s_red[w]);
    __syncthreads();
    float s = 0.f;
    row_pass(x, V, vec, [&](float v) { s += __expf((v - m) * inv_temp); });
    s = block_sum(s, s_red);
    // probs may be logits (every read of the sum is behind the block's barriers); 16-byte stores: the scalar loop took 45 of the 67 us of 64 rows of 152064
    const float inv = 1.f / s;
    if constexpr (WIDE) {
        const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
        f32x4* y4 = reinterpret_cast<f32x4*>(y);
#pragma unroll 4
        for (int j = threadIdx.x; j < V >> 2; j += kThreads) {
            f32x4 v = x4[j];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = __expf((v[r] - m) * inv_temp) * inv;
            y4[j] = v;
        }
    } else {
        int j = threadIdx.x;
        for (; j + 3 * kThreads < V; j += 4 * kThreads) {     // four loads in front of their stores: 3 rows of 27258 13.5 -> 10.9 us, 13.1 with pointers that cannot be the same
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = x[j + u * kThreads];
#pragma unroll
            for (int u = 0; u < 4; ++u) y[j + u * kThreads] = __expf((v[u] - m) * inv_temp) * inv;
        }
        for (; j < V; j += kThreads) y[j] = __expf((x[j] - m) * inv_temp) * inv;
    }
}

// (a, b) summed over the block in a fixed order (wave butterfly, then 16 partials added by every thread): deterministic.
__device__ __forceinline__ void block_sum2(float& a, float& b, float (*s_pair)[2]) {
    a = wave_sum(a); b = wave_sum(b);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) { s_pair[wave][0] = a; s_pair[wave][1] = b; }
    __syncthreads();
    float ta = 0.f, tb = 0.f;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) { ta += s_pair[w][0]; tb += s_pair[w][1]; }
    __syncthreads();
    a = ta; b = tb;
}

// Temperature, then repetition / presence / frequency penalties, in place on fp32 logits.
//   batchApplyTemperaturePenalty (sampling_penalty_kernels.cu:26-54): logit *= 1 / (T[row] + 1e-6)
//   batchApplyPenaltyLongSeq (:129-180): every vocabulary id seen among output_ids[0 .. step)[row] (padding positions
//   [input_length, max_input_length) skipped, ids outside [0, V) skipped) is penalised ONCE:
//   logit = logit < 0 ? logit * rep : logit / rep;  logit -= presence;  logit -= frequency * count.
// Temperature runs over the row in a launch of its own, the penalties in one behind it.
struct PenaltyParams {
    float*         logits;
    int            V, ld;
    const float   *temperature, *repetition, *presence, *frequency;
    const int32_t* output_ids;     // [step][batch]
    const int32_t* input_lengths;  // [batch] or null
    int            batch, max_input_length, step;
    int32_t*       counts;         // [batch][V]: histories of more than kShortHistory entries
};

// Of the n values of x a thread's own (start, start + stride, ..) by its row's temperature; vec: x lies on 16 bytes, start and stride count fours there.
__device__ __forceinline__ void scale_row(const PenaltyParams& p, int row, float* x, int n, bool vec, int start, int stride) {
    const float inv_t = 1.0f / (p.temperature[row] + 1e-6f);
    int done = 0;
    if (vec) {
        f32x4* x4 = reinterpret_cast<f32x4*>(x);
        done = n & ~3;
#pragma unroll 4
        for (int j = start; j < n >> 2; j += stride) {
            f32x4 v = x4[j];
            v[0] *= inv_t; v[1] *= inv_t; v[2] *= inv_t; v[3] *= inv_t;
            x4[j] = v;
        }
    }
    for (int j = done + start; j < n; j += stride) x[j] *= inv_t;
}

// Temperature alone: blockIdx.x splits the row.
template <bool WHOLE>
__global__ __launch_bounds__(kThreads) void temperature_kernel(const PenaltyParams p) {
    const int row = WHOLE ? blockIdx.x : blockIdx.y, start = (WHOLE ? 0 : blockIdx.x * kThreads) + threadIdx.x, stride = WHOLE ? kThreads : gridDim.x * kThreads;
    scale_row(p, row, p.logits + (size_t)row * p.ld, p.V, (p.ld & 3) == 0 && (reinterpret_cast<uintptr_t>(p.logits) & 15) == 0, start, stride);
}

__device__ __forceinline__ float penalised(const PenaltyParams& p, int row, float logit, int count) {
    if (p.repetition) logit = logit < 0.0f ? logit * p.repetition[row] : logit / p.repetition[row];
    if (p.presence) logit -= p.presence[row];
    if (p.frequency) logit -= p.frequency[row] * (float)count;
    return logit;
}

// A history of at most kShortHistory entries is counted in LDS: a table of at least twice as many slots, hashed by the id, probed in line.  No [batch][V] counters to clear (39 MB at
// 64 rows of 152064, more than all the other work of the launch), and no entry is compared with every other.
// us with such comparisons / here / with counters in memory: 16 rows of 1627 entries 343 / 7.7 / 15, 1 row of 300 20 / 3.1 / 5.5, 64 rows of 256 11.5 / 5.7 / 12.4; in the joint
// launches below 64 rows of 2000 253 / 32.
constexpr int kShortHistory = 2048;
struct HistoryTable { int key[2 * kShortHistory], count[2 * kShortHistory]; };      // key -1: free

// A thread's entries of the row's history, -1: padding or none.
template <int NT>
struct HistoryIds {
    static constexpr int E = (kShortHistory + NT - 1) / NT;
    int tok[E];
    __device__ __forceinline__ void load(const PenaltyParams& p, int row, int id_step, int id_row) {
        const int input_length = p.input_lengths ? p.input_lengths[row] : p.max_input_length;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = threadIdx.x + e * NT;
            tok[e] = i < p.step && !(i >= input_length && i < p.max_input_length) ? p.output_ids[(size_t)i * id_step + (size_t)row * id_row] : -1;
        }
    }
};
// Counts the ids in [lo, lo + n), 2^bits slots; seen(i) for each entry, i = its id - lo.  Whole block of NT threads; ends with a barrier.
template <int NT, class Seen>
__device__ __forceinline__ void count_history(const HistoryIds<NT>& ids, HistoryTable& t, int bits, int lo, int n, Seen&& seen) {
    const int size = 1 << bits;
    for (int i = threadIdx.x; i < size; i += NT) { t.key[i] = -1; t.count[i] = 0; }
    __threadfence_block();
    __syncthreads();                                        // also: the row's scaling by other threads is done
#pragma unroll
    for (int e = 0; e < HistoryIds<NT>::E; ++e) {
        const int tok = ids.tok[e];
        if (tok < lo || tok >= lo + n) continue;
        int at = (int)(((uint32_t)tok * 2654435761u) >> (32 - bits));
        for (int probe = 0; probe < size; ++probe) {        // ends: there are more slots than entries
            const int was = atomicCAS(&t.key[at], -1, tok);
            if (was == -1 || was == tok) { atomicAdd(&t.count[at], 1); break; }
            at = (at + 1) & (size - 1);
        }
        seen(tok - lo);
    }
    __syncthreads();
}
__device__ __forceinline__ int history_bits(int step) {
    int bits = 6;
    while ((1 << bits) < 2 * step) ++bits;
    return bits;
}
// how often the id is in the history
__device__ __forceinline__ int history_count(const HistoryTable& t, int bits, int tok) {
    const int size = 1 << bits;
    int at = (int)(((uint32_t)tok * 2654435761u) >> (32 - bits));
    for (int probe = 0; probe < size; ++probe) {
        const int key = t.key[at];
        if (key == tok) return t.count[at];
        if (key == -1) break;
        at = (at + 1) & (size - 1);
    }
    return 0;
}

// Penalises the history's ids in [lo, lo + n) once each, x = the row from lo on.  Whole block of NT threads; ends without a barrier.
template <int NT>
__device__ __forceinline__ void penalise_history(const PenaltyParams& p, HistoryTable& t, int row, int id_step, int id_row, int lo, int n, float* x) {
    const int bits = history_bits(p.step);
    HistoryIds<NT> ids;
    ids.load(p, row, id_step, id_row);
    count_history<NT>(ids, t, bits, lo, n, [](int) {});
    for (int i = threadIdx.x; i < 1 << bits; i += NT) {
        const int tok = t.key[i];
        if (tok >= 0) x[tok - lo] = penalised(p, row, x[tok - lo], t.count[i]);
    }
}

template <int NT>
__global__ __launch_bounds__(NT) void penalties_short_kernel(const PenaltyParams p) {
    __shared__ HistoryTable table;
    penalise_history<NT>(p, table, blockIdx.x, p.batch, 1, 0, p.V, p.logits + (size_t)blockIdx.x * p.ld);
}

// Temperature, penalties and softmax of the sampler in two launches, every row split over blocks.  One block per row, the softmax alone took 36 us of 64 rows of 152064 (its
// three passes at what one CU pulls), behind 14 of temperature and 14 of penalties; the two take 29 and 11.
// A slice of up to kHeld aligned values stays in registers between its uses.  The history is counted while the slice is on its way; a bitmap names the fours with an id of it, whose
// threads look their ids up.  64 rows of 152064: 24.7 us walked three times, with the penalties behind the scaled values in memory; held 22.4 (without the writing, and the same
// again in the next launch: 18.6, and 18.3 there in place of 12.6).
constexpr int kHeld = 20 * kThreads, kHeldRounds = kHeld / (4 * kThreads);
struct HeldShared { HistoryTable table; uint32_t seen[kHeld / 128]; };      // a bit per four values
struct HeldSlice {
    f32x4 v[kHeldRounds];
    float tail;                                                             // the last n % 4 values: threads 0 to 2
    int n, n4;
    __device__ __forceinline__ bool has(int i) const { return (int)threadIdx.x + i * kThreads < n4; }
    __device__ __forceinline__ bool has_tail() const { return (n4 << 2) + (int)threadIdx.x < n; }
    __device__ __forceinline__ void load(const PenaltyParams& p, HeldShared& sh, int row, int id_step, int id_row, int lo, float* x) {
        const int tx = threadIdx.x, rest = (n4 << 2) + tx;
        f32x4* x4 = reinterpret_cast<f32x4*>(x);
        HistoryIds<kThreads> ids;                                           // in front of the slice: loads come back in order
        if (p.output_ids) { ids.load(p, row, id_step, id_row); __builtin_amdgcn_sched_barrier(0); }
#pragma unroll
        for (int i = 0; i < kHeldRounds; ++i) v[i] = has(i) ? x4[tx + i * kThreads] : f32x4{0.f, 0.f, 0.f, 0.f};
        tail = has_tail() ? x[rest] : 0.f;
        const int bits = history_bits(p.step);
        if (p.output_ids) {
            for (int i = tx; i < kHeld / 128; i += kThreads) sh.seen[i] = 0u;
            count_history<kThreads>(ids, sh.table, bits, lo, n, [&](int at) { atomicOr(&sh.seen[at >> 7], 1u << (at >> 2 & 31)); });
        }
        const float scale = p.temperature ? 1.0f / (p.temperature[row] + 1e-6f) : 1.f;
        auto penalise = [&](float f, int at) { const int c = history_count(sh.table, bits, lo + at); return c ? penalised(p, row, f, c) : f; };
#pragma unroll
        for (int i = 0; i < kHeldRounds; ++i) {
            const int j = tx + i * kThreads;
            if (!has(i)) continue;
            if (p.temperature) v[i] *= scale;
            const bool seen = p.output_ids && (sh.seen[j >> 5] >> (j & 31) & 1u);
            if (seen) {
#pragma unroll
                for (int r = 0; r < 4; ++r) v[i][r] = penalise(v[i][r], 4 * j + r);
            }
            if (p.temperature || seen) x4[j] = v[i];
        }
        if (has_tail()) {
            if (p.temperature) tail *= scale;
            if (p.output_ids) tail = penalise(tail, rest);
            x[rest] = tail;
        }
    }
};

// Prepare: scales and penalises the slice, leaves its maximum and sum of exponentials.
template <bool HELD>
__global__ __launch_bounds__(kThreads) void sampling_prepare_kernel(const PenaltyParams p, float2* parts, int id_step, int id_row, int slice) {
    __shared__ std::conditional_t<HELD, HeldShared, HistoryTable> sh;
    __shared__ float s_red[kThreads / 64];
    const int row = blockIdx.y, tx = threadIdx.x, lo = min(p.V, (int)blockIdx.x * slice), n = min(p.V, lo + slice) - lo;
    float* x = p.logits + (size_t)row * p.ld + lo;
    const bool vec = (p.ld & 3) == 0 && (reinterpret_cast<uintptr_t>(p.logits) & 15) == 0;       // lo is a multiple of 4
    HeldSlice held;
    if constexpr (HELD) {
        held.n = n; held.n4 = n >> 2;
        held.load(p, sh, row, id_step, id_row, lo, x);
    } else {
        if (p.temperature) scale_row(p, row, x, n, vec, tx, kThreads);
        if (p.output_ids) penalise_history<kThreads>(p, sh, row, id_step, id_row, lo, n, x);
        __threadfence_block();
        __syncthreads();
    }
    auto each = [&](auto&& g) {
        if constexpr (HELD) {
#pragma unroll
            for (int i = 0; i < kHeldRounds; ++i)
                if (held.has(i)) { g(held.v[i][0]); g(held.v[i][1]); g(held.v[i][2]); g(held.v[i][3]); }
            if (held.has_tail()) g(held.tail);
        } else row_pass(x, n, vec, g);
    };
    float m = -3.0e38f;
    each([&](float f) { m = fmaxf(m, f); });
    m = wave_max(m);
    if ((tx & 63) == 0) s_red[tx >> 6] = m;
    __syncthreads();
    m = s_red[0];
    for (int w = 1; w < kThreads / 64; ++w) m = fmaxf(m, s_red[w]);
    __syncthreads();
    float s = 0.f;
    each([&](float f) { s += __expf(f - m); });
    s = block_sum(s, s_red);
    if (tx == 0) parts[(size_t)row * gridDim.x + blockIdx.x] = make_float2(m, s);
}

// A probability's place among kDrawBins bins of a sixteenth of an octave down from 1, 0: below them (2^-32 and less, negative, NaN); and its exact value in units of 2^-56.
constexpr int kDrawBins = 512, kDrawShift = 19, kDrawBase = (127 << 4) - (kDrawBins - 1), kList = 8 * kThreads;
__device__ __forceinline__ int draw_bin(uint32_t b) { return min(max((int)(b >> kDrawShift) - kDrawBase, 0), kDrawBins - 1); }
__device__ __forceinline__ unsigned long long draw_fixed(uint32_t b) { return (unsigned long long)((b & 0x7FFFFFu) | 0x800000u) << ((b >> 23) - 94u); }

// Rows so flat that the list of a bin (kList values, see draw_listed_kernel) cannot hold what is there: their mean lies 16 log2(V / sum) bins below their maximum, sum = that of
// exp(x - max), and most values within about twice that.  They are not counted: their thousands of values meet in a few words of LDS.  Us of the joint draw counted / not / of the
// separate launches: 64 rows of 152064 equal values 811 / 784 / 778, of deviation 0.05 402 / 392 / 389; 237 x 32000 equal 274 / 248 / 244.  A flatness that the rule does not see costs the difference,
// one that it sees wrongly (deviation 0.2, top-p 0.95) the gain.
__device__ __forceinline__ bool draw_is_flat(int V, float sum) { return (float)V > kList * (1.f + 16.f * __log2f((float)V / sum)); }

// Probabilities in place: exp(x - m) / sum from the slices' maxima and sums.  HIST: with a histogram of the slice's probabilities, count << 40 | sum of the bits below the bin's;
// bin 0, which counts nothing, says 1 for a flat row.
template <bool HIST>
__global__ __launch_bounds__(kThreads) void sampling_probs_kernel(float* logits, int V, int ld, const float2* parts, int slice, unsigned long long* hist) {
    __shared__ unsigned long long s_hist[HIST ? kDrawBins : 1];
    const int row = blockIdx.y, tx = threadIdx.x, lo = min(V, (int)blockIdx.x * slice), n = min(V, lo + slice) - lo;
    float* x = logits + (size_t)row * ld + lo;
    if (HIST) { for (int i = tx; i < kDrawBins; i += kThreads) s_hist[i] = 0ull; __syncthreads(); }
    const float2* pr = parts + (size_t)row * gridDim.x;
    float m = pr[0].x, s = 0.f;
    for (int i = 1; i < (int)gridDim.x; ++i) m = fmaxf(m, pr[i].x);
    for (int i = 0; i < (int)gridDim.x; ++i) s += pr[i].y * __expf(pr[i].x - m);
    const float inv = 1.f / s;
    const bool flat = HIST && draw_is_flat(V, s);
    auto count = [&](float v) {
        if (flat) return;
        const uint32_t b = v > 0.f ? __float_as_uint(v) : 0u;
        const int bin = draw_bin(b);
        if (bin > 0) atomicAdd(&s_hist[bin], (1ull << 40) + (unsigned long long)(b & ((1u << kDrawShift) - 1u)));
    };
    auto four = [&](f32x4 v) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = __expf(v[r] - m) * inv;
        if (HIST) { count(v[0]); count(v[1]); count(v[2]); count(v[3]); }
        return v;
    };
    auto one = [&](float f) {
        const float v = __expf(f - m) * inv;
        if (HIST) count(v);
        return v;
    };
    int done = 0;
    if ((ld & 3) == 0 && (reinterpret_cast<uintptr_t>(logits) & 15) == 0) {
        f32x4* x4 = reinterpret_cast<f32x4*>(x);
#pragma unroll 4
        for (int j = tx; j < n >> 2; j += kThreads) x4[j] = four(x4[j]);
        done = n & ~3;
    }
    for (int j = done + tx; j < n; j += kThreads) x[j] = one(x[j]);
    if constexpr (HIST) {
        __syncthreads();
        for (int i = tx; i < kDrawBins; i += kThreads) hist[((size_t)row * gridDim.x + blockIdx.x) * kDrawBins + i] = i == 0 ? (unsigned long long)flat : s_hist[i];
    }
}

// Longer histories: counters in memory, cleared by the first of two launches.
__global__ __launch_bounds__(kThreads) void clear_counts_kernel(int32_t* counts, size_t n) {
    for (size_t i = (size_t)blockIdx.x * kThreads + threadIdx.x; i < n; i += (size_t)gridDim.x * kThreads) counts[i] = 0;
}
__global__ __launch_bounds__(kThreads) void penalties_kernel(const PenaltyParams p) {
    const int row = blockIdx.x, tx = threadIdx.x;
    float* x = p.logits + (size_t)row * p.ld;
    int32_t* cnt = p.counts + (size_t)row * p.V;
    // count the ids of the history; the lane whose increment found a zero owns the id and penalises it once the counts are final -- the work is
    // proportional to the history, not to the vocabulary (histories beyond 32 entries per lane fall back to a scan of the row)
    const int input_length = p.input_lengths ? p.input_lengths[row] : p.max_input_length;
    uint32_t mine = 0;                                     // bit s: the s-th history entry of this lane was the first of its id
    int s = 0;
    for (int index = tx; index < p.step; index += kThreads, ++s) {
        if (index >= input_length && index < p.max_input_length) continue;
        const int tok = p.output_ids[(size_t)index * p.batch + row];
        if (tok >= p.V || tok < 0) continue;
        const int old = atomicAdd(&cnt[tok], 1);
        if (old == 0 && s < 32) mine |= 1u << s;
    }
    __syncthreads();
    if (p.step <= 32 * kThreads) {
        s = 0;
        for (int index = tx; index < p.step; index += kThreads, ++s) {
            if (!((mine >> s) & 1u)) continue;
            const int tok = p.output_ids[(size_t)index * p.batch + row];
            x[tok] = penalised(p, row, x[tok], __hip_atomic_load(&cnt[tok], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
    } else {
        for (int j = tx; j < p.V; j += kThreads) {
            const int c = __hip_atomic_load(&cnt[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (c > 0) x[j] = penalised(p, row, x[j], c);
        }
    }
}

// Top-k / top-p filter and draw on probability rows (CudaSampleOp.cc:748-786), one block per row:
//   k = top_k[row] (<= 0 or >= V: no filter): entries below the k-th largest value are dropped (ties with it stay, :755-760);
//   p = top_p[row] (|p| < 1e-7 reads as 1; |p - 1| < 1e-7: no filter): in descending order (equal values in index order) an
//       entry is dropped when the mass before it exceeds p (:768-775).  Only the smallest surviving value v can lose part of
//       its equals: with S = mass of all strictly larger entries, its j-th occurrence stays while S + j v <= p;
//   the survivors are renormalised by max(sum, 1e-10) (probs_out, optional) and one index is drawn by inverse CDF in index order
//   with uniform[row] (torch.multinomial in the reference: same distribution, explicit randomness).
// No sort.  What bounds it is the number of passes over the row: bit by bit from the top of the fp32 pattern (non-negative floats order like their bits) the
// two thresholds took 31 passes of 24 us over 152064 values on one CU.  A histogram of the pattern's top 12 bits (a sixteenth of an octave per bin) with the
// count and the mass of every bin names the one bin each threshold lies in; the values of those two bins go to LDS and the low 19 bits are searched there.  The
// values of a bin share their exponent, so its mass is a sum of integers, exact whatever the order of the atomics, and packs with the count into one 64-bit
// word: one LDS atomic a value.  The draw reads the row twice more, a wave per contiguous sixteenth.  Where a bin holds more than kSet values (flat rows), a second
// histogram of it gives the next 12 bits; runs of more than kSet equal values are searched bit by bit over the row for the
// last 7.  Infinities, p < 0 and rows of more than 2^20 values are searched bit by bit as a whole.
// 64 rows of 152064, top-k 0..100, top-p 0.8..0.95 of a distribution with a heavy tail: 827 -> 97 us; flat ones (softmax of logits of deviation 0.5) 508 -> 134.
struct TopKPParams {
    const float*   probs;
    int            V, ld;
    const int32_t* top_k;
    const float*   top_p;
    const float*   uniform;
    int32_t*       ids;
    float*         probs_out;
    int            ld_out;
};

constexpr int kSet = 4096, kBinShift = 19, kBins = 1 << (31 - kBinShift), kWaves = kThreads / 64;

// (16-byte aligned, so that a wave reads the sixteen waves' results 16 bytes at a time: 31 against 38 us for a row of 1001)
#define ALIGN16 __attribute__((aligned(16)))
struct DrawShared { ALIGN16 float red[kWaves]; int found; };
struct SampleShared : DrawShared {
    ALIGN16 float    pair[kWaves][2];
    ALIGN16 float    scan[kThreads];
    ALIGN16 unsigned long long hist[kBins];  // count << 40 | sum of the bits below the bin's
    ALIGN16 uint32_t set_k[kSet];
    ALIGN16 uint32_t set_q[kSet];
    ALIGN16 uint32_t wave_n[kWaves];
    ALIGN16 unsigned long long wave_m[kWaves];
    ALIGN16 double   wave_d[kWaves];
    int      n_k, n_q, bin_k, bin_q;
    uint32_t above_k;                        // entries in the bins above bin_k
    double   above_q;                        // mass in the bins above bin_q
};
#undef ALIGN16

__device__ __forceinline__ float sample_pos(float v) { return v > 0.f ? v : 0.f; }   // +0 for -0, negatives and NaN: the bit pattern is the order

// four values of [lo, hi) from index j on (a multiple of 4 from a 16-byte address); outside: zeros
__device__ __forceinline__ f32x4 row4(const float* q, int j, int lo, int hi) {
    if (j >= lo && j + 3 < hi) return *reinterpret_cast<const f32x4*>(q + j);
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) if (j + r >= lo && j + r < hi) v[r] = q[j + r];
    return v;
}

// sum over the wave without the LDS crossbar (row operations, then the swaps of 16 and 32 lanes): every lane gets it
__device__ __forceinline__ float lane_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, true));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, true));
    return xor32_sum(xor16_sum(v));
}
__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// One index of the row by inverse CDF over w(value), one contiguous run of the row per wave: the runs' sums, their prefix, and a second walk of the run that
// holds u.  The same rule as block_draw (a run that the rounding of the second walk leaves without a crossing gives its last index of positive weight).  Rows that start off
// 16 bytes (an odd V) are walked from the address before them on: value by value 41 rows of 84055 took 33 us, 16 this way.
template <class W>
__device__ __forceinline__ float row_draw(const float* row, int V, float u01, DrawShared& sh, W&& weight) {
    const int tx = threadIdx.x, lane = tx & 63, wave = tx >> 6;
    const int off = (int)(reinterpret_cast<uintptr_t>(row) >> 2 & 3), end = V + off;             // value i of the row is q[off + i]
    const float* q = row - off;
    const int chunk = ((end + kWaves - 1) / kWaves + 255) & ~255;               // 256 values per step
    const int w0 = min(end, wave * chunk), w1 = min(end, w0 + chunk);
    float s = 0.f;
#pragma unroll 4
    for (int j = w0 + lane * 4; j < w1; j += 256) {
        const f32x4 v = row4(q, j, off, w1);
        s += (weight(v[0]) + weight(v[1])) + (weight(v[2]) + weight(v[3]));
    }
    s = lane_sum(s);
    if (lane == 0) sh.red[wave] = s;
    if (tx == 0) sh.found = V - 1;
    __syncthreads();
    float total = 0.f, excl = 0.f;
    for (int w = 0; w < kWaves; ++w) { if (w == wave) excl = total; total += sh.red[w]; }
    const float u = u01 * total, incl = excl + s;
    if (s > 0.f && excl <= u && incl > u) {                                     // the same for every lane of the wave
        float c = excl;
        int hit = -1, last = -1;
        for (int j = w0 + lane * 4; j - lane * 4 < w1; j += 256) {
            const f32x4 v = row4(q, j, off, w1);
            float t[4], mine = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) { t[r] = weight(v[r]); mine += t[r]; }
            const unsigned long long any = __ballot(mine > 0.f);
            if (any == 0ull) continue;
            float pre = mine;                                                   // inclusive over the lanes
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) { const float y = __shfl_up(pre, o); if (lane >= o) pre += y; }
            float at = c + (pre - mine);
            int h = -1;
#pragma unroll
            for (int r = 0; r < 4; ++r) { at += t[r]; if (t[r] > 0.f && h < 0 && at > u) h = j + r; }
            const unsigned long long crossed = __ballot(h >= 0);
            if (crossed) { hit = __shfl(h, __ffsll((unsigned long long)crossed) - 1); break; }
            int l = -1;
#pragma unroll
            for (int r = 0; r < 4; ++r) if (t[r] > 0.f) l = j + r;
            last = __shfl(l, 63 - __clzll((long long)any));
            c += __shfl(pre, 63);
        }
        if (lane == 0) sh.found = (hit >= 0 ? hit : last) - off;
    }
    __syncthreads();
    return total;
}

// The filter and the draw over the row with equals of the top-p boundary value dropped from some index on; kept(j), for j of this thread's segment
// [lo, hi), is what stays of value j.
template <class Out>
__device__ __forceinline__ void filter_and_draw(const float* q, int V, uint32_t kb, uint32_t vbits, bool use_p, float tp, float u, SampleShared& sh, Out&& out) {
    const int tx = threadIdx.x;
    // top-p boundary value (an entry's value: the mass above a threshold only changes at entries).  Its equals are ranked in index order over the
    // contiguous segments block_draw uses; `cut` = first index of this thread's segment from which they are dropped.
    const int seg = draw_segment(V);
    const int lo = min(V, tx * seg), hi = min(V, lo + seg);
    int cut = hi;
    if (use_p) {
        float sb = 0.f, ties = 0.f;
        for (int j = lo; j < hi; ++j) {
            const float v = sample_pos(q[j]);
            const uint32_t b = __float_as_uint(v);
            sb += (b > vbits) ? v : 0.f;
            ties += (b == vbits) ? 1.f : 0.f;
        }
        const float mine = ties;
        float z = 0.f;
        block_sum2(sb, z, sh.pair);
        sh.scan[tx] = mine;                       // inclusive scan of the tie counts over threads (exact: counts < 2^24)
        __syncthreads();
        for (int off = 1; off < kThreads; off <<= 1) {
            const float add = (tx >= off) ? sh.scan[tx - off] : 0.f;
            __syncthreads();
            sh.scan[tx] += add;
            __syncthreads();
        }
        float rank = sh.scan[tx] - mine;
        __syncthreads();
        const float vb = __uint_as_float(vbits);
        for (int j = lo; j < hi; ++j) {
            if (__float_as_uint(sample_pos(q[j])) != vbits) continue;
            if (sb + rank * vb > tp) { cut = j; break; }
            rank += 1.f;
        }
    }
    auto kept = [&](int j) {      // j inside this thread's segment
        const float v = sample_pos(q[j]);
        const uint32_t b = __float_as_uint(v);
        return (b >= kb && (b > vbits || (b == vbits && j < cut))) ? v : 0.f;
    };
    const float total = block_draw(kept, V, u, sh.red, sh.scan, &sh.found);
    out(kept, lo, hi, total);
}

// Both thresholds from the histogram: kb = the k-th largest value's bits (0: every entry), vbits = the smallest value's bits that top-p keeps.  use_p is cleared when the
// whole row's mass fits.  Returns 0 when the row has to be searched bit by bit, 1 when all equals of the boundary value stay, 2 when some of them go.
__device__ __forceinline__ int search_histogram(const float* q, int V, bool vec, bool use_k, int k, bool& use_p, float tp, uint32_t& kb, uint32_t& vbits,
                                                SampleShared& sh) {
    const int tx = threadIdx.x, lane = tx & 63, wave = tx >> 6;
    if (V > (1 << 20) || (use_p && tp < 0.f)) return 0;                         // the packed sums hold 2^21 values
    auto bits_of = [](float x) { return __float_as_uint(sample_pos(x)); };
    // the values above zero whose bits from `up` on are `top`, by their bits [shift, up)
    auto count = [&](int shift, int up, uint32_t top) {
        for (int i = tx; i < kBins; i += kThreads) sh.hist[i] = 0ull;
        if (tx == 0) { sh.bin_k = sh.bin_q = -1; sh.n_k = sh.n_q = 0; }
        __syncthreads();
        const uint32_t low = (1u << shift) - 1u;
        row_pass(q, V, vec, [&](float x) {
            const uint32_t b = bits_of(x);
            if (b != 0u && b >> up == top) atomicAdd(&sh.hist[b >> shift & (kBins - 1)], (1ull << 40) + (unsigned long long)(b & low));
        });
        __syncthreads();
    };
    // The bins that hold the k-th largest value (sh.bin_k) and the crossing of p (sh.bin_q), c0 values and m0 mass above the histogram: from the largest values down, a thread takes
    // kBins / kThreads bins, prefixes over the lanes and the waves.  Returns the histogram's mass.
    auto locate = [&](int shift, uint32_t base, bool want_k, uint32_t c0, bool want_p, double m0, bool only_above_p) {
        constexpr int PB = kBins / kThreads;
        uint32_t c[PB], ci = 0;
        double m[PB], mi = 0.0;
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const uint32_t bin = kBins - 1 - (tx * PB + i), at = base | bin << shift, e = at >> 23;
            const unsigned long long h = sh.hist[bin], mant = (at & 0x7FFFFFu) | (e ? 0x800000u : 0u);
            c[i] = (uint32_t)(h >> 40);
            m[i] = (double)(c[i] * mant + (h & ((1ull << 40) - 1ull))) * __builtin_ldexp(1.0, (int)(e ? e : 1) - 150);
            if (at >= 0x7F800000u) { if (c[i]) sh.bin_k = -2; m[i] = 0.0; }         // an infinity
            ci += c[i]; mi += m[i];
        }
        const uint32_t c_own = ci;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t yc = __shfl_up(ci, o);
            const double ym = __shfl_up(mi, o);
            if (lane >= o) { ci += yc; mi += ym; }
        }
        if (lane == 63) { sh.wave_n[wave] = ci; sh.wave_d[wave] = mi; }
        __syncthreads();
        if (sh.bin_k == -2) return -1.0;
        uint32_t c_at = c0 + ci - c_own;
        double m_at = 0.0, total = 0.0;
        for (int w = 0; w < kWaves; ++w) {
            if (w < wave) c_at += sh.wave_n[w];
            if (w == wave) m_at = total;
            total += sh.wave_d[w];
        }
        const double m_lane = __shfl_up(mi, 1);
        if (lane > 0) m_at += m_lane;
        m_at += m0;
        if (only_above_p) want_p = want_p && total > (double)tp;
        // The prefix up to a thread's bins and the sum over the bins of the thread before it round differently: both may see p crossed.  The larger values' bin has it, with the sum
        // of the thread that it belongs to.
        int mine_q = -1;
        double mine_above = 0.0;
#pragma unroll
        for (int i = 0; i < PB; ++i) {
            const int bin = kBins - 1 - (tx * PB + i);
            if (want_k && c_at < (uint32_t)k && c_at + c[i] >= (uint32_t)k) { sh.bin_k = bin; sh.above_k = c_at; }
            if (want_p && m_at <= (double)tp && m_at + m[i] > (double)tp) { mine_q = bin; mine_above = m_at; }
            c_at += c[i]; m_at += m[i];
        }
        if (mine_q >= 0) atomicMax(&sh.bin_q, mine_q);
        __syncthreads();
        if (mine_q >= 0 && mine_q == sh.bin_q) sh.above_q = mine_above;             // to be read behind another barrier
        return total;
    };
    count(kBinShift, 31, 0);
    const double total = locate(kBinShift, 0, use_k, 0, use_p, 0.0, true);
    if (total < 0.0) return 0;
    if (use_p) use_p = total > (double)tp;                                      // nothing to drop when even the mass above 0 fits
    const int bin_k = use_k ? sh.bin_k : -1, bin_q = use_p ? sh.bin_q : -1;     // bin_k -1: fewer than k entries are above zero
    if (use_p && bin_q < 0) return 0;                                           // the sums crossed p between a thread's last bin and the next thread's first
    kb = 0; vbits = 0;
    if (bin_k < 0 && bin_q < 0) return 1;
    int left_k = kBinShift, left_q = kBinShift;                                 // bits of the thresholds that are not known
    if (bin_k >= 0) kb = (uint32_t)bin_k << kBinShift; else left_k = 0;
    if (bin_q >= 0) vbits = (uint32_t)bin_q << kBinShift; else left_q = 0;
    auto in_k = [&](uint32_t b) { return bin_k >= 0 && b != 0u && b >> left_k == kb >> left_k; };
    auto in_q = [&](uint32_t b) { return bin_q >= 0 && b != 0u && b >> left_q == vbits >> left_q; };
    auto gather = [&]() {                                                       // the values that share a threshold's known bits
        row_pass(q, V, vec, [&](float x) {
            const uint32_t b = bits_of(x);
            if (in_k(b)) { const int at = atomicAdd(&sh.n_k, 1); if (at < kSet) sh.set_k[at] = b; }
            if (in_q(b)) { const int at = atomicAdd(&sh.n_q, 1); if (at < kSet) sh.set_q[at] = b; }
        });
        __syncthreads();
    };
    gather();
    uint32_t above_k = sh.above_k;
    double above_q = sh.above_q;
    if (sh.n_k > kSet || sh.n_q > kSet) {                                       // flat rows: the next 12 bits from a histogram of the bin
        const bool again_k = sh.n_k > kSet, again_q = sh.n_q > kSet;
        constexpr int REST = kBinShift - 12;
        __syncthreads();                                                        // the counts have been read
        if (again_k) {
            count(REST, kBinShift, (uint32_t)bin_k);
            locate(REST, kb, true, above_k, false, 0.0, false);
            kb |= (uint32_t)sh.bin_k << REST; above_k = sh.above_k; left_k = REST;
        }
        if (again_q) {
            __syncthreads();                                                    // bin_k has been read
            count(REST, kBinShift, (uint32_t)bin_q);
            locate(REST, vbits, false, 0, true, above_q, false);
            if (sh.bin_q < 0) return 0;                                         // rounding took the crossing out of the bin
            __syncthreads();
            vbits |= (uint32_t)sh.bin_q << REST; above_q = sh.above_q; left_q = REST;
        }
        __syncthreads();
        gather();
    }
    const int n_k = sh.n_k, n_q = sh.n_q;
    const bool whole = n_k > kSet || n_q > kSet;                                // long runs of one value: the last bits from the row
    const int e_q = (int)(vbits >> 23);
    const uint32_t implicit = e_q ? 0x800000u : 0u;
    const double unit = __builtin_ldexp(1.0, (e_q ? e_q : 1) - 150);
    auto mantissa = [&](uint32_t b) { return (unsigned long long)((b & 0x7FFFFFu) | implicit); };
    auto over_waves = [&](uint32_t& cnt, unsigned long long& mass) {            // of every wave's sums
        if (bin_q >= 0) mass = wave_sum_u64(mass);
        if (lane == 0) { sh.wave_n[wave] = cnt; sh.wave_m[wave] = mass; }
        __syncthreads();
        cnt = 0; mass = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) { cnt += sh.wave_n[w]; mass += sh.wave_m[w]; }
        __syncthreads();
    };
    // the rest, most significant bit first: the largest threshold that leaves k entries (more mass than p) at or above it
    uint32_t ties = 0;
    unsigned long long mass = 0;
    if (!whole) {                                                               // the sets lie in registers
        constexpr int PT = kSet / kThreads;
        uint32_t vk[PT], vq[PT];
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            const int j = tx + i * kThreads;
            vk[i] = j < n_k ? sh.set_k[j] : 0u;
            vq[i] = j < n_q ? sh.set_q[j] : 0u;
        }
        for (int bit = max(left_k, left_q) - 1; bit >= 0; --bit) {
            const uint32_t ck = kb | (1u << bit), cq = vbits | (1u << bit);
            uint32_t cnt = 0;
            mass = 0;
#pragma unroll
            for (int i = 0; i < PT; ++i) {
                cnt += (uint32_t)__popcll(__ballot(vk[i] >= ck));
                if (vq[i] >= cq) mass += mantissa(vq[i]);
            }
            over_waves(cnt, mass);
            if (bin_k >= 0 && bit < left_k && above_k + cnt >= (uint32_t)k) kb = ck;
            if (bin_q >= 0 && bit < left_q && above_q + (double)mass * unit > (double)tp) vbits = cq;
        }
        if (bin_q < 0) return 1;
        mass = 0;
#pragma unroll
        for (int i = 0; i < PT; ++i) {
            ties += (uint32_t)__popcll(__ballot(vq[i] == vbits && vq[i] != 0u));
            if (vq[i] > vbits) mass += mantissa(vq[i]);
        }
        over_waves(ties, mass);
    } else {
        const uint32_t top_k = bin_k >= 0 ? kb >> left_k : ~0u, top_q = bin_q >= 0 ? vbits >> left_q : ~0u;
        for (int bit = max(left_k, left_q) - 1; bit >= 0; --bit) {
            const uint32_t ck = kb | (1u << bit), cq = vbits | (1u << bit);
            uint32_t cnt = 0;
            mass = 0;
            row_pass(q, V, vec, [&](float x) {
                const uint32_t b = bits_of(x);
                if (b >> left_k == top_k && b >= ck) ++cnt;
                if (b >> left_q == top_q && b >= cq) mass += mantissa(b);
            });
            cnt = (uint32_t)wave_sum_u64(cnt);
            over_waves(cnt, mass);
            if (bin_k >= 0 && bit < left_k && above_k + cnt >= (uint32_t)k) kb = ck;
            if (bin_q >= 0 && bit < left_q && above_q + (double)mass * unit > (double)tp) vbits = cq;
        }
        if (bin_q < 0) return 1;
        mass = 0;
        row_pass(q, V, vec, [&](float x) {
            const uint32_t b = bits_of(x);
            if (b == vbits && b != 0u) ++ties;
            if (b >> left_q == top_q && b > vbits) mass += mantissa(b);
        });
        ties = (uint32_t)wave_sum_u64(ties);
        over_waves(ties, mass);
    }
    // equals of the boundary value: the j-th of T stays while S + j v <= p, S = the mass above it
    return ties <= 1u || above_q + (double)(mass + (unsigned long long)(ties - 1u) * mantissa(vbits)) * unit <= (double)tp ? 1 : 2;
}

__device__ __forceinline__ void sample_row(const TopKPParams& p, int row, SampleShared& sh) {
    const int tx = threadIdx.x, V = p.V;
    const float* q = p.probs + (size_t)row * p.ld;
    const int k = p.top_k ? p.top_k[row] : 0;
    const bool use_k = k > 0 && k < V;
    float tp = p.top_p ? p.top_p[row] : 1.0f;
    if (fabsf(tp) < 1e-7f) tp = 1.0f;
    bool use_p = fabsf(tp - 1.0f) >= 1e-7f;
    const bool vec = ((p.ld & 3) == 0) && ((reinterpret_cast<uintptr_t>(p.probs) & 15) == 0);
    uint32_t kb = 0, vbits = 0;
    int how = 1;                                       // 0: bit by bit over the row, 1: kept are the values at or above kb and vbits, 2: some equals of vbits go
    if (use_k || use_p) {
        how = search_histogram(q, V, vec, use_k, k, use_p, tp, kb, vbits, sh);
        if (how == 0) {
            use_p = fabsf(tp - 1.0f) >= 1e-7f;
            if (use_p) {                               // nothing to drop when even the mass above 0 fits
                float m = 0.f, z = 0.f;
                row_pass(q, V, vec, [&](float x) { m += sample_pos(x); });
                block_sum2(m, z, sh.pair);
                use_p = m > tp;
            }
            uint32_t tk = 0, tq = 0;                   // tk: largest t with #(bits >= t) >= k;  tq: largest t with mass(bits > t) > p
            if (use_k || use_p) {
                for (int bit = 30; bit >= 0; --bit) {
                    const uint32_t ck = tk | (1u << bit), cq = tq | (1u << bit);
                    float cnt = 0.f, mass = 0.f;
                    row_pass(q, V, vec, [&](float x) {
                        const float v = sample_pos(x);
                        const uint32_t b = __float_as_uint(v);
                        cnt += (b >= ck) ? 1.f : 0.f;
                        mass += (b > cq) ? v : 0.f;
                    });
                    block_sum2(cnt, mass, sh.pair);
                    if (use_k && cnt >= (float)k) tk = ck;
                    if (use_p && mass > tp) tq = cq;
                }
            }
            kb = use_k ? tk : 0u; vbits = use_p ? tq + 1u : 0u;
            how = 2;
        }
    }
    float* y = p.probs_out ? p.probs_out + (size_t)row * p.ld_out : nullptr;
    if (how == 1) {
        const uint32_t floor_bits = max(kb, vbits);
        auto weight = [&](float x) { const float v = sample_pos(x); return __float_as_uint(v) >= floor_bits ? v : 0.f; };
        const float total = row_draw(q, V, p.uniform[row], sh, weight);
        if (tx == 0) p.ids[row] = sh.found;
        if (y) {
            const float den = fmaxf(total, 1e-10f);
            for (int j = tx; j < V; j += kThreads) y[j] = weight(q[j]) / den;
        }
    } else {
        filter_and_draw(q, V, kb, vbits, use_p, tp, p.uniform[row], sh, [&](auto& kept, int lo, int hi, float total) {
            if (tx == 0) p.ids[row] = sh.found;
            if (!y) return;
            const float den = fmaxf(total, 1e-10f);
            for (int j = lo; j < hi; ++j) y[j] = kept(j) / den;
        });
    }
}

__global__ __launch_bounds__(kThreads) void top_k_top_p_sample_kernel(const TopKPParams p) {
    __shared__ SampleShared sh;
    sample_row(p, blockIdx.x, sh);
}

// The same behind sampling_probs_kernel<true>.  Its histograms name the bin that the higher of the two thresholds lies in, and give every slice's mass above it; the values of
// that bin (1300 of 152064 where logits have a deviation of 2) are copied to the row's list by sampling_list_kernel, every row split over blocks as in the launches before.
// draw_listed_kernel, one block per row, finds the threshold among them, with it every slice's mass and the slice that the draw falls into, and walks that slice alone.
// Counts and masses are integers (units of 2^-56): exact, whatever the order.  Rows without such a bin (no filter, a threshold below 2^-32) or with more than kList values
// in it take sample_row.
// 64 rows of 152064, top-k 0..100, top-p 0.8..0.95: 103 us of top_k_top_p_sample_kernel (one compute unit pulls a row three times) -> 12.8 and 16.8.
__device__ __host__ __forceinline__ int draw_list(int V) { return V < kList ? V : kList; }        // a row's list

struct DrawFilter { int k; bool use_k, use_p; float tp; };
__device__ __forceinline__ DrawFilter draw_filter(const TopKPParams& p, int row) {
    DrawFilter f;
    f.k = p.top_k ? p.top_k[row] : 0;
    f.use_k = f.k > 0 && f.k < p.V;
    f.tp = p.top_p ? p.top_p[row] : 1.0f;
    if (fabsf(f.tp) < 1e-7f) f.tp = 1.0f;
    f.use_p = !(fabsf(f.tp - 1.0f) < 1e-7f);
    return f;
}
// mass <= p as mass <= draw_limit(p), p >= 0
__device__ __forceinline__ unsigned long long draw_limit(float tp) { return tp >= 64.f ? ~0ull >> 1 : (unsigned long long)((double)tp * 72057594037927936.0); }
// The mass of c values that share the exponent and the four bits behind it, at = those, low = the sum of the bits below; c at most 2^20.  In 32 bits: of c times the whole mantissa
// in 64 bits the compiler (hipcc 7.2) lost the mantissa's mask.
__device__ __forceinline__ unsigned long long draw_mass(uint32_t at, uint32_t c, unsigned long long low) {
    return (((unsigned long long)(c * (16u + (at & 15u))) << kDrawShift) + low) << ((at >> 4) - 94u);
}

struct DrawRow { int n; uint32_t low, above; unsigned long long mass; };        // values in the list (-1: none is made), their top bits, how many and how much lies above them

struct DrawScan {                                                               // where the filter's thresholds cross, from the largest values down, a bin a thread
    uint32_t c[kWaves];
    unsigned long long m[kWaves];
    int bin;
};
// ci / mi: the bin's count and mass with all above it, from c0 and m0 on.  Returns the higher crossing's bin (0 to `most`, -1: none).  Whole block.
__device__ __forceinline__ int draw_cross(const DrawFilter& f, unsigned long long limit, int bin, uint32_t c, unsigned long long m, uint32_t c0, unsigned long long m0, uint32_t& ci,
                                          unsigned long long& mi, bool& of_p, DrawScan& sc) {
    const int tx = threadIdx.x, lane = tx & 63, wave = tx >> 6;
    if (tx == 0) sc.bin = -1;
    ci = c; mi = m;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t yc = __shfl_up(ci, o);
        const unsigned long long ym = __shfl_up(mi, o);
        if (lane >= o) { ci += yc; mi += ym; }
    }
    if (lane == 63) { sc.c[wave] = ci; sc.m[wave] = mi; }
    __syncthreads();
    ci += c0; mi += m0;
    for (int w = 0; w < wave; ++w) { ci += sc.c[w]; mi += sc.m[w]; }
    const bool of_k = f.use_k && ci - c < (uint32_t)f.k && ci >= (uint32_t)f.k;
    of_p = f.use_p && mi - m <= limit && mi > limit;
    if (bin >= 0 && (of_k || of_p)) atomicMax(&sc.bin, bin);
    __syncthreads();
    return sc.bin;
}

__global__ __launch_bounds__(kThreads) void sampling_list_kernel(const TopKPParams p, const unsigned long long* hist, int slice, DrawRow* rows, unsigned long long* above, uint2* list) {
    __shared__ DrawScan sc;
    __shared__ unsigned long long s_mass, s_above;
    __shared__ uint32_t s_over;
    __shared__ int s_n, s_base, s_at;
    const int row = blockIdx.y, S = gridDim.x, tx = threadIdx.x, lane = tx & 63, wave = tx >> 6;
    const DrawFilter f = draw_filter(p, row);
    const unsigned long long* hr = hist + (size_t)row * S * kDrawBins;
    if (hr[0]) {
        if (blockIdx.x == 0 && tx == 0) rows[row] = DrawRow{-1, 0u, 0u, 0ull};
        return;
    }
    if (tx == 0) { s_n = -1; s_base = 0; s_at = 0; s_above = 0; }
    uint32_t c = 0, ci;
    unsigned long long m = 0, mi, own = 0;                                      // the row's bin, what of its mass lies in this slice
    bool of_p;
    const int bin = kDrawBins - 1 - tx;
    if (bin > 0) {
        unsigned long long h = 0;
#pragma unroll 4
        for (int s = 0; s < S; ++s) h += hr[s * kDrawBins + bin];
        c = (uint32_t)(h >> 40);
        m = draw_mass((uint32_t)(bin + kDrawBase), c, h & ((1ull << 40) - 1ull));
        h = hr[blockIdx.x * kDrawBins + bin];
        own = draw_mass((uint32_t)(bin + kDrawBase), (uint32_t)(h >> 40), h & ((1ull << 40) - 1ull));
    }
    const bool negative = f.use_p && !(f.tp >= 0.f);
    const int low = draw_cross(f, f.use_p && !negative ? draw_limit(f.tp) : 0ull, bin > 0 ? bin : -1, c, m, 0u, 0ull, ci, mi, of_p, sc);
    if (bin == low && low > 0 && !negative && c <= (uint32_t)kList) { s_n = (int)c; s_over = ci - c; s_mass = mi - m; }
    if (low > 0) {
        own = wave_sum_u64(bin > low ? own : 0ull);
        if (lane == 0 && own) atomicAdd(&s_above, own);
    }
    for (int s = wave; s < (int)blockIdx.x; s += kWaves)                        // where the slice's part of the list begins
        if (lane == 0 && low > 0) atomicAdd(&s_base, (int)(hr[s * kDrawBins + low] >> 40));
    __syncthreads();
    if (tx == 0) {
        if (blockIdx.x == 0) rows[row] = DrawRow{s_n, (uint32_t)(max(low, 0) + kDrawBase), s_over, s_mass};
        above[(size_t)row * S + blockIdx.x] = s_above;
    }
    if (s_n < 0) return;
    uint2* out = list + (size_t)row * draw_list(p.V) + s_base;
    const int lo = min(p.V, (int)blockIdx.x * slice), n = min(p.V, lo + slice) - lo;
    const float* x = p.probs + (size_t)row * p.ld + lo;
    const float least = __uint_as_float((uint32_t)(low + kDrawBase) << kDrawShift), next = __uint_as_float((uint32_t)(low + 1 + kDrawBase) << kDrawShift);
    auto take = [&](float v, int j) {
        if (v >= least && (v < next || low == kDrawBins - 1)) out[atomicAdd(&s_at, 1)] = make_uint2(__float_as_uint(v), (uint32_t)(lo + j));
    };
    int done = 0;
    if ((p.ld & 3) == 0 && (reinterpret_cast<uintptr_t>(p.probs) & 15) == 0) {
        const f32x4* x4 = reinterpret_cast<const f32x4*>(x);
#pragma unroll 4
        for (int j = tx; j < n >> 2; j += kThreads) {
            const f32x4 v = x4[j];
            take(v[0], 4 * j); take(v[1], 4 * j + 1); take(v[2], 4 * j + 2); take(v[3], 4 * j + 3);
        }
        done = n & ~3;
    }
    for (int j = done + tx; j < n; j += kThreads) take(x[j], j);
}

__global__ __launch_bounds__(kThreads) void draw_listed_kernel(const TopKPParams p, int S, int slice, const DrawRow* rows, const unsigned long long* above, const uint2* list) {
    __shared__ SampleShared sh;
    __shared__ DrawScan sc;
    __shared__ unsigned long long s_slice[kMostSplits], s_over;
    __shared__ uint32_t s_ties, s_stay;
    const int row = blockIdx.x, tx = threadIdx.x, lane = tx & 63, wave = tx >> 6;
    const DrawRow r = rows[row];
    if (r.n < 0) { sample_row(p, row, sh); return; }
    const DrawFilter f = draw_filter(p, row);
    const unsigned long long limit = f.use_p ? draw_limit(f.tp) : 0ull;
    constexpr int PT = kList / kThreads, REST = 9;                              // values of a thread; bits behind the first 10 of the 19 that the list's values differ in
    uint2 e[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) e[i] = tx + i * kThreads < r.n ? list[(size_t)row * draw_list(p.V) + tx + i * kThreads] : make_uint2(0u, 0u);
    sh.hist[tx] = 0ull; sh.hist[kThreads + tx] = 0ull;
    if (tx < S) s_slice[tx] = above[(size_t)row * S + tx];
    __syncthreads();
    constexpr uint32_t LOW = (1u << kDrawShift) - 1u;
#pragma unroll
    for (int i = 0; i < PT; ++i)
        if (e[i].x) atomicAdd(&sh.hist[(e[i].x & LOW) >> REST], (1ull << 40) + (unsigned long long)(e[i].x & LOW));
    __syncthreads();
    uint32_t ci;
    unsigned long long mi;
    bool of_p;
    unsigned long long h = sh.hist[kThreads - 1 - tx];
    uint32_t c = (uint32_t)(h >> 40);
    unsigned long long m = draw_mass(r.low, c, h & ((1ull << 40) - 1ull));
    const int first = draw_cross(f, limit, kThreads - 1 - tx, c, m, r.above, r.mass, ci, mi, of_p, sc);
    if (kThreads - 1 - tx == first) { s_ties = ci - c; s_over = mi - m; }       // counted so far, and their mass
    __syncthreads();
    const uint32_t c1 = s_ties;
    const unsigned long long m1 = s_over;
#pragma unroll
    for (int i = 0; i < PT; ++i)
        if (e[i].x && (int)((e[i].x & LOW) >> REST) == first) atomicAdd(&sh.hist[kThreads + (e[i].x & ((1u << REST) - 1u))], 1ull);
    __syncthreads();
    const int bin = (1 << REST) - 1 - tx;
    c = bin >= 0 ? (uint32_t)sh.hist[kThreads + bin] : 0u;
    const uint32_t mine = r.low << kDrawShift | (uint32_t)(first << REST) | (uint32_t)max(bin, 0);      // the bits of the bin's value
    m = c * draw_fixed(mine);
    const int last = draw_cross(f, limit, bin, c, m, c1, m1, ci, mi, of_p, sc);
    if (bin == last) {                                                          // equals of the boundary value: the j-th stays while S + j v <= p, S = the mass above it
        s_ties = c;
        s_stay = of_p ? (uint32_t)min((unsigned long long)c, (limit - (mi - m)) / draw_fixed(mine) + 1ull) : c;
    }
    __syncthreads();
    const uint32_t bound = r.low << kDrawShift | (uint32_t)(first << REST) | (uint32_t)last, ties = s_ties, stay = s_stay;
    uint32_t cut = (uint32_t)p.V;                                               // equals from this index on go
    if (stay < ties) {                                                          // the largest index with at most `stay` of them in front of it
        cut = 0;
        for (int bit = 31 - __clz(p.V); bit >= 0; --bit) {
            const uint32_t at = cut | 1u << bit;
            uint32_t before = 0;
#pragma unroll
            for (int i = 0; i < PT; ++i) before += (uint32_t)__popcll(__ballot(e[i].x == bound && e[i].y < at));
            if (lane == 0) sc.c[wave] = before;
            __syncthreads();
            before = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) before += sc.c[w];
            __syncthreads();
            if (before <= stay) cut = at;
        }
    }
#pragma unroll
    for (int i = 0; i < PT; ++i)
        if (e[i].x && (e[i].x > bound || (e[i].x == bound && e[i].y < cut))) atomicAdd(&s_slice[e[i].y / (uint32_t)slice], draw_fixed(e[i].x));
    __syncthreads();
    unsigned long long total = 0, front = 0;                                    // mass in front of the slice with the draw
    for (int s = 0; s < S; ++s) total += s_slice[s];
    const double u = (double)p.uniform[row] * (double)total;
    int hit = 0;
    while (hit < S && !((double)(front + s_slice[hit]) > u)) front += s_slice[hit++];
    if (hit == S || !(u >= 0.0)) {
        if (tx == 0) p.ids[row] = p.V - 1;
        return;
    }
    // the slice: a contiguous run of it a thread, the runs' masses, their prefix, the run that u lies in
    const int lo = hit * slice, end = min(p.V, lo + slice), run = ((slice / 4 + kThreads - 1) / kThreads) * 4, j0 = min(end, lo + tx * run), j1 = min(end, j0 + run);
    const float* q = p.probs + (size_t)row * p.ld;
    auto weight = [&](float v, int j) -> unsigned long long {
        const uint32_t b = v > 0.f ? __float_as_uint(v) : 0u;
        return b > bound || (b == bound && (uint32_t)j < cut) ? draw_fixed(b) : 0ull;
    };
    unsigned long long sum = 0;
    int j = j0;
    if ((p.ld & 3) == 0 && (reinterpret_cast<uintptr_t>(p.probs) & 15) == 0) {
#pragma unroll 4
        for (; j + 3 < j1; j += 4) {
            const f32x4 v = *reinterpret_cast<const f32x4*>(q + j);
            sum += (weight(v[0], j) + weight(v[1], j + 1)) + (weight(v[2], j + 2) + weight(v[3], j + 3));
        }
    }
    for (; j < j1; ++j) sum += weight(q[j], j);
    unsigned long long incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long y = __shfl_up(incl, o);
        if (lane >= o) incl += y;
    }
    if (lane == 63) sc.m[wave] = incl;
    __syncthreads();
    for (int w = 0; w < wave; ++w) incl += sc.m[w];
    incl += front;
    if (sum && !((double)(incl - sum) > u) && (double)incl > u) {
        unsigned long long at = incl - sum;
        for (j = j0; j < j1; ++j) {
            at += weight(q[j], j);
            if ((double)at > u) { p.ids[row] = j; break; }
        }
    }
}


// ids[r] = inverse-CDF sample of probs[r, :] with uniform[r] (the top_k = 0 / top_p = 1 branch of the sampler:
// softmax, then sampling from the probabilities, bindings/core/CudaSampleOp.cc:702-737)
__global__ __launch_bounds__(kThreads) void sample_rows_kernel(const float* __restrict__ probs, int V, int ld,
                                                               const float* __restrict__ uniform, int32_t* __restrict__ ids) {
    __shared__ DrawShared sh;
    row_draw(probs + (size_t)blockIdx.x * ld, V, uniform[blockIdx.x], sh, [](float v) { return fmaxf(v, 0.f); });
    if (threadIdx.x == 0) ids[blockIdx.x] = sh.found;
}

// no_repeat_ngram_size: ban_repeat_ngram (bindings/common/kernels/banRepeatNgram.cu:30-136, greedy case beam_width = 1; called from
// CudaSampleOp.cc:242-283).  With N = last_index[row] + 1 tokens so far and n = ngram[row]: every position i <= N - n whose n - 1
// tokens equal the last n - 1 tokens of the sequence bans the token that followed it there (logit = -inf), so that no n-gram of
// the sequence can be produced a second time.  n == 0 or N < n: nothing.  One block per row; the history is read from global
// memory (N n int32 reads per row: nothing next to the vocabulary row the sampler touches anyway).
__global__ __launch_bounds__(256) void ban_repeat_ngram_kernel(float* __restrict__ logits, int V, int ld, const int32_t* __restrict__ token_ids,
                                                               int token_ld, const int32_t* __restrict__ last_index,
                                                               const int32_t* __restrict__ ngram) {
    const int row = blockIdx.x;
    const int n = ngram[row], N = last_index[row] + 1;
    if (n <= 0 || N < n || N > token_ld) return;
    const int32_t* tok = token_ids + (size_t)row * token_ld;
    const int32_t* last = tok + (N - n + 1);                // the n - 1 most recent tokens
    for (int i = threadIdx.x; i <= N - n; i += 256) {
        bool match = true;
        for (int k = 0; k < n - 1; ++k)
            if (tok[i + k] != last[k]) { match = false; break; }
        if (!match) continue;
        const int banned = tok[i + n - 1];
        if (banned >= 0 && banned < V) logits[(size_t)row * ld + banned] = -INFINITY;
    }
}

} // namespace

extern "C" int mi355_sample_rows(const float* probs, int32_t rows, int32_t V, int32_t ld, const float* uniform_samples,
                                 int32_t* ids, mi355_stream_t stream) {
    MI355_CHECK_ARG(probs && uniform_samples && ids && rows > 0 && V > 0 && ld >= V, "sample_rows: bad args");
    hipLaunchKernelGGL(sample_rows_kernel, dim3(rows), dim3(kThreads), 0, (hipStream_t)stream, probs, V, ld, uniform_samples, ids);
    MI355_CHECK_LAUNCH("sample_rows_kernel");
    return MI355_OK;
}

extern "C" int mi355_softmax_rows(const float* logits, int32_t rows, int32_t V, int32_t ld, float temperature, float* probs,
                                  mi355_stream_t stream) {
    MI355_CHECK_ARG(logits && probs && rows > 0 && V > 0 && ld >= V && temperature > 0.f, "softmax_rows: bad args");
    if (V % 4 == 0 && ld % 4 == 0 && ((uintptr_t)logits | (uintptr_t)probs) % 16 == 0)
        hipLaunchKernelGGL(softmax_rows_kernel<true>, dim3(rows), dim3(kThreads), 0, (hipStream_t)stream, logits, V, ld, 1.f / temperature, probs);
    else
        hipLaunchKernelGGL(softmax_rows_kernel<false>, dim3(rows), dim3(kThreads), 0, (hipStream_t)stream, logits, V, ld, 1.f / temperature, probs);
    MI355_CHECK_LAUNCH("softmax_rows_kernel");
    return MI355_OK;
}

extern "C" int mi355_rejection_sample(const float* draft_probs, const int32_t* draft_token_ids, const float* uniform_samples,
                                      const float* target_probs, const int32_t* target_token_ids, int32_t target_token_stride,
                                      int32_t* output_token_ids, int32_t* output_accepted_token_num, const uint8_t* do_sample,
                                      int32_t batch_size, int32_t num_speculative_tokens, int32_t vocab_size,
                                      int32_t draft_probs_point_mass, mi355_stream_t stream) {
    if (batch_size == 0) return MI355_OK; // as invokeRejectionSampling (sampling.cu:491-493)
    MI355_CHECK_ARG(draft_token_ids && uniform_samples && target_probs && target_token_ids && output_token_ids &&
                        output_accepted_token_num && do_sample,
                    "rejection_sample: null pointer");
    MI355_CHECK_ARG(draft_probs || draft_probs_point_mass, "rejection_sample: draft_probs missing (and not point-mass)");
    MI355_CHECK_ARG(batch_size > 0 && num_speculative_tokens > 0 && vocab_size > 0 && target_token_stride > 0,
                    "rejection_sample: batch=%d gamma=%d vocab=%d stride=%d", batch_size, num_speculative_tokens, vocab_size,
                    target_token_stride);
    RejectParams p{draft_probs, draft_token_ids, uniform_samples, target_probs, target_token_ids, target_token_stride,
                   output_token_ids, output_accepted_token_num, do_sample, batch_size, num_speculative_tokens, vocab_size,
                   draft_probs_point_mass ? 1 : 0};
    hipLaunchKernelGGL(rejection_sample_kernel, dim3(batch_size), dim3(kThreads), 0, (hipStream_t)stream, p);
    MI355_CHECK_LAUNCH("rejection_sample_kernel");
    return MI355_OK;
}

// Blocks of a row: about one block per compute unit in all, none with less than a pass of its threads.  Temperature alone, us with 1 / 2 / 4 / 8 / 16 blocks a row:
// 1 x 152064 11.9 / 6.6 / 4.3 / 3.2 / 2.7, 64 x 152064 18.3 / 12.5 / 11.6 / 12.2 / 12.4, 64 x 6952 2.8 / 2.8 / 2.9 / 3.6 / 4.5, 237 x 32000 8.3 / 8.2 / 8.8 / 9.6 / 13.1.
static int row_splits(int rows, int V) {
    const int most = rows >= 256 ? 1 : 256 / rows < kMostSplits ? 256 / rows : kMostSplits, full = (V + 4 * kThreads - 1) / (4 * kThreads);
    return most < full ? most : full;
}
// The joint launches: of long rows as many blocks as hold their slices in registers.  64 x 152064, us of prepare, probabilities and list with 8 blocks a row (one round of two a compute
// unit) 21.8 + 12.7 + 12.9, with 9 24.2 + 14.8 + 14.3; with 4, walked from memory, the first two took 31.7 before against 28.1 with 9.
static int held_splits(int V) { const int held = (V + kHeld - 1) / kHeld; return held < kMostSplits ? held : kMostSplits; }
static int joint_splits(int rows, int V) {
    const int least = row_splits(rows, V), near = held_splits(V);
    return least > near ? least : near;
}

extern "C" int mi355_apply_penalties(float* logits, int32_t batch_size, int32_t V, int32_t ld, const float* temperature,
                                     const float* repetition_penalty, const float* presence_penalty, const float* frequency_penalty,
                                     const int32_t* output_ids, const int32_t* input_lengths, int32_t max_input_length,
                                     int32_t step, int32_t* penalty_ws, mi355_stream_t stream) {
    if (batch_size == 0) return MI355_OK;
    MI355_CHECK_ARG(logits && batch_size > 0 && V > 0 && ld >= V, "apply_penalties: bad args");
    const bool pen = repetition_penalty || presence_penalty || frequency_penalty;
    MI355_CHECK_ARG(!pen || (output_ids && penalty_ws && step >= 0 && max_input_length >= 0),
                    "apply_penalties: penalties need output_ids [step][batch] and a [batch][V] int32 workspace");
    if (!pen && !temperature) return MI355_OK;
    PenaltyParams p{logits, V, ld, temperature, repetition_penalty, presence_penalty, frequency_penalty,
                    pen ? output_ids : nullptr, input_lengths, batch_size, max_input_length, step, penalty_ws};
    hipStream_t st = (hipStream_t)stream;
    if (temperature) {
        const int split = row_splits(batch_size, V);
        if (split > 1) hipLaunchKernelGGL(temperature_kernel<false>, dim3(split, batch_size), dim3(kThreads), 0, st, p);
        else           hipLaunchKernelGGL(temperature_kernel<true>, dim3(batch_size), dim3(kThreads), 0, st, p);
        MI355_CHECK_LAUNCH("temperature_kernel");
    }
    if (pen && step > kShortHistory) {
        const size_t n = (size_t)batch_size * V;
        hipLaunchKernelGGL(clear_counts_kernel, dim3((unsigned)(n / (16 * kThreads) < 1024 ? n / (16 * kThreads) + 1 : 1024)), dim3(kThreads), 0, st, penalty_ws, n);
        MI355_CHECK_LAUNCH("clear_counts_kernel");
        hipLaunchKernelGGL(penalties_kernel, dim3(batch_size), dim3(kThreads), 0, st, p);
        MI355_CHECK_LAUNCH("penalties_kernel");
    } else if (pen && step > 0) {
        if (step <= 256) hipLaunchKernelGGL(penalties_short_kernel<256>, dim3(batch_size), dim3(256), 0, st, p);
        else             hipLaunchKernelGGL(penalties_short_kernel<kThreads>, dim3(batch_size), dim3(kThreads), 0, st, p);
        MI355_CHECK_LAUNCH("penalties_short_kernel");
    }
    return MI355_OK;
}

namespace {
template <bool HIST>
int launch_probs(const PenaltyParams& p, void* parts, int id_step, int id_row, int S, int slice, unsigned long long* hist, hipStream_t st) {
    const dim3 grid(S, p.batch), block(kThreads);
    const bool held = slice <= kHeld && p.ld % 4 == 0 && (uintptr_t)p.logits % 16 == 0;
    if (held) hipLaunchKernelGGL(sampling_prepare_kernel<true>, grid, block, 0, st, p, (float2*)parts, id_step, id_row, slice);
    else      hipLaunchKernelGGL(sampling_prepare_kernel<false>, grid, block, 0, st, p, (float2*)parts, id_step, id_row, slice);
    MI355_CHECK_LAUNCH("sampling_prepare_kernel");
    hipLaunchKernelGGL(sampling_probs_kernel<HIST>, grid, block, 0, st, p.logits, p.V, p.ld, (const float2*)parts, slice, hist);
    MI355_CHECK_LAUNCH("sampling_probs_kernel");
    return MI355_OK;
}
} // namespace

extern "C" size_t mi355_sampling_probs_workspace_bytes(int32_t rows) { return rows > 0 ? (size_t)rows * kMostSplits * sizeof(float2) : 0; }

extern "C" int mi355_sampling_probs(float* logits, int32_t rows, int32_t V, int32_t ld, const float* temperature, const float* repetition, const float* presence,
                                    const float* frequency, const int32_t* output_ids, int32_t id_step, int32_t id_row, const int32_t* input_lengths, int32_t max_input_length,
                                    int32_t step, void* workspace, mi355_stream_t stream) {
    MI355_CHECK_ARG(logits && workspace && rows > 0 && V > 0 && ld >= V && step >= 0 && (uintptr_t)workspace % 8 == 0, "sampling_probs: bad args");
    if (output_ids && step > kShortHistory) return MI355_ERR_UNSUPPORTED;      // apply_penalties counts those in memory
    const bool pen = output_ids && step > 0 && (repetition || presence || frequency);
    const int S = joint_splits(rows, V), slice = ((V + S - 1) / S + 3) & ~3;
    const PenaltyParams p{logits, V, ld, temperature, repetition, presence, frequency, pen ? output_ids : nullptr, input_lengths, rows, max_input_length, step, nullptr};
    return launch_probs<false>(p, workspace, id_step, id_row, S, slice, nullptr, (hipStream_t)stream);
}

// mi355_sampling_probs and mi355_top_k_top_p_sample (without its probabilities) in one: the logits become the probabilities, ids[row] is drawn from what the filter leaves.
namespace {
struct DrawWorkspace { size_t hist, above, list, listed, bytes; };                     // the slices' (maximum, sum) lie in front
constexpr int kDrawRows = 1024;                                                       // rows of a round of launches: four blocks a compute unit and more, at most 130 MB
DrawWorkspace draw_workspace(int rows, int V) {                                       // no smaller for more rows
    DrawWorkspace w;
    rows = rows < kDrawRows ? rows : kDrawRows;
    const int most = rows * held_splits(V) > 256 ? rows * held_splits(V) : 256, slices = rows * kMostSplits < most ? rows * kMostSplits : most;         // rows * joint_splits at most
    w.hist = ((size_t)rows * kMostSplits * sizeof(float2) + 15) & ~(size_t)15;
    w.above = w.hist + (size_t)slices * kDrawBins * sizeof(unsigned long long);
    w.list = w.above + (size_t)slices * sizeof(unsigned long long);
    w.listed = w.list + (size_t)rows * draw_list(V) * sizeof(uint2);
    w.bytes = w.listed + (size_t)rows * sizeof(DrawRow);
    return w;
}
} // namespace
extern "C" size_t mi355_sampling_draw_workspace_bytes(int32_t rows, int32_t V) { return rows > 0 && V > 0 ? draw_workspace(rows, V).bytes : 0; }

extern "C" int mi355_sampling_draw(float* logits, int32_t rows, int32_t V, int32_t ld, const float* temperature, const float* repetition, const float* presence,
                                   const float* frequency, const int32_t* output_ids, int32_t id_step, int32_t id_row, const int32_t* input_lengths, int32_t max_input_length,
                                   int32_t step, const int32_t* top_k, const float* top_p, const float* uniform_samples, int32_t* ids, void* workspace, mi355_stream_t stream) {
    MI355_CHECK_ARG(logits && workspace && rows > 0 && V > 0 && ld >= V && step >= 0 && (uintptr_t)workspace % 16 == 0 && uniform_samples && ids, "sampling_draw: bad args");
    if (V > 1 << 20) {                                                          // the packed sums of a bin
        if (int e = mi355_sampling_probs(logits, rows, V, ld, temperature, repetition, presence, frequency, output_ids, id_step, id_row, input_lengths, max_input_length, step, workspace, stream)) return e;
        return mi355_top_k_top_p_sample(logits, rows, V, ld, top_k, top_p, uniform_samples, ids, nullptr, 0, stream);
    }
    if (output_ids && step > kShortHistory) return MI355_ERR_UNSUPPORTED;
    const bool pen = output_ids && step > 0 && (repetition || presence || frequency);
    const int S = joint_splits(rows, V), slice = ((V + S - 1) / S + 3) & ~3;
    const DrawWorkspace w = draw_workspace(rows, V);
    char* ws = (char*)workspace;
    hipStream_t st = (hipStream_t)stream;
    for (int r0 = 0; r0 < rows; r0 += kDrawRows) {
        const int n = rows - r0 < kDrawRows ? rows - r0 : kDrawRows;
        auto from = [r0](auto* v) { return v ? v + r0 : v; };
        float* x = logits + (size_t)r0 * ld;
        const PenaltyParams p{x, V, ld, from(temperature), from(repetition), from(presence), from(frequency), pen ? output_ids + (size_t)r0 * id_row : nullptr, from(input_lengths), n,
                              max_input_length, step, nullptr};
        if (int e = launch_probs<true>(p, workspace, id_step, id_row, S, slice, (unsigned long long*)(ws + w.hist), st)) return e;
        const TopKPParams t{x, V, ld, from(top_k), from(top_p), uniform_samples + r0, ids + r0, nullptr, 0};
        auto* above = (unsigned long long*)(ws + w.above);
        hipLaunchKernelGGL(sampling_list_kernel, dim3(S, n), dim3(kThreads), 0, st, t, (const unsigned long long*)(ws + w.hist), slice, (DrawRow*)(ws + w.listed), above, (uint2*)(ws + w.list));
        MI355_CHECK_LAUNCH("sampling_list_kernel");
        hipLaunchKernelGGL(draw_listed_kernel, dim3(n), dim3(kThreads), 0, st, t, S, slice, (const DrawRow*)(ws + w.listed), above, (const uint2*)(ws + w.list));
        MI355_CHECK_LAUNCH("draw_listed_kernel");
    }
    return MI355_OK;
}

// The host's part of a step in one place: of 184 us for 64 rows of 152064 values 110 were Python looking at the vectors and packing them, a copy from pageable memory and one back (108 us now).
namespace {
struct Filters { bool greedy, some; };
Filters filters(const int32_t* top_k, const float* top_p, int rows, int V) {
    bool greedy = true, some_k = false, some_p = false;
    for (int r = 0; r < rows; ++r) {
        greedy = greedy && top_k[r] == 1;
        some_k = some_k || (top_k[r] > 0 && top_k[r] < V);
        some_p = some_p || (top_p[r] != 1.f && !(fabsf(top_p[r]) < 1e-7f));
    }
    return {greedy, some_k || some_p};
}
struct HostLook { bool takes, scale, pen; };
HostLook look(const mi355_sampler_host_t& h, int rows, int V) {
    const Filters f = filters(h.top_k, h.top_p, rows, V);
    bool scale = false, pen = false;
    for (int r = 0; r < rows; ++r) {
        scale = scale || h.temperature[r] != 1.f;
        if (h.repetition) pen = pen || h.repetition[r] != 1.f || h.presence[r] != 0.f || h.frequency[r] != 0.f;
    }
    return {!f.greedy && f.some && h.step < kShortHistory && rows <= 65535, scale, pen};
}
} // namespace

// bit 0: every row greedy (top_k 1); bit 1: some row has a filter.  Of 110 us of Python for a step that this file does not take, looking at the vectors for it was 4 to 8.
extern "C" int mi355_sampler_filters(const int32_t* top_k, const float* top_p, int32_t rows, int32_t V) {
    if (!top_k || !top_p || rows <= 0) return 1;
    const Filters f = filters(top_k, top_p, rows, V);
    return f.greedy | f.some << 1;
}
extern "C" size_t mi355_sampler_step_stage_bytes(int32_t rows, int32_t step) { return rows > 0 && step >= 0 ? (size_t)rows * ((size_t)step + 10) * 4 : 0; }
extern "C" int mi355_sampler_step_takes(const mi355_sampler_host_t* host, int32_t rows, int32_t V) {
    return host && host->temperature && host->top_k && host->top_p && rows > 0 && host->step >= 0 && !host->repetition == !host->presence && !host->repetition == !host->frequency &&
           look(*host, rows, V).takes;
}

extern "C" int mi355_sampler_step(float* logits, int32_t rows, int32_t V, int32_t ld, const mi355_sampler_host_t* host, void* pinned, void* device, int32_t* ids, void* workspace,
                                  mi355_stream_t stream) {
    MI355_CHECK_ARG(logits && host && pinned && device && ids && workspace && rows > 0 && V > 0 && ld >= V, "sampler_step: bad args");
    const mi355_sampler_host_t& h = *host;
    MI355_CHECK_ARG(h.temperature && h.top_k && h.top_p && h.uniform && h.token_ids && h.step >= 0 && !h.repetition == !h.presence && !h.repetition == !h.frequency &&
                    (!h.repetition || (h.input_lengths && h.n_sequences >= 0 && h.n_sequences <= rows && (h.n_sequences == 0 || h.sequence_lengths))), "sampler_step: bad vectors");
    const HostLook seen = look(h, rows, V);
    if (!seen.takes) return MI355_ERR_UNSUPPORTED;
    int32_t* at = (int32_t*)pinned;
    auto put = [&](const void* v, size_t n) {                                   // -> where it will be on the device
        void* there = (char*)device + ((char*)at - (char*)pinned);
        memcpy(at, v, n * 4);
        at += n;
        return there;
    };
    const float* temperature = seen.scale ? (const float*)put(h.temperature, rows) : nullptr;
    const float *rep = nullptr, *pres = nullptr, *freq = nullptr;
    const int32_t *lengths = nullptr, *history = nullptr;
    if (seen.pen) {
        rep = (const float*)put(h.repetition, rows); pres = (const float*)put(h.presence, rows); freq = (const float*)put(h.frequency, rows);
        int32_t* first = at;
        lengths = (const int32_t*)put(h.input_lengths, rows);
        if (h.n_sequences > 0) memcpy(first, h.sequence_lengths, (size_t)h.n_sequences * 4);
        history = (const int32_t*)put(h.token_ids, (size_t)rows * (h.step + 1));
    }
    const int32_t* top_k = (const int32_t*)put(h.top_k, rows);
    float* p = (float*)at;
    const float* top_p = (const float*)put(h.top_p, rows);
    for (int r = 0; r < rows; ++r) if (fabsf(p[r]) < 1e-7f) p[r] = 1.f;
    const float* uniform = (const float*)put(h.uniform, rows);
    int32_t* back = at;                                                         // the ids land behind what is sent
    hipStream_t st = (hipStream_t)stream;
    int rc = MI355_ERR_HIP;
    hipError_t e = hipMemcpyAsync(device, pinned, (char*)at - (char*)pinned, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) {
        rc = mi355_sampling_draw(logits, rows, V, ld, temperature, rep, pres, freq, history, 1, h.step + 1, lengths, h.step + 1, h.step + 1, top_k, top_p, uniform, ids, workspace, stream);
        if (rc == MI355_OK) e = hipMemcpyAsync(back, ids, (size_t)rows * 4, hipMemcpyDeviceToHost, st);
    }
    const hipError_t done = hipStreamSynchronize(st);                           // also after an error: the caller's buffers are free again
    if (e == hipSuccess) e = done;
    if (e != hipSuccess) { mi355_set_error("sampler_step: %s", hipGetErrorString(e)); return MI355_ERR_HIP; }
    if (rc != MI355_OK) return rc;
    for (int r = 0; r < rows; ++r) h.token_ids[(size_t)r * (h.step + 1) + h.step] = back[r];
    return MI355_OK;
}

extern "C" int mi355_top_k_top_p_sample(const float* probs, int32_t rows, int32_t V, int32_t ld, const int32_t* top_k,
                                        const float* top_p, const float* uniform_samples, int32_t* ids, float* probs_out,
                                        int32_t ld_out, mi355_stream_t stream) {
    if (rows == 0) return MI355_OK;
    MI355_CHECK_ARG(probs && uniform_samples && ids && rows > 0 && V > 0 && ld >= V, "top_k_top_p_sample: bad args");
    MI355_CHECK_ARG(!probs_out || ld_out >= V, "top_k_top_p_sample: ld_out %d < V %d", ld_out, V);
    TopKPParams p{probs, V, ld, top_k, top_p, uniform_samples, ids, probs_out, ld_out};
    hipLaunchKernelGGL(top_k_top_p_sample_kernel, dim3(rows), dim3(kThreads), 0, (hipStream_t)stream, p);
    MI355_CHECK_LAUNCH("top_k_top_p_sample_kernel");
    return MI355_OK;
}

extern "C" int mi355_ban_repeat_ngram(float* logits, int32_t batch_size, int32_t V, int32_t ld, const int32_t* token_ids,
                                      int32_t token_ld, const int32_t* sequence_last_index, const int32_t* no_repeat_ngram_size,
                                      mi355_stream_t stream) {
    if (batch_size == 0) return MI355_OK;
    MI355_CHECK_ARG(logits && token_ids && sequence_last_index && no_repeat_ngram_size && batch_size > 0 && V > 0 && ld >= V && token_ld > 0,
                    "ban_repeat_ngram: bad args");
    hipLaunchKernelGGL(ban_repeat_ngram_kernel, dim3(batch_size), dim3(256), 0, (hipStream_t)stream, logits, V, ld, token_ids, token_ld,
                       sequence_last_index, no_repeat_ngram_size);
    MI355_CHECK_LAUNCH("ban_repeat_ngram_kernel");
    return MI355_OK;
}
