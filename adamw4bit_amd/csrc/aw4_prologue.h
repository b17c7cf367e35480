// The step's prologue: the global gradient norm and clipping coefficient of
// torch.nn.utils.clip_grad_norm_ (norm type 2), which the reference's training examples
// run before every step (an HF Trainer with max_grad_norm=1.0,
// examples/train_gpt_small.py:214), optionally of the gradients GradScaler.unscale_ would leave
// (the loss scale's inverse applied in the same read).  One pass over the gradients: each
// workgroup sums the squares of one segment of one gradient in float64; the last workgroup of a
// gradient then combines its segments, and the last of all adds the per-gradient squares, both in a
// fixed order, with torch's rounding points (clip_grad.py _get_total_norm /
// _clip_grads_with_norm_):
//   g'     = grad_dtype(fp32(g * u))                   (unscaling: _amp_foreach_non_finite_check_and_unscale_)
//   norm_t = grad_dtype(fp32(sqrt(sum of g'^2)))       (torch._foreach_norm)
//   total  = R(fp32(sqrt(sum_t norm_t^2)))             (vector_norm of the stacked norms)
//   coef   = min(R(R(1 / R(total + 1e-6)) * max_norm), 1)
// with R the promotion of the gradient dtypes and every operation in fp32 rounded to R; with
// unscaling, found_inf = 1 if any g (the scaled value, as torch checks it) is not finite.  The
// unscaling and the coefficient are applied by the step itself (AW4_TENSOR_GRAD_UNSCALE,
// AW4_TENSOR_GRAD_SCALE), so neither the unscaled nor the clipped gradients are written.
#pragma once

#include "aw4_step.h"

namespace aw4 {

constexpr int kNormThreads = 256;
// Gradient values per workgroup of the norm pass: 2^13 (one batch of eight vector loads per thread) to
// 2^18, the host's choice by the total (norm_segment_shift).
constexpr int kNormShiftMin = 13, kNormShiftMax = 18;

// One gradient of the pass (24 bytes: the rows of 156 gradients fit a launch's arguments).
struct NormRow {
    uint64_t grad;      // device address
    int64_t numel;
    int32_t seg_start;  // first of its segments
    int32_t dtype;      // AW4_* of the gradient, with kNormVec where 4-value vector access is allowed and
                        // kNormKeep where the loads go through the caches
};
constexpr int kNormVec = 0x100, kNormKeep = 0x200;

struct NormHeader {
    int32_t count;
    int32_t result_dtype;  // R
    float max_norm;
    int32_t unscale;       // nonzero: unscale by *inv_scale, and report found_inf
    int32_t total_segments;
    int32_t segment_shift;
    uint64_t partials;     // device address, double[total_segments]
    uint64_t norm_sq;      // device address, double[count]: norm_t^2 of each gradient
    uint64_t tickets;      // device address, the gradients' tickets and the launch's (norm_ticket_words), zero
                           // before and after the launch
    uint64_t groups;       // device address, the segment groups' (norm_group_words), likewise
    uint64_t norm_out;     // device address, float
    uint64_t coef_out;     // device address, float
    uint64_t inv_scale;    // device address, float u (unscale)
    uint64_t nonfinite;    // device address, uint32[total_segments]: a segment holds a non-finite g (unscale)
    uint64_t found_out;    // device address, float found_inf (unscale)
};
// followed by NormRow rows[count]

// Every ticket is in a cache line of its own, and whoever draws a ticket's last number clears it: atomics on one
// line follow one another at about 14 ns, and a launch's workgroups finish together (2 GB in 64 fp32 gradients of
// 32 segments: 357 us with their tickets in two lines).  For the same reason a gradient of more than kNormGroup
// segments counts them in two levels, a ticket for each aligned run of kNormGroup segments (the gradient's part
// of it) and the gradient's for its runs.  A run holds parts of at most two such gradients, one that starts in
// it and one before: two tickets each.
constexpr int kNormGroup = 32, kNormTicketStride = 32;
__host__ __device__ constexpr int64_t norm_ticket_words(int64_t gradients) { return kNormTicketStride * (gradients + 1); }
__host__ __device__ constexpr int64_t norm_group_words(int64_t segments) {
    return 2 * kNormTicketStride * (segments / kNormGroup + 1);
}
// Finished gradients likewise, from kNormManyGradients on: a ticket for each aligned run of kNormGroup of
// them, behind the segments' runs.  (From 64 on measured the same at 150 and 200 gradients, whose one counter
// is no longer than the further level's latency.)
constexpr int kNormManyGradients = 256;
__host__ __device__ constexpr int64_t norm_many_words(int64_t gradients) {
    return gradients < kNormManyGradients ? 0 : kNormTicketStride * (gradients / kNormGroup + 1);
}

__device__ __forceinline__ double wave_sum_f64(double v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// One gradient value's contribution: its square, after unscaling (kUnscale: g' = G(fp32(g * u)),
// with a non-finite g recorded in `bad`, as torch checks the scaled value).
template <int G, bool kUnscale>
__device__ __forceinline__ double sq1(float f, float u, bool& bad) {
    if constexpr (kUnscale) {
        bad = bad | !__builtin_isfinite(f);
        f = round_to_dtype(f * u, G);
    }
    return (double)f * (double)f;
}

// Sum of squares of 4 consecutive gradient values starting at element e (all in range).
template <int G, bool kUnscale, bool kKeep>
__device__ __forceinline__ double sq4(uint64_t grad, int64_t e, bool vec, float u, bool& bad) {
    uint32_t w[4];
    float f[4];
    load_words<G, kKeep>(grad, e, vec, w);
    words_to_f32<G>(w, f);
    double s = 0.0;
#pragma unroll
    for (int t = 0; t < 4; ++t) s += sq1<G, kUnscale>(f[t], u, bad);
    return s;
}

template <int G, bool kUnscale, bool kKeep>
__device__ __forceinline__ double segment_sum(uint64_t grad, int64_t e0, int64_t e1, bool vec, float u,
                                              bool& bad) {
    // Full groups of 4 values: thread i takes groups i, i + 256, ... (8 loads in flight per
    // thread: 4 KB per workgroup per load instruction; 4 where fp16 values are unscaled, which with 8 took the
    // kernel from 44 to 69 VGPRs and an eighth workgroup from each CU).
    constexpr int kLoads = kUnscale && G == D_F16 ? 4 : 8;
    double acc = 0.0;
    const int64_t groups = (e1 - e0) >> 2;
    int64_t k = threadIdx.x;
    for (; k + (kLoads - 1) * kNormThreads < groups; k += kLoads * kNormThreads) {
        double s[kLoads];
#pragma unroll
        for (int v = 0; v < kLoads; ++v) s[v] = sq4<G, kUnscale, kKeep>(grad, e0 + 4 * (k + v * kNormThreads), vec, u, bad);
#pragma unroll
        for (int v = 0; v < kLoads; ++v) acc += s[v];
    }
    for (; k < groups; k += kNormThreads) acc += sq4<G, kUnscale, kKeep>(grad, e0 + 4 * k, vec, u, bad);
    // the tail of the tensor (fewer than 4 values)
    const int64_t tail = e0 + 4 * groups;
    if ((int64_t)threadIdx.x < e1 - tail) {
        float f;
        if (G == D_F32) f = gaddr<const float>(grad)[tail + threadIdx.x];
        else {
            const uint32_t h = gaddr<const uint16_t>(grad)[tail + threadIdx.x];
            f = G == D_BF16 ? bf16_to_f32(h) : f16_to_f32(h);
        }
        acc += sq1<G, kUnscale>(f, u, bad);
    }
    return acc;
}

template <bool kUnscale, bool kKeep>
__device__ __forceinline__ double segment_sum_any(uint64_t grad, int dtype, int64_t e0, int64_t e1, bool vec, float u,
                                                  bool& bad) {
    if (dtype == D_F32) return segment_sum<D_F32, kUnscale, kKeep>(grad, e0, e1, vec, u, bad);
    if (dtype == D_BF16) return segment_sum<D_BF16, kUnscale, kKeep>(grad, e0, e1, vec, u, bad);
    return segment_sum<D_F16, kUnscale, kKeep>(grad, e0, e1, vec, u, bad);
}

// What one workgroup leaves for another goes through device-scope atomic accesses only (the XCDs' L2
// caches are not coherent for plain ones within a launch): a store written through, complete when
// draw_last's wait returns, then the ticket, and loads past the caches by whoever drew the last one.
// A release and an acquire in their place would also write back and invalidate an L2 per workgroup, for
// plain stores that none of them reads: 195 us a pass more for GPT-2-small, after a step's dirty lines.
template <class T>
__device__ __forceinline__ T agent_load(gptr<T> p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void agent_store(gptr<T> p, T v) {
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Whether this was the last of `drawers` draws of a ticket, which it then leaves cleared.
__device__ __forceinline__ bool draw_last(gptr<uint32_t> p, uint32_t drawers) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // keeps the order in the compiler
    __builtin_amdgcn_s_waitcnt(0x0F70);                     // vmcnt(0): this thread's stores are complete
    const uint32_t drawn = __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (drawn != drawers - 1u) return false;
    agent_store(p, 0u);
    return true;
}

// Draws for one finished segment of gradient t (segments start .. end - 1); whether it was the gradient's last.
__device__ __forceinline__ bool norm_last_of_gradient(const NormHeader* hdr, int t, int seg, int start, int end) {
    uint32_t drawers = (uint32_t)(end - start);
    if (drawers == 1u) return true;
    if (drawers > (uint32_t)kNormGroup) {
        const int run = seg / kNormGroup, run0 = run * kNormGroup;
        const gptr<uint32_t> group =
            gaddr<uint32_t>(hdr->groups) + kNormTicketStride * (2 * (int64_t)run + (start > run0 ? 1 : 0));
        if (!draw_last(group, (uint32_t)(min(end, run0 + kNormGroup) - max(start, run0)))) return false;
        drawers = (uint32_t)((end - 1) / kNormGroup - start / kNormGroup + 1);
    }
    return draw_last(gaddr<uint32_t>(hdr->tickets) + kNormTicketStride * (int64_t)t, drawers);
}

// Draws for finished gradient t; whether it was the launch's last.
__device__ __forceinline__ bool norm_last_of_all(const NormHeader* hdr, int t, int count) {
    uint32_t drawers = (uint32_t)count;
    if (count >= kNormManyGradients) {
        const int run = t / kNormGroup, run0 = run * kNormGroup;
        const gptr<uint32_t> group =
            gaddr<uint32_t>(hdr->groups) + norm_group_words(hdr->total_segments) + kNormTicketStride * (int64_t)run;
        if (!draw_last(group, (uint32_t)(min(count, run0 + kNormGroup) - run0))) return false;
        drawers = (uint32_t)((count - 1) / kNormGroup + 1);
    }
    return draw_last(gaddr<uint32_t>(hdr->tickets) + kNormTicketStride * (int64_t)count, drawers);
}

// The index of the gradient that holds a segment.
__device__ __forceinline__ int norm_row_of(const NormRow* rows, int count, int seg) {
    int lo = 0, hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (rows[mid].seg_start <= seg) lo = mid; else hi = mid - 1;
    }
    return lo;
}

__device__ __forceinline__ double norm_sq_of(double s, int dtype) {
    const float norm_t = round_to_dtype((float)__builtin_sqrt(s), dtype);
    return (double)norm_t * (double)norm_t;  // exact
}

// norm_t^2 of one gradient from its segments' sums (lanes stride over them): wave 0 of its last workgroup.
__device__ __forceinline__ double norm_tensor_sq(const NormHeader* hdr, int first, int end, int dtype) {
    const gptr<double> partials = gaddr<double>(hdr->partials);
    double s = 0.0;
    int k = first + (int)threadIdx.x;
    for (; k + 7 * 64 < end; k += 8 * 64) {  // eight loads in flight (they pass the caches, about a us each)
        double v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = agent_load(partials + k + 64 * i);
#pragma unroll
        for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; k < end; k += 64) s += agent_load(partials + k);
    return norm_sq_of(wave_sum_f64(s), dtype);
}

// The total norm and the coefficient, by the whole of the launch's last workgroup: thread i adds
// norm_sq[i], norm_sq[i + 256], ...; the sums of the 4 waves are added in order.
__device__ __forceinline__ void norm_finish(const NormHeader* hdr, double* wave_sq, uint32_t* wave_bad_any) {
    const int count = hdr->count;
    const gptr<double> norm_sq = gaddr<double>(hdr->norm_sq);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double sq = 0.0;
    int at = threadIdx.x;
    for (; at + 7 * kNormThreads < count; at += 8 * kNormThreads) {
        double v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = agent_load(norm_sq + at + kNormThreads * i);
#pragma unroll
        for (int i = 0; i < 8; ++i) sq += v[i];
    }
    for (; at < count; at += kNormThreads) sq += agent_load(norm_sq + at);
    sq = wave_sum_f64(sq);
    uint32_t bad = 0;
    if (hdr->unscale) {
        const gptr<uint32_t> nonfinite = gaddr<uint32_t>(hdr->nonfinite);
        int k = threadIdx.x;
        for (; k + 7 * kNormThreads < hdr->total_segments; k += 8 * kNormThreads) {
            uint32_t b[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) b[i] = agent_load(nonfinite + k + kNormThreads * i);
#pragma unroll
            for (int i = 0; i < 8; ++i) bad |= b[i];
        }
        for (; k < hdr->total_segments; k += kNormThreads) bad |= agent_load(nonfinite + k);
    }
    const bool wave_bad = __builtin_amdgcn_ballot_w64(bad != 0) != 0;
    __syncthreads();  // the arrays' earlier contents have been read
    if (lane == 0) {
        wave_sq[wave] = sq;
        wave_bad_any[wave] = wave_bad ? 1u : 0u;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = wave_sq[0];
#pragma unroll
        for (int w = 1; w < kNormThreads / 64; ++w) s += wave_sq[w];
        if (hdr->unscale) {
            uint32_t b = 0;
#pragma unroll
            for (int w = 0; w < kNormThreads / 64; ++w) b |= wave_bad_any[w];
            *gaddr<float>(hdr->found_out) = b ? 1.0f : 0.0f;
        }
        const int R = hdr->result_dtype;
        const float total = round_to_dtype((float)__builtin_sqrt(s), R);
        const float shifted = round_to_dtype(total + 1e-6f, R);
        const float inv = round_to_dtype(div_cr(1.0f, shifted), R);
        float coef = round_to_dtype(inv * hdr->max_norm, R);
        coef = coef > 1.0f ? 1.0f : coef;  // torch.clamp(max=1): NaN stays NaN
        *gaddr<float>(hdr->norm_out) = total;
        *gaddr<float>(hdr->coef_out) = coef;
    }
}

// One workgroup per segment: the float64 sum of squares of its values -> partials[seg].  The workgroup
// that draws a gradient's last ticket adds up that gradient's segments, and the one that then draws the
// last gradient's ticket the whole (no workgroup waits for another; the sums' order is fixed, whichever
// workgroups those are).  Bound by the read of the gradients; as three launches behind a staged table
// (segments, gradients, total) the last two took 5 us each for GPT-2-small's 148 gradients, and longer
// than the read for a small model's.  Clip and step: GPT-2-small 431 -> 428 us, a tiny GPT-2 (host bound)
// 135 -> 127 us, 9 MB of bf16 gradients in seven tensors 82 -> 73 us.
// With tickets in two levels and the partials loaded eight at a time: one 4096^2 fp32 gradient's pass 40 us
// (1.7 TB/s) -> 16, clip and step 89.8 -> 65.9 us; two bf16 ones 124.4 -> 104.2 us.
// Many gradients, host and pass (fp32, of 1,000 values): drawing from one counter each 1,000 gradients took
// 24.7 us, 5,000 78.0 and 20,000 275; in runs, and without tickets for a gradient's only segment, 14.7, 27.5
// and 79.  With every ticket in a line of its own: 512 MB of bf16 gradients in 64 tensors 178 -> 165 us, 2 GB of
// fp32 ones 357 -> 311 (both read past the caches).
__device__ __forceinline__ void norm_body(const NormHeader* hdr) {
    const NormRow* rows = (const NormRow*)(hdr + 1);
    const int count = hdr->count;
    const int seg = (int)blockIdx.x;
    const int t = norm_row_of(rows, count, seg);
    const NormRow& T = rows[t];
    const int end = t + 1 < count ? rows[t + 1].seg_start : hdr->total_segments;
    const int dtype = T.dtype & (kNormVec - 1);
    const int64_t e0 = (int64_t)(seg - T.seg_start) << hdr->segment_shift;
    const int64_t e1 = min(e0 + ((int64_t)1 << hdr->segment_shift), T.numel);
    const bool vec = (T.dtype & kNormVec) != 0;
    double acc;
    bool bad = false;
    const bool keep = (T.dtype & kNormKeep) != 0;
    if (hdr->unscale) {
        const float u = *gaddr<const float>(hdr->inv_scale);
        acc = keep ? segment_sum_any<true, true>(T.grad, dtype, e0, e1, vec, u, bad)
                   : segment_sum_any<true, false>(T.grad, dtype, e0, e1, vec, u, bad);
    } else {
        acc = keep ? segment_sum_any<false, true>(T.grad, dtype, e0, e1, vec, 1.0f, bad)
                   : segment_sum_any<false, false>(T.grad, dtype, e0, e1, vec, 1.0f, bad);
    }
    acc = wave_sum_f64(acc);
    const bool wave_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    __shared__ double wave_acc[kNormThreads / 64];
    __shared__ uint32_t wave_bad_any[kNormThreads / 64];
    __shared__ uint32_t last_of_gradient, last_of_all;  // this workgroup drew the last ticket
    const bool whole = end - T.seg_start == 1;          // the gradient's only segment
    if ((threadIdx.x & 63) == 0) {
        wave_acc[threadIdx.x >> 6] = acc;
        wave_bad_any[threadIdx.x >> 6] = wave_bad ? 1u : 0u;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = wave_acc[0];
        uint32_t b = wave_bad_any[0];
#pragma unroll
        for (int w = 1; w < kNormThreads / 64; ++w) {
            s += wave_acc[w];
            b |= wave_bad_any[w];
        }
        if (whole) wave_acc[0] = s;
        else agent_store(gaddr<double>(hdr->partials) + seg, s);
        if (hdr->unscale) agent_store(gaddr<uint32_t>(hdr->nonfinite) + seg, b);
        last_of_gradient = norm_last_of_gradient(hdr, t, seg, T.seg_start, end) ? 1u : 0u;
    }
    __syncthreads();
    if (!last_of_gradient) return;
    if (threadIdx.x < 64) {
        const double norm_sq =
            whole ? norm_sq_of(wave_acc[0], dtype) : norm_tensor_sq(hdr, T.seg_start, end, dtype);
        if (threadIdx.x == 0) {
            agent_store(gaddr<double>(hdr->norm_sq) + t, norm_sq);
            last_of_all = norm_last_of_all(hdr, t, count) ? 1u : 0u;
        }
    }
    __syncthreads();
    if (last_of_all) norm_finish(hdr, wave_acc, wave_bad_any);
}

__global__ void __launch_bounds__(kNormThreads) norm_kernel(const NormHeader* hdr) { norm_body(hdr); }

// The same with header and rows in the launch's arguments (few gradients: no staging copy before it).
constexpr int kNormInlineBytes = 3840;
struct __align__(16) NormInlineArgs {
    unsigned char table[kNormInlineBytes];
};
__global__ void __launch_bounds__(kNormThreads) norm_kernel_inline(const NormInlineArgs a) {
    norm_body((const NormHeader*)((const char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(NormInlineArgs, table)));
}

}  // namespace aw4
