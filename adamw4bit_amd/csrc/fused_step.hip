// Fused 4-bit AdamW step for MI355X (gfx950): a multi-tensor launch for each kernel an optimizer step needs.
//
// Work decomposition
//   * A 128-value block (one fp32 scale per moment) is owned by 8 lanes of a 64-lane
//     wave; a wave owns 8 consecutive blocks (a 1024-value wave tile).
//   * Lane j (0..7) of a block owns the 16 values at offsets 32q + 4j + t (q, t = 0..3):
//     every parameter/gradient access is a 4-value vector (16 B for fp32) and each
//     quarter q of a block is one contiguous 128 B segment across the 8 lanes.  The same
//     split makes the reference's per-block sum order (ATen's 8-lane x 4-accumulator
//     reduction) mostly lane-local (block_sum_cross in aw4_math.h).
//   * Tiles of all tensors form one index space; each wave takes up to 4 tiles (in grid
//     order for the memory-bound kernels, consecutive ones for the update-SR kernels) and
//     the grid covers all of them, so the hardware dispatcher keeps the tiles in flight a
//     narrow moving window of memory.  fp32-state tensors join a launch of their dtype or
//     take one of their own (plan_values).
//   * Kernels are specialised on (m1 rounding kind, m2 rounding kind, parameter dtype);
//     a launch table whose tensors share one such combination (every recipe) runs the
//     specialised kernel, any other table the generic one.
//
// Arithmetic contract (the reference's ATen CPU operations, in order):
//   decode    m = cb[code] * scale                       (_optimized_quantization.py:91-107)
//   moments   m1 = fma(w1, g - m1, m1); m2 = fma(w2, g*g - m2, m2)   (ATen lerp)
//   denom     d = sqrt(m2) / sqrt(bc2) + eps             (_optimized.py:219-220)
//   param     p = p * (1 - lr*wd); p = p + (step_coef * m1) / d      (_optimized.py:221-222)
//   encode    s = max(max|m|, 1e-12); x = m / s; round; [dyn4_nz floor]; [EDEN]
//             (_optimized_quantization.py:46-88, _compiled_quantization.py:30-109)
// The file is compiled with -ffp-contract=off: every fused multiply-add is explicit.

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <map>
#include <mutex>
#include <string>
#include <algorithm>
#include <type_traits>
#include <vector>

#include "adamw4bit_hip.h"
#ifndef AW4_SCHED_ILP_TU
#include "aw4_prologue.h"  // its kernels belong to the main object only
#endif
#include "aw4_step.h"

// Device memory the library holds without allocating it: file-scope arrays, one copy per GPU,
// kept until the process ends.  g_tables_mem holds the codebook and lookup tables every kernel
// reads; `scratch` holds the launch tables of aw4_fused_step_noalloc.  In host code these names
// are stand-ins, not device addresses: the host takes each GPU's address of them with
// hipGetSymbolAddress (device_state) and uses only that.  (Only the main object holds them: the
// second compile of this file, AW4_SCHED_ILP_TU below, emits kernels and nothing else.)
#ifndef AW4_SCHED_ILP_TU
static __device__ __align__(256) uint8_t g_tables_mem[sizeof(aw4::Tables) + sizeof(aw4::SpecTables)];
// Launch tables of AW4_NOALLOC_TABLE_BYTES, and beyond them the header and the padding of every launch after
// the first that such a table can split into: whether a call fits depends on its rows alone.
constexpr size_t kNoallocGroupBytes = 1 << 17;
static __device__ __align__(256) uint8_t scratch[AW4_NOALLOC_TABLE_BYTES + kNoallocGroupBytes];
#endif

namespace {

using namespace aw4;

static_assert(sizeof(aw4_moment) == 104, "aw4_moment layout");
static_assert(sizeof(aw4_tensor) == 296, "aw4_tensor layout");

// Codebooks as fp32 bit patterns (ascending; code = index).  Values of the reference's
// closed forms: NF4 table (quantization.py:401-422), signed and unsigned dynamic maps
// with 3 exponent bits (:201-237), linspace grids (:457-497).
constexpr uint32_t kCodebookBits[AW4_NUM_CODEBOOKS][16] = {
    {0xBF800000u, 0xBF3239B1u, 0xBF066B31u, 0xBECA32A0u, 0xBE91A24Eu, 0xBE3D353Du, 0xBDBA786Cu, 0x00000000u,
     0x3DA2FAFFu, 0x3E24CAE3u, 0x3E7C04DDu, 0x3EAD0339u, 0x3EE1A4B7u, 0x3F1007ABu, 0x3F3913B2u, 0x3F800000u},
    {0xBF633333u, 0xBF29999Au, 0xBEE00000u, 0xBE599999u, 0xBD9EB852u, 0xBD051EB9u, 0xBBB43958u, 0x00000000u,
     0x3BB43958u, 0x3D051EB9u, 0x3D9EB852u, 0x3E599999u, 0x3EE00000u, 0x3F29999Au, 0x3F633333u, 0x3F800000u},
    {0x00000000u, 0x3B54FDF4u, 0x3BFDF3B5u, 0x3CAE147Bu, 0x3D333333u, 0x3D87AE15u, 0x3DB5C28Fu, 0x3E200000u,
     0x3E89999Au, 0x3EC33333u, 0x3EFCCCCDu, 0x3F1B3334u, 0x3F380000u, 0x3F54CCCCu, 0x3F71999Au, 0x3F800000u},
    {0x00000000u, 0x3D888889u, 0x3E088889u, 0x3E4CCCCEu, 0x3E888889u, 0x3EAAAAABu, 0x3ECCCCCEu, 0x3EEEEEF0u,
     0x3F088888u, 0x3F199999u, 0x3F2AAAAAu, 0x3F3BBBBCu, 0x3F4CCCCDu, 0x3F5DDDDEu, 0x3F6EEEEFu, 0x3F800000u},
    {0x3D800000u, 0x3E000000u, 0x3E400000u, 0x3E800000u, 0x3EA00000u, 0x3EC00000u, 0x3EE00000u, 0x3F000000u,
     0x3F100000u, 0x3F200000u, 0x3F300000u, 0x3F400000u, 0x3F500000u, 0x3F600000u, 0x3F700000u, 0x3F800000u},
};

// Lookup table a moment encodes with: round-to-nearest (dyn4_nz: floored) or level count.
__host__ __device__ inline int lut_id_of(int rounding, int codebook, int flags) {
    if (rounding == AW4_ROUND_RTN)
        return ((flags & AW4_MOMENT_ZERO_FLOOR) && codebook == AW4_CB_DYN4) ? kLutRtnDyn4Floor : kLutRtn[codebook];
    return kLutLevels[codebook];
}

// ---------------------------------------------------------------------------
// LDS layouts
// ---------------------------------------------------------------------------

// The specialised kernels' tables, behind those that every kernel reads.
__host__ __device__ inline const SpecTables* spec_tables(const Tables* g) { return (const SpecTables*)(g + 1); }

// Specialised kernels: the tables of the one codebook each moment uses.
template <bool kUpd, bool kSsr>
struct LdsSlots {
    float cb[2][16];
    UsrPair usr[2][kPairs];
    PairEntry pairs[2][kPairs];
    SsrEntry ssr[kSsr ? 2 : 1][kPairs];
    float2 dec[2][256];
    __align__(16) LinEntry lin[2][kLinSlots];
    WaveScratch scratch[kWavesPerGroup];
    f32x4 m2_stage[kUpd ? kWavesPerGroup * 4 * 64 : 1];  // second moments of a tile (update-SR kernels)

    __device__ __forceinline__ MomentTables moment(const aw4_moment&, int which, const StepHeader* h) const {
        const float magic = h->lin_magic[which];
        const uint32_t at = (uint32_t)(uintptr_t)(LinLds)(&lin[which][0]);
        return MomentTables{cb[which], pairs[which], dec[which], nullptr, usr[which], ssr[kSsr ? which : 0], magic,
                            at + ((uint32_t)h->lin_zero[which] << 3) - (f2u(magic) << 3)};
    }
    __device__ f32x4* wave_m2_stage(int wslot) { return kUpd ? &m2_stage[wslot * 4 * 64] : nullptr; }
    // Every load is issued before the first store to LDS, from addresses that depend on the header alone
    // (a lookup table is copied whole, whatever its count; a moment without codes copies codebook 0's
    // tables, which nothing reads): loops over the tables, with a lookup table's count read first, waited
    // for memory six times in a row at the start of every workgroup.  One fp32 tensor of 2048 x 4096, us so and
    // with loops: ZIP-SR 26.2 / 28.1, read back after its encode 41.5 / 43.9.
    __device__ void load(const Tables* g, const StepHeader* h) {
        const int i = threadIdx.x;
        const int i16 = min(i, 15), ip = min(i, kPairs - 1);
        float cb_v[2];
        u32x4 usr_v[2], pair_v[2], ssr_v[2], lin_v[2], lin_last[2];
        u32x2 dec_v[2];
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const int c = max(w ? h->cb2 : h->cb1, 0), l = max(w ? h->lut2 : h->lut1, 0);
            cb_v[w] = g->codebook[c][i16];
            usr_v[w] = *(const u32x4*)&g->usr[c][ip];
            pair_v[w] = *(const u32x4*)&g->pairs[c][ip];
            if (kSsr) ssr_v[w] = *(const u32x4*)&spec_tables(g)->ssr[c][ip];
            dec_v[w] = *(const u32x2*)&g->dec[c][i];
            const u32x4* e = (const u32x4*)spec_tables(g)->lin[l].e;
            lin_v[w] = e[i];
            lin_last[w] = e[kThreads];
        }
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            if (i < 16) cb[w][i] = cb_v[w];
            if (i < kPairs) {
                *(u32x4*)&usr[w][i] = usr_v[w];
                *(u32x4*)&pairs[w][i] = pair_v[w];
                if (kSsr) *(u32x4*)&ssr[w][i] = ssr_v[w];
            }
            *(u32x2*)&dec[w][i] = dec_v[w];
            *(u32x4*)&lin[w][2 * i] = lin_v[w];
            if (i == 0) *(u32x4*)&lin[w][2 * kThreads] = lin_last[w];
        }
        __syncthreads();
    }
    static_assert(kThreads == 256 && kLinSlots == 2 * kThreads + 2, "two lookup entries per thread, and two more");
};

// Generic kernels: every table.
struct LdsAll {
    Tables t;
    WaveScratch scratch[kWavesPerGroup];

    __device__ __forceinline__ MomentTables moment(const aw4_moment& m, int, const StepHeader*) const {
        const int cbid = m.rounding == AW4_ROUND_FP32 ? 0 : m.codebook;
        return MomentTables{t.codebook[cbid], t.pairs[cbid], t.dec[cbid],
                            t.lut[m.rounding == AW4_ROUND_FP32 ? 0 : lut_id_of(m.rounding, cbid, m.flags)],
                            t.usr[cbid], nullptr, 0.0f, 0u};
    }
    __device__ f32x4* wave_m2_stage(int) { return nullptr; }
    __device__ void load(const Tables* g, const StepHeader*) {
        const uint32_t* src = (const uint32_t*)g;
        uint32_t* dst = (uint32_t*)&t;
        for (int i = threadIdx.x; i < (int)(sizeof(Tables) / 4); i += kThreads) dst[i] = src[i];
        __syncthreads();
    }
};

template <int M1K, int M2K, int D>
struct KernelTraits {
    static constexpr int K1 = kind_of(M1K), K2 = kind_of(M2K);
    static constexpr bool kGeneric = K1 == K_ANY || K2 == K_ANY || D == D_ANY;
    static constexpr bool kSsr = K1 == K_SSR || K2 == K_SSR;
    static constexpr bool kUpd = K1 == K_USR || K2 == K_USR || K1 == K_ANY || K2 == K_ANY;
    using Lds = typename std::conditional<kGeneric, LdsAll, LdsSlots<kUpd, kSsr>>::type;
};

template <int M1K, int M2K, int D>
__device__ __forceinline__ void step_body(const StepHeader* __restrict__ hdr, const Tables* __restrict__ tables) {
    using Lds = typename KernelTraits<M1K, M2K, D>::Lds;
    __shared__ Lds lds;
    const int wslot = threadIdx.x >> 6;
    run_tiles<M1K, M2K, D>(hdr, lds, lds.scratch[wslot], lds.wave_m2_stage(wslot), [&] { lds.load(tables, hdr); });
}

template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) step_kernel(const StepHeader* __restrict__ hdr,
                                                         const Tables* __restrict__ tables) {
    step_body<M1K, M2K, D>(hdr, tables);
}

// The same kernel held to 128 VGPRs, four waves per SIMD (the fp32 recipes fit without spills;
// the fourth wave hides memory latency the third leaves exposed).
template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
step_kernel_4w(const StepHeader* __restrict__ hdr, const Tables* __restrict__ tables) {
    step_body<M1K, M2K, D>(hdr, tables);
}

// The same kernel held to 256 VGPRs, two waves per SIMD: the generic research instance (every
// m2 kind, read back or lookahead, with run-time dtypes) needed 270 otherwise, one wave per SIMD;
// it takes 243, without spills, and the second wave took the pending lookahead from 108 to
// 66 ms on the Llama-3-8B set.
template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2)))
step_kernel_2w(const StepHeader* __restrict__ hdr, const Tables* __restrict__ tables) {
    step_body<M1K, M2K, D>(hdr, tables);
}

// The same kernel held to 168 VGPRs, three waves per SIMD: the pending lookahead instance needed
// 178 otherwise (two waves); it takes 166, without spills, and the third wave took its step on the
// Llama-3-8B set from 37.8 to 34.8 ms.
template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3)))
step_kernel_3w(const StepHeader* __restrict__ hdr, const Tables* __restrict__ tables) {
    step_body<M1K, M2K, D>(hdr, tables);
}

// Small steps: the launch table travels in the kernel arguments, so that the step is one launch
// with no staging copy before it and no staging buffer to recycle after it (the launch packet
// holds its own copy of the arguments).  The kernel reads the table where the arguments are, so
// its fields still come through scalar loads.  Instances exist for the two recipes' kernels.
constexpr int kInlineTableBytes = 3584;

struct __align__(16) InlineArgs {
    const Tables* tables;
    uint64_t reserved;
    unsigned char table[kInlineTableBytes];
};

template <int M1K, int M2K, int D>
__device__ __forceinline__ void step_body_inline(const InlineArgs& a) {
    const StepHeader* hdr =
        (const StepHeader*)((const char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(InlineArgs, table));
    step_body<M1K, M2K, D>(hdr, a.tables);
}

template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
step_kernel_inline_4w(const InlineArgs a) {
    step_body_inline<M1K, M2K, D>(a);
}

// A launch of fp32-state tensors only (run_value_tiles).
template <int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
values_kernel(const StepHeader* __restrict__ hdr, const Tables* __restrict__) {
    run_value_tiles<D>(hdr);
}

template <int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
values_kernel_inline(const InlineArgs a) {
    run_value_tiles<D>(
        (const StepHeader*)((const char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(InlineArgs, table)));
}

}  // namespace

// The bf16 update-SR kernels (ZIP-SR and its nf4_sr head), the fp16 round-to-nearest ones and the
// code-storing lookahead ones come from a second compile of this file, with AW4_SCHED_ILP_TU defined and
// LLVM's max-ilp machine scheduler (-mllvm -amdgpu-sched-strategy=max-ilp); that object holds nothing else.
// Bound by their instruction issue, they run faster under it: the bf16 update-SR ones 1.2-1.5%; one
// Llama-3-8B layer under the proxy lookahead fp32 735.7 -> 714.4 us, bf16 724.3 -> 690.4 us; under ZE-EDEN
// fp16 385.9 -> 383.0 us, sdyn4 / dyn4 fp16 373.0 -> 370.9 us.  The bf16 round-to-nearest kernels gain
// nothing beyond a run's spread (374.4 and 373.7 us), and ZE-EDEN fp32 spilled (4% slower).  Since the
// update-SR encode is one stretch of code (encode_quick), the fp32 one and the EDEN-m2 ablation spill under
// it too (37 and 4 registers); all of these keep the default scheduler.  The main object declares these
// kernels and launches them through the variant table.
namespace aw4_ilp {
template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4)))
step_kernel_4w(const aw4::StepHeader* __restrict__ hdr, const aw4::Tables* __restrict__ tables)
#ifdef AW4_SCHED_ILP_TU
{
    step_body<M1K, M2K, D>(hdr, tables);
}
#else
    ;
#endif

template <int M1K, int M2K, int D>
__global__ void __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(3)))
step_kernel_3w(const aw4::StepHeader* __restrict__ hdr, const aw4::Tables* __restrict__ tables)
#ifdef AW4_SCHED_ILP_TU
{
    step_body<M1K, M2K, D>(hdr, tables);
}
#else
    ;
#endif
}  // namespace aw4_ilp

namespace {

// The instantiated kernels; the host groups a step's tensors by the variant whose moment
// specs and dtype they match (optimized-path flags).  ZE-EDEN: NF4 round-to-nearest m1,
// Dyn4 round-to-nearest m2 with EDEN.  ZIP-SR: NF4 round-to-nearest m1, Dyn4 update-SR m2
// with the exact-level guards; its nf4_sr head (value-space SR m1).  QuantizedAdamW
// ablations of ZIP-SR: an fp32 m2, EDEN on the update-SR m2.  Plain round-to-nearest moments (the
// ablation of both recipes; nf4 or sdyn4 first moments, any round-to-nearest second moment).
constexpr int kRtn = mspec(K_RTN), kRtnEden = mspec(K_RTN, AW4_MOMENT_EDEN), kFp32 = mspec(K_FP32);
constexpr int kSsrGuarded = mspec(K_SSR, AW4_MOMENT_GUARDS);
constexpr int kUsrGuarded = mspec(K_USR, AW4_MOMENT_GUARDS);
constexpr int kUsrGuardedEden = mspec(K_USR, AW4_MOMENT_GUARDS | AW4_MOMENT_EDEN);
// The reference step's update-SR m2 read back after its encode: dyn4_upd_sr / lin4_upd_sr,
// and *_upd_sr_store_eden (read at the scale before EDEN, EDEN on the stored scale).
constexpr int kUsrRead = mspec(K_USR, AW4_MOMENT_SAMPLED_READ);
constexpr int kUsrReadEden = mspec(K_USR, AW4_MOMENT_SAMPLED_READ | AW4_MOMENT_READ_RAW_SCALE | AW4_MOMENT_EDEN);
// Lookahead update-SR m2 stored as codes (dyn4_proxy_la_upd_sr, dyn4_vproxy_la_upd_sr).
constexpr int kLaStore = mspec(K_LA);
// ... and the pending form (dyn4_la_upd_sr): fp32 state sampled before the update.
constexpr int kLaPending = mspec(K_LA, AW4_MOMENT_PENDING);
// Any m2 kind of the research schemes (read-back and lookahead), any dtype.
constexpr int kAnyResearch = mspec(K_ANY, AW4_MOMENT_SAMPLED_READ);

#ifdef AW4_SCHED_ILP_TU
}  // namespace

template __global__ void aw4_ilp::step_kernel_4w<kRtn, kUsrGuarded, D_BF16>(const aw4::StepHeader*, const aw4::Tables*);
template __global__ void aw4_ilp::step_kernel_4w<kSsrGuarded, kUsrGuarded, D_BF16>(const aw4::StepHeader*,
                                                                                   const aw4::Tables*);
template __global__ void aw4_ilp::step_kernel_4w<kRtn, kRtnEden, D_F16>(const aw4::StepHeader*, const aw4::Tables*);
template __global__ void aw4_ilp::step_kernel_4w<kRtn, kRtn, D_F16>(const aw4::StepHeader*, const aw4::Tables*);
template __global__ void aw4_ilp::step_kernel_3w<kRtn, kLaStore, D_F32>(const aw4::StepHeader*, const aw4::Tables*);
template __global__ void aw4_ilp::step_kernel_3w<kRtn, kLaStore, D_BF16>(const aw4::StepHeader*, const aw4::Tables*);
template __global__ void aw4_ilp::step_kernel_3w<kRtn, kLaStore, D_F16>(const aw4::StepHeader*, const aw4::Tables*);
#else

struct KernelVariant {
    int m1, m2, dtype;
    const void* fn;
    const void* fn_inline;  // the instance taking its table in the arguments, or null
};
#define AW4_VARIANT(M1, M2, D) {M1, M2, D, (const void*)&step_kernel<M1, M2, D>, nullptr}
#define AW4_VARIANT_4W(M1, M2, D) {M1, M2, D, (const void*)&step_kernel_4w<M1, M2, D>, nullptr}
#define AW4_VARIANT_2W(M1, M2, D) {M1, M2, D, (const void*)&step_kernel_2w<M1, M2, D>, nullptr}
#define AW4_VARIANT_3W(M1, M2, D) {M1, M2, D, (const void*)&step_kernel_3w<M1, M2, D>, nullptr}
#define AW4_VARIANT_I4W(M1, M2, D) \
    {M1, M2, D, (const void*)&step_kernel_4w<M1, M2, D>, (const void*)&step_kernel_inline_4w<M1, M2, D>}
// the max-ilp instances of the second object (their small-step instances stay in this one)
#define AW4_VARIANT_ILP(M1, M2, D) {M1, M2, D, (const void*)&aw4_ilp::step_kernel_4w<M1, M2, D>, nullptr}
#define AW4_VARIANT_ILP_3W(M1, M2, D) {M1, M2, D, (const void*)&aw4_ilp::step_kernel_3w<M1, M2, D>, nullptr}
#define AW4_VARIANT_ILP_I4W(M1, M2, D) \
    {M1, M2, D, (const void*)&aw4_ilp::step_kernel_4w<M1, M2, D>, (const void*)&step_kernel_inline_4w<M1, M2, D>}
// launches of fp32-state tensors of one dtype
#define AW4_VARIANT_VALUES(D) \
    {kFp32, kFp32, D, (const void*)&values_kernel<D>, (const void*)&values_kernel_inline<D>}
// The fp16 recipes are bound as the bf16 ones are (memory for round-to-nearest, issue for update-SR)
// and take the same tiles; before they had instances they ran the generic kernel, bound by its two
// waves per SIMD: one Llama-3-8B layer (218M values) under ZE-EDEN 1,299 us there, 391-394 us here
// (4.5 TB/s).  The fp16 update-SR ones spill under the max-ilp scheduler and keep the default one.
// Plain round-to-nearest pairs likewise: the GPT-2-small fp32 set 545 -> 312 us (5.6 TB/s), a 4.3 GB
// bf16 set 3,590 -> 2,245 us.  And 16-bit parameters under the research second moments that keep codes: a
// 1.1 GB bf16 set under the proxy lookahead 1,147 -> 479 us, a 568 MB one with clipping 444 -> 166 us.
const KernelVariant kVariants[] = {
    AW4_VARIANT_I4W(kRtn, kRtnEden, D_F32),       AW4_VARIANT_I4W(kRtn, kUsrGuarded, D_F32),
    AW4_VARIANT_I4W(kRtn, kRtnEden, D_BF16),      AW4_VARIANT_ILP_I4W(kRtn, kUsrGuarded, D_BF16),
    AW4_VARIANT(kSsrGuarded, kUsrGuarded, D_F32), AW4_VARIANT_ILP(kSsrGuarded, kUsrGuarded, D_BF16),
    AW4_VARIANT(kRtn, kFp32, D_F32),              AW4_VARIANT(kRtn, kFp32, D_BF16),
    AW4_VARIANT(kRtn, kUsrGuardedEden, D_F32),    AW4_VARIANT_4W(kRtn, kUsrGuardedEden, D_BF16),
    AW4_VARIANT_ILP(kRtn, kRtnEden, D_F16),       AW4_VARIANT_4W(kRtn, kUsrGuarded, D_F16),
    AW4_VARIANT_4W(kSsrGuarded, kUsrGuarded, D_F16),
    AW4_VARIANT(kRtn, kFp32, D_F16),              AW4_VARIANT_4W(kRtn, kUsrGuardedEden, D_F16),
    AW4_VARIANT_4W(kRtn, kRtn, D_F32),            AW4_VARIANT_4W(kRtn, kRtn, D_BF16),
    AW4_VARIANT_ILP(kRtn, kRtn, D_F16),
    AW4_VARIANT_VALUES(D_F32), AW4_VARIANT_VALUES(D_BF16), AW4_VARIANT_VALUES(D_F16),
    AW4_VARIANT(kRtn, kUsrRead, D_F32),           AW4_VARIANT(kRtn, kUsrReadEden, D_F32),
    AW4_VARIANT_ILP_3W(kRtn, kLaStore, D_F32),    AW4_VARIANT_3W(kRtn, kLaPending, D_F32),
    AW4_VARIANT(kRtn, kUsrRead, D_BF16),          AW4_VARIANT(kRtn, kUsrRead, D_F16),
    AW4_VARIANT_ILP_3W(kRtn, kLaStore, D_BF16),   AW4_VARIANT_ILP_3W(kRtn, kLaStore, D_F16),
    AW4_VARIANT_2W(K_ANY, kAnyResearch, D_ANY),
    AW4_VARIANT(K_ANY, K_ANY, D_ANY),
};
#undef AW4_VARIANT
#undef AW4_VARIANT_VALUES
#undef AW4_VARIANT_4W
#undef AW4_VARIANT_2W
#undef AW4_VARIANT_3W
#undef AW4_VARIANT_I4W
#undef AW4_VARIANT_ILP
#undef AW4_VARIANT_ILP_3W
#undef AW4_VARIANT_ILP_I4W
constexpr int kNumVariants = sizeof(kVariants) / sizeof(kVariants[0]);
constexpr int kGenericVariant = kNumVariants - 1;
constexpr int kResearchVariant = kNumVariants - 2;  // generic, for read-back and lookahead m2
constexpr int kNumSpecialised = kResearchVariant;

// Stand-alone codec kernels.  They stream (encode reads 4 bytes and writes 0.53 a value, decode the
// reverse), so a workgroup's LDS holds only the tables its one moment needs (3 to 3.6 KB of tables and the
// four waves' scratch, 8.3 KB, to encode, 2 KB to decode; all codebooks' tables are 36 KB and left three
// workgroups to a CU), and the grid covers every tile at kCodecTiles per wave, which share the table fill.
// Decode's stores are non-temporal, as the other kernels' are: dirty lines left in the L2s were written
// back while the next launch waited.
// Measured, nf4, us encode / decode: 2^24 values 26.5 / 27.6 with all tables, a grid of eight workgroups per
// CU and plain stores, 13.6 / 12.1 so (5.6 / 6.3 TB/s); 2^27 values 140 / 160 and 111 / 89 us (5.5 / 6.8 TB/s).
// A kernel that reads the decoded values next loses nothing: decode and a copy of 2^20, 2^22, 2^24 and 2^27
// values 10.6, 30.7, 54.9 and 347 us before, 8.8, 16.1, 39.2 and 294 so.  Encoding nf4_sr is bound by its draws
// (24.0 us of 2^24 values).
constexpr int kCodecTiles = 4;

// Encode tables of the codebook a moment uses, those its kind of rounding reads, and the waves' scratch.
template <int KIND>
struct LdsEncode {
    float cb[16];
    UsrPair usr[KIND == K_USR ? kPairs : 1];
    PairEntry pairs[KIND != K_RTN ? kPairs : 1];
    LutEntry lut[AW4_LUT_ENTRIES];
    WaveScratch scratch[kWavesPerGroup];

    __device__ void load(const Tables* g, int codebook, int lut_id) {
        if (threadIdx.x < 16) cb[threadIdx.x] = g->codebook[codebook][threadIdx.x];
        if (threadIdx.x < kPairs) {
            if constexpr (KIND == K_USR) usr[threadIdx.x] = g->usr[codebook][threadIdx.x];
            if constexpr (KIND != K_RTN) pairs[threadIdx.x] = g->pairs[codebook][threadIdx.x];
        }
        if (threadIdx.x < AW4_LUT_ENTRIES) lut[threadIdx.x] = g->lut[lut_id][threadIdx.x];
        __syncthreads();
    }
};
static_assert(AW4_LUT_ENTRIES <= kThreads, "one thread per lookup entry");

// KIND: the moment's rounding (its flags are read at run time).  Wave w of W encodes tiles w, w + W, ...,
// the next tile's values loaded while this one is encoded.
template <int KIND>
__global__ void __launch_bounds__(kThreads) quantize_kernel(const float* __restrict__ values, int64_t numel,
                                                            aw4_moment M, const Tables* __restrict__ tables) {
    __shared__ LdsEncode<KIND> lds;
    const int lane = threadIdx.x & 63;
    const int wslot = threadIdx.x >> 6;
    const int j = lane & 7, grp = lane >> 3;
    const int64_t nblocks = numel / kBlock;
    const int64_t tiles = (nblocks + kBlocksPerWave - 1) / kBlocksPerWave;
    const int64_t nwaves = (int64_t)gridDim.x * kWavesPerGroup;
    int64_t tile = (int64_t)blockIdx.x * kWavesPerGroup + __builtin_amdgcn_readfirstlane(wslot);
    auto load = [&](int64_t t, float (&m)[16]) {
        const int64_t blk = t * kBlocksPerWave + grp;
        // a lane past the last block reads the tile's first block, which exists; nothing of it is stored
        const float* v = values + (blk < nblocks ? blk : t * kBlocksPerWave) * kBlock + 4 * j;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const f32x4 x = *(gptr<const f32x4>)gaddr<const float>((uint64_t)(v + 32 * q));
            m[4 * q] = x.x; m[4 * q + 1] = x.y; m[4 * q + 2] = x.z; m[4 * q + 3] = x.w;
        }
    };
    float next[16];
    if (tile < tiles) load(tile, next);
    lds.load(tables, M.codebook, lut_id_of(M.rounding, M.codebook, M.flags));
    const MomentTables L{lds.cb, lds.pairs, nullptr, lds.lut, lds.usr, nullptr, 0.0f, 0u};
    while (tile < tiles) {
        float m[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) m[i] = next[i];
        const int64_t blk0 = tile * kBlocksPerWave;
        tile += nwaves;
        if (tile < tiles) load(tile, next);
        // stand-alone encodes accept any sign (a first moment or a caller's values)
        encode_block<mspec(KIND, kFlagsAtRunTime), false>(M, L, blk0, grp, j, blk0 + grp < nblocks, RegValues{m},
                                                          lds.scratch[wslot].block(grp));
    }
}

// Wave w of W decodes tiles w, w + W, ...; in a tile, load q of lane l is the two code bytes of values
// 256 q + 4 l .. + 3, so a wave's loads and stores are contiguous (128 bytes and 1 KB).
__global__ void __launch_bounds__(kThreads) dequantize_kernel(aw4_moment M, int64_t numel, float* __restrict__ out,
                                                              const Tables* __restrict__ tables) {
    __shared__ float2 dec[256];
    static_assert(kThreads == 256, "one thread per decode entry");
    dec[threadIdx.x] = tables->dec[M.codebook][threadIdx.x];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int64_t tiles = (numel + kWaveTile - 1) / kWaveTile;
    const int64_t nwaves = (int64_t)gridDim.x * kWavesPerGroup;
    const gptr<const uint8_t> codes = gaddr<const uint8_t>(M.codes);
    const gptr<const float> scales = gaddr<const float>(M.scales);
    for (int64_t tile = (int64_t)blockIdx.x * kWavesPerGroup + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
         tile < tiles; tile += nwaves) {
        const int64_t e0 = tile * kWaveTile + 4 * lane;
        uint32_t w[4];
        float scale[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t e = e0 + 256 * q;
            const int64_t at = e < numel ? e : 4 * (lane & 31);  // past the end: the first block's, not stored
            w[q] = *(gptr<const uint16_t>)(codes + at / 2);
            scale[q] = scales[at / kBlock];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int64_t e = e0 + 256 * q;
            float m[4];
            decode4(dec, w[q], scale[q], m);
            if (e < numel)
                __builtin_nontemporal_store(f32x4{m[0], m[1], m[2], m[3]}, (gptr<f32x4>)gaddr<float>((uint64_t)(out + e)));
        }
    }
}

// Uniforms at positions offset .. offset+n-1 (n > 0): one thread per (position group, lane).
__global__ void __launch_bounds__(kThreads) uniforms_kernel(uint64_t seed, uint64_t offset, int64_t n,
                                                            float* __restrict__ out) {
    const uint64_t g0 = offset >> 7, end = offset + (uint64_t)n;
    const int64_t lanes = (int64_t)(((end - 1) >> 7) - g0 + 1) * 8;
    for (int64_t l = (int64_t)blockIdx.x * kThreads + threadIdx.x; l < lanes; l += (int64_t)gridDim.x * kThreads) {
        const uint64_t group = g0 + (uint64_t)(l >> 3);
        const int j = (int)(l & 7);
        uint32_t w[12];
#pragma unroll
        for (int r = 0; r < 3; ++r) philox_lane_call(seed, group, j, r, &w[4 * r]);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float u[4];
            lane_fields4(&w[3 * q], u);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint64_t pos = group * kBlock + (uint64_t)(32 * q + 4 * j + t);
                if (pos >= offset && pos < end) out[pos - offset] = u[t] * 0x1p-24f;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

thread_local std::string g_error;
thread_local int g_fail_after = -1;  // aw4_inject_launch_failure

int set_error(int code, const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    g_error = buf;
    return code;
}

#define AW4_HIP_CHECK(expr)                                                                             \
    do {                                                                                                \
        hipError_t err_ = (expr);                                                                       \
        if (err_ != hipSuccess) return set_error(AW4_EHIP, "%s: %s", #expr, hipGetErrorString(err_)); \
    } while (0)

float host_f(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }

int count_less(const float* cb, float x) {
    int c = 0;
    for (int k = 0; k < 16; ++k) c += cb[k] < x ? 1 : 0;
    return c;
}

// Round-to-nearest code of the reference (ties to the upper level), in fp32.
int rtn_code(const float* cb, float x, bool floor_zero) {
    const int idx = count_less(cb, x);
    const int lo = idx > 0 ? idx - 1 : 0;
    const int hi = idx < 15 ? idx : 15;
    const float da = fabsf(x - cb[lo]);
    const float db = fabsf(cb[hi] - x);
    int code = da < db ? lo : hi;
    if (floor_zero && code == 0) code = 1;
    return code;
}

static_assert(kLinSlots == AW4_LINEAR_SLOTS && sizeof(LinTable) == 16 + 8 * AW4_LINEAR_SLOTS, "aw4_linear_tables");

struct HostTables {
    Tables t;
    SpecTables spec;  // behind `t`, as in device memory
    bool ok = false;
    std::string error;
};

// Build one lookup table: bucket -> (threshold, base) such that f(x) = base + (x >= threshold)
// for every fp32 x of the bucket, where f is monotone non-decreasing in x.  Fails if a
// bucket holds more than one change of f.  The entry's levels are cb[min(f, 15)] for both
// outcomes: the code's level (round-to-nearest) or the upper neighbour b of x (level count).
template <class F>
bool build_lut(LutEntry* out, F f, const float* cb, std::string& err) {
    for (int sign = 0; sign < 2; ++sign) {
        for (int k = 0; k < AW4_LUT_HALF; ++k) {
            uint32_t alo, ahi;
            if (k == 0) {
                alo = 0u;
                ahi = ((uint32_t)AW4_LUT_EXP0 << 20) - 1u;
            } else if (k < AW4_LUT_HALF - 1) {
                alo = (uint32_t)(AW4_LUT_EXP0 - 1 + k) << 20;
                ahi = alo + (1u << 20) - 1u;
            } else {
                alo = (uint32_t)(AW4_LUT_EXP0 - 1 + k) << 20;
                ahi = 0x7f800000u;
            }
            auto val = [&](uint32_t a) { return sign ? -host_f(a) : host_f(a); };
            // x increases with a for sign 0 and decreases for sign 1
            const uint32_t amin = sign ? ahi : alo, amax = sign ? alo : ahi;
            const int base = f(val(amin));
            const int top = f(val(amax));
            LutEntry e;
            e.base = (uint32_t)base;
            if (top == base) {
                // NaN: x >= thr is false for every x (an infinite threshold would still
                // increment at x = +inf, one past the bucket's count)
                e.thr = host_f(0x7fc00000u);
            } else if (top == base + 1) {
                // smallest x (in value order) with f(x) == base + 1
                uint32_t good = amax, bad = amin;
                while ((sign ? bad - good : good - bad) > 1u) {
                    const uint32_t mid = sign ? good + (bad - good) / 2u : bad + (good - bad) / 2u;
                    if (f(val(mid)) == base + 1) good = mid; else bad = mid;
                }
                e.thr = val(good);
            } else {
                char buf[160];
                snprintf(buf, sizeof(buf), "lookup bucket %d (sign %d) spans %d code changes", k, sign, top - base);
                err = buf;
                return false;
            }
            e.lv_lo = cb[base < 15 ? base : 15];
            e.lv_hi = cb[base + 1 < 15 ? base + 1 : 15];
            out[k + sign * AW4_LUT_HALF] = e;
        }
    }
    return true;
}

// The LinTable of f, monotone non-decreasing, over [0, 1] or (is_signed) [-1, 1]: the widest buckets that
// hold at most one change of f each.
template <class F>
bool build_linear_lut(LinTable& out, F f, bool is_signed, std::string& err) {
    // floats of the range in order, and back
    auto value = [](int32_t k) { return k < 0 ? -host_f((uint32_t)-k) : host_f((uint32_t)k); };
    const int32_t one = 0x3f800000;
    for (int inv = 16; inv <= 512; inv *= 2) {
        const int count = is_signed ? 2 * inv + 1 : inv + 1;
        if (count > kLinSlots) break;
        memset(&out, 0, sizeof(out));
        out.magic = 1.5f * (float)(1 << 23) / (float)inv;
        out.count = count;
        out.zero = is_signed ? inv : 0;
        auto bucket = [&](int32_t k) {
            const volatile float sum = value(k) + out.magic;  // rounded to fp32, as the kernel's addition
            const float s = sum;
            uint32_t a, b;
            memcpy(&a, &s, 4);
            memcpy(&b, &out.magic, 4);
            return (int)(a - b) + out.zero;
        };
        // first float of the range at or above bucket b
        auto first = [&](int b) {
            int32_t lo = is_signed ? -one : 0, hi = one + 1;
            while (lo < hi) {
                const int32_t mid = lo + (hi - lo) / 2;
                if (bucket(mid) >= b) hi = mid; else lo = mid + 1;
            }
            return lo;
        };
        bool ok = bucket(is_signed ? -one : 0) == 0 && bucket(one) == count - 1;
        for (int b = 0; b < count && ok; ++b) {
            const int32_t lo = first(b), hi = first(b + 1) - 1;
            const int base = f(value(lo)), top = f(value(hi));
            out.e[b].base = (uint32_t)base;
            out.e[b].thr = host_f(0x7fc00000u);  // never reached
            if (top == base + 1) {
                int32_t bad = lo, good = hi;
                while (good - bad > 1) {
                    const int32_t mid = bad + (good - bad) / 2;
                    if (f(value(mid)) == base + 1) good = mid; else bad = mid;
                }
                out.e[b].thr = value(good);
            }
            ok = lo <= hi && top <= base + 1;
        }
        if (ok) return true;
    }
    err = "no linear lookup table holds one code change per bucket";
    return false;
}

const HostTables& host_tables() {
    static HostTables h;
    static std::once_flag once;
    std::call_once(once, [] {
        Tables& t = h.t;
        memset(&t, 0, sizeof(t));
        for (int c = 0; c < AW4_NUM_CODEBOOKS; ++c) {
            for (int k = 0; k < 16; ++k) t.codebook[c][k] = host_f(kCodebookBits[c][k]);
            // square roots of the levels and of their gaps, in double, rounded once to fp32
            float sqrt_level[16];
            for (int k = 0; k < 16; ++k) {
                const double l = (double)t.codebook[c][k];
                sqrt_level[k] = l > 0.0 ? (float)sqrt(l) : 0.0f;
            }
            for (int i = 0; i < kPairs; ++i) {
                const int lo = i > 0 ? i - 1 : 0, hi = i < 15 ? i : 15;
                const double a = (double)t.codebook[c][lo], b = (double)t.codebook[c][hi];
                const float gap = (a >= 0.0 && b > a) ? (float)(sqrt(b) - sqrt(a)) : 0.0f;
                t.usr[c][i] = UsrPair{sqrt_level[lo], sqrt_level[hi], ldexpf(gap, -24),
                                      t.codebook[c][hi] > t.codebook[c][lo] ? 1.0f : 0.0f};
                PairEntry& p = t.pairs[c][i];
                p.a = t.codebook[c][lo];
                p.b = t.codebook[c][hi];
                const float w = p.b - p.a;
                p.width_rcp = 1.0f / (w < 1e-12f ? 1e-12f : w);
                p.lohi = (uint32_t)lo | ((uint32_t)hi << 8);
                // (the 1e-12 floor of the width binds only where lo == hi: index 0, and 16, which no x <= 1 has)
                SsrEntry& e = h.spec.ssr[c][i];
                if (i > 0) {
                    e.a = p.a;
                    e.width = ldexpf(w < 1e-12f ? 1e-12f : w, -24);
                } else {
                    e.a = -8.0f;
                    e.width = 0x1p-24f;
                }
                e.width_rcp = 1.0f / e.width;
            }
            for (int b = 0; b < 256; ++b) t.dec[c][b] = make_float2(t.codebook[c][b & 15], t.codebook[c][b >> 4]);
        }
        bool ok = true;
        for (int c = 0; c < AW4_NUM_CODEBOOKS && ok; ++c) {
            const float* cb = t.codebook[c];
            ok = build_lut(t.lut[kLutRtn[c]], [cb](float x) { return rtn_code(cb, x, false); }, cb, h.error) &&
                 build_lut(t.lut[kLutLevels[c]], [cb](float x) { return count_less(cb, x); }, cb, h.error);
        }
        if (ok) {
            const float* cb = t.codebook[AW4_CB_DYN4];
            ok = build_lut(t.lut[kLutRtnDyn4Floor], [cb](float x) { return rtn_code(cb, x, true); }, cb, h.error) &&
                 build_linear_lut(h.spec.lin[kLutRtnDyn4Floor], [cb](float x) { return rtn_code(cb, x, true); }, false, h.error);
        }
        for (int c = 0; c < AW4_NUM_CODEBOOKS && ok; ++c) {
            const float* cb = t.codebook[c];
            const bool is_signed = cb[0] < 0.0f;
            ok = build_linear_lut(h.spec.lin[kLutRtn[c]], [cb](float x) { return rtn_code(cb, x, false); }, is_signed, h.error) &&
                 build_linear_lut(h.spec.lin[kLutLevels[c]], [cb](float x) { return count_less(cb, x); }, is_signed, h.error);
        }
        h.ok = ok;
    });
    return h;
}

struct StagingSlot {
    void* host = nullptr;            // pinned, mapped and coherent: the host writes the table here
    const void* host_dev = nullptr;  // the device's address of `host`
    void* dev = nullptr;             // device copy the kernels read
    size_t cap = 0;
    uint32_t* counters = nullptr;    // the norm pass's (norm_counters), zero outside its launches
    size_t counter_words = 0;
    hipEvent_t done = nullptr;
    bool pending = false;
};

constexpr int kSlots = 4;

struct DeviceState {
    Tables* tables = nullptr;    // this GPU's address of g_tables_mem
    uint8_t* scratch = nullptr;  // this GPU's address of `scratch`
    int num_cus = 0;
    StagingSlot slots[kSlots];
    int next = 0;
    // Host buffers of slots that have grown.  The device has read them uncached; they are kept
    // until the process ends rather than freed and their pages handed out again.
    std::vector<void*> retired_host;
    std::vector<uint8_t> noalloc_host;  // host image of the tables aw4_fused_step_noalloc stages
    std::vector<uint8_t> inline_host;   // host image of the tables of small steps (launch arguments)
};

std::mutex g_mutex;
std::map<int, DeviceState> g_devices;

int device_state(DeviceState** out) {
    const HostTables& ht = host_tables();
    if (!ht.ok) return set_error(AW4_EINVAL, "encode tables: %s", ht.error.c_str());
    int dev = 0;
    AW4_HIP_CHECK(hipGetDevice(&dev));
    DeviceState& ds = g_devices[dev];
    if (!ds.tables) {
        // Once per device, with that device current: its addresses of the file-scope arrays, and
        // the codebook tables copied into them (one synchronous copy; nothing is allocated).
        hipDeviceProp_t prop;
        AW4_HIP_CHECK(hipGetDeviceProperties(&prop, dev));
        ds.num_cus = prop.multiProcessorCount;
        void* tables = nullptr;
        void* stage = nullptr;
        AW4_HIP_CHECK(hipGetSymbolAddress(&tables, HIP_SYMBOL(g_tables_mem)));
        AW4_HIP_CHECK(hipGetSymbolAddress(&stage, HIP_SYMBOL(scratch)));
        static_assert(offsetof(HostTables, spec) == sizeof(Tables), "one copy of both");
        AW4_HIP_CHECK(hipMemcpy(tables, &ht.t, sizeof(Tables) + sizeof(SpecTables), hipMemcpyHostToDevice));
        ds.scratch = (uint8_t*)stage;
        ds.tables = (Tables*)tables;
    }
    *out = &ds;
    return AW4_OK;
}

bool aligned(uint64_t addr, uint64_t a) { return (addr % a) == 0; }

int check_moment(const aw4_moment& m, int64_t numel, int index, const char* name) {
    const bool la = m.rounding == AW4_ROUND_LOOKAHEAD_SR;
    if ((m.flags & (AW4_MOMENT_FRESH_PROXY | AW4_MOMENT_PENDING)) && !la)
        return set_error(AW4_EINVAL, "tensor %d: %s lookahead flags without lookahead rounding", index, name);
    if (m.rounding == AW4_ROUND_FP32) {
        if (!m.values) return set_error(AW4_EINVAL, "tensor %d: %s fp32 state without values", index, name);
        if (!aligned(m.values, 16)) return set_error(AW4_EALIGN, "tensor %d: %s values not 16-byte aligned", index, name);
        return AW4_OK;
    }
    if (m.rounding < AW4_ROUND_RTN || m.rounding > AW4_ROUND_LOOKAHEAD_SR)
        return set_error(AW4_EINVAL, "tensor %d: %s has rounding %d", index, name, m.rounding);
    if (m.codebook < 0 || m.codebook >= AW4_NUM_CODEBOOKS)
        return set_error(AW4_EINVAL, "tensor %d: %s has codebook %d", index, name, m.codebook);
    if (numel % kBlock != 0)
        return set_error(AW4_EINVAL, "tensor %d: %s quantized but numel %lld is not a multiple of %d", index, name,
                         (long long)numel, kBlock);
    if (la) {
        // lookahead update-SR (quantize_dyn4_la_upd_sr): m2 on the dyn4 codebook only
        if (strcmp(name, "m2") != 0 || m.codebook != AW4_CB_DYN4)
            return set_error(AW4_EINVAL, "tensor %d: lookahead update-SR is for a dyn4 m2 only", index);
        if ((m.flags & AW4_MOMENT_FRESH_PROXY) && (m.flags & AW4_MOMENT_PENDING))
            return set_error(AW4_EINVAL, "tensor %d: m2 FRESH_PROXY and PENDING together", index);
        if (m.flags & (AW4_MOMENT_SAMPLED_READ | AW4_MOMENT_READ_RAW_SCALE | AW4_MOMENT_EDEN))
            return set_error(AW4_EINVAL, "tensor %d: lookahead m2 with read-back or EDEN flags", index);
        if (!(m.la_bias > 0.0) || !(m.la_beta2 >= 0.0 && m.la_beta2 < 1.0) || !(m.la_eps >= 0.0))
            return set_error(AW4_EINVAL, "tensor %d: lookahead m2 needs bias > 0, beta2 in [0, 1), eps >= 0", index);
    }
    if (la && (m.flags & AW4_MOMENT_PENDING)) {
        if (!m.values || !aligned(m.values, 16))
            return set_error(AW4_EINVAL, "tensor %d: pending lookahead m2 without 16-byte aligned values", index);
    } else {
        if (!m.codes || !m.scales)
            return set_error(AW4_EINVAL, "tensor %d: %s quantized without codes/scales", index, name);
        // codes: each lane stores its 16 codes as one 8-byte word
        if (!aligned(m.codes, 8) || !aligned(m.scales, 4))
            return set_error(AW4_EALIGN, "tensor %d: %s codes not 8-byte or scales not 4-byte aligned", index, name);
    }
    if (m.rounding != AW4_ROUND_RTN) {
        if (m.flags & AW4_MOMENT_EXT_DRAWS) {
            if (!m.draws || !aligned(m.draws, 16))
                return set_error(AW4_EINVAL, "tensor %d: %s external draws missing or misaligned", index, name);
        } else if (m.rng_offset % kBlock != 0) {
            return set_error(AW4_EINVAL, "tensor %d: %s rng_offset not a multiple of 128", index, name);
        }
    }
    if (m.rounding == AW4_ROUND_UPDATE_SR && !(m.sr_bias > 0.0f))
        return set_error(AW4_EINVAL, "tensor %d: %s update-SR bias must be positive", index, name);
    if (m.flags & (AW4_MOMENT_SAMPLED_READ | AW4_MOMENT_READ_RAW_SCALE)) {
        if (strcmp(name, "m2") != 0)
            return set_error(AW4_EINVAL, "tensor %d: only m2 can be read back after its encode", index);
        if (!(m.flags & AW4_MOMENT_SAMPLED_READ))
            return set_error(AW4_EINVAL, "tensor %d: m2 READ_RAW_SCALE without SAMPLED_READ", index);
        if (m.values && !aligned(m.values, 16))
            return set_error(AW4_EALIGN, "tensor %d: m2 preconditioner output not 16-byte aligned", index);
    }
    return AW4_OK;
}

int check_tensor(const aw4_tensor& t, int index) {
    if (!t.param || !t.grad) return set_error(AW4_EINVAL, "tensor %d: null param or grad", index);
    if (t.numel <= 0) return set_error(AW4_EINVAL, "tensor %d: numel %lld", index, (long long)t.numel);
    for (int dt : {t.param_dtype, t.grad_dtype})
        if (dt != AW4_F32 && dt != AW4_BF16 && dt != AW4_F16 && dt != AW4_F64)
            return set_error(AW4_EINVAL, "tensor %d: dtype %d", index, dt);
    if (t.flags & AW4_TENSOR_VEC_ALIGNED) {
        // 4-value vector access: 16 bytes (fp32, and float64 as two 16-byte halves) or 8 bytes
        const uint64_t pa = t.param_dtype == AW4_F32 || t.param_dtype == AW4_F64 ? 16 : 8;
        const uint64_t ga = t.grad_dtype == AW4_F32 || t.grad_dtype == AW4_F64 ? 16 : 8;
        if (!aligned(t.param, pa) || !aligned(t.grad, ga))
            return set_error(AW4_EALIGN, "tensor %d: VEC_ALIGNED but param/grad misaligned", index);
    }
    const bool scaled = (t.flags & (AW4_TENSOR_GRAD_SCALE | AW4_TENSOR_GRAD_UNSCALE)) != 0;
    if (scaled && (!t.grad_scale || !aligned(t.grad_scale, 4)))
        return set_error(AW4_EINVAL, "tensor %d: GRAD_SCALE/GRAD_UNSCALE without a 4-byte aligned grad_scale", index);
    if (scaled && t.grad_dtype == AW4_F64)
        return set_error(AW4_EINVAL, "tensor %d: GRAD_SCALE/GRAD_UNSCALE with a float64 gradient", index);
    int rc = check_moment(t.m1, t.numel, index, "m1");
    if (rc) return rc;
    return check_moment(t.m2, t.numel, index, "m2");
}

bool host_values_only(const aw4_tensor& t) {
    return (t.m1.rounding == AW4_ROUND_FP32 && t.m2.rounding == AW4_ROUND_FP32) || t.numel % kBlock != 0;
}

// m2 of the reference step's research variants, stepped by the research kernel instance.
bool research_m2(const aw4_moment& m) {
    return (m.flags & AW4_MOMENT_SAMPLED_READ) || m.rounding == AW4_ROUND_LOOKAHEAD_SR;
}

// One launch of a step: a kernel variant, the tables its LDS slots load, and its tensors.
struct LaunchGroup {
    int variant = kGenericVariant;
    int cb1 = -1, lut1 = -1, cb2 = -1, lut2 = -1;
    std::vector<int> members;
};

// fp32-state tensors of one dtype join the step's first launch of that dtype or take one of their own
// (values_kernel).  Beside blocks a tile of them goes value by value, 10-20 us for its wave, at nobody's
// expense while the launch has waves to spare; their own launch is faster per tile and costs about 1 us
// (3 us of host time for a staged table) and a boundary on the stream.  Measured, us a step joined /
// own, one block tensor and fp32-state tiles, ZIP-SR fp32 and bf16:
//   1024^2 and 16-512 tiles: 15.9-16.2 / 17.1 and 15.8-16.9 / 17.1; 1024 tiles: 17.1 / 17.2 and
//     17.4 / 17.5; 2048: 27.6 / 20.6 and 24.2 / 19.6; 4096: 47.6 / 30.1 and 44.2 / 29.9;
//   8 tiles, which end the launch: 2048 x 3072 (24 tiles per CU, 2 fp32-state tiles) 25.5 / 30.0 and
//     24.6 / 30.2; 2048 x 4096 (32) 37.9 / 32.3 and 41.7 / 32.2; 4096^2 (64) 53.3 / 54.5 and
//     67.9 / 48.8 (a wave of consecutive tiles takes several of them); 14336 x 4096 157.6 / 158.7 and
//     144.8 / 133.2;
//   4096^2 and 16 tiles: 64.1 / 53.9 and 78.2 / 48.7;
//   1 and 2 tiles beside a large launch, where a wave of consecutive tiles meets two at most: 2048 x 4096 bf16
//     25.9 / 32.0 and 33.9 / 32.2 (3 and 4: 36.7 / 33.6 and later), 4096^2 40.7 / 47.7 and 46.1 / 47.8,
//     14336 x 4096 124.2 / 130.1 and 123.1 / 128.9; not so beside the generic kernel, whose one tile takes
//     longer than a launch: sdyn4_sr / dyn4_sr fp32 2048 x 4096 75.6 / 67.1;
//   the code-storing lookahead kernels, slower per block tile, hide more of them: fp32 2048 x 4096 and 8 tiles
//     50.4 / 55.4, bf16 51.0 / 56.0; 16 tiles bf16 4096^2 93.4 / 90.8.
constexpr int64_t kValuesLaunchTiles = 1024;   // own launch from this many fp32-state tiles on
constexpr int64_t kValuesBlockTiles = 8192;    // beside this many block tiles (32 per CU): own launch
constexpr int64_t kValuesFewTiles = 16;        // ... unless they are fewer than this, in grid order or lookahead
constexpr int64_t kValuesFewConsecutive = 3;   // ... or than this, where waves take consecutive tiles

bool values_variant(const KernelVariant& kv) { return kv.m1 == kFp32 && kv.m2 == kFp32; }

int64_t tiles_of(const aw4_tensor* ts, const std::vector<int>& members) {
    int64_t n = 0;
    for (int i : members) n += (ts[i].numel + kWaveTile - 1) / kWaveTile;
    return n;
}

void plan_values(const aw4_tensor* ts, const std::vector<int>& values, std::vector<LaunchGroup>& groups,
                 LaunchGroup& generic) {
    const size_t block_groups = groups.size();
    for (int dtype : {AW4_F32, AW4_BF16, AW4_F16, AW4_F64}) {
        std::vector<int> of;
        for (int i : values)
            if (ts[i].param_dtype == dtype) of.push_back(i);
        if (of.empty()) continue;
        int own = -1;  // this dtype's values_kernel (none for float64, which joins the generic launch)
        for (int k = 0; k < kNumSpecialised; ++k)
            if (kVariants[k].dtype == dtype && values_variant(kVariants[k])) own = k;
        LaunchGroup* g = nullptr;
        for (size_t k = 0; k < block_groups && !g; ++k)
            if (kVariants[groups[k].variant].dtype == dtype) g = &groups[k];
        if (!g && (own < 0 || !generic.members.empty())) g = &generic;
        if (g && own >= 0) {
            const KernelVariant& kv = kVariants[g->variant];
            const int64_t tiles = tiles_of(ts, of);
            const bool hidden = tile_order_grid(kv.m1, kv.m2, kv.dtype) || kind_of(kv.m2) == K_LA;
            const int64_t few = g == &generic ? 1 : hidden ? kValuesFewTiles : kValuesFewConsecutive;
            const bool large = tiles_of(ts, g->members) >= kValuesBlockTiles && tiles >= few;
            if (tiles >= kValuesLaunchTiles || large) g = nullptr;
        }
        if (!g) {
            groups.emplace_back();
            g = &groups.back();
            g->variant = own;
        }
        g->members.insert(g->members.end(), of.begin(), of.end());
    }
}

// Split a step's tensors into launches: tensors that share a specialised kernel and its
// tables form one launch each; fp32-state tensors join one of their dtype or form their own
// (plan_values); everything else (other scheme mixes, float64, mixed dtypes) runs in one launch of
// the generic kernel.  A recipe's table is one launch, or two with many fp32-state tensors or some beside a
// large launch; a step of several can fail after the first of them (AW4_ELAUNCHED).
std::vector<LaunchGroup> plan_launches(const aw4_tensor* ts, int32_t count) {
    std::vector<LaunchGroup> groups;
    LaunchGroup generic, research;
    generic.variant = kGenericVariant;
    research.variant = kResearchVariant;
    std::vector<int> values;
    for (int i = 0; i < count; ++i) {
        const aw4_tensor& t = ts[i];
        if (host_values_only(t)) {
            if (t.param_dtype != t.grad_dtype) generic.members.push_back(i); else values.push_back(i);
            continue;
        }
        const bool research_tensor = research_m2(t.m2);
        const int s1 = mspec(t.m1.rounding, t.m1.flags & spec_flags_mask(t.m1.rounding));
        const int s2 = mspec(t.m2.rounding, t.m2.flags & spec_flags_mask(t.m2.rounding));
        // Specialised kernels access parameters and gradients as 4-value vectors, and those that
        // store parameters through LDS as 16-byte pieces; a row whose addresses do not allow that
        // (a view at an odd offset into a flat buffer) runs the generic kernel, which reads the
        // flag at run time.
        int v = kGenericVariant;
        const bool vec16 = aligned(t.param, 16);
        // ... and their lookup tables hold [-1, 1] for signed codebooks only: a first moment on an
        // unsigned one (no scheme has it) runs the generic kernel.
        const bool m1_signed = t.m1.rounding == AW4_ROUND_FP32 || t.m1.codebook == AW4_CB_NF4 || t.m1.codebook == AW4_CB_SDYN4;
        if (t.param_dtype == t.grad_dtype && (t.flags & AW4_TENSOR_VEC_ALIGNED) && m1_signed)
            for (int k = 0; k < kNumSpecialised; ++k)
                if (kVariants[k].dtype == t.param_dtype && kVariants[k].m1 == s1 && kVariants[k].m2 == s2 &&
                    (vec16 || !lds_tile_io(kVariants[k].m1, kVariants[k].m2, kVariants[k].dtype))) {
                    v = k;
                    break;
                }
        if (v == kGenericVariant) { (research_tensor ? research : generic).members.push_back(i); continue; }
        const bool f1 = t.m1.rounding == AW4_ROUND_FP32, f2 = t.m2.rounding == AW4_ROUND_FP32;
        const int c1 = f1 ? -1 : t.m1.codebook, c2 = f2 ? -1 : t.m2.codebook;
        const int l1 = f1 ? -1 : lut_id_of(t.m1.rounding, c1, t.m1.flags);
        const int l2 = f2 ? -1 : lut_id_of(t.m2.rounding, c2, t.m2.flags);
        LaunchGroup* g = nullptr;
        for (LaunchGroup& c : groups)
            if (c.variant == v && c.cb1 == c1 && c.lut1 == l1 && c.cb2 == c2 && c.lut2 == l2) { g = &c; break; }
        if (!g) {
            groups.emplace_back();
            g = &groups.back();
            g->variant = v; g->cb1 = c1; g->lut1 = l1; g->cb2 = c2; g->lut2 = l2;
        }
        g->members.push_back(i);
    }
    plan_values(ts, values, groups, generic);
    if (!research.members.empty()) groups.push_back(std::move(research));
    if (!generic.members.empty()) groups.push_back(std::move(generic));
    for (LaunchGroup& g : groups) std::sort(g.members.begin(), g.members.end());
    return groups;
}

// The next staging slot with at least `bytes` of pinned host and device memory, once the
// launch that last used it has completed.
// Upload of a staged table: a copy kernel on the launch stream reads the pinned host buffer
// directly.  A DMA copy (hipMemcpyAsync) runs on another engine, and the hand-over to it and
// back cost about 20 us each way between consecutive steps (GPT-2-small: 45 us of idle GPU
// per 330 us step, measured).  `cap` is a power of two >= 4096, so the copy's round-up to
// 16 bytes stays inside both buffers.
constexpr int kStageThreads = 256;

__global__ void __launch_bounds__(kStageThreads) stage_copy_kernel(const uint4* src, uint4* dst, int64_t n16) {
    for (int64_t i = (int64_t)blockIdx.x * kStageThreads + threadIdx.x; i < n16;
         i += (int64_t)gridDim.x * kStageThreads)
        dst[i] = src[i];
}

int upload_slot(const StagingSlot& slot, size_t bytes, hipStream_t s) {
    const int64_t n16 = (int64_t)((bytes + 15) / 16);
    if (n16 <= 0) return AW4_OK;
    if ((size_t)n16 * 16 > slot.cap) return set_error(AW4_EINVAL, "staging: %zu bytes exceed the slot", bytes);
    const int64_t blocks = std::min<int64_t>((n16 + kStageThreads - 1) / kStageThreads, 1024);
    hipLaunchKernelGGL(stage_copy_kernel, dim3((unsigned)blocks), dim3(kStageThreads), 0, s,
                       (const uint4*)slot.host_dev, (uint4*)slot.dev, n16);
    AW4_HIP_CHECK(hipGetLastError());
    return AW4_OK;
}

int acquire_slot(DeviceState* ds, size_t bytes, StagingSlot** out) {
    StagingSlot& slot = ds->slots[ds->next];
    ds->next = (ds->next + 1) % kSlots;
    if (slot.pending) {
        AW4_HIP_CHECK(hipEventSynchronize(slot.done));
        slot.pending = false;
    }
    if (slot.cap < bytes) {
        if (slot.host) ds->retired_host.push_back(slot.host);
        if (slot.dev) AW4_HIP_CHECK(hipFree(slot.dev));
        slot.host = slot.dev = nullptr;
        slot.host_dev = nullptr;
        slot.cap = 0;
        size_t cap = 4096;
        while (cap < bytes) cap *= 2;
        // Coherent: the device reads it uncached, so a slot reused four launches later is never
        // read from a stale cache line.
        AW4_HIP_CHECK(hipHostMalloc(&slot.host, cap, hipHostMallocMapped | hipHostMallocCoherent));
        void* mapped = nullptr;
        AW4_HIP_CHECK(hipHostGetDevicePointer(&mapped, slot.host, 0));
        slot.host_dev = mapped;
        AW4_HIP_CHECK(hipMalloc(&slot.dev, cap));
        slot.cap = cap;
    }
    // The event only tells the host that the launch which read the slot has finished; no data
    // flows from the device to the host through it, so it records without a system-scope fence
    // (a cache write-back between consecutive launches).
    if (!slot.done)
        AW4_HIP_CHECK(hipEventCreateWithFlags(&slot.done, hipEventDisableTiming | hipEventDisableSystemFence));
    *out = &slot;
    return AW4_OK;
}

// One step's launches: the kernel groups and where each group's table sits in the staged bytes.
struct StepLaunch {
    std::vector<LaunchGroup> plan;
    std::vector<size_t> offset;
    std::vector<int64_t> grid;
    size_t bytes = 0;
};

// Bytes of the launch table of n tensors (header, rows, tile starts), and with its padding to 256 bytes.
size_t table_bytes(size_t n) { return sizeof(StepHeader) + sizeof(aw4_tensor) * n + sizeof(int64_t) * (n + 1); }
size_t padded_table_bytes(size_t n) { return (table_bytes(n) + 255) & ~(size_t)255; }

// A step has at most one launch for each specialised variant, the two codebooks of a specialised first
// moment and the second moment's five and floored dyn4, and the two generic ones.
static_assert((12 * kNumSpecialised + 2) * (sizeof(StepHeader) + sizeof(int64_t) + 255) <= kNoallocGroupBytes,
              "the table area of aw4_fused_step_noalloc holds every split of a call that fits it unsplit");

// Validate the rows and plan the launches (no device work, no lock needed).
int prepare_step(const aw4_tensor* tensors, int32_t count, StepLaunch& sl) {
    if (count < 0 || (count > 0 && !tensors)) return set_error(AW4_EINVAL, "aw4_fused_step: bad tensor list");
    if (count == 0) return AW4_OK;
    for (int i = 0; i < count; ++i) {
        const int rc = check_tensor(tensors[i], i);
        if (rc) return rc;
    }
    sl.plan = plan_launches(tensors, count);
    // Launch table of each group, 256-byte aligned: header, tensors[n], tile_start[n + 1].
    sl.offset.resize(sl.plan.size());
    sl.grid.assign(sl.plan.size(), 0);
    sl.bytes = 0;
    for (size_t g = 0; g < sl.plan.size(); ++g) {
        sl.offset[g] = sl.bytes;
        sl.bytes += padded_table_bytes(sl.plan[g].members.size());
    }
    return AW4_OK;
}

// Tiles per wave of a large launch (per_cu: tiles per CU, at least 128): three for the kernels
// that take their tiles in grid order (all specialised ones but the bf16 update-SR and research
// kernels; bound by memory, or memory and issue together); up to twelve for the
// bf16 update-SR kernels and the research m2 kernels, which are bound by their instruction issue
// and gain from loading each workgroup's tables for more tiles, while a launch keeps at least 128
// tiles per CU for each tile of a wave (several rounds of workgroups, so the last round is a
// small share); four for the rest.  Measured on the Llama-3-8B sets with alternating processes,
// ranked as the first process on a fresh box (where the fp32 set streams slower; two boxes per
// variant), which is how the benchmark runs:
//   ZIP-SR fp32: grid order 2 tiles 21.80-22.09 ms, 3 20.83-21.01, 4 21.10-21.16, 12 21.89-21.90;
//     consecutive tiles 2 21.47, 3 21.16-21.19, 4 21.25-21.37, 8 21.90, 12 21.99-22.00 (in later
//     processes on a box grid order at 4-24 tiles ran 19.1-19.6 ms, consecutive 4 19.7-19.8);
//   ZE-EDEN: grid order 2 20.24-20.44, 3 20.33-20.52, 4 20.49-20.50, 12 as 3 in later processes;
//     consecutive 4 21.14-21.16;
//   the bf16 mixed set (consecutive tiles, later processes): 2 tiles 17.87 ms, 4 16.98-17.07,
//     6 16.80-16.83, 8 16.44-16.65, 12 16.35-16.37, 16 16.28-16.38; in grid order at 12, 2% slower;
//   the research kernels (first process), four -> twelve tiles: proxy lookahead 28.4-28.5 ->
//     27.2-27.4 ms, v-proxy 28.0-28.3 -> 27.4-27.5, pending lookahead 33.5-33.6 -> 32.6-32.7,
//     read-back 23.5-23.7 -> 22.6, store-EDEN 28.0 -> 26.4.
int large_tiles_per_wave(int variant, int64_t per_cu) {
    if (variant < kNumSpecialised) {
        const KernelVariant& kv = kVariants[variant];
        if (values_variant(kv)) return 1;
        if (tile_order_grid(kv.m1, kv.m2, kv.dtype)) return 3;
        if ((kind_of(kv.m2) == K_USR && is_16bit(kv.dtype)) || research_kernel(kv.m2))
            return (int)std::max<int64_t>(kTilesPerWave, std::min<int64_t>(12, per_cu / 128));
    }
    return kTilesPerWave;
}

// Write each group's launch table into `dst` (host memory of sl.bytes) and set its grid.
//
// A few tiles per wave and a grid covering all of them: the hardware dispatcher hands each free
// slot the next workgroup, so the tiles in flight stay a narrow, moving window of the index
// space (HBM page locality) and no CU waits on a static share at the end.  Measured on MI355X
// against persistent grids of contiguous per-wave ranges, which stream from thousands of
// far-apart addresses at once and leave a load-imbalance tail.  The kernel picks which tiles a
// wave takes (consecutive ones, or one per grid-sized stride); either way the grid is
// ceil(tiles / tiles per wave) waves.
int fill_step_tables(const aw4_tensor* tensors, StepLaunch& sl, int num_cus, void* dst) {
    for (size_t g = 0; g < sl.plan.size(); ++g) {
        const LaunchGroup& lg = sl.plan[g];
        const int n = (int)lg.members.size();
        StepHeader* h = (StepHeader*)((char*)dst + sl.offset[g]);
        memset(h, 0, sizeof(*h));
        aw4_tensor* rows = (aw4_tensor*)(h + 1);
        int64_t* starts = (int64_t*)(rows + n);
        int64_t acc = 0;
        for (int k = 0; k < n; ++k) {
            rows[k] = tensors[lg.members[k]];
            starts[k] = acc;
            acc += (rows[k].numel + kWaveTile - 1) / kWaveTile;
        }
        starts[n] = acc;
        // Smaller launches take fewer tiles per wave so that their waves still spread over every
        // CU: from 128 tiles per CU 3 or 4; below, one per 16 tiles per CU (16 waves per CU, the
        // four 256-thread workgroups the recipe kernels keep resident: one round of waves), at
        // least 1.  Measured on one 4096^2 ZIP-SR tensor (64 tiles per CU): 4 tiles per wave
        // 52.1-52.2 us, 2 52.7-52.9, 3 56.4-56.6, 1 57.1-57.3; one 1024^2 tensor (4 per CU): 1.
        const int64_t per_cu = acc / (int64_t)num_cus;
        const int tiles_per_wave = per_cu >= 128 || values_variant(kVariants[lg.variant])
                                       ? large_tiles_per_wave(lg.variant, per_cu)
                                                 : (int)std::max<int64_t>(1, std::min<int64_t>(4, per_cu / 16));
        const int64_t waves = (acc + tiles_per_wave - 1) / tiles_per_wave;
        sl.grid[g] = (waves + kWavesPerGroup - 1) / kWavesPerGroup;
        if (sl.grid[g] > 0x7fffffff)
            return set_error(AW4_EINVAL, "aw4_fused_step: %lld tiles exceed one launch", (long long)acc);
        h->count = n;
        h->cb1 = lg.cb1; h->lut1 = lg.lut1; h->cb2 = lg.cb2; h->lut2 = lg.lut2;
        for (int w = 0; w < 2; ++w) {
            const int lut = w == 0 ? lg.lut1 : lg.lut2;
            if (lut < 0) continue;
            h->lin_magic[w] = host_tables().spec.lin[lut].magic;
            h->lin_zero[w] = host_tables().spec.lin[lut].zero;
        }
        h->total_tiles = acc;
        h->tiles_per_wave = tiles_per_wave;
    }
    return AW4_OK;
}

// One step kernel launch of a call that has made `launched` of them: a failure after the first
// is AW4_ELAUNCHED (the step's tensors may be partly updated).  aw4_inject_launch_failure makes
// the launch fail here without attempting it.
int launch_one(const void* fn, unsigned grid, void** args, hipStream_t s, int& launched) {
    const int code = launched > 0 ? AW4_ELAUNCHED : AW4_EHIP;
    if (g_fail_after >= 0 && launched >= g_fail_after) {
        g_fail_after = -1;
        return set_error(code, "step kernel launch %d: failure injected by aw4_inject_launch_failure", launched + 1);
    }
    const hipError_t err = hipLaunchKernel(fn, dim3(grid), dim3(kThreads), args, 0, s);
    if (err != hipSuccess)
        return set_error(code, "step kernel launch %d: %s%s", launched + 1, hipGetErrorString(err),
                         launched > 0 ? " (earlier launches of this step were enqueued)" : "");
    ++launched;
    return AW4_OK;
}

// Launch every group whose table is at dev_base + offset.
int launch_step(const StepLaunch& sl, const char* dev_base, const Tables* tables, hipStream_t s, int& launched) {
    for (size_t g = 0; g < sl.plan.size(); ++g) {
        if (sl.grid[g] == 0) continue;
        const StepHeader* dh = (const StepHeader*)(dev_base + sl.offset[g]);
        void* args[] = {(void*)&dh, (void*)&tables};
        const int rc = launch_one(kVariants[sl.plan[g].variant].fn, (unsigned)sl.grid[g], args, s, launched);
        if (rc) return rc;
    }
    return AW4_OK;
}

// Bytes of group g's launch table, without the padding.
size_t group_table_bytes(const StepLaunch& sl, size_t g) { return table_bytes(sl.plan[g].members.size()); }

// Whether every group can take its table in its launch's arguments.
bool fits_inline(const StepLaunch& sl) {
    for (size_t g = 0; g < sl.plan.size(); ++g)
        if (!kVariants[sl.plan[g].variant].fn_inline || group_table_bytes(sl, g) > (size_t)kInlineTableBytes)
            return false;
    return true;
}

// Launch every group with its table (at host + offset) in the launch's arguments.
int launch_step_inline(const StepLaunch& sl, const uint8_t* host, const Tables* tables, hipStream_t s) {
    InlineArgs a;
    a.tables = tables;
    a.reserved = 0;
    int launched = 0;
    for (size_t g = 0; g < sl.plan.size(); ++g) {
        if (sl.grid[g] == 0) continue;
        memcpy(a.table, host + sl.offset[g], group_table_bytes(sl, g));
        void* args[] = {(void*)&a};
        const int rc = launch_one(kVariants[sl.plan[g].variant].fn_inline, (unsigned)sl.grid[g], args, s, launched);
        if (rc) return rc;
    }
    return AW4_OK;
}

// Staging through kernel arguments: each launch carries up to kArgBytes of the table by value
// and copies them to their place in device memory, so the bytes need no device buffer of the
// host's and no copy engine, and the host's buffer is free again when the call returns (the
// launch packet holds its own copy).  Kernel arguments are limited to 4 KB per launch.
constexpr int kArgBytes = 3584;

struct __align__(16) ArgChunk {
    uint64_t dst;    // device address, 16-byte aligned
    uint32_t n16;    // 16-byte words to copy (at most kArgBytes / 16)
    uint32_t reserved;
    uint4 data[kArgBytes / 16];
};

__global__ void __launch_bounds__(256) stage_args_kernel(const ArgChunk chunk) {
    const uint4* src = (const uint4*)((const char*)__builtin_amdgcn_kernarg_segment_ptr() + offsetof(ArgChunk, data));
    for (uint32_t i = threadIdx.x; i < chunk.n16; i += 256) gaddr<u32x4>(chunk.dst)[i] = ((const u32x4*)src)[i];
}

int upload_by_arguments(const void* src, size_t bytes, uint8_t* dst, hipStream_t s) {
    ArgChunk chunk;
    for (size_t off = 0; off < bytes; off += kArgBytes) {
        const size_t n = std::min<size_t>(kArgBytes, bytes - off);
        memset(&chunk, 0, sizeof(chunk));
        chunk.dst = (uint64_t)(dst + off);
        chunk.n16 = (uint32_t)((n + 15) / 16);
        memcpy(chunk.data, (const char*)src + off, n);
        hipLaunchKernelGGL(stage_args_kernel, dim3(1), dim3(256), 0, s, chunk);
        AW4_HIP_CHECK(hipGetLastError());
    }
    return AW4_OK;
}

// Workgroups of a codec launch: kCodecTiles tiles per wave once that leaves every CU eight workgroups,
// fewer below (the kernels' waves stride over whatever tiles the grid leaves).
unsigned codec_groups(int64_t numel, int num_cus) {
    const int64_t tiles = (numel + kWaveTile - 1) / kWaveTile;
    const int64_t per_wave = std::max<int64_t>(1, std::min<int64_t>(kCodecTiles, tiles / (num_cus * 8 * kWavesPerGroup)));
    const int64_t groups = (tiles + per_wave * kWavesPerGroup - 1) / (per_wave * kWavesPerGroup);
    return (unsigned)std::min<int64_t>(groups, 0x7fffffff);
}

}  // namespace

extern "C" {

int aw4_abi_version(void) { return AW4_ABI_VERSION; }

const char* aw4_last_error(void) { return g_error.c_str(); }

int64_t aw4_encode_tables(void* out, int64_t bytes) {
    const HostTables& ht = host_tables();
    if (!ht.ok) return set_error(AW4_EINVAL, "encode tables: %s", ht.error.c_str());
    const int64_t size = (int64_t)sizeof(ht.t.lut);
    if (!out) return size;
    if (bytes < size) return set_error(AW4_EINVAL, "aw4_encode_tables: need %lld bytes", (long long)size);
    memcpy(out, ht.t.lut, (size_t)size);
    return size;
}

int64_t aw4_linear_tables(void* out, int64_t bytes) {
    const HostTables& ht = host_tables();
    if (!ht.ok) return set_error(AW4_EINVAL, "encode tables: %s", ht.error.c_str());
    const int64_t size = (int64_t)sizeof(ht.spec.lin);
    if (!out) return size;
    if (bytes < size) return set_error(AW4_EINVAL, "aw4_linear_tables: need %lld bytes", (long long)size);
    memcpy(out, ht.spec.lin, (size_t)size);
    return size;
}

int aw4_fused_step(const aw4_tensor* tensors, int32_t count, void* stream) {
    g_error.clear();
    StepLaunch sl;
    int rc = prepare_step(tensors, count, sl);
    if (rc || sl.plan.empty()) return rc;
    std::lock_guard<std::mutex> lock(g_mutex);
    DeviceState* ds = nullptr;
    rc = device_state(&ds);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (fits_inline(sl)) {
        std::vector<uint8_t>& host = ds->inline_host;
        host.resize(sl.bytes);
        rc = fill_step_tables(tensors, sl, ds->num_cus, host.data());
        if (rc) return rc;
        return launch_step_inline(sl, host.data(), ds->tables, s);
    }
    StagingSlot* sp = nullptr;
    rc = acquire_slot(ds, sl.bytes, &sp);
    if (rc) return rc;
    StagingSlot& slot = *sp;
    rc = fill_step_tables(tensors, sl, ds->num_cus, slot.host);
    if (rc) return rc;
    rc = upload_slot(slot, sl.bytes, s);
    if (rc) return rc;
    int launched = 0;
    rc = launch_step(sl, (const char*)slot.dev, ds->tables, s, launched);
    // the slot is in use by whatever was enqueued: it is not reused before that completes
    const hipError_t err = hipEventRecord(slot.done, s);
    slot.pending = err == hipSuccess;
    if (rc) return rc;
    if (err != hipSuccess)
        return set_error(AW4_ELAUNCHED, "hipEventRecord after the step's launches: %s", hipGetErrorString(err));
    return AW4_OK;
}

int aw4_fused_step_noalloc(const aw4_tensor* tensors, int32_t count, void* stream) {
    g_error.clear();
    StepLaunch sl;
    int rc = prepare_step(tensors, count, sl);
    if (rc || sl.plan.empty()) return rc;
    // By the rows, not by how many launches they split into (the area has room for those, kNoallocGroupBytes).
    const size_t unsplit = padded_table_bytes((size_t)count);
    if (unsplit > (size_t)AW4_NOALLOC_TABLE_BYTES || sl.bytes > sizeof(scratch))
        return set_error(AW4_EINVAL,
                         "aw4_fused_step_noalloc: the launch tables of %d tensors need %zu bytes, more than its "
                         "%d-byte table area (use aw4_fused_step)",
                         count, std::max(unsplit, sl.bytes), AW4_NOALLOC_TABLE_BYTES);
    std::lock_guard<std::mutex> lock(g_mutex);
    DeviceState* ds = nullptr;
    rc = device_state(&ds);
    if (rc) return rc;
    std::vector<uint8_t>& host = ds->noalloc_host;
    host.assign(sl.bytes, 0);
    rc = fill_step_tables(tensors, sl, ds->num_cus, host.data());
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    rc = upload_by_arguments(host.data(), sl.bytes, ds->scratch, s);
    if (rc) return rc;
    int launched = 0;
    return launch_step(sl, (const char*)ds->scratch, ds->tables, s, launched);
}

void aw4_inject_launch_failure(int32_t after) { g_fail_after = after < 0 ? -1 : after; }

int aw4_quantize(const float* values, int64_t numel, const aw4_moment* m, void* stream) {
    g_error.clear();
    if (!values || !m || numel <= 0 || numel % kBlock != 0)
        return set_error(AW4_EINVAL, "aw4_quantize: bad arguments (numel %lld)", (long long)numel);
    if (((uint64_t)values) % 16 != 0) return set_error(AW4_EALIGN, "aw4_quantize: values not 16-byte aligned");
    if (m->rounding == AW4_ROUND_FP32) return set_error(AW4_EINVAL, "aw4_quantize: fp32 moment");
    if (m->rounding == AW4_ROUND_LOOKAHEAD_SR)
        return set_error(AW4_EINVAL, "aw4_quantize: lookahead update-SR reads gradients (fused step only)");
    int rc = check_moment(*m, numel, 0, "moment");
    if (rc) return rc;
    std::lock_guard<std::mutex> lock(g_mutex);
    DeviceState* ds = nullptr;
    rc = device_state(&ds);
    if (rc) return rc;
    auto kernel = m->rounding == AW4_ROUND_RTN ? quantize_kernel<K_RTN>
                : m->rounding == AW4_ROUND_STATE_SR ? quantize_kernel<K_SSR> : quantize_kernel<K_USR>;
    hipLaunchKernelGGL(kernel, dim3(codec_groups(numel, ds->num_cus)), dim3(kThreads), 0, (hipStream_t)stream, values, numel, *m,
                       (const Tables*)ds->tables);
    AW4_HIP_CHECK(hipGetLastError());
    return AW4_OK;
}

int aw4_dequantize(const aw4_moment* m, int64_t numel, float* out, void* stream) {
    g_error.clear();
    if (!m || !out || numel <= 0 || numel % kBlock != 0)
        return set_error(AW4_EINVAL, "aw4_dequantize: bad arguments (numel %lld)", (long long)numel);
    if (((uint64_t)out) % 16 != 0) return set_error(AW4_EALIGN, "aw4_dequantize: out not 16-byte aligned");
    if (m->rounding == AW4_ROUND_FP32) return set_error(AW4_EINVAL, "aw4_dequantize: fp32 moment");
    if (m->codebook < 0 || m->codebook >= AW4_NUM_CODEBOOKS || !m->codes || !m->scales)
        return set_error(AW4_EINVAL, "aw4_dequantize: bad moment");
    if (!aligned(m->codes, 2) || !aligned(m->scales, 4)) return set_error(AW4_EALIGN, "aw4_dequantize: misaligned");
    std::lock_guard<std::mutex> lock(g_mutex);
    DeviceState* ds = nullptr;
    int rc = device_state(&ds);
    if (rc) return rc;
    hipLaunchKernelGGL(dequantize_kernel, dim3(codec_groups(numel, ds->num_cus)), dim3(kThreads), 0,
                       (hipStream_t)stream, *m, numel, out, (const Tables*)ds->tables);
    AW4_HIP_CHECK(hipGetLastError());
    return AW4_OK;
}

}  // extern "C"

namespace {

// Segments of 2^18 gradient values for large models, shorter ones (to 2^13) while the launch would have
// fewer than eight workgroups per CU: at 2^18 one 4096^2 gradient is 64 workgroups for 256 CUs, and
// GPT-2-small's 124M values 585, an uneven two or three per CU.
int norm_segment_shift(int64_t values) {
    int shift = kNormShiftMin;
    while (shift < kNormShiftMax && (values >> (shift + 1)) >= 2048) ++shift;
    return shift;
}

// Up to this many gradient values in all the norm pass reads them through the caches, where the step that
// follows finds some of them again; more it reads past the caches, which is faster (2 GB of fp32 gradients 355 ->
// 311 us), and the step finds less.  Measured, us clip and step under ZE-EDEN, through / past the caches:
//   fp32, 16M values 63.1 / 64.4, 64M 211.0 / 217.7, 128M 414.3 / 422.1, 160M 520.3 / 522.8, 192M 619.3 / 621.3,
//     256M 829.8 / 821.1, 512M 1,656 / 1,628;
//   bf16, 64M 165.1 / 165.7, 128M 319.2 / 319.6, 160M 397.0 / 396.9, 192M 472.8 / 470.0, 256M 625.4 / 616.8,
//     512M 1,233 / 1,214.
constexpr int64_t kNormKeepValues = (int64_t)160 << 20;

int64_t norm_segments(int64_t numel, int shift) { return (numel + ((int64_t)1 << shift) - 1) >> shift; }

__global__ void __launch_bounds__(kStageThreads) zero_words_kernel(uint32_t* dst, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * kStageThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kStageThreads)
        dst[i] = 0;
}

// The workgroup counters of a norm pass over `slot` (acquired: its last launch has completed), at least
// `words` of them.  Only the norm pass allocates them, and a kernel before its launch clears new ones: a
// synchronous copy of zeros would have the host wait for all work queued so far.
int norm_counters(StagingSlot& slot, size_t words, hipStream_t s) {
    if (slot.counter_words >= words) return AW4_OK;
    slot.counter_words = 0;
    if (slot.counters) AW4_HIP_CHECK(hipFree(slot.counters));
    slot.counters = nullptr;
    size_t cap = 1024;
    while (cap < words) cap *= 2;
    void* p = nullptr;
    AW4_HIP_CHECK(hipMalloc(&p, cap * sizeof(uint32_t)));
    slot.counters = (uint32_t*)p;
    const size_t blocks = std::min<size_t>((cap + kStageThreads - 1) / kStageThreads, 1024);
    hipLaunchKernelGGL(zero_words_kernel, dim3((unsigned)blocks), dim3(kStageThreads), 0, s, slot.counters, (int64_t)cap);
    AW4_HIP_CHECK(hipGetLastError());
    slot.counter_words = cap;
    return AW4_OK;
}

// The norm pass and coefficient of aw4_clip_coefficient (inv_scale null) and
// aw4_unscale_clip_coefficient.
int norm_prologue(const char* what, const aw4_tensor* tensors, int32_t count, const float* inv_scale,
                  float max_norm, float* norm_out, float* coef_out, float* found_out, void* stream) {
    g_error.clear();
    const bool unscale = inv_scale != nullptr;
    if (count <= 0 || !tensors || !norm_out || !coef_out || (unscale && !found_out))
        return set_error(AW4_EINVAL, "%s: bad arguments", what);
    if (!aligned((uint64_t)norm_out, 4) || !aligned((uint64_t)coef_out, 4) ||
        (unscale && (!aligned((uint64_t)inv_scale, 4) || !aligned((uint64_t)found_out, 4))))
        return set_error(AW4_EALIGN, "%s: device floats not 4-byte aligned", what);
    int result_dtype = tensors[0].grad_dtype;
    int64_t values = 0;
    for (int i = 0; i < count; ++i) {
        const aw4_tensor& t = tensors[i];
        if (!t.grad || t.numel <= 0) return set_error(AW4_EINVAL, "tensor %d: null grad or numel %lld", i,
                                                      (long long)t.numel);
        if (t.grad_dtype != AW4_F32 && t.grad_dtype != AW4_BF16 && t.grad_dtype != AW4_F16)
            return set_error(AW4_EINVAL, "tensor %d: grad dtype %d", i, t.grad_dtype);
        if ((t.flags & AW4_TENSOR_VEC_ALIGNED) && !aligned(t.grad, t.grad_dtype == AW4_F32 ? 16 : 8))
            return set_error(AW4_EALIGN, "tensor %d: VEC_ALIGNED but grad misaligned", i);
        if (t.grad_dtype != result_dtype) result_dtype = AW4_F32;  // torch.stack promotes mixed dtypes
        values += t.numel;
    }
    const int shift = norm_segment_shift(values);
    int64_t segments = 0;
    for (int i = 0; i < count; ++i) segments += norm_segments(tensors[i].numel, shift);
    if (segments > 0x7fffffff) return set_error(AW4_EINVAL, "%s: too many segments", what);
    // header and rows (in the launch's arguments where they fit, else staged), then on the device the
    // partial sums, the per-gradient squared norms and (unscaling) the per-segment non-finite flags
    const size_t table = sizeof(NormHeader) + sizeof(NormRow) * (size_t)count;
    const bool in_args = table <= (size_t)kNormInlineBytes;
    const size_t scratch_at = in_args ? 0 : (table + 255) & ~(size_t)255;
    const size_t bytes = scratch_at + sizeof(double) * ((size_t)segments + (size_t)count) +
                         (unscale ? sizeof(uint32_t) * (size_t)segments : 0);

    std::lock_guard<std::mutex> lock(g_mutex);
    DeviceState* ds = nullptr;
    int rc = device_state(&ds);
    if (rc) return rc;
    StagingSlot* slot = nullptr;
    rc = acquire_slot(ds, bytes, &slot);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int64_t ticket_words = norm_ticket_words(count);
    rc = norm_counters(*slot, (size_t)(ticket_words + norm_group_words(segments) + norm_many_words(count)), s);
    if (rc) return rc;
    NormInlineArgs args;
    NormHeader* h = (NormHeader*)(in_args ? (void*)args.table : slot->host);
    memset(h, 0, sizeof(*h));
    NormRow* rows = (NormRow*)(h + 1);
    int64_t acc = 0;
    const int32_t keep = values <= kNormKeepValues ? kNormKeep : 0;
    for (int i = 0; i < count; ++i) {
        const aw4_tensor& t = tensors[i];
        rows[i] = NormRow{t.grad, t.numel, (int32_t)acc,
                          t.grad_dtype | keep | ((t.flags & AW4_TENSOR_VEC_ALIGNED) ? kNormVec : 0)};
        acc += norm_segments(t.numel, shift);
    }
    h->count = count;
    h->result_dtype = result_dtype;
    h->max_norm = max_norm;
    h->unscale = unscale ? 1 : 0;
    h->total_segments = (int32_t)segments;
    h->segment_shift = shift;
    h->partials = (uint64_t)slot->dev + scratch_at;
    h->norm_sq = h->partials + sizeof(double) * (uint64_t)segments;
    h->tickets = (uint64_t)slot->counters;
    h->groups = (uint64_t)(slot->counters + ticket_words);
    h->norm_out = (uint64_t)norm_out;
    h->coef_out = (uint64_t)coef_out;
    if (unscale) {
        h->inv_scale = (uint64_t)inv_scale;
        h->nonfinite = h->norm_sq + sizeof(double) * (uint64_t)count;
        h->found_out = (uint64_t)found_out;
    }
    if (in_args) {
        hipLaunchKernelGGL(norm_kernel_inline, dim3((unsigned)segments), dim3(kNormThreads), 0, s, args);
    } else {
        rc = upload_slot(*slot, table, s);
        if (!rc)
            hipLaunchKernelGGL(norm_kernel, dim3((unsigned)segments), dim3(kNormThreads), 0, s, (const NormHeader*)slot->dev);
    }
    const hipError_t launched = rc ? hipSuccess : hipGetLastError();
    // the slot is in use by whatever was enqueued; if that cannot be waited for, its counters are not used again
    const hipError_t err = hipEventRecord(slot->done, s);
    slot->pending = err == hipSuccess;
    if (err != hipSuccess) slot->counter_words = 0;
    if (rc) return rc;
    AW4_HIP_CHECK(launched);
    AW4_HIP_CHECK(err);
    return AW4_OK;
}

}  // namespace

extern "C" {

int aw4_clip_coefficient(const aw4_tensor* tensors, int32_t count, float max_norm, float* norm_out,
                         float* coef_out, void* stream) {
    return norm_prologue("aw4_clip_coefficient", tensors, count, nullptr, max_norm, norm_out, coef_out, nullptr,
                         stream);
}

int aw4_unscale_clip_coefficient(const aw4_tensor* tensors, int32_t count, const float* inv_scale, float max_norm,
                                 float* norm_out, float* coef_out, float* found_inf_out, void* stream) {
    if (!inv_scale) return set_error(AW4_EINVAL, "aw4_unscale_clip_coefficient: null inv_scale");
    return norm_prologue("aw4_unscale_clip_coefficient", tensors, count, inv_scale, max_norm, norm_out, coef_out,
                         found_inf_out, stream);
}

int aw4_uniforms(uint64_t seed, uint64_t offset, int64_t n, float* out, void* stream) {
    g_error.clear();
    if (!out || n < 0 || offset > UINT64_MAX - (uint64_t)n) return set_error(AW4_EINVAL, "aw4_uniforms: bad arguments");
    if (n == 0) return AW4_OK;
    const int64_t lanes = (int64_t)(((offset + (uint64_t)n - 1) >> 7) - (offset >> 7) + 1) * 8;
    int64_t groups = (lanes + kThreads - 1) / kThreads;
    if (groups > 4096) groups = 4096;
    hipLaunchKernelGGL(uniforms_kernel, dim3((unsigned)groups), dim3(kThreads), 0, (hipStream_t)stream, seed, offset,
                       n, out);
    AW4_HIP_CHECK(hipGetLastError());
    return AW4_OK;
}

}  // extern "C"

#endif  // AW4_SCHED_ILP_TU
