// What the 16-bit grouped GEMM sources share: element types and their MFMA operands, kernel arguments,
// wave-uniform loads, the 4-byte direct-to-LDS load and the activations of the epilogues.
#pragma once

#include "amoe_common.h"

#include <atomic>
#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 mfma_bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 mfma_f16x8;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float mfma_f32x16;

// What the kernel needs to know about its 16-bit element type: the MFMA operand vector and
// instruction, and the conversions of the epilogues (round to nearest even on the way out).
// Addresses, tiles and the LDS layout only depend on the element size, which the two types share.
template <typename ET>
struct Elem16;
template <>
struct Elem16<bf16_t> {
    typedef mfma_bf16x8 frag_t;
    __device__ static __forceinline__ float lo(uint32_t w) { return bf16_lo(w); }
    __device__ static __forceinline__ float hi(uint32_t w) { return bf16_hi(w); }
    __device__ static __forceinline__ uint32_t pack2(float a, float b) { return pack_bf16x2(a, b); }
    __device__ static __forceinline__ mfma_f32x16 mfma(frag_t a, frag_t b, mfma_f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Elem16<f16_t> {
    typedef mfma_f16x8 frag_t;
    __device__ static __forceinline__ float lo(uint32_t w) { return f16_lo(w); }
    __device__ static __forceinline__ float hi(uint32_t w) { return f16_hi(w); }
    __device__ static __forceinline__ uint32_t pack2(float a, float b) { return pack_f16x2(a, b); }
    __device__ static __forceinline__ mfma_f32x16 mfma(frag_t a, frag_t b, mfma_f32x16 c)
    {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

struct GemmArgs {
    const bf16_t* A;
    const bf16_t* B;
    bf16_t* C;
    bf16_t* C2;
    const int32_t* a_row_map;
    const int32_t* b_row_map;  // weight gradient only
    const float* row_scale;  // gated epilogues: the per-row factor of the gated activation (null = 1)
    const bf16_t* G;         // gated-backward epilogue: gate_up [R, 2N] of the forward pass
    float* partials;         // gated-backward epilogue: [n_ntiles][part_stride] row sums, or null
    int ldg, part_stride;
    const int32_t* offsets;
    const int4* tile_map;
    const int32_t* n_mtiles;
    int lda, ldb, ldc, ldc2;
    long long strideB, strideC;
    int E;
    int Kd;       // rows mode: reduction length
    int M;        // wgrad mode: output rows per expert
    int N;        // output columns
    int n_ntiles;
    int n_mt;     // wgrad mode: M tiles per expert
    int rows_total;  // weight gradient: length of the row maps; gemm_skinny.hip: rows of B (0: Kd)
    int gm, gn;   // blocks of one XCD work on super-tiles of gm x gn tiles
    int sn;       // super-tiles along N
    uint32_t inv_gn, inv_super;                   // ceil(2^32 / gn), .. gm gn (0 for a divisor of 1; weight gradients: see their launches)
    uint32_t inv_gm, inv_sn;                      // weight gradients only
    uint32_t inv_group, inv_n, inv_last, inv_kt;  // gemm_pp.hip, .. gm n_ntiles, n_ntiles, width of the last super-column, Kd / 64
    int first_step;  // gemm_pp.hip: K tile at which the reduction of expert 1 starts, of e times that, modulo Kd / 64 (0: all at the first)
    int max_mtiles;  // rows mode: entries of tile_map (those past the last tile hold expert -1)
    float* split_out;   // EPI_PART: partial sums [splits][M][N]
    int splits, n_real;  // EPI_PART: parts of the reduction, N tiles of one part (n_ntiles counts the tiles of all)
    uint32_t inv_splits, inv_real;   // ceil(2^32 / splits), .. n_real (0 for a divisor of 1)
    int stream_from;  // rows mode: from this number of tiles on B is loaded past the caches (0: never; gemm_skinny.hip: always otherwise)
    int pairs_cus, pairs_always;  // gemm_skinny.hip: compute units; workgroups of two column groups from which on there are always such
    int f16;         // host side only: the operands are float16 (launch the f16 instance), else bf16
};

enum { EPI_STORE = 0, EPI_GATED = 1, EPI_GATED_BWD = 2, EPI_PART = 3, EPI_STORE_PAST = 4 /* gemm_pp.hip: past the caches */ };

namespace {

// Wave-uniform load of one int32 from memory this kernel never writes: read through the
// constant address space, which makes it a scalar load (its own counter, tracked by the
// compiler) instead of a vector load.
__device__ __forceinline__ int scalar_load_i32(const int32_t* ptr)
{
    return *(const __attribute__((address_space(4))) int32_t*)ptr;
}

typedef __attribute__((address_space(3))) void* lptr_t;

// One direct-to-LDS load of 4 bytes per lane: a wave-uniform 64-bit base, a 32-bit byte offset per lane, the
// wave's LDS destination in M0 (lane l lands at M0 + 4 l).  The load is not known to the compiler: whoever
// issues it waits for it (vmcnt) before the data is read.
__device__ __forceinline__ void dma4_sbase(const void* base, uint32_t lane_offset, uint32_t lds_addr)
{
    // (operands the compiler may hold in vector registers although they are wave-uniform)
    const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds_addr);
    const uint64_t b64 = (uint64_t)(uintptr_t)base;
    const uint64_t sb = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b64) |
                        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b64 >> 32)) << 32);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(m0v), "v"(lane_offset), "s"(sb)
                 : "memory");
}

// Phi(g), the normal distribution function of the exact gelu, and exp(-g^2 / 2), which its derivative needs as well.
// |g| < 1.484375: 0.5 + g S(g^2), S of degree 6, off by 2.0e-9 at most.  Beyond it the tail on the far side, exp(-g^2 / 2) times
// a polynomial of degree 7 without a constant term in t = 1 / (1 + 0.4 |g|), off by 4.9e-8 of itself (both fitted to the least
// largest error, coefficients rounded one after the other): below 0 Phi itself, above it 1 less it.  The tail's form alone
// will not do: 1 less a tail of nearly 0.5 keeps every rounding of the tail's chain.
// Error of gelu(g) / g in float32 over all float16 gates up to 8, with erff / with that form alone / so: largest 1.05e-7 / 1.95e-7 /
// 0.90e-7, root mean square 2.06e-8 / 4.73e-8 / 1.89e-8, and in the lower tail 1.5e-6 of its value, where 1 + erff(z) has no
// digit left.  Infinities and NaN come out as with erff: gelu(inf) = inf, gelu(-inf) = -inf * 0 = NaN, the derivative of both
// inf * 0 = NaN.  (No step from |g| to t may meet inf * 0: a Newton step on the reciprocal would.)
// Bound by vector instructions, of which erff takes some 60 and both sides of a branch.  With erff / so, gated backward
// product of 10650 rows, 21 experts, 896 x 4320 321 / 191 us (the tail's form alone 183), of 7512 rows, 114 experts, 3072 x 608
// 201 / 151 (145), of 3969 rows, 6 experts, 1504 x 128 (a tile for every tenth compute unit) 71 / 49 (46); gate_up of the
// first 254 / 232 (225).
__device__ __forceinline__ void gelu_parts(float g, float& phi, float& ex)
{
    const float a = fabsf(g), u = g * g, t = __builtin_amdgcn_rcpf(__builtin_fmaf(0.4f, a, 1.0f));
    ex = __builtin_amdgcn_exp2f(-0.72134752f * u);
    float h = 0.0687517524f;
    h = __builtin_fmaf(h, t, -0.18816857f);
    h = __builtin_fmaf(h, t, 0.10725268f);
    h = __builtin_fmaf(h, t, 0.0545073859f);
    h = __builtin_fmaf(h, t, 0.139302209f);
    h = __builtin_fmaf(h, t, 0.159056231f);
    h = __builtin_fmaf(h, t, 0.159598291f);
    float s = 3.58700191e-07f;
    s = __builtin_fmaf(s, u, -8.34226012e-06f);
    s = __builtin_fmaf(s, u, 0.000113329719f);
    s = __builtin_fmaf(s, u, -0.00118514698f);
    s = __builtin_fmaf(s, u, 0.00997239258f);
    s = __builtin_fmaf(s, u, -0.0664901063f);
    s = __builtin_fmaf(s, u, 0.398942262f);
    const float q = t * ex, tail = g < 0.f ? h * q : __builtin_fmaf(-h, q, 1.0f);
    phi = a < 1.484375f ? __builtin_fmaf(g, s, 0.5f) : tail;
}

// Activation for the bf16 epilogue: the sigmoid's division by the hardware reciprocal (1 ulp; the
// result is rounded to bf16 next) instead of the ten-instruction IEEE division sequence.
template <int ACT>
__device__ __forceinline__ float act_fwd_fast(float g)
{
    if (ACT == AMOE_ACT_SILU) return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g));
    if (ACT == AMOE_ACT_GPT_OSS) return g * __builtin_amdgcn_rcpf(1.0f + __expf(-1.702f * g));
    if (ACT == AMOE_ACT_GELU) {
        float phi, ex;
        gelu_parts(g, phi, ex);
        return g * phi;
    }
    return act_fwd<ACT>(g);
}
// act(g) and act'(g) for the backward epilogue, sharing one sigmoid (hardware reciprocal, see above)
template <int ACT>
__device__ __forceinline__ void act_both_fast(float g, float& f, float& df)
{
    if (ACT == AMOE_ACT_SILU || ACT == AMOE_ACT_GPT_OSS) {
        const float a = ACT == AMOE_ACT_SILU ? 1.0f : 1.702f;
        const float sg = __builtin_amdgcn_rcpf(1.0f + __expf(-a * g));
        f = g * sg;
        df = sg * (1.0f + a * g * (1.0f - sg));
    } else if (ACT == AMOE_ACT_GELU) {
        float phi, ex;
        gelu_parts(g, phi, ex);
        f = g * phi;
        df = phi + g * (0.39894228f * ex);
    } else {
        f = act_fwd<ACT>(g);
        df = act_bwd<ACT>(g);
    }
}

}  // namespace
