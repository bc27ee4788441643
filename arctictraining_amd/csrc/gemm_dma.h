// What the 16-bit GEMM kernels with direct-to-LDS loads through buffer descriptors share (gemm_pp.hip, gemm_short.hip): the
// matrix instruction, the loads, waits and stores, and the lane exchanges of the epilogues.
#pragma once

#include "gemm_common.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float mfma_f32x4;
typedef short i16x4_t __attribute__((ext_vector_type(4)));

namespace {

constexpr uint32_t PP_NOWHERE = 0xFFFFFFF0u;         // a load offset past every operand: the lane receives zeros
constexpr uint32_t PP_DROP = 0x80000000u;            // a store offset past the tile: the lane stores nothing

using T_ = std::true_type;
using F_ = std::false_type;

typedef uint32_t srd_t __attribute__((ext_vector_type(4)));

template <typename ET>
struct Mfma16;
template <>
struct Mfma16<bf16_t> {
    __device__ static __forceinline__ mfma_f32x4 run(mfma_bf16x8 a, mfma_bf16x8 b, mfma_f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
    }
};
template <>
struct Mfma16<f16_t> {
    __device__ static __forceinline__ mfma_f32x4 run(mfma_f16x8 a, mfma_f16x8 b, mfma_f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
    }
};

// 16 bytes per lane from global memory straight into LDS (lane l lands at lds_addr + 16 l): a wave-uniform base,
// a 32-bit byte offset per lane.  Through a buffer descriptor, whose range check returns zeros for PP_NOWHERE:
// rows past an expert's end, columns past the matrix and the K remainder need no clamping and no masking.
// Not known to the compiler: the kernel's own vmcnt waits cover it.
// (lds_addr = lds_base + LDS_OFF is formed in M0 itself)
// STREAM: non-temporal, for what is read once
template <uint32_t LDS_OFF, bool STREAM = false>
__device__ __forceinline__ void pp_dma16(const srd_t& d, uint32_t off, uint32_t lds_base)
{
    if constexpr (STREAM)
        asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen nt lds"
                     :
                     : "s"(lds_base), "v"(off), "s"(d), "n"(LDS_OFF)
                     : "memory", "scc");
    else
        asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                     :
                     : "s"(lds_base), "v"(off), "s"(d), "n"(LDS_OFF)
                     : "memory", "scc");
}
__device__ __forceinline__ srd_t pp_srd(const void* base)
{
    const uint64_t b = (uint64_t)(uintptr_t)base;
    return srd_t{(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b), (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)),
                 PP_NOWHERE, 0x00020000u};
}
// move a descriptor's base on
__device__ __forceinline__ void pp_advance(srd_t& d, uint32_t bytes)
{
    const uint64_t b = (((uint64_t)d[1] << 32) | d[0]) + bytes;
    d[0] = (uint32_t)b;
    d[1] = (uint32_t)(b >> 32);
}

__device__ __forceinline__ void pp_go_back(srd_t& d, uint32_t bytes)
{
    const uint64_t b = (((uint64_t)d[1] << 32) | d[0]) - bytes;
    d[0] = (uint32_t)b;
    d[1] = (uint32_t)(b >> 32);
}

template <int N>
__device__ __forceinline__ void pp_vmwait()
{
    static_assert(N >= 0 && N <= 63, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void pp_fence() { __builtin_amdgcn_sched_barrier(0); }
__device__ __forceinline__ void pp_barrier()
{
    pp_fence();
    __builtin_amdgcn_s_barrier();
    pp_fence();
}
// Between a wavefront's writes to LDS and its reads of what other lanes wrote, and back: the LDS serves a wavefront in order,
// so that only the compiler has to keep the order
__device__ __forceinline__ void pp_lds_turn()
{
    pp_fence();
    asm volatile("" ::: "memory");
}
template <typename T>
__device__ __forceinline__ T pp_lds(uint32_t addr)
{
    return *(const __attribute__((address_space(3))) T*)(uintptr_t)addr;
}

// (x, y) = four consecutive columns each of two 16-column tiles, lane quarter q holding columns 4q..4q+3 of both;
// afterwards quarter q holds columns 8q..8q+7 of the 32: x the first four of them, y the second four.
__device__ __forceinline__ void pp_join(uint32_t& x, uint32_t& y)
{
    auto a = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    auto b = __builtin_amdgcn_permlane16_swap(a[0], a[1], false, false);
    x = b[0];
    y = b[1];
}
// sum over the four lane quarters, in every lane
__device__ __forceinline__ float pp_quarter_sum(float v)
{
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    const float s = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(s), __float_as_uint(s), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// STREAM: written through the L2 (sc1 nt), not into it
template <bool STREAM = false>
__device__ __forceinline__ void pp_store16(__amdgpu_buffer_rsrc_t d, u32x4_t v, uint32_t off, uint32_t soff)
{
    __builtin_amdgcn_raw_buffer_store_b128(v, d, off, soff, STREAM ? 18 : 0);
    // (a 16-byte store reads its data a wait state after it issues, and not only without a scalar offset as the
    // compiler assumes: with the next instruction writing the first of the four registers, lanes 12-15 of each 16
    // stored that instruction's result, in about one row of 200)
    pp_fence();
    asm volatile("s_nop 1");
    pp_fence();
}

// The kernel's arguments, read again from the kernel argument segment at each place that uses them between two
// K loops: held in scalar registers across the loops they would spill.  (The argument struct is the only one.)
typedef const __attribute__((address_space(4))) GemmArgs args_t;
__device__ __forceinline__ args_t& pp_args()
{
    auto k = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(k));
    return *(args_t*)k;
}
// a value the compiler cannot trace: what is derived from it is computed here, not hoisted out of the tile loop
__device__ __forceinline__ int pp_here(int v)
{
    asm volatile("" : "+v"(v));
    return v;
}

}  // namespace
