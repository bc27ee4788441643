// Ragged grouped GEMMs on bf16 / f16 MFMA (v_mfma_f32_32x32x16_bf16 / _f16), f32 accumulate.
//
// Two kernel templates cover the three operand layouts of the expert FFN:
//   grouped_gemm_rows_body (persistent, one workgroup per CU)
//     rows / NN   C[rows_e,:] = A[rows_e,:] @ B[e]        (forward; B is [Kd,N], N contiguous)
//     rows / NT   C[rows_e,:] = A[rows_e,:] @ B[e]^T      (data gradient; B is [N',Kd'] so both K-contiguous)
//   grouped_gemm_wgrad_body (one tile per workgroup)
//     wgrad / TN  C[e] = A[rows_e,:]^T @ B[rows_e,:]      (weight gradient; the reduction runs over the ragged rows)
//
// Tiles of BM x BN x 32 move from global memory straight into LDS (global_load_lds, 16 bytes
// per lane, four stages in flight); the XOR swizzle of the LDS layout is applied on the source
// side.  Fragments are read back with
//   * ds_read_b128 when the operand is K-contiguous in LDS.  A 32-wide K row is 4 chunks of
//     16 bytes; chunk kc of row r sits at position kc ^ ((r >> 2) & 3), which makes the 32
//     rows a half-wave reads cover every group of 4 banks exactly twice and the 4 lanes of
//     each quad distinct groups: conflict-free on the 64-bank LDS of gfx950;
//   * two ds_read_b64_tr_b16 (the transposing LDS read of gfx950) when it is K-strided, i.e.
//     stored [k][column] with the columns contiguous.  The 16 lanes of a group together read a
//     4 (k) x 16 (columns) block -- lane j supplies the address of k row j/4, columns
//     4*(j%4)..+3 -- and lane i of the group receives column i for the 4 k rows, which is the
//     MFMA operand layout.  16-byte chunk c of k row k sits at position c ^ ((k & 3) << 2), so
//     the four k rows a half-wave reads fall into the four different quarters of the banks.
// Every operand layout therefore yields the same accumulator layout: lane l of a 32x32 tile
// holds column l%32.  In the epilogue neighbouring lanes swap one value (DPP) so that each
// lane stores a packed pair of adjacent columns of ONE row; for the gate_up GEMM that pair is
// (gate, up) of one intermediate column, so the gated activation runs on registers.
//
// Row-grouped launches take their (expert, first row, end row) per M tile from a tile map
// that a small kernel builds on the device from the expert offsets: no host sync, empty
// experts simply own no tile.  Tiles are dealt to the 8 XCDs so that the ~32 workgroups resident
// on one XCD cover one super-tile of gm x gn tiles (shared A and B panels in that XCD's L2),
// and super-tiles rotate over the XCDs, which keeps them evenly loaded whatever the routing
// skew.
#include "gemm_common.h"
#include "gemm_calls.h"
#include "gemm_launch.h"

#include <algorithm>

// This file is compiled once per group of entry points (-DAMOE_GEMM_PART=0..3), in parallel: the
// kernels of all groups are instances of the same two templates.
//   0: gate_up forward with the gated activation   1: plain row-grouped products (NN, NT)
//   2: data gradient of down + gated-activation backward   3: weight gradients, tile map, shared host helpers
#ifndef AMOE_GEMM_PART
#define AMOE_GEMM_PART -1   // everything in one translation unit
#endif
#define AMOE_PART(n) (AMOE_GEMM_PART < 0 || AMOE_GEMM_PART == (n))

namespace {

constexpr int BK = 32;      // K extent of one LDS stage
constexpr int NSTAGE = 4;   // LDS stages: one being consumed, the others landed or in flight.  (5 stages fit
                            // the 160 KB of LDS and were measured: no faster.)

#if AMOE_PART(3)
// tile map of a caller that brings its own expert offsets (amoe_emit_tile_map has the layout)
__global__ void __launch_bounds__(512)
tile_map_kernel(const int32_t* __restrict__ offsets, int E, int bm, int4* __restrict__ tile_map,
                int32_t* __restrict__ header, int max_mtiles)
{
    __shared__ int32_t row_end[AMOE_MAX_EXPERTS];
    __shared__ int32_t tscan[AMOE_MAX_EXPERTS];
    const int e = threadIdx.x;  // 512 threads, one per possible expert
    if (e < E) row_end[e] = offsets[e + 1] - offsets[0];
    __syncthreads();
    amoe_emit_tile_map<512>(row_end, offsets[0], E, bm, tile_map, header, max_mtiles, tscan);
}
#endif

typedef short tr_i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) tr_i16x4* tr_lptr_t;

// value of the lane whose index differs in bit 0 / bit 1 (DPP quad permutes, no LDS traffic)
__device__ __forceinline__ float lane_xor1(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, true));  // quad_perm [1,0,3,2]
}
__device__ __forceinline__ float lane_xor2(float x)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xF, 0xF, true));  // quad_perm [2,3,0,1]
}

// 16 zero bytes that masked lanes of a direct-to-LDS load read instead of out-of-range rows
static __device__ __attribute__((aligned(16))) uint32_t g_zero_chunk[4] = {0u, 0u, 0u, 0u};

typedef const __attribute__((address_space(1))) void* gptr_t;

// wave-level half of a workgroup barrier for LDS data: this wave's LDS reads have returned and
// all but N of its loads have landed; then the hardware barrier.  (No memory fence: LDS is not
// cached and the direct-to-LDS loads are tracked by vmcnt.)
template <int N>
__device__ __forceinline__ void lds_barrier()
{
    static_assert(N >= 0 && N <= 63, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (0 << 8) | ((N >> 4) << 14));
    __builtin_amdgcn_s_barrier();
}
// One direct-to-LDS load of 16 bytes per lane in its scalar-base form: a wave-uniform 64-bit base, a
// 32-bit byte offset per lane, the wave's LDS destination in M0 (lane l lands at M0 + 16 l).  The
// builtin only produces the form with a 64-bit address per lane, which costs a register pair per
// load and a 64-bit vector add per issue.  The load is not known to the compiler: whoever issues it
// waits for it (vmcnt) before the data is read.  M0 is written and consumed inside one asm statement
// (the compiler reserves M0 and sets it anew before each use of its own; the build's assembly check
// verifies that every write of M0 in these kernels is followed at once by the load that reads it).
__device__ __forceinline__ void dma16_sbase(const void* base, uint32_t lane_offset, uint32_t lds_addr)
{
    // (operands the compiler may hold in vector registers although they are wave-uniform)
    const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds_addr);
    const uint64_t b64 = (uint64_t)(uintptr_t)base;
    const uint64_t sb = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b64) |
                        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b64 >> 32)) << 32);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(m0v), "v"(lane_offset), "s"(sb)
                 : "memory");
}
// workgroup barrier for data exchanged through LDS by ordinary LDS accesses: this wave's LDS traffic
// has completed, then the hardware barrier (loads and stores to global memory stay in flight)
__device__ __forceinline__ void lds_sync()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}
using T_ = std::true_type;
using F_ = std::false_type;

// ------------------------------------------------------------------ weight gradient: one tile per workgroup
// C[e] = A[rows_e,:]^T @ B[rows_e,:]: the reduction runs over the expert's rows, both operands are
// K-strided ([k][column] in LDS, transposing reads).
// MAPS: 1 = the rows of A, 2 = the rows of B are gathered through a row map
// ET: the 16-bit element type (bf16_t or f16_t); GemmArgs names its pointers bf16_t for both
// OUT32: C is float32 (partial sums)
template <int BM, int BN, int WGM, int WGN, int MAPS, typename ET, bool OUT32 = false>
__device__ __forceinline__ void grouped_gemm_wgrad_body(const GemmArgs& p)
{
    typedef typename Elem16<ET>::frag_t frag_t;
    constexpr int NT = WGM * WGN * 64;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int TM = WTM / 32, TN = WTN / 32;
    constexpr bool A_MAP = (MAPS & 1) != 0, B_MAP = (MAPS & 2) != 0;
    static_assert(BM >= 128 && BN >= 128, "K-strided swizzle needs 16 chunks per row");
    constexpr int A_CH = BM * 4, B_CH = BN * 4;   // 16-byte chunks per stage (a 32-wide K row is 4 chunks)
    constexpr int STAGE = A_CH + B_CH;
    constexpr int PER_A = A_CH / NT, PER_B = B_CH / NT;
    static_assert(A_CH % NT == 0 && B_CH % NT == 0, "tile must split evenly over the block");

    extern __shared__ u32x4_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int lj = lane & 31, lg = lane >> 5;

    // ------------------------------------------------------------ block -> tile
    // Workgroups are dealt to the 8 XCDs round-robin.  The ~32 workgroups resident on one XCD
    // are made to cover one gm x gn super-tile, so its gm A panels and gn B panels are fetched
    // into that XCD's L2 once and shared; super-tiles themselves rotate over the XCDs.
    const int b = blockIdx.x;
    const int xcd = b & 7;
    const int q = b >> 3;
    const int per_super = p.gm * p.gn;
    const int sid = (q / per_super) * 8 + xcd;
    const int w = q % per_super;
    const int sm = sid / p.sn, sn_i = sid - sm * p.sn;
    const int pm = sm * p.gm + w / p.gn;
    const int nt = sn_i * p.gn + w % p.gn;
    if (nt >= p.n_ntiles) return;
    const int e = pm / p.n_mt;
    if (e >= p.E) return;
    const int m0 = (pm - e * p.n_mt) * BM;
    const int mend = p.M;   // output rows per expert
    const int r0 = p.offsets[e], r1 = p.offsets[e + 1];
    const int kt_count = (r1 - r0 + BK - 1) / BK;
    const int n0 = nt * BN;

    // ------------------------------------------------------------ global load plans
    // Loads go straight from global memory into LDS: lane l of a wave fills the 16-byte chunk
    // (wave's base + l), so chunk c = tid + NT*i of a stage is filled by thread tid in its i-th
    // load.  The XOR swizzle of the LDS layout is applied on the SOURCE side: the thread that
    // fills physical chunk c fetches the logical chunk that belongs there.
    uint32_t aoff[PER_A], boff[PER_B];
    int a_kr[PER_A], b_kr[PER_B];  // wgrad: k row of the chunk, for the ragged-end mask
    const bf16_t* Ab = p.A;
    const bf16_t* Bb = p.B;
#pragma unroll
    for (int i = 0; i < PER_A; ++i) {
        const int c = tid + NT * i;
        constexpr int CPR = BM / 8;
        const int krow = c / CPR, mc = (c % CPR) ^ ((krow & 3) << 2);
        const int col = min(m0 + mc * 8, p.lda - 8);
        aoff[i] = A_MAP ? (uint32_t)col : (uint32_t)krow * (uint32_t)p.lda + col;
        a_kr[i] = krow;
    }
#pragma unroll
    for (int i = 0; i < PER_B; ++i) {
        const int c = tid + NT * i;
        constexpr int CPR = BN / 8;
        const int krow = c / CPR, nc = (c % CPR) ^ ((krow & 3) << 2);
        const int col = min(n0 + nc * 8, p.N - 8);
        boff[i] = B_MAP ? (uint32_t)col : (uint32_t)krow * (uint32_t)p.ldb + col;
        b_kr[i] = krow;
    }
    if (!A_MAP) Ab += (long long)r0 * p.lda;
    if (!B_MAP) Bb += (long long)r0 * p.ldb;
    const int k_rows = r1 - r0;  // rows of this expert

    // Gathered operands of the weight gradient: the source row of a chunk changes with every K
    // tile.  One wave-wide load covers RPW consecutive k rows starting at a wave-uniform row, so
    // the row indices are fetched with SCALAR loads (their own counter: a vector load here would
    // have to be awaited together with every direct-to-LDS load issued before it; the maps are
    // only ever read by this kernel, which is what a scalar load requires) into a_snx /
    // b_snx one tile ahead, and spread to the lanes (a_use / b_use) right after the fragment
    // wait at the start of the step whose loads use them.
    constexpr int RPW_A = 64 / (BM / 8), RPW_B = 64 / (BN / 8);
    int a_use[PER_A], b_use[PER_B];
    int a_snx[PER_A][RPW_A], b_snx[PER_B][RPW_B];
    auto sfetch_a = [&](int kt, int (&dst)[PER_A][RPW_A]) {
#pragma unroll
        for (int i = 0; i < PER_A; ++i)
#pragma unroll
            for (int q = 0; q < RPW_A; ++q)
                dst[i][q] = scalar_load_i32(p.a_row_map + min(r0 + kt * BK + (wave * 64 + NT * i) / (BM / 8) + q, p.rows_total - 1));
    };
    auto sfetch_b = [&](int kt, int (&dst)[PER_B][RPW_B]) {
#pragma unroll
        for (int i = 0; i < PER_B; ++i)
#pragma unroll
            for (int q = 0; q < RPW_B; ++q)
                dst[i][q] = scalar_load_i32(p.b_row_map + min(r0 + kt * BK + (wave * 64 + NT * i) / (BN / 8) + q, p.rows_total - 1));
    };
    // Each fetched index passes through an empty asm statement as a scalar register first: a
    // select between two values that are still loads from the index array would be folded into
    // one load at a selected address, which turns the array into scratch memory.
    auto spread_a = [&](const int (&src)[PER_A][RPW_A], int (&dst)[PER_A]) {
#pragma unroll
        for (int i = 0; i < PER_A; ++i) {
            int v = 0;
#pragma unroll
            for (int q = 0; q < RPW_A; ++q) {
                int sq = src[i][q];
                asm("" : "+s"(sq));
                v = (q == 0 || lane / (BM / 8) == q) ? sq : v;
            }
            dst[i] = v;
        }
    };
    auto spread_b = [&](const int (&src)[PER_B][RPW_B], int (&dst)[PER_B]) {
#pragma unroll
        for (int i = 0; i < PER_B; ++i) {
            int v = 0;
#pragma unroll
            for (int q = 0; q < RPW_B; ++q) {
                int sq = src[i][q];
                asm("" : "+s"(sq));
                v = (q == 0 || lane / (BN / 8) == q) ? sq : v;
            }
            dst[i] = v;
        }
    };

    const bf16_t* zero_src = reinterpret_cast<const bf16_t*>(g_zero_chunk);
    asm volatile("" : "+s"(zero_src));  // keep the address in registers (not re-derived per load)
    // wgrad: rows past the end of the expert read a block of zeros instead (only the last K
    // tile of an expert can be ragged, the select costs two VALU ops per load)
    auto dma_a = [&](int kt, auto LO, auto HI, const int (&idx)[PER_A]) {
        constexpr int lo = decltype(LO)::value, hi = decltype(HI)::value;
        const int k0 = kt * BK;
        u32x4_t* sa = smem + (kt % NSTAGE) * STAGE + wave * 64;
        const bf16_t* a_base = A_MAP ? Ab : Ab + (long long)k0 * p.lda;
#pragma unroll
        for (int i = lo; i < hi; ++i) {
            const bf16_t* src = a_base + aoff[i];
            if (A_MAP) src += (long long)idx[i] * p.lda;
            src = (k0 + a_kr[i] < k_rows) ? src : zero_src;
            __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(sa + NT * i), 16, 0, 0);
        }
    };
    auto dma_b = [&](int kt, auto LO, auto HI, const int (&idx)[PER_B]) {
        constexpr int lo = decltype(LO)::value, hi = decltype(HI)::value;
        const int k0 = kt * BK;
        u32x4_t* sb = smem + (kt % NSTAGE) * STAGE + A_CH + wave * 64;
        const bf16_t* b_base = B_MAP ? Bb : Bb + (long long)k0 * p.ldb;
#pragma unroll
        for (int i = lo; i < hi; ++i) {
            const bf16_t* src = b_base + boff[i];
            if (B_MAP) src += (long long)idx[i] * p.ldb;
            src = (k0 + b_kr[i] < k_rows) ? src : zero_src;
            __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(sb + NT * i), 16, 0, 0);
        }
    };
    auto issue_a = [&](int kt, auto LO, auto HI) { dma_a(kt, LO, HI, a_use); };
    auto issue_b = [&](int kt, auto LO, auto HI) { dma_b(kt, LO, HI, b_use); };

    mfma_f32x16 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // ------------------------------------------------------------ fragment readers
    // One 16-byte register quad per 32-wide tile and 16-deep K step.  Lane -> (k row, 4 columns) inside the 4x16 block its 16-lane group
    // transposes; groups 0/1 take columns 0-15 / 16-31 of the tile, groups 2/3 the k rows 8-15.
    // The transposing read is issued as inline assembly: through the builtin the compiler treats
    // it as possibly aliasing the direct-to-LDS loads in flight and drains them all (vmcnt(0))
    // before every read.  The compiler therefore does not track these reads; settle() below
    // waits for them and ties the fragments to the wait.
    const int tr_j = lane & 15, tr_blk = lane >> 4;
    const int tr_col = 16 * (tr_blk & 1) + 4 * (tr_j & 3);   // first of this lane's 4 columns in the tile
    const int tr_k = 8 * (tr_blk >> 1) + (tr_j >> 2);        // its k row inside the K step (+4 for the second read)
    auto read_tr = [&](const u32x4_t* st, auto CPR_, int col0, auto KS) -> u32x4_t {
        constexpr int cpr = decltype(CPR_)::value, ks = decltype(KS)::value;
        const int col = col0 + tr_col;
        const int chunk = (col >> 3) ^ ((tr_j >> 2) << 2);
        const uint32_t addr = (uint32_t)(uintptr_t)(lptr_t)st + (uint32_t)((tr_k * cpr + chunk) * 16 + (col & 7) * 2);
        u32x2_t lo, hi;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "i"(ks * 16 * cpr * 16));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "i"((ks * 16 + 4) * cpr * 16));
        return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    };
    auto read_a = [&](const u32x4_t* sa, auto KS, frag_t (&fa)[TM], auto LIVE) {
        [[maybe_unused]] constexpr int ks = decltype(KS)::value;
#pragma unroll
        for (int t = 0; t < decltype(LIVE)::value; ++t) {
            fa[t] = __builtin_bit_cast(frag_t, read_tr(sa, std::integral_constant<int, BM / 8>{}, wm * WTM + t * 32, KS));
        }
    };
    auto read_b = [&](const u32x4_t* sb, auto KS, frag_t (&fb)[TN]) {
        constexpr int ks = decltype(KS)::value;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            fb[t] = __builtin_bit_cast(frag_t, read_tr(sb, std::integral_constant<int, BN / 8>{}, wn * WTN + t * 32, KS));
        }
    };
    // Called before the first MFMA that consumes fragments fetched by read_tr: waits for this
    // wave's LDS reads and makes the fragments depend on the wait (an MFMA is otherwise free to
    // be scheduled ahead of it).
    auto settle = [&](frag_t (&fa)[TM], frag_t (&fb)[TN], auto LIVE) {
        asm volatile("s_waitcnt lgkmcnt(0)");
#pragma unroll
        for (int t = 0; t < decltype(LIVE)::value; ++t) asm volatile("" : "+v"(fa[t]));   // only the blocks that were read
#pragma unroll
        for (int t = 0; t < TN; ++t) asm volatile("" : "+v"(fb[t]));
    };
    // quarter Q of a K step's MFMAs (A tile outer, B tile inner)
    constexpr int N_MFMA = TM * TN;
    static_assert(N_MFMA % 4 == 0, "a K step is issued in four chunks");
    auto mma_quarter = [&](const frag_t (&fa)[TM], const frag_t (&fb)[TN], auto Q, auto LIVE) {
        constexpr int q = decltype(Q)::value;
#pragma unroll
        for (int f = q * (N_MFMA / 4); f < (q + 1) * (N_MFMA / 4); ++f) {
            const int i = f / TN, j = f % TN;
            if (i >= decltype(LIVE)::value) continue;   // a 32-row block past the end of the expert
            acc[i][j] = Elem16<ET>::mfma(fa[i], fb[j], acc[i][j]);
        }
    };

    // ------------------------------------------------------------ main loop
    // NSTAGE LDS stages of one 32-wide K tile each (two MFMA K steps); the offsets below are
    // those of NSTAGE = 4.  Iteration j works on tile j (stage j % 4):
    //   step A: MFMAs on the ks=0 fragments | fetch the ks=1 fragments of tile j
    //           | issue the B half of the loads of tile j+3
    //   wait until tile j+1 has landed (the loads of tiles j+2, j+3 may stay in flight), barrier:
    //           tile j+1 is visible and stage j % 4 is free (every wave holds its last fragments)
    //   step B: MFMAs on the ks=1 fragments | fetch the ks=0 fragments of tile j+1
    //           | issue the A half of the loads of tile j+4 into the stage just freed
    // so the direct-to-LDS loads trickle out evenly (the L1 path moves 64 bytes a clock, half of
    // what the MFMAs consume at full rate) and each has about two iterations to land.
    // A step is written as four chunks fenced by scheduling barriers, each pairing a quarter of
    // the MFMAs with one kind of side work: A-fragment reads, B-fragment reads, loads, loads.
    // Fragments are double-buffered: a step's reads fill the set the other step consumes.
    constexpr int PER = PER_A + PER_B;
    static_assert((NSTAGE - 2) * PER + PER_A <= 63, "vmcnt is a 6-bit counter");
    using IC0 = std::integral_constant<int, 0>;
    using IC1 = std::integral_constant<int, 1>;
    using IC2 = std::integral_constant<int, 2>;
    using IC3 = std::integral_constant<int, 3>;
    using A_HALF = std::integral_constant<int, (PER_A + 1) / 2>;
    using A_ALL = std::integral_constant<int, PER_A>;
    using B_HALF = std::integral_constant<int, (PER_B + 1) / 2>;
    using B_ALL = std::integral_constant<int, PER_B>;
    frag_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];

    // prologue: tiles 0..2 and the A half of tile 3 go out, tile 0 is awaited
    {
        // row lookups of the first four tiles go out together, ahead of their loads
        int sa4[NSTAGE][PER_A][RPW_A], sb4[NSTAGE][PER_B][RPW_B];
#pragma unroll
        for (int t = 0; t < NSTAGE; ++t) {
            if (A_MAP) sfetch_a(t, sa4[t]);
            if (B_MAP && t < NSTAGE - 1) sfetch_b(t, sb4[t]);
        }
        if (A_MAP) sfetch_a(NSTAGE, a_snx);      // next A tile to go out in the loop
        if (B_MAP) sfetch_b(NSTAGE - 1, b_snx);  // next B tile to go out in the loop
#pragma unroll
        for (int t = 0; t < NSTAGE - 1; ++t) {
            if (t < kt_count) {
                if (A_MAP) spread_a(sa4[t], a_use);
                if (B_MAP) spread_b(sb4[t], b_use);
                // B first: its addresses are known, those of A may still wait for the row map
                dma_b(t, IC0{}, B_ALL{}, b_use);
                dma_a(t, IC0{}, A_ALL{}, a_use);
            }
        }
        if (kt_count > NSTAGE - 1) {
            if (A_MAP) spread_a(sa4[NSTAGE - 1], a_use);
            dma_a(NSTAGE - 1, IC0{}, A_ALL{}, a_use);
        }
    }
    if (kt_count > NSTAGE - 1) {
        lds_barrier<(NSTAGE - 2) * PER + PER_A>();
    } else {
        lds_barrier<0>();
    }
    __builtin_amdgcn_sched_barrier(0);

    // LOAD_B: tile kt+3 exists; LOAD_A: tile kt+4 exists; WAITN: loads younger than tile kt+1
    auto k_tile = [&](auto LIVE, auto LOAD_B, auto LOAD_A, auto WAITN, auto NEXT, int kt) {
        constexpr bool idle = decltype(LIVE)::value == 0;   // this wave owns no live row: it only takes part in the loads
        constexpr bool load_b = decltype(LOAD_B)::value, load_a = decltype(LOAD_A)::value;
        constexpr bool next = decltype(NEXT)::value;
        constexpr int waitn = decltype(WAITN)::value;
        const u32x4_t* sa = smem + (kt % NSTAGE) * STAGE;
        const u32x4_t* sb = sa + A_CH;
        // ---- step A: MFMAs on (fa0, fb0)
        if (!idle) settle(fa0, fb0, LIVE);
        if (B_MAP && load_b) {
            spread_b(b_snx, b_use);     // rows of the B tile whose loads go out in this step
            sfetch_b(kt + NSTAGE, b_snx);
        }
        read_a(sa, IC1{}, fa1, LIVE);
        mma_quarter(fa0, fb0, IC0{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (!idle) read_b(sb, IC1{}, fb1);
        mma_quarter(fa0, fb0, IC1{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (load_b) issue_b(kt + NSTAGE - 1, IC0{}, B_HALF{});
        mma_quarter(fa0, fb0, IC2{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (load_b) issue_b(kt + NSTAGE - 1, B_HALF{}, B_ALL{});
        mma_quarter(fa0, fb0, IC3{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier<waitn>();
        __builtin_amdgcn_sched_barrier(0);
        // ---- step B: MFMAs on (fa1, fb1)
        const u32x4_t* na = smem + ((kt + 1) % NSTAGE) * STAGE;
        if (!idle) settle(fa1, fb1, LIVE);
        if (A_MAP && load_a) {
            spread_a(a_snx, a_use);     // rows of the A tile whose loads go out in this step
            sfetch_a(kt + NSTAGE + 1, a_snx);
        }
        if (next) read_a(na, IC0{}, fa0, LIVE);
        mma_quarter(fa1, fb1, IC0{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (next && !idle) read_b(na + A_CH, IC0{}, fb0);
        mma_quarter(fa1, fb1, IC1{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (load_a) issue_a(kt + NSTAGE, IC0{}, A_HALF{});
        mma_quarter(fa1, fb1, IC2{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (load_a) issue_a(kt + NSTAGE, A_HALF{}, A_ALL{});
        mma_quarter(fa1, fb1, IC3{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
    };
    // Every path through this block ends in the final k_tile, whose first action waits for the
    // fragment reads still outstanding: none is in flight when the epilogue reuses the registers.
    auto run_tiles = [&](auto LIVE) {
    if (kt_count > 0) {
        // W<r>: loads younger than tile kt+1 when r tiles (kt included) remain and none is left to issue
        using W0 = std::integral_constant<int, 0>;
        using W1 = std::integral_constant<int, PER>;
        using W2 = std::integral_constant<int, 2 * PER>;
        using WFULL = std::integral_constant<int, (NSTAGE - 2) * PER>;
        static_assert(NSTAGE == 4 || NSTAGE == 5, "the drain below is written out for 4 or 5 stages");
        read_a(smem, IC0{}, fa0, LIVE);
        if (decltype(LIVE)::value) read_b(smem + A_CH, IC0{}, fb0);
        __builtin_amdgcn_sched_barrier(0);
        int kt = 0;
        for (; kt + NSTAGE < kt_count; ++kt) k_tile(LIVE, T_{}, T_{}, WFULL{}, T_{}, kt);
        if (kt + NSTAGE == kt_count) { k_tile(LIVE, T_{}, F_{}, WFULL{}, T_{}, kt); ++kt; }
        if (NSTAGE == 5) {
            if (kt + 4 == kt_count) { k_tile(LIVE, F_{}, F_{}, W2{}, T_{}, kt); ++kt; }
        }
        if (kt + 3 == kt_count) { k_tile(LIVE, F_{}, F_{}, W1{}, T_{}, kt); ++kt; }
        if (kt + 2 == kt_count) { k_tile(LIVE, F_{}, F_{}, W0{}, T_{}, kt); ++kt; }
        k_tile(LIVE, F_{}, F_{}, W0{}, F_{}, kt);  // kt + 1 == kt_count here, whichever way it was reached
    }
    };
    // Only the 32-row blocks of this wave that hold live rows are read and multiplied: the last tile
    // of an expert is often a sliver, and a block of clamped duplicate rows costs as much as a live
    // one.  The count is wave-uniform and picks one copy of the loop; a wave without live rows still
    // issues its share of the loads and meets the barriers.  (Tests inside one shared loop were
    // measured slower than no skipping at all: they cost the full tiles more than the slivers gain.)
    {
        // (weight gradient: mend is the number of output rows per expert; a wave whose columns all lie
        // past the matrix edge has nothing to multiply either)
        const int live_rows = n0 + wn * WTN < p.N ? min(max(mend - (m0 + wm * WTM), 0), WTM) : 0;
        const int live = (live_rows + 31) >> 5;
        static_assert(TM == 2 || TM == 4, "the dispatch below is written for two or four 32-row blocks per wave");
        if (live >= TM) {
            run_tiles(std::integral_constant<int, TM>{});
        } else if (live == 0) {
            run_tiles(std::integral_constant<int, 0>{});
        } else if (live == 1) {
            run_tiles(std::integral_constant<int, 1>{});
        } else {
            if constexpr (TM == 4) {
                if (live == 2) run_tiles(std::integral_constant<int, 2>{});
                else run_tiles(std::integral_constant<int, 3>{});
            }
        }
    }

    // ------------------------------------------------------------ epilogue
    // Lane l of tile (i, j) holds column j*32 + l%32 for 16 rows; registers v, v+1 (v even) are
    // rows r, r+1.  Each lane converts its two values to one packed pair, lanes 2c and 2c+1
    // exchange the pairs (DPP) and a byte permute leaves the even lane with columns (2c, 2c+1) of
    // row r and the odd lane with those of row r+1: three VALU operations per 4-byte store.
    // Addresses are a wave-uniform row base (scalar arithmetic) plus one per-lane 32-bit offset;
    // tiles that lie entirely inside the matrix take the FULL form without per-store bounds tests.
    if constexpr (OUT32) {
        float* const C32 = reinterpret_cast<float*>(p.C) + (long long)e * p.strideC;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int row = m0 + wm * WTM + i * 32 + 8 * (v >> 2) + 4 * lg + (v & 3), col = n0 + wn * WTN + j * 32 + lj;
                    if (row < mend && col < p.N) C32[(long long)row * p.ldc + col] = acc[i][j][v];
                }
        return;
    }
    bf16_t* Cb = p.C + (long long)e * p.strideC;
    const int odd1 = lj & 1;
    const uint32_t swap_sel = odd1 ? 0x03020706u : 0x05040100u;
    // wave-uniform origin of this wave's part of the tile, and the lane's offset from it (bytes)
    const long long worg = (long long)(m0 + wm * WTM) * p.ldc + n0 + wn * WTN;
    char* cbase = reinterpret_cast<char*>(Cb + worg);
    const uint32_t loff = (uint32_t)((4 * lg + odd1) * p.ldc + (lj & ~1)) * 2u;
    auto epilogue = [&](auto FULL) {
        constexpr bool full = decltype(FULL)::value;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const bool col_ok = full || (n0 + wn * WTN + j * 32 + (lj & ~1) < p.N);
#pragma unroll
                for (int v = 0; v < 16; v += 4) {
                    const int rq = i * 32 + 8 * (v >> 2);           // first of 8 rows, relative to the wave's origin
                    const int rt = wm * WTM + rq + 4 * lg;          // rows rt..rt+3 of the tile
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const uint32_t own = Elem16<ET>::pack2(acc[i][j][v + 2 * u], acc[i][j][v + 2 * u + 1]);
                        const uint32_t got = __builtin_amdgcn_update_dpp(0, own, 0xB1, 0xF, 0xF, true);
                        const uint32_t pk = __builtin_amdgcn_perm(got, own, swap_sel);
                        const bool ok = full || (col_ok && m0 + rt + 2 * u + odd1 < mend);
                        if (ok) {
                            char* rowp = cbase + ((long long)(rq + 2 * u) * p.ldc + j * 32) * 2;
                            *reinterpret_cast<uint32_t*>(rowp + loff) = pk;
                        }
                    }
                }
            }
        }
    };
    if (m0 + BM <= mend && n0 + BN <= p.N) epilogue(T_{}); else epilogue(F_{});
}

// ------------------------------------------------------------------ row-grouped GEMMs: persistent kernel
// One workgroup per CU walks over its share of the tiles (virtual block b, b + grid, b + 2 grid, ...
// with the same virtual block -> tile mapping a one-tile-per-workgroup launch would use, so the
// workgroups of one XCD still work on one super-tile at a time).  The K loops of consecutive tiles
// form one software pipeline: the last four iterations of a tile issue the loads of the first four
// K tiles of the next one, so a tile starts with its operands already in LDS, and what remains
// between two tiles is the epilogue.  What the next tile needs is fetched a tile ahead: its entry
// of the tile map by a scalar load, its gathered row indices by a direct-to-LDS load at the start
// of the current tile (a vector load to registers would have to be awaited together with every
// operand load issued after it).  The row scales of the gated epilogues arrive the same way.
template <int BM, int BN, int WGM, int WGN, bool B_KC, int EPI, int ACT, typename ET>
__device__ __forceinline__ void grouped_gemm_rows_body(const GemmArgs& p)
{
    typedef typename Elem16<ET>::frag_t frag_t;
    constexpr int NT = WGM * WGN * 64;
    constexpr int WTM = BM / WGM, WTN = BN / WGN;
    constexpr int TM = WTM / 32, TN = WTN / 32;
    static_assert(NSTAGE == 4, "the cross-tile pipeline is written for four stages");
    static_assert(BM >= 128 && BN >= 128, "K-strided swizzle needs 16 chunks per row");
    static_assert(NT >= BM, "one thread per tile row for the row-index and row-scale loads");
    constexpr int A_CH = BM * 4, B_CH = BN * 4;   // 16-byte chunks per stage (a 32-wide K row is 4 chunks)
    constexpr int STAGE = A_CH + B_CH;
    constexpr int PER_A = A_CH / NT, PER_B = B_CH / NT;
    constexpr int PER = PER_A + PER_B;
    static_assert(A_CH % NT == 0 && B_CH % NT == 0, "tile must split evenly over the block");
    static_assert((NSTAGE - 2) * PER + PER_A <= 63, "vmcnt is a 6-bit counter");
    // stores every wave issues in the epilogue of a tile without edge tests (at least)
    constexpr int EPI_STORES = EPI == EPI_GATED_BWD ? TM * TN * 16 : (EPI == EPI_GATED ? TM * TN * 4 : TM * TN * 8);
    constexpr int W_AFTER_STORES = -1;
    constexpr int W_LOOSE = (NSTAGE - 2) * PER + EPI_STORES < 63 ? (NSTAGE - 2) * PER + EPI_STORES : 63;

    extern __shared__ u32x4_t smem[];
    // LDS: the stages | row indices of the next tile [NT] | row scales of two tiles [2][BM] | row-sum partials [2 WGN][BM]
    int32_t* s_idx = reinterpret_cast<int32_t*>(smem + NSTAGE * STAGE);
    float* s_rs2 = reinterpret_cast<float*>(s_idx + NT);
    float* s_part = s_rs2 + 2 * BM;

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int lj = lane & 31, lg = lane >> 5;
    const int KT = p.Kd / BK;

    // ------------------------------------------------------------ this workgroup's tiles
    // Virtual blocks b, b + grid, b + 2 grid, ...; virtual block v belongs to XCD v % 8 (the hardware deals
    // workgroups to the XCDs round-robin) and is slot (v / 8) % (gm gn) of super-tile ((v / 8) / (gm gn)) * 8
    // + v % 8: the workgroups resident on one XCD work on one super-tile of gm x gn tiles at a time (its gm A
    // panels and gn B panels are shared in that XCD's L2) and the super-tiles rotate over the XCDs.  Only whole
    // groups of 8 super-tiles are dealt that way: the up to 7 left over would give some XCDs a whole super-tile
    // (about one round of tiles) more than the others, so their tiles go to the XCDs one by one.
    const int per_super = p.gm * p.gn;
    const int n_mtiles = min(scalar_load_i32(p.n_mtiles), p.max_mtiles);
    const int supers = ((n_mtiles + p.gm - 1) / p.gm) * p.sn;
    const int vb_rot = (supers >> 3) * 8 * per_super;      // virtual blocks of the rotated part
    const int vb_total = supers * per_super;
    int vb_next = blockIdx.x;
    auto advance = [&](int& pm, int& nt) -> bool {  // this workgroup's next tile; false: none is left
        while (vb_next < vb_total) {
            const int vb = vb_next;
            vb_next += gridDim.x;
            int sid, w;
            if (vb < vb_rot) {
                const int xcd = vb & 7, q = vb >> 3;
                sid = (q / per_super) * 8 + xcd;
                w = q % per_super;
            } else {
                sid = vb / per_super;
                w = vb - sid * per_super;
            }
            const int sm = sid / p.sn, sn_i = sid - sm * p.sn;
            pm = sm * p.gm + w / p.gn;
            nt = sn_i * p.gn + w % p.gn;
            if (nt < p.n_ntiles && pm < n_mtiles) return true;
        }
        return false;
    };
    auto load_entry = [&](int pm) -> int4 {
        const int32_t* ent = reinterpret_cast<const int32_t*>(p.tile_map + pm);
        int4 v;
        v.x = scalar_load_i32(ent);
        v.y = scalar_load_i32(ent + 1);
        v.z = scalar_load_i32(ent + 2);
        v.w = 0;
        return v;
    };

    // ------------------------------------------------------------ load plans
    // Lane l of a wave fills the 16-byte chunk (wave's base + l) of a stage, so chunk c = tid + NT*i is
    // filled by thread tid in its i-th load; the XOR swizzle of the LDS layout is applied on the
    // source side.  A plan is one 32-bit BYTE offset per load, from the operand's base (A) or the
    // expert's base (B): the loads then take a wave-uniform 64-bit base that moves along K by scalar
    // arithmetic plus that constant per-lane offset, and the K loop spends no vector instruction on
    // addresses.  (The host side rejects operands of 4 GiB or more.)
    auto plan_a = [&](int m0, int mend, bool from_lds, uint32_t (&aoff)[PER_A]) {
#pragma unroll
        for (int i = 0; i < PER_A; ++i) {
            const int c = tid + NT * i;
            const int row = c >> 2, kc = (c & 3) ^ ((row >> 2) & 3);
            int gr = min(m0 + row, mend - 1);
            if (p.a_row_map) gr = from_lds ? s_idx[row] : p.a_row_map[gr];
            aoff[i] = ((uint32_t)gr * (uint32_t)p.lda + kc * 8) * 2u;
        }
    };
    auto plan_b = [&](int n0, uint32_t (&boff)[PER_B]) {
#pragma unroll
        for (int i = 0; i < PER_B; ++i) {
            const int c = tid + NT * i;
            if (B_KC) {
                const int row = c >> 2, kc = (c & 3) ^ ((row >> 2) & 3);
                const int gn = min(n0 + row, p.N - 1);
                boff[i] = ((uint32_t)gn * (uint32_t)p.ldb + kc * 8) * 2u;
            } else {
                constexpr int CPR = BN / 8;
                const int krow = c / CPR, nc = (c % CPR) ^ ((krow & 3) << 2);
                const int col = min(n0 + nc * 8, p.N - 8);
                boff[i] = ((uint32_t)krow * (uint32_t)p.ldb + col) * 2u;
            }
        }
    };
    auto dma_a = [&](int stage, int k0, const uint32_t (&off)[PER_A], auto LO, auto HI) {
        u32x4_t* sa = smem + stage * STAGE + wave * 64;
        const char* a_base = reinterpret_cast<const char*>(p.A + k0);
#pragma unroll
        for (int i = decltype(LO)::value; i < decltype(HI)::value; ++i)
            dma16_sbase(a_base, off[i], (uint32_t)(uintptr_t)(lptr_t)(sa + NT * i));
    };
    auto dma_b = [&](int stage, int k0, const bf16_t* Bb, const uint32_t (&off)[PER_B], auto LO, auto HI) {
        u32x4_t* sb = smem + stage * STAGE + A_CH + wave * 64;
        const char* b_base = reinterpret_cast<const char*>(B_KC ? Bb + k0 : Bb + (long long)k0 * p.ldb);
#pragma unroll
        for (int i = decltype(LO)::value; i < decltype(HI)::value; ++i)
            dma16_sbase(b_base, off[i], (uint32_t)(uintptr_t)(lptr_t)(sb + NT * i));
    };

    mfma_f32x16 acc[TM][TN];

    // ------------------------------------------------------------ fragment readers (see grouped_gemm_wgrad_body)
    const int tr_j = lane & 15, tr_blk = lane >> 4;
    const int tr_col = 16 * (tr_blk & 1) + 4 * (tr_j & 3);
    const int tr_k = 8 * (tr_blk >> 1) + (tr_j >> 2);
    auto read_tr = [&](const u32x4_t* st, auto CPR_, int col0, auto KS) -> u32x4_t {
        constexpr int cpr = decltype(CPR_)::value, ks = decltype(KS)::value;
        const int col = col0 + tr_col;
        const int chunk = (col >> 3) ^ ((tr_j >> 2) << 2);
        const uint32_t addr = (uint32_t)(uintptr_t)(lptr_t)st + (uint32_t)((tr_k * cpr + chunk) * 16 + (col & 7) * 2);
        u32x2_t lo, hi;
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "i"(ks * 16 * cpr * 16));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "i"((ks * 16 + 4) * cpr * 16));
        return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    };
    auto read_a = [&](const u32x4_t* sa, auto KS, frag_t (&fa)[TM], auto LIVE) {
        [[maybe_unused]] constexpr int ks = decltype(KS)::value;
#pragma unroll
        for (int t = 0; t < decltype(LIVE)::value; ++t) {
            const int row = wm * WTM + t * 32 + lj;
            const int kc = ks * 2 + lg;
            fa[t] = __builtin_bit_cast(frag_t, sa[row * 4 + (kc ^ ((row >> 2) & 3))]);
        }
    };
    auto read_b = [&](const u32x4_t* sb, auto KS, frag_t (&fb)[TN]) {
        constexpr int ks = decltype(KS)::value;
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            u32x4_t r;
            if (B_KC) {
                const int row = wn * WTN + t * 32 + lj;
                const int kc = ks * 2 + lg;
                r = sb[row * 4 + (kc ^ ((row >> 2) & 3))];
            } else {
                r = read_tr(sb, std::integral_constant<int, BN / 8>{}, wn * WTN + t * 32, KS);
            }
            fb[t] = __builtin_bit_cast(frag_t, r);
        }
    };
    auto settle = [&](frag_t (&fb)[TN]) {
        if (B_KC) return;
        asm volatile("s_waitcnt lgkmcnt(0)");
#pragma unroll
        for (int t = 0; t < TN; ++t) asm volatile("" : "+v"(fb[t]));
    };
    constexpr int N_MFMA = TM * TN;
    static_assert(N_MFMA % 4 == 0, "a K step is issued in four chunks");
    auto mma_quarter = [&](const frag_t (&fa)[TM], const frag_t (&fb)[TN], auto Q, auto LIVE) {
        constexpr int q = decltype(Q)::value;
#pragma unroll
        for (int f = q * (N_MFMA / 4); f < (q + 1) * (N_MFMA / 4); ++f) {
            const int i = f / TN, j = f % TN;
            if (i >= decltype(LIVE)::value) continue;
            acc[i][j] = Elem16<ET>::mfma(fa[i], fb[j], acc[i][j]);
        }
    };

    using IC0 = std::integral_constant<int, 0>;
    using IC1 = std::integral_constant<int, 1>;
    using IC2 = std::integral_constant<int, 2>;
    using IC3 = std::integral_constant<int, 3>;
    using A_HALF = std::integral_constant<int, (PER_A + 1) / 2>;
    using A_ALL = std::integral_constant<int, PER_A>;
    using B_HALF = std::integral_constant<int, (PER_B + 1) / 2>;
    using B_ALL = std::integral_constant<int, PER_B>;
    frag_t fa0[TM], fb0[TN], fa1[TM], fb1[TN];

    // ------------------------------------------------------------ tile state
    // this tile
    int e, m0, mend, nt, n0;
    uint32_t aoff[PER_A], boff[PER_B];
    const bf16_t* Bb;
    // the next tile of this workgroup, if it has one
    bool have_n;
    int pm_n = 0, nt_n = 0;
    int4 tm_n;
    uint32_t aoff_n[PER_A], boff_n[PER_B];
    const bf16_t* Bb_n = p.B;
#pragma unroll
    for (int i = 0; i < PER_A; ++i) aoff_n[i] = 0;
#pragma unroll
    for (int i = 0; i < PER_B; ++i) boff_n[i] = 0;
    {
        int pm = 0;
        nt = 0;
        if (!advance(pm, nt)) return;
        const int4 tm = load_entry(pm);
        e = tm.x;
        m0 = tm.y;
        mend = tm.z;
        have_n = advance(pm_n, nt_n);
        tm_n = have_n ? load_entry(pm_n) : make_int4(0, 0, 1, 0);
    }
    n0 = nt * BN;
    plan_a(m0, mend, false, aoff);
    plan_b(n0, boff);
    Bb = p.B + (long long)e * p.strideB;

    bool loose = false;     // the previous tile issued this tile's first loads and its epilogue stored without edge tests

    // One 32-wide K tile kt of the current tile; g = running K-tile count of this workgroup (stage g % 4).
    //   step A: MFMAs on the ks=0 fragments | fetch the ks=1 fragments | issue the B loads of K tile g+3
    //   wait until K tile g+1 has landed (the loads of g+2, g+3 may stay in flight), barrier
    //   step B: MFMAs on the ks=1 fragments | fetch the ks=0 fragments of K tile g+1 | issue the A loads
    //           of K tile g+4 into the stage just freed
    // LB / LA: 0 = nothing to load, 1 = K tile kt+3 / kt+4 of this tile, 2 = K tile kt+3-KT / kt+4-KT of the next
    auto k_tile = [&](auto LIVE, auto LB, auto LA, auto WAITN, auto NEXT, int kt, int g) {
        constexpr bool idle = decltype(LIVE)::value == 0;
        constexpr int lb = decltype(LB)::value, la = decltype(LA)::value;
        constexpr bool next = decltype(NEXT)::value;
        constexpr int waitn = decltype(WAITN)::value;
        const u32x4_t* sa = smem + (g & 3) * STAGE;
        const u32x4_t* sb = sa + A_CH;
        const int kb = (lb == 2 ? kt + 3 - KT : kt + 3) * BK;
        const int ka = (la == 2 ? kt + 4 - KT : kt + 4) * BK;
        // ---- step A
        if (!idle) settle(fb0);
        read_a(sa, IC1{}, fa1, LIVE);
        mma_quarter(fa0, fb0, IC0{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (!idle) read_b(sb, IC1{}, fb1);
        mma_quarter(fa0, fb0, IC1{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (lb == 1) dma_b((g + 3) & 3, kb, Bb, boff, IC0{}, B_HALF{});
        if (lb == 2) dma_b((g + 3) & 3, kb, Bb_n, boff_n, IC0{}, B_HALF{});
        mma_quarter(fa0, fb0, IC2{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (lb == 1) dma_b((g + 3) & 3, kb, Bb, boff, B_HALF{}, B_ALL{});
        if (lb == 2) dma_b((g + 3) & 3, kb, Bb_n, boff_n, B_HALF{}, B_ALL{});
        mma_quarter(fa0, fb0, IC3{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (waitn == W_AFTER_STORES) {
            // first two K tiles of a tile whose loads went out before the previous tile's epilogue: the
            // stores of that epilogue are younger than the loads awaited here.  When their number is
            // known (a tile without edge tests stores unconditionally) they may stay in flight.
            if (loose) lds_barrier<W_LOOSE>(); else lds_barrier<(NSTAGE - 2) * PER>();
        } else {
            lds_barrier<waitn>();
        }
        __builtin_amdgcn_sched_barrier(0);
        // ---- step B
        const u32x4_t* na = smem + ((g + 1) & 3) * STAGE;
        if (!idle) settle(fb1);
        if (next) read_a(na, IC0{}, fa0, LIVE);
        mma_quarter(fa1, fb1, IC0{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (next && !idle) read_b(na + A_CH, IC0{}, fb0);
        mma_quarter(fa1, fb1, IC1{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (la == 1) dma_a(g & 3, ka, aoff, IC0{}, A_HALF{});
        if (la == 2) dma_a(g & 3, ka, aoff_n, IC0{}, A_HALF{});
        mma_quarter(fa1, fb1, IC2{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
        if (la == 1) dma_a(g & 3, ka, aoff, A_HALF{}, A_ALL{});
        if (la == 2) dma_a(g & 3, ka, aoff_n, A_HALF{}, A_ALL{});
        mma_quarter(fa1, fb1, IC3{}, LIVE);
        __builtin_amdgcn_sched_barrier(0);
    };
    using W0 = std::integral_constant<int, 0>;
    using W1 = std::integral_constant<int, PER>;
    using WFULL = std::integral_constant<int, (NSTAGE - 2) * PER>;
    using WDYN = std::integral_constant<int, W_AFTER_STORES>;
    // The K loop of one tile, for a wave with LIVE 32-row blocks of live rows.  chain: the loop ends by
    // issuing the first loads of the next tile (whose plan is made here, once its row indices are in LDS).
    auto run_tile = [&](auto LIVE, bool chain, int g0) {
        read_a(smem + (g0 & 3) * STAGE, IC0{}, fa0, LIVE);
        if (decltype(LIVE)::value) {
            read_b(smem + (g0 & 3) * STAGE + A_CH, IC0{}, fb0);
            settle(fb0);   // (nothing to overlap with here; every path below then starts with no read outstanding)
        }
        __builtin_amdgcn_sched_barrier(0);
        int kt = 0;
        if (chain) {
            k_tile(LIVE, IC1{}, IC1{}, WDYN{}, T_{}, kt, g0 + kt); ++kt;
            k_tile(LIVE, IC1{}, IC1{}, WDYN{}, T_{}, kt, g0 + kt); ++kt;
            for (; kt < KT - 4; ++kt) k_tile(LIVE, IC1{}, IC1{}, WFULL{}, T_{}, kt, g0 + kt);
            if (decltype(LIVE)::value) settle(fb0);   // before the plan of the next tile is made in this wave's registers
            plan_a(tm_n.y, tm_n.z, true, aoff_n);
            plan_b(nt_n * BN, boff_n);
            Bb_n = p.B + (long long)tm_n.x * p.strideB;
            __builtin_amdgcn_sched_barrier(0);
            k_tile(LIVE, IC1{}, IC2{}, WFULL{}, T_{}, kt, g0 + kt); ++kt;
            k_tile(LIVE, IC2{}, IC2{}, WFULL{}, T_{}, kt, g0 + kt); ++kt;
            k_tile(LIVE, IC2{}, IC2{}, WFULL{}, T_{}, kt, g0 + kt); ++kt;
            k_tile(LIVE, IC2{}, IC2{}, WFULL{}, F_{}, kt, g0 + kt);
        } else {
            for (; kt + NSTAGE < KT; ++kt) k_tile(LIVE, IC1{}, IC1{}, WFULL{}, T_{}, kt, g0 + kt);
            if (kt + NSTAGE == KT) { k_tile(LIVE, IC1{}, IC0{}, WFULL{}, T_{}, kt, g0 + kt); ++kt; }
            if (kt + 3 == KT) { k_tile(LIVE, IC0{}, IC0{}, W1{}, T_{}, kt, g0 + kt); ++kt; }
            if (kt + 2 == KT) { k_tile(LIVE, IC0{}, IC0{}, W0{}, T_{}, kt, g0 + kt); ++kt; }
            k_tile(LIVE, IC0{}, IC0{}, W0{}, F_{}, kt, g0 + kt);
        }
    };

    // ------------------------------------------------------------ the workgroup's tiles
    int g0 = 0, par = 0;
    bool chained = false;   // the previous tile issued this tile's first loads
    for (;;) {
        const bool have_next = have_n;
        const bool chain = have_next && KT >= 8;
        float* s_rs = s_rs2 + par * BM;
        // the row scales of this tile, parked in LDS for its epilogue (visible after the loop's barriers)
        if (EPI != EPI_STORE) {
            if (p.row_scale) {
                dma4_sbase(p.row_scale, (uint32_t)min(m0 + tid % BM, mend - 1) * 4u,
                           (uint32_t)(uintptr_t)(lptr_t)(s_rs + (wave * 64) % BM));
            } else if (tid < BM) {
                s_rs[tid] = 1.0f;
            }
        }
        // the gathered row indices of the next tile
        if (chain && p.a_row_map) {
            dma4_sbase(p.a_row_map, (uint32_t)min(tm_n.y + tid % BM, tm_n.z - 1) * 4u,
                       (uint32_t)(uintptr_t)(lptr_t)(s_idx + wave * 64));
        }
        // and the tile after the next: which one it is, and its entry of the tile map
        int pm_nn = 0, nt_nn = 0;
        const bool have_nn = have_next && advance(pm_nn, nt_nn);
        const int4 tm_nn = have_nn ? load_entry(pm_nn) : make_int4(0, 0, 1, 0);

        if (!chained) {
            // tiles 0..2 and the A half of tile 3 go out, tile 0 is awaited
#pragma unroll
            for (int t = 0; t < NSTAGE - 1; ++t) {
                if (t < KT) {
                    dma_b((g0 + t) & 3, t * BK, Bb, boff, IC0{}, B_ALL{});
                    dma_a((g0 + t) & 3, t * BK, aoff, IC0{}, A_ALL{});
                }
            }
            if (KT > NSTAGE - 1) {
                dma_a((g0 + NSTAGE - 1) & 3, (NSTAGE - 1) * BK, aoff, IC0{}, A_ALL{});
                lds_barrier<(NSTAGE - 2) * PER + PER_A>();
            } else {
                lds_barrier<0>();
            }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
        {
            // Only the 32-row blocks of this wave that hold live rows are read and multiplied; the count
            // is wave-uniform and picks one copy of the loop (a wave without live rows still issues its
            // share of the loads and meets the barriers).
            const int live_rows = n0 + wn * WTN < p.N ? min(max(mend - (m0 + wm * WTM), 0), WTM) : 0;
            const int live = (live_rows + 31) >> 5;
            static_assert(TM == 2 || TM == 4, "the dispatch below is written for two or four 32-row blocks per wave");
            if (live >= TM) {
                run_tile(std::integral_constant<int, TM>{}, chain, g0);
            } else if (live == 0) {
                run_tile(std::integral_constant<int, 0>{}, chain, g0);
            } else if (live == 1) {
                run_tile(std::integral_constant<int, 1>{}, chain, g0);
            } else {
                if constexpr (TM == 4) {
                    if (live == 2) run_tile(std::integral_constant<int, 2>{}, chain, g0);
                    else run_tile(std::integral_constant<int, 3>{}, chain, g0);
                }
            }
        }

        // ---------------------------------------------------------- epilogue
        // Lane l of tile (i, j) holds column j*32 + l%32 for 16 rows; registers v, v+1 (v even) are
        // rows r, r+1.  Each lane converts its two values to one packed pair, lanes 2c and 2c+1
        // exchange the pairs (DPP) and a byte permute leaves the even lane with columns (2c, 2c+1) of
        // row r and the odd lane with those of row r+1: three VALU operations per 4-byte store.
        // Gated: that pair is (gate, up) of intermediate column c; a second exchange between lanes l
        // and l^2 over two row pairs packs two neighbouring intermediate columns of one row.
        // Addresses are a wave-uniform row base (scalar arithmetic) plus one per-lane 32-bit offset;
        // tiles that lie entirely inside their expert's rows and the matrix take the FULL form
        // without per-store bounds tests.
        const bool tile_full = m0 + BM <= mend && n0 + BN <= p.N;
        // (the lane index passes through an empty asm statement: everything the epilogue derives from
        // it would otherwise be hoisted out of the tile loop and held in registers across the K loops)
        int lane_e = lane;
        asm volatile("" : "+v"(lane_e));
        const int lj = lane_e & 31, lg = lane_e >> 5;
        const int odd1 = lj & 1, odd2 = (lj >> 1) & 1;
        const uint32_t swap_sel = odd1 ? 0x03020706u : 0x05040100u;
        if (EPI == EPI_GATED_BWD) {
            // The accumulators are d_inter[r, c] (c = intermediate column); nothing of it is stored.
            // With (gate, up) = gate_up[r, 2c], gate_up[r, 2c+1] re-read from the forward pass and
            // s = row_scale[r]:  d_gate_up[r, 2c] = s * d * up * act'(gate),  d_gate_up[r, 2c+1] =
            // s * d * act(gate)  (one packed pair per element, no lane exchange needed), and the row
            // sums  sum_c d * up * act(gate)  -- the gradient of s -- are reduced over the tile's columns
            // in a fixed order and written to partials[N tile][row].
            const long long gorg = (long long)(m0 + wm * WTM) * p.ldg + 2 * (n0 + wn * WTN);
            const char* gbase = reinterpret_cast<const char*>(p.G + gorg);
            char* dbase = reinterpret_cast<char*>(p.C + gorg);
            const uint32_t goff = (uint32_t)(4 * lg * p.ldg + 2 * lj) * 2u;
            auto run = [&](auto FULL) {
                constexpr bool full = decltype(FULL)::value;
                // a block = 8 of the 16 values a lane holds of one 32x32 tile (half hh: registers 8hh..8hh+7)
                auto load_block = [&](int i, int j, int hh, uint32_t (&g)[8]) {
                    const bool col_ok = full || (n0 + wn * WTN + j * 32 + lj < p.N);
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        const int v = 8 * hh + u;
                        const int rr = i * 32 + 8 * (v >> 2) + (v & 3);   // row relative to the wave's origin (+ 4*lg in goff)
                        const bool ok = full || (col_ok && m0 + wm * WTM + rr + 4 * lg < mend);
                        const char* rowp = gbase + ((long long)rr * p.ldg + 2 * j * 32) * 2;
                        g[u] = ok ? *reinterpret_cast<const uint32_t*>(rowp + goff) : 0u;
                    }
                };
                uint32_t gcur[8], gnxt[8];
                load_block(0, 0, 0, gcur);
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    float dot[16];
#pragma unroll
                    for (int v = 0; v < 16; ++v) dot[v] = 0.f;
#pragma unroll
                    for (int jh = 0; jh < 2 * TN; ++jh) {
                        const int j = jh >> 1, hh = jh & 1;
                        // the next block's pairs are requested before this block is worked on
                        constexpr int NB = TM * TN * 2;
                        const int b_next = i * 2 * TN + jh + 1;
                        if (b_next < NB) load_block(b_next / (2 * TN), (b_next % (2 * TN)) >> 1, b_next & 1, gnxt);
                        __builtin_amdgcn_sched_barrier(0);
                        const bool col_ok = full || (n0 + wn * WTN + j * 32 + lj < p.N);
#pragma unroll
                        for (int u = 0; u < 8; ++u) {
                            // (fenced every four elements: left alone, the scheduler interleaves all the
                            // activation chains and their temporaries no longer fit beside the accumulators)
                            if (u == 4) __builtin_amdgcn_sched_barrier(0);
                            const int v = 8 * hh + u;
                            const int rr = i * 32 + 8 * (v >> 2) + (v & 3);
                            const float d = acc[i][j][v];
                            const float gate = Elem16<ET>::lo(gcur[u]), up = Elem16<ET>::hi(gcur[u]);
                            float f, df;
                            act_both_fast<ACT>(gate, f, df);
                            const float sd = s_rs[wm * WTM + rr + 4 * lg] * d;
                            dot[v] += d * up * f;
                            const bool ok = full || (col_ok && m0 + wm * WTM + rr + 4 * lg < mend);
                            if (ok) {
                                char* rowp = dbase + ((long long)rr * p.ldg + 2 * j * 32) * 2;
                                *reinterpret_cast<uint32_t*>(rowp + goff) = Elem16<ET>::pack2(sd * up * df, sd * f);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                        if (b_next < NB) {
#pragma unroll
                            for (int u = 0; u < 8; ++u) gcur[u] = gnxt[u];
                        }
                    }
                    if (p.partials) {
                        // sum over the 16 lanes of a row group (its 16 columns), then one slot per
                        // (wave column, half-wave group) and tile row
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            float x = dot[v];
                            x += dpp_f32<AMOE_DPP_QUAD_XOR1>(x);
                            x += dpp_f32<AMOE_DPP_QUAD_XOR2>(x);
                            x += dpp_f32<AMOE_DPP_HALF_MIRROR>(x);
                            x += dpp_f32<AMOE_DPP_MIRROR>(x);
                            if ((lane_e & 15) == 0)
                                s_part[(wn * 2 + ((lane_e >> 4) & 1)) * BM + wm * WTM + i * 32 + 8 * (v >> 2) + 4 * lg + (v & 3)] = x;
                        }
                    }
                }
            };
            if (tile_full) run(T_{}); else run(F_{});
            if (p.partials) {
                lds_sync();
                if (tid < BM && m0 + tid < mend) {
                    float tot = 0.f;
#pragma unroll
                    for (int q = 0; q < 2 * WGN; ++q) tot += s_part[q * BM + tid];
                    p.partials[(long long)nt * p.part_stride + m0 + tid] = tot;
                }
            }
        } else {
            // wave-uniform origin of this wave's part of the tile, and the lane's offset from it (bytes)
            const long long worg = (long long)(m0 + wm * WTM) * p.ldc + n0 + wn * WTN;
            const long long worg2 = (long long)(m0 + wm * WTM) * p.ldc2 + ((n0 + wn * WTN) >> 1);
            char* cbase = reinterpret_cast<char*>(p.C + worg);
            char* c2base = EPI == EPI_GATED ? reinterpret_cast<char*>(p.C2 + worg2) : nullptr;
            const uint32_t loff = (uint32_t)((4 * lg + odd1) * p.ldc + (lj & ~1)) * 2u;
            const uint32_t loff2 = EPI == EPI_GATED ? (uint32_t)((4 * lg + 2 * odd2 + odd1) * p.ldc2 + ((lj >> 1) & ~1)) * 2u : 0u;
            const bool want_c = EPI != EPI_GATED || p.C != nullptr;
            auto epilogue = [&](auto FULL) {
                constexpr bool full = decltype(FULL)::value;
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    // gated: the scales of this lane's 8 rows of tile row i, fetched together ahead of
                    // the column loop (one wait for the batch instead of one per use)
                    float sc[4][2];
                    if (EPI == EPI_GATED) {
#pragma unroll
                        for (int v4 = 0; v4 < 4; ++v4)
#pragma unroll
                            for (int u = 0; u < 2; ++u) sc[v4][u] = s_rs[wm * WTM + i * 32 + 8 * v4 + 4 * lg + 2 * u + odd1];
                    }
#pragma unroll
                    for (int j = 0; j < TN; ++j) {
                        const bool col_ok = full || (n0 + wn * WTN + j * 32 + (lj & ~1) < p.N);
#pragma unroll
                        for (int v = 0; v < 16; v += 4) {
                            const int rq = i * 32 + 8 * (v >> 2);           // first of 8 rows, relative to the wave's origin
                            const int rt = wm * WTM + rq + 4 * lg;          // rows rt..rt+3 of the tile
                            float h[2];
#pragma unroll
                            for (int u = 0; u < 2; ++u) {
                                const uint32_t own = Elem16<ET>::pack2(acc[i][j][v + 2 * u], acc[i][j][v + 2 * u + 1]);
                                const uint32_t got = __builtin_amdgcn_update_dpp(0, own, 0xB1, 0xF, 0xF, true);
                                const uint32_t pk = __builtin_amdgcn_perm(got, own, swap_sel);
                                const bool ok = full || (col_ok && m0 + rt + 2 * u + odd1 < mend);
                                if (EPI == EPI_GATED)
                                    h[u] = sc[v >> 2][u] * Elem16<ET>::hi(pk) * act_fwd_fast<ACT>(Elem16<ET>::lo(pk));
                                if (want_c && ok) {
                                    char* rowp = cbase + ((long long)(rq + 2 * u) * p.ldc + j * 32) * 2;
                                    *reinterpret_cast<uint32_t*>(rowp + loff) = pk;
                                }
                            }
                            if (EPI == EPI_GATED) {
                                // lanes with bit 1 clear keep the first row pair, the others the second
                                const float got = lane_xor2(odd2 ? h[0] : h[1]);
                                const uint32_t hp = odd2 ? Elem16<ET>::pack2(got, h[1]) : Elem16<ET>::pack2(h[0], got);
                                const bool ok = full || (col_ok && m0 + rt + 2 * odd2 + odd1 < mend);
                                if (ok) {
                                    char* rowp = c2base + ((long long)rq * p.ldc2 + j * 16) * 2;
                                    *reinterpret_cast<uint32_t*>(rowp + loff2) = hp;
                                }
                            }
                        }
                    }
                }
            };
            if (tile_full) epilogue(T_{}); else epilogue(F_{});
        }

        if (!have_next) break;
        // ---- the next tile becomes this tile
        e = tm_n.x;
        m0 = tm_n.y;
        mend = tm_n.z;
        nt = nt_n;
        n0 = nt * BN;
        if (chain) {
#pragma unroll
            for (int i = 0; i < PER_A; ++i) aoff[i] = aoff_n[i];
#pragma unroll
            for (int i = 0; i < PER_B; ++i) boff[i] = boff_n[i];
            Bb = Bb_n;
        } else {
            plan_a(m0, mend, false, aoff);
            plan_b(n0, boff);
            Bb = p.B + (long long)e * p.strideB;
        }
        have_n = have_nn;
        pm_n = pm_nn;
        nt_n = nt_nn;
        tm_n = tm_nn;
        chained = chain;
        loose = chain && tile_full;
        g0 += KT;
        par ^= 1;
    }
}

// ------------------------------------------------------------------ host side

template <int BM, int BN, int WGM, int WGN, int MAPS>
__global__ void __launch_bounds__(WGM * WGN * 64)
grouped_gemm_wgrad_bf16_kernel(GemmArgs p)
{
    grouped_gemm_wgrad_body<BM, BN, WGM, WGN, MAPS, bf16_t>(p);
}

// the same kernel on float16 operands (v_mfma_f32_32x32x16_f16)
template <int BM, int BN, int WGM, int WGN, int MAPS>
__global__ void __launch_bounds__(WGM * WGN * 64)
grouped_gemm_wgrad_f16_kernel(GemmArgs p)
{
    grouped_gemm_wgrad_body<BM, BN, WGM, WGN, MAPS, f16_t>(p);
}

// partial sums in float32
__global__ void __launch_bounds__(256)
grouped_gemm_wgrad_parts_bf16_kernel(GemmArgs p)
{
    grouped_gemm_wgrad_body<128, 128, 2, 2, 0, bf16_t, true>(p);
}
__global__ void __launch_bounds__(256)
grouped_gemm_wgrad_parts_f16_kernel(GemmArgs p)
{
    grouped_gemm_wgrad_body<128, 128, 2, 2, 0, f16_t, true>(p);
}

template <int BM, int BN, int WGM, int WGN, bool B_KC, int EPI, int ACT>
__global__ void __launch_bounds__(WGM * WGN * 64)
grouped_gemm_rows_bf16_kernel(GemmArgs p)
{
    grouped_gemm_rows_body<BM, BN, WGM, WGN, B_KC, EPI, ACT, bf16_t>(p);
}
template <int BM, int BN, int WGM, int WGN, bool B_KC, int EPI, int ACT>
__global__ void __launch_bounds__(WGM * WGN * 64)
grouped_gemm_rows_f16_kernel(GemmArgs p)
{
    grouped_gemm_rows_body<BM, BN, WGM, WGN, B_KC, EPI, ACT, f16_t>(p);
}

// F16_OK = false leaves the float16 instance of this shape out of the library
template <int BM, int BN, int WGM, int WGN, bool A_KC, bool B_KC, int EPI, int ACT, int MAPS = 0, bool F16_OK = true>
int launch_cfg(const GemmArgs& a, int grid, hipStream_t s)
{
    constexpr int NT = WGM * WGN * 64;
    constexpr int stage_bytes = NSTAGE * (BM + BN) * BK * 2;
    if (a.f16 && !F16_OK) {
        amoe_set_error("grouped_gemm: this tile_cfg is not available for float16 with this epilogue");
        return AMOE_ERR_UNSUPPORTED;
    }
    if constexpr (A_KC) {
        // row-grouped: persistent workgroups, as many as fit on the device at once
        constexpr int lds_bytes = stage_bytes + NT * 4 + 2 * BM * 4 + (EPI == EPI_GATED_BWD ? 2 * WGN * BM * 4 : 0);
        constexpr int per_cu = (lds_bytes <= 80 * 1024 && NT <= 256) ? 2 : 1;
        const int cus = device_cu_count();
        AMOE_REQUIRE(cus > 0, AMOE_ERR_LAUNCH, "grouped_gemm: cannot read the number of compute units");
        // (a multiple of 8: every XCD then runs the same number of workgroups; `grid` bounds the number of tiles)
        int g = grid < cus * per_cu ? grid : cus * per_cu;
        g = (g + 7) & ~7;
        if constexpr (F16_OK) {
            if (a.f16) return launch_kernel<grouped_gemm_rows_f16_kernel<BM, BN, WGM, WGN, B_KC, EPI, ACT>, NT, lds_bytes>(a, g, s);
        }
        return launch_kernel<grouped_gemm_rows_bf16_kernel<BM, BN, WGM, WGN, B_KC, EPI, ACT>, NT, lds_bytes>(a, g, s);
    } else {
        if constexpr (F16_OK) {
            if (a.f16) return launch_kernel<grouped_gemm_wgrad_f16_kernel<BM, BN, WGM, WGN, MAPS>, NT, stage_bytes>(a, grid, s);
        }
        return launch_kernel<grouped_gemm_wgrad_bf16_kernel<BM, BN, WGM, WGN, MAPS>, NT, stage_bytes>(a, grid, s);
    }
}

struct TileCfg {
    int bm, bn;
};

inline TileCfg pick_cfg(int tile_cfg)
{
    switch (tile_cfg) {
        case 1: return {128, 128};
        case 2: return {256, 128};
        case 3: return {256, 256};
        case 5: return {256, 256};
        default: return {256, 256};
    }
}

template <bool A_KC, bool B_KC, int EPI, int ACT, int MAPS = 0>
int launch_any(const GemmArgs& a, int tile_cfg, int grid, hipStream_t s)
{
    switch (tile_cfg) {
        case 1: return launch_cfg<128, 128, 2, 2, A_KC, B_KC, EPI, ACT, MAPS>(a, grid, s);
        case 3:
            // four waves with 256 accumulator registers each leave the gated-backward epilogue no
            // room for its operands: that shape is not built for it
            if constexpr (EPI == EPI_GATED_BWD) {
                amoe_set_error("grouped_gemm: tile_cfg 3 is not available with the gated-backward epilogue");
                return AMOE_ERR_UNSUPPORTED;
            } else {
                // (in float16 the conversions of the epilogues do not fit beside 256 accumulators in the
                // row-grouped kernel: bfloat16 only there)
                return launch_cfg<256, 256, 2, 2, A_KC, B_KC, EPI, ACT, MAPS, !A_KC>(a, grid, s);
            }
        case 5:
            if constexpr (EPI == EPI_GATED_BWD) {   // spills as well (four tile columns per wave)
                amoe_set_error("grouped_gemm: tile_cfg 5 is not available with the gated-backward epilogue");
                return AMOE_ERR_UNSUPPORTED;
            } else {
                return launch_cfg<256, 256, 4, 2, A_KC, B_KC, EPI, ACT, MAPS>(a, grid, s);
            }
        case 2: return launch_cfg<256, 128, 2, 2, A_KC, B_KC, EPI, ACT, MAPS>(a, grid, s);
        default:
            return AMOE_ERR_BAD_ARG;   // (the default shape is in gemm_pp.hip)
    }
}

}  // namespace

// super-tile shape and grid size for `m_tiles` (upper bound) x `n_ntiles` tiles
static int set_supertiles(GemmArgs& a, long long m_tiles, long long* grid)
{
    // at most 8 N tiles per super-tile, the N super-columns of equal width (11 -> 6 + 5, not 8 + 3)
    const int n_super = (a.n_ntiles + 7) / 8;
    a.gn = (a.n_ntiles + n_super - 1) / n_super;
    a.gm = 32 / a.gn;
    // weight gradient: when all tiles of one expert fit in one round of an XCD's 32 CUs, the
    // expert is the super-tile, so its rows are fetched into one L2 only
    if (a.n_mt > 0 && (long long)a.n_mt * a.n_ntiles <= 32) {
        a.gm = a.n_mt;
        a.gn = a.n_ntiles;
    }
    a.sn = (a.n_ntiles + a.gn - 1) / a.gn;
    const long long sm = (m_tiles + a.gm - 1) / a.gm;
    const long long supers = sm * a.sn;
    *grid = 8 * ((supers + 7) / 8) * a.gm * a.gn;
    auto inverse = [](int d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; };
    a.inv_gn = inverse(a.gn);
    a.inv_super = inverse(a.gm * a.gn);
    // (n / d by multiplication with these is exact while n d < 2^32; every n here is a tile index)
    AMOE_REQUIRE(*grid < (1ll << 31) / 32 && *grid * a.sn < (1ll << 32), AMOE_ERR_UNSUPPORTED, "grouped_gemm: grid too large");
    return AMOE_OK;
}

// workspace: [0,16) tile count, then one int4 per M tile
static inline int ws_max_mtiles(int R, int E, int bm) { return R / bm + E + 1; }

// Tile height of the row-grouped products: that of the tile shape, and with the default one a lower one where an
// expert has few rows on average (gemm_skinny.hip reads the weights once per such tile and is bound by that).
// 128 experts of 2048 x 768, A B[e] of both products, this tile height against 256 rows: 1 row an expert 142 against
// 160 us, 4 rows 219 / 230, 8 rows 232 / 230, 16 rows 248 / 236; 64 experts of 2048 x 1408 (whose 256-column tiles fill
// the last round of workgroups badly) 8 rows 209 / 236, 16 rows 219 / 239; 32 experts of 1024 x 1024 8 rows 39 / 50.
// Uneven loads set the limits: where a sixteenth of the experts has half of the rows, their low tiles read the weights
// again, at 6 rows an expert and 16-row tiles 13 % in the products with B^T (153 / 135 us), at 8 and 32-row tiles
// nothing (135 / 136), at 12 again 14 %.
// Loads that are more uneven than that gain: the rows of 4 an expert all on top_k = 8 of 128 experts of 2048 x 768, gate_up
// and down products 34 / 48 us, those with B^T 63 / 62; all on one expert 26 / 60 and 62 / 77 (more workgroups than 256-row
// tiles make, and the weights that they read again are in the caches).  What is lost is a launch of a few tiles more than
// there are compute units: half of 3 rows an expert on a sixteenth of 64 experts of 2048 x 1408, one product 84 / 51 us,
// the four 316 / 324.  Tiles of their own for the products with B^T, of 32 or 128 rows, win these and lose 2-6 % elsewhere.
static inline int rows_tile_height(int R, int E, int tile_cfg)
{
    if (tile_cfg == 0) {
        if (R <= 4ll * E) return 16;
        if (R <= 8ll * E) return 32;
    }
    return pick_cfg(tile_cfg).bm;
}

int amoe_build_tile_map(const int32_t* offsets, int R, int E, int bm, void* workspace, size_t workspace_bytes,
                        const int4** tile_map, const int32_t** n_mtiles, int* max_mtiles, hipStream_t s, bool ready);

static inline size_t map_bytes(int max_mtiles) { return 16 + sizeof(int4) * (size_t)max_mtiles; }

#if AMOE_PART(3)
// What any of the products needs for any number of rows up to R: a workspace made for the largest call serves the
// smaller ones, some of which have more tiles.  (64: no tile of another type or shape is lower)
AMOE_EXPORT size_t amoe_grouped_gemm_workspace_bytes(int R, int E)
{
    if (R <= 0 || E <= 0) return 0;
    const int lowest = (int)std::min<long long>(R, 4ll * E);
    return map_bytes(std::max(ws_max_mtiles(R, E, 64), ws_max_mtiles(lowest, E, 16)));
}

// What one call asks for: R rows, this type and tile shape (float32: what its 64-row tiles needed, its 128-row ones use less)
size_t amoe_rows_map_bytes(int R, int E, int dtype, int tile_cfg)
{
    return map_bytes(ws_max_mtiles(R, E, dtype == AMOE_F32 ? 64 : rows_tile_height(R, E, tile_cfg & ~AMOE_TILE_MAP_READY)));
}

// ready: the workspace already holds the map for these arguments (AMOE_TILE_MAP_READY); nothing is launched
int amoe_build_tile_map(const int32_t* offsets, int R, int E, int bm, void* workspace, size_t workspace_bytes,
                        const int4** tile_map, const int32_t** n_mtiles, int* max_mtiles, hipStream_t s, bool ready)
{
    int32_t* cnt = (int32_t*)workspace;
    int4* map = (int4*)((char*)workspace + 16);
    *max_mtiles = ws_max_mtiles(R, E, bm);
    AMOE_REQUIRE(workspace_bytes >= map_bytes(*max_mtiles), AMOE_ERR_WORKSPACE, "grouped_gemm: workspace %zu < %zu bytes",
                 workspace_bytes, map_bytes(*max_mtiles));
    *tile_map = map;
    *n_mtiles = cnt;
    if (ready) return AMOE_OK;
    hipLaunchKernelGGL(tile_map_kernel, dim3(1), dim3(512), 0, s, offsets, E, bm, map, cnt, *max_mtiles);
    return amoe_check_launch("tile_map");
}

// Where the tile map of a row-grouped GEMM lives inside its workspace and how tall its tiles are, for a
// caller that builds the map itself (the permutation plan): the float32 kernels use 128-row tiles.
int amoe_tile_map_layout(int R, int E, int dtype, int tile_cfg, void* workspace, size_t workspace_bytes, int4** tile_map,
                         int32_t** n_mtiles, int* bm, int* max_mtiles)
{
    AMOE_REQUIRE(dtype == AMOE_F32 || dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_BAD_ARG, "tile map: bad dtype %d", dtype);
    const int shape = tile_cfg & ~AMOE_TILE_MAP_READY;
    AMOE_REQUIRE(tile_cfg >= 0 && shape <= 5 && shape != 4, AMOE_ERR_BAD_ARG, "tile map: bad tile_cfg %d", tile_cfg);
    AMOE_REQUIRE(R > 0 && E > 0 && E <= AMOE_MAX_EXPERTS, AMOE_ERR_BAD_ARG, "tile map: bad sizes R=%d E=%d", R, E);
    *bm = dtype == AMOE_F32 ? 128 : rows_tile_height(R, E, shape);
    *max_mtiles = ws_max_mtiles(R, E, *bm);
    AMOE_REQUIRE(workspace_bytes >= amoe_rows_map_bytes(R, E, dtype, shape), AMOE_ERR_WORKSPACE, "tile map: workspace %zu < %zu bytes",
                 workspace_bytes, amoe_rows_map_bytes(R, E, dtype, shape));
    *n_mtiles = (int32_t*)workspace;
    *tile_map = (int4*)((char*)workspace + 16);
    return AMOE_OK;
}

#endif

// the default tile shape (gemm_pp.hip)
int amoe_pp_gateup_act(const GemmArgs& a, int act, hipStream_t s);
int amoe_pp_rows(const GemmArgs& a, bool b_kc, hipStream_t s);
int amoe_pp_gated_bwd(const GemmArgs& a, int act, hipStream_t s);
int amoe_pp_wgrad(GemmArgs a, hipStream_t s);
// few rows to reduce over (gemm_short.hip)
int amoe_short_wgrad(GemmArgs a, hipStream_t s);
// few tiles of a deep reduction (gemm_split.hip)
int amoe_split_rows(const GemmArgs& a, bool b_kc, int epi, int act, hipStream_t s);
// few rows per expert (gemm_skinny.hip)
int amoe_skinny_gateup_act(const GemmArgs& a, int act, int bm, hipStream_t s);
int amoe_skinny_nn(const GemmArgs& a, int bm, hipStream_t s);
int amoe_skinny_gateup_routed(const GemmArgs& a, int act, const AmoeRoute& r, hipStream_t s);
int amoe_skinny_nn_combined(const GemmArgs& a, const AmoeCombine& c, hipStream_t s);

// From how many tiles of rows on a product's weights are loaded past the caches (0: never).
// Weights that are read once and that the last-level cache (256 MiB in front of all XCDs) cannot hold until the next call
// are: a read of 1 GB takes 6.3 TB/s with ordinary loads, 7.1 with non-temporal ones, and what lies in the cache stays (of
// weights that fit, the ordinary loads are faster: of 8 experts of 2048 x 768 for one token 10 %).
// Once means one tile of rows; the kernel of 256-row tiles leaves the experts with more to the caches (with 384 rows an expert
// the products of 128 experts of 2048 x 768 were 13 % slower past them).  How many experts have rows at all only the GPU
// knows, so that the kernel of 256-row tiles compares their number: of 154 experts of 960 x 1152 of which a skewed router uses
// some twenty, 1679 tokens took 160 us past the caches and 154 through them.  (The kernel for few rows goes by the bound: with
// both forms in one its registers spill.)
// A gate_up product of a short reduction and many rows is not bound by the reading: it gains nothing, and the caches' dirty
// lines, which ordinary loads would push out meanwhile, are then written under the next product.  K = 352, 79 rows an expert
// 523 us with and 504 without, K = 288, 31 rows 522 / 507, K = 992, 46 rows 298 / 294; past the lines K = 768, 19 rows 227 / 232,
// K = 672, 24 rows 143 / 147.
// Before and after, bf16, K=8 of 128 experts of 2048 x 768: 64 tokens 242 -> 219 us, 3001 tokens 365 -> 341, a training step
// of 509 tokens 905 -> 827; 124 other sizes of such weights 0.98 to 1.19 times faster, 1.04 on average.  Whether a single
// product gains depends on what it finds in the cache and has to displace: only whole passes say something.
static int stream_from(int R, int E, long long strideB, int Kred, bool gate_up)
{
    const long long least = (256ll << 20) / (strideB * 2) + 1;
    if (R > 256ll * E || (R < E ? R : E) < least || (gate_up && Kred < 1024 && R > 28ll * E)) return 0;
    return (int)least;
}

// rows mode driver shared by the three row-grouped entry points
// split, split_bytes: where the parts of a reduction that is cut into parts go (null: it is not cut)
template <bool B_KC, int EPI, int ACT>
static int run_rows_bf16(const void* A, const int32_t* a_row_map, const void* B, const int32_t* offsets, void* C,
                         void* C2, const float* row_scale, int R, int E, int Kred, int N, int ldb, long long strideB, void* workspace,
                         size_t workspace_bytes, int tile_cfg, hipStream_t s, int dtype, float* split, size_t split_bytes, const void* G = nullptr,
                         float* partials = nullptr)
{
    const bool map_ready = (tile_cfg & AMOE_TILE_MAP_READY) != 0;
    tile_cfg &= ~AMOE_TILE_MAP_READY;
    TileCfg tc = pick_cfg(tile_cfg);
    // the kernel addresses A (at most R source rows) and one expert of B with 32-bit byte offsets
    AMOE_REQUIRE((unsigned long long)R * (unsigned long long)Kred * 2ull < (1ull << 32) &&
                     (unsigned long long)Kred * (unsigned long long)N * 2ull < (1ull << 32),
                 AMOE_ERR_UNSUPPORTED, "grouped_gemm: operand of 4 GiB or more (R=%d, K=%d, N=%d)", R, Kred, N);
    GemmArgs a = {};
    int max_mtiles = 0;
    const int bm = rows_tile_height(R, E, tile_cfg);
    int rc = amoe_build_tile_map(offsets, R, E, bm, workspace, workspace_bytes, &a.tile_map, &a.n_mtiles,
                                 &max_mtiles, s, map_ready);
    if (rc) return rc;
    a.A = (const bf16_t*)A;
    a.B = (const bf16_t*)B;
    a.C = (bf16_t*)C;
    a.C2 = (bf16_t*)C2;
    a.f16 = dtype == AMOE_F16;
    a.a_row_map = a_row_map;
    a.row_scale = row_scale;
    a.offsets = offsets;
    a.lda = Kred;
    a.ldb = ldb;
    a.ldc = EPI == EPI_GATED_BWD ? 2 * N : N;
    a.ldc2 = N / 2;
    a.G = (const bf16_t*)G;
    a.ldg = 2 * N;
    a.partials = partials;
    a.part_stride = R;
    a.strideB = strideB;
    a.strideC = 0;
    a.E = E;
    a.Kd = Kred;
    a.M = R;
    a.N = N;
    a.n_ntiles = (N + tc.bn - 1) / tc.bn;
    a.n_mt = 0;
    long long grid = 0;
    a.max_mtiles = max_mtiles;
    // a map that is there already may have been built for another bound of the rows, and then with tiles of another
    // height: the workspace limits their number
    if (map_ready && tile_cfg == 0) {
        const size_t fit = (workspace_bytes - 16) / sizeof(int4);
        a.max_mtiles = fit < (1u << 20) ? (int)fit : 1 << 20;
    }
    a.stream_from = stream_from(R, E, strideB, Kred, EPI == EPI_GATED);
    if (bm < tc.bm) {
        if constexpr (EPI == EPI_GATED) return amoe_skinny_gateup_act(a, ACT, bm, s);
        else if constexpr (EPI == EPI_STORE && !B_KC) return amoe_skinny_nn(a, bm, s);
        // (the products with B^T run on the default kernel, which takes tiles of any height up to its own)
    }
    const int splits = tile_cfg == 0 && split && bm == tc.bm ? amoe_split_count(R, E, Kred, N) : 1;
    if (splits > 1) {
        AMOE_REQUIRE(split_bytes >= (size_t)splits * R * N * sizeof(float), AMOE_ERR_WORKSPACE, "grouped_gemm: %zu bytes for %d parts",
                     split_bytes, splits);
        auto inverse = [](int d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; };
        a.split_out = split;
        a.splits = splits;
        a.n_real = a.n_ntiles;
        a.inv_splits = inverse(splits);
        a.inv_real = inverse(a.n_real);
        a.n_ntiles *= splits;
    }
    rc = set_supertiles(a, max_mtiles, &grid);
    if (rc) return rc;
    if (splits > 1) return amoe_split_rows(a, B_KC, EPI, ACT, s);
    if (tile_cfg == 0) {
        if constexpr (EPI == EPI_GATED) return amoe_pp_gateup_act(a, ACT, s);
        else if constexpr (EPI == EPI_GATED_BWD) return amoe_pp_gated_bwd(a, ACT, s);
        else return amoe_pp_rows(a, B_KC, s);
    }
    return launch_any<true, B_KC, EPI, ACT>(a, tile_cfg, (int)grid, s);
}

#if AMOE_PART(0)
int amoe_bf16_gateup_act(const void* xp, const int32_t* a_row_map, const void* w, const int32_t* offsets, void* gate_up,
                         void* inter, const float* row_scale, int R, int E, int H, int I, int act, void* workspace, size_t workspace_bytes,
                         int tile_cfg, hipStream_t s, int dtype, float* split, size_t split_bytes)
{
    AMOE_DISPATCH_ACT(act, return (run_rows_bf16<false, EPI_GATED, ACT>(xp, a_row_map, w, offsets, gate_up, inter, row_scale, R, E, H,
                                                                        2 * I, 2 * I, (long long)H * 2 * I, workspace,
                                                                        workspace_bytes, tile_cfg, s, dtype, split, split_bytes)))
    return AMOE_ERR_BAD_ARG;
}

#endif

#if AMOE_PART(0)
// Up to 8 tokens: each of the product's workgroups selects for itself and walks over the rows, which pays while that takes less
// than the two launches that it saves, 7 us.  `steps`: how many experts are selected one after the other on a compute unit, which
// holds two workgroups of eight wavefronts or four of four; a wavefront takes the tokens in turn.  One forward pass, us, logits /
// routing / gate_up / down / sums as five launches and as three (T tokens, K of E experts of H x I):
//   more workgroups than are held: 243 experts of 288 x 3712, T=4 K=8 (steps 16) 58 / 58, K=16 (64) 103 / 121, T=8 K=16 (192) 157 / 268
//   two tokens in turn: 64 of 1024 x 512, T=6 K=6 (12) 34 / 35, T=8 K=8 (16) 42 / 45; 128 of 2048 x 768, T=8 K=4 (8) 66 / 67; 243 of
//     288 x 3712, T=8 K=2 (4) 39 / 36
//   R + 3 K: 256 of 512 x 256, T=5 K=10 (80) 32 / 31, T=6 (90) 32 / 33, T=8 K=16 (176) 39 / 48; 64 of 1024 x 512, K=16, T=2 (80)
//     39 / 36, T=3 (96) 44 / 45
//   long rows, whose reading hides it: 32 of 4096 x 1408, T=1 K=8 72 / 66, T=8 K=16 (steps 32) 201 / 199; 32 of 2880 x 2880, T=5 K=8
//     (32) 221 / 216, T=8 K=16 (64) 265 / 268
// One token of 8 of 128 experts of 2048 x 768 34 / 29; passes that are bound by the host 33 / 26.
int amoe_routed_fits(int dtype, int T, int K, int E, int H, int I, int tile_cfg)
{
    if ((dtype != AMOE_BF16 && dtype != AMOE_F16) || tile_cfg != 0 || T > 8 || T * K > 128 || E > 256 || K > E || K > AMOE_MAX_TOPK ||
        rows_tile_height(T * K, E, 0) != 16 || H % 32 || I % 32 || (unsigned long long)H * 2 * I * 2 >= (1ull << 32))
        return 0;
    const int R = T * K, m_tiles = E < R ? E : R, cus = device_cu_count();
    if (cus <= 0) return 0;
    const bool narrow = skinny_narrow(m_tiles, 2 * I, cus);
    const int in_turn = (T + (narrow ? 7 : 3)) / (narrow ? 8 : 4), held = cus * (narrow ? 2 : 4), cols = narrow ? 64 : 128;
    const long long steps = in_turn * K * (((long long)m_tiles * ((2 * I + cols - 1) / cols) + held - 1) / held);
    const bool pays = H >= 2560 ? steps <= 32 : steps <= (in_turn > 1 ? 6 : 16) && R + 3 * K <= 80;
    return pays ? cus : 0;
}

int amoe_run_gateup_routed(const void* x, const void* w_gate_up, void* gate_up, void* inter, const AmoeRoute& r, int dtype, int E, int H, int I,
                           int act, void* workspace, size_t workspace_bytes, hipStream_t s)
{
    AMOE_REQUIRE(x && w_gate_up && inter && r.logits && act >= AMOE_ACT_SILU && act <= AMOE_ACT_GPT_OSS, AMOE_ERR_BAD_ARG,
                 "gateup_routed: bad argument");
    const int R = r.T * r.K;
    GemmArgs a = {};
    AmoeRoute route = r;
    const int4* map = nullptr;
    const int32_t* count = nullptr;
    int rc = amoe_build_tile_map(nullptr, R, E, 16, workspace, workspace_bytes, &map, &count, &a.max_mtiles, s, true);
    if (rc) return rc;
    route.tile_map = const_cast<int4*>(map);
    route.n_mtiles = const_cast<int32_t*>(count);
    a.A = (const bf16_t*)x;
    a.B = (const bf16_t*)w_gate_up;
    a.C = (bf16_t*)gate_up;
    a.C2 = (bf16_t*)inter;
    a.f16 = dtype == AMOE_F16;
    a.lda = a.Kd = H;
    a.ldb = a.ldc = a.N = 2 * I;
    a.ldc2 = I;
    a.strideB = (long long)H * 2 * I;
    a.E = E;
    a.M = R;
    a.stream_from = stream_from(R, E, a.strideB, H, true);
    return amoe_skinny_gateup_routed(a, act, route, s);
}

int amoe_run_down_combined(const void* inter, const void* w_down, void* out, const AmoeCombine& c, int dtype, int E, int H, int I, void* workspace,
                           size_t workspace_bytes, hipStream_t s)
{
    AMOE_REQUIRE(inter && w_down && out && c.arrived && c.row_of && c.y, AMOE_ERR_BAD_ARG, "down_combined: null pointer");
    GemmArgs a = {};
    a.M = c.T * c.K;
    int rc = amoe_build_tile_map(nullptr, a.M, E, 16, workspace, workspace_bytes, &a.tile_map, &a.n_mtiles, &a.max_mtiles, s, true);
    if (rc) return rc;
    a.A = (const bf16_t*)inter;
    a.B = (const bf16_t*)w_down;
    a.C = (bf16_t*)out;
    a.f16 = dtype == AMOE_F16;
    a.lda = a.Kd = I;
    a.ldb = a.ldc = a.N = H;
    a.strideB = (long long)I * H;
    a.E = E;
    a.stream_from = stream_from(a.M, E, a.strideB, I, false);
    return amoe_skinny_nn_combined(a, c, s);
}
#endif

#if AMOE_PART(1)
int amoe_bf16_nn(const void* A, const int32_t* a_row_map, const void* B, const int32_t* offsets, void* C, int R, int E,
                 int Kd, int N, void* workspace, size_t workspace_bytes, int tile_cfg, hipStream_t s, int dtype, float* split,
                 size_t split_bytes)
{
    return run_rows_bf16<false, EPI_STORE, 0>(A, a_row_map, B, offsets, C, nullptr, nullptr, R, E, Kd, N, N, (long long)Kd * N,
                                              workspace, workspace_bytes, tile_cfg, s, dtype, split, split_bytes);
}

// C[rows_e, :Kd] = A[rows_e, :N] @ B[e]^T with B [E, Kd, N]: the reduction runs over N
int amoe_bf16_nt(const void* A, const int32_t* a_row_map, const void* B, const int32_t* offsets, void* C, int R, int E,
                 int Kd, int N, void* workspace, size_t workspace_bytes, int tile_cfg, hipStream_t s, int dtype, float* split,
                 size_t split_bytes)
{
    return run_rows_bf16<true, EPI_STORE, 0>(A, a_row_map, B, offsets, C, nullptr, nullptr, R, E, /*Kred=*/N, /*N out=*/Kd,
                                             /*ldb=*/N, (long long)Kd * N, workspace, workspace_bytes, tile_cfg, s, dtype, split,
                                             split_bytes);
}

#endif

#if AMOE_PART(2)
// d_gate_up [R, 2I] and the row sums of the score gradient from dy rows [., H], w_down [E, I, H] and the
// forward's gate_up [R, 2I]: the data gradient of the down projection with the backward of the gated
// activation as its epilogue.  The reduction runs over H, the output columns are the I intermediate columns.
int amoe_bf16_nt_gated_bwd(const void* dy, const int32_t* a_row_map, const void* w_down, const int32_t* offsets,
                           const void* gate_up, const float* row_scale, void* d_gate_up, float* partials, int R, int E,
                           int I, int H, int act, void* workspace, size_t workspace_bytes, int tile_cfg, hipStream_t s, int dtype,
                           float* split, size_t split_bytes)
{
    AMOE_DISPATCH_ACT(act, return (run_rows_bf16<true, EPI_GATED_BWD, ACT>(dy, a_row_map, w_down, offsets, d_gate_up, nullptr,
                                                                           row_scale, R, E, /*Kred=*/H, /*N out=*/I, /*ldb=*/H,
                                                                           (long long)I * H, workspace, workspace_bytes,
                                                                           tile_cfg, s, dtype, split, split_bytes, gate_up, partials)))
    return AMOE_ERR_BAD_ARG;
}

#endif

#if AMOE_PART(3)
// number of row-sum partials per routed row that amoe_bf16_nt_gated_bwd writes: one per N tile
int amoe_bf16_gated_bwd_parts(int I, int tile_cfg)
{
    TileCfg tc = pick_cfg(tile_cfg & ~AMOE_TILE_MAP_READY);
    return (I + tc.bn - 1) / tc.bn;
}

// lda: elements from one row of A to the next, a multiple of 8; the Kd of the output may be fewer (not with tile_cfg 0)
// out32: C is float32 (tile_cfg 1, nothing gathered)
int amoe_bf16_wgrad(const void* A, const int32_t* a_row_map, const void* B, const int32_t* b_row_map,
                    const int32_t* offsets, void* C, int R, int E, int Kd, int N, int tile_cfg, hipStream_t s, int dtype, int lda, bool out32)
{
    const bool offsets32 = !(a_row_map || b_row_map) || (tile_cfg & AMOE_SOURCE_BELOW_4GIB);
    tile_cfg &= ~(AMOE_TILE_MAP_READY | AMOE_SOURCE_BELOW_4GIB);   // no tile map in the weight gradient
    TileCfg tc = pick_cfg(tile_cfg);
    GemmArgs a = {};
    a.f16 = dtype == AMOE_F16;
    a.A = (const bf16_t*)A;
    a.B = (const bf16_t*)B;
    a.C = (bf16_t*)C;
    a.a_row_map = a_row_map;
    a.b_row_map = b_row_map;
    a.rows_total = R;
    a.offsets = offsets;
    a.lda = lda;
    a.ldb = N;
    a.ldc = N;
    a.strideC = (long long)Kd * N;
    a.E = E;
    a.M = Kd;
    a.N = N;
    a.n_ntiles = (N + tc.bn - 1) / tc.bn;
    a.n_mt = (Kd + tc.bm - 1) / tc.bm;
    // The default kernel addresses a gathered operand with 32-bit byte offsets and numbers its tiles in 32 bits; where the
    // caller does not vouch for the operand's size (the length of the map says nothing about it), and beyond that many
    // tiles, the kernel with 64-bit addresses runs.
    const long long per = (long long)a.n_mt * a.n_ntiles;
    if (tile_cfg == 0) {
        // Up to 128 rows per expert the product is bound by the gradients' stores: gemm_short.hip, where its 32-bit tile
        // numbers reach (with a fourth of these tiles' size).  Beyond, gemm_pp.hip, whose tiles are never done in less than three
        // K tiles: with uneven loads the deep ones, four times as large as the short kernel's, fall to a few compute units.  (Below 704 rows an expert
        // it deals tiles by number.)  The two gradients, short / pp, us: 128 experts of 2048 x 768, 96 rows, even 298 / 306, 105 rows 337 / 309, 128 rows 354 /
        // 317, Zipf loads 342 / 418 and 379 / 454; 64 of 2048 x 1408, even, 96 rows 266 / 283, 105 rows 302 / 286, 128 rows 319 / 290, a sixteenth of the
        // experts with half of the rows 290 / 308, 302 / 316, 357 / 326, Zipf loads 310 / 338, 321 / 345, 353 / 370; 32 of 1024 x 2048, 105 rows 116 / 114, 105 /
        // 132, 105 / 139, 128 rows 118 / 113, 123 / 139, 119 / 145; 27 of 1024 x 4608, 105 rows 231 / 207, 241 / 245, 229 / 233.  Of six such layers, from 105
        // to 128 rows, even loads are 1.00 to 1.13 times as fast on the large tiles, a sixteenth 0.78 to 1.12, Zipf loads 0.73 to 1.03: the line
        // lies where uneven loads still lose, not where even ones begin to gain.
        if (R <= 128ll * E && offsets32 && 16 * per * per * E < (1ll << 32)) return amoe_short_wgrad(a, s);
        if (offsets32 && per * per * E < (1ll << 32)) return amoe_pp_wgrad(a, s);
        tile_cfg = 5;
    }
    long long grid = 0;
    int rc = set_supertiles(a, (long long)E * a.n_mt, &grid);
    if (rc) return rc;
    if (out32) {
        constexpr int lds_bytes = NSTAGE * (128 + 128) * BK * 2;
        AMOE_REQUIRE(tile_cfg == 1 && !a_row_map && !b_row_map, AMOE_ERR_BAD_ARG, "grouped_gemm_wgrad: float32 sums of gathered rows");
        if (a.f16) return launch_kernel<grouped_gemm_wgrad_parts_f16_kernel, 256, lds_bytes>(a, (int)grid, s);
        return launch_kernel<grouped_gemm_wgrad_parts_bf16_kernel, 256, lds_bytes>(a, (int)grid, s);
    }
    if (a_row_map) return launch_any<false, false, EPI_STORE, 0, 1>(a, tile_cfg, (int)grid, s);
    if (b_row_map) return launch_any<false, false, EPI_STORE, 0, 2>(a, tile_cfg, (int)grid, s);
    return launch_any<false, false, EPI_STORE, 0>(a, tile_cfg, (int)grid, s);
}
#endif
