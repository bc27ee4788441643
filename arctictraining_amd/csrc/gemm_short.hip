// Weight gradients of experts with few rows: C[e] = A[rows_e,:]^T @ B[rows_e,:], a reduction of a few K tiles and then 32 KB of
// output for every 128 x 128 of the gradient.
//
// Bound by writing the gradients (a plain write in this pattern takes 5.7 TB/s).  A wavefront's loads and stores complete in
// order, so that one which stores a tile and loads the next waits for its stores: here the fifth wavefront of a workgroup
// loads, K tiles of 32 into three LDS stages, on from tile to tile, and the other four (64 x 64 each) multiply and store and
// never wait for memory.  Three workgroups on a compute unit, as many as the LDS holds, for as long as there are tiles.
// The stores are written through the L2 and past what lies in the last-level cache (sc1 nt): the rows stay there, and so do
// the weights that the kernels beside and behind this one read.  With ordinary stores 32 rows of 128 experts of 2048 x 768 took
// 112 us for down's gradient, with these 75.
//
// Lines are whole: eight lanes store a row's 128 bytes, which the accumulators reach through 1 KB of LDS a wavefront.  Out of a cold
// cache, bf16, the rows of one operand gathered, us, with 16 bytes of 16 rows an instruction (a request a lane) / so:
//   128 experts,  32 rows, 2048 x 1536  285 / 173 (4.7 TB/s),  768 x 2048  132 /  90
//   146 experts,   2 rows,  384 x 6208  142 / 139,            3104 x  384   97 /  70
//    51 experts,  23 rows, 2848 x 2944  237 / 162 (5.3 TB/s)
//    64 experts,  60 rows, 1408 x 2048  147 / 105;   8 experts, 100 rows, 4096 x 4096  117 / 93
// and a training step of 509 tokens of 128 experts of 2048 x 768 751 / 735.  The same step with 256 x 256 tiles and ordinary 4-byte
// stores took 93 us longer than with the former, 64 experts of 2048 x 1408 with 250 rows (not taken) 285 us less.
#include "gemm_dma.h"
#include "gemm_launch.h"

namespace {

constexpr int SH_THREADS = 320, SH_WGS = 3;      // (workgroups on a compute unit)
constexpr int SH_BM = 128, SH_BN = 128, SH_BK = 32, SH_NS = 3;
constexpr uint32_t SH_OPERAND = SH_BM * SH_BK * 2, SH_STAGE = 2 * SH_OPERAND;
constexpr uint32_t SH_TURN = 1024;               // a wavefront's for its epilogue

// MAPS: 1 = the rows of A, 2 = the rows of B are gathered through a row map
template <int MAPS, typename ET>
__device__ __forceinline__ void short_wgrad_body(const GemmArgs& p)
{
    typedef typename Elem16<ET>::frag_t frag_t;
    __shared__ __attribute__((aligned(1024))) char smem[SH_NS * SH_STAGE + 4 * SH_TURN + 64];
    const uint32_t lds = (uint32_t)(uintptr_t)(lptr_t)smem;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr bool A_MAP = MAPS == 1, B_MAP = MAPS == 2;
    constexpr uint32_t END = SH_NS * SH_STAGE, FLAGS = END + 4 * SH_TURN;      // per stage: whether it is its tile's last

    // ------------------------------------------------------------ this workgroup's tiles
    // Tiles are numbered expert by expert, row by row inside one; XCD x (workgroups with blockIdx % 8 == x) works through chunks
    // x, x + 8, ... of 16 consecutive tiles, which share rows in its L2; those left over from the last whole group of chunks are
    // dealt one by one.  (chunks of 1 to 64: within 5 % of each other, either way)
    auto divide = [](int n, uint32_t inv) -> int { return inv ? (int)(((uint64_t)(uint32_t)n * inv) >> 32) : n; };
    const int per = p.n_mt * p.n_ntiles, total = p.E * per, whole = total & ~127;
    const int xcd = blockIdx.x & 7, gq = gridDim.x >> 3;
    auto number = [&](int q) -> int {     // of the q-th tile of this XCD
        const int v = ((q >> 4) << 7) + (xcd << 4) + (q & 15);
        return v < whole ? v : whole + ((q - (whole >> 3)) << 3) + xcd;
    };
    struct Tile { int e, m0, n0; };
    auto decode = [&](int v) -> Tile {
        const int e = divide(v, p.inv_super), i = v - e * per;
        const int mt = divide(i, p.inv_gn);
        return {e, mt * SH_BM, (i - mt * p.n_ntiles) * SH_BN};
    };
    int q = blockIdx.x >> 3, qd = q, v = number(q);
    if (v >= total) return;

    if (wave == SH_THREADS / 64 - 1) {
        // ------------------------------------------------------------ the loading wavefront
        // A stage is 32 rows of 16 16-byte chunks of either operand, chunk c of row k at c ^ 2 ((k & 3) | (((k >> 3) & 1) << 2)).
        // A load takes four rows: row 4 i + lane / 16, one of two columns.
        const int lr = lane >> 4;
        const uint32_t lda2 = (uint32_t)p.lda * 2u, ldb2 = (uint32_t)p.ldb * 2u;
        auto add_sat = [](uint32_t a, uint32_t b) { return __builtin_elementwise_add_sat(a, b); };
        srd_t ad, bd;
        uint32_t acol[2], bcol[2], aoff[8], boff[8];
        int idx[32];                          // rows of the map, fetched a stage ahead by scalar loads
        int left = 0, row_n = 0;              // rows of the expert from the stage that is requested next, and where they begin
        auto fetch_idx = [&]() {
            if constexpr (MAPS != 0) {
                const int32_t* map = A_MAP ? p.a_row_map : p.b_row_map;
                typedef int i32x16_t __attribute__((ext_vector_type(16), aligned(4)));
                if (row_n + 32 <= p.rows_total) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const i32x16_t x = *(const __attribute__((address_space(4))) i32x16_t*)(map + row_n + 16 * j);
#pragma unroll
                        for (int k = 0; k < 16; ++k) idx[16 * j + k] = x[k];
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 32; ++k) idx[k] = scalar_load_i32(map + min(row_n + k, p.rows_total - 1));
                }
            }
        };
        auto plan = [&]() {                   // the stages of the next tile; an expert without rows has one, of zeros
            const int v = number(q);
            q += gq;
            left = 0;
            if (v < total) {
                const Tile t = decode(v);
                const int r0 = __builtin_amdgcn_readfirstlane(scalar_load_i32(p.offsets + t.e)), r1 = __builtin_amdgcn_readfirstlane(scalar_load_i32(p.offsets + t.e + 1));
                ad = pp_srd(A_MAP ? p.A : p.A + (long long)r0 * p.lda);
                bd = pp_srd(B_MAP ? p.B : p.B + (long long)r0 * p.ldb);
                left = r1 - r0;
                row_n = r0;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int col = ((lane & 15) ^ (2 * (lr | (h << 2)))) * 8;
                    acol[h] = t.m0 + col < p.M ? (uint32_t)(t.m0 + col) * 2u : PP_NOWHERE;
                    bcol[h] = t.n0 + col < p.N ? (uint32_t)(t.n0 + col) * 2u : PP_NOWHERE;
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    if (!A_MAP) aoff[i] = add_sat((uint32_t)(4 * i + lr) * lda2, acol[(i >> 1) & 1]);
                    if (!B_MAP) boff[i] = add_sat((uint32_t)(4 * i + lr) * ldb2, bcol[(i >> 1) & 1]);
                }
            }
            if (left > 0) fetch_idx();
        };
        uint32_t ends = 0;                    // bit i: the i-th last stage requested was the last of its tile
        auto issue = [&](uint32_t at) {
            // rows past the expert's end read as zeros: the descriptors of operands in place end with them
            const uint32_t rows = (uint32_t)__builtin_amdgcn_readfirstlane(min(max(left, 0), SH_BK));
            if (!A_MAP) ad[2] = rows * lda2;
            if (!B_MAP) bd[2] = rows * ldb2;
            if constexpr (MAPS != 0) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int i01 = lr & 1 ? idx[4 * i + 1] : idx[4 * i], i23 = lr & 1 ? idx[4 * i + 3] : idx[4 * i + 2];
                    const uint32_t o = 4 * i + lr < left ? (uint32_t)(lr & 2 ? i23 : i01) * (A_MAP ? lda2 : ldb2) : PP_NOWHERE;
                    if (A_MAP) aoff[i] = add_sat(o, acol[(i >> 1) & 1]);
                    else boff[i] = add_sat(o, bcol[(i >> 1) & 1]);
                }
            }
#define SH_LOAD(i) pp_dma16<(i) * 1024>(ad, aoff[i], lds + at); pp_dma16<SH_OPERAND + (i) * 1024>(bd, boff[i], lds + at);
            SH_LOAD(0) SH_LOAD(1) SH_LOAD(2) SH_LOAD(3) SH_LOAD(4) SH_LOAD(5) SH_LOAD(6) SH_LOAD(7)
#undef SH_LOAD
            if (!A_MAP) pp_advance(ad, SH_BK * lda2);
            if (!B_MAP) pp_advance(bd, SH_BK * ldb2);
            left -= SH_BK;
            row_n += SH_BK;
            const uint32_t last = left <= 0 ? 1u : 0u;
            ends = (ends << 1) | last;
            *(__attribute__((address_space(3))) uint32_t*)(uintptr_t)(lds + FLAGS + at / SH_STAGE * 4u) = last;
            if (left > 0) fetch_idx();
            else plan();
        };
        plan();
#pragma unroll
        for (int t = 0; t < SH_NS - 1; ++t) issue(t * SH_STAGE);
        uint32_t to = (SH_NS - 1) * SH_STAGE;
        for (;;) {
            pp_vmwait<(SH_NS - 2) * 16>();                 // this stage has landed
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            pp_barrier();
            if ((ends >> (SH_NS - 2)) & 1) {               // it is its tile's last: of the workgroup's last tile?
                v = number(qd += gq);
                if (v >= total) break;
            }
            issue(to);                                     // (past the last tile: zeros)
            to = to + SH_STAGE == END ? 0 : to + SH_STAGE;
        }
        pp_vmwait<0>();   // (loads past the last tile wrote zeros into LDS: landed before the workgroup leaves)
        return;
    }

    // ------------------------------------------------------------ the multiplying ones
    const int wm = wave >> 1, wn = wave & 1, l16 = lane & 15, lq = lane >> 4;
    uint32_t ra[4], rb[4];
    {
        const int k = 8 * lq + (l16 >> 2), key = 2 * ((l16 >> 2) | ((lq & 1) << 2));
        const uint32_t base = lds + (uint32_t)(k * 256 + (l16 & 1) * 8);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            ra[t] = base + (uint32_t)((wm * 8 + 2 * t + ((l16 & 3) >> 1)) ^ key) * 16u;
            rb[t] = base + SH_OPERAND + (uint32_t)((wn * 8 + 2 * t + ((l16 & 3) >> 1)) ^ key) * 16u;
        }
    }
    auto read_tr = [&](uint32_t at) -> frag_t {
        typedef __attribute__((address_space(3))) i16x4_t* tr_ptr;
        const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)at));
        const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)(at + 1024u)));
        return __builtin_bit_cast(frag_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
    };
    uint32_t at = 0;
    do {
        const Tile t = decode(v);
        mfma_f32x4 acc[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = 0; b < 4; ++b) acc[a][b] = mfma_f32x4{0.f, 0.f, 0.f, 0.f};
        uint32_t last;
        do {
            pp_barrier();                   // the stage has landed, and nobody reads the one before it any more
            frag_t fa[4], fb[4];
            last = *(const __attribute__((address_space(3))) uint32_t*)(uintptr_t)(lds + FLAGS + at / SH_STAGE * 4u);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                fb[u] = read_tr(at + rb[u]);
                fa[u] = read_tr(at + ra[u]);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            pp_fence();
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = Mfma16<ET>::run(fb[b], fa[a], acc[a][b]);
            pp_fence();
            at = at + SH_STAGE == END ? 0 : at + SH_STAGE;
        } while (!__builtin_amdgcn_readfirstlane(last));
        // Lane (lq, l16) holds columns 4 lq .. + 3 of row l16 of each 16 x 16 tile.  Eight rows of 128 bytes at a time go through LDS
        // (chunk c of row r at c ^ r), after which eight lanes hold a row's and a store writes whole lines.
        bf16_t* const c = p.C + (long long)t.e * p.strideC + (long long)(t.m0 + wm * 64) * p.ldc + t.n0 + wn * 64;
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(c, (short)0, (int)PP_DROP, 0x00020000);
        const uint32_t ldc2 = (uint32_t)p.ldc * 2u;
        const int r8 = lane >> 3, c8 = lane & 7;
        const uint32_t off = 8 * c8 < p.N - t.n0 - wn * 64 ? (uint32_t)r8 * ldc2 + 16u * c8 : PP_DROP;
        const int rows = p.M - t.m0 - wm * 64 - r8;
        const uint32_t turn = lds + END + (uint32_t)wave * SH_TURN;
        const uint32_t wr = turn + (uint32_t)((l16 & 7) * 128 + ((lq >> 1) ^ (l16 & 7)) * 16 + (lq & 1) * 8);
        const uint32_t rd = turn + (uint32_t)(r8 * 128 + (c8 ^ r8) * 16);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            u32x2_t x[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) x[b] = u32x2_t{Elem16<ET>::pack2(acc[a][b][0], acc[a][b][1]), Elem16<ET>::pack2(acc[a][b][2], acc[a][b][3])};
            u32x4_t y[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (l16 >> 3 == h) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) *(__attribute__((address_space(3))) u32x2_t*)(uintptr_t)(wr ^ (32u * b)) = x[b];
                }
                pp_lds_turn();
                y[h] = pp_lds<u32x4_t>(rd);
                pp_lds_turn();
            }
#pragma unroll
            for (int h = 0; h < 2; ++h) pp_store16<true>(d, y[h], a * 16 + h * 8 < rows ? off : PP_DROP, (uint32_t)(a * 16 + h * 8) * ldc2);
        }
        v = number(q += gq);
    } while (v < total);
}

template <int MAPS>
__global__ void __launch_bounds__(SH_THREADS, 4) grouped_gemm_short_wgrad_bf16_kernel(GemmArgs p)
{
    short_wgrad_body<MAPS, bf16_t>(p);
}
template <int MAPS>
__global__ void __launch_bounds__(SH_THREADS, 4) grouped_gemm_short_wgrad_f16_kernel(GemmArgs p)
{
    short_wgrad_body<MAPS, f16_t>(p);
}

template <int MAPS>
int launch_short(const GemmArgs& a, int grid, hipStream_t s)
{
    if (a.f16) hipLaunchKernelGGL(grouped_gemm_short_wgrad_f16_kernel<MAPS>, dim3(grid), dim3(SH_THREADS), 0, s, a);
    else hipLaunchKernelGGL(grouped_gemm_short_wgrad_bf16_kernel<MAPS>, dim3(grid), dim3(SH_THREADS), 0, s, a);
    return amoe_check_launch("grouped_gemm_short_wgrad");
}

}  // namespace

int amoe_short_wgrad(GemmArgs a, hipStream_t s)
{
    a.n_mt = (a.M + SH_BM - 1) / SH_BM;
    a.n_ntiles = (a.N + SH_BN - 1) / SH_BN;
    const long long per = (long long)a.n_mt * a.n_ntiles, total = a.E * per;
    AMOE_REQUIRE(total * per < (1ll << 32), AMOE_ERR_UNSUPPORTED, "grouped_gemm_wgrad: too many tiles");
    const int cus = device_cu_count();
    AMOE_REQUIRE(cus > 0, AMOE_ERR_LAUNCH, "grouped_gemm: cannot read the number of compute units");
    auto inverse = [](int d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; };
    a.inv_super = inverse((int)per);
    a.inv_gn = inverse(a.n_ntiles);
    const int most = cus * SH_WGS;
    const int grid = (int)(((total < most ? total : most) + 7) & ~7ll);
    if (a.a_row_map) return launch_short<1>(a, grid, s);
    if (a.b_row_map) return launch_short<2>(a, grid, s);
    return launch_short<0>(a, grid, s);
}
