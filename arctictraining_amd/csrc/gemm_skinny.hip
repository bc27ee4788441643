// The 16-bit grouped products C[rows_e,:] = A[rows_e,:] @ B[e] where an expert has a few rows (decoding, short prompts).
//
// Bound by reading the weights once: with 256-row tiles eight wavefronts wait at the same barriers for the same stage,
// a tile has one workgroup's loads in flight, and one token of K = 8 experts fills 48 compute units.  Here a wavefront
// streams its part of the weights straight into registers: no LDS and no barrier before the last sum, so every wavefront
// on a compute unit has its own two 8 KB steps in flight.
//
// A workgroup owns MT x 16 rows of an expert and 16 * CPL columns, its NW wavefronts take every NW-th step of 32 k; or two groups of
// NW / 2 wavefronts stand side by side in the columns, and a wavefront takes two such parts of the reduction, one after the other
// (with a barrier in between; skinny_pairs).
// Lane (lq, l16) loads, for each of the 8 k of its quarter lq, the CPL columns l16 * CPL .. of the row of B (256 or 128
// contiguous bytes per row and quarter); byte permutes of two such rows give the MFMA operands: fragment j holds column
// l16 * CPL + j.  The NW parts' sums meet in LDS, in the order of the parts: the two forms give the same bits.
//
// One MI355X, bf16, gate_up and down product, against 256-row tiles: 128 experts of 2048 x 768, 1 row an expert 105 and
// 55 -> 99 and 43 us, 4 rows 152 and 78 -> 145 and 74 (5.5 TB/s, what a read of that size reaches); 8 experts of
// 4096 x 14336, 1 row 292 and 184 -> 256 and 129, 4 rows 334 and 195 -> 330 and 149; 16 experts of 512 x 512, 4 rows 17
// and 12 -> 11 and 9.  A 64-row form at 32 rows an expert of the first took 222 and 90 us (one-tile workgroups of 256 rows
// 204 and 83) and is not kept.
#include "gemm_calls.h"
#include "gemm_common.h"
#include "gemm_launch.h"
#include "router_topk.h"

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float sk_f32x4;

namespace {

constexpr uint32_t SK_NOWHERE = 0xFFFFFFF0u;   // a load offset past every operand: the lane receives zeros

template <typename ET>
struct MfmaSkinny;
template <>
struct MfmaSkinny<bf16_t> {
    __device__ static __forceinline__ sk_f32x4 run(u32x4_t a, u32x4_t b, sk_f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(mfma_bf16x8, a), __builtin_bit_cast(mfma_bf16x8, b), c, 0, 0, 0);
    }
};
template <>
struct MfmaSkinny<f16_t> {
    __device__ static __forceinline__ sk_f32x4 run(u32x4_t a, u32x4_t b, sk_f32x4 c)
    {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(mfma_f16x8, a), __builtin_bit_cast(mfma_f16x8, b), c, 0, 0, 0);
    }
};

// source_of(row): the row of A that stands for a row; scale_of(row): its factor in the gated epilogue
// SHARED: C is stored where workgroups of other XCDs see it (agent scope: through the L2s)
// PAIRS: two groups of wavefronts stand side by side in the columns, n0 is the first one's
// FORMS: the kernel holds one or both of the forms in a loop over a tile's parts (0: no loop)
template <int MT, int CPL, int NW, int EPI, int ACT, bool STREAM, typename ET, bool SHARED = false, bool PAIRS = false, int FORMS = 0, typename SourceOf, typename ScaleOf>
__device__ __forceinline__ void skinny_tile(const GemmArgs& p, sk_f32x4 (&red_all)[NW][CPL * 64], int e, int m0, int mend, int n0,
                                            SourceOf source_of, ScaleOf scale_of)
{
    constexpr int W = CPL / 2, H = CPL / 4;           // dwords of a lane's row, groups of four columns
    int tid = threadIdx.x % (NW * 64);
    if constexpr (FORMS == 2) asm volatile("" : "+v"(tid));   // (or what both forms need is worked out ahead of the branch between them, held across the reduction, and spills)
    const int lane = tid & 63, l16 = lane & 15, lq = lane >> 4;
    constexpr int GW = PAIRS ? NW / 2 : NW;           // wavefronts of a group
    int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int group = PAIRS ? wave / GW : 0;
    if (PAIRS) wave %= GW;
    static_assert(!PAIRS || (GW == 2 && MT <= GW), "a row of red for every 16 rows");
    sk_f32x4 (*const red)[CPL * 64] = red_all + group * GW;
    n0 += group * 16 * CPL;

    const int steps = p.Kd / 32;                      // (the reduction length is a multiple of 32)
    const uint32_t row_bytes = (uint32_t)p.ldb * 2u;
    const __amdgpu_buffer_rsrc_t bd = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<bf16_t*>(p.B) + (long long)e * p.strideB, (short)0, (int)((uint32_t)(p.rows_total ? p.rows_total : p.Kd) * row_bytes),
        0x00020000);
    const __amdgpu_buffer_rsrc_t ad = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(p.A), (short)0, (int)SK_NOWHERE, 0x00020000);
    const int n = n0 + l16 * CPL;
    const uint32_t boff = n < p.N ? (uint32_t)(lq * 8) * row_bytes + (uint32_t)n * 2u : SK_NOWHERE;
    uint32_t aoff[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int row = m0 + i * 16 + l16;
        aoff[i] = row < mend ? ((uint32_t)source_of(row) * (uint32_t)p.lda + lq * 8) * 2u : SK_NOWHERE;
    }

    struct Step {
        uint32_t b[8][W];
        u32x4_t a[MT];
    };
    // a step past the last loads zeros
    auto load = [&](Step& s, int step) {
        const bool live = step < steps;
        const uint32_t sb = live ? (uint32_t)step * 32u * row_bytes : 0u, sa = live ? (uint32_t)step * 64u : 0u;
        const uint32_t vb = live ? boff : SK_NOWHERE;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            if constexpr (CPL == 8) {
                const u32x4_t v = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(bd, vb, sb + k * row_bytes, STREAM ? 2 : 0));
#pragma unroll
                for (int w = 0; w < 4; ++w) s.b[k][w] = v[w];
            } else {
                const u32x2_t v = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(bd, vb, sb + k * row_bytes, STREAM ? 2 : 0));
                s.b[k][0] = v[0];
                s.b[k][1] = v[1];
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
            s.a[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ad, live ? aoff[i] : SK_NOWHERE, sa, 0));
    };
    sk_f32x4 acc[MT][CPL];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < CPL; ++j) acc[i][j] = sk_f32x4{0.f, 0.f, 0.f, 0.f};
    };
    clear();
    auto multiply = [&](const Step& s) {
#pragma unroll
        for (int w = 0; w < W; ++w) {
            u32x4_t f0, f1;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                f0[k] = __builtin_amdgcn_perm(s.b[2 * k + 1][w], s.b[2 * k][w], 0x05040100u);
                f1[k] = __builtin_amdgcn_perm(s.b[2 * k + 1][w], s.b[2 * k][w], 0x07060302u);
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                acc[i][2 * w] = MfmaSkinny<ET>::run(f0, s.a[i], acc[i][2 * w]);
                acc[i][2 * w + 1] = MfmaSkinny<ET>::run(f1, s.a[i], acc[i][2 * w + 1]);
            }
        }
    };

    // Lane (lq, l16) holds columns (4 lq + v) * CPL + j of row l16.
    auto sums = [&](int i, auto use) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int h = 0; h < H; ++h)
                use((v * H + h) * 64 + lane, sk_f32x4{acc[i][4 * h][v], acc[i][4 * h + 1][v], acc[i][4 * h + 2][v], acc[i][4 * h + 3][v]});
    };
    // Part p of the reduction is the steps p, p + NW, .. (those past the last are zeros).
    const int rounds = (steps + NW - 1) / NW;
    Step s0, s1;
    load(s0, wave);
    if constexpr (!PAIRS) {
        for (int r = 0; r < rounds; r += 2) {
            load(s1, (r + 1) * NW + wave);
            multiply(s0);
            load(s0, (r + 2) * NW + wave);
            multiply(s1);
        }
    } else {
        // Row i of red takes ((part 0 + part 1) + part 2) + part 3 of rows 16 i ..+15, in two halves, of which the two
        // wavefronts add to one each.
        auto half = [&](int which, auto use) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
                if (MT == 1 || i == which) sums(i, [&](int u, sk_f32x4 c) {
                    if (MT > 1 || u / (2 * H * 64) == which) use(red[i][u], c);
                });
        };
        const auto put = [](sk_f32x4& at, sk_f32x4 c) { at = c; };
        const auto add = [](sk_f32x4& at, sk_f32x4 c) { at += c; };
#pragma unroll 1
        for (int part = wave;; part += GW) {
            const bool last = part >= GW;
            for (int r = 0; r + 1 < rounds; r += 2) {
                load(s1, (r + 1) * NW + part);
                multiply(s0);
                load(s0, r + 2 < rounds || last ? (r + 2) * NW + part : part + GW);
                multiply(s1);
            }
            if (rounds & 1) {
                multiply(s0);
                if (!last) load(s0, part + GW);
            }
            if (last) break;
            if (wave == 0) half(1, put);
            else half(0, put);
            __syncthreads();
            if (wave == 0) half(0, add);
            else half(1, add);
            clear();
        }
        if (wave == 0) half(0, add);
        __syncthreads();
        if (wave == 0) half(1, add);
        else half(0, add);
        __syncthreads();
        if (wave == 1) half(1, add);
        __syncthreads();
    }
    // 16 rows at a time
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (m0 + i * 16 >= mend) break;
        if constexpr (!PAIRS) {
            if (i) __syncthreads();
            sums(i, [&](int u, sk_f32x4 c) { red[wave][u] = c; });
            __syncthreads();
        }
        int first = tid;
        if constexpr (FORMS > 0) {
            first = threadIdx.x;   // (worked out here: held across the reduction it spills)
            asm volatile("" : "+v"(first));
        }
        for (int u = first % (GW * 64); u < 4 * H * 64; u += GW * 64) {
            sk_f32x4 c = red[PAIRS ? i : 0][u];
            if constexpr (!PAIRS) {
#pragma unroll
                for (int w = 1; w < NW; ++w) c += red[w][u];
            }
            const int l = u & 63, q = u >> 6;
            const int row = m0 + i * 16 + (l & 15);
            const int col = n0 + ((l >> 4) * 4 + q / H) * CPL + (q % H) * 4;
            if (row < mend && col < p.N) {
                const uint32_t x = Elem16<ET>::pack2(c[0], c[1]), y = Elem16<ET>::pack2(c[2], c[3]);
                bf16_t* const at = p.C + (long long)row * p.ldc + col;
                if constexpr (SHARED)
                    __hip_atomic_store(reinterpret_cast<uint64_t*>(at), (uint64_t)y << 32 | x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else if (EPI != EPI_GATED || p.C) *reinterpret_cast<u32x2_t*>(at) = u32x2_t{x, y};
                if constexpr (EPI == EPI_GATED) {
                    const float s = scale_of(row);
                    *reinterpret_cast<uint32_t*>(p.C2 + (long long)row * p.ldc2 + (col >> 1)) =
                        Elem16<ET>::pack2(s * Elem16<ET>::hi(x) * act_fwd_fast<ACT>(Elem16<ET>::lo(x)),
                                          s * Elem16<ET>::hi(y) * act_fwd_fast<ACT>(Elem16<ET>::lo(y)));
                }
            }
        }
    }
}

// Two column groups of two wavefronts instead of four wavefronts on one: a workgroup reads 512 bytes of each row together, not
// 256 (reads alone, 128 matrices of 2048 rows of 3072 bytes: 7.0 TB/s instead of 6.5; 1024 bytes 6.5, neighbouring workgroups on
// one XCD 6.3), and takes twice as long.  By the tiles that the map holds, which only the device knows: with all rows on a few experts there are
// few, whatever the host's bound says.  w: workgroups of two groups for a compute unit.  Where whole ones of them and halves of one
// round up to the same, two groups are faster, otherwise the most loaded compute unit has half a workgroup more: products of
// K x N = 256 x 1024 to 4096 x 2048, 2.5 and 6 rows an expert, times as fast: w 0.5 to 1.3 0.72 .. 1.06; 1.56 1.05 .. 1.24; 1.7 to 2 1.00 .. 1.21;
// 2.02 to 2.5 0.91 .. 1.12 (median 0.99); 2.6 to 3 1.02 .. 1.13; 3.1 to 3.5 0.96 .. 1.05 (1.00); 3.52 to 4 0.98 .. 1.12 (1.05).  With several rounds of
// them that no longer counts: 4.1 to 4.5 0.98 .. 1.05, 4.6 to 8 1.00 .. 1.20 (1.05).
__device__ __forceinline__ bool skinny_pairs(const GemmArgs& p, int tiles, int n_pairs)
{
    const int workgroups = tiles * n_pairs, cus = p.pairs_cus;
    return 2 * workgroups >= 3 * cus && (workgroups > p.pairs_always || (2 * workgroups + cus - 1) / cus % 2 == 0);
}

// A map's tile is 16 * MT rows where the launch's own rule built it; the taller tiles of a map that was built for another
// bound of the rows are walked in parts.
template <int MT, int CPL, int NW, bool PAIRS, int EPI, int ACT, bool STREAM, typename ET>
__device__ __forceinline__ void skinny_body(const GemmArgs& p)
{
    __shared__ sk_f32x4 red[NW][CPL * 64];
    int pm = blockIdx.x / p.n_ntiles, nt = blockIdx.x - pm * p.n_ntiles;
    int e = 0, m0 = pm * 16 * MT, mend = min(m0 + 16 * MT, p.M);   // without a map: one expert that has all p.M rows
    bool two = false;
    if (p.tile_map) {
        const int tiles = min(scalar_load_i32(p.n_mtiles), p.max_mtiles);
        const int32_t* ent = reinterpret_cast<const int32_t*>(p.tile_map + pm);
        e = scalar_load_i32(ent);
        m0 = scalar_load_i32(ent + 1);
        mend = scalar_load_i32(ent + 2);
        if constexpr (PAIRS) {
            // (the entries of both forms are read beside the number of tiles, not after it)
            const int n_pairs = p.n_ntiles / 2, pm2 = blockIdx.x / n_pairs;
            const int32_t* ent2 = reinterpret_cast<const int32_t*>(p.tile_map + min(pm2, p.max_mtiles - 1));
            const int e2 = scalar_load_i32(ent2), from2 = scalar_load_i32(ent2 + 1), to2 = scalar_load_i32(ent2 + 2);
            two = skinny_pairs(p, tiles, n_pairs);
            if (two) {
                pm = pm2;
                nt = 2 * ((int)blockIdx.x - pm2 * n_pairs);
                e = e2;
                m0 = from2;
                mend = to2;
            }
        }
        if (pm >= tiles) return;
    }
    const int n0 = nt * 16 * CPL;
    const auto source_of = [&](int row) { return p.a_row_map ? p.a_row_map[row] : row; };
    const auto scale_of = [&](int row) { return p.row_scale ? p.row_scale[row] : 1.0f; };
    auto part = [&](auto TWO) {
        skinny_tile<MT, CPL, NW, EPI, ACT, STREAM, ET, false, decltype(TWO)::value, PAIRS ? 2 : 1>(p, red, e, m0, mend, n0, source_of, scale_of);
    };
    auto walk = [&](auto TWO) {
#pragma unroll 1
        for (;;) {
            part(TWO);
            if ((m0 += 16 * MT) >= mend) break;
            __syncthreads();   // (the sums are read before the next part's are written)
        }
    };
    if constexpr (PAIRS) {
        if (two) walk(std::integral_constant<bool, true>{});
        else walk(std::integral_constant<bool, false>{});
    } else {
        part(std::integral_constant<bool, false>{});
#pragma unroll 1
        for (m0 += 16 * MT; m0 < mend; m0 += 16 * MT) {
            __syncthreads();
            part(std::integral_constant<bool, false>{});
        }
    }
}

// (at least 4 wavefronts per SIMD with 16 rows, 3 with 32)
// STREAM: B is loaded past the caches
template <int MT, int CPL, int NW, bool PAIRS, int EPI, int ACT, bool STREAM>
__global__ void __launch_bounds__(NW * 64, MT == 1 ? 4 : 3) grouped_gemm_skinny_bf16_kernel(GemmArgs p)
{
    skinny_body<MT, CPL, NW, PAIRS, EPI, ACT, STREAM, bf16_t>(p);
}
template <int MT, int CPL, int NW, bool PAIRS, int EPI, int ACT, bool STREAM>
__global__ void __launch_bounds__(NW * 64, MT == 1 ? 4 : 3) grouped_gemm_skinny_f16_kernel(GemmArgs p)
{
    skinny_body<MT, CPL, NW, PAIRS, EPI, ACT, STREAM, f16_t>(p);
}

template <int MT, int CPL, int NW, bool PAIRS, int EPI, int ACT, bool STREAM>
int launch_skinny(const GemmArgs& a, int grid, hipStream_t s)
{
    if (a.f16)
        hipLaunchKernelGGL((grouped_gemm_skinny_f16_kernel<MT, CPL, NW, PAIRS, EPI, ACT, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a);
    else
        hipLaunchKernelGGL((grouped_gemm_skinny_bf16_kernel<MT, CPL, NW, PAIRS, EPI, ACT, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a);
    return amoe_check_launch("grouped_gemm_skinny");
}

template <int MT, int CPL, int NW, bool PAIRS, int EPI, int ACT>
int launch_skinny(GemmArgs a, int m_tiles, hipStream_t s)
{
    a.n_ntiles = (a.N + 16 * CPL - 1) / (16 * CPL);
    long long grid = (long long)m_tiles * a.n_ntiles;
    if (PAIRS && grid / 2 > a.pairs_always)   // (of one column group there are at most as many as skinny_pairs lets be)
        grid = grid / 2 > 2ll * a.pairs_always ? grid / 2 : 2ll * a.pairs_always;
    AMOE_REQUIRE(grid < (1ll << 31), AMOE_ERR_UNSUPPORTED, "grouped_gemm: grid too large");
    if (a.stream_from) return launch_skinny<MT, CPL, NW, PAIRS, EPI, ACT, true>(a, (int)grid, s);
    return launch_skinny<MT, CPL, NW, PAIRS, EPI, ACT, false>(a, (int)grid, s);
}

// Whether there can be workgroups of two column groups (skinny_pairs).  Rows that are no multiple of 512 bytes lose: 3968 bytes 131 / 143 us,
// 22272 191 / 202.  Up to 128 rows, which may be in as few experts: 8 tokens, 8 of 256 experts of 2560 x 768 84 / 93 and 41 / 47.
static bool skinny_may_pair(GemmArgs& a, int m_tiles, int fit, int cus)
{
    a.pairs_cus = cus;
    a.pairs_always = (fit + 1) * cus;
    const long long workgroups = (long long)m_tiles * (a.N / 256);
    return cus && a.tile_map && a.N % 256 == 0 && a.M > 128 && 2 * workgroups >= 3ll * cus && workgroups < (1 << 29);
}

// bm: height of the map's tiles; R rows of a.E experts
template <int EPI, int ACT>
int launch_height(GemmArgs a, int bm, hipStream_t s)
{
    const int R = a.M;
    // every expert with a row has at most rows / 16 + 1 tiles, whatever rule built the map
    int m_tiles = R / 16 + (a.E < R ? a.E : R);
    if (m_tiles > R) m_tiles = R;
    if (m_tiles > a.max_mtiles) m_tiles = a.max_mtiles;
    AMOE_REQUIRE(bm == 16 || bm == 32, AMOE_ERR_UNSUPPORTED, "grouped_gemm: no kernel for tiles of %d rows", bm);
    const int cus = device_cu_count();
    if (bm == 32) {
        if (skinny_may_pair(a, m_tiles, 3, cus)) return launch_skinny<2, 8, 4, true, EPI, ACT>(a, m_tiles, s);
        return launch_skinny<2, 8, 4, false, EPI, ACT>(a, m_tiles, s);
    }
    if (skinny_narrow(m_tiles, a.N, cus)) return launch_skinny<1, 4, 8, false, EPI, ACT>(a, m_tiles, s);
    if (skinny_may_pair(a, m_tiles, 4, cus)) return launch_skinny<1, 8, 4, true, EPI, ACT>(a, m_tiles, s);
    return launch_skinny<1, 8, 4, false, EPI, ACT>(a, m_tiles, s);
}

// ------------------------------------------------------------------ gate_up product with the routing of a few tokens
// Softmax, top-k and the plan of a few tokens (one wavefront a token, then a walk over the at most kRoutedRows selected slots in
// LDS) cost a launch of one workgroup 6 us, most of it the launch and memory round trips that the product then waits for.
// Here every workgroup of the product selects for itself and finds its own expert and rows; what the other products and backward
// read of the routing is written by one more workgroup, which multiplies nothing.
// (At amoe_routed_fits: where this pays, and what it measured.)
constexpr int kRoutedRows = 128, kRoutedExperts = 256;

template <int CPL, int NW, int ACT, bool STREAM, typename ET>
__device__ __forceinline__ void skinny_routed_body(const GemmArgs& p, const AmoeRoute& r)
{
    constexpr int VPT = kRoutedExperts / 64, WORDS = kRoutedExperts / 32;
    __shared__ sk_f32x4 red[NW][CPL * 64];
    __shared__ __attribute__((aligned(16))) int sel[kRoutedRows];      // expert of flat slot k * T + t
    __shared__ float score[kRoutedRows], row_score[kRoutedRows];
    __shared__ int row_token[kRoutedRows];
    __shared__ uint32_t met[WORDS];                                    // experts that have a row
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int T = r.T, K = r.K, E = p.E, R = T * K;
    const bool writer = blockIdx.x == 0;
    if (tid < WORDS) met[tid] = 0;
    if (tid < kRoutedRows) sel[tid] = kRoutedExperts;                  // (past the last slot: of no expert)
    __syncthreads();
    for (int t = wave; t < T; t += NW) {
        int e;
        float s;
        router_topk_token<ET, VPT>((const ET*)r.logits + (size_t)t * E, E, K, r.normalize, lane, writer ? r.probs + (size_t)t * E : nullptr, e, s);
        if (lane < K) {
            e = min(max(e, 0), E - 1);
            sel[lane * T + t] = e;
            score[lane * T + t] = s;
            atomicOr(&met[e >> 5], 1u << (e & 31));
            if (writer) {
                r.topk_idx[t * K + lane] = e;
                r.scores[t * K + lane] = s;
            }
        }
    }
    __syncthreads();
    // slots of smaller experts, and of this one before slot f
    auto walk = [&](int e, int f, int& smaller, int& before) {
        smaller = before = 0;
        for (int g = 0; g < R; g += 4) {
            const int4 v = *reinterpret_cast<const int4*>(sel + g);
            const int x[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                smaller += x[i] < e;
                before += x[i] == e && g + i < f;
            }
        }
    };
    auto experts_below = [&](int e) {
        int n = 0;
#pragma unroll
        for (int w = 0; w < WORDS; ++w) {
            const int left = e - 32 * w;
            n += __popc(left >= 32 ? met[w] : left > 0 ? met[w] & ((1u << left) - 1u) : 0u);
        }
        return n;
    };
    if (writer) {
        if (tid < R) {
            const int e = sel[tid], k = tid / T, t = tid - k * T;
            int smaller, before;
            walk(e, tid, smaller, before);
            const int row = smaller + before;
            r.token_of[row] = t;
            r.slot_of[row] = tid;
            r.row_of[t * K + k] = row;
            r.scores_perm[row] = score[tid];
        }
        for (int e = tid; e < E; e += NW * 64) {
            int smaller, rows;
            walk(e, R, smaller, rows);
            r.counts[e] = rows;
            r.offsets[e + 1] = smaller + rows;
            // (an expert's rows are at most the T tokens: one tile)
            if (rows) r.tile_map[experts_below(e)] = make_int4(e, smaller, smaller + rows, 0);
        }
        const int tiles = experts_below(E);
        for (int i = tiles + tid; i < p.max_mtiles; i += NW * 64) r.tile_map[i] = make_int4(-1, 0, 0, 0);
        if (tid == 0) r.offsets[0] = 0;
        if (tid < 4) r.n_mtiles[tid] = tid ? 0 : tiles;
        for (int i = tid; i < r.n_arrived; i += NW * 64) r.arrived[i] = 0;
        return;
    }
    const int pm = (int)(blockIdx.x - 1) / p.n_ntiles;
    const int n0 = ((int)(blockIdx.x - 1) - pm * p.n_ntiles) * 16 * CPL;
    if (pm >= experts_below(E)) return;
    int e = 0, skip = pm;                // the pm-th expert that has a row
#pragma unroll
    for (int w = 0; w < WORDS; ++w) {
        const int n = __popc(met[w]);
        if (skip >= 0 && skip < n) {
            uint32_t m = met[w];
            for (; skip; --skip) m &= m - 1;
            e = 32 * w + __builtin_ctz(m);
            skip = -1;
        } else if (skip >= 0) skip -= n;
    }
    e = __builtin_amdgcn_readfirstlane(e);
    int m0, rows, rank;
    walk(e, R, m0, rows);
    if (tid < R && sel[tid] == e) {
        walk(e, tid, m0, rank);
        row_token[rank] = tid % T;
        row_score[rank] = score[tid];
    }
    m0 = __builtin_amdgcn_readfirstlane(m0);
    rows = __builtin_amdgcn_readfirstlane(rows);
    __syncthreads();
    skinny_tile<1, CPL, NW, EPI_GATED, ACT, STREAM, ET>(p, red, e, m0, m0 + rows, n0, [&](int row) { return row_token[row - m0]; },
                                                        [&](int row) { return row_score[row - m0]; });
}

template <int CPL, int NW, int ACT, bool STREAM>
__global__ void __launch_bounds__(NW * 64, 4) grouped_gemm_skinny_routed_bf16_kernel(GemmArgs p, AmoeRoute r)
{
    skinny_routed_body<CPL, NW, ACT, STREAM, bf16_t>(p, r);
}
template <int CPL, int NW, int ACT, bool STREAM>
__global__ void __launch_bounds__(NW * 64, 4) grouped_gemm_skinny_routed_f16_kernel(GemmArgs p, AmoeRoute r)
{
    skinny_routed_body<CPL, NW, ACT, STREAM, f16_t>(p, r);
}

template <int CPL, int NW, int ACT, bool STREAM>
int launch_routed(const GemmArgs& a, const AmoeRoute& r, int grid, hipStream_t s)
{
    if (a.f16) hipLaunchKernelGGL((grouped_gemm_skinny_routed_f16_kernel<CPL, NW, ACT, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a, r);
    else hipLaunchKernelGGL((grouped_gemm_skinny_routed_bf16_kernel<CPL, NW, ACT, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a, r);
    return amoe_check_launch("grouped_gemm_skinny_routed");
}
template <int CPL, int NW, int ACT>
int launch_routed(GemmArgs a, const AmoeRoute& r, int m_tiles, hipStream_t s)
{
    a.n_ntiles = (a.N + 16 * CPL - 1) / (16 * CPL);
    const long long grid = (long long)m_tiles * a.n_ntiles + 1;
    AMOE_REQUIRE(grid < (1ll << 31), AMOE_ERR_UNSUPPORTED, "grouped_gemm: grid too large");
    if (a.stream_from) return launch_routed<CPL, NW, ACT, true>(a, r, (int)grid, s);
    return launch_routed<CPL, NW, ACT, false>(a, r, (int)grid, s);
}

// ------------------------------------------------------------------ down product with the sums over a token's rows
// As grouped_gemm_skinny with a map of 16-row tiles; the last of a column tile's workgroups to arrive adds up the tokens' rows
// there, as stored and in the order of k (gather_reduce_kernel's sum, bit for bit), instead of a launch of its own that waits for all of them.
template <int CPL, int NW, bool STREAM, typename ET>
__device__ __forceinline__ void skinny_combine_body(const GemmArgs& p, const AmoeCombine& c)
{
    __shared__ sk_f32x4 red[NW][CPL * 64];
    __shared__ int before;
    const int pm = blockIdx.x / p.n_ntiles, nt = blockIdx.x - pm * p.n_ntiles, n0 = nt * 16 * CPL;
    const int tiles = min(scalar_load_i32(p.n_mtiles), p.max_mtiles);
    if (pm >= tiles) return;
    const int32_t* ent = reinterpret_cast<const int32_t*>(p.tile_map + pm);
    skinny_tile<1, CPL, NW, EPI_STORE, 0, STREAM, ET, true>(p, red, scalar_load_i32(ent), scalar_load_i32(ent + 1), scalar_load_i32(ent + 2), n0,
                                                            [](int row) { return row; }, [](int) { return 1.0f; });
    // Rows are stored and read past the L2s, and every wavefront awaits its stores before the workgroup arrives: a release would
    // write out all of the XCD's L2 besides, a microsecond or more in every workgroup (4 tokens of 8 of 128 experts of 2048 x
    // 768, the whole pass 75 us with a launch of its own for the sums, 89 with a release, 75 so; 1 token 30.8, 32.3, 29.9).
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0) before = __hip_atomic_fetch_add(c.arrived + nt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (before != tiles - 1) return;
    constexpr int PIECES = 4 * CPL;                     // of four columns
    for (int i = threadIdx.x; i < c.T * PIECES; i += NW * 64) {
        const int t = i / PIECES, col = n0 + (i - t * PIECES) * 4;
        if (col >= p.N) continue;
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < c.K; ++k) {
            const u32x2_t v = __builtin_bit_cast(u32x2_t, __hip_atomic_load(reinterpret_cast<const uint64_t*>(p.C + (long long)c.row_of[t * c.K + k] * p.ldc + col),
                                                                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                sum[2 * j] += Elem16<ET>::lo(v[j]);
                sum[2 * j + 1] += Elem16<ET>::hi(v[j]);
            }
        }
        *reinterpret_cast<u32x2_t*>((bf16_t*)c.y + (long long)t * p.ldc + col) =
            u32x2_t{Elem16<ET>::pack2(sum[0], sum[1]), Elem16<ET>::pack2(sum[2], sum[3])};
    }
}

template <int CPL, int NW, bool STREAM>
__global__ void __launch_bounds__(NW * 64, 4) grouped_gemm_skinny_combine_bf16_kernel(GemmArgs p, AmoeCombine c)
{
    skinny_combine_body<CPL, NW, STREAM, bf16_t>(p, c);
}
template <int CPL, int NW, bool STREAM>
__global__ void __launch_bounds__(NW * 64, 4) grouped_gemm_skinny_combine_f16_kernel(GemmArgs p, AmoeCombine c)
{
    skinny_combine_body<CPL, NW, STREAM, f16_t>(p, c);
}

template <int CPL, int NW, bool STREAM>
int launch_combine(const GemmArgs& a, const AmoeCombine& c, int grid, hipStream_t s)
{
    if (a.f16) hipLaunchKernelGGL((grouped_gemm_skinny_combine_f16_kernel<CPL, NW, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a, c);
    else hipLaunchKernelGGL((grouped_gemm_skinny_combine_bf16_kernel<CPL, NW, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a, c);
    return amoe_check_launch("grouped_gemm_skinny_combine");
}
template <int CPL, int NW>
int launch_combine(GemmArgs a, const AmoeCombine& c, int m_tiles, hipStream_t s)
{
    a.n_ntiles = (a.N + 16 * CPL - 1) / (16 * CPL);
    const long long grid = (long long)m_tiles * a.n_ntiles;
    AMOE_REQUIRE(grid < (1ll << 31), AMOE_ERR_UNSUPPORTED, "grouped_gemm: grid too large");
    if (a.stream_from) return launch_combine<CPL, NW, true>(a, c, (int)grid, s);
    return launch_combine<CPL, NW, false>(a, c, (int)grid, s);
}

// ------------------------------------------------------------------ the router's linear map for few tokens
// logits [T,E] = x [T,H] @ w [E,H]^T, both operands K-contiguous and read straight into MFMA operands.  A workgroup is a
// 16 x 16 tile, its 16 wavefronts share the reduction (every 16th step of 32 k).  Bound by latency: the tile's
// steps are requested all at once.
// (The caller's rule for using it holds the measurements.)
constexpr int kLogitWaves = 16;

template <typename ET>
__global__ void __launch_bounds__(kLogitWaves * 64)
router_logits_kernel(const ET* __restrict__ x, const ET* __restrict__ w, ET* __restrict__ logits, int T, int E, int H)
{
    __shared__ sk_f32x4 red[kLogitWaves][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l16 = lane & 15, lq = lane >> 4;
    const int n_et = (E + 15) >> 4;
    const int t0 = (int)(blockIdx.x / n_et) * 16, e0 = (int)(blockIdx.x % n_et) * 16;
    // (rows past the last are copies of it; their products are not stored)
    const ET* const xr = x + (size_t)min(t0 + l16, T - 1) * H + lq * 8;
    const ET* const wr = w + (size_t)min(e0 + l16, E - 1) * H + lq * 8;
    sk_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k = wave * 32; k < H; k += kLogitWaves * 32)
        acc = MfmaSkinny<ET>::run(*reinterpret_cast<const u32x4_t*>(wr + k), *reinterpret_cast<const u32x4_t*>(xr + k), acc);
    red[wave][lane] = acc;
    __syncthreads();
    // thread (q, l, v): logit of token l and expert 4 q + v
    if (threadIdx.x < 256) {
        const int l = threadIdx.x & 63, v = threadIdx.x >> 6;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < kLogitWaves; ++i) sum += red[i][l][v];
        const int t = t0 + (l & 15), e = e0 + (l >> 4) * 4 + v;
        if (t < T && e < E) ElemTraits<ET>::store1(logits + (size_t)t * E + e, sum);
    }
}

}  // namespace

AMOE_EXPORT int amoe_router_logits(const void* x, const void* w, void* logits, int dtype, int T, int E, int H, void* stream)
{
    AMOE_REQUIRE(x && w && logits, AMOE_ERR_BAD_ARG, "router_logits: null pointer");
    AMOE_REQUIRE(T > 0 && E > 0 && H > 0, AMOE_ERR_BAD_ARG, "router_logits: sizes must be positive (T=%d E=%d H=%d)", T, E, H);
    AMOE_REQUIRE(dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_UNSUPPORTED, "router_logits: bf16 and float16 only");
    AMOE_REQUIRE(H % 32 == 0 && ((uintptr_t)x | (uintptr_t)w) % 16 == 0, AMOE_ERR_UNSUPPORTED,
                 "router_logits: H=%d must be a multiple of 32, the operands aligned to 16 bytes", H);
    const long long grid = (long long)((T + 15) / 16) * ((E + 15) / 16);
    AMOE_REQUIRE(grid < (1ll << 31), AMOE_ERR_UNSUPPORTED, "router_logits: grid too large");
    if (dtype == AMOE_F16)
        hipLaunchKernelGGL((router_logits_kernel<f16_t>), dim3((int)grid), dim3(kLogitWaves * 64), 0, (hipStream_t)stream,
                           (const f16_t*)x, (const f16_t*)w, (f16_t*)logits, T, E, H);
    else
        hipLaunchKernelGGL((router_logits_kernel<bf16_t>), dim3((int)grid), dim3(kLogitWaves * 64), 0, (hipStream_t)stream,
                           (const bf16_t*)x, (const bf16_t*)w, (bf16_t*)logits, T, E, H);
    return amoe_check_launch("router_logits");
}

int amoe_skinny_gateup_act(const GemmArgs& a, int act, int bm, hipStream_t s)
{
    AMOE_DISPATCH_ACT(act, return (launch_height<EPI_GATED, ACT>(a, bm, s)))
    return AMOE_ERR_BAD_ARG;
}

// a: as for amoe_skinny_gateup_act, without the maps and scales that the routing gives
int amoe_skinny_gateup_routed(const GemmArgs& a, int act, const AmoeRoute& r, hipStream_t s)
{
    const int R = r.T * r.K, m_tiles = a.E < R ? a.E : R;
    AMOE_REQUIRE(r.T <= 16 && R <= kRoutedRows && a.E <= kRoutedExperts, AMOE_ERR_UNSUPPORTED,   // (a tile holds 16 rows)
                 "grouped_gemm: routing of %d rows of %d experts", R, a.E);
    AMOE_DISPATCH_ACT(act, return skinny_narrow(m_tiles, a.N, r.cus) ? (launch_routed<4, 8, ACT>(a, r, m_tiles, s)) : (launch_routed<8, 4, ACT>(a, r, m_tiles, s)))
    return AMOE_ERR_BAD_ARG;
}

// c.arrived holds a count for every 64 columns
int amoe_skinny_nn_combined(const GemmArgs& a, const AmoeCombine& c, hipStream_t s)
{
    const int m_tiles = a.E < a.M ? a.E : a.M;
    return skinny_narrow(m_tiles, a.N, c.cus) ? launch_combine<4, 8>(a, c, m_tiles, s) : launch_combine<8, 4>(a, c, m_tiles, s);
}

int amoe_skinny_nn(const GemmArgs& a, int bm, hipStream_t s) { return launch_height<EPI_STORE, 0>(a, bm, s); }

// out [T,H] = d_logits [T,E] @ w [E,H], the router's part of the gradient of the input: the product above with one
// expert that has every row.  ld: elements from one row of d_logits to the next; those past E are zero, and the rows of w
// that they would meet read as zeros.
AMOE_EXPORT int amoe_router_input_grad_rows(const void* d_logits, int ld, const void* w, void* out, int dtype, int T, int E, int H,
                                            void* stream)
{
    AMOE_REQUIRE(d_logits && w && out, AMOE_ERR_BAD_ARG, "router_input_grad: null pointer");
    AMOE_REQUIRE(T > 0 && E > 0 && H > 0, AMOE_ERR_BAD_ARG, "router_input_grad: sizes must be positive (T=%d E=%d H=%d)", T, E, H);
    AMOE_REQUIRE(ld >= E, AMOE_ERR_BAD_ARG, "router_input_grad: rows of %d elements for %d experts", ld, E);
    AMOE_REQUIRE(dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_UNSUPPORTED, "router_input_grad: bf16 and float16 only");
    AMOE_REQUIRE(ld % 32 == 0 && H % 8 == 0 && ((uintptr_t)d_logits | (uintptr_t)w | (uintptr_t)out) % 16 == 0, AMOE_ERR_UNSUPPORTED,
                 "router_input_grad: E=%d must be a multiple of 32, H=%d of 8, the operands aligned to 16 bytes", ld, H);
    AMOE_REQUIRE((unsigned long long)T * ld * 2ull < (1ull << 31) && (unsigned long long)E * H * 2ull < (1ull << 31), AMOE_ERR_UNSUPPORTED,
                 "router_input_grad: operand of 2 GiB or more");
    GemmArgs a = {};
    a.A = (const bf16_t*)d_logits;
    a.B = (const bf16_t*)w;
    a.C = (bf16_t*)out;
    a.f16 = dtype == AMOE_F16;
    a.lda = a.Kd = ld;
    a.rows_total = E;
    a.ldb = a.ldc = a.N = H;
    a.E = 1;
    a.M = T;
    if (T <= 16) return launch_skinny<1, 4, 8, false, EPI_STORE, 0>(a, 1, (hipStream_t)stream);
    return launch_skinny<2, 8, 4, false, EPI_STORE, 0>(a, (T + 31) / 32, (hipStream_t)stream);
}

AMOE_EXPORT int amoe_router_input_grad(const void* d_logits, const void* w, void* out, int dtype, int T, int E, int H, void* stream)
{
    return amoe_router_input_grad_rows(d_logits, E, w, out, dtype, T, E, H, stream);
}
