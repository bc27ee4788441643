// The 16-bit grouped products C[rows_e,:] = A[rows_e,:] @ B[e] where an expert has a few rows (decoding, short prompts).
//
// Bound by reading the weights once: with 256-row tiles eight wavefronts wait at the same barriers for the same stage,
// a tile has one workgroup's loads in flight, and one token of K = 8 experts fills 48 compute units.  Here a wavefront
// streams its part of the weights straight into registers: no LDS and no barrier before the last sum, so every wavefront
// on a compute unit has its own two 8 KB steps in flight.
//
// A workgroup owns MT x 16 rows of an expert and 16 * CPL columns, its NW wavefronts take every NW-th step of 32 k.
// Lane (lq, l16) loads, for each of the 8 k of its quarter lq, the CPL columns l16 * CPL .. of the row of B (256 or 128
// contiguous bytes per row and quarter); byte permutes of two such rows give the MFMA operands: fragment j holds column
// l16 * CPL + j.  The wavefronts' partial sums meet in LDS, in a fixed order.
//
// One MI355X, bf16, gate_up and down product, against 256-row tiles: 128 experts of 2048 x 768, 1 row an expert 105 and
// 55 -> 99 and 43 us, 4 rows 152 and 78 -> 145 and 74 (5.5 TB/s, what a read of that size reaches); 8 experts of
// 4096 x 14336, 1 row 292 and 184 -> 256 and 129, 4 rows 334 and 195 -> 330 and 149; 16 experts of 512 x 512, 4 rows 17
// and 12 -> 11 and 9.  A 64-row form at 32 rows an expert of the first took 222 and 90 us (one-tile workgroups of 256 rows
// 204 and 83) and is not kept.
#include "gemm_common.h"
#include "gemm_launch.h"

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

template <int MT, int CPL, int NW, int EPI, int ACT, bool STREAM, typename ET>
__device__ __forceinline__ void skinny_tile(const GemmArgs& p, sk_f32x4 (&red)[NW][CPL * 64], int e, int m0, int mend, int n0)
{
    constexpr int W = CPL / 2, H = CPL / 4;           // dwords of a lane's row, groups of four columns
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;

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
        const int src = row < mend && p.a_row_map ? p.a_row_map[row] : row;
        aoff[i] = row < mend ? ((uint32_t)src * (uint32_t)p.lda + lq * 8) * 2u : SK_NOWHERE;
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
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j) acc[i][j] = sk_f32x4{0.f, 0.f, 0.f, 0.f};
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

    const int rounds = (steps + NW - 1) / NW;
    Step s0, s1;
    load(s0, wave);
    for (int r = 0; r < rounds; r += 2) {
        load(s1, (r + 1) * NW + wave);
        multiply(s0);
        load(s0, (r + 2) * NW + wave);
        multiply(s1);
    }

    // the wavefronts' sums, 16 rows at a time.  Lane (lq, l16) holds columns (4 lq + v) * CPL + j of row l16.
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (m0 + i * 16 >= mend) break;
        if (i) __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; ++v)
#pragma unroll
            for (int h = 0; h < H; ++h)
                red[wave][(v * H + h) * 64 + lane] =
                    sk_f32x4{acc[i][4 * h][v], acc[i][4 * h + 1][v], acc[i][4 * h + 2][v], acc[i][4 * h + 3][v]};
        __syncthreads();
        for (int u = tid; u < 4 * H * 64; u += NW * 64) {
            sk_f32x4 c = red[0][u];
#pragma unroll
            for (int w = 1; w < NW; ++w) c += red[w][u];
            const int l = u & 63, q = u >> 6;
            const int row = m0 + i * 16 + (l & 15);
            const int col = n0 + ((l >> 4) * 4 + q / H) * CPL + (q % H) * 4;
            if (row < mend && col < p.N) {
                const uint32_t x = Elem16<ET>::pack2(c[0], c[1]), y = Elem16<ET>::pack2(c[2], c[3]);
                if (EPI != EPI_GATED || p.C) *reinterpret_cast<u32x2_t*>(p.C + (long long)row * p.ldc + col) = u32x2_t{x, y};
                if constexpr (EPI == EPI_GATED) {
                    const float s = p.row_scale ? p.row_scale[row] : 1.0f;
                    *reinterpret_cast<uint32_t*>(p.C2 + (long long)row * p.ldc2 + (col >> 1)) =
                        Elem16<ET>::pack2(s * Elem16<ET>::hi(x) * act_fwd_fast<ACT>(Elem16<ET>::lo(x)),
                                          s * Elem16<ET>::hi(y) * act_fwd_fast<ACT>(Elem16<ET>::lo(y)));
                }
            }
        }
    }
}

// A map's tile is 16 * MT rows where the launch's own rule built it; the taller tiles of a map that was built for another
// bound of the rows are walked in parts.
template <int MT, int CPL, int NW, int EPI, int ACT, bool STREAM, typename ET>
__device__ __forceinline__ void skinny_body(const GemmArgs& p)
{
    __shared__ sk_f32x4 red[NW][CPL * 64];
    const int pm = blockIdx.x / p.n_ntiles;
    const int n0 = (blockIdx.x - pm * p.n_ntiles) * 16 * CPL;
    int e = 0, m0 = pm * 16 * MT, mend = min(m0 + 16 * MT, p.M);   // without a map: one expert that has all p.M rows
    if (p.tile_map) {
        if (pm >= min(scalar_load_i32(p.n_mtiles), p.max_mtiles)) return;
        const int32_t* ent = reinterpret_cast<const int32_t*>(p.tile_map + pm);
        e = scalar_load_i32(ent);
        m0 = scalar_load_i32(ent + 1);
        mend = scalar_load_i32(ent + 2);
    }
    skinny_tile<MT, CPL, NW, EPI, ACT, STREAM, ET>(p, red, e, m0, mend, n0);
#pragma unroll 1
    for (m0 += 16 * MT; m0 < mend; m0 += 16 * MT) {
        __syncthreads();   // (the sums are read before the next part's are written)
        skinny_tile<MT, CPL, NW, EPI, ACT, STREAM, ET>(p, red, e, m0, mend, n0);
    }
}

// (at least 4 wavefronts per SIMD with 16 rows, 3 with 32)
// STREAM: B is loaded past the caches
template <int MT, int CPL, int NW, int EPI, int ACT, bool STREAM>
__global__ void __launch_bounds__(NW * 64, MT == 1 ? 4 : 3) grouped_gemm_skinny_bf16_kernel(GemmArgs p)
{
    skinny_body<MT, CPL, NW, EPI, ACT, STREAM, bf16_t>(p);
}
template <int MT, int CPL, int NW, int EPI, int ACT, bool STREAM>
__global__ void __launch_bounds__(NW * 64, MT == 1 ? 4 : 3) grouped_gemm_skinny_f16_kernel(GemmArgs p)
{
    skinny_body<MT, CPL, NW, EPI, ACT, STREAM, f16_t>(p);
}

template <int MT, int CPL, int NW, int EPI, int ACT, bool STREAM>
int launch_skinny(const GemmArgs& a, int grid, hipStream_t s)
{
    if (a.f16)
        hipLaunchKernelGGL((grouped_gemm_skinny_f16_kernel<MT, CPL, NW, EPI, ACT, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a);
    else
        hipLaunchKernelGGL((grouped_gemm_skinny_bf16_kernel<MT, CPL, NW, EPI, ACT, STREAM>), dim3(grid), dim3(NW * 64), 0, s, a);
    return amoe_check_launch("grouped_gemm_skinny");
}

template <int MT, int CPL, int NW, int EPI, int ACT>
int launch_skinny(GemmArgs a, int m_tiles, hipStream_t s)
{
    a.n_ntiles = (a.N + 16 * CPL - 1) / (16 * CPL);
    const long long grid = (long long)m_tiles * a.n_ntiles;
    AMOE_REQUIRE(grid < (1ll << 31), AMOE_ERR_UNSUPPORTED, "grouped_gemm: grid too large");
    if (a.stream_from) return launch_skinny<MT, CPL, NW, EPI, ACT, true>(a, (int)grid, s);
    return launch_skinny<MT, CPL, NW, EPI, ACT, false>(a, (int)grid, s);
}

// bm: height of the map's tiles; R rows of a.E experts
template <int EPI, int ACT>
int launch_height(const GemmArgs& a, int bm, hipStream_t s)
{
    const int R = a.M;
    // every expert with a row has at most rows / 16 + 1 tiles, whatever rule built the map
    int m_tiles = R / 16 + (a.E < R ? a.E : R);
    if (m_tiles > R) m_tiles = R;
    if (m_tiles > a.max_mtiles) m_tiles = a.max_mtiles;
    AMOE_REQUIRE(bm == 16 || bm == 32, AMOE_ERR_UNSUPPORTED, "grouped_gemm: no kernel for tiles of %d rows", bm);
    if (bm == 32) return launch_skinny<2, 8, 4, EPI, ACT>(a, m_tiles, s);
    // too few tiles of 128 columns for the compute units (one token): half as wide, twice as many wavefronts each
    const int cus = device_cu_count();
    if ((long long)m_tiles * ((a.N + 127) / 128) < cus) return launch_skinny<1, 4, 8, EPI, ACT>(a, m_tiles, s);
    return launch_skinny<1, 8, 4, EPI, ACT>(a, m_tiles, s);
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
    if (T <= 16) return launch_skinny<1, 4, 8, EPI_STORE, 0>(a, 1, (hipStream_t)stream);
    return launch_skinny<2, 8, 4, EPI_STORE, 0>(a, (T + 31) / 32, (hipStream_t)stream);
}

AMOE_EXPORT int amoe_router_input_grad(const void* d_logits, const void* w, void* out, int dtype, int T, int E, int H, void* stream)
{
    return amoe_router_input_grad_rows(d_logits, E, w, out, dtype, T, E, H, stream);
}
