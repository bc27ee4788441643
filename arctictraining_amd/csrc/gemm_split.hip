// Row-grouped 16-bit products whose tiles leave most compute units idle: the reduction is cut into parts, each a tile of its
// own on the default kernel (gemm_pp.hip, EPI_PART), and the parts, in float32, are added here, with the epilogue of the
// product behind the sum.
//
// Bound by memory: splits x 4 bytes read for every output.  One MI355X, us, whole tiles / parts + sum: 744 rows of 5 experts
// and of a shared one beside them, A B of K = 11648, N = 864 198 / 47 + 7 each, A B^T of K = 23296 370 / 76 + 7; 472 rows of 7
// experts, K = 3200, N = 640 40 / 17 + 4; 3165 rows of 7 experts, A B^T of K = 13568, N = 1152 268 / 120 + 9; 3390 rows of 6
// experts, the gated product of K = 6560, N = 896 114 / 55 + 8.
#include "gemm_common.h"
#include "gemm_calls.h"
#include "gemm_launch.h"

int amoe_pp_part(const GemmArgs& a, bool b_kc, hipStream_t s);

namespace {

constexpr int kBlock = 256;

// eight columns of one row, added in the parts' order
__device__ __forceinline__ void sum8(const float* __restrict__ parts, int splits, long long stride, long long at, float (&c)[8])
{
    f32x4_t a = {0.f, 0.f, 0.f, 0.f}, b = a;
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
        const f32x4_t* p = reinterpret_cast<const f32x4_t*>(parts + s * stride + at);
        a += p[0];
        b += p[1];
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        c[v] = a[v];
        c[4 + v] = b[v];
    }
}

template <typename ET>
__global__ void __launch_bounds__(kBlock)
split_store_kernel(const float* __restrict__ parts, int splits, long long stride, ET* __restrict__ out, long long n8)
{
    const long long i = blockIdx.x * (long long)kBlock + threadIdx.x;
    if (i >= n8) return;
    float c[8];
    sum8(parts, splits, stride, i * 8, c);
    reinterpret_cast<u32x4_t*>(out)[i] = u32x4_t{Elem16<ET>::pack2(c[0], c[1]), Elem16<ET>::pack2(c[2], c[3]), Elem16<ET>::pack2(c[4], c[5]),
                                                 Elem16<ET>::pack2(c[6], c[7])};
}

// a packed pair is (gate, up) of one intermediate column
template <typename ET, int ACT>
__global__ void __launch_bounds__(kBlock)
split_gated_kernel(const float* __restrict__ parts, int splits, long long stride, const float* __restrict__ row_scale,
                   ET* __restrict__ gate_up, ET* __restrict__ inter, long long n8, int row8)
{
    const long long i = blockIdx.x * (long long)kBlock + threadIdx.x;
    if (i >= n8) return;
    float c[8];
    sum8(parts, splits, stride, i * 8, c);
    const float s = row_scale ? row_scale[i / row8] : 1.0f;
    u32x4_t g;
    float h[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        g[v] = Elem16<ET>::pack2(c[2 * v], c[2 * v + 1]);
        h[v] = s * Elem16<ET>::hi(g[v]) * act_fwd_fast<ACT>(Elem16<ET>::lo(g[v]));
    }
    if (gate_up) reinterpret_cast<u32x4_t*>(gate_up)[i] = g;
    reinterpret_cast<u32x2_t*>(inter)[i] = u32x2_t{Elem16<ET>::pack2(h[0], h[1]), Elem16<ET>::pack2(h[2], h[3])};
}

// one wavefront per row and 256 columns, whose sum is a row-sum partial as the fused epilogue leaves them
template <typename ET, int ACT>
__global__ void __launch_bounds__(kBlock)
split_gated_bwd_kernel(const float* __restrict__ parts, int splits, long long stride, const float* __restrict__ row_scale,
                       const ET* __restrict__ gate_up, ET* __restrict__ d_gate_up, float* __restrict__ partials, int R, int I, int n_blocks)
{
    const long long unit = blockIdx.x * (long long)(kBlock / AMOE_WAVE) + (threadIdx.x >> 6);
    if (unit >= (long long)R * n_blocks) return;
    const int row = (int)(unit / n_blocks), nb = (int)(unit - (long long)row * n_blocks);
    const int lane = threadIdx.x & 63, c = nb * 256 + lane * 4;
    float dot = 0.f;
    if (c < I) {
        f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
        for (int s = 0; s < splits; ++s) d += *reinterpret_cast<const f32x4_t*>(parts + s * stride + (long long)row * I + c);
        const long long at = ((long long)row * I + c) * 2;
        const u32x4_t gu = *reinterpret_cast<const u32x4_t*>(gate_up + at);
        const float sc = row_scale ? row_scale[row] : 1.0f;
        u32x4_t o;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float gate = Elem16<ET>::lo(gu[v]), up = Elem16<ET>::hi(gu[v]);
            float f, df;
            act_both_fast<ACT>(gate, f, df);
            dot += d[v] * up * f;
            const float sd = sc * d[v];
            o[v] = Elem16<ET>::pack2(sd * up * df, sd * f);
        }
        *reinterpret_cast<u32x4_t*>(d_gate_up + at) = o;
    }
    if (partials) {
        dot = wave_sum(dot);
        if (lane == 0) partials[(long long)nb * R + row] = dot;
    }
}

}  // namespace

// Into how many parts the reduction over K of R rows of E experts, N columns, is cut (1: not at all).  A tile's K tile takes
// 0.9 us whether one compute unit works or half of them do; the parts cost their bytes, written and read at 5 TB/s, and one
// more launch.  No more tiles than compute units (an expert's last tile counts half: they are not all there), six K tiles a
// part at least.
int amoe_split_count(int R, int E, int K, int N)
{
    if (R <= 8ll * E) return 1;          // (low tiles: gemm_skinny.hip, and many of them)
    const long long tiles = ((long long)R / 256 + E / 2 + 1) * ((N + 255) / 256), kt = (K + 63) / 64;
    const int cus = device_cu_count();
    int best = 1;
    double most = 0.0;
    for (int s = 2; s <= 16 && kt / s >= 6 && tiles * s <= cus; ++s) {
        const double gain = 0.9 * (double)(kt - (kt + s - 1) / s) - (5.0 + 8e-6 * (double)s * R * N / 5.0);
        if (gain > most) {
            most = gain;
            best = s;
        }
    }
    return best;
}

size_t amoe_split_bytes(int R, int E, int K, int N)
{
    const int s = amoe_split_count(R, E, K, N);
    return s > 1 ? (size_t)s * R * N * sizeof(float) : 0;
}

// a: the product as for the default kernel, super-tiles set for n_ntiles = n_real * splits
int amoe_split_rows(const GemmArgs& a, bool b_kc, int epi, int act, hipStream_t s)
{
    int rc = amoe_pp_part(a, b_kc, s);
    if (rc) return rc;
    const long long n = (long long)a.M * a.N, n8 = n / 8;
    const dim3 grid((unsigned)((n8 + kBlock - 1) / kBlock)), block(kBlock);
#define AMOE_SPLIT(...)                                               \
    if (a.f16) { typedef f16_t ET; __VA_ARGS__; }                     \
    else { typedef bf16_t ET; __VA_ARGS__; }
    if (epi == EPI_STORE) {
        AMOE_SPLIT(hipLaunchKernelGGL(split_store_kernel<ET>, grid, block, 0, s, a.split_out, a.splits, n, (ET*)a.C, n8))
    } else if (epi == EPI_GATED) {
        AMOE_DISPATCH_ACT(act, AMOE_SPLIT(hipLaunchKernelGGL((split_gated_kernel<ET, ACT>), grid, block, 0, s, a.split_out, a.splits, n,
                                                             a.row_scale, (ET*)a.C, (ET*)a.C2, n8, a.N / 8)))
    } else {
        const int blocks = (a.N + 255) / 256;
        const long long units = (long long)a.M * blocks;
        const dim3 waves((unsigned)((units + kBlock / AMOE_WAVE - 1) / (kBlock / AMOE_WAVE)));
        AMOE_DISPATCH_ACT(act, AMOE_SPLIT(hipLaunchKernelGGL((split_gated_bwd_kernel<ET, ACT>), waves, block, 0, s, a.split_out, a.splits, n,
                                                             a.row_scale, (const ET*)a.G, (ET*)a.C, a.partials, a.M, a.N, blocks)))
    }
#undef AMOE_SPLIT
    return amoe_check_launch("grouped_gemm_split");
}
