// Router softmax / top-k and its backward: one 64-lane wavefront per token, expert values
// spread over lanes (expert e lives in lane e % 64, register e / 64), reductions by
// cross-lane shuffles.  HBM-bound: T*E logits in, T*E probabilities + T*K pairs out.
#include "router_topk.h"

namespace {

constexpr int kTokensPerBlock = 4;  // 4 wavefronts

template <typename T, int VPT>
__global__ void __launch_bounds__(kTokensPerBlock * AMOE_WAVE)
router_topk_fwd_kernel(const T* __restrict__ logits, int n_tokens, int E, int K, int normalize,
                       float* __restrict__ probs, int32_t* __restrict__ topk_idx, float* __restrict__ scores)
{
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * kTokensPerBlock + (threadIdx.x >> 6);
    if (t >= n_tokens) return;
    int top_e;
    float s;
    router_topk_token<T, VPT>(logits + (size_t)t * E, E, K, normalize, lane, probs + (size_t)t * E, top_e, s);
    if (lane < K) {
        topk_idx[(size_t)t * K + lane] = top_e;
        scores[(size_t)t * K + lane] = s;
    }
}

template <typename T, int VPT>
__global__ void __launch_bounds__(kTokensPerBlock * AMOE_WAVE)
router_bwd_kernel(const float* __restrict__ d_scores, const float* __restrict__ probs,
                  const int32_t* __restrict__ topk_idx, const int32_t* __restrict__ counts, int n_tokens, int E,
                  int K, int normalize, float lb_coeff, T* __restrict__ d_logits, int ld)
{
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * kTokensPerBlock + (threadIdx.x >> 6);
    if (t >= n_tokens) return;
    const float* prow = probs + (size_t)t * E;

    float p[VPT], dp[VPT];
    float cnt_part = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        int e = lane + 64 * j;
        bool ok = e < E;
        p[j] = ok ? prow[e] : 0.f;
        float c = ok ? (float)counts[e] : 0.f;
        dp[j] = c;  // scaled below once the total is known
        cnt_part += c;
    }
    const float total = wave_sum(cnt_part);
    const float lb = total > 0.f ? lb_coeff / total : 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) dp[j] *= lb;

    // lanes 0..K-1 hold one selected slot each
    int e_k = 0;
    float ds_k = 0.f, p_k = 0.f;
    if (lane < K) {
        e_k = topk_idx[(size_t)t * K + lane];
        ds_k = d_scores[(size_t)t * K + lane];
        p_k = prow[e_k];
    }
    float dptop = ds_k;
    if (normalize) {
        float S = wave_sum(p_k);
        float dot = wave_sum(ds_k * (p_k / S));
        dptop = (ds_k - dot) / S;
    }
    for (int k = 0; k < K; ++k) {
        int e = __shfl(e_k, k, AMOE_WAVE);
        float g = __shfl(dptop, k, AMOE_WAVE);
#pragma unroll
        for (int j = 0; j < VPT; ++j)
            if (lane + 64 * j == e) dp[j] += g;
    }
    float part = 0.f;
#pragma unroll
    for (int j = 0; j < VPT; ++j) part += p[j] * dp[j];
    const float inner = wave_sum(part);
    T* out = d_logits + (size_t)t * ld;
#pragma unroll
    for (int j = 0; j < VPT; ++j) {
        int e = lane + 64 * j;
        if (e < ld) ElemTraits<T>::store1(out + e, e < E ? p[j] * (dp[j] - inner) : 0.f);
    }
}

int check_router_shape(int T, int E, int K)
{
    AMOE_REQUIRE(T > 0 && E > 0 && K > 0, AMOE_ERR_BAD_ARG, "router: T, E, K must be positive (T=%d E=%d K=%d)", T, E, K);
    AMOE_REQUIRE(E <= AMOE_MAX_EXPERTS, AMOE_ERR_UNSUPPORTED, "router: E=%d exceeds %d", E, AMOE_MAX_EXPERTS);
    AMOE_REQUIRE(K <= E && K <= AMOE_MAX_TOPK, AMOE_ERR_UNSUPPORTED, "router: K=%d must be <= min(E=%d, %d)", K, E,
                 AMOE_MAX_TOPK);
    return AMOE_OK;
}

}  // namespace

AMOE_EXPORT int amoe_router_topk_fwd(const void* logits, int dtype, int T, int E, int K, int normalize, float* probs,
                                     int32_t* topk_idx, float* scores, void* stream)
{
    AMOE_REQUIRE(logits && probs && topk_idx && scores, AMOE_ERR_BAD_ARG, "router_topk_fwd: null pointer");
    AMOE_REQUIRE(dtype == AMOE_F32 || dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_BAD_ARG, "router_topk_fwd: bad dtype %d", dtype);
    int rc = check_router_shape(T, E, K);
    if (rc) return rc;
    dim3 grid((T + kTokensPerBlock - 1) / kTokensPerBlock), block(kTokensPerBlock * AMOE_WAVE);
    hipStream_t s = (hipStream_t)stream;
    ROUTER_DISPATCH_VPT(E, {
        AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL((router_topk_fwd_kernel<ELEM, VPT>), grid, block, 0, s,
                                                     (const ELEM*)logits, T, E, K, normalize, probs, topk_idx, scores))
    })
    return amoe_check_launch("router_topk_fwd");
}

// ld: elements from one row of d_logits to the next, at most 32 past E; those past E are set to zero
int amoe_launch_router_bwd(const float* d_scores, const float* probs, const int32_t* topk_idx, const int32_t* counts, int dtype, int T,
                           int E, int K, int normalize, float lb_coeff, void* d_logits, int ld, hipStream_t s)
{
    AMOE_REQUIRE(d_scores && probs && topk_idx && counts && d_logits, AMOE_ERR_BAD_ARG, "router_bwd: null pointer");
    AMOE_REQUIRE(dtype == AMOE_F32 || dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_BAD_ARG, "router_bwd: bad dtype %d", dtype);
    int rc = check_router_shape(T, E, K);
    if (rc) return rc;
    AMOE_REQUIRE(ld >= E && ld <= (E + 31) / 32 * 32, AMOE_ERR_BAD_ARG, "router_bwd: rows of %d elements for %d experts", ld, E);
    dim3 grid((T + kTokensPerBlock - 1) / kTokensPerBlock), block(kTokensPerBlock * AMOE_WAVE);
    ROUTER_DISPATCH_VPT(E, {
        AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL((router_bwd_kernel<ELEM, VPT>), grid, block, 0, s, d_scores, probs,
                                                     topk_idx, counts, T, E, K, normalize, lb_coeff, (ELEM*)d_logits, ld))
    })
    return amoe_check_launch("router_bwd");
}

AMOE_EXPORT int amoe_router_bwd(const float* d_scores, const float* probs, const int32_t* topk_idx,
                                const int32_t* counts, int dtype, int T, int E, int K, int normalize, float lb_coeff,
                                void* d_logits, void* stream)
{
    return amoe_launch_router_bwd(d_scores, probs, topk_idx, counts, dtype, T, E, K, normalize, lb_coeff, d_logits, E, (hipStream_t)stream);
}
