// HBM-bound row kernels: gather, weighted gather-reduce (combine / gather backward),
// combine backward, and the backward of the gated activation
// (float32, and the shared expert).  All move 16-byte vectors per lane; a row of H elements is walked by
// the 256 lanes of a block in steps of 256 vectors so every access is fully coalesced.
#include "amoe_common.h"
#include <type_traits>

namespace {

constexpr int kBlock = 256;

// xp[r,:] = x[token_of[r],:]
template <typename T>
__global__ void __launch_bounds__(kBlock)
gather_rows_kernel(const T* __restrict__ x, const int32_t* __restrict__ token_of, T* __restrict__ xp, int R, int H)
{
    constexpr int V = ElemTraits<T>::kVec;
    const int nvec = H / V;
    for (int r = blockIdx.x; r < R; r += gridDim.x) {
        const u32x4_t* src = reinterpret_cast<const u32x4_t*>(x + (size_t)token_of[r] * H);
        u32x4_t* dst = reinterpret_cast<u32x4_t*>(xp + (size_t)r * H);
        for (int i = threadIdx.x; i < nvec; i += kBlock) dst[i] = src[i];
    }
}

// dst[t,:] = (addend ? addend[t,:] : 0) + sum_k w[t,k] * src[row_of[t,k],:]   (w == null -> 1)
// SHARED adds what a shared expert gives the gradient of the input: second[t,:] + coef[t] * vec[:]
// STREAM: the rows of src are loaded past the caches
template <typename T, int KMAX, bool SHARED, bool STREAM>
__global__ void __launch_bounds__(kBlock)
gather_reduce_kernel(const T* __restrict__ src, const int32_t* __restrict__ row_of, const float* __restrict__ w,
                     const T* __restrict__ addend, T* __restrict__ dst, int n_tokens, int K, int H,
                     const T* __restrict__ second, const T* __restrict__ coef, const T* __restrict__ vec)
{
    constexpr int V = ElemTraits<T>::kVec;
    const int nvec = H / V;
    for (int t = blockIdx.x; t < n_tokens; t += gridDim.x) {
        int rows[KMAX];
        float wk[KMAX];
        const float c = SHARED ? ElemTraits<T>::load1(coef + t) : 0.f;
#pragma unroll
        for (int k = 0; k < KMAX; ++k) {
            bool ok = k < K;
            rows[k] = ok ? row_of[(size_t)t * K + k] : 0;
            wk[k] = ok ? (w ? w[(size_t)t * K + k] : 1.0f) : 0.f;
        }
        for (int i = threadIdx.x; i < nvec; i += kBlock) {
            float acc[V];
            if (addend) {
                u32x4_t a = reinterpret_cast<const u32x4_t*>(addend + (size_t)t * H)[i];
                ElemTraits<T>::unpack(a, acc);
            } else {
#pragma unroll
                for (int j = 0; j < V; ++j) acc[j] = 0.f;
            }
            if (SHARED) {
                float a[V], b[V];
                ElemTraits<T>::unpack(reinterpret_cast<const u32x4_t*>(second + (size_t)t * H)[i], a);
                ElemTraits<T>::unpack(reinterpret_cast<const u32x4_t*>(vec)[i], b);
#pragma unroll
                for (int j = 0; j < V; ++j) acc[j] += a[j] + c * b[j];
            }
#pragma unroll
            for (int k = 0; k < KMAX; ++k) {
                if (k < K) {
                    const u32x4_t* const at = reinterpret_cast<const u32x4_t*>(src + (size_t)rows[k] * H) + i;
                    const u32x4_t v = STREAM ? __builtin_nontemporal_load(at) : *at;
                    float f[V];
                    ElemTraits<T>::unpack(v, f);
#pragma unroll
                    for (int j = 0; j < V; ++j) acc[j] += wk[k] * f[j];
                }
            }
            reinterpret_cast<u32x4_t*>(dst + (size_t)t * H)[i] = ElemTraits<T>::pack(acc);
        }
    }
}

// d_out[row_of[t,k],:] = dy[t,:] * s[t,k];  d_s[t,k] = <dy[t,:], out[row_of[t,k],:]>
template <typename T>
__global__ void __launch_bounds__(kBlock)
combine_bwd_kernel(const T* __restrict__ dy, const T* __restrict__ out, const int32_t* __restrict__ row_of,
                   const float* __restrict__ scores, T* __restrict__ d_out, float* __restrict__ d_scores,
                   int n_tokens, int K, int H)
{
    constexpr int V = ElemTraits<T>::kVec;
    __shared__ float red[kBlock / AMOE_WAVE];
    const int nvec = H / V;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int t = blockIdx.x; t < n_tokens; t += gridDim.x) {
        const u32x4_t* g = reinterpret_cast<const u32x4_t*>(dy + (size_t)t * H);
        for (int k = 0; k < K; ++k) {
            const int row = row_of[(size_t)t * K + k];
            const float s = scores[(size_t)t * K + k];
            const u32x4_t* o = reinterpret_cast<const u32x4_t*>(out + (size_t)row * H);
            u32x4_t* d = d_out ? reinterpret_cast<u32x4_t*>(d_out + (size_t)row * H) : nullptr;
            float part = 0.f;
            for (int i = threadIdx.x; i < nvec; i += kBlock) {
                float gv[V], ov[V], dv[V];
                ElemTraits<T>::unpack(g[i], gv);
                ElemTraits<T>::unpack(o[i], ov);
#pragma unroll
                for (int j = 0; j < V; ++j) {
                    part += gv[j] * ov[j];
                    dv[j] = gv[j] * s;
                }
                if (d) d[i] = ElemTraits<T>::pack(dv);
            }
            part = wave_sum(part);
            __syncthreads();  // red[] free again
            if (lane == 0) red[wv] = part;
            __syncthreads();
            if (threadIdx.x == 0) {
                float tot = 0.f;
#pragma unroll
                for (int i = 0; i < kBlock / AMOE_WAVE; ++i) tot += red[i];
                d_scores[(size_t)t * K + k] = tot;
            }
        }
    }
}

// Backward of inter[r,i] = scale[r] * up * act(gate)   (one wavefront per row):
//   d_gu[r,2i]   = scale[r] * d_inter[r,i] * up * act'(gate)
//   d_gu[r,2i+1] = scale[r] * d_inter[r,i] * act(gate)
//   d_scale[r]   = sum_i d_inter[r,i] * up * act(gate)        written at slot (t,k) of row r
template <typename T, int ACT>
__global__ void __launch_bounds__(kBlock)
gated_act_bwd_kernel(const T* __restrict__ gu, const T* __restrict__ d_inter, const float* __restrict__ scale,
                     const int32_t* __restrict__ slot_of, int n_tokens, int K, T* __restrict__ d_gu,
                     float* __restrict__ d_scale_tk, int R, int I)
{
    constexpr int V = ElemTraits<T>::kVec;
    const int lane = threadIdx.x & 63;
    const int nvec = I / V;
    for (int r = blockIdx.x * (kBlock / AMOE_WAVE) + (threadIdx.x >> 6); r < R; r += gridDim.x * (kBlock / AMOE_WAVE)) {
        const float sc = scale ? scale[r] : 1.0f;
        const u32x4_t* g = reinterpret_cast<const u32x4_t*>(gu + (size_t)r * 2 * I);
        const u32x4_t* di = reinterpret_cast<const u32x4_t*>(d_inter + (size_t)r * I);
        u32x4_t* o = reinterpret_cast<u32x4_t*>(d_gu + (size_t)r * 2 * I);
        float dot = 0.f;
        for (int i = lane; i < nvec; i += AMOE_WAVE) {
            float a[V], b[V], d[V], oa[V], ob[V];
            ElemTraits<T>::unpack(g[2 * i], a);
            ElemTraits<T>::unpack(g[2 * i + 1], b);
            ElemTraits<T>::unpack(di[i], d);
#pragma unroll
            for (int j = 0; j < V / 2; ++j) {
                const float fa = act_fwd<ACT>(a[2 * j]), fb = act_fwd<ACT>(b[2 * j]);
                dot += d[j] * a[2 * j + 1] * fa + d[V / 2 + j] * b[2 * j + 1] * fb;
                oa[2 * j] = sc * d[j] * a[2 * j + 1] * act_bwd<ACT>(a[2 * j]);
                oa[2 * j + 1] = sc * d[j] * fa;
                ob[2 * j] = sc * d[V / 2 + j] * b[2 * j + 1] * act_bwd<ACT>(b[2 * j]);
                ob[2 * j + 1] = sc * d[V / 2 + j] * fb;
            }
            o[2 * i] = ElemTraits<T>::pack(oa);
            o[2 * i + 1] = ElemTraits<T>::pack(ob);
        }
        if (d_scale_tk) {
            dot = wave_sum(dot);
            if (lane == 0) {
                const int f = slot_of ? slot_of[r] : r;   // (null: one slot per row, in row order)
                const int k = f / n_tokens;
                d_scale_tk[(size_t)(f - k * n_tokens) * K + k] = dot;
            }
        }
    }
}

// d_scores[t,k] = sum_p partials[p][row_of[t,k]] (+ extra[row_of[t,k]])  (fixed order over p), added to what d_scores
// holds if `accumulate`
__global__ void __launch_bounds__(kBlock)
score_grad_gather_kernel(const float* __restrict__ partials, int n_parts, long long part_stride, const float* __restrict__ extra,
                         const int32_t* __restrict__ row_of, float* __restrict__ d_scores, int n_slots, int accumulate)
{
    const int s = blockIdx.x * kBlock + threadIdx.x;
    if (s >= n_slots) return;
    const int row = row_of[s];
    float tot = accumulate ? d_scores[s] : 0.f;
    for (int p = 0; p < n_parts; ++p) tot += partials[p * part_stride + row];
    if (extra) tot += extra[row];
    d_scores[s] = tot;
}

// sig[t] = sigmoid(<x[t,:], w>), rounded to the element type after the product and after the sigmoid as the library's
// two steps round (moe.py:311-312); one wavefront per token
template <typename T>
__global__ void __launch_bounds__(kBlock)
shared_gate_kernel(const T* __restrict__ x, const T* __restrict__ w, float* __restrict__ sig, int n_tokens, int H)
{
    constexpr int V = ElemTraits<T>::kVec;
    const int lane = threadIdx.x & 63;
    const int t = blockIdx.x * (kBlock / AMOE_WAVE) + (threadIdx.x >> 6);
    if (t >= n_tokens) return;
    float dot = 0.f;
    for (int i = lane; i < H / V; i += AMOE_WAVE) {
        float a[V], b[V];
        ElemTraits<T>::unpack(reinterpret_cast<const u32x4_t*>(x + (size_t)t * H)[i], a);
        ElemTraits<T>::unpack(reinterpret_cast<const u32x4_t*>(w)[i], b);
#pragma unroll
        for (int j = 0; j < V; ++j) dot += a[j] * b[j];
    }
    dot = ElemTraits<T>::round(wave_sum(dot));
    if (lane == 0) sig[t] = ElemTraits<T>::round(1.0f / (1.0f + expf(-dot)));
}

// d_pre[t] = d_sig[t] * sig[t] * (1 - sig[t])
template <typename T>
__global__ void __launch_bounds__(kBlock)
shared_gate_bwd_kernel(const float* __restrict__ d_sig, const float* __restrict__ sig, T* __restrict__ d_pre, int n_tokens)
{
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t < n_tokens) ElemTraits<T>::store1(d_pre + t, d_sig[t] * sig[t] * (1.0f - sig[t]));
}

// parts[s][h] = sum over the tokens t of chunk s of coef[t] * x[t,h] (chunk s: tokens s * chunk ..): the weight gradient
// of a map onto one column.  A block takes 64 vectors of columns, its wavefronts every fourth token of the chunk each;
// their sums meet in a fixed order.
// Bound by reading x once.  The library's product with one column, which this replaces: float16, T = 4001, H = 2048 32 us
// beside nothing else; in bfloat16 with some thousand tokens (6165 x 384, 13373 x 992) it kept the host busy for 11 ms a
// call.  Here: 6 us and 5 for the sum of the parts.
template <typename T>
__global__ void __launch_bounds__(kBlock)
column_grad_kernel(const T* __restrict__ x, const T* __restrict__ coef, float* __restrict__ parts, int n_tokens, int H, int chunk)
{
    constexpr int V = ElemTraits<T>::kVec, W = kBlock / AMOE_WAVE;
    __shared__ float red[W][V * AMOE_WAVE];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int i = blockIdx.x * AMOE_WAVE + lane, nvec = H / V;
    const int first = blockIdx.y * chunk, last = min(first + chunk, n_tokens);
    float acc[V] = {};
    if (i < nvec) {
#pragma unroll 4
        for (int t = first + wv; t < last; t += W) {
            const float c = ElemTraits<T>::load1(coef + t);
            float f[V];
            ElemTraits<T>::unpack(reinterpret_cast<const u32x4_t*>(x + (size_t)t * H)[i], f);
#pragma unroll
            for (int j = 0; j < V; ++j) acc[j] += c * f[j];
        }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) red[wv][j * AMOE_WAVE + lane] = acc[j];
    __syncthreads();
    for (int u = threadIdx.x; u < V * AMOE_WAVE; u += kBlock) {
        const int h = (blockIdx.x * AMOE_WAVE + (u & 63)) * V + (u >> 6);
        if (h >= H) continue;
        float s = red[0][u];
#pragma unroll
        for (int w = 1; w < W; ++w) s += red[w][u];
        parts[(size_t)blockIdx.y * H + h] = s;
    }
}

// out[h] = sum_s parts[s][h]
template <typename T>
__global__ void __launch_bounds__(AMOE_WAVE)
column_sum_kernel(const float* __restrict__ parts, int n_parts, T* __restrict__ out, int H)
{
    const int h = blockIdx.x * AMOE_WAVE + threadIdx.x;
    if (h >= H) return;
    float s = 0.f;
#pragma unroll 8
    for (int p = 0; p < n_parts; ++p) s += parts[(size_t)p * H + h];
    ElemTraits<T>::store1(out + h, s);
}

// Chunks of the tokens: 64 tokens at least, 64 chunks at most (with 2048 columns a block for every compute unit)
inline int column_grad_chunk(int T) { return T <= 64 * 64 ? 64 : (T + 63) / 64; }

// out[i] = sum_p parts[p][i] in float32, one rounding
template <typename P, typename T>
__global__ void __launch_bounds__(kBlock)
sum_parts_kernel(const P* __restrict__ parts, int n_parts, T* __restrict__ out, long long n_vec)
{
    constexpr int V = ElemTraits<T>::kVec, W = V / ElemTraits<P>::kVec;
    const u32x4_t* src = reinterpret_cast<const u32x4_t*>(parts);
    for (long long i = blockIdx.x * (long long)kBlock + threadIdx.x; i < n_vec; i += (long long)gridDim.x * kBlock) {
        float acc[V] = {};
#pragma unroll 4
        for (int p = 0; p < n_parts; ++p) {
            float f[V];
#pragma unroll
            for (int w = 0; w < W; ++w) ElemTraits<P>::unpack(src[(p * n_vec + i) * W + w], f + w * ElemTraits<P>::kVec);
#pragma unroll
            for (int j = 0; j < V; ++j) acc[j] += f[j];
        }
        reinterpret_cast<u32x4_t*>(out)[i] = ElemTraits<T>::pack(acc);
    }
}

int check_rows(const char* what, int dtype, int rows, int H)
{
    AMOE_REQUIRE(dtype == AMOE_F32 || dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_BAD_ARG, "%s: bad dtype %d", what, dtype);
    AMOE_REQUIRE(rows > 0 && H > 0, AMOE_ERR_BAD_ARG, "%s: sizes must be positive (rows=%d H=%d)", what, rows, H);
    const int vec = dtype != AMOE_F32 ? 8 : 4;
    AMOE_REQUIRE(H % vec == 0, AMOE_ERR_UNSUPPORTED, "%s: row length %d must be a multiple of %d", what, H, vec);
    return AMOE_OK;
}

inline int row_grid(int rows) { return rows < 65536 ? rows : 65536; }

}  // namespace

AMOE_EXPORT int amoe_gather_rows_fwd(const void* x, const int32_t* token_of, void* xp, int dtype, int R, int H,
                                     void* stream)
{
    AMOE_REQUIRE(x && token_of && xp, AMOE_ERR_BAD_ARG, "gather_rows_fwd: null pointer");
    int rc = check_rows("gather_rows_fwd", dtype, R, H);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL(gather_rows_kernel<ELEM>, dim3(row_grid(R)), dim3(kBlock), 0, s,
                                                 (const ELEM*)x, token_of, (ELEM*)xp, R, H))
    return amoe_check_launch("gather_rows_fwd");
}

template <typename T, bool SHARED>
static void launch_gather_reduce(const void* src, const int32_t* row_of, const float* w, const void* addend, void* dst,
                                 int T_, int K, int H, hipStream_t s, const void* second = nullptr, const void* coef = nullptr,
                                 const void* vec = nullptr)
{
    dim3 grid(row_grid(T_)), block(kBlock);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, (const T*)src, row_of, w, (const T*)addend, (T*)dst, T_, K, H, (const T*)second,
                           (const T*)coef, (const T*)vec);
    };
    auto pick = [&](auto stream) {
        constexpr bool STREAM = decltype(stream)::value;
        if (K <= 2) go(gather_reduce_kernel<T, 2, SHARED, STREAM>);
        else if (K <= 4) go(gather_reduce_kernel<T, 4, SHARED, STREAM>);
        else if (K <= 8) go(gather_reduce_kernel<T, 8, SHARED, STREAM>);
        else go(gather_reduce_kernel<T, AMOE_MAX_TOPK, SHARED, STREAM>);
    };
    // Rows that are read once and that the last-level cache (256 MiB) cannot hold, past the caches: bf16, 8 rows of 2048 for each
    // of 16384 tokens 134 -> 112 us (6.0 TB/s), 4 for 32768 157 -> 120, 7 of 4288 for 17484 271 -> 249.  (what fits is faster
    // out of the cache: 2 of 4096 for 8192 tokens, 134 MB, 40 us, 6.7 TB/s)
    if ((size_t)T_ * K * H * sizeof(T) > (size_t)256 << 20) pick(std::true_type{});
    else pick(std::false_type{});
}

AMOE_EXPORT int amoe_gather_rows_bwd(const void* d_xp, const int32_t* row_of, const void* addend, void* dx, int dtype,
                                     int T, int K, int H, void* stream)
{
    AMOE_REQUIRE(d_xp && row_of && dx, AMOE_ERR_BAD_ARG, "gather_rows_bwd: null pointer");
    int rc = check_rows("gather_rows_bwd", dtype, T, H);
    if (rc) return rc;
    AMOE_REQUIRE(K > 0 && K <= AMOE_MAX_TOPK, AMOE_ERR_UNSUPPORTED, "gather_rows_bwd: K=%d outside 1..%d", K,
                 AMOE_MAX_TOPK);
    AMOE_DISPATCH_ELEM(dtype, (launch_gather_reduce<ELEM, false>(d_xp, row_of, nullptr, addend, dx, T, K, H, (hipStream_t)stream)))
    return amoe_check_launch("gather_rows_bwd");
}

AMOE_EXPORT int amoe_combine_fwd(const void* moe_out, const int32_t* row_of, const float* scores, void* y, int dtype,
                                 int T, int K, int H, void* stream)
{
    AMOE_REQUIRE(moe_out && row_of && y, AMOE_ERR_BAD_ARG, "combine_fwd: null pointer");
    int rc = check_rows("combine_fwd", dtype, T, H);
    if (rc) return rc;
    AMOE_REQUIRE(K > 0 && K <= AMOE_MAX_TOPK, AMOE_ERR_UNSUPPORTED, "combine_fwd: K=%d outside 1..%d", K, AMOE_MAX_TOPK);
    AMOE_DISPATCH_ELEM(dtype, (launch_gather_reduce<ELEM, false>(moe_out, row_of, scores, nullptr, y, T, K, H, (hipStream_t)stream)))
    return amoe_check_launch("combine_fwd");
}

AMOE_EXPORT int amoe_combine_bwd(const void* dy, const void* moe_out, const int32_t* row_of, const float* scores,
                                 void* d_moe_out, float* d_scores, int dtype, int T, int K, int H, void* stream)
{
    AMOE_REQUIRE(dy && moe_out && row_of && scores && d_scores, AMOE_ERR_BAD_ARG, "combine_bwd: null pointer");
    int rc = check_rows("combine_bwd", dtype, T, H);
    if (rc) return rc;
    AMOE_REQUIRE(K > 0 && K <= AMOE_MAX_TOPK, AMOE_ERR_UNSUPPORTED, "combine_bwd: K=%d outside 1..%d", K, AMOE_MAX_TOPK);
    hipStream_t s = (hipStream_t)stream;
    AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL(combine_bwd_kernel<ELEM>, dim3(row_grid(T)), dim3(kBlock), 0, s,
                                                 (const ELEM*)dy, (const ELEM*)moe_out, row_of, scores, (ELEM*)d_moe_out,
                                                 d_scores, T, K, H))
    return amoe_check_launch("combine_bwd");
}

static void launch_act_bwd(const void* gate_up, const void* d_inter, const float* row_scale, const int32_t* slot_of, void* d_gate_up,
                           float* d_row_scale, int dtype, int R, int I, int T, int K, int act, hipStream_t s)
{
    const int rows_per_block = kBlock / AMOE_WAVE;
    const int grid = (R + rows_per_block - 1) / rows_per_block < 65536 ? (R + rows_per_block - 1) / rows_per_block : 65536;
    AMOE_DISPATCH_ACT(act, {
        AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL((gated_act_bwd_kernel<ELEM, ACT>), dim3(grid), dim3(kBlock), 0, s,
                                                     (const ELEM*)gate_up, (const ELEM*)d_inter, row_scale, slot_of, T, K,
                                                     (ELEM*)d_gate_up, d_row_scale, R, I))
    })
}

// the same with the gradient of row_scale in row order (a shared expert: one row per token)
int amoe_launch_gated_act_bwd_rows(const void* gate_up, const void* d_inter, const float* row_scale, void* d_gate_up, float* d_scale,
                                   int dtype, int R, int I, int act, hipStream_t s)
{
    launch_act_bwd(gate_up, d_inter, row_scale, nullptr, d_gate_up, d_scale, dtype, R, I, R, 1, act, s);
    return amoe_check_launch("gated_act_bwd");
}

AMOE_EXPORT int amoe_gated_act_bwd(const void* gate_up, const void* d_inter, const float* row_scale,
                                   const int32_t* slot_of, void* d_gate_up, float* d_row_scale, int dtype, int R, int I,
                                   int T, int K, int act, void* stream)
{
    AMOE_REQUIRE(gate_up && d_inter && d_gate_up, AMOE_ERR_BAD_ARG, "gated_act_bwd: null pointer");
    int rc = check_rows("gated_act_bwd", dtype, R, I);
    if (rc) return rc;
    AMOE_REQUIRE(act >= AMOE_ACT_SILU && act <= AMOE_ACT_GPT_OSS, AMOE_ERR_BAD_ARG, "gated_act_bwd: bad activation %d",
                 act);
    if (d_row_scale) {
        AMOE_REQUIRE(slot_of, AMOE_ERR_BAD_ARG, "gated_act_bwd: d_row_scale needs slot_of");
        AMOE_REQUIRE(T > 0 && K > 0 && (long long)T * K == (long long)R, AMOE_ERR_BAD_ARG,
                     "gated_act_bwd: T*K must equal R (T=%d K=%d R=%d)", T, K, R);
    }
    launch_act_bwd(gate_up, d_inter, row_scale, slot_of, d_gate_up, d_row_scale, dtype, R, I, T, K, act, (hipStream_t)stream);
    return amoe_check_launch("gated_act_bwd");
}

int amoe_launch_score_grad(const float* partials, int n_parts, const float* extra, const int32_t* row_of, float* d_scores,
                           int n_slots, bool accumulate, hipStream_t s)
{
    hipLaunchKernelGGL(score_grad_gather_kernel, dim3((n_slots + kBlock - 1) / kBlock), dim3(kBlock), 0, s, partials, n_parts,
                       (long long)n_slots, extra, row_of, d_scores, n_slots, (int)accumulate);
    return amoe_check_launch("score_grad_gather");
}

int amoe_launch_shared_gate(const void* x, const void* w, float* sig, int dtype, int T, int H, hipStream_t s)
{
    int rc = check_rows("shared_gate", dtype, T, H);
    if (rc) return rc;
    const dim3 grid((T + kBlock / AMOE_WAVE - 1) / (kBlock / AMOE_WAVE));
    AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL(shared_gate_kernel<ELEM>, grid, dim3(kBlock), 0, s, (const ELEM*)x, (const ELEM*)w,
                                                 sig, T, H))
    return amoe_check_launch("shared_gate");
}

int amoe_launch_shared_gate_bwd(const float* d_sig, const float* sig, void* d_pre, int dtype, int T, hipStream_t s)
{
    AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL(shared_gate_bwd_kernel<ELEM>, dim3((T + kBlock - 1) / kBlock), dim3(kBlock), 0, s,
                                                 d_sig, sig, (ELEM*)d_pre, T))
    return amoe_check_launch("shared_gate_bwd");
}

// dx[t,:] = dense[t,:] + sum_k d_xp[row_of[t,k],:]  (+ shared[t,:] + d_pre[t] * gate[:] with a shared expert)
int amoe_launch_input_grad(const void* d_xp, const int32_t* row_of, const void* dense, const void* shared, const void* d_pre,
                           const void* gate, void* dx, int dtype, int T, int K, int H, hipStream_t s)
{
    if (!shared) return amoe_gather_rows_bwd(d_xp, row_of, dense, dx, dtype, T, K, H, s);
    int rc = check_rows("input_grad", dtype, T, H);
    if (rc) return rc;
    AMOE_DISPATCH_ELEM(dtype, (launch_gather_reduce<ELEM, true>(d_xp, row_of, nullptr, dense, dx, T, K, H, s, shared, d_pre, gate)))
    return amoe_check_launch("input_grad");
}

int amoe_launch_sum_parts(const void* parts, int n_parts, void* out, int parts_dtype, int dtype, long long n, hipStream_t s)
{
    const int vec = dtype != AMOE_F32 ? 8 : 4;
    AMOE_REQUIRE(n % vec == 0, AMOE_ERR_UNSUPPORTED, "sum_parts: %lld elements are no multiple of %d", n, vec);
    const long long blocks = (n / vec + kBlock - 1) / kBlock;
    const dim3 grid((unsigned)(blocks < 8192 ? blocks : 8192));
    if (parts_dtype == AMOE_F32) {
        AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL((sum_parts_kernel<float, ELEM>), grid, dim3(kBlock), 0, s, (const float*)parts,
                                                     n_parts, (ELEM*)out, n / vec))
    } else {
        AMOE_REQUIRE(parts_dtype == dtype, AMOE_ERR_BAD_ARG, "sum_parts: parts of another type");
        AMOE_DISPATCH_ELEM(dtype, hipLaunchKernelGGL((sum_parts_kernel<ELEM, ELEM>), grid, dim3(kBlock), 0, s, (const ELEM*)parts,
                                                     n_parts, (ELEM*)out, n / vec))
    }
    return amoe_check_launch("sum_parts");
}

AMOE_EXPORT size_t amoe_column_grad_workspace_bytes(int T, int H)
{
    if (T <= 0 || H <= 0) return 0;
    const int chunk = column_grad_chunk(T);
    return (size_t)((T + chunk - 1) / chunk) * H * sizeof(float);
}

AMOE_EXPORT int amoe_column_grad(const void* x, const void* coef, void* out, int dtype, int T, int H, void* workspace,
                                 size_t workspace_bytes, void* stream)
{
    AMOE_REQUIRE(x && coef && out && workspace, AMOE_ERR_BAD_ARG, "column_grad: null pointer");
    int rc = check_rows("column_grad", dtype, T, H);
    if (rc) return rc;
    AMOE_REQUIRE(workspace_bytes >= amoe_column_grad_workspace_bytes(T, H), AMOE_ERR_WORKSPACE, "column_grad: workspace %zu < %zu bytes",
                 workspace_bytes, amoe_column_grad_workspace_bytes(T, H));
    hipStream_t s = (hipStream_t)stream;
    const int chunk = column_grad_chunk(T), parts = (T + chunk - 1) / chunk;
    AMOE_DISPATCH_ELEM(dtype, {
        const int nvec = H / ElemTraits<ELEM>::kVec;
        hipLaunchKernelGGL(column_grad_kernel<ELEM>, dim3((nvec + AMOE_WAVE - 1) / AMOE_WAVE, parts), dim3(kBlock), 0, s, (const ELEM*)x,
                           (const ELEM*)coef, (float*)workspace, T, H, chunk);
        hipLaunchKernelGGL(column_sum_kernel<ELEM>, dim3((H + AMOE_WAVE - 1) / AMOE_WAVE), dim3(AMOE_WAVE), 0, s,
                           (const float*)workspace, parts, (ELEM*)out, H);
    })
    return amoe_check_launch("column_grad");
}

AMOE_EXPORT int amoe_score_grad_gather(const float* partials, int n_parts, const int32_t* row_of, float* d_scores, int T,
                                       int K, void* stream)
{
    AMOE_REQUIRE(partials && row_of && d_scores, AMOE_ERR_BAD_ARG, "score_grad_gather: null pointer");
    AMOE_REQUIRE(n_parts > 0 && T > 0 && K > 0, AMOE_ERR_BAD_ARG, "score_grad_gather: sizes must be positive");
    AMOE_REQUIRE((long long)T * K < (1ll << 31), AMOE_ERR_UNSUPPORTED, "score_grad_gather: T*K does not fit int32");
    return amoe_launch_score_grad(partials, n_parts, nullptr, row_of, d_scores, T * K, false, (hipStream_t)stream);
}
