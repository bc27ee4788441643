// Deterministic token-to-expert permutation plan: a stable counting sort of the k-major
// flattened assignment vector, in one launch of one block for few rows and otherwise in three launches
//   1. per-chunk expert histograms (LDS counters),
//   2. a one-block scan over chunks and experts (counts, offsets, per-chunk bases),
//   3. per-chunk ranking in ascending slot order (ballot match inside a wavefront, LDS
//      running counters across steps) and the scatter of the three index maps.
// A chunk is kChunk consecutive flat slots f = k*T + t handled by ONE wavefront, so the
// order inside an expert is ascending f by construction, with no global atomics.
#include "router_topk.h"

#include <atomic>

namespace {

constexpr int kChunk = 512;         // flat slots per wavefront
constexpr int kWavesPerBlock = 4;   // independent chunks per block

__device__ __forceinline__ int load_expert(const int32_t* assign, int f, int T, int K, int E)
{
    int k = f / T;
    int t = f - k * T;
    int e = assign[(size_t)t * K + k];
    return min(max(e, 0), E - 1);  // memory safety for caller-supplied assignments
}

__global__ void __launch_bounds__(kWavesPerBlock * AMOE_WAVE)
permute_hist_kernel(const int32_t* __restrict__ assign, int T, int K, int E, int R, int n_chunks,
                    int32_t* __restrict__ chunk_counts)
{
    __shared__ int32_t cnt[kWavesPerBlock][AMOE_MAX_EXPERTS];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = blockIdx.x * kWavesPerBlock + w;
    for (int e = lane; e < E; e += 64) cnt[w][e] = 0;
    __syncthreads();
    if (c < n_chunks) {
        const int f0 = c * kChunk;
        const int f1 = min(f0 + kChunk, R);
        for (int f = f0 + lane; f < f1; f += 64) atomicAdd(&cnt[w][load_expert(assign, f, T, K, E)], 1);
    }
    __syncthreads();
    if (c < n_chunks)
        for (int e = lane; e < E; e += 64) chunk_counts[(size_t)c * E + e] = cnt[w][e];
}

// Inclusive scan over the experts of the row counts, by ONE wavefront (lane t): 8 consecutive entries per lane
// serially, the lane sums by cross-lane shuffles (a block-wide Hillis-Steele scan costs 18 barriers of 16 wavefronts).
__device__ __forceinline__ void scan_row_counts(int32_t* tot, int t)
{
    static_assert(AMOE_MAX_EXPERTS == 8 * AMOE_WAVE, "one wavefront scans 8 entries per lane");
    int r[8];
    int s_rows = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        r[i] = tot[t * 8 + i];
        s_rows += r[i];
    }
    int in_rows = s_rows;
#pragma unroll
    for (int o = 1; o < AMOE_WAVE; o <<= 1) {
        const int u = __shfl_up(in_rows, o, AMOE_WAVE);
        if (t >= o) in_rows += u;
    }
    int run_rows = in_rows - s_rows;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        run_rows += r[i];
        tot[t * 8 + i] = run_rows;
    }
}

// rank of this lane among the lanes below it that hold the same expert, and whether it is the last of them
__device__ __forceinline__ int rank_of(int e, bool valid, int lane, bool* last)
{
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 9; ++b) {
        const unsigned long long bits = __ballot((e >> b) & 1);
        same &= ((e >> b) & 1) ? bits : ~bits;
    }
    *last = valid && (same >> lane) == 1ull;
    return __popcll(same & ((1ull << lane) - 1ull));
}

// One block of 1024 threads: with EP = E rounded up to a power of two, thread t works for
// expert t % EP on the (t / EP)-th slice of the chunks, so that the walk over chunks (the only
// sequential part) is 1024 / EP ways parallel and every load is coalesced over experts.  A
// thread holds its slice of counts in registers between the two passes (kScanBatch at a time):
// the exclusive bases overwrite the counts in place, and loads issued after such a store cannot
// be moved ahead of it, which would turn the second pass into a chain of dependent round trips.
// When tile_map is non-null the block also writes the row-grouped GEMMs' tile map (one int4
// {expert, first row, end row, 0} per `bm`-row tile, {-1,0,0,0} past the last) and its tile count.
constexpr int kScanThreads = 1024;
constexpr int kScanBatch = 16;

__global__ void __launch_bounds__(kScanThreads)
permute_scan_kernel(int32_t* __restrict__ chunk_counts /* in: counts, out: exclusive base inside expert */,
                    int E, int EP, int n_chunks, int32_t* __restrict__ counts, int32_t* __restrict__ offsets,
                    int4* __restrict__ tile_map, int32_t* __restrict__ n_mtiles, int bm, int max_mtiles)
{
    __shared__ int32_t part[kScanThreads];       // [slice][EP]
    __shared__ int32_t tot[AMOE_MAX_EXPERTS + 1];
    __shared__ int32_t tstart[AMOE_MAX_EXPERTS + 1];
    const int t = threadIdx.x;
    const int e = t & (EP - 1);
    const int g = t / EP;
    const int G = kScanThreads / EP;
    const int per = (n_chunks + G - 1) / G;
    const int c0 = min(g * per, n_chunks), c1 = min(c0 + per, n_chunks);
    int sum = 0;
    if (e < E)
        for (int cb = c0; cb < c1; cb += kScanBatch) {
            int v[kScanBatch];
#pragma unroll
            for (int i = 0; i < kScanBatch; ++i) v[i] = cb + i < c1 ? chunk_counts[(size_t)(cb + i) * E + e] : 0;
#pragma unroll
            for (int i = 0; i < kScanBatch; ++i) sum += v[i];
        }
    part[t] = sum;
    __syncthreads();
    int run = 0;
    for (int gg = 0; gg < g; ++gg) run += part[gg * EP + e];
    if (g == G - 1 && e < E) {
        counts[e] = run + sum;
        tot[e] = run + sum;
    }
    if (e < E)
        for (int cb = c0; cb < c1; cb += kScanBatch) {
            int v[kScanBatch];
#pragma unroll
            for (int i = 0; i < kScanBatch; ++i) v[i] = cb + i < c1 ? chunk_counts[(size_t)(cb + i) * E + e] : 0;
#pragma unroll
            for (int i = 0; i < kScanBatch; ++i) {
                if (cb + i < c1) chunk_counts[(size_t)(cb + i) * E + e] = run;
                run += v[i];
            }
        }
    if (t < AMOE_MAX_EXPERTS && t >= E) tot[t] = 0;
    __syncthreads();
    if (t < AMOE_WAVE) scan_row_counts(tot, t);
    __syncthreads();
    if (t < E) offsets[t + 1] = tot[t];
    if (t == 0) offsets[0] = 0;
    if (tile_map == nullptr) return;
    // tot[e] = end row of expert e
    amoe_emit_tile_map<kScanThreads>(tot, 0, E, bm, tile_map, n_mtiles, max_mtiles, tstart);
}

__global__ void __launch_bounds__(kWavesPerBlock * AMOE_WAVE)
permute_scatter_kernel(const int32_t* __restrict__ assign, int T, int K, int E, int R, int n_chunks,
                       const int32_t* __restrict__ chunk_base, const int32_t* __restrict__ offsets,
                       const float* __restrict__ scores, int32_t* __restrict__ token_of, int32_t* __restrict__ slot_of,
                       int32_t* __restrict__ row_of, float* __restrict__ scores_perm)
{
    __shared__ int32_t run[kWavesPerBlock][AMOE_MAX_EXPERTS];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int c = blockIdx.x * kWavesPerBlock + w;
    if (c >= n_chunks) return;  // no block-wide barrier below: every wavefront is independent
    for (int e = lane; e < E; e += 64) run[w][e] = offsets[e] + chunk_base[(size_t)c * E + e];
    __builtin_amdgcn_wave_barrier();
    const int f0 = c * kChunk;
    const int f1 = min(f0 + kChunk, R);
    for (int fb = f0; fb < f1; fb += 64) {
        const int f = fb + lane;
        const bool valid = f < f1;
        const int e = valid ? load_expert(assign, f, T, K, E) : 0;
        bool last;
        const int rank = rank_of(e, valid, lane, &last);
        int row = 0;
        if (valid) row = run[w][e] + rank;
        __builtin_amdgcn_wave_barrier();
        // the highest lane of each group advances the running counter
        if (last) run[w][e] = row + 1;
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            int k = f / T;
            int t = f - k * T;
            token_of[row] = t;
            slot_of[row] = f;
            row_of[(size_t)t * K + k] = row;
            if (scores_perm) scores_perm[row] = scores[(size_t)t * K + k];
        }
    }
}

// The whole plan in one block, for up to kSmallRows routed rows: the three kernels above are 2-8 us each there, most
// of it their launches and the chain of memory round trips between them (one token 8.7 us, 512 rows 17 us).  Sixteen
// wavefronts take consecutive chunks of the slots, so an expert's rows come in ascending slot order as above; the
// chunk counts stay in LDS and the experts of a wavefront's slots in its registers.  One MI355X:
// one token of 8 experts 8.7 -> 4.8 us, 4096 rows 20 -> 11 us, and two launches fewer for the host.
constexpr int kSmallWaves = 16, kSmallSteps = 8;
constexpr int kSmallRows = kSmallWaves * kSmallSteps * AMOE_WAVE;

struct PlanOut {
    int32_t *counts, *offsets, *token_of, *slot_of, *row_of;
    float* scores_perm;
    int4* tile_map;
    int32_t* n_mtiles;
    int bm, max_mtiles;
};

// expert_of(flat slot), score_of(token, k)
template <typename ExpertOf, typename ScoreOf>
__device__ __forceinline__ void plan_in_block(ExpertOf expert_of, ScoreOf score_of, int T, int K, int E, int R,
                                              int steps /* of 64 slots per wavefront */, const PlanOut& o)
{
    __shared__ int32_t run[kSmallWaves][AMOE_MAX_EXPERTS];
    __shared__ int32_t tot[AMOE_MAX_EXPERTS + 1];
    __shared__ int32_t tstart[AMOE_MAX_EXPERTS + 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const int f0 = w * steps * AMOE_WAVE + lane;
    int ex[kSmallSteps];
#pragma unroll
    for (int i = 0; i < kSmallSteps; ++i) {
        const int f = f0 + i * AMOE_WAVE;
        ex[i] = i < steps && f < R ? expert_of(f) : -1;
    }
    for (int e = lane; e < E; e += AMOE_WAVE) run[w][e] = 0;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kSmallSteps; ++i)
        if (ex[i] >= 0) atomicAdd(&run[w][ex[i]], 1);
    __syncthreads();
    if (t < AMOE_MAX_EXPERTS) {
        int sum = 0;
        if (t < E) {
            // counts of the chunks -> exclusive bases inside the expert
#pragma unroll
            for (int c = 0; c < kSmallWaves; ++c) {
                const int v = run[c][t];
                run[c][t] = sum;
                sum += v;
            }
            o.counts[t] = sum;
        }
        tot[t] = sum;
    }
    __syncthreads();
    if (t < AMOE_WAVE) scan_row_counts(tot, t);
    __syncthreads();
    if (t < E) o.offsets[t + 1] = tot[t];
    if (t == 0) o.offsets[0] = 0;
#pragma unroll
    for (int i = 0; i < kSmallSteps; ++i) {
        if (i >= steps) break;
        const bool valid = ex[i] >= 0;
        const int e = valid ? ex[i] : 0;
        bool last;
        const int rank = rank_of(e, valid, lane, &last);
        int in_expert = 0;
        if (valid) in_expert = run[w][e] + rank;
        __builtin_amdgcn_wave_barrier();
        if (last) run[w][e] = in_expert + 1;
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            const int f = f0 + i * AMOE_WAVE;
            const int k = f / T, tok = f - k * T;
            const int row = in_expert + (e ? tot[e - 1] : 0);
            o.token_of[row] = tok;
            o.slot_of[row] = f;
            o.row_of[(size_t)tok * K + k] = row;
            if (o.scores_perm) o.scores_perm[row] = score_of(tok, k);
        }
    }
    if (o.tile_map) amoe_emit_tile_map<kSmallWaves * AMOE_WAVE>(tot, 0, E, o.bm, o.tile_map, o.n_mtiles, o.max_mtiles, tstart);
}

__global__ void __launch_bounds__(kSmallWaves * AMOE_WAVE)
permute_small_kernel(const int32_t* __restrict__ assign, int T, int K, int E, int R, int steps, const float* __restrict__ scores, PlanOut o)
{
    plan_in_block([&](int f) { return load_expert(assign, f, T, K, E); }, [&](int t, int k) { return scores[(size_t)t * K + k]; }, T, K, E, R,
                  steps, o);
}

// Softmax, top-k and the plan of at most one token per wavefront of the block: the selection reaches the plan through LDS.
// (One token through 128 experts of 2048 x 768, the whole forward: 41 us with two launches, 37 with this one.)
template <typename T, int VPT>
__global__ void __launch_bounds__(kSmallWaves * AMOE_WAVE)
route_small_kernel(const T* __restrict__ logits, int n_tokens, int E, int K, int normalize, float* __restrict__ probs,
                   int32_t* __restrict__ topk_idx, float* __restrict__ scores, PlanOut o)
{
    __shared__ int32_t sel[kSmallWaves][AMOE_MAX_TOPK];
    __shared__ float sc[kSmallWaves][AMOE_MAX_TOPK];
    const int lane = threadIdx.x & 63, t = threadIdx.x >> 6;
    if (t < n_tokens) {
        int e;
        float s;
        router_topk_token<T, VPT>(logits + (size_t)t * E, E, K, normalize, lane, probs + (size_t)t * E, e, s);
        if (lane < K) {
            topk_idx[(size_t)t * K + lane] = e;
            scores[(size_t)t * K + lane] = s;
            sel[t][lane] = min(max(e, 0), E - 1);
            sc[t][lane] = s;
        }
    }
    __syncthreads();
    const int R = n_tokens * K;
    auto expert_of = [&](int f) {
        const int k = f / n_tokens;
        return sel[f - k * n_tokens][k];
    };
    plan_in_block(expert_of, [&](int tok, int k) { return sc[tok][k]; }, n_tokens, K, E, R,
                  (R + kSmallWaves * AMOE_WAVE - 1) / (kSmallWaves * AMOE_WAVE), o);
}

}  // namespace

static inline int permute_chunks(int R) { return (R + kChunk - 1) / kChunk; }

AMOE_EXPORT size_t amoe_permute_workspace_bytes(int R, int E)
{
    if (R <= 0 || E <= 0) return 0;
    return (size_t)permute_chunks(R) * (size_t)E * sizeof(int32_t);
}

// argument checks shared by the two entry points (all before the first HIP call)
static int check_plan_args(const int32_t* assign, const float* scores, int T, int K, int E, int32_t* counts,
                           int32_t* offsets, int32_t* token_of, int32_t* slot_of, int32_t* row_of, float* scores_perm)
{
    AMOE_REQUIRE(assign && counts && offsets && token_of && slot_of && row_of, AMOE_ERR_BAD_ARG,
                 "permute_plan: null pointer");
    AMOE_REQUIRE(!scores_perm || scores, AMOE_ERR_BAD_ARG, "permute_plan: scores_perm needs scores");
    AMOE_REQUIRE(T > 0 && K > 0 && E > 0, AMOE_ERR_BAD_ARG, "permute_plan: T, K, E must be positive");
    AMOE_REQUIRE(E <= AMOE_MAX_EXPERTS, AMOE_ERR_UNSUPPORTED, "permute_plan: E=%d exceeds %d", E, AMOE_MAX_EXPERTS);
    AMOE_REQUIRE((long long)T * K < (1ll << 31), AMOE_ERR_UNSUPPORTED, "permute_plan: T*K does not fit int32");
    return AMOE_OK;
}

// the three launches; cc = per-chunk expert counts, permute_chunks(R) * E int32 (every entry is
// written by the histogram kernel before it is read: nothing has to be cleared)
static int launch_plan(const int32_t* assign, const float* scores, int T, int K, int E, int32_t* counts,
                       int32_t* offsets, int32_t* token_of, int32_t* slot_of, int32_t* row_of, float* scores_perm,
                       int32_t* cc, hipStream_t s, int4* tile_map = nullptr, int32_t* n_mtiles = nullptr, int bm = 1,
                       int max_mtiles = 0)
{
    const int R = T * K;
    if (R <= kSmallRows) {
        const int steps = (R + kSmallWaves * AMOE_WAVE - 1) / (kSmallWaves * AMOE_WAVE);
        hipLaunchKernelGGL(permute_small_kernel, dim3(1), dim3(kSmallWaves * AMOE_WAVE), 0, s, assign, T, K, E, R, steps, scores,
                           PlanOut{counts, offsets, token_of, slot_of, row_of, scores_perm, tile_map, n_mtiles, bm, max_mtiles});
        return amoe_check_launch("permute_plan");
    }
    const int n_chunks = permute_chunks(R);
    const int n_blocks = (n_chunks + kWavesPerBlock - 1) / kWavesPerBlock;
    hipLaunchKernelGGL(permute_hist_kernel, dim3(n_blocks), dim3(kWavesPerBlock * AMOE_WAVE), 0, s, assign, T, K, E, R,
                       n_chunks, cc);
    int EP = 1;
    while (EP < E) EP <<= 1;
    hipLaunchKernelGGL(permute_scan_kernel, dim3(1), dim3(kScanThreads), 0, s, cc, E, EP, n_chunks, counts, offsets,
                       tile_map, n_mtiles, bm, max_mtiles);
    hipLaunchKernelGGL(permute_scatter_kernel, dim3(n_blocks), dim3(kWavesPerBlock * AMOE_WAVE), 0, s, assign, T, K, E,
                       R, n_chunks, cc, offsets, scores, token_of, slot_of, row_of, scores_perm);
    return amoe_check_launch("permute_plan");
}

AMOE_EXPORT int amoe_permute_plan(const int32_t* assign, const float* scores, int T, int K, int E, int32_t* counts,
                                  int32_t* offsets, int32_t* token_of, int32_t* slot_of, int32_t* row_of,
                                  float* scores_perm, void* workspace, size_t workspace_bytes, void* stream)
{
    int rc = check_plan_args(assign, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm);
    if (rc) return rc;
    AMOE_REQUIRE(workspace, AMOE_ERR_BAD_ARG, "permute_plan: null workspace");
    AMOE_REQUIRE(workspace_bytes >= amoe_permute_workspace_bytes(T * K, E), AMOE_ERR_WORKSPACE,
                 "permute_plan: workspace %zu < %zu bytes", workspace_bytes, amoe_permute_workspace_bytes(T * K, E));
    return launch_plan(assign, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm,
                       (int32_t*)workspace, (hipStream_t)stream);
}

// The plan together with the tile map of the row-grouped GEMMs that will run over its offsets: the
// scan kernel holds the offsets anyway, so the map costs no launch of its own.
int amoe_tile_map_layout(int R, int E, int dtype, int tile_cfg, void* workspace, size_t workspace_bytes, int4** tile_map,
                         int32_t** n_mtiles, int* bm, int* max_mtiles);

AMOE_EXPORT int amoe_permute_plan_tiled(const int32_t* assign, const float* scores, int T, int K, int E, int32_t* counts,
                                        int32_t* offsets, int32_t* token_of, int32_t* slot_of, int32_t* row_of,
                                        float* scores_perm, void* workspace, size_t workspace_bytes, void* gemm_workspace,
                                        size_t gemm_workspace_bytes, int dtype, int tile_cfg, void* stream)
{
    int rc = check_plan_args(assign, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm);
    if (rc) return rc;
    AMOE_REQUIRE(workspace && gemm_workspace, AMOE_ERR_BAD_ARG, "permute_plan_tiled: null workspace");
    AMOE_REQUIRE(workspace_bytes >= amoe_permute_workspace_bytes(T * K, E), AMOE_ERR_WORKSPACE,
                 "permute_plan_tiled: workspace %zu < %zu bytes", workspace_bytes, amoe_permute_workspace_bytes(T * K, E));
    int4* tile_map = nullptr;
    int32_t* n_mtiles = nullptr;
    int bm = 0, max_mtiles = 0;
    rc = amoe_tile_map_layout(T * K, E, dtype, tile_cfg, gemm_workspace, gemm_workspace_bytes, &tile_map, &n_mtiles, &bm,
                              &max_mtiles);
    if (rc) return rc;
    return launch_plan(assign, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm,
                       (int32_t*)workspace, (hipStream_t)stream, tile_map, n_mtiles, bm, max_mtiles);
}

// amoe_router_topk_fwd and amoe_permute_plan_tiled of its selection, in one launch where one block has a wavefront per token.
int amoe_launch_route(const void* logits, int logits_dtype, int T, int K, int E, int normalize, float* probs, int32_t* topk_idx,
                      float* scores, int32_t* counts, int32_t* offsets, int32_t* token_of, int32_t* slot_of, int32_t* row_of,
                      float* scores_perm, void* workspace, size_t workspace_bytes, void* gemm_workspace,
                      size_t gemm_workspace_bytes, int dtype, int tile_cfg, hipStream_t s)
{
    if (T > kSmallWaves || E > AMOE_MAX_EXPERTS || K > E || K > AMOE_MAX_TOPK) {
        const int rc = amoe_router_topk_fwd(logits, logits_dtype, T, E, K, normalize, probs, topk_idx, scores, s);
        if (rc) return rc;
        return amoe_permute_plan_tiled(topk_idx, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm, workspace,
                                       workspace_bytes, gemm_workspace, gemm_workspace_bytes, dtype, tile_cfg, s);
    }
    AMOE_REQUIRE(logits && probs, AMOE_ERR_BAD_ARG, "route: null pointer");
    AMOE_REQUIRE(logits_dtype == AMOE_F32 || logits_dtype == AMOE_BF16 || logits_dtype == AMOE_F16, AMOE_ERR_BAD_ARG,
                 "route: bad dtype %d", logits_dtype);
    int rc = check_plan_args(topk_idx, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm);
    if (rc) return rc;
    PlanOut o{counts, offsets, token_of, slot_of, row_of, scores_perm, nullptr, nullptr, 0, 0};
    rc = amoe_tile_map_layout(T * K, E, dtype, tile_cfg, gemm_workspace, gemm_workspace_bytes, &o.tile_map, &o.n_mtiles, &o.bm,
                              &o.max_mtiles);
    if (rc) return rc;
    ROUTER_DISPATCH_VPT(E, {
        AMOE_DISPATCH_ELEM(logits_dtype, hipLaunchKernelGGL((route_small_kernel<ELEM, VPT>), dim3(1), dim3(kSmallWaves * AMOE_WAVE), 0, s,
                                                            (const ELEM*)logits, T, E, K, normalize, probs, topk_idx, scores, o))
    })
    return amoe_check_launch("route");
}

// ------------------------------------------------------------------ the variant that allocates nothing
// The per-chunk counts live in a fixed array in device memory that belongs to the library (each
// GPU the library runs on holds its own copy until the process ends).  Host code never uses the
// array's name as an address: the device address is looked up once per device and kept.
static __device__ __align__(256) int32_t scratch[AMOE_PERMUTE_STATIC_MAX_COUNTS];

static constexpr int kMaxDevices = 64;
static std::atomic<int32_t*> g_scratch_ptr[kMaxDevices];

// device address of `scratch` on the current device (resolved on the first call per device)
static int static_scratch(int32_t** out)
{
    int dev = -1;
    hipError_t err = hipGetDevice(&dev);
    if (err != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        amoe_set_error("permute_plan_static: no usable current device (%s)", hipGetErrorString(err));
        return AMOE_ERR_LAUNCH;
    }
    int32_t* ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!ptr) {
        void* sym = nullptr;
        err = hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !sym) {
            amoe_set_error("permute_plan_static: cannot resolve the scratch array on device %d: %s", dev,
                           hipGetErrorString(err));
            return AMOE_ERR_LAUNCH;
        }
        ptr = (int32_t*)sym;
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);  // racing threads store the same address
    }
    *out = ptr;
    return AMOE_OK;
}

AMOE_EXPORT int amoe_permute_plan_static(const int32_t* assign, const float* scores, int T, int K, int E,
                                         int32_t* counts, int32_t* offsets, int32_t* token_of, int32_t* slot_of,
                                         int32_t* row_of, float* scores_perm, void* stream)
{
    int rc = check_plan_args(assign, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm);
    if (rc) return rc;
    const long long need = (long long)permute_chunks(T * K) * E;
    AMOE_REQUIRE(need <= (long long)AMOE_PERMUTE_STATIC_MAX_COUNTS, AMOE_ERR_UNSUPPORTED,
                 "permute_plan_static: ceil(T*K/%d)*E = %lld exceeds the built-in scratch of %d counters; "
                 "use amoe_permute_plan with a caller workspace",
                 kChunk, need, AMOE_PERMUTE_STATIC_MAX_COUNTS);
    int32_t* cc = nullptr;
    rc = static_scratch(&cc);
    if (rc) return rc;
    return launch_plan(assign, scores, T, K, E, counts, offsets, token_of, slot_of, row_of, scores_perm, cc,
                       (hipStream_t)stream);
}
