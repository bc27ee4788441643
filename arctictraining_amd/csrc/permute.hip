// Deterministic token-to-expert permutation plan: a stable counting sort of the k-major
// flattened assignment vector, in one launch up to 65536 rows and otherwise in three launches
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
constexpr int kWavesPerBlock = 1;   // independent chunks per block (a compute unit takes a cycle for every scattered element it stores)

constexpr int kSteps = kChunk / AMOE_WAVE;

// place of flat slot f in the [T,K] arrays; the token is `t`
__device__ __forceinline__ int place_of(int f, int T, int K, int& t)
{
    const int k = f / T;
    t = f - k * T;
    return t * K + k;
}
__device__ __forceinline__ int load_expert(const int32_t* assign, int place, int E)
{
    return min(max(assign[place], 0), E - 1);  // memory safety for caller-supplied assignments
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
        int e[kSteps];
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            const int f = c * kChunk + i * 64 + lane;
            int t;
            e[i] = f < R ? load_expert(assign, place_of(f, T, K, t), E) : -1;
        }
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
            if (e[i] >= 0) atomicAdd(&cnt[w][e[i]], 1);
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
// thread holds its slice of counts in registers (kScanBatch at a time; one batch from pass to pass):
// the exclusive bases overwrite the counts in place, and loads issued after such a store cannot
// be moved ahead of it, which would turn the second pass into a chain of dependent round trips.
// When tile_map is non-null the block also writes the row-grouped GEMMs' tile map (one int4
// {expert, first row, end row, 0} per `bm`-row tile, {-1,0,0,0} past the last) and its tile count.
constexpr int kScanThreads = 1024;
constexpr int kScanBatch = 32;

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
    int sum = 0, v[kScanBatch];
    if (e < E)
        for (int cb = c0; cb < c1; cb += kScanBatch) {
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
            if (per > kScanBatch) {
#pragma unroll
                for (int i = 0; i < kScanBatch; ++i) v[i] = cb + i < c1 ? chunk_counts[(size_t)(cb + i) * E + e] : 0;
            }
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
    // (all that a chunk reads is requested before the chain of its steps, and a block is one wavefront: 131072 rows 13.6 -> 9.8 us)
    int ex[kSteps], tok[kSteps], at[kSteps];
    float sc[kSteps];
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
        const int f = c * kChunk + i * 64 + lane;
        ex[i] = -1;
        sc[i] = 0.f;
        if (f < R) {
            at[i] = place_of(f, T, K, tok[i]);
            ex[i] = load_expert(assign, at[i], E);
            if (scores_perm) sc[i] = scores[at[i]];
        }
    }
    for (int e = lane; e < E; e += 64) run[w][e] = offsets[e] + chunk_base[(size_t)c * E + e];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
        const bool valid = ex[i] >= 0;
        const int e = valid ? ex[i] : 0;
        bool last;
        const int rank = rank_of(e, valid, lane, &last);
        int row = 0;
        if (valid) row = run[w][e] + rank;
        __builtin_amdgcn_wave_barrier();
        // the highest lane of each group advances the running counter
        if (last) run[w][e] = row + 1;
        __builtin_amdgcn_wave_barrier();
        if (valid) {
            token_of[row] = tok[i];
            slot_of[row] = c * kChunk + i * 64 + lane;
            row_of[at[i]] = row;
            if (scores_perm) scores_perm[row] = sc[i];
        }
    }
}

// The whole plan in one launch, for up to kOneLaunchRows routed rows: the three kernels above are 5-8 us each there, most
// of it their launches and the chain of memory round trips between them.  A block of sixteen wavefronts owns 1024 consecutive
// slots, one to a thread, and counts ALL slots by itself, told apart as before its own, its own by wavefront, and after them:
// that gives every wavefront the bases of its rows without a word between blocks.  (The slots are counted in the order in which
// they are stored, 16 bytes a lane.)  Up to 8192 rows one block did all of it before, a store of a scattered element a cycle.
// Launches back to back, us, before / so: 512 rows of 128 experts 5.1 / 4.3, 4072 14.5 / 7.3, 8000 24.9 / 7.7, 24008 18.6 / 10.3,
// 65536 20.0 / 16.3, all of them to 8 experts 18.9 / 15.6, 4096 rows of 8 experts 9.5 / 6.3; with 131072 rows, which each of 128
// blocks would count, 27 / 30.
constexpr int kSmallWaves = 16;
constexpr int kSmallRows = kSmallWaves * AMOE_WAVE;
constexpr int kOneLaunchRows = 1 << 16;
// Lanes add to one of 8 copies of the counters, in banks of their own: where all slots go to one expert they would else wait for
// each other (65536 slots 59 us, so 15).
constexpr int kCopies = 8, kCopyStride = AMOE_MAX_EXPERTS + 1;

struct PlanOut {
    int32_t *counts, *offsets, *token_of, *slot_of, *row_of;
    float* scores_perm;
    int4* tile_map;
    int32_t* n_mtiles;
    int bm, max_mtiles;
};

// count_others(before, after): adds the slots that are not this block's.  e, tok, at, score: this thread's slot, its expert
// (-1: none), token, place t K + k and score
template <typename CountOthers>
__device__ __forceinline__ void plan_in_block(CountOthers count_others, int e, int slot, int tok, int at, float score, int E, const PlanOut& o)
{
    __shared__ int32_t run[kSmallWaves][AMOE_MAX_EXPERTS];
    __shared__ int32_t before[kCopies * kCopyStride], after[kCopies * kCopyStride];
    __shared__ int32_t tot[AMOE_MAX_EXPERTS + 1];
    __shared__ int32_t tstart[AMOE_MAX_EXPERTS + 1];
    const int t = threadIdx.x, w = t >> 6, lane = t & 63;
    const bool valid = e >= 0, first = blockIdx.x == 0, alone = gridDim.x == 1;
    for (int i = lane; i < E; i += AMOE_WAVE) run[w][i] = 0;
    if (!alone)
        for (int i = t; i < kCopies * kCopyStride; i += kSmallRows) before[i] = after[i] = 0;
    __syncthreads();
    if (valid) atomicAdd(&run[w][e], 1);
    if (!alone) count_others(before, after);
    __syncthreads();
    if (t < AMOE_MAX_EXPERTS) {
        int sum = 0;
        if (t < E) {
            // counts of the wavefronts -> exclusive bases inside the expert
            int rest = 0;
            if (!alone) {
#pragma unroll
                for (int c = 0; c < kCopies; ++c) {
                    sum += before[c * kCopyStride + t];
                    rest += after[c * kCopyStride + t];
                }
            }
#pragma unroll
            for (int c = 0; c < kSmallWaves; ++c) {
                const int v = run[c][t];
                run[c][t] = sum;
                sum += v;
            }
            sum += rest;
            if (first) o.counts[t] = sum;
        }
        tot[t] = sum;
    }
    __syncthreads();
    if (t < AMOE_WAVE) scan_row_counts(tot, t);
    __syncthreads();
    if (first) {
        if (t < E) o.offsets[t + 1] = tot[t];
        if (t == 0) o.offsets[0] = 0;
    }
    bool last;
    const int rank = rank_of(valid ? e : 0, valid, lane, &last);
    if (valid) {
        const int row = run[w][e] + rank + (e ? tot[e - 1] : 0);
        o.token_of[row] = tok;
        o.slot_of[row] = slot;
        o.row_of[at] = row;
        if (o.scores_perm) o.scores_perm[row] = score;
    }
    if (first && o.tile_map) amoe_emit_tile_map<kSmallWaves * AMOE_WAVE>(tot, 0, E, o.bm, o.tile_map, o.n_mtiles, o.max_mtiles, tstart);
}

// inv_k: 2^32 / K rounded up (0 for K = 1); VEC: assign lies on 16 bytes
template <bool VEC>
__global__ void __launch_bounds__(kSmallWaves * AMOE_WAVE)
permute_small_kernel(const int32_t* __restrict__ assign, int T, int K, uint32_t inv_k, int E, int R, const float* __restrict__ scores, PlanOut o)
{
    const int lo = blockIdx.x * kSmallRows, hi = lo + kSmallRows, slot = lo + threadIdx.x;
    int e = -1, tok = 0, at = 0;
    float score = 0.f;
    if (slot < R) {
        at = place_of(slot, T, K, tok);
        e = load_expert(assign, at, E);
        if (o.scores_perm) score = scores[at];
    }
    auto count_others = [&](int32_t* before, int32_t* after) {
        const int copy = threadIdx.x % kCopies * kCopyStride;
        auto count = [&](int place, int expert) {
            const int token = inv_k ? (int)(((uint64_t)(uint32_t)place * inv_k) >> 32) : place;
            const int f = (place - token * K) * T + token;
            if (f < lo || f >= hi) atomicAdd((f < lo ? before : after) + copy + min(max(expert, 0), E - 1), 1);
        };
        constexpr int W = VEC ? 4 : 1, BATCH = VEC ? 4 : 8;
        typedef int32_t vec_t __attribute__((ext_vector_type(W)));
        for (int p0 = threadIdx.x * W; p0 < R; p0 += kSmallRows * W * BATCH) {
            int32_t v[BATCH][W];
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
                const int p = p0 + i * kSmallRows * W;
                if (p + W <= R) {
                    const vec_t q = *reinterpret_cast<const vec_t*>(assign + p);
#pragma unroll
                    for (int j = 0; j < W; ++j) v[i][j] = q[j];
                } else {
#pragma unroll
                    for (int j = 0; j < W; ++j) v[i][j] = p + j < R ? assign[p + j] : 0;
                }
            }
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
#pragma unroll
                for (int j = 0; j < W; ++j)
                    if (p0 + i * kSmallRows * W + j < R) count(p0 + i * kSmallRows * W + j, v[i][j]);
        }
    };
    plan_in_block(count_others, e, slot, tok, at, score, E, o);
}

// Softmax, top-k and the plan of at most one token per wavefront of the block: the selection reaches the plan through LDS.
// (One token through 128 experts of 2048 x 768, the whole forward: 41 us with two launches, 37 with this one.)
template <typename T, int VPT>
__global__ void __launch_bounds__(kSmallWaves * AMOE_WAVE)
route_small_kernel(const T* __restrict__ logits, int n_tokens, int E, int K, int normalize, float* __restrict__ probs,
                   int32_t* __restrict__ topk_idx, float* __restrict__ scores, PlanOut o)
{
    __shared__ int32_t sel[kSmallWaves * AMOE_MAX_TOPK];    // [token][K]
    __shared__ float sc[kSmallWaves * AMOE_MAX_TOPK];
    const int lane = threadIdx.x & 63, t = threadIdx.x >> 6;
    if (t < n_tokens) {
        int e;
        float s;
        router_topk_token<T, VPT>(logits + (size_t)t * E, E, K, normalize, lane, probs + (size_t)t * E, e, s);
        if (lane < K) {
            topk_idx[(size_t)t * K + lane] = e;
            scores[(size_t)t * K + lane] = s;
            sel[t * K + lane] = min(max(e, 0), E - 1);
            sc[t * K + lane] = s;
        }
    }
    __syncthreads();
    const int slot = threadIdx.x;
    int tok = 0, at = 0;
    const bool valid = slot < n_tokens * K;        // (16 tokens of 16 at most)
    if (valid) at = place_of(slot, n_tokens, K, tok);
    plan_in_block([](int32_t*, int32_t*) {}, valid ? sel[at] : -1, slot, tok, at, valid ? sc[at] : 0.f, E, o);
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
    if (R <= kOneLaunchRows) {
        const dim3 grid((R + kSmallRows - 1) / kSmallRows), block(kSmallRows);
        const uint32_t inv_k = K > 1 ? (uint32_t)(((1ull << 32) + K - 1) / K) : 0u;      // (exact: R K < 2^32)
        const PlanOut o{counts, offsets, token_of, slot_of, row_of, scores_perm, tile_map, n_mtiles, bm, max_mtiles};
        if (((uintptr_t)assign & 15) == 0) hipLaunchKernelGGL(permute_small_kernel<true>, grid, block, 0, s, assign, T, K, inv_k, E, R, scores, o);
        else hipLaunchKernelGGL(permute_small_kernel<false>, grid, block, 0, s, assign, T, K, inv_k, E, R, scores, o);
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
