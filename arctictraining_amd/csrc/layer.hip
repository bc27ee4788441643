// The expert layer's forward and backward as a few native calls.  A pass of a small layer is bound by the host: each
// stage called from Python costs an output allocation per tensor, argument checks, a crossing into the library and a
// crossing back, 10-15 us of host time against 2-10 us on the GPU.  Here the caller makes one buffer for what backward
// needs and one for what only this call needs, and the stages run over addresses cut from them.  The plain linear maps
// of the router stay with the caller, between the calls.
// (One token through 128 experts of 2048 x 768: 144 us of host time a forward stage by stage, 70 us this way.)
#include "amoe_common.h"
#include "gemm_calls.h"

#include <algorithm>
#include <mutex>
#include <vector>

int amoe_launch_route(const void* logits, int logits_dtype, int T, int K, int E, int normalize, float* probs, int32_t* topk_idx,
                      float* scores, int32_t* counts, int32_t* offsets, int32_t* token_of, int32_t* slot_of, int32_t* row_of,
                      float* scores_perm, void* workspace, size_t workspace_bytes, void* gemm_workspace,
                      size_t gemm_workspace_bytes, int dtype, int tile_cfg, hipStream_t s);
int amoe_launch_score_grad(const float* partials, int n_parts, const float* extra, const int32_t* row_of, float* d_scores,
                           int n_slots, bool accumulate, hipStream_t s);
int amoe_launch_shared_gate(const void* x, const void* w, float* sig, int dtype, int T, int H, hipStream_t s);
int amoe_launch_shared_gate_bwd(const float* d_sig, const float* sig, void* d_pre, int dtype, int T, hipStream_t s);
int amoe_launch_input_grad(const void* d_xp, const int32_t* row_of, const void* dense, const void* shared, const void* d_pre,
                           const void* gate, void* dx, int dtype, int T, int K, int H, hipStream_t s);
int amoe_launch_gated_act_bwd_rows(const void* gate_up, const void* d_inter, const float* row_scale, void* d_gate_up, float* d_scale,
                                   int dtype, int R, int I, int act, hipStream_t s);
int amoe_launch_router_bwd(const float* d_scores, const float* probs, const int32_t* topk_idx, const int32_t* counts, int dtype, int T,
                           int E, int K, int normalize, float lb_coeff, void* d_logits, int ld, hipStream_t s);
int amoe_launch_sum_parts(const void* parts, int n_parts, void* out, int parts_dtype, int dtype, long long n, hipStream_t s);

namespace {

struct Shape {
    int E, K, H, I, act, dtype, normalize, tile_cfg, shared;
    size_t esz() const { return dtype == AMOE_F32 ? 4 : 2; }
    bool fused_bwd() const { return dtype != AMOE_F32 && tile_cfg <= 2; }
};

struct Cut {
    uintptr_t base;
    size_t used = 0;
    template <typename T>
    T* take(size_t n)
    {
        T* p = reinterpret_cast<T*>(base + used);
        used += (n * sizeof(T) + 255) & ~(size_t)255;
        return p;
    }
};

// what backward reads
struct Saved {
    float *probs, *scores, *scores_perm, *sh_sig;
    int32_t *topk_idx, *counts, *offsets, *token_of, *slot_of, *row_of;
    char *gemm_ws, *sh_ws, *gate_up, *inter, *sh_gate_up, *sh_inter;
    size_t gemm_ws_bytes, sh_ws_bytes, bytes;
};

Saved cut_saved(const Shape& c, int T, void* base, bool keep)
{
    Saved s = {};
    Cut b{(uintptr_t)base};
    const size_t R = (size_t)T * c.K, E = c.E;
    s.probs = b.take<float>((size_t)T * E);
    s.scores = b.take<float>(R);
    s.scores_perm = b.take<float>(R);
    s.topk_idx = b.take<int32_t>(R);
    s.counts = b.take<int32_t>(E);
    s.offsets = b.take<int32_t>(E + 1);
    s.token_of = b.take<int32_t>(R);
    s.slot_of = b.take<int32_t>(R);
    s.row_of = b.take<int32_t>(R);
    s.gemm_ws_bytes = amoe_grouped_gemm_workspace_bytes((int)R, c.E);
    s.gemm_ws = b.take<char>(s.gemm_ws_bytes);
    s.inter = b.take<char>(R * c.I * c.esz());
    // float32 gate_up products store it whether backward reads it or not: rows that are worked out again are activated from it
    if (keep || c.dtype == AMOE_F32) s.gate_up = b.take<char>(R * 2 * c.I * c.esz());
    if (c.shared) {
        s.sh_sig = b.take<float>(T);
        s.sh_ws_bytes = amoe_grouped_gemm_workspace_bytes(T, 1);
        s.sh_ws = b.take<char>(s.sh_ws_bytes);
        s.sh_inter = b.take<char>((size_t)T * c.I * c.esz());
        if (keep || c.dtype == AMOE_F32) s.sh_gate_up = b.take<char>((size_t)T * 2 * c.I * c.esz());
    }
    s.bytes = b.used;
    return s;
}

// room for the parts of the products of `R` rows of `E` experts, K[i] x N[i]
size_t split_room(const Shape& c, int T, int K0, int N0, int K1, int N1)
{
    if (c.dtype == AMOE_F32 || c.tile_cfg != 0) return 0;
    const int R = T * c.K;
    size_t n = std::max(amoe_split_bytes(R, c.E, K0, N0), amoe_split_bytes(R, c.E, K1, N1));
    if (c.shared) n = std::max({n, amoe_split_bytes(T, 1, K0, N0), amoe_split_bytes(T, 1, K1, N1)});
    return n;
}

struct FwdScratch {
    char *plan_ws, *out, *sh_out;
    int32_t* arrived;
    float* split;
    size_t plan_ws_bytes, split_bytes, bytes;
};

FwdScratch cut_fwd(const Shape& c, int T, void* base)
{
    FwdScratch f = {};
    Cut b{(uintptr_t)base};
    const size_t R = (size_t)T * c.K;
    f.plan_ws_bytes = amoe_permute_workspace_bytes((int)R, c.E);
    f.plan_ws = b.take<char>(f.plan_ws_bytes);
    f.out = b.take<char>(R * c.H * c.esz());
    if (c.shared) f.sh_out = b.take<char>((size_t)T * c.H * c.esz());
    f.arrived = b.take<int32_t>((c.H + 63) / 64);
    f.split_bytes = split_room(c, T, c.H, 2 * c.I, c.I, c.H);
    if (f.split_bytes) f.split = (float*)b.take<char>(f.split_bytes);
    f.bytes = b.used;
    return f;
}

struct BwdScratch {
    float *parts, *d_scores, *sh_d_sig;
    char *d_gate_up, *d_rows /* d_inter, later d_xp */, *sh_d_gate_up, *sh_d_rows;
    float* split;
    size_t split_bytes, bytes;
};

BwdScratch cut_bwd(const Shape& c, int T, void* base)
{
    BwdScratch w = {};
    Cut b{(uintptr_t)base};
    const size_t R = (size_t)T * c.K, wide = c.I > c.H ? c.I : c.H;
    if (c.fused_bwd()) w.parts = b.take<float>((size_t)amoe_gated_bwd_score_parts(c.I, c.tile_cfg) * R);
    w.d_scores = b.take<float>(R);
    w.d_gate_up = b.take<char>(R * 2 * c.I * c.esz());
    w.d_rows = b.take<char>(R * (c.fused_bwd() ? c.H : wide) * c.esz());
    if (c.shared) {
        w.sh_d_sig = b.take<float>(T);
        w.sh_d_gate_up = b.take<char>((size_t)T * 2 * c.I * c.esz());
        w.sh_d_rows = b.take<char>((size_t)T * wide * c.esz());
    }
    w.split_bytes = split_room(c, T, c.H, c.I, 2 * c.I, c.H);
    if (w.split_bytes) w.split = (float*)b.take<char>(w.split_bytes);
    w.bytes = b.used;
    return w;
}

int read_shape(const char* what, const int32_t* config, int T, Shape* c)
{
    AMOE_REQUIRE(config, AMOE_ERR_BAD_ARG, "%s: null config", what);
    *c = {config[0], config[1], config[2], config[3], config[4], config[5], config[6], config[7], config[8]};
    AMOE_REQUIRE(T > 0 && c->E > 0 && c->K > 0 && c->H > 0 && c->I > 0, AMOE_ERR_BAD_ARG,
                 "%s: sizes must be positive (T=%d E=%d K=%d H=%d I=%d)", what, T, c->E, c->K, c->H, c->I);
    AMOE_REQUIRE(c->dtype == AMOE_F32 || c->dtype == AMOE_BF16 || c->dtype == AMOE_F16, AMOE_ERR_BAD_ARG, "%s: bad dtype %d", what,
                 c->dtype);
    AMOE_REQUIRE((long long)T * c->K < (1ll << 31), AMOE_ERR_UNSUPPORTED, "%s: T*K does not fit int32", what);
    return AMOE_OK;
}

// Events that order the second stream after the first and back.  A wait takes the event's state as it is when the wait is
// queued, so an event is free for its next use as soon as the call that queued both is over: the pool never holds more
// than the number of threads that were inside a backward at the same time.
class OrderEvent {
public:
    OrderEvent()
    {
        (void)hipGetDevice(&device_);
        std::lock_guard<std::mutex> lock(mutex());
        auto& free = pool();
        for (size_t i = 0; i < free.size(); ++i)
            if (free[i].device == device_) {
                event_ = free[i].event;
                free[i] = free.back();
                free.pop_back();
                return;
            }
        if (hipEventCreateWithFlags(&event_, hipEventDisableTiming) != hipSuccess) event_ = nullptr;
    }
    ~OrderEvent()
    {
        if (!event_) return;
        std::lock_guard<std::mutex> lock(mutex());
        if (pool().size() < kKept) pool().push_back({device_, event_});
        else (void)hipEventDestroy(event_);
    }
    // everything queued on `later` from here on runs after everything queued on `first` so far
    bool order(hipStream_t first, hipStream_t later)
    {
        return event_ && hipEventRecord(event_, first) == hipSuccess && hipStreamWaitEvent(later, event_, 0) == hipSuccess;
    }

private:
    static constexpr size_t kKept = 64;
    struct Entry {
        int device;
        hipEvent_t event;
    };
    static std::mutex& mutex()
    {
        static std::mutex m;
        return m;
    }
    static std::vector<Entry>& pool()
    {
        static std::vector<Entry>* p = new std::vector<Entry>;   // (never destroyed: the HIP runtime may be gone before it)
        return *p;
    }
    int device_ = 0;
    hipEvent_t event_ = nullptr;
};

}  // namespace

#define AMOE_TRY(expr)              \
    do {                            \
        const int rc_ = (expr);     \
        if (rc_ != AMOE_OK) return rc_; \
    } while (0)

AMOE_EXPORT int amoe_layer_sizes(const int32_t* config, int T, int keep, long long* out)
{
    Shape c;
    AMOE_TRY(read_shape("layer_sizes", config, T, &c));
    AMOE_REQUIRE(out, AMOE_ERR_BAD_ARG, "layer_sizes: null pointer");
    const Saved s = cut_saved(c, T, nullptr, keep != 0);
    const void* fields[] = {s.probs, s.scores, s.scores_perm, s.topk_idx, s.counts, s.offsets, s.token_of, s.slot_of, s.row_of};
    out[0] = (long long)s.bytes;
    out[1] = (long long)cut_fwd(c, T, nullptr).bytes;
    out[2] = (long long)cut_bwd(c, T, nullptr).bytes;
    for (int i = 0; i < 9; ++i) out[3 + i] = (long long)(uintptr_t)fields[i];
    out[12] = (long long)(uintptr_t)cut_bwd(c, T, nullptr).d_scores;
    return AMOE_OK;
}

AMOE_EXPORT int amoe_layer_fwd(const int32_t* config, int T, const void* x, const void* logits, int logits_dtype,
                               const int32_t* assign, const void* w_gate_up, const void* w_down, const void* sh_gate_up,
                               const void* sh_down, const void* sh_out_gate, const int32_t* all_rows, void* saved,
                               int keep, void* scratch, void* y, int stages, void* stream)
{
    Shape c;
    AMOE_TRY(read_shape("layer_fwd", config, T, &c));
    AMOE_REQUIRE(x && logits && w_gate_up && w_down && saved && scratch && y, AMOE_ERR_BAD_ARG, "layer_fwd: null pointer");
    AMOE_REQUIRE(!c.shared || (sh_gate_up && sh_down && sh_out_gate && all_rows), AMOE_ERR_BAD_ARG, "layer_fwd: null shared expert");
    const Saved s = cut_saved(c, T, saved, keep != 0);
    const FwdScratch f = cut_fwd(c, T, scratch);
    const int R = T * c.K, ready = c.tile_cfg | AMOE_TILE_MAP_READY;
    if (stages & AMOE_STAGE_ROUTE) {
        // the row-grouped products share one tile map: the plan builds it, backward uses it again
        if (assign) {
            AMOE_TRY(amoe_router_topk_fwd(logits, logits_dtype, T, c.E, c.K, c.normalize, s.probs, s.topk_idx, s.scores, stream));
            AMOE_TRY(amoe_permute_plan_tiled(assign, s.scores, T, c.K, c.E, s.counts, s.offsets, s.token_of, s.slot_of, s.row_of,
                                             s.scores_perm, f.plan_ws, f.plan_ws_bytes, s.gemm_ws, s.gemm_ws_bytes, c.dtype,
                                             c.tile_cfg, stream));
        } else {
            AMOE_TRY(amoe_launch_route(logits, logits_dtype, T, c.K, c.E, c.normalize, s.probs, s.topk_idx, s.scores, s.counts,
                                       s.offsets, s.token_of, s.slot_of, s.row_of, s.scores_perm, f.plan_ws, f.plan_ws_bytes,
                                       s.gemm_ws, s.gemm_ws_bytes, c.dtype, c.tile_cfg, (hipStream_t)stream));
        }
    }
    if (stages & AMOE_STAGE_EXPERTS) {
        // the rows x[token_of] are gathered inside the product's loads; a row's score multiplies its intermediate
        // activation (the down projection is linear), so that the combine is a plain sum
        AMOE_TRY(amoe_run_gateup_act_fwd(x, s.token_of, w_gate_up, s.offsets, s.scores_perm, s.gate_up, s.inter, c.dtype, R, c.E, c.H, c.I,
                                         c.act, s.gemm_ws, s.gemm_ws_bytes, ready, stream, f.split, f.split_bytes));
        AMOE_TRY(amoe_run_nn(s.inter, nullptr, w_down, s.offsets, f.out, c.dtype, R, c.E, c.I, c.H, s.gemm_ws, s.gemm_ws_bytes, ready, stream,
                             f.split, f.split_bytes));
    }
    if (c.shared && (stages & AMOE_STAGE_SHARED)) {
        // the shared expert is one more expert that owns every token, sigmoid(x @ gate) in the role of the score
        AMOE_TRY(amoe_launch_shared_gate(x, sh_out_gate, s.sh_sig, c.dtype, T, c.H, (hipStream_t)stream));
        AMOE_TRY(amoe_run_gateup_act_fwd(x, nullptr, sh_gate_up, all_rows, s.sh_sig, s.sh_gate_up, s.sh_inter, c.dtype, T, 1, c.H, c.I, c.act,
                                         s.sh_ws, s.sh_ws_bytes, c.tile_cfg, stream, f.split, f.split_bytes));
        AMOE_TRY(amoe_run_nn(s.sh_inter, nullptr, sh_down, all_rows, f.sh_out, c.dtype, T, 1, c.I, c.H, s.sh_ws, s.sh_ws_bytes, ready, stream,
                             f.split, f.split_bytes));
    }
    if (stages & AMOE_STAGE_COMBINE)
        AMOE_TRY(amoe_gather_rows_bwd(f.out, s.row_of, c.shared ? f.sh_out : nullptr, y, c.dtype, T, c.K, c.H, stream));
    return AMOE_OK;
}

// The forward pass that forms the logits [T,E] itself, of 16-bit x with rows of a multiple of 32.
AMOE_EXPORT int amoe_layer_fwd_router(const int32_t* config, int T, const void* x, const void* router_gate, void* logits,
                                      const int32_t* assign, const void* w_gate_up, const void* w_down, const void* sh_gate_up,
                                      const void* sh_down, const void* sh_out_gate, const int32_t* all_rows, void* saved, int keep,
                                      void* scratch, void* y, int stages, void* stream)
{
    Shape c;
    AMOE_TRY(read_shape("layer_fwd_router", config, T, &c));
    if (stages & AMOE_STAGE_ROUTE) AMOE_TRY(amoe_router_logits(x, router_gate, logits, c.dtype, T, c.E, c.H, stream));
    const int fused = AMOE_STAGE_ROUTE | AMOE_STAGE_EXPERTS;
    const int cus = !assign && (stages & fused) == fused ? amoe_routed_fits(c.dtype, T, c.K, c.E, c.H, c.I, c.tile_cfg) : 0;
    if (cus) {
        AMOE_REQUIRE(x && w_gate_up && w_down && saved && scratch && y, AMOE_ERR_BAD_ARG, "layer_fwd_router: null pointer");
        // (a few tokens: their routing inside the gate_up product)
        const Saved s = cut_saved(c, T, saved, keep != 0);
        const FwdScratch f = cut_fwd(c, T, scratch);
        const AmoeRoute route = {logits, T, c.K, c.normalize, s.probs, s.scores, s.scores_perm, s.topk_idx, s.counts, s.offsets, s.token_of,
                                 s.slot_of, s.row_of, nullptr, nullptr, f.arrived, (c.H + 63) / 64, cus};
        AMOE_TRY(amoe_run_gateup_routed(x, w_gate_up, s.gate_up, s.inter, route, c.dtype, c.E, c.H, c.I, c.act, s.gemm_ws, s.gemm_ws_bytes,
                                        (hipStream_t)stream));
        stages &= ~fused;
        if (!c.shared && (stages & AMOE_STAGE_COMBINE)) {
            const AmoeCombine combine = {f.arrived, s.row_of, y, T, c.K, cus};
            return amoe_run_down_combined(s.inter, w_down, f.out, combine, c.dtype, c.E, c.H, c.I, s.gemm_ws, s.gemm_ws_bytes, (hipStream_t)stream);
        }
        AMOE_TRY(amoe_run_nn(s.inter, nullptr, w_down, s.offsets, f.out, c.dtype, T * c.K, c.E, c.I, c.H, s.gemm_ws, s.gemm_ws_bytes,
                             c.tile_cfg | AMOE_TILE_MAP_READY, stream, f.split, f.split_bytes));
    }
    return amoe_layer_fwd(config, T, x, logits, c.dtype, assign, w_gate_up, w_down, sh_gate_up, sh_down, sh_out_gate, all_rows, saved,
                          keep, scratch, y, stages, stream);
}

static int layer_bwd(const int32_t* config, int T, const void* x, const void* dy, const void* w_down, const void* saved, void* scratch,
                     const float* d_scores_rows, float lb_coeff, void* d_w_gate_up, void* d_w_down, void* d_logits, int ld, void* stream,
                     void* side_stream)
{
    Shape c;
    AMOE_TRY(read_shape("layer_bwd", config, T, &c));
    AMOE_REQUIRE(x && dy && w_down && saved && scratch && d_logits, AMOE_ERR_BAD_ARG, "layer_bwd: null pointer");
    const Saved s = cut_saved(c, T, const_cast<void*>(saved), true);
    const BwdScratch w = cut_bwd(c, T, scratch);
    const int R = T * c.K, ready = c.tile_cfg | AMOE_TILE_MAP_READY;
    const hipStream_t main = (hipStream_t)stream, side = (hipStream_t)side_stream;
    const bool overlap = side_stream && side_stream != stream && (d_w_gate_up || d_w_down);
    // d(out)[r] = dy[token_of[r]]: the rows of dy are gathered inside the products' loads
    if (c.fused_bwd()) {
        // data gradient of the down projection with the backward of the gated activation as its epilogue; the score
        // gradients come back as sums over the columns of one tile each
        AMOE_TRY(amoe_run_nt_gated_bwd(dy, s.token_of, w_down, s.offsets, s.gate_up, s.scores_perm, w.d_gate_up, w.parts, c.dtype, R, c.E, c.I,
                                       c.H, c.act, s.gemm_ws, s.gemm_ws_bytes, ready, stream, w.split, w.split_bytes));
    } else {
        AMOE_TRY(amoe_grouped_gemm_nt(dy, s.token_of, w_down, s.offsets, w.d_rows, c.dtype, R, c.E, c.I, c.H, s.gemm_ws,
                                      s.gemm_ws_bytes, ready, stream));
        AMOE_TRY(amoe_gated_act_bwd(s.gate_up, w.d_rows, s.scores_perm, s.slot_of, w.d_gate_up, w.d_scores, c.dtype, R, c.I, T, c.K,
                                    c.act, stream));
    }
    // The expert weight gradients feed nothing else here.  On the second stream, and queued ahead of the rest, they start as the
    // gated backward's workgroups end; the kernels of this stream then run on what the weight gradients leave, which is little
    // before their workgroups end (from 129 rows an expert on these take two tiles each, from 704 on all that fall to them): with
    // 16384 tokens of 128 experts of 2048 x 768 the router's weight gradient and the sum of its parts last 422 and 759 us, of which
    // 24 and 5 are their own.  A step with the second stream / without, us: those 3700 / 3706, 8192 tokens of 8 experts of 4096 x 14336
    // 13560 / 13575, 4001 tokens of 64 experts and a shared one, float16, 1542 / 1581, 2048 tokens in float32 373 / 399, 128, 509, 1024,
    // 1600, 2000 and 2400 tokens of the first 690 / 697, 735 / 740, 798 / 799, 934 / 905, 1002 / 970, 984 / 990.
    OrderEvent event;
    if (overlap) AMOE_REQUIRE(event.order(main, side), AMOE_ERR_LAUNCH, "layer_bwd: cannot order the second stream after the first");
    void* const wstream = overlap ? side_stream : stream;
    // (the rows that are gathered are the T tokens')
    const auto gathered = [&](int width) {
        return c.tile_cfg | ((size_t)T * width * c.esz() < (1ull << 32) ? AMOE_SOURCE_BELOW_4GIB : 0);
    };
    if (d_w_down)
        AMOE_TRY(amoe_grouped_gemm_wgrad(s.inter, nullptr, dy, s.token_of, s.offsets, d_w_down, c.dtype, R, c.E, c.I, c.H,
                                         gathered(c.H), wstream));
    if (d_w_gate_up)
        AMOE_TRY(amoe_grouped_gemm_wgrad(x, s.token_of, w.d_gate_up, nullptr, s.offsets, d_w_gate_up, c.dtype, R, c.E, c.H, 2 * c.I,
                                         gathered(c.H), wstream));
    if (c.fused_bwd())
        AMOE_TRY(amoe_launch_score_grad(w.parts, amoe_gated_bwd_score_parts(c.I, c.tile_cfg), d_scores_rows, s.row_of, w.d_scores, R,
                                        false, main));
    else if (d_scores_rows)
        AMOE_TRY(amoe_launch_score_grad(nullptr, 0, d_scores_rows, s.row_of, w.d_scores, R, true, main));
    return amoe_launch_router_bwd(w.d_scores, s.probs, s.topk_idx, s.counts, c.dtype, T, c.E, c.K, c.normalize, lb_coeff, d_logits,
                                  ld ? ld : c.E, main);
}

AMOE_EXPORT int amoe_layer_bwd(const int32_t* config, int T, const void* x, const void* dy, const void* w_down, const void* saved,
                               void* scratch, const float* d_scores_rows, float lb_coeff, void* d_w_gate_up, void* d_w_down,
                               void* d_logits, void* stream, void* side_stream)
{
    return layer_bwd(config, T, x, dy, w_down, saved, scratch, d_scores_rows, lb_coeff, d_w_gate_up, d_w_down, d_logits, 0, stream,
                     side_stream);
}

// The same with rows of d_logits that are a multiple of 32 long, whatever E is (what is past E: zeros), so that the
// router's gradients run on kernels that read 8 or 32 elements at a time, and with the router's weight gradient [E,H] in
// the same call (see amoe_dense_wgrad for the chunks; the parts [splits][E][H] are float32).
AMOE_EXPORT int amoe_layer_bwd_router(const int32_t* config, int T, const void* x, const void* dy, const void* w_down, const void* saved,
                                      void* scratch, const float* d_scores_rows, float lb_coeff, void* d_w_gate_up, void* d_w_down,
                                      void* d_logits, const int32_t* chunk_offsets, int splits, void* parts, void* d_router_gate,
                                      void* stream, void* side_stream)
{
    Shape c;
    AMOE_TRY(read_shape("layer_bwd_router", config, T, &c));
    AMOE_REQUIRE(c.dtype != AMOE_F32, AMOE_ERR_UNSUPPORTED, "layer_bwd_router: bf16 and float16 only");
    AMOE_REQUIRE(c.H % 8 == 0, AMOE_ERR_UNSUPPORTED, "layer_bwd_router: H=%d must be a multiple of 8", c.H);
    const int ld = (c.E + 31) / 32 * 32;
    AMOE_TRY(layer_bwd(config, T, x, dy, w_down, saved, scratch, d_scores_rows, lb_coeff, d_w_gate_up, d_w_down, d_logits, ld, stream,
                       side_stream));
    if (!d_router_gate) return AMOE_OK;
    AMOE_REQUIRE(chunk_offsets && splits > 0 && (splits == 1 || parts), AMOE_ERR_BAD_ARG, "layer_bwd_router: null pointer");
    AMOE_TRY(amoe_bf16_wgrad(d_logits, nullptr, x, nullptr, chunk_offsets, splits > 1 ? parts : d_router_gate, T, splits, c.E, c.H, 1,
                             (hipStream_t)stream, c.dtype, ld, splits > 1));
    if (splits == 1) return AMOE_OK;
    return amoe_launch_sum_parts(parts, splits, d_router_gate, AMOE_F32, c.dtype, (long long)c.E * c.H, (hipStream_t)stream);
}

// C [Kd,N] = A [T,Kd]^T @ B [T,N], the weight gradient of a map that every token takes: few output tiles and a deep
// reduction, so the tokens are cut into `splits` chunks (chunk_offsets [splits+1]) that play the role of experts, and the
// partial products, in the operands' type, are added in float32.
AMOE_EXPORT int amoe_dense_wgrad(const void* A, const void* B, const int32_t* chunk_offsets, int splits, void* parts, void* C,
                                 int dtype, int T, int Kd, int N, int tile_cfg, void* stream)
{
    AMOE_REQUIRE(C && splits > 0 && (splits == 1 || parts), AMOE_ERR_BAD_ARG, "dense_wgrad: null pointer");
    AMOE_TRY(amoe_grouped_gemm_wgrad(A, nullptr, B, nullptr, chunk_offsets, splits > 1 ? parts : C, dtype, T, splits, Kd, N, tile_cfg,
                                     stream));
    if (splits == 1) return AMOE_OK;
    return amoe_launch_sum_parts(parts, splits, C, dtype, dtype, (long long)Kd * N, (hipStream_t)stream);
}

AMOE_EXPORT int amoe_layer_bwd_shared(const int32_t* config, int T, const void* x, const void* dy, const void* sh_down,
                                      const int32_t* all_rows, const void* saved, void* scratch, void* parts,
                                      const int32_t* gate_up_chunks, int gate_up_splits, void* d_sh_gate_up,
                                      const int32_t* down_chunks, int down_splits, void* d_sh_down, void* d_pre, void* stream)
{
    Shape c;
    AMOE_TRY(read_shape("layer_bwd_shared", config, T, &c));
    AMOE_REQUIRE(x && dy && sh_down && all_rows && saved && scratch && d_pre && c.shared, AMOE_ERR_BAD_ARG,
                 "layer_bwd_shared: null pointer");
    const Saved s = cut_saved(c, T, const_cast<void*>(saved), true);
    const BwdScratch w = cut_bwd(c, T, scratch);
    const hipStream_t main = (hipStream_t)stream;
    // the chain of amoe_layer_bwd for the expert that owns every token; its score gradient goes on through the sigmoid
    AMOE_TRY(amoe_run_nt(dy, nullptr, sh_down, all_rows, w.sh_d_rows, c.dtype, T, 1, c.I, c.H, s.sh_ws, s.sh_ws_bytes,
                         c.tile_cfg | AMOE_TILE_MAP_READY, stream, w.split, w.split_bytes));
    if (d_sh_down)
        AMOE_TRY(amoe_dense_wgrad(s.sh_inter, dy, down_chunks, down_splits, parts, d_sh_down, c.dtype, T, c.I, c.H, c.tile_cfg, stream));
    AMOE_TRY(amoe_launch_gated_act_bwd_rows(s.sh_gate_up, w.sh_d_rows, s.sh_sig, w.sh_d_gate_up, w.sh_d_sig, c.dtype, T, c.I, c.act, main));
    if (d_sh_gate_up)
        AMOE_TRY(amoe_dense_wgrad(x, w.sh_d_gate_up, gate_up_chunks, gate_up_splits, parts, d_sh_gate_up, c.dtype, T, c.H, 2 * c.I,
                                  c.tile_cfg, stream));
    return amoe_launch_shared_gate_bwd(w.sh_d_sig, s.sh_sig, d_pre, c.dtype, T, main);
}

AMOE_EXPORT int amoe_layer_bwd_input(const int32_t* config, int T, const void* w_gate_up, const void* sh_gate_up,
                                     const void* sh_out_gate, const int32_t* all_rows, const void* saved, void* scratch,
                                     const void* dx_router, const void* d_pre, void* dx, void* stream, void* side_stream)
{
    Shape c;
    AMOE_TRY(read_shape("layer_bwd_input", config, T, &c));
    AMOE_REQUIRE(saved && scratch, AMOE_ERR_BAD_ARG, "layer_bwd_input: null pointer");
    const Saved s = cut_saved(c, T, const_cast<void*>(saved), true);
    const BwdScratch w = cut_bwd(c, T, scratch);
    const int R = T * c.K, ready = c.tile_cfg | AMOE_TILE_MAP_READY;
    const hipStream_t main = (hipStream_t)stream;
    if (dx) {
        AMOE_REQUIRE(w_gate_up && dx_router, AMOE_ERR_BAD_ARG, "layer_bwd_input: null pointer");
        AMOE_REQUIRE(!c.shared || (sh_gate_up && sh_out_gate && all_rows && d_pre), AMOE_ERR_BAD_ARG,
                     "layer_bwd_input: null shared expert");
        AMOE_TRY(amoe_run_nt(w.d_gate_up, nullptr, w_gate_up, s.offsets, w.d_rows, c.dtype, R, c.E, c.H, 2 * c.I, s.gemm_ws, s.gemm_ws_bytes,
                             ready, stream, w.split, w.split_bytes));
        if (c.shared)
            AMOE_TRY(amoe_run_nt(w.sh_d_gate_up, nullptr, sh_gate_up, all_rows, w.sh_d_rows, c.dtype, T, 1, c.H, 2 * c.I, s.sh_ws,
                                 s.sh_ws_bytes, ready, stream, w.split, w.split_bytes));
        AMOE_TRY(amoe_launch_input_grad(w.d_rows, s.row_of, dx_router, c.shared ? w.sh_d_rows : nullptr, d_pre, sh_out_gate, dx,
                                        c.dtype, T, c.K, c.H, main));
    }
    if (side_stream && side_stream != stream) {
        OrderEvent event;   // the caller's next work sees the weight gradients
        AMOE_REQUIRE(event.order((hipStream_t)side_stream, main), AMOE_ERR_LAUNCH, "layer_bwd_input: cannot join the second stream");
    }
    return AMOE_OK;
}
