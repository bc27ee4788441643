// Grouped products as the layer's calls and the exported entry points share them.
#pragma once

#include "amoe_common.h"

// With room for the parts of a reduction (gemm_split.hip), none if split is null: amoe_split_bytes of the same rows, experts,
// reduction length K and columns N as the product has, or the call is refused.
int amoe_run_gateup_act_fwd(const void* xp, const int32_t* a_row_map, const void* w_gate_up, const int32_t* offsets, const float* row_scale,
                            void* gate_up, void* inter, int dtype, int R, int E, int H, int I, int act, void* workspace,
                            size_t workspace_bytes, int tile_cfg, void* stream, float* split, size_t split_bytes);
int amoe_run_nn(const void* A, const int32_t* a_row_map, const void* B, const int32_t* offsets, void* C, int dtype, int R, int E, int Kd,
                int N, void* workspace, size_t workspace_bytes, int tile_cfg, void* stream, float* split, size_t split_bytes);
int amoe_run_nt(const void* A, const int32_t* a_row_map, const void* B, const int32_t* offsets, void* C, int dtype, int R, int E, int Kd,
                int N, void* workspace, size_t workspace_bytes, int tile_cfg, void* stream, float* split, size_t split_bytes);
int amoe_run_nt_gated_bwd(const void* dy, const int32_t* a_row_map, const void* w_down, const int32_t* offsets, const void* gate_up,
                          const float* row_scale, void* d_gate_up, float* score_partials, int dtype, int R, int E, int I, int H, int act,
                          void* workspace, size_t workspace_bytes, int tile_cfg, void* stream, float* split, size_t split_bytes);
int amoe_split_count(int R, int E, int K, int N);
size_t amoe_split_bytes(int R, int E, int K, int N);

// weight gradients in 16 bits (gemm_bf16.hip)
int amoe_bf16_wgrad(const void* A, const int32_t* a_row_map, const void* B, const int32_t* b_row_map, const int32_t* offsets, void* C, int R,
                    int E, int Kd, int N, int tile_cfg, hipStream_t s, int dtype, int lda, bool out32);

// Routing of a few tokens inside the gate_up product: what it reads, and what it leaves for the other kernels (as
// amoe_router_topk_fwd and amoe_permute_plan_tiled do).
struct AmoeRoute {
    const void* logits;      // [T,E], of the product's type
    int T, K, normalize;
    float *probs, *scores, *scores_perm;
    int32_t *topk_idx, *counts, *offsets, *token_of, *slot_of, *row_of;
    int4* tile_map;
    int32_t* n_mtiles;
    int32_t* arrived;        // AmoeCombine's, which it sets to zero
    int n_arrived;
    int cus;                 // compute units of the device
};
// The sums over a token's K rows inside the down product: the workgroup of a column tile that is the last to arrive adds them up.
struct AmoeCombine {
    int32_t* arrived;        // workgroups of a column tile that have stored their rows, zero before
    const int32_t* row_of;   // [T,K]
    void* y;                 // [T,N]
    int T, K, cus;
};
// compute units of the device if it takes them (and then the product does, with every check of amoe_run_gateup_act_fwd on its sizes
// made), else 0
int amoe_routed_fits(int dtype, int T, int K, int E, int H, int I, int tile_cfg);
int amoe_run_gateup_routed(const void* x, const void* w_gate_up, void* gate_up, void* inter, const AmoeRoute& r, int dtype, int E, int H, int I,
                           int act, void* workspace, size_t workspace_bytes, hipStream_t s);
// out [T*K,H] = inter @ w_down[e] by the map that amoe_run_gateup_routed left, and y as above
int amoe_run_down_combined(const void* inter, const void* w_down, void* out, const AmoeCombine& c, int dtype, int E, int H, int I, void* workspace,
                           size_t workspace_bytes, hipStream_t s);
