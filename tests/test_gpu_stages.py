"""Stage-level parity of the HIP kernels (through the C ABI) against the CPU oracle.

Integer results (top-k indices, counts, offsets, the three index maps) must be bit-exact;
floating-point results are compared by relative L2 error against the oracle evaluated in
float64 from the same (already rounded) inputs: <= 1e-2 for bf16 data, <= 1e-5 for float32.
"""
import numpy as np
import pytest
import torch

from oracle import moe_oracle as O

pytestmark = pytest.mark.gpu

BF16_TOL = 1e-2
F32_TOL = 1e-5


@pytest.fixture(scope="module")
def ops(gpu_device):
    from arctictraining_amd import ops as _ops

    return _ops


def _pick(dtype, bf16_tol, f32_tol):
    """tolerance by element type; float16 carries 3 more mantissa bits than bf16, it gets a quarter of bf16's"""
    return {torch.bfloat16: bf16_tol, torch.float16: bf16_tol / 4}.get(dtype, f32_tol)


def _tol(dtype):
    return _pick(dtype, BF16_TOL, F32_TOL)


def _say(*a):
    print(*a, flush=True)


# ------------------------------------------------------------------ router
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("E,K", [(8, 2), (64, 4), (128, 8), (60, 6), (256, 8), (384, 1), (512, 16), (5, 5)])
@pytest.mark.parametrize("normalize", [True, False])
def test_router_topk(ops, gpu_device, dtype, E, K, normalize):
    _say("router_topk", dtype, E, K, normalize)
    g = torch.Generator().manual_seed(E * 131 + K)
    T = 777
    logits = (torch.randn(T, E, generator=g) * 0.9).to(dtype)
    # rows with forced ties, including across the k / k+1 boundary and an all-equal row
    logits[0] = 0.0
    logits[1, : E // 2] = 1.5
    logits[2, :5] = torch.tensor([0.25, -0.0, 0.0, 0.25, 0.5]).to(dtype)
    probs, idx, scores = ops.router_topk_fwd(logits.to(gpu_device), K, normalize)
    torch.cuda.synchronize()
    ref_p = O.softmax_probs(logits)
    _, ref_idx = O.topk_canonical(logits.to(torch.float64) + 0.0, K)
    assert torch.equal(idx.cpu().to(torch.int64), ref_idx), "top-k indices must be bit-exact"
    assert torch.allclose(probs.cpu(), ref_p, atol=2e-7, rtol=2e-6)
    ref_s = O.normalize_and_cast(torch.gather(ref_p, -1, ref_idx), normalize, dtype).float()
    got_s = scores.cpu()
    # the scores went through the model dtype: allow one unit in the last place of it
    ulp = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10}.get(dtype, 2.0 ** -21)
    assert torch.all((got_s - ref_s).abs() <= ulp * ref_s.abs() + 1e-9)
    if dtype != torch.float32:
        assert torch.equal(got_s, got_s.to(dtype).float()), "scores are representable in the model dtype"


def test_router_topk_matches_selection_on_probabilities(ops, gpu_device):
    """On configuration-shaped logits the selection on logits equals the reference's
    selection on float32 probabilities (with the lowest-index tie rule)."""
    x, wr, *_ = O.make_inputs(4096, 256, 128, 8, 8, torch.bfloat16, seed=12)
    logits = O.router_linear(x, wr)
    assert O.selection_agrees(logits, 8)
    _, idx, _ = ops.router_topk_fwd(logits.to(gpu_device), 8, True)
    _, ref = O.topk_canonical(O.softmax_probs(logits), 8)
    assert torch.equal(idx.cpu().long(), ref)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("E,K,normalize", [(8, 2, True), (128, 8, True), (64, 4, False), (300, 3, True)])
def test_router_bwd(ops, gpu_device, dtype, E, K, normalize):
    _say("router_bwd", dtype, E, K, normalize)
    g = torch.Generator().manual_seed(E + K)
    T = 333
    logits = (torch.randn(T, E, generator=g)).to(dtype)
    probs = O.softmax_probs(logits)
    _, idx = O.topk_canonical(logits.double(), K)
    d_scores = torch.randn(T, K, generator=g)
    counts = torch.randint(0, 50, (E,), generator=g, dtype=torch.int32)
    lb = 0.37 / T
    got = ops.router_bwd(
        d_scores.to(gpu_device), probs.to(gpu_device), idx.to(torch.int32).to(gpu_device), counts.to(gpu_device), dtype,
        normalize, lb,
    )
    p = probs.double()
    pt = torch.gather(p, -1, idx)
    ds = d_scores.double()
    if normalize:
        S = pt.sum(-1, keepdim=True)
        dpt = (ds - (ds * pt / S).sum(-1, keepdim=True)) / S
    else:
        dpt = ds
    dp = torch.zeros_like(p).scatter_add(-1, idx, dpt) + lb * counts.double()[None] / counts.sum()
    ref = p * (dp - (p * dp).sum(-1, keepdim=True))
    assert O.rel_l2(got.cpu(), ref) <= _pick(dtype, 4e-3, F32_TOL)


# ------------------------------------------------------------------ permutation
def _check_plan(ops, dev, assign, E):
    T, K = assign.shape
    g = torch.Generator().manual_seed(T * 7 + K)
    s_tk = torch.rand(T, K, generator=g)
    counts, offsets, token_of, slot_of, row_of, s_perm = ops.permute_plan(assign.to(torch.int32).to(dev), E, s_tk.to(dev))
    torch.cuda.synchronize()
    perm, tok, cnt = O.permutation(assign.long(), E)
    assert torch.equal(s_perm.cpu(), s_tk.t().reshape(-1)[perm]), "scores in row order (moe.py:379)"
    assert ops.permute_plan(assign.to(torch.int32).to(dev), E)[5] is None
    assert torch.equal(counts.cpu().long(), cnt), "counts"
    assert torch.equal(offsets.cpu().long(), torch.cat([torch.zeros(1, dtype=torch.int64), cnt.cumsum(0)])), "offsets"
    assert torch.equal(slot_of.cpu().long(), perm), "permutation order"
    assert torch.equal(token_of.cpu().long(), tok), "token ids"
    assert torch.equal(row_of.cpu().long(), O.inverse_row_map(perm, T, K)), "inverse map"


@pytest.mark.parametrize(
    "T,K,E",
    [(3, 2, 2), (1, 1, 1), (64, 1, 8), (1000, 2, 8), (1025, 4, 64), (4096, 8, 128), (777, 3, 300), (5000, 6, 512)],
)
def test_permute_plan_random(ops, gpu_device, T, K, E):
    _say("permute_plan", T, K, E)
    g = torch.Generator().manual_seed(T + K + E)
    assign = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)])
    _check_plan(ops, gpu_device, assign, E)


def test_permute_plan_worked_example(ops, gpu_device):
    assign = torch.tensor([[1, 0], [0, 1], [1, 0]])
    counts, offsets, token_of, slot_of, row_of, _ = ops.permute_plan(assign.to(torch.int32).to(gpu_device), 2)
    assert slot_of.tolist() == [1, 3, 5, 0, 2, 4]
    assert token_of.tolist() == [1, 0, 2, 0, 2, 1]
    assert counts.tolist() == [3, 3] and offsets.tolist() == [0, 3, 6]


def test_permute_plan_skewed_and_empty(ops, gpu_device):
    g = torch.Generator().manual_seed(3)
    T, K, E = 6000, 4, 64
    # 4 hot experts take about half, the last 8 experts receive nothing
    w = torch.ones(E)
    w[:4] = 13.0
    w[-8:] = 0.0
    assign = torch.multinomial(w.expand(T, E), K, replacement=False, generator=g)
    _check_plan(ops, gpu_device, assign, E)
    # everything to one expert per k
    assign = torch.tensor([[5, 9]]).expand(3000, 2).contiguous()
    _check_plan(ops, gpu_device, assign, 16)


def test_permute_plan_full_size_headline(ops, gpu_device):
    """T=16384, K=8, E=128 (the headline shape): bit-exact against the oracle."""
    g = torch.Generator().manual_seed(7)
    T, K, E = 16384, 8, 128
    assign = torch.multinomial(torch.ones(T, E), K, replacement=False, generator=g)
    _check_plan(ops, gpu_device, assign, E)


# ------------------------------------------------------------------ row kernels
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("T,K,H,E", [(50, 2, 64, 4), (300, 8, 2048, 16), (129, 4, 520, 8)])
def test_gather_and_combine(ops, gpu_device, dtype, T, K, H, E):
    _say("rows", dtype, T, K, H, E)
    g = torch.Generator().manual_seed(T + H)
    assign = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)])
    perm, tok, _ = O.permutation(assign, E)
    row_of = O.inverse_row_map(perm, T, K)
    R = T * K
    x = torch.randn(T, H, generator=g).to(dtype)
    d = gpu_device
    tok_d, row_d = tok.to(torch.int32).to(d), row_of.to(torch.int32).to(d)

    xp = ops.gather_rows_fwd(x.to(d), tok_d)
    assert torch.equal(xp.cpu(), x[tok]), "gather is a copy: bit-exact"

    d_xp = torch.randn(R, H, generator=g).to(dtype)
    addend = torch.randn(T, H, generator=g).to(dtype)
    dx = ops.gather_rows_bwd(d_xp.to(d), row_d, addend.to(d))
    ref = addend.double().index_add(0, tok, d_xp.double())
    assert O.rel_l2(dx.cpu(), ref) <= _tol(dtype)
    dx = ops.gather_rows_bwd(d_xp.to(d), row_d, None)
    ref = torch.zeros(T, H, dtype=torch.float64).index_add(0, tok, d_xp.double())
    assert O.rel_l2(dx.cpu(), ref) <= _tol(dtype)

    out = torch.randn(R, H, generator=g).to(dtype)
    s_tk = torch.rand(T, K, generator=g).to(dtype).float()
    s_perm = s_tk.t().reshape(-1)[perm]
    y = ops.combine_fwd(out.to(d), row_d, s_tk.to(d))
    ref = O.combine(out.double(), tok, s_perm.double(), K)
    assert O.rel_l2(y.cpu(), ref) <= _tol(dtype)
    y1 = ops.combine_fwd(out.to(d), row_d, None)
    assert O.rel_l2(y1.cpu(), O.combine(out.double(), tok, torch.ones(R, dtype=torch.float64), K)) <= _tol(dtype)

    dy = torch.randn(T, H, generator=g).to(dtype)
    d_out, d_s = ops.combine_bwd(dy.to(d), out.to(d), row_d, s_tk.to(d))
    ref_d_out = dy.double()[tok] * s_perm.double()[:, None]
    ref_ds_perm = (dy.double()[tok] * out.double()).sum(-1)
    ref_ds = torch.zeros(R, dtype=torch.float64)
    ref_ds[perm] = ref_ds_perm
    assert O.rel_l2(d_out.cpu(), ref_d_out) <= _tol(dtype)
    assert O.rel_l2(d_s.cpu(), ref_ds.view(K, T).t()) <= 1e-5
    _, d_s2 = ops.combine_bwd(dy.to(d), out.to(d), row_d, s_tk.to(d), need_d_out=False)
    assert torch.equal(d_s2, d_s)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("act", ["silu", "gelu", "relu", "gpt_oss"])
def test_gated_act_bwd(ops, gpu_device, dtype, act):
    code = {"silu": 0, "gelu": 1, "relu": 2, "gpt_oss": 3}[act]
    g = torch.Generator().manual_seed(4)
    R, I = 100, 96
    gu = torch.randn(R, 2 * I, generator=g).to(dtype)
    di = torch.randn(R, I, generator=g).to(dtype)
    got = ops.gated_act_bwd(gu.to(gpu_device), di.to(gpu_device), code)
    gu64 = gu.double().requires_grad_(True)
    inter = gu64[:, 1::2] * O.activation(act)(gu64[:, 0::2])
    inter.backward(di.double())
    assert O.rel_l2(got.cpu(), gu64.grad) <= _pick(dtype, 5e-3, 2e-5)
    # with the score folded in: inter = s_r * up * act(gate); also the score gradient per slot
    T, K = 25, 4
    assign = torch.stack([torch.randperm(8, generator=g)[:K] for _ in range(T)])
    perm, tok, _ = O.permutation(assign, 8)
    s_perm = torch.rand(R, generator=g) + 0.1
    got, d_s = ops.gated_act_bwd(
        gu.to(gpu_device), di.to(gpu_device), code, row_scale=s_perm.to(gpu_device),
        slot_of=perm.to(torch.int32).to(gpu_device), tk=(T, K),
    )
    gu64 = gu.double().requires_grad_(True)
    s64 = s_perm.double().requires_grad_(True)
    inter = s64[:, None] * gu64[:, 1::2] * O.activation(act)(gu64[:, 0::2])
    inter.backward(di.double())
    assert O.rel_l2(got.cpu(), gu64.grad) <= _pick(dtype, 5e-3, 2e-5)
    ref_ds = torch.zeros(R, dtype=torch.float64)
    ref_ds[perm] = s64.grad
    assert O.rel_l2(d_s.cpu(), ref_ds.view(K, T).t()) <= 2e-5


# ------------------------------------------------------------------ grouped GEMMs
def _ragged_counts(name, R, E, g):
    if name == "uniform":
        c = torch.full((E,), R // E)
        c[0] += R - int(c.sum())
    elif name == "ragged":
        w = torch.rand(E, generator=g) + 0.05
        c = torch.floor(w / w.sum() * R).long()
        c[-1] += R - int(c.sum())
    elif name == "holes":  # empty experts, one-row experts, one dominant expert
        c = torch.zeros(E, dtype=torch.long)
        c[1] = 1
        c[E // 2] = 3
        c[E - 2] = R - 4
    else:
        raise ValueError(name)
    assert int(c.sum()) == R and bool((c >= 0).all())
    return c


def _offsets(counts, dev):
    return torch.cat([torch.zeros(1, dtype=torch.int64), counts.cumsum(0)]).to(torch.int32).to(dev)


GEMM_CASES = [
    # dtype, R, E, Kd, N, counts, tile_cfg
    (torch.bfloat16, 512, 4, 64, 64, "uniform", 0),
    (torch.bfloat16, 200, 3, 32, 96, "ragged", 0),
    (torch.bfloat16, 900, 7, 96, 160, "holes", 2),
    (torch.bfloat16, 1000, 8, 128, 192, "ragged", 1),
    (torch.bfloat16, 1000, 8, 128, 192, "ragged", 2),
    (torch.bfloat16, 1000, 8, 128, 192, "ragged", 3),
    (torch.bfloat16, 1000, 8, 128, 192, "ragged", 5),
    (torch.bfloat16, 1500, 3, 448, 704, "ragged", 0),
    (torch.bfloat16, 2100, 9, 832, 256, "holes", 0),
    (torch.bfloat16, 3000, 5, 320, 576, "ragged", 0),
    (torch.bfloat16, 3000, 5, 320, 576, "holes", 5),
    (torch.bfloat16, 777, 6, 256, 320, "holes", 0),
    (torch.bfloat16, 2500, 16, 512, 384, "ragged", 0),
    (torch.bfloat16, 300, 3, 192, 1096, "ragged", 0),
    (torch.float16, 200, 3, 32, 96, "ragged", 0),
    (torch.float16, 1000, 8, 128, 192, "ragged", 1),
    (torch.float16, 1000, 8, 128, 192, "ragged", 2),
    (torch.float16, 1000, 8, 128, 192, "ragged", 3),
    (torch.float16, 1000, 8, 128, 192, "ragged", 5),
    (torch.float16, 2100, 9, 832, 256, "holes", 0),
    (torch.float16, 3000, 5, 320, 576, "ragged", 0),
    (torch.float32, 512, 4, 64, 64, "uniform", 0),
    (torch.float32, 777, 6, 100, 76, "holes", 0),
    (torch.float32, 1000, 8, 128, 192, "ragged", 0),
]


@pytest.mark.parametrize("dtype,R,E,Kd,N,cname,cfg", GEMM_CASES)
def test_grouped_gemm_nn_nt_wgrad(ops, gpu_device, dtype, R, E, Kd, N, cname, cfg):
    _say("gemm", dtype, R, E, Kd, N, cname, cfg)
    g = torch.Generator().manual_seed(R + E + Kd + N)
    counts = _ragged_counts(cname, R, E, g)
    cs = counts.cumsum(0)
    offs = _offsets(counts, gpu_device)
    A = torch.randn(R, Kd, generator=g).to(dtype)
    B = (torch.randn(E, Kd, N, generator=g) * 0.1).to(dtype)
    d = gpu_device
    tol = _pick(dtype, 4e-3, F32_TOL)
    # float16 with tile_cfg 3 exists for the weight gradient only: the row-grouped products reject it
    rows_ok = not (dtype == torch.float16 and cfg == 3)
    if not rows_ok:
        with pytest.raises(RuntimeError, match="float16"):
            ops.grouped_gemm_nn(A.to(d), B.to(d), offs, tile_cfg=cfg)
        with pytest.raises(RuntimeError, match="float16"):
            ops.grouped_gemm_nt(torch.randn(R, N).to(dtype).to(d), B.to(d), offs, tile_cfg=cfg)

    # NN: C = A @ B[e]
    C = ops.grouped_gemm_nn(A.to(d), B.to(d), offs, tile_cfg=cfg if rows_ok else 0)
    ref = O.grouped_gemm(A.double(), B.double(), cs)
    assert O.rel_l2(C.cpu(), ref) <= tol, "nn"

    # NN with the row gather folded in
    if dtype == torch.bfloat16 or True:
        Tn = max(R // 2, 1)
        src = torch.randn(Tn, Kd, generator=g).to(dtype)
        rmap = torch.randint(0, Tn, (R,), generator=g)
        C2 = ops.grouped_gemm_nn(src.to(d), B.to(d), offs, a_row_map=rmap.to(torch.int32).to(d), tile_cfg=cfg if rows_ok else 0)
        ref2 = O.grouped_gemm(src.double()[rmap], B.double(), cs)
        assert O.rel_l2(C2.cpu(), ref2) <= tol, "nn + row map"

    # NT: D = G @ B[e]^T
    G = torch.randn(R, N, generator=g).to(dtype)
    if dtype == torch.float32 or (N % 32 == 0 and Kd % 8 == 0):
        D = ops.grouped_gemm_nt(G.to(d), B.to(d), offs, tile_cfg=cfg if rows_ok else 0)
        refD = O.grouped_gemm(G.double(), B.double().transpose(1, 2).contiguous(), cs)
        assert O.rel_l2(D.cpu(), refD) <= tol, "nt"

    # wgrad: W[e] = A_e^T @ G_e, zeros for empty experts
    W = ops.grouped_gemm_wgrad(A.to(d), G.to(d), offs, E, tile_cfg=cfg)
    refW = torch.zeros(E, Kd, N, dtype=torch.float64)
    start = 0
    for e in range(E):
        end = int(cs[e])
        refW[e] = A.double()[start:end].t() @ G.double()[start:end]
        start = end
    assert O.rel_l2(W.cpu(), refW) <= tol, "wgrad"
    for e in range(E):
        if int(counts[e]) == 0:
            assert bool((W[e] == 0).all()), "empty expert must produce exact zeros"
    # weight gradient with one operand gathered through a row map inside the kernel
    Tn = max(R // 2, 1)
    rmap = torch.randint(0, Tn, (R,), generator=g)
    rmap_d = rmap.to(torch.int32).to(d)
    srcA = torch.randn(Tn, Kd, generator=g).to(dtype)
    Wa = ops.grouped_gemm_wgrad(srcA.to(d), G.to(d), offs, E, tile_cfg=cfg, a_row_map=rmap_d)
    srcB = torch.randn(Tn, N, generator=g).to(dtype)
    Wb = ops.grouped_gemm_wgrad(A.to(d), srcB.to(d), offs, E, tile_cfg=cfg, b_row_map=rmap_d)
    refA = torch.zeros(E, Kd, N, dtype=torch.float64)
    refB = torch.zeros(E, Kd, N, dtype=torch.float64)
    start = 0
    for e in range(E):
        end = int(cs[e])
        refA[e] = srcA.double()[rmap[start:end]].t() @ G.double()[start:end]
        refB[e] = A.double()[start:end].t() @ srcB.double()[rmap[start:end]]
        start = end
    assert O.rel_l2(Wa.cpu(), refA) <= tol, "wgrad + A row map"
    assert O.rel_l2(Wb.cpu(), refB) <= tol, "wgrad + B row map"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 5])
@pytest.mark.parametrize("act", ["silu", "gpt_oss"])
def test_gateup_activation_fused(ops, gpu_device, dtype, cfg, act):
    _say("gateup", dtype, cfg, act)
    code = {"silu": 0, "gelu": 1, "relu": 2, "gpt_oss": 3}[act]
    g = torch.Generator().manual_seed(17)
    R, E, H, I = 900, 5, 128, 96
    counts = _ragged_counts("ragged", R, E, g)
    offs = _offsets(counts, gpu_device)
    xp = torch.randn(R, H, generator=g).to(dtype)
    w = (torch.randn(E, H, 2 * I, generator=g) * 0.1).to(dtype)
    if dtype == torch.float16 and cfg == 3:
        # four waves of 256 accumulators leave the float16 conversions of this epilogue no registers: not built
        with pytest.raises(RuntimeError, match="float16"):
            ops.grouped_gemm_gateup_act_fwd(xp.to(gpu_device), w.to(gpu_device), offs, code, tile_cfg=cfg)
        return
    gu, inter = ops.grouped_gemm_gateup_act_fwd(xp.to(gpu_device), w.to(gpu_device), offs, code, tile_cfg=cfg)
    ref_gu = O.grouped_gemm(xp.double(), w.double(), counts.cumsum(0))
    tol = _pick(dtype, 4e-3, F32_TOL)
    assert O.rel_l2(gu.cpu(), ref_gu) <= tol
    ref_inter = ref_gu[:, 1::2] * O.activation(act)(ref_gu[:, 0::2])
    assert O.rel_l2(inter.cpu(), ref_inter) <= _pick(dtype, BF16_TOL, 2e-5)
    # inter is exactly the activation of the stored (rounded) gate_up
    gu_s = gu.cpu().double()
    chk = gu_s[:, 1::2] * O.activation(act)(gu_s[:, 0::2])
    assert O.rel_l2(inter.cpu(), chk) <= _pick(dtype, 4e-3, 2e-6)
    if dtype != torch.float32:
        _, inter2 = ops.grouped_gemm_gateup_act_fwd(
            xp.to(gpu_device), w.to(gpu_device), offs, code, tile_cfg=cfg, want_gate_up=False
        )
        assert torch.equal(inter2, inter)
    # row scale folded into the epilogue
    rs = torch.rand(R, generator=g) + 0.25
    gu3, inter3 = ops.grouped_gemm_gateup_act_fwd(
        xp.to(gpu_device), w.to(gpu_device), offs, code, tile_cfg=cfg, row_scale=rs.to(gpu_device)
    )
    assert torch.equal(gu3, gu)
    assert O.rel_l2(inter3.cpu(), ref_inter * rs.double()[:, None]) <= _pick(dtype, BF16_TOL, 2e-5)


@pytest.mark.parametrize("el", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("cfg", [0, 1, 2])
@pytest.mark.parametrize("act", ["silu", "gpt_oss", "gelu"])
def test_dgrad_down_with_gated_activation_backward(ops, gpu_device, cfg, act, el):
    """The data gradient of the down projection with the gated-activation backward as its epilogue
    (autograd of moe.py:187-192 and of the score multiply of moe.py:460): d_gate_up and the score
    gradients against float64 autograd over the same rounded inputs, and against the two-kernel
    path it replaces."""
    _say("dgrad_down+gated_bwd", cfg, act, el)
    tol = _pick(el, 5e-3, 0.0)
    code = {"silu": 0, "gelu": 1, "relu": 2, "gpt_oss": 3}[act]
    g = torch.Generator().manual_seed(23)
    T, K, E, H, I = 230, 4, 6, 128, 352          # I: two N tiles of 256 (the second ragged), or three of 128
    R = T * K
    assign = torch.stack([torch.randperm(E, generator=g)[:K] for _ in range(T)])
    assign[assign == 2] = 3                       # an empty expert
    perm, tok, counts = O.permutation(assign, E)
    offs = _offsets(counts, gpu_device)
    row_of = O.inverse_row_map(perm, T, K).to(torch.int32).to(gpu_device)
    bf = el
    dy = torch.randn(T, H, generator=g).to(bf)
    wd = (torch.randn(E, I, H, generator=g) * 0.1).to(bf)
    gu = torch.randn(R, 2 * I, generator=g).to(bf)
    s_perm = torch.rand(R, generator=g) + 0.1
    d = gpu_device
    d_gu, parts = ops.grouped_gemm_nt_gated_bwd(dy.to(d), wd.to(d), offs, gu.to(d), code, row_scale=s_perm.to(d),
                                                a_row_map=tok.to(torch.int32).to(d), n_rows=R, tile_cfg=cfg)
    d_s = ops.score_grad_gather(parts, row_of)
    torch.cuda.synchronize()
    # float64 autograd of inter_s = s * up * act(gate), out = inter_s @ W_down[e], loss = <dy[tok], out>
    gu64 = gu.double().requires_grad_(True)
    s64 = s_perm.double().requires_grad_(True)
    inter = s64[:, None] * gu64[:, 1::2] * O.activation(act)(gu64[:, 0::2])
    out = O.grouped_gemm(inter, wd.double(), counts.cumsum(0))
    (out * dy.double()[tok]).sum().backward()
    assert O.rel_l2(d_gu.cpu(), gu64.grad) <= tol, "d_gate_up"
    ref_ds = torch.zeros(R, dtype=torch.float64)
    ref_ds[perm] = s64.grad
    assert O.rel_l2(d_s.cpu(), ref_ds.view(K, T).t()) <= tol, "score gradients"
    # the two kernels it replaces (they round d_inter to the model dtype in between)
    d_inter = ops.grouped_gemm_nt(dy.to(d), wd.to(d), offs, a_row_map=tok.to(torch.int32).to(d), n_rows=R, tile_cfg=cfg)
    d_gu2, d_s2 = ops.gated_act_bwd(gu.to(d), d_inter, code, row_scale=s_perm.to(d),
                                    slot_of=perm.to(torch.int32).to(d), tk=(T, K))
    assert O.rel_l2(d_gu.cpu(), d_gu2.cpu().double()) <= tol
    assert O.rel_l2(d_s.cpu(), d_s2.cpu().double()) <= tol
    # without the partials, and without a row scale
    d_gu3, none = ops.grouped_gemm_nt_gated_bwd(dy.to(d), wd.to(d), offs, gu.to(d), code, row_scale=s_perm.to(d),
                                                a_row_map=tok.to(torch.int32).to(d), n_rows=R, tile_cfg=cfg,
                                                want_score_parts=False)
    assert none is None and torch.equal(d_gu3, d_gu)
    d_gu4, _ = ops.grouped_gemm_nt_gated_bwd(dy.to(d)[tok.to(d)].contiguous(), wd.to(d), offs, gu.to(d), code, tile_cfg=cfg)
    gu64b = gu.double().requires_grad_(True)
    inter = gu64b[:, 1::2] * O.activation(act)(gu64b[:, 0::2])
    (O.grouped_gemm(inter, wd.double(), counts.cumsum(0)) * dy.double()[tok]).sum().backward()
    assert O.rel_l2(d_gu4.cpu(), gu64b.grad) <= tol
    with pytest.raises(RuntimeError, match="tile_cfg 3"):
        ops.grouped_gemm_nt_gated_bwd(dy.to(d), wd.to(d), offs, gu.to(d), code, a_row_map=tok.to(torch.int32).to(d),
                                      n_rows=R, tile_cfg=3)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cfg", [0, 1, 3, 5])
def test_grouped_gemm_every_sliver_height(ops, gpu_device, dtype, cfg):
    """An expert's last tile may hold any number of live rows; a wavefront only works on its 32-row
    blocks that hold some (one copy of the K loop per count).  Experts whose row counts leave every
    remainder class around the block boundaries, through the plain, the transposed-weight, the fused
    gate_up and the fused gated-backward products."""
    _say("sliver heights", dtype, cfg)
    if dtype == torch.float16 and cfg == 3:
        pytest.skip("float16 with tile_cfg 3 exists for the weight gradient only")
    g = torch.Generator().manual_seed(77)
    rems = [1, 31, 32, 33, 63, 64, 65, 96, 97, 127, 128, 129, 160, 161, 191, 192, 193, 224, 255, 256, 0, 300]
    counts = torch.tensor(rems)
    E, R = len(rems), int(counts.sum())
    cs = counts.cumsum(0)
    offs = _offsets(counts, gpu_device)
    H, I = 64, 160
    d = gpu_device
    tol = _pick(dtype, 4e-3, F32_TOL)
    A = torch.randn(R, H, generator=g).to(dtype)
    W = (torch.randn(E, H, 2 * I, generator=g) * 0.1).to(dtype)
    C = ops.grouped_gemm_nn(A.to(d), W.to(d), offs, tile_cfg=cfg)
    ref = O.grouped_gemm(A.double(), W.double(), cs)
    assert O.rel_l2(C.cpu(), ref) <= tol, "nn"
    # per expert as well: a wrong sliver would drown in the whole-matrix norm
    start = 0
    for e in range(E):
        end = int(cs[e])
        if end > start:
            assert O.rel_l2(C[start:end].cpu(), ref[start:end]) <= 2 * tol, f"nn, expert {e} with {end - start} rows"
        start = end
    G = torch.randn(R, 2 * I, generator=g).to(dtype)
    D = ops.grouped_gemm_nt(G.to(d), W.to(d), offs, tile_cfg=cfg)
    refD = O.grouped_gemm(G.double(), W.double().transpose(1, 2).contiguous(), cs)
    start = 0
    for e in range(E):
        end = int(cs[e])
        if end > start:
            assert O.rel_l2(D[start:end].cpu(), refD[start:end]) <= 2 * tol, f"nt, expert {e} with {end - start} rows"
        start = end
    if not (dtype == torch.float16 and cfg == 3):
        rs = torch.rand(R, generator=g) + 0.25
        gu, inter = ops.grouped_gemm_gateup_act_fwd(A.to(d), W.to(d), offs, 0, tile_cfg=cfg, row_scale=rs.to(d))
        assert O.rel_l2(gu.cpu(), ref) <= tol
        ref_inter = ref[:, 1::2] * O.activation("silu")(ref[:, 0::2]) * rs.double()[:, None]
        assert O.rel_l2(inter.cpu(), ref_inter) <= _pick(dtype, BF16_TOL, 2e-5)
    if cfg in (0, 1):
        Wd = (torch.randn(E, I, H, generator=g) * 0.1).to(dtype)
        dy = torch.randn(R, H, generator=g).to(dtype)
        gu_in = torch.randn(R, 2 * I, generator=g).to(dtype)
        s_perm = torch.rand(R, generator=g) + 0.1
        d_gu, parts = ops.grouped_gemm_nt_gated_bwd(dy.to(d), Wd.to(d), offs, gu_in.to(d), 0, row_scale=s_perm.to(d), tile_cfg=cfg)
        gu64 = gu_in.double().requires_grad_(True)
        s64 = s_perm.double().requires_grad_(True)
        inter64 = s64[:, None] * gu64[:, 1::2] * O.activation("silu")(gu64[:, 0::2])
        (O.grouped_gemm(inter64, Wd.double(), cs) * dy.double()).sum().backward()
        assert O.rel_l2(d_gu.cpu(), gu64.grad) <= _pick(dtype, 5e-3, 0.0)
        assert O.rel_l2(parts.sum(0).cpu(), s64.grad) <= _pick(dtype, 5e-3, 0.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cfg", [0, 1, 3, 5])
def test_weight_gradient_every_edge_class(ops, gpu_device, dtype, cfg):
    """The weight gradient's live-block dispatch: output rows (Kd) that end in every remainder class of a
    32-row block in the last row tile, output columns (N) that leave waves of the last column tile without
    work, experts with ragged and empty row ranges.  Per expert, so that one wrong edge tile cannot hide
    in the norm of the whole gradient."""
    _say("wgrad edges", dtype, cfg)
    g = torch.Generator().manual_seed(123)
    counts = torch.tensor([1, 31, 64, 0, 97, 300, 33])
    E, R = len(counts), int(counts.sum())
    cs = counts.cumsum(0)
    offs = _offsets(counts, gpu_device)
    d = gpu_device
    tol = _pick(dtype, 4e-3, F32_TOL)
    for Kd, N in ((32, 72), (96, 104), (160, 200), (288, 328)):
        A = torch.randn(R, Kd, generator=g).to(dtype)
        G = torch.randn(R, N, generator=g).to(dtype)
        W = ops.grouped_gemm_wgrad(A.to(d), G.to(d), offs, E, tile_cfg=cfg).cpu()
        start = 0
        for e in range(E):
            end = int(cs[e])
            if end == start:
                assert bool((W[e] == 0).all()), f"Kd={Kd} N={N}: expert {e} has no rows"
            else:
                ref = A[start:end].double().t() @ G[start:end].double()
                assert O.rel_l2(W[e], ref) <= 2 * tol, f"Kd={Kd} N={N}: expert {e} with {end - start} rows"
            start = end


def test_grouped_gemm_rows_outside_groups_untouched(ops, gpu_device):
    """Rows past offsets[E] are never written (the tile map covers only routed rows)."""
    g = torch.Generator().manual_seed(5)
    R, E, Kd, N = 640, 4, 64, 128
    counts = torch.tensor([100, 0, 250, 90])  # 440 of 640 rows in use
    offs = _offsets(counts, gpu_device)
    A = torch.randn(R, Kd, generator=g).to(torch.bfloat16).to(gpu_device)
    B = torch.randn(E, Kd, N, generator=g).to(torch.bfloat16).to(gpu_device)
    lib_ops = ops
    C = lib_ops.grouped_gemm_nn(A, B, offs)
    ref = O.grouped_gemm(A.cpu().double()[:440], B.cpu().double(), counts.cumsum(0))
    assert O.rel_l2(C[:440].cpu(), ref) <= 4e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32, torch.float16])
def test_grouped_gemm_shared_tile_map(ops, gpu_device, dtype):
    """Row-grouped GEMMs over the same offsets may share one workspace: calls after the first pass
    map_ready (AMOE_TILE_MAP_READY) and reuse the tile map it holds; results are unchanged."""
    g = torch.Generator().manual_seed(9)
    R, E, Kd, N = 1500, 6, 96, 160
    counts = torch.tensor([300, 0, 517, 255, 1, 427])
    offs = _offsets(counts, gpu_device)
    A = torch.randn(R, Kd, generator=g).to(dtype).to(gpu_device)
    A2 = torch.randn(R, N, generator=g).to(dtype).to(gpu_device)
    B = (torch.randn(E, Kd, N, generator=g) * 0.1).to(dtype).to(gpu_device)
    ws = ops.gemm_workspace(R, E, gpu_device)
    c_first = ops.grouped_gemm_nn(A, B, offs, workspace=ws)                      # builds the map
    c_again = ops.grouped_gemm_nn(A, B, offs, workspace=ws, map_ready=True)      # reuses it
    d_again = ops.grouped_gemm_nt(A2, B, offs, workspace=ws, map_ready=True)
    assert torch.equal(c_first, ops.grouped_gemm_nn(A, B, offs))
    assert torch.equal(c_again, c_first)
    assert torch.equal(d_again, ops.grouped_gemm_nt(A2, B, offs))
    with pytest.raises(RuntimeError, match="workspace"):
        ops.grouped_gemm_nn(A, B, offs, map_ready=True)


@pytest.mark.parametrize("dtype,cfg", [(torch.bfloat16, 0), (torch.bfloat16, 1), (torch.float32, 0), (torch.float16, 0)])
def test_permute_plan_builds_the_gemm_tile_map(ops, gpu_device, dtype, cfg):
    """The plan can build the row-grouped GEMMs' tile map as a by-product of its scan kernel: a GEMM
    that reuses it (map_ready) gives exactly the result of one that builds its own, with empty
    experts, one-row experts and experts of several tiles; the plan's own outputs are unchanged."""
    g = torch.Generator().manual_seed(31)
    T, K, E, Kd, N = 1700, 3, 9, 96, 160
    assign = torch.randint(0, E, (T, K), generator=g)
    assign[assign == 4] = 5            # expert 4 empty
    assign[assign == 7] = 0
    assign[0, 0] = 7                   # expert 7 holds one row
    a32 = assign.to(torch.int32).to(gpu_device)
    R = T * K
    ws = ops.gemm_workspace(R, E, gpu_device)
    ws.fill_(0xAB)                     # stale bytes must not survive
    plain = ops.permute_plan(a32, E)
    tiled = ops.permute_plan(a32, E, gemm_workspace=ws, gemm_dtype=dtype, tile_cfg=cfg)
    for a, b in zip(plain[:5], tiled[:5]):
        assert torch.equal(a, b)
    offs = tiled[1]
    assert int(tiled[0][4]) == 0 and int(tiled[0][7]) == 1
    A = torch.randn(R, Kd, generator=g).to(dtype).to(gpu_device)
    B = (torch.randn(E, Kd, N, generator=g) * 0.1).to(dtype).to(gpu_device)
    assert torch.equal(ops.grouped_gemm_nn(A, B, offs, tile_cfg=cfg, workspace=ws, map_ready=True),
                       ops.grouped_gemm_nn(A, B, offs, tile_cfg=cfg))
    A2 = torch.randn(R, N, generator=g).to(dtype).to(gpu_device)
    assert torch.equal(ops.grouped_gemm_nt(A2, B, offs, tile_cfg=cfg, workspace=ws, map_ready=True),
                       ops.grouped_gemm_nt(A2, B, offs, tile_cfg=cfg))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("copies", [1, 40])
def test_gelu_of_the_epilogues(gpu_device, dtype, copies):
    """gelu and its derivative over the range where they are not 0 or g, the lower tail included, through products that
    hand the epilogues g itself.  One rounding of the result (of 8 or 11 significant bits: 2^-8, 2^-11 of it at most)
    and 1e-5 of the tail's value."""
    from arctictraining_amd import ops

    print("gelu epilogues", dtype, copies, flush=True)
    g = torch.linspace(-6 if dtype == torch.bfloat16 else -3, 12, 2048).to(dtype)
    H, I, R = 32, 64, 32
    w = torch.zeros(1, H, 2 * I, dtype=dtype)
    w[0, 1, 1::2] = 1.0                       # up = 1
    wd = torch.zeros(1, I, H, dtype=dtype)
    wd[0, :, 0] = 1.0                         # d_inter = 1
    for part in g.view(-1, R):
        x = torch.zeros(R, H, dtype=dtype)
        x[:, 0], x[:, 1] = part, 1.0
        x = x.repeat(copies, 1).to(gpu_device)
        w[0, 0, 0::2] = 1.0                   # gate = the row's value
        off = torch.tensor([0, R * copies], dtype=torch.int32, device=gpu_device)
        gu, inter = ops.grouped_gemm_gateup_act_fwd(x, w.to(gpu_device), off, ops.ACT_GELU)
        dy = torch.zeros(R * copies, H, dtype=dtype, device=gpu_device)
        dy[:, 0] = 1.0
        dg, _ = ops.grouped_gemm_nt_gated_bwd(dy, wd.to(gpu_device), off, gu, ops.ACT_GELU)
        v = part.double().repeat(copies).view(-1, 1)
        phi = torch.special.ndtr(v)
        ref = v * phi
        eps = 2.0 ** (-8 if dtype == torch.bfloat16 else -11) + 1e-5
        tiny = 1e-7 if dtype == torch.float16 else 0.0   # (float16 below its normal range)
        assert ((inter.cpu().double() - ref).abs() <= eps * ref.abs() + tiny).all()
        d = phi + v * torch.exp(-v * v / 2) * 0.3989422804014327
        got = dg.cpu().double()
        assert ((got[:, 0::2] - d).abs() <= eps * d.abs() + 1e-6).all()
        assert ((got[:, 1::2] - ref).abs() <= eps * ref.abs() + tiny).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("cfg", [0, 1])
def test_gelu_is_no_further_off_than_with_erff(gpu_device, dtype, cfg):
    """Every 16-bit gate up to 8, in float32: with one column of d_inter and of up that is not zero, a score partial is
    gelu of that column's gate.  0.5 (1 + erff(z)), of roundings of half a place of 1 + erff and of erff and of z, is off by
    up to 6.1e-8; the product with the gate is rounded once more."""
    from arctictraining_amd import ops

    print("gelu against erff", dtype, cfg, flush=True)
    v = torch.arange(-(1 << 15), 1 << 15, dtype=torch.int32).to(torch.int16).view(dtype)
    v = v[v.float().abs() <= 8]
    R, H, I = v.numel(), 32, 64
    gu = torch.zeros(R, 2 * I, dtype=dtype)
    gu[:, 0], gu[:, 1] = v, 1.0
    wd = torch.zeros(1, I, H, dtype=dtype)
    wd[0, 0, 0] = 1.0
    dy = torch.zeros(R, H, dtype=dtype)
    dy[:, 0] = 1.0
    off = torch.tensor([0, R], dtype=torch.int32, device=gpu_device)
    _, parts = ops.grouped_gemm_nt_gated_bwd(dy.to(gpu_device), wd.to(gpu_device), off, gu.to(gpu_device), ops.ACT_GELU, tile_cfg=cfg)
    got, ref = parts.sum(0).cpu().double(), v.double() * torch.special.ndtr(v.double())
    assert ((got - ref).abs() <= 6.1e-8 * v.double().abs() + 2.0**-24 * ref.abs() + 2.0**-126).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("copies,cfg", [(1, 0), (40, 0), (40, 1)])
def test_gelu_of_gates_without_end(gpu_device, dtype, copies, cfg):
    """Gates that are infinite (by overflow: each sum of two terms), the largest that there are, NaN, and where the
    exponential ends: as 0.5 g (1 + erff(g / sqrt 2)) and its derivative have them."""
    from arctictraining_amd import ops

    print("gelu without end", dtype, copies, cfg, flush=True)
    top = torch.finfo(dtype).max
    pairs = torch.tensor([(top, top), (-top, -top), (top, 0), (-top, 0), (14, 0), (-14, 0), (40, 0), (-40, 0), (0, 0), (-0.0, 0)])
    x = torch.zeros(len(pairs), 32, dtype=dtype)
    x[:, 0], x[:, 1], x[:, 2] = pairs[:, 0].to(dtype), pairs[:, 1].to(dtype), 1.0
    w = torch.zeros(1, 32, 128, dtype=dtype)
    w[0, :2, 0::2] = 1.0
    w[0, 2, 1::2] = 1.0
    x = x.repeat(copies, 1).to(gpu_device)
    off = torch.tensor([0, x.shape[0]], dtype=torch.int32, device=gpu_device)
    gu, inter = ops.grouped_gemm_gateup_act_fwd(x, w.to(gpu_device), off, ops.ACT_GELU, tile_cfg=cfg)
    g = gu[:, 0].cpu().float()
    assert g.isinf().sum() == 2 * copies

    def same(got, ref):
        got, ref = got.cpu().float(), ref.to(dtype).float()
        assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
        ok = ref.isfinite()
        # (a tail that 1 + erff has lost is not 0 here: below 1e-40 it is in neither type)
        assert ((got - ref)[ok].abs() <= 2.0**-7 * ref[ok].abs() + 1e-40).all() and torch.equal(got[ref.isinf()], ref[ref.isinf()])

    def former(g):
        phi = 0.5 * (1.0 + torch.erf(g * 0.7071067811865476))
        return g * phi, phi + g * (0.3989422804014327 * torch.exp(-0.5 * g * g))

    for col in (0, 63):
        same(inter[:, col], former(g)[0])
    gu[3, 0::2] = float("nan")
    g = gu[:, 0].cpu().float()
    wd = torch.zeros(1, 64, 32, dtype=dtype)
    wd[0, :, 0] = 1.0
    dy = torch.zeros(x.shape[0], 32, dtype=dtype, device=gpu_device)
    dy[:, 0] = 1.0
    dg, _ = ops.grouped_gemm_nt_gated_bwd(dy, wd.to(gpu_device), off, gu, ops.ACT_GELU, tile_cfg=cfg)
    f, df = former(g)
    same(dg[:, 0], df)
    same(dg[:, 127], f)
