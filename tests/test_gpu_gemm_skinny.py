"""The row-grouped products where an expert has few rows: each tile height, its remainders, the narrow tiles of a
single token, matrix edges, and loads so uneven that one expert fills many tiles.  Reference: the per-expert
product in float32 of the 16-bit operands; the tolerance is a few roundings of the 16-bit result."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 1e-2, torch.float16: 2e-3}


def _counts(kind, E):
    if kind == "token":       # one token of four experts
        return [1 if e in (0, 3, 4, E - 1) else 0 for e in range(E)]
    if kind == "16":
        return [(e * 7) % 17 // 3 + (9 if e == 2 else 0) for e in range(E)]
    if kind == "32":
        return [(0, 1, 15, 0, 17, 0, 31, 0)[e % 8] for e in range(E)]
    if kind == "more":        # past the limit: the default tiles
        return [(33, 64, 65, 0, 63, 48, 1, 16)[e % 8] for e in range(E)]
    return [0] * (E - 1) + [6 * E - 1] if kind == "one" else [E * 4] + [0] * (E - 1)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kind", ["token", "16", "32", "more", "one", "first"])
@pytest.mark.parametrize("Kd,N", [(32, 8), (96, 136), (160, 520), (1024, 264)])
def test_few_rows(gpu_device, dtype, kind, Kd, N):
    from arctictraining_amd import ops

    print("skinny", dtype, kind, Kd, N, flush=True)
    E = 24
    counts = _counts(kind, E)
    R = sum(counts)
    low = {"token": 4, "16": 4, "32": 8, "one": 8, "first": 4}.get(kind)
    assert R <= low * E if low else R > 8 * E
    g = torch.Generator(device=gpu_device).manual_seed(Kd + N)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    src = torch.randn(max(R // 3, 1), Kd, device=gpu_device, generator=g).to(dtype)
    rows = torch.randint(0, src.shape[0], (R,), device=gpu_device, generator=g, dtype=torch.int32)
    w = (torch.randn(E, Kd, N, device=gpu_device, generator=g) * 0.05).to(dtype)
    w[E - 2] = float("nan") if counts[E - 2] == 0 else w[E - 2]   # an expert without rows is not read
    a = src[rows.long()]
    ref = torch.cat([p.float() @ w[e].float() for e, p in enumerate(a.split(counts)) if counts[e]])

    def check(got, want):
        assert torch.isfinite(got).all()
        norm = want.norm(dim=-1)
        err = (got.float() - want).norm(dim=-1) / torch.maximum(norm, norm.pow(2).mean().sqrt())
        assert float(err.max()) <= TOL[dtype], f"worst row {float(err.max()):.2e}"

    check(ops.grouped_gemm_nn(a, w, offs), ref)
    check(ops.grouped_gemm_nn(src, w, offs, a_row_map=rows), ref)
    # (the products with the transposed weights take the same tile map)
    check(ops.grouped_gemm_nt(src, w.transpose(1, 2).contiguous(), offs, a_row_map=rows), ref)
    scale = torch.rand(R, device=gpu_device)
    for act, fn in enumerate((torch.nn.functional.silu, torch.nn.functional.gelu, torch.relu, lambda v: v * torch.sigmoid(1.702 * v))):
        gu, inter = ops.grouped_gemm_gateup_act_fwd(src, w, offs, act, a_row_map=rows, row_scale=scale)
        check(gu, ref)
        check(inter, scale[:, None] * gu[:, 1::2].float() * fn(gu[:, 0::2].float()))
        only = ops.grouped_gemm_gateup_act_fwd(src, w, offs, act, a_row_map=rows, row_scale=scale, want_gate_up=False)
        assert only[0] is None and torch.equal(only[1], inter)


@pytest.mark.parametrize("plan_rows,call_rows", [(4, 8), (4, 40), (8, 4), (40, 4), (40, 8)])
def test_map_of_another_bound(gpu_device, plan_rows, call_rows):
    """A tile map built for one bound of the rows serves a product that states another one: the same expert offsets,
    the rows past the last expert's unused."""
    from arctictraining_amd import ops

    E, Kd, N = 24, 96, 264
    bound = [plan_rows * E, call_rows * E]
    counts = [(e * 5) % 8 if min(bound) > 4 * E else (e * 5) % 5 for e in range(E)]
    counts[3] += min(bound) - sum(counts)
    print("map of another bound", plan_rows, call_rows, counts, flush=True)
    assert min(counts) >= 0
    g = torch.Generator(device=gpu_device).manual_seed(plan_rows)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    x = torch.randn(max(bound), Kd, device=gpu_device, generator=g).bfloat16()
    w = (torch.randn(E, Kd, N, device=gpu_device, generator=g) * 0.05).bfloat16()
    ws = ops.gemm_workspace(max(bound), E, gpu_device)   # (a workspace of the larger call serves the smaller one)
    ops.grouped_gemm_nn(x[: bound[0]].contiguous(), w, offs, workspace=ws)
    a = x[: bound[1]].contiguous()
    n = sum(counts)
    ref = torch.cat([p.float() @ w[e].float() for e, p in enumerate(a[:n].split(counts))])
    for got in (
        ops.grouped_gemm_nn(a, w, offs, workspace=ws, map_ready=True)[:n],
        ops.grouped_gemm_nt(a, w.transpose(1, 2).contiguous(), offs, workspace=ws, map_ready=True)[:n],
        ops.grouped_gemm_gateup_act_fwd(a, w, offs, workspace=ws, map_ready=True)[0][:n],
    ):
        assert (got.float() - ref).norm() <= 1e-2 * ref.norm()
