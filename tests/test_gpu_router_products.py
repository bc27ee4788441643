"""The router's products for few tokens against float64, at the edges of their tiles, and the layer on both sides of
the rule that chooses them.  Tolerance: one rounding of the 16-bit result (2^-9 and 2^-12 of the value) and the order of
the float32 sums."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 4e-3, torch.float16: 5e-4}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 33, 256, 300, 511, 513])
@pytest.mark.parametrize("E,H", [(1, 32), (8, 544), (60, 1024), (128, 2048), (32, 4096), (512, 96)])
def test_products(gpu_device, dtype, T, E, H):
    from arctictraining_amd import moe, ops

    print("router products", dtype, T, E, H, flush=True)
    g = torch.Generator(gpu_device).manual_seed(T + E + H)
    x = torch.randn(T, H, device=gpu_device, generator=g).to(dtype)
    w = (torch.randn(E, H, device=gpu_device, generator=g) * 0.02).to(dtype)
    dl = torch.randn(T, E, device=gpu_device, generator=g).to(dtype)

    def check(got, ref):
        assert got.dtype == dtype and (got.double() - ref).norm() <= TOL[dtype] * ref.norm()

    check(ops.router_logits(x, w), x.double() @ w.double().t())
    if E % 32 == 0:
        check(ops.router_input_grad(dl, w), dl.double() @ w.double())
    check(moe._router_weight_grad(dl, x), dl.double().t() @ x.double())


def test_refused(gpu_device):
    from arctictraining_amd import moe, ops

    x = torch.randn(4, 40, device=gpu_device).bfloat16()
    w = torch.randn(8, 40, device=gpu_device).bfloat16()
    with pytest.raises(RuntimeError):
        ops.router_logits(x, w)
    with pytest.raises(RuntimeError):
        ops.router_input_grad(torch.randn(4, 8, device=gpu_device).bfloat16(), w)
    assert moe._router_logits(x, w).shape == (4, 8)   # (the library takes it)
    odd = torch.randn(8 * 64 + 1, device=gpu_device).bfloat16()[1:].view(8, 64)   # two bytes off
    x = torch.randn(4, 64, device=gpu_device).bfloat16()
    assert not moe._router_kernel_fits(x, odd)
    ref = x.double() @ odd.double().t()
    assert (moe._router_logits(x, odd).double() - ref).norm() <= 4e-3 * ref.norm()
    with torch.autocast("cuda", dtype=torch.float16):
        assert moe._router_logits(x, odd.clone()).dtype == torch.float16
    with pytest.raises(RuntimeError):
        moe._router_logits(x, odd.float())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("E,K", [(5, 1), (64, 8), (65, 16), (128, 8), (300, 3), (512, 16)])
@pytest.mark.parametrize("T", [1, 5, 16, 17])
def test_route_in_one_launch(gpu_device, dtype, E, K, T):
    """The layer's routing of a few tokens equals the stages on their own (whole numbers exactly)."""
    from arctictraining_amd import ArcticMoE, MoEConfig, ops

    if K > E:
        pytest.skip("top_k above the number of experts")
    print("route", dtype, E, K, T, flush=True)
    torch.manual_seed(E + T)
    with gpu_device:
        layer = ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=dtype, intermediate_dim=32, model_dim=32, normalize_topk_scores=T % 2 == 0,
                                    num_experts=E, top_k=K))
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.1)
        layer.capture = got = {}
        layer(torch.randn(T, 32, device=gpu_device).to(dtype))
        probs, idx, scores = ops.router_topk_fwd(got["logits"], K, T % 2 == 0)
        counts, offsets, token_of, slot_of, row_of, _ = ops.permute_plan(idx, E, scores)
    for name, want in dict(probs=probs, topk_idx=idx, scores=scores, counts=counts, offsets=offsets, token_of=token_of, slot_of=slot_of,
                           row_of=row_of).items():
        assert torch.equal(got[name], want), name
