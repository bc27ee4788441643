"""The layer as native calls: its own small kernels at their edges, and forward alone against forward for backward."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,Kd,N,splits", [(5, 8, 16, 1), (300, 40, 264, 3), (4096, 256, 8, 16)])
def test_dense_weight_gradient(gpu_device, dtype, T, Kd, N, splits):
    from arctictraining_amd import moe, ops

    print("dense_wgrad", dtype, T, Kd, N, splits, flush=True)
    g = torch.Generator(gpu_device).manual_seed(T + N)
    a = torch.randn(T, Kd, device=gpu_device, generator=g).to(dtype)
    b = torch.randn(T, N, device=gpu_device, generator=g).to(dtype)
    got = ops.dense_wgrad(a, b, moe._token_offsets(T, splits, gpu_device))
    ref = a.double().t() @ b.double()
    tol = {torch.bfloat16: 1e-2, torch.float16: 2e-3, torch.float32: 1e-5}[dtype]
    assert (got.double() - ref).norm() <= tol * ref.norm()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,H", [(1, 8), (63, 520), (65, 512), (4096, 2048), (4097, 1032), (9556, 320)])
def test_gradient_of_one_column(gpu_device, dtype, T, H):
    """One rounding of the result (2^-9, 2^-12, 2^-24 of the value) and the order of float32 sums."""
    from arctictraining_amd import ops

    print("column_grad", dtype, T, H, flush=True)
    g = torch.Generator(gpu_device).manual_seed(T + H)
    x = torch.randn(T, H, device=gpu_device, generator=g).to(dtype)
    coef = torch.randn(T, 1, device=gpu_device, generator=g).to(dtype)
    got = ops.column_grad(x, coef)
    ref = x.double().t() @ coef.double()
    assert got.shape == (H, 1) and got.dtype == dtype
    assert (got.double() - ref).norm() <= {torch.bfloat16: 4e-3, torch.float16: 5e-4, torch.float32: 2e-6}[dtype] * ref.norm()
    with pytest.raises(RuntimeError):
        ops.column_grad(x, coef[:0])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("T", [1, 7, 260])
def test_forward_alone_equals_forward_for_backward(gpu_device, dtype, shared, T):
    from arctictraining_amd import ArcticMoE, MoEConfig

    print("layer", dtype, shared, T, flush=True)
    torch.manual_seed(T)
    cfg = MoEConfig(act_fn=F.silu, input_dtype=dtype, intermediate_dim=96, model_dim=160, normalize_topk_scores=True, num_experts=5,
                    top_k=2, use_shared_expert=shared, return_router_scores=True)
    with gpu_device:
        layer = ArcticMoE(cfg)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.1)
    x = torch.randn(T, 160, device=gpu_device).to(dtype)
    y, scores = layer(x)
    with torch.no_grad():
        y0, scores0 = layer(x)
        # the shared expert's part against a plain computation of it
        if shared:
            plain = ArcticMoE(MoEConfig(**{**cfg.__dict__, "use_shared_expert": False})).to(gpu_device)
            for n, p in plain.named_parameters():
                p.copy_(getattr(layer, n))
            h = x.float() @ layer.shared_expert_gate_up.float()
            want = (F.silu(h[:, 0::2]) * h[:, 1::2]) @ layer.shared_expert_down.float()
            want = want * torch.sigmoid(x.float() @ layer.shared_expert_output_gate.float())
            got = y0.float() - plain(x)[0].float()
            assert (got - want).norm() <= (2e-2 if dtype == torch.bfloat16 else 1e-5) * (want.norm() + y0.float().norm())
    assert torch.equal(y, y0) and torch.equal(scores, scores0)
    assert y.requires_grad and not y0.requires_grad


def test_failure_in_backward_joins_the_second_stream(gpu_device, monkeypatch):
    """An error between the fork and the join of the second stream: the main stream still waits for it."""
    from arctictraining_amd import ArcticMoE, MoEConfig, moe

    with gpu_device:
        layer = ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=torch.bfloat16, intermediate_dim=32, model_dim=64,
                                    normalize_topk_scores=True, num_experts=4, top_k=2))
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.1)
    x = torch.randn(8, 64, device=gpu_device).bfloat16().requires_grad_(True)
    waited = []
    wait = torch.cuda.Stream.wait_stream

    def spy(self, other):
        waited.append(other.cuda_stream)
        return wait(self, other)

    def fail(*a):
        raise RuntimeError("planted on the host")

    y = layer(x)
    monkeypatch.setattr(torch.cuda.Stream, "wait_stream", spy)
    monkeypatch.setattr(moe, "_router_input_grad", fail)
    with pytest.raises(RuntimeError, match="planted on the host"):
        y.sum().backward()
    assert moe._side_stream(x.device).cuda_stream in waited
    torch.cuda.synchronize()


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("T", [3, 70])
def test_router_of_fewer_experts(gpu_device, gated, T):
    """A router_gate with fewer rows than the layer has experts: the layer of the first experts alone."""
    from arctictraining_amd import ArcticMoE, MoEConfig

    print("router of fewer experts", gated, T, flush=True)
    torch.manual_seed(T)

    def layer(E):
        return ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=torch.bfloat16, intermediate_dim=32, model_dim=64, normalize_topk_scores=True,
                                   num_experts=E, top_k=2, is_gated=gated, loss_coeff=0.5)).to(gpu_device)

    few, wide = layer(5), layer(8)
    with torch.no_grad():
        for n, p in few.named_parameters():
            p.normal_(0.0, 0.1)
            getattr(wide, n).normal_(0.0, 0.1)[:5].copy_(p)
    wide.router_gate = torch.nn.Parameter(few.router_gate.detach().clone())
    x, dy = torch.randn(2, T, 64, device=gpu_device).bfloat16()
    out = []
    for m in (few, wide):
        xg = x.clone().requires_grad_(True)
        y = m(xg)
        y.backward(dy)
        out.append((y.detach(), xg.grad, *(p.grad[:5] for p in m.parameters())))
    assert all(torch.equal(a, b) for a, b in zip(*out))
    for p in (wide.expert_gate_up, wide.expert_down):
        assert bool((p.grad[5:] == 0).all())
