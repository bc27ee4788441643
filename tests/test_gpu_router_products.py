"""The router's products for few tokens against float64, at the edges of their tiles, and the layer on both sides of
the rule that chooses them.  Tolerance: one rounding of the 16-bit result (2^-9 and 2^-12 of the value) and the order of
the float32 sums."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 4e-3, torch.float16: 5e-4}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 33, 256])
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
