"""Few rows an expert where workgroups of two column groups run (rows of whole 512 bytes, enough of them): both tile heights, none to several
tiles an expert, reductions of one step, of an odd number of them and of a few, in one round of workgroups and in more, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows", [(0, 1, 2, 16, 3, 0), (17, 0, 1, 16, 5, 4)])   # tiles of 16 and of 32 rows
@pytest.mark.parametrize("Kd,N", [(32, 1024), (96, 1280), (160, 1024), (512, 3584)])
def test_two_column_groups(gpu_device, dtype, rows, Kd, N):
    from arctictraining_amd import ops

    print("two column groups", dtype, rows, Kd, N, flush=True)
    E = 102
    counts = [rows[e % 6] for e in range(E)]
    counts[5] = 33 if sum(rows) == 22 else 70   # (several tiles)
    R = sum(counts)
    assert R <= 4 * E if sum(rows) == 22 else 4 * E < R <= 8 * E
    g = torch.Generator(device=gpu_device).manual_seed(Kd + N)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    src = torch.randn(R // 3, Kd, device=gpu_device, generator=g).to(dtype)
    row_of = torch.randint(0, R // 3, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    w = (torch.randn(E, Kd, N, device=gpu_device, generator=g) * 0.05).to(dtype)
    a = src[row_of.long()]
    ref = torch.cat([p.double() @ w[e].double() for e, p in enumerate(a.split(counts)) if counts[e]])
    size = torch.cat([p.double().abs() @ w[e].double().abs() for e, p in enumerate(a.split(counts)) if counts[e]])
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    # rounded once, the products summed in float32 (float16 rounds what is below 2^-14 to multiples of 2^-24)
    bound = u * ref.abs() + Kd * 2.0 ** -24 * size + (2.0 ** -25 if dtype == torch.float16 else 0.0)

    got = ops.grouped_gemm_nn(src, w, offs, a_row_map=row_of)
    assert bool(((got.double() - ref).abs() <= bound).all())
    assert torch.equal(got, ops.grouped_gemm_nn(a, w, offs))
    scale = torch.rand(R, device=gpu_device)
    gate_up, inter = ops.grouped_gemm_gateup_act_fwd(src, w, offs, 0, a_row_map=row_of, row_scale=scale)
    assert torch.equal(gate_up, got)
    gate, up = gate_up[:, 0::2].double(), gate_up[:, 1::2].double()
    want = scale[:, None].double() * up * gate * torch.sigmoid(gate)
    # (exponential, reciprocal and three products in float32: a few units of 2^-24)
    assert bool(((inter.double() - want).abs() <= (u + 2.0 ** -20) * want.abs() + (2.0 ** -25 if dtype == torch.float16 else 0.0)).all())
