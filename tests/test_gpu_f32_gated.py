"""float32 gate_up products, whose epilogue applies the gated activation: each of the three kernel forms, columns that end inside
a tile and inside a vector, rows without a scale, and rows that are worked out again for an infinity, a NaN or a product past
the parts' range.  The intermediate activation against its formula in float64 on the gate_up that the same call returns."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = {
    "few_tiles": ([40, 0, 33, 1], 64, 36),          # eight wavefronts share a reduction
    "two_groups": ([700, 0, 129, 671], 512, 320),   # two groups of wavefronts
    "many_tiles": ([500, 513, 0, 987], 128, 1012),
    "few_rows": ([1, 2, 16, 17, 33, 0] * 10, 64, 320),   # tiles of a row on, blocks of 16 without a live row
}


def _act(act, g):
    if act == 0:
        return g * torch.sigmoid(g)
    if act == 1:
        return 0.5 * g * (1 + torch.erf(g * 0.5 ** 0.5))
    return g.relu() if act == 2 else g * torch.sigmoid(1.702 * g)


@pytest.mark.parametrize("special", [False, True])
@pytest.mark.parametrize("act", range(4))
@pytest.mark.parametrize("name", list(CASES))
def test_gated(gpu_device, name, act, special):
    from arctictraining_amd import ops

    counts, H, I = CASES[name]
    print("float32 gated", name, act, special, flush=True)
    R, E = sum(counts), len(counts)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    g = torch.Generator(device=gpu_device).manual_seed(R + act)
    x = torch.randn(R // 2, H, device=gpu_device, generator=g)
    rows = torch.randint(0, R // 2, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    if special:
        x[int(rows[0]), 3], x[int(rows[R - 1]), 0], x[int(rows[R // 2]), H - 1] = float("inf"), float("nan"), 3.0e36
    w = torch.randn(E, H, 2 * I, device=gpu_device, generator=g) * 0.1
    scale = torch.rand(R, device=gpu_device, generator=g) if act % 2 == 0 else None
    gu, inter = ops.grouped_gemm_gateup_act_fwd(x, w, off, act, a_row_map=rows, row_scale=scale)
    a = x[rows.long()]
    ref = torch.cat([p.double() @ w[e].double() for e, p in enumerate(a.split(counts))])
    fine = torch.isfinite(ref).all(1) & (ref.abs().amax(1) < 1e30)
    assert float((gu[fine].double() - ref[fine]).norm() / ref[fine].norm()) <= 1e-6
    gate, up = gu[:, 0::2].double(), gu[:, 1::2].double()
    s = torch.ones(R, 1, device=gpu_device, dtype=torch.float64) if scale is None else scale.double()[:, None]
    want = s * up * _act(act, gate)
    # float32 throughout: the exponential's argument is off by |gate| 2^-24 of itself, gelu by that of 1 + erf's roundings
    bound = 1e-5 * want.abs() + 2e-7 * (s * up * gate).abs()
    near = (inter.double() - want).abs() <= bound
    usual = torch.isfinite(want) & (gate.abs() < 80) & fine[:, None]
    assert bool(near[usual].all())
    if special:
        # what is not finite came out of the formula in float32, whatever form of it the rows took
        bad = ~torch.isfinite(gu).all(1)
        assert bool(bad.any()) and not bool((bad & fine).any())
        f32 = (s.float() * gu[:, 1::2]) * _act(act, gu[:, 0::2])
        lost = ~torch.isfinite(gu[:, 0::2]) | ~torch.isfinite(gu[:, 1::2])
        assert bool((torch.isfinite(inter[lost]) <= torch.isfinite(f32[lost])).all())
        kept = bad[:, None] & ~lost & (gate.abs() < 80)
        assert bool(near[kept].all())
    again = ops.grouped_gemm_gateup_act_fwd(x, w, off, act, a_row_map=rows, row_scale=scale)[1]
    assert torch.equal(inter.view(torch.int32), again.view(torch.int32))
