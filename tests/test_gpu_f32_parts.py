"""float32 row-grouped products whose last round of tiles is worked off in parts of 32 rows (256 compute units): a few tiles past one and past
two whole rounds, tiles of all heights among them, either B, gathered rows, the gated epilogue, values without parts, against float64.
Tolerance as for the other forms: 2^-24 of an operand in the parts, K / 32 * 2^-24 of the sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-6

# rows of each expert, K, N: 264 tiles of 128 x 64; 266 that end in tiles of 43, 1, 33 and 97 rows; 666; 360
CASES = [
    ([128] * 7 + [5], 548, 2056),
    ([128, 0, 129, 64, 1, 33, 97], 100, 2376),
    ([128] * 12 + [31, 96, 65, 127, 1, 32], 36, 2312),
    ([256, 300, 90], 1024, 3840),
]


@pytest.mark.parametrize("counts,K,N", CASES)
def test_last_round_in_parts(gpu_device, counts, K, N):
    from arctictraining_amd import ops

    print("float32 parts", counts, K, N, flush=True)
    R, E = sum(counts), len(counts)
    g = torch.Generator(gpu_device).manual_seed(R + N)
    rand = lambda *s: torch.randn(s, device=gpu_device, generator=g)  # noqa: E731
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    src, b, scale = rand(R + 5, K), rand(E, K, N), rand(R)
    rows = torch.randint(0, R + 5, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    a = src[rows.long()]
    parts = a.split(counts)
    ref = torch.cat([x.double() @ b[e].double() for e, x in enumerate(parts)])
    got = ops.grouped_gemm_nn(src, b, off, a_row_map=rows)
    for x, want in zip(got.split(counts), ref.split(counts)):
        assert (x.double() - want).norm() <= TOL * want.norm()
    got_t = ops.grouped_gemm_nt(a, b.transpose(1, 2).contiguous(), off)
    for x, want in zip(got_t.split(counts), ref.split(counts)):
        assert (x.double() - want).norm() <= TOL * want.norm()
    gate_up, inter = ops.grouped_gemm_gateup_act_fwd(src, b, off, 0, a_row_map=rows, row_scale=scale)
    assert torch.equal(gate_up, got)
    gate, up = gate_up[:, 0::2].double(), gate_up[:, 1::2].double()
    want = scale[:, None].double() * up * gate * torch.sigmoid(gate)
    # (exponential, reciprocal and three products: a few units of 2^-24)
    assert (inter.double() - want).abs().max() <= 2.0 ** -20 * want.abs().max()

    # an infinity and a NaN in the last tile's rows
    bad = a.clone()
    bad[R - 1, 0], bad[R - 2 if counts[-1] > 1 else 0, K - 1] = float("inf"), float("nan")
    last = len(counts) - 1
    want = (bad[R - counts[last]:].double() @ b[last].double()).float()
    got = ops.grouped_gemm_nn(bad, b, off)[R - counts[last]:]
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    assert (got[fine].double() - want[fine].double()).norm() <= TOL * max(float(want[fine].double().norm()), 1e-30)
