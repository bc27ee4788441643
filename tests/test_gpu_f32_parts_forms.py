"""float32 row-grouped products whose last round of tiles is worked off in parts of 32 rows, by the lines of each product: behind one, two and three whole
rounds, up to the line and just past it; infinities and NaN in the parts' rows with B^T and under the gated epilogue, where one wavefront does the part
again.  Tolerance as for the other forms: 2^-24 of an operand in the parts, K / 32 * 2^-24 of the sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _line(rounds, kind):
    """sixteenths of a round up to which it is worked off in parts"""
    if kind == "nt":
        return {1: 4, 2: 8}.get(rounds, 5)
    return 7 if rounds == 1 else {2: 10}.get(rounds, 8)


# rows of each expert, K, N, products whose last round is in parts
CASES = [
    ([128] * 7 + [5], 548, 2056, ("nn", "nt", "gated")),            # 264 tiles
    ([200, 128, 64, 1, 33, 97], 100, 2880, ("nn", "nt", "gated")),   # 315
    ([256, 300, 90], 516, 3648, ("nn", "gated")),                   # 342
    ([256, 300, 90], 2052, 3968, ()),                               # 372, deep
    ([128] * 12 + [31, 96, 65, 127, 1, 32], 36, 2176, ("nn", "nt", "gated")),   # 612
    ([128] * 12 + [31, 96, 65, 127, 1, 32], 260, 2312, ("nn", "gated")),        # 666
    ([128] * 12 + [31, 96, 65, 127, 1, 32], 36, 2944, ("nn", "nt", "gated")),   # 828
    ([128] * 12 + [31, 96, 65, 127, 1, 32], 132, 3136, ("nn", "gated")),        # 882
    ([128] * 12 + [31, 96, 65, 127, 1, 32], 36, 3264, ()),                      # 918
]


@pytest.mark.parametrize("counts,K,N,parts", CASES)
def test_lines_and_values_without_parts(gpu_device, counts, K, N, parts):
    from arctictraining_amd import ops

    print("float32 parts, forms", counts, K, N, flush=True)
    cus = torch.cuda.get_device_properties(gpu_device).multi_processor_count
    if cus != 256:
        pytest.skip(f"sized for 256 compute units, not {cus}")
    tiles = sum(-(-c // 128) for c in counts) * -(-N // 64)
    rounds, last = tiles // cus, tiles % cus
    for kind in ("nn", "nt", "gated"):
        assert (0 < last <= cus * _line(rounds, kind) // 16) == (kind in parts), (kind, tiles)
    R, E = sum(counts), len(counts)
    g = torch.Generator(gpu_device).manual_seed(R + N)
    rand = lambda *s: torch.randn(s, device=gpu_device, generator=g)  # noqa: E731
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    a, b, scale = rand(R, K), rand(E, K, N), rand(R)
    bt = b.transpose(1, 2).contiguous()
    bad = a.clone()   # in the last tile's rows, the first and the last of its parts
    last_rows = (counts[-1] - 1) % 128 + 1
    bad[R - 1, 0], bad[R - last_rows, K - 1] = float("inf"), float("nan")
    for x in (a, bad):
        ref = torch.cat([p.double() @ b[e].double() for e, p in enumerate(x.split(counts))])
        fine = ref.isfinite()
        gate_up, inter = ops.grouped_gemm_gateup_act_fwd(x, b, off, 0, row_scale=scale)
        assert x is bad or torch.equal(gate_up, ops.grouped_gemm_nn(x, b, off))
        for got in (ops.grouped_gemm_nn(x, b, off), ops.grouped_gemm_nt(x, bt, off), gate_up):
            assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
            for p, want, ok in zip(got.split(counts), ref.split(counts), fine.split(counts)):
                assert (p[ok].double() - want[ok]).norm() <= TOL * max(float(want[ok].norm()), 1e-30)
        gate, up = gate_up[:, 0::2].double(), gate_up[:, 1::2].double()
        want = scale[:, None].double() * up * gate * torch.sigmoid(gate)
        ok = gate.isfinite() & up.isfinite()
        assert bool(inter[ok].isfinite().all()) and bool(inter.isfinite()[~ok].logical_not().any()) == bool((~ok).any())
        # (exponential, reciprocal and three products: a few units of 2^-24)
        assert (inter[ok].double() - want[ok]).abs().max() <= 2.0 ** -20 * want[ok].abs().max()
