"""Weight gradients whose tiles are dealt by depth, over the range of experts: more than a wavefront of them, numbers that are no multiple of four, as many as
the kernel has threads, gradients that the L2s hold (stored the ordinary way), and Zipf loads.  Every element against float64; the outputs'
memory holds NaN before."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows of the experts, M, N (256 x 256 tiles: 12, 9, 36, 16 and 35 an expert)
CASES = {
    "67": ([{3: 9000, 40: 9000, 41: 90000, 66: 200000}.get(e, 900 * (e % 7)) for e in range(67)], 520, 1000),
    "130": ([2600 + 37 * e for e in range(126)] + [180000, 0, 150000, 1], 520, 704),
    "512": ([900] * 200 + [45500] * 8 + [64 * (e % 30) for e in range(304)], 1496, 1480),
    "held": ([26000 if e in (0, 5, 16, 21) else 500 + 20 * e for e in range(30)], 264, 2048),
    "zipf": ([int(90000 * (e + 1) ** -1.2) for e in range(35)], 1544, 1064),
}


@pytest.mark.parametrize("name", list(CASES))
def test_every_tile_is_dealt(gpu_device, name):
    from arctictraining_amd import ops

    counts, M, N = CASES[name]
    R, E = sum(counts), len(counts)
    assert R >= 704 * E and (2 * E * M * N <= 32 << 20) == (name == "held")
    print("weight gradient, dealing", name, E, R, flush=True)
    off = torch.tensor([0] + counts, dtype=torch.int64).cumsum(0).to(torch.int32)
    g = torch.Generator(device=gpu_device).manual_seed(M)
    draw = lambda *shape: torch.empty(shape, dtype=torch.bfloat16, device=gpu_device).normal_(generator=g)  # noqa: E731
    few = 5000
    rows = torch.randint(0, few, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    a, b = draw(few, M), draw(R, N)
    torch.cuda.empty_cache()
    torch.full((E, M, N), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    got = ops.grouped_gemm_wgrad(a, b, off.to(gpu_device), E, a_row_map=rows)
    for e in range(E):
        lo, hi = int(off[e]), int(off[e + 1])
        p, q = a[rows[lo:hi].long()].double(), b[lo:hi].double()
        ref, size = p.t() @ q, p.t().abs() @ q.abs()
        # (rounded once, the rows' products summed in float32)
        bound = 2.0 ** -8 * ref.abs() + counts[e] * 2.0 ** -24 * size
        assert bool(((got[e].double() - ref).abs() <= bound).all()), e
