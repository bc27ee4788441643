"""Weight gradients of uneven loads, whose tiles are dealt by depth: a deep expert first, last and in the middle, several of them, many of equal depth
behind, experts without rows, ragged last tiles, either operand gathered or none, and loads just too even for it.  Every element against float64;
the outputs' memory holds NaN before, which a tile that nobody takes would leave."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows of the experts, M, N (256 x 256 tiles: 48 to 96 an expert)
CASES = {
    "first": ([6000, 400, 300, 200, 0, 500, 65, 64, 700, 350, 129, 800], 1928, 2952),
    "last": ([400, 300, 0, 0, 500, 65, 64, 700, 350, 1, 800, 7000], 2048, 2816),
    "several": ([300, 3000, 200, 0, 5000, 100, 100, 100, 100, 1500, 100, 100, 1600, 90, 80, 70], 1544, 2056),
    "two_depths": ([192] * 10 + [9000] + [192] * 5, 2048, 3072),
    "too_even": ([1500] * 3 + [700] * 9, 1928, 2952),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(CASES))
def test_every_tile_is_dealt(gpu_device, name, dtype):
    from arctictraining_amd import ops

    counts, M, N = CASES[name]
    R, E = sum(counts), len(counts)
    tiles = -(-M // 256) * -(-N // 256)
    depths = [max(3, -(-c // 64)) + 3 for c in counts]
    assert R >= 704 * E and tiles * E > 256 and sum(depths) * tiles >= 1024 * E
    assert (max(depths) * E > 2 * sum(depths)) == (name != "too_even")
    print("weight gradient, dealing", name, dtype, flush=True)
    off = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32)
    g = torch.Generator(device=gpu_device).manual_seed(M)
    draw = lambda *shape: torch.empty(shape, dtype=dtype, device=gpu_device).normal_(generator=g)
    rows = torch.randint(0, R, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    a, b = draw(R, M), draw(R, N)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for kw, xg, yg in (({}, a, b), (dict(a_row_map=rows), a[rows.long()], b), (dict(b_row_map=rows), a, b[rows.long()])):
        torch.cuda.empty_cache()
        torch.full((E, M, N), float("nan"), dtype=dtype, device=gpu_device)
        got = ops.grouped_gemm_wgrad(a, b, off.to(gpu_device), E, **kw)
        for e in range(E):
            p, q = (t[int(off[e]):int(off[e + 1])].double() for t in (xg, yg))
            ref, size = p.t() @ q, p.t().abs() @ q.abs()
            # rounded once, the rows' products summed in float32 (float16 rounds what is below 2^-14 to multiples of 2^-24)
            bound = u * ref.abs() + counts[e] * 2.0 ** -24 * size + (2.0 ** -25 if dtype == torch.float16 and counts[e] else 0.0)
            assert bool(((got[e].double() - ref).abs() <= bound).all()), (kw.keys(), e)
