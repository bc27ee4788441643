"""Weight gradients on the large tiles: row indices are requested three K tiles ahead, across the turns from tile to tile.  Experts of every
number of K tiles from none to eight in turn, one row more and one less, several tiles a workgroup, lower halves that lie past the matrix,
either operand gathered or none, against float64, out of a cold cache."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# (rows of the experts, M, N): M leaves whole, half and nearly empty last tiles
CASES = {
    "turns": ([1, 64, 65, 128, 129, 191, 192, 193, 256, 257, 0, 320, 321, 449, 512, 63] * 3, 512, 768),
    "half": ([130, 260, 64, 0, 390, 200, 1, 515] * 9, 392, 1032),
    "one_tile_each": ([129, 300, 511], 136, 264),
    "deep_among_short": ([65] * 20 + [4000] + [65] * 20, 768, 520),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(CASES))
def test_indices_across_tiles(gpu_device, name, dtype):
    from arctictraining_amd import ops

    counts, M, N = CASES[name]
    R, E = sum(counts), len(counts)
    assert R > 128 * E   # (few rows have a kernel of their own)
    print("weight gradient, indices", name, dtype, flush=True)
    off = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32)
    g = torch.Generator(device=gpu_device).manual_seed(E + M)
    draw = lambda *shape: torch.empty(shape, dtype=dtype, device=gpu_device).normal_(generator=g)
    rows = torch.randint(0, R, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    a, b = draw(R, M), draw(R, N)
    flush = torch.empty(320 << 20, dtype=torch.uint8, device=gpu_device)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for kw, xg, yg in (({}, a, b), (dict(a_row_map=rows), a[rows.long()], b), (dict(b_row_map=rows), a, b[rows.long()])):
        got = []
        for _ in range(3):
            flush.fill_(1)
            got.append(ops.grouped_gemm_wgrad(a, b, off.to(gpu_device), E, **kw))
        assert all(torch.equal(got[0], c) for c in got[1:])
        for e in range(E):
            p, q = (t[int(off[e]):int(off[e + 1])].double() for t in (xg, yg))
            ref, size = p.t() @ q, p.t().abs() @ q.abs()
            # rounded once, the rows' products summed in float32 (float16 rounds what is below 2^-14 to multiples of 2^-24)
            bound = u * ref.abs() + counts[e] * 2.0 ** -24 * size + (2.0 ** -25 if dtype == torch.float16 and counts[e] else 0.0)
            assert bool(((got[0][e].double() - ref).abs() <= bound).all()), (kw.keys(), e)
