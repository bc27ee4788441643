"""Weight gradients of 129 rows per expert and more, whose epilogue takes a wavefront's 64 columns through LDS and stores whole
lines: edges of the 8-column pieces and 16-row blocks it writes, half tiles, one, two and all tiles a workgroup, uneven loads, gradients
that the caches hold and that they do not (stored past them), either operand gathered, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = {
    "pieces": ([130, 0, 257, 300, 1], 264, 328),             # 8 rows and 8 columns past a tile, an expert without rows
    "blocks": ([129, 200, 140], 8, 72),                      # less than one 16-row block, 8 columns past 64
    "half": ([192, 193, 64, 300], 392, 1416),                # a lower half of 8 rows; columns end inside a wavefront's
    "past_the_caches": ([150] * 30, 520, 1096),              # 34 MB, 450 tiles: two a workgroup, of 256
    "two_of_four": ([130] * 40, 776, 1096),                  # 800 tiles: two a workgroup, the second 256 workgroups not all filled
    "uneven": ([0, 3000, 1, 0, 64, 1500, 7] * 6, 776, 1032), # 840 tiles of 3 to 47 K tiles, two a workgroup
    "all_of_three": ([720] * 8, 2056, 2056),                 # 648 tiles of 11 K tiles and more: three a workgroup
    "all_to_one": ([0, 900, 0], 136, 520),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(CASES))
def test_whole_lines(gpu_device, name, dtype):
    from arctictraining_amd import ops

    counts, M, N = CASES[name]
    print("weight gradient, whole lines", name, dtype, flush=True)
    R, E = sum(counts), len(counts)
    assert R > 128 * E   # (few rows have a kernel of their own)
    assert name != "past_the_caches" or 2 * E * M * N > 32 << 20
    off = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32)
    g = torch.Generator(device=gpu_device).manual_seed(R)
    draw = lambda *shape: torch.empty(shape, dtype=dtype, device=gpu_device).normal_(generator=g)
    rows = torch.randint(0, R + 7, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    a, b, a_src, b_src = draw(R, M), draw(R, N), draw(R + 7, M), draw(R + 7, N)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for kw, x, y, xg, yg in (({}, a, b, a, b), (dict(a_row_map=rows), a_src, b, a_src[rows.long()], b),
                             (dict(b_row_map=rows), a, b_src, a, b_src[rows.long()])):
        c = ops.grouped_gemm_wgrad(x, y, off.to(gpu_device), E, **kw)
        assert torch.equal(c, ops.grouped_gemm_wgrad(x, y, off.to(gpu_device), E, **kw))
        for e in range(E):
            p, q = (t[int(off[e]):int(off[e + 1])].double() for t in (xg, yg))
            ref, size = p.t() @ q, p.t().abs() @ q.abs()
            # rounded once, and the rows' products summed in float32; an expert without rows has zeros (float16 rounds what is
            # below 2^-14 to multiples of 2^-24)
            bound = u * ref.abs() + counts[e] * 2.0 ** -24 * size + (2.0 ** -25 if dtype == torch.float16 and counts[e] else 0.0)
            assert bool(((c[e].double() - ref).abs() <= bound).all()), (kw.keys(), e)
