"""Weight gradients at the ends of the few-row kernel's range, 128 rows an expert and 129, whose epilogues take eight rows at a
time through LDS: extents that end inside a line, a block of eight rows or a wavefront's columns, either operand gathered,
against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = {
    "edge": ([64, 63, 0, 128, 385], 136, 120),
    "hot": ([0, 512, 0, 0], 264, 8),
    "past": ([0, 513, 0, 0], 264, 8),              # 256-column tiles
    "ragged": ([128, 1, 200, 7], 72, 200),
    "wide": ([33, 0, 97], 8, 1032),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(CASES))
def test_lines(gpu_device, name, dtype):
    from arctictraining_amd import ops

    counts, M, N = CASES[name]
    print("few rows, whole lines", name, dtype, flush=True)
    R, E = sum(counts), len(counts)
    assert (R <= 128 * E) == (name != "past")
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


@pytest.mark.parametrize("counts,kernel", [([0, 512, 0, 0], "short_wgrad"), ([128] * 4, "short_wgrad"), ([0, 513, 0, 0], "pp_wgrad")])
def test_which_kernel(gpu_device, launched, counts, kernel):
    """Up to 128 rows an expert the few-row kernel, whatever the loads: with all rows on one of 64 experts of 1024 x 2048 the large
    tiles take 1.9 times as long."""
    from arctictraining_amd import ops

    print("few rows, which kernel", counts, flush=True)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    a, b = (torch.zeros(sum(counts), n, dtype=torch.bfloat16, device=gpu_device) for n in (64, 72))
    names = launched(lambda: ops.grouped_gemm_wgrad(a, b, off, len(counts)))
    assert any(kernel in n for n in names) and sum("wgrad" in n for n in names) == 1, names
