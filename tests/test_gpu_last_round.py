"""Dealing of the 16-bit row-grouped products' tiles: fewer tiles than a round, in 4, 2 or 1 pieces each, rounds with a few tiles
left over, groups of tile rows that end short, super-columns of unequal width, low tiles that stay whole.  Operands are small
integers, whose float32 sums are exact in any order: results equal the reference bit for bit, on repetition too."""
import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = {
    "one": ([250], 128, 256),                                    # a single tile, in quarters
    "five": ([256, 200, 256, 31, 225], 64, 256),
    "quarters": ([256, 250, 193, 225], 128, 320),                # 4 x 2 tiles
    "halves": ([300, 225, 512, 768], 64, 2560),                  # 8 x 10, two super-columns of 5
    "whole": ([192, 190, 64, 1], 96, 4608),                      # 4 x 18, none of them tall
    "one_round": ([256] * 16, 96, 4096),                         # 16 x 16 = 256
    "few_left": ([257, 250, 255] * 8, 64, 2200),                 # 32 x 9, super-columns of 5 and 4, 32 left, in quarters
    "many_left": ([200, 256, 0, 7] * 13, 64, 2816),              # 39 x 11, super-columns of 6 and 5, 173 left
    "past_the_caches": ([1000, 31, 2000, 0, 5200], 64, 8200),    # 128 MiB and more, which are stored past the caches, but not
    "whole_lines": ([1000, 31, 2000, 0, 5200], 64, 8192),        # .. in rows of 16400 bytes: these are
    "turned_2048": ([200, 31, 0, 256, 257, 90], 2048, 264),      # reductions that start at another K tile for every expert (B^T)
    "turned_6144": ([40, 300] * 4, 6144, 72),
    "tall": ([224, 225, 256, 255], 64, 10240),                   # 4 x 40, not cut: the last 32 rows of a tile dead, begun and full
    "short_group": ([256, 31] * 19 + [250], 64, 1904),           # 39 x 8, groups of 4
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(CASES))
def test_every_tile_once(gpu_device, name, dtype):
    from arctictraining_amd import ops

    counts, K, N = CASES[name]
    print("last round", name, dtype, flush=True)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    R, E = sum(counts), len(counts)
    g = torch.Generator(device=gpu_device).manual_seed(R)
    draw = lambda *shape: torch.randint(-2, 3, shape, device=gpu_device, generator=g).to(dtype)
    src, w = draw(R // 2, K), draw(E, K, N)
    rows = torch.randint(0, R // 2, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    a = src[rows.long()]
    ref = torch.cat([p.float() @ w[e].float() for e, p in enumerate(a.split(counts))])      # |sums| <= 4 K: exact
    wt = w.transpose(1, 2).contiguous()
    for _ in range(2):
        assert torch.equal(ops.grouped_gemm_nn(a, w, off), ref.to(dtype))
        assert torch.equal(ops.grouped_gemm_nt(src, wt, off, a_row_map=rows), ref.to(dtype))
        gate_up, _ = ops.grouped_gemm_gateup_act_fwd(src, w, off, a_row_map=rows)
        assert torch.equal(gate_up, ref.to(dtype))
    # gated backward, relu: d_gate_up = (d up 1[gate > 0], d relu(gate)) and row sums of d up relu(gate), all of integers; up to 4 K * 2
    # * 2, which 8 significant bits do not hold, so that the products are rounded once
    fwd = draw(R, 2 * N)
    d_gu, parts = ops.grouped_gemm_nt_gated_bwd(src, wt, off, fwd, 2, a_row_map=rows)
    gate, up = fwd[:, 0::2].float(), fwd[:, 1::2].float()
    want = torch.stack((ref * up * (gate > 0), ref * gate.relu()), -1).flatten(1).to(dtype)
    assert torch.equal(d_gu, want)
    assert torch.equal(parts.sum(0), (ref * up * gate.relu()).sum(1))


def test_more_columns_than_the_reciprocal_divides(gpu_device):
    """Tile numbers of a short group are divided by the number of column tiles with its reciprocal rounded up, which is one too many
    for the last one of the third row of 37927: that tile would lie in a row that does not exist.  Three rows, 1.9 GB of weights."""
    from arctictraining_amd import ops

    n_tiles = 37927
    last, inv = 3 * n_tiles - 1, -(-2 ** 32 // n_tiles)
    assert last * inv >> 32 == last // n_tiles + 1
    print("many columns", n_tiles, flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(1)
    draw = lambda *shape: torch.randint(-2, 3, shape, device=gpu_device, generator=g, dtype=torch.int8).to(torch.bfloat16)
    a, w = draw(3, 32), draw(3, 256 * n_tiles, 32)
    got = ops.grouped_gemm_nt(a, w, torch.arange(4, dtype=torch.int32, device=gpu_device))
    for e in range(3):
        assert torch.equal(got[e], (w[e].float() @ a[e].float()).to(torch.bfloat16)), e


@pytest.mark.parametrize("name,epilogue", [("whole_lines", 4), ("past_the_caches", 0), ("whole", 0)])
def test_which_go_past_the_caches(gpu_device, launched, name, epilogue):
    """Large outputs, if their rows are whole lines: stores of parts of lines past the caches take longer than ordinary ones."""
    from arctictraining_amd import ops

    counts, K, N = CASES[name]
    print("past the caches", name, flush=True)
    off = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    a, w = (torch.zeros(*shape, dtype=torch.bfloat16, device=gpu_device) for shape in ((sum(counts), K), (len(counts), K, N)))
    names = launched(lambda: (ops.grouped_gemm_nn(a, w, off), ops.grouped_gemm_nt(a, w.view(len(counts), N, K), off)))
    for b_kc in ("false", "true"):
        assert any(f"pp_rows_bf16_kernel<{b_kc}, {epilogue}, 0," in n for n in names), names
