"""Few rows an expert: a row's result does not depend on how many others a call has, that is whether its workgroups are one column group of four
wavefronts (up to 128 rows) or two of two, on the height of a map's tiles, or on where the rows are.  Bit for bit, infinities and NaN among the values."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _chunks(counts, most=128):
    """experts [lo, hi) of up to `most` rows each that cover all, the last ones reaching back over those before"""
    out, lo = [], 0
    while lo < len(counts):
        hi = lo
        while hi < len(counts) and sum(counts[lo:hi + 1]) <= most:
            hi += 1
        if hi == len(counts):
            while lo and sum(counts[lo - 1:hi]) <= most:
                lo -= 1
        assert hi > lo
        out.append((lo, hi))
        lo = hi
    return out


def _two_groups(gpu_device, tiles, N, rounds):
    """whether that many tiles run as workgroups of two column groups, of which `rounds` run on a compute unit at a time"""
    cus = torch.cuda.get_device_properties(gpu_device).multi_processor_count
    if cus != 256:
        pytest.skip(f"sized for 256 compute units, not {cus}")
    w = tiles * (N // 256)
    return 2 * w >= 3 * cus and (w > (rounds + 1) * cus or -(-2 * w // cus) % 2 == 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,N", [((0, 1, 2, 16, 3, 0), 1536), ((0, 1, 2, 16, 3, 0), 3584), ((0, 1, 2, 16, 3, 0), 1280),   # tiles of 16 rows
                                    ((17, 0, 1, 16, 5, 4), 1280), ((17, 0, 1, 16, 5, 4), 3584), ((17, 0, 1, 16, 5, 4), 1536)])   # and of 32
@pytest.mark.parametrize("Kd", [32, 96, 160, 224, 512, 2048])
def test_rows_of_larger_and_smaller_calls(gpu_device, dtype, rows, Kd, N):
    from arctictraining_amd import ops

    print("few rows, order of sums", dtype, rows, Kd, N, flush=True)
    E = 102
    counts = [rows[e % 6] for e in range(E)]
    counts[5] = 33 if sum(rows) == 22 else 70   # (several tiles)
    R = sum(counts)
    high = 16 if sum(rows) == 22 else 32
    two = _two_groups(gpu_device, sum(-(-c // high) for c in counts), N, 4 if high == 16 else 3)
    assert two == ((high, N) not in ((16, 1280), (32, 1536)))   # (those with one group, as the smaller calls)
    g = torch.Generator(device=gpu_device).manual_seed(Kd + N)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    a = torch.randn(R, Kd, device=gpu_device, generator=g).to(dtype)
    w = (torch.randn(E, Kd, N, device=gpu_device, generator=g) * 0.05).to(dtype)
    scale = torch.rand(R, device=gpu_device, generator=g)
    bad = a.clone()
    bad[3, Kd - 1], bad[R - 1, 0], bad[R // 2, Kd // 2] = float("inf"), float("nan"), float("-inf")
    same = lambda x, y: torch.equal(x.isnan(), y.isnan()) and torch.equal(x.nan_to_num(0.0), y.nan_to_num(0.0))  # noqa: E731

    whole = [ops.grouped_gemm_nn(a, w, offs), ops.grouped_gemm_nn(bad, w, offs), *ops.grouped_gemm_gateup_act_fwd(a, w, offs, 0, row_scale=scale)]
    assert bool(whole[0].isfinite().all()) and bool(whole[1][3].isnan().logical_or(whole[1][3].isinf()).all())
    for lo, hi in _chunks(counts):
        r0, r1 = sum(counts[:lo]), sum(counts[:hi])
        assert r1 - r0 <= 128
        empty = max(0, (r1 - r0 + 5) // 6 - (hi - lo))   # (experts without rows, as many rows an expert as the few-row kernel takes)
        part_offs = torch.cat([offs[lo:hi + 1], offs[hi:hi + 1].expand(empty)]) - offs[lo]
        x, b, we = a[r0:r1].contiguous(), bad[r0:r1].contiguous(), torch.cat([w[lo:hi], w[:empty]])
        got = [ops.grouped_gemm_nn(x, we, part_offs), ops.grouped_gemm_nn(b, we, part_offs),
               *ops.grouped_gemm_gateup_act_fwd(x, we, part_offs, 0, row_scale=scale[r0:r1].contiguous())]
        for p, q in zip(got, whole):
            assert same(p, q[r0:r1]), (lo, hi, float((p.double() - q[r0:r1].double()).abs().nan_to_num(0.0).max()))


@pytest.mark.parametrize("plan_rows,call_rows", [(4, 8), (4, 40), (8, 4), (40, 4), (40, 8)])
def test_map_of_another_bound(gpu_device, plan_rows, call_rows):
    """taller or lower tiles in the map than the call's own rule makes, enough workgroups for two column groups"""
    from arctictraining_amd import ops

    E, Kd, N = 104, 96, 1536
    counts = [(0, 1, 2, 7, 3, 0, 5, 0)[e % 8] for e in range(E)]
    counts[3] += 41
    R = sum(counts)
    print("few rows, map of another bound", plan_rows, call_rows, R, flush=True)
    assert R <= min(plan_rows, call_rows) * E and R > 128
    assert all(_two_groups(gpu_device, sum(-(-c // high) for c in counts), N, rounds) for high, rounds in ((16, 4), (16, 3), (32, 4), (32, 3)))
    g = torch.Generator(device=gpu_device).manual_seed(plan_rows)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    x = torch.randn(max(plan_rows, call_rows) * E, Kd, device=gpu_device, generator=g).bfloat16()
    w = (torch.randn(E, Kd, N, device=gpu_device, generator=g) * 0.05).bfloat16()
    want = ops.grouped_gemm_nn(x[:R].contiguous(), w, offs)
    ws = ops.gemm_workspace(x.shape[0], E, gpu_device)
    ops.grouped_gemm_nn(x[:plan_rows * E].contiguous(), w, offs, workspace=ws)   # (leaves its map)
    got = ops.grouped_gemm_nn(x[:call_rows * E].contiguous(), w, offs, workspace=ws, map_ready=True)[:R]
    if max(plan_rows, call_rows) <= 8:
        assert torch.equal(got, want)
    else:   # (the default tiles' order of sums)
        assert (got.double() - want.double()).norm() <= 2.0 ** -7 * want.double().norm()


@pytest.mark.parametrize("rows", [1000, 1900])   # tiles of 16 and of 32 rows
@pytest.mark.parametrize("on", [1, 7, 64, 100, 130, 180, 205, 230, 260, 275, 300])
def test_rows_on_some_of_the_experts(gpu_device, rows, on):
    """one or two column groups by the tiles that there are, and every tile by some workgroup: the memory of the output holds NaN before"""
    from arctictraining_amd import ops

    print("few rows on some of the experts", rows, on, flush=True)
    E, Kd, N = 300, 64, 1024
    counts = [0] * E
    for r in range(rows):
        counts[(r % on) * E // on] += 1
    high, rounds = (16, 4) if rows == 1000 else (32, 3)
    two = {1000: (100, 180, 230, 300), 1900: (100, 180, 230, 260, 275, 300)}[rows]
    assert _two_groups(gpu_device, sum(-(-c // high) for c in counts), N, rounds) == (on in two)
    assert sum(c > 0 for c in counts) == on and (rows <= 4 * E) == (rows == 1000) and rows <= 8 * E
    g = torch.Generator(device=gpu_device).manual_seed(on)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    a = torch.randn(rows, Kd, device=gpu_device, generator=g).bfloat16()
    w = (torch.randn(E, Kd, N, device=gpu_device, generator=g) * 0.05).bfloat16()
    ref = torch.cat([p.double() @ w[e].double() for e, p in enumerate(a.split(counts)) if counts[e]])
    size = torch.cat([p.double().abs() @ w[e].double().abs() for e, p in enumerate(a.split(counts)) if counts[e]])
    torch.cuda.empty_cache()
    torch.full((rows, N), float("nan"), dtype=torch.bfloat16, device=gpu_device)
    got = ops.grouped_gemm_nn(a, w, offs)
    # (rounded once, the products summed in float32)
    assert bool(((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + Kd * 2.0 ** -24 * size).all())
