"""The float32 grouped products against float64, on both sides of the rules that choose their forms and at the edges of
their tiles.  Tolerance: the parts that are kept hold 2^-24 of an operand, a float32 accumulator of K / 32 steps (two groups of
wavefronts or eight halve or shorten the chain) errs by at most K / 32 * 2^-24 of the largest partial sum; 1e-6 of the
2-norm covers K <= 1024."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-6


def _offsets(counts, device):
    return torch.from_numpy(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)).to(device)


# rows of each expert, K, N: the eight-wave form, two groups, one group; remainders of 32, 64 and 128
CASES = [
    ([1], 4, 4),
    ([0, 33, 1, 0, 31], 100, 68),
    ([128, 129, 0, 127], 36, 64),
    ([300, 180], 1024, 132),
    ([513, 255, 0], 548, 2052),
    ([700, 96, 640], 260, 1028),
]


@pytest.mark.parametrize("counts,K,N", CASES)
@pytest.mark.parametrize("gather", [False, True])
def test_products(gpu_device, counts, K, N, gather):
    from arctictraining_amd import ops

    print("float32 products", counts, K, N, gather, flush=True)
    R, E = sum(counts), len(counts)
    g = torch.Generator(gpu_device).manual_seed(R + K + N)
    rand = lambda *s: torch.randn(s, device=gpu_device, generator=g)  # noqa: E731
    off = _offsets(counts, gpu_device)
    b, bt, d = rand(E, K, N), rand(E, N, K), rand(R, N)
    rows = torch.randint(0, R + 5, (R,), device=gpu_device, generator=g, dtype=torch.int32) if gather else None
    a = rand(R + 5, K) if gather else rand(R, K)
    full = a[rows.long()] if gather else a
    kw = dict(a_row_map=rows) if gather else {}
    nn = ops.grouped_gemm_nn(a, b, off, **kw)
    nt = ops.grouped_gemm_nt(a, bt, off, **kw)
    wa = ops.grouped_gemm_wgrad(a, d, off, E, **kw)
    src = rand(R + 5, N) if gather else d
    wb = ops.grouped_gemm_wgrad(full, src, off, E, b_row_map=rows)
    dfull = src[rows.long()] if gather else d
    for e in range(E):
        s = slice(sum(counts[:e]), sum(counts[: e + 1]))
        x = full[s].double()
        for got, ref in ((nn[s], x @ b[e].double()), (nt[s], x @ bt[e].double().t()), (wa[e], x.t() @ d[s].double()),
                         (wb[e], x.t() @ dfull[s].double())):
            assert (got.double() - ref).norm() <= TOL * ref.norm()


@pytest.mark.parametrize("counts,K,N", [([40, 3], 64, 68), ([300, 180], 1024, 132), ([700, 96, 640], 64, 1028)])
def test_values_that_have_no_parts(gpu_device, counts, K, N):
    """Infinities, NaN and values next to the largest, which round to infinity in bfloat16: as in float64, rounded."""
    from arctictraining_amd import ops

    print("float32 special values", counts, K, N, flush=True)
    R, E = sum(counts), len(counts)
    g = torch.Generator(gpu_device).manual_seed(R)
    a = torch.randn(R, K, device=gpu_device, generator=g)
    b = torch.randn(E, K, N, device=gpu_device, generator=g)
    d = torch.randn(R, N, device=gpu_device, generator=g)
    a[0, 1], a[1, 0], a[2, 3], a[R - 1, K - 1] = float("inf"), float("nan"), 3.4e38, -float("inf")
    a[2, 4:] *= 1e-3
    b[0, 3] *= 1e-3
    b[0, 3, 0], b[E - 1, 5, N - 1] = 0.0, float("inf")
    d[3, 7], d[2] = -float("inf"), d[2] * 1e-3
    off = _offsets(counts, gpu_device)
    bt = b.transpose(1, 2).contiguous()
    nn, nt, w = ops.grouped_gemm_nn(a, b, off), ops.grouped_gemm_nt(a, bt, off), ops.grouped_gemm_wgrad(a, d, off, E)

    def same(got, ref):
        ref32 = ref.float()
        assert torch.equal(got.isnan(), ref32.isnan()) and torch.equal(got.isinf(), ref32.isinf())
        assert torch.equal(got[got.isinf()], ref32[got.isinf()])
        ok = ref32.isfinite()
        # (of a sum next to a term of 3e35 what is left is that term's rounding: compared line by line of the scale)
        scale = torch.where(ok, ref, 0).abs().amax()
        assert ((got.double() - ref)[ok].abs() <= 1e-5 * scale).all()

    for e in range(E):
        s = slice(sum(counts[:e]), sum(counts[: e + 1]))
        same(nn[s], a[s].double() @ b[e].double())
        same(nt[s], a[s].double() @ b[e].double())
        same(w[e], a[s].double().t() @ d[s].double())


@pytest.mark.parametrize("counts,K,N", [([40, 3], 64, 68), ([300, 180], 1024, 132), ([700, 96, 640], 64, 1028)])
@pytest.mark.parametrize("ea,eb", [(-118, 100), (100, -122), (-126, 110), (120, -140), (-62, -60), (60, 50)])
def test_values_near_the_ends_of_the_range(gpu_device, counts, K, N, ea, eb):
    """Operands around 2^ea and 2^eb, subnormal ones among them, as exact as any others; rows of zeros give zeros."""
    from arctictraining_amd import ops

    print("float32 range", counts, K, N, ea, eb, flush=True)
    R, E = sum(counts), len(counts)
    g = torch.Generator(gpu_device).manual_seed(R)

    def rand(e, *s):
        return (torch.randn(s, device=gpu_device, generator=g).double() * 2.0**e).float()

    a, b, d = rand(ea, R, K), rand(eb, E, K, N), rand(eb, R, N)
    a[1], a[:, 2] = 0.0, 0.0
    off = _offsets(counts, gpu_device)
    nn, nt = ops.grouped_gemm_nn(a, b, off), ops.grouped_gemm_nt(a, b.transpose(1, 2).contiguous(), off)
    w = ops.grouped_gemm_wgrad(a, d, off, E)
    assert not nn[1].any() and not nt[1].any() and not w[:, 2].any()
    for e in range(E):
        s = slice(sum(counts[:e]), sum(counts[: e + 1]))
        for got, ref in ((nn[s], a[s].double() @ b[e].double()), (nt[s], a[s].double() @ b[e].double()),
                         (w[e], a[s].double().t() @ d[s].double())):
            # (and half of the smallest float32 for each)
            assert (got.double() - ref).norm() <= TOL * ref.norm() + 2.0**-150 * ref.numel() ** 0.5
