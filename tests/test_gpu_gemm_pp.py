"""The default tile shape of the 16-bit row-grouped products at the sizes where it can go wrong: reductions
of less than one K tile up to several with a remainder, tiles of every height class, matrix edges, and
launches in which a workgroup walks several tiles.  Reference: the per-expert product in float32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

COUNTS = [0, 1, 31, 32, 33, 128, 129, 0, 160, 200, 225, 255, 256, 257, 300, 513]


@pytest.fixture(scope="module")
def ops(gpu_device):
    from arctictraining_amd import ops as _ops

    return _ops


def _problem(counts, Kd, N, dtype, dev, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(dev)
    R, E = sum(counts), len(counts)
    src = torch.randn(max(R // 3, 1), Kd, device=dev, generator=g).to(dtype)
    rows = torch.randint(0, src.shape[0], (R,), device=dev, generator=g, dtype=torch.int32)
    w = (torch.randn(E, Kd, N, device=dev, generator=g) * 0.05).to(dtype)
    return offs, src, rows, w


def _reference(a, w, counts):
    return torch.cat([p.float() @ w[e].float() for e, p in enumerate(a.split(counts))])


def _check(got, ref, tol):
    assert torch.isfinite(got).all()
    rows = ref.norm(dim=-1)
    err = (got.float() - ref).norm(dim=-1) / torch.maximum(rows, rows.pow(2).mean().sqrt())
    assert float(err.max()) <= tol, f"worst row {float(err.max()):.2e}"


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1e-2), (torch.float16, 2e-3)])
@pytest.mark.parametrize("Kd,N", [(32, 8), (64, 136), (96, 256), (128, 264), (160, 520), (192, 96), (256, 1000), (352, 256)])
def test_edges(ops, gpu_device, dtype, tol, Kd, N):
    print("pp edges", dtype, Kd, N, flush=True)
    offs, src, rows, w = _problem(COUNTS, Kd, N, dtype, gpu_device, Kd + N)
    a = src[rows.long()]
    ref = _reference(a, w, COUNTS)
    wt = w.transpose(1, 2).contiguous()
    _check(ops.grouped_gemm_nn(a, w, offs), ref, tol)
    _check(ops.grouped_gemm_nn(src, w, offs, a_row_map=rows), ref, tol)
    _check(ops.grouped_gemm_nt(a, wt, offs), ref, tol)
    _check(ops.grouped_gemm_nt(src, wt, offs, a_row_map=rows), ref, tol)
    scale = torch.rand(a.shape[0], device=gpu_device)
    gu, inter = ops.grouped_gemm_gateup_act_fwd(src, w, offs, a_row_map=rows, row_scale=scale)
    _check(gu, ref, tol)
    want = scale[:, None] * gu[:, 1::2].float() * torch.nn.functional.silu(gu[:, 0::2].float())
    _check(inter, want, tol)
    only = ops.grouped_gemm_gateup_act_fwd(src, w, offs, a_row_map=rows, row_scale=scale, want_gate_up=False)
    assert only[0] is None and torch.equal(only[1], inter)
    # gated backward: d_inter = a @ w, gate_up of the forward pass given
    fwd = torch.randn(a.shape[0], 2 * N, device=gpu_device).to(dtype)
    d_gu, parts = ops.grouped_gemm_nt_gated_bwd(src, wt, offs, fwd, row_scale=scale, a_row_map=rows)
    gate, up = fwd[:, 0::2].float(), fwd[:, 1::2].float()
    sg = torch.sigmoid(gate)
    want = torch.stack((scale[:, None] * ref * up * (sg * (1 + gate * (1 - sg))), scale[:, None] * ref * gate * sg), -1)
    _check(d_gu, want.flatten(1), tol)
    dots = (ref * up * gate * sg).sum(1)
    assert float((parts.sum(0) - dots).norm() / dots.norm()) <= tol


@pytest.mark.parametrize("E,Kd,N", [(40, 320, 1536), (3, 704, 4096)])
def test_many_tiles_per_workgroup(ops, gpu_device, E, Kd, N):
    """More tiles than compute units: the loads of a tile's first K tiles go out during the previous tile."""
    print("pp many tiles", E, Kd, N, flush=True)
    counts = [(37 * e) % 700 + (900 if E < 8 else 60) for e in range(E)]
    offs, src, rows, w = _problem(counts, Kd, N, torch.bfloat16, gpu_device, E)
    ref = _reference(src[rows.long()], w, counts)
    for _ in range(3):
        _check(ops.grouped_gemm_nn(src, w, offs, a_row_map=rows), ref, 1e-2)
        _check(ops.grouped_gemm_nt(src, w.transpose(1, 2).contiguous(), offs, a_row_map=rows), ref, 1e-2)


@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 1e-2), (torch.float16, 2e-3)])
@pytest.mark.parametrize("M,N,counts", [
    (256, 256, [0, 1, 700, 513, 0, 400]),            # empty and one-row experts, remainders of a K tile
    (136, 1032, [1100, 64, 65, 0, 200, 900]),        # edges in both extents
    (1408, 520, [257] * 9 + [0, 600]),               # a last row tile of half height; 198 tiles, one a workgroup
])
def test_weight_gradient(ops, gpu_device, dtype, tol, M, N, counts):
    print("pp wgrad", dtype, M, N, flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(M + N)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    R, E = sum(counts), len(counts)
    assert R >= 256 * E   # (test_gpu_wgrad_lines.py has fewer rows)
    T = R // 3
    rows = torch.randint(0, T, (R,), device=gpu_device, generator=g, dtype=torch.int32)
    rnd = lambda *s: torch.randn(*s, device=gpu_device, generator=g).to(dtype)
    A, B, As, Bs = rnd(R, M), rnd(R, N), rnd(T, M), rnd(T, N)

    def ref(a, b):
        return torch.stack([p.float().t() @ q.float() for p, q in zip(a.split(counts), b.split(counts))])

    for got, want in (
        (ops.grouped_gemm_wgrad(A, B, offs, E), ref(A, B)),
        (ops.grouped_gemm_wgrad(As, B, offs, E, a_row_map=rows), ref(As[rows.long()], B)),
        (ops.grouped_gemm_wgrad(A, Bs, offs, E, b_row_map=rows), ref(A, Bs[rows.long()])),
    ):
        for e in range(E):
            if counts[e]:
                _check(got[e], want[e], tol)
            else:
                assert bool((got[e] == 0).all())


@pytest.mark.parametrize("operand", ["A", "B"])
def test_weight_gradient_gathered_from_4_gib(ops, gpu_device, operand):
    """A gathered operand of more than 4 GiB behind a short row map: the rows past 4 GiB are the ones that are read."""
    print("pp wgrad of 4 GiB", operand, flush=True)
    M, N, counts = 264, 256, [300, 0, 500]
    width = M if operand == "A" else N
    R, T = sum(counts), (1 << 32) // (2 * width) + 1000
    g = torch.Generator(device=gpu_device).manual_seed(1)
    offs = torch.tensor([0] + counts).cumsum(0).to(torch.int32).to(gpu_device)
    rnd = lambda *s: torch.randn(*s, device=gpu_device, generator=g).bfloat16()
    source = torch.zeros(T, width, device=gpu_device, dtype=torch.bfloat16)
    rows = (T - 1 - torch.arange(R, device=gpu_device)).to(torch.int32)
    dense = rnd(R, width)
    source[rows.long()] = dense
    other = rnd(R, N if operand == "A" else M)
    if operand == "A":
        got, (a, b) = ops.grouped_gemm_wgrad(source, other, offs, 3, a_row_map=rows), (dense, other)
    else:
        got, (a, b) = ops.grouped_gemm_wgrad(other, source, offs, 3, b_row_map=rows), (other, dense)
    for e, (p, q) in enumerate(zip(a.split(counts), b.split(counts))):
        if counts[e]:
            _check(got[e], p.float().t() @ q.float(), 1e-2)
        else:
            assert bool((got[e] == 0).all())
