"""Products whose weights are more than the last-level cache holds and are loaded past the caches: 302 MB of nine experts,
against the same products of five and four of them (168 and 134 MB, loaded through the caches), bit by bit: experts without
rows, with one tile of 256 rows and with more.  The kernel for few rows sums in another order for fewer tiles: there
against float64.  The sums of rows over the same bound as well."""
import pytest
import torch

pytestmark = pytest.mark.gpu

E, K, N = 9, 4128, 4064


@pytest.fixture(scope="module")
def ops(gpu_device):
    from arctictraining_amd import ops as _ops

    return _ops


def _case(gpu_device, dtype, counts):
    g = torch.Generator(device=gpu_device).manual_seed(sum(counts))
    draw = lambda *shape: torch.empty(shape, dtype=dtype, device=gpu_device).normal_(0.0, 0.1, generator=g)
    off = torch.tensor([0] + counts, dtype=torch.int32).cumsum(0).to(torch.int32)
    return draw, off, int(off[-1])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts", [
    [256, 257, 0, 255, 1, 300, 32, 90, 511],
    [33, 8, 12, 3, 1, 9, 4, 1, 256],          # nine tiles, the fewest whose weights are more than the cache holds
    [200, 90, 0, 255, 1, 90, 14, 1, 1],       # eight: loaded through the caches
])
def test_tall_tiles(ops, gpu_device, dtype, counts):
    draw, off, R = _case(gpu_device, dtype, counts)
    wide, deep = draw(E, K, N), draw(E, N, K)
    a, b, gate_up, scale = draw(R, K), draw(R, N), draw(R, 2 * N), torch.rand(R, device=gpu_device)
    products = {
        "gate_up": lambda e, r, o: ops.grouped_gemm_gateup_act_fwd(a[r], wide[e], o, row_scale=scale[r]),
        "nn": lambda e, r, o: ops.grouped_gemm_nn(a[r], wide[e], o),
        "nt": lambda e, r, o: ops.grouped_gemm_nt(b[r], wide[e], o),
        "gated_bwd": lambda e, r, o: ops.grouped_gemm_nt_gated_bwd(a[r], deep[e], o, gate_up[r], row_scale=scale[r]),
    }
    for name, run in products.items():
        print("streamed weights", dtype, name, flush=True)
        whole = run(slice(0, E), slice(0, R), off.to(gpu_device))
        whole = whole if isinstance(whole, tuple) else (whole,)
        for lo, hi in ((0, 5), (5, E)):
            rows = slice(int(off[lo]), int(off[hi]))
            part = run(slice(lo, hi), rows, (off[lo:hi + 1] - off[lo]).to(gpu_device))
            for w, p in zip(whole, part if isinstance(part, tuple) else (part,)):
                assert torch.equal(w[:, rows] if w.dim() == 2 and w.shape[0] != R else w[rows], p), name


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("counts", [[1, 0, 16, 3, 0, 8, 5, 2, 0], [17, 8, 0, 31, 1, 2, 0, 4, 7]])   # tiles of 16 and of 32 rows
def test_low_tiles(ops, gpu_device, dtype, counts):
    print("streamed weights", dtype, counts, flush=True)
    draw, off, R = _case(gpu_device, dtype, counts)
    w, a = draw(E, K, N), draw(R, K)
    offsets = off.to(gpu_device)
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    got = ops.grouped_gemm_nn(a, w, offsets)
    gate_up, inter = ops.grouped_gemm_gateup_act_fwd(a, w, offsets)
    assert torch.equal(gate_up, got)
    gate, up = gate_up[:, 0::2].double(), gate_up[:, 1::2].double()
    h = up * gate * torch.sigmoid(gate)
    # rounded once, and float32's exponential and reciprocal
    assert bool(((inter.double() - h).abs() <= (u + 2.0 ** -20) * h.abs() + 2.0 ** -24).all())
    for e in range(E):
        r = slice(int(off[e]), int(off[e + 1]))
        x, y = a[r].double(), w[e].double()
        ref, size = x @ y, x.abs() @ y.abs()
        # rounded once, and K products summed in float32
        assert bool(((got[r].double() - ref).abs() <= u * ref.abs() + K * 2.0 ** -24 * size).all()), e


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("top_k", [2, 4, 7, 9])
def test_row_sums(ops, gpu_device, dtype, top_k):
    """Sums of more rows than the last-level cache holds, against the same in two halves, bit by bit."""
    size, H = torch.finfo(dtype).bits // 8, 4104
    T = (300 << 20) // (top_k * H * size)
    print("streamed rows", dtype, top_k, T, flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(top_k)
    rows = torch.empty((T * top_k, H), dtype=dtype, device=gpu_device).normal_(generator=g)
    row_of = torch.randperm(T * top_k, device=gpu_device, generator=g).view(T, top_k).to(torch.int32)
    scores = torch.rand((T, top_k), device=gpu_device, generator=g)
    addend = torch.empty((T, H), dtype=dtype, device=gpu_device).normal_(generator=g)
    for run in (lambda t: ops.combine_fwd(rows, row_of[t].contiguous(), scores[t].contiguous()),
                lambda t: ops.gather_rows_bwd(rows, row_of[t].contiguous(), addend[t].contiguous())):
        assert torch.equal(run(slice(0, T)), torch.cat([run(slice(0, T // 2)), run(slice(T // 2, T))]))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_parts_of_a_reduction(gpu_device, dtype):
    """Products of few tiles that the layer cuts into parts (down projection and last data gradient, 294 and 587 MB), past the
    caches with rows of all ten experts and through them with rows of nine: bit by bit for the tokens that both have."""
    from arctictraining_amd import ArcticMoE, MoEConfig, moe

    T, H, E, K, I = 100, 512, 10, 2, 28672
    print("streamed weights", dtype, "parts", flush=True)
    # (the layer's scratch has room for parts)
    assert moe._layer_sizes((E, K, H, I, 0, 1, True, 0, False), T, False)[1] - T * K * H * 2 >= 2 * T * K * H * 4
    cfg = MoEConfig(input_dtype=dtype, intermediate_dim=I, model_dim=H, num_experts=E, top_k=K, loss_coeff=0.0, normalize_topk_scores=True,
                    act_fn=torch.nn.functional.silu, enable_routing_replay=True)
    layer = ArcticMoE(cfg).to(gpu_device)
    g = torch.Generator(device=gpu_device).manual_seed(9)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.02, generator=g)
    x, dy = (torch.empty((T, H), dtype=dtype, device=gpu_device).normal_(generator=g) for _ in range(2))
    t = torch.arange(T, device=gpu_device)
    some = torch.stack([t % 8, (t + 3) % 8], 1).to(torch.int32)
    some[90:] = torch.tensor([8, 7], dtype=torch.int32, device=gpu_device)
    every = some.clone()
    every[90:, 1] = 9
    got = []
    for assign in (every, some):
        xg = x.clone().requires_grad_(True)
        out = layer(xg, assign)
        y = out[0] if isinstance(out, tuple) else out
        y.backward(dy)
        got.append((y.detach()[:90], xg.grad[:90]))
    for a, b in zip(*got):
        assert torch.equal(a, b)
    # token 0 goes to experts 0 and 3
    with torch.no_grad():
        p = torch.softmax((x[:1] @ layer.router_gate.t()).float(), -1).topk(K, -1).values
        w = (p / p.sum()).to(dtype).double()[0]
        ref = 0.0
        for e, s in zip((0, 3), w):
            h = x[:1].double() @ layer.expert_gate_up[e].double()
            ref = ref + s * ((torch.nn.functional.silu(h[:, 0::2]) * h[:, 1::2]) @ layer.expert_down[e].double())
        assert (got[0][0][:1].double() - ref).norm() <= 1e-2 * ref.norm()
