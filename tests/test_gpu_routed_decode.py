"""A few tokens: the routing inside the gate_up product and the sums over a token's rows inside the down product, against the same
pass with the selection handed over as a replay, which routes and sums in kernels of their own: every result, every field of the
routing and every gradient bit for bit, on both sides of the lines at which the path is taken."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

CASES = {
    "one": (1, 64, 5, 3, 32),                 # 15 columns tiles, most of them past the end
    "wide": (1, 2048, 128, 8, 768),           # half-width tiles
    "all_alike": (4, 96, 2, 2, 64),           # both experts have every token, four rows an expert on average
    "limits": (8, 2560, 256, 16, 96),         # the most rows and experts
    "many_rows": (8, 544, 256, 7, 96),        # the most of them where rows are short
    "two_in_turn": (8, 288, 64, 2, 1056),     # four wavefronts select eight tokens
    "full_width": (7, 4096, 64, 6, 1056),     # 128-column tiles, columns past the end
}
PAST = {                                      # past the lines: the launches of their own on both sides
    "experts": (8, 64, 257, 2, 32),
    "tokens": (9, 64, 64, 2, 32),
    "rows": (6, 96, 256, 12, 96),             # each workgroup would walk over 72 rows
    "in_turn": (8, 64, 128, 4, 768),          # a wavefront would select two tokens, four experts each
    "workgroups": (3, 64, 243, 10, 3712),     # a compute unit would select more than once
}
NAMES = list(CASES) + list(PAST)


def _layer(device, dtype, H, E, K, I, normalize=True, shared=False):
    from arctictraining_amd import ArcticMoE, MoEConfig

    with torch.device(device):
        layer = ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=dtype, intermediate_dim=I, model_dim=H, normalize_topk_scores=normalize,
                                    num_experts=E, top_k=K, loss_coeff=0.001, use_shared_expert=shared))
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.05)
    return layer


def _run(layer, x, dy, replay=None, grad=True):
    layer.zero_grad(set_to_none=True)
    layer.capture = {}
    layer.enable_routing_replay = replay is not None
    xi = x.clone().requires_grad_(grad)
    with torch.set_grad_enabled(grad):
        y = layer(xi, routing_replay_assignments=replay)
    out = dict(y=y.detach().clone(), **{k: v.clone() for k, v in layer.capture.items() if torch.is_tensor(v)})
    if grad:
        y.backward(dy)
        out.update({n: p.grad.clone() for n, p in layer.named_parameters()}, dx=xi.grad.clone())
    return out


def _bits(t):
    return t.contiguous().view({2: torch.int16, 4: torch.int32, 8: torch.int64}[t.element_size()])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("name", NAMES)
def test_same_as_with_launches_of_their_own(gpu_device, launched, name, shared, dtype):
    T, H, E, K, I = CASES.get(name) or PAST[name]
    print("few tokens", name, shared, dtype, flush=True)
    torch.manual_seed(T + H)
    layer = _layer(gpu_device, dtype, H, E, K, I, T != 7, shared)
    x = torch.randn(1, T, H, device=gpu_device).to(dtype)
    if T > 2:
        x[0, 1] = x[0, 0]                     # two tokens that route alike
    dy = torch.randn(1, T, H, device=gpu_device).to(dtype)
    own = _run(layer, x, dy)
    replay = own["topk_idx"].clone()
    for grad in (True, False):
        got, want = _run(layer, x, dy, grad=grad), _run(layer, x, dy, replay, grad)
        assert got.keys() == want.keys()
        for k in want:
            assert torch.equal(got[k], want[k]), (k, grad)
    again = _run(layer, x, dy, grad=False)    # (who arrives last does not matter)
    assert torch.equal(again["y"], own["y"])
    # which path took which
    inside = lambda names, what: any(what in n for n in names)
    names = launched(lambda: _run(layer, x, dy, grad=False))
    assert inside(names, "skinny_routed") == (name in CASES), names
    assert inside(names, "skinny_combine") == (name in CASES and not shared), names
    names = launched(lambda: _run(layer, x, dy, replay, False))
    assert not inside(names, "skinny_routed") and not inside(names, "skinny_combine"), names
    # and the replay is what the other path goes by
    moved = _run(layer, x, dy, (replay + 1) % E, False)
    assert E == K or not torch.equal(moved["y"], own["y"])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("value", [float("nan"), float("inf"), -float("inf")])
def test_logits_without_a_value(gpu_device, launched, value, dtype):
    """Experts whose logits are NaN or infinite for some tokens or all: selection, scores and results as in the launches of their own, bit
    for bit (a NaN's too)."""
    print("few tokens, logits", value, dtype, flush=True)
    T, H, E, K, I = 5, 64, 40, 3, 64
    torch.manual_seed(5)
    layer = _layer(gpu_device, dtype, H, E, K, I)
    x = torch.randn(1, T, H, device=gpu_device).to(dtype)
    x[0, :, 0], x[0, 1, 0] = 1.0, 0.0         # (0 inf is NaN: that token has one whatever the value)
    with torch.no_grad():
        layer.router_gate[7, 0] = value
        layer.router_gate[2, 0] = value
        x[0, 3, 5] = value                    # every logit of this token
    own = _run(layer, x, None, grad=False)
    assert bool((own["topk_idx"] >= 0).all()) and bool((own["topk_idx"] < E).all())
    want = _run(layer, x, None, own["topk_idx"].clone(), False)
    for k in want:
        assert torch.equal(_bits(own[k]), _bits(want[k])), k
    assert any("skinny_routed" in n for n in launched(lambda: _run(layer, x, None, grad=False)))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_under_graph_capture(gpu_device, dtype):
    """The counters of the arrivals are cleared inside the pass: every replay finds them at zero."""
    from arctictraining_amd import ArcticMoE, MoEConfig

    print("few tokens, captured", dtype, flush=True)
    T, H, E, K, I = 3, 256, 32, 4, 96
    torch.manual_seed(3)
    with torch.device(gpu_device):
        layer = ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=dtype, intermediate_dim=I, model_dim=H, normalize_topk_scores=True,
                                    num_experts=E, top_k=K))
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.05)
        x = torch.randn(1, T, H, device=gpu_device).to(dtype)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            layer(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layer(x)
        for i in range(4):
            x.copy_(torch.randn(1, T, H, device=gpu_device).to(dtype))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, layer(x)), i
            torch.cuda.synchronize()
