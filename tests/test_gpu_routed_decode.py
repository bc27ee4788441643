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
    "limits": (8, 544, 256, 16, 96),          # the most rows and experts
    "full_width": (7, 4096, 64, 6, 1056),     # 128-column tiles, columns past the end
    "past_experts": (8, 64, 257, 2, 32),      # past the lines: the launches of their own on both sides
    "past_tokens": (9, 64, 64, 2, 32),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_same_as_with_launches_of_their_own(gpu_device, name, shared, dtype):
    from arctictraining_amd import ArcticMoE, MoEConfig

    T, H, E, K, I = CASES[name]
    print("few tokens", name, shared, dtype, flush=True)
    torch.manual_seed(T + H)
    with torch.device(gpu_device):
        layer = ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=dtype, intermediate_dim=I, model_dim=H, normalize_topk_scores=T != 7,
                                    num_experts=E, top_k=K, loss_coeff=0.001, use_shared_expert=shared))
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.05)
    x = torch.randn(1, T, H, device=gpu_device).to(dtype)
    if T > 2:
        x[0, 1] = x[0, 0]                     # two tokens that route alike
    dy = torch.randn(1, T, H, device=gpu_device).to(dtype)

    def run(replay=None, grad=True):
        layer.zero_grad(set_to_none=True)
        layer.capture = {}
        xi = x.clone().requires_grad_(grad)
        with torch.set_grad_enabled(grad):
            y = layer(xi) if replay is None else layer(xi, routing_replay_assignments=replay)
        out = dict(y=y.detach().clone(), **{k: v.clone() for k, v in layer.capture.items() if torch.is_tensor(v)})
        if grad:
            y.backward(dy)
            out.update({n: p.grad.clone() for n, p in layer.named_parameters()}, dx=xi.grad.clone())
        return out

    own = run()
    for grad in (True, False):
        got, want = run(grad=grad), run(own["topk_idx"], grad=grad)
        assert got.keys() == want.keys()
        for k in want:
            assert torch.equal(got[k], want[k]), (k, grad)
    again = run(grad=False)                   # (who arrives last does not matter)
    assert torch.equal(again["y"], own["y"])


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
