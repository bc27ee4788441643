"""What the layer refuses before an address reaches the library (the kernels trust the shapes they are told)."""
import ctypes

import pytest
import torch
import torch.nn.functional as F

from arctictraining_amd import ArcticMoE, MoEConfig, _lib, moe, ops

T, H, E, K = 8, 32, 4, 2


class _Library:
    """Stands where the native library does: every entry point succeeds and notes that it was reached."""

    def __init__(self):
        self.reached = []

    def __getattr__(self, name):
        return lambda *a: self.reached.append(name) or 0


@pytest.fixture
def on_host(monkeypatch):
    """The layer on CPU tensors: its input, the logits and the incoming gradient pass for GPU tensors, the library is a stub."""
    lib = _Library()
    check = ops._chk
    monkeypatch.setattr(ops, "_chk", lambda t, name, *a, **k: t if name in ("x", "logits", "dy") else check(t, name, *a, **k))
    monkeypatch.setattr(ops, "_stream", lambda: 0)
    monkeypatch.setattr(_lib, "load", lambda: lib)
    monkeypatch.setattr(moe, "_layer_sizes", lambda *a: (4096,) * 13)
    return lib


def _layer(gated=True, **options):
    layer = ArcticMoE(MoEConfig(act_fn=F.silu, input_dtype=torch.float32, intermediate_dim=32, model_dim=H, normalize_topk_scores=True,
                                num_experts=E, top_k=K, is_gated=gated, **options))
    with torch.no_grad():
        for p in layer.parameters():
            p.zero_()
    return layer


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("shape", [(T, K), (T - 1, K), (T, K - 1), (T, K + 1), (1, T, K), (T * K,)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_replayed_assignments(on_host, gated, shape, dtype):
    """A tensor in host memory and one of another shape than [tokens, top_k] end in an error, checked ids or not."""
    layer = _layer(gated, enable_routing_replay=True)
    for layer.check_replay in (True, False):
        with torch.no_grad(), pytest.raises(RuntimeError, match="routing_replay_assignments"):
            layer(torch.zeros(T, H), torch.zeros(shape, dtype=dtype))
    assert "amoe_layer_fwd" not in on_host.reached


@pytest.mark.parametrize("gated", [True, False])
def test_router_of_more_experts_than_the_layer_has(on_host, gated):
    """Its logits would choose experts that have no weights."""
    layer = _layer(gated)
    layer.router_gate = torch.nn.Parameter(torch.zeros(E + 1, H))
    with torch.no_grad(), pytest.raises(RuntimeError, match="router_gate"):
        layer(torch.zeros(T, H))
    assert not on_host.reached


def test_router_of_fewer_experts(on_host, monkeypatch):
    """The kernels read logits [tokens, experts]: the experts that the router leaves out get -inf, a probability of 0."""
    layer = _layer()
    layer.router_gate = torch.nn.Parameter(torch.ones(E - 1, H))
    seen = {}

    def forward(config, tokens, x, logits, *rest):
        seen["logits"] = torch.frombuffer((ctypes.c_float * (tokens * E)).from_address(logits), dtype=torch.float32).clone()
        return 0

    monkeypatch.setattr(on_host, "amoe_layer_fwd", forward, raising=False)
    with torch.no_grad():
        layer(torch.ones(T, H))
    want = torch.full((T, E), float("-inf"))
    want[:, : E - 1] = H
    assert torch.equal(seen["logits"].view(T, E), want)


@pytest.mark.parametrize("unpack", [lambda t: t.half(), lambda t: t[..., :-1], lambda t: t.transpose(0, -1)],
                         ids=["type", "shape", "strides"])
@pytest.mark.parametrize("which", range(6))
def test_saved_tensors_come_back_as_they_were(on_host, unpack, which):
    """Backward reads what the unpack hook returns: another type, shape or layout ends in an error."""
    layer = _layer(use_shared_expert=True)
    layer.overlap_weight_grads = False
    saved = [None, layer.expert_gate_up, layer.expert_down, layer.shared_expert_gate_up, layer.shared_expert_down,
             layer.shared_expert_output_gate][which]
    x = torch.zeros(T, H, requires_grad=True)
    planted = []

    def hook(t):
        if t.shape == (x if which == 0 else saved).shape:
            planted.append(unpack(t))
            return planted[-1]
        return t

    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, hook):
        y = layer(x)
    ops_reached = len(on_host.reached)
    with pytest.raises(RuntimeError, match="must"):
        y.sum().backward()
    assert planted and len(on_host.reached) == ops_reached


@pytest.mark.parametrize("dual", ["x", "expert_down"])
def test_forward_mode_without_gradients(monkeypatch, dual):
    """The layer has no forward-mode derivative: a tangent ends in an error also where gradients are switched off, and is
    not dropped.  An open dual level without a tangent changes nothing."""
    import torch.autograd.forward_ad as fwAD

    layer = _layer()
    key = (E, K, H, 32, 0, 0, True, 0, False)
    monkeypatch.setattr(moe, "_layer_forward", lambda x, *a, **k: (x + 1, torch.zeros(64, dtype=torch.uint8), key))
    x = torch.zeros(T, H)
    with torch.no_grad(), fwAD.dual_level():
        assert torch.equal(layer(x), x + 1)
        if dual == "x":
            x = fwAD.make_dual(x, torch.ones(T, H))
        else:
            tangent = fwAD.make_dual(layer.expert_down.detach(), torch.ones_like(layer.expert_down))
            del layer.expert_down
            layer.expert_down = tangent
        with pytest.raises(NotImplementedError, match="jvp"):
            layer(x)
    with torch.no_grad():
        assert torch.equal(layer(torch.zeros(T, H)), torch.ones(T, H))
