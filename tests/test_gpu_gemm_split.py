"""Products of few tiles and a deep reduction, which the layer cuts into parts, against the oracle in float64: reductions that
no part divides evenly and with a half K tile at the end, ragged columns, every epilogue and activation, the shared expert,
an expert without rows.  Tolerances are the layer's."""
import pytest
import torch
import torch.nn.functional as F

from oracle import moe_oracle as O
from test_gpu_layer import TOL, build_layer, check_against_oracle, run_layer

pytestmark = pytest.mark.gpu

# T, H, E, K, I: gate_up and the gated backward reduce over H, down over I, the last data gradient over 2 I.
# Which of gate_up, down, gated backward and gate_up's gradient are cut is told by `cut`.
CASES = {
    "all": (150, 2080, 4, 2, 1568, F.silu, (1, 1, 1, 1)),
    "deep_intermediate": (130, 96, 3, 2, 4128, F.gelu, (0, 1, 0, 1)),
    "wide_model": (700, 4128, 2, 2, 160, lambda x: x * torch.sigmoid(1.702 * x), (1, 0, 1, 0)),
    "starved": (130, 1056, 5, 2, 2080, F.silu, (0, 1, 1, 1)),
}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", list(CASES))
def test_parts_of_a_reduction(gpu_device, name, dtype):
    T, H, E, K, I, act, cut = CASES[name]
    print("split products", name, dtype, flush=True)
    extra = dict(bias_hot=0.55, n_hot=1, n_dead=2) if name == "starved" else {}
    x, wr, wgu, wd, dy = O.make_inputs(T, H, E, K, I, dtype, seed=31, **extra)
    layer = build_layer(dtype, H, E, K, I, gpu_device, act=act)
    got = run_layer(layer, x, wr, wgu, wd, dy, gpu_device)
    again = run_layer(layer, x, wr, wgu, wd, dy, gpu_device)
    for k in ("y", "dx", "d_router_gate", "d_expert_gate_up", "d_expert_down"):
        assert torch.equal(got[k], again[k]), k
    with torch.no_grad():
        assert torch.equal(layer(x.to(gpu_device)).cpu(), got["y"])
    name_of = {F.silu: "silu", F.gelu: "gelu"}.get(act, "gpt_oss")
    ocfg = O.OracleConfig(model_dim=H, intermediate_dim=I, num_experts=E, top_k=K, loss_coeff=0.001, act=name_of)
    check_against_oracle(got, x, wr, wgu, wd, dy, ocfg, dtype)


@pytest.mark.parametrize("T", [65, 300])
def test_shared_expert_in_parts(gpu_device, T):
    """(its products have one expert and T rows: cut also where the experts' are not)"""
    from test_gpu_layer import test_layer_shared_expert

    test_layer_shared_expert(gpu_device, torch.bfloat16, T, 1056, 64, 4, 1568, "silu")


@pytest.mark.parametrize("name", list(CASES))
def test_the_cases_are_cut(gpu_device, name):
    """The rule, by the room that the layer's scratch has for the parts."""
    from arctictraining_amd import moe

    T, H, E, K, I, _, cut = CASES[name]
    for keep, which, whole, (n0, n1) in ((False, 1, T * K * H * 2, (2 * I, H)), (True, 2, T * K * (2 * I + H) * 2, (I, H))):
        room = moe._layer_sizes((E, K, H, I, 0, 1, True, 0, False), T, keep)[which] - whole
        flags = cut[:2] if which == 1 else cut[2:]
        need = max([2 * T * K * n * 4 for n, f in zip((n0, n1), flags) if f], default=0)
        assert room >= need
