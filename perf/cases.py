"""The work that a user of the expert layer has it do, as cases that can be timed and compared.

Five kinds, each through the public entry points of the package:
  forward   ArcticMoE under no_grad: decoding, prefill, evaluation
  train     ArcticMoE forward and backward: the output and every gradient
  experts   the grouped expert FFN, forward and backward, on rows that arrive already assigned to the
            experts (one expert-parallel rank's share)
  import    filling an ArcticMoE from the original block's per-expert nn.Linear weights
  export    the inverse, for a checkpoint in the original format

A case is a dict of plain values: kind, dtype, tokens (routed rows for `experts`), hidden, experts, top_k,
inter, and the options act, normalize, shared (a shared expert), skew (a few experts take about half of the
rows, some take none).
"""
import math

import numpy as np
import torch
import torch.nn.functional as F

from arctictraining_amd import ArcticMoE, MoEConfig, ops
from arctictraining_amd.remap import fill_arctic_moe_from_orig_mlp, fill_orig_mlp_from_arctic_moe

_DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}
_ACTS = {"silu": F.silu, "gelu": F.gelu, "gpt_oss": lambda x: x * torch.sigmoid(x * 1.702)}
_LOSS_COEFF = 0.001
_ZIPF = 1.2


def _case(kind, dtype, tokens, hidden, experts, top_k, inter, **options):
    c = dict(kind=kind, dtype=dtype, tokens=tokens, hidden=hidden, experts=experts, top_k=top_k, inter=inter,
             act="silu", normalize=True, shared=False, skew=False)
    c.update(options)
    return c


def listed():
    wide = dict(hidden=2048, experts=128, top_k=8, inter=768)    # many small experts: the headline layer shape
    hot = dict(hidden=2048, experts=64, top_k=4, inter=1408)
    cases = {
        # one sequence decoded token by token: eight experts' weights are all there is to read
        "decode_1": _case("forward", "bfloat16", 1, **wide),
        # a decoding batch: nearly every expert gets a handful of rows
        "decode_64": _case("forward", "bfloat16", 64, **wide),
        # a prompt (or an evaluation batch) of an odd length
        "prefill_3001": _case("forward", "bfloat16", 3001, **wide),
        # a short packed batch, a few dozen rows an expert: weights and their gradients dominate
        "train_509": _case("train", "bfloat16", 509, **wide),
        # the headline training step
        "train_16k_e128": _case("train", "bfloat16", 16384, **wide),
        # few wide experts: the largest matrix products
        "train_8k_e8": _case("train", "bfloat16", 8192, 4096, 8, 2, 14336),
        # a router that has not balanced yet
        "train_32k_skew": _case("train", "bfloat16", 32768, skew=True, **hot),
        # the full-precision layer
        "train_2k_f32": _case("train", "float32", 2048, 512, 8, 2, 1024),
        # half precision, a shared expert, scores as the softmax left them, an odd token count
        "train_4001_f16_shared": _case("train", "float16", 4001, shared=True, normalize=False, **hot),
        # one expert-parallel rank of a wide layer: rows come in grouped, loads follow a Zipf law
        "experts_64k": _case("experts", "bfloat16", 65536, 7168, 32, 1, 2048),
        # loading and saving one layer in the original checkpoint format
        "import_e128": _case("import", "bfloat16", 0, **wide),
        "export_e128": _case("export", "bfloat16", 0, **wide),
    }
    return [dict(c, name=n) for n, c in cases.items()]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(("forward", "train", "experts", "import", "export"), (35, 42, 9, 7, 7))[0]
    dtype = rng.choices(("bfloat16", "float16", "float32"), (70, 15, 15))[0]
    if kind == "experts" and dtype == "float32":
        dtype = "bfloat16"   # the fused backward of grouped rows is a 16-bit entry point
    f32 = dtype == "float32"
    while True:
        experts = _log_uniform(rng, 4, 256)
        top_k = rng.randint(1, min(8, experts))
        hidden = 32 * _log_uniform(rng, 8, 32 if f32 else 224)
        inter = 32 * _log_uniform(rng, 4, 64 if f32 else 448)
        tokens = _log_uniform(rng, 1 if kind == "forward" else 64, 4096 if f32 else 32768)
        c = _case(kind, dtype, tokens, hidden, experts, top_k, inter, act=rng.choice(("silu", "silu", "gelu", "gpt_oss")),
                  normalize=rng.random() < 0.7)
        if kind in ("forward", "train"):
            c["shared"] = rng.random() < 0.2
            c["skew"] = experts >= 16 and tokens >= 1024 and rng.random() < 0.25
        elif kind == "experts":
            c["tokens"], c["top_k"] = tokens * top_k, 1
        else:
            c.update(tokens=0, top_k=min(top_k, experts), act="silu", normalize=True)
        weights = 3 * experts * hidden * inter
        rows = c["tokens"] * c["top_k"]
        if not 2e6 <= weights <= (1e8 if f32 else 1.2e9):
            continue
        if work(c)["flops"] > (4e11 if f32 else 1.5e13) or rows > 262144 or rows * max(hidden, 2 * inter) > 1.2e9:
            continue
        return c


# ---------------------------------------------------------------------------------------------- states
class _Linear(torch.nn.Module):
    """The part of nn.Linear that a checkpoint holds: weight [out, in]."""

    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)


class _Expert(torch.nn.Module):
    def __init__(self, gate, up, down):
        super().__init__()
        self.gate_proj, self.up_proj, self.down_proj = _Linear(gate), _Linear(up), _Linear(down)


class _OrigBlock(torch.nn.Module):
    """An MoE block as the original model holds it: a router and a ModuleList of per-expert MLPs."""

    def __init__(self, router, gate, up, down):
        super().__init__()
        self.gate = _Linear(router)
        self.experts = torch.nn.ModuleList(_Expert(*w) for w in zip(gate, up, down))


def _layer(case, device):
    cfg = MoEConfig(
        act_fn=_ACTS[case["act"]], input_dtype=_DTYPES[case["dtype"]], intermediate_dim=case["inter"], model_dim=case["hidden"],
        normalize_topk_scores=case["normalize"], num_experts=case["experts"], top_k=case["top_k"], loss_coeff=_LOSS_COEFF,
        use_shared_expert=case["shared"],
    )
    with torch.device(device):
        return ArcticMoE(cfg)


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    dtype = _DTYPES[case["dtype"]]
    g = torch.Generator(device).manual_seed(seed)
    kind, T, H, E, K, I = (case[k] for k in ("kind", "tokens", "hidden", "experts", "top_k", "inter"))

    def normal(*shape, std=1.0):
        return torch.empty(shape, dtype=dtype, device=device).normal_(0.0, std, generator=g)

    def weight(*shape):
        return normal(*shape, std=0.02)

    state = dict(kind=kind)
    if kind == "experts":
        p = np.arange(1, E + 1, dtype=np.float64) ** -_ZIPF
        counts = np.random.Generator(np.random.PCG64(seed)).multinomial(T, p / p.sum())
        offsets = torch.from_numpy(np.concatenate([[0], counts.cumsum()]).astype(np.int32)).to(device)
        state.update(
            x=normal(T, H), dy=normal(T, H), gate_up=weight(E, H, 2 * I), down=weight(E, I, H), offsets=offsets,
            scores=torch.empty(T, device=device).uniform_(generator=g), act=("silu", "gelu", "relu", "gpt_oss").index(case["act"]),
            row_of=torch.arange(T, dtype=torch.int32, device=device).view(T, 1),
        )
        return state
    layer = state["layer"] = _layer(case, device)
    with torch.no_grad():
        for p in layer.parameters():
            p.normal_(0.0, 0.02, generator=g)
    if kind in ("import", "export"):
        if kind == "import":   # a checkpoint's tensors: each weight in memory of its own
            of_experts = [[weight(*shape) for _ in range(E)] for shape in ((I, H), (I, H), (H, I))]
            state["block"] = _OrigBlock(weight(E, H), *of_experts)
        else:                  # a block about to be saved: the weights of its experts sit side by side
            state["saved"] = [torch.empty(shape, dtype=dtype, device=device) for shape in ((E, H), (E, I, H), (E, I, H), (E, H, I))]
            state["block"] = _OrigBlock(*state["saved"])
        state["device"] = device
        return state
    x = normal(1, T, H)
    if case["skew"]:
        # a constant input channel biases the router: a sixteenth of the experts is hot, an eighth is never chosen
        with torch.no_grad():
            x[..., H - 1] = 1.0
            layer.router_gate[:, H - 1] = 0.0
            layer.router_gate[: E // 16, H - 1] = 1.6
            layer.router_gate[E - E // 8:, H - 1] = -1.0e4
    state["x"] = x
    if kind == "train":
        x.requires_grad_(True)
        state["dy"] = normal(1, T, H)
    return state


# ---------------------------------------------------------------------------------------------- one pass
def _experts_step(s):
    R, E = s["x"].shape[0], s["gate_up"].shape[0]
    ws = ops.gemm_workspace(R, E, s["x"].device)
    gate_up, inter = ops.grouped_gemm_gateup_act_fwd(s["x"], s["gate_up"], s["offsets"], s["act"], row_scale=s["scores"], workspace=ws)
    y = ops.grouped_gemm_nn(inter, s["down"], s["offsets"], workspace=ws, map_ready=True)
    d_gate_up, parts = ops.grouped_gemm_nt_gated_bwd(s["dy"], s["down"], s["offsets"], gate_up, s["act"], row_scale=s["scores"],
                                                     workspace=ws, map_ready=True)
    d_scores = ops.score_grad_gather(parts, s["row_of"])
    d_down = ops.grouped_gemm_wgrad(inter, s["dy"], s["offsets"], E)
    d_w_gate_up = ops.grouped_gemm_wgrad(s["x"], d_gate_up, s["offsets"], E)
    dx = ops.grouped_gemm_nt(d_gate_up, s["gate_up"], s["offsets"], workspace=ws, map_ready=True)
    return dict(y=y, dx=dx, d_gate_up=d_w_gate_up, d_down=d_down, d_scores=d_scores)


def run(state):
    kind = state["kind"]
    if kind == "forward":
        with torch.no_grad():
            return state["layer"](state["x"])
    if kind == "train":
        layer, x = state["layer"], state["x"]
        layer.zero_grad(set_to_none=True)
        x.grad = None
        y = layer(x)
        y.backward(state["dy"])
        out = {name: p.grad for name, p in layer.named_parameters()}
        out.update(y=y.detach(), dx=x.grad)
        return out
    if kind == "experts":
        return _experts_step(state)
    layer, block = state["layer"], state["block"]
    if kind == "import":
        fill_arctic_moe_from_orig_mlp(layer, block, state["device"])
        return [layer.router_gate.detach(), layer.expert_gate_up.detach(), layer.expert_down.detach()]
    fill_orig_mlp_from_arctic_moe(block, layer)
    return state["saved"]


# ---------------------------------------------------------------------------------------------- what a pass is worth
def work(case):
    kind, T, H, E, K, I = (case[k] for k in ("kind", "tokens", "hidden", "experts", "top_k", "inter"))
    size = 4 if case["dtype"] == "float32" else 2
    ffn = 3 * H * I                                   # weights of one expert
    if kind in ("import", "export"):
        return dict(bytes=2.0 * size * E * (ffn + H), flops=0.0)
    rows = T * K
    extra = 1 if case["shared"] else 0
    router = 0 if kind == "experts" else E * H
    if kind == "forward":
        met = E * (1.0 - (1.0 - K / E) ** T)          # experts that get a row
        return dict(bytes=float(size) * ((met + extra) * ffn + router + 2 * T * H),
                    flops=2.0 * (rows + extra * T) * ffn + 2.0 * T * router)
    weights = (E + extra) * ffn + router
    return dict(bytes=float(size) * (2 * weights + 4 * T * H), flops=6.0 * (rows + extra * T) * ffn + 6.0 * T * router)


def tolerance(case):
    if case["kind"] in ("import", "export"):
        return "exact"
    return {"rel": {"bfloat16": 1e-2, "float16": 2e-3, "float32": 1e-5}[case["dtype"]]}
