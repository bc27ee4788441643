"""MI355X-native ArcticMoE layer: the reference's module surface
(arctic_training/model/moe/moe.py:33-51 `MoEConfig`, :63-323 `ArcticMoE`) over hand-written
HIP kernels reached through the C ABI of libarctic_moe_hip.so.

Same constructor argument, parameter names / shapes / layouts (they are checkpoint keys,
arctic_training/model/moe/utils.py:563-566), forward signature and return type as the
reference, so the trainer's `layer.mlp = ArcticMoE(config)` (utils.py:320) works unchanged.
The whole routed-expert computation of a gated layer is one torch.autograd.Function: forward is one
native call, backward three at most, over one saved and one scratch buffer; a layer without a gate calls the
kernels stage by stage.  Neither synchronises with the host.
"""
import contextlib
import ctypes
import functools
import math
import time
from collections import OrderedDict, defaultdict
from dataclasses import dataclass
from typing import Any, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad

from . import _lib, ops


@dataclass(kw_only=True)
class MoEConfig:
    """Field for field the reference's MoEConfig (moe.py:33-51)."""

    act_fn: object
    ep_group: Any = None
    ep_size: int = 1
    ep_rank: int = 0
    input_dtype: torch.dtype
    intermediate_dim: int
    is_gated: bool = True
    loss_coeff: float = 0.01
    model_dim: int
    normalize_topk_scores: bool
    num_experts: int
    return_router_scores: bool = False
    top_k: int
    use_triton: bool = True  # accepted for compatibility; the HIP kernels are always used
    use_shared_expert: bool = False
    # accepted for compatibility and IGNORED: the reference's capacity-padded custom-kernel path (moe.py:140-149,
    # 413-448) differs from its default path by design (atomic row order, no load-balance gradient, scores
    # normalised inside the gather); this layer always computes the default path and warns once when the flag is set
    use_custom_moe_kernel: bool = False
    enable_routing_replay: bool = False


def classify_activation(act_fn) -> int:
    """Map the callable the reference config carries (utils.py:118-127) to the kernel's
    activation code by evaluating it on a few points."""
    if isinstance(act_fn, int):
        return act_fn
    if isinstance(act_fn, str):
        return {"silu": ops.ACT_SILU, "gelu": ops.ACT_GELU, "relu": ops.ACT_RELU, "gpt_oss": ops.ACT_GPT_OSS}[act_fn]
    probe = torch.tensor([-2.0, -0.5, 0.3, 1.7], dtype=torch.float32, device="cpu")  # also under a meta-device context
    got = act_fn(probe)
    candidates = {
        ops.ACT_SILU: F.silu(probe),
        ops.ACT_GELU: F.gelu(probe),
        ops.ACT_RELU: F.relu(probe),
        ops.ACT_GPT_OSS: probe * torch.sigmoid(probe * 1.702),
    }
    for code, ref in candidates.items():
        if torch.allclose(got, ref, atol=1e-6):
            return code
    raise ValueError("unsupported activation: expected silu, gelu, relu or x*sigmoid(1.702x)")


class PhaseTimers:
    """The attributes of the reference's SynchronizedWallClockTimerSimple that its callers
    touch (arctic_training/model/moe/timers.py:44-72): start/stop/elapsed, `times`,
    `token_counts`, and the `wall_clock_breakdown` switch.  A no-op unless switched on."""

    def __init__(self, wall_clock_breakdown: bool = False):
        self.wall_clock_breakdown = wall_clock_breakdown
        self.times = defaultdict(float)
        self.token_counts = defaultdict(int)
        self._t0 = {}

    def start(self, name):
        if self.wall_clock_breakdown:
            torch.cuda.synchronize()
            self._t0[name] = time.perf_counter()

    def stop(self, name):
        if self.wall_clock_breakdown:
            torch.cuda.synchronize()
            self.times[name] = (time.perf_counter() - self._t0.pop(name, time.perf_counter())) * 1000.0
        else:
            self.times[name] = 0

    def skip(self, names):
        """What start and stop of each leave behind while switched off."""
        for name in names:
            self.times[name] = 0

    def elapsed(self, name):
        return self.times[name]


class _SmallTensorCache:
    """A few small index tensors keyed by (size, kind, device), least recently used evicted first:
    the token count changes from step to step with packed variable-length batches, so the cache
    must not grow with the number of distinct sizes seen.  Nothing is stored while a HIP graph is
    being captured (a tensor created there lives in the graph's private pool and only holds its
    values after a replay)."""

    def __init__(self, max_entries: int = 8):
        self.max_entries = max_entries
        self._d = OrderedDict()

    def get(self, key, make):
        t = self._d.get(key)
        if t is not None:
            self._d.move_to_end(key)
            return t
        t = make()
        if not (t.is_cuda and torch.cuda.is_current_stream_capturing()):
            self._d[key] = t
            while len(self._d) > self.max_entries:
                self._d.popitem(last=False)
        return t

    def __len__(self):
        return len(self._d)


_INDEX_CACHE = _SmallTensorCache()


_side_streams: dict = {}


def _side_stream(device) -> "torch.cuda.Stream":
    """One extra stream per device (default priority) for the expert weight gradients of the
    backward pass: they feed nothing else in the layer, and every grouped GEMM here is one
    workgroup per compute unit that ends with part of the chip idle -- launched from a second
    stream, the next kernel's workgroups start on the compute units as the previous kernel's leave."""
    idx = device.index if device.index is not None else torch.cuda.current_device()
    st = _side_streams.get(idx)
    if st is None:
        st = _side_streams[idx] = torch.cuda.Stream(device=idx)
    return st


def _token_offsets(T: int, parts: int, device) -> torch.Tensor:
    """int32 [parts + 1]: the T tokens cut into `parts` nearly equal consecutive chunks."""
    return _INDEX_CACHE.get(
        (T, parts, str(device)),
        lambda: (torch.arange(parts + 1, dtype=torch.int64, device=device) * T // parts).to(torch.int32),
    )


def _dense_splits(T: int, Kd: int, N: int, dtype, tile: int = 256) -> int:
    """Chunks of the tokens for the weight gradient [Kd,N] of a dense (not routed) linear map."""
    tiles = -(-Kd // tile) * -(-N // tile)
    return max(1, min(16, 512 // tiles, T // 256)) if dtype != torch.float32 else 1


def _dense_weight_grad(a: torch.Tensor, b: torch.Tensor, tile_cfg: int = 0, tile: int = 256) -> torch.Tensor:
    """C [Kd,N] = a^T [Kd,T] @ b [T,N]: the weight gradient of a dense (not routed) linear map.

    Few output tiles and a deep reduction over the tokens: run as a split-K on the grouped
    weight-gradient kernel -- the tokens are cut into chunks that play the role of experts,
    C[s] = a[chunk s]^T @ b[chunk s].  The kernel accumulates each partial product in float32 and
    stores it in the operands' 16-bit type; the (at most 16) partials are then added in float32
    and the sum is rounded once more."""
    splits = _dense_splits(a.shape[0], a.shape[1], b.shape[1], a.dtype, tile)
    return ops.dense_wgrad(a, b, _token_offsets(a.shape[0], splits, a.device), tile_cfg=tile_cfg)


# The router's products on the package's kernels, up to this many (16 x 16 tiles of logits) * H: a pass with so few tokens
# (256 at 128 experts and H = 2048) is usually bound by the host, and a call of torch.matmul costs it 19 us against 8 us of
# a launch of the kernels, which take about as long on the GPU (logits, then input gradient, against the library: 128
# experts, H = 2048, 200 tokens 6.0 / 5.7 us, 4.9 / 4.4, at 1024 tokens 9.8 / 6.5, 8.1 / 5.6; 64 experts, H = 512, 2048
# tokens 4.4 / 5.7, 5.2 / 4.3).
_ROUTER_KERNEL_WORK = 1 << 18


def _router_kernel_fits(a: torch.Tensor, w: torch.Tensor) -> bool:
    """Whether a product of a [T, .] with the router's weight w [E,H] may run on the package's kernels: few tokens, both
    dense (a: its rows), of one 16-bit type, on one device, aligned, and no autocast that would change a type."""
    return (
        -(-a.shape[0] // 16) * -(-w.shape[0] // 16) * w.shape[1] <= _ROUTER_KERNEL_WORK
        and a.dtype in (torch.bfloat16, torch.float16)
        and w.dtype is a.dtype
        and a.stride(1) == 1
        and w.is_contiguous()
        and w.get_device() == a.get_device()
        and (a.data_ptr() | w.data_ptr()) % 16 == 0
        and not torch.is_autocast_enabled("cuda")
    )


def _router_logits(x: torch.Tensor, router_gate: torch.Tensor) -> torch.Tensor:
    """x [T,H] @ router_gate [E,H]^T (moe.py:233)."""
    # (longer rows are more than 12 steps in a row for a wavefront of the kernel: 64 tokens, H = 7168 11.8 us against 7.5,
    # H = 5728 7.5 against 13.0)
    if _router_logits_fit(x, router_gate):
        return ops.router_logits(x, router_gate)
    return torch.matmul(x, router_gate.t())


def _router_logits_fit(x: torch.Tensor, router_gate: torch.Tensor) -> bool:
    return (
        x.shape[1] == router_gate.shape[1] <= 6144
        and x.shape[1] % 32 == 0
        and x.is_contiguous()
        and _router_kernel_fits(x, router_gate)
    )


def _fit_logits(logits: torch.Tensor, opts, pad: bool = True) -> torch.Tensor:
    """The logits of a router_gate that has not one row for each of the layer's experts, as the kernels read them: [T,E],
    an expert that the router leaves out with a probability of 0 (not padded for the stages, which take E from them)."""
    n, E, K = logits.shape[1], opts["num_experts"], opts["top_k"]
    if n > E:   # (their counts, weights and gradients do not exist)
        raise RuntimeError(f"router_gate must have one row for each of at most {E} experts, got {n}")
    if n < K:
        raise RuntimeError(f"router_gate must have at least top_k = {K} rows, got {n}")
    return F.pad(logits, (0, E - n), value=float("-inf")) if pad else logits


def _router_input_grad(d_logits: torch.Tensor, router_gate: torch.Tensor, padded: bool = False) -> torch.Tensor:
    """d_logits [T,E] @ router_gate [E,H] (autograd of moe.py:233).  padded: the rows of d_logits are a multiple of 32 elements
    apart, with zeros between them."""
    E, H = router_gate.shape
    if (padded or (E % 32 == 0 and d_logits.is_contiguous())) and H % 8 == 0 and _router_kernel_fits(d_logits, router_gate):
        return ops.router_input_grad(d_logits, router_gate)
    return torch.matmul(d_logits, router_gate)


def _router_weight_grad(d_logits: torch.Tensor, x: torch.Tensor) -> torch.Tensor:
    """dW_router [E,H] = d_logits^T [E,T] @ x [T,H] (autograd of moe.py:233), where the layer's native call does not form it:
    experts without a gate, a router in another type or of fewer rows than experts, float32.  Skinny (E rows) and deep (T), so
    that the library GEMM leaves most of the chip idle on it (128 experts, H = 2048: 4096 tokens 35 us against 17, 16384 tokens 135
    against 21, the sum of the parts included)."""
    if x.dtype == torch.float32 or d_logits.shape[1] % 8:
        return torch.matmul(d_logits.t(), x)
    return _dense_weight_grad(d_logits, x, tile_cfg=1, tile=128)  # 128x128 tiles


def _replayed(replay, T: int, opts) -> torch.Tensor:
    """The replayed assignments as int32 [T,K] on the current device: the kernels read them at that shape."""
    E, K = opts["num_experts"], opts["top_k"]
    if tuple(replay.shape) != (T, K):
        raise RuntimeError(f"routing_replay_assignments must be [{T}, {K}] (tokens, top_k), got {list(replay.shape)}")
    ops._chk(replay, "routing_replay_assignments", contiguous=False)
    assign = replay.to(torch.int32).contiguous()
    if opts.get("check_replay", True) and not torch.cuda.is_current_stream_capturing():
        # The reference's one_hot(..., num_classes=E) raises on an expert id outside [0, E)
        # (moe.py:374).  The same error here, at the price of one host synchronisation per replayed
        # forward; `ArcticMoE.check_replay = False` (and a HIP graph capture, which cannot
        # synchronise) skips it, the permutation kernels then clamp such ids for memory safety.
        bad = ((assign < 0) | (assign >= E)).any()
        if bool(bad):
            raise RuntimeError(f"routing_replay_assignments holds expert ids outside [0, {E})")
    return assign


def _route(x, router_gate, replay, opts):
    """Router linear map, softmax / top-k, and the permutation plan with the tile map of the
    row-grouped GEMMs (moe.py:231-233, 359-382).  Returns logits, probs, topk_idx, scores [T,K],
    the GEMM workspace that holds the tile map, and the plan (counts, offsets, token_of, slot_of,
    row_of, scores_perm)."""
    T = x.shape[0]
    E, K = opts["num_experts"], opts["top_k"]
    timers: PhaseTimers = opts["timers"]
    timers.start("router")
    logits = _fit_logits(_router_logits(x, router_gate), opts, pad=False)
    probs, topk_idx, scores = ops.router_topk_fwd(logits, K, opts["normalize"])
    assign = topk_idx if replay is None else _replayed(replay, T, opts)
    # the row-grouped GEMMs of a step share one tile map: the permutation plan builds it (its
    # scan kernel holds the offsets), the workspace is kept for backward
    ws = ops.gemm_workspace(T * K, E, x.device)
    plan = ops.permute_plan(assign, E, scores, gemm_workspace=ws, gemm_dtype=x.dtype, tile_cfg=opts["tile_cfg"])
    timers.stop("router")
    return logits, probs, topk_idx, scores, ws, plan


@functools.lru_cache(maxsize=64)
def _layer_config(E, K, H, I, act, dtype, normalize, tile_cfg, shared):
    return (ctypes.c_int32 * 9)(E, K, H, I, act, dtype, normalize, tile_cfg, shared)


# byte offsets and element counts inside the saved buffer, in the order the library lists them
_SAVED_FIELDS = ("probs", "scores", "scores_perm", "topk_idx", "counts", "offsets", "token_of", "slot_of", "row_of")


@functools.lru_cache(maxsize=256)
def _layer_sizes(config_key, T: int, keep: bool):
    out = (ctypes.c_longlong * (4 + len(_SAVED_FIELDS)))()
    _lib.check(_lib.load().amoe_layer_sizes(_layer_config(*config_key), T, int(keep), out), "amoe_layer_sizes")
    return tuple(out)


def _saved_view(saved, name, config_key, T: int):
    """One of _SAVED_FIELDS as a tensor over the saved buffer."""
    E, K = config_key[:2]
    shape = {"probs": (T, E), "scores": (T, K), "topk_idx": (T, K), "counts": (E,), "offsets": (E + 1,), "row_of": (T, K)}.get(name, (T * K,))
    dtype = torch.float32 if name in ("probs", "scores", "scores_perm") else torch.int32
    start = _layer_sizes(config_key, T, True)[3 + _SAVED_FIELDS.index(name)]
    return saved[start : start + 4 * math.prod(shape)].view(dtype).view(shape)


@functools.lru_cache(maxsize=256)
def _overlap_pays(config_key, T: int) -> bool:
    """Whether the expert weight gradients go on the second stream.  The events that order the streams cost the host 40-60 us a
    step; a step that the GPU takes less time for than the host is longer by that much (20 of 60 steps drawn over the sizes of
    this layer: 12-39 %), one that it takes longer for is mostly 3-15 % shorter with the second stream.  The line lies where
    the products at 800 TFLOP/s (float32 100), their columns rounded up to whole tiles, and the weights, read twice and their
    gradients written, at 3 TB/s make 150 us: T=556 H=1760 E=8 K=6 I=672 (143 us) 250 us with it, 220 without; T=3065 H=320 E=19
    K=5 I=1088 (243) 268 and 283.  (Not all: T=95 H=2336 E=12 K=2 I=1536 (193), whose kernels have become faster than the host,
    takes 261 and 228; about 110 rows an expert of 128 experts of 2048 x 768, bound by memory on both streams, 3 % longer with it.)"""
    E, K, H, I, dtype, shared = *config_key[:4], config_key[5], config_key[8]
    size, rate = (4, 1e8) if dtype == ops.F32 else (2, 8e8)
    rows, weights = T * K + (T if shared else 0), (E + (1 if shared else 0)) * H * I
    padded = -(-H // 256) * 256 * -(-I // 128) * 128
    return 18.0 * rows * padded / rate + 6.0 * size * weights / 3e6 > 150.0


def _check_operand(t, name, like, shape) -> None:
    """t has to be dense, of `like`'s type, on the current device (like's), and of the given shape."""
    if t.dtype is not like.dtype or t.get_device() != like.get_device() or not t.is_contiguous():
        ops._chk(t, name, like.dtype)
    if t.shape != shape:
        raise RuntimeError(f"{name} must be {list(shape)}, got {list(t.shape)}")


def _layer_forward(x, router_gate, w_gate_up, w_down, shared, replay, opts, keep: bool):
    """Router linear map, then the whole layer in one native call (moe.py:231-233, 340-411, 176-193, 450-461).  Returns y,
    the buffer of what backward reads (keep) or of what a caller that only runs forward may look at, and the
    config key."""
    T, H = x.shape
    E, K = opts["num_experts"], opts["top_k"]
    ops._chk(x, "x")
    _check_operand(w_gate_up, "w_gate_up", x, (E, H, w_gate_up.shape[-1]))
    I = w_gate_up.shape[2] // 2
    _check_operand(w_down, "w_down", x, (E, I, H))
    sh_gate_up, sh_down, sh_out_gate = shared
    all_rows = None
    if sh_gate_up is not None:
        _check_operand(sh_gate_up, "shared_expert_gate_up", x, (H, 2 * I))
        _check_operand(sh_down, "shared_expert_down", x, (I, H))
        _check_operand(sh_out_gate, "shared_expert_output_gate", x, (H, 1))
        all_rows = _token_offsets(T, 1, x.device)
    timers: PhaseTimers = opts["timers"]
    key = (E, K, H, I, opts["act"], ops._dtype_code(x), opts["normalize"], opts["tile_cfg"], all_rows is not None)
    sizes = _layer_sizes(key, T, keep)
    if timers.wall_clock_breakdown:
        timers.start("router")
    # few tokens: the logits are formed inside the native call, behind its scratch; else the library's product
    native = router_gate.shape[0] == E and _router_logits_fit(x, router_gate)
    if not native:
        logits = routed = _router_logits(x, router_gate)
        if routed.shape != (T, E) or not routed.is_contiguous():
            logits = _fit_logits(routed, opts).contiguous()
    assign = None if replay is None else _replayed(replay, T, opts)
    y = torch.empty_like(x)
    extra = T * E * x.element_size() if native else 0
    buf = torch.empty(sizes[0] + (0 if keep else sizes[1] + extra), dtype=torch.uint8, device=x.device)
    base = buf.data_ptr()
    scratch = torch.empty(sizes[1] + extra, dtype=torch.uint8, device=x.device) if keep else None
    scratch_ptr = scratch.data_ptr() if keep else base + sizes[0]

    def run(stages):
        if native:
            call, routing = _lib.load().amoe_layer_fwd_router, (router_gate.data_ptr(), scratch_ptr + sizes[1])
        else:
            call, routing = _lib.load().amoe_layer_fwd, (logits.data_ptr(), ops._dtype_code(logits))
        _lib.check(
            call(
                _layer_config(*key), T, x.data_ptr(), *routing, ops._ptr(assign),
                w_gate_up.data_ptr(), w_down.data_ptr(), ops._ptr(sh_gate_up), ops._ptr(sh_down), ops._ptr(sh_out_gate),
                ops._ptr(all_rows), base, keep, scratch_ptr, y.data_ptr(), stages, ops._stream(),
            ),
            "amoe_layer_fwd",
        )

    if not timers.wall_clock_breakdown:
        run(_STAGE_ALL)
        timers.skip(_PHASES)
    else:
        for name, stage in zip(_PHASES, (1, 2, 4, 8)):
            if name != "router":
                if name == "shared-expert" and all_rows is None:
                    continue
                timers.start(name)
            run(stage)
            timers.stop(name)
    cap = opts.get("capture")
    if cap is not None:
        if native:
            at = sizes[1] if keep else sizes[0] + sizes[1]
            routed = (scratch if keep else buf)[at : at + extra].view(x.dtype).view(T, E).clone()
        cap.update(logits=routed, **{n: _saved_view(buf, n, key, T).clone() for n in _SAVED_FIELDS if n != "scores_perm"})
    return y, buf, key


_STAGE_ALL = 15
_PHASES = ("router", "groupGeMM", "shared-expert", "moe-combine")


class _ExpertLayerFn(torch.autograd.Function):
    """router top-k -> permutation -> grouped gated FFN -> weighted combine, and the
    gradients of all of it (the autograd of moe.py:231-233, 340-411, 176-193, 450-461 plus
    the load-balance hook :393-406).  A shared expert (moe.py:305-314) runs through the same
    kernels as one more expert that owns every token, the sigmoid of its output gate in the role of
    the routing score."""

    @staticmethod
    def forward(ctx, x, router_gate, w_gate_up, w_down, sh_gate_up, sh_down, sh_out_gate, replay, opts):
        y, saved, key = _layer_forward(
            x, router_gate, w_gate_up, w_down, (sh_gate_up, sh_down, sh_out_gate), replay, opts, keep=True
        )
        ctx.opts, ctx.key, ctx.device, ctx.tokens = opts, key, x.device, x.shape[0]
        ctx.save_for_backward(x, router_gate, w_gate_up, w_down, sh_gate_up, sh_down, sh_out_gate, saved)
        ctx.set_materialize_grads(False)  # no zero-filled gradient for an output the loss does not use
        if not opts["want_scores"]:
            return y
        # scores in routed-row order, in the model dtype, as the reference returns them (moe.py:323,
        # only when return_router_scores); they stay attached to the graph like the reference's
        return y, _saved_view(saved, "scores_perm", key, x.shape[0]).to(x.dtype, copy=True)

    @staticmethod
    def backward(ctx, dy, ds_perm=None):
        if dy is None and ds_perm is None:  # neither output took part in the loss
            return (None,) * 9
        # The two expert weight gradients run on a second stream beside the chain of data gradients.  It
        # starts on them behind everything the main stream has queued up to their operands, and the main
        # stream waits for it at the end, so the tensors either stream uses outlive the kernels that use them.
        overlap = ctx.opts["overlap_weight_grads"] and (ctx.needs_input_grad[2] or ctx.needs_input_grad[3])
        side = _side_stream(ctx.device) if overlap and _overlap_pays(ctx.key, ctx.tokens) else None
        try:
            return _ExpertLayerFn._backward(ctx, dy, ds_perm, None if side is None else side.cuda_stream)
        except BaseException:
            # (memory may run out between the fork and the join: what is freed here is used again on the main stream; of a
            # second stream without work the wait is nothing)
            if overlap:
                torch.cuda.current_stream(ctx.device).wait_stream(_side_stream(ctx.device))
            raise

    @staticmethod
    def _backward(ctx, dy, ds_perm, side):
        x, router_gate, w_gate_up, w_down, sh_gate_up, sh_down, sh_out_gate, saved = ctx.saved_tensors
        opts, key, T = ctx.opts, ctx.key, ctx.tokens
        E, K, H, I = key[:4]
        # (what a saved-tensor hook returned, read below at the shapes of the forward pass)
        if ops._dtype_code(ops._chk(x, "x")) != key[5] or x.shape != (T, H):
            raise RuntimeError(f"saved x must come back as the forward pass had it, got {x.dtype} {list(x.shape)}")
        _check_operand(w_gate_up, "saved w_gate_up", x, (E, H, 2 * I))
        _check_operand(w_down, "saved w_down", x, (E, I, H))
        if sh_gate_up is not None:
            _check_operand(sh_gate_up, "saved shared_expert_gate_up", x, (H, 2 * I))
            _check_operand(sh_down, "saved shared_expert_down", x, (I, H))
            _check_operand(sh_out_gate, "saved shared_expert_output_gate", x, (H, 1))
        ops._chk(saved, "saved routing and activations", torch.uint8)
        if saved.numel() != _layer_sizes(key, T, True)[0]:
            raise RuntimeError("saved routing and activations must come back at their size")
        dy = torch.zeros_like(x) if dy is None else dy.contiguous()
        ops._chk(dy, "dy", x.dtype)
        lib, config, stream, need = _lib.load(), _layer_config(*key), ops._stream(), ctx.needs_input_grad
        shared = sh_gate_up is not None
        scratch = torch.empty(_layer_sizes(key, T, True)[2], dtype=torch.uint8, device=x.device)
        d_w_gate_up = torch.empty_like(w_gate_up) if need[2] else None
        d_w_down = torch.empty_like(w_down) if need[3] else None
        if ds_perm is not None:
            ds_perm = ds_perm.float().contiguous()
        bwd = (config, T, x.data_ptr(), dy.data_ptr(), w_down.data_ptr(), saved.data_ptr(), scratch.data_ptr(), ops._ptr(ds_perm),
               opts["loss_coeff"] / T / opts["ep_size"], ops._ptr(d_w_gate_up), ops._ptr(d_w_down))
        # 16 bits: rows of d_logits of a multiple of 32 (zeros past E), whatever E is, and the router's weight gradient in
        # the same call
        padded = x.dtype is not torch.float32 and router_gate.shape == (E, H) and router_gate.dtype is x.dtype
        d_router_gate = None
        if padded:
            d_logits = torch.empty((T, -(-E // 32) * 32), dtype=x.dtype, device=x.device)
            chunks = parts = None
            splits = 1
            if need[1]:
                d_router_gate = torch.empty((E, H), dtype=x.dtype, device=x.device)
                splits = _dense_splits(T, E, H, x.dtype, 128)
                chunks = _token_offsets(T, splits, x.device)
                parts = torch.empty(splits * E * H, dtype=torch.float32, device=x.device) if splits > 1 else None
            _lib.check(
                lib.amoe_layer_bwd_router(
                    *bwd, d_logits.data_ptr(), ops._ptr(chunks), splits, ops._ptr(parts), ops._ptr(d_router_gate), stream, side
                ),
                "amoe_layer_bwd",
            )
            if d_logits.shape[1] != E:
                d_logits = d_logits[:, :E]
        else:
            d_logits = torch.empty((T, E), dtype=x.dtype, device=x.device)
            _lib.check(lib.amoe_layer_bwd(*bwd, d_logits.data_ptr(), stream, side), "amoe_layer_bwd")
            if router_gate.shape[0] != E:
                d_logits = d_logits[:, : router_gate.shape[0]].contiguous()
            if need[1]:
                d_router_gate = _router_weight_grad(d_logits, x)
        cap = opts.get("capture")
        if cap is not None:
            start = _layer_sizes(key, T, True)[-1]
            cap.update(d_logits=d_logits, d_scores=scratch[start : start + 4 * T * K].view(torch.float32).view(T, K).clone())

        d_sh_gate_up = d_sh_down = d_sh_out_gate = d_pre = all_rows = None
        if shared:
            all_rows = _token_offsets(T, 1, x.device)
            d_pre = torch.empty((T, 1), dtype=x.dtype, device=x.device)
            n_gu, n_dn = _dense_splits(T, H, 2 * I, x.dtype), _dense_splits(T, I, H, x.dtype)
            d_sh_gate_up = torch.empty_like(sh_gate_up) if need[4] else None
            d_sh_down = torch.empty_like(sh_down) if need[5] else None
            parts = torch.empty(max(2 * n_gu, n_dn) * H * I, dtype=x.dtype, device=x.device) if max(n_gu, n_dn) > 1 else None
            _lib.check(
                lib.amoe_layer_bwd_shared(
                    config, T, x.data_ptr(), dy.data_ptr(), sh_down.data_ptr(), all_rows.data_ptr(), saved.data_ptr(),
                    scratch.data_ptr(), ops._ptr(parts), _token_offsets(T, n_gu, x.device).data_ptr(), n_gu, ops._ptr(d_sh_gate_up),
                    _token_offsets(T, n_dn, x.device).data_ptr(), n_dn, ops._ptr(d_sh_down), d_pre.data_ptr(), stream,
                ),
                "amoe_layer_bwd_shared",
            )
            if need[6]:
                d_sh_out_gate = ops.column_grad(x, d_pre)

        dx = dx_router = None
        if need[0]:
            dx = torch.empty_like(x)
            dx_router = _router_input_grad(d_logits, router_gate, padded)
        if dx is not None or side is not None:
            _lib.check(
                lib.amoe_layer_bwd_input(
                    config, T, w_gate_up.data_ptr(), ops._ptr(sh_gate_up), ops._ptr(sh_out_gate), ops._ptr(all_rows),
                    saved.data_ptr(), scratch.data_ptr(), ops._ptr(dx_router), ops._ptr(d_pre), ops._ptr(dx), stream, side,
                ),
                "amoe_layer_bwd_input",
            )
        return dx, d_router_gate, d_w_gate_up, d_w_down, d_sh_gate_up, d_sh_down, d_sh_out_gate, None, None


class _UngatedExpertLayerFn(torch.autograd.Function):
    """The layer with is_gated=False (moe.py:101-106, 188-191, 306-311): an expert is two plain
    linear maps, out = (x @ W_up[e]) @ W_down[e] with W_up [E,H,I] -- the reference applies its
    activation only inside the gated branch -- and the routing scores weight the combine
    (moe.py:450-461).  Same routing, permutation, load-balance hook and gradients as the gated
    layer; the grouped GEMMs run without an activation epilogue."""

    @staticmethod
    def forward(ctx, x, router_gate, w_up, w_down, sh_up, sh_down, sh_out_gate, replay, opts):
        T, H = x.shape
        K = opts["top_k"]
        timers: PhaseTimers = opts["timers"]
        cfg = opts["tile_cfg"]
        logits, probs, topk_idx, scores, ws, (counts, offsets, token_of, slot_of, row_of, scores_perm) = _route(
            x, router_gate, replay, opts
        )
        timers.start("groupGeMM")
        inter = ops.grouped_gemm_nn(x, w_up, offsets, a_row_map=token_of, n_rows=T * K, tile_cfg=cfg, workspace=ws,
                                    map_ready=True)
        out = ops.grouped_gemm_nn(inter, w_down, offsets, tile_cfg=cfg, workspace=ws, map_ready=True)
        timers.stop("groupGeMM")
        timers.start("moe-combine")
        y = ops.combine_fwd(out, row_of, scores)
        timers.stop("moe-combine")

        shared = sh_up is not None
        sh_inter = sh_out = sh_sig = None
        if shared:
            # dense linear maps over all T tokens: plain library GEMMs, like the reference's
            timers.start("shared-expert")
            sh_inter = torch.matmul(x, sh_up)
            sh_out = torch.matmul(sh_inter, sh_down)
            sh_sig = torch.sigmoid(torch.matmul(x, sh_out_gate))  # [T,1]
            y = y + sh_out * sh_sig
            timers.stop("shared-expert")

        ctx.opts = opts
        ctx.shared = shared
        ctx.gemm_ws = ws
        ctx.save_for_backward(x, router_gate, w_up, w_down, probs, topk_idx, counts, offsets, row_of, token_of, scores,
                              inter, out, sh_up, sh_down, sh_out_gate, sh_inter, sh_out, sh_sig)
        if opts["want_scores"]:
            scores_out = scores_perm.to(x.dtype)
        else:
            scores_out = scores_perm.new_empty(0)
            ctx.mark_non_differentiable(scores_out)
        ctx.set_materialize_grads(False)
        cap = opts.get("capture")
        if cap is not None:
            cap.update(logits=logits, probs=probs, topk_idx=topk_idx, scores=scores, counts=counts, offsets=offsets,
                       token_of=token_of, slot_of=slot_of, row_of=row_of)
        return y, scores_out

    @staticmethod
    def backward(ctx, dy, ds_perm):
        (x, router_gate, w_up, w_down, probs, topk_idx, counts, offsets, row_of, token_of, scores,
         inter, out, sh_up, sh_down, sh_out_gate, sh_inter, sh_out, sh_sig) = ctx.saved_tensors
        opts = ctx.opts
        E, K = opts["num_experts"], opts["top_k"]
        T = x.shape[0]
        cfg = opts["tile_cfg"]
        if dy is None and ds_perm is None:
            return (None,) * 9
        dy = torch.zeros_like(x) if dy is None else dy.contiguous()
        ws = ctx.gemm_ws  # still holds the forward's tile map

        # d_out[r] = s_r * dy[token_of[r]],  d_scores[t,k] = <dy[t], out[row_of[t,k]]>
        d_out, d_scores = ops.combine_bwd(dy, out, row_of, scores)
        if ds_perm is not None:
            d_scores = d_scores + ds_perm.float()[row_of.long()]
        d_inter = ops.grouped_gemm_nt(d_out, w_down, offsets, tile_cfg=cfg, workspace=ws, map_ready=True)
        d_w_down = ops.grouped_gemm_wgrad(inter, d_out, offsets, E, tile_cfg=cfg) if ctx.needs_input_grad[3] else None
        d_w_up = None
        if ctx.needs_input_grad[2]:
            d_w_up = ops.grouped_gemm_wgrad(x, d_inter, offsets, E, tile_cfg=cfg, a_row_map=token_of)

        d_logits = ops.router_bwd(
            d_scores, probs, topk_idx, counts, x.dtype, opts["normalize"], opts["loss_coeff"] / T / opts["ep_size"]
        )
        d_router_gate = _router_weight_grad(d_logits, x) if ctx.needs_input_grad[1] else None
        cap = opts.get("capture")
        if cap is not None:
            cap.update(d_scores=d_scores, d_logits=d_logits)

        d_sh_up = d_sh_down = d_sh_out_gate = d_sh_inter = d_pre = None
        if ctx.shared:
            d_sh_out = dy * sh_sig
            d_sig = (dy.float() * sh_out.float()).sum(dim=1, keepdim=True)
            sig = sh_sig.float()
            d_pre = (d_sig * sig * (1.0 - sig)).to(x.dtype)  # [T,1]
            d_sh_inter = torch.matmul(d_sh_out, sh_down.t())
            if ctx.needs_input_grad[5]:
                d_sh_down = torch.matmul(sh_inter.t(), d_sh_out)
            if ctx.needs_input_grad[4]:
                d_sh_up = torch.matmul(x.t(), d_sh_inter)
            if ctx.needs_input_grad[6]:
                d_sh_out_gate = ops.column_grad(x, d_pre)

        dx = None
        if ctx.needs_input_grad[0]:
            d_xp = ops.grouped_gemm_nt(d_inter, w_up, offsets, tile_cfg=cfg, workspace=ws, map_ready=True)
            dx_dense = _router_input_grad(d_logits, router_gate)
            if ctx.shared:
                dx_dense.addmm_(d_pre, sh_out_gate.t())
                dx_dense.addmm_(d_sh_inter, sh_up.t())
            dx = ops.gather_rows_bwd(d_xp, row_of, addend=dx_dense)
        return dx, d_router_gate, d_w_up, d_w_down, d_sh_up, d_sh_down, d_sh_out_gate, None, None


class ArcticMoE(nn.Module):
    """Mixture-of-experts layer with the reference's surface (moe.py:63-323).

    Args:
        config: MoEConfig (or any object with the same attributes; the reference passes a
                SimpleNamespace, utils.py:107-161)

    Attributes beyond the reference's, all optional:
        tile_cfg: tile shape of the grouped GEMMs (0 = the library's default; 1, 2, 3, 5 for tuning)
        check_replay: raise on a replayed expert id outside [0, E), as the reference's one_hot does
                (one host synchronisation per replayed forward; skipped under graph capture)
        overlap_weight_grads: run the two expert weight gradients of the backward on a second stream where the step is long
                enough for it to pay
        capture: a dict that receives the routing intermediates of each forward (tests)
    """

    def __init__(self, config):
        super().__init__()
        self._config = config
        self.act_fn = config.act_fn
        self.ep_group = getattr(config, "ep_group", None)
        self.ep_rank = getattr(config, "ep_rank", 0)
        self.ep_size = getattr(config, "ep_size", 1)
        self.input_dtype = config.input_dtype
        self.intermediate_dim = config.intermediate_dim
        self.model_dim = config.model_dim
        self.num_experts = config.num_experts
        self.top_k = config.top_k
        self.use_custom_kernel = getattr(config, "use_custom_moe_kernel", False)
        if self.use_custom_kernel:
            import warnings

            warnings.warn(
                "ArcticMoE: use_custom_moe_kernel=True is ignored -- the layer computes the reference's default path "
                "(ragged rows, load-balance gradient, scores normalised in the gate), not its capacity-padded one",
                stacklevel=2,
            )
        if self.ep_size != 1:
            raise NotImplementedError("this build runs the expert layer on one GPU (ep_size must be 1)")
        self.is_gated = bool(getattr(config, "is_gated", True))
        self._act_code = classify_activation(config.act_fn)

        self.timers = PhaseTimers()
        self.wall_clock_breakdown = False
        self.gate_time = 0.0
        self.num_local_experts = self.num_experts // self.ep_size
        self.tile_cfg = 0  # 0 = library default tile shape; other values are for tuning
        # replayed expert ids outside [0, E) raise like the reference's one_hot (one host synchronisation per
        # replayed forward); False: no check, the permutation kernels clamp them
        self.check_replay = True
        self.capture = None  # set to a dict to receive the routing intermediates of each forward

        dt = self.input_dtype
        # gate and up projection interleaved when gated, one plain projection otherwise (moe.py:101-106)
        up_cols = (2 if self.is_gated else 1) * self.intermediate_dim
        self.router_gate = nn.Parameter(torch.empty((self.num_experts, self.model_dim), dtype=dt))
        self.expert_gate_up = nn.Parameter(
            torch.empty((self.num_local_experts, self.model_dim, up_cols), dtype=dt)
        )
        self.gate_scale = 1.0
        self.up_scale = 0.0
        self.expert_down = nn.Parameter(torch.empty((self.num_local_experts, self.intermediate_dim, self.model_dim), dtype=dt))
        if getattr(config, "use_shared_expert", False):
            self.shared_expert_gate_up = nn.Parameter(torch.empty((self.model_dim, up_cols), dtype=dt))
            self.shared_expert_down = nn.Parameter(torch.empty((self.intermediate_dim, self.model_dim), dtype=dt))
            self.shared_expert_output_gate = nn.Parameter(torch.empty(self.model_dim, 1, dtype=dt))
        self.enable_routing_replay = getattr(config, "enable_routing_replay", False)
        # backward: the two expert weight gradients on a second stream (see _side_stream)
        self.overlap_weight_grads = True

    def enable_wall_clock_breakdown(self):
        """activate the phase timers (moe.py:153-156)"""
        self.wall_clock_breakdown = True
        self.timers.wall_clock_breakdown = True

    def extra_repr(self):
        lines = [
            f"(router_gate): Parameter({tuple(self.router_gate.shape)})",
            f"(expert_gate_up): Parameter({tuple(self.expert_gate_up.shape)})",
            f"(expert_down): Parameter({tuple(self.expert_down.shape)})",
        ]
        if getattr(self._config, "use_shared_expert", False):
            lines += [
                f"(shared_expert_gate_up): Parameter({tuple(self.shared_expert_gate_up.shape)})",
                f"(shared_expert_down): Parameter({tuple(self.shared_expert_down.shape)})",
                f"(shared_expert_output_gate): Parameter({tuple(self.shared_expert_output_gate.shape)})",
            ]
        return "\n".join(lines)

    def forward(self, hidden_states, routing_replay_assignments: Optional[torch.Tensor] = None):
        if self.enable_routing_replay:
            assert (
                routing_replay_assignments is not None
            ), "Routing replay assignments must be provided when routing replay is enabled"
        self.timers.start("amoe e2e")
        orig_shape = hidden_states.shape
        x = hidden_states.reshape(-1, hidden_states.shape[-1]).contiguous()
        opts = dict(
            num_experts=self.num_experts,
            top_k=self.top_k,
            normalize=bool(self._config.normalize_topk_scores),
            loss_coeff=float(getattr(self._config, "loss_coeff", 0.01)),
            ep_size=self.ep_size,
            act=self._act_code,
            tile_cfg=self.tile_cfg,
            check_replay=self.check_replay,
            overlap_weight_grads=self.overlap_weight_grads,
            want_scores=bool(getattr(self._config, "return_router_scores", False)),
            timers=self.timers,
            capture=self.capture,
        )
        replay = routing_replay_assignments if self.enable_routing_replay else None
        if self.tile_cfg == 3 and x.dtype == torch.float16:
            # (the row-grouped products are not built for that combination; the default shape is)
            raise RuntimeError("ArcticMoE: tile_cfg 3 is not available for float16 layers")
        if x.shape[0] == 0:
            # no tokens (the reference returns an empty tensor from the same code path): nothing to
            # launch; the result still hangs off every parameter so that their gradients are zeros
            output = (x + sum(p.sum() for p in self.parameters()) * 0).reshape(orig_shape)
            self.timers.stop("amoe e2e")
            return (output, x.new_zeros(0)) if getattr(self._config, "return_router_scores", False) else output
        shared = (None, None, None)
        if getattr(self._config, "use_shared_expert", False):
            shared = (self.shared_expert_gate_up, self.shared_expert_down, self.shared_expert_output_gate)
        # the kernels are launched on the current device's current stream: make x's device current
        elsewhere = x.is_cuda and x.device.index != torch.cuda.current_device()
        with torch.cuda.device(x.device) if elsewhere else contextlib.nullcontext():
            if self.is_gated:
                output, scores = self._run_gated(x, shared, replay, opts)
            else:
                output, scores = _UngatedExpertLayerFn.apply(
                    x, self.router_gate, self.expert_gate_up, self.expert_down, *shared, replay, opts
                )
        output = output.reshape(orig_shape)
        self.timers.stop("amoe e2e")
        return (output, scores) if getattr(self._config, "return_router_scores", False) else output

    def _run_gated(self, x, shared, replay, opts):
        weights = (self.router_gate, self.expert_gate_up, self.expert_down)
        # (forward-mode runs without gradients too: inside a dual level the autograd function decides on the tangents)
        if torch.is_grad_enabled() or getattr(forward_ad, "_current_level", 0) >= 0:
            out = _ExpertLayerFn.apply(x, *weights, *shared, replay, opts)
            return out if opts["want_scores"] else (out, None)
        y, saved, key = _layer_forward(x, *weights, shared, replay, opts, keep=False)
        return y, _saved_view(saved, "scores_perm", key, x.shape[0]).to(x.dtype, copy=True) if opts["want_scores"] else None
