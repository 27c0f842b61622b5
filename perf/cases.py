"""The work that a program has this package do, as cases to be timed.

A case is one call, or a short run of calls, through the package's public
entry points:

  linear   BlockFP8Linear: a dense FP8 projection (attention, shared expert)
           over `rows` token rows, from one decode token to a prefill chunk
  mlp      ClampedMLP: gate, up, SwiGLU and down of a dense FP8 MLP
  decode   one token through `layers` MoE layers, each by its own DecodePlan
           with bound weights (router, routed and shared experts)
  moe      SortedGroupedFP8MoE over `tokens` tokens: a short batch (a few
           sequences decoding together, or speculative tokens) up to a long
           prefill chunk, routing skewed or not, either reduction
  blocks   the prefill composed from its building blocks, as a program does
           that keeps its own routing: route plan, tile plan, grouped gate/up,
           SwiGLU, grouped down, restore and reduce

Weights are N(0, 0.02) quantised per 128 x 128 block with scale amax / 448,
router weights N(0, 0.02), router bias U(-0.01, 0.01) (plus a Zipf-like slope
for a skewed layer), activations N(0, 1) in bf16.  All are made with torch on
the GPU from the seed.
"""

import importlib
import math
from types import SimpleNamespace

import numpy as np
import torch

moe53 = importlib.import_module("glm53-flash-mlx_amd")

BLOCK = 128
LIMIT = 10.0
DEVICE = "cuda"


def listed():
    return [
        # one decode token through one dense projection: the smallest call
        {"name": "linear 1x4096x4096", "kind": "linear", "rows": 1, "n": 4096, "k": 4096},
        # 16 sequences decoding together through the same projection
        {"name": "linear 16x4096x4096", "kind": "linear", "rows": 16, "n": 4096, "k": 4096},
        # a short ragged prompt through a projection of the shared expert's size
        {"name": "linear 300x1536x4096", "kind": "linear", "rows": 300, "n": 1536, "k": 4096},
        # a prefill chunk through a square projection
        {"name": "linear 2048x4096x4096", "kind": "linear", "rows": 2048, "n": 4096, "k": 4096},
        # a dense MLP over a short prompt
        {"name": "mlp 96x4096x1536", "kind": "mlp", "tokens": 96, "hidden": 4096, "inter": 1536},
        # batch-1 decode, four layers of the 288-expert configuration
        {"name": "decode 4 layers", "kind": "decode", "layers": 4, "hidden": 4096, "inter": 1536, "experts": 288},
        # eight tokens at once: a small decode batch, or speculative tokens
        {"name": "moe 8 tokens", "kind": "moe", "tokens": 8, "hidden": 4096, "inter": 1536, "experts": 288,
         "skew": False, "reduction": "grouped"},
        # a short prompt, combined in the Direct order
        {"name": "moe 64 tokens direct", "kind": "moe", "tokens": 64, "hidden": 4096, "inter": 1536, "experts": 288,
         "skew": False, "reduction": "direct"},
        # the 256-token prefill configuration (2,048 routes)
        {"name": "moe 256 tokens", "kind": "moe", "tokens": 256, "hidden": 4096, "inter": 1536, "experts": 288,
         "skew": False, "reduction": "grouped"},
        # the 2,048-token configuration with Zipf-skewed routing
        {"name": "moe 2048 tokens zipf", "kind": "moe", "tokens": 2048, "hidden": 4096, "inter": 1536, "experts": 288,
         "skew": True, "reduction": "grouped"},
        # a long prefill chunk: the largest call
        {"name": "moe 8192 tokens", "kind": "moe", "tokens": 8192, "hidden": 4096, "inter": 1536, "experts": 288,
         "skew": False, "reduction": "grouped"},
        # 512 tokens through the building blocks at the real checkpoint's width (I = 2048)
        {"name": "blocks 512 tokens", "kind": "blocks", "tokens": 512, "hidden": 4096, "inter": 2048, "experts": 288},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# (hidden, intermediate) of the layers in the repository's configurations and tests
_DECODE_WIDTHS = [(4096, 1536), (4096, 2048), (7168, 2048), (6144, 2048), (2048, 1024), (2048, 1536)]
_MOE_WIDTHS = _DECODE_WIDTHS + [(1024, 512), (2048, 768), (3072, 1024), (5120, 1536)]


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "decode", "moe", "moe", "moe", "blocks"])
    if kind == "linear":
        return {"kind": kind, "rows": _log_uniform(rng, 1, 4096), "n": 16 * _log_uniform(rng, 32, 512),
                "k": 128 * _log_uniform(rng, 4, 56)}
    if kind == "mlp":
        return {"kind": kind, "tokens": _log_uniform(rng, 1, 2048), "hidden": 128 * _log_uniform(rng, 8, 48),
                "inter": 128 * _log_uniform(rng, 4, 32)}
    if kind == "decode":
        hidden, inter = rng.choice(_DECODE_WIDTHS)
        return {"kind": kind, "layers": rng.choice([2, 3, 4]), "hidden": hidden, "inter": inter,
                "experts": rng.randint(32, 288)}
    hidden, inter = rng.choice(_MOE_WIDTHS)
    experts = rng.randint(32, 288)
    tokens = _log_uniform(rng, 32, 2048) if kind == "blocks" else _log_uniform(rng, 2, 4096)
    case = {"kind": kind, "tokens": tokens, "hidden": hidden, "inter": inter, "experts": experts}
    if kind == "moe":
        case.update(skew=rng.random() < 0.4, reduction=rng.choice(["grouped", "grouped", "direct"]))
    return case


# ------------------------------------------------------------------ inputs --


class _Rng:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEVICE)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device=DEVICE, dtype=torch.float32).mul_(std)

    def uniform(self, *shape, lo, hi):
        return torch.rand(shape, generator=self.g, device=DEVICE, dtype=torch.float32).mul_(hi - lo).add_(lo)


def _fill(rng, codes, scale):
    """Quantised N(0, 0.02) matrices into codes u8 [E, rows, cols] and scale
    f32 [E, ceil(rows / 128), cols / 128] (rows may be ragged)."""
    experts, rows, cols = codes.shape
    rb = scale.shape[1]
    step = max(1, (1 << 28) // (rb * BLOCK * cols))
    for e in range(0, experts, step):
        n = min(step, experts - e)
        w = rng.normal(n, rb * BLOCK, cols, std=0.02)
        if rows < rb * BLOCK:
            w[:, rows:] = 0.0
        blocks = w.view(n, rb, BLOCK, cols // BLOCK, BLOCK)
        amax = torch.amax(blocks.abs(), dim=(2, 4))
        s = (amax / 448.0).clamp_min_(1e-12)
        blocks.div_(s[:, :, None, :, None]).clamp_(-448.0, 448.0)
        codes[e:e + n] = w.to(torch.float8_e4m3fn).view(torch.uint8)[:, :rows]
        scale[e:e + n] = s


def _matrices(rng, experts, shapes):
    """One bank buffer pair of matrices [rows, cols] stacked by rows."""
    cols = shapes[0][1]
    rows = sum(r for r, _ in shapes)
    codes = torch.empty((experts, rows, cols), dtype=torch.uint8, device=DEVICE)
    scale = torch.empty((experts, sum(-(-r // BLOCK) for r, _ in shapes), cols // BLOCK), dtype=torch.float32,
                        device=DEVICE)
    r0 = s0 = 0
    for r, _ in shapes:
        sb = -(-r // BLOCK)
        _fill(rng, codes[:, r0:r0 + r], scale[:, s0:s0 + sb])
        r0, s0 = r0 + r, s0 + sb
    return codes, scale


def _linear(rng, module):
    _fill(rng, module.weight[None], module.weight_scale_inv[None])
    return module


def _mlp(rng, hidden, inter):
    mlp = moe53.ClampedMLP(hidden, inter, LIMIT, device=DEVICE)
    for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj):
        _linear(rng, m)
    return mlp


def _bank(rng, case):
    e, h, i = case["experts"], case["hidden"], case["inter"]
    gate_up, gate_up_scale = _matrices(rng, e, [(i, h), (i, h)])
    down, down_scale = _matrices(rng, e, [(h, i)])
    leased = [moe53.owned_tensor(t, layout=moe53.TensorLayout.ROW_MAJOR_CONTIGUOUS)
              for t in (gate_up, gate_up_scale, down, down_scale)]
    return moe53.PackedFP8ExpertBank(*leased, intermediate_size=i)


def _gate(rng, case):
    e, h = case["experts"], case["hidden"]
    weight = rng.normal(e, h, std=0.02)
    bias = rng.uniform(e, lo=-0.01, hi=0.01)
    if case.get("skew"):
        rank = torch.randperm(e, generator=rng.g, device=DEVICE)
        bias = -0.12 * 1.1 * torch.log1p(rank.to(torch.float32))
    return moe53.Float32Gate(weight, bias, top_k=8, routed_scaling_factor=1.0, norm_topk_prob=True)


def _layer(rng, case):
    bank = _bank(rng, case)
    shared = _mlp(rng, case["hidden"], case["inter"])
    return bank, shared, _gate(rng, case)


def _tokens(rng, n, hidden):
    return rng.normal(n, hidden).to(torch.bfloat16)


def prepare(case, seed):
    rng = _Rng(seed)
    kind = case["kind"]
    if kind == "linear":
        x = _tokens(rng, case["rows"], case["k"])
        return SimpleNamespace(kind=kind, x=x, linear=_linear(rng, moe53.BlockFP8Linear(case["k"], case["n"],
                                                                                      device=DEVICE)))
    if kind == "mlp":
        x = _tokens(rng, case["tokens"], case["hidden"])
        return SimpleNamespace(kind=kind, x=x, mlp=_mlp(rng, case["hidden"], case["inter"]))
    if kind == "decode":
        layers = []
        for _ in range(case["layers"]):
            bank, shared, gate = _layer(rng, case)
            plan = moe53.DecodePlan(case["hidden"], case["inter"], case["inter"], case["experts"], 8, LIMIT)
            plan.bind_weights(bank, shared, gate)
            layers.append(SimpleNamespace(plan=plan, bank=bank, shared=shared, gate=gate,
                                          x=_tokens(rng, 1, case["hidden"])[0]))
        return SimpleNamespace(kind=kind, layers=layers)
    if kind == "moe":
        bank, shared, gate = _layer(rng, case)
        config = SimpleNamespace(hidden_size=case["hidden"], moe_intermediate_size=case["inter"], swiglu_limit=LIMIT,
                                 n_routed_experts=case["experts"], num_experts_per_tok=8, n_shared_experts=1)
        layer = moe53.SortedGroupedFP8MoE(bank, config, gate, shared, reduction=case["reduction"])
        return SimpleNamespace(kind=kind, layer=layer, bank=bank, shared=shared, gate=gate,
                               x=_tokens(rng, case["tokens"], case["hidden"])[None])
    bank = _bank(rng, case)
    x = _tokens(rng, case["tokens"], case["hidden"])
    noise = rng.normal(case["tokens"], case["experts"])
    chosen, ids = torch.topk(torch.sigmoid(noise), 8, dim=-1)
    return SimpleNamespace(kind=kind, bank=bank, x=x, ids=ids.to(torch.int32), scores=chosen / chosen.sum(-1, True))


# --------------------------------------------------------------------- run --


def run(state):
    if state.kind == "linear":
        return state.linear(state.x)
    if state.kind == "mlp":
        return state.mlp(state.x)
    if state.kind == "decode":
        return [layer.plan.execute_bound_router(layer.x) for layer in state.layers]
    if state.kind == "moe":
        return state.layer(state.x)
    bank = state.bank
    sorted_x, sorted_experts, sorted_scores, inverse = moe53.build_route_plan(state.x, state.ids, state.scores,
                                                                              expert_count=bank.expert_count)
    tiles = moe53.build_grouped_tile_plan(sorted_experts, bank.expert_count)
    gate_up = moe53.grouped_fp8_linear(sorted_x, tiles, bank.gate_up_weight, bank.gate_up_scale_inv)
    hidden = moe53.activate_gate_up(gate_up, bank.intermediate_size, LIMIT)
    routed = moe53.grouped_fp8_linear(hidden, tiles, bank.down_weight, bank.down_scale_inv)
    return moe53.restore_and_reduce(routed, sorted_scores, inverse, state.x.shape, 8)


# ------------------------------------------------------------ what it takes --


def _touched(case):
    """Experts that a call of this size touches (a fixed sample of the
    routing distribution)."""
    g = np.random.default_rng(0)
    e, h = case["experts"], case["hidden"]
    score = 1.0 / (1.0 + np.exp(-g.standard_normal((case.get("tokens", 1), e)) * 0.02 * math.sqrt(h)))
    if case.get("skew"):
        score = score - 0.12 * 1.1 * np.log1p(g.permutation(e))
    return int(np.unique(np.argpartition(-score, 7, axis=1)[:, :8]).size)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k + 4 * -(-n // BLOCK) * (k // BLOCK) + 2 * m * (n + k), "flops": 2 * m * n * k}
    t = case.get("tokens", 1)
    h, i = case["hidden"], case["inter"]
    expert = 3 * h * i + 4 * 3 * (h // BLOCK) * (i // BLOCK)
    if kind == "mlp":
        return {"bytes": expert + 4 * t * h, "flops": 6 * t * h * i}
    e = case["experts"]
    router = 4 * e * h + 4 * e
    if kind == "decode":
        return {"bytes": case["layers"] * (9 * expert + router + 4 * h),
                "flops": case["layers"] * (9 * 6 * h * i + 2 * e * h)}
    touched = _touched(case)
    if kind == "moe":
        return {"bytes": (touched + 1) * expert + router + 4 * t * h, "flops": 9 * t * 6 * h * i + 2 * t * e * h}
    return {"bytes": touched * expert + 4 * t * h + 64 * t, "flops": 8 * t * 6 * h * i}


def tolerance(case):
    # bf16 results of fp32 sums: another order of the sums moves some results
    # by one bf16 step (2^-8 relative); a MoE or MLP rounds three times in a row
    return {"rel": 4e-3 if case["kind"] == "linear" else 1e-2}


# ------------------------------------------------------------- 64-bit answer --


def _dequant(codes, scale):
    """float64 [rows, cols] of one matrix."""
    rows, cols = codes.shape
    w = codes.view(torch.float8_e4m3fn).to(torch.float64)
    s = scale.to(torch.float64)
    return w * s.repeat_interleave(BLOCK, 0)[:rows].repeat_interleave(BLOCK, 1)[:, :cols]


def _swiglu(g, u):
    g = torch.clamp(g, max=LIMIT)
    return g * torch.sigmoid(g) * torch.clamp(u, -LIMIT, LIMIT)


def _mlp64(mlp, x):
    g, u, d = (_dequant(m.weight, m.weight_scale_inv) for m in (mlp.gate_proj, mlp.up_proj, mlp.down_proj))
    return _swiglu(x @ g.T, x @ u.T) @ d.T


def _routed64(bank, x, ids, scores):
    inter = bank.intermediate_size
    srows = bank.gate_up_scale_inv.shape[1] // 2
    out = torch.zeros_like(x)
    for e in torch.unique(ids).tolist():
        token, slot = torch.nonzero(ids == e, as_tuple=True)
        gate = _dequant(bank.gate_up_weight[e, :inter], bank.gate_up_scale_inv[e, :srows])
        up = _dequant(bank.gate_up_weight[e, inter:], bank.gate_up_scale_inv[e, srows:])
        down = _dequant(bank.down_weight[e], bank.down_scale_inv[e])
        rows = x[token]
        out.index_add_(0, token, (_swiglu(rows @ gate.T, rows @ up.T) @ down.T) * scores[token, slot, None])
    return out


def _moe64(bank, shared, gate, x):
    score = torch.sigmoid(x @ gate.weight.to(torch.float64).T)
    choice = score + gate.e_score_correction_bias.to(torch.float64)
    ids = torch.topk(choice, gate.top_k, dim=-1).indices
    chosen = torch.gather(score, 1, ids)
    return _routed64(bank, x, ids, chosen / chosen.sum(-1, True)) + _mlp64(shared, x)


def exact(case, seed):
    state = prepare(case, seed)
    if state.kind == "linear":
        return state.x.to(torch.float64) @ _dequant(state.linear.weight, state.linear.weight_scale_inv).T
    if state.kind == "mlp":
        return _mlp64(state.mlp, state.x.to(torch.float64))
    if state.kind == "decode":
        return [_moe64(l.bank, l.shared, l.gate, l.x.to(torch.float64)[None])[0] for l in state.layers]
    if state.kind == "moe":
        return _moe64(state.bank, state.shared, state.gate, state.x[0].to(torch.float64))[None]
    return _routed64(state.bank, state.x.to(torch.float64), state.ids.to(torch.int64), state.scores.to(torch.float64))
