"""Performance cases of the sparse-MLP path: what a program built on this framework has it do, through its public
entry points (``SparseMLPStack``, ``SparseDecodeLayer``, ``SkipMLP``, ``WeightCache`` and ``sparse_mlp_forward``).

Kinds of case
  stack     one token through ``SparseMLPStack.step_staged``, replayed from its HIP graph: the decode loop of bench.py
  layers    ``SparseDecodeLayer.step`` once per layer, launched call by call, every layer with inputs of its own: a model
            whose attention and norms sit between the calls.  The same calls with many rows are a prefill.
  module    the drop-in ``SkipMLP`` as a decoder layer drives it: predictor mask, ``update_active_weights``, forward
  operator  the reference's call sequence on one layer: update, two getters, ``sparse_mlp_forward``
  rebuild   ``SkipMLP.reset_cache``, which a generation starts with

In all of them but the last the masks change from pass to pass: every layer's predictor inputs follow an AR(1) sequence
that is walked forwards and backwards, so that each pass swaps about ``churn`` of the active set.  The predictors'
thresholds (k, standard deviations) are placed in a gap between scores near their nominal value, so that a score which
is rounded differently does not change a mask.
"""
import math

import torch

import sparse_transformers_amd as st

STEPS = 6    # inputs of a sequence: passes run 1, 2, ... 5, 4, ... 0, 1, ...


def listed():
    llama1b = dict(hidden=2048, intermediate=8192, rank=64)
    llama3b = dict(hidden=3072, intermediate=8192, rank=128)
    mistral = dict(hidden=4096, intermediate=14336, rank=256)
    relullama = dict(hidden=4096, intermediate=11008, rank=440)
    opt = dict(hidden=2560, intermediate=10240, rank=104)

    def case(name, kind, shape, layers, rows, dtype, act="silu", gated=True, method="threshold", active=0.35, churn=0.10,
             shared=0.0):
        return dict(name=name, kind=kind, **shape, layers=layers, rows=rows, dtype=dtype, act=act, gated=gated,
                    method=method, active=active, churn=churn, shared=shared)

    return [
        # a single fp32 layer called like the reference's operator: the smallest call, where the host counts
        case("operator_llama1b_fp32", "operator", llama1b, 1, 1, "float32", active=0.30),
        # the decode loops of bench.py: one token (eight rows of a batch) through a stack, replayed from a graph.  Gated
        # stacks are kept short: without the model's norms every layer doubles the relative difference of its input.
        case("stack_llama3b_fp16", "stack", llama3b, 4, 1, "float16"),
        case("stack_mistral7b_bf16_b8", "stack", mistral, 4, 8, "bfloat16", active=0.25),
        # very sparse ReLU model at its full depth
        case("stack_relullama7b_ungated_fp16", "stack", relullama, 32, 1, "float16", act="relu", gated=False, active=0.10,
             churn=0.20),
        # a 3B model's 28 MLPs for one token, launched from the model's own Python loop
        case("layers_llama3b_fp16", "layers", llama3b, 28, 1, "float16"),
        # the same through the drop-in module, with the row-statistic mask of the Gemma-3n configuration
        case("module_mistral7b_bf16_statistical", "module", mistral, 8, 1, "bfloat16", method="statistical_topk",
             active=0.25),
        # small batches: the union of per-row masks that share most of their indices
        case("layers_llama3b_bf16_b4_topk", "layers", llama3b, 8, 4, "bfloat16", method="topk", active=0.30, shared=0.65),
        case("layers_llama3b_bf16_b16", "layers", llama3b, 8, 16, "bfloat16", active=0.70, churn=0.20, shared=0.65),
        # prefills: a short ragged prompt, 512 tokens, and the largest call
        case("prefill_opt2b7_ungated_fp16_77", "layers", opt, 4, 77, "float16", act="relu", gated=False, active=0.60,
             shared=0.9),
        case("prefill_llama3b_bf16_512", "layers", llama3b, 2, 512, "bfloat16", active=0.80, shared=0.9),
        case("prefill_mistral7b_bf16_2048", "layers", mistral, 1, 2048, "bfloat16", active=0.90, shared=0.9),
        # a new generation starts: one layer's cache is dropped and built again from the module's weights
        case("rebuild_llama3b_fp16", "rebuild", llama3b, 1, 1, "float16"),
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["operator", "stack", "stack", "layers", "layers", "module", "prefill", "prefill", "rebuild"])
    hidden = 128 * round(_log_uniform(rng, 6, 40))
    intermediate = min(16384, int(hidden * rng.uniform(2.0, 4.0)))
    if rng.random() < 0.75:       # model sizes are round; a quarter of the draws is not
        intermediate = intermediate // 64 * 64
    rank = max(16, int(hidden * rng.uniform(0.02, 0.11)) // 8 * 8)
    act, gated = rng.choice([("silu", True), ("silu", True), ("relu", True), ("gelu_pytorch_tanh", True), ("relu", False)])
    dtype = rng.choice(["float16", "bfloat16"] if kind == "prefill" else ["float16", "float16", "bfloat16", "bfloat16", "float32"])
    rows, layers, method = 1, 1, "threshold"
    active, churn, shared = rng.uniform(0.08, 0.5), rng.uniform(0.05, 0.4), 0.0
    if kind in ("stack", "layers", "module", "operator"):
        rows = round(_log_uniform(rng, 1, 8 if dtype == "float32" else 32))
        shared = rng.uniform(0.5, 0.8) if rows > 1 else 0.0
        if kind != "operator":
            # at most as much as the deepest listed stack streams
            per_layer = (3 if gated else 2) * active * intermediate * hidden * (4 if dtype == "float32" else 2)
            layers = max(1, min(rng.randint(2, 4 if kind == "stack" and gated else 8), int(6e8 / per_layer)))
        if kind in ("layers", "module"):
            method = rng.choice(["threshold", "threshold", "topk", "statistical_topk"])
    if kind == "prefill":
        kind, shared, active = "layers", 0.9, rng.uniform(0.5, 0.95)
        rows = round(_log_uniform(rng, 33, min(2048, 1.0e11 / (hidden * intermediate))))
    return dict(kind=kind, hidden=hidden, intermediate=intermediate, rank=rank, layers=layers, rows=rows, dtype=dtype, act=act,
                gated=gated, method=method, active=round(active, 4), churn=round(churn, 4), shared=round(shared, 4))


# ---------------------------------------------------------------------------------------------------- preparation
# root mean square of act(g) * u (act(u) ungated) for independent standard normal g, u: a layer's down projection is
# scaled by it, so that a stack's activations stay of order one
_ACT_RMS = {"silu": 0.597, "relu": 0.707, "gelu_pytorch_tanh": 0.652}


def _predictor_inputs(c, gen, dev):
    """[STEPS, layers, rows, hidden]: AR(1) along the steps, rows of a layer with a shared part.  For normal scores at a
    third active the set changes by 0.61 sqrt(1 - rho) of itself per step."""
    rho = max(0.0, 1.0 - (c["churn"] / 0.61) ** 2)
    L, B, H = c["layers"], c["rows"], c["hidden"]

    def fresh():
        own = torch.randn(L, B, H, generator=gen, device=dev)
        if c["shared"] == 0.0:
            return own
        return math.sqrt(c["shared"]) * torch.randn(L, 1, H, generator=gen, device=dev) + math.sqrt(1 - c["shared"]) * own

    x = fresh()
    steps = [x]
    for _ in range(STEPS - 1):
        x = rho * x + math.sqrt(1.0 - rho * rho) * fresh()
        steps.append(x)
    return torch.stack(steps).to(getattr(torch, c["dtype"]))


def _place_cut(c, scores):
    """The layer's threshold, k or standard-deviation multiplier: of 65 values around the nominal one, the value whose
    cut lies farthest from every score.  scores: fp32 [STEPS, rows, I]."""
    dev, I = scores.device, scores.size(-1)
    if c["method"] == "threshold":
        s = scores.amax(1).sort(-1).values                     # the union over rows sees the largest score only
        at = min(max(int((1.0 - c["active"]) * s.numel()), 40), s.numel() - 40)
        flat = s.flatten().sort().values
        values = 0.5 * (flat[at - 33:at + 32] + flat[at - 32:at + 33])
        cuts = values[:, None].expand(-1, s.size(0))
    else:
        s = scores.flatten(0, 1).sort(-1).values
        if c["method"] == "topk":
            k = min(max(int(c["active"] * I), 40), I - 40)
            values = torch.arange(k - 32, k + 33, device=dev)
            cuts = 0.5 * (s[:, I - values] + s[:, I - 1 - values]).t()
        else:
            z = float(torch.distributions.Normal(0.0, 1.0).icdf(torch.tensor(1.0 - c["active"])))
            values = z + 0.002 * torch.arange(-32, 33, device=dev)
            mean, std = s.mean(-1), s.std(-1, unbiased=False)
            cuts = mean + std * values[:, None]
    cuts = cuts.t().contiguous()                               # [row, candidate]
    i = torch.searchsorted(s, cuts).clamp(1, I - 1)
    margin = torch.minimum((cuts - s.gather(1, i - 1)).abs(), (s.gather(1, i) - cuts).abs()).amin(0)
    return values[margin.argmax()]


def prepare(case, seed):
    c = dict(case)
    dev, dt = torch.device("cuda"), getattr(torch, c["dtype"])
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    L, B, H, I, r = c["layers"], c["rows"], c["hidden"], c["intermediate"], c["rank"]

    def weight(rows, cols, std):
        return torch.randn(rows, cols, generator=gen, device=dev, dtype=dt).mul_(std)

    state = {"case": c, "pass": 0}
    x_pred = None if c["kind"] == "rebuild" else _predictor_inputs(c, gen, dev)
    predictors, caches, modules, cuts = [], [], [], []
    down_std = (c["active"] * I) ** -0.5 / (_ACT_RMS[c["act"]] if c["gated"] else 0.707)
    ones = torch.ones(I, dtype=torch.bool, device=dev)
    x = torch.randn(STEPS, *(() if c["kind"] == "stack" else (L,)), B, H, generator=gen, device=dev).to(dt)
    for l in range(L):
        gate = weight(I, H, H ** -0.5) if c["gated"] else None
        up, down = weight(I, H, H ** -0.5), weight(H, I, down_std)
        A, Bm = weight(r, H, H ** -0.5), weight(I, r, r ** -0.5)
        if x_pred is not None:
            predictors.append(st.FastLoRAProjection(A, Bm))
            scores = ((x_pred[:, l].flatten(0, 1).float() @ A.float().t()) @ Bm.float().t()).view(STEPS, B, I)
            cuts.append(_place_cut(c, scores))
            del scores
        if c["kind"] in ("module", "rebuild"):
            m = st.SkipMLP.from_weights(gate, up, down, sparsity=1.0 - c["active"], act_fn=c["act"], has_gate=c["gated"])
            m.initialize_weight_cache()
            modules.append(m)
        else:
            caches.append(st.WeightCache(ones, H, gate, up, down, c["gated"]))
        del gate, up, down
    cuts = [v.item() for v in cuts]

    if c["kind"] == "rebuild":
        state["module"] = modules[0]
        return state
    state["x_pred"], state["x"] = x_pred, x

    if c["kind"] in ("stack", "layers"):
        layers = [st.SparseDecodeLayer(p, k, c["act"], method=c["method"], **_cut_args(c, cut))
                  for p, k, cut in zip(predictors, caches, cuts)]
        if c["kind"] == "layers":
            state["layers"] = layers
            for l, layer in enumerate(layers):                 # the step before the first pass: from all rows to the first mask
                layer.step(x_pred[0, l], state["x"][0, l])
            return state
        stack = state["stack"] = st.SparseMLPStack(layers)
        for l, layer in enumerate(layers):
            layer.cache.update_active_weights(layer.predict_mask(x_pred[0, l]))
        stack.prepare(B)
        stack.use_trace_masks = False                          # the layers' own masks drive the caches
        stack.step_staged(state["x"][0], x_pred[0])            # one eager step before the capture
        torch.cuda.synchronize()
        stack.capture()
        return state
    if c["kind"] == "module":
        state["modules"], state["predictors"] = modules, predictors
        state["cut_args"] = [_cut_args(c, cut) for cut in cuts]
        for l, m in enumerate(modules):
            m.weight_cache.update_active_weights(predictors[l].mask(x_pred[0, l], c["method"], **state["cut_args"][l]))
            m(state["x"][0, l])
        return state
    # operator: the masks of a sequence in hand, the caller's two buffers as the reference registers them
    state["cache"] = caches[0]
    state["masks"] = [predictors[0].mask(x_pred[t, 0], c["method"], **_cut_args(c, cuts[0])) for t in range(STEPS)]
    caches[0].update_active_weights(state["masks"][0])
    state["down_proj_buffer"] = torch.zeros(B, H, dtype=dt, device=dev)
    state["combined_proj_buffer"] = torch.zeros(B, (2 if c["gated"] else 1) * int(c["active"] * I), dtype=dt, device=dev)
    return state


def _cut_args(c, cut):
    return {"threshold": {"thr": cut}, "topk": {"k": int(cut)}, "statistical_topk": {"std_multiplier": cut}}[c["method"]]


# ----------------------------------------------------------------------------------------------------------- one pass
def run(state):
    c = state["case"]
    if c["kind"] == "rebuild":
        module = state["module"]
        module.reset_cache()
        return {"concat": module.weight_cache.get_concat_weight(), "down": module.weight_cache.get_active_down_weight()}
    state["pass"] += 1
    t = state["pass"] % (2 * STEPS - 2)
    t = min(t, 2 * STEPS - 2 - t)
    if c["kind"] == "stack":
        stack = state["stack"]
        out = stack.step_staged(state["x"][t], state["x_pred"][t], replay=True)
        return {"out": out, "masks": [layer.mask for layer in stack.layers]}
    if c["kind"] == "layers":
        outs = [layer.step(xp, x) for layer, xp, x in zip(state["layers"], state["x_pred"][t], state["x"][t])]
        return {"out": outs, "masks": [layer.mask for layer in state["layers"]]}
    if c["kind"] == "module":
        outs, masks = [], []
        for module, predictor, args, xp, x in zip(state["modules"], state["predictors"], state["cut_args"],
                                                  state["x_pred"][t], state["x"][t]):
            mask = predictor.mask(xp, c["method"], **args)
            module.weight_cache.update_active_weights(mask)
            outs.append(module(x))
            masks.append(mask)
        return {"out": outs, "masks": masks}
    cache = state["cache"]
    cache.update_active_weights(state["masks"][t])
    out = st.sparse_mlp_forward(state["x"][t, 0], cache.get_concat_weight(), cache.get_active_down_weight(),
                                state["down_proj_buffer"], state["combined_proj_buffer"], c["act"], c["gated"])
    return {"out": out}


# --------------------------------------------------------------------------------------------------- work, tolerance
def work(case):
    """Of one pass: the active rows, the changed rows once from the pool and once into the packed buffers, the
    predictor's weights, inputs, outputs and masks."""
    c = case
    s = 4 if c["dtype"] == "float32" else 2
    mats = 3 if c["gated"] else 2
    H, I, r, B, L = c["hidden"], c["intermediate"], c["rank"], c["rows"], c["layers"]
    if c["kind"] == "rebuild":        # the module's weights once, the pools and the packed rows once
        return {"bytes": 3 * mats * I * H * s, "flops": 0}
    n = c["active"] * I
    if c["method"] != "threshold" and B > 1:      # a selection per row: their union is larger (rows share most of it)
        n = min(I, n * (1.0 + (1.0 - c["shared"]) * (B - 1) * 0.5))
    predictor = 0 if c["kind"] == "operator" else (r * H + I * r) * s + B * H * s + I
    mlp = mats * n * H * s + 2 * mats * min(c["churn"], 1.0) * n * H * s + 2 * B * H * s + 2 * I
    flops = 2.0 * B * n * H * mats + (0 if c["kind"] == "operator" else 2.0 * B * (r * H + I * r))
    if c["kind"] == "operator":
        mlp += B * mats * n * s
    return {"bytes": L * (predictor + mlp), "flops": L * flops}


def tolerance(case):
    """Four times what a pass differs by from float64 sums with the inputs, weights, outputs and act(g) * u rounded to the
    storage type (the kernels keep the last in fp32 for one or two rows of x): 1.9e-7 / 3.5e-4 / 2.6e-3 for a single
    layer in fp32 / fp16 / bf16; 5e-7 / 2e-3 / 1.1e-2 for stacks, which pass rounded activations on and whose gated
    layers, of second order in their input, double a deviation."""
    if case["kind"] == "rebuild":
        return "exact"
    if case["kind"] == "stack":
        return {"float32": {"rel": 2e-6, "max": 1e-5, "differ": 2e-4}, "float16": {"rel": 8e-3, "max": 4e-2, "differ": 2e-4},
                "bfloat16": {"rel": 3e-2, "max": 2.5e-1, "differ": 2e-4}}[case["dtype"]]
    return {"float32": {"rel": 8e-7, "max": 4e-6, "differ": 2e-4}, "float16": {"rel": 1.4e-3, "max": 5e-3, "differ": 2e-4},
            "bfloat16": {"rel": 1e-2, "max": 5e-2, "differ": 2e-4}}[case["dtype"]]
