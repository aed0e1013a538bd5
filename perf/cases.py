"""Timed workloads of the gfx950 attention path: what a synthesis server has this framework do.

The model is the one the repository's tests and benchmark run: hidden 1024, 16 query / 2 KV heads of 64, FFN 4096,
Q8_0 weights drawn from N(0, 0.02), 24 layers (the backbone) or 4 / 8 (the LocDiT decoder).  Weights, caches and
activations are seeded N(0, 1) data of those shapes, made on the GPU.

A program keeps its weights (declared constant, as the plugin declares ggml's weight buffers), its caches and its plan.
What recurs with the same shapes and buffers -- a decode step's plan, a CFM solve, a LocDiT pass, the attention calls of
a step -- is replayed from a HIP graph, as bench.py and the plugin's recognition of recurring graphs do; a prompt is
issued call by call, since its length is its own.

  listed()         the fixed cases
  draw(rng)        one more case of the same ranges
  prepare(c, s)    what the program has in hand before the call, from the seed s
  run(state)       one pass; returns every result, the written cache slots among them
  work(c)          bytes and operations that the pass cannot do without
  tolerance(c)     how far another correct implementation at the same precision may be off
"""
import math

import numpy as np
import torch

import __graft_entry__

pkg = __graft_entry__.load_package()
from voxcpm_cpp_amd.backbone import WEIGHT_NAMES, MiniCPMBackbone  # noqa: E402
from voxcpm_cpp_amd.cfm import LocDiTCfmSolver  # noqa: E402

HIDDEN, HEADS, KV_HEADS, HEAD_DIM, FFN, FEAT = 1024, 16, 2, 64, 4096, 64
SHAPES = {"q_proj": (HEADS * HEAD_DIM, HIDDEN), "k_proj": (KV_HEADS * HEAD_DIM, HIDDEN), "v_proj": (KV_HEADS * HEAD_DIM, HIDDEN),
          "o_proj": (HIDDEN, HEADS * HEAD_DIM), "gate_proj": (FFN, HIDDEN), "up_proj": (FFN, HIDDEN), "down_proj": (HIDDEN, FFN)}
LAYER_WEIGHTS = sum(m * k for m, k in SHAPES.values())
LAYERS = 24          # the backbone
F16_LAYERS = 8       # layers of the F16-weight products: 56 of them
SCALE = 1.0 / math.sqrt(HEAD_DIM)


def listed():
    return [
        # one stream right after a short prompt, the reference's own cache type: the smallest decode step, all latency
        {"name": "step_b1_kv37_f32", "kind": "step", "batch": 1, "past": 37, "f16": False},
        # the CFG pair of one request in the middle of an utterance, f16 cache
        {"name": "step_b2_kv700_f16", "kind": "step", "batch": 2, "past": 700, "f16": True},
        # eight streams x CFG pair at long context: the largest decode step the benchmark runs
        {"name": "step_b16_kv6144_f16", "kind": "step", "batch": 16, "past": 6144, "f16": True},
        # a sentence of text as the prompt of one stream
        {"name": "prompt_1x45_f32", "kind": "prompt", "batch": 1, "tokens": 45, "f16": False},
        # a paragraph, or a sentence behind a few seconds of prompt audio
        {"name": "prompt_1x203_f32", "kind": "prompt", "batch": 1, "tokens": 203, "f16": False},
        # the CFG pair's prompt with prompt audio (the benchmark's 512-token prefill)
        {"name": "prompt_2x512_f16", "kind": "prompt", "batch": 2, "tokens": 512, "f16": True},
        # eight streams x CFG pair, long prompt audio: the largest prefill
        {"name": "prompt_16x4096_f16", "kind": "prompt", "batch": 16, "tokens": 4096, "f16": True},
        # one request's CFM solve: ten Euler steps over the 14-token CFG-pair sequence, 4 LocDiT layers
        {"name": "solve_p2_c4", "kind": "solve", "layers": 4, "patch": 2, "prefix": 4, "steps": 10},
        # one estimator pass of eight concurrent requests
        {"name": "locdit_r8_l7", "kind": "locdit", "requests": 8, "branch": 7, "layers": 4},
        # the operator itself at decode: the 24 attention calls of a batch-16 step over 8192 cached keys
        {"name": "attn_b16_kv8192", "kind": "attn", "batch": 16, "keys": 8192},
        # the operator itself at prefill: one sequence, causal mask, f16 keys and values
        {"name": "causal_1x4096", "kind": "causal", "batch": 1, "tokens": 4096},
        # the projections of eight layers with F16 weights (an unquantised model file) over a prompt
        {"name": "f16_weights_n337", "kind": "products", "tokens": 337},
    ]


def draw(rng):
    def spread(lo, hi):      # over the logarithm, ends included, odd sizes as likely as even ones
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["step", "step", "prompt", "prompt", "prompt", "solve", "locdit", "attn", "causal", "products"])
    if kind == "step":
        return {"kind": kind, "batch": spread(1, 16), "past": spread(16, 8190), "f16": rng.random() < 0.5}
    if kind == "prompt":
        return {"kind": kind, "batch": spread(1, 16), "tokens": spread(17, 4096), "f16": rng.random() < 0.5}
    if kind == "solve":
        patch = rng.choice([2, 3, 4])       # (the solver assembles a CFG pair of at most 16 tokens)
        return {"kind": kind, "layers": rng.choice([4, 8]), "patch": patch, "prefix": rng.randint(2, 7 - patch), "steps": rng.randint(4, 10)}
    if kind == "locdit":
        return {"kind": kind, "requests": spread(1, 32), "branch": rng.randint(5, 9), "layers": rng.choice([4, 8])}
    if kind == "attn":
        return {"kind": kind, "batch": spread(1, 16), "keys": spread(65, 8192)}
    if kind == "causal":
        return {"kind": kind, "batch": spread(1, 16), "tokens": spread(256, 4096)}
    return {"kind": kind, "tokens": spread(17, 2048)}


# ---- inputs -----------------------------------------------------------------------------------------------------------
def _randn(gen, *shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _q8_0(w):
    """Q8_0 rows (blocks of an f16 scale and 32 int8) of a float matrix, as uint8 (rows, K / 32 * 34)."""
    b = w.view(w.shape[0], -1, 32)
    d = b.abs().amax(2, keepdim=True) / 127.0
    q = torch.round(b * torch.where(d > 0, 1.0 / d, torch.zeros_like(d))).to(torch.int8)
    return torch.cat([d.to(torch.float16).view(torch.uint8), q.view(torch.uint8)], dim=2).view(w.shape[0], -1)


def _stack(gen, layers, batch, max_length, f16, mup):
    m = MiniCPMBackbone(n_layer=layers, max_length=max_length, batch=batch, use_mup=mup, kv_f16=f16)
    for li in range(layers):
        for name in WEIGHT_NAMES:
            m.set_weight(li, name, _q8_0(_randn(gen, *SHAPES[name]) * 0.02), SHAPES[name][1])
        for name in ("input_layernorm", "post_layernorm"):
            m.set_norm(li, name, 1.0 + 0.1 * _randn(gen, HIDDEN))
    m.set_norm(-1, "norm", 1.0 + 0.1 * _randn(gen, HIDDEN))
    m.rope_factors = 1.0 + torch.rand(HEAD_DIM // 2, generator=gen, device="cuda")
    m.pin_weights()
    return m


def _causal_mask(n):
    return torch.triu(torch.full((n, n), float("-inf"), dtype=torch.float16, device="cuda"), 1)


_side = []


def _recorded(fn):
    """fn's launches as a HIP graph (two plain runs first: the library's workspace grows then, not under the capture)."""
    if not _side:
        _side.append(torch.cuda.Stream())
    side = _side[0]
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
        fn()
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    return graph.replay


def _slots(m, start, n):
    return [c[:, :, start:start + n] for c in m.k_cache + m.v_cache]


def prepare(case, seed):
    pkg.check(pkg.lib().vx_init(0), "vx_init")
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return globals()["_prepare_" + case["kind"]](case, gen)


def _prepare_step(case, gen):
    b, past = case["batch"], case["past"]
    m = _stack(gen, LAYERS, b, past + 1, case["f16"], True)
    for c in m.k_cache + m.v_cache:
        c[:, :, :past] = _randn(gen, b, KV_HEADS, past, HEAD_DIM)
    x = _randn(gen, b, 1, HIDDEN)
    run_plan, out = m.plan(x, 1, past)
    return {"run": _recorded(run_plan), "out": [out] + _slots(m, past, 1), "keep": (m, run_plan)}


def _prepare_prompt(case, gen):
    b, n = case["batch"], case["tokens"]
    m = _stack(gen, LAYERS, b, n, case["f16"], True)
    x, mask = _randn(gen, b, n, HIDDEN), _causal_mask(n)
    run_plan, out = m.plan(x, n, 0, mask)
    return {"run": run_plan, "out": [out] + _slots(m, 0, n), "keep": (m, mask)}


def _prepare_solve(case, gen):
    patch, prefix, steps = case["patch"], case["prefix"], case["steps"]
    dec = _stack(gen, case["layers"], 1, 2 * (1 + prefix + patch), False, False)
    proj = [(_q8_0(_randn(gen, m, k) * 0.02), k, 0.1 * _randn(gen, m)) for m, k in ((HIDDEN, FEAT), (HIDDEN, FEAT), (FEAT, HIDDEN))]
    solver = LocDiTCfmSolver(dec, FEAT, *proj)
    t = np.linspace(1.0, 0.0, steps + 1, dtype=np.float32)
    t_span = (t + (np.cos(np.pi / 2 * t) - 1 + t)).astype(np.float32)
    inputs = (_randn(gen, patch, FEAT), _randn(gen, HIDDEN), _randn(gen, prefix, FEAT), _randn(gen, steps, HIDDEN))
    run_plan, x = solver.plan(*inputs, t_span, cfg_value=2.0)
    return {"run": _recorded(run_plan), "out": [x], "keep": (solver, inputs, run_plan)}


def _prepare_locdit(case, gen):
    r, half = case["requests"], case["branch"]
    n = 2 * half
    m = _stack(gen, case["layers"], r, n, False, False)
    i = torch.arange(n, device="cuda")
    mask = torch.where((i[None, :] < half) != (i[:, None] < half), float("-inf"), 0.0).to(torch.float16).contiguous()
    x = _randn(gen, r, n, HIDDEN)
    run_plan, out = m.plan(x, n, 0, mask, write_kv=False, positions=(i % half).to(torch.int32))
    return {"run": _recorded(run_plan), "out": [out], "keep": (m, mask, run_plan)}


def _prepare_attn(case, gen):
    b, keys = case["batch"], case["keys"]
    caches = [[_randn(gen, b, KV_HEADS, keys, HEAD_DIM).half() for _ in range(2)] for _ in range(LAYERS)]
    qs = [_randn(gen, b, HEADS, 1, HEAD_DIM) for _ in range(LAYERS)]
    outs = [torch.empty((b, 1, HEADS, HEAD_DIM), device="cuda") for _ in range(LAYERS)]

    def calls():
        for q, (k, v), out in zip(qs, caches, outs):
            pkg.flash_attn_ext(q, k, v, None, SCALE, out=out)

    return {"run": _recorded(calls), "out": outs, "keep": (caches, qs, calls)}


def _prepare_causal(case, gen):
    b, n = case["batch"], case["tokens"]
    q = _randn(gen, b, HEADS, n, HEAD_DIM)
    k, v = (_randn(gen, b, KV_HEADS, n, HEAD_DIM).half() for _ in range(2))
    mask, out = _causal_mask(n), torch.empty((b, n, HEADS, HEAD_DIM), device="cuda")
    return {"run": lambda: pkg.flash_attn_ext(q, k, v, mask, SCALE, out=out), "out": [out]}


def _prepare_products(case, gen):
    n = case["tokens"]
    xs = {k: _randn(gen, n, k) for k in (HIDDEN, FFN)}
    todo = [((_randn(gen, *SHAPES[name]) * 0.02).half(), xs[SHAPES[name][1]], torch.empty((n, SHAPES[name][0]), device="cuda"))
            for _ in range(F16_LAYERS) for name in WEIGHT_NAMES]

    def calls():
        for w, x, out in todo:
            pkg.mul_mat(w, x, out=out)

    return {"run": _recorded(calls), "out": [out for _, _, out in todo], "keep": (todo, calls)}


def run(state):
    state["run"]()
    return state["out"]


# ---- what a pass cannot do without -----------------------------------------------------------------------------------
def _stack_work(layers, rows, es_written, attn_flops, kv_read_bytes):
    """layers x (every Q8_0 weight once, its products over `rows` tokens, attention), the hidden states in and out."""
    kv_values = rows * 2 * KV_HEADS * HEAD_DIM
    return {"bytes": layers * (LAYER_WEIGHTS * 34 // 32 + kv_read_bytes + kv_values * es_written) + 2 * rows * HIDDEN * 4,
            "flops": layers * (2 * LAYER_WEIGHTS * rows + attn_flops)}


def work(case):
    kind = case["kind"]
    if kind == "step":
        b, past, es = case["batch"], case["past"], 2 if case["f16"] else 4
        return _stack_work(LAYERS, b, es, 4 * b * HEADS * HEAD_DIM * (past + 1), 2 * b * KV_HEADS * HEAD_DIM * past * es)
    if kind == "prompt":
        b, n = case["batch"], case["tokens"]
        return _stack_work(LAYERS, b * n, 2 if case["f16"] else 4, 4 * b * HEADS * HEAD_DIM * n * (n + 1) // 2, 0)
    if kind == "solve":
        half = 1 + case["prefix"] + case["patch"]
        passes = case["steps"] - 1        # the first Euler step skips the estimator under CFG-zero-star
        one = _stack_work(case["layers"], 2 * half, 0, 2 * 4 * HEADS * HEAD_DIM * half * half, 0)
        return {"bytes": one["bytes"], "flops": passes * one["flops"]}      # (the weights stay in the caches between passes)
    if kind == "locdit":
        r, half = case["requests"], case["branch"]
        return _stack_work(case["layers"], 2 * r * half, 0, 2 * r * 4 * HEADS * HEAD_DIM * half * half, 0)
    if kind == "attn":
        b, keys = case["batch"], case["keys"]
        return {"bytes": LAYERS * b * (2 * KV_HEADS * keys * HEAD_DIM * 2 + 2 * HEADS * HEAD_DIM * 4), "flops": LAYERS * 4 * b * HEADS * HEAD_DIM * keys}
    if kind == "causal":
        b, n = case["batch"], case["tokens"]
        return {"bytes": b * n * (2 * HEADS * HEAD_DIM * 4 + 2 * KV_HEADS * HEAD_DIM * 2) + n * n * 2,
                "flops": 4 * b * HEADS * HEAD_DIM * n * (n + 1) // 2}
    n = case["tokens"]
    rows = sum(m for m, _ in SHAPES.values())
    return {"bytes": F16_LAYERS * (LAYER_WEIGHTS * 2 + n * rows * 4) + n * (HIDDEN + FFN) * 4, "flops": F16_LAYERS * 2 * LAYER_WEIGHTS * n}


def tolerance(case):
    """About four times what was measured: the larger of the distance to a float64 evaluation of the same inputs and of
    the change that one unit in the last place of the float inputs makes (it moves the roundings to f16 on the way:
    activations in front of a product, probabilities, f16 cache slots)."""
    if case["kind"] in ("attn", "causal"):      # 3.1e-4 / 8.1e-3 (f16 probabilities; the first causal rows see few keys)
        return {"rel": 1.2e-3, "max": 0.03}
    if case["kind"] == "products":              # 2.1e-4 / 1.1e-3
        return {"rel": 9e-4, "max": 4.5e-3}
    return {"rel": 1.7e-3, "max": 6e-3}         # stacks and solves: 4.3e-4 (cache slots of the last layers) / 1.5e-3
