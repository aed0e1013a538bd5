"""The resident stack launch (vx_stack_run) against the separate calls: the same bits, cache slots included."""
import os

import numpy as np
import pytest

import reflib
from reflib import rng

pytestmark = pytest.mark.gpu


def say(what):
    print(what, flush=True)


def build(gpu, layers, batch, max_length, f16, mup=True, **dims):
    import torch
    from voxcpm_cpp_amd import backbone as bb
    m = bb.MiniCPMBackbone(n_layer=layers, max_length=max_length, batch=batch, use_mup=mup, kv_f16=f16, act_mode=gpu.ACT_FLOAT, **dims)
    H, q, kv, F = m.hidden, m.n_heads * 64, m.n_kv * 64, m.ffn
    shapes = {"q_proj": (q, H), "k_proj": (kv, H), "v_proj": (kv, H), "o_proj": (H, q), "gate_proj": (F, H), "up_proj": (F, H), "down_proj": (H, F)}
    for li in range(layers):
        for n, (r, k) in shapes.items():
            w = rng("stack", n, li, r, k).standard_normal((r, k)).astype(np.float32) * 0.02
            m.set_weight(li, n, torch.from_numpy(reflib.quantize_q8_0(w)).cuda().view(torch.uint8).view(r, -1), k)
        for n in ("input_layernorm", "post_layernorm"):
            m.set_norm(li, n, torch.from_numpy((1 + 0.1 * rng("stack", n, li).standard_normal(H)).astype(np.float32)).cuda())
    m.set_norm(-1, "norm", torch.from_numpy((1 + 0.1 * rng("stack", "norm").standard_normal(H)).astype(np.float32)).cuda())
    m.rope_factors = torch.from_numpy(rng("stack", "ff").uniform(1, 2, 32).astype(np.float32)).cuda()
    return m


def same(a, b):
    import torch
    return torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a.float().nan_to_num(7.0, 8.0, 9.0), b.float().nan_to_num(7.0, 8.0, 9.0))


@pytest.fixture
def env():
    keep = {k: os.environ.get(k) for k in ("VX_STACK", "VX_STACK_GROUPS")}
    yield os.environ
    for k, v in keep.items():
        if v is None:
            os.environ.pop(k, None)
        else:
            os.environ[k] = v


def both(env, m, x, T, past, mask=None, groups=(None,), **kw):
    """The separate calls, then the one launch with each number of work-groups: outputs and written slots."""
    import torch
    from voxcpm_cpp_amd import lib
    slots = lambda: [c[:, :, past:past + T].clone() for c in m.k_cache + m.v_cache] if kw.get("write_kv", True) else []
    res = []
    for g in ("separate",) + tuple(groups):
        env.pop("VX_STACK_GROUPS", None)
        env.pop("VX_STACK", None)
        if g == "separate":
            env["VX_STACK"] = "0"
        elif g:
            env["VX_STACK_GROUPS"] = str(g)
        if kw.get("write_kv", True):
            for c in m.k_cache + m.v_cache:
                c[:, :, past:past + T] = 0
        run, out = m.plan(x, T, past, mask, **kw)
        if g != "separate":
            assert lib().vx_supports_stack(m._stack(x, out, run._keep[0], T, past, mask, kw.get("write_kv", True), 1.0)), "the shape is one the launch takes"
        out.fill_(3.0)
        run()
        torch.cuda.synchronize()
        res.append((g, out.clone(), slots()))
    want = res[0]
    for g, o, c in res[1:]:
        assert same(want[1], o), f"{g}: output"
        assert all(same(p, q) for p, q in zip(want[2], c)), f"{g}: cache"
    return want[1]


# one key range up to 256 keys, several beyond; 64 / 65 keys: the f16 cache's two kernels; the step's own key opens a tile (past a
# multiple of 32) or closes one; 4 / 5 rows: the products' slots; 8 / 9 rows: a row a wave, sixteen waves
@pytest.mark.parametrize("batch,past,f16", [(1, 1, False), (1, 37, False), (1, 63, True), (1, 64, True), (2, 255, False), (2, 256, False), (4, 700, True),
                                            (5, 700, False), (8, 31, True), (8, 513, True), (9, 100, True), (9, 40, True), (16, 255, False), (16, 1000, True), (3, 8100, True)])
def test_decode_steps(gpu, env, batch, past, f16):
    import torch
    say(f"stack: {batch} sequences behind {past} keys, f16 cache {f16}")
    m = build(gpu, 2, batch, past + 1, f16)
    gen = torch.Generator(device="cuda").manual_seed(past)
    for c in m.k_cache + m.v_cache:
        c[:, :, :past] = torch.randn((batch, 2, past, 64), generator=gen, device="cuda")
    x = torch.randn((batch, 1, 1024), generator=gen, device="cuda")
    out = both(env, m, x, 1, past, groups=(None, 256, 255, 100) if past < 1000 else (None, 37))
    assert bool(torch.isfinite(out).all())


@pytest.mark.parametrize("batch,T,masked", [(1, 2, True), (1, 7, False), (1, 10, True), (1, 14, True), (2, 5, True), (3, 1, False)])
def test_sequences_without_a_cache(gpu, env, batch, T, masked):
    import torch
    say(f"stack: {batch} sequences of {T} tokens, mask {masked}")
    m = build(gpu, 3, batch, 16, False, mup=False)
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn((batch, T, 1024), generator=gen, device="cuda")
    i = torch.arange(T, device="cuda")
    mask = torch.where((i[None, :] * 2 < T) != (i[:, None] * 2 < T), float("-inf"), 0.0).to(torch.float16).contiguous() if masked else None
    out = both(env, m, x, T, 0, mask, groups=(None, 200, 1), write_kv=False, positions=(i % 5).to(torch.int32))
    assert bool(torch.isfinite(out).all())


def test_other_dimensions(gpu, env):
    """Four KV heads, half the FFN: other numbers of rows a work-group."""
    import torch
    say("stack: 16 / 4 heads, FFN 2048")
    m = build(gpu, 2, 3, 301, True, n_kv_heads=4, ffn=2048)
    gen = torch.Generator(device="cuda").manual_seed(3)
    for c in m.k_cache + m.v_cache:
        c[:, :, :300] = torch.randn((3, 4, 300, 64), generator=gen, device="cuda")
    both(env, m, torch.randn((3, 1, 1024), generator=gen, device="cuda"), 1, 300, groups=(None, 50))


@pytest.mark.parametrize("value", [float("inf"), "all ones"])
def test_values_that_are_no_numbers_arrive(gpu, env, value):
    """An activation that is infinite, or the NaN whose bits mark an empty slot of the exchange: every wait ends, NaN where the
    separate calls have NaN."""
    import torch
    say(f"stack: an input value {value}")
    m = build(gpu, 2, 2, 41, False)
    gen = torch.Generator(device="cuda").manual_seed(5)
    for c in m.k_cache + m.v_cache:
        c[:, :, :40] = torch.randn((2, 2, 40, 64), generator=gen, device="cuda")
    x = torch.randn((2, 1, 1024), generator=gen, device="cuda")
    if value == "all ones":
        x.view(torch.int32)[1, 0, 5] = -1
    else:
        x[1, 0, 5] = value
    both(env, m, x, 1, 40)


def test_first_call_under_a_capture_and_replays(gpu, env):
    """A stream whose first call is recorded: every replay clears the plan's exchange area."""
    import torch
    say("stack: captured and replayed")
    m = build(gpu, 2, 2, 301, True)
    gen = torch.Generator(device="cuda").manual_seed(6)
    for c in m.k_cache + m.v_cache:
        c[:, :, :300] = torch.randn((2, 2, 300, 64), generator=gen, device="cuda")
    x = torch.randn((2, 1, 1024), generator=gen, device="cuda")
    env["VX_STACK"] = "0"
    run, out = m.plan(x, 1, 300)
    run()
    torch.cuda.synchronize()
    want = out.clone()
    env.pop("VX_STACK")
    run, out = m.plan(x, 1, 300)
    s = torch.cuda.Stream()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        run()
    for _ in range(4):
        out.zero_()
        (torch.randn(1 << 20, device="cuda") * 2).sum().item()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_two_streams_at_once(gpu, env):
    """Two of these launches on streams of their own, together with other kernels: whoever gets fewer compute units gives the same bits."""
    import torch
    say("stack: two streams")
    env.pop("VX_STACK", None)
    gen = torch.Generator(device="cuda").manual_seed(8)
    jobs = []
    for i in range(2):
        m = build(gpu, 4, 2, 201, True)
        for c in m.k_cache + m.v_cache:
            c[:, :, :200] = torch.randn((2, 2, 200, 64), generator=gen, device="cuda")
        run, out = m.plan(torch.randn((2, 1, 1024), generator=gen, device="cuda"), 1, 200)
        run()
        torch.cuda.synchronize()
        jobs.append((torch.cuda.Stream(), run, out, out.clone(), m))
    noise = torch.randn(2048, 2048, device="cuda")
    torch.cuda.synchronize()
    for _ in range(5):
        for s, run, out, _, _ in jobs:
            with torch.cuda.stream(s):
                for _ in range(6):
                    run()
        noise = (noise * 1.0001).contiguous()
    torch.cuda.synchronize()
    for _, _, out, want, _ in jobs:
        assert torch.equal(out, want)


# A process of its own each, since the library reads the switch once.
MANY_TOKENS = """
import os, sys
sys.path[:0] = [{root!r}, {tests!r}]
import torch, __graft_entry__, test_gpu_stack as t
gpu = __graft_entry__.load_package()
gpu.check(gpu.lib().vx_init(0), "vx_init")
def taken(batch, T, past):
    m = t.build(gpu, 1, batch, past + T, True)
    x = torch.zeros((batch, T, 1024), device="cuda")
    pos = torch.arange(past, past + T, dtype=torch.int32, device="cuda")
    return m._stack(x, torch.empty_like(x), pos, T, past, None, past > 0, 1.0) is not None
print([taken(*s) for s in ((1, 1, 40), (4, 1, 40), (8, 1, 40), (9, 1, 40), (16, 1, 700), (1, 8, 0), (1, 9, 0), (2, 7, 0))])
"""


def test_slots_that_no_instance_has_are_refused(gpu):
    """VX_GEMV_MANY_TOKENS above the row count gives products of 9 to 16 rows eight slots; the launch for more than eight rows has sixteen."""
    import subprocess
    import sys
    say("stack: VX_GEMV_MANY_TOKENS")
    tests = os.path.dirname(os.path.abspath(__file__))
    code = MANY_TOKENS.format(root=os.path.dirname(tests), tests=tests)
    for many, want in ((None, [True] * 8), ("100", [True, True, True, False, False, True, False, False])):
        env = {k: v for k, v in os.environ.items() if k not in ("VX_GEMV_MANY_TOKENS", "VX_STACK")}
        if many:
            env["VX_GEMV_MANY_TOKENS"] = many
        got = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
        assert got.returncode == 0, got.stderr[-2000:]
        assert got.stdout.strip().splitlines()[-1] == str(want), (many, got.stdout)


def test_graphs_of_one_stream_replay_side_by_side(gpu, env):
    """Two plans recorded on the same stream and replayed on two others at once: a plan's exchange area is its own."""
    import torch
    say("stack: two graphs of one capture stream on two streams")
    env.pop("VX_STACK", None)
    gen = torch.Generator(device="cuda").manual_seed(9)
    side, jobs = torch.cuda.Stream(), []
    for i in range(2):
        m = build(gpu, 4, 2, 41, False)     # (one key range: nothing of the separate calls' lies in the workspace either)
        for c in m.k_cache + m.v_cache:
            c[:, :, :40] = torch.randn((2, 2, 40, 64), generator=gen, device="cuda")
        run, out = m.plan(torch.randn((2, 1, 1024), generator=gen, device="cuda"), 1, 40)
        run()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            run()
        jobs.append((torch.cuda.Stream(), g, out, out.clone(), m, run))
    for _ in range(5):
        for _, _, out, _, _, _ in jobs:
            out.zero_()
        torch.cuda.synchronize()
        for _ in range(8):
            for s, g, _, _, _, _ in jobs:
                with torch.cuda.stream(s):
                    g.replay()
        torch.cuda.synchronize()
        for _, _, out, want, _, _ in jobs:
            assert torch.equal(out, want)


def test_areas_that_do_not_fit_are_refused(gpu, env):
    import torch
    from voxcpm_cpp_amd import lib
    say("stack: the caller's area")
    env.pop("VX_STACK", None)
    m = build(gpu, 1, 2, 41, False)
    x = torch.zeros((2, 1, 1024), device="cuda")
    run, out = m.plan(x, 1, 40)
    st = m._stack(x, out, run._keep[0], 1, 40, None, True, 1.0)
    n = lib().vx_stack_area_bytes(st)
    area = torch.empty(n + 16, dtype=torch.uint8, device="cuda")
    assert n > 256
    for at, size in ((0, n), (area.data_ptr(), n - 1), (area.data_ptr() + 8, n)):
        assert lib().vx_stack_run_in(st, at, size, None) == 3   # VX_ERR_INVALID
    assert lib().vx_stack_run_in(st, area.data_ptr() + 16, n, None) == 0
    torch.cuda.synchronize()
    st.n_tokens = 17
    assert lib().vx_stack_area_bytes(st) == 0 and lib().vx_stack_run_in(st, area.data_ptr(), n, None) == 2


def test_ordering_scalar_is_the_graphs(gpu, env):
    """The sums over k and v are formed in another order than the separate calls': right where the scale is zero, refused elsewhere."""
    import torch
    from voxcpm_cpp_amd import lib
    say("stack: the ordering scalar's scale")
    env.pop("VX_STACK", None)
    m = build(gpu, 1, 2, 41, False)
    x = torch.zeros((2, 1, 1024), device="cuda")
    run, out = m.plan(x, 1, 40)
    st = m._stack(x, out, run._keep[0], 1, 40, None, True, 1.0)
    for scale, bias, want in ((0.0, 0.0, 1), (0.0, 0.5, 1), (0.125, 0.0, 0), (0.125, 0.5, 0), (float("nan"), 0.0, 0)):
        st.sync_scale, st.sync_bias = scale, bias
        assert lib().vx_supports_stack(st) == want, (scale, bias)


def test_norm_weights_of_another_layout_stay_with_the_separate_calls(gpu, env):
    """The launch reads dense F32 norm weights; what the separate calls refuse or read otherwise is not its own."""
    import torch
    say("stack: norm weights")
    env.pop("VX_STACK", None)
    m = build(gpu, 2, 2, 41, False)
    x = torch.zeros((2, 1, 1024), device="cuda")
    pos = torch.full((1,), 40, dtype=torch.int32, device="cuda")
    taken = lambda: m._stack(x, torch.empty_like(x), pos, 1, 40, None, True, 1.0) is not None
    assert taken()
    for li, name in ((-1, "norm"), (1, "input_layernorm"), (0, "post_layernorm")):
        good = m.final_norm if li < 0 else m.norms[li][name]
        for bad in (good[:8].contiguous(), good.half(), torch.stack([good, good], 1)[:, 0]):
            m.set_norm(li, name, bad)
            assert not taken(), (name, bad.dtype, bad.shape, bad.stride())
        m.set_norm(li, name, good)
    assert taken()


def test_a_plan_can_keep_the_separate_calls(gpu, env):
    import torch
    say("stack: resident = False")
    env.pop("VX_STACK", None)
    m = build(gpu, 2, 2, 41, False)
    gen = torch.Generator(device="cuda").manual_seed(11)
    for c in m.k_cache + m.v_cache:
        c[:, :, :40] = torch.randn((2, 2, 40, 64), generator=gen, device="cuda")
    x = torch.randn((2, 1, 1024), generator=gen, device="cuda")
    outs = []
    for resident in (True, False):
        m.resident = resident
        run, out = m.plan(x, 1, 40)
        areas = [t for t in run._keep if isinstance(t, torch.Tensor) and t.dtype == torch.uint8]
        assert len(areas) == int(resident)
        run()
        outs.append(out)
    torch.cuda.synchronize()
    assert torch.equal(*outs)


@pytest.mark.parametrize("n_kv,batch,past,f16", [(1, 4, 70, True), (1, 5, 40, False), (8, 4, 300, False), (8, 3, 33, True), (16, 1, 40, True), (16, 1, 20, False)])
def test_numbers_of_kv_heads(gpu, env, n_kv, batch, past, f16):
    """One to sixteen query heads to a KV head: other pairs a work-group, other columns of an attention unit."""
    import torch
    say(f"stack: 16 / {n_kv} heads, {batch} sequences behind {past} keys, f16 cache {f16}")
    m = build(gpu, 2, batch, past + 1, f16, n_kv_heads=n_kv)
    gen = torch.Generator(device="cuda").manual_seed(past)
    for c in m.k_cache + m.v_cache:
        c[:, :, :past] = torch.randn((batch, n_kv, past, 64), generator=gen, device="cuda")
    x = torch.randn((batch, 1, 1024), generator=gen, device="cuda")
    both(env, m, x, 1, past, groups=(None, 77))


def test_the_streams_workspace_as_area_grows_beside_a_capture(gpu, env):
    """vx_stack_run, whose area lies in the stream's workspace: recorded as the stream's first call, then replayed."""
    import torch
    from voxcpm_cpp_amd import lib
    say("stack: vx_stack_run captured on a fresh stream")
    env.pop("VX_STACK", None)
    m = build(gpu, 2, 3, 301, True)
    gen = torch.Generator(device="cuda").manual_seed(12)
    for c in m.k_cache + m.v_cache:
        c[:, :, :300] = torch.randn((3, 2, 300, 64), generator=gen, device="cuda")
    x = torch.randn((3, 1, 1024), generator=gen, device="cuda")
    run, out = m.plan(x, 1, 300)
    run()
    torch.cuda.synchronize()
    want = out.clone()
    st = m._stack(x, out, run._keep[0], 1, 300, None, True, 1.0)
    s, g = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        assert lib().vx_stack_run(st, torch.cuda.current_stream().cuda_stream) == 0
    for _ in range(4):
        out.zero_()
        (torch.randn(1 << 20, device="cuda") * 2).sum().item()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
