"""GPU: the product kernel for 17 to 3072 tokens (F16 weights: 1152) (csrc/gemm_mid.hip) at the edges of its tiles -- ragged token and row tiles,
the shortest and longest K it takes, a batch, both weight types -- and the groups built on it against their separate calls."""
import ctypes as C

import numpy as np
import pytest

from reflib import rng
from test_gpu_fused import dev, ok, q8_dev, same_bits, say

pytestmark = pytest.mark.gpu


def dequant(q, K):
    b = q.reshape(q.shape[0], K // 32, 34)
    d = np.ascontiguousarray(b[:, :, :2]).view(np.float16).astype(np.float64)
    return (np.ascontiguousarray(b[:, :, 2:]).view(np.int8).astype(np.float64) * d).reshape(q.shape[0], K)


@pytest.mark.parametrize("M,K,N,nb", [(16, 1024, 17, 1), (1000, 1024, 33, 1), (128, 768, 64, 2), (1024, 1024, 203, 1), (40, 2304, 31, 3),
                                      (1024, 4096, 129, 1), (520, 4096, 17, 1), (4096, 1024, 65, 1), (1024, 1024, 1024, 1), (72, 16384, 100, 1),
                                      (136, 1024, 1152, 1), (136, 1024, 1153, 1), (72, 4096, 1536, 2), (136, 1024, 3073, 1)])
@pytest.mark.parametrize("wtype", ["q8", "f16"])
def test_products(pkg, gpu, monkeypatch, M, K, N, nb, wtype):
    import torch
    say(f"product of some tens of tokens M={M} K={K} N={N} batch={nb} weights={wtype}")
    L, d = pkg.lib(), pkg.desc
    g = rng("mid", M, K, N, nb)
    w = (0.05 * g.standard_normal((M, K))).astype(np.float32)
    if wtype == "q8":
        wg, _ = q8_dev(w)
        wd, w64 = pkg.desc_q8(wg, K), dequant(wg.cpu().numpy(), K)
    else:
        wg = dev(w.astype(np.float16))
        wd, w64 = d(wg), w.astype(np.float16).astype(np.float64)
    x = g.standard_normal((nb, N, K)).astype(np.float32)
    xd = dev(x)
    out = torch.full((nb, N + 2, M), 7.0, dtype=torch.float32, device="cuda")   # a strided destination: rows past N must stay
    dst = out[:, :N].unsqueeze(1) if nb > 1 else out[0, :N]
    ok(pkg, L.vx_mul_mat(wd, d(xd.unsqueeze(1) if nb > 1 else xd[0]), d(dst), pkg.ACT_FLOAT, None), "mul_mat")
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert (got[:, N:] == 7.0).all()
    x16 = x.astype(np.float16).astype(np.float64)
    # fp32 sums of exact products: 32 terms inside an instruction, K / 128 scaled additions per group of blocks, four groups
    bound = (32 + K // 128 + 4) * 2.0 ** -24 * np.einsum("bnk,mk->bnm", np.abs(x16), np.abs(w64), optimize=True)
    assert (np.abs(got[:, :N] - np.einsum("bnk,mk->bnm", x16, w64, optimize=True)) <= bound + 1e-30).all()
    # the residual update is the product's value, scaled and added with a rounding each
    res = dev(g.standard_normal((nb, N, M)).astype(np.float32))
    upd = torch.empty_like(res)
    v = (lambda t: t.unsqueeze(1)) if nb > 1 else (lambda t: t[0])
    ok(pkg, L.vx_mul_mat_scale_add(wd, d(v(xd)), d(v(res)), d(v(upd)), 0.7, pkg.ACT_FLOAT, None), "mul_mat_scale_add")
    torch.cuda.synchronize()
    prod = torch.from_numpy(got[:, :N]).cuda()
    assert same_bits(upd, (res + prod * np.float32(0.7)).contiguous())
    if K in (768, 1024) and M <= 1024 and N <= 448:   # the streaming kernel's shapes: the same order of every sum
        monkeypatch.setenv("VX_GEMM_MID", "0")
        old = torch.empty((nb, N, M), dtype=torch.float32, device="cuda")
        ok(pkg, L.vx_mul_mat(wd, d(v(xd)), d(v(old)), pkg.ACT_FLOAT, None), "mul_mat")
        torch.cuda.synchronize()
        assert same_bits(old, prod.contiguous())


@pytest.mark.parametrize("T,B", [(17, 1), (45, 1), (64, 1), (203, 1), (300, 3), (1024, 1)])
@pytest.mark.parametrize("wtype", ["q8", "f16"])
def test_groups_equal_their_separate_calls(pkg, gpu, T, B, wtype):
    """norm + q/k/v + rope and the MLP with its residual update, sequences flattened into one token dimension."""
    import torch
    say(f"layer groups of some tens of tokens T={T} B={B} weights={wtype}")
    L, d = pkg.lib(), pkg.desc
    K, H, Hkv, F, N = 1024, 16, 2, 4096, T * B
    g = rng("mid-groups", T, B)
    keep = []

    def weight(m, k):
        w = (0.05 * g.standard_normal((m, k))).astype(np.float32)
        t = q8_dev(w)[0] if wtype == "q8" else dev(w.astype(np.float16))
        keep.append(t)
        return pkg.desc_q8(t, k) if wtype == "q8" else d(t)

    wq, wk, wv, wg, wu, wd = weight(K, K), weight(128, K), weight(128, K), weight(F, K), weight(F, K), weight(K, F)
    x, nw = dev((2 * g.standard_normal((N, K))).astype(np.float32)), dev((1 + 0.1 * g.standard_normal(K)).astype(np.float32))
    pos, ff = dev((np.arange(T) + 5).astype(np.int32)), dev((1 + g.random(32)).astype(np.float32))
    new = lambda *s: torch.full(s, float("nan"), dtype=torch.float32, device="cuda")
    rope = (64, 2, 32768, 10000.0, 1.0, 0.0, 1.0, 32.0, 1.0)
    n, q1, k1, v1, q2, k2, v2 = new(N, K), new(B, T, H, 64), new(B, T, Hkv, 64), new(N, 128), new(B, T, H, 64), new(B, T, Hkv, 64), new(N, 128)
    ok(pkg, L.vx_rms_norm_mul(d(x), d(nw), d(n), 1e-5, None), "norm")
    for w, t, rot in ((wq, q1, True), (wk, k1, True), (wv, v1, False)):
        ok(pkg, L.vx_mul_mat(w, d(n), d(t.view(N, -1)), pkg.ACT_FLOAT, None), "mul_mat")
        if rot:
            ok(pkg, L.vx_rope(d(t), pos.data_ptr(), ff.data_ptr(), d(t), *rope, None), "rope")
    assert L.vx_supports_norm_qkv_proj_rope_tiled(d(x), d(nw), wq, wk, wv, d(q2), d(k2), d(v2), 64, 2, pkg.ACT_FLOAT) == 1
    ok(pkg, L.vx_norm_qkv_proj_rope(d(x), d(nw), 1e-5, wq, wk, wv, pos.data_ptr(), ff.data_ptr(), d(q2), d(k2), d(v2), *rope, pkg.ACT_FLOAT, None), "qkv")
    torch.cuda.synchronize()
    assert same_bits(q1, q2) and same_bits(k1, k2) and same_bits(v1, v2)
    gate, up, act, o1, o2 = new(N, F), new(N, F), new(N, F), new(N, K), new(N, K)
    ok(pkg, L.vx_mul_mat(wg, d(n), d(gate), pkg.ACT_FLOAT, None), "gate")
    ok(pkg, L.vx_mul_mat(wu, d(n), d(up), pkg.ACT_FLOAT, None), "up")
    ok(pkg, L.vx_glu(pkg.GLU_SWIGLU, d(gate), d(up), d(act), 0, None), "glu")
    ok(pkg, L.vx_mul_mat_scale_add(wd, d(act), d(x), d(o1), 0.3, pkg.ACT_FLOAT, None), "down")
    assert L.vx_supports_mlp_tiled(d(x), d(nw), wg, wu, wd, d(x), d(o2), pkg.ACT_FLOAT) == 1
    ok(pkg, L.vx_mlp_tiled(d(x), d(nw), 1e-5, wg, wu, wd, d(x), 0.3, d(o2), pkg.ACT_FLOAT, None), "mlp_tiled")
    torch.cuda.synchronize()
    assert same_bits(o1, o2)


@pytest.mark.parametrize("T,B,wtype", [(1500, 2, "q8"), (3072, 1, "q8"), (1152, 1, "f16")])
def test_groups_at_the_last_token_counts(pkg, gpu, T, B, wtype):
    test_groups_equal_their_separate_calls(pkg, gpu, T, B, wtype)


@pytest.mark.parametrize("N", [45, 100, 300, 1024])
def test_kernel_switches_mean_what_they_say(pkg, gpu, monkeypatch, N):
    """The switches that name another kernel, at shapes of this one: VX_GEMM_LDS=2 rounds q * d once to f16 on the tiled kernels, 0 is the
    register-operand kernels, VX_GEMM_Q8T chooses between the prefill kernels; a switch set to its default changes nothing."""
    import torch
    say(f"kernel switches at N={N}")
    L, d = pkg.lib(), pkg.desc
    K, M = 4096, 1024
    g = rng("mid-switches", N)
    w = (0.05 * g.standard_normal((M, K))).astype(np.float32)
    wd = pkg.desc_q8(wq := q8_dev(w)[0], K)
    x = dev(g.standard_normal((N, K)).astype(np.float32))

    def product(**env):
        for name in ("VX_GEMM_MID", "VX_GEMM_LDS", "VX_GEMM_Q8T"):
            monkeypatch.delenv(name, raising=False)
        for name, value in env.items():
            monkeypatch.setenv(name, value)
        out = torch.empty((N, M), dtype=torch.float32, device="cuda")
        ok(pkg, L.vx_mul_mat(wd, d(x), d(out), pkg.ACT_FLOAT, None), "mul_mat")
        torch.cuda.synchronize()
        return out

    plain = product()
    for name, value in (("VX_GEMM_MID", "1"), ("VX_GEMM_LDS", "1"), ("VX_GEMM_Q8T", "1")):
        assert same_bits(plain, product(**{name: value})), (name, value)
    for value in ("0", "2"):
        assert same_bits(product(VX_GEMM_LDS=value), product(VX_GEMM_LDS=value, VX_GEMM_MID="0")), value
        if N >= 1024:
            assert same_bits(product(VX_GEMM_Q8T=value), product(VX_GEMM_Q8T=value, VX_GEMM_MID="0")), value
    # the folded scale is another rounding of every weight: about 2^-12 of the result away, the sums' order some 2^-22
    x16, w64 = x.half().double(), torch.from_numpy(dequant(wq.cpu().numpy(), K)).cuda()
    away = lambda t: float((t.double() - x16 @ w64.T).norm() / (x16 @ w64.T).norm())
    assert away(plain) < 1e-6 and away(product(VX_GEMM_LDS="2")) > 2e-5


@pytest.mark.parametrize("K,M,N,wtype", [(1024, 1024, 45, "q8"), (1024, 1024, 1100, "q8"), (1024, 4096, 1100, "f16")])
def test_first_call_of_a_stream_under_capture(pkg, gpu, K, M, N, wtype):
    """Products whose other kernels use no scratch memory: a graph may begin with one on a stream that never ran anything, and so may
    the gate/up pair.  Replayed with direct calls of another size (the workspace grows) between the replays."""
    import torch
    say(f"capture without a reservation K={K} M={M} N={N} weights={wtype}")
    L, d = pkg.lib(), pkg.desc
    g = rng("mid-capture", K, M, N)
    keep = []

    def weight():
        w = (0.05 * g.standard_normal((M, K))).astype(np.float32)
        keep.append(q8_dev(w)[0] if wtype == "q8" else dev(w.astype(np.float16)))
        return pkg.desc_q8(keep[-1], K) if wtype == "q8" else d(keep[-1])

    w, up = weight(), weight()
    x, big = (dev(g.standard_normal((n, K)).astype(np.float32)) for n in (N, 1152))
    want, want2, out, out2, other = (torch.zeros(n, M, device="cuda") for n in (N, N, N, N, 1152))
    ok(pkg, L.vx_mul_mat(w, d(x), d(want), pkg.ACT_FLOAT, None), "direct")
    ok(pkg, L.vx_mul_mat_swiglu(w, up, d(x), d(want2), pkg.ACT_FLOAT, None), "direct pair")
    torch.cuda.synchronize()
    s = C.c_void_p()        # (a stream of its own: torch's come from a pool and may have a workspace already)
    ok(pkg, L.vx_stream_create(C.byref(s)), "stream")
    ok(pkg, L.vx_graph_begin(s), "begin")
    rc = L.vx_mul_mat(w, d(x), d(out), pkg.ACT_FLOAT, s), L.vx_mul_mat_swiglu(w, up, d(x), d(out2), pkg.ACT_FLOAT, s)
    graph = C.c_void_p()
    ok(pkg, L.vx_graph_end(s, C.byref(graph)), "end")
    assert rc == (0, 0) and graph.value
    for _ in range(3):
        out.zero_(), out2.zero_()
        torch.cuda.synchronize()
        ok(pkg, L.vx_graph_launch(graph, s), "replay")
        ok(pkg, L.vx_stream_synchronize(s), "sync")
        assert same_bits(out, want) and same_bits(out2, want2)
        ok(pkg, L.vx_mul_mat(w, d(big), d(other), pkg.ACT_FLOAT, s), "direct call between")
        ok(pkg, L.vx_stream_synchronize(s), "sync")
    ok(pkg, L.vx_graph_destroy(graph), "graph")
    ok(pkg, L.vx_stream_destroy(s), "stream")
    # the same under a capture that forbids other threads' unsafe calls as well (torch's)
    ok(pkg, L.vx_stream_create(C.byref(s)), "stream")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=torch.cuda.ExternalStream(s.value)):
        rc = L.vx_mul_mat(w, d(x), d(out), pkg.ACT_FLOAT, s)
    assert rc == 0
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert same_bits(out, want)
    del g
    ok(pkg, L.vx_stream_destroy(s), "stream")


@pytest.mark.parametrize("M,last,wtype", [(1024, 192, "q8"), (4096, 48, "q8"), (1024, 64, "f16"), (128, 1024, "f16")])
def test_small_products_keep_the_streaming_kernel(pkg, gpu, monkeypatch, M, last, wtype):
    """Where both kernels give the same bits the streaming one runs up to `last` tokens: it needs no scratch memory, so a stream that
    never ran anything else still has none.  The two sides of the line against the streaming kernel alone."""
    import torch
    say(f"streaming kernel up to {last} tokens x {M} rows, weights={wtype}")
    L, d = pkg.lib(), pkg.desc
    K = 1024
    g = rng("mid-small", M, last)
    w = (0.05 * g.standard_normal((M, K))).astype(np.float32)
    wg = q8_dev(w)[0] if wtype == "q8" else dev(w.astype(np.float16))
    wd = pkg.desc_q8(wg, K) if wtype == "q8" else d(wg)
    for N in (17, last, last + 1):
        x, res = dev(g.standard_normal((N, K)).astype(np.float32)), dev(g.standard_normal((N, M)).astype(np.float32))
        out, upd, old, old_upd = (torch.empty(N, M, device="cuda") for _ in range(4))
        torch.cuda.synchronize()
        s, ptr, size = C.c_void_p(), C.c_void_p(), C.c_size_t()
        ok(pkg, L.vx_stream_create(C.byref(s)), "stream")
        ok(pkg, L.vx_mul_mat(wd, d(x), d(out), pkg.ACT_FLOAT, s), "mul_mat")
        ok(pkg, L.vx_mul_mat_scale_add(wd, d(x), d(res), d(upd), 0.7, pkg.ACT_FLOAT, s), "mul_mat_scale_add")
        ok(pkg, L.vx_stream_synchronize(s), "sync")
        ok(pkg, L.vx_workspace_info(s, C.byref(ptr), C.byref(size), None), "info")
        assert (size.value == 0) == (N <= last), (N, size.value)
        ok(pkg, L.vx_stream_destroy(s), "stream")
        with monkeypatch.context() as m:
            m.setenv("VX_GEMM_MID", "0")
            if M * N <= 256 * 1024 or (M <= 1024 and N <= 448):     # (what the streaming kernel takes at all)
                ok(pkg, L.vx_mul_mat(wd, d(x), d(old), pkg.ACT_FLOAT, None), "streaming")
                ok(pkg, L.vx_mul_mat_scale_add(wd, d(x), d(res), d(old_upd), 0.7, pkg.ACT_FLOAT, None), "streaming")
                torch.cuda.synchronize()
                assert same_bits(out, old) and same_bits(upd, old_upd), N


@pytest.mark.parametrize("K,M,N,wtype", [(1024, 8192, 2048, "q8"), (1024, 16384, 400, "q8"), (4096, 11264, 1024, "q8"), (4096, 128, 600, "q8"),
                                         (8192, 200, 45, "q8"), (1024, 50000, 97, "q8"), (1024, 8200, 500, "f16")])
def test_rows_that_other_kernels_serve(pkg, gpu, monkeypatch, K, M, N, wtype):
    """Wide matrices at many tokens and few rows with a long K: the kernels behind VX_GEMM_MID=0, alone and (where it is one call) as a pair."""
    import torch
    say(f"rows outside the mid-size kernel K={K} M={M} N={N} weights={wtype}")
    L, d = pkg.lib(), pkg.desc
    gen = torch.Generator(device="cuda").manual_seed(M + N)

    def weight():
        if wtype == "f16":
            w = (0.05 * torch.randn(M, K, generator=gen, device="cuda")).half()
            return w, d(w)
        w = torch.randint(0, 256, (M, K // 32, 34), generator=gen, device="cuda", dtype=torch.uint8)
        w[:, :, :2] = torch.tensor([0, 0x10], dtype=torch.uint8, device="cuda")     # scales of 2^-11
        w = w.view(M, -1)
        return w, pkg.desc_q8(w, K)

    (w, wd), (u, ud) = weight(), weight()
    x = torch.randn(N, K, generator=gen, device="cuda")
    outs = []
    for mid in (None, "0"):
        if mid:
            monkeypatch.setenv("VX_GEMM_MID", mid)
        out, pair = torch.full((N, M), 5.0, device="cuda"), torch.full((N, M), 5.0, device="cuda")
        ok(pkg, L.vx_mul_mat(wd, d(x), d(out), pkg.ACT_FLOAT, None), "mul_mat")
        if L.vx_supports_mul_mat_swiglu_tiled(wd, ud, d(x), d(pair), pkg.ACT_FLOAT):
            ok(pkg, L.vx_mul_mat_swiglu(wd, ud, d(x), d(pair), pkg.ACT_FLOAT, None), "pair")
        torch.cuda.synchronize()
        outs.append((out, pair))
    assert same_bits(outs[0][0], outs[1][0]) and same_bits(outs[0][1], outs[1][1])


# (rows wide enough for the pre-tiled kernel on the side that is not the mid-size kernel's: K 512, an ffn width off the 256s)
@pytest.mark.parametrize("K,F,M,N", [(1024, 5504, 5504, 3072), (512, 11008, 5632, 3000), (1024, 5632, 5504, 3072)])
def test_mlp_with_one_product_on_each_kernel(pkg, gpu, K, F, M, N):
    """norm + gate/up + SwiGLU + down + update as one call where the two products by themselves run on different kernels."""
    import torch
    say(f"mlp K={K} ffn={F} rows={M} tokens={N}")
    L, d = pkg.lib(), pkg.desc
    gen = torch.Generator(device="cuda").manual_seed(F + N)

    def weight(m, k):
        w = torch.randint(0, 256, (m, k // 32, 34), generator=gen, device="cuda", dtype=torch.uint8)
        w[:, :, :2] = torch.tensor([0, 0x0c], dtype=torch.uint8, device="cuda")     # scales of 2^-12
        return w.view(m, -1)

    wg, wu, wd = weight(F, K), weight(F, K), weight(M, F)
    gd, ud, dd = pkg.desc_q8(wg, K), pkg.desc_q8(wu, K), pkg.desc_q8(wd, F)
    x, nw = torch.randn(N, K, generator=gen, device="cuda"), 1 + 0.1 * torch.randn(K, generator=gen, device="cuda")
    res = torch.randn(N, M, generator=gen, device="cuda")
    act, o1, o2 = torch.empty(N, F, device="cuda"), torch.empty(N, M, device="cuda"), torch.full((N, M), 5.0, device="cuda")
    ok(pkg, L.vx_norm_mul_mat_swiglu(d(x), d(nw), 1e-5, gd, ud, d(act), pkg.ACT_FLOAT, None), "pair")
    ok(pkg, L.vx_mul_mat_scale_add(dd, d(act), d(res), d(o1), 0.3, pkg.ACT_FLOAT, None), "down")
    assert L.vx_supports_mlp_tiled(d(x), d(nw), gd, ud, dd, d(res), d(o2), pkg.ACT_FLOAT) == 1
    ok(pkg, L.vx_mlp_tiled(d(x), d(nw), 1e-5, gd, ud, dd, d(res), 0.3, d(o2), pkg.ACT_FLOAT, None), "mlp")
    torch.cuda.synchronize()
    assert same_bits(o1, o2)


@pytest.mark.parametrize("F,N,shift", [(4096, 20, 4), (4096, 24, 2), (4096, 100, 4), (4096, 1500, 8), (5504, 3072, 4)])
@pytest.mark.parametrize("which", ["gate", "up"])
def test_pair_with_one_matrix_off_the_16_bytes(pkg, gpu, F, N, shift, which):
    """Taken as before and with the bits of gate and up by themselves, of which one runs on another kernel then; with the norm in front and
    with the down projection behind where those are one call."""
    import torch
    say(f"split pair ffn={F} tokens={N} shift={shift} {which}")
    L, d = pkg.lib(), pkg.desc
    K, M = 1024, 5504
    gen = torch.Generator(device="cuda").manual_seed(F + N)

    def weight(m, k, at=0):
        w = torch.randint(0, 256, (m, k // 32, 34), generator=gen, device="cuda", dtype=torch.uint8)
        w[:, :, :2] = torch.tensor([0, 0x0c], dtype=torch.uint8, device="cuda")
        flat = torch.zeros(w.numel() + 16, dtype=torch.uint8, device="cuda")
        flat[at:at + w.numel()] = w.view(-1)
        return flat[at:at + w.numel()].view(m, -1)

    wg, wu, wd = weight(F, K, shift if which == "gate" else 0), weight(F, K, shift if which == "up" else 0), weight(M, F)
    gd, ud, dd = pkg.desc_q8(wg, K), pkg.desc_q8(wu, K), pkg.desc_q8(wd, F)
    x, nw = torch.randn(N, K, generator=gen, device="cuda"), 1 + 0.1 * torch.randn(K, generator=gen, device="cuda")
    res = torch.randn(N, M, generator=gen, device="cuda")
    new = lambda m: torch.full((N, m), 5.0, device="cuda")
    n, want, got, got_n, o1, o2 = new(K), new(F), new(F), new(F), new(M), new(M)
    ok(pkg, L.vx_rms_norm_mul(d(x), d(nw), d(n), 1e-5, None), "norm")

    def apart(src):
        g, u, out = new(F), new(F), new(F)
        ok(pkg, L.vx_mul_mat(gd, d(src), d(g), pkg.ACT_FLOAT, None), "gate")
        ok(pkg, L.vx_mul_mat(ud, d(src), d(u), pkg.ACT_FLOAT, None), "up")
        ok(pkg, L.vx_glu(pkg.GLU_SWIGLU, d(g), d(u), d(out), 0, None), "glu")
        return out

    want = apart(x)
    ok(pkg, L.vx_mul_mat_swiglu(gd, ud, d(x), d(got), pkg.ACT_FLOAT, None), "pair")
    torch.cuda.synchronize()
    assert same_bits(got, want)
    if N in (20, 24, 3072):
        want = apart(n)
        ok(pkg, L.vx_norm_mul_mat_swiglu(d(x), d(nw), 1e-5, gd, ud, d(got_n), pkg.ACT_FLOAT, None), "norm + pair")
        torch.cuda.synchronize()
        assert same_bits(got_n, want)
    if N == 3072:
        ok(pkg, L.vx_mul_mat_scale_add(dd, d(want), d(res), d(o1), 0.3, pkg.ACT_FLOAT, None), "down")
        ok(pkg, L.vx_mlp_tiled(d(x), d(nw), 1e-5, gd, ud, dd, d(res), 0.3, d(o2), pkg.ACT_FLOAT, None), "mlp")
        torch.cuda.synchronize()
        assert same_bits(o1, o2)


@pytest.mark.parametrize("T,B", [(17, 3), (45, 2), (203, 2), (517, 2)])
@pytest.mark.parametrize("wtype", ["q8", "f16"])
@pytest.mark.parametrize("poison", [False, True])
def test_groups_by_sequence(pkg, gpu, T, B, wtype, poison):
    """norm + q/k/v + rope, k + v + rope and the MLP with the sequences in a dimension of their own and strided rows, against separate calls;
    a NaN and an infinity stay in their tokens."""
    import torch
    say(f"layer groups by sequence T={T} B={B} weights={wtype} poison={poison}")
    L, d = pkg.lib(), pkg.desc
    K, H, Hkv, F = 1024, 16, 2, 2304
    gen = torch.Generator(device="cuda").manual_seed(T * B)
    keep = []

    def weight(m, k):
        w = 0.05 * torch.randn(m, k, generator=gen, device="cuda")
        keep.append(q8_dev(w.cpu().numpy())[0] if wtype == "q8" else w.half())
        return pkg.desc_q8(keep[-1], k) if wtype == "q8" else d(keep[-1])

    wq, wk, wv, wg, wu, wd = weight(K, K), weight(128, K), weight(128, K), weight(F, K), weight(F, K), weight(K, F)
    wide = torch.randn(B, T + 2, K + 32, generator=gen, device="cuda")
    if poison:
        wide[0, T // 2, 5], wide[B - 1, T - 1, 7] = float("nan"), float("inf")
    x, nw = wide[:, :T, :K], 1 + 0.1 * torch.randn(K, generator=gen, device="cuda")
    x4 = x.unsqueeze(1)                                             # [K, T, 1, B]
    pos, ff = torch.arange(5, 5 + T, dtype=torch.int32, device="cuda"), 1 + torch.rand(32, generator=gen, device="cuda")
    rope = (64, 2, 32768, 10000.0, 1.0, 0.0, 1.0, 32.0, 1.0)
    new = lambda *s: torch.full(s, 9.0, device="cuda")
    n, q1, k1, v1, q2, k2, v2, k3, v3 = (new(B, 1, T, K), new(B, T, H, 64), new(B, T, Hkv, 64), new(B, 1, T, 128), new(B, T, H, 64), new(B, T, Hkv, 64),
                                         new(B, 1, T, 128), new(B, T, Hkv, 64), new(B, 1, T, 128))
    ok(pkg, L.vx_rms_norm_mul(d(x4), d(nw), d(n), 1e-5, None), "norm")
    for w, t in ((wq, q1), (wk, k1), (wv, v1)):
        ok(pkg, L.vx_mul_mat(w, d(n), d(t.view(B, 1, T, -1)), pkg.ACT_FLOAT, None), "mul_mat")
        if t is not v1:
            ok(pkg, L.vx_rope(d(t), pos.data_ptr(), ff.data_ptr(), d(t), *rope, None), "rope")
    ok(pkg, L.vx_norm_qkv_proj_rope(d(x4), d(nw), 1e-5, wq, wk, wv, pos.data_ptr(), ff.data_ptr(), d(q2), d(k2), d(v2), *rope, pkg.ACT_FLOAT, None), "qkv")
    ok(pkg, L.vx_kv_proj_rope(wk, wv, d(n), pos.data_ptr(), ff.data_ptr(), d(k3), d(v3), *rope, pkg.ACT_FLOAT, None), "kv")
    gate, up, act, o1, o2 = new(B, T, F), new(B, T, F), new(B, T, F), new(B, T, K), new(B, T, K)
    n3 = n[:, 0]
    ok(pkg, L.vx_mul_mat(wg, d(n3), d(gate), pkg.ACT_FLOAT, None), "gate")
    ok(pkg, L.vx_mul_mat(wu, d(n3), d(up), pkg.ACT_FLOAT, None), "up")
    ok(pkg, L.vx_glu(pkg.GLU_SWIGLU, d(gate), d(up), d(act), 0, None), "glu")
    ok(pkg, L.vx_mul_mat_scale_add(wd, d(act), d(x), d(o1), 0.3, pkg.ACT_FLOAT, None), "down")
    assert L.vx_supports_mlp_tiled(d(x), d(nw), wg, wu, wd, d(x), d(o2), pkg.ACT_FLOAT) == (B * T <= (3072 if wtype == "q8" else 1152))
    if B * T <= 1152 or wtype == "q8":
        ok(pkg, L.vx_mlp_tiled(d(x), d(nw), 1e-5, wg, wu, wd, d(x), 0.3, d(o2), pkg.ACT_FLOAT, None), "mlp")
    torch.cuda.synchronize()
    for a, b in ((q1, q2), (k1, k2), (v1, v2), (k1, k3), (v1, v3), (o1, o2)):
        assert torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a.nan_to_num(3.0, 4.0, 5.0), b.nan_to_num(3.0, 4.0, 5.0))
    bad = {(0, T // 2), (B - 1, T - 1)} if poison else set()
    assert {tuple(i) for i in torch.nonzero(~torch.isfinite(o2).all(2)).tolist()} == bad
    assert {tuple(i) for i in torch.nonzero(~torch.isfinite(v2[:, 0]).all(2)).tolist()} == bad
