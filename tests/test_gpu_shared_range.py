"""GPU: attention by four waves that share a column tile's keys (csrc/fattn.hip, fattn_cols16_kernel's NW) against float64: waves
with one tile, two or none, ragged last tiles, a wave whose keys are all hidden, rows that see nothing, both sides of the rule."""
import pytest

from reflib import rng
from test_gpu_fused import dev, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("B,H,Hkv,n_q,n_kv,kind,sinks", [
    (1, 16, 2, 17, 33, "causal", False), (1, 16, 2, 45, 45, "causal", True), (1, 16, 2, 64, 65, "causal", False), (2, 16, 2, 96, 96, "hidden", True),
    (1, 16, 2, 97, 97, "causal", False), (1, 16, 2, 128, 128, "tiles", False), (1, 16, 2, 129, 129, "hidden", False), (1, 16, 2, 203, 203, "causal", False),
    (1, 16, 2, 250, 256, "values", True), (1, 4, 4, 33, 100, "tiles", False), (1, 6, 2, 40, 77, "causal", False), (2, 16, 2, 128, 128, "causal", False),
    (3, 16, 2, 86, 86, "causal", False), (1, 16, 2, 203, 203, None, True), (1, 16, 2, 40, 64, None, False), (2, 16, 1, 21, 255, None, False)])
def test_waves_share_a_range(pkg, gpu, B, H, Hkv, n_q, n_kv, kind, sinks, f16):
    import torch
    say(f"attention, waves share a range: {B} x {n_q}/{n_kv} heads {H}/{Hkv} {kind} sinks={sinks} f16={f16}")
    scale, log2e = 0.125, 1.44269504088896341
    g = rng("shared", B, n_q, n_kv)
    q, k, v = (dev(g.standard_normal((B, h, n, 64)).astype("float32")) for h, n in ((H, n_q), (Hkv, n_kv), (Hkv, n_kv)))
    if f16:
        k, v = k.half(), v.half()
    mask = None
    if kind:
        i, j = torch.arange(n_q)[:, None] + (n_kv - n_q), torch.arange(n_kv)[None]
        vis = {"causal": j <= i, "tiles": (j // 32 % 4 != 1) & (i % 9 > 0) | (j // 32 % 4 == 2), "hidden": (j <= i) & (i % 7 > 0), "values": j <= i + 40}[kind]
        m = torch.where(vis, torch.from_numpy(g.standard_normal((n_q, n_kv)).astype("float32")) if kind == "values" else torch.tensor(0.0), torch.tensor(float("-inf")))
        mask = m.half().view(1, 1, n_q, n_kv).contiguous().cuda()
    sk = dev(g.standard_normal(H).astype("float32")) if sinks else None
    got = gpu.flash_attn_ext(q, k, v, mask, scale, sinks=sk).double()
    streamed = f16 and mask is None and n_kv > 64      # (the streaming kernel's: f16 q and probabilities, none of this test's)
    for b in range(B):
        for h in range(H):
            qq, kk, vv = q[b, h].double(), k[b, h // (H // Hkv)].double(), v[b, h // (H // Hkv)].double()
            s = qq @ kk.t().contiguous() * scale
            size = (qq.abs() @ kk.abs().t().contiguous()).max() * scale
            if mask is not None:
                s = s + mask[0, 0].double()
            if sk is not None:
                s = torch.cat([s, sk[h].double().expand(n_q, 1)], 1)
            top = s.max(1, keepdim=True).values
            p = torch.exp(s - torch.where(top == float("-inf"), torch.zeros_like(top), top))
            tot = p.sum(1, keepdim=True)
            want = (p[:, :n_kv] @ vv) / torch.where(tot == 0, torch.ones_like(tot), tot)
            # q, k, the probabilities and v as two halves each (2^-22 lost) and fp32 sums: a score is off by 2^-20 of its terms' sum at
            # most, a weight by twice that of itself, the result by 2^-20 of v more.  The streaming kernel rounds q and the weights to f16.
            bound = (2.0 ** -10 * (2 + size) if streamed else 2.0 ** -20 * (2 * size + 1)) * vv.abs().max()
            err = (got[b, :, h] - want).abs().max()
            assert float(err) <= float(bound), (b, h, float(err), float(bound))


@pytest.mark.parametrize("kinds", ["f32", "f16", "f16 cache, f32 step"])
@pytest.mark.parametrize("B,H,Hkv,T,n_past,masked", [
    (1, 16, 2, 40, 100, True), (2, 16, 2, 17, 17, True), (1, 16, 2, 33, 160, False), (1, 16, 2, 64, 31, True), (1, 16, 2, 20, 128, True),
    (1, 16, 2, 100, 5, True), (1, 6, 2, 45, 66, False), (1, 16, 2, 128, 128, True), (2, 16, 2, 127, 129, True), (3, 16, 2, 86, 50, True),
    (1, 16, 2, 17, 47, True), (1, 16, 2, 17, 48, True), (1, 16, 2, 16, 100, True)])
def test_two_segments_are_shared_as_one(pkg, gpu, B, H, Hkv, T, n_past, masked, kinds):
    """Cached keys and the step's own as two pairs of tensors against the two joined: the same bits, on both sides of the rule (17 rows,
    33 / 65 keys, 256 tiles), with the boundary on a multiple of 32, beside it, in the first tile and in each wave's tiles."""
    import torch
    say(f"attention over two segments, waves share a range: {B} x {T}/{n_past}+{T} heads {H}/{Hkv} mask={masked} {kinds}")
    L, d, n_kv = pkg.lib(), pkg.desc, n_past + T
    g = rng("shared2", B, T, n_past)
    first = torch.float32 if kinds == "f32" else torch.float16
    second = torch.float16 if kinds == "f16" else torch.float32
    q = dev(g.standard_normal((B, H, T, 64)).astype("float32"))
    kp, vp = (dev(g.standard_normal((B, Hkv, n_past + 7, 64)).astype("float32")).to(first)[:, :, :n_past] for _ in range(2))
    kc, vc = (dev(g.standard_normal((B, T, Hkv, 64)).astype("float32")).to(second).transpose(1, 2) for _ in range(2))
    i, j = torch.arange(T)[:, None] + n_past, torch.arange(n_kv)[None]
    mask = torch.where((j <= i) & (i % 7 > 0), 0.0, float("-inf")).half().view(1, 1, T, n_kv).contiguous().cuda() if masked else None
    kall, vall = (torch.cat([p, c.to(first)], 2).contiguous() for p, c in ((kp, kc), (vp, vc)))
    want = gpu.flash_attn_ext(q, kall, vall, mask, 0.125)
    got = torch.full_like(want, 3.0)
    assert L.vx_supports_flash_attn_ext_kv2(d(q), d(kp), d(kc), d(vp), d(vc), d(mask), d(got)) == 1
    pkg.check(L.vx_flash_attn_ext_kv2(d(q), d(kp), d(kc), d(vp), d(vc), d(mask), None, d(got), 0.125, 0.0, 0.0, None), "kv2")
    torch.cuda.synchronize()
    assert torch.equal(want, got)
