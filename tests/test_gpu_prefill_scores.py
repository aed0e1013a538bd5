"""GPU: prefill attention (csrc/fattn_prefill.hip, pf_kernel) against the same attention in float64: two teams of waves with one tile
or none for the second, an odd last tile, columns that one team or nobody sees, both sides of the rule's line; scores far below zero there and
in the decode kernel (csrc/fattn.hip, fattn_dec64_kernel)."""
import pytest

from reflib import rng
from test_gpu_fused import dev, say

pytestmark = pytest.mark.gpu

LOG2E = 1.44269504088896341


def check(q, k, v, mask, scale, sinks, got):
    """q (scaled, in the log2 domain) and k enter the kernel as f16: what is left are the probabilities' roundings."""
    import torch
    (B, H, n_q, _), Hkv, n_kv = q.shape, k.shape[1], k.shape[2]
    qh, kh = (q * torch.tensor(scale * LOG2E, dtype=torch.float32)).half().double(), k.half().double()
    for b in range(B):
        for h in range(H):
            s = qh[b, h] @ kh[b, h // (H // Hkv)].t().contiguous()
            if mask is not None:
                s = s + mask[0, 0].double() * LOG2E
            if sinks is not None:
                s = torch.cat([s, (sinks[h].double() * LOG2E).expand(n_q, 1)], 1)
            top = s.max(1, keepdim=True).values
            p = torch.exp2(s - torch.where(top == float("-inf"), torch.zeros_like(top), top))
            vv, tot = v[b, h // (H // Hkv)].double(), p.sum(1, keepdim=True)
            want = (p[:, :n_kv] @ vv) / torch.where(tot == 0, torch.ones_like(tot), tot)
            # a probability is off by 2^-10 of itself at most, in the sums above and below alike (2^-9 of |v - o|); the sum below is
            # formed in eight f16 additions of 2^-11 each (2^-8 of o).  A score of 2^10 and more has a 2^-13 step in fp32.
            bound = 2.0 ** -9 * (vv.abs().max() + want.abs()) + 2.0 ** -8 * want.abs() + 1e-5
            if bool((top.abs() > 1024).any()):
                far = (top.abs() > 1024) & (top != float("-inf"))
                bound = bound + far * 4 * 2.0 ** -24 * torch.where(far, top.abs(), torch.zeros_like(top)) * vv.abs().max()
            err = (got[b, :, h].double() - want).abs()
            assert bool((err <= bound).all()), (b, h, float((err - bound).max()), float(err.max()))


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("B,n_q,n", [(1, 300, 300), (4, 1200, 1200), (2, 1, 700), (1, 4, 2000)])
@pytest.mark.parametrize("case", ["scores below -128", "lowest finite mask"])
def test_first_scores_far_below_zero(pkg, gpu, B, n_q, n, case, f16):
    import torch
    say(f"attention {case}: {B} x {n_q}/{n} f16={f16}")
    g = rng("far", B, n_q, n)
    q, k, v = (dev(g.standard_normal((B, h, m, 64)).astype("float32")) for h, m in ((16, n_q), (2, n), (2, n)))
    mask = None
    if case == "lowest finite mask":
        mask = torch.zeros((1, 1, n_q, n), dtype=torch.float16, device="cuda")
        mask[0, 0, 3 % n_q::11] = -65504.0
    else:
        q[:, :, ::3] = -16.0
        k = k * 0.25 + 2.0      # every third row's scores lie around -16 * 2 * 64 / 8 = -256
    if f16:
        k, v = k.half(), v.half()
    check(q, k, v, mask, 0.125, None, gpu.flash_attn_ext(q, k, v, mask, 0.125))


def masks(kind, n_q, n_kv, g):
    import torch
    i, j = torch.arange(n_q)[:, None] + (n_kv - n_q), torch.arange(n_kv)[None]
    vis = {"causal": j <= i, "one tile": (j // 64 == min(3, (n_kv - 1) // 64)) & (i >= 0), "second team only": (j // 64 == 1) & (i % 3 > 0),
           "either team": (j // 64) % 2 == (i // 5) % 2, "hidden rows": (j <= i) & (i % 7 > 0), "all hidden": (j < 0) & (i >= 0), "values": j <= i + 100}[kind]
    m = torch.where(vis, torch.from_numpy(g.standard_normal((n_q, n_kv)).astype("float32")) if kind == "values" else torch.tensor(0.0), torch.tensor(float("-inf")))
    if kind == "either team":
        m[3::11] = -65504.0     # the lowest finite value is a value, not a hidden key
    return m.half().view(1, 1, n_q, n_kv).contiguous().cuda()


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("B,n_q,n_kv,kind,sinks", [
    (1, 512, 512, "causal", False), (1, 257, 64, "one tile", False), (1, 300, 333, "one tile", True), (1, 260, 100, "second team only", True),
    (2, 270, 460, "either team", False), (1, 523, 523, "hidden rows", True), (1, 256, 300, "all hidden", False), (1, 400, 777, "values", False),
    (1, 513, 1025, None, True), (1, 2048, 2048, "causal", False), (1, 2049, 2049, "causal", False), (2, 1170, 1170, "causal", False),
    (2, 1500, 1500, "causal", False), (2, 1700, 1700, "causal", False), (4, 520, 520, "causal", False), (1, 2049, 2049, None, False)])
def test_prefill_attention_by_two_teams(pkg, gpu, B, n_q, n_kv, kind, sinks, f16):
    import torch
    say(f"prefill attention, two teams: {B} x {n_q}/{n_kv} {kind} sinks={sinks} f16={f16}")
    H, Hkv, D, scale = 16, 2, 64, 0.125
    g = rng("teams", B, n_q, n_kv)
    q, k, v = (dev(g.standard_normal((B, h, n, D)).astype("float32")) for h, n in ((H, n_q), (Hkv, n_kv), (Hkv, n_kv)))
    if f16:
        k, v = k.half(), v.half()
    mask = masks(kind, n_q, n_kv, g) if kind else None
    sk = dev(g.standard_normal(H).astype("float32")) if sinks else None
    check(q, k, v, mask, scale, sk, gpu.flash_attn_ext(q, k, v, mask, scale, sinks=sk))


def wide_mask(kind, n):
    import torch
    i, j = torch.arange(n, device="cuda")[:, None], torch.arange(n, device="cuda")[None]
    vis = {"causal": j <= i, "all": j < n + 0 * i, "late hidden": (j <= i + n) & (i < n - n // 10), "early hidden": (j >= 0) & (i >= n // 5), "nothing": (j < 0) & (i >= 0),
           "window": (j <= i) & (j > i - 300), "prefix": (j <= i) | (j < n // 2), "values": j <= i + n}[kind]
    m = torch.where(vis, torch.randn((n, n), generator=torch.Generator(device="cuda").manual_seed(n), device="cuda") if kind == "values" else torch.tensor(0.0, device="cuda"),
                    torch.tensor(float("-inf"), device="cuda"))
    return m.half().view(1, 1, n, n).contiguous()


# more row blocks than compute units: 258 (two second teams with a block), 288, 376, 512, 264 dealt by XCD (8 KV heads); 532: one team
@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("B,H,Hkv,n,kind,sinks", [
    (1, 16, 2, 2064, "all", False), (1, 16, 2, 2065, "window", True), (1, 16, 2, 2300, "late hidden", False), (1, 16, 2, 2300, "early hidden", True),
    (1, 16, 2, 2300, "nothing", True), (1, 16, 2, 2300, "causal", False), (1, 16, 2, 2290, "prefix", False), (1, 16, 2, 3001, "values", False),
    (1, 16, 2, 4096, "all", False), (1, 16, 2, 4095, "window", False), (1, 8, 8, 4200, "all", False), (1, 8, 8, 4200, "early hidden", True), (1, 32, 4, 2113, "late hidden", False)])
def test_teams_with_a_row_block_each(pkg, gpu, B, H, Hkv, n, kind, sinks, f16):
    import torch
    say(f"prefill attention, a row block a team: {B} x {n} heads {H}/{Hkv} {kind} sinks={sinks} f16={f16}")
    g = rng("parted", B, n, H)
    q, k, v = (dev(g.standard_normal((B, h, n, 64)).astype("float32")) for h in (H, Hkv, Hkv))
    if f16:
        k, v = k.half(), v.half()
    mask = wide_mask(kind, n)
    sk = dev(g.standard_normal(H).astype("float32")) if sinks else None
    out = torch.full((B, n, H, 64), 7.0, device="cuda")
    check(q, k, v, mask, 0.125, sk, gpu.flash_attn_ext(q, k, v, mask, 0.125, sinks=sk, out=out))


@pytest.mark.parametrize("kind", ["all", "causal", "late hidden"])
def test_cache_write_with_a_row_block_a_team(pkg, gpu, kind):
    """The cache write's scalar joins both teams' rows: the bits of the call without a write (the scale is zero)."""
    import torch
    n, H, Hkv = 2300, 16, 2
    say(f"prefill attention with a cache write, a row block a team: {kind}")
    L, d = pkg.lib(), pkg.desc
    g = rng("parted store", n)
    q = dev(g.standard_normal((1, H, n, 64)).astype("float32"))
    k, v = (dev(g.standard_normal((1, n, Hkv, 64)).astype("float32")) for _ in range(2))
    mask = wide_mask(kind, n)
    kt, vt = k.transpose(1, 2), v.transpose(1, 2)
    want = gpu.flash_attn_ext(q, kt, vt, mask, 0.125)
    kc, vc = (torch.zeros((1, Hkv, n + 3, 64), device="cuda") for _ in range(2))
    kw, vw = kc[:, :, :n].transpose(1, 2), vc[:, :, :n].transpose(1, 2)
    got = torch.full_like(want, 7.0)
    assert L.vx_supports_flash_attn_ext_store(d(q), d(kt), d(vt), d(mask), d(k), d(kw), d(v), d(vw), d(got), 0.0) == 1
    pkg.check(L.vx_flash_attn_ext_store(d(q), d(kt), d(vt), d(mask), None, d(k), d(kw), d(v), d(vw), d(got), 0.125, 0.0, 0.0, 0.0, 0.0, None), "store")
    torch.cuda.synchronize()
    assert torch.equal(want, got) and torch.equal(kc[:, :, :n], kt) and torch.equal(vc[:, :, :n], vt)


@pytest.mark.parametrize("f16", [True, False])
@pytest.mark.parametrize("B,H,Hkv,n_q,n_kv,kind", [
    (1, 8, 8, 512, 512, "causal"), (2, 8, 4, 400, 431, "causal"), (1, 16, 16, 300, 333, "hidden rows"), (1, 8, 8, 513, 513, "either team"), (1, 8, 4, 1025, 1025, None),
    (8, 16, 4, 1024, 1024, "causal"), (8, 16, 4, 1000, 1030, "hidden rows"), (4, 8, 8, 2048, 2048, "causal"), (2, 12, 3, 512, 512, "causal")])
def test_blocks_of_many_rows(pkg, gpu, B, H, Hkv, n_q, n_kv, kind, f16):
    """Few heads to a KV head: more rows in a block than there are visibility bits in LDS (32), in blocks of 128 columns and of 256."""
    import torch
    say(f"prefill attention, blocks of many rows: {B} x {n_q}/{n_kv} heads {H}/{Hkv} {kind} f16={f16}")
    g = rng("many rows", B, n_q, n_kv, H, Hkv)
    q, k, v = (dev(g.standard_normal((B, h, n, 64)).astype("float32")) for h, n in ((H, n_q), (Hkv, n_kv), (Hkv, n_kv)))
    if f16:
        k, v = k.half(), v.half()
    mask = masks(kind, n_q, n_kv, g) if kind else None
    check(q, k, v, mask, 0.125, None, gpu.flash_attn_ext(q, k, v, mask, 0.125))
