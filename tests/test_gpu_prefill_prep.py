"""GPU: the launch in front of the prefill attention (csrc/fattn_prefill.hip, pf_prep_kernel): the cache write's stores and sums at
the edges of their forms -- 16 Ki units and 64 block totals a side, ragged last blocks -- and a slot that the attention reads."""
import pytest

from reflib import rng
from test_gpu_fused import dev, ok, say

pytestmark = pytest.mark.gpu


# 32 units of four values a token: 512 tokens are 16 Ki units (the last sum of one block), 2048 are 64 block totals
@pytest.mark.parametrize("B,T", [(1, 512), (1, 513), (4, 512), (3, 683), (1, 4097)])
@pytest.mark.parametrize("f16,aligned", [(False, True), (False, False), (True, True)])
def test_cache_write_forms(pkg, gpu, B, T, f16, aligned):
    import torch
    say(f"prefill cache write B={B} T={T} f16 cache={f16} aligned slots={aligned}")
    L, d = pkg.lib(), pkg.desc
    H, Hkv, D = 16, 2, 64
    g = rng("prep", B, T)
    q, k, v = (dev(g.standard_normal((B, T, h, D)).astype("float32")) for h in (H, Hkv, Hkv))
    cdt = torch.float16 if f16 else torch.float32
    pad = 0 if aligned else 1    # (F32 slots off the 16-byte boundaries are written and summed value by value)
    flat = [torch.zeros(B * Hkv * (T + 2) * D + 1, dtype=cdt, device="cuda") for _ in range(4)]
    kc1, vc1, kc2, vc2 = (f[pad:pad + B * Hkv * (T + 2) * D].view(B, Hkv, T + 2, D) for f in flat)
    slot = lambda c: c[:, :, 1:1 + T].transpose(1, 2)
    a, b = torch.empty((B, T, H, D), device="cuda"), torch.empty((B, T, H, D), device="cuda")
    qd, kd, vd = d(q.transpose(1, 2)), d(k.transpose(1, 2)), d(v.transpose(1, 2))
    ok(pkg, L.vx_flash_attn_ext(qd, kd, vd, None, None, d(a), 0.125, 0.0, 0.0, None), "flash_attn_ext")
    ok(pkg, L.vx_kv_store_sync(d(k), d(slot(kc1)), d(v), d(slot(vc1)), d(a), d(a), 0.25, 0.5, None), "kv_store_sync")
    assert L.vx_supports_flash_attn_ext_store(qd, kd, vd, None, d(k), d(slot(kc2)), d(v), d(slot(vc2)), d(b), 0.0) == 1
    ok(pkg, L.vx_flash_attn_ext_store(qd, kd, vd, None, None, d(k), d(slot(kc2)), d(v), d(slot(vc2)), d(b), 0.125, 0.0, 0.0, 0.25, 0.5, None), "store")
    torch.cuda.synchronize()
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2) and torch.equal(a, b)


def test_attention_reads_the_written_slots(pkg, gpu):
    """F32 K / V that lie in the slots being written: the write comes first, as it does for F16 ones."""
    import torch
    say("prefill attention over the slots that its cache write fills")
    L, d = pkg.lib(), pkg.desc
    B, T, H, Hkv, D = 2, 640, 16, 2, 64
    g = rng("prep-alias")
    q, k, v = (dev(g.standard_normal((B, T, h, D)).astype("float32")) for h in (H, Hkv, Hkv))
    kc, vc = (torch.full((B, Hkv, T, D), 3.0, device="cuda") for _ in range(2))
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    slot = lambda c: c.transpose(1, 2)
    a, b = torch.empty((B, T, H, D), device="cuda"), torch.empty((B, T, H, D), device="cuda")
    ok(pkg, L.vx_flash_attn_ext_store(d(q.transpose(1, 2)), d(k.transpose(1, 2)), d(v.transpose(1, 2)), None, None, d(k), d(slot(kc2)), d(v), d(slot(vc2)),
                                      d(a), 0.125, 0.0, 0.0, 0.0, 0.0, None), "apart")
    ok(pkg, L.vx_flash_attn_ext_store(d(q.transpose(1, 2)), d(kc), d(vc), None, None, d(k), d(slot(kc)), d(v), d(slot(vc)), d(b), 0.125, 0.0, 0.0, 0.0, 0.0,
                                      None), "over the slots")
    torch.cuda.synchronize()
    assert torch.equal(kc, kc2) and torch.equal(vc, vc2) and torch.equal(a, b)


@pytest.mark.parametrize("B,T", [(1, 17), (1, 32), (1, 33), (1, 45), (2, 64), (1, 129), (3, 100), (1, 203), (1, 256), (5, 203), (12, 256), (13, 256)])
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("poison", [False, True])
def test_short_prompt_block(pkg, gpu, B, T, f16, poison):
    """A prompt's attention, cache write, o projection and update as one call against the calls it stands for, bit for bit."""
    import torch
    from test_gpu_fused import q8_dev
    say(f"short prompt's attention block as one call B={B} T={T} f16 cache={f16} poison={poison}")
    L, d = pkg.lib(), pkg.desc
    H, Hkv, D, hidden = 16, 2, 64, 1024
    g = rng("prep-short", B, T)
    q, k, v = (dev(g.standard_normal((B, T, h, D)).astype("float32")) for h in (H, Hkv, Hkv))
    if poison:
        v[B - 1, T // 2, 1, 3] = float("nan")
    res = dev(g.standard_normal((B * T, hidden)).astype("float32"))
    wd = pkg.desc_q8(w := q8_dev((0.05 * g.standard_normal((hidden, hidden))).astype("float32"))[0], hidden)
    mask = torch.full((T, T), float("-inf"), dtype=torch.float16, device="cuda").triu(1).contiguous()
    kc1, vc1, kc2, vc2 = (torch.zeros((B, Hkv, T + 3, D), dtype=torch.float16 if f16 else torch.float32, device="cuda") for _ in range(4))
    slot = lambda c: c[:, :, 2:2 + T].transpose(1, 2)
    qkv = [d(t.transpose(1, 2)) for t in (q, k, v)]
    a, o1 = torch.empty((B, T, H, D), device="cuda"), torch.empty_like(res)
    ok(pkg, L.vx_flash_attn_ext(*qkv, d(mask), None, d(a), 0.125, 0.0, 0.0, None), "flash_attn_ext")
    ok(pkg, L.vx_kv_store_sync(d(k), d(slot(kc1)), d(v), d(slot(vc1)), d(a), d(a), 0.25, 0.5, None), "kv_store_sync")
    ok(pkg, L.vx_mul_mat_scale_add(wd, d(a.view(B * T, hidden)), d(res), d(o1), 0.7, pkg.ACT_FLOAT, None), "mul_mat_scale_add")
    b, o2 = torch.full((B * T, hidden), 7.0, device="cuda"), torch.full_like(res, 5.0)
    tail = (d(k), d(slot(kc2)), d(v), d(slot(vc2)), d(b), wd, d(res), d(o2))
    one = L.vx_supports_flash_attn_ext_store_proj(*qkv, d(mask), *tail, 0.0, pkg.ACT_FLOAT)
    assert one == (B * T <= 3072)   # (the product kernel's last token count)
    ok(pkg, L.vx_flash_attn_ext_store_proj(*qkv, d(mask), None, *tail, 0.125, 0.0, 0.0, 0.25, 0.5, 0.7, pkg.ACT_FLOAT, None), "one call")
    torch.cuda.synchronize()
    assert torch.equal(kc1.view(torch.uint8), kc2.view(torch.uint8)) and torch.equal(vc1.view(torch.uint8), vc2.view(torch.uint8))
    assert torch.equal(torch.isnan(o1), torch.isnan(o2)) and torch.equal(o1.nan_to_num(3.0), o2.nan_to_num(3.0))
    assert bool(torch.isnan(o2).any()) == poison and (not one or bool((b == 7.0).all()))


@pytest.mark.parametrize("B,T,H,M", [(2, 1536, 64, 8192), (2, 600, 16, 1024), (3, 517, 16, 1000)])
@pytest.mark.parametrize("batched", [True, False])
def test_prefill_block_by_sequence(pkg, gpu, B, T, H, M, batched):
    """Attention, cache write, o projection and update as one call, the attention's result a batch of sequences or flattened: the bits
    of the three calls either way, whichever product kernel a single call of that shape runs on."""
    import torch
    from test_gpu_fused import q8_dev
    say(f"prefill attention block as one call B={B} T={T} heads={H} rows={M} batched={batched}")
    L, d = pkg.lib(), pkg.desc
    Hkv, D, hidden = H // 8, 64, H * 64
    g = rng("prep-batch", B, T, H)
    q, k, v = (dev(g.standard_normal((B, T, h, D)).astype("float32")) for h in (H, Hkv, Hkv))
    shape = (B, 1, T, hidden) if batched else (B * T, hidden)
    res = dev(g.standard_normal((B, 1, T, M) if batched else (B * T, M)).astype("float32"))
    wd = pkg.desc_q8(w := q8_dev((0.05 * g.standard_normal((M, hidden))).astype("float32"))[0], hidden)
    kc1, vc1, kc2, vc2 = (torch.zeros((B, Hkv, T, D), device="cuda") for _ in range(4))
    slot = lambda c: c.transpose(1, 2)
    qkv = [d(t.transpose(1, 2)) for t in (q, k, v)]
    a, o1, b, o2 = torch.empty(shape, device="cuda"), torch.empty_like(res), torch.empty(shape, device="cuda"), torch.full_like(res, 5.0)
    ok(pkg, L.vx_flash_attn_ext(*qkv, None, None, d(a.view(B, T, H, D)), 0.125, 0.0, 0.0, None), "flash_attn_ext")
    ok(pkg, L.vx_kv_store_sync(d(k), d(slot(kc1)), d(v), d(slot(vc1)), d(a.view(B, T, H, D)), d(a.view(B, T, H, D)), 0.25, 0.5, None), "kv_store_sync")
    ok(pkg, L.vx_mul_mat_scale_add(wd, d(a), d(res), d(o1), 0.7, pkg.ACT_FLOAT, None), "mul_mat_scale_add")
    tail = (d(k), d(slot(kc2)), d(v), d(slot(vc2)), d(b), wd, d(res), d(o2))
    assert batched or L.vx_supports_flash_attn_ext_store_proj(*qkv, None, *tail, 0.0, pkg.ACT_FLOAT) == 1
    ok(pkg, L.vx_flash_attn_ext_store_proj(*qkv, None, None, *tail, 0.125, 0.0, 0.0, 0.25, 0.5, 0.7, pkg.ACT_FLOAT, None), "one call")
    torch.cuda.synchronize()
    assert torch.equal(kc1, kc2) and torch.equal(vc1, vc2) and torch.equal(o1, o2)
