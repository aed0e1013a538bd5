"""GPU: the launch in front of the prefill attention (csrc/fattn_prefill.hip, pf_prep_kernel): the cache write's stores and sums at
the edges of their forms -- 16 Ki units and 64 block totals a side, ragged last blocks -- and a slot that the attention reads."""
import pytest

from reflib import rng
from test_gpu_fused import dev, ok, say

pytestmark = pytest.mark.gpu


# 32 units of four values a token: 512 tokens are 16 Ki units (the last sum of one block), 2048 are 64 block totals
@pytest.mark.parametrize("B,T", [(1, 512), (1, 513), (4, 512), (3, 683), (1, 4097)])
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("aligned", [True, False])
def test_cache_write_forms(pkg, gpu, B, T, f16, aligned):
    import torch
    say(f"prefill cache write B={B} T={T} f16 cache={f16} aligned slots={aligned}")
    L, d = pkg.lib(), pkg.desc
    H, Hkv, D = 4, 2, 64
    g = rng("prep", B, T)
    q, k, v = (dev(g.standard_normal((B, T, h, D)).astype("float32")) for h in (H, Hkv, Hkv))
    cdt = torch.float16 if f16 else torch.float32
    pad = 0 if aligned or f16 else 1    # (F32 slots off the 16-byte boundaries are written and summed value by value)
    flat = [torch.zeros(B * Hkv * (T + 2) * D + 1, dtype=cdt, device="cuda") for _ in range(4)]
    kc1, vc1, kc2, vc2 = (f[pad:pad + B * Hkv * (T + 2) * D].view(B, Hkv, T + 2, D) for f in flat)
    slot = lambda c: c[:, :, 1:1 + T].transpose(1, 2)
    a, b = torch.empty((B, T, H, D), device="cuda"), torch.empty((B, T, H, D), device="cuda")
    qd, kd, vd = d(q.transpose(1, 2)), d(k.transpose(1, 2)), d(v.transpose(1, 2))
    ok(pkg, L.vx_flash_attn_ext(qd, kd, vd, None, None, d(a), 0.125, 0.0, 0.0, None), "flash_attn_ext")
    ok(pkg, L.vx_kv_store_sync(d(k), d(slot(kc1)), d(v), d(slot(vc1)), d(a), d(a), 0.25, 0.5, None), "kv_store_sync")
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
