"""GPU: prefill attention (csrc/fattn_prefill.hip, pf_kernel) against the same attention in float64; scores far below zero there and
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
