"""GPU: products of some hundred tokens on the 96- and 112-token tiles of csrc/gemm_mid.hip (their last passes hold two and three token
tiles) and activation passes of several 1024-column pieces, against float64."""
import numpy as np
import pytest

from reflib import rng
from test_gpu_fused import dev, ok, q8_dev, say
from test_gpu_gemm_mid import dequant

pytestmark = pytest.mark.gpu


# 96 tokens a tile: 4096 rows x 337, 380; 112: 4096 x 203, 224 (both with a ragged and a whole last tile); K of 2, 3 and 4 pieces and a ragged one
@pytest.mark.parametrize("M,K,N", [(4096, 1024, 337), (4096, 1024, 384), (4096, 1024, 203), (4096, 1024, 224), (4064, 768, 333),
                                   (512, 4096, 33), (520, 2304, 31), (264, 3072, 65), (136, 3328, 50)])
@pytest.mark.parametrize("wtype", ["q8", "f16"])
def test_products_on_the_middle_tiles(pkg, gpu, M, K, N, wtype):
    import torch
    say(f"middle tiles M={M} K={K} N={N} weights={wtype}")
    L, d = pkg.lib(), pkg.desc
    g = rng("mid-tiles", M, K, N)
    w = (0.05 * g.standard_normal((M, K))).astype(np.float32)
    if wtype == "q8":
        wg, _ = q8_dev(w)
        wd, w64 = pkg.desc_q8(wg, K), dequant(wg.cpu().numpy(), K)
    else:
        wg = dev(w.astype(np.float16))
        wd, w64 = d(wg), w.astype(np.float16).astype(np.float64)
    x = g.standard_normal((N, K)).astype(np.float32)
    xd = dev(x)
    out = torch.full((N + 2, M), 7.0, dtype=torch.float32, device="cuda")   # rows past N must stay
    ok(pkg, L.vx_mul_mat(wd, d(xd), d(out[:N]), pkg.ACT_FLOAT, None), "mul_mat")
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert (got[N:] == 7.0).all()
    x16 = x.astype(np.float16).astype(np.float64)
    # fp32 sums of exact products: 32 terms inside an instruction, K / 128 scaled additions per group of blocks, four groups
    bound = (32 + K // 128 + 4) * 2.0 ** -24 * (np.abs(x16) @ np.abs(w64).T)
    assert (np.abs(got[:N] - x16 @ w64.T) <= bound + 1e-30).all()
