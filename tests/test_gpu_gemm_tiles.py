"""GPU: products, pairs and q/k/v groups on the 96- and 112-token tiles of csrc/gemm_mid.hip (their last passes hold two and three token
tiles) and on the 32 x 32 tile of three stages, and activation passes of several 1024-column pieces: products against float64, groups
against their separate calls.  Which tile each of the cases runs on is held by tests/test_cpu_gemm_tiles.py."""
import numpy as np
import pytest

from reflib import rng
from test_gpu_fused import dev, ok, q8_dev, same_bits, say
from test_gpu_gemm_mid import dequant, test_groups_equal_their_separate_calls as groups_equal_their_separate_calls

pytestmark = pytest.mark.gpu

# (ragged and whole last tiles) 96 tokens: 4096 rows x 337, 384, 333; 112: x 397, 448, 770; 32 x 32 with three stages (Q8_0): 520 x 2304 x 400, 3072 x 768 x 150;
# K of 2, 3 and 4 pieces and a ragged one
PRODUCTS = [(4096, 1024, 337), (4096, 1024, 384), (4064, 768, 333), (4096, 1024, 397), (4096, 1024, 448), (4088, 1024, 770), (520, 2304, 400), (3072, 768, 150),
            (4096, 1024, 203), (4096, 1024, 224), (512, 4096, 33), (520, 2304, 31), (264, 3072, 65), (136, 3328, 50)]
# rows of each matrix, tokens, weights
PAIRS = [(4096, 140, "q8"), (4096, 140, "f16"), (4096, 203, "q8"), (4096, 203, "f16"), (4096, 448, "q8"), (4064, 1030, "f16"), (5504, 17, "q8"), (5496, 31, "q8")]
# tokens of a sequence, sequences, weights
GROUPS = [(800, 1, "q8"), (411, 2, "f16"), (1153, 1, "q8"), (431, 3, "q8")]


@pytest.mark.parametrize("M,K,N", PRODUCTS)
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


@pytest.mark.parametrize("M,N,wtype", PAIRS)
def test_pairs_on_the_middle_tiles(pkg, gpu, M, N, wtype):
    """gate / up and SwiGLU as one call, the two products and the GLU as three."""
    import torch
    say(f"pairs on middle tiles M={M} N={N} weights={wtype}")
    L, d, K = pkg.lib(), pkg.desc, 1024
    g = rng("mid-pairs", M, N)
    keep = [(0.05 * g.standard_normal((M, K))).astype(np.float32) for _ in range(2)]
    keep = [q8_dev(w)[0] if wtype == "q8" else dev(w.astype(np.float16)) for w in keep]
    wg, wu = (pkg.desc_q8(w, K) if wtype == "q8" else d(w) for w in keep)
    x = dev(g.standard_normal((N, K)).astype(np.float32))
    gate, up, want = (torch.empty((N, M), dtype=torch.float32, device="cuda") for _ in range(3))
    got = torch.full((N + 2, M), 7.0, dtype=torch.float32, device="cuda")
    ok(pkg, L.vx_mul_mat(wg, d(x), d(gate), pkg.ACT_FLOAT, None), "gate")
    ok(pkg, L.vx_mul_mat(wu, d(x), d(up), pkg.ACT_FLOAT, None), "up")
    ok(pkg, L.vx_glu(pkg.GLU_SWIGLU, d(gate), d(up), d(want), 0, None), "glu")
    ok(pkg, L.vx_mul_mat_swiglu(wg, wu, d(x), d(got[:N]), pkg.ACT_FLOAT, None), "mul_mat_swiglu")
    torch.cuda.synchronize()
    assert same_bits(got[:N], want) and bool((got[N:] == 7.0).all())


@pytest.mark.parametrize("T,B,wtype", GROUPS)
def test_groups_on_the_middle_tiles(pkg, gpu, T, B, wtype):
    groups_equal_their_separate_calls(pkg, gpu, T, B, wtype)
