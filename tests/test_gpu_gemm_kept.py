"""GPU: products of some hundred to a few thousand tokens from the kept tiles of pinned Q8_0 weights (csrc/gemm_mid.hip, gd_kernel):
the bits of the kernel that reads the Q8_0 rows, at whole and ragged row and token tiles, the shortest and a long K, a batch."""
import ctypes as C

import numpy as np
import pytest

from reflib import rng
from test_gpu_fused import dev, ok, q8_dev, same_bits, say

pytestmark = pytest.mark.gpu


def kept_bytes(L):
    v = [C.c_size_t() for _ in range(3)]
    L.vx_weights_info(*[C.byref(t) for t in v])
    return [t.value for t in v]


@pytest.mark.parametrize("M,K,N,nb", [(4096, 1024, 768, 1), (4096, 1024, 1024, 1), (4064, 768, 1001, 1), (6144, 1024, 513, 1), (1000, 1024, 3071, 1),
                                      (1024, 4096, 3072, 1), (2080, 2304, 450, 3), (4096, 1024, 65, 6)])
def test_products_from_kept_tiles(pkg, gpu, M, K, N, nb):
    import torch
    say(f"products from kept tiles M={M} K={K} N={N} batch={nb}")
    L, d = pkg.lib(), pkg.desc
    g = rng("kept", M, K, N, nb)
    raw = [q8_dev((0.05 * g.standard_normal((M, K))).astype(np.float32))[0] for _ in range(2)]
    pool = torch.stack(raw).contiguous()
    wd, wd2 = pkg.desc_q8(pool[0], K), pkg.desc_q8(pool[1], K)
    x, res = dev(g.standard_normal((nb, N, K)).astype(np.float32)), dev(g.standard_normal((nb, N, M)).astype(np.float32))
    v = (lambda t: t.unsqueeze(1)) if nb > 1 else (lambda t: t[0])

    def all_three():
        outs = [torch.full((nb, N, M), 7.0, dtype=torch.float32, device="cuda") for _ in range(3)]
        ok(pkg, L.vx_mul_mat(wd, d(v(x)), d(v(outs[0])), pkg.ACT_FLOAT, None), "mul_mat")
        ok(pkg, L.vx_mul_mat_scale_add(wd, d(v(x)), d(v(res)), d(v(outs[1])), 0.7, pkg.ACT_FLOAT, None), "mul_mat_scale_add")
        if L.vx_supports_mul_mat_swiglu_tiled(wd, wd2, d(v(x)), d(v(outs[2])), pkg.ACT_FLOAT):
            ok(pkg, L.vx_mul_mat_swiglu(wd, wd2, d(v(x)), d(v(outs[2])), pkg.ACT_FLOAT, None), "mul_mat_swiglu")
        torch.cuda.synchronize()
        return outs

    want = all_three()
    base = kept_bytes(L)
    pkg.check(L.vx_weights_pin(pool.data_ptr(), pool.numel()), "pin")
    try:
        for turn in range(2):   # the copies are made, then used again
            assert all(same_bits(a, b) for a, b in zip(want, all_three())), turn
        assert kept_bytes(L) != base
    finally:
        L.vx_weights_unpin(pool.data_ptr())


@pytest.mark.parametrize("T", [768, 1000, 1024, 2048])
def test_mlp_from_kept_tiles(pkg, gpu, T):
    """The whole MLP: the pair leaves its result as the down projection's tiles."""
    import torch
    say(f"MLP from kept tiles T={T}")
    L, d = pkg.lib(), pkg.desc
    K, F = 1024, 4096
    g = rng("kept-mlp", T)
    mk = lambda m, k: q8_dev((0.05 * g.standard_normal((m, k))).astype(np.float32))[0]
    pair, down = torch.stack([mk(F, K), mk(F, K)]).contiguous(), mk(K, F)
    wg, wu, wd = pkg.desc_q8(pair[0], K), pkg.desc_q8(pair[1], K), pkg.desc_q8(down, F)
    x, nw = dev((2 * g.standard_normal((T, K))).astype(np.float32)), dev((1 + 0.1 * g.standard_normal(K)).astype(np.float32))

    def mlp():
        out = torch.full((T, K), float("nan"), dtype=torch.float32, device="cuda")
        ok(pkg, L.vx_mlp_tiled(d(x), d(nw), 1e-5, wg, wu, wd, d(x), 0.3, d(out), pkg.ACT_FLOAT, None), "mlp_tiled")
        torch.cuda.synchronize()
        return out

    want = mlp()
    for t in (pair, down):
        pkg.check(L.vx_weights_pin(t.data_ptr(), t.numel()), "pin")
    try:
        assert same_bits(want, mlp()) and same_bits(want, mlp())
    finally:
        for t in (pair, down):
            L.vx_weights_unpin(t.data_ptr())


def test_copies_share_allocations(pkg, gpu):
    """The first product over each of many pinned matrices does not allocate by itself; rewriting one of them again and again, its neighbours'
    copies in use, takes no more and more memory, and all of it goes back when the range is unpinned."""
    import torch
    say("kept tiles: several copies to an allocation")
    L, d = pkg.lib(), pkg.desc
    M, K, N, W = 4096, 1024, 768, 9
    g = rng("kept-blocks")
    pool = torch.stack([q8_dev((0.05 * g.standard_normal((M, K))).astype(np.float32))[0] for _ in range(W)]).contiguous()
    spare = torch.stack([pool[1].clone(), pool[2].clone()])
    x = dev(g.standard_normal((N, K)).astype(np.float32))
    out = torch.empty((N, M), dtype=torch.float32, device="cuda")

    def product(w):
        ok(pkg, L.vx_mul_mat(pkg.desc_q8(w, K), d(x), d(out), pkg.ACT_FLOAT, None), "mul_mat")
        torch.cuda.synchronize()
        return out

    free = lambda: torch.cuda.mem_get_info()[0]
    want = [product(w).clone() for w in pool]
    start, copies = free(), kept_bytes(L)[1]
    pkg.check(L.vx_weights_pin(pool.data_ptr(), pool.numel()), "pin")
    try:
        seen = set()
        for w, r in zip(pool, want):
            assert same_bits(product(w), r)
            seen.add(free())
        assert kept_bytes(L)[1] == copies + W
        assert len(seen) <= 2 and start - min(seen) <= 300 << 20
        for turn in range(100):   # 100 more copies of 9 MB
            pool[0].copy_(spare[turn % 2])
            pkg.check(L.vx_weights_changed(pool[0].data_ptr(), pool[0].numel()), "changed")
            assert same_bits(product(pool[0]), want[1 + turn % 2]) and same_bits(product(pool[5]), want[5])
        assert kept_bytes(L)[1] == copies + W and start - free() <= 600 << 20
    finally:
        L.vx_weights_unpin(pool.data_ptr())
    assert kept_bytes(L)[1] == copies and free() >= start


def test_copy_filled_on_one_stream_read_on_another(pkg, gpu):
    import torch
    say("kept tiles: filled on one stream, read on another at once")
    L, d = pkg.lib(), pkg.desc
    M, K, N, W = 4096, 1024, 768, 6
    g = rng("kept-streams")
    pool = torch.stack([q8_dev((0.05 * g.standard_normal((M, K))).astype(np.float32))[0] for _ in range(W)]).contiguous()
    x = dev(g.standard_normal((N, K)).astype(np.float32))
    outs = torch.empty((3, W, N, M), dtype=torch.float32, device="cuda")
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]

    def product(i, w, stream):
        pkg.check(L.vx_mul_mat(pkg.desc_q8(pool[w], K), d(x), d(outs[i, w]), pkg.ACT_FLOAT, stream), "mul_mat")

    for s in streams:
        product(0, 0, s.cuda_stream)   # (the streams' workspaces)
    for w in range(W):
        product(0, w, None)
    torch.cuda.synchronize()
    pkg.check(L.vx_weights_pin(pool.data_ptr(), pool.numel()), "pin")
    try:
        for w in range(W):
            product(1, w, streams[w % 2].cuda_stream)
            product(2, w, streams[1 - w % 2].cuda_stream)
        torch.cuda.synchronize()
        assert same_bits(outs[0], outs[1]) and same_bits(outs[0], outs[2])
    finally:
        L.vx_weights_unpin(pool.data_ptr())
