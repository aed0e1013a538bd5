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


# rows (of each matrix), K, tokens, batch; whether the single product and the pair run on gd_kernel (tests/test_cpu_gemm_tiles.py holds this
# against the rule): whole and ragged 256-row tiles of both, the shortest K and long ones, batches
PRODUCTS = [(4096, 1024, 768, 1, True, True), (4096, 1024, 1024, 1, True, True), (4064, 1024, 1001, 1, True, True), (6144, 1024, 513, 1, True, True),
            (1000, 1024, 3071, 1, True, False), (2784, 1024, 513, 1, False, True), (2048, 4096, 1857, 1, True, True), (2080, 2560, 450, 3, True, True),
            (4096, 1024, 65, 6, True, True), (1536, 8192, 2310, 1, True, True), (1024, 4096, 3072, 1, False, True), (4096, 768, 1001, 1, False, False)]


@pytest.mark.parametrize("M,K,N,nb,single,pair", PRODUCTS)
def test_products_from_kept_tiles(pkg, gpu, M, K, N, nb, single, pair):
    import torch
    say(f"products from kept tiles M={M} K={K} N={N} batch={nb}")
    L, d = pkg.lib(), pkg.desc
    g = rng("kept", M, K, N, nb)
    raw = [q8_dev((0.05 * g.standard_normal((M, K))).astype(np.float32))[0] for _ in range(2)]
    pool = torch.stack(raw).contiguous()
    wd, wd2 = pkg.desc_q8(pool[0], K), pkg.desc_q8(pool[1], K)
    x, res = dev(g.standard_normal((nb, N, K)).astype(np.float32)), dev(g.standard_normal((nb, N, M)).astype(np.float32))
    v = (lambda t: t.unsqueeze(1)) if nb > 1 else (lambda t: t[0])
    calls = [lambda o: L.vx_mul_mat(wd, d(v(x)), d(v(o)), pkg.ACT_FLOAT, None),
             lambda o: L.vx_mul_mat_scale_add(wd, d(v(x)), d(v(res)), d(v(o)), 0.7, pkg.ACT_FLOAT, None)]
    if L.vx_supports_mul_mat_swiglu_tiled(wd, wd2, d(v(x)), d(v(res)), pkg.ACT_FLOAT):
        calls.append(lambda o: L.vx_mul_mat_swiglu(wd, wd2, d(v(x)), d(v(o)), pkg.ACT_FLOAT, None))
    assert len(calls) == 3 or not pair

    def run(call):
        out = torch.full((nb, N, M), 7.0, dtype=torch.float32, device="cuda")
        ok(pkg, call(out), "product")
        torch.cuda.synchronize()
        return out

    want = [run(c) for c in calls]
    pkg.check(L.vx_weights_pin(pool.data_ptr(), pool.numel()), "pin")
    try:
        base = held = kept_bytes(L)[1:]
        for turn in range(2):   # the copies are made, then used again
            for c, w, copies in zip(calls, want, (single, single, single + pair)):
                assert same_bits(w, run(c)), turn
                before, held = held, kept_bytes(L)[1:]
                if turn == 0:
                    assert held[0] == base[0] + copies
                    assert held == before or held[1] - before[1] >= 2 * M * K * (held[0] - base[0])    # (f16 values; the pair's are two matrices')
                else:
                    assert held == before
    finally:
        L.vx_weights_unpin(pool.data_ptr())
    assert kept_bytes(L)[1:] == base


# tokens, rows behind the down projection; copies: the pair's, and down's where that runs on gd_kernel as well, from the tiles that the pair left
MLPS = [(768, 1024, 1), (1000, 1024, 1), (1024, 1024, 1), (2048, 1024, 1), (3072, 1024, 1), (1801, 2048, 2), (1856, 2040, 2)]


@pytest.mark.parametrize("T,M,copies", MLPS)
def test_mlp_from_kept_tiles(pkg, gpu, T, M, copies):
    """The whole MLP: the pair leaves its result as the down projection's tiles."""
    import torch
    say(f"MLP from kept tiles T={T} rows={M}")
    L, d = pkg.lib(), pkg.desc
    K, F = 1024, 4096
    g = rng("kept-mlp", T, M)
    mk = lambda m, k: q8_dev((0.05 * g.standard_normal((m, k))).astype(np.float32))[0]
    pair, down = torch.stack([mk(F, K), mk(F, K)]).contiguous(), mk(M, F)
    wg, wu, wd = pkg.desc_q8(pair[0], K), pkg.desc_q8(pair[1], K), pkg.desc_q8(down, F)
    x, nw = dev((2 * g.standard_normal((T, K))).astype(np.float32)), dev((1 + 0.1 * g.standard_normal(K)).astype(np.float32))
    res = dev(g.standard_normal((T, M)).astype(np.float32))

    def mlp():
        out = torch.full((T, M), float("nan"), dtype=torch.float32, device="cuda")
        ok(pkg, L.vx_mlp_tiled(d(x), d(nw), 1e-5, wg, wu, wd, d(res), 0.3, d(out), pkg.ACT_FLOAT, None), "mlp_tiled")
        torch.cuda.synchronize()
        return out

    want = mlp()
    base = kept_bytes(L)[1]
    for t in (pair, down):
        pkg.check(L.vx_weights_pin(t.data_ptr(), t.numel()), "pin")
    try:
        for turn in range(2):
            assert same_bits(want, mlp()) and kept_bytes(L)[1] == base + copies, turn
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


def test_dropping_one_of_several_copies_waits_for_its_readers(pkg, gpu):
    """As dropping an allocation of its own does: the caller may write to or free the weights next."""
    import torch
    say("kept tiles: a copy dropped with kernels in flight, its neighbour staying")
    L, d = pkg.lib(), pkg.desc
    M, K, N = 4096, 1024, 2048
    g = rng("kept-drop")
    pool = torch.stack([q8_dev((0.05 * g.standard_normal((M, K))).astype(np.float32))[0] for _ in range(2)]).contiguous()
    x = dev(g.standard_normal((N, K)).astype(np.float32))
    outs = torch.empty((2, N, M), dtype=torch.float32, device="cuda")
    side, done = torch.cuda.Stream(), torch.cuda.Event()

    def product(w):
        pkg.check(L.vx_mul_mat(pkg.desc_q8(pool[w], K), d(x), d(outs[w]), pkg.ACT_FLOAT, side.cuda_stream), "mul_mat")

    copies = kept_bytes(L)[1]
    pkg.check(L.vx_weights_pin(pool.data_ptr(), pool.numel()), "pin")
    try:
        product(0)
        product(1)
        torch.cuda.synchronize()
        assert kept_bytes(L)[1] == copies + 2
        for _ in range(400):   # some 13 ms of kernels
            product(0)
        done.record(side)
        pkg.check(L.vx_weights_changed(pool[0].data_ptr(), pool[0].numel()), "changed")
        assert done.query() and kept_bytes(L)[1] == copies + 1
    finally:
        L.vx_weights_unpin(pool.data_ptr())
