"""CPU: the tile rules of the mid-size products (csrc/gm_tiles.hpp)."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
Q8, F16 = 0, 1
PLAIN, SWIGLU, SEGS = 0, 1, 2


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("gm_tiles") / "gm_tiles_check.so")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests", "gm_tiles_check.cpp")])
    return C.CDLL(so)


def choice(rules, wtype, epi, rows, K, N, nb=1):
    out = (C.c_int64 * 8)()
    m = (C.c_int64 * len(rows))(*rows)
    rules.gm_choice(wtype, epi, m, len(rows), C.c_int64(K), C.c_int64(N), C.c_int64(nb), out)
    return dict(zip(("tile", "rows", "toks", "lone", "xr", "nx", "ny", "rounds"), out))


SHAPES = [(PLAIN, [m], k) for m, k in ((16, 1024), (128, 1024), (520, 2304), (1000, 4096), (1024, 1024), (1536, 3072), (4096, 1024), (6144, 768))] + \
         [(SWIGLU, [m], 1024) for m in (512, 2816, 4096, 5504)] + [(SEGS, [1024, 128, 128], 1024), (SEGS, [2048, 512, 512], 1024)]


@pytest.mark.parametrize("wtype", [Q8, F16])
@pytest.mark.parametrize("epi,rows,K", SHAPES)
def test_work_groups_cover_every_tile_once_and_rounds_are_an_xcds(rules, wtype, epi, rows, K):
    """gm_kernel's mapping of work-groups to tiles, written out: every tile once, and no XCD with more rounds than the choice counted."""
    for N in (17, 45, 100, 203, 337, 416, 448, 777, 1152, 3072):
        for nb in (1, 3):
            c = choice(rules, wtype, epi, rows, K, N, nb)
            mul = 2 if epi == SWIGLU else 1
            gx, gy = sum(-(-mul * m // c["rows"]) for m in rows), -(-N // c["toks"])
            seen, load = set(), [0] * 8
            for y in range(c["ny"]):
                for x in range(8 * c["nx"]):
                    xcd = x & 7
                    tx, ty = ((x >> 3) << c["xr"]) + (xcd & ((1 << c["xr"]) - 1)), (y << (3 - c["xr"])) + (xcd >> c["xr"])
                    load[xcd] += 1
                    if tx < gx and ty < gy:
                        assert (tx, ty) not in seen
                        seen.add((tx, ty))
            assert len(seen) == gx * gy, (N, c)
            assert -(-max(load) * nb // 32) == c["rounds"], (N, c)


@pytest.mark.parametrize("wtype", [Q8, F16])
@pytest.mark.parametrize("M,K,N", [(520, 2304, 416), (520, 2304, 448), (520, 2304, 480), (520, 2304, 850), (520, 2304, 950)])
def test_an_odd_number_of_row_tiles_does_not_take_a_second_round(rules, wtype, M, K, N):
    """Just under 256 work-groups of a tile that has a compute unit to itself, of which an XCD's share is more than its 32 units."""
    c = choice(rules, wtype, PLAIN, [M], K, N)
    assert c["rounds"] == 1 or not c["lone"], c


@pytest.mark.parametrize("epi,rows,K,N", [(SWIGLU, [5504], 1024, 24), (SWIGLU, [5504], 1024, 32), (PLAIN, [3072], 768, 160)])
def test_small_tiles_share_a_compute_unit(rules, epi, rows, K, N):
    """Q8_0, a little more than a work-group for each compute unit: the 32 x 32 tiles that run there leave room for a second one."""
    c = choice(rules, Q8, epi, rows, K, N)
    assert c["rows"] == c["toks"] == 32 and not c["lone"], c


@pytest.mark.parametrize("epi,M,K,N,nb,kept", [
    (PLAIN, 4096, 1024, 700, 1, 0), (PLAIN, 4096, 1024, 768, 1, 1), (PLAIN, 4096, 768, 1000, 1, 0), (SWIGLU, 4096, 1024, 256, 1, 0), (SWIGLU, 4096, 1024, 257, 1, 1),
    (SWIGLU, 2800, 1024, 3000, 1, 0), (SWIGLU, 2784, 1024, 3000, 1, 1), (PLAIN, 1024, 4096, 3072, 1, 0), (PLAIN, 2048, 4096, 1536, 1, 0), (SWIGLU, 1024, 4096, 1400, 1, 0),
    (PLAIN, 2048, 4096, 1856, 1, 1), (PLAIN, 1536, 4096, 2560, 1, 1), (PLAIN, 1536, 4096, 2688, 1, 0), (PLAIN, 2048, 4096, 2304, 1, 0), (PLAIN, 2048, 4096, 2432, 1, 1),
    (PLAIN, 2048, 16384, 1792, 1, 0), (PLAIN, 2048, 16384, 1856, 1, 1), (SWIGLU, 2048, 2560, 400, 3, 1), (SWIGLU, 768, 3072, 896, 3, 0)])
def test_products_from_kept_tiles(rules, epi, M, K, N, nb, kept):
    """Where gd_kernel was measured to be the faster kernel it is taken, elsewhere not."""
    assert rules.gm_kept(Q8, epi, C.c_int64(M), C.c_int64(K), C.c_int64(N), C.c_int64(nb)) == kept


def test_the_gpu_cases_run_on_the_tiles_they_name(rules):
    """tests/test_gpu_gemm_tiles.py: 96 and 112 tokens in every form, the 32 x 32 tile that shares a compute unit."""
    import test_gpu_gemm_tiles as cases
    types = {"q8": Q8, "f16": F16}

    def tile(wtype, epi, rows, K, N):
        c = choice(rules, wtype, epi, rows, K, N)
        return c["rows"], c["toks"], bool(c["lone"])

    for wtype in (Q8, F16):
        at = {(m, k, n): tile(wtype, PLAIN, [m], k, n) for m, k, n in cases.PRODUCTS}
        assert [at[c][1] for c in cases.PRODUCTS[:6]] == [96, 96, 96, 112, 112, 112]
        if wtype == Q8:
            assert [at[c] for c in cases.PRODUCTS[6:8]] == [(32, 32, False)] * 2
        assert {at[c][1] for c in cases.PRODUCTS[8:10]} == {64}
    pairs = [tile(types[w], SWIGLU, [m], 1024, n) for m, n, w in cases.PAIRS]
    assert [t[1] for t in pairs] == [96, 96, 112, 112, 112, 112, 32, 32] and not pairs[6][2] and not pairs[7][2]
    assert [tile(types[w], SEGS, [1024, 128, 128], 1024, t * b)[1] for t, b, w in cases.GROUPS] == [96, 96, 112, 112]


def test_the_gpu_cases_of_kept_tiles_run_on_gd_kernel(rules):
    """tests/test_gpu_gemm_kept.py says which of its products and pairs do."""
    import test_gpu_gemm_kept as cases
    kept = lambda *a: bool(rules.gm_kept(Q8, a[0], *(C.c_int64(v) for v in a[1:])))
    for M, K, N, nb, single, pair in cases.PRODUCTS:
        assert (kept(PLAIN, M, K, N, nb), kept(SWIGLU, M, K, N, nb)) == (single, pair), (M, K, N, nb)
    for T, M, copies in cases.MLPS:
        assert kept(SWIGLU, 4096, 1024, T, 1) + kept(PLAIN, M, 4096, T, 1) == copies, (T, M)
    assert any(copies == 2 for _, _, copies in cases.MLPS)
    assert any(pair and 2 * M % 256 for M, _, _, _, _, pair in cases.PRODUCTS) and any(single and M % 256 for M, _, _, _, single, _ in cases.PRODUCTS)
