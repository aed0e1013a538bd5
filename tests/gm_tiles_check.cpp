// Host-only access to the tile rules of the mid-size products (voxcpm.cpp_amd/csrc/gm_tiles.hpp) for tests/test_cpu_gemm_tiles.py.
#include "../voxcpm.cpp_amd/csrc/gm_tiles.hpp"

extern "C" {
// out: tile, rows, tokens, lone, xr, nx, ny, rounds of the fullest XCD
void gm_choice(int wtype, int epi, const int64_t * m, int nmat, int64_t k, int64_t n, int64_t nbatch, int64_t * out) {
    gm_product p = { wtype, epi, nmat, {}, k, n, nbatch };
    for (int i = 0; i < nmat; ++i) p.M[i] = m[i];
    gm_share s = {};
    const int t = gm_tile_choice(p, s);
    const int64_t all[8] = { t, gm_tiles[t].rows, gm_tiles[t].toks, gm_tiles[t].lone[wtype], s.xr, s.nx, s.ny, s.rounds };
    for (int i = 0; i < 8; ++i) out[i] = all[i];
}
int gm_kept(int wtype, int epi, int64_t m, int64_t k, int64_t n, int64_t nbatch) { return gd_takes({ wtype, epi, 1, { m, 0, 0 }, k, n, nbatch }); }
}
