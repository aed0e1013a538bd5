// gm_tiles.hpp -- which tile of gm_kernel (or gd_kernel's) a product of gemm_mid.hip runs on, and which XCD takes which of its tiles.
// Free of HIP calls, so that the rules can be asked on a host without a device.
#pragma once

#include <cstdint>

enum { VX_GM_Q8 = 0, VX_GM_F16 = 1 };
enum { GM_PLAIN = 0, GM_SWIGLU = 1, GM_SEGS = 2 };

constexpr int GM_KG = 4; // waves of a row group, over the k blocks: the streaming kernel's four waves

// gm_kernel's tile: row tiles of 16 a wave, token tiles of 16, row groups, 128-k chunks a stage, stages
template <int WT, int MT, int NT, int RW, int CH, int S>
struct gm_shape {
    static constexpr int NC = GM_KG * RW, NWAVES = NC + 2;    // compute waves; one wave brings the weights, one the activations
    static constexpr int ROWS = 16 * MT * RW, TOKS = 16 * NT;
    static constexpr int PIECES = WT == VX_GM_Q8 ? (CH == 1 ? 9 : 17) : 16 * CH; // 16-byte pieces of a row per stage
    static constexpr int PITCH = PIECES * 16;
    static constexpr int WINST = (ROWS * PIECES + 63) / 64, XINST = 4 * CH * NT;
    static constexpr int WBYTES = WINST * 1024, XBYTES = XINST * 1024, STAGE = WBYTES + XBYTES;
    static constexpr int STEPS = 4 * CH / GM_KG;              // k blocks of a stage per compute wave
    static constexpr int NP = NT < 4 ? NT : 4;                // token tiles per pass of the final sum
    static constexpr int RED = GM_KG * RW * MT * NP * 1024;
    static constexpr int LDS = S * STAGE > RED ? S * STAGE : RED;
};

// ---- tile choice -----------------------------------------------------------------------------------------------------
// (row tiles per wave, token tiles, row groups, 128-k chunks a stage; stages with Q8_0 and with F16 weights, 0: not built; what a
// work-group costs beside the other tiles': microseconds per 128 of K and fixed)
//   Stages.  Three, or more where that gains within one round of work-groups; measured as kernels of 256 and 512 work-groups (K 1024 /
// 4352) and as whole products (1024 x 4096), microseconds with three and with these:
//   * 16 x 16, five: two share a unit's LDS with either type; 256: Q8_0 K 4352 7.4 / 7.1, F16 7.4 / 6.7; 45 tokens: 9.4 / 9.3, F16 9.3 / 8.8;
//   * 32 x 32, four: alone on a unit; 256: Q8_0 5.6 / 5.8 and 11.7 / 10.4, F16 5.1 / 5.0 and 12.8 / 12.5; 203 tokens: 13.9 / 13.5, F16 13.1 / 12.7.
//     F16 does not share with three either.  Q8_0 does: a tile of its own (8) for more work-groups than units, 512: 7.3 / 10.5, pairs of 5504 rows
//     by 24 tokens 10.2 / 10.8;
//   * 32 x 64, five: alone on a unit; 256: Q8_0 6.4 / 6.6 and 14.2 / 12.8, F16 6.2 / 5.9 and 16.2 / 15.1; 337 tokens: 17.4 / 17.5, F16 17.6 / 16.5; a
//     prompt of 45 tokens, whose gate/up pair is one round of it, 974 / 963.  With three two share a unit (512: 8.8 / 11.7), but from there on
//     the larger tiles are the faster.
//   Costs.  Those of the tiles up to 64 x 128 come from kernels with Q8_0 weights and three stages, without what every tile pays alike; 96
// and 112 tokens lie on the line between 64 and 128.  They only serve to compare: over 994 products, pairs and q/k/v groups of 17 to 3072 tokens,
// both types, the tile chosen takes 0.5 % longer than the fastest one on average, more than 3 % in 66 of them, at most 14 (520 rows x 416 tokens of
// K 2304); no other pair of values for 96 or 112 tokens does better by more than 0.03 %.
#define GM_TILES(X) \
    X(0, 1, 1, 1, 2, 5, 5, 0.127f, 0.95f) \
    X(1, 1, 2, 1, 2, 3, 3, 0.135f, 1.10f) \
    X(2, 2, 2, 1, 2, 4, 4, 0.190f, 1.40f) \
    X(3, 2, 4, 1, 1, 5, 5, 0.276f, 1.30f) \
    X(4, 2, 4, 2, 1, 3, 3, 0.355f, 2.15f) \
    X(5, 2, 8, 2, 1, 3, 3, 0.505f, 2.85f) \
    X(6, 2, 6, 2, 1, 3, 3, 0.430f, 2.50f) \
    X(7, 2, 7, 2, 1, 3, 3, 0.468f, 2.68f) \
    X(8, 2, 2, 1, 2, 3, 0, 0.190f, 1.40f)
constexpr int GM_N_TILES = 9;
// lone: a compute unit's LDS holds one work-group (F16 rows are twice the bytes: more of the tiles)
struct gm_tile { int rows, toks, mt; float per_step, fixed; bool lone[2], built[2]; };
constexpr gm_tile gm_tiles[GM_N_TILES] = {
#define X(I, MT, NT, RW, CH, SQ, SF, A_, B_)                                                          \
    { 16 * MT * RW, 16 * NT, MT, A_, B_, { 2 * gm_shape<VX_GM_Q8, MT, NT, RW, CH, SQ>::LDS > 160 * 1024, \
                                           2 * gm_shape<VX_GM_F16, MT, NT, RW, CH, SF>::LDS > 160 * 1024 }, { SQ > 0, SF > 0 } },
    GM_TILES(X)
#undef X
};
static_assert(!gm_tiles[0].lone[VX_GM_Q8] && !gm_tiles[0].lone[VX_GM_F16] && !gm_tiles[1].lone[VX_GM_Q8] && !gm_tiles[1].lone[VX_GM_F16] &&
              !gm_tiles[8].lone[VX_GM_Q8], "two of these share a compute unit: more stages would end that");

// gd_kernel's tile, and the work-groups that share a compute unit
constexpr int GD_CT = 4, GD_ROWS = 256, GD_TOKS = 16 * GD_CT, GD_PER_CU = 2;

struct gm_product { int wtype, epi, nmat; int64_t M[3], K, N, nbatch; }; // (a pair: M[0] rows of each matrix)

// Which tiles an XCD takes: 1, 2, 4 or all 8 of them (2^xr) share out the gx row tiles, the rest the gy token tiles -- nx by ny tiles an
// XCD and batch entry.  What the eight L2s bring in is every weight once per group of token tiles and every activation once per group of
// row tiles: the fewest bytes of those divisions that leave the fullest XCD (32 compute units, per_cu work-groups each at a time) the
// fewest rounds.
struct gm_share { int xr; int64_t nx, ny, rounds, tiles; }; // tiles: of the whole product
static inline gm_share gm_share_out(int64_t gx, int64_t gy, int64_t nbatch, double wbytes, double xbytes, int per_cu) {
    gm_share s = { 0, 0, 0, 0, gx * gy * nbatch };
    double least = 0.0;
    for (int r = 3; r >= 0; --r) {
        const int64_t nx = (gx + (1 << r) - 1) >> r, ny = (gy + (8 >> r) - 1) / (8 >> r), rounds = (nx * ny * nbatch + 32 * per_cu - 1) / (32 * per_cu);
        const double bytes = wbytes * (8 >> r) + xbytes * (1 << r);
        if (s.nx && (rounds > s.rounds || (rounds == s.rounds && bytes >= least))) continue;
        s = { r, nx, ny, rounds, s.tiles };
        least = bytes;
    }
    return s;
}

static inline gm_share gm_tile_share(const gm_product & p, int tile) {
    const gm_tile & g = gm_tiles[tile];
    int64_t gx = 0;
    if (p.epi == GM_SWIGLU) gx = (2 * p.M[0] + g.rows - 1) / g.rows;
    else for (int i = 0; i < p.nmat; ++i) gx += (p.M[i] + g.rows - 1) / g.rows;
    return gm_share_out(gx, (p.N + g.toks - 1) / g.toks, p.nbatch, (double) gx * g.rows * (double) (p.K / 32) * (p.wtype == VX_GM_Q8 ? 34 : 64), (double) p.N * p.K * 2, 1);
}

// The tile whose work-groups finish first by the costs.  One that has a compute unit to itself: on the XCD that has most of them.  (Counted
// over the chip, 238 work-groups of 520 rows x 448 tokens of K 2304 seemed one round of 256; at least 34 are an XCD's, which has 32 compute
// units: 16.0 us where another tile takes 12.7.)  Where two share one, an XCD's last few join others and cost far less than a round: over the chip.
static inline int gm_tile_choice(const gm_product & p, gm_share & share) {
    int best = -1;
    float best_us = 0.0f;
    for (int t = 0; t < GM_N_TILES; ++t) {
        const gm_tile & g = gm_tiles[t];
        if (!g.built[p.wtype] || (p.epi != GM_PLAIN && g.mt % 2)) continue;
        const gm_share s = gm_tile_share(p, t);
        const float steps = g.per_step * (float) (p.K / 128), one = g.fixed + steps, rounds = (float) (g.lone[p.wtype] ? s.rounds : (s.tiles + 255) / 256);
        // (work-groups that share a compute unit share its vector units: the fixed part of one hides behind the other's products)
        const float us = g.lone[p.wtype] ? rounds * one : one + (rounds - 1.0f) * (steps + 0.3f * g.fixed);
        if (best < 0 || us < best_us) { best = t; best_us = us; share = s; }
    }
    return best;
}

// Single products and pairs that gd_kernel takes where the weights' tiles are kept: from the number of its 256 x 64 tiles on at which it
// beats gm_kernel.  gm_kernel / here, microseconds, activation pass included, by the tokens (tiles):
//   * K 1024, single: 4096 rows 512 (128) 15.1 / 19.8, 768 (192) 21.4 / 21.6, 1024 (256) 24.4 / 24.0, 1088 (272) 30.1 / 27.9, 2048 (512) 45.9 / 33.6; 6144
//     rows 512 (192) 21.9 / 22.1, 640 (240) 24.8 / 23.5; 2048 rows 1536 (192) 22.4 / 21.9;
//   * K 1024, a pair with its down projection behind it: 4096 rows 256 (128) 27.9 / 31.9, 300 (160) 37.0 / 35.4, 512 (256) 41.7 / 36.7, 576 (288) 50.6 /
//     47.7, 1024 (512) 66.4 / 54.6, 1280 (640) 83.2 / 69.8, 3072 (1536) 179 / 133;
//   * a long K, on which few work-groups take longer: K 4096, 1024 rows 3072 (192) 61.4 / 65.5, 1536 rows 2240 (210) 60.4 / 62.3, 2304 (216) 64.9 / 62.8,
//     2048 rows 1664 (208) 59.9 / 58.7, 2048 (256) 66.4 / 63.0, 4096 rows 2048 (512) 119 / 100; K 16384, 2048 rows 1792 (224) 206 / 225, 1856 (232) 225 / 226;
//   * and just over a work-group for each of an XCD's compute units there: K 4096, 1536 rows 2688 (252, no XCD fewer than 33) 70.7 / 81.2, 2048 rows
//     2304 (288, 36) 80.4 / 80.5, 2432 (304, 38) 87.3 / 81.4.
static inline bool gd_takes(const gm_product & p) {
    if (p.wtype != VX_GM_Q8 || p.epi == GM_SEGS || p.K % 512) return false; // (a group's k blocks in whole fours)
    const bool pair = p.epi == GM_SWIGLU;
    const int64_t MV = pair ? 2 * p.M[0] : p.M[0], gx = (MV + GD_ROWS - 1) / GD_ROWS, gy = (p.N + GD_TOKS - 1) / GD_TOKS, tiles = gx * gy * p.nbatch;
    if ((pair && p.M[0] % 32) || (MV + 15) / 16 * (p.K / 32) >= (1 << 22)) return false;
    if (p.K <= 1024) return tiles >= (pair ? 160 : 192);
    if (tiles < (p.K > 8192 ? 232 : 216)) return false;
    int64_t fullest = INT64_MAX; // XCD's work-groups, of the most even division
    for (int r = 0; r < 4; ++r) {
        const int64_t n = ((gx + (1 << r) - 1) >> r) * ((gy + (8 >> r) - 1) / (8 >> r)) * p.nbatch;
        fullest = n < fullest ? n : fullest;
    }
    return fullest <= 32 || fullest > 36;
}
