// gemm_mid.hpp -- the product kernel for some tens to a few thousand tokens (gemm_mid.hip), as mul_mat.hip calls it.
#pragma once
#include "vx_common.hpp"
#include "gm_tiles.hpp"
#include "rope_common.hpp"

struct vx_gm_mat {        // one weight matrix of a launch and where its product goes
    const char * w;
    char *       dst;
    int          M, wg0;  // rows; first row tile of the grid (filled in by the launcher)
    uint64_t     nb01;    // weight row stride
    uint64_t     nb1, nb2, nb3; // dst strides of token, ne2, ne3
    int          rope;    // rotate (d, d + 32) of every head of 64 rows before storing
};

struct vx_gm_call {
    int           wtype;          // VX_GM_*
    int           nmat;           // 1 .. 3 matrices over the same activations
    vx_gm_mat     mat[3];
    const char *  w2;             // second matrix of a gate/up pair (mat[0]'s shape and stride): dst = silu(W x) * (W2 x)
    int64_t       K, N;
    int           ne12, ne13;     // batch of the activations; the weights are the same for every entry
    // activations: F32 (x, strides), normalised on the way when norm_w is set, or the f16 tiles a kernel in front left (tile_in)
    const char *  x;
    uint64_t      nb11, nb12, nb13;
    const float * norm_w;
    float         norm_eps;
    const double * add_totals;    // a cache write's wave totals, whose ordering scalar is added to every activation (no norm), or null
    float         add_scale, add_bias;
    const void *  tile_in;
    int           tile_tt;        // 16-token tiles per k block of tile_in / tile_out
    void *        tile_out;       // gate/up pair: results as the next product's f16 activation tiles instead of dst
    const char *  res;            // residual update dst = res + res_scale * (W x), or null
    uint64_t      rnb1, rnb2, rnb3;
    float         res_scale;
    // rotation (mat[i].rope): positions of rope_T tokens per sequence, flattened sequences taken modulo
    const int32_t * pos; const float * ff;
    rope_params   rp;
    int           rope_T;
    size_t        ws_offset;      // bytes at the start of the stream's workspace that the caller keeps
};

// Whether this kernel serves a product of M rows, K columns and N * nbatch tokens.  The rows of one matrix decide, for a gate/up pair
// as for gate or up alone, and a group of several matrices needs the answer for each: a product and every group it is part of
// are formed by the same kernel, in the same order of every sum.
bool vx_gm_shape(int wtype, int64_t K, int64_t N, int64_t nbatch, int64_t M);
bool vx_gm_on(int64_t N); // and whether the environment leaves it in place
static inline bool vx_gm_region(int wtype, int64_t K, int64_t N, int64_t nbatch, int64_t M) { return vx_gm_shape(wtype, K, N, nbatch, M) && vx_gm_on(N); }
// region, and operands on the boundaries its loads need (dst only needs 4-byte aligned values)
bool vx_gm_takes(const vx_gm_call & c);
// Weights as mul_mat.hip's weight pass lays them out for the pre-tiled kernel (f16 integers in operand tiles, the block scales apart;
// a pair's 16-row tiles alternate), kept for pinned weights: false where there is no such copy to be had.
bool vx_qt_kept_tiles(const char * w, const char * w2, int64_t K, int64_t M, uint64_t nb01, hipStream_t st, const void ** tiles, const float ** scales);
size_t vx_gm_tile_bytes(int64_t K, int64_t N, int64_t nbatch); // f16 activation tiles of a product
vx_status vx_gm_run(const vx_gm_call & c, hipStream_t st);
