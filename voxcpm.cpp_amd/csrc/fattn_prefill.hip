// fattn_prefill.hip -- GGML_OP_FLASH_ATTN_EXT for many query rows (prefill) on gfx950: a
// tiled flash-attention kernel on f16 MFMA with K/V tiles staged in LDS and the online
// softmax in fp32.
//
// A work-group (4 waves) owns 256 (or 128) *columns* of one (batch, KV head): RB = 256 / gqa
// consecutive query rows times the gqa query heads that share the KV head, so one K/V tile
// in LDS serves all of them (the GQA reuse).  Keys are walked in tiles of 64.
//
// The mask is data, not a flag: a small pre-pass classifies every (row block, key tile) of it
// as all -inf (tile skipped: the causal upper triangle costs nothing), all zero (no mask
// arithmetic) or mixed (mask values are applied element-wise), so the result equals
// ggml-cpu's for any mask while a causal mask gets causal cost.
//
// Roofline: MFMA-bound in principle (4 * D flops per score); at D = 64 the exp, the rounding
// and the row sums of a score (VALU) need about as many issue cycles as its share of the
// matrix instructions, so the two pipes have to run side by side to come near the peak.
#include "kvs_common.hpp"
#include "vx_common.hpp"

#include <algorithm>
#include <cmath>

namespace {

constexpr int PF_WAVES = 4;
constexpr int PF_COLS  = 256; // columns per work-group
constexpr int PF_KT    = 64;  // keys per tile
constexpr int PF_MAX_TILES = 1024;
constexpr int PF_BIT_ROWS = 32; // rows whose visibility bits of a tile fit the block's LDS: blocks of more rows (few heads to a KV head) take the mask's values
constexpr int PF_PART = 256; // compute units: work-groups that stay where two teams walk a row block each
constexpr int PF_TOTALS = VX_KVS_V_AT;       // block totals of one sum of a cache write, at most
constexpr int PF_TOTALS_INLINE = 64; // up to here a wave of every attention work-group adds them (two sequences of 512 tokens: 32 a side; beside
                                     // the tile list that takes less than the 4.5 us of a launch for one number), beyond pf_scalar_kernel does

struct pf_args {
    const char * q; const char * k; const char * v; const char * vl; const char * mask;
    const float * sinks;
    const float * add1; // optional scalar added to every output element (a fused GGML_OP_ADD1)
    _Float16 * tile_out; // optional: the result as f16 activation tiles of the product that follows, instead of dst
    uint32_t tile_tt, tile_bs, tile_ts;
    float * dst;
    const uint8_t * flags; // [nem3][nem2][n_rb][n_tiles]: 0 skip, 1 no mask, 2 apply mask values, 3 apply visibility bits
    const uint8_t * bits;  // [nem3][nem2][n_q][n_tiles] 8 bytes each: one bit per key of the tile (flag 3)
    uint64_t nbq1, nbq2, nbq3, nbk1, nbk2, nbk3, nbv1, nbv2, nbv3, nbm1, nbm2, nbm3;
    int n_q, n_kv, Hq, Hkv, gqa, ne3, rk3, nem2, nem3;
    int RB, n_rb, n_tiles, n_groups, xcd_map;
    int gqa_sh; // gqa divides 128: a power of two, gqa == 1 << gqa_sh
    float scale2, max_bias, m0, m1; // scale2 = scale * log2(e)
    uint32_t n_head_log2;
    int kv_f32;
    const double * totals; // instead of add1 the block totals of a cache write's two sums (n_tk of k at 0, n_tv of v at PF_TOTALS), which give that scalar
    int n_tk, n_tv;
    float sync_scale, sync_bias;
};

// What the launch in front of the attention kernel prepares, each by work-groups of its own: the cache write of the same
// attention block (n_store work-groups), the mask's tile flags (n_mask), the f16 images of F32 K / V (the rest).
struct pf_mask_args {
    const char * mask;
    uint64_t nbm1, nbm2, nbm3;
    int nem2, n_q, n_kv, RB, n_rb, n_tiles, vec_ok, n_units;
    uint8_t * flags; uint8_t * bits;
};
struct pf_prep_args {
    kvs_side ks, vs;
    double * totals;
    int store_large, n_tk, n_store; // the SUMs' form (below); work-groups (large) or totals of the k side; work-groups of both
    pf_mask_args m;
    int n_mask, n_kv;
    const char * k; const char * v;
    uint64_t nbk1, nbk2, nbk3, nbv1, nbv2, nbv3;
    int Hkv, key_blocks;
    _Float16 * k16; _Float16 * vhi; _Float16 * vlo;
};

// classifies mask tiles: one wave per (key tile, row block, mask batch).  A lane reads 8 keys
// (16 bytes) of a row, so the wave covers 8 rows of the 64-key tile per step.  Flags: 0 no key of the tile is visible to
// any row of the block; 1 every entry is zero; 2 some entry is a finite non-zero value; 3 zeros and -inf only.  For the
// last kind the rows' visibility is also left as one bit per key (bits[mask batch][row][tile], keys past n_kv cleared),
// so that the attention kernel applies such a tile -- a causal mask's diagonal -- from 8 bytes per row.
__device__ __forceinline__ void pf_mask_unit(const pf_mask_args & a, int tile, int rb, int mb, int lane) {
    const char * mp = a.mask + (uint64_t) (mb % a.nem2) * a.nbm2 + (uint64_t) (mb / a.nem2) * a.nbm3;
    const int r0 = rb * a.RB, r1 = min(a.n_q, (rb + 1) * a.RB);
    bool any_visible = false, any_nonzero = false, any_hidden = false;
    if (a.vec_ok && (tile + 1) * PF_KT <= a.n_kv) {
        const int sub = lane >> 3, part = lane & 7; // row within the step, 8-key group
        for (int r = r0 + sub; r < r1; r += 8) {
            const int4_t v = *(const int4_t *) (mp + (uint64_t) r * a.nbm1 + ((uint64_t) tile * PF_KT + part * 8) * 2);
            uint32_t byte = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t w = (uint32_t) v[i];
                const bool v0 = (w & 0xFFFFu) != 0xFC00u, v1 = (w >> 16) != 0xFC00u;
                byte |= (v0 ? 1u : 0u) << (2 * i) | (v1 ? 1u : 0u) << (2 * i + 1);
                any_nonzero |= (v0 && (w & 0x7FFFu) != 0) || (v1 && (w & 0x7FFF0000u) != 0);
            }
            any_visible |= byte != 0;
            any_hidden  |= byte != 0xFFu;
            a.bits[(((uint64_t) mb * a.n_q + r) * a.n_tiles + tile) * 8 + part] = (uint8_t) byte;
        }
    } else {
        const int key = tile * PF_KT + lane;
        for (int r = r0; r < r1; ++r) {
            bool vis = false;
            if (key < a.n_kv) {
                const uint16_t h = ((const uint16_t *) (mp + (uint64_t) r * a.nbm1))[key];
                vis = h != 0xFC00u;
                any_nonzero |= vis && (h & 0x7FFFu) != 0;
            }
            any_visible |= vis;
            any_hidden  |= !vis;
            const uint64_t row_bits = __builtin_amdgcn_ballot_w64(vis);
            if (lane == 0) *(uint64_t *) (a.bits + (((uint64_t) mb * a.n_q + r) * a.n_tiles + tile) * 8) = row_bits;
        }
    }
    const bool vis = __builtin_amdgcn_ballot_w64(any_visible) != 0;
    const bool nz  = __builtin_amdgcn_ballot_w64(any_nonzero) != 0;
    const bool hid = __builtin_amdgcn_ballot_w64(any_hidden) != 0;
    if (lane == 0) a.flags[((uint64_t) mb * a.n_rb + rb) * a.n_tiles + tile] = !vis ? 0 : (nz ? 2 : (hid ? 3 : 1));
}

// ---- the tiled kernel ---------------------------------------------------------------------------------------------
// A work-group (4 waves) owns 128 * NCB columns of one (batch, KV head); a wave owns NCB blocks of 32 columns and walks
// 64-key tiles as two blocks of 32 keys with v_mfma_f32_32x32x16_f16:
//     S^T = K Q^T     A = 32 keys x 16 d from LDS (one 16-byte read), B = Q^T resident in registers, C = -reference, so the
//                     matrix core hands back score - reference and the common path is exp2, convert, nothing else
//     O^T += V^T P^T  A = 32 d x 16 keys, read from the row-major V tile with the transposing LDS read
//                     (ds_read_b64_tr_b16: a lane of a 16-lane group receives one d of four consecutive keys), B = P^T
//                     straight from the S^T accumulator registers: lane-half h of the S^T result holds keys 4h .. 4h+3 of
//                     every group of 8, which is the order the V^T reads are issued in
// K and V tiles never pass through registers: every wave copies its share of a tile into LDS with direct loads
// (global_load_lds_dwordx4, 64 lanes x 16 bytes = 8 rows per instruction), four tiles deep (three with a low image of
// V), one barrier per tile.  The 16-byte chunks of a row are stored xor-swizzled (the permutation is applied on the
// global address, the LDS side of a direct load is always lane-linear): K by the row's low three bits, 8-row blocks 128
// bytes apart, so the 32 rows of an A operand fall into different banks; V by twice the row's low two bits, so the
// 4 rows x 32 bytes a 16-lane group transposes do (the bank-conflict counter reads zero).  F32 K/V are converted by a
// pass of their own beforehand (K rounded to f16 as Q is; V as a high and a low f16 image whose products are both
// added, so a value is carried to about 22 bits).
// What bounds the walk is instruction issue, not the matrix core: a SIMD issues from its two waves about three
// quarters of the time, so every instruction that is not an exp2, a convert, a packed add or a matrix instruction
// is kept out of the steady state (no divisions, one LDS wait per step, no wait states behind transcendentals).
constexpr int PF_STAGES_MAX = 4;       // tiles in LDS: being read, landed, and two in flight (one with the low image of V)
constexpr int PF_KBLK    = 1152;            // bytes of an 8-row block of a K tile in LDS (8 x 128 + 128)
constexpr int PF_KSTAGE  = 8 * PF_KBLK;     // a 64-key K tile
constexpr int PF_VSTAGE  = 64 * 128;        // a 64-key V tile, rows back to back
constexpr float PF_SUM_LIMIT = 2048.0f;     // a lane's 16 probabilities of a block may add up to this before the reference moves

typedef __attribute__((address_space(3))) char lds_char;

__device__ __forceinline__ float16_t mfma32(half8_t a, half8_t b, float16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
}

// 16 bytes per lane from global memory (uniform base + per-lane 32-bit offset) straight into LDS: lane l's land at
// lds + 16 l (lds uniform).  M0 carries the LDS address.
__device__ __forceinline__ void pf_dma16(const char * base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory");
}

__device__ __forceinline__ void pf_dma4(const char * base, uint32_t off, uint32_t lds) { // 4 bytes per lane, at lds + 4 l
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory");
}

// Two probabilities to f16, to nearest (v_cvt_pk_f16_f32).  Rounded toward zero, a column's reference key alone would keep its value,
// 1, while all others lose half a unit on average: with two references a column (two teams) that was 0.8 % of the whole error, and to
// nearest the error is 10 % below either.  It costs 0.2 to 0.6 % (causal, toward zero / to nearest: 1 x 1024 20.9 / 21.0 us, 1 x 4096
// 65.1 / 65.5, 16 x 1024 68.5 / 68.9, 16 x 2048 197.0 / 198.2).
__device__ __forceinline__ half2_t pf_cvt2(float a, float b) {
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_convertvector(f2{a, b}, half2_t);
}

__device__ __forceinline__ half8_t pf_tr8(const lds_char * p) {
    typedef short short4_t __attribute__((ext_vector_type(4)));
    typedef short short8_t __attribute__((ext_vector_type(8)));
    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3))) *) p);
    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3))) *) (p + 8 * 128));
    return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// F32 K and V of one (batch entry, KV head) as f16 planes [key][64]: K rounded, V as high and low halves
__device__ __forceinline__ void pf_convert_unit(const pf_prep_args & a, int unit, int g, int b) { // 8 values each
    const int key = unit >> 3, part = unit & 7;
    if (key >= a.n_kv) return;
    const float4_t * kp = (const float4_t *) (a.k + (uint64_t) key * a.nbk1 + (uint64_t) g * a.nbk2 + (uint64_t) b * a.nbk3) + 2 * part;
    const float4_t * vp = (const float4_t *) (a.v + (uint64_t) key * a.nbv1 + (uint64_t) g * a.nbv2 + (uint64_t) b * a.nbv3) + 2 * part;
    const float4_t k0 = kp[0], k1 = kp[1], v0 = vp[0], v1 = vp[1];
    half8_t kh, vh, vl;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        kh[i] = (_Float16) k0[i]; kh[4 + i] = (_Float16) k1[i];
        vh[i] = (_Float16) v0[i]; vh[4 + i] = (_Float16) v1[i];
        vl[i]     = (_Float16) (v0[i] - (float) vh[i]);
        vl[4 + i] = (_Float16) (v1[i] - (float) vh[4 + i]);
    }
    const uint64_t o = (((uint64_t) b * a.Hkv + g) * a.n_kv + key) * 64 + 8 * part;
    *(half8_t *) (a.k16 + o) = kh;
    *(half8_t *) (a.vhi + o) = vh;
    *(half8_t *) (a.vlo + o) = vl;
}

// One cache write and its sum in the order of GGML_OP_SUM's kernels here (glue.hip).  Beyond 16 Ki units that is blocks of
// 1024 threads: block b's thread t walks units 1024 b + t, + 128 * 1024, ..., a wave adds its lanes by butterfly, a block's 16
// wave totals are added in order.  A work-group of 256 threads stands for one such block, each of its waves for four of the
// block's: four units of a thread are requested together.
template <bool VEC>
__device__ __forceinline__ void pf_store_large(const kvs_side & s, uint32_t b, double * total, double * part) {
    const uint32_t n = kvs_units(s, VEC);
    double acc[4] = { 0.0, 0.0, 0.0, 0.0 };
    for (uint32_t base = b * 1024 + threadIdx.x; base < n; base += PF_TOTALS * 1024) {
        float v[4][VEC ? 4 : 1];
#pragma unroll
        for (int p = 0; p < 4; ++p) if (base + 256 * p < n) kvs_fetch<VEC>(s, base + 256 * p, v[p]);
#pragma unroll
        for (int p = 0; p < 4; ++p) if (base + 256 * p < n) kvs_apply<VEC>(s, base + 256 * p, true, v[p], acc[p]);
    }
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        const double t = vx_wave_sum(acc[p]);
        if ((threadIdx.x & 63) == 0) part[4 * p + (threadIdx.x >> 6)] = t;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int w = 0; w < 16; ++w) t += part[w];
        *total = t;
    }
}

// One launch for what three did (the cache write, the mask's flags, the f16 images): each is a trip to memory and its
// latency at a prompt's size.  Two sequences of 512 tokens: 4.8 + 4.1 + 3.9 us as launches of their own, and 4.5 for the
// scalar that the attention now adds up itself; 24 layers 3067 -> 2876 us (16 x 4096 tokens: no difference beyond noise).
// STORE is a parameter of its own because the write's four units in flight cost every wave of the launch 98 registers, half
// the waves a SIMD can hold (F32 keys and values without a write are left for the other instance).
template <bool STORE>
__global__ __launch_bounds__(256) void pf_prep_kernel(const pf_prep_args a) {
    __shared__ double part[16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    int i = blockIdx.x;
    if (STORE && i < a.n_store) {
        if (a.store_large) {
            const bool second = i >= a.n_tk; // (uniform)
            const kvs_side & s = second ? a.vs : a.ks;
            const uint32_t b = (uint32_t) (second ? i - a.n_tk : i);
            double * total = a.totals + (second ? PF_TOTALS : 0) + b;
            if (s.vec) pf_store_large<true>(s, b, total, part);
            else       pf_store_large<false>(s, b, total, part);
        } else { // 16 waves a side
            const bool second = i >= 4;
            const kvs_side & s = second ? a.vs : a.ks;
            const uint32_t w = (uint32_t) (4 * (i & 3) + wave);
            const double t = s.vec ? kvs_mid_wave<true>(s, w, (uint32_t) lane) : kvs_mid_wave<false>(s, w, (uint32_t) lane);
            if (lane == 0) a.totals[(second ? PF_TOTALS : 0) + w] = t;
        }
        return;
    }
    if constexpr (STORE) i -= a.n_store;
    if (i < a.n_mask) {
        const int unit = 4 * i + wave;
        if (unit < a.m.n_units) pf_mask_unit(a.m, unit % a.m.n_tiles, (unit / a.m.n_tiles) % a.m.n_rb, unit / a.m.n_tiles / a.m.n_rb, lane);
        return;
    }
    i -= a.n_mask;
    const int kb = i % a.key_blocks, bg = i / a.key_blocks;
    pf_convert_unit(a, kb * 256 + (int) threadIdx.x, bg % a.Hkv, bg / a.Hkv);
}

// The mask's units alone (f16 keys and values, no cache write): the grid is (W key tiles, row block, mask batch), a wave a tile.
// (Arguments one by one: the first of them come in registers, where a struct's fields are a trip to memory, 0.2 of 3 us.)
template <int W>
__global__ __launch_bounds__(64 * W) void pf_mask_kernel(const char * mask, uint64_t nbm1, uint64_t nbm2, uint64_t nbm3, int nem2, int n_q, int n_kv, int RB,
                                                         int n_rb, int n_tiles, int vec_ok, uint8_t * flags, uint8_t * bits) {
    const pf_mask_args a = { mask, nbm1, nbm2, nbm3, nem2, n_q, n_kv, RB, n_rb, n_tiles, vec_ok, 0, flags, bits };
    const int tile = W * (int) blockIdx.x + __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    if (tile < n_tiles) pf_mask_unit(a, tile, blockIdx.y, blockIdx.z, threadIdx.x & 63);
}

// the ordering scalar of a large write's totals, for every work-group of the attention kernel to read
__global__ __launch_bounds__(128) void pf_scalar_kernel(const double * totals, int n_tk, int n_tv, float scale, float bias, float * out) {
    __shared__ double part[2][PF_TOTALS];
    __shared__ double sum[2];
    const int t = threadIdx.x;
    part[0][t] = t < n_tk ? totals[t] : 0.0;
    part[1][t] = t < n_tv ? totals[PF_TOTALS + t] : 0.0;
    __syncthreads();
    if ((t & 63) == 0) { // a wave a side
        double s = 0.0;
        const int n = t ? n_tv : n_tk;
        for (int i = 0; i < n; ++i) s += part[t >> 6][i];
        sum[t >> 6] = s;
    }
    __syncthreads();
    if (t == 0) *out = kvs_scalar((float) sum[0], (float) sum[1], scale, bias);
}

// VLO: V comes with a low-half image (a.vl).  NCB: 32-column blocks per wave.  SUMS: the addend is the ordering scalar of a.totals
// (an instance of its own: as a test in every instance it cost the calls without a cache write 1 %, 2048 causal tokens 38.7 -> 39.1 us).
// TEAMS: sets of PF_WAVES waves over the same columns, each with every TEAMS-th active tile and stages of its own, their (O, sum,
// reference) joined through LDS at the end -- or, in a grid of more work-groups than compute units whose walks are alike (pf_two_teams),
// over a row block each.  A wave alone on its SIMD leaves half of the issue slots empty (0.92 us a tile; two that
// share the SIMD take 0.62 us each), so a row block walks 64 tiles in about 45 us where one team takes 62; against a cut of the
// key range into work-groups of their own nothing goes through memory and no launch follows.  One sequence of 4096 tokens 72 -> 64 us.
// PART: whether a team may have a row block of its own (an instance of its own: in the others' code the choice cost 0.6 us of a call).
template <bool VLO, int NCB, bool SUMS = false, int TEAMS = 1, bool PART = false>
__global__ __launch_bounds__(64 * PF_WAVES * TEAMS) __attribute__((amdgpu_waves_per_eu(2, 2))) void pf_kernel(const pf_args a) {
    constexpr int D = 64;
    constexpr int PF_STAGES = VLO ? 3 : PF_STAGES_MAX; // (three stages of K, V and V low leave room for two work-groups on a compute unit)
    constexpr int NL = VLO ? 6 : 4; // direct loads per wave and tile (a tile that needs its visibility bits has one more)
    __shared__ __attribute__((aligned(1024))) char k_lds[TEAMS][PF_STAGES][PF_KSTAGE];
    __shared__ __attribute__((aligned(1024))) char v_lds[TEAMS][PF_STAGES][PF_VSTAGE];
    __shared__ __attribute__((aligned(1024))) char vl_lds[VLO ? TEAMS : 1][VLO ? PF_STAGES : 1][VLO ? PF_VSTAGE : 16];
    __shared__ __attribute__((aligned(256))) uint32_t bits_lds[TEAMS][PF_STAGES][2 * PF_BIT_ROWS]; // visibility bits of the block's rows: 8 bytes per row
    __shared__ uint16_t tile_list[PART ? 2 * PF_MAX_TILES : PF_MAX_TILES];
    __shared__ uint8_t  tile_flag[PART ? 2 * PF_MAX_TILES : PF_MAX_TILES];
    __shared__ int      n_active_s[2];
    __shared__ float    y_s; // SUMS

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid  = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = TEAMS == 1 ? wid : wid % PF_WAVES, team = TEAMS == 1 ? 0 : wid / PF_WAVES;
    const int hl = lane >> 5, cl = lane & 31;

    // ---- which (batch, kv head, row block): heavy (late) row blocks first; blocks of one
    //      (batch, kv head) stay on one XCD (work-groups are dealt round-robin to 8 XCDs)
    int rb, g, b, row0, ncols_blk; // (ncols_blk: valid columns of the block)
    auto block = [&](int i) {
        int grp;
        if (a.xcd_map) {
            const int xcd = i & 7, slot = i >> 3;
            grp = (slot / a.n_rb) * 8 + xcd;
            rb  = a.n_rb - 1 - slot % a.n_rb;
        } else {
            grp = i % a.n_groups;
            rb  = a.n_rb - 1 - i / a.n_groups;
        }
        g = grp % a.Hkv;
        b = grp / a.Hkv;
        row0 = rb * a.RB;
        ncols_blk = min(a.n_q - row0, a.RB) * a.gqa;
    };
    block(blockIdx.x);

    // whether the teams walk a row block each: 64 of the mask's flags (4 row blocks x 16 tiles) say, see pf_two_teams
    uint8_t sample = 0;
    auto alike = [&]() {
        const uint64_t bal = __builtin_amdgcn_ballot_w64(sample != 0);
        int most = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) most = max(most, __builtin_popcountll((bal >> (16 * q)) & 0xFFFF));
        return 3 * most <= __builtin_popcountll(bal);
    };
    if constexpr (PART) sample = a.flags[(((2 * (lane >> 4) + 1) * a.n_rb) >> 3) * a.n_tiles + (((2 * (lane & 15) + 1) * a.n_tiles) >> 5)];

    // ---- this wave's columns: lane (hl, cl) holds column cl of each block as the B operand's d = 16 kk + 8 hl .. + 7.
    //      The loads are issued before anything else (the tile list and the first tiles' copies are built while they fly).
    float4_t qraw[NCB][4][2];
    auto load_q = [&]() {
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const int  col = wave * (32 * NCB) + cb * 32 + cl;
            const bool ok  = col < ncols_blk;
            const int  row = row0 + (ok ? (col >> a.gqa_sh) : 0);
            const int  hd  = g * a.gqa + (ok ? (col & (a.gqa - 1)) : 0);
            const float * qp = (const float *) (a.q + (uint64_t) row * a.nbq1 + (uint64_t) hd * a.nbq2 + (uint64_t) b * a.nbq3) + 8 * hl;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                qraw[cb][kk][0] = ((const float4_t *) (qp + 16 * kk))[0];
                qraw[cb][kk][1] = ((const float4_t *) (qp + 16 * kk))[1];
            }
        }
    };
    load_q();
    if constexpr (PART) {
        if (blockIdx.x >= PF_PART && alike()) return; // (the second team of an earlier work-group has its block)
    }

    // ---- active key tiles of this row block, by one wave: list and flags from `at` on, their number
    auto list_tiles = [&](int at) {
        int base = 0;
        for (int t0 = 0; t0 < a.n_tiles; t0 += 64) {
            const int t = t0 + lane;
            uint8_t f = 0;
            if (t < a.n_tiles) {
                if (a.flags) {
                    // a tile is active if any head of the group sees it; mixed if any head needs the mask
                    for (int hd = 0; hd < a.gqa; ++hd) {
                        const int mb = ((b % a.nem3) * a.nem2) + ((g * a.gqa + hd) % a.nem2);
                        const uint8_t ff = a.flags[((uint64_t) mb * a.n_rb + rb) * a.n_tiles + t];
                        f = ff > f ? ff : f;
                        if (a.nem2 == 1) break;
                    }
                    if (a.nem2 > 1 && f) f = 2; // heads may disagree: let the element-wise path decide
                } else {
                    f = 1;
                }
                if (f == 1 && (t + 1) * PF_KT > a.n_kv) f = 3; // partial tile: the bounds are visibility bits
                if (f == 3 && a.flags && a.RB > PF_BIT_ROWS) f = 2; // (the values themselves say the same)
            }
            const uint64_t bal = __builtin_amdgcn_ballot_w64(f != 0);
            const int pos = base + __builtin_popcountll(bal & ((1ull << lane) - 1));
            if (f) { tile_list[at + pos] = (uint16_t) t; tile_flag[at + pos] = f; }
            base += __builtin_popcountll(bal);
        }
        return base;
    };
    if (wid == 0) {
        const int n = list_tiles(0);
        if (lane == 0) n_active_s[0] = n;
    } else if (SUMS && wid == 1) { // the cache write's ordering scalar: k's totals in the low half of the wave, v's in the high
        const int n = hl ? a.n_tv : a.n_tk;
        double tot[PF_TOTALS_INLINE / 32];
#pragma unroll
        for (int u = 0; u < PF_TOTALS_INLINE / 32; ++u) tot[u] = 32 * u + cl < n ? a.totals[hl * PF_TOTALS + 32 * u + cl] : 0.0;
        double t = 0.0;
        const int nmax = max(a.n_tk, a.n_tv); // (zeros behind a side's own count change nothing: a sum from +0.0 is never -0.0)
#pragma unroll
        for (int u = 0; u < PF_TOTALS_INLINE / 32; ++u) {
            if (32 * u >= nmax) break;
            for (int i2 = 0; i2 < min(32, nmax - 32 * u); ++i2) t += __shfl(tot[u], (lane & 32) + i2, 64);
        }
        const float sum = (float) t, sv = __shfl(sum, 32, 64);
        if (lane == 0) y_s = kvs_scalar(sum, sv, a.sync_scale, a.sync_bias);
    }
    bool apart = false, idle = false; // (idle: a second team without a row block)
    if constexpr (PART) {
        static_assert(TEAMS == 2, "teams");
        apart = alike();
        if (apart && team == 1) {
            idle = (int) blockIdx.x + PF_PART >= a.n_rb * a.n_groups;
            if (!idle) {
                block((int) blockIdx.x + PF_PART);
                load_q();
            }
            if (wave == 0) {
                const int n = idle ? 0 : list_tiles(PF_MAX_TILES);
                if (lane == 0) n_active_s[1] = n;
            }
        }
    }
    __syncthreads();
    const int n_first = __builtin_amdgcn_readfirstlane(n_active_s[0]);
    const int n_all = apart ? max(n_first, __builtin_amdgcn_readfirstlane(n_active_s[1])) : n_first;
    // this team's tiles: team, team + TEAMS, ... of the list, or the whole of its own
    const int n_active = TEAMS == 1 ? n_all : apart ? __builtin_amdgcn_readfirstlane(n_active_s[team]) : (n_all - team + TEAMS - 1) / TEAMS;
    const int list_step = apart ? 1 : TEAMS, list_at = apart ? team * PF_MAX_TILES : team;

    // Softmax bookkeeping.  Probabilities are taken relative to a per-column *reference* that trails the running maximum:
    // the S^T accumulator starts at -reference (the same value in a lane's 16 registers: a lane holds one column).  The
    // row sums are formed from the *rounded* probabilities, so numerator and denominator see the same values: the 16 of a
    // unit are added as packed halves (v_pk_add_f16: one instruction per pair; a dot2 or two fp32 additions per pair cost the
    // loop a fifth of its speed, measured), the two partial sums then join the fp32 total.  A unit's contribution doubles
    // as the test for "some score ran far above its reference": only then (or when the tile carries mask values, or a column has not seen a key yet) does the slow
    // block run, which moves the reference up, rescales O and forms the block's probabilities again.
    half8_t   qb[NCB][4];
    float16_t o[NCB][2], negm[NCB];
    float     l[NCB];
    bool      seen[NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
        l[cb] = 0.0f;
        seen[cb] = false;
#pragma unroll
        for (int r = 0; r < 16; ++r) { negm[cb][r] = 0.0f; o[cb][0][r] = 0.0f; o[cb][1][r] = 0.0f; }
    }
    bool all_seen = false; // wave-uniform

    if (n_active > 0) {
        const char * kg = a.k + (uint64_t) g * a.nbk2 + (uint64_t) (b / a.rk3) * a.nbk3;
        const char * vg = a.v + (uint64_t) g * a.nbv2 + (uint64_t) (b / a.rk3) * a.nbv3;
        const char * vlg = VLO ? a.vl + (uint64_t) g * a.nbv2 + (uint64_t) (b / a.rk3) * a.nbv3 : nullptr;
        const uint32_t k_base = (uint32_t) (uintptr_t) (lds_char *) &k_lds[team][0][0];
        const uint32_t v_base = (uint32_t) (uintptr_t) (lds_char *) &v_lds[team][0][0];
        const uint32_t vl_base = (uint32_t) (uintptr_t) (lds_char *) &vl_lds[VLO ? team : 0][0][0];
        const uint32_t bits_base = (uint32_t) (uintptr_t) (lds_char *) &bits_lds[team][0][0];
        // the rows' visibility bits of a tile (used when the tile's flag is 3): lane = (row lane / 2, dword lane % 2); every
        // wave fetches the block's 256 bytes (the same bytes to the same place), only for tiles that need them
        const char * bits_src = a.bits ? (const char *) a.bits + ((uint64_t) (b % a.nem3) * a.nem2 * a.n_q) * a.n_tiles * 8 : a.q;
        // (this lane's offset into them, worked out where it is used: see apply_mask)
        auto bits_row = [&]() {
            int ln = lane;
            asm volatile("" : "+v"(ln));
            return (uint32_t) min(row0 + (ln >> 1), a.n_q - 1) * (uint32_t) a.n_tiles * 8 + 4 * (ln & 1);
        };

        // ---- direct loads: this wave copies rows 16 wave .. 16 wave + 15 of a tile, 8 rows per instruction; lane = (row
        //      lane / 8, chunk position lane % 8), the chunk it fetches is the position un-swizzled
        const int dr = lane >> 3, dp = lane & 7;
        const uint32_t kch = (uint32_t) ((dp ^ dr) << 4), vch = (uint32_t) ((dp ^ (2 * (dr & 3))) << 4);
        uint32_t kof[2], vof[2]; // this lane's byte offsets inside a whole tile, per 8-row block
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            kof[u] = (uint32_t) (16 * wave + 8 * u + dr) * (uint32_t) a.nbk1 + kch;
            vof[u] = (uint32_t) (16 * wave + 8 * u + dr) * (uint32_t) a.nbv1 + vch;
        }
        // A tile's copy is NOPS instructions per wave (K and V, two 8-row blocks each; with VLO the low image too).  They are
        // not issued in one burst: the memory pipeline takes a hundred cycles and more to accept one when all eight waves of
        // a compute unit arrive together, and a wave waits in line.  issue_setup fixes the tile and its stage, issue_op(j)
        // sends instruction j; the steps of the walk send one or two each.
        constexpr int NOPS = VLO ? 6 : 4;
        const char * dma_kt = nullptr, * dma_vt = nullptr, * dma_vlt = nullptr;
        uint32_t dma_kl = 0, dma_vl = 0;
        int dma_last = 0, dma_stage = 0, dma_tile = 0;
        bool dma_bits = false;
        auto issue_setup = [&](int idx, int stage) {
            const int at = list_step * min(idx, n_active - 1) + list_at;
            const int tile = __builtin_amdgcn_readfirstlane(tile_list[at]);
            dma_kt = kg + (uint64_t) tile * PF_KT * a.nbk1;
            dma_vt = vg + (uint64_t) tile * PF_KT * a.nbv1;
            dma_vlt = VLO ? vlg + (uint64_t) tile * PF_KT * a.nbv1 : nullptr;
            dma_kl = k_base + stage * PF_KSTAGE + 2 * wave * PF_KBLK;
            dma_vl = stage * PF_VSTAGE + 2 * wave * 1024;
            dma_last = a.n_kv - 1 - tile * PF_KT; // rows past it are clamped (their scores are masked by the bounds)
            dma_stage = stage;
            dma_tile = tile;
            dma_bits = a.bits && __builtin_amdgcn_readfirstlane(tile_flag[at]) == 3;
        };
        auto issue_op = [&](int j) {
            const int u = j & 1, what = j >> 1; // 0 K, 1 V, 2 V low
            uint32_t off = what == 0 ? kof[u] : vof[u];
            if (dma_last < PF_KT - 1) { // wave-uniform: a ragged last tile
                const int r = min(16 * wave + 8 * u + dr, dma_last);
                off = what == 0 ? (uint32_t) r * (uint32_t) a.nbk1 + kch : (uint32_t) r * (uint32_t) a.nbv1 + vch;
            }
            if (what == 0) pf_dma16(dma_kt, off, dma_kl + u * PF_KBLK);
            if (what == 1) pf_dma16(dma_vt, off, v_base + dma_vl + u * 1024);
            if (what == 2) pf_dma16(dma_vlt, off, vl_base + dma_vl + u * 1024);
            // the rows' visibility bits ride behind the first instruction of a tile that needs them (a further load only
            // makes the waits below more conservative: they count what may still be in flight)
            if (j == 0 && dma_bits) pf_dma4(bits_src + (uint64_t) ((uint32_t) dma_tile * 8u), bits_row(), bits_base + dma_stage * 256);
        };
        auto issue = [&](int idx, int stage) {
            issue_setup(idx, stage);
#pragma unroll
            for (int j = 0; j < NOPS; ++j) issue_op(j);
        };

        for (int t = 0; t < PF_STAGES - 1; ++t) issue(t, t);

        // ---- Q, pre-scaled by scale * log2(e) and rounded to f16
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const bool ok = wave * (32 * NCB) + cb * 32 + cl < ncols_blk;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) {
                float4_t x0 = qraw[cb][kk][0], x1 = qraw[cb][kk][1];
                if (!ok) { x0 = float4_t{0, 0, 0, 0}; x1 = float4_t{0, 0, 0, 0}; }
                x0 *= a.scale2;
                x1 *= a.scale2;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    qb[cb][kk][i]     = (_Float16) x0[i];
                    qb[cb][kk][4 + i] = (_Float16) x1[i];
                }
            }
        }

        // ---- operand addresses inside a stage
        uint32_t kad[4], vad[2];
        {
            const int r8 = cl & 7;
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) kad[kk] = (uint32_t) (team * PF_STAGES * PF_KSTAGE + (cl >> 3) * PF_KBLK + r8 * 128 + (((2 * kk + hl) ^ r8) << 4));
            const int i = lane & 15, gg = (lane >> 4) & 1;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
                vad[dt] = (uint32_t) (team * PF_STAGES * PF_VSTAGE + (4 * hl + (i >> 2)) * 128 + (((4 * dt + 2 * gg + ((i & 3) >> 1)) ^ (2 * (i >> 2))) << 4) + 8 * (i & 1));
        }
        const lds_char * const k_lds0 = (const lds_char *) &k_lds[0][0][0]; // (a team's own lie in the lane's offset)
        const lds_char * const v_lds0 = (const lds_char *) &v_lds[0][0][0];
        const lds_char * const vl_lds0 = (const lds_char *) &vl_lds[0][0][0];

        // The walk is a software pipeline over *units* (a 32-key block x one of the wave's 32-column blocks; 2 NCB per tile,
        // column blocks alternating).  A step handles unit u as 8 groups of { one matrix instruction; exp2, exp2, convert,
        // dot2 of two of u's scores }: the matrix instructions of a step are the 4 of S(u + 1) and the 4 of O += V^T P(u - 1),
        // neither of which depends on the vector work they run beside.  The K operands of a block are read right after the
        // last S instruction that needs the previous ones has issued, the V^T operands likewise behind the O instructions.
        constexpr int NU = 2 * NCB;            // units (steps) per tile
        constexpr int KBAR = NU - 2;           // the step that waits for the next tile (its tail reads that tile's K)
        float16_t sbuf[2];                     // scores of the current and of the next unit (alternating)
        int4_t    pbuf[2][2];                  // probabilities of the current and of the previous unit: [parity][16-key half]
        half8_t   ak[4], av[2][2], avl[2][2];
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) {
                pbuf[x][y] = int4_t{0, 0, 0, 0};
#pragma unroll
                for (int i = 0; i < 8; ++i) { av[x][y][i] = (_Float16) 0.0f; avl[x][y][i] = (_Float16) 0.0f; }
            }

        auto load_ak = [&](int stage, int kb) {
#pragma unroll
            for (int kk = 0; kk < 4; ++kk) ak[kk] = *(const __attribute__((address_space(3))) half8_t *) (k_lds0 + stage * PF_KSTAGE + kad[kk] + kb * 4 * PF_KBLK);
        };
        auto load_av = [&](int stage, int kb) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) {
                    av[dt][ks] = pf_tr8(v_lds0 + stage * PF_VSTAGE + vad[dt] + (32 * kb + 16 * ks) * 128);
                    if constexpr (VLO) avl[dt][ks] = pf_tr8(vl_lds0 + stage * PF_VSTAGE + vad[dt] + (32 * kb + 16 * ks) * 128);
                }
        };
        // the slow block of unit (kb, cb) of `tile`: mask and bounds, the column maxima, the reference moved, O rescaled
        // the mask of unit (kb, cb) of `tile` applied to its scores (tiles flagged 2 or 3 only)
        auto apply_mask = [&](int tile, int stage, int flag, int kb, int cb, float16_t & s) {
            // (the column's row and head are worked out here, behind an opaque statement: hoisted out of the walk they would be
            // held in registers the walk does not have, i.e. spilled)
            int clo = cl;
            asm volatile("" : "+v"(clo));
            if (flag == 3) { // zeros and -inf only (a causal diagonal, a ragged last tile): one bit per key
                const int col = wave * (32 * NCB) + cb * 32 + clo;
                const int rl  = col < ncols_blk ? (col >> a.gqa_sh) : 0;
                uint32_t w;
                if (a.bits) {
                    w = bits_lds[team][stage][2 * rl + kb];
                } else { // no mask: the bounds
                    const int left = a.n_kv - tile * PF_KT - 32 * kb;
                    w = left >= 32 ? 0xFFFFFFFFu : (left <= 0 ? 0u : (1u << left) - 1u);
                }
                w >>= 4 * hl;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = ((w >> (8 * (r >> 2) + (r & 3))) & 1u) ? s[r] : -INFINITY;
            } else { // element-wise mask values / bounds
                const int col  = wave * (32 * NCB) + cb * 32 + clo;
                const bool ok  = col < ncols_blk;
                const int row  = row0 + (ok ? (col >> a.gqa_sh) : 0);
                const int hd   = g * a.gqa + (ok ? (col & (a.gqa - 1)) : 0);
                const float slope = vx_alibi_slope(a.max_bias, (uint32_t) hd, a.n_head_log2, a.m0, a.m1) * 1.44269504088896341f;
                const __half * mrow = a.mask ? (const __half *) (a.mask + (uint64_t) row * a.nbm1 + (uint64_t) (hd % a.nem2) * a.nbm2 + (uint64_t) (b % a.nem3) * a.nbm3) : nullptr;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = tile * PF_KT + 32 * kb + 8 * (r >> 2) + 4 * hl + (r & 3);
                    float x = 0.0f;
                    if (mrow) x = slope * __half2float(mrow[min(key, a.n_kv - 1)]);
                    s[r] += key < a.n_kv ? x : -INFINITY;
                }
            }
        };
        // the slow block: the column maxima of a unit's scores, the reference moved, O rescaled
        auto move_reference = [&](int cb, float16_t & s, float16_t & s_inflight, bool same_cb_inflight) {
            float cm = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) cm = fmaxf(cm, s[r]);
            cm = fmaxf(cm, __shfl_xor(cm, 32, 64));
            // move the reference: up to the new maximum, or (first visible key of the column) onto it wherever it lies
            const bool  vis   = cm != -INFINITY;
            const float delta = !vis ? 0.0f : (seen[cb] ? fmaxf(cm, 0.0f) : cm);
            seen[cb] = seen[cb] || vis;
            if (__builtin_amdgcn_ballot_w64(delta != 0.0f) == 0) return; // nothing moves (wave-uniform)
            // (a column's first reference may lie anywhere below zero -- scores of -200, a mask of the lowest finite value -- and what it
            // would scale is zero: by 1, not by an exponential that overflows, 0 * inf)
            const float f = __builtin_amdgcn_exp2f(-fmaxf(delta, 0.0f));
            s -= delta;
            if (same_cb_inflight) s_inflight -= delta; // scores already formed against the old reference
            negm[cb] -= delta;
            o[cb][0] *= f;
            o[cb][1] *= f;
            l[cb] *= f;
        };
        auto probs = [&](const float16_t & s, int4_t (&pb)[2], float & lt) {
            half2_t acc = half2_t{(_Float16) 0.0f, (_Float16) 0.0f};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const half2_t pr = pf_cvt2(__builtin_amdgcn_exp2f(s[2 * i]), __builtin_amdgcn_exp2f(s[2 * i + 1]));
                pb[i >> 2][i & 3] = __builtin_bit_cast(int, pr);
                acc += pr;
            }
            lt = (float) acc[0] + (float) acc[1];
        };
        // O += V^T P of one unit (outside the pipelined steps: the very last unit)
        auto pv_all = [&](int cb, const int4_t (&pb)[2]) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const half8_t p = __builtin_bit_cast(half8_t, pb[ks]);
#pragma unroll
                for (int dt = 0; dt < 2; ++dt) {
                    o[cb][dt] = mfma32(av[dt][ks], p, o[cb][dt]);
                    if constexpr (VLO) o[cb][dt] = mfma32(avl[dt][ks], p, o[cb][dt]);
                }
            }
        };

        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NL * (PF_STAGES - 2)) : "memory"); // tile 0 has landed
        load_ak(0, 0);
        sbuf[0] = negm[0];
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) sbuf[0] = mfma32(ak[kk], qb[0][kk], sbuf[0]);
        if constexpr (NCB == 1) load_ak(0, 1); // the next unit is the tile's second block already

        for (int it = 0; it < n_active; ++it) {
            const int  stage  = it % PF_STAGES, stage1 = (it + 1) % PF_STAGES;
            const int  tile   = __builtin_amdgcn_readfirstlane(tile_list[list_step * it + list_at]);
            const int  flag   = __builtin_amdgcn_readfirstlane(tile_flag[list_step * it + list_at]); // 1 plain, 2 mask values, 3 visibility bits

#pragma unroll
            for (int k = 0; k < NU; ++k) {
                const int kb = k / NCB, cb = k % NCB;             // this step's unit
                const int cbn = (k + 1) % NCB;                    // the next unit's column block
                const int cbp = (k + NU - 1) % NCB;               // the previous unit's
                const int cur = k & 1, nxt = cur ^ 1;             // NU is even: parities line up across tiles
                if (k == KBAR) {
                    // the next tile has landed for everybody, and everybody is past the previous tile: its stage is refilled,
                    // the copy's instructions spread over this step and the NU - 1 that follow
                    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(NL * (PF_STAGES - 3)) : "memory");
                    issue_setup(it + PF_STAGES - 1, (it + PF_STAGES - 1) % PF_STAGES);
                }
                {   // with four stages the copy has until the wait after next and spreads over a whole round of steps (those
                    // ahead of the first wait belong to a tile the prologue has sent); with three it must be under way before
                    // the next wait and takes the steps that are left of this round
                    constexpr int SPREAD = PF_STAGES >= 4 ? NU : NU - KBAR;
                    constexpr int PER = NOPS / SPREAD; // 4 or 6 instructions over 2 or 4 steps: 1, 2 or 3 a step
                    static_assert(PER * SPREAD == NOPS, "the copy's instructions must divide over its steps");
                    const int sl = (k - KBAR + NU) % NU; // which step of the copy this is
                    if (sl < SPREAD && (k >= KBAR || it > 0)) {
#pragma unroll
                        for (int j = PER * sl; j < PER * sl + PER; ++j) issue_op(j);
                    }
                }
                float lt = 0.0f;
                half2_t acc2 = half2_t{(_Float16) 0.0f, (_Float16) 0.0f};
                // matrix instruction i of the step, and the operand reads that follow it
                auto mat = [&](int i) {
                    if (i < 4) {
                        sbuf[nxt] = mfma32(ak[i], qb[cbn][i], i == 0 ? negm[cbn] : sbuf[nxt]);
                    } else {
                        const int ks = (i - 4) >> 1, dt = (i - 4) & 1;
                        const half8_t p = __builtin_bit_cast(half8_t, pbuf[nxt][ks]); // the previous unit wrote the other parity
                        o[cbp][dt] = mfma32(av[dt][ks], p, o[cbp][dt]);
                        if constexpr (VLO) o[cbp][dt] = mfma32(avl[dt][ks], p, o[cbp][dt]);
                    }
                    if (i == 3) { // the K operands the S instructions after the next step's need
                        if (NCB == 2 && k == 0) load_ak(stage, 1);
                        if (NCB == 2 && k == 2) load_ak(stage1, 0);
                        if (NCB == 1 && k == 0) load_ak(stage1, 0);
                        if (NCB == 1 && k == 1) load_ak(stage1, 1);
                    }
                    // the V^T operands of this unit's block, for the O instructions of the next step (and the one after)
                    if (i == 7 && cb == 0) load_av(stage, kb);
                };
                // One path for every tile: on a masked tile, and while a column has not seen a key, the probabilities
                // formed here are thrown away (the slow block forms them again from the corrected scores), which keeps the
                // matrix instructions in one place; `lt` passes through an opaque statement so that the vector work stays
                // where it is written instead of being moved under the condition.
                // (everything a step's matrix instructions read from LDS was requested a step ago: one wait, stated here, in
                // place of one in front of every instruction; and a pair's conversion trails its exponentials by a group, so
                // that no wait state is needed between a transcendental and its reader)
                __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0)
                float ea = 0.0f, eb = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    mat(i);
                    const float na = __builtin_amdgcn_exp2f(sbuf[cur][2 * i]), nb = __builtin_amdgcn_exp2f(sbuf[cur][2 * i + 1]);
                    if (i > 0) {
                        const half2_t pr = pf_cvt2(ea, eb);
                        pbuf[cur][(i - 1) >> 2][(i - 1) & 3] = __builtin_bit_cast(int, pr);
                        acc2 += pr;
                    }
                    ea = na;
                    eb = nb;
                    __builtin_amdgcn_sched_barrier(0);
                }
                {
                    const half2_t pr = pf_cvt2(ea, eb);
                    pbuf[cur][1][3] = __builtin_bit_cast(int, pr);
                    acc2 += pr;
                }
                lt = (float) acc2[0] + (float) acc2[1];
                asm volatile("" : "+v"(lt));
                bool redo = !all_seen || __builtin_amdgcn_ballot_w64(!(lt <= PF_SUM_LIMIT)) != 0;
                if (flag != 1) { // a masked tile: what was formed above is void, the scores take the mask first
                    apply_mask(tile, stage, flag, kb, cb, sbuf[cur]);
                    redo = true;
                    if (all_seen) {
                        probs(sbuf[cur], pbuf[cur], lt);
                        redo = __builtin_amdgcn_ballot_w64(!(lt <= PF_SUM_LIMIT)) != 0;
                    }
                }
                if (redo) {
                    move_reference(cb, sbuf[cur], sbuf[nxt], NCB == 1);
                    probs(sbuf[cur], pbuf[cur], lt);
                    if (!all_seen) {
                        bool every = true;
#pragma unroll
                        for (int c2 = 0; c2 < NCB; ++c2) every = every && seen[c2];
                        all_seen = __builtin_amdgcn_ballot_w64(!every) == 0;
                    }
                }
                l[cb] += lt;
            }
        }
        pv_all(NCB - 1, pbuf[(NU - 1) & 1]); // the last unit's
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the loads issued past the last tile
    }
    if constexpr (TEAMS == 2) {
        // The walk's barriers are the work-group's: one in front, one a tile.  A team makes up for the tiles it has
        // not, or for a walk it has not at all.  (A loop of its own: a wave's count is uniform.)
        const int mine = n_active > 0 ? n_active + 1 : 0, most = n_all > 0 ? (apart ? n_all : (n_all + 1) / 2) + 1 : 0;
        for (int i = mine; i < most; ++i) asm volatile("s_barrier" ::: "memory");
        if (idle) return;
        l[0] += __shfl_xor(l[0], 32, 64); // (the two lanes of a column hold disjoint keys)
    }
    if (TEAMS == 2 && !apart) {
        static_assert(TEAMS == 1 || NCB == 1, "the hand-over below is one column block's");
        __syncthreads(); // nobody reads a stage any more, and every direct load has landed
        // the second team's sums through its own stages: o by register and lane, then the column's L and reference
        float * const po = (float *) &k_lds[TEAMS - 1][0][0] + wave * (16 + 2) * 64, * const po1 = (float *) &v_lds[TEAMS - 1][0][0] + wave * 16 * 64;
        static_assert(PF_WAVES * 18 * 64 * 4 <= PF_STAGES * PF_KSTAGE && PF_WAVES * 16 * 64 * 4 <= PF_STAGES * PF_VSTAGE, "room for a team's sums");
        if (team == 1) {
#pragma unroll
            for (int r = 0; r < 16; ++r) { po[r * 64 + lane] = o[0][0][r]; po1[r * 64 + lane] = o[0][1][r]; }
            po[16 * 64 + lane] = l[0];
            po[17 * 64 + lane] = -negm[0][0];
        }
        __syncthreads();
        if (team == 1) return;
        const float L1 = po[16 * 64 + lane], M1 = po[17 * 64 + lane], M0 = -negm[0][0];
        // (a column that saw no key has the sum 0 and no reference; one that did has at least its largest score's 1)
        const float m  = l[0] == 0.0f ? M1 : L1 == 0.0f ? M0 : fmaxf(M0, M1);
        const float f0 = l[0] == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(M0 - m), f1 = L1 == 0.0f ? 0.0f : __builtin_amdgcn_exp2f(M1 - m);
        l[0] = l[0] * f0 + L1 * f1;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            o[0][0][r] = o[0][0][r] * f0 + po[r * 64 + lane] * f1;
            o[0][1][r] = o[0][1][r] * f0 + po1[r * 64 + lane] * f1;
            negm[0][r] = -m;
        }
    }

    // ---- finish: lane (hl, cl), d block dt, register r holds d = 32 dt + 8 (r / 4) + 4 hl + r % 4 of column cl
    int lane_e = threadIdx.x & 63; // (worked out again rather than kept alive through the walk)
    asm volatile("" : "+v"(lane_e));
    const int hl_e = lane_e >> 5, cl_e = lane_e & 31;
    const bool  has_add = SUMS || a.add1;
    const float addend = SUMS ? y_s : a.add1 ? *a.add1 : 0.0f;
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
        const int  col = wave * (32 * NCB) + cb * 32 + cl_e;
        const bool ok  = col < ncols_blk;
        const int  row = row0 + (ok ? (col >> a.gqa_sh) : 0);
        const int  hd  = g * a.gqa + (ok ? (col & (a.gqa - 1)) : 0);
        float L = TEAMS == 2 ? l[cb] : l[cb] + __shfl_xor(l[cb], 32, 64); // the two lanes of a column hold disjoint keys
        float M = -negm[cb][0]; // the reference the sums are relative to
        float ms = 1.0f;
        if (a.sinks) { // ggml/src/ggml-cpu/ops.cpp:8598-8615, in the log2 domain
            const float sk = a.sinks[hd] * 1.44269504088896341f;
            float vs = 1.0f;
            if (sk > M) { ms = __builtin_amdgcn_exp2f(M - sk); } else { vs = __builtin_amdgcn_exp2f(sk - M); }
            L = L * ms + vs;
        }
        const float inv = L == 0.0f ? 0.0f : ms / L;
        if (ok && a.tile_out) { // (uniform choice) rounded to f16 as the product's activation pass would round the stored value
            // k = hd * 64 + d: tile (k block 2 hd + dt, 16 tokens), slot (q4, token mod 16), halves 4 hl .. 4 hl + 3
            const uint32_t tokf = (uint32_t) b * a.tile_ts + (uint32_t) row;
            _Float16 * tb = a.tile_out + ((((uint64_t) b * a.tile_bs + (uint64_t) (2 * hd) * a.tile_tt + (tokf >> 4)) * 64 + (tokf & 15)) * 8 + 4 * hl_e);
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
#pragma clang fp contract(off) // (the normalised value is rounded before the addend joins it, as two nodes would)
                    float4_t r = float4_t{o[cb][dt][4 * q4], o[cb][dt][4 * q4 + 1], o[cb][dt][4 * q4 + 2], o[cb][dt][4 * q4 + 3]} * inv;
                    if (has_add) r += addend;
                    asm volatile("" : "+v"(r)); // the fp32 value the node holds, formed as such, then rounded
                    *(half4_t *) (tb + ((uint64_t) dt * a.tile_tt * 64 + 16 * q4) * 8) = half4_t{(_Float16) r[0], (_Float16) r[1], (_Float16) r[2], (_Float16) r[3]};
                }
        } else if (ok) {
            float * out = a.dst + (((uint64_t) b * a.n_q + row) * a.Hq + hd) * D;
#pragma unroll
            for (int dt = 0; dt < 2; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
#pragma clang fp contract(off) // (the normalised value is rounded before the addend joins it, as two nodes would)
                    float4_t r = float4_t{o[cb][dt][4 * q4], o[cb][dt][4 * q4 + 1], o[cb][dt][4 * q4 + 2], o[cb][dt][4 * q4 + 3]} * inv;
                    if (has_add) r += addend;
                    *(float4_t *) (out + 32 * dt + 8 * q4 + 4 * hl_e) = r;
                }
        }
    }
}

} // namespace

// Called by vx_flash_attn_ext when the shape suits this kernel; returns VX_ERR_UNSUPPORTED
// (without touching the error string) when the caller should use the general kernel.
bool vx_fattn_prefill_accepts(const vx_tensor * q, const vx_tensor * k, float logit_softcap) {
    if (q->ne[0] != 64 || logit_softcap != 0.0f) return false;
    // F32 K/V (the reference's own cache type, and what a prefill sees: the keys straight from the projections) are
    // staged as f16 here -- K rounded like Q is, V as a high and a low half, so the result carries the same error as with
    // an f16 cache (the rounding of P, about 1.3e-3 on unit-scale data against the 2e-3 bar).  The general kernel keeps
    // hi + lo parts of everything (1e-6) and is 10 - 20 times slower on such shapes; VX_FA_F32_PREFILL=0 sends F32 K/V
    // there (read on every call).
    if (k->type == VX_TYPE_F32) {
        const char * e = getenv("VX_FA_F32_PREFILL");
        if (e && atoi(e) == 0) return false;
    } else if (k->type != VX_TYPE_F16) {
        return false;
    }
    const int Hq = (int) q->ne[2], Hkv = (int) k->ne[2], gqa = Hq / Hkv;
    if (gqa > PF_COLS / 2 || ((PF_COLS / 2) % gqa) != 0) return false;
    const int n_q = (int) q->ne[1], n_kv = (int) k->ne[1];
    const int RB = PF_COLS / gqa, n_rb = (n_q + RB - 1) / RB, n_tiles = (n_kv + PF_KT - 1) / PF_KT;
    const int n_groups = (int) q->ne[3] * Hkv;
    if (n_q * gqa < PF_COLS || n_tiles > PF_MAX_TILES) return false;
    if (k->type == VX_TYPE_F16 && k->nb[1] >= (1u << 25)) return false; // a tile's rows are addressed by 32-bit offsets
    // too few work-groups: the wave kernel spreads wider (one stream of 512 tokens, 32 blocks of 256 columns run as 64 of
    // 128: 19 us here against 28 us there; 256 tokens, 16 blocks: 15 us against 14 us)
    return (int64_t) n_rb * n_groups >= 32;
}

// Whether a grid of 128-column work-groups runs with two teams of waves (pf_kernel's TEAMS) instead of one.
// Up to a work-group for each of 256 compute units the second team runs on what would be idle issue slots, over the same columns; it
// costs nothing where the walk is a few tiles.  Beyond, such work-groups come one after another where two of one team would share a
// compute unit.  That repays itself where a few long walks end the call, as under a causal mask, and costs a prologue where all
// walks are alike; which it is stands in the mask's flags, so the kernel decides: 64 of them, spread over rows and keys, and where
// the longest of the four sampled walks is not a third longer than their mean, a work-group's teams take a row block each, placed as one
// team's work-groups would be.  Us a call, f16 keys and values, one team / two over the same columns:
//   256 work-groups: 2048 causal tokens 38.2 / 31.1, no mask 32.8 / 27.9, 2 x 1024 24.3 / 21.5, 4 x 512 17.7 / 17.7; 512 new of 4096 keys
//   (64) 62.7 / 45.5.  No mask, beyond: 2300 tokens (288) 47.6 / 54.3, 4096 (512) 91.3 / 93.2.
// One team / two over the same columns / by the flags:
//   tokens (work-groups)   2064 (258)           2300 (288)           2700 (338)           3300 (414)           4096 (512)
//   causal                 42.3  35.2  34.4     48.1  40.2  39.3     57.6  48.5  48.1     68.0  59.8  59.0     72.3  65.8  65.3
//   all visible            52.6  61.4  52.8     60.1  68.7  60.1     73.0  81.3  73.4     87.5  93.7  84.8     99.9  103.6 98.8
//   a third hidden behind  40.7  48.4  41.3     46.9  54.5  47.1     56.9  65.1  58.4     67.6  74.3  66.6     74.1  79.0  74.3
//   half, then causal      41.4  43.4  42.2     47.4  47.9  46.6     57.0  57.5  57.3     68.8  71.1  70.6     76.6  80.0  79.5
//   4 causal sequences     28.9  27.4  29.3     35.2  32.0  35.7     43.4  40.0  44.6     51.1  53.4  52.8     37.6  41.8  38.3
//   window of 512          23.4  27.5  25.7     26.9  34.7  30.3     35.7  43.1  38.1     38.6  46.0  39.8     31.1  38.7  34.7
// (the short walks lose what the second team's list and rows cost behind the decision).  F32 keys and values alike: causal 2300 59.9 / 49.8 /
// 49.1, all visible 76.4 / 87.6 / 77.7.  With fewer tiles the causal call gains little and the others lose more: 2 x 1200 (300) causal
// 29.7 / 28.4 / 29.0, half then causal 29.5 / 34.0; and towards 512 work-groups the causal walks are no longer few: 2 x 1700 (428) 39.2 /
// 40.3, 2 x 2048 (512) 40.1 / 41.3.
static bool pf_two_teams(int64_t n_wg, int n_tiles, bool masked) {
    if (n_wg <= PF_PART) return true;
    return masked && n_wg <= 2 * PF_PART && n_tiles >= 32 && n_tiles * (700 - n_wg) >= 7500;
}

vx_status vx_fattn_prefill(const vx_tensor * q, const vx_tensor * k, const vx_tensor * v, const vx_tensor * mask,
                           const float * sinks, const float * addend, const vx_tensor * dst, float scale, float max_bias,
                           float logit_softcap, hipStream_t st, const vx_pf_front * front) {
    if (!vx_fattn_prefill_accepts(q, k, logit_softcap)) return VX_ERR_UNSUPPORTED;
    const int Hq = (int) q->ne[2], Hkv = (int) k->ne[2], gqa = Hq / Hkv;
    const int n_q = (int) q->ne[1], n_kv = (int) k->ne[1];
    const int n_groups = (int) q->ne[3] * Hkv;
    // work-groups of 256 columns; of 128 while 256 would put fewer than two work-groups on every CU
    // (with the low image of V a wave of 64 columns does not fit two to a SIMD: F32 K/V always take the 128-column form)
    const bool half_cols = k->type == VX_TYPE_F32 || (int64_t) ((n_q + PF_COLS / gqa - 1) / (PF_COLS / gqa)) * n_groups < 512;
    const int cols = half_cols ? PF_COLS / 2 : PF_COLS;
    const int RB = cols / gqa, n_rb = (n_q + RB - 1) / RB, n_tiles = (n_kv + PF_KT - 1) / PF_KT;

    pf_args a;
    a.q = (const char *) q->data; a.k = (const char *) k->data; a.v = (const char *) v->data;
    a.mask = mask ? (const char *) mask->data : nullptr;
    a.sinks = sinks;
    a.add1 = addend;
    a.tile_out = nullptr; a.tile_tt = a.tile_bs = a.tile_ts = 0;
    a.dst = (float *) dst->data;
    a.flags = nullptr;
    a.bits = nullptr;
    a.nbq1 = q->nb[1]; a.nbq2 = q->nb[2]; a.nbq3 = q->nb[3];
    a.nbk1 = k->nb[1]; a.nbk2 = k->nb[2]; a.nbk3 = k->nb[3];
    a.nbv1 = v->nb[1]; a.nbv2 = v->nb[2]; a.nbv3 = v->nb[3];
    a.nbm1 = mask ? mask->nb[1] : 0; a.nbm2 = mask ? mask->nb[2] : 0; a.nbm3 = mask ? mask->nb[3] : 0;
    a.n_q = n_q; a.n_kv = n_kv; a.Hq = Hq; a.Hkv = Hkv; a.gqa = gqa;
    a.gqa_sh = 0;
    while ((1 << a.gqa_sh) < gqa) ++a.gqa_sh;
    a.ne3 = (int) q->ne[3]; a.rk3 = (int) (q->ne[3] / k->ne[3]);
    a.nem2 = mask ? (int) mask->ne[2] : 1; a.nem3 = mask ? (int) mask->ne[3] : 1;
    a.RB = RB; a.n_rb = n_rb; a.n_tiles = n_tiles; a.n_groups = n_groups;
    a.xcd_map = (n_groups % 8 == 0);
    a.scale2 = scale * 1.44269504088896341f;
    a.max_bias = max_bias;
    a.n_head_log2 = 1u << (uint32_t) floor(log2((double) Hq));
    a.m0 = powf(2.0f, -(max_bias) / a.n_head_log2);
    a.m1 = powf(2.0f, -(max_bias / 2.0f) / a.n_head_log2);
    a.kv_f32 = k->type == VX_TYPE_F32;
    a.vl = nullptr;

    // one workspace block: the mask's tile flags, then (F32 K/V) the f16 images of K, V high and V low
    const size_t bits_bytes = mask ? (size_t) a.nem2 * a.nem3 * n_q * n_tiles * 8 : 0;
    const size_t flag_bytes = mask ? ((bits_bytes + (size_t) a.nem2 * a.nem3 * n_rb * n_tiles + 255) & ~(size_t) 255) : 0;
    const size_t plane = a.kv_f32 ? (size_t) k->ne[3] * Hkv * n_kv * 64 * sizeof(_Float16) : 0;
    char * ws = nullptr;
    const size_t front_bytes = front ? front->bytes : 0;
    if (front_bytes + flag_bytes + 3 * plane) {
        void * p = nullptr;
        vx_status rc = vx_workspace(st, front_bytes + flag_bytes + 3 * plane, &p);
        if (rc != VX_OK) return rc;
        ws = (char *) p;
    }
    pf_prep_args p = {};
    p.key_blocks = 1;
    a.totals = nullptr; a.n_tk = a.n_tv = 0; a.sync_scale = a.sync_bias = 0.0f;
    if (front) { // the cache write's totals and scalar lie at the front of the block
        p.ks = *front->ks; p.vs = *front->vs;
        if (front->base) *front->base = ws;
        p.totals = (double *) ws;
        p.store_large = front->store_large;
        const int64_t uk = kvs_host_units(p.ks), uv = kvs_host_units(p.vs);
        a.n_tk = p.store_large ? (int) std::min<int64_t>(PF_TOTALS, (uk + 1023) / 1024) : 16;
        a.n_tv = p.store_large ? (int) std::min<int64_t>(PF_TOTALS, (uv + 1023) / 1024) : 16;
        p.n_tk = a.n_tk;
        p.n_store = p.store_large ? a.n_tk + a.n_tv : 8;
        if (std::max(a.n_tk, a.n_tv) <= PF_TOTALS_INLINE) a.totals = p.totals;
        else a.add1 = (const float *) (ws + VX_PF_SCALAR_AT);
        a.sync_scale = front->scale; a.sync_bias = front->bias;
        if (front->tiles) {
            a.tile_out = (_Float16 *) (ws + front->tiles_at);
            a.tile_tt = front->tile_tt; a.tile_bs = front->tile_bs; a.tile_ts = front->tile_ts;
        }
        ws += front_bytes;
    }
    int64_t blocks = p.n_store;
    p.n_kv = n_kv;
    p.m.n_q = n_q; p.m.n_kv = n_kv; p.m.RB = RB; p.m.n_rb = n_rb; p.m.n_tiles = n_tiles;
    if (mask) {
        p.m.mask = a.mask; p.m.nbm1 = a.nbm1; p.m.nbm2 = a.nbm2; p.m.nbm3 = a.nbm3; p.m.nem2 = a.nem2;
        p.m.vec_ok = (uintptr_t) a.mask % 16 == 0 && a.nbm1 % 16 == 0 && a.nbm2 % 16 == 0 && a.nbm3 % 16 == 0;
        p.m.bits = (uint8_t *) ws; p.m.flags = (uint8_t *) ws + bits_bytes;
        const int64_t units = (int64_t) n_tiles * n_rb * a.nem2 * a.nem3;
        if (units > 0x7ffffff0) return vx_fail(VX_ERR_UNSUPPORTED, "flash_attn_ext: launch too large");
        p.m.n_units = (int) units;
        p.n_mask = (int) ((units + 3) / 4);
        blocks += p.n_mask;
        a.bits = p.m.bits;
        a.flags = p.m.flags;
    }
    if (a.kv_f32) {
        p.k16 = (_Float16 *) (ws + flag_bytes); p.vhi = (_Float16 *) (ws + flag_bytes + plane); p.vlo = (_Float16 *) (ws + flag_bytes + 2 * plane);
        p.k = a.k; p.v = a.v;
        p.nbk1 = a.nbk1; p.nbk2 = a.nbk2; p.nbk3 = a.nbk3; p.nbv1 = a.nbv1; p.nbv2 = a.nbv2; p.nbv3 = a.nbv3;
        p.Hkv = Hkv; p.key_blocks = (n_kv * 8 + 255) / 256;
        blocks += (int64_t) p.key_blocks * Hkv * k->ne[3];
        a.k = (const char *) p.k16; a.v = (const char *) p.vhi; a.vl = (const char *) p.vlo;
        a.nbk1 = a.nbv1 = 128; a.nbk2 = a.nbv2 = (uint64_t) n_kv * 128; a.nbk3 = a.nbv3 = (uint64_t) Hkv * n_kv * 128;
    }
    if (blocks > 0x7fffffff) return vx_fail(VX_ERR_UNSUPPORTED, "flash_attn_ext: launch too large");
    if (p.n_store && (kvs_overlaps(p.ks, k) || kvs_overlaps(p.ks, v) || kvs_overlaps(p.vs, k) || kvs_overlaps(p.vs, v) ||
                      (mask && (kvs_overlaps(p.ks, mask) || kvs_overlaps(p.vs, mask))))) { // (what the rest reads is being written: one after the other)
        pf_prep_args first = p;
        first.n_mask = 0;
        vx_launch(pf_prep_kernel<true>, dim3((unsigned) p.n_store), dim3(256), 0, st, first);
        VX_LAUNCH_CHECK();
        blocks -= p.n_store;
        p.n_store = 0;
    }
    if (blocks && blocks == p.n_mask && n_rb <= 65535 && a.nem2 * a.nem3 <= 65535) {
        // Up to four units a compute unit go out one by one (a causal call of 512 tokens 16.2 us against 16.3 with four to a work-group,
        // 16 x 256 18.5 / 18.9), more of them by fours (2048: 38.4 us against 39.1, 4096: 72.1 / 73.8).
        const dim3 grid((unsigned) n_tiles, (unsigned) n_rb, (unsigned) (a.nem2 * a.nem3));
        const pf_mask_args & m = p.m;
        if (m.n_units <= 1024) vx_launch(pf_mask_kernel<1>, grid, dim3(64), 0, st, m.mask, m.nbm1, m.nbm2, m.nbm3, m.nem2, m.n_q, m.n_kv, m.RB, m.n_rb, m.n_tiles, m.vec_ok, m.flags, m.bits);
        else vx_launch(pf_mask_kernel<4>, dim3((grid.x + 3) / 4, grid.y, grid.z), dim3(256), 0, st, m.mask, m.nbm1, m.nbm2, m.nbm3, m.nem2, m.n_q, m.n_kv, m.RB, m.n_rb, m.n_tiles, m.vec_ok, m.flags, m.bits);
        VX_LAUNCH_CHECK();
    } else if (blocks) {
        if (p.n_store) vx_launch(pf_prep_kernel<true>, dim3((unsigned) blocks), dim3(256), 0, st, p);
        else           vx_launch(pf_prep_kernel<false>, dim3((unsigned) blocks), dim3(256), 0, st, p);
        VX_LAUNCH_CHECK();
    }
    if (front && !a.totals) {
        vx_launch(pf_scalar_kernel, dim3(1), dim3(PF_TOTALS), 0, st, (const double *) p.totals, a.n_tk, a.n_tv, a.sync_scale, a.sync_bias, (float *) a.add1);
        VX_LAUNCH_CHECK();
    }
    const dim3 grid((unsigned) (n_rb * n_groups)), block(64 * PF_WAVES), block2(2 * 64 * PF_WAVES);
    const bool two = half_cols && pf_two_teams((int64_t) n_rb * n_groups, n_tiles, mask != nullptr);
    const bool part = two && n_rb * n_groups > PF_PART; // (with a mask only)
    if (a.totals) {
        if (!half_cols)            vx_launch(pf_kernel<false, 2, true>, grid, block, 0, st, a);
        else if (a.kv_f32 && part) vx_launch(pf_kernel<true, 1, true, 2, true>, grid, block2, 0, st, a);
        else if (part)             vx_launch(pf_kernel<false, 1, true, 2, true>, grid, block2, 0, st, a);
        else if (a.kv_f32 && two)  vx_launch(pf_kernel<true, 1, true, 2>, grid, block2, 0, st, a);
        else if (two)              vx_launch(pf_kernel<false, 1, true, 2>, grid, block2, 0, st, a);
        else if (a.kv_f32)         vx_launch(pf_kernel<true, 1, true>, grid, block, 0, st, a);
        else                       vx_launch(pf_kernel<false, 1, true>, grid, block, 0, st, a);
    } else if (half_cols) {
        if (a.kv_f32 && part)      vx_launch(pf_kernel<true, 1, false, 2, true>, grid, block2, 0, st, a);
        else if (part)             vx_launch(pf_kernel<false, 1, false, 2, true>, grid, block2, 0, st, a);
        else if (a.kv_f32 && two)  vx_launch(pf_kernel<true, 1, false, 2>, grid, block2, 0, st, a);
        else if (two)              vx_launch(pf_kernel<false, 1, false, 2>, grid, block2, 0, st, a);
        else if (a.kv_f32)         vx_launch(pf_kernel<true, 1>, grid, block, 0, st, a);
        else                       vx_launch(pf_kernel<false, 1>, grid, block, 0, st, a);
    } else {
        vx_launch(pf_kernel<false, 2>, grid, block, 0, st, a);
    }
    VX_LAUNCH_CHECK();
    return VX_OK;
}
