// stack.hip -- a whole decoder stack over a few token rows (a decode step, one LocDiT pass) as one resident launch.
//
// What bounds a decode step issued operator by operator is not its bytes (24 layers of Q8_0 weights: 0.3 GB, 55 us) but its
// chain of some 145 dependent kernels: every boundary costs 1.7 us before the next kernel's first instruction, another
// microsecond until its weights' first bytes, and a drain at the end -- 31 us a layer.  Here one work-group per compute unit
// stays for the whole stack.  Every work-group owns the same few rows of every matrix of a layer:
//   * weights do not depend on the tokens, so a work-group's rows (64 KB a layer) are loaded into LDS a whole layer ahead,
//     straight from memory, by waves that have nothing to wait for at that point;
//   * activations pass between the compute units through memory past the L2s (device-scope loads and stores).  There is no
//     barrier across the grid and no flag: each exchanged value has a slot of its own, filled with a pattern that no result
//     has (all ones, a NaN that is never published) by a small kernel in front, and a consumer re-reads its values until none
//     of them is the pattern.  A value is on its way for one store and one load: 1.4 us from all compute units to all compute
//     units (16 KB; 2.5 for 64), against 4.6 to 6.2 us for data behind flags and 10.6 us for a release / acquire barrier.
// Steps of 24 layers (us, separate calls / here): one sequence over 37 keys 767 / 524, over 8000 keys 729 / 534; two over 700 keys 718 /
// 528; four 791 / 559; eight 846 / 693.  A layer of the one-token step is 20 us now: 6 of the attention, and for each product 1.4 of the
// exchange, the sums' ends and the next activations' norm (1.0) and 0.5 to 1.4 of the products.  Waves wait for 78 % of their cycles; a
// SIMD issues vector work for 16 % of the time and matrix work for 2 %, LDS bank conflicts take 1 to 4 %: trips bound it.
// Beside other work (one row, separate / here): next to a stream of large products 3358 / 663 us, of 203-token prompts 919 / 537, of
// elementwise passes over 1 GiB 2635 / 1142 -- the launch keeps its compute units once it has them.  Next to others of its kind: one
// step on each of two streams 895 / 1019, three 968 / 1700 (two that wait for the chip get half of it each, and without a whole
// one nothing is loaded ahead), eight rows on each of three 1217 / 3264: a program that steps several streams keeps the separate calls.
// The arithmetic is that of the separate kernels, sum by sum: products in the order of gemv_dma_kernel's waves, RMS_NORM by
// one wave a row, the key ranges and the merge of fattn.hip.  The results are the same bits.
//
// Residency.  Waiting on another work-group needs that work-group to be running.  Nothing promises that all of the grid is:
// another stream's kernels may hold compute units, and two of these launches may share the chip.  So a work-group that
// starts takes a number; the first one waits until all have come or 100 us have passed and then closes the entrance.  The
// work-groups inside deal the work among themselves -- all of them are running, so every wait ends -- and one that comes later
// leaves at once.  Which work-group does what does not change any sum.
#include "mm_common.hpp"
#include "rope_common.hpp"
#include "stack.hpp"

#include <cstdlib>
#include <cstring>
#include <type_traits>

namespace {

constexpr int VS_DEV = 16;                  // buffer access with device scope (sc1): past the L2s
constexpr uint32_t VS_CLOSED = 0x80000000u; // bit of the arrival count: the entrance is closed
constexpr uint32_t VS_ENTER_TICKS = 10000;  // of the 100 MHz clock
constexpr int VS_SPIN_LIMIT = 1 << 18;      // polls of a wait that cannot take that long (some 200 ms)

// which attention a launch has
enum { VS_F16 = 0, VS_F32 = 1, VS_F16_SHORT = 2, VS_SELF = 3 };

// A layer's four products: q / k / v, o, gate / up, down
enum { VS_QKV = 0, VS_O = 1, VS_GU = 2, VS_D = 3 };

struct vs_layer {
    const char *  w[4];          // q, o, gate, down
    const char *  wk, * wv, * wu;
    const float * nin, * npost;
    char *        kc, * vc;
};
// what a product's code needs, laid out so that one scalar load brings it
struct vs_prod {
    int in_at, out_at;           // the layer's part of the exchange area: activations read, results written
    int row_bytes, pieces;       // an activation row: bytes, 16-byte pieces per lane
    int kp;                      // halfs between staged rows in LDS
    int img, slot, cols;         // weight rows in LDS: first, bytes of one, how many a tile has
    int units;
    int nw, per;                 // slots of a sum, blocks of one (of a staged half)
    int sfar;                    // gate and up: from the one's rows to the other's in LDS
    int gain;                    // norm weights in LDS
    int nap;                     // 64-clock pauses in front of the first look at the activations
    int reserved;
};
struct vs_args {
    vs_prod       P[4];
    vs_layer      L[VX_STACK_MAX_LAYERS];
    const float * x;
    float *       out;
    const float * norm;
    const int32_t * pos;
    const float * ff;
    const char *  mask;
    uint64_t      nbm1;
    uint32_t *    ctl;               // [0] arrivals, [1] work-groups inside
    char *        xch;               // exchange area
    uint32_t      xch_bytes, layer_bytes;
    uint32_t      o_qkv, o_attn, o_h, o_act, o_x; // offsets in a layer's part
    uint32_t      o_part, o_ml;      // key-range partials (one set for all layers)
    uint64_t      nbc1, nbc2, nbc3;  // cache strides: row, head, sequence
    rope_params   rp;
    float         eps, res_scale, scale, sync_scale, sync_bias;
    int           n_layer, N, T, hidden, ffn, hq, hkv, gqa, n_past, n_splits, chunk, n_col_tiles;
    int           pp, ro, rf;        // pairs of q / k / v rows, rows of o and down, gate/up pairs of a work-group
    int           l_red, l_rcs;      // LDS offsets
    int           nap_q, nap_part;   // 64-clock pauses in front of the first look at q, at the partials
};
static_assert(sizeof(vs_prod) <= 64 && sizeof(vs_args) <= 4096, "kernel arguments");

typedef __attribute__((address_space(3))) char vs_lds_char;

__device__ __forceinline__ void vs_barrier() { // LDS traffic done, direct loads into LDS left in flight
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
__device__ __forceinline__ void vs_nap(int n) { // n times 64 clocks
    for (; n > 0; --n) __builtin_amdgcn_s_sleep(1);
}
__device__ __forceinline__ void vs_wait_vm0() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// 16 bytes per lane from global memory into LDS at lds + 16 lane (one statement: the compiler may use M0 between two)
__device__ __forceinline__ void vs_dma16(const char * g, uint32_t lds) {
    const uint32_t base = (uint32_t) __builtin_amdgcn_readfirstlane((int) lds);
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(base) : "memory");
}
__device__ __forceinline__ void vs_dma16_nt(const char * base, uint32_t off, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" ::"v"(off), "s"(base), "s"(lds) : "memory");
}

// ---- the exchange
struct vs_xch {
    __amdgpu_buffer_rsrc_t r;
    // a wait was given up (uniform per wave): nothing waits any more, so that the grid drains.  What is missing stays the pattern, a NaN in
    // F32 and in f16, and every use of it -- norm, product, softmax weight, sum, residual -- gives NaN: the token rows that depend on it end
    // as NaN in all their columns (the next norm's sum is NaN), the others are right.
    int dead;
    __device__ __forceinline__ int4_t ld(uint32_t off) const { return __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, VS_DEV); }
    __device__ __forceinline__ void st(uint32_t off, float v) const {
        const int b = __builtin_bit_cast(int, v);
        __builtin_amdgcn_raw_buffer_store_b32(b == -1 ? 0x7fffffff : b, r, off, 0, VS_DEV);
    }
    __device__ __forceinline__ void st4(uint32_t off, float4_t v) const {
        int4_t b = __builtin_bit_cast(int4_t, v);
#pragma unroll
        for (int i = 0; i < 4; ++i) b[i] = b[i] == -1 ? 0x7fffffff : b[i];
        __builtin_amdgcn_raw_buffer_store_b128(b, r, off, 0, VS_DEV);
    }
    __device__ __forceinline__ void st_h2(uint32_t off, _Float16 lo, _Float16 hi) const {
        const int b = __builtin_bit_cast(int, half2_t{lo, hi});
        __builtin_amdgcn_raw_buffer_store_b32(b == -1 ? 0x7fff7fff : b, r, off, 0, VS_DEV);
    }
    __device__ __forceinline__ void clear4(uint32_t off) const { // (the pattern is made where it is stored: kept, it is four registers of every lane)
        int m = -1;
        asm volatile("" : "+v"(m));
        __builtin_amdgcn_raw_buffer_store_b128(int4_t{m, m, m, m}, r, off, 0, VS_DEV);
    }
    __device__ __forceinline__ void clear2(uint32_t off) const {
        typedef int int2_v __attribute__((ext_vector_type(2)));
        int m = -1;
        asm volatile("" : "+v"(m));
        __builtin_amdgcn_raw_buffer_store_b64(int2_v{m, m}, r, off, 0, VS_DEV);
    }
};
// (as arithmetic: a chain of tests becomes a branch each)
__device__ __forceinline__ int vs_miss(const int4_t & v) { return (int) (v[0] == -1) | (int) (v[1] == -1) | (int) (v[2] == -1) | (int) (v[3] == -1); }

// NC chunks of 16 bytes per lane at base + c * step, chunk c wanted where c < n and the lane takes part; returns when all of
// a wave's chunks are there
template <int NC>
__device__ __forceinline__ void vs_load(const vs_xch & x, uint32_t base, uint32_t step, int n, bool lane_on, int4_t (&v)[NC]) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (c < n && lane_on) v[c] = x.ld(base + (uint32_t) c * step);
        else                  v[c] = int4_t{0, 0, 0, 0};
    }
}
template <int NC>
__device__ __forceinline__ bool vs_all(const int4_t (&v)[NC]) {
    int miss = 0;
#pragma unroll
    for (int c = 0; c < NC; ++c) miss |= vs_miss(v[c]);
    return miss == 0;
}
template <int NC>
__device__ __forceinline__ void vs_await(vs_xch & x, uint32_t base, uint32_t step, int n, bool lane_on, int4_t (&v)[NC]) { // v: loaded once already
    for (int spin = 0; __builtin_amdgcn_ballot_w64(!vs_all(v)) != 0 && !x.dead; ++spin) {
        if (spin >= VS_SPIN_LIMIT) { x.dead = 1; break; }
        asm volatile("" ::: "memory");
        vs_load(x, base, step, n, lane_on, v);
    }
}
template <int NC>
__device__ __forceinline__ void vs_poll(vs_xch & x, uint32_t base, uint32_t step, int n, bool lane_on, int4_t (&v)[NC]) {
    asm volatile("" ::: "memory");
    vs_load(x, base, step, n, lane_on, v);
    vs_await(x, base, step, n, lane_on, v);
}
__device__ __forceinline__ float4_t vs_f4(const int4_t & v) { return __builtin_bit_cast(float4_t, v); }

// a value as it is, rounded to F32: no conversion or addition behind it may take over the operation that made it
__device__ __forceinline__ void vs_round32(float4_t & v) {
    asm volatile("" : "+v"(v));
}

// ---- products: one k block (32 values) of a weight row's LDS image against the staged activations.  sh: 16 where the block
// starts on a dword (its quants then sit 2 bytes in), 0 where it starts 2 bytes past one
struct vs_block { uint32_t w0, w1, w2; _Float16 d; half8_t x; };
__device__ __forceinline__ void vs_block_load(vs_block & b, const vs_lds_char * sd, const vs_lds_char * sq, const vs_lds_char * xp) {
    const __attribute__((address_space(3))) uint32_t * q = (const __attribute__((address_space(3))) uint32_t *) sq;
    b.w0 = q[0]; b.w1 = q[1]; b.w2 = q[2];
    b.d  = *(const __attribute__((address_space(3))) _Float16 *) sd;
    b.x  = *(const __attribute__((address_space(3))) half8_t *) xp;
}
__device__ __forceinline__ float4_t vs_block_mul(const vs_block & b, uint32_t sh) {
    return mfma16(b.x, q8_to_half8(__builtin_amdgcn_alignbit(b.w1, b.w0, sh), __builtin_amdgcn_alignbit(b.w2, b.w1, sh)), float4_t{0, 0, 0, 0});
}
// `per` blocks of each of a wave's sums, NW blocks apart, four blocks at a time: two of acc0, two of acc1 whose operands lie sfar / xfar
// bytes further on -- or (SINGLE) four of acc0.  sd, sq, xp: LDS addresses of the first block's scale, its quants, its activations.
template <int NW, bool SINGLE>
__device__ __forceinline__ void vs_blocks(uint32_t sd, uint32_t sq, uint32_t xp, int per, uint32_t sfar, uint32_t xfar, uint32_t sh, float4_t & acc0, float4_t & acc1) {
    constexpr uint32_t SS = NW * VX_Q8_BLOCK, XS = NW * 64;
#pragma unroll 1
    for (int i = 0; i < per; i += SINGLE ? 4 : 2) {
        const vs_lds_char * const d0 = (const vs_lds_char *) (uintptr_t) sd, * const q0 = (const vs_lds_char *) (uintptr_t) sq, * const x0 = (const vs_lds_char *) (uintptr_t) xp;
        vs_block b[4];
        vs_block_load(b[0], d0, q0, x0);
        vs_block_load(b[1], d0 + SS, q0 + SS, x0 + XS);
        if constexpr (SINGLE) {
            vs_block_load(b[2], d0 + 2 * SS, q0 + 2 * SS, x0 + 2 * XS);
            vs_block_load(b[3], d0 + 3 * SS, q0 + 3 * SS, x0 + 3 * XS);
        } else {
            vs_block_load(b[2], d0 + sfar, q0 + sfar, x0 + xfar);
            vs_block_load(b[3], d0 + sfar + SS, q0 + sfar + SS, x0 + xfar + XS);
        }
        float4_t y[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = vs_block_mul(b[e], sh);
        acc0 += y[0] * (float) b[0].d;
        acc0 += y[1] * (float) b[1].d;
        float4_t & far = SINGLE ? acc0 : acc1;
        far += y[2] * (float) b[2].d;
        far += y[3] * (float) b[3].d;
        sd += (SINGLE ? 4 : 2) * SS;
        sq += (SINGLE ? 4 : 2) * SS;
        xp += (SINGLE ? 4 : 2) * XS;
    }
}

template <int NW> // one sum, two blocks at a time
__device__ __forceinline__ void vs_sum_of(uint32_t sd, uint32_t sq, uint32_t xp, int per, uint32_t sh, float4_t & acc) {
    constexpr uint32_t SS = NW * VX_Q8_BLOCK, XS = NW * 64;
#pragma unroll 1
    for (int i = 0; i < per; i += 2, sd += 2 * SS, sq += 2 * SS, xp += 2 * XS) {
        const vs_lds_char * const d0 = (const vs_lds_char *) (uintptr_t) sd, * const q0 = (const vs_lds_char *) (uintptr_t) sq, * const x0 = (const vs_lds_char *) (uintptr_t) xp;
        vs_block b[2];
        vs_block_load(b[0], d0, q0, x0);
        vs_block_load(b[1], d0 + SS, q0 + SS, x0 + XS);
        float4_t y[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) y[e] = vs_block_mul(b[e], sh);
        acc += y[0] * (float) b[0].d;
        acc += y[1] * (float) b[1].d;
    }
}

// ---- attention over registers: one tile of 32 keys (NH = 1: its first 16), the arithmetic of fattn_cols16_kernel
__device__ __forceinline__ void vs_pk2(half8_t & dst, int i, float a, float b) {
    typedef __fp16 fp16x2 __attribute__((ext_vector_type(2)));
    const fp16x2 v = __builtin_amdgcn_cvt_pkrtz(a, b);
    dst[i]     = (_Float16) v[0];
    dst[i + 1] = (_Float16) v[1];
}
__device__ __forceinline__ void vs_split(const float4_t & a, const float4_t & b, half8_t & hi, half8_t & lo) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        hi[i]     = (_Float16) a[i];
        lo[i]     = (_Float16) (a[i] - (float) hi[i]);
        hi[4 + i] = (_Float16) b[i];
        lo[4 + i] = (_Float16) (b[i] - (float) hi[4 + i]);
    }
}
template <int NH> struct vs_kv {
    half8_t khi[NH][2], klo[NH][2], vhi[NH][2], vlo[NH][2];
};
struct vs_soft {
    float4_t o[2][2];
    float    m, l;
};
template <bool F32, int NH>
__device__ __forceinline__ void vs_consume(const vs_kv<NH> & t, int kb, int kv1, const float (&mask)[NH][4], const half8_t (&qhi)[2], const half8_t (&qlo)[2],
                                           float scale, int lane, vs_soft & st) {
    const int j = lane >> 4, c = lane & 15;
    const bool tail = NH == 1 || kb + 32 > kv1;
    float4_t s[NH];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
        float4_t acc = {0, 0, 0, 0};
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            acc = mfma16(t.khi[h][p], qlo[p], acc);
            if constexpr (F32) acc = mfma16(t.klo[h][p], qhi[p], acc);
            acc = mfma16(t.khi[h][p], qhi[p], acc);
        }
        s[h] = acc;
    }
    float cmax = -INFINITY;
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float x = s[h][r] * scale;
            if (tail) x += kb + 16 * h + 4 * j + r < kv1 ? mask[h][r] : -INFINITY;
            s[h][r] = x;
            cmax = fmaxf(cmax, x);
        }
    cmax = fmaxf(cmax, __shfl_xor(cmax, 16, 64));
    cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
    const float m_new = fmaxf(st.m, cmax);
    const float shift = (m_new == -INFINITY) ? 0.0f : m_new;
    const float alpha = __builtin_amdgcn_exp2f(st.m - shift);
    float   psum = 0.0f, pvv[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    half8_t phi, plo;
#pragma unroll
    for (int h = 0; h < NH; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            pvv[4 * h + r] = __builtin_amdgcn_exp2f(s[h][r] - shift);
            psum += pvv[4 * h + r];
        }
#pragma unroll
    for (int i = 0; i < 8; i += 2) vs_pk2(phi, i, pvv[i], pvv[i + 1]);
#pragma unroll
    for (int i = 0; i < 8; i += 2) vs_pk2(plo, i, pvv[i] - (float) phi[i], pvv[i + 1] - (float) phi[i + 1]);
    st.l = st.l * alpha + psum;
    st.m = m_new;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
        for (int p = 0; p < 2; ++p) { st.o[p][0] *= alpha; st.o[p][1] *= alpha; }
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        half8_t sel;
#pragma unroll
        for (int i = 0; i < 8; ++i) sel[i] = (j == 2 * u + (c >> 3) && i == (c & 7)) ? (_Float16) 1.0f : (_Float16) 0.0f;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            float4_t t0 = mfma16(t.vhi[0][p], sel, float4_t{0, 0, 0, 0}), t1 = float4_t{0, 0, 0, 0};
            if constexpr (NH == 2) t1 = mfma16(t.vhi[NH - 1][p], sel, t1);
            if constexpr (F32) {
                t0 = mfma16(t.vlo[0][p], sel, t0);
                if constexpr (NH == 2) t1 = mfma16(t.vlo[NH - 1][p], sel, t1);
            }
            half8_t vt;
#pragma unroll
            for (int r = 0; r < 4; r += 2) { vs_pk2(vt, r, t0[r], t0[r + 1]); vs_pk2(vt, 4 + r, t1[r], t1[r + 1]); }
            st.o[p][u] = mfma16(vt, plo, st.o[p][u]);
            st.o[p][u] = mfma16(vt, phi, st.o[p][u]);
            if constexpr (F32) {
                half8_t vl;
#pragma unroll
                for (int r = 0; r < 4; r += 2) {
                    vs_pk2(vl, r, t0[r] - (float) vt[r], t0[r + 1] - (float) vt[r + 1]);
                    vs_pk2(vl, 4 + r, t1[r] - (float) vt[4 + r], t1[r + 1] - (float) vt[4 + r + 1]);
                }
                st.o[p][u] = mfma16(vl, phi, st.o[p][u]);
            }
        }
    }
}

// the normalised result of 4 consecutive d, plus the cache write's ordering scalar, as the o projection's f16 activations
__device__ __forceinline__ void vs_finish(const vs_xch & x, float4_t acc, float L, bool has_addend, float addend, uint32_t off) {
#pragma clang fp contract(off)
    const float inv = L == 0.0f ? 0.0f : 1.0f / L;
    float4_t r = acc * inv;
    if (has_addend) r += addend;
    x.st_h2(off, (_Float16) r[0], (_Float16) r[1]);
    x.st_h2(off + 4, (_Float16) r[2], (_Float16) r[3]);
}

// The ordering scalar of a layer's cache write (kvs_scalar): the sums over all tokens' k and v.  With the graph's scale and
// bias of zero it is zero or NaN, whatever the order of the sums.
struct vs_kvs { int4_t v[4]; }; // four pieces of 16 bytes a lane
__device__ __forceinline__ void vs_addend_load(const vs_args & a, const vs_xch & x, uint32_t qkv, int e0, int lane, vs_kvs & s) {
    const int per_tok = 32 * a.hkv, total = a.N * per_tok;
    const uint32_t row = (uint32_t) (a.hq + 2 * a.hkv) * 256u, kv_at = qkv + (uint32_t) a.hq * 256u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int e = e0 + lane + 64 * i, tok = e / per_tok;
        s.v[i] = int4_t{0, 0, 0, 0};
        if (e < total) s.v[i] = x.ld(kv_at + (uint32_t) tok * row + (uint32_t) (e - tok * per_tok) * 16u);
    }
}
template <bool F16> // s: the first pieces, loaded once already
__device__ __forceinline__ float vs_addend(const vs_args & a, vs_xch & x, uint32_t qkv, int lane, vs_kvs & s) {
    const int per_tok = 32 * a.hkv, total = a.N * per_tok;
    double k = 0.0, v = 0.0;
#pragma unroll 1
    for (int e0 = 0;;) {
        for (int spin = 0; __builtin_amdgcn_ballot_w64(!vs_all(s.v)) != 0 && !x.dead; ++spin) {
            if (spin >= VS_SPIN_LIMIT) { x.dead = 1; break; }
            asm volatile("" ::: "memory");
            vs_addend_load(a, x, qkv, e0, lane, s);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int e = e0 + lane + 64 * i;
            float4_t f = vs_f4(s.v[i]);
            if constexpr (F16) {
#pragma unroll
                for (int r = 0; r < 4; ++r) f[r] = (float) (_Float16) f[r];
            }
            const double t = (double) f[0] + (double) f[1] + (double) f[2] + (double) f[3];
            if (e % per_tok < 16 * a.hkv) k += t; else v += t;
        }
        e0 += 256;
        if (e0 >= total) break;
        vs_addend_load(a, x, qkv, e0, lane, s);
    }
    const float sk = (float) vx_wave_sum(k), sv = (float) vx_wave_sum(v);
    const float t = sk + sv;
    return a.sync_bias == 0.0f ? t * a.sync_scale : fmaf(t, a.sync_scale, a.sync_bias);
}

// ---- the streaming attention of an f16 cache (fattn_dec64_kernel), one wave = one key range of one (sequence, KV head)
constexpr int VD_STAGES = 3, VD_KBLK = 1152, VD_KTILE = 4 * VD_KBLK, VD_VTILE = 32 * 128;
constexpr int VD_WAVE_LDS = (VD_STAGES + 1) * (VD_KTILE + VD_VTILE);
constexpr int VD_WAVES = 2;
constexpr float VD_SUM_LIMIT = 2048.0f;

__device__ __forceinline__ half8_t vd_tr8(const vs_lds_char * p) {
    typedef short short4_t __attribute__((ext_vector_type(4)));
    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3))) *) p);
    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((short4_t __attribute__((address_space(3))) *) (p + 16 * 128));
    return __builtin_bit_cast(half8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// where a key range's result goes: the partials, or (one range) the attention's output
__device__ __forceinline__ uint32_t vs_part(const vs_args & a, int bg, int sp, int c) { return (uint32_t) ((bg * a.n_splits + sp) * a.gqa + c); }

__device__ __forceinline__ void vd_range(const vs_args & a, vs_xch & x, const vs_layer & Ly, uint32_t layer, int bg, int sp, char * lds, int lane) {
    const int j = lane >> 4, c = lane & 15;
    const int b = bg / a.hkv, g = bg - b * a.hkv;
    const bool col_ok = c < a.gqa;
    const uint32_t qkv_row = layer + a.o_qkv + (uint32_t) b * (uint32_t) (a.hq + 2 * a.hkv) * 256u;
    const int n_kv = a.n_past + 1;
    const int kv0 = sp * a.chunk, kv1 = min(n_kv, kv0 + a.chunk);
    const int ntile = (kv1 - kv0 + 31) / 32;
    const int ndma = min(ntile, max(0, (a.n_past - kv0) / 32));
    char * const k_lds = lds, * const v_lds = lds + (VD_STAGES + 1) * VD_KTILE;
    const char * kg = Ly.kc + (uint64_t) g * a.nbc2 + (uint64_t) b * a.nbc3;
    const char * vg = Ly.vc + (uint64_t) g * a.nbc2 + (uint64_t) b * a.nbc3;
    const uint32_t k_base = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (uintptr_t) (vs_lds_char *) k_lds);
    const uint32_t v_base = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (uintptr_t) (vs_lds_char *) v_lds);
    const int dr = lane >> 3, dp = lane & 7;
    const int ck = dp ^ dr, cv = dp ^ (2 * (dr & 3));
    const uint32_t kof = (uint32_t) dr * (uint32_t) a.nbc1 + (uint32_t) (ck << 4), vof = (uint32_t) dr * (uint32_t) a.nbc1 + (uint32_t) (cv << 4);
    const uint64_t row8 = 8 * a.nbc1;
    const char * knext = kg + (uint64_t) kv0 * a.nbc1;
    const char * vnext = vg + (uint64_t) kv0 * a.nbc1;
    auto issue = [&](int stage) { // the next tile of the range (every streamed tile lies wholly in the cache)
        const uint32_t kl = k_base + (uint32_t) (stage * VD_KTILE), vl = v_base + (uint32_t) (stage * VD_VTILE);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            vs_dma16_nt(knext, kof, kl + u * VD_KBLK);
            vs_dma16_nt(vnext, vof, vl + u * 1024);
            knext += row8;
            vnext += row8;
        }
    };
#pragma unroll
    for (int t = 0; t < VD_STAGES; ++t)
        if (t < ndma) issue(t);

    // the cached rows of the tile that ends in the step's own key go to its buffer before the wait for that key
    const int kbm = kv0 + 32 * ndma;
    const bool mixed = ndma < ntile;
    char * const kmix = k_lds + VD_STAGES * VD_KTILE + lane * 16, * const vmix = v_lds + VD_STAGES * VD_VTILE + lane * 16;
    if (mixed) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int key = min(kbm + 8 * u + dr, a.n_past - 1);
            *(half8_t *) (kmix + u * VD_KBLK) = *(const half8_t *) (kg + (uint64_t) key * a.nbc1 + ck * 16);
            *(half8_t *) (vmix + u * 1024)    = *(const half8_t *) (vg + (uint64_t) key * a.nbc1 + cv * 16);
        }
    }
    int4_t qv[4];
    vs_nap(a.nap_q);
    vs_poll(x, qkv_row + (uint32_t) (g * a.gqa + c) * 256u + (uint32_t) j * 64u, 16, 4, col_ok, qv);
    if (mixed) {
        int4_t kn[2], vn[2];
        const uint32_t kat = qkv_row + (uint32_t) (a.hq + g) * 256u, vat = kat + (uint32_t) a.hkv * 256u;
        vs_load(x, kat + (uint32_t) ck * 32u, 16, 2, true, kn);
        vs_load(x, vat + (uint32_t) cv * 32u, 16, 2, true, vn);
        vs_await(x, kat + (uint32_t) ck * 32u, 16, 2, true, kn);
        vs_await(x, vat + (uint32_t) cv * 32u, 16, 2, true, vn);
        half8_t k1, v1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            k1[i] = (_Float16) vs_f4(kn[0])[i]; k1[4 + i] = (_Float16) vs_f4(kn[1])[i];
            v1[i] = (_Float16) vs_f4(vn[0])[i]; v1[4 + i] = (_Float16) vs_f4(vn[1])[i];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int key = kbm + 8 * u + dr;
            if (key == a.n_past) { // the cache write
                *(half8_t *) (const_cast<char *>(kg) + (uint64_t) key * a.nbc1 + ck * 16) = k1;
                *(half8_t *) (const_cast<char *>(vg) + (uint64_t) key * a.nbc1 + cv * 16) = v1;
            }
            if (key >= a.n_past) {
                *(half8_t *) (kmix + u * VD_KBLK) = k1;
                *(half8_t *) (vmix + u * 1024)    = v1;
            }
        }
    }
    half8_t qh[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        float4_t x0 = vs_f4(qv[2 * p]) * a.scale, x1 = vs_f4(qv[2 * p + 1]) * a.scale;
        vs_round32(x0);
        vs_round32(x1);
#pragma unroll
        for (int i = 0; i < 4; ++i) { qh[p][i] = col_ok ? (_Float16) x0[i] : (_Float16) 0.0f; qh[p][4 + i] = col_ok ? (_Float16) x1[i] : (_Float16) 0.0f; }
    }
    uint32_t kad[2], vad[4];
    {
        const int r8 = c & 7;
#pragma unroll
        for (int p = 0; p < 2; ++p) kad[p] = (uint32_t) ((c >> 3) * VD_KBLK + r8 * 128 + (((2 * j + p) ^ r8) << 4));
#pragma unroll
        for (int dt = 0; dt < 4; ++dt)
            vad[dt] = (uint32_t) ((4 * j + (c >> 2)) * 128 + (((2 * dt + ((c & 3) >> 1)) ^ (2 * (c >> 2))) << 4) + 8 * (c & 1));
    }
    const vs_lds_char * const k_lds0 = (const vs_lds_char *) k_lds;
    const vs_lds_char * const v_lds0 = (const vs_lds_char *) v_lds;
    float4_t o[4], negm = float4_t{0, 0, 0, 0};
#pragma unroll
    for (int dt = 0; dt < 4; ++dt) o[dt] = float4_t{0, 0, 0, 0};
    float l = 0.0f;
    bool  seen = false, all_seen = false;
    typedef __fp16 fp16x2 __attribute__((ext_vector_type(2)));
    auto probs = [&](const float4_t (&s)[2], int4_t & pb, float & lt) {
        half2_t acc = half2_t{(_Float16) 0.0f, (_Float16) 0.0f};
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 4; r += 2) {
                const fp16x2 pr = __builtin_amdgcn_cvt_pkrtz(__builtin_amdgcn_exp2f(s[h][r]), __builtin_amdgcn_exp2f(s[h][r + 1]));
                pb[2 * h + (r >> 1)] = __builtin_bit_cast(int, pr);
                acc += __builtin_bit_cast(half2_t, pr);
            }
        lt = (float) acc[0] + (float) acc[1];
    };
    for (int t = 0; t < ntile; ++t) {
        const bool streamed = t < ndma; // wave-uniform
        const int stage = streamed ? t % VD_STAGES : VD_STAGES;
        const int kb = kv0 + 32 * t;
        if (streamed) {
            const int younger = min(VD_STAGES - 1, ndma - 1 - t);
            if (younger >= 2)      asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
            else if (younger == 1) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
            else                   asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        half8_t kk[2][2], vv[4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int p = 0; p < 2; ++p) kk[h][p] = *(const __attribute__((address_space(3))) half8_t *) (k_lds0 + stage * VD_KTILE + kad[p] + h * 2 * VD_KBLK);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) vv[dt] = vd_tr8(v_lds0 + stage * VD_VTILE + vad[dt]);
        __builtin_amdgcn_s_waitcnt(0xC07F); // lgkmcnt(0): the stage is in registers, the tile three ahead may overwrite it
        if (t + VD_STAGES < ndma) issue(stage);
        float4_t s[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            s[h] = mfma16(kk[h][0], qh[0], negm);
            s[h] = mfma16(kk[h][1], qh[1], s[h]);
        }
        int4_t pb;
        float  lt;
        probs(s, pb, lt);
        const bool tail = kb + 32 > kv1; // wave-uniform
        if (tail || !all_seen || __builtin_amdgcn_ballot_w64(!(lt <= VD_SUM_LIMIT)) != 0) {
            if (tail) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[h][r] = kb + 16 * h + 4 * j + r < kv1 ? s[h][r] : -INFINITY;
            }
            float cm = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])), fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
            cm = fmaxf(cm, __shfl_xor(cm, 16, 64));
            cm = fmaxf(cm, __shfl_xor(cm, 32, 64));
            const bool  vis   = cm != -INFINITY;
            const float delta = !vis ? 0.0f : (seen ? fmaxf(cm, 0.0f) : cm);
            seen = seen || vis;
            const float f = __builtin_amdgcn_exp2f(-fmaxf(delta, 0.0f)); // (a first reference below zero scales sums of zero: by 1, not by what may be inf)
            s[0] -= delta;
            s[1] -= delta;
            negm -= delta;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) o[dt] *= f;
            l *= f;
            probs(s, pb, lt);
            all_seen = __builtin_amdgcn_ballot_w64(!seen) == 0;
        }
        l += lt;
        const half8_t p8 = __builtin_bit_cast(half8_t, pb);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) o[dt] = mfma16(vv[dt], p8, o[dt]);
    }
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    const float m = seen ? -negm[0] : -INFINITY;
    if (a.n_splits == 1) {
        vs_kvs kvs;
        vs_addend_load(a, x, layer + a.o_qkv, 0, lane, kvs);
        const float addend = vs_addend<true>(a, x, layer + a.o_qkv, lane, kvs);
        if (col_ok) {
            const uint32_t at = layer + a.o_attn + ((uint32_t) b * (uint32_t) a.hq + (uint32_t) (g * a.gqa + c)) * 128u;
#pragma unroll
            for (int dt = 0; dt < 4; ++dt) vs_finish(x, o[dt], l, true, addend, at + (uint32_t) (16 * dt + 4 * j) * 2u);
        }
    } else if (col_ok) {
        const uint32_t p = vs_part(a, bg, sp, c);
#pragma unroll
        for (int dt = 0; dt < 4; ++dt) x.st4(a.o_part + p * 256u + (uint32_t) (16 * dt + 4 * j) * 4u, o[dt]);
        if (j == 0) { x.st(a.o_ml + p * 8u, m); x.st(a.o_ml + p * 8u + 4u, l); }
    }
}

// A key range in registers: an F32 cache (F32), or an f16 cache of at most 64 keys; the step's own key behind the cached ones
template <bool F32>
__device__ __forceinline__ void vr_range(const vs_args & a, vs_xch & x, const vs_layer & Ly, uint32_t layer, int bg, int sp, char * lds, int lane) {
    constexpr int ES = F32 ? 4 : 2, NV = F32 ? 4 : 2; // bytes per value; 16-byte pieces of a lane's 16 values
    const int j = lane >> 4, c = lane & 15;
    const int b = bg / a.hkv, g = bg - b * a.hkv;
    const bool col_ok = c < a.gqa;
    const uint32_t qkv_row = layer + a.o_qkv + (uint32_t) b * (uint32_t) (a.hq + 2 * a.hkv) * 256u;
    const int n_kv = a.n_past + 1;
    const int kv0 = sp * a.chunk, kv1 = min(n_kv, kv0 + a.chunk);
    const bool last = kv1 == n_kv; // the step's own key is in this range
    char * kg = Ly.kc + (uint64_t) g * a.nbc2 + (uint64_t) b * a.nbc3 + (uint64_t) (16 * j) * ES;
    char * vg = Ly.vc + (uint64_t) g * a.nbc2 + (uint64_t) b * a.nbc3 + (uint64_t) (16 * j) * ES;
    int4_t kr[2][NV], vr[2][NV];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int key = min(kb + 16 * h + c, a.n_past - 1);
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                kr[h][i] = *(const int4_t *) (kg + (uint64_t) key * a.nbc1 + i * 16);
                vr[h][i] = *(const int4_t *) (vg + (uint64_t) key * a.nbc1 + i * 16);
            }
        }
    };
    // a tile's cached rows as operands; then (once it is there) the step's own key in the lanes whose row it is
    auto cached = [&](vs_kv<2> & t) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                if constexpr (F32) {
                    vs_split(vs_f4(kr[h][2 * p]), vs_f4(kr[h][2 * p + 1]), t.khi[h][p], t.klo[h][p]);
                    vs_split(vs_f4(vr[h][2 * p]), vs_f4(vr[h][2 * p + 1]), t.vhi[h][p], t.vlo[h][p]);
                } else {
                    t.khi[h][p] = __builtin_bit_cast(half8_t, kr[h][p]);
                    t.vhi[h][p] = __builtin_bit_cast(half8_t, vr[h][p]);
                }
            }
    };
    fetch(kv0);
    int4_t qv[4];
    const uint32_t kat = qkv_row + (uint32_t) (a.hq + g) * 256u + (uint32_t) j * 64u, vat = kat + (uint32_t) a.hkv * 256u;
    const uint32_t qat = qkv_row + (uint32_t) (g * a.gqa + c) * 256u + (uint32_t) j * 64u;
    int4_t * const kn = (int4_t *) (lds + 64 * j), * const vn = (int4_t *) (lds + 256 + 64 * j); // the step's own key and value
    vs_kv<2> t;
    cached(t); // (in the shadow of the wait for q)
    vs_nap(a.nap_q);
    asm volatile("" ::: "memory");
    vs_load(x, qat, 16, 4, col_ok, qv);
    {
        int4_t k1[4], v1[4];
        vs_load(x, kat, 16, 4, last, k1);
        vs_load(x, vat, 16, 4, last, v1);
        vs_await(x, qat, 16, 4, col_ok, qv);
        vs_await(x, kat, 16, 4, last, k1);
        vs_await(x, vat, 16, 4, last, v1);
        if (c == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i) { kn[i] = k1[i]; vn[i] = v1[i]; }
        }
    }
    vs_kvs kvs;
    if (a.n_splits == 1) vs_addend_load(a, x, layer + a.o_qkv, 0, lane, kvs); // (under way while the tiles are worked on)
    half8_t qhi[2], qlo[2];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        float4_t x0 = vs_f4(qv[2 * p]), x1 = vs_f4(qv[2 * p + 1]);
        if (!col_ok) { x0 = float4_t{0, 0, 0, 0}; x1 = float4_t{0, 0, 0, 0}; }
        vs_split(x0, x1, qhi[p], qlo[p]);
    }
    vs_soft st;
    st.m = -INFINITY; st.l = 0.0f;
#pragma unroll
    for (int p = 0; p < 2; ++p) { st.o[p][0] = float4_t{0, 0, 0, 0}; st.o[p][1] = float4_t{0, 0, 0, 0}; }
    const float no_mask[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll 1
    for (int kb = kv0;;) {
        if (kb + 32 < kv1) fetch(kb + 32);
        if (kb + 32 > a.n_past) { // uniform: the tile has rows beyond the cache (the step's own key, clamped rows included)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (kb + 16 * h + c >= a.n_past) {
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        if constexpr (F32) {
                            vs_split(vs_f4(kn[2 * p]), vs_f4(kn[2 * p + 1]), t.khi[h][p], t.klo[h][p]);
                            vs_split(vs_f4(vn[2 * p]), vs_f4(vn[2 * p + 1]), t.vhi[h][p], t.vlo[h][p]);
                        } else {
#pragma unroll
                            for (int i = 0; i < 4; ++i) {
                                t.khi[h][p][i] = (_Float16) vs_f4(kn[2 * p])[i]; t.khi[h][p][4 + i] = (_Float16) vs_f4(kn[2 * p + 1])[i];
                                t.vhi[h][p][i] = (_Float16) vs_f4(vn[2 * p])[i]; t.vhi[h][p][4 + i] = (_Float16) vs_f4(vn[2 * p + 1])[i];
                            }
                        }
                    }
                }
        }
        vs_consume<F32, 2>(t, kb, kv1, no_mask, qhi, qlo, a.scale, lane, st);
        kb += 32;
        if (kb >= kv1) break;
        cached(t);
    }
    if (last && c == 0) { // the cache write: lane-group j holds 16 values of the row
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            int4_t k1, v1;
            if constexpr (F32) { k1 = kn[i]; v1 = vn[i]; }
            else {
                half8_t hk, hv;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    hk[r] = (_Float16) vs_f4(kn[2 * i])[r]; hk[4 + r] = (_Float16) vs_f4(kn[2 * i + 1])[r];
                    hv[r] = (_Float16) vs_f4(vn[2 * i])[r]; hv[4 + r] = (_Float16) vs_f4(vn[2 * i + 1])[r];
                }
                k1 = __builtin_bit_cast(int4_t, hk); v1 = __builtin_bit_cast(int4_t, hv);
            }
            *(int4_t *) (kg + (uint64_t) a.n_past * a.nbc1 + i * 16) = k1;
            *(int4_t *) (vg + (uint64_t) a.n_past * a.nbc1 + i * 16) = v1;
        }
    }
    st.l += __shfl_xor(st.l, 16, 64);
    st.l += __shfl_xor(st.l, 32, 64);
    float addend = 0.0f;
    if (a.n_splits == 1) addend = vs_addend<!F32>(a, x, layer + a.o_qkv, lane, kvs);
    if (!col_ok) return;
    const uint32_t p_at = vs_part(a, bg, sp, c);
    const uint32_t at = layer + a.o_attn + ((uint32_t) b * (uint32_t) a.hq + (uint32_t) (g * a.gqa + c)) * 128u;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int d0 = 16 * (2 * u + (j >> 1)) + 8 * p + 4 * (j & 1);
            if (a.n_splits == 1) {
                vs_finish(x, st.o[p][u], st.l, true, addend, at + (uint32_t) d0 * 2u);
            } else {
                x.st4(a.o_part + p_at * 256u + (uint32_t) d0 * 4u, st.o[p][u]);
            }
        }
    if (a.n_splits != 1 && j == 0) { x.st(a.o_ml + p_at * 8u, st.m); x.st(a.o_ml + p_at * 8u + 4u, st.l); }
}

// A sequence of at most 16 tokens that attends to itself (no cache): one wave = 16 (token, head) columns of one KV head
__device__ __forceinline__ void vr_self(const vs_args & a, vs_xch & x, uint32_t layer, int tile, int lane) {
    const int j = lane >> 4, c = lane & 15;
    const int bg = tile / a.n_col_tiles, ct = tile - bg * a.n_col_tiles;
    const int b = bg / a.hkv, g = bg - b * a.hkv;
    const int col = ct * 16 + c;
    const bool col_ok = col < a.T * a.gqa;
    const int iq1 = col_ok ? col / a.gqa : 0, head = g * a.gqa + (col_ok ? col - iq1 * a.gqa : 0);
    const uint32_t row = (uint32_t) (a.hq + 2 * a.hkv) * 256u, seq = layer + a.o_qkv + (uint32_t) (b * a.T) * row;
    float mask[1][4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        mask[0][r] = a.mask ? 1.44269504088896341f * __half2float(((const __half *) (a.mask + (uint64_t) iq1 * a.nbm1))[min(4 * j + r, a.T - 1)]) : 0.0f;
    int4_t qv[4], kr[4], vr[4];
    const uint32_t qat = seq + (uint32_t) iq1 * row + (uint32_t) head * 256u + (uint32_t) j * 64u;
    const uint32_t kat = seq + (uint32_t) min(c, a.T - 1) * row + (uint32_t) (a.hq + g) * 256u + (uint32_t) j * 64u, vat = kat + (uint32_t) a.hkv * 256u;
    vs_nap(a.nap_q);
    asm volatile("" ::: "memory");
    vs_load(x, kat, 16, 4, true, kr);
    vs_load(x, vat, 16, 4, true, vr);
    vs_load(x, qat, 16, 4, true, qv);
    vs_await(x, kat, 16, 4, true, kr);
    vs_await(x, vat, 16, 4, true, vr);
    vs_await(x, qat, 16, 4, true, qv);
    half8_t qhi[2], qlo[2];
    vs_kv<1> t;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        float4_t x0 = vs_f4(qv[2 * p]), x1 = vs_f4(qv[2 * p + 1]);
        if (!col_ok) { x0 = float4_t{0, 0, 0, 0}; x1 = float4_t{0, 0, 0, 0}; }
        vs_split(x0, x1, qhi[p], qlo[p]);
        vs_split(vs_f4(kr[2 * p]), vs_f4(kr[2 * p + 1]), t.khi[0][p], t.klo[0][p]);
        vs_split(vs_f4(vr[2 * p]), vs_f4(vr[2 * p + 1]), t.vhi[0][p], t.vlo[0][p]);
    }
    vs_soft st;
    st.m = -INFINITY; st.l = 0.0f;
#pragma unroll
    for (int p = 0; p < 2; ++p) { st.o[p][0] = float4_t{0, 0, 0, 0}; st.o[p][1] = float4_t{0, 0, 0, 0}; }
    vs_consume<true, 1>(t, 0, a.T, mask, qhi, qlo, a.scale, lane, st);
    st.l += __shfl_xor(st.l, 16, 64);
    st.l += __shfl_xor(st.l, 32, 64);
    if (!col_ok) return;
    const uint32_t at = layer + a.o_attn + ((uint32_t) (b * a.T + iq1) * (uint32_t) a.hq + (uint32_t) head) * 128u;
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int u = 0; u < 2; ++u) vs_finish(x, st.o[p][u], st.l, false, 0.0f, at + (uint32_t) (16 * (2 * u + (j >> 1)) + 8 * p + 4 * (j & 1)) * 2u);
}

// The key ranges of one column (sequence, head) merged as fattn_merge_kernel<64> does; the partials' slots are emptied for the
// next layer.  They are refilled only by waves that hold that layer's q, which needs every work-group's part of this layer's
// later products, and this one's come after the clearing stores have arrived.
template <bool F16, int NB> // NB: ranges a lane holds, at least a fourth of all
__device__ __forceinline__ void vs_merge(const vs_args & a, vs_xch & x, uint32_t layer, int column, int lane) {
    constexpr int DU = 16, PH = 4;
    const int b = column / a.hq, head = column - b * a.hq, g = head / a.gqa, c = head - g * a.gqa, bg = b * a.hkv + g;
    const int q = lane / DU, dl = lane % DU;
    vs_kvs kvs;
    vs_addend_load(a, x, layer + a.o_qkv, 0, lane, kvs);
    const float addend = vs_addend<F16>(a, x, layer + a.o_qkv, lane, kvs);
    typedef int int2_v __attribute__((ext_vector_type(2)));
    int4_t rows[NB];
    int2_v ml[NB];
    vs_nap(a.nap_part);
    for (int spin = 0;; ++spin) {
        asm volatile("" ::: "memory");
        int miss = 0;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int s = q + PH * i;
            if (s < a.n_splits) {
                const uint32_t p = vs_part(a, bg, s, c);
                ml[i]   = __builtin_amdgcn_raw_buffer_load_b64(x.r, a.o_ml + p * 8u, 0, VS_DEV);
                rows[i] = x.ld(a.o_part + p * 256u + (uint32_t) dl * 16u);
            } else {
                ml[i]   = int2_v{(int) 0xff800000, 0};
                rows[i] = int4_t{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) miss |= (int) (ml[i][0] == -1) | (int) (ml[i][1] == -1) | vs_miss(rows[i]);
        if (__builtin_amdgcn_ballot_w64(miss != 0) == 0 || x.dead) break;
        if (spin >= VS_SPIN_LIMIT) { x.dead = 1; break; }
    }
    float M = -INFINITY;
#pragma unroll
    for (int i = 0; i < NB; ++i) M = fmaxf(M, __int_as_float(ml[i][0]));
#pragma unroll
    for (int off = DU; off < 64; off <<= 1) M = fmaxf(M, __shfl_xor(M, off, 64));
    const float shift = (M == -INFINITY) ? 0.0f : M;
    float    L   = 0.0f;
    float4_t acc = {0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const float wgt = __builtin_amdgcn_exp2f(__int_as_float(ml[i][0]) - shift);
        L   += __int_as_float(ml[i][1]) * wgt;
        acc += vs_f4(rows[i]) * wgt;
    }
#pragma unroll
    for (int off = DU; off < 64; off <<= 1) {
        L += __shfl_xor(L, off, 64);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] += __shfl_xor(acc[r], off, 64);
    }
    if (q == 0) vs_finish(x, acc, L, true, addend, layer + a.o_attn + (uint32_t) (b * a.hq + head) * 128u + (uint32_t) dl * 8u);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int s = q + PH * i;
        if (s < a.n_splits) {
            const uint32_t p = vs_part(a, bg, s, c);
            x.clear4(a.o_part + p * 256u + (uint32_t) dl * 16u);
            if (dl == 0) x.clear2(a.o_ml + p * 8u);
        }
    }
    vs_wait_vm0();
}

// ---- the phases of a layer.  Each is a function of the arguments, the layer and the lane, and is given both afresh by every
// layer through an opaque copy: what it derives from them stays inside the phase instead of being carried, in more registers
// than there are, around the loop over the layers.
typedef const __attribute__((address_space(4))) vs_args vs_const_args;
__device__ __forceinline__ const vs_args & vs_fresh(vs_const_args * p) {
    asm volatile("" : "+s"(p));
    return *(const vs_args *) p;
}
__device__ __forceinline__ int vs_fresh(int v) {
    asm volatile("" : "+v"(v));
    return v;
}
struct vs_ctx {
    char *   smem;
    uint32_t lds0;
    int      wid, n, vid;
    bool     full;
    vs_xch   x;
};
// Of W waves, wave W - 4 + p loads product p's rows, a layer ahead; the wave that loads the next product's rows (its loads were issued long ago)
// finishes product p.

// column cc < 2 pp of a q / k / v unit: matrix and row; the two rows of a rotated pair sit pp columns apart
__device__ __forceinline__ bool vs_qkv_col(const vs_args & a, int u, int cc, int & mat, int & row, int & pair) {
    const int half = cc >= a.pp ? 1 : 0, p = u * a.pp + cc - half * a.pp;
    const int nq = a.hq * 32, nk = a.hkv * 32;
    pair = p & 31;
    if (p < nq)           { mat = 0; row = (p >> 5) * 64 + pair + 32 * half; }
    else if (p < nq + nk) { mat = 1; row = ((p - nq) >> 5) * 64 + pair + 32 * half; }
    else                  { mat = 2; row = 2 * (p - nq - nk) + half; }
    return p < nq + 2 * nk;
}
// `rows` rows of `bytes` bytes (a multiple of 16) that lie one behind the other in memory into LDS, `slot` bytes apart
__device__ __forceinline__ void vs_rows(const vs_ctx & k, const char * g, int rows, int bytes, int slot, int at, int lane) {
    const int  whole = bytes >> 10, rest = bytes & 1023;
    const bool part = lane * 16 < rest;
    const char * p = g + lane * 16;
    uint32_t     d = k.lds0 + (uint32_t) at;
#pragma unroll 1
    for (int r = 0; r < rows; ++r) {
        uint32_t e = d;
#pragma unroll 1
        for (int w = 0; w < whole; ++w, p += 1024, e += 1024) vs_dma16(p, e);
        if (part) vs_dma16(p, e);
        p += rest;
        d += (uint32_t) slot;
    }
}
// Unit u's rows of product p in layer l, and the norm weights in front of it, into LDS.
__device__ __forceinline__ void vs_fetch(const vs_args & a, const vs_ctx & k, int p, int l, int u, int lane) {
    const vs_layer & Ly = a.L[l];
    const char * const w = Ly.w[p];
    const int slot = a.P[p].slot, cols = a.P[p].cols, img = a.P[p].img, gain = a.P[p].gain, bytes = ((p == VS_D ? a.ffn : a.hidden) >> 5) * VX_Q8_BLOCK;
    if (p == VS_QKV) {
#pragma unroll 1
        for (int cc = 0; cc < cols; ++cc) {
            int mat, row, pair;
            if (!vs_qkv_col(a, u, cc, mat, row, pair)) continue;
            vs_rows(k, (mat == 0 ? w : mat == 1 ? Ly.wk : Ly.wv) + (uint64_t) row * bytes, 1, bytes, slot, img + cc * slot, lane);
        }
    } else {
        const uint64_t off = (uint64_t) u * cols * bytes;
        vs_rows(k, w + off, cols, bytes, slot, img, lane);
        if (p == VS_GU) vs_rows(k, Ly.wu + off, cols, bytes, slot, img + cols * slot, lane);
    }
    if (gain >= 0) vs_rows(k, (const char *) (p == VS_QKV ? Ly.nin : Ly.npost), 1, a.hidden * 4, 0, gain, lane);
}
// the rotation of a q / k / v unit's columns, four token slots per lane (the same in every layer), by one wave
__device__ __forceinline__ void vs_angles(const vs_args & a, const vs_ctx & k, int u, int lane) {
    const int j = lane >> 4, c = lane & 15;
    int mat = 2, row = 0, pair = 0;
    const bool ok = c < 2 * a.pp && vs_qkv_col(a, u, c, mat, row, pair);
    const float ffv = a.ff && ok ? a.ff[pair] : 1.0f;
    float2 * rcs = (float2 *) (k.smem + a.l_rcs);
#pragma unroll 1
    for (int r = 0; r < 4; ++r) {
        float cv = 1.0f, sv = 0.0f;
        if (ok && mat != 2 && 4 * j + r < a.N) rope_cos_sin(a.rp, (float) a.pos[(4 * j + r) % a.T], pair, ffv, cv, sv);
        rcs[r * 64 + lane] = float2{cv, sv};
    }
}

// A product's end, by one wave: the slots' sums in slot order, then what the separate launch has in its epilogue
template <int NWA>
__device__ __forceinline__ void vs_finish_product(const vs_args & a, const vs_ctx & k, int p, int l, int u, int lane, const float (&res)[4]) {
    const int j = lane >> 4, c = lane & 15;
    const bool pair = p == VS_GU, two = pair || p == VS_D || NWA == 16;
    const uint32_t layer = (uint32_t) l * a.layer_bytes, out = layer + (uint32_t) a.P[p].out_at;
    const float4_t * const red = (const float4_t *) (k.smem + a.l_red);
    // ---- the slots' sums in slot order, by one wave
    float4_t part[8], acc, up;
#pragma unroll
    for (int s = 0; s < 8; ++s) part[s] = red[s * 64 + lane];
    acc = part[0];
#pragma unroll
    for (int s = 1; s < 8; ++s) acc += part[s];
    if (two) {
#pragma unroll
        for (int s = 0; s < 8; ++s) part[s] = red[(8 + s) * 64 + lane];
        up = pair ? part[0] : acc + part[0];
#pragma unroll
        for (int s = 1; s < 8; ++s) up += part[s];
        if (!pair) acc = up;
    }
    if (p == VS_QKV) {
        int mat = 2, row = 0, ip = 0;
        const bool ok = c < 2 * a.pp && vs_qkv_col(a, u, c, mat, row, ip);
        const bool lead = c < a.pp;
        const uint32_t to = out + (uint32_t) ((mat == 0 ? 0 : mat == 1 ? a.hq * 64 : (a.hq + a.hkv) * 64) + row) * 4u;
        const float2 * rcs = (const float2 *) (k.smem + a.l_rcs);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float other = __shfl(acc[r], lane + (lead ? a.pp : -a.pp), 64);
            const float2 cs = rcs[r * 64 + lane];
            float y0, y1;
            rope_rotate(lead ? acc[r] : other, lead ? other : acc[r], cs.x, cs.y, y0, y1);
            if (ok && 4 * j + r < a.N) k.x.st(to + (uint32_t) (4 * j + r) * (uint32_t) (a.hq + 2 * a.hkv) * 256u, mat == 2 ? acc[r] : lead ? y0 : y1);
        }
    } else if (p == VS_GU) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float y  = (acc[r] / (1.0f + expf(-acc[r]))) * up[r];
            const float y1 = __shfl(y, lane + 1, 64);
            if (!(c & 1) && c < a.rf && 4 * j + r < a.N)
                k.x.st_h2(out + (uint32_t) (((4 * j + r) * a.ffn + u * a.rf + c) * 2), (_Float16) y, (_Float16) y1);
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (c < a.ro && 4 * j + r < a.N) k.x.st(out + (uint32_t) (((4 * j + r) * a.hidden + u * a.ro + c) * 4), scaled_residual(acc[r], a.res_scale, res[r]));
    }
}

// Product p of layer l: the activations' rows (one wave a row; in front of q / k / v and gate / up normalised in the order of
// RMS_NORM), the products in the order of gemv_dma_kernel's waves, and what the separate launch has in its epilogue.  One body
// for all four, with uniform branches where they differ: four bodies of their own were more code than a compute unit's
// instruction cache holds, and every layer fetched all of it again (28 us a layer instead of 17 for one token).
template <int W, int TPW, int NWA>
__device__ __forceinline__ void vs_product(vs_const_args * ap, vs_ctx & k, int p, int l, int lane0) {
    const int wid = k.wid, end = W - 4 + ((p + 1) & 3), units = vs_fresh(ap).P[p].units;
    if (wid == end) vs_wait_vm0(); // the next product's rows (and its norm weights) are there when this product's barriers are passed
    int4_t v[TPW][8];
#pragma unroll 1
    for (int u = k.vid; u < units; u += k.n) {
        const vs_args & a = vs_fresh(ap);
        const int lane = vs_fresh(lane0), j = lane >> 4, c = lane & 15;
        const vs_prod P = a.P[p];
        const bool norm = p == VS_QKV || p == VS_GU, input = p == VS_QKV && l == 0; // (the stack's input: a plain tensor, nothing to wait for)
        const uint32_t layer = (uint32_t) l * a.layer_bytes, x_at = layer - a.layer_bytes + a.o_x;
        const uint32_t in_at = input ? 0u : layer + (uint32_t) P.in_at;
        const int row_bytes = P.row_bytes, pieces = P.pieces, KP = P.kp;
        const int halves = W * TPW > 8 && p == VS_D ? 2 : 1; // sixteen rows of K = ffn do not fit beside the weights: half of K at a time
        _Float16 * const xs  = (_Float16 *) k.smem;
        float4_t * const red = (float4_t *) (k.smem + a.l_red);
        __amdgpu_buffer_rsrc_t in = k.x.r;
        if (input) in = __builtin_amdgcn_make_buffer_rsrc((void *) a.x, 0, (uint32_t) (a.N * a.hidden * 4), 0x00020000);
        if (!k.full) {
            vs_barrier();
            if (wid == W - 4 + p) { vs_fetch(a, k, p, l, u, lane); vs_wait_vm0(); }
            if (p == VS_QKV && wid == 1) vs_angles(a, k, u, lane);
            vs_barrier();
        }
        if (u == k.vid && wid < a.N) {
            auto load = [&](auto aux) {
#pragma unroll
                for (int i = 0; i < TPW; ++i) {
                    const int t = wid + W * i;
                    const uint32_t off = in_at + (uint32_t) (t * row_bytes + lane * 16);
#pragma unroll
                    for (int cc = 0; cc < 8; ++cc) {
                        v[i][cc] = int4_t{0, 0, 0, 0};
                        if (t < a.N && cc < pieces) v[i][cc] = __builtin_amdgcn_raw_buffer_load_b128(in, off + (uint32_t) cc * 1024u, 0, decltype(aux)::value);
                    }
                }
            };
            asm volatile("" ::: "memory");
            if (input) {
                load(std::integral_constant<int, 0>{});
            } else {
                vs_nap(P.nap);
                asm volatile("" ::: "memory");
                load(std::integral_constant<int, VS_DEV>{});
                for (int spin = 0; !k.x.dead; ++spin) {
                    int miss = 0;
#pragma unroll
                    for (int i = 0; i < TPW; ++i)
#pragma unroll
                        for (int cc = 0; cc < 8; ++cc) miss |= vs_miss(v[i][cc]);
                    if (__builtin_amdgcn_ballot_w64(miss != 0) == 0) break;
                    if (spin >= VS_SPIN_LIMIT) { k.x.dead = 1; break; }
                    asm volatile("" ::: "memory");
                    load(std::integral_constant<int, VS_DEV>{});
                }
            }
            if (norm) {
                float sc[TPW];
                vx_rms_row r[TPW];
#pragma unroll
                for (int i = 0; i < TPW; ++i)
#pragma unroll
                    for (int cc = 0; cc < 8; ++cc) r[i].v[cc] = __builtin_bit_cast(float4, v[i][cc]);
                if constexpr (TPW == 2) vx_rms_row_scale2(r[0], r[1], a.hidden, lane, a.eps, sc[0], sc[1]);
                else                    sc[0] = vx_rms_row_scale(r[0], a.hidden, lane, a.eps);
                const float4_t * gain = (const float4_t *) (k.smem + P.gain);
#pragma unroll
                for (int cc = 0; cc < 8; ++cc) {
                    if (cc >= pieces) break;
                    const float4_t g = gain[lane + 64 * cc];
#pragma unroll
                    for (int i = 0; i < TPW; ++i) {
                        const int t = wid + W * i;
                        if (t >= a.N) continue;
                        float4_t f = vs_f4(v[i][cc]) * sc[i] * g; // RMS_NORM's product, then the MUL node's
                        vs_round32(f);
                        *(half4_t *) (xs + (size_t) t * KP + 4 * (lane + 64 * cc)) = half4_t{(_Float16) f[0], (_Float16) f[1], (_Float16) f[2], (_Float16) f[3]};
                    }
                }
            }
        }
        float res[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if (wid == end && (p == VS_O || p == VS_D)) { // the residual values of this work-group's rows, its own stores: lane (j, c) has tokens 4 j .. 4 j + 3 of column c
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t e = (uint32_t) ((4 * j + r) * a.hidden + u * a.ro + c);
                if (c < a.ro && 4 * j + r < a.N)
                    res[r] = p == VS_O && l == 0 ? a.x[e] : __int_as_float((int) __builtin_amdgcn_raw_buffer_load_b32(k.x.r, (p == VS_O ? x_at : layer + a.o_h) + e * 4u, 0, VS_DEV));
            }
        }
        float4_t acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
#pragma unroll 1
        for (int h = 0; h < halves; ++h) {
            if (!norm && (u == k.vid || halves > 1)) { // f16 rows as they are
                if (h || u != k.vid) vs_barrier();     // (the products of the half before are done)
                const int np = pieces / halves;
#pragma unroll
                for (int i = 0; i < TPW; ++i) {
                    const int t = wid + W * i;
                    if (t >= a.N) continue;
#pragma unroll
                    for (int cc = 0; cc < 8; ++cc) {
                        const int q = cc - h * np;
                        if (q >= 0 && q < np) *(int4_t *) (xs + (size_t) t * KP + 8 * (lane + 64 * q)) = v[i][cc];
                    }
                }
            }
            vs_barrier();
            // slot wid of eight; of two tiles (gate and up); slots wid and wid + 8 of sixteen
            const int tile = W == 16 && p == VS_GU ? wid >> 3 : 0, s0 = wid - 8 * tile; // (sixteen waves: a sum each)
            const uint32_t sd = k.lds0 + (uint32_t) (P.img + tile * P.sfar + min(c, P.cols - 1) * P.slot + (h * P.per * P.nw + s0) * VX_Q8_BLOCK);
            const uint32_t sq = sd + (uint32_t) (8 * j + (wid & 1 ? 2 : 0)), sh = wid & 1 ? 0u : 16u;
            const uint32_t xp = k.lds0 + (uint32_t) (2 * (min(c, a.N - 1) * KP + 8 * j + s0 * 32));
            if constexpr (W == 16) {
                static_assert(W == 8 || NWA == 16, "a wave a slot");
                if (p == VS_GU) vs_sum_of<8>(sd, sq, xp, P.per, sh, acc0);
                else            vs_sum_of<16>(sd, sq, xp, P.per, sh, acc0);
            } else if (NWA == 8 && (p == VS_QKV || p == VS_O)) vs_blocks<8, true>(sd, sq, xp, P.per, 0, 0, sh, acc0, acc1);
            else if (p == VS_GU)                        vs_blocks<8, false>(sd, sq, xp, P.per, (uint32_t) P.sfar, 0, sh, acc0, acc1);
            else                                        vs_blocks<16, false>(sd, sq, xp, P.per, 8 * VX_Q8_BLOCK, 8 * 64, sh, acc0, acc1);
        }
        red[wid * 64 + lane] = acc0;
        if constexpr (W == 8) red[(wid + 8) * 64 + lane] = acc1;
        vs_barrier();
        if (k.full && wid == W - 4 + p && l + 1 < a.n_layer) vs_fetch(vs_fresh(ap), k, p, l + 1, u, vs_fresh(lane0));
        if (wid != end) continue;
        vs_finish_product<NWA>(vs_fresh(ap), k, p, l, u, vs_fresh(lane0), res);
        // The o projection of the next layer reads these values back as its residual, by another wave and without a look: they are in memory
        // before this wave passes a barrier.  (Everybody else waits for the same trip: 550 -> 551.5 us a step of two rows, where looking for
        // the empty slot's pattern at the o projection's end took 567.  What down reads back has been seen by this work-group's gate / up rows.)
        if (p == VS_D) vs_wait_vm0();
    }
}

template <int MODE, int W>
__device__ __forceinline__ void vs_attention(vs_const_args * ap, vs_ctx & k, int l, int lane) {
    const vs_args & a0 = vs_fresh(ap);
    const uint32_t layer = (uint32_t) l * a0.layer_bytes;
    const int n_units = MODE == VS_SELF ? a0.N / a0.T * a0.hkv * a0.n_col_tiles : a0.N * a0.hkv * a0.n_splits;
    constexpr int AW = MODE == VS_F16 ? VD_WAVES : 7;
    if (k.wid < AW) {
#pragma unroll 1
        for (int u = k.vid + k.wid * k.n; u < n_units; u += AW * k.n) {
            const vs_args & a = vs_fresh(ap);
            if constexpr (MODE == VS_SELF) {
                vr_self(a, k.x, layer, u, vs_fresh(lane));
            } else {
                const int bg = u / a.n_splits, sp = u - bg * a.n_splits;
                if constexpr (MODE == VS_F16) vd_range(a, k.x, a.L[l], layer, bg, sp, k.smem + k.wid * VD_WAVE_LDS, vs_fresh(lane));
                else                          vr_range<MODE == VS_F32>(a, k.x, a.L[l], layer, bg, sp, k.smem + k.wid * 512, vs_fresh(lane));
            }
        }
    }
    if constexpr (MODE == VS_F16 || MODE == VS_F32) {
        if (a0.n_splits > 1 && k.wid == W - 1) {
#pragma unroll 1
            for (int m = k.n - 1 - k.vid; m < a0.N * a0.hq; m += k.n) vs_merge<MODE == VS_F16, W == 16 ? 8 : 16>(vs_fresh(ap), k.x, layer, m, vs_fresh(lane));
        }
    }
    vs_barrier();
}

// MODE: which attention; TPW: token rows a wave stages (8 rows in all, or 16); NWA: slots of a sum over K = hidden in q, k, v, o
template <int MODE, int W, int TPW, int NWA>
__global__ __launch_bounds__(64 * W) void stack_kernel(const vs_args) {
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    vs_const_args * const ap = (vs_const_args *) __builtin_amdgcn_kernarg_segment_ptr();
    const int lane = threadIdx.x & 63;
    vs_ctx k;
    k.smem = smem;
    k.lds0 = (uint32_t) (uintptr_t) (vs_lds_char *) smem;
    k.wid  = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    {   // the entrance; the first layer's weights are already on their way for the case that everybody comes
        const vs_args & a = vs_fresh(ap);
        int * const sh = (int *) (smem + a.l_rcs + 4 * 64 * sizeof(float2));
        const int G = (int) gridDim.x, v0 = (int) blockIdx.x;
        k.vid = v0;
        if (k.wid >= W - 4 && v0 < a.P[k.wid - (W - 4)].units) vs_fetch(a, k, k.wid - (W - 4), 0, v0, lane);
        if (threadIdx.x == 0) {
            const uint32_t r = __hip_atomic_fetch_add(a.ctl, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            uint32_t n = 0;
            if (r == 0) {
                const uint64_t t0 = wall_clock64();
                while (__hip_atomic_load(a.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < (uint32_t) G && wall_clock64() - t0 < VS_ENTER_TICKS) {}
                n = __hip_atomic_fetch_or(a.ctl, VS_CLOSED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(a.ctl + 1, n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            } else if (r < (uint32_t) G) { // (the entrance was open)
                for (int spin = 0; n == 0 && spin < VS_SPIN_LIMIT; ++spin) n = __hip_atomic_load(a.ctl + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            sh[0] = (int) min(n, (uint32_t) G);
            sh[1] = (int) r;
        }
        if (k.wid == 1) vs_angles(a, k, v0, lane);
        vs_barrier();
        k.n    = __builtin_amdgcn_readfirstlane(sh[0]);
        k.full = k.n == a.P[VS_O].units; // (one unit a work-group)
        if (!k.full) {
            k.vid = __builtin_amdgcn_readfirstlane(sh[1]);
            vs_wait_vm0(); // (direct loads for another number's rows are still under way into this work-group's LDS)
            if (k.n == 0 || k.vid < 0 || k.vid >= k.n) return; // closed before this one came
            vs_barrier();
        }
        k.x.r    = __builtin_amdgcn_make_buffer_rsrc(a.xch, 0, a.xch_bytes, 0x00020000);
        k.x.dead = 0;
        if (k.wid == W - 4) vs_wait_vm0(); // q / k / v rows and norm weights
        vs_barrier();
    }
    const int n_layer = vs_fresh(ap).n_layer;
#pragma unroll 1
    for (int l = 0; l < n_layer; ++l) {
#pragma unroll 1
        for (int p = 0; p < 4; ++p) {
            if (p == VS_O) vs_attention<MODE, W>(ap, k, l, lane);
            vs_product<W, TPW, NWA>(ap, k, p, l, lane);
        }
    }
    // ---- the final norm: a row each for the first work-groups
    const vs_args & a = vs_fresh(ap);
    if (k.wid == 0) {
        const int nv = a.hidden >> 8;
        const uint32_t x_at = (uint32_t) (n_layer - 1) * a.layer_bytes + a.o_x;
        for (int t = k.vid; t < a.N; t += k.n) {
            int4_t v[8];
            vs_poll(k.x, x_at + (uint32_t) (t * a.hidden * 4 + lane * 16), 1024, nv, true, v);
            vx_rms_row r;
#pragma unroll
            for (int cc = 0; cc < 8; ++cc) r.v[cc] = __builtin_bit_cast(float4, v[cc]);
            const float sc = vx_rms_row_scale(r, a.hidden, lane, a.eps);
#pragma unroll
            for (int cc = 0; cc < 8; ++cc)
                if (cc < nv) ((float4_t *) (a.out + (size_t) t * a.hidden))[lane + 64 * cc] = vs_f4(v[cc]) * sc * ((const float4_t *) a.norm)[lane + 64 * cc];
        }
    }
}

// every slot of the exchange area to the pattern that no result has, the counters to zero
__global__ __launch_bounds__(256) void stack_clear_kernel(int4_t * p, uint32_t n16) {
    for (uint32_t e = blockIdx.x * 256u + threadIdx.x; e < n16; e += gridDim.x * 256u)
        p[e] = e < 16 ? int4_t{0, 0, 0, 0} : int4_t{-1, -1, -1, -1}; // (the first 256 bytes are the counters)
}

int vs_cus() {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) { (void) hipGetLastError(); return 0; }
    return n;
}

size_t align16(size_t v) { return (v + 15) / 16 * 16; }

struct vs_plan {
    int    mode, tpw, halves, nwa, grid;
    size_t ws_bytes, lds;
};

bool al16(const void * p) { return (uintptr_t) p % 16 == 0; }

// Whether the launch takes this stack, and its arguments.  All it needs beyond sizes that fit the LDS is that the separate
// calls would run the kernels whose sums it repeats.
bool vs_fill(const vx_stack * s, vs_args & a, vs_plan & p) {
    const char * off = getenv("VX_STACK"); // read on every call; 0 keeps every stack on the separate calls
    if (off && atoi(off) == 0) return false;
    if (!s || !s->layers || !s->x || !s->out || !s->norm || !s->positions) return false;
    if (s->n_layer < 1 || s->n_layer > VX_STACK_MAX_LAYERS || s->batch < 1 || s->n_tokens < 1 || s->n_past < 0) return false;
    const int64_t N = (int64_t) s->batch * s->n_tokens;
    if (N > 16 || s->head_dim != 64 || s->n_kv_heads < 1 || s->n_heads % s->n_kv_heads || s->n_heads / s->n_kv_heads > 16) return false;
    // (the slots below are those of sums over 1024 values)
    if (s->hidden != 1024 || s->n_heads != 16 || (s->ffn != 2048 && s->ffn != 4096)) return false;
    if (N * s->n_kv_heads > 32) return false;
    const bool decode = s->write_kv != 0;
    if (decode && s->sync_scale != 0.0f) return false; // (vs_addend's order of sums shows in any but a product with zero)
    if (decode ? (s->n_tokens != 1 || s->n_past < 1 || s->mask != nullptr) : s->n_past != 0) return false;
    if (s->kv_type != VX_TYPE_F32 && s->kv_type != VX_TYPE_F16) return false;
    if (!al16(s->x) || !al16(s->out) || !al16(s->norm) || (s->mask && ((uintptr_t) s->mask % 2 || s->mask_nb1 % 2))) return false;
    memset(&a, 0, sizeof(a));
    const int cus = vs_cus();
    int g = cus;
    while (g > 0 && (s->hidden % g || s->ffn % g || (s->ffn / g) % 2)) --g;
    if (g < 16) return false;
    a.n_layer = s->n_layer; a.N = (int) N; a.T = s->n_tokens; a.hidden = s->hidden; a.ffn = s->ffn;
    a.hq = s->n_heads; a.hkv = s->n_kv_heads; a.gqa = a.hq / a.hkv; a.n_past = s->n_past;
    const int n_pairs = (a.hq + 2 * a.hkv) * 32;
    a.pp = (n_pairs + g - 1) / g; a.ro = a.hidden / g; a.rf = a.ffn / g;
    if (2 * a.pp > 16 || a.ro > 16 || a.rf > 16) return false; // (one tile of sixteen columns)
    // the slots that the separate products' sums have
    p.nwa = vx_gemv_waves(a.hidden, N, a.hidden);
    if ((p.nwa != 8 && p.nwa != 16) || vx_gemv_waves(a.hidden, N, a.hkv * 64) != p.nwa) return false;
    if (vx_gemv_waves(a.hidden, N, a.ffn) != 8 || vx_gemv_waves(a.ffn, N, a.hidden) != 16) return false;
    if (N > 8 && p.nwa != 16) return false; // (the instances for more than eight rows have sixteen; VX_GEMV_MANY_TOKENS may ask for eight)
    p.tpw = N > 8 ? 2 : 1;
    p.halves = p.tpw;
    for (int l = 0; l < s->n_layer; ++l) {
        const vx_stack_layer & L = s->layers[l];
        const void * need[] = { L.q_proj, L.k_proj, L.v_proj, L.o_proj, L.gate_proj, L.up_proj, L.down_proj, L.input_norm, L.post_norm };
        for (const void * q : need) if (!q || !al16(q)) return false;
        if (decode && (!L.k_cache || !L.v_cache || !al16(L.k_cache) || !al16(L.v_cache))) return false;
        a.L[l] = vs_layer{ { (const char *) L.q_proj, (const char *) L.o_proj, (const char *) L.gate_proj, (const char *) L.down_proj }, (const char *) L.k_proj,
                           (const char *) L.v_proj, (const char *) L.up_proj, (const float *) L.input_norm, (const float *) L.post_norm, (char *) L.k_cache, (char *) L.v_cache };
    }
    a.x = (const float *) s->x; a.out = (float *) s->out; a.norm = (const float *) s->norm;
    a.pos = s->positions; a.ff = s->rope_factors; a.mask = (const char *) s->mask; a.nbm1 = s->mask_nb1;
    a.eps = s->eps; a.res_scale = s->residual_scale;
    a.rp = rope_make_params(64, 2, s->rope_n_ctx_orig, s->rope_base, s->rope_freq_scale, s->rope_ext_factor, s->rope_attn_factor, s->rope_beta_fast, s->rope_beta_slow);
    a.scale = s->attn_scale * 1.44269504088896341f;
    a.sync_scale = s->sync_scale; a.sync_bias = s->sync_bias;
    a.nbc1 = s->cache_nb1; a.nbc2 = s->cache_nb2; a.nbc3 = s->cache_nb3;
    a.n_splits = 1; a.n_col_tiles = (a.T * a.gqa + 15) / 16;
    if (decode) {
        if (a.nbc1 % 16 || a.nbc2 % 16 || a.nbc3 % 16 || a.nbc1 >= (1u << 28)) return false;
        if (!vx_fattn_stack_plan((int64_t) N * a.hkv, a.n_past + 1, s->kv_type == VX_TYPE_F16, &a.n_splits, &a.chunk) || a.n_splits > 64) return false;
        const bool f32 = s->kv_type == VX_TYPE_F32;
        p.mode = f32 ? VS_F32 : a.n_past + 1 > 64 ? VS_F16 : VS_F16_SHORT;
        // Where the separate calls are the faster ones (us a step of 24 layers, separate / here): with more than eight rows what every
        // work-group stages outweighs the launches -- 16 rows over 6144 keys of an f16 cache 1070 / 1131, over 700 keys 953 / 912, over 40
        // keys 1260 / 890; 9 rows of an F32 cache over 300 keys 853 / 862, 16 over 200 keys 1436 / 1100.  Up to eight rows, an F32 cache
        // (the attention's tiles in registers are seven waves' work here and a whole grid's there) over 300, 2000, 4000 and 8000 keys:
        //   rows 1  675 / 538   712 / 552   763 / 598   826 / 647      5  789 / 688   858 / 832   918 / 879  1032 / 963
        //        2  703 / 583   754 / 641   794 / 683   867 / 741      6  802 / 695   878 / 869   940 / 910  1080 / 1022
        //        4  777 / 621   829 / 718   880 / 768   970 / 840      7  822 / 739   911 / 963   980 / 1023 1157 / 1164
        // seven rows over 1000 keys 849 / 822, over 1400 878 / 873, over 1535 879 / 885; eight over 400 831 / 756, over 1023 874 / 843, over 2000 934 / 949.
        // An f16 cache over 300, 2000 and 8000 keys: one row 717 / 499, 716 / 519, 706 / 549; five 794 / 602, 786 / 723, 847 / 823; eight
        // 800 / 666, 841 / 808, 979 / 936.
        const int most = N > 8 ? (f32 ? 256 : 1024) : !f32 || N < 7 ? 1 << 30 : N == 7 ? 1408 : 1024;
        if (a.n_past + 1 > most || (N > 8 && a.n_splits > 32)) return false;
    } else {
        // (14 rows, a ten-step solve: 1352 / 1280 us; one pass of 16 rows 130 / 133)
        if (!vx_fattn_stack_self(a.T, a.gqa) || N > 14) return false;
        p.mode = VS_SELF;
    }
    // the exchange area: counters, partials, then a part per layer
    const size_t qw = (size_t) (a.hq + 2 * a.hkv) * 256;
    size_t at = 0;
    a.o_qkv = (uint32_t) at;  at += (size_t) N * qw;
    a.o_attn = (uint32_t) at; at += (size_t) N * a.hq * 128;
    a.o_h = (uint32_t) at;    at += (size_t) N * a.hidden * 4;
    a.o_act = (uint32_t) at;  at += (size_t) N * a.ffn * 2;
    a.o_x = (uint32_t) at;    at += (size_t) N * a.hidden * 4;
    a.layer_bytes = (uint32_t) at;
    const size_t layers = at * a.n_layer;
    size_t part = 0, ml = 0;
    if (a.n_splits > 1) { part = (size_t) N * a.hkv * a.n_splits * a.gqa * 256; ml = (size_t) N * a.hkv * a.n_splits * a.gqa * 8; }
    a.o_part = (uint32_t) layers; a.o_ml = (uint32_t) (layers + part);
    a.xch_bytes = (uint32_t) (layers + part + align16(ml));
    p.ws_bytes = 256 + a.xch_bytes;
    p.grid = g;
    // LDS: activations (or the streamed attention's tiles), the slots' sums, angles, norm weights, the four images
    size_t act = (size_t) N * (a.hidden + 8) * 2;
    const size_t actf = (size_t) N * (a.ffn / p.halves + 8) * 2;
    act = act > actf ? act : actf;
    if (p.mode == VS_F16 && act < (size_t) VD_WAVES * VD_WAVE_LDS) act = (size_t) VD_WAVES * VD_WAVE_LDS;
    size_t o = align16(act);
    a.l_red = (int) o;   o += 16 * 64 * sizeof(float4_t);
    a.l_rcs = (int) o;   o += 4 * 64 * sizeof(float2) + 16;
    const int row_h = vx_gemv_dma_slot(a.hidden), row_f = vx_gemv_dma_slot(a.ffn); // (padded: the columns' reads fall into different banks)
    int gain[2];
    for (int & at_ : gain) { at_ = (int) o; o += (size_t) a.hidden * 4; }
    for (int q = 0; q < 4; ++q) {
        vs_prod & P = a.P[q];
        const int K = q == VS_D ? a.ffn : a.hidden, halves = q == VS_D ? p.halves : 1;
        P.in_at  = (int) (q == VS_QKV ? a.o_x - a.layer_bytes : q == VS_O ? a.o_attn : q == VS_GU ? a.o_h : a.o_act); // (q / k / v: the layer before)
        P.out_at = (int) (q == VS_QKV ? a.o_qkv : q == VS_O ? a.o_h : q == VS_GU ? a.o_act : a.o_x);
        P.row_bytes = K * (q == VS_QKV || q == VS_GU ? 4 : 2);
        P.pieces    = P.row_bytes / 1024;
        P.kp        = K / halves + 8;
        P.img  = (int) o;
        P.slot = q == VS_D ? row_f : row_h;
        P.cols = q == VS_QKV ? 2 * a.pp : q == VS_GU ? a.rf : a.ro;
        o += (size_t) P.cols * P.slot * (q == VS_GU ? 2 : 1);
        P.units = q == VS_QKV ? (n_pairs + a.pp - 1) / a.pp : g;
        P.nw    = q == VS_D ? 16 : q == VS_GU ? 8 : p.nwa;
        P.per   = K / 32 / halves / P.nw;
        P.sfar = a.rf * row_h;
        // The first look comes when the values should be there: one that comes too early is answered a round trip later (0.7 us) and another
        // has to follow, and the early ones of 256 work-groups hold up the stores they wait for (a bare exchange of 4 KB: 2.35 us a round
        // looking at once, 1.38 after a pause of 0.25 us).  Measured, steps of 24 layers, without pauses / with these: one token 637 / 524 us,
        // two 688 / 528; every further row takes the finishing wave a little longer.  (o: the attention's end is not known; look at once.)
        const int nap = 22 + 6 * (int) N, most = q == VS_D ? 48 : 40;
        P.nap = q == VS_O ? 0 : nap < most ? nap : most;
        P.gain = q == VS_QKV ? gain[0] : q == VS_GU ? gain[1] : -1;
        if (P.per % (P.nw == 8 && q != VS_GU ? 4 : 2)) return false;
    }
    a.nap_q = decode ? 24 : 8; a.nap_part = 24;
    o += 16; // (the last block's reads go four bytes past it)
    p.lds = o;
    return o <= 160 * 1024;
}

template <int MODE, int W, int TPW, int NWA>
vx_status vs_go(const vs_args & a, const vs_plan & p, hipStream_t st) {
    auto kern = stack_kernel<MODE, W, TPW, NWA>;
    static bool raised = false; // above 64 KiB of LDS a kernel has to be told once that it may be given that much
    if (!raised) {
        VX_HIP(hipFuncSetAttribute((const void *) kern, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised = true;
    }
    vx_launch(kern, dim3((unsigned) p.grid), dim3(64 * W), p.lds, st, a);
    VX_LAUNCH_CHECK();
    return VX_OK;
}
template <int MODE>
vx_status vs_launch(const vs_args & a, const vs_plan & p, hipStream_t st) {
    // Sixteen waves where more than eight rows are to be staged: a row a wave instead of two (solve of 14 rows: 1435 us a ten-step solve
    // with eight waves, 1280 with sixteen).  Not where the attention
    // works on tiles in registers: they need more than a sixteenth of the file.
    constexpr bool eight = MODE == VS_F32 || MODE == VS_F16_SHORT;
    if (a.N > 8) return vs_go<MODE, eight ? 8 : 16, eight ? 2 : 1, 16>(a, p, st);
    return p.nwa == 16 ? vs_go<MODE, 8, 1, 16>(a, p, st) : vs_go<MODE, 8, 1, 8>(a, p, st);
}

} // namespace

extern "C" int vx_supports_stack(const vx_stack * s) {
    vs_args a;
    vs_plan p;
    return vs_fill(s, a, p) ? 1 : 0;
}

extern "C" size_t vx_stack_area_bytes(const vx_stack * s) {
    vs_args a;
    vs_plan p;
    return vs_fill(s, a, p) ? p.ws_bytes : 0;
}

static vx_status vs_refused() {
    return vx_fail(VX_ERR_UNSUPPORTED, "stack: at most 16 token rows; a decode step of one token a sequence, or sequences without a cache; Q8_0 weights on 16-byte boundaries");
}
static vx_status vs_run(vs_args & a, vs_plan & p, void * area, hipStream_t st) {
    a.ctl = (uint32_t *) area;
    a.xch = (char *) area + 256;
    const uint32_t n16 = (uint32_t) (p.ws_bytes / 16);
    const unsigned blocks = (n16 + 255) / 256 < 2048 ? (n16 + 255) / 256 : 2048;
    vx_launch(stack_clear_kernel, dim3(blocks), dim3(256), 0, st, (int4_t *) area, n16);
    VX_LAUNCH_CHECK();
    // fewer work-groups than compute units leave the others to other streams (read on every call; any number gives the same bits)
    if (const char * e = getenv("VX_STACK_GROUPS")) { const int n = atoi(e); if (n >= 1 && n < p.grid) p.grid = n; }
    switch (p.mode) {
        case VS_F16:       return vs_launch<VS_F16>(a, p, st);
        case VS_F32:       return vs_launch<VS_F32>(a, p, st);
        case VS_F16_SHORT: return vs_launch<VS_F16_SHORT>(a, p, st);
        default:           return vs_launch<VS_SELF>(a, p, st);
    }
}

extern "C" vx_status vx_stack_run(const vx_stack * s, vx_stream stream) {
    vs_args a;
    vs_plan p;
    if (!vs_fill(s, a, p)) return vs_refused();
    void * ws = nullptr;
    const vx_status rc = vx_workspace((hipStream_t) stream, p.ws_bytes, &ws, true);
    return rc != VX_OK ? rc : vs_run(a, p, ws, (hipStream_t) stream);
}

extern "C" vx_status vx_stack_run_in(const vx_stack * s, void * area, size_t bytes, vx_stream stream) {
    vs_args a;
    vs_plan p;
    if (!vs_fill(s, a, p)) return vs_refused();
    if (!area || !al16(area) || bytes < p.ws_bytes)
        return vx_fail(VX_ERR_INVALID, "stack: the area must be %zu bytes on a 16-byte boundary", p.ws_bytes);
    return vs_run(a, p, area, (hipStream_t) stream);
}
