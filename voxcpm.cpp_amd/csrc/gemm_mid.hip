// gemm_mid.hip -- MUL_MAT for some tens to a few thousand tokens (a prompt, concurrent LocDiT requests): Q8_0 / F16 weights.
//
// What bounds these products is neither the matrix cores nor HBM (a 203-token layer is 6 GFLOP and 16 MB of weights) but
// what each of the chip's 256 compute units has to bring in and issue for its small tile, and the time until its first
// bytes arrive.  Hence:
//   * the activations are rounded to f16 once, by a pass of their own that also applies a fused norm and fills the
//     rotation's angle table (gm_acts_kernel), and laid out as 1 KB operand tiles: a work-group brings in half the bytes
//     and converts nothing;
//   * weights come as raw Q8_0 rows (1.06 bytes a weight), both by direct loads into LDS issued by two waves that do
//     nothing else -- with every wave loading and multiplying, two fifths of a step's 218 instructions were address,
//     branch and M0 bookkeeping in front of the products (64 x 64 tile: 0.54 us per 128 of K, 0.36 now);
//   * four waves of a row group share the k blocks (block kb: group kb mod 4), so that small tiles keep a compute unit's
//     four SIMDs busy; their sums are added in group order at the end -- the order of the streaming kernel's four waves
//     (mul_mat.hip), whose products of more than 16 tokens come out with the same bits here;
//   * a step's products are interleaved with their scaled additions and with the next step's conversion: a SIMD issues one
//     vector instruction every four cycles, so an exactly scaled 16 x 16 x 32 product costs its own slot and four
//     additions, 20 cycles against the matrix core's 16, plus the conversions -- 7 slots in all at two row tiles x eight
//     token tiles a wave.
// Under the tracer, microseconds a launch in a stack of 24 layers (the activation pass, which the norm's launch was before, is
// 3.4 to 4.8 of its own): 45 tokens: norm + q / k / v + rope 6.6, gate/up pair 7.6, o and down 7.5 on average; 1024 tokens: 12, 39, o
// 10, down 23.  Whole prompts against the streaming / LDS-tiled kernels of mul_mat.hip and the launches around them: 45 tokens
// 1729 -> 1108 us, 203 2329 -> 1579, 2 x 512 4408 -> 2850.  Counters of the pair at 1024 tokens: 10.4 vector instructions a matrix
// instruction, epilogue and GLU included; they issue in half of the SIMDs' cycles and the matrix cores are busy in a fifth.
#include "gemm_mid.hpp"
#include "kvs_common.hpp"
#include "mm_common.hpp"

#include <cstdlib>
#include <type_traits>

namespace {

struct gm_args {
    vx_gm_mat     mat[3];
    int           nmat;
    const char *  w2;
    const half8_t * xt;            // [batch][k block][n_tt][64] operand tiles
    int           n_tt, n_kb;
    int           N, ne12;
    const half8_t * wt;            // gd_kernel: the weights as operand tiles [k block][n_rt][64] ...
    const float * wdt;             // ... and their scales, per 64 rows [16][4]
    int           n_rt;            // 16-row tiles (of a pair's alternating ones)
    int           xr;              // log2 of the XCDs that share out the row tiles (the others share out the token tiles)
    const char *  res;
    uint64_t      rnb1, rnb2, rnb3;
    float         res_scale;
    _Float16 *    tile_out;
    int           out_tt;
    const float2 * rope_tab;       // [token][32] cos, sin
};

// N consecutive 1 KB tiles from global memory (uniform base + lane offset) into LDS at lds + 16 lane: one statement, since the
// compiler may write M0 between two
template <int N> __device__ __forceinline__ void gm_dma_tiles(uint32_t off, const char * base, uint32_t lds) {
    static_assert(N >= 1 && N <= 4, "one statement's loads");
    if constexpr (N == 1)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds) : "memory");
    else if constexpr (N == 2)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024" ::"v"(off), "s"(base), "s"(lds)
                     : "memory");
    else if constexpr (N == 3)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                     "global_load_lds_dwordx4 %0, %1 offset:2048" ::"v"(off), "s"(base), "s"(lds) : "memory");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1\n\tglobal_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                     "global_load_lds_dwordx4 %0, %1 offset:2048\n\tglobal_load_lds_dwordx4 %0, %1 offset:3072" ::"v"(off), "s"(base), "s"(lds) : "memory");
}

template <int N> __device__ __forceinline__ void gm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory"); }

// a stage of L loads has landed once only those of the stages behind it, at most MOST of them, are outstanding
template <int L, int MOST> __device__ __forceinline__ void gm_wait_younger(int younger) {
    if constexpr (MOST > 0) {
        if (younger < MOST) { gm_wait_younger<L, MOST - 1>(younger); return; }
    }
    gm_wait<L * MOST>();
}

constexpr int KG = GM_KG;

template <int WT, int MT, int NT, int RW, int CH, int S, int EPI>
__global__ __launch_bounds__(64 * (KG * RW + 2)) void gm_kernel(const gm_args a) {
    using sh = gm_shape<WT, MT, NT, RW, CH, S>;
    static_assert((CH == 1 || CH == 2) && 4 * CH % KG == 0, "stages of 128 or 256 k, whole steps");
    static_assert(EPI == GM_PLAIN || MT == 2, "pairs of row tiles inside a wave");
    extern __shared__ __align__(1024) char gm_smem[];
    typedef __attribute__((address_space(3))) char lds_char;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    const int j = lane >> 4, c = lane & 15;
    const int g = wid % KG, rw = wid / KG; // k group (block kb belongs to group kb mod KG), row group

    // (work-groups are dealt to the eight XCDs in turn, the grid's width is a multiple of 8)
    const int xcd = blockIdx.x & 7;
    int mi = 0, tx = (((int) blockIdx.x >> 3) << a.xr) + (xcd & ((1 << a.xr) - 1));
    const int ty = ((int) blockIdx.y << (3 - a.xr)) + (xcd >> a.xr);
    if constexpr (EPI == GM_SEGS) {
        if (a.nmat > 1 && tx >= a.mat[1].wg0) mi = 1;
        if (a.nmat > 2 && tx >= a.mat[2].wg0) mi = 2;
        tx -= a.mat[mi].wg0;
    }
    const vx_gm_mat & mt = a.mat[mi];
    const int M = mt.M;
    if (tx * sh::ROWS >= (EPI == GM_SWIGLU ? 2 * M : M) || ty * sh::TOKS >= a.N) return; // padding of the grid
    const int tt0 = ty * NT;
    const int batch = blockIdx.z;
    const int nst = a.n_kb / (4 * CH);

    // first row of local row tile lt (wave row rw holds lt = rw * MT + m)
    auto row_of = [&](int lt) {
        if constexpr (EPI == GM_SWIGLU) return tx * (sh::ROWS / 2) + 16 * (lt >> 1);      // even tiles W, odd tiles the same rows of W2
        if constexpr (EPI == GM_SEGS) { // 32 rows a wave: (d .. d + 15, d + 32 .. d + 47) of one head
            const int q = tx * RW + lt / MT;
            return (q >> 1) * 64 + 16 * (q & 1) + 32 * (lt % MT);
        }
        return tx * sh::ROWS + 16 * lt;
    };

    const uint32_t smem0 = (uint32_t) (uintptr_t) (lds_char *) gm_smem;
    float4_t acc[MT][NT];
    if (wid >= sh::NC) {
        // ---- the two waves that fill the stages.  Stage st is announced by barrier st; the stage that takes its buffer
        // again is requested after barrier st + 1, when every compute wave holds stage st's operands in registers.
        if (wid == sh::NC) {
            const char * wptr[sh::WINST];
#pragma unroll
            for (int i = 0; i < sh::WINST; ++i) {
                const int P = i * 64 + lane, row = min(P / sh::PIECES, sh::ROWS - 1); // (the last load's spare lanes: into the stage's padding)
                int piece = P % sh::PIECES;
                const int lt = row >> 4, cc = row & 15;
                if constexpr (WT == VX_GM_F16) piece ^= cc; // the sixteen rows' pieces over the banks
                const char * wsel = EPI == GM_SWIGLU && (lt & 1) ? a.w2 : mt.w;
                wptr[i] = wsel + (uint64_t) (uint32_t) min(row_of(lt) + cc, M - 1) * mt.nb01 + piece * 16;
            }
            auto issue = [&](int st, int buf) {
                const uint32_t base = smem0 + (uint32_t) buf * sh::STAGE;
                const int woff = WT == VX_GM_F16 ? 256 * CH * st : CH == 2 ? 272 * st : 136 * st - 8 * (st & 1);
#pragma unroll
                for (int i = 0; i < sh::WINST; ++i)
                    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(wptr[i] + woff), "s"(base + (uint32_t) i * 1024) : "memory");
            };
            constexpr int L = sh::WINST;
            static_assert(L * (S - 2) <= 63, "loads in flight are counted in six bits");
#pragma unroll
            for (int s = 0; s < S; ++s) if (s < nst) issue(s, s);
            int buf = S - 1; // where the stage before last lies (st = 0: unused)
            for (int st = 0; st < nst; ++st) {
                gm_wait_younger<L, S - 2>(nst - 1 - st);
                __builtin_amdgcn_s_barrier();
                if (st > 0 && st - 1 + S < nst) issue(st - 1 + S, buf);
                buf = buf + 1 == S ? 0 : buf + 1;
            }
        } else {
            const char * xsrc = (const char *) (a.xt + ((int64_t) batch * a.n_kb * a.n_tt + tt0) * 64);
            const uint32_t loff = (uint32_t) lane * 16;
            auto issue = [&](int st, int buf) {
                const uint32_t base = smem0 + (uint32_t) buf * sh::STAGE + sh::WBYTES;
#pragma unroll
                for (int kb = 0; kb < 4 * CH; ++kb) { // NT consecutive tiles of a k block (past the last token tile: the next block's, dropped at the store)
                    const char * p = xsrc + (int64_t) (st * 4 * CH + kb) * a.n_tt * 1024;
#pragma unroll
                    for (int t0 = 0; t0 + 4 <= NT; t0 += 4) gm_dma_tiles<4>(loff, p + t0 * 1024, base + (uint32_t) (kb * NT + t0) * 1024);
                    constexpr int rest = NT & 3;
                    if constexpr (rest) gm_dma_tiles<rest>(loff, p + (NT - rest) * 1024, base + (uint32_t) (kb * NT + NT - rest) * 1024);
                }
            };
            constexpr int L = sh::XINST;
            static_assert(L * (S - 2) <= 63, "loads in flight are counted in six bits");
#pragma unroll
            for (int s = 0; s < S; ++s) if (s < nst) issue(s, s);
            int buf = S - 1;
            for (int st = 0; st < nst; ++st) {
                gm_wait_younger<L, S - 2>(nst - 1 - st);
                __builtin_amdgcn_s_barrier();
                if (st > 0 && st - 1 + S < nst) issue(st - 1 + S, buf);
                buf = buf + 1 == S ? 0 : buf + 1;
            }
        }
    } else {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[m][n] = float4_t{0, 0, 0, 0};
        // this lane's operand addresses inside a stage: its row of row tile 0, its slot of token tile 0
        const uint32_t wl = (uint32_t) ((rw * MT * 16 + c) * sh::PITCH + (WT == VX_GM_Q8 ? VX_Q8_BLOCK * g : 0));
        const uint32_t xl = (uint32_t) (sh::WBYTES + g * NT * 1024 + lane * 16);
        const uint32_t sh16 = g & 1 ? 0u : 16u;                       // an even block's quants sit 2 bytes into their dwords
        const uint32_t qoff = 8u * (uint32_t) j + (g & 1 ? 2u : 0u);
        typedef const __attribute__((address_space(3))) uint32_t lds_u32;
        typedef const __attribute__((address_space(3))) half8_t  lds_half8;
        // The operands of a step are in registers before it begins: the weights' as f16 (bop, with the block scales d), the
        // activations' (x).  While it is multiplied the next step's bytes are read, x[n] as soon as its last product has
        // been issued, and the weights' are turned into f16 between the second half of the products.
        struct wops { half8_t bop[MT]; float d[MT]; } A, B;
        half8_t  x[NT];
        uint32_t wq[MT][3]; _Float16 wd[MT];
        auto read_w = [&](wops & o, int st, int sp, int buf) {
            const lds_char * base = (const lds_char *) gm_smem + buf * sh::STAGE;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if constexpr (WT == VX_GM_Q8) {
                    const lds_char * p = base + wl + (CH == 1 ? 8 * (st & 1) : 0) + sp * (KG * VX_Q8_BLOCK) + m * 16 * sh::PITCH;
                    lds_u32 * qp = (lds_u32 *) (p + qoff);
                    wq[m][0] = qp[0]; wq[m][1] = qp[1]; wq[m][2] = qp[2];
                    wd[m] = *(const __attribute__((address_space(3))) _Float16 *) p;
                } else {
                    const uint32_t piece = (uint32_t) (4 * (KG * sp + g) + j) ^ (uint32_t) c;
                    o.bop[m] = *(lds_half8 *) (base + (rw * MT * 16 + m * 16 + c) * sh::PITCH + piece * 16);
                }
            }
        };
        auto convert = [&](wops & o, int m) {
            o.bop[m] = q8_to_half8(__builtin_amdgcn_alignbit(wq[m][1], wq[m][0], sh16), __builtin_amdgcn_alignbit(wq[m][2], wq[m][1], sh16));
            o.d[m] = (float) wd[m];
            asm volatile("" : "+v"(o.d[m]));
        };
        auto read_x = [&](int n, int sp, int buf) { x[n] = *(lds_half8 *) ((const lds_char *) gm_smem + buf * sh::STAGE + xl + (sp * KG * NT + n) * 1024); };
        auto step = [&](auto MORE, const wops & o, wops & nx, int st1, int sp1, int buf1) {
            constexpr bool more = decltype(MORE)::value;
            if constexpr (more) read_w(nx, st1, sp1, buf1);
            constexpr int T = MT * NT, LAG = T < 2 ? T : 2; // the scaled additions of a product follow the MFMA LAG further on
            float4_t blk[LAG];
#pragma unroll
            for (int i = 0; i < T + (WT == VX_GM_Q8 ? LAG : 0); ++i) {
                if constexpr (WT == VX_GM_Q8) {
                    if (i >= LAG) {
                        const int q = i - LAG;
#pragma unroll
                        for (int r = 0; r < 4; ++r) acc[q % MT][q / MT][r] = __builtin_fmaf(blk[q % LAG][r], o.d[q % MT], acc[q % MT][q / MT][r]);
                    }
                    if (i < T) blk[i % LAG] = mfma16(x[i / MT], o.bop[i % MT], float4_t{0, 0, 0, 0});
                } else if (i < T) {
                    acc[i % MT][i / MT] = mfma16(x[i / MT], o.bop[i % MT], acc[i % MT][i / MT]);
                }
                if constexpr (more) {
                    if (i < T && i % MT == MT - 1) read_x(i / MT, sp1, buf1);
                    if constexpr (WT == VX_GM_Q8) {
                        constexpr int H = T / 2, E = (T - H) / MT > 0 ? (T - H) / MT : 1; // convert tile m behind product H + E m
                        if constexpr (T >= 2 * MT) { if (i >= H && (i - H) % E == 0 && (i - H) / E < MT) convert(nx, (i - H) / E); }
                        else if (i == T - 1) { _Pragma("unroll") for (int m = 0; m < MT; ++m) convert(nx, m); }
                    }
                }
            }
        };
        auto barrier = [&]() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
        barrier();
        read_w(A, 0, 0, 0);
#pragma unroll
        for (int n = 0; n < NT; ++n) read_x(n, 0, 0);
        if constexpr (WT == VX_GM_Q8) {
#pragma unroll
            for (int m = 0; m < MT; ++m) convert(A, m);
        }
        int buf = 0;
        using more = std::true_type;
        using last = std::false_type;
        auto advance = [&]() { buf = buf + 1 == S ? 0 : buf + 1; barrier(); };
        // (two steps a turn and no branch inside a turn: across one the compiler would sink a step's additions)
        if constexpr (sh::STEPS == 1) {
            for (int st = 0; st + 2 < nst; st += 2) {
                advance();
                step(more{}, A, B, st + 1, 0, buf);
                advance();
                step(more{}, B, A, st + 2, 0, buf);
            }
            advance();
            step(more{}, A, B, nst - 1, 0, buf);
        } else {
            for (int st = 0; st + 1 < nst; ++st) {
                step(more{}, A, B, st, 1, buf);
                advance();
                step(more{}, B, A, st + 1, 0, buf);
            }
            step(more{}, A, B, nst - 1, 1, buf);
        }
        step(last{}, B, A, 0, 0, 0);
    }

    // ---- the k groups' sums, in group order; wave (rw, g) finishes token tiles n = g mod 4 of its row group
    const int  i12 = batch % a.ne12, i13 = batch / a.ne12;
    float4_t * red = (float4_t *) gm_smem; // [group][row group][m][n - 4 p][lane]
#pragma unroll
    for (int p = 0; p < (NT + 3) / 4; ++p) {
        constexpr int NP = sh::NP;
        __syncthreads();
        if (wid < sh::NC) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int n = 0; n < NP; ++n)
                    if (4 * p + n < NT) red[(((g * RW + rw) * MT + m) * NP + n) * 64 + lane] = acc[m][4 * p + n];
        }
        __syncthreads();
        const int n = g;
        if (wid >= sh::NC || n >= NP || 4 * p + n >= NT) continue; // (uniform; nothing below synchronises)
        const int tok0 = 16 * (tt0 + 4 * p + n);
        if (tok0 >= a.N) continue;
        float4_t v[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            v[m] = red[((rw * MT + m) * NP + n) * 64 + lane];
#pragma unroll
            for (int gg = 1; gg < KG; ++gg) v[m] += red[(((gg * RW + rw) * MT + m) * NP + n) * 64 + lane];
        }
        char * db = mt.dst + (uint64_t) i12 * mt.nb2 + (uint64_t) i13 * mt.nb3;
        if constexpr (EPI == GM_SWIGLU) {
#pragma unroll
            for (int m = 0; m < MT; m += 2) {
                const int row = row_of(rw * MT + m) + c;
                if (row >= M) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int   tok = tok0 + 4 * j + r;
                    const float gt = v[m][r], u = v[m + 1][r];
                    float h = (gt / (1.0f + expf(-gt))) * u;
                    if (a.tile_out) { // (uniform) rounded to f16 as the next product's activation pass would round it; whole tiles are written
                        asm volatile("" : "+v"(h)); // the fp32 value the GLU node holds, formed as such
                        const uint64_t tile = ((uint64_t) batch * (uint32_t) (M >> 5) + (uint32_t) (row >> 5)) * (uint32_t) a.out_tt + (uint32_t) (tok >> 4);
                        a.tile_out[(tile * 64 + ((row >> 3) & 3) * 16 + (tok & 15)) * 8 + (row & 7)] = (_Float16) h;
                    } else if (tok < a.N) {
                        *(float *) (db + (uint64_t) tok * mt.nb1 + (uint64_t) row * 4) = h;
                    }
                }
            }
        } else {
            if constexpr (EPI == GM_SEGS) {
                if (mt.rope) { // (uniform) tile m holds d = row mod 64 < 32, tile m + MT / 2 the partners d + 32
#pragma unroll
                    for (int m = 0; m < MT / 2; ++m) {
                        const int d = (row_of(rw * MT + m) + c) & 31;
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int    tok = min(tok0 + 4 * j + r, a.N - 1);
                            const float2 cs = a.rope_tab[tok * 32 + d];
                            float y0, y1;
                            rope_rotate(v[m][r], v[m + MT / 2][r], cs.x, cs.y, y0, y1);
                            v[m][r] = y0; v[m + MT / 2][r] = y1;
                        }
                    }
                }
            }
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int row = row_of(rw * MT + m) + c;
                if (row >= M) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int tok = tok0 + 4 * j + r;
                    if (tok >= a.N) continue;
                    float val = v[m][r];
                    if (EPI == GM_PLAIN && a.res)
                        val = scaled_residual(val, a.res_scale, *(const float *) (a.res + (uint64_t) i12 * a.rnb2 + (uint64_t) i13 * a.rnb3 + (uint64_t) tok * a.rnb1 + (uint64_t) row * 4));
                    *(float *) (db + (uint64_t) tok * mt.nb1 + (uint64_t) row * 4) = val;
                }
            }
        }
    }
}

// ---- the same product from weights that are laid out already ----------------------------------------------------------
// Pinned Q8_0 weights may be at hand as f16 operand tiles (vx_qt_kept_tiles).  Then a compute wave has nothing to convert, which
// is two of gm_kernel's seven vector slots a product, and owns 64 rows by itself: it fetches their tiles from memory straight into
// the operand registers, four k blocks ahead, so that only the activations (which its three neighbours need as well) and the scales
// pass through LDS, in stages of two k blocks with one barrier a stage.  What bounds it is the matrix core and the four scaled
// additions of every product, which a SIMD overlaps only in part (25 cycles measured for the five, 16.5 and 9 for the two sides alone);
// two work-groups a compute unit.  In a layer of 1024 tokens the pair of 4096 rows takes 28 us, 42.5 on gm_kernel; 24 layers 2769 -> 2481.
// The k blocks are walked group by group (0, 4, 8 ..., then 1, 5, ...) and a group's sum is added to the total before the next
// begins: gm_kernel's order of every sum, so which of the two runs does not show in the result.
constexpr int GD_ST = 3;
constexpr int GD_BLOCK = GD_CT * 1024, GD_STAGE = 2 * GD_BLOCK + 4 * 1024; // two blocks of token tiles, 1 KB of scales per wave (512 bytes of it read)
constexpr int GD_LDS = GD_ST * GD_STAGE;

template <int EPI>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gd_kernel(const gm_args a) {
    extern __shared__ __align__(1024) char gm_smem[];
    typedef __attribute__((address_space(3))) char lds_char;
    typedef const __attribute__((address_space(3))) half8_t  lds_half8;
    typedef const __attribute__((address_space(3))) float4_t lds_float4;
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    const int j = lane >> 4, c = lane & 15;
    const int xcd = blockIdx.x & 7;
    const int tx = (((int) blockIdx.x >> 3) << a.xr) + (xcd & ((1 << a.xr) - 1)), ty = ((int) blockIdx.y << (3 - a.xr)) + (xcd >> a.xr);
    if (tx * (GD_ROWS / 16) >= a.n_rt || ty * GD_TOKS >= a.N) return; // padding of the grid
    const int batch = blockIdx.z, nkb = a.n_kb;
    const int rtw = tx * (GD_ROWS / 16) + 4 * wid, tt0 = ty * GD_CT; // the wave's first row tile, the work-group's first token tile
    const int n_rt4 = (a.n_rt + 3) & ~3;
    const uint32_t smem0 = (uint32_t) (uintptr_t) (lds_char *) gm_smem, loff = (uint32_t) lane * 16;

    // The k blocks in the order of the sums: in steps of four, from a group's last block to the next group's first (behind the last
    // group blocks 4 and 8 again: one stage, requested for nothing).
    const int n4 = nkb / 4;
    // ---- a stage: wave w brings token tiles 2 (w mod 2), + 1 of block w / 2, and its own rows' scales of both blocks
    // (past the last token tile: that one again, dropped at the store)
    const int64_t xstr = (int64_t) a.n_tt * 1024;
    const char * xsrc = (const char *) a.xt + ((int64_t) batch * nkb + (wid < 2 ? 0 : 4)) * xstr;
    const uint32_t xo0 = (uint32_t) min(tt0 + 2 * (wid & 1), a.n_tt - 1) * 1024 + loff, xo1 = (uint32_t) min(tt0 + 2 * (wid & 1) + 1, a.n_tt - 1) * 1024 + loff;
    const char * dsrc = (const char *) (a.wdt + min(rtw, n_rt4 - 4) * 16);
    const int64_t dstr = (int64_t) n_rt4 * 64;
    const uint32_t doff = (uint32_t) (lane & 16 ? 4 * dstr : 0) + (uint32_t) c * 16; // (lanes 32 on: the same again)
    const uint32_t sdst = smem0 + (uint32_t) ((wid >> 1) * GD_BLOCK + 2 * (wid & 1) * 1024);
    int sleft = n4 / 2; // stages of the group that are still to be requested
    uint32_t ibuf = 0;
    auto request = [&](int i) {
        if (i < 2) {
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(i ? xo1 : xo0), "s"(xsrc), "s"(sdst + ibuf + i * 1024) : "memory");
        } else {
            asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(doff), "s"(dsrc), "s"(smem0 + ibuf + 2 * GD_BLOCK + wid * 1024) : "memory");
            const int64_t step = --sleft ? 8 : 9 - nkb;
            sleft = sleft ? sleft : n4 / 2;
            xsrc += step * xstr;
            dsrc += step * dstr;
            ibuf = ibuf + GD_STAGE == GD_ST * GD_STAGE ? 0 : ibuf + GD_STAGE;
        }
    };
    // ---- the wave's weights: four row tiles a block
    // (buffer loads: a base that stays, one 32-bit offset a lane and row tile, one scalar that walks the blocks; gd_takes keeps the
    // matrix below 4 GiB)
    const auto wrsrc = __builtin_amdgcn_make_buffer_rsrc((void *) a.wt, (short) 0, (int) ((uint32_t) nkb * (uint32_t) a.n_rt * 1024u), 0x00027000);
    const uint32_t wstr = (uint32_t) a.n_rt * 1024u, wstep = 4 * wstr, wback = (uint32_t) (5 - nkb) * wstr;
    uint32_t wsoff = 0;
    int wleft = n4;
    uint32_t woff[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) woff[rt] = (uint32_t) min(rtw + rt, a.n_rt - 1) * 1024 + loff;
    half8_t b[4][4], x[GD_CT];
    float4_t d[2];
    auto fetch = [&](int set, int rt) {
        b[set][rt] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, (int) woff[rt], (int) wsoff, 0));
        if (rt == 3) {
            wsoff += --wleft ? wstep : wback;
            wleft = wleft ? wleft : n4;
        }
    };
    float4_t acc[4][GD_CT], tot[4][GD_CT];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int tt = 0; tt < GD_CT; ++tt) { acc[rt][tt] = float4_t{0, 0, 0, 0}; tot[rt][tt] = float4_t{-0.0f, -0.0f, -0.0f, -0.0f}; } // (-0 + s is s)
    auto stage_wait = [&](auto NC) { asm volatile("s_waitcnt vmcnt(%0)" ::"i"(decltype(NC)::value) : "memory"); };
    auto barrier = [&]() { __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); };
#pragma unroll
    for (int i = 0; i < 4; ++i) fetch(0, i);
#pragma unroll
    for (int i = 0; i < 6; ++i) request(i % 3);
#pragma unroll
    for (int i = 4; i < 16; ++i) fetch(i >> 2, i & 3);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 3; ++i) request(i);
    stage_wait(std::integral_constant<int, 18>{}); // younger than stage 0: stages 1 and 2, the weight tiles of three blocks
    barrier();
    uint32_t rbuf = 0;
#pragma unroll
    for (int n = 0; n < GD_CT; ++n) x[n] = *(lds_half8 *) ((const lds_char *) gm_smem + n * 1024 + loff);
    const uint32_t dof = 2 * GD_BLOCK + wid * 1024 + c * 16;
    d[0] = *(lds_float4 *) ((const lds_char *) gm_smem + dof);
    __builtin_amdgcn_sched_barrier(0);

    // A block: its operands (set P of the weights and scales, the tokens) are in registers; row by row its products are issued, their
    // scaled additions two products behind, and what the row leaves free takes the next blocks' bytes.  The last turn's four blocks
    // (ENDING) bring in nothing: every weight they need is in registers or on its way there, the last stage is requested.
    auto block = [&](auto SET, auto ENDING) {
        constexpr int Q = decltype(SET)::value, P = Q & 1, T = 4 * GD_CT, LAG = 2;
        constexpr bool ending = decltype(ENDING)::value, more = !(ending && Q == 3);
        const uint32_t nbuf = rbuf + GD_STAGE == GD_ST * GD_STAGE ? 0 : rbuf + GD_STAGE;
        const lds_char * nx = (const lds_char *) gm_smem + (P ? nbuf : rbuf + GD_BLOCK) + loff;
        const lds_char * nd = (const lds_char *) gm_smem + (P ? nbuf : rbuf + 256) + dof;
        float4_t blk[LAG + 1];
#pragma unroll
        for (int i = 0; i < T + LAG; ++i) {
            const int rt = i / GD_CT, n = i % GD_CT;
            if (i < T) {
                blk[i % (LAG + 1)] = mfma16(x[n], b[Q][rt], float4_t{0, 0, 0, 0});
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (more) {
                    if (P == 1 && i == GD_CT - 1) {
                        // The next stage has landed once at most these are outstanding: younger than stage 1 are 19 loads, than stage 2 the
                        // 15 of blocks 0 to 2, later 16.  In the last turn 12: behind the last stage's third load the turn before fetched nine
                        // tiles and requested three loads (with 8 allowed, four of the nine may go or move).  Behind the barrier every wave has
                        // this stage's operands in registers: its buffer takes the stage after next.
                        stage_wait(std::integral_constant<int, ending ? 8 : 15>{});
                        barrier();
                    }
                    if (!ending && P == 1 && i > GD_CT && i % GD_CT == 1) request(rt - 1);
                    if (rt == 3) x[n] = *(lds_half8 *) (nx + n * 1024);
                    if (rt == 2 && n == GD_CT - 1) d[1 - P] = *(lds_float4 *) nd;
                    if (!ending && n == GD_CT - 1) fetch(Q, rt);
                }
            }
            if (i >= LAG) {
                const int p = i - LAG;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[p / GD_CT][p % GD_CT][r] = __builtin_fmaf(blk[p % (LAG + 1)][r], d[P][p / GD_CT], acc[p / GD_CT][p % GD_CT][r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (P) rbuf = nbuf;
    };
    auto add_group = [&]() {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int n = 0; n < GD_CT; ++n) {
#pragma unroll
                for (int r = 0; r < 4; ++r) { tot[rt][n][r] += acc[rt][n][r]; acc[rt][n][r] = 0.0f; }
                asm volatile("" : "+v"(tot[rt][n]), "+v"(acc[rt][n]));
            }
    };
    using set0 = std::integral_constant<int, 0>;
    using set1 = std::integral_constant<int, 1>;
    using set2 = std::integral_constant<int, 2>;
    using set3 = std::integral_constant<int, 3>;
    auto four = [&](auto ENDING) { block(set0{}, ENDING); block(set1{}, ENDING); block(set2{}, ENDING); block(set3{}, ENDING); };
    const int turns = nkb / 16; // of a group
    for (int g = 0; g < 3; ++g) {
        for (int s = 0; s < turns; ++s) four(std::false_type{});
        add_group();
    }
    for (int s = 0; s < turns - 1; ++s) four(std::false_type{});
    four(std::true_type{});
    add_group();
    stage_wait(std::integral_constant<int, 0>{}); // (stages requested past the end have landed before the work-group's LDS is given back or used again)

    // lane (j, c), tile (rt, n), register r: token 16 (tt0 + n) + 4 j + r, virtual row 16 (rtw + rt) + c
    const int i12 = batch % a.ne12, i13 = batch / a.ne12;
    const vx_gm_mat & mt = a.mat[0];
    const int M = mt.M;
    char * db = mt.dst + (uint64_t) i12 * mt.nb2 + (uint64_t) i13 * mt.nb3;
    if constexpr (EPI == GM_SWIGLU) {
        const int row0 = 8 * rtw; // the wave's 32 rows
        if (a.tile_out) { // (uniform) rounded to f16 as the next product's activation pass would round it; whole tiles are written
            __syncthreads(); // (the stages are read out: 4 KB of them for each wave's four tiles)
            lds_char * mine = (lds_char *) gm_smem + wid * GD_CT * 1024;
            if (row0 >= M) return;
#pragma unroll
            for (int n = 0; n < GD_CT; ++n)
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float gt = tot[2 * p][n][r], u = tot[2 * p + 1][n][r];
                        float h = (gt / (1.0f + expf(-gt))) * u;
                        asm volatile("" : "+v"(h)); // the fp32 value the GLU node holds, formed as such
                        *(__attribute__((address_space(3))) _Float16 *) (mine + n * 1024 + ((2 * p + (c >> 3)) * 16 + 4 * j + r) * 16 + (c & 7) * 2) = (_Float16) h;
                    }
            char * out = (char *) a.tile_out + (((uint64_t) batch * (uint32_t) (M >> 5) + (uint32_t) (row0 >> 5)) * (uint32_t) a.out_tt + (uint32_t) tt0) * 1024 + loff;
#pragma unroll
            for (int n = 0; n < GD_CT; ++n)
                if (16 * (tt0 + n) < a.N) *(half8_t *) (out + n * 1024) = *(lds_half8 *) (mine + n * 1024 + loff);
            return;
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int row = row0 + 16 * p + c;
            if (row >= M) continue;
#pragma unroll
            for (int n = 0; n < GD_CT; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int   tok = 16 * (tt0 + n) + 4 * j + r;
                    const float gt = tot[2 * p][n][r], u = tot[2 * p + 1][n][r];
                    if (tok < a.N) *(float *) (db + (uint64_t) tok * mt.nb1 + (uint64_t) row * 4) = (gt / (1.0f + expf(-gt))) * u;
                }
        }
    } else {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) {
            const int row = 16 * (rtw + rt) + c;
            if (row >= M) continue;
#pragma unroll
            for (int n = 0; n < GD_CT; ++n)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int tok = 16 * (tt0 + n) + 4 * j + r;
                    if (tok >= a.N) continue;
                    float val = tot[rt][n][r];
                    if (a.res)
                        val = scaled_residual(val, a.res_scale, *(const float *) (a.res + (uint64_t) i12 * a.rnb2 + (uint64_t) i13 * a.rnb3 + (uint64_t) tok * a.rnb1 + (uint64_t) row * 4));
                    *(float *) (db + (uint64_t) tok * mt.nb1 + (uint64_t) row * 4) = val;
                }
        }
    }
}

// ---- activations -> operand tiles ------------------------------------------------------------------------------------
struct gm_acts {
    const char *  x;
    uint64_t      nb11, nb12, nb13;
    int           ne12, N, K, n_tt, n_kb, row_blocks;
    const float * norm_w;
    float         eps;
    const double * totals;  // a cache write's wave totals: its scalar joins every value before the rounding
    float         sync_scale, sync_bias;
    half8_t *     xt;
    // rotation angles of the launch behind (blocks from row_blocks on)
    const int32_t * pos; const float * ff;
    rope_params   rp;
    int           rope_T;
    float2 *      tab;
};

// One wave = one token: its row rounded to f16 (normalised first: RMS_NORM in the RMS_NORM kernel's wave-per-row order, then
// the MUL node, each rounded as the separate kernels round) and stored as its sixteen-byte pieces of the tiles.  Four tokens
// a work-group and no LDS: with some tens to a thousand tokens the pass is one trip to memory and its latency, and a tile's
// sixteen rows in one work-group of 1024 threads (as qt_acts_norm_kernel has it for prefill sizes) leave most of the chip idle.
template <bool NORM>
__global__ __launch_bounds__(256) void gm_acts_kernel(const gm_acts a) {
    const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
    if ((int) blockIdx.x >= a.row_blocks) { // the angle table: (cos, sin) of (token, pair), a chain of multiplications and two trigonometric evaluations each
        const int idx = ((int) blockIdx.x - a.row_blocks) * 256 + (int) threadIdx.x;
        if (idx >= a.N * 32 || blockIdx.y || blockIdx.z) return;
        const int tok = idx >> 5, ip = idx & 31;
        float c, sn;
        rope_cos_sin(a.rp, (float) a.pos[tok % a.rope_T], ip, a.ff ? a.ff[ip] : 1.0f, c, sn);
        a.tab[idx] = make_float2(c, sn);
        return;
    }
    const int tok = (int) blockIdx.x * 4 + wid, batch = blockIdx.y;
    if (tok >= 16 * a.n_tt) return;
    const int i12 = batch % a.ne12, i13 = batch / a.ne12;
    const int nvec = a.K / 4, iv0 = 256 * (int) blockIdx.z + lane; // (nvec is a multiple of 64: whole waves)
    char * out = (char *) (a.xt + ((int64_t) batch * a.n_kb * a.n_tt + (tok >> 4)) * 64) + (tok & 15) * 16;
    auto put = [&](int iv, half4_t h) { // columns 4 iv .. + 3: half a piece of k block iv / 8
        *(half4_t *) (out + (int64_t) (iv >> 3) * a.n_tt * 1024 + ((iv >> 1) & 3) * 256 + (iv & 1) * 8) = h;
    };
    if (tok >= a.N) { // (uniform) the last tile's missing tokens
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (iv0 + 64 * u < nvec) put(iv0 + 64 * u, half4_t{0, 0, 0, 0});
        return;
    }
    const float * row = (const float *) (a.x + (uint64_t) i12 * a.nb12 + (uint64_t) i13 * a.nb13 + (uint64_t) tok * a.nb11);
    if constexpr (NORM) {
        vx_rms_row r;
        float4     gn[4];
        vx_rms_row_load(r, row, a.K, lane);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc)
            if (lane + 64 * cc < nvec) gn[cc] = ((const float4 *) a.norm_w)[lane + 64 * cc];
        const float sc = vx_rms_row_scale(r, a.K, lane, a.eps);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            if (lane + 64 * cc >= nvec) break;
            float       v[4]  = { r.v[cc].x, r.v[cc].y, r.v[cc].z, r.v[cc].w };
            const float gg[4] = { gn[cc].x, gn[cc].y, gn[cc].z, gn[cc].w };
            half4_t h;
#pragma unroll
            for (int i = 0; i < 4; ++i) { v[i] *= sc; v[i] *= gg[i]; h[i] = (_Float16) v[i]; }
            put(lane + 64 * cc, h);
        }
    } else {
        // (blockIdx.z: 1024 columns of the row.  As one wave a row, four trips one after the other, the pass made products of K 4096 over 203 tokens
        // 14.5 us, 13.1 now; 337 tokens 17.5 / 16.6)
        float4_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = ((const float4_t *) row)[min(iv0 + 64 * u, nvec - 1)];
        if (a.totals) { // (uniform) the ADD1 node
            const float y = kvs_scalar_of_16(a.totals, lane, a.sync_scale, a.sync_bias);
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] += y;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (iv0 + 64 * u >= nvec) break;
            half4_t h;
#pragma unroll
            for (int i = 0; i < 4; ++i) h[i] = (_Float16) v[u][i];
            put(iv0 + 64 * u, h);
        }
    }
}

template <int WT, int MT, int NT, int RW, int CH, int S, int EPI>
bool gm_launch(const gm_args & a, int gx, int gy, int nbatch, hipStream_t st) {
    using sh = gm_shape<WT, MT, NT, RW, CH, S>;
    auto kern = gm_kernel<WT, MT, NT, RW, CH, S, EPI>;
    static bool raised = false;
    if (!raised && sh::LDS > 64 * 1024) {
        if (hipFuncSetAttribute((const void *) kern, hipFuncAttributeMaxDynamicSharedMemorySize, sh::LDS) != hipSuccess) { (void) hipGetLastError(); return false; }
        raised = true;
    }
    vx_launch(kern, dim3((unsigned) gx, (unsigned) gy, (unsigned) nbatch), dim3(64 * sh::NWAVES), (size_t) sh::LDS, st, a);
    return true;
}

template <int WT>
bool gm_go(int tile, int epi, const gm_args & a, int gx, int gy, int nbatch, hipStream_t st) {
    switch (tile) {
#define X(I, MT, NT, RW, CH, SQ, SF, A_, B_)                                                                            \
        case I: {                                                                                                       \
            constexpr int S = WT == VX_GM_Q8 ? SQ : SF;                                                                 \
            if constexpr (S > 0) {                                                                                      \
                if (epi == GM_PLAIN) return gm_launch<WT, MT, NT, RW, CH, S, GM_PLAIN>(a, gx, gy, nbatch, st);          \
                if constexpr (MT % 2 == 0) {                                                                            \
                    if (epi == GM_SWIGLU) return gm_launch<WT, MT, NT, RW, CH, S, GM_SWIGLU>(a, gx, gy, nbatch, st);    \
                    return gm_launch<WT, MT, NT, RW, CH, S, GM_SEGS>(a, gx, gy, nbatch, st);                            \
                }                                                                                                       \
            }                                                                                                           \
            return false;                                                                                               \
        }
        GM_TILES(X)
#undef X
    }
    return false;
}

} // namespace

// Rows of a matrix that the kernels of mul_mat.hip serve better (`tokens` of the whole call; a gate/up pair goes by one matrix's rows).
// Measured with graphs of several weights and, for the pre-tiled kernel, pinned ones; these / here, microseconds:
//   * over 6144 rows and from 1024 tokens on, where the pre-tiled kernel fills the chip with the pair's 256 x 128 tiles: K 4096, pairs of
//     11264 rows x 1024 tokens 215 / 294, 14336 x 2048 499 / 739; 16384 rows x 2048 299 / 421 (8192 x 1024: 121 / 108);
//   * over 6144 rows with K up to 1024, where the 128 x 128 tiles of the LDS-tiled kernel fill it: Q8_0 16384 rows x 300 tokens 32 / 30,
//     x 512 37 / 43; F16 16384 x 200 23.7 / 25.0, x 448 32 / 44, 8192 x 200 17.6 / 14.9, x 337 17.5 / 20.8, x 800 31 / 40;
//   * a vocabulary's 73448 rows: K 1024 x 64 tokens 1.4 of the time here, x 100 0.96, x 512 0.84, K 4096 x 100 1.3, x 300 0.93;
//   * few rows and a long K, which those kernels cut across work-groups: K 4096, 128 rows x 300 tokens 1.33, x 512 0.91, x 2048 0.77;
//     K 8192, 128 rows x 45 0.97, x 512 0.74.
static bool gm_rows_ok(int wtype, int64_t K, int64_t tokens, int64_t M) {
    if (M <= 256 && (K >= 8192 || (K >= 4096 && tokens >= 512))) return false;
    if (M <= 6144) return true;
    if (M > 49152 && tokens > 96) return false;
    const int64_t tiles = (M + 255) / 256 * ((tokens + 127) / 128);
    if (wtype == VX_GM_Q8 && tokens >= 1024 && tiles >= 320 && tiles * K >= 512 * 1024) return false;
    return K > 1024 || M * tokens <= (wtype == VX_GM_Q8 ? 5120 : 2560) * 1024;
}

bool vx_gm_shape(int wtype, int64_t K, int64_t N, int64_t nbatch, int64_t M) {
    // Up to where this kernel's 64 x 128 tiles beat the LDS-tiled and pre-tiled kernels' larger ones in a layer of 1024 / 4096 rows.
    // Q8_0, 24 layers of one prompt: 1200 tokens 6270 -> 3818 us, 2048 6834 -> 5205, 2600 8990 -> 7156, but 4000 9639 -> 10114;
    // F16, 56 products: 1100 tokens 1343 -> 1260 us, 1537 1417 -> 1463.
    if (N <= 16 || N * nbatch > (wtype == VX_GM_Q8 ? 3072 : 1152) || nbatch > 65535) return false;
    // K of whole 256s (the stages).  Up to 16 tokens are the streaming kernel's; what it takes beyond them with K of 513 to
    // 1024 it sums in this kernel's order, and with K above 2048 it takes nothing beyond them: elsewhere a call that one of
    // the two had to decline (alignment, VX_ACT_Q8's groups) would differ from its neighbours in the last bit.
    return K % 256 == 0 && ((K > 512 && K <= 1024) || (K > 2048 && K <= 16384)) && gm_rows_ok(wtype, K, N * nbatch, M);
}

bool vx_gm_on(int64_t N) {
    // Switches, read on every call.  VX_GEMM_MID=0: the kernels of mul_mat.hip for these shapes.  VX_GEMM_LDS other than 1 and, from
    // 1024 tokens on, VX_GEMM_Q8T other than 1 ask for one of those kernels by name (another rounding of the weights, the older
    // kernels, one prefill kernel or the other): then it is that kernel that runs.
    auto is = [](const char * name, int by_default) { const char * e = getenv(name); return e ? atoi(e) : by_default; };
    return is("VX_GEMM_MID", 1) != 0 && is("VX_GEMM_LDS", 1) == 1 && (N < 1024 || is("VX_GEMM_Q8T", 1) == 1);
}

bool vx_gm_takes(const vx_gm_call & c) {
    auto al16 = [](const void * p, uint64_t s) { return (uintptr_t) p % 16 == 0 && s % 16 == 0; };
    for (int i = 0; i < c.nmat; ++i) {
        if (!vx_gm_shape(c.wtype, c.K, c.N, (int64_t) c.ne12 * c.ne13, c.mat[i].M)) return false;
        if (!al16(c.mat[i].w, c.mat[i].nb01) || c.mat[i].M < 1) return false;
        if (c.nmat > 1 && c.mat[i].M % 64) return false;
    }
    if (c.w2 && !al16(c.w2, 0)) return false;
    if (!c.tile_in && !(al16(c.x, c.nb11) && c.nb12 % 16 == 0 && c.nb13 % 16 == 0)) return false;
    if (c.norm_w && (c.K > 1024 || (uintptr_t) c.norm_w % 16)) return false;
    return vx_gm_on(c.N);
}

size_t vx_gm_tile_bytes(int64_t K, int64_t N, int64_t nbatch) {
    // (a work-group's last stage may read up to 7 tiles past the last token tile: their products are dropped)
    return (size_t) nbatch * (size_t) (K / 32) * (size_t) ((N + 15) / 16) * 1024 + 8192;
}

static void gd_launch(int epi, dim3 grid, const gm_args & a, hipStream_t st);

vx_status vx_gm_run(const vx_gm_call & c, hipStream_t st) {
    const int nbatch = c.ne12 * c.ne13;
    gm_args a = {};
    for (int i = 0; i < c.nmat; ++i) a.mat[i] = c.mat[i];
    a.nmat = c.nmat; a.w2 = c.w2;
    a.n_kb = (int) (c.K / 32); a.N = (int) c.N; a.ne12 = c.ne12;
    a.n_tt = c.tile_in ? c.tile_tt : (int) ((c.N + 15) / 16);
    a.res = c.res; a.rnb1 = c.rnb1; a.rnb2 = c.rnb2; a.rnb3 = c.rnb3; a.res_scale = c.res_scale;
    a.tile_out = (_Float16 *) c.tile_out; a.out_tt = c.tile_tt;
    bool rotate = false;
    for (int i = 0; i < c.nmat; ++i) rotate = rotate || c.mat[i].rope;
    const size_t xt_bytes = c.tile_in ? 0 : vx_gm_tile_bytes(c.K, c.N, nbatch), tab_bytes = rotate ? (size_t) c.N * 32 * sizeof(float2) : 0;
    void * ws = nullptr;
    if (xt_bytes + tab_bytes) {
        const vx_status rc = vx_workspace(st, c.ws_offset + xt_bytes + tab_bytes, &ws, true);
        if (rc != VX_OK) return rc;
    }
    char * base = (char *) ws + c.ws_offset;
    a.xt = c.tile_in ? (const half8_t *) c.tile_in : (const half8_t *) base;
    if (!c.tile_in) {
        gm_acts p = {};
        p.x = c.x; p.nb11 = c.nb11; p.nb12 = c.nb12; p.nb13 = c.nb13; p.ne12 = c.ne12;
        p.N = a.N; p.K = (int) c.K; p.n_tt = a.n_tt; p.n_kb = a.n_kb;
        p.row_blocks = 4 * a.n_tt;
        p.norm_w = c.norm_w; p.eps = c.norm_eps;
        p.totals = c.add_totals; p.sync_scale = c.add_scale; p.sync_bias = c.add_bias;
        p.xt = (half8_t *) base;
        int blocks = p.row_blocks;
        if (rotate) {
            p.pos = c.pos; p.ff = c.ff; p.rp = c.rp; p.rope_T = c.rope_T;
            p.tab = (float2 *) (base + xt_bytes);
            a.rope_tab = p.tab;
            blocks += (a.N * 32 + 255) / 256;
        }
        if (c.norm_w) vx_launch(gm_acts_kernel<true>, dim3((unsigned) blocks, (unsigned) nbatch), dim3(256), 0, st, p); // (K of at most 1024)
        else          vx_launch(gm_acts_kernel<false>, dim3((unsigned) blocks, (unsigned) nbatch, (unsigned) ((c.K + 1023) / 1024)), dim3(256), 0, st, p);
    }
    const int epi = c.w2 ? GM_SWIGLU : c.nmat > 1 ? GM_SEGS : GM_PLAIN;
    gm_product shape = { c.wtype, epi, c.nmat, {}, c.K, c.N, nbatch };
    for (int i = 0; i < c.nmat; ++i) shape.M[i] = c.mat[i].M;
    auto fits = [](const gm_share & s) { return 8 * s.nx <= 0x7fffffff && s.ny <= 65535; };
    if (gd_takes(shape)) {
        const void * tiles = nullptr;
        const float * scales = nullptr;
        const int64_t MV = c.w2 ? 2 * (int64_t) c.mat[0].M : c.mat[0].M;
        const gm_share s = gm_share_out((MV + GD_ROWS - 1) / GD_ROWS, (c.N + GD_TOKS - 1) / GD_TOKS, nbatch, (double) MV * c.K * 2, (double) c.N * c.K * 2, GD_PER_CU);
        if (fits(s) && vx_qt_kept_tiles(c.mat[0].w, c.w2, c.K, c.mat[0].M, c.mat[0].nb01, st, &tiles, &scales)) {
            a.wt = (const half8_t *) tiles; a.wdt = scales; a.n_rt = (int) ((MV + 15) / 16); a.xr = s.xr;
            gd_launch(epi, dim3((unsigned) (8 * s.nx), (unsigned) s.ny, (unsigned) nbatch), a, st);
            return VX_OK;
        }
    }
    gm_share s = {};
    const int tile = gm_tile_choice(shape, s);
    if (!fits(s)) return vx_fail(VX_ERR_UNSUPPORTED, "mul_mat: launch too large");
    a.xr = s.xr;
    if (epi != GM_SWIGLU) for (int i = 0, wg = 0; i < c.nmat; ++i) { a.mat[i].wg0 = wg; wg += (c.mat[i].M + gm_tiles[tile].rows - 1) / gm_tiles[tile].rows; }
    const int gx = (int) (8 * s.nx), gy = (int) s.ny;
    const bool ok = c.wtype == VX_GM_Q8 ? gm_go<VX_GM_Q8>(tile, epi, a, gx, gy, nbatch, st) : gm_go<VX_GM_F16>(tile, epi, a, gx, gy, nbatch, st);
    return ok ? VX_OK : vx_fail(VX_ERR_HIP, "mul_mat: the kernel could not be given its LDS");
}

// (last: gm_kernel's instances keep their places in the code object)
static void gd_launch(int epi, dim3 grid, const gm_args & a, hipStream_t st) {
    if (epi == GM_SWIGLU) vx_launch(gd_kernel<GM_SWIGLU>, grid, dim3(256), (size_t) GD_LDS, st, a);
    else                  vx_launch(gd_kernel<GM_PLAIN>, grid, dim3(256), (size_t) GD_LDS, st, a);
}
