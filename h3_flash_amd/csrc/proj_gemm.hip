// Projection GEMM of the H3 attention block with the q/k RMSNorm + RoPE
// prologue as its epilogue (gfx950).
//
//   y[m, f] = sum_k x[m, k] * w[f, k] (+ bias[f])            (nn.Linear)
//   q / k sections: per (token m, head of 128 features) the result, rounded
//   to bf16 as the module's linear outputs it, is RMS-normalised in fp32,
//   scaled by the norm weight and rotated (rotate-half RoPE over the first R
//   features, table row m mod seqlen), then rounded to bf16 again: the
//   reference's order of a projection followed by fused_qknorm_rope; v and
//   out-projection sections are stored as they are.
//
// x (M tokens x K) and w (N features x K) are bf16 with K contiguous (the
// nn.Linear layout). The product is computed transposed, C^T = W X^T, on
// v_mfma_f32_16x16x32_bf16: the W fragment is the A operand (16 features x
// 32 K) and the X fragment the B operand (32 K x 16 tokens), so every lane of
// the result holds one token and 4 consecutive features per 16-feature block.
//
// Tiling: one workgroup of 4 waves per CU computes TF features x 16*NT tokens
// (proj_gemm_kernel<TF, NT, SW, SX>), one wave per SIMD. Large tiles split the waves
// 2 x 2 (128 features x 8*NT tokens each), small ones 4 x 1 (TF/4 features x
// all tokens), whichever reads fewer LDS bytes per MFMA; the accumulators are
// held in the accumulation registers (256 per lane at TF = 256, NT = 16).
//
// K advances 64 at a time through rings of SW (W rows) and SX (X rows) LDS
// stages, as many as fit in 160 KB, filled HBM -> LDS by buffer_load ... lds (16 bytes per lane, no VGPR
// staging; each load covers whole 128-byte lines of 8 rows). LDS rows are 128
// bytes; the 16-byte chunk c of row r sits at c ^ ((r >> 1) & 7), so the 16
// rows a quarter-wave's fragment read touches hit 16 distinct bank groups.
// One barrier per K step of 64, in its middle (see the step below).
#include <math.h>

#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace h3a {
namespace {

constexpr int kPK = 64;                   // K per stage (two MFMA K steps of 32)
constexpr int kPWaves = 4;
constexpr int kPThreads = kPWaves * 64;
constexpr int kPRow = kPK * 2;            // LDS bytes per tile row

typedef __attribute__((address_space(3))) char lds_char;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) i32x4 lds_i32x4;
typedef __attribute__((address_space(3))) i32x2 lds_i32x2;

// vmcnt(N) and lgkmcnt(0): the wave's own DMA loads beyond the newest N have
// landed and its LDS reads have completed.
template <int N>
__device__ __forceinline__ void wait_vm_lgkm() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
}

__device__ __forceinline__ void barrier() { asm volatile("s_barrier" ::: "memory"); }

// acc += A B on v_mfma_f32_16x16x32_bf16 with the accumulator pinned to the
// accumulation registers: with the builtin, the 256 accumulators of a lane
// are split between VGPRs and AGPRs and copied around the loop back edge.
__device__ __forceinline__ void mfma_acc(f32x4& acc, const bf16x8& a, const bf16x8& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}

// f(0), ..., f(N - 1) with compile-time indices.
template <int... I, typename F>
__device__ __forceinline__ void static_for_seq(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_seq(std::make_integer_sequence<int, N>{}, f);
}

// Section i of the launch, selected field by field (indexing the kernel
// argument with a runtime index would copy the whole argument block into
// private memory).
__device__ __forceinline__ ProjSection section(const ProjGemmParams& p, int i) {
    auto pick = [&](auto f0, auto f1, auto f2) { return i == 0 ? f0 : i == 1 ? f1 : f2; };
#define H3A_FIELD(f) pick(p.sec[0].f, p.sec[1].f, p.sec[2].f)
    return ProjSection{H3A_FIELD(w),    H3A_FIELD(bias), H3A_FIELD(norm_w), H3A_FIELD(y),    H3A_FIELD(w_rs),
                       H3A_FIELD(y_rs), H3A_FIELD(n),    H3A_FIELD(tiles),  H3A_FIELD(mode), H3A_FIELD(eps)};
#undef H3A_FIELD
}

// Tile t of the grouped order: groups of p.group_m token tiles x every feature
// tile, token tile fastest.
struct TileCoord {
    int sec;  // section of the feature tile
    int f0;   // first feature of the tile, within the section
    int m0;   // first token of the tile
};
__device__ __forceinline__ TileCoord tile_coord(const ProjGemmParams& p, int tile, int tile_f, int tile_m) {
    const int in_group = p.group_m * p.n_tiles;
    const int first_m = (tile / in_group) * p.group_m;
    const int group_m = min(p.m_tiles - first_m, p.group_m);
    const int mt = first_m + (tile % in_group) % group_m;
    int nt = (tile % in_group) / group_m;
    int sec = 0;
    if (p.n_sections > 1 && nt >= p.sec[0].tiles) {
        nt -= p.sec[0].tiles;
        sec = 1;
        if (p.n_sections > 2 && nt >= p.sec[1].tiles) {
            nt -= p.sec[1].tiles;
            sec = 2;
        }
    }
    return TileCoord{sec, nt * tile_f, mt * tile_m};
}

__device__ __forceinline__ void unpack8(const i32x4& raw, float* f) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float((uint32_t)raw[i] << 16);
        f[2 * i + 1] = __uint_as_float((uint32_t)raw[i] & 0xffff0000u);
    }
}

// Eight norm weights, of which only 8-byte alignment is known.
__device__ __forceinline__ void load_w8(const void* w, int col0, float* f) {
    const i32x2* const a = (const i32x2*)((const uint16_t*)w + col0);
    const i32x2 lo = a[0], up = a[1];
    unpack8(i32x4{lo.x, lo.y, up.x, up.y}, f);
}

// A tile shape: TF features x 16*NT tokens; SW stages of W rows, SX of X rows.
template <int TF, int NT, int SW, int SX>
struct Tile {
    static constexpr int kTokens = 16 * NT;
    // Waves over features x tokens. LDS reads per MFMA K step: 2 x 2 reads
    // 4 * (8 + NT/2) KB, 4 x 1 reads 4 * (TF/64 + NT) KB.
    static constexpr int WN = TF == 256 && NT >= 10 ? 2 : 4, WM = kPWaves / WN;
    static constexpr int NA = TF / 16 / WN, NB = NT / WM;  // 16 x 16 MFMA blocks of a wave
    static constexpr int kWBytes = TF * kPRow, kXBytes = kTokens * kPRow;
    static constexpr int kXBase = SW * kWBytes, kStages = kXBase + SX * kXBytes;  // X stages follow the W stages
    // DMA loads (1 KB: 8 rows) per wave and stage
    static constexpr int kLoadsW = TF / 8 / kPWaves, kLoadsX = kTokens / 8 / kPWaves;
    // Epilogue: the tile's bf16 output rows over the (then idle) stages, and
    // a row buffer per 16-lane group for RoPE partners across lanes.
    static constexpr int kOutRow = TF * 2;
    static constexpr int kOutBytes = kTokens * kOutRow;
    static constexpr int kPartner = any_r_row_bytes(16);
    static constexpr int kEpiBytes = kOutBytes + kPThreads / 16 * kPartner;
    static constexpr int kLds = kStages > kEpiBytes ? kStages : kEpiBytes;
    static_assert(NT % 2 == 0 && TF % 128 == 0, "DMA map: whole loads per wave");
    static_assert(NB * WM == NT && NA * NB >= 4, "wave map; an accumulator is next used 4 MFMAs later at the least");
    static_assert(SX >= 2 && SW > SX, "the waits below count loads in this order");
    static_assert(kLds <= 160 * 1024, "LDS of one workgroup");
};

// Epilogue of one tile, in two passes. First every wave adds the bias to its
// accumulators, rounds to bf16 (as the module's linear outputs it) and writes
// the values into the tile's output rows in LDS: token t, head h of the tile
// (128 features) at byte t * 2 TF + 256 h, its 16-byte chunk c at c ^ (t & 15)
// (both passes bank-conflict free). Then rows go out: plain ones as they are,
// 16 lanes each; norm rows are RMS-normalised in fp32 (sum of squares over the
// row's lanes by DPP), scaled by the norm weight, rotated and rounded once more,
// as the reference's separate steps do (dense_fa4.py:123-140,
// transformer.py:146-173; normalising the unrounded accumulator moves the LSE of
// the attention that follows by up to about 2e-3 against that order). With R a
// multiple of 16, 8 lanes take a row and each holds both columns of its pairs;
// otherwise 16 lanes, the partners c +- R/2 through any_r_partners. Stores are
// non-temporal (no later tile reads the rows), whole 128-byte lines. cos / sin
// of the next token are loaded before the current one is computed, once for the
// heads of the tile.
// Bound by VALU issue (one wave per SIMD, the matrix cores idle), and on long
// launches by the power it draws. So the weights are multiplied into the token's
// tables once for the tile's heads, and a pair's two values are unpacked and
// scaled once: with 16 lanes a row, each unpacking its partners again, 49,920
// tokens x 40 heads took 5,730 us, 6,240 x 40 725, 6,240 x 5 26.6; now 5,600,
// 712 and 23.5 (the epilogue in the accumulator layout, 4 lanes x 32 columns of
// a head, 5,624, 722 and 25.9). At R = 126, where that layout read partners and
// tables element by element, 1,296 x 40 went from 322 to 226 us, in part by the
// tile shape.
template <typename T>
__device__ __forceinline__ void epilogue(const ProjGemmParams& p, const TileCoord& tc, const f32x4 (&acc)[T::NA][T::NB],
                                         int wn, int wm, int tid, char* smem) {
    constexpr int kHeads = T::kOutRow / 256;
    // Opaque here, so that no lane-derived value of the epilogue is hoisted
    // and held (or spilled) across the K loop.
    asm volatile("" : "+v"(tid));
    const int lane = tid & 63;
    const ProjSection sec = section(p, tc.sec);
    lds_char* const out = (lds_char*)smem;
    {
        // Lane l holds, for token block b (token 16 (NB wm + b) + (l & 15)) and
        // feature block a, features 16 (NA wn + a) + 4 * (l >> 4) + e.
        const int f_wave = 16 * T::NA * wn, q = lane >> 4;
        const bool has_bias = sec.bias != nullptr;
        lds_char* const row = out + (16 * T::NB * wm + (lane & 15)) * T::kOutRow + (f_wave >> 7) * 256 + (q & 1) * 8;
        const int swz = ((lane & 15) ^ (q >> 1)) << 4;
#pragma unroll
        for (int a = 0; a < T::NA; ++a) {
            // (Features past the section, in the second half of a last tile,
            // read the section's first ones; their rows are not stored.)
            const int f = tc.f0 + f_wave + 16 * a + 4 * q;
            const i32x2 br = has_bias ? *(const i32x2*)((const uint16_t*)sec.bias + (f < sec.n ? f : 0)) : i32x2{0, 0};
            const float b0 = __uint_as_float((uint32_t)br.x << 16), b1 = __uint_as_float((uint32_t)br.x & 0xffff0000u);
            const float b2 = __uint_as_float((uint32_t)br.y << 16), b3 = __uint_as_float((uint32_t)br.y & 0xffff0000u);
            const int c = (((f_wave & 127) >> 3) + 2 * a) << 4;
#pragma unroll
            for (int b = 0; b < T::NB; ++b) {
                const f32x4 v = acc[a][b];
                *(lds_i32x2*)(row + b * 16 * T::kOutRow + (swz ^ c)) =
                    i32x2{(int)pack_bf16x2(v.x + b0, v.y + b1), (int)pack_bf16x2(v.z + b2, v.w + b3)};
            }
        }
    }
    __syncthreads();

    const int g = tid >> 4, j = tid & 15;  // row group, lane of the row
    const int heads = min(kHeads, (sec.n - tc.f0) >> 7);
    const int tokens = min(T::kTokens, p.m - tc.m0);
    char* const yb = (char*)sec.y + (int64_t)tc.m0 * sec.y_rs + (int64_t)tc.f0 * 2 + j * 16;
    auto load_row = [&](int t, int h, int chunk) {
        return *(const lds_i32x4*)(out + t * T::kOutRow + h * 256 + ((chunk ^ (t & 15)) << 4));
    };
    auto store_row = [&](int t, int h, const i32x4& v) {
        __builtin_nontemporal_store(v, (i32x4*)(yb + (int64_t)t * sec.y_rs + h * 256));
    };
    const int R = sec.mode != 0 ? p.rotary_dim : 0;
    if (sec.mode == 0) {
#pragma unroll 4
        for (int t = g; t < tokens; t += 16)
#pragma unroll
            for (int h = 0; h < kHeads; ++h)
                if (h < heads) store_row(t, h, load_row(t, h, j));
        return;
    }
    const float eps = sec.eps;
    const bool tab16 = (((uintptr_t)p.cos | (uintptr_t)p.sin) & 15) == 0 && (p.table_stride & 3) == 0;
    auto table_row = [&](int t) {
        int s = tc.m0 + min(t, tokens - 1);
        s = s < p.seqlen ? s : s % p.seqlen;
        return (int64_t)s * p.table_stride;
    };

    // R a multiple of 16 and tables with 16-byte rows: eight lanes take a row,
    // each one two 16-byte chunks that rotate with each other (columns 8 j and
    // R/2 on), or two of those past R. kAll: R = 128, every lane rotary. kFull:
    // the tables are read at both chunks' columns, else at the first's, the
    // halves being equal. A wave's eight rows of one access are two tokens' t
    // and t + 8 over, so that each 16 lanes read 16 different bank groups.
    auto pair_rows = [&](auto all_c, auto full_c) __attribute__((always_inline)) {
        constexpr bool kAll = decltype(all_c)::value, kFull = decltype(full_c)::value;
        const int j8 = lane & 7, g8 = lane >> 3, wave = tid >> 6;
        const int row0 = 16 * (wave >> 1) + 4 * (wave & 1) + (g8 >> 1) + 8 * (g8 & 1);  // of every 32 tokens
        const int np = kAll ? 8 : R >> 4;
        const bool rot = kAll || j8 < np;
        const int ca = rot ? j8 : 2 * j8, cb = rot ? j8 + np : 2 * j8 + 1;
        float wa[8], wb[8];
        load_w8(sec.norm_w, 8 * ca, wa);
        load_w8(sec.norm_w, 8 * cb, wb);
        constexpr int kTabs = kFull ? 4 : 2;
        struct Tabs {
            f32x4 c[kTabs], s[kTabs];
        };
        const int ta_col = rot ? 8 * ca : 0, tb_col = rot ? 8 * cb : 0;
        auto load_tables = [&](int t) __attribute__((always_inline)) {
            Tabs w;
            const float* const cr = p.cos + table_row(t);
            const float* const sr = p.sin + table_row(t);
#pragma unroll
            for (int i = 0; i < kTabs; ++i) {
                const int c = (i < 2 ? ta_col : tb_col) + 4 * (i & 1);
                w.c[i] = *(const f32x4*)(cr + c);
                w.s[i] = *(const f32x4*)(sr + c);
            }
            return w;
        };
        auto token = [&](int t, const Tabs& tab) __attribute__((always_inline)) {
            // y = (x r) (w cos) + (x' r) (w' sin): the weights times the tables
            // are the token's, shared by its heads. r comes first, as in the
            // separate steps: a row whose squares overflow fp32 (r = 0) gives
            // zeros, and small rows lose no bits to a subnormal product.
            float ta[8], tb[8], sa[8], sb[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float c0 = tab.c[e >> 2][e & 3], s0 = tab.s[e >> 2][e & 3];
                const float c1 = tab.c[(kFull ? 2 : 0) + (e >> 2)][e & 3], s1 = tab.s[(kFull ? 2 : 0) + (e >> 2)][e & 3];
                ta[e] = rot ? wa[e] * c0 : wa[e];
                tb[e] = rot ? wb[e] * c1 : wb[e];
                sa[e] = rot ? -(wb[e] * s0) : -0.f;
                sb[e] = rot ? wa[e] * s1 : -0.f;
            }
            char* const yr = (char*)sec.y + (int64_t)(tc.m0 + t) * sec.y_rs + (int64_t)tc.f0 * 2;
#pragma unroll
            for (int h = 0; h < kHeads; ++h) {
                if (h >= heads) break;
                float xa[8], xb[8];
                unpack8(load_row(t, h, ca), xa);
                unpack8(load_row(t, h, cb), xb);
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += xa[e] * xa[e];
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += xb[e] * xb[e];
                const float r = rsqrtf(group_sum<8>(ss) * (1.0f / 128.0f) + eps);
                float oa[8], ob[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float na = xa[e] * r, nb = xb[e] * r;
                    oa[e] = na * ta[e] + (rot ? nb : 0.f) * sa[e];
                    ob[e] = nb * tb[e] + (rot ? na : 0.f) * sb[e];
                }
                i32x4 va, vb;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    va[e] = (int)pack_bf16x2(oa[2 * e], oa[2 * e + 1]);
                    vb[e] = (int)pack_bf16x2(ob[2 * e], ob[2 * e + 1]);
                }
                if (t < tokens) {
                    __builtin_nontemporal_store(va, (i32x4*)(yr + h * 256 + 16 * ca));
                    __builtin_nontemporal_store(vb, (i32x4*)(yr + h * 256 + 16 * cb));
                }
            }
        };
        const int n = (tokens + 31) / 32;
        Tabs t0 = load_tables(row0);
        int it = 0, t = row0;
        for (; it + 2 <= n; it += 2, t += 64) {
            const Tabs t1 = load_tables(t + 32);
            token(t, t0);
            t0 = load_tables(t + 64);
            token(t + 32, t1);
        }
        if (it < n) token(t, t0);
    };
    if (R > 0 && (R & 15) == 0 && tab16) {
        if (R == 128 && p.rope_full_tables == 0)
            pair_rows(std::true_type{}, std::false_type{});
        else if (R == 128)
            pair_rows(std::true_type{}, std::true_type{});
        else if (p.rope_full_tables == 0)
            pair_rows(std::false_type{}, std::false_type{});
        else
            pair_rows(std::false_type{}, std::true_type{});
        return;
    }

    // No rotary columns, or (kRope) any even R and tables at any alignment:
    // sixteen lanes a row.
    const int half = R >> 1, col0 = 8 * j;
    float wv[8], wp[8];
    load_w8(sec.norm_w, col0, wv);
    auto rows = [&](auto rope_c) __attribute__((always_inline)) {
        constexpr bool kRope = decltype(rope_c)::value;
        uint32_t pmask[4];
        if constexpr (kRope) {
            // Partner weights with the rotation's sign, zero past R.
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int c = min(col0 + e, R - 1);
                const float w = bf16_to_f32(((const uint16_t*)sec.norm_w)[c < half ? c + half : c - half]);
                wp[e] = c < half ? -w : w;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) pmask[i] = col0 + 2 * i < R ? 0xffffffffu : 0u;
        }
        const bool pairs = (((uintptr_t)p.cos | (uintptr_t)p.sin) & 7) == 0 && (p.table_stride & 1) == 0;  // uniform
        struct Tabs {
            f32x4 c[2], s[2];  // cos and sin of the lane's 8 columns
        };
        auto load_tables = [&](int t) __attribute__((always_inline)) {
            Tabs w{};
            if constexpr (kRope) {
                const float* const cr = p.cos + table_row(t);
                const float* const sr = p.sin + table_row(t);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int c0 = min(col0 + 4 * i, R - 2), c1 = min(col0 + 4 * i + 2, R - 2);
                    if (pairs) {
                        const f32x2 a = *(const f32x2*)(cr + c0), b = *(const f32x2*)(cr + c1);
                        const f32x2 c = *(const f32x2*)(sr + c0), d = *(const f32x2*)(sr + c1);
                        w.c[i] = f32x4{a.x, a.y, b.x, b.y};
                        w.s[i] = f32x4{c.x, c.y, d.x, d.y};
                    } else {
                        w.c[i] = f32x4{cr[c0], cr[c0 + 1], cr[c1], cr[c1 + 1]};
                        w.s[i] = f32x4{sr[c0], sr[c0 + 1], sr[c1], sr[c1 + 1]};
                    }
                }
            }
            return w;
        };
        // A wave's four groups are four consecutive tokens: the loop bound is
        // the wave's, so every lane joins the row sums and partner reads.
        const int t_end = (tokens - 4 * (g >> 2) + 15) / 16;  // iterations of this wave
        auto token = [&](int t, const Tabs& tab) __attribute__((always_inline)) {
            float tc_[8], ts_[8];  // as above
            if constexpr (kRope) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const bool in = col0 + e < R;
                    tc_[e] = in ? wv[e] * tab.c[e >> 2][e & 3] : wv[e];
                    ts_[e] = in ? wp[e] * tab.s[e >> 2][e & 3] : -0.f;
                }
            }
#pragma unroll
            for (int h = 0; h < kHeads; ++h) {
                if (h >= heads) break;
                const i32x4 x = load_row(t, h, j);
                float xv[8], o[8];
                unpack8(x, xv);
                float ss = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) ss += xv[e] * xv[e];
                const float r = rsqrtf(group_sum<16>(ss) * (1.0f / 128.0f) + eps);
                if constexpr (!kRope) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = (xv[e] * r) * wv[e];
                } else {
                    i32x4 px = any_r_partners(out + T::kOutBytes + g * T::kPartner, x, j, R);
#pragma unroll
                    for (int i = 0; i < 4; ++i) px[i] &= (int)pmask[i];
                    float xp[8];
                    unpack8(px, xp);
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = (xv[e] * r) * tc_[e] + (xp[e] * r) * ts_[e];
                }
                i32x4 w;
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = (int)pack_bf16x2(o[2 * e], o[2 * e + 1]);
                if (t < tokens) store_row(t, h, w);
            }
        };
        Tabs t0 = load_tables(g);
        int it = 0, t = g;
        for (; it + 2 <= t_end; it += 2, t += 32) {
            const Tabs t1 = load_tables(t + 16);
            token(t, t0);
            t0 = load_tables(t + 32);
            token(t + 16, t1);
        }
        if (it < t_end) token(t, t0);
    };
    if (R == 0)
        rows(std::false_type{});
    else
        rows(std::true_type{});
}

template <int TF, int NT, int SW, int SX>
__global__ __launch_bounds__(kPThreads, 1) void proj_gemm_kernel(ProjGemmParams p) {
    using T = Tile<TF, NT, SW, SX>;
    __shared__ __attribute__((aligned(1024))) char smem[T::kLds];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave / T::WM, wm = wave % T::WM;

    // One workgroup per tile. Workgroup b runs on XCD b mod 8 (round-robin
    // dispatch) as that XCD's (b / 8)-th; each XCD owns one contiguous range
    // of the grouped tile order, so the ~32 tiles an XCD runs at a time are
    // consecutive in it and share their X and W panels in the XCD's L2. (A
    // persistent grid of one workgroup per CU looping over its XCD's range
    // measured from 1% faster to 4% slower, and is not used.)
    const int total = p.m_tiles * p.n_tiles;
    const int bid = blockIdx.x;
    const int xcd = bid & 7, local = bid >> 3;
    const int per = total >> 3, rem = total & 7;
    const int tile = xcd * per + min(xcd, rem) + local;
    const TileCoord tc = tile_coord(p, tile, TF, T::kTokens);

    // Operand resources, based at the tile's first row: rows past the section
    // or the token range are outside their records and load as zeros.
    const ProjSection sec = section(p, tc.sec);
    const int32_t w_rs = (int32_t)sec.w_rs, x_rs = (int32_t)p.x_rs;
    i32x4 rw = make_rsrc_words((const char*)sec.w + (int64_t)tc.f0 * sec.w_rs,
                                     (uint32_t)((int64_t)(min(TF, sec.n - tc.f0) - 1) * sec.w_rs + p.k * 2));
    i32x4 rx = make_rsrc_words((const char*)p.x + (int64_t)tc.m0 * p.x_rs,
                                     (uint32_t)((int64_t)(min(T::kTokens, p.m - tc.m0) - 1) * p.x_rs + p.k * 2));
    // DMA map: load i of wave w fills rows 8 (4i + w) .. +8 of an operand's
    // stage; lane L writes LDS chunk (L & 7) of row r = 8 (4i + w) + (L >> 3),
    // which holds the row's 16-byte chunk (L & 7) ^ ((r >> 1) & 7) =
    // (L & 7) ^ (4 (w & 1) + (L >> 4)). Everything that depends on the lane is
    // the same for every load; i and the K step go into the scalar offset.
    const int chunk = ((lane & 7) ^ (4 * (wave & 1) + (lane >> 4))) << 4;
    const int row0 = 8 * wave + (lane >> 3);
    const uint32_t dw = (uint32_t)(row0 * w_rs + chunk), dx = (uint32_t)(row0 * x_rs + chunk);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(const lds_char*)smem;
    const uint32_t lds_wave = lds0 + (uint32_t)wave * 1024u;
    // Load j of this wave's share of a K step's rows (32 j rows on from the
    // wave's first), into LDS at dst + 4096 j. buffer_load ... lds writes 16
    // bytes per lane to LDS address M0 + 16*lane; M0 needs one wait state
    // before the load reads it. The row offsets stay in scalar registers and
    // the resources' bases move along K: three instructions a load, which fit
    // between two MFMAs (offsets formed per load took six, and held up the
    // lone wave's MFMAs).
    auto dma1 = [&](const i32x4& rsrc, uint32_t voff, uint32_t soff, uint32_t dst, int j) __attribute__((always_inline)) {
        asm volatile("s_add_u32 m0, %0, %1\n\ts_nop 0\n\tbuffer_load_dwordx4 %2, %3, %4 offen lds"
                     :
                     : "s"(dst), "i"(j * 4096), "v"(voff), "s"(rsrc), "s"(soff)
                     : "memory", "scc");
    };
    uint32_t sow[T::kLoadsW], sox[T::kLoadsX];
#pragma unroll
    for (int j = 0; j < T::kLoadsW; ++j) sow[j] = (uint32_t)(32 * j * w_rs);
#pragma unroll
    for (int j = 0; j < T::kLoadsX; ++j) sox[j] = (uint32_t)(32 * j * x_rs);
    auto dma_w1 = [&](const i32x4& r, uint32_t stage, int j) __attribute__((always_inline)) {
        dma1(r, dw, sow[j], lds_wave + stage, j);
    };
    auto dma_x1 = [&](const i32x4& r, uint32_t stage, int j) __attribute__((always_inline)) {
        dma1(r, dx, sox[j], lds_wave + T::kXBase + stage, j);
    };
    // The resource one K step further along its rows. The records stay: a
    // lane's offset in its row is under 128 bytes and a row is at least the
    // reduction long, so the row after the last one is out of range at every
    // base.
    auto advance = [](i32x4& r) __attribute__((always_inline)) {
        const uint64_t base = ((uint64_t)(uint32_t)r.y << 32 | (uint32_t)r.x) + kPRow;
        r.x = (int)(uint32_t)base;
        r.y = (int)((uint32_t)(base >> 32) & 0xffffu);
    };

    // Fragment reads: lane l takes row (16*block + (l & 15)) of the wave's
    // operand rows and, for MFMA K step h of the stage, logical chunk
    // 4h + (l >> 4) (K 32h + 8*(l>>4) .. +8); swz(row) = ((l & 15) >> 1) & 7.
    const int sl = (lane >> 1) & 7;
    const int fo0 = (lane & 15) * kPRow + (((lane >> 4) ^ sl) << 4);
    const int fo1 = (lane & 15) * kPRow + (((4 + (lane >> 4)) ^ sl) << 4);
    const lds_char* const lds = (const lds_char*)smem;
    const lds_char* const wfr0 = lds + wn * 16 * T::NA * kPRow + fo0;
    const lds_char* const wfr1 = lds + wn * 16 * T::NA * kPRow + fo1;
    const lds_char* const xfr0 = lds + T::kXBase + wm * 16 * T::NB * kPRow + fo0;
    const lds_char* const xfr1 = lds + T::kXBase + wm * 16 * T::NB * kPRow + fo1;

    f32x4 acc[T::NA][T::NB];
    bf16x8 fw[2][T::NA], fx[2][T::NB];
    constexpr int kReads = T::NA + T::NB, kMfmas = T::NA * T::NB;

    // Fragment j of MFMA K step h of the stages at byte offsets sw, sx.
    auto read1 = [&](uint32_t sw, uint32_t sx, int h, int j) __attribute__((always_inline)) {
        const lds_char* const xf = (h ? xfr1 : xfr0) + sx;
        const lds_char* const wf = (h ? wfr1 : wfr0) + sw;
        if (j < T::NB)
            fx[h][j] = *(const lds_bf16x8*)(xf + j * 16 * kPRow);
        else
            fw[h][j - T::NB] = *(const lds_bf16x8*)(wf + (j - T::NB) * 16 * kPRow);
    };
    // The MFMAs of fragment set h, feature block major, token blocks snaking,
    // with `extra(t)` issued after MFMA t.
    auto mfmas = [&](int h, auto&& extra) __attribute__((always_inline)) {
        static_for<kMfmas>([&](auto tc_) __attribute__((always_inline)) {
            constexpr int t = decltype(tc_)::value, a = t / T::NB, r = t % T::NB, b = (a & 1) ? T::NB - 1 - r : r;
            mfma_acc(acc[a][b], fw[h][a], fx[h][b]);
            extra(tc_);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // n items spread over the first `over` MFMAs: those that follow MFMA t.
    auto spread = [](auto tc_, auto n_c, auto over_c, auto&& item) __attribute__((always_inline)) {
        constexpr int t = decltype(tc_)::value, n = decltype(n_c)::value, over = decltype(over_c)::value;
        constexpr int lo = t < over ? t * n / over : n, hi = t < over ? (t + 1) * n / over : n;
        static_for<hi - lo>([&](auto i) __attribute__((always_inline)) { item(lo + decltype(i)::value); });
    };
    using Reads = std::integral_constant<int, kReads>;
    using LoadsW = std::integral_constant<int, T::kLoadsW>;
    using LoadsX = std::integral_constant<int, T::kLoadsX>;
    using Most = std::integral_constant<int, kMfmas * 3 / 4>;
    using All = std::integral_constant<int, kMfmas>;

    const int nk = p.k / kPK;
    // K step i of W is loaded in the first half of step i + 1 - SW, of X in the
    // second half of step i - SX. Those before step 0 come here, in that order
    // (steps past the end of a short reduction through an empty resource: they
    // load zeros, so that the waits count the same).
    const i32x4 none{0, 0, 0, kBufferWord3};
#pragma unroll
    for (int i = 0; i < SW - 1; ++i) {
        const int ix = i + 1 - SW + SX;
#pragma unroll
        for (int j = 0; j < T::kLoadsW; ++j) dma_w1(i < nk ? rw : none, (uint32_t)(i * T::kWBytes), j);
        advance(rw);
        if (ix < 0) continue;
#pragma unroll
        for (int j = 0; j < T::kLoadsX; ++j) dma_x1(ix < nk ? rx : none, (uint32_t)(ix * T::kXBytes), j);
        advance(rx);
    }
#pragma unroll
    for (int a = 0; a < T::NA; ++a)
#pragma unroll
        for (int b = 0; b < T::NB; ++b) {
            acc[a][b] = f32x4{};
            asm volatile("" : "+a"(acc[a][b]));
        }
    wait_vm_lgkm<(SX - 1) * (T::kLoadsW + T::kLoadsX)>();  // K step 0 (own loads) landed
    barrier();
#pragma unroll
    for (int j = 0; j < kReads; ++j) read1(0, 0, 0, j);

    // K step kt in the stages at `cw` and `cx`, its first-half fragments in set
    // 0. First half: MFMAs of set 0 while set 1 is read from the same stages,
    // and the W rows of step kt+SW-1 go into the W stage before `cw`. Then the
    // wave's own loads of step kt+1 are waited for (later ones stay in flight),
    // with its reads of the stages; after the barrier every wave's part of
    // step kt+1 is in LDS and step kt's stages are no longer read by anyone.
    // Second half: MFMAs of set 1 while step kt+1's first-half fragments are
    // read into set 0 and the X rows of step kt+SX go into `cx`. The loads of a
    // step are thus spread over it (the CU's address path takes 64 bytes a
    // clock, and a lone wave that finds it busy holds up its MFMAs), and W, the
    // operand that comes from HBM, has SW - 1 steps to land.
    // `left` K steps follow; the last steps run out of loads, the last one
    // reads nothing.
    uint32_t cw = 0, pw = (SW - 1) * T::kWBytes, cx = 0;
    int kt = 0;
    auto step = [&](auto left_c) __attribute__((always_inline)) {
        constexpr int left = decltype(left_c)::value;  // SW: that many or more
        constexpr int kAheadW = left - (SW - SX) < SX - 1 ? left - (SW - SX) : SX - 1;
        constexpr int kAheadX = left - 1 < SX - 2 ? left - 1 : SX - 2;
        const uint32_t nw = cw == (SW - 1) * T::kWBytes ? 0u : cw + T::kWBytes;
        const uint32_t nx = cx == (SX - 1) * T::kXBytes ? 0u : cx + T::kXBytes;
        mfmas(0, [&](auto t) __attribute__((always_inline)) {
            spread(t, Reads{}, Most{}, [&](int i) __attribute__((always_inline)) { read1(cw, cx, 1, i); });
            if constexpr (left >= SW - 1)
                spread(t, LoadsW{}, All{}, [&](int i) __attribute__((always_inline)) { dma_w1(rw, pw, i); });
        });
        wait_vm_lgkm<(kAheadW > 0 ? kAheadW : 0) * T::kLoadsW + (kAheadX > 0 ? kAheadX : 0) * T::kLoadsX>();
        barrier();
        mfmas(1, [&](auto t) __attribute__((always_inline)) {
            if constexpr (left > 0)
                spread(t, Reads{}, All{}, [&](int i) __attribute__((always_inline)) { read1(nw, nx, 0, i); });
            if constexpr (left >= SX)
                spread(t, LoadsX{}, Most{}, [&](int i) __attribute__((always_inline)) { dma_x1(rx, cx, i); });
        });
        advance(rw);
        advance(rx);
        pw = cw;
        cw = nw;
        cx = nx;
        ++kt;
    };
    while (kt < nk - SW) step(std::integral_constant<int, SW>{});
    // The last min(SW, nk) steps.
    auto tail = [&](auto self, auto left_c) __attribute__((always_inline)) -> void {
        constexpr int left = decltype(left_c)::value;
        if (left < nk) step(left_c);
        if constexpr (left > 0) self(self, std::integral_constant<int, left - 1>{});
    };
    tail(tail, std::integral_constant<int, SW - 1>{});
    // No load is in flight and no wave reads the stages any more (the last
    // step's barrier followed every wave's last fragment read). The MFMAs are
    // inline asm, outside the compiler's hazard tracking: give the last ones
    // time to write their results before they are read.
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    epilogue<T>(p, tc, acc, wn, wm, tid, smem);
}

template <int TF, int NT, int SW, int SX>
hipError_t launch_tile(ProjGemmParams& p, hipStream_t stream) {
    using T = Tile<TF, NT, SW, SX>;
    p.m_tiles = (p.m + T::kTokens - 1) / T::kTokens;
    p.n_tiles = 0;
    for (int i = 0; i < p.n_sections; ++i) p.n_tiles += p.sec[i].tiles = (p.sec[i].n + TF - 1) / TF;
    // Token tiles of a group: all of a short launch (every W row is then read
    // from HBM once), else about 1,024 tokens, a little less in a long one.
    // 1,296 x 5,120 x 5,120 at 128 tokens a tile: 69.9 us with groups of 2, 63.6
    // with 8, 61.5 with all 11; at 256 tokens and 15,360 x 5,120, 3,000 tokens:
    // 382 (2), 371 (4), 386 (12); 6,240: 742 (1), 698 (2), 697 (4), 739 (16);
    // 49,920: 5,767 (2), 5,751 (3), 5,826 (4), 6,041 (8).
    const int group_tokens = p.m <= 2048 ? 2048 : p.m <= 16384 ? 1024 : 768;
    p.group_m = group_tokens / T::kTokens < p.m_tiles ? group_tokens / T::kTokens : p.m_tiles;
    hipLaunchKernelGGL((proj_gemm_kernel<TF, NT, SW, SX>), dim3((unsigned)(p.m_tiles * p.n_tiles)), dim3(kPThreads), 0, stream, p);
    return hipGetLastError();
}

// The tile shapes, with the time of one K step of 64 when most CUs run one
// (measured: 6,240 x 15,360 x 5,120 q/k/v launches, time per round of tiles
// over 80 steps). Small tiles read more operand bytes per MFMA, so a step costs
// more than its share; they win where larger ones leave CUs idle: a launch of
// few tiles, or a last round that is nearly empty. Below about 128 tokens the
// step time is that of the W rows alone (a CU gets about 60 GB/s from HBM), so
// 128-feature tiles on twice as many CUs win.
struct Shape {
    int tf, nt;
    float step_us;
    hipError_t (*launch)(ProjGemmParams&, hipStream_t);
};
constexpr Shape kShapes[] = {
    {256, 16, 1.33f, launch_tile<256, 16, 3, 2>}, {256, 14, 1.21f, launch_tile<256, 14, 3, 2>},
    {256, 12, 1.07f, launch_tile<256, 12, 3, 2>}, {256, 10, 0.95f, launch_tile<256, 10, 3, 2>},
    {256, 8, 0.78f, launch_tile<256, 8, 4, 2>},   {256, 6, 0.70f, launch_tile<256, 6, 4, 2>},
    {128, 8, 0.49f, launch_tile<128, 8, 6, 4>},   {128, 4, 0.33f, launch_tile<128, 4, 7, 5>},
    {128, 2, 0.27f, launch_tile<128, 2, 8, 6>},
};

// The shape with the least expected time: rounds of tiles over the CUs, times
// a tile's K steps and its start and epilogue. Past three rounds the tiles no
// longer run in step, and the last round costs about half of one.
const Shape& pick_shape(const ProjGemmParams& p, int cus) {
    const Shape* best = &kShapes[0];
    float best_us = 0.f;
    for (const Shape& s : kShapes) {
        int64_t tiles = 0;
        for (int i = 0; i < p.n_sections; ++i) tiles += (p.sec[i].n + s.tf - 1) / s.tf;
        tiles *= (p.m + 16 * s.nt - 1) / (16 * s.nt);
        if (tiles >= ((int64_t)1 << 31)) continue;
        const float r = (float)tiles / (float)cus;
        const float rounds = r > 3.f ? r + 0.5f : ceilf(r);
        const float us = rounds * ((float)(p.k / kPK) * s.step_us + 3.f + (float)(s.nt * s.tf) / 1024.f);
        if (s.nt == 16 || us < best_us) {
            best = &s;
            best_us = us;
        }
    }
    return *best;
}

}  // namespace

hipError_t launch_proj_gemm(ProjGemmParams p, int cus, hipStream_t stream) {
    return pick_shape(p, cus > 0 ? cus : 256).launch(p, stream);
}

int proj_gemm_tile() { return 256; }
int proj_gemm_k_multiple() { return 2 * kPK; }

}  // namespace h3a
