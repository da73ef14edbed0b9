// Batched dequant-GEMM Y = X W^T for many rows of X (prompts, large decode
// batches): gemm.hip's arithmetic (the integer codes exact in bf16, each
// block's scale and zero point in fp32, X as packed bf16 or as hi + lo bf16
// terms, xpack.h) on v_mfma_f32_32x32x16_bf16. It serves wpcg_linear_gemm
// above 64 rows of X and every projection of the prefill.
//
// k_gemm re-unpacks a matrix's codes for every 64 (SPLIT: 32) rows of X and
// pays a pack and a reduce launch for each; here one launch covers every
// row, a workgroup of up to 16 waves up to 256 x 128 outputs. X is the first
// operand and the weights the second, so a lane holds 16 rows of X of ONE
// weight row: one scale a lane and block instead of one per output, and
// stores of whole 128-byte runs. The zero points of a pair of blocks are one fp32
// v_mfma_f32_32x32x2_f32 (k = the two blocks).
//
// What bounds it: the matrix cores under this load. A timing copy with
// nothing but the products and the barriers ran 112 us where the whole ran
// 150 (15360 x 3840 matrix, 1024 rows of bf16; a plain library product of
// 8192^3 reaches 1.2 PFLOP/s on the same card); the code unpack (28 vector
// instructions per 32 codes) and the scale (16 per 32 x 32 x 128 products)
// are most of the rest. Hence 16 waves of small tiles (four a
// SIMD), whose vector work hides under the other waves' products: 8 waves
// of 64 x 64 outputs each took 158-171 us, two groups of waves alternating
// between vector and matrix phases 160-197.
//
// Measured, us a call, before -> now (two cards): 15360 x 3840 v4 at 1024 rows
// of bf16 383-396 -> 128-135, 9728 x 2560 v3 at 777 rows SPLIT 541 -> 84-91;
// in the prefill (Qwen3-4B shape, 1000 tokens, per layer) gate and up 350 ->
// 208, q/k/v 142 -> 76, o and down 310 -> 200.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "wide_shape.h"
#include "wpcg_internal.hpp"
#include "xpack.h"

namespace wpcg {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float h2f(uint32_t bits)
{
    _Float16 h;
    uint16_t b = (uint16_t)bits;
    __builtin_memcpy(&h, &b, 2);
    return (float)h;
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void* base, int bytes)
{
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, bytes, 0x00020000);
}
constexpr int PAST = 1 << 30;  // added to a buffer offset: past every range, reads zero (ranges are shorter)

// One matrix of a launch: its tiles (times kg slices) start at t0.
struct WideMat {
    const uint8_t* codes;
    const uint8_t* hp;
    const uint32_t* params;
    float* y;           // [M][rows]
    const float* bias;  // [rows] or null
    int rows, rows_pad, rgs, t0;
    int rope;         // GEMM_ROPE_*: the prefill's q, k or v epilogue
    float* cache;     // k, v: the layer's cache [head][max_pos][128]
    const float* nw;  // q, k: the head norm's weights [128]
};
constexpr int WIDE_MATS = sizeof(GemmRope::mode) / sizeof(int);
struct WideArgs {
    WideMat mat[WIDE_MATS];
    const u32x4* xf;    // packed X, [nb][xt][4][64] fragments
    const float* xsum;  // [nb][xt*16]
    const float* res;   // [M][rows] added to Y (may be y itself) or null (one matrix only)
    float* part;        // kg > 1: [kg][M][rows_pad] sums of the K-slices (one matrix only)
    int nmat, nb, M, xt, cgs, total, kg, nbk;  // nbk: blocks of a slice
    // rope: the rotation tables and positions of the rows of X
    const float* cos_t;  // [max_pos][64]
    const float* sin_t;
    int pos0, max_pos;
    float eps;
};

// Eight codes, one byte each, as bf16. v4: a byte 0..15 is the fp8 (e4m3)
// number code * 2^-9 (subnormal below 8), so the fp8 conversion scaled by
// 2^9 gives the code itself, two an instruction, and the sums carry no
// offset (15360 x 3840 at 1024 rows of bf16: error against float64 1.6e-6
// with 128 + code, 1.5e-7 with the codes, at the same time). v3 (codes to 63): 128 +
// code, whose bit patterns are 0x4300 | code, one byte permute for two; the
// products are then D + 128 S and the zero point zp - 128 scale.
constexpr float code_offset(int scheme) { return scheme == 4 ? 0.0f : 128.0f; }
template <int SCHEME>
__device__ __forceinline__ bf16x8 codes_bf16(uint32_t a, uint32_t b)
{
    bf16x8 o;
    if constexpr (SCHEME == 4) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        const bf16x2 r[4] = {__builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 512.0f, false),
                             __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(a, 512.0f, true),
                             __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 512.0f, false),
                             __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(b, 512.0f, true)};
        __builtin_memcpy(&o, r, 16);
    } else {
        u32x4 r;
        r.x = __builtin_amdgcn_perm(0x43434343u, a, 0x04010400u);
        r.y = __builtin_amdgcn_perm(0x43434343u, a, 0x04030402u);
        r.z = __builtin_amdgcn_perm(0x43434343u, b, 0x04010400u);
        r.w = __builtin_amdgcn_perm(0x43434343u, b, 0x04030402u);
        __builtin_memcpy(&o, &r, 16);
    }
    return o;
}

// Wave (wr, wc, kw) of WR x WC x KW computes 32 weight rows x CT * 32 rows
// of X over the blocks kw, kw + KW, ...: KW > 1 splits K inside the
// workgroup where the outputs alone would leave CUs idle, the K groups'
// sums joining in group order. A round is KW blocks: its X goes through LDS
// (two buffers, one barrier a round), fetched into registers a round ahead,
// the codes straight into registers two rounds ahead.
//
// KS also splits K over kg workgroups, where even so there are too few (2560
// weight rows and 24 rows of X are 40 workgroups of the smallest shape): each
// takes a run of blocks and leaves its sums in part, which the next launch
// (launch_gemm_reduce) adds in slice order: o_proj and down of a 24-token
// Qwen3-4B-shaped prompt 51.6 us together without slices, 20.1 and 8.2 for the
// reduces with them; 512 x 12288 at 33 rows SPLIT 39.6 -> 23.7 us a call. (A
// form of its own: with the slice in the other launches too, the small v3
// ones were 1 us slower.)
//
// ROPE (the prefill's q, k and v; WR % 4 == 0): four row tiles are one
// 128-wide head. The sums go to LDS as [token][d], and 16 threads take a
// token of a head: the head RMSNorm (FAST: squares by fused multiply-adds,
// then exchanges), (x * scale) * w, the rotation at the token's position
// (d < 64 and d + 64 are a pair: y c - y' s and y' c + y s), q into Y, k
// and v (v as computed) into the cache rows, all as 16-byte pieces.
template <int SCHEME, bool SPLIT, int CT, int WR, int WC, int KW, bool ROPE, bool KS>
__global__ __launch_bounds__(WR * WC * KW * 64, WR * WC * KW == 16 ? 4 : 2) void k_gemm_wide(const WideArgs P0)
{
    constexpr int WG = WR * WC * KW * 64;
    constexpr int PARTS = SPLIT ? 2 : 1;
    constexpr int C32 = WC * CT;           // 32-column groups of the workgroup
    constexpr int FW = C32 * PARTS * 512;  // 16-byte X words per block
    constexpr int XV = KW * FW / WG;       // per thread and round
    static_assert(KW * FW % WG == 0, "whole words per thread");
    static_assert((KW - 1) * WR * WC * CT * 256 <= 2 * KW * FW, "the K groups' sums fit the X buffers");
    static_assert(!ROPE || (WR % 4 == 0 && CT == 1), "whole heads");
    constexpr int HS = 132;                      // floats per token of a head's stage
    constexpr int HW = ROPE ? 32 * HS / 4 : 0;   // 16-byte words per (head, column group)
    constexpr int XW = 2 * KW * FW > WR / 4 * C32 * HW ? 2 * KW * FW : WR / 4 * C32 * HW;
    __shared__ __align__(16) u32x4 xw[XW];
    u32x4* const xb[2] = {xw, xw + KW * FW};

    // XCD x (workgroups x, x + 8, ...) takes a contiguous run of tiles, the
    // column groups of one row group next to each other
    const int per = (P0.total + 7) / 8;
    const int t = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (t >= P0.total) return;
    int e = 0;
    for (int i = 1; i < P0.nmat; i++) e = t >= P0.mat[i].t0 ? i : e;
    const WideMat P = P0.mat[e];
    const int tl = t - P.t0;
    const int rk = __builtin_amdgcn_readfirstlane(tl / P0.cgs), cg = tl - rk * P0.cgs;  // the division runs on lanes
    const int rg = KS ? __builtin_amdgcn_readfirstlane(rk / P0.kg) : rk, ks = KS ? rk - rg * P0.kg : 0;
    const int nbt = P0.nb, XT = P0.xt;
    const int b0 = KS ? ks * P0.nbk : 0, nb = KS ? min(P0.nbk, nbt - b0) : nbt;  // the slice (none is empty)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int kw = wave / (WR * WC), wrc = wave % (WR * WC), wr = wrc / WC, wc = wrc % WC;
    const int half = lane >> 5, jj = lane & 31, j = jj & 15;
    const int ntiles = P.rows_pad / TILE_ROWS;
    const int T0 = (rg * WR + wr) * 2;  // the wave's first 16-row tile
    const int live = __builtin_amdgcn_readfirstlane(max(0, min(2, ntiles - T0)));
    // (every range starts at the slice's first block and ends with the second tile's slice)
    const size_t rec0 = (size_t)min(T0, ntiles - 1) * nbt + b0;
    const int recs = !KS ? live * nb : live ? (live - 1) * nbt + nb : 0;
    const auto crs = buf_rsrc(P.codes + rec0 * CODE_REC, recs * (int)CODE_REC);
    const auto hrs = buf_rsrc((SCHEME == 3 ? P.hp : P.codes) + rec0 * HP_REC, SCHEME == 3 ? recs * (int)HP_REC : 0);
    const auto prs = buf_rsrc(P.params + rec0 * TILE_ROWS, recs * TILE_ROWS * 4);
    const auto xrs = buf_rsrc(P0.xf + (size_t)b0 * XT * 256, nb * XT * 4096);
    const auto srs = buf_rsrc(P0.xsum + (size_t)b0 * XT * 16, nb * XT * 64);

    // the wave's codes of one block: word ga is lane group g = 2 ga + half of
    // 16-row tile jj / 16
    u32x4 cw[2][2];
    u32x2 hw[2][2];
    uint32_t pw[2];
    const int crec = (jj >> 4) * nbt;  // record of block 0
    auto load_word = [&](int u, int ga, int b) {
        const int past = b < nb ? 0 : PAST;
        cw[u][ga] = __builtin_amdgcn_raw_buffer_load_b128(
            crs, crec * (int)CODE_REC + half * 256 + j * 16 + (b * (int)CODE_REC + past) + ga * 512, 0, 0);
        if constexpr (SCHEME == 3)
            hw[u][ga] = __builtin_amdgcn_raw_buffer_load_b64(
                hrs, crec * (int)HP_REC + half * 128 + j * 8 + (b * (int)HP_REC + past) + ga * 256, 0, 0);
    };
    auto load_par = [&](int u, int b) {
        pw[u] = __builtin_amdgcn_raw_buffer_load_b32(prs, crec * 64 + j * 4 + (b * 64 + (b < nb ? 0 : PAST)), 0, 0);
    };
    const int xbase = cg * C32 * 2 * PARTS;  // the workgroup's first 16-column tile
    u32x4 xr[XV];
    auto load_x = [&](int r) {
#pragma unroll
        for (int v = 0; v < XV; v++) {
            // (the block of a word is the same for a whole wave)
            const int w = (int)threadIdx.x + v * WG, b = r * KW + __builtin_amdgcn_readfirstlane(w / FW);
            xr[v] = __builtin_amdgcn_raw_buffer_load_b128(
                xrs, w % FW * 16 + ((b * XT + xbase) * 4096 + (b < nb ? 0 : PAST)), 0, 0);
        }
    };
    // a fragment's words in the lane order of the 32-wide operand: word
    // (tile, i, lane group g, column c) goes to fragment (tile / 2, i, g / 2),
    // lane (g % 2) * 32 + (tile % 2) * 16 + c
    auto store_x = [&](int buf) {
#pragma unroll
        for (int v = 0; v < XV; v++) {
            const int w = (int)threadIdx.x + v * WG, f = w % FW;
            const int tile = f >> 8, i = (f >> 6) & 3, l = f & 63;
            xb[buf][w / FW * FW + (((tile >> 1) * 4 + i) * 2 + (l >> 5)) * 64 + ((l >> 4) & 1) * 32 + (tile & 1) * 16 +
                    (l & 15)] = xr[v];
        }
    };
    float sx[CT];  // block sums: lane half h holds the pair's block h
    auto load_sums = [&](int r) {
#pragma unroll
        for (int ct = 0; ct < CT; ct++) {
            const int b = (r + half) * KW + kw, tile = xbase + (wc * CT + ct) * 2 * PARTS + (jj >> 4);
            const int o = (b * XT + tile) * 64 + j * 4 + (b < nb ? 0 : PAST);
            float s = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, o, 0, 0));
            if constexpr (SPLIT) s += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(srs, o + 128, 0, 0));
            sx[ct] = s;
        }
    };

    f32x16 acc[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int q = 0; q < 16; q++) acc[ct][q] = 0.0f;

    load_x(0);
#pragma unroll
    for (int u = 0; u < 2; u++) {
        load_word(u, 0, u * KW + kw);
        load_word(u, 1, u * KW + kw);
        load_par(u, u * KW + kw);
    }
    store_x(0);
    load_x(1);
    __syncthreads();

    const int rounds = (nb + KW - 1) / KW;
    for (int r = 0; r < rounds; r += 2) {
        load_sums(r);
        float zo;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            store_x(u ^ 1);
            load_x(r + u + 2);
            f32x16 D[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int q = 0; q < 16; q++) D[ct][q] = 0.0f;
            const float sc = h2f(pw[u] >> 16), z = __builtin_fmaf(-code_offset(SCHEME), sc, h2f(pw[u] & 0xFFFFu));
            zo = u == 1 && half == 0 ? zo : z;
            load_par(u, (r + u + 2) * KW + kw);
            const u32x4* xl = &xb[u][kw * FW + wc * CT * PARTS * 512 + lane];
            bf16x8 W[2][4];
            auto unpack = [&](int ga) {
                const u32x4 U = cw[u][ga];
                const uint32_t MK = 0x0F0F0F0Fu;
                u32x4 lo = {U.x & MK, U.y & MK, U.z & MK, U.w & MK};
                u32x4 hi = {(U.x >> 4) & MK, (U.y >> 4) & MK, (U.z >> 4) & MK, (U.w >> 4) & MK};
                if constexpr (SCHEME == 3) {
                    const uint32_t T6 = 0x30303030u, hx = hw[u][ga].x, hy = hw[u][ga].y;
                    lo.x |= (hx << 4) & T6; lo.y |= (hx << 2) & T6;
                    lo.z |= (hy << 4) & T6; lo.w |= (hy << 2) & T6;
                    hi.x |= hx & T6;        hi.y |= (hx >> 2) & T6;
                    hi.z |= hy & T6;        hi.w |= (hy >> 2) & T6;
                }
                W[ga][0] = codes_bf16<SCHEME>(lo.x, lo.y);
                W[ga][1] = codes_bf16<SCHEME>(lo.z, lo.w);
                W[ga][2] = codes_bf16<SCHEME>(hi.x, hi.y);
                W[ga][3] = codes_bf16<SCHEME>(hi.z, hi.w);
                load_word(u, ga, (r + u + 2) * KW + kw);
            };
            // part p of X against the codes of word ga. The lo terms of SPLIT
            // go first: their sums are 2^-9 of the hi terms', so only the hi
            // terms' products are rounded at full size.
            auto products = [&](int p, int ga) {
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int ct = 0; ct < CT; ct++) {
                        bf16x8 X;
                        const u32x4 w = xl[((ct * PARTS + p) * 8 + i * 2 + ga) * 64];
                        __builtin_memcpy(&X, &w, 16);
                        D[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X, W[ga][i], D[ct], 0, 0, 0);
                    }
            };
            unpack(0);
            products(PARTS - 1, 0);
            unpack(1);
            products(PARTS - 1, 1);
            if constexpr (SPLIT) {
                products(0, 0);
                products(0, 1);
            }
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int q = 0; q < 16; q++) acc[ct][q] = __builtin_fmaf(sc, D[ct][q], acc[ct][q]);
            __syncthreads();
        }
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
            acc[ct] = __builtin_amdgcn_mfma_f32_32x32x2f32(sx[ct], zo, acc[ct], 0, 0, 0);
    }

    // the K groups' sums, in group order
    if constexpr (KW > 1) {
        float* red = reinterpret_cast<float*>(xw);
        if (kw > 0) {
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int q = 0; q < 16; q++)
                    red[((((kw - 1) * WR * WC + wrc) * CT + ct) * 16 + q) * 64 + lane] = acc[ct][q];
        }
        __syncthreads();
        if (!ROPE && kw > 0) return;
        if (kw == 0) {
#pragma unroll
            for (int k = 1; k < KW; k++)
#pragma unroll
                for (int ct = 0; ct < CT; ct++)
#pragma unroll
                    for (int q = 0; q < 16; q++)
                        acc[ct][q] += red[((((k - 1) * WR * WC + wrc) * CT + ct) * 16 + q) * 64 + lane];
        }
    }

    // lane (half, jj) holds weight row jj for the rows 8 (q / 4) + 4 half + q % 4 of X
    const int row = T0 * TILE_ROWS + jj;
    if constexpr (ROPE) {
        float* ex = reinterpret_cast<float*>(xw);
        if constexpr (KW > 1) __syncthreads();  // the K groups' sums are read
        if (kw == 0) {
            const float bias = P.bias && row < P.rows ? P.bias[row] : 0.0f;
#pragma unroll
            for (int q = 0; q < 16; q++)
                ex[((wr / 4 * C32 + wc) * 32 + 8 * (q >> 2) + 4 * half + (q & 3)) * HS + (wr & 3) * 32 + jj] =
                    acc[0][q] + bias;
        }
        __syncthreads();
        const int d1 = 4 * (threadIdx.x & 15);
        for (int i = (int)threadIdx.x >> 4; i < WR / 4 * C32 * 32; i += WG / 16) {
            const int hd = i / (C32 * 32), tok = i % (C32 * 32);
            const int m = cg * C32 * 32 + tok, head = rg * (WR / 4) + hd;
            const float4 y1 = *reinterpret_cast<const float4*>(&ex[i * HS + d1]);
            const float4 y2 = *reinterpret_cast<const float4*>(&ex[i * HS + d1 + 64]);
            float4 o1 = y1, o2 = y2;
            // (the sixteen lanes of a token are all live: their exchanges are whole)
            if (P.rope != GEMM_ROPE_V) {
                float ss = fmaf(y1.w, y1.w, fmaf(y1.z, y1.z, fmaf(y1.y, y1.y, y1.x * y1.x)));
                ss = fmaf(y2.w, y2.w, fmaf(y2.z, y2.z, fmaf(y2.y, y2.y, fmaf(y2.x, y2.x, ss))));
                ss += __shfl_xor(ss, 1);
                ss += __shfl_xor(ss, 2);
                ss += __shfl_xor(ss, 4);
                ss += __shfl_xor(ss, 8);
                const float sc = __fdiv_rn(1.0f, __builtin_sqrtf(__fadd_rn(__fdiv_rn(ss, 128.0f), P0.eps)));
                const int pos = min(P0.pos0 + m, P0.max_pos - 1);
                const float4 w1 = *reinterpret_cast<const float4*>(P.nw + d1);
                const float4 w2 = *reinterpret_cast<const float4*>(P.nw + d1 + 64);
                const float4 c = *reinterpret_cast<const float4*>(P0.cos_t + (size_t)pos * 64 + d1);
                const float4 sn = *reinterpret_cast<const float4*>(P0.sin_t + (size_t)pos * 64 + d1);
                const float4 n1 = make_float4((y1.x * sc) * w1.x, (y1.y * sc) * w1.y, (y1.z * sc) * w1.z, (y1.w * sc) * w1.w);
                const float4 n2 = make_float4((y2.x * sc) * w2.x, (y2.y * sc) * w2.y, (y2.z * sc) * w2.z, (y2.w * sc) * w2.w);
                o1 = make_float4(fmaf(n1.x, c.x, -(n2.x * sn.x)), fmaf(n1.y, c.y, -(n2.y * sn.y)),
                                 fmaf(n1.z, c.z, -(n2.z * sn.z)), fmaf(n1.w, c.w, -(n2.w * sn.w)));
                o2 = make_float4(fmaf(n2.x, c.x, n1.x * sn.x), fmaf(n2.y, c.y, n1.y * sn.y),
                                 fmaf(n2.z, c.z, n1.z * sn.z), fmaf(n2.w, c.w, n1.w * sn.w));
            }
            if (m < P0.M && head * 128 < P.rows) {
                float* dst = P.rope == GEMM_ROPE_Q ? P.y + (size_t)m * P.rows + head * 128
                                                   : P.cache + ((size_t)head * P0.max_pos + P0.pos0 + m) * 128;
                *reinterpret_cast<float4*>(dst + d1) = o1;
                *reinterpret_cast<float4*>(dst + d1 + 64) = o2;
            }
        }
        return;
    }
    if constexpr (KS) {
        if (row >= P.rows_pad) return;
#pragma unroll
        for (int ct = 0; ct < CT; ct++)
#pragma unroll
            for (int q = 0; q < 16; q++) {
                const int m = ((cg * WC + wc) * CT + ct) * 32 + 8 * (q >> 2) + 4 * half + (q & 3);
                if (m < P0.M) P0.part[((size_t)ks * P0.M + m) * P.rows_pad + row] = acc[ct][q];
            }
        return;
    }
    if (row >= P.rows) return;
    const float bias = P.bias ? P.bias[row] : 0.0f;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int m = ((cg * WC + wc) * CT + ct) * 32 + 8 * (q >> 2) + 4 * half + (q & 3);
            if (m >= P0.M) continue;
            float v = acc[ct][q];
            if (P.bias) v += bias;
            const size_t at = (size_t)m * P.rows + row;
            if (P0.res) v += P0.res[at];
            P.y[at] = v;
        }
}


template <int SCHEME, bool SPLIT, int CT, int WR, int WC, int KW, bool ROPE = false, bool KS = false>
hipError_t launch_cfg(WideArgs a, hipStream_t s)
{
    a.cgs = ((a.M + 31) / 32 + CT * WC - 1) / (CT * WC);
    a.total = 0;
    for (int e = 0; e < a.nmat; e++) {
        WideMat& m = a.mat[e];
        m.rgs = ((m.rows_pad + 31) / 32 + WR - 1) / WR;
        m.t0 = a.total;
        a.total += m.rgs * a.cgs * a.kg;
    }
    hipLaunchKernelGGL((k_gemm_wide<SCHEME, SPLIT, CT, WR, WC, KW, ROPE, KS>), dim3((unsigned)((a.total + 7) / 8 * 8)),
                       dim3(WR * WC * KW * 64), 0, s, a);
    return hipGetLastError();
}

// M: the rows of X that pick the shape (the whole batch of a pass); part
// holds part_floats, for K-slices
template <int SCHEME, bool SPLIT>
hipError_t launch_any(WideArgs& a, uint32_t M, bool rope, float* part, uint64_t part_floats, hipStream_t s)
{
    int tiles32[WIDE_MATS] = {};
    for (int e = 0; e < a.nmat; e++) tiles32[e] = (a.mat[e].rows_pad + 31) / 32;
    const WidePick p = pick_wide(SPLIT, rope, SCHEME, tiles32, a.nmat, (int)((M + 31) / 32), a.nb,
                                 (uint64_t)M * a.mat[0].rows_pad, part ? part_floats : 0);
    a.kg = p.kg;
    a.nbk = (a.nb + p.kg - 1) / p.kg;
    a.part = part;
    if (p.kg > 1) {  // (pick_wide slices these two only)
        if constexpr (!SPLIT)
            return p.shape == 3 ? launch_cfg<SCHEME, SPLIT, 1, 4, 1, 4, false, true>(a, s)
                                : launch_cfg<SCHEME, SPLIT, 1, 2, 1, 8, false, true>(a, s);
        else
            return p.shape == 1 ? launch_cfg<SCHEME, SPLIT, 1, 4, 1, 2, false, true>(a, s)
                                : launch_cfg<SCHEME, SPLIT, 1, 2, 1, 4, false, true>(a, s);
    }
    if constexpr (!SPLIT) {
        switch (p.shape) {
        case 0: return launch_cfg<SCHEME, SPLIT, 2, 8, 2, 1>(a, s);
        case 1: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 1>(a, s);
        case 2: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 2>(a, s);
        case 3: return launch_cfg<SCHEME, SPLIT, 1, 4, 1, 4>(a, s);
        default: return launch_cfg<SCHEME, SPLIT, 1, 2, 1, 8>(a, s);
        }
    } else {
        if (rope) {
            switch (p.shape) {
            case 0: return launch_cfg<SCHEME, SPLIT, 1, 16, 1, 1, true>(a, s);
            case 1: return launch_cfg<SCHEME, SPLIT, 1, 4, 1, 2, true>(a, s);
            default: return launch_cfg<SCHEME, SPLIT, 1, 8, 1, 2, true>(a, s);
            }
        }
        switch (p.shape) {
        case 0: return launch_cfg<SCHEME, SPLIT, 1, 16, 1, 1>(a, s);
        case 1: return launch_cfg<SCHEME, SPLIT, 1, 4, 1, 2>(a, s);
        case 2: return launch_cfg<SCHEME, SPLIT, 1, 8, 1, 2>(a, s);
        case 3: return launch_cfg<SCHEME, SPLIT, 1, 2, 1, 4>(a, s);
        default: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 2>(a, s);
        }
    }
}

// The slices' sums, the bias and the residual into Y, where there are slices
hipError_t finish(const WideArgs& a, hipStream_t s)
{
    const WideMat& m = a.mat[0];
    if (a.kg == 1) return hipSuccess;
    return launch_gemm_reduce(a.part, a.kg, a.M, m.rows_pad, m.rows, a.M, m.bias, a.res, m.y, s);
}

WideMat wide_mat(const DeviceMatrix& m, const float* bias, float* y)
{
    WideMat w{};
    w.codes = m.codes;
    w.hp = m.hp;
    w.params = m.params;
    w.y = y;
    w.bias = bias;
    w.rows = (int)m.rows;
    w.rows_pad = (int)m.rows_pad;
    return w;
}

}  // namespace

hipError_t launch_gemm_wide(const DeviceMatrix& m, void* xf, float* xsum, int tiles, const void* x, int x_mode,
                            uint32_t M, const float* bias, float* y, float* part, uint64_t part_floats, hipStream_t s)
{
    const bool split = x_mode == GX_SPLIT;
    // (the shape is picked from the whole batch, so that the order of an
    // output's sum does not depend on the passes)
    const uint32_t cap = (uint32_t)gemm_wide_cols(x_mode, tiles);
    if (M < 1 || m.nb == 0 || cap < 1 || m.nb * (uint64_t)tiles * 4096 >= (uint64_t)PAST) return hipErrorInvalidValue;
    const uint64_t es = x_mode == GX_BF16 ? 2 : 4;
    for (uint32_t c = 0; c < M; c += cap) {
        const int mc = (int)std::min(cap, M - c);
        const int xt = split ? gemm_rows_tiles(mc) : (mc + 31) / 32 * 2;
        hipError_t e = launch_gemm_pack(static_cast<const uint8_t*>(x) + (uint64_t)c * m.cols * es, x_mode, mc,
                                        (int)m.cols, xt, split ? 4 : xt, xf, xsum, s);
        if (e != hipSuccess) return e;
        WideArgs a{};
        a.mat[0] = wide_mat(m, bias, y + (uint64_t)c * m.rows);
        a.nmat = 1;
        a.xf = static_cast<const u32x4*>(xf);
        a.xsum = xsum;
        a.nb = (int)m.nb;
        a.M = mc;
        a.xt = xt;
        if (split) e = m.scheme == 4 ? launch_any<4, true>(a, M, false, part, part_floats, s)
                                     : launch_any<3, true>(a, M, false, part, part_floats, s);
        else e = m.scheme == 4 ? launch_any<4, false>(a, M, false, part, part_floats, s)
                               : launch_any<3, false>(a, M, false, part, part_floats, s);
        if (e == hipSuccess) e = finish(a, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_gemm_packed_rows(const DeviceMatrix* const* ms, const float* const* biases, float* const* ys,
                                   int count, const void* xf, const float* xsum, int M, const float* res,
                                   hipStream_t s, const GemmRope* rope, float* part, uint64_t part_floats)
{
    if (M < 1 || count < 1 || count > WIDE_MATS || (res && count > 1)) return hipErrorInvalidValue;
    if (ms[0]->nb * (uint64_t)gemm_rows_tiles(M) * 4096 >= (uint64_t)PAST) return hipErrorInvalidValue;
    WideArgs a{};
    for (int e = 0; e < count; e++) {
        if (ms[e]->nb == 0 || ms[e]->nb != ms[0]->nb || ms[e]->scheme != ms[0]->scheme) return hipErrorInvalidValue;
        a.mat[e] = wide_mat(*ms[e], biases[e], ys[e]);
        if (!rope) continue;
        // whole 128-row heads; q and k have norm weights, k and v a cache
        const int md = rope->mode[e];
        if (md < GEMM_ROPE_Q || md > GEMM_ROPE_V || ms[e]->rows % 128 || (md != GEMM_ROPE_V && !rope->nw[e]) ||
            (md != GEMM_ROPE_Q && !rope->cache[e]))
            return hipErrorInvalidValue;
        a.mat[e].rope = md;
        a.mat[e].cache = rope->cache[e];
        a.mat[e].nw = rope->nw[e];
    }
    if (rope) {
        if (!rope->cos_t || !rope->sin_t || rope->pos0 < 0 || rope->pos0 + M > rope->max_pos)
            return hipErrorInvalidValue;
        a.cos_t = rope->cos_t;
        a.sin_t = rope->sin_t;
        a.pos0 = rope->pos0;
        a.max_pos = rope->max_pos;
        a.eps = rope->eps;
    }
    (void)hipGetLastError();
    a.nmat = count;
    a.xf = static_cast<const u32x4*>(xf);
    a.xsum = xsum;
    a.res = res;
    a.nb = (int)ms[0]->nb;
    a.M = M;
    a.xt = gemm_rows_tiles(M);
    const hipError_t e = ms[0]->scheme == 4 ? launch_any<4, true>(a, (uint32_t)M, rope != nullptr, part, part_floats, s)
                                            : launch_any<3, true>(a, (uint32_t)M, rope != nullptr, part, part_floats, s);
    return e == hipSuccess ? finish(a, s) : e;
}

}  // namespace wpcg
