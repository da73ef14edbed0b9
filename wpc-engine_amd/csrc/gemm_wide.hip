// Batched dequant-GEMM Y = X W^T for many rows of X (prompts, large decode
// batches): gemm.hip's arithmetic (the integer codes as the exact bf16
// values 128 + code, each block's scale and zero point in fp32, X as packed
// bf16 or as hi + lo bf16 terms, xpack.h) on v_mfma_f32_32x32x16_bf16.
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
// Measured, us a call, before -> now: 15360 x 3840 v4 at 1024 rows of bf16
// 384 -> 128, 9728 x 2560 v3 at 777 rows SPLIT 541 -> 90.
#include <hip/hip_runtime.h>

#include <algorithm>

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

struct WideArgs {
    const uint8_t* codes;
    const uint8_t* hp;
    const uint32_t* params;
    const u32x4* xf;    // packed X, [nb][xt][4][64] fragments
    const float* xsum;  // [nb][xt*16]
    float* y;           // [M][rows]
    const float* bias;  // [rows] or null
    const float* res;   // [M][rows] added to Y (may be y itself) or null
    int rows, rows_pad, nb, M, xt, rgs, cgs;
};

// eight codes (one byte each, < 128) as the bf16 values 128 + code
__device__ __forceinline__ bf16x8 codes_bf16(uint32_t a, uint32_t b)
{
    u32x4 r;
    r.x = __builtin_amdgcn_perm(0x43434343u, a, 0x04010400u);
    r.y = __builtin_amdgcn_perm(0x43434343u, a, 0x04030402u);
    r.z = __builtin_amdgcn_perm(0x43434343u, b, 0x04010400u);
    r.w = __builtin_amdgcn_perm(0x43434343u, b, 0x04030402u);
    bf16x8 o;
    __builtin_memcpy(&o, &r, 16);
    return o;
}

// Wave (wr, wc, kw) of WR x WC x KW computes 32 weight rows x CT * 32 rows
// of X over the blocks kw, kw + KW, ...: KW > 1 splits K inside the
// workgroup where the outputs alone would leave CUs idle, the K groups'
// sums joining in group order. A round is KW blocks: its X goes through LDS
// (two buffers, one barrier a round), fetched into registers a round ahead,
// the codes straight into registers two rounds ahead.
template <int SCHEME, bool SPLIT, int CT, int WR, int WC, int KW>
__global__ __launch_bounds__(WR * WC * KW * 64, WR * WC * KW == 16 ? 4 : 2) void k_gemm_wide(const WideArgs P)
{
    constexpr int WG = WR * WC * KW * 64;
    constexpr int PARTS = SPLIT ? 2 : 1;
    constexpr int C32 = WC * CT;           // 32-column groups of the workgroup
    constexpr int FW = C32 * PARTS * 512;  // 16-byte X words per block
    constexpr int XV = KW * FW / WG;       // per thread and round
    static_assert(KW * FW % WG == 0, "whole words per thread");
    static_assert((KW - 1) * WR * WC * CT * 256 <= 2 * KW * FW, "the K groups' sums fit the X buffers");
    __shared__ __align__(16) u32x4 xb[2][KW * FW];

    // XCD x (workgroups x, x + 8, ...) takes a contiguous run of tiles, the
    // column groups of one row group next to each other
    const int total = P.rgs * P.cgs, per = (total + 7) / 8;
    const int t = ((int)blockIdx.x & 7) * per + ((int)blockIdx.x >> 3);
    if (t >= total) return;
    const int rg = __builtin_amdgcn_readfirstlane(t / P.cgs), cg = t - rg * P.cgs;  // the division runs on lanes
    const int nb = P.nb, XT = P.xt;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int kw = wave / (WR * WC), wrc = wave % (WR * WC), wr = wrc / WC, wc = wrc % WC;
    const int half = lane >> 5, jj = lane & 31, j = jj & 15;
    const int ntiles = P.rows_pad / TILE_ROWS;
    const int T0 = (rg * WR + wr) * 2;  // the wave's first 16-row tile
    const int live = __builtin_amdgcn_readfirstlane(max(0, min(2, ntiles - T0)));
    const size_t rec0 = (size_t)min(T0, ntiles - 1) * nb;
    const auto crs = buf_rsrc(P.codes + rec0 * CODE_REC, live * nb * (int)CODE_REC);
    const auto hrs = buf_rsrc((SCHEME == 3 ? P.hp : P.codes) + rec0 * HP_REC, SCHEME == 3 ? live * nb * (int)HP_REC : 0);
    const auto prs = buf_rsrc(P.params + rec0 * TILE_ROWS, live * nb * TILE_ROWS * 4);
    const auto xrs = buf_rsrc(P.xf, nb * XT * 4096);
    const auto srs = buf_rsrc(P.xsum, nb * XT * 64);

    // the wave's codes of one block: word ga is lane group g = 2 ga + half of
    // 16-row tile jj / 16
    u32x4 cw[2][2];
    u32x2 hw[2][2];
    uint32_t pw[2];
    const int crec = (jj >> 4) * nb;  // record of block 0
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
            const float sc = h2f(pw[u] >> 16), z = __builtin_fmaf(-128.0f, sc, h2f(pw[u] & 0xFFFFu));
            zo = u == 1 && half == 0 ? zo : z;
            load_par(u, (r + u + 2) * KW + kw);
            const u32x4* xl = &xb[u][kw * FW + wc * CT * PARTS * 512 + lane];
#pragma unroll
            for (int ga = 0; ga < 2; ga++) {
                bf16x8 W[4];
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
                W[0] = codes_bf16(lo.x, lo.y);
                W[1] = codes_bf16(lo.z, lo.w);
                W[2] = codes_bf16(hi.x, hi.y);
                W[3] = codes_bf16(hi.z, hi.w);
                load_word(u, ga, (r + u + 2) * KW + kw);
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int ct = 0; ct < CT; ct++)
#pragma unroll
                        for (int p = 0; p < PARTS; p++) {
                            bf16x8 X;
                            const u32x4 w = xl[((ct * PARTS + p) * 8 + i * 2 + ga) * 64];
                            __builtin_memcpy(&X, &w, 16);
                            D[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(X, W[i], D[ct], 0, 0, 0);
                        }
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
        float* red = reinterpret_cast<float*>(&xb[0][0]);
        if (kw > 0) {
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int q = 0; q < 16; q++)
                    red[((((kw - 1) * WR * WC + wrc) * CT + ct) * 16 + q) * 64 + lane] = acc[ct][q];
        }
        __syncthreads();
        if (kw > 0) return;
#pragma unroll
        for (int k = 1; k < KW; k++)
#pragma unroll
            for (int ct = 0; ct < CT; ct++)
#pragma unroll
                for (int q = 0; q < 16; q++)
                    acc[ct][q] += red[((((k - 1) * WR * WC + wrc) * CT + ct) * 16 + q) * 64 + lane];
    }

    // lane (half, jj) holds weight row jj for the rows 8 (q / 4) + 4 half + q % 4 of X
    const int row = T0 * TILE_ROWS + jj;
    if (row >= P.rows) return;
    const float bias = P.bias ? P.bias[row] : 0.0f;
#pragma unroll
    for (int ct = 0; ct < CT; ct++)
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int m = ((cg * WC + wc) * CT + ct) * 32 + 8 * (q >> 2) + 4 * half + (q & 3);
            if (m >= P.M) continue;
            float v = acc[ct][q];
            if (P.bias) v += bias;
            const size_t at = (size_t)m * P.rows + row;
            if (P.res) v += P.res[at];
            P.y[at] = v;
        }
}


template <int SCHEME, bool SPLIT, int CT, int WR, int WC, int KW>
hipError_t launch_cfg(WideArgs a, hipStream_t s)
{
    const int tiles32 = (a.rows_pad + 31) / 32;
    a.rgs = (tiles32 + WR - 1) / WR;
    a.cgs = ((a.M + 31) / 32 + CT * WC - 1) / (CT * WC);
    const int total = a.rgs * a.cgs;
    hipLaunchKernelGGL((k_gemm_wide<SCHEME, SPLIT, CT, WR, WC, KW>), dim3((unsigned)((total + 7) / 8 * 8)),
                       dim3(WR * WC * KW * 64), 0, s, a);
    return hipGetLastError();
}

// A tile shape: 32-row and 32-column tiles of a workgroup, and what one
// K-block of a round of 256 workgroups takes in hundredths of a microsecond
// (v4, v3), measured over 512..15360 rows, K 768..15360 and 40..1024 rows of
// X; the shape with the fewest rounds x time wins. Large outputs fill the
// chip with the widest tile (15360 x 3840, 1024 rows: 256 x 128 144 us,
// 128 x 64 164, 64 x 32 357), small ones need the narrow, K-split ones
// (3840 x 15360, 128 rows: 64 x 32 37 us, 128 x 64 97, 256 x 128 197).
struct Shape {
    int rows32, cols32;
    int cost[2];
    bool shared;  // workgroups of 8 waves share a CU: the chip fills by fractions of a round
};

int pick(const Shape* sh, int n, int tiles32, int cols32, int scheme)
{
    int best = 0;
    int64_t best_t = INT64_MAX;
    for (int i = 0; i < n; i++) {
        const int64_t wgs = (int64_t)((tiles32 + sh[i].rows32 - 1) / sh[i].rows32) *
                            ((cols32 + sh[i].cols32 - 1) / sh[i].cols32);
        const int64_t c = sh[i].cost[scheme == 3];
        const int64_t t = sh[i].shared ? std::max(c * 4 / 3 * 256, c * (wgs + 128)) : (wgs + 255) / 256 * 256 * c;
        if (t < best_t) {
            best_t = t;
            best = i;
        }
    }
    return best;
}

template <int SCHEME, bool SPLIT>
hipError_t launch_any(const WideArgs& a, uint32_t M, hipStream_t s)
{
    const int tiles32 = (a.rows_pad + 31) / 32, cols32 = (int)((M + 31) / 32);
    if constexpr (!SPLIT) {
        static constexpr Shape sh[] = {{8, 4, {200, 220}, false}, {4, 2, {62, 69}, true}, {4, 2, {70, 80}, false},
                                       {4, 1, {39, 60}, false}, {2, 1, {33, 57}, false}};
        switch (pick(sh, 5, tiles32, cols32, SCHEME)) {
        case 0: return launch_cfg<SCHEME, SPLIT, 2, 8, 2, 1>(a, s);
        case 1: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 1>(a, s);
        case 2: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 2>(a, s);
        case 3: return launch_cfg<SCHEME, SPLIT, 1, 4, 1, 4>(a, s);
        default: return launch_cfg<SCHEME, SPLIT, 1, 2, 1, 8>(a, s);
        }
    } else {
        static constexpr Shape sh[] = {{16, 1, {160, 165}, false}, {4, 2, {110, 118}, true}, {4, 2, {100, 110}, false},
                                       {4, 1, {65, 80}, false}, {8, 1, {88, 105}, false}, {2, 1, {60, 70}, false}};
        switch (pick(sh, 6, tiles32, cols32, SCHEME)) {
        case 0: return launch_cfg<SCHEME, SPLIT, 1, 16, 1, 1>(a, s);
        case 1: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 1>(a, s);
        case 2: return launch_cfg<SCHEME, SPLIT, 1, 4, 2, 2>(a, s);
        case 3: return launch_cfg<SCHEME, SPLIT, 1, 4, 1, 4>(a, s);
        case 4: return launch_cfg<SCHEME, SPLIT, 1, 8, 1, 2>(a, s);
        default: return launch_cfg<SCHEME, SPLIT, 1, 2, 1, 4>(a, s);
        }
    }
}

}  // namespace

hipError_t launch_gemm_wide(const DeviceMatrix& m, void* xf, float* xsum, int tiles, const void* x, int x_mode,
                            uint32_t M, const float* bias, const float* res, float* y, hipStream_t s)
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
        a.codes = m.codes;
        a.hp = m.hp;
        a.params = m.params;
        a.xf = static_cast<const u32x4*>(xf);
        a.xsum = xsum;
        a.y = y + (uint64_t)c * m.rows;
        a.bias = bias;
        a.res = res ? res + (uint64_t)c * m.rows : nullptr;
        a.rows = (int)m.rows;
        a.rows_pad = (int)m.rows_pad;
        a.nb = (int)m.nb;
        a.M = mc;
        a.xt = xt;
        if (split) e = m.scheme == 4 ? launch_any<4, true>(a, M, s) : launch_any<3, true>(a, M, s);
        else e = m.scheme == 4 ? launch_any<4, false>(a, M, s) : launch_any<3, false>(a, M, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace wpcg
