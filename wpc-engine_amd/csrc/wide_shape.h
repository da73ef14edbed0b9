// Which workgroup shape, and how many K-slices, a launch of the many-row
// GEMM (gemm_wide.hip) runs with. Host code only, no HIP: the CPU tests
// compile it to see which shapes the GPU tests reach.
#pragma once

#include <algorithm>
#include <cstdint>

namespace wpcg {

// A tile shape: 32-row and 32-column tiles of a workgroup, and what one
// K-block of a round of 256 workgroups takes in hundredths of a microsecond
// (v4, v3), measured over 512..15360 rows, K 768..15360 and 40..1024 rows of
// X; the shape with the fewest rounds x time wins. Large outputs fill the
// chip with the widest tile (15360 x 3840, 1024 rows: 256 x 128 144 us,
// 128 x 64 164, 64 x 32 357), small ones need the narrow, K-split ones
// (3840 x 15360, 128 rows: 64 x 32 37 us, 128 x 64 97, 256 x 128 197). The
// 16-wave forms are held to 128 registers and some spill, which their costs
// contain (registers spilled, v4 and v3: SPLIT 128 x 64 18 and 21, 64 x 32 8
// and 18). SPLIT 128 x 32 has two K groups in 8 waves: with four in 16 waves,
// whose cost this is, it spilled 10 and 16 and took a tenth to a quarter longer
// wherever it is picked (9728 x 2560 at 33 rows, weights in HBM: v4 22.9 us,
// now 18.3, v3 27.6 and 20.9; gate and up of a 24-token Qwen3-4B-shaped prompt
// 22.7 and 17.2).
struct WideShape {
    int rows32, cols32;
    int cost[2];
    bool shared;  // workgroups of 8 waves share a CU: the chip fills by fractions of a round
    bool slices;  // has a form for K-slices over workgroups
};
constexpr WideShape WIDE_BF16[] = {{8, 4, {200, 220}, false, false}, {4, 2, {62, 69}, true, false},
                                   {4, 2, {70, 80}, false, false},   {4, 1, {39, 60}, false, true},
                                   {2, 1, {33, 57}, false, true}};
// (128 x 64 in 8 waves is not among these: it holds 132-137 registers, so no two
// of them share a CU, and where it was picked it took 5-18 % longer than what is
// picked without it. The last two have no form for the q/k/v epilogue: no whole
// heads, and no launch that would pick it.)
constexpr WideShape WIDE_SPLIT[] = {{16, 1, {160, 165}, false, false},
                                    {4, 1, {65, 80}, false, true},
                                    {8, 1, {88, 105}, false, false},
                                    {2, 1, {60, 70}, false, true},
                                    {4, 2, {100, 110}, false, false}};

// K-slices over workgroups, where the chip has room for all of them at once:
// slices of at least WIDE_SLICE blocks, whose partials cost a second launch
// (k_gemm_reduce, 4.1-4.8 us in a trace, and the gap before it), their way
// through memory, and the start of a short run of blocks (a quarter more a
// block). Up to 256 of the 64 x 32 tiles; us without and with: 512 x 12288 v3,
// 24 tiles, SPLIT 96 rows 43.2 and 24.4; 2560 x 9728 v3, 160, bf16 100 rows
// 31.9 and 25.1, SPLIT 37.5 and 29.4; 3840 x 15360 v3, 180, bf16 65 rows 44.6
// and 34.6, SPLIT 96 rows 49.4 and 43.8.
constexpr int WIDE_SLICE = 8;
constexpr int64_t WIDE_REDUCE = 550;            // hundredths of a microsecond
constexpr int64_t WIDE_PART_FLOATS = 5000;      // partial sums written and read in one of those

struct WidePick {
    int shape, kg;
};

// tiles32: 32-row tiles of each of the nmat matrices; cols32: 32-row tiles of
// X; nb: K-blocks; outs: outputs (rows of X times padded weight rows), whose
// partials must fit part_floats (0: no slices).
// rope (SPLIT only): with the q/k/v epilogue.
inline WidePick pick_wide(bool split, bool rope, int scheme, const int* tiles32, int nmat, int cols32, int nb,
                          uint64_t outs, uint64_t part_floats)
{
    const WideShape* sh = split ? WIDE_SPLIT : WIDE_BF16;
    const int n = rope ? 3 : 5;
    int64_t small = 0;  // 64 x 32 tiles
    for (int e = 0; e < nmat; e++) small += (int64_t)((tiles32[e] + 1) / 2) * cols32;
    const int most = rope || nmat > 1 || small > 256
                         ? 1
                         : (int)std::min<uint64_t>(part_floats / std::max<uint64_t>(outs, 1),
                                                                     (uint64_t)std::max(nb / WIDE_SLICE, 1));
    WidePick best{0, 1};
    int64_t best_t = INT64_MAX;
    for (int i = 0; i < n; i++) {
        int64_t wgs = 0;
        for (int e = 0; e < nmat; e++) wgs += (tiles32[e] + sh[i].rows32 - 1) / sh[i].rows32;
        wgs *= (cols32 + sh[i].cols32 - 1) / sh[i].cols32;
        const int64_t c = sh[i].cost[scheme == 3];
        for (int k = 1; k == 1 || (sh[i].slices && k <= most && k * wgs <= 256); k++) {
            const int nbk = (nb + k - 1) / k;
            if ((nb + nbk - 1) / nbk != k) continue;  // an empty slice: the same as fewer
            const int64_t w = wgs * k;
            const int64_t round = sh[i].shared ? std::max(c * 4 / 3 * 256, c * (w + 128)) : (w + 255) / 256 * 256 * c;
            const int64_t t = k == 1 ? round * nbk
                                     : round * nbk * 5 / 4 + 256 * (WIDE_REDUCE + k * (int64_t)outs / WIDE_PART_FLOATS);
            if (t < best_t) {
                best_t = t;
                best = {i, k};
            }
        }
    }
    return best;
}

}  // namespace wpcg
