// Reads launches of the many-row GEMM, one a line (split rope scheme rows_of_X
// K part_floats nmat rows...), and prints the shape and the K-slices that
// csrc/wide_shape.h picks for each.
#include "../../wpc-engine_amd/csrc/wide_shape.h"

#include <cstdio>

int main()
{
    int split, rope, scheme, m, k, nmat;
    unsigned long long part;
    while (std::scanf("%d %d %d %d %d %llu %d", &split, &rope, &scheme, &m, &k, &part, &nmat) == 7) {
        int tiles[3] = {}, rows = 0, rows_pad = 0;
        for (int e = 0; e < nmat && e < 3; e++) {
            if (std::scanf("%d", &rows) != 1) return 1;
            tiles[e] = ((rows + 15) / 16 * 16 + 31) / 32;
            if (e == 0) rows_pad = (rows + 15) / 16 * 16;
        }
        const wpcg::WidePick p = wpcg::pick_wide(split, rope, scheme, tiles, nmat, (m + 31) / 32, k / 128,
                                                 (unsigned long long)m * rows_pad, part);
        std::printf("%d %d\n", p.shape, p.kg);
    }
    return 0;
}
