/*
 * rows_shape.h - the block shapes of rows_gemm_kernel and the choice between them (host only).
 */
#ifndef W4A16_ROWS_SHAPE_H
#define W4A16_ROWS_SHAPE_H

#include <algorithm>

namespace w4a16 {

struct RowsShape {
    int rows, tile_pairs, groups; /* a block's rows / 16 and tile pairs, groups a step */
    float base, first, more;      /* us */
};

constexpr RowsShape kRowsShapes[] = {
    {1, 1, 16, 6.02f, 0.60f, 2.11f}, {1, 2, 8, 4.05f, 0.77f, 1.33f},  {1, 3, 8, 4.40f, 0.89f, 1.55f},
    {1, 4, 4, 3.62f, 0.63f, 0.65f},  {1, 6, 4, 4.13f, 0.80f, 1.18f},  {1, 8, 4, 4.18f, 0.98f, 1.42f},
    {1, 10, 2, 4.13f, 0.65f, 0.85f}, {2, 4, 4, 4.13f, 0.94f, 1.34f},  {2, 6, 4, 5.07f, 1.09f, 1.77f},
    {2, 9, 4, 6.50f, 1.45f, 2.33f},  {2, 10, 2, 5.46f, 0.94f, 1.31f}, {2, 6, 2, 4.85f, 0.74f, 0.64f},
    {4, 10, 2, 6.89f, 1.67f, 2.32f},
};

/* The index of the shape whose estimated time for M rows of N x K is least: base + steps * (first + more *
 * (rounds - 1)), with steps = ceil(groups / groups a step) and rounds the blocks of the fullest CU, counted on
 * the fullest XCD (column blocks go round the eight XCDs, a column block's row slices stay on one).
 * A shape's three constants are a least-squares fit (relative error 3 to 8 %) to its times over 22
 * weights, K 1024 to 17408 and N 1024 to 34816, and 16 to 128 rows; the choice is on average within
 * 1 % of the best shape there and never more than 20 % off. No shape serves all: at 32 rows
 * 9728 x 2560 takes 12.0 us as 1 x 2 x 8 (row tiles x tile pairs x groups a step) and 20 as 2 x 6 x
 * 4, which takes 12.1 us where 2560 x 19456 takes 17 as 1 x 2 x 8. */
inline int rows_shape(int M, int N, int K, int cus) {
    const int G = K / 128, tile_pairs = (N / 8 + 1) / 2, xcd_cus = std::max(1, cus / 8);
    int best = 0;
    float least = 0.0f;
    for (int i = 0; i < (int)(sizeof(kRowsShapes) / sizeof(kRowsShapes[0])); ++i) {
        const RowsShape &c = kRowsShapes[i];
        const long long blocks = ((long long)(tile_pairs + c.tile_pairs - 1) / c.tile_pairs + 7) / 8 *
                                 ((M + 16 * c.rows - 1) / (16 * c.rows));
        const float rounds = (float)((blocks + xcd_cus - 1) / xcd_cus);
        const float t = c.base + (float)((G + c.groups - 1) / c.groups) * (c.first + c.more * (rounds - 1.0f));
        if (i == 0 || t < least) {
            best = i;
            least = t;
        }
    }
    return best;
}

}  // namespace w4a16

#endif
