/*
 * rows_shape.h - host-only rules of the multi-row dispatch: the block shapes of rows_gemm_kernel and the choice
 * between them, which linears rows_stream_kernel and gemv_rows16w_kernel take, and the RMSNorm's block.
 */
#ifndef W4A16_ROWS_SHAPE_H
#define W4A16_ROWS_SHAPE_H

#include <algorithm>
#include <cstddef>

namespace w4a16 {

constexpr std::size_t kMaxLds = 163840; /* LDS a block can allocate on gfx950 */

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

/* The few-row kernel's LDS: both groups of every pair of the M rows (whole 1 KiB load instructions) and the
 * wave reduction. */
inline std::size_t rows_smem(int M, int K, int waves) {
    const int P = (K / 128 + 1) / 2;
    return (std::size_t)((P * 32 * M + 63) / 64) * 1024 + (std::size_t)waves * 256;
}

/* Whether an N x K linear of M <= 16 row-major rows that no LDS-staged tile-pair kernel takes runs on
 * rows_stream_kernel (or past its LDS on the row-tiled GEMM): with more than one tile pair a CU, from a K that falls
 * with the rows (17408 x 5120 M = 2 / 3 / 8 18.9 / 19.4 / 31.1 us in the few-row form, 17.6 / 17.1 / 21.5 there;
 * 8704 x 5120 M = 5 / 8 11.9 / 12.6, 10.2 / 10.8). With up to two tile pairs a CU the few-row form keeps 4 rows a
 * little longer (8704 x 5120 10.4 / 10.4) and up to 64 KB of rows (5 rows of 5248 x 4224 7.3 / 7.8, of 6144 x 8192
 * 9.2 / 9.5, but 6 of 6144 x 5120 8.4 / 8.2, and 5 of 5248 x 9728 11.5 / 10.0); and just past one tile pair a CU, where
 * the streamed kernel leaves half of the CUs without a block, as long as two blocks of it fit a CU (5 rows of
 * 7168 x 4104 8.2 / 9.0). */
inline bool rows_streams(int M, int N, int K, int cus) {
    const int pairs = (K / 128 + 1) / 2, tile_pairs = (N / 8 + 1) / 2;
    const bool narrow = tile_pairs <= 2 * cus;
    if (tile_pairs <= cus || pairs <= (M == 2 ? 48 : M == 3 ? 40 : M == 4 ? (narrow ? 36 : 32) : 20)) return false;
    const std::size_t staged = rows_smem(M, K, 16);
    if (M >= 5 && narrow && staged <= 68 * 1024) return false; /* the rows and the waves' sums */
    return !(M >= 4 && tile_pairs < cus + cus / 32 && staged <= kMaxLds / 2);
}

/* Tile pairs a block (1, 2 or 4) of gemv_rows16w_kernel for a linear of more than 16 rows, 0 where the row-tiled
 * GEMM takes it. The registers-fed slices win while they are one round of blocks and K is no more than two groups a
 * wave, except where K fills the steps of the GEMM's small shapes (24 rows, N = 1024, registers-fed / row-tiled: K = 1024
 * 4.0 / 4.3 us, 1536 4.4 / 5.4, 2048 5.0 / 4.8, 2560 5.3 / 6.1, 3712 6.1 / 6.5, 4096 6.5 / 6.5; two tile pairs, 128
 * rows: 1024 4.5 / 4.4, 1536 5.0 / 5.4, 2560 5.9 / 6.3); in fours only as a nearly full round (K = 3200, N = 2048, 128 / 80
 * rows 7.6 / 8.2, 7.8 / 7.5). */
inline int rows_slices(int M, int N, int K, int cus) {
    const int G = K / 128;
    if ((G > 12 && G <= 16) || G > 30) return 0;
    const long long tile_pairs = (N / 8 + 1) / 2, slices = (M + 15) / 16;
    if (tile_pairs * slices <= cus) return 1;
    if (G > 5 && G <= 8) return 0;
    if ((tile_pairs + 1) / 2 * slices <= cus) return G <= 28 ? 2 : 0;
    const long long fours = (tile_pairs + 3) / 4 * slices;
    return fours <= cus && fours > cus * 7 / 8 ? 4 : 0;
}

/* Chunks of 8 values a thread of rmsnorm_kernel. One keeps a row's FP64 chain shortest; of blocks past 512 threads,
 * though, too few fit a CU once there are more rows than that (5120 columns, one / two chunks: 384 rows and fewer one is
 * ahead, 768 4.7 / 4.2 us, 2048 8.7 / 7.9, 16384 69 / 58). */
inline int rmsnorm_chunks(int cols, int rows, int cus) {
    const int chunks = cols / 8;
    return chunks > 1024 || (chunks > 512 && rows > cus + cus / 2) ? 2 : 1;
}

}  // namespace w4a16

#endif
