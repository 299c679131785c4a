// split3_plan.h -- how an fp32 product on the bf16 matrix cores (gemm_split3.hip) is divided into passes over the rows, row tiles and
// pieces of K.  Host arithmetic on sizes alone, so it is checked on the CPU over all sizes.
#pragma once

#include <cstddef>

namespace rlh {

constexpr int kS3K = 32;      // k values per K-tile
constexpr int kS3Cols = 128;  // columns of a workgroup's tile
constexpr int kS3RowMax = 256; // rows of the highest tile
constexpr int kS3MaxPieces = 16;

struct Split3Plan {
    int rows = 0;      // rows of A of the next pass over B (0: the work memory is too small)
    int tiles = 0;     // 32-row tiles per workgroup
    int m_pad = 0;     // rows of the planes: row tiles x 32 tiles
    int pieces = 1;    // along K
    size_t planes_bytes = 0;
};

// Row tiles of equal height over `rows` rows: sets tiles and m_pad.
inline void split3_row_tiles(int rows, Split3Plan &q) {
    const int row_tiles = (rows + kS3RowMax - 1) / kS3RowMax;
    q.rows = rows;
    q.tiles = ((rows + row_tiles - 1) / row_tiles + 31) / 32;
    q.m_pad = row_tiles * q.tiles * 32;
}

// The next pass over B for the `m` rows that are left.  All of them if their planes, padding included, fit the work memory; else as
// many whole tiles of 256 rows as fit, which pad to themselves.  The rows that then remain can be planned the same way (at worst as
// whole tiles of 256 rows again), so a product whose first pass has a plan has one for every pass.
//
// Pieces along K by a model of the time in microseconds -- rounds of workgroups x (K-tiles of a piece x its cycles + 4 us to start and
// drain), and for a cut product the partial sums written and read back at 4 TB/s and the launch that adds them.  Cycles of a K-tile:
// 384 MFMA cycles per SIMD and 32-row tile + 400 for the barrier and the decomposition of B's first fragments.  That is what a K-tile
// costs its compute unit.  It takes longer (0.5 / 1.2 / 2.2 us with one / four / eight 32-row tiles, where this counts 0.36 / 0.88 / 1.6)
// because all workgroups share the bandwidth that feeds them, and that part does not shrink when more of them run, so it is left out:
// with it the model cuts finer, which loses (11008 x 4096, 8 / 200 rows 53 / 154 -> 63 / 157 us).
inline Split3Plan plan_split3(int m, int n, int k, int ldc, size_t workspace_bytes, int n_cu) {
    Split3Plan best;
    const size_t row_bytes = (size_t)k * 6;
    split3_row_tiles(m, best);
    if ((size_t)best.m_pad * row_bytes > workspace_bytes) {
        const size_t whole = workspace_bytes / row_bytes / kS3RowMax * kS3RowMax;
        if (whole == 0) return Split3Plan();
        split3_row_tiles((int)whole, best); // fewer than m: m rows in tiles of 256 did not fit
    }
    best.planes_bytes = row_bytes * best.m_pad;
    const int kt = k / kS3K;
    const long tiles = (long)((n + kS3Cols - 1) / kS3Cols) * (best.m_pad / (best.tiles * 32));
    const double us_kt = (384.0 * best.tiles + 400.0) / 2200.0;
    const size_t room = workspace_bytes - best.planes_bytes, per = (size_t)best.rows * n * 4;
    double best_t = 0.0;
    for (int s = 1; s <= kS3MaxPieces && (s == 1 || kt / s >= 4); s++) {
        if (s > 1 && ((size_t)s * per > room || n % 4 != 0 || ldc % 4 != 0)) break;
        const long rounds = (tiles * s + n_cu - 1) / n_cu;
        const double t = rounds * (((kt + s - 1) / s) * us_kt + 4.0) + (s > 1 ? 5.0 + s * (double)per * 2.0 / 4e6 : 0.0);
        if (s == 1 || t < best_t) {
            best.pieces = s;
            best_t = t;
        }
    }
    return best;
}

// Microseconds of all passes, to compare with another kernel: rounds of workgroups, partial sums with their launch, and the kernel that takes
// A apart.  Negative: no plan.  Fitted to lone calls (10 % standard deviation), so a K-tile counts in full here; see plan_split3.
inline double split3_us(int m, int n, int k, int ldc, size_t workspace_bytes, int n_cu) {
    double us = 0.0;
    for (int left = m; left > 0;) {
        const Split3Plan q = plan_split3(left, n, k, ldc, workspace_bytes, n_cu);
        if (q.rows <= 0) return -1.0;
        const long blocks = (long)((n + kS3Cols - 1) / kS3Cols) * (q.m_pad / (q.tiles * 32)) * q.pieces, rounds = (blocks + n_cu - 1) / n_cu;
        us += rounds * (5.7 + (k / kS3K + q.pieces - 1) / q.pieces * 0.25 * (q.tiles + 1)) + 2.5 + 3.3e-6 * q.m_pad * (double)k;
        if (q.pieces > 1) us += 2.9 + 0.62e-6 * q.pieces * 4.0 * q.rows * n;
        left -= q.rows;
    }
    return us;
}

// The most work memory that a product of up to `m` rows makes use of: with that much or more its plan is the same.
inline size_t split3_work_bytes(int m, int n, int k) {
    const size_t tile = m > kS3RowMax ? kS3RowMax : 32, padded = ((size_t)m + tile - 1) / tile * tile;
    return padded * k * 6 + (size_t)kS3MaxPieces * m * n * 4;
}

} // namespace rlh
