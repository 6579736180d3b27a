// small_batch_plan.h -- which calls the small-batch matrix-core kernel takes
// and how it splits them.  Plain host arithmetic on the shape, in a header of
// its own so that the host tests compile the same rules.
#pragma once

#include <stdint.h>

#include <algorithm>

namespace iq4xs {

// The choices that fix a row's summation order count row blocks against
// MI355X's 256 CUs, so that a device or partition with another CU count gives
// the same bits; grid shapes use the device's own count.
constexpr int64_t GM_CHOICE_CUS = 256;

constexpr int64_t GM_MAX_COLS = 64;

// Calls of the GEMM entry (M > 8) that the small-batch kernel takes: those
// where neither the matrix alone, nor a pair of it (gate and up), nor it with
// two eighths of its rows (q, k, v) is slower than on the GEMM.  The route
// follows the matrix alone, since a grouped call has the bits of single ones;
// up to 8192 rows it follows K and M alone, so that q, k and v go together.
//   * The GEMM reads a weight once for all columns but needs about 256 tiles
//     of 128 rows to fill the chip; this kernel fills it with 32-row blocks,
//     and its time grows with the columns.  So it wins on few columns
//     everywhere (us, GEMM / here: a pair of 17408 x 5120, M = 16 62 / 29), on
//     many only where the GEMM's tiles are few (4096 x 17408, M = 64 79 / 46)
//     or just past a round: pairs of 16384 to 24576 rows (17408 x 5120: M = 40
//     71 / 51, M = 48 71 / 58), but not of 13312 (M = 40 40 / 47, M = 64 41 /
//     52), and not a single matrix of 28672 (M = 40 41 / 47).
//   * Short rows: with 5 to about 15 super-blocks most waves have one or two,
//     and a second round of workgroups costs a full one (K = 1280: 28672 rows,
//     M = 24 12.7 / 16.5, M = 32 13.0 / 20.1; a pair of 6144, M = 48 13.2 /
//     17.3; K = 2304: a pair of 9216, M = 32 18.1 / 21.4, a pair of 8192, M =
//     64 19.3 / 23.3), hence the least K, though a single matrix of 4096 rows
//     is faster here below it too (K = 2304, M = 64 14.5 / 12.4).  Up to four
//     super-blocks a workgroup has four waves, and more of them fit a CU.
//   * The limits of the kernel's 32-bit offsets.
inline bool use_small_batch(int64_t N, int64_t K, int64_t M) {
    if (M > GM_MAX_COLS || N >= ((int64_t)1 << 30) || K >= ((int64_t)1 << 24)) return false;
    constexpr int64_t kRound = 32 * GM_CHOICE_CUS;  // rows of one 32-row block per CU: 8192
    if (M <= 24) return N <= 3 * kRound / 2 || K <= 1024 || K >= 1792;
    if (M <= 32) return N <= kRound || K <= 1024 || K >= (N <= 3 * kRound / 2 ? 4608 : 5120);
    if (M <= 40 && N <= kRound && (K <= 1024 || K >= 1792)) return true;
    if (K < 4096) return false;
    return N <= kRound || (M <= 48 && (N <= 3 * kRound / 2 || (N > 2 * kRound && N <= 3 * kRound)));
}

// Most waves of a workgroup at G groups of 8 columns (gm_split).
constexpr int gm_max_waves(int G) { return G == 1 ? 16 : G <= 6 ? 12 : 8; }

// How K is split over the waves of a workgroup: `waves` waves, each with one
// partial sum or (`two`) one for its even and one for its odd super-blocks.
struct GmSplit {
    int waves;
    bool two;
    bool operator==(const GmSplit& o) const { return waves == o.waves && two == o.two; }
};

// The split of an N-row matrix.  It fixes a row's fp32 summation order, so it
// follows the matrix's own shape and M, never the launch.
//   * From 384 row blocks on (gate/up, N = 17408) the blocks alone nearly fill
//     the chip: 8 waves each.  Past 32 tokens, where a workgroup of 8 leaves
//     no room for a second one, 4 waves as soon as there are more blocks than
//     CUs (up to 48 tokens: use_small_batch).
//   * Below, K is split further so that every CU has loads in flight: 12
//     waves, 8 past 48 tokens (226 and 246 registers leave two waves per
//     SIMD), 16 up to 8 tokens from K = 8192 on (as fast, with shorter sums).
// Measured, us per launch with 4 / 8 / 12 waves: gate + up M = 8 30.6 / 30.3 /
// 33.4, M = 32 48.5 / 47.7 / 55.2, M = 33 55 / 75 / 70; 17408 -> 5120 M = 8
// 32.5 / 21.0 / 18.7 (16 waves 19.1), M = 32 50 / 33 / 29, M = 33 66 / 43 /
// 36, M = 64 59 / 44.
//
// Precision at M <= 8: sixteen partial sums below 512 row blocks have the
// shorter chains (K = 17408: 1.33e-7 against 1.59e-7 with eight, rel. 2-norm
// against 64 bits).  From 384 blocks on 8 waves keep them as two sums each,
// added in the order of sixteen waves, with the bits and without the time of
// those (12288 x 3328, M = 8: 9.3 us, 16 waves 11.2) -- where sixteen are
// closer: with 9 to 15 super-blocks eight have up to 1.05 times their error,
// with 16 to 24 as much (0.99 to 1.00), with more 1.02 times and rising.
// Twelve waves add their sums in two chains (gemv_mfma.hip), which is closer
// than sixteen in one (K = 3584: 0.83e-7 against 0.89e-7; one chain of twelve
// 0.93e-7).
inline GmSplit gm_split(int64_t N, int64_t K, int G) {
    const int64_t bpr = K / 256, blocks = (N + 31) / 32;
    constexpr int64_t kLarge = 3 * GM_CHOICE_CUS / 2;  // 384 row blocks
    int waves = G == 1 && bpr < 32 ? 12 : gm_max_waves(G);
    if (G <= 4 && blocks >= kLarge) waves = 8;
    if (G >= 5 && blocks > GM_CHOICE_CUS) waves = 4;
    const bool longer = (bpr > 8 && bpr < 16) || bpr > 24;  // eight sums against sixteen, see above
    return {(int)std::max<int64_t>(4, std::min<int64_t>(waves, bpr)),
            G == 1 && blocks >= kLarge && blocks < 2 * GM_CHOICE_CUS && longer};
}

// Rows per workgroup of a launch of `count` matrices on `cus` CUs: the fewest
// that give every CU at most one workgroup (N = 5120: 20 rows on 256 CUs
// against 160 blocks of 32), 32 where that many do not fit.  Each matrix has a
// ragged last block of its own, so the total alone does not tell: q/k/v of
// 4096 + 512 + 512 rows have 257 workgroups of 20, and the last one is a
// second round (K = 5120, M = 64: 29.1 us, with 21 rows 16.7).  At least 8,
// since each workgroup decodes all 32 MFMA rows whatever it keeps (N = 1024,
// M = 8: 6.6 us with 8 rows against 7.0 with 4).
inline int64_t gm_rows(int count, const int64_t* N, int64_t cus) {
    int64_t total = 0;
    for (int i = 0; i < count; ++i) total += N[i];
    int64_t rows = std::max<int64_t>(8, std::min<int64_t>(32, (total + cus - 1) / cus));
    for (; rows < 32; ++rows) {
        int64_t wgs = 0;
        for (int i = 0; i < count; ++i) wgs += (N[i] + rows - 1) / rows;
        if (wgs <= cus) break;
    }
    return rows;
}

}  // namespace iq4xs
