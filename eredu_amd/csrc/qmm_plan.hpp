// Host-side rules of the prefill-shaped quantized matmul's launches: plain C++,
// so that they can be checked without a GPU.
#pragma once
#include <cstdint>

namespace eq {

constexpr int kBM = 128, kBN = 256, kBK = 64;  // the default tile (rows, columns) and the K chunk

// Whether a launch may read its scales and biases as whole words (two groups
// each): both arrays 4-byte aligned, rows of an even number of groups (always so
// below group size 64) and, with a split of K, splits that start at an even
// group.  A view at an odd element of a larger buffer is only 2-byte aligned;
// such a call reads its parameters two bytes at a time instead (4-bit group 32,
// 14336 x 4096: M = 512 80 us against 67 with windows, M = 64 28 against 23).
inline bool qmm_param_words(int gs, int K, int cps, const void* s, const void* b) {
    if ((reinterpret_cast<uintptr_t>(s) | reinterpret_cast<uintptr_t>(b)) % 4 != 0) return false;  // (no biases: null)
    return gs == 16 || gs == 32 || (gs == 64 && (K / 64) % 2 == 0 && cps % 2 == 0) ||
           (gs == 128 && (K / 128) % 2 == 0 && cps % 4 == 0);
}

// Tile shape and split of K of one launch on `cu` compute units.  Up to 128 rows: one of the narrow
// tiles, by qmm_plan_few_rows.  Above: 128 x 256 tiles when there are at least
// 3/4 as many as CUs, or when K split to fill the CUs still leaves each split
// 32 chunks or more; otherwise 64 x 128 tiles (four times as many, each
// dequantized code used by 64 rows instead of 128) when the large tiles would
// split K 8 ways or more, or at group sizes 32 and above (whose dequantization
// is the cheapest per code), unless the 128 x 128 tiles below take the call.  K is split so that the grid fills the CUs without exceeding
// them (a second round would double the time), at least 8 chunks per split (4
// per K-group).  Measured with weights rotated from HBM, 4-bit: M = 512, 4096 x
// 4096, the large tiles' 4 splits against the 128 x 128 tiles' two: group 32
// 43.5 -> 32.0 us, group 128 40.0 -> 29.0; at group 16 (the 2/3/5/6-bit
// re-packed codes included) the small tiles' per-code work made them 2-8 %
// slower there.  Not so up to 128 rows: group 16, 14336 x 4096, M = 64, 128 x 256
// tiles split four ways against the narrow plan, 4-bit 39.1 -> 28.5 us, 8-bit 47.7
// -> 33.0.  M = 96, 4096 x 4096, group 32, 64 x 128 tiles and 4 splits against 96 x
// 128 and 8: 15.4 against 19.7 us; M = 77, 14336 x 4096, 96 x 128 against 128 x 128
// tiles, both split twice: 24.8 against 26.2.
struct QmmPlan {
    int tm, tn;  // 32-row and 128-column blocks of a tile
    int mtiles, ntiles, splits;
};
inline int qmm_splits(int tiles, int slots, int nchunks) {
    int s = slots / (tiles > 0 ? tiles : 1);
    s = s > nchunks / 8 ? nchunks / 8 : s;
    return s < 1 ? 1 : s;
}
// The cheapest plan of at most 128 rows, in microseconds: a workgroup walks
// its steps of two chunks in `step` each (64, 96 and 128 rows measured at
// 0.70, 0.87 and 1.0 us, whether or not a second workgroup shares the CU)
// after 5 us of launch, first loads and reduction; partials are written and
// read back at 4 MB/us, and their reduction is a launch of 2.5 us.  Where the
// 64 x 128 tiles cover more than half the CUs and K is short, K is split only if
// the pieces stay at 24 chunks, fill 3/4 of the CUs and write partials of at
// most N K bytes: such calls otherwise need no workspace, and may be captured
// without an eager call before.  (Not at group size 16 where 128 x 256 tiles
// would split K 2 to 7 ways: 4-bit, M = 87, 12160 x 5248 61 -> 42 us, 8-bit, M =
// 128, 10240 x 3072 39.9 -> 27.6.)
inline QmmPlan qmm_plan_few_rows(int M, int N, int gs, int bits, int cu, int nchunks, bool may_split) {
    QmmPlan best{};
    double least = 0;
    const int nt = (N + 127) / 128, big_splits = qmm_splits((N + 255) / 256, cu, nchunks);
    const bool short_k = qmm_splits((M + 63) / 64 * nt, cu, nchunks) == 1 && nchunks / big_splits < 32 &&
                         (gs > 16 || big_splits == 1 || big_splits >= 8);
    const double step[3] = {0.70, 0.87, 1.0};
    for (int tm = 2; tm <= 4; tm++) {
        const int mt = (M + 32 * tm - 1) / (32 * tm);
        const int most = may_split ? qmm_splits(mt * nt, cu, nchunks) : 1;
        for (int s = 1; s <= most; s++) {
            if (s > 1 && short_k &&
                (nchunks / s < 24 || 4 * mt * nt * s < 3 * cu || int64_t(s) * M * 4 > int64_t(nchunks) * kBK))
                continue;
            const int rounds = (mt * nt * s + cu - 1) / cu, steps = (nchunks + 2 * s - 1) / (2 * s);
            const double us = rounds * (5.0 + steps * step[tm - 2]) + (s > 1 ? 2.5 + 8.0 * s * M * N / 4e6 : 0.0);
            if (!best.tm || us < least) least = us, best = QmmPlan{tm, 1, mt, nt, s};
        }
    }
    // 8-bit codes above 96 rows: unsplit 64 x 128 tiles, which read each code for
    // two row tiles, lose to split 128 x 128 ones (group 64, K = 4096: M = 128 14336
    // rows 34.1 -> 31.9 us, M = 100 15872 rows 35.1 -> 31.6, M = 112 12288 rows 33.8 ->
    // 28.9; group 16, M = 128, 10240 x 3072 39.9 -> 27.6; with 4-bit codes 27.4 against
    // 29.0 at M = 128, 14336 x 4096), but need longer pieces where they fill the CUs
    // exactly (M = 120, 16384 x 3072, 24 chunks: 27.6 against 29.2).
    const int ms = may_split ? qmm_splits(nt, cu, nchunks) : 1;
    const int least_chunks = gs == 16 && !short_k ? 16 : 2 * nt >= cu ? 32 : 24;
    if (bits == 8 && M > 96 && best.splits == 1 && ms > 1 && 4 * nt * ms >= 3 * cu && nchunks / ms >= least_chunks &&
        int64_t(ms) * M * 4 <= int64_t(nchunks) * kBK)
        best = QmmPlan{4, 1, 1, nt, ms};
    return best;
}
inline QmmPlan qmm_plan(int M, int N, int K, int gs, int bits, bool may_split, int cu) {
    const int nchunks = K / kBK;
    if (M <= 128) return qmm_plan_few_rows(M, N, gs, bits, cu, nchunks, may_split);
    QmmPlan p{4, 2, 0, 0, 1};
    const int big = ((M + 127) / 128) * ((N + 255) / 256);
    const int big_splits = may_split ? qmm_splits(big, cu, nchunks) : 1;
    const bool big_ok = 4 * big >= 3 * cu || nchunks / big_splits >= 32;
    const bool small_ok = big_splits >= 8 || gs >= 32;
    if (!big_ok && small_ok) p.tm = 2, p.tn = 1;
    // 128 x 128 tiles (group sizes 32 and above) in place of the
    // small tiles, or of large tiles that split K, when their own split leaves
    // each piece at least 24 chunks, fills 3/4 of the CUs and writes f32
    // partials of at most twice the weight bytes: every code then feeds 128
    // rows, as in the large tile, with twice the large tile's workgroups.
    // Group size 16: in place of small tiles that split K, at 16 chunks and any
    // partials (4-bit, M = 955, 768 x 13952: 71 -> 43 us, M = 323, 1152 x 10368:
    // 33.6 -> 27.3; M = 539, 896 x 6784, 17 chunks, 8-bit: 25.0 against 25.2).
    const int mid = ((M + 127) / 128) * ((N + 127) / 128), ms = qmm_splits(mid, cu, nchunks);
    const bool fills = 4 * mid * ms >= 3 * cu;
    if (may_split && gs == 16) {
        if (p.tm == 2 && qmm_splits(((M + 63) / 64) * ((N + 127) / 128), cu, nchunks) > 1 && fills && nchunks / ms >= 16)
            p.tm = 4, p.tn = 1;
    } else if (may_split && (p.tm == 2 || big_splits > 1)) {
        const bool long_k = nchunks / ms >= 24;
        const bool partials_ok = ms == 1 || double(ms) * M * N * 4.0 <= 2.0 * double(N) * double(K) * bits / 8.0;
        if (fills && long_k && partials_ok && (p.tm == 2 || ms < big_splits)) p.tm = 4, p.tn = 1;
    }
    p.mtiles = (M + 32 * p.tm - 1) / (32 * p.tm), p.ntiles = (N + 128 * p.tn - 1) / (128 * p.tn);
    p.splits = may_split ? qmm_splits(p.mtiles * p.ntiles, cu, nchunks) : 1;
    return p;
}

}  // namespace eq
