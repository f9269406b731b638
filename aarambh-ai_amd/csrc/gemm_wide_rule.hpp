// Which many-row products take the wide wave tiles (gemm_wide.hip).
// Plain C++, so that a host test can ask for the choice.
#pragma once

namespace aarh {

inline int wide_blocks(int N, int M, int cols, int rows) { return ((N + cols - 1) / cols) * ((M + rows - 1) / rows); }

// INT4: time in us of a launch with cn = 2 or 3 weight tiles per wave (128 or 192 columns x 64
// rows per block) without k-splits, from the measured cost of a block (10 us of ramp, K
// reduction and epilogue, then 0.93 or 1.22 us per 128-column group) and the dispatch rounds.
inline double wide_time(int N, int K, int M, int cn, int cus) {
    const int rounds = (wide_blocks(N, M, 64 * cn, 64) + cus - 1) / cus;
    return rounds * (10.0 + (K >> 7) * (cn == 3 ? 1.22 : 0.93));
}

// gemm.hip's plans take about 5 us plus 1.75e-7 us per 32 rows, weight row and column (0.5 us
// per 32 rows x 2048 columns x 1408 weight rows), measured within 20% for the d4096 projections
// from 72 to 500 rows; shapes outside its table (`tuned`) also have blocks of 64 rows x 192 or
// 256 columns (12.5 us, then 1.33 or 1.7 us per group; gate/up 16384 x 3072 at 250 rows 57 us
// against 65 wide, at 500 rows 108 against 122, at 333 rows 102 against 95).  The wide tiles win
// where their blocks fill the dispatch rounds.  The d4096 projections up to 513 rows: gate/up at
// 65 to 128, 161 to 256 and from 289 rows, qkv from 225, down from 321 and wo from 353; wo and
// down at 256 rows (128 blocks) measured 34 and 76 us against 27 and 57.
inline bool wide_wins_int4(int N, int K, int M, bool tuned, int cus) {
    if (M <= 64) return false;
    double narrow = 5.0 + 1.75e-7 * ((M + 31) / 32) * (double)N * K;
    if (!tuned)
        for (int tpw = 3; tpw <= 4; tpw++) {
            const int rounds = (wide_blocks(N, M, 64 * tpw, 64) + cus - 1) / cus;
            const double t = rounds * (12.5 + (K >> 7) * (tpw == 4 ? 1.7 : 1.33));
            if (t < narrow) narrow = t;
        }
    return wide_time(N, K, M, 2, cus) < narrow || wide_time(N, K, M, 3, cus) < narrow;
}

// The BF16 LM head's blocks cover 128 rows against 64: they win where that halves the row blocks
// (183 rows, which it does not: 174 us against 141) and fills the dispatch rounds to nine
// tenths, or to three quarters where one row block reads the weights from HBM once.  50304 x
// 3072, 200 rows (786 blocks, four rounds for three): forward 888 us wide, 853 narrow; 50304 x
// 4096, 70 rows (393 blocks): 755 wide, 794 narrow.  32000 x 4096: 65 to 128, 193 to 256, 321
// to 384 and 449 to 512 rows.
inline bool wide_wins_head(int N, int M, int cus) {
    const int nb = wide_blocks(N, M, 128, 128), slots = (nb + cus - 1) / cus * cus;
    return M > 64 && ((M + 63) / 64) % 2 == 0 && nb * 20 >= slots * (M <= 128 ? 15 : 18);
}

}  // namespace aarh
