// Which logits row each workgroup of the acceptance kernel takes.
// Plain C++ once __host__, __device__ and __forceinline__ are defined: the host test includes it.
#pragma once

struct RowSlot {
    int seq, row;
};

// Workgroup `block` of `blocks` = sequences x `rows`; `cus` compute units hold two workgroups
// each.  Workgroups cus .. 2 cus - 1 join the ones already on compute units 0 .. cus - 1, and the
// two slow each other down, so they are the last of their sequences to finish and resolve them.
// In row order the pair belongs to two sequences, and both resolve on the one compute unit: 32
// sequences x 9 rows of 32 000 logits 232 us against 180 us of 28 sequences (252 workgroups), 20
// x 13 of 50 000 341 against 252 of 19.  So pairs are formed of rows of one sequence, which
// leaves its resolver alone: 187 and 254 us, 128 x 9 rows of 32 000 420 -> 320.
__host__ __device__ __forceinline__ RowSlot row_slot(int block, int blocks, int rows, int cus) {
    const int half = rows / 2;  // pairs per sequence
    if (blocks <= cus || half == 0) return {block / rows, block % rows};
    int pairs = blocks / rows * half;
    if (pairs > blocks - cus) pairs = blocks - cus;
    if (pairs > cus) pairs = cus;
    if (block < pairs) return {block / half, 2 * (block % half)};
    if (block >= cus && block < cus + pairs) return {(block - cus) / half, 2 * ((block - cus) % half) + 1};
    // the other rows in order: the odd row of each paired sequence, the rest of the one paired
    // in part, whole sequences
    const int t = block < cus ? block - pairs : block - 2 * pairs;
    const int paired = pairs / half, odd = rows - 2 * half;
    if (t < paired * odd) return {t, rows - 1};
    const int at = t - paired * odd + 2 * (pairs % half);
    return {paired + at / rows, at % rows};
}
