// Checks csrc/row_slot.hpp on the host: every row is taken once, pairs are of one sequence.
#include <stdio.h>

#include <vector>
#define __host__ static
#define __device__
#define __forceinline__ inline
#include "../../aarambh-ai_amd/csrc/row_slot.hpp"

int main() {
    long wrong = 0, split = 0, n = 0;
    for (int cus : {1, 2, 7, 256, 304})
        for (int rows = 1; rows <= 20; rows++)
            for (int seqs = 1; seqs <= 150; seqs++) {
                const int blocks = seqs * rows;
                std::vector<int> taken(blocks, 0), seq(blocks);
                for (int i = 0; i < blocks; i++) {
                    const RowSlot s = row_slot(i, blocks, rows, cus);
                    if (s.seq < 0 || s.seq >= seqs || s.row < 0 || s.row >= rows) {
                        wrong++;
                        continue;
                    }
                    wrong += taken[s.seq * rows + s.row]++;
                    seq[i] = s.seq;
                }
                // pairs of one sequence, as far as the sequences' rows give whole pairs
                int differ = 0;
                for (int i = cus; i < blocks && i < 2 * cus; i++) differ += seq[i] != seq[i - cus];
                const int could = seqs * (rows / 2), joined = blocks < 2 * cus ? blocks - cus : cus;
                if (joined > 0) split += differ > (joined > could ? joined - could : 0);
                n++;
            }
    printf("%ld %ld %ld\n", n, wrong, split);
    return 0;
}
