// For each "fmt N K M" of the command line: 1 where csrc/gemm_wide_rule.hpp takes the wide tiles.
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "../../aarambh-ai_amd/csrc/gemm_wide_rule.hpp"

int main(int argc, char** argv) {
    for (int i = 1; i + 3 < argc; i += 4) {
        const int n = atoi(argv[i + 1]), k = atoi(argv[i + 2]), m = atoi(argv[i + 3]);
        printf("%d\n", strcmp(argv[i], "head") == 0 ? aarh::wide_wins_head(n, m, 256)
                                                    : aarh::wide_wins_int4(n, k, m, strcmp(argv[i], "tuned") == 0, 256));
    }
    return 0;
}
