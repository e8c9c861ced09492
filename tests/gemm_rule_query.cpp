// Prints the tile that gemm_rule.hpp picks for each launch named on the command line (0: none
// fits). Test infrastructure: built with g++ by tests/gemm_launches.py.
//
// Usage: gemm_rule_query N_CU [DTYPE M N K NCOL ROWS_PER_BATCH]...   (dtype 0 fp32, 1 bf16)
#include <cstdio>
#include <cstdlib>

#include "../slime_amd/csrc/gemm_rule.hpp"

int main(int argc, char** argv) {
    if (argc < 8 || (argc - 2) % 6) return 2;
    for (int i = 2; i < argc; i += 6) {
        int v[6];
        for (int k = 0; k < 6; ++k) v[k] = std::atoi(argv[i + k]);
        std::printf("%d\n", slime::gemm_rule::pick({v[0], v[1], v[2], v[3], v[4], v[5]}, std::atoi(argv[1])));
    }
    return 0;
}
