// Prints the form an M > 1 product takes (llm-kv260_amd/csrc/gemm_route.h) for
// each "m rows k cus" line of its input.
#include <cstdio>

#include "gemm_route.h"

using namespace w4a8;

int main() {
    const char *const forms[] = {"split", "rows", "tiles"};
    int m, rows, k, cus;
    while (std::scanf("%d %d %d %d", &m, &rows, &k, &cus) == 4)
        std::printf("split%d rows%d %s\n", gemm_route::split_tokens(m, rows, k, cus),
                    gemm_route::split_rows(m, rows, k, cus), forms[gemm_route::form(m, rows, k, cus)]);
    return 0;
}
