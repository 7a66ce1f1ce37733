// Prints chs::tdma_thread_per_line for each "kind n nl alloc" line of stdin.
#include <cstdio>

#include "../../chapsim1.0_amd/csrc/chs_tdma_rule.h"

int main()
{
    int kind, n, nl, alloc;
    while (std::scanf("%d %d %d %d", &kind, &n, &nl, &alloc) == 4)
        std::printf("%d\n", (int)chs::tdma_thread_per_line(kind, n, nl, alloc != 0));
}
