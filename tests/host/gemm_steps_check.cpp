// CPU check of how the mode GEMM walks its channels (turbofno_amd/csrc/gemm_steps.h): for each "K Kw nt threads cap" on
// standard input, prints the channels per run and whether its steps go in halves.
#include "../../turbofno_amd/csrc/gemm_steps.h"
#include <cstdio>
int main()
{
    int K, Kw, nt, threads, cap;
    while (std::scanf("%d %d %d %d %d", &K, &Kw, &nt, &threads, &cap) == 5) {
        const tfno::GemmWalk walk = tfno::gemm_walk(K, Kw, nt, threads, cap);
        std::printf("%d %d\n", walk.run, (int)walk.halves);
    }
    return 0;
}
