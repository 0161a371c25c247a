// CPU check of how the mode GEMM walks its channels (turbofno_amd/csrc/gemm_steps.h). On standard input lines of numbers, their kind
// first: "0 K Kw nt threads cap" prints the channels per run and whether its steps go in halves; "1 nblocks most K" the persistent blocks
// per tile of outputs.
#include "../../turbofno_amd/csrc/gemm_steps.h"
#include <cstdio>
int main()
{
    int kind;
    while (std::scanf("%d", &kind) == 1) {
        int K, Kw, nt, threads, cap;
        long nblocks, most;
        if (kind == 0 && std::scanf("%d %d %d %d %d", &K, &Kw, &nt, &threads, &cap) == 5) {
            const tfno::GemmWalk walk = tfno::gemm_walk(K, Kw, nt, threads, cap);
            std::printf("%d %d\n", walk.run, (int)walk.halves);
        } else if (kind == 1 && std::scanf("%ld %ld %d", &nblocks, &most, &K) == 3) {
            std::printf("%ld\n", tfno::gemm_persistent_blocks(nblocks, most, K));
        } else {
            return 1;
        }
    }
    return 0;
}
