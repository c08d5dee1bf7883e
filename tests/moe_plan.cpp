// Asks the plan of the persistent gathered GEMM, from the header that its launcher and its kernel share.
// Input, a problem per line: tokens K N experts w_kcontig CUs.  Output: whether it fits, the tiles that a workgroup's list has
// room for, the end of that list in LDS, and the largest byte offsets into the tokens and into the weights of a tile.
#include <cstdio>
#include "moe_plan.hpp"

using namespace spx;

int main() {
    int n_tok, K, N, n_exp, w_kcontig, n_cu;
    while (std::scanf("%d %d %d %d %d %d", &n_tok, &K, &N, &n_exp, &w_kcontig, &n_cu) == 6) {
        const int64_t rounds = persist_rounds(n_tok, N, n_exp, persist_workgroups(n_cu));
        const int64_t tokens = (int64_t)(n_tok - 1) * K * 2 + 128, cols = N < 256 ? N : 256;
        const int64_t weights = w_kcontig ? (cols - 1) * K * 2 + 128 : ((int64_t)63 * N + N) * 2;
        std::printf("%d %lld %lld %lld %lld\n", persist_fits(n_tok, K, N, n_exp, w_kcontig != 0, n_cu) ? 1 : 0, (long long)rounds,
                    (long long)(kPersistList + rounds * (int64_t)sizeof(PersistTile)), (long long)tokens, (long long)weights);
    }
    return 0;
}
