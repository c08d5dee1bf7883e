// Walks the launches of the LDS-ring kernel on the host, from the header that the launcher and the kernel share.
// Input, a launch per line: elem_bytes TM BN swap M K N batch cover.  Output: slots, LDS bytes, the fewest and the most
// tiles of a workgroup over the XCDs, the most LDS that a workgroup's list reaches to, where `cover` is set whether
// every tile has exactly one workgroup (-1: not walked), the workgroups of the launch that are side by side on the chip
// (over the batch), and how many the choice of a tile height counts on; then, for 64-row tiles (0 otherwise), the log2 of the
// parts that a block-column is cut into, `cover` of that launch, whether each of its tiles has a workgroup to itself, the groups of
// wavefronts that share a long walk there, the LDS of a workgroup with them, and how many of them a CU has to hold; last, whether results with an
// activation are written through (16-bit rows of 64 bytes).
#include <cstdio>
#include <vector>
#include "matmul_spmm_ring_plan.hpp"

using namespace spx;

static int covered(const RingLaunch& launch, int nb) {
    std::vector<int> seen((size_t)launch.list.n_mtiles * nb, 0);
    const bool one = launch.n_pos == launch.n_list;
    for (int xcd = 0; xcd < 8; ++xcd) {
        const RingShare share = ring_share(launch.list, xcd, launch.n_pos);
        for (int pos = 0; pos < launch.n_pos && pos < share.n_list; ++pos)
            for (int r = 0; r < (one ? 1 : share.n_rounds); ++r) {
                int mt = 0, o = 0;
                if (one ? ring_place<true>(launch.list, share, xcd, pos, launch.n_pos, nb, r, mt, o)
                        : ring_place<false>(launch.list, share, xcd, pos, launch.n_pos, nb, r, mt, o)) {
                    if (mt < 0 || mt >= launch.list.n_mtiles || o < 0) return 0;
                    ++seen[(size_t)mt * nb + o];
                }
            }
    }
    for (const int n : seen)
        if (n != 1) return 0;
    return 1;
}

int main() {
    int es, TM, BN, swap, M, K, N, batch, cover;
    while (std::scanf("%d %d %d %d %d %d %d %d %d", &es, &TM, &BN, &swap, &M, &K, &N, &batch, &cover) == 9) {
        const RingLaunch launch = ring_launch(es, TM, BN, swap != 0, M, K, N, batch);
        int fewest = 0x7fffffff, most = 0, reach = 0;
        for (int xcd = 0; xcd < 8; ++xcd) {
            const RingShare share = ring_share(launch.list, xcd, launch.n_pos);
            if (share.n_list == 0) continue;   // no workgroup gets that far
            if (share.n_rounds < fewest) fewest = share.n_rounds;
            if (share.n_rounds > most) most = share.n_rounds;
            const int end = ring_lds(es, TM, BN, swap != 0).list + (share.listed ? share.n_rounds * (int)sizeof(RingTile) : 0);
            if (end > reach) reach = end;
        }
        const bool low = TM == 64;
        const int sub = low ? ring_sub_log2(es, BN, swap != 0, M, K, N, batch) : 0, part = BN >> sub;
        const RingLaunch cut = ring_launch(es, TM, part, swap != 0, M, K, N, batch);
        const bool one = low && cut.n_pos == cut.n_list;
        const int groups = one ? ring_groups(es, part, swap != 0, cut.n_pos * batch, 100.0) : 0;
        const RingLds lds = ring_lds(es, TM, part, swap != 0);
        std::printf("%d %d %d %d %d %d %d %d", launch.list.slots, launch.smem, fewest, most, reach,
                    cover ? covered(launch, N / BN) : -1, 8 * launch.n_pos * batch, ring_slots(es, TM, BN, swap != 0));
        std::printf(" %d %d %d %d %d %d %d\n", sub, cover && low ? covered(cut, N / part) : -1, (int)one, groups,
                    groups ? cut.smem + (groups - 1) * ring_stages(es) * lds.stage : 0, (cut.n_pos * batch + 31) / 32,
                    (int)ring_results_through(M, K, N, launch.list.parts_log2));
    }
    return 0;
}
