// What the host and the workgroups of the LDS-ring kernel (matmul_spmm_ring.hpp) have to agree on: the LDS layout, the
// division of the tiles among the workgroups, and whether a workgroup keeps the list of its tiles in LDS.  Each of these
// is worked out here and nowhere else.  Plain C++ without device code, so that a host program can walk every workgroup.
#pragma once
#include <cstdint>

namespace spx {

constexpr int kRingThreads = 320;     // four multiplying wavefronts and the loader
constexpr int kRingTableMax = 1024;   // block-columns whose order and pointers fit the ring before it is filled (8 KB)
constexpr int kRingListMax = 128;     // tiles of a workgroup that fit its list (2 KB)
constexpr int kRingLdsOfCu = 160 * 1024, kRingLdsPiece = 1280;   // LDS is given out in pieces
struct alignas(16) RingTile {
    int m0, j, e0, n_blk;             // n_blk < 0: no tile
};

// Stages: two keep a third or fourth workgroup on the CU, which 16-bit types gain more from (8192 x 3072 -> 768
// at 10 %: 15.0 against 16.4 us with three); fp32 works longer on a stage and wants the deeper ring.
constexpr int ring_stages(int elem_bytes) { return elem_bytes == 2 ? 2 : 3; }

// LDS layout: the ring, the output tile, then the list of tiles.  swap: the tile lies as [m][n] in LDS.
struct RingLds {
    int stage;        // bytes of a stage
    int rows, cols;   // output tile
    int pitch;        // elements from row to row of it
    int list;         // where the list of tiles begins: all that a workgroup without one needs
};
constexpr RingLds ring_lds(int elem_bytes, int TM, int BN, bool swap) {
    const int stage = (TM + BN) * 128, rows = swap ? TM : BN, cols = swap ? BN : TM, pitch = cols + 16 / elem_bytes;
    return {stage, rows, cols, pitch, ring_stages(elem_bytes) * stage + rows * pitch * elem_bytes};
}

// The list of tiles of an XCD (workgroup L runs on XCD L % 8).  A unit is a panel of TM dense rows with
// every `parts`-th block-column of the launch order (parts > 1: fewer panels than fill the XCDs evenly);
// unit u belongs to XCD u % 8.  `group` units at a time - what their dense rows take in the XCD's L2
// - are walked column by column, longest first, so the list falls in length group by group and
// workgroups that take it there and back end up with equal sums.
struct RingList {
    int n_mtiles, parts_log2, cols, group;   // cols: block-columns of a unit, rounded up
    // Tiles that the launch has LDS for in the list of a workgroup, 0: none, every tile is looked up when it is needed.
    // The XCDs' lists differ in length, so only the host, which sizes LDS by the longest, may decide this: a workgroup
    // never has more tiles than slots, but it may have fewer, and even one.
    int slots;
};
constexpr int ring_units(const RingList& l, int xcd) { return ((l.n_mtiles << l.parts_log2) - xcd + 7) >> 3; }
constexpr int ring_rounds(int n_list, int n_pos) { return n_pos == 0 ? 0 : (n_list + n_pos - 1) / n_pos; }

// What falls to an XCD, and to each of its n_pos workgroups.
struct RingShare {
    int n_units, n_list;   // its units, and the tiles in its list
    int n_rounds;          // tiles of a workgroup, rounded up
    bool listed;           // ... which it keeps in LDS
};
constexpr RingShare ring_share(const RingList& l, int xcd, int n_pos) {
    const int n_units = ring_units(l, xcd), n_list = n_units * l.cols;
    return {n_units, n_list, ring_rounds(n_list, n_pos), l.slots > 0};
}
// The place of the r-th tile of workgroup `pos` of an XCD: its row tile and its position in the launch order of the nb
// block-columns; false: none.  One: no workgroup has more than one tile.
template <bool ONE>
constexpr bool ring_place(const RingList& l, const RingShare& share, int xcd, int pos, int n_pos, int nb, int r, int& mt, int& o) {
    const int id = r * n_pos + (r & 1 ? n_pos - 1 - pos : pos);   // there and back along the list
    if (id >= share.n_list) return false;
    int first = 0, size = share.n_units;   // (with one tile to a workgroup all of them run side by side: one group)
    if constexpr (!ONE) {
        first = id / (l.group * l.cols) * l.group;
        size = share.n_units - first < l.group ? share.n_units - first : l.group;
    }
    const int in = id - first * l.cols, i = in / size;
    const int unit = (first + in - i * size) * 8 + xcd;
    mt = unit >> l.parts_log2;
    o = (i << l.parts_log2) + unit - (mt << l.parts_log2);
    return o < nb;
}

// Whether the tiles of a workgroup are listed, all at once by a thread each: what a wavefront then needs of the next one
// is a single read, where looking it up takes three divisions and three dependent reads between two tiles.  fp16 us
// before / after, 32 x 64 blocks, 64-row and 128-row tiles: 8192 x 768 -> 3072 at 10 % 28.1 / 21.3 and 22.2 / 20.3, 16384 x
// 512 -> 2048 at 20 % 37.1 / 29.2 and 28.4 / 27.0, 8192 x 768 -> 2304 at 20 % 24.7 / 20.4 and 20.4 / 18.5; with two tiles to a
// workgroup 18.9 / 18.1 and 16.2 / 16.2 (8192 x 3072 -> 768), 64-row tiles 11.9 / 10.0 (4518 x 1472 -> 1024 at 20 %) and no size behind.
constexpr bool ring_listed(int n_rounds) { return n_rounds > 1 && n_rounds <= kRingListMax; }

struct RingLaunch {
    RingList list;
    int n_list;   // tiles in the longest of the eight lists
    int n_pos;    // workgroups per XCD
    int smem;     // bytes of LDS of a workgroup
};
// The launch with `per_cu` workgroups to a CU (the batch entries share the device).
constexpr RingLaunch ring_launch_of(RingList l, int lds, int per_cu, int batch) {
    const int n_list = ring_units(l, 0) * l.cols, fit = 32 * per_cu / batch;
    const int n_pos = fit < 1 ? 1 : fit > n_list ? n_list : fit;
    const int n_rounds = ring_rounds(n_list, n_pos);
    l.slots = ring_listed(n_rounds) ? n_rounds : 0;
    return {l, n_list, n_pos, lds + l.slots * (int)sizeof(RingTile)};
}
constexpr bool ring_fits(int smem, int per_cu) {
    return per_cu * ((smem + kRingLdsPiece - 1) / kRingLdsPiece * kRingLdsPiece) <= kRingLdsOfCu;
}
// Workgroups that fit the chip's 256 CUs at a time, at most five to a CU.
constexpr int ring_slots(int elem_bytes, int TM, int BN, bool swap) {
    int per_cu = 5;
    while (per_cu > 1 && !ring_fits(ring_lds(elem_bytes, TM, BN, swap).list, per_cu)) --per_cu;
    return 256 * per_cu;
}
constexpr RingLaunch ring_launch(int elem_bytes, int TM, int BN, bool swap, int Mc, int K, int Nc, int batch) {
    RingList l = {};
    const int nb = Nc / BN, lds = ring_lds(elem_bytes, TM, BN, swap).list;
    l.n_mtiles = (Mc + TM - 1) / TM;
    int parts = 1;
    // panels that do not deal out evenly are cut by columns, unless the copies of the dense operand that
    // every further XCD then reads cost more than the idle ones (64 MB: about 10 us)
    if (l.n_mtiles < 64)
        while (parts < 8 && (int64_t)l.n_mtiles * parts % 8 != 0 &&
               (int64_t)Mc * K * elem_bytes * 2 * parts <= (64 << 20)) parts *= 2;
    l.parts_log2 = parts == 8 ? 3 : parts >> 1;
    l.cols = (nb + parts - 1) / parts;
    const int64_t panel = (int64_t)TM * K * elem_bytes;
    l.group = panel >= (2 << 20) ? 1 : (int)((2 << 20) / panel);
    // At most four workgroups to a CU, and a fifth where it saves a round: 64-row tiles of 2992 x 768 -> 3072 bf16 13.4 ->
    // 11.6 us with it, of 5000 x 2048 -> 1024 fp16 20.9 -> 18.1, of 3713 x 1280 -> 640 bf16 11.9 -> 9.1; but of 3699 x 3328 -> 832
    // bf16 20.0 -> 22.7, two rounds either way.
    const RingLaunch four = ring_launch_of(l, lds, 4, batch), five = ring_launch_of(l, lds, 5, batch);
    int per_cu = ring_rounds(five.n_list, five.n_pos) < ring_rounds(four.n_list, four.n_pos) ? 5 : 4;
    while (per_cu > 1 && !ring_fits(ring_launch_of(l, lds, per_cu, batch).smem, per_cu)) --per_cu;
    return ring_launch_of(l, lds, per_cu, batch);
}

// Live blocks of a sparse operand that the choice of a kernel and of its launch counts on: every eighth place where they are not
// counted on the host (a dense operand under a mask, a compressed one kept at the capacity of its index).
constexpr int64_t spmm_live_blocks(bool counted, int64_t stored, int64_t places) { return counted ? stored : places / 8; }

// 64-row tiles, log2 of the parts that a block-column is cut into, each a tile of its own, where every tile then still has a
// workgroup to itself.  fp32: as narrow as it gets, a tile's MFMAs are most of its time (64 x 64 blocks at 30 - 40 %, us: 52 x 1600 -> 3584
// 20.9, in halves 13.6, in quarters 10.4; gradients of the input 64 x 2688 -> 1408 24.9 / 15.1 / 12.8, 304 x 1856 -> 1088 21.7 / 13.8 /
// 12.8; 1024^3 at 20 % 12.4 / 10.4 / 9.9; 32 x 64 blocks 903 x 3200 -> 512 12.4 / 11.8; no size behind).  16-bit types: 64-wide blocks in
// halves, where that fills idle CUs (1 x 1024 -> 4096 (64 tiles) 7.0 / 5.8, 109 x 2944 -> 576 9.5 / 8.4, 185 x 1536 -> 1728 (81) 6.0 / 5.4;
// 129 x 640 -> 2688 (126) 4.1 / 4.5, 208 x 2432 -> 3264 (204) 10.2 / 11.0; 32-wide blocks lose, 304 x 896 -> 2944 7.8 / 8.3).
constexpr int ring_sub_log2(int elem_bytes, int BN, bool swap, int Mc, int K, int Nc, int batch) {
    int sub = elem_bytes == 4 ? (BN == 64 ? 2 : BN == 32 ? 1 : 0) : BN == 64 && (int64_t)((Mc + 63) / 64) * (Nc / BN) * batch <= 96 ? 1 : 0;
    for (; sub > 0; --sub) {
        const RingLaunch l = ring_launch(elem_bytes, 64, BN >> sub, swap, Mc, K, Nc, batch);
        if (l.n_pos == l.n_list) break;
    }
    return sub;
}
// Groups of wavefronts that share the walk of a tile out, where each tile has a workgroup to itself: three where the workgroups have
// a CU each, two where two share one (`n_pos`: workgroups of an XCD, 32 CUs).  stages: of a walk, on the average.  One, two and
// three groups, us: fp16 64 x 64 blocks at 30 - 40 %, gradient of the input 416 x 4032 -> 1152 (126 tiles) 18.4 / 13.6 / 11.6, 416 x 1152 -> 4032 (441) 8.8 /
// 7.0 / 11.2, 816 x 4032 -> 1472 (663) 11.4 / 12.8 / 16.5, 128 x 3392 -> 2816 12.0 / 9.0 / 8.2, 4 x 3264 -> 2112 9.5 / 7.2 / 6.6; bf16 32 x 32 blocks, gradient of
// 304 x 2944 -> 896 15.2 / 9.8 / 8.4; fp32 46 x 4096 -> 960 at 34 % 15.4 / 12.4 / 12.0, 512 x 1408 -> 896 (448) 7.6 / 7.6 / 9.4, 304 x 1088 -> 1856 (580)
// 10.5 / 11.4 / 13.6.  Walks of two stages: 288 x 2112 -> 2560 at 6 % 5.7 / - / 6.5.
// fp32 tiles wider than 16: one.  Block-columns are cut narrower wherever every tile then still has a workgroup, so there are
// over 64 of these to an XCD.
constexpr int ring_most_groups(int elem_bytes, int BN) { return elem_bytes == 4 && BN > 16 ? 1 : 3; }
constexpr int ring_groups(int elem_bytes, int BN, bool swap, int n_pos, double stages) {
    if (ring_most_groups(elem_bytes, BN) == 1) return 1;
    const RingLds lds = ring_lds(elem_bytes, 64, BN, swap);
    int groups = stages < 2.5 ? 1 : n_pos <= 32 ? 3 : n_pos <= 64 ? 2 : 1;
    while (groups > 1 && !ring_fits(lds.list + (groups - 1) * ring_stages(elem_bytes) * lds.stage, n_pos <= 32 ? 1 : 2)) --groups;
    return groups;
}

// 16-bit results in rows of 64 bytes, k-contiguous operands, with an activation: whether they are written through to the last-level
// cache, which non-temporal stores go past.  The next product then reads them from there.  Feed-forward blocks K -> N -> K, fp16, both products
// with the hint / with this, us: 8192 x 768 -> 3072 38.4 / 33.4, 8192 x 1024 -> 2048 38.3 / 35.5, 8192 x 512 -> 2048 32.7 / 30.1, 12345 x 1024 -> 2048
// 55.0 / 50.3; between 5121 and 8192 rows level (5200 x 768 -> 3072 32.5 / 32.6, 6000 rows 32.9 / 33.3, 7000 rows 35.8 / 35.4, 6500 x 1024 -> 2048 37.4 / 37.8,
// 5700 x 1024 -> 4096 42.1 / 41.7), with blocks of depth 32 too (8192 x 768 -> 3072 49.1 / 49.0).
// Refused, as a product on its own takes up to 7 % longer: fewer rows (4096 x 768 -> 2304 10.8 / 11.5, 4000 x 1024 -> 4096 15.0 / 15.7, though
// some pairs would gain, 4096 x 1024 -> 4096 33.6 / 30.6 and 2767 x 512 -> 1024 12.4 / 11.3) and results that are no wider than twice the depth
// (8192 x 2048 -> 1024 19.1 / 20.1, 16384 x 1024 -> 1024 16.5 / 17.2); and panels whose columns, and with them the lines of a row, several
// XCDs share out (2314 x 704 -> 1408 in eight parts, the pair 18.2 / 19.4).  Results without an activation keep the hint, from which a product
// on its own gains 1 - 3 % (9235 x 1024 -> 2176 24.0 / 24.4, 2423 x 2176 -> 2624 20.1 / 20.7); plain stores take 0.4 - 2 us longer than either.
constexpr bool ring_results_through(int Mc, int K, int Nc, int parts_log2) { return Mc > 5120 && Nc >= 2 * K && parts_log2 <= 1; }

}  // namespace spx
