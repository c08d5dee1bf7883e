// What the launcher and the workgroups of the persistent gathered GEMM (moe_persist.hip) have to agree on: the LDS layout, the
// length of a workgroup's list of tiles, and which problems fit it.  Plain C++ without device code, so that a host program can
// ask it about any size.
#pragma once
#include <cstdint>

namespace spx {

constexpr int kPersistThreads = 512, kPersistSlot = 512 * 128;   // a stage: rows of 128 bytes, 256 of tokens and 256 of weights
constexpr int kPersistTok = 2 * kPersistSlot;                    // token ids of two tiles
constexpr int kPersistList = kPersistTok + 2 * 256 * 4;          // the workgroup's tiles
constexpr int kPersistLds = 160 * 1024;
struct alignas(16) PersistTile {
    int expert, row0, rows, n0;   // expert < 0: no tile
};

constexpr int persist_workgroups(int n_cu) { return n_cu < 8 ? 8 : n_cu & ~7; }

// Tiles of a workgroup, at most: of 256 rows (a last one to every expert, and to the tokens without one) and 256 columns, dealt out
// over all workgroups, and one round of pieces.
constexpr int64_t persist_rounds(int n_tok, int N, int n_exp, int n_wg) {
    const int64_t row_tiles = n_tok / 256 + (int64_t)n_exp + 1, col_tiles = ((int64_t)N + 255) / 256;
    return (row_tiles * col_tiles + n_wg - 1) / n_wg + 1;
}

// Four stages to a tile: the token ids of the next one arrive meanwhile.  Byte offsets in 32 bits: of all tokens, and of the weights of
// a tile, 64 rows of k ([E, in, out]) or 256 rows of columns ([E, out, in]).  The list of tiles in LDS.
constexpr bool persist_fits(int n_tok, int K, int N, int n_exp, bool w_kcontig, int n_cu) {
    const int64_t limit = (int64_t)1 << 32;
    return K >= 256 && (int64_t)n_tok * K * 2 < limit && (w_kcontig ? (int64_t)K * 512 : (int64_t)N * 128) < limit &&
           persist_rounds(n_tok, N, n_exp, persist_workgroups(n_cu)) * (int64_t)sizeof(PersistTile) <= kPersistLds - kPersistList;
}

}  // namespace spx
