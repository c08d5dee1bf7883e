// What the gathered GEMM kernels of the mixture of experts share: launch parameters and the list of tiles.
#pragma once
#include "common.hpp"
#include "mma.hpp"

namespace spx {

struct MoeParams {
    const void* tokens;
    const void* weight;
    void* out;
    const int32_t* expert_offset;
    const int32_t* token_perm;
    int n_tok, K, N, n_exp;
    int w_kcontig;  // weight [E, N, K] if set, else [E, K, N]
    int col_groups; // direct kernel: 0: tile (x, y) is workgroup (x, y); else see moe_tile_of_workgroup
};

// Which (expert, row tile) belongs to tile index y: one wavefront scans the per-expert
// tile counts.  Expert n_exp is the pseudo expert of the tokens whose id was out of
// range (token_perm[expert_offset[n_exp] .. n_tok)): its tiles are zero-filled instead
// of multiplied.  found_e = -1 when y is past the last tile.
//
// The row tiles are numbered with every expert's full tiles first
// and the partly filled last tiles of the experts behind them (longest first).  Workgroups start in the order
// of their tile numbers, so the short tiles (a partly filled tile skips the work of its empty
// 64-row groups) fill the end of the launch, where the long ones would leave most CUs idle.
template <int TM>
__device__ __forceinline__ void moe_find_tile(const MoeParams& p, int y, int lane,
                                                     int& found_e, int& found_row0, int& found_rows) {
    int total_full = 0;
    for (int e0 = 0; e0 <= p.n_exp; e0 += 64) {
        const int e = e0 + lane;
        int cnt = 0;
        if (e <= p.n_exp) cnt = (e < p.n_exp ? p.expert_offset[e + 1] : p.n_tok) - p.expert_offset[e];
        total_full += __shfl(wave_inclusive_scan(cnt / TM), 63, 64);
    }
    const bool part = y >= total_full;   // looking for a partly filled tile
    const int want = part ? y - total_full : y;
    int before = 0;
    found_e = -1; found_row0 = 0; found_rows = 0;
    if (part && p.n_exp < 64) {
        // at most 64 candidates: the partly filled tiles go out longest first (rank = number of
        // experts whose last tile holds more rows, ties in expert order)
        int cnt = 0, off = 0;
        if (lane <= p.n_exp) {
            off = p.expert_offset[lane];
            cnt = (lane < p.n_exp ? p.expert_offset[lane + 1] : p.n_tok) - off;
        }
        const int full = cnt / TM, rest = cnt - full * TM;
        int rank = 0;
        for (int o = 0; o <= p.n_exp; ++o) {
            const int r = __shfl(rest, o, 64);
            rank += (r > rest || (r == rest && o < lane)) ? 1 : 0;
        }
        const unsigned long long hit = __ballot(rest > 0 && rank == want);
        if (hit) {
            const int src = __ffsll((long long)hit) - 1;
            found_e = src;
            found_row0 = __shfl(off, src, 64) + __shfl(full, src, 64) * TM;
            found_rows = __shfl(rest, src, 64);
        }
        return;
    }
    for (int e0 = 0; e0 <= p.n_exp; e0 += 64) {
        const int e = e0 + lane;
        int cnt = 0, off = 0;
        if (e <= p.n_exp) {
            off = p.expert_offset[e];
            cnt = (e < p.n_exp ? p.expert_offset[e + 1] : p.n_tok) - off;
        }
        const int full = cnt / TM, rest = cnt - full * TM;
        const int tiles = part ? (rest ? 1 : 0) : full;
        const int inc = wave_inclusive_scan(tiles);
        const int excl = before + inc - tiles;
        const unsigned long long hit = __ballot(want >= excl && want < excl + tiles);
        if (hit) {
            const int src = __ffsll((long long)hit) - 1;
            const int lt = want - __shfl(excl, src, 64);
            found_e = e0 + src;
            found_row0 = __shfl(off, src, 64) + (part ? __shfl(full, src, 64) : lt) * TM;
            found_rows = part ? __shfl(rest, src, 64) : TM;
            return;
        }
        before += __shfl(inc, 63, 64);
    }
}

// Zero rows token_perm[row0 .. row0 + rows) of `out`, columns n0 .. n0 + TN (16-byte stores).
template <typename T>
__device__ __forceinline__ void moe_zero_tile(const MoeParams& p, int row0, int rows, int n0, int TN, int nthreads) {
    constexpr int VE = 16 / (int)sizeof(T);
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    T* out = reinterpret_cast<T*>(p.out);
    const int ncol = (min(n0 + TN, p.N) - n0) / VE;  // N is a multiple of VE
    for (int v = threadIdx.x; v < rows * ncol; v += nthreads) {
        const int r = v / ncol, c = v - r * ncol;
        const int tok = p.token_perm[row0 + r];
        *reinterpret_cast<u32x4*>(out + (int64_t)tok * p.N + n0 + c * VE) = u32x4{0u, 0u, 0u, 0u};
    }
}

// moe_persist.hip: 256 x 256 tiles by workgroups that stay on their CU (16-bit types; what persist_fits takes)
template <typename T> int launch_moe_persist(const MoeParams& p, int n_cu, hipStream_t st);

}  // namespace spx
