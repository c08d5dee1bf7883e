// Backward pass of fused block-sparse attention without stored probabilities: 32 queries (row side) or
// 32 keys (column side) per wavefront, 32 x 32 x 16 MFMAs.
#include <type_traits>
#include "attention.hpp"

namespace spx {

// ---- the two kernels ---------------------------------------------------------------------------------
// One workgroup per block row (row side: dQ) or block column (column side: dK, dV) and batch entry, a wavefront per
// 32 queries (keys).  The other side is walked in tiles of 32 rows, K and V or Q and dO, which go global -> LDS
// directly through a ring of three stages; the wavefronts share the loads of a stage and meet at one barrier per stage.
// The slots of the ring are constants (the walk is unrolled by three), so LDS addresses cost no arithmetic.
//   row side, per 32 keys:      S^T = K Q^T, dP^T = V dO^T, dS = P o (dP - D) / T, dQ^T += K^T dS^T
//   column side, per 32 queries: S = Q K^T, dP = dO V^T, dV^T += dO^T P, dK^T += Q^T dS
// P = exp2(S log2(e) / T - L) from the row statistic of the forward kernel; the accumulators hold P and dS in the
// layout that the last products read as B operand.
// Without an element mask Q and dO (K and V) are scaled to 16 bits first and the accumulators start at -L and
// -D / T, as in the kernels with 16 queries per wavefront; the row side scales S in fp32 instead (F32S) where the row
// statistic is of such scores.  With a mask all scaling stays in fp32, as it was where the probabilities were stored (relative error of dQ, dK, dV, causal window fp16: 4.2e-4, 4.1e-4, 3.5e-4 there,
// 3.1e-4, 3.1e-4, 3.0e-4 here).  The scaling in fp32 costs 10 % of the time.
// The element mask is the [Nt, Ns] tensor, or its live blocks one after the other in BCSR order (a training step keeps
// those: the caller's tensor may hold another mask by then, and all of it is more than a long sequence can spare).
//
// What bounds them: the matrix cores at the clock the chip holds.  Per 32 x 32 scores a wavefront spends 384 (512) clocks on
// MFMAs and reads 12 (16) KB of LDS, half of what 16 queries per wavefront need; a stage of the column side takes
// 2400 clocks with three wavefronts on a SIMD, i.e. 63 % of its MFMA rate, and the clock falls to 1.75 GHz
// (2.2 in kernels with fewer MFMAs).  96 x 4096 x 64 fp16, 392 blocks of 64 x 64: row side 87 -> 77 us, column side 111 -> 93
// (58 and 77 GFLOP: 750 and 830 TFLOP/s); without the tile loads 66 and 82, without exponentials 92, without LDS reads 88.
// Left out, no gain: four stages, two stages, loads requested later in a stage, raised wave priority.
// Head dim 128, row side only: two stages, for four workgroups of two wavefronts to a CU.  24 x 3200 positions, 202 blocks of
// 64 x 64 to a head, fp16 38.3 (16 queries per wavefront) -> 34.2 us, with an element mask 37.8 (stored probabilities) -> 37.7.  On
// the column side the accumulators of 32 keys and their rows of K and V are 192 registers: what is spilled is read
// back behind the loads of the next stage (41 -> 45 us), and with one wavefront to a SIMD nothing covers it.  Two wavefronts to
// 32 queries that share the keys out lose as well (34 -> 39 us, though 12 x 1024 12.7 -> 11.8).
constexpr int bwd_stages(int E) { return E == 64 ? 3 : 2; }
template <int E, int WAVES, bool HAS_MASK, bool STATS> struct BwdLds {
    static constexpr int NB = bwd_stages(E);
    static constexpr int MASK = 2 * AttnTile<E>::BYTES;                          // 32 x 32 bytes per wavefront
    static constexpr int STAT = MASK + (HAS_MASK ? WAVES * 1024 : 0);            // 32 + 32 floats per wavefront
    static constexpr int STAGE = STAT + (STATS ? WAVES * 256 : 0);
    static constexpr int OUT = WAVES * 32 * (AttnTile<E>::ROW + 16);             // output rows, in the same space
    static constexpr int TOTAL = NB * STAGE > OUT ? NB * STAGE : OUT;
};

// ---- row side -----------------------------------------------------------------------------------
template <typename T, int E, int WAVES, bool HAS_MASK, bool F32S>
__global__ __launch_bounds__(64 * WAVES, HAS_MASK || E == 128 ? 2 : 3) void attention_bwd_row_wide_kernel(AttnParams p, int nbr, int log_sub, int batch) {
    typedef AttnTile<E> Tile;
    typedef BwdLds<E, WAVES, HAS_MASK, false> Lds;
    constexpr int EC = Tile::EC, ET = Tile::ET, NB = Lds::NB;
    constexpr int LPT = 2 * Tile::LOADS / WAVES;             // tile loads of a wavefront and stage
    constexpr int LPW = LPT + (HAS_MASK ? 1 : 0);
    typedef typename MmaW<T>::frag Frag;
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    extern __shared__ __align__(16) char smem[];

    // workgroup L runs on XCD L % 8: give each XCD whole batch*head entries
    const int L = blockIdx.x;
    const int slot = L >> 3;
    const int64_t b = (slot / nbr) * 8 + (L & 7);
    const int br = slot % nbr;
    if (b >= batch) return;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Tile tile(lane);
    const int l32 = tile.l32, h2 = tile.h2;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

    const int row0 = br * (32 * WAVES) + wave * 32;
    const int64_t qoff = (b * p.Nt + row0 + l32) * E;
    const T* Kg = reinterpret_cast<const T*>(p.k) + b * (int64_t)p.Ns * E;
    const T* Vg = reinterpret_cast<const T*>(p.v) + b * (int64_t)p.Ns * E;

    // what the wavefront keeps is requested ahead of the index and of the first tiles
    Frag gf[EC], qf[EC], o_raw[EC];
#pragma unroll
    for (int c = 0; c < EC; ++c) {
        const int64_t at = qoff + c * 16 + h2 * 8;
        gf[c] = *reinterpret_cast<const Frag*>(reinterpret_cast<const T*>(p.grad_out) + at);
        qf[c] = *reinterpret_cast<const Frag*>(reinterpret_cast<const T*>(p.q) + at);
        o_raw[c] = *reinterpret_cast<const Frag*>(reinterpret_cast<const T*>(p.out) + at);
    }
    const float lse = p.row_lse[b * p.Nt + row0 + l32];
    const int e_begin = p.row_ptr[br];
    const int n_ent = p.row_ptr[br + 1] - e_begin;
    const int n = n_ent << log_sub;
    int bc_vec = 0;
    if (lane < n_ent) bc_vec = p.bcsr_idx[e_begin + lane] & 0xffff;
    auto key0_at = [&](int i) {
        const int e = i >> log_sub;
        const int col = e < 64 ? __builtin_amdgcn_readlane(bc_vec, e) : __builtin_amdgcn_readfirstlane(p.bcsr_idx[e_begin + e] & 0xffff);
        return ((col << log_sub) + (i & ((1 << log_sub) - 1))) * 32;
    };
    // the rows of this wavefront in the mask, or in the live blocks of its block row, which follow each other
    const int mask_ld = p.mask_blocks ? 32 << log_sub : p.Ns;
    const uint8_t* const mask = p.mask + (p.mask_blocks ? (int64_t)e_begin * (32 * WAVES) + wave * 32 : (int64_t)row0) * mask_ld;
    auto mask_column = [&](int i, int key0) {
        return p.mask_blocks ? ((((i >> log_sub) * (32 * WAVES)) << log_sub) + (i & ((1 << log_sub) - 1))) * 32 : key0;
    };
    auto issue = [&](int i, int at) {
        const int key0 = key0_at(i);
        const uint32_t to = lds0 + at;
        if constexpr (WAVES == 1) {
            tile.template request<LPT / 2>(Kg + (int64_t)key0 * E, 0, to);
            tile.template request<LPT / 2>(Vg + (int64_t)key0 * E, 0, to + Tile::BYTES);
        } else {   // the first half of the wavefronts brings K, the others V
            const T* from = wave < WAVES / 2 ? Kg : Vg;
            tile.template request<LPT>(from + (int64_t)key0 * E, (wave & (WAVES / 2 - 1)) * LPT, to + (wave < WAVES / 2 ? 0 : Tile::BYTES));
        }
        if constexpr (HAS_MASK)
            lds_direct_load16_at(mask + mask_column(i, key0), (lane >> 1) * mask_ld + (lane & 1) * 16, to + Lds::MASK + wave * 1024);
    };

#pragma unroll
    for (int s = 0; s < NB - 1; ++s)
        if (s < n) issue(s, s * Lds::STAGE);
    const float c2 = p.inv_t * 1.4426950408889634f;
    float d_part = 0.f;
#pragma unroll
    for (int c = 0; c < EC; ++c) {
        f32x8 gs, qs;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            gs[j] = (float)gf[c][j] * p.inv_t;
            qs[j] = (float)qf[c][j] * c2;
            d_part += gs[j] * (float)o_raw[c][j];
        }
        if constexpr (!HAS_MASK) gf[c] = AttnPack<T>::pack(gs);
        if constexpr (!F32S) qf[c] = AttnPack<T>::pack(qs);
    }
    const float d_row = xor32_sum(d_part);   // D / T
    if (p.row_dot && h2 == 0) p.row_dot[b * p.Nt + row0 + l32] = d_row;
    f32x16 s0, dp0;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        s0[j] = F32S ? 0.f : -lse;
        dp0[j] = HAS_MASK ? 0.f : -d_row;
    }
    f32x16 qacc[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) qacc[t][j] = 0.f;

    // the slots are constants, so the offsets of the LDS reads are too
    auto step = [&](int i, auto slot) {
        constexpr int at = slot * Lds::STAGE, fill = (slot + NB - 1) % NB * Lds::STAGE;
        if (NB > 2 && i + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();   // stage i has landed, stage i - 1 has been read
        const char* kt = smem + at;
        const char* vt = kt + Tile::BYTES;
        if (i + NB - 1 < n) issue(i + NB - 1, fill);

        f32x16 s = s0, dp = dp0;
#pragma unroll
        for (int c = 0; c < EC; ++c) s = MmaW<T>::mma(tile.template row_frag<Frag>(kt, c), qf[c], s);
#pragma unroll
        for (int c = 0; c < EC; ++c) dp = MmaW<T>::mma(tile.template row_frag<Frag>(vt, c), gf[c], dp);
#pragma unroll
        for (int j = 0; j < 16; ++j) s[j] = __builtin_amdgcn_exp2f(F32S ? __builtin_fmaf(s[j], c2, -lse) : s[j]);
        if constexpr (HAS_MASK) {
            unsigned live[4];
            const char* m = kt + Lds::MASK + wave * 1024 + l32 * 32 + h2 * 4;
#pragma unroll
            for (int a = 0; a < 4; ++a) live[a] = *reinterpret_cast<const uint32_t*>(m + a * 8);
            if (__builtin_amdgcn_ballot_w64((live[0] & live[1] & live[2] & live[3]) != 0x01010101u) != 0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) s[j] = ((live[j >> 2] >> (8 * (j & 3))) & 0xffu) ? s[j] : 0.f;
            }
        }
        Frag sf[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f32x8 ds;
#pragma unroll
            for (int j = 0; j < 8; ++j) ds[j] = s[8 * u + j] * (HAS_MASK ? __builtin_fmaf(dp[8 * u + j], p.inv_t, -d_row) : dp[8 * u + j]);
            sf[u] = AttnPack<T>::pack(ds);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int t = 0; t < ET; ++t) qacc[t] = MmaW<T>::mma(tile.template tr_frag<Frag>(kt, t, u), sf[u], qacc[t]);
    };
    for (int i = 0; i < n; i += NB) {
        step(i, std::integral_constant<int, 0>());
        if (i + 1 < n) step(i + 1, std::integral_constant<int, 1>());
        if constexpr (NB > 2)
            if (i + 2 < n) step(i + 2, std::integral_constant<int, 2>());
    }
    __syncthreads();   // the tiles are dead: their space carries the output rows
    store_rows32<T, E>(smem + wave * (32 * (E * 2 + 16)), reinterpret_cast<T*>(p.grad_q) + (b * p.Nt + row0) * E, qacc, lane);
}

// ---- column side --------------------------------------------------------------------------------
template <typename T, int WAVES, bool HAS_MASK>
__global__ __launch_bounds__(64 * WAVES, HAS_MASK ? 2 : 3) void attention_bwd_col_wide_kernel(AttnParams p, int nbc, int log_sub, int batch) {
    typedef AttnTile<64> Tile;
    typedef BwdLds<64, WAVES, HAS_MASK, true> Lds;
    constexpr int E = 64, EC = Tile::EC, ET = Tile::ET, NB = Lds::NB;
    constexpr int LPT = 2 * Tile::LOADS / WAVES;
    constexpr int LPW = LPT + 1 + (HAS_MASK ? 1 : 0);
    typedef typename MmaW<T>::frag Frag;
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) char smem[];

    const int L = blockIdx.x;
    const int slot = L >> 3;
    const int64_t b = (slot / nbc) * 8 + (L & 7);
    const int bc = slot % nbc;
    if (b >= batch) return;
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const Tile tile(lane);
    const int l32 = tile.l32, h2 = tile.h2;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

    const int key0 = bc * (32 * WAVES) + wave * 32;
    const T* Qg = reinterpret_cast<const T*>(p.q) + b * (int64_t)p.Nt * E;
    const T* Gg = reinterpret_cast<const T*>(p.grad_out) + b * (int64_t)p.Nt * E;
    // lanes 0 .. 31 fetch L of the queries of a tile, lanes 32 .. 63 their D / T
    const float* stat = (h2 ? p.row_dot : p.row_lse) + b * (int64_t)p.Nt + l32;

    Frag vf[EC], kf[EC];   // rows of this lane's key: requested ahead of the index and of the first tiles
#pragma unroll
    for (int c = 0; c < EC; ++c) {
        const int64_t at = (b * p.Ns + key0 + l32) * E + c * 16 + h2 * 8;
        vf[c] = *reinterpret_cast<const Frag*>(reinterpret_cast<const T*>(p.v) + at);
        kf[c] = *reinterpret_cast<const Frag*>(reinterpret_cast<const T*>(p.k) + at);
    }
    const int e_begin = p.col_ptr[bc];
    const int n_ent = p.col_ptr[bc + 1] - e_begin;
    const int n = n_ent << log_sub;
    struct Entry {
        int row, place;   // block row, and the place among the live blocks
    };
    auto entry = [&](int e) -> Entry {
        if (p.bcsc_wide) {
            const long long v = reinterpret_cast<const long long*>(p.bcsc_idx)[e];
            return {(int)(v & 0xffff), (int)(v >> 32)};
        }
        return {reinterpret_cast<const int32_t*>(p.bcsc_idx)[e] & 0xffff, e};
    };
    Entry mine = {0, 0};
    if (lane < n_ent) mine = entry(e_begin + lane);
    const int br_vec = mine.row, mask_vec = p.mask_blocks ? mine.place : mine.row;
    auto query0_at = [&](int i) {
        const int e = i >> log_sub;
        const int row = e < 64 ? __builtin_amdgcn_readlane(br_vec, e) : __builtin_amdgcn_readfirstlane(entry(e_begin + e).row);
        return ((row << log_sub) + (i & ((1 << log_sub) - 1))) * 32;
    };
    const int mask_ld = p.mask_blocks ? 32 * WAVES : p.Ns;
    const uint8_t* const mask = p.mask + (p.mask_blocks ? wave * 32 : key0);
    auto mask_row = [&](int i) -> int64_t {
        const int e = i >> log_sub;
        int block = __builtin_amdgcn_readlane(mask_vec, e & 63);
        if (e >= 64) {
            const Entry far = entry(e_begin + e);
            block = __builtin_amdgcn_readfirstlane(p.mask_blocks ? far.place : far.row);
        }
        return (((int64_t)block << log_sub) + (i & ((1 << log_sub) - 1))) * 32;
    };
    auto issue = [&](int i, int at) {
        const int q0 = query0_at(i);
        const uint32_t to = lds0 + at;
        if constexpr (WAVES == 1) {
            tile.request<LPT / 2>(Qg + (int64_t)q0 * E, 0, to);
            tile.request<LPT / 2>(Gg + (int64_t)q0 * E, 0, to + Tile::BYTES);
        } else {
            const T* from = wave < WAVES / 2 ? Qg : Gg;
            tile.request<LPT>(from + (int64_t)q0 * E, (wave & (WAVES / 2 - 1)) * LPT, to + (wave < WAVES / 2 ? 0 : Tile::BYTES));
        }
        lds_direct_load4(stat + q0, to + Lds::STAT + wave * 256);
        if constexpr (HAS_MASK)
            lds_direct_load16_at(mask + mask_row(i) * mask_ld, (lane >> 1) * mask_ld + (lane & 1) * 16, to + Lds::MASK + wave * 1024);
    };

#pragma unroll
    for (int s = 0; s < NB - 1; ++s)
        if (s < n) issue(s, s * Lds::STAGE);
    const float c2 = p.inv_t * 1.4426950408889634f;
    if constexpr (!HAS_MASK) {
        // -K * log2(e) / T and -V / T: the accumulators start at L and D / T and end as L - S and (D - dP) / T,
        // whose signs are free modifiers of the exponential and of the product
#pragma unroll
        for (int c = 0; c < EC; ++c) {
            f32x8 vs, ks;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                vs[j] = (float)vf[c][j] * -p.inv_t;
                ks[j] = (float)kf[c][j] * -c2;
            }
            vf[c] = AttnPack<T>::pack(vs);
            kf[c] = AttnPack<T>::pack(ks);
        }
    }
    f32x16 kacc[ET], vacc[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) kacc[t][j] = vacc[t][j] = 0.f;

    // the slots are constants, so the offsets of the LDS reads are too
    auto step = [&](int i, auto slot) {
        constexpr int at = slot * Lds::STAGE, fill = (slot + NB - 1) % NB * Lds::STAGE;
        if (i + 1 < n) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const char* qt = smem + at;
        const char* gt = qt + Tile::BYTES;
        if (i + NB - 1 < n) issue(i + NB - 1, fill);

        // register j of lane (l32, h2): query 8 (j / 4) + 4 h2 + j % 4, key l32
        const char* st = qt + Lds::STAT + wave * 256 + h2 * 16;
        f32x16 s, dp;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const f32x4 lse = *reinterpret_cast<const f32x4*>(st + a * 32), dot = *reinterpret_cast<const f32x4*>(st + 128 + a * 32);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                s[4 * a + x] = HAS_MASK ? 0.f : lse[x];
                dp[4 * a + x] = HAS_MASK ? 0.f : dot[x];
            }
        }
#pragma unroll
        for (int c = 0; c < EC; ++c) s = MmaW<T>::mma(tile.row_frag<Frag>(qt, c), kf[c], s);
#pragma unroll
        for (int c = 0; c < EC; ++c) dp = MmaW<T>::mma(tile.row_frag<Frag>(gt, c), vf[c], dp);
        if constexpr (HAS_MASK) {
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 lse = *reinterpret_cast<const f32x4*>(st + a * 32);
#pragma unroll
                for (int x = 0; x < 4; ++x) s[4 * a + x] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * a + x], c2, -lse[x]));
            }
            const char* m = qt + Lds::MASK + wave * 1024;
            const u32x4 mine = *reinterpret_cast<const u32x4*>(m + lane * 16);
            if (__builtin_amdgcn_ballot_w64((mine[0] & mine[1] & mine[2] & mine[3]) != 0x01010101u) != 0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) s[j] = m[(8 * (j >> 2) + 4 * h2 + (j & 3)) * 32 + l32] ? s[j] : 0.f;
            }
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                const f32x4 dot = *reinterpret_cast<const f32x4*>(st + 128 + a * 32);
#pragma unroll
                for (int x = 0; x < 4; ++x) dp[4 * a + x] = s[4 * a + x] * __builtin_fmaf(dp[4 * a + x], p.inv_t, -dot[x]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                s[j] = __builtin_amdgcn_exp2f(-s[j]);
                dp[j] = s[j] * -dp[j];
            }
        }
        Frag pf[2], sf[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            f32x8 pv, ds;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                pv[j] = s[8 * u + j];
                ds[j] = dp[8 * u + j];
            }
            pf[u] = AttnPack<T>::pack(pv);
            sf[u] = AttnPack<T>::pack(ds);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int t = 0; t < ET; ++t) {
                vacc[t] = MmaW<T>::mma(tile.tr_frag<Frag>(gt, t, u), pf[u], vacc[t]);
                kacc[t] = MmaW<T>::mma(tile.tr_frag<Frag>(qt, t, u), sf[u], kacc[t]);
            }
    };
    for (int i = 0; i < n; i += NB) {
        step(i, std::integral_constant<int, 0>());
        if (i + 1 < n) step(i + 1, std::integral_constant<int, 1>());
        if (i + 2 < n) step(i + 2, std::integral_constant<int, 2>());
    }
    __syncthreads();
    char* rows = smem + wave * (32 * (E * 2 + 16));
    const int64_t out = (b * p.Ns + key0) * E;
    store_rows32<T, E>(rows, reinterpret_cast<T*>(p.grad_v) + out, vacc, lane);
    store_rows32<T, E>(rows, reinterpret_cast<T*>(p.grad_k) + out, kacc, lane);
}

template <typename T, int E, int WAVES, bool HAS_MASK, bool F32S>
static int launch_bwd_row_wide_inst(const AttnParams& p, int batch, int BW, hipStream_t st) {
    constexpr int smem = BwdLds<E, WAVES, HAS_MASK, false>::TOTAL;
    const int nbr = p.Nt / p.BH;
    const int64_t groups = ((int64_t)batch + 7) / 8 * 8 * nbr;
    if (groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)groups);
    SPX_GRANT_LDS((attention_bwd_row_wide_kernel<T, E, WAVES, HAS_MASK, F32S>), smem, "attention_bwd_row_wide_kernel");
    hipLaunchKernelGGL((attention_bwd_row_wide_kernel<T, E, WAVES, HAS_MASK, F32S>), dim3((unsigned)groups), dim3(64 * WAVES), smem, st, p, nbr, ilog2(BW / 32), batch);
    SPX_LAUNCH_CHECK("attention_bwd_row_wide_kernel");
    return 0;
}

template <typename T, int WAVES, bool HAS_MASK>
static int launch_bwd_col_wide_inst(const AttnParams& p, int batch, int BW, hipStream_t st) {
    constexpr int smem = BwdLds<64, WAVES, HAS_MASK, true>::TOTAL;
    const int nbc = p.Ns / BW;
    const int64_t groups = ((int64_t)batch + 7) / 8 * 8 * nbc;
    if (groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)groups);
    SPX_GRANT_LDS((attention_bwd_col_wide_kernel<T, WAVES, HAS_MASK>), smem, "attention_bwd_col_wide_kernel");
    hipLaunchKernelGGL((attention_bwd_col_wide_kernel<T, WAVES, HAS_MASK>), dim3((unsigned)groups), dim3(64 * WAVES), smem, st, p, nbc, ilog2(p.BH / 32), batch);
    SPX_LAUNCH_CHECK("attention_bwd_col_wide_kernel");
    return 0;
}

template <typename T>
static int launch_bwd_row_wide_typed(const AttnParams& p, int batch, int BW, int E, bool fp32_scores, hipStream_t st) {
#define SPX_BWD_CASE(bh)                                                                                   \
    if (p.BH == bh && E == 64)                                                                             \
        return p.mask        ? launch_bwd_row_wide_inst<T, 64, bh / 32, true, true>(p, batch, BW, st)      \
               : fp32_scores ? launch_bwd_row_wide_inst<T, 64, bh / 32, false, true>(p, batch, BW, st)     \
                             : launch_bwd_row_wide_inst<T, 64, bh / 32, false, false>(p, batch, BW, st);   \
    if (p.BH == bh && E == 128 && p.mask) return launch_bwd_row_wide_inst<T, 128, bh / 32, true, true>(p, batch, BW, st);
    SPX_BWD_CASE(32) SPX_BWD_CASE(64)
#undef SPX_BWD_CASE
    if (p.BH == 64 && E == 128 && fp32_scores) return launch_bwd_row_wide_inst<T, 128, 2, false, true>(p, batch, BW, st);
    return fail(SPX_E_CONFIG, "the attention backward kernel does not cover query blocks of %d with head dim %d", p.BH, E);
}

template <typename T>
static int launch_bwd_col_wide_typed(const AttnParams& p, int batch, int BW, hipStream_t st) {
#define SPX_BWD_CASE(bw)                                                                        \
    if (BW == bw)                                                                               \
        return p.mask ? launch_bwd_col_wide_inst<T, bw / 32, true>(p, batch, BW, st) : launch_bwd_col_wide_inst<T, bw / 32, false>(p, batch, BW, st);
    SPX_BWD_CASE(32) SPX_BWD_CASE(64)
#undef SPX_BWD_CASE
    return fail(SPX_E_CONFIG, "the attention backward kernel does not cover key blocks of %d", BW);
}

int launch_attention_bwd_row_wide(int dtype, const AttnParams& p, int batch, int BW, int E, bool fp32_scores, hipStream_t st) {
    if (dtype == SPX_F16) return launch_bwd_row_wide_typed<_Float16>(p, batch, BW, E, fp32_scores, st);
    return launch_bwd_row_wide_typed<bf16_t>(p, batch, BW, E, fp32_scores, st);
}

int launch_attention_bwd_col_wide(int dtype, const AttnParams& p, int batch, int BW, hipStream_t st) {
    if (dtype == SPX_F16) return launch_bwd_col_wide_typed<_Float16>(p, batch, BW, st);
    return launch_bwd_col_wide_typed<bf16_t>(p, batch, BW, st);
}

}  // namespace spx
