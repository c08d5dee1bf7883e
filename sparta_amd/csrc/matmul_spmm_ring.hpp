// Sparse-operand matmul through a ring of LDS stages filled by direct loads:
//     out[m, n] = sum_k D[m, k] S[k, n]   (canonical problem of matmul_spmm.hpp, every layout).
//
// A workgroup is four multiplying wavefronts and a loader.  It walks its list of TM x BN output tiles; a
// multiplying wavefront owns TM / 4 rows of a tile.  The walk over the live blocks of a block-column
// is cut into halves of 64 bytes of k (16 fp32 or 32 16-bit values); a stage holds two halves - of one block
// or of two - of the TM dense rows and of the sparse block.  The loader brings stages global -> LDS
// directly (global_load_lds_dwordx4), one or two ahead of the multiplications and across tile
// boundaries; one barrier per stage hands them over.
//
// What bounds it.  fp32: the matrix cores (a 16x16x4 MFMA takes 32 clocks), 57 % of their rate on the
// 4096 x 3072 x 768 product at 20 %.  16-bit types: the L1s, as in the other kernels of this family, or the
// output.  Why a loader wavefront: loads and stores of a wavefront share one in-order counter, so a
// workgroup that loads its own next tile waits for the stores of the last one first, and the
// index look-ups and addresses (some 90 scalar instructions per stage) stand between the barrier and the
// MFMAs.  Measured on that product (fp32): the kernel without a pipeline it replaces 110 us; each wavefront
// loading its share, a workgroup per tile 51; the same walking several tiles 52; with the loader 44, with the
// balanced tile list below 38.  Fragments fetched one stage ahead of the MFMAs, and a fourth stage, were slower.
//
// Layouts in LDS (bytes are the same for every type: 64 per row and half):
//   * k-contiguous operand: rows of 128 bytes (two halves); 16-byte chunk c of row r sits at
//     c ^ ((r >> 1) & 7), so that the 16 lanes of a fragment read hit 16 different places of
//     two rows' 256 bytes;
//   * the other way round ([k][m] or [k][n]): the k-rows of a half as they are in memory, 32-byte
//     (16-bit types, LDS transpose reads) or 64-byte units (fp32, 4-byte reads) permuted by the
//     k-row so that rows read together differ in their banks where the row is long enough.
// The permutation is applied to the source address: a direct load writes lane after lane.
//
#pragma once
#include <type_traits>
#include "matmul_spmm_panel.hpp"
#include "matmul_spmm_ring_plan.hpp"

namespace spx {

// unit permutation of k-row k for rows of PITCH bytes; UNITS = units per row (power of two)
template <typename T, int PITCH> __device__ __forceinline__ int ring_row_swizzle(int k) {
    if constexpr (sizeof(T) == 2) {   // 32-byte units; a transpose read touches k-rows 0..3 (+4) of groups of 8
        if constexpr (PITCH >= 256) return (k & 3) | (((k >> 3) & 1) << 2);
        else if constexpr (PITCH == 128) return ((k >> 1) & 1) | (((k >> 3) & 1) << 1);
        else if constexpr (PITCH == 64) return (k >> 3) & 1;
        else return 0;
    } else {                          // 64-byte units; a read touches one k-row of each group of 4
        if constexpr (PITCH >= 256) return (k >> 2) & 3;
        else if constexpr (PITCH == 128) return (k >> 2) & 1;
        else return 0;
    }
}

// One fragment (16 rows, 64 bytes of k) of an operand part in LDS.  KC: k-contiguous rows.
// `row0`: first of the 16 rows; `half`: which half; ROWS: rows of the part.
template <typename T, int ROWS, bool KC, typename Frag>
__device__ __forceinline__ Frag ring_frag(const char* part, int row0, int half, int r16, int g4) {
    if constexpr (KC) {
        const int row = row0 + r16;
        return *reinterpret_cast<const Frag*>(part + row * 128 + (((half * 4 + g4) ^ ((row >> 1) & 7)) << 4));
    } else if constexpr (sizeof(T) == 2) {
        typedef short s16x8_t __attribute__((ext_vector_type(8)));
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;
        constexpr int PITCH = ROWS * 2;
        const int k = g4 * 8 + (r16 >> 2);           // and k + 4, which has the same permutation but for bit 2
        const char* base = part + half * ROWS * 64 + k * PITCH + (r16 & 3) * 8;
        const int u = row0 >> 4;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(base + ((u ^ ring_row_swizzle<T, PITCH>(k)) << 5)));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(base + 4 * PITCH + ((u ^ ring_row_swizzle<T, PITCH>(k + 4)) << 5)));
        return __builtin_bit_cast(Frag, (s16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
        constexpr int PITCH = ROWS * 4;
        Frag f;
        const char* base = part + half * ROWS * 64 + r16 * 4;
        const int u = row0 >> 4;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = g4 * 4 + j;
            f[j] = *reinterpret_cast<const float*>(base + k * PITCH + ((u ^ ring_row_swizzle<T, PITCH>(k)) << 6));
        }
        return f;
    }
}

// ONE: no workgroup has more than one tile.  GROUPS (then only): so many times four multiplying wavefronts, a loader and a ring
// share the blocks of the tile out; the first group adds up what the others hold.  CUT: a tile may be a part of a block-column
// (p.sub_log2); without it the loader has fewer scalar instructions to a stage (1024^3 fp32 at 35 %, blocks of 16 x 16, 15.2 -> 14.4 us).
template <typename T, int TM, int BN, int BK, bool DK, bool SK, bool SWAP, bool ONE, bool CUT = false, int GROUPS = 1>
__global__ __launch_bounds__(kRingThreads * GROUPS, 3) void spmm_ring_kernel(SpmmParams p, RingList l) {
    static_assert((GROUPS == 1 && !CUT) || (ONE && TM == 64), "the walk of a single 64-row tile is shared out, and its block-column cut");
    typedef typename PanelMma<T>::M MMA;
    typedef typename MMA::frag Frag;
    constexpr int ES = (int)sizeof(T), E16 = 16 / ES;
    constexpr RingLds LDS = ring_lds(ES, TM, BN, SWAP);
    constexpr int KC = 64 / ES;               // k per half
    constexpr int CH = BK / KC;               // halves per block
    constexpr int MT = TM / 64, NT = BN / 16; // 16 x 16 tiles of a wavefront
    // fp32 blocks 16 wide: the sum of a tile in four chains of MFMAs, by half and by the parity of their k-step, added up at
    // the end.  They are as long as those of four wavefronts that share a block-column (matmul_spmm_ksplit.hpp), and
    // neighbouring MFMAs of a wavefront with one tile do not wait for each other.  1024^3 at 35 %: relative error 3.4e-7 in one
    // chain, 1.8e-7 in four, 15.3 and 15.0 us (split columns 16.4).
    constexpr int CHAINS = ES == 4 && NT == 1 ? 4 : 1;
    constexpr int NB = ring_stages(ES), D_BYTES = TM * 128, STAGE = LDS.stage;
    constexpr int ND = TM / 8, NS = BN / 8;   // load instructions of a stage: dense and sparse part
    constexpr int NL = ND + NS;
    // Blocks of an even number of halves: a stage is one piece of one block.  Blocks of one half: a stage
    // is two blocks, and the last one may be half empty.
    constexpr bool PAIR = CH == 1;
    constexpr int SPB = PAIR ? 1 : CH / 2;    // stages per block
    constexpr int HK = PAIR ? 0 : KC;         // k between the halves of a stage
    static_assert(BK % KC == 0, "block depth must be a multiple of the half stage");
    typedef const __attribute__((address_space(4))) int32_t* const_i32;     // read through the scalar cache
    typedef const __attribute__((address_space(4))) int64_t* const_i64;
    extern __shared__ __align__(16) char smem[];
    constexpr int TILE = GROUPS * NB * STAGE;   // the output tile, behind the rings

    const int nb = p.Nc / BN;
    // the tiles of this workgroup's XCD, and its place among the workgroups there
    const int xcd = blockIdx.x & 7, pos = blockIdx.x >> 3, n_pos = gridDim.x >> 3;
    const RingShare share = ring_share(l, xcd, n_pos);
    if (pos >= share.n_list) return;
    const int64_t b = blockIdx.y;
    const int lane = lane_id();
    const int wave_of = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int group = GROUPS > 1 ? wave_of / 5 : 0, wave = GROUPS > 1 ? wave_of % 5 : wave_of;
    char* const ring = smem + group * (NB * STAGE);

    const int n_rounds = ONE ? 1 : share.n_rounds;
    const bool listed = !ONE && share.listed, table = listed && nb <= kRingTableMax;
    RingTile* const list = reinterpret_cast<RingTile*>(smem + LDS.list);
    struct Tile {
        int m0, j, e0, n_blk, n_st, n_bar;   // n_bar: stages of the group that has most
    };
    auto stages = [](int n_blk) { return PAIR ? (n_blk + 1) >> 1 : n_blk * SPB; };
    // launch order and column pointers while the list is made: in the ring, which is empty yet
    int* const tab_ptr = reinterpret_cast<int*>(smem);
    int* const tab_order = tab_ptr + nb + 1;
    auto place = [&](int r, int& mt, int& o) __attribute__((always_inline)) -> bool {
        return ring_place<ONE>(l, share, xcd, pos, n_pos, nb, r, mt, o);
    };
    auto look_up = [&](int r) __attribute__((always_inline)) -> RingTile {
        int mt, o;
        if (!place(r, mt, o)) return {0, 0, 0, -1};
        const int j = table ? tab_order[o] : p.sched ? p.sched[o] : o;
        const int* const ptr = table ? tab_ptr : p.ptr;
        const int e0 = ptr[j];
        return {mt * TM, j, e0, ptr[j + 1] - e0};
    };
    // all tiles of this workgroup at once, a thread each (ring_listed says where)
    if (listed) {
        if (table) {
            for (int i = threadIdx.x; i <= nb; i += kRingThreads) tab_ptr[i] = p.ptr[i];
            for (int i = threadIdx.x; i < nb; i += kRingThreads) tab_order[i] = p.sched ? p.sched[i] : i;
            __syncthreads();
        }
        for (int r = threadIdx.x; r < n_rounds; r += kRingThreads) list[r] = look_up(r);
        __syncthreads();
    }
    auto tile_at = [&](int r, Tile& t) __attribute__((always_inline)) -> bool {
        RingTile e = {0, 0, 0, -1};
        int mt, o;
        if (listed) {
            e = list[r];
        } else if (place(r, mt, o)) {   // (through the scalar cache)
            e.m0 = mt * TM;
            const int sub = CUT ? p.sub_log2 : 0, column = o >> sub;
            e.j = p.sched ? ((const_i32)p.sched)[column] : column;
            e.e0 = ((const_i32)p.ptr)[e.j];
            e.n_blk = ((const_i32)p.ptr)[e.j + 1] - e.e0;
            if constexpr (CUT) e.j = (e.j << sub) + (o & ((1 << sub) - 1));   // in tiles
        }
        t.n_blk = __builtin_amdgcn_readfirstlane(e.n_blk);
        t.m0 = __builtin_amdgcn_readfirstlane(e.m0);
        t.j = __builtin_amdgcn_readfirstlane(e.j);
        t.e0 = __builtin_amdgcn_readfirstlane(e.e0);
        const bool exists = t.n_blk >= 0;
        if constexpr (GROUPS > 1) {
            const int most = (t.n_blk + GROUPS - 1) / GROUPS, first = group * most;
            t.n_bar = stages(most);
            t.e0 += first;
            t.n_blk = t.n_blk - first < most ? t.n_blk - first : most;
            if (t.n_blk < 0) t.n_blk = 0;
        }
        t.n_st = stages(t.n_blk);
        return exists;
    };

    // Barriers, the same sequence in every wavefront: one per stage (its data has landed, and the slot
    // that is filled next has been read), one more per tile (the output tile is complete in LDS), and one
    // ahead of that for a tile without a stage (the output tile before it has left).
    if (wave == 4) {
        __builtin_amdgcn_s_setprio(3);
        // ---- the loader --------------------------------------------------------------------------------
        const T* D = reinterpret_cast<const T*>(p.D) + b * p.d_batch;
        const T* S = reinterpret_cast<const T*>(p.S) + b * p.s_batch;
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
        constexpr int USH = ES == 2 ? 5 : 6;   // log2 of a unit
        // byte offsets of this lane in the load instructions of the dense part, from the tile's first row
        // (column) and the stage's k; they fit 32 bits (checked on the host)
        uint32_t d_off[ND];
        int d_upper = 0;                       // bit q: the lane's piece belongs to the second half
        auto set_rows = [&](int m0) {
            const int last = p.Mc - 1 - m0;    // rows past the end re-read the last one; never stored
            d_upper = 0;
#pragma unroll
            for (int q = 0; q < ND; ++q) {
                if constexpr (DK) {
                    const int row = q * 8 + (lane >> 3);
                    const int chunk = (lane & 7) ^ ((row >> 1) & 7);
                    d_off[q] = ((uint32_t)(row < last ? row : last) * (uint32_t)p.d_ld + (chunk & 3) * E16 + (chunk >> 2) * HK) * ES;
                    d_upper |= (chunk >> 2) << q;
                } else {
                    constexpr int PITCH = TM * ES, IPH = TM / 16;   // instructions per half
                    const int o = (q % IPH) * 1024 + lane * 16;
                    const int k = o / PITCH + q / IPH * HK, at = o % PITCH;
                    const int col = ((((at >> USH) ^ ring_row_swizzle<T, PITCH>(o / PITCH)) << USH) + (at & ((1 << USH) - 1))) / ES;
                    d_off[q] = ((uint32_t)k * (uint32_t)p.d_ld + (col <= last ? col : 0)) * ES;
                }
            }
        };
        const int sub = CUT ? p.sub_log2 : 0;
        const int64_t sld = p.compressed ? (SK ? BK : BN << sub) : p.s_ld;
        uint32_t s_off[NS];
        int s_upper = 0;
#pragma unroll
        for (int q = 0; q < NS; ++q) {
            if constexpr (SK) {
                const int row = q * 8 + (lane >> 3);
                const int chunk = (lane & 7) ^ ((row >> 1) & 7);
                s_off[q] = ((uint32_t)row * (uint32_t)sld + (chunk & 3) * E16 + (chunk >> 2) * HK) * ES;
                s_upper |= (chunk >> 2) << q;
            } else {
                constexpr int PITCH = BN * ES, IPH = BN / 16;
                const int o = (q % IPH) * 1024 + lane * 16;
                const int k = o / PITCH + q / IPH * HK, at = o % PITCH;
                const int col = ((((at >> USH) ^ ring_row_swizzle<T, PITCH>(o / PITCH)) << USH) + (at & ((1 << USH) - 1))) / ES;
                s_off[q] = ((uint32_t)k * (uint32_t)sld + col) * ES;
            }
        }
        // ---- the load cursor: runs NB - 1 stages ahead of the multiplications, across tiles
        int ld_round = -1, ld_st = 0;
        Tile ld;
        ld.n_st = 0;
        ld.m0 = -1;
        int64_t ent_a = 0, ent_b = 0;   // index entries of its stage: (slot << 32) | k block
        auto entry = [&](int e) -> int64_t {
            if (p.idx_kind == SPX_IDX_BCSC_I64) {
                const int64_t v = ((const_i64)p.idx)[e];
                return (v & ~(int64_t)0xffffffff) | (v & 0xffff);
            }
            return ((int64_t)e << 32) | (((const_i32)p.idx)[e] & 0xffff);
        };
        auto seek = [&]() {             // to the next stage there is
            while (ld_st >= ld.n_st) {
                if (++ld_round >= n_rounds) return;
                const int m0 = ld.m0;
                ld_st = 0;
                if (!tile_at(ld_round, ld)) ld.n_st = 0;
                else if (ld.m0 != m0) set_rows(ld.m0);
            }
            if constexpr (PAIR) {
                const int e = ld.e0 + 2 * ld_st;
                ent_a = entry(e);
                ent_b = 2 * ld_st + 1 < ld.n_blk ? entry(e + 1) : ent_a;   // an odd last block: loaded twice, used once
            } else if (ld_st % SPB == 0) {
                ent_a = entry(ld.e0 + ld_st / SPB);
            }
        };
        auto s_block = [&](int64_t ent, int ch) {
            const int k = (int)(ent & 0xffff) * BK + ch * KC;
            if (p.compressed)
                return S + (ent >> 32) * (BK * BN << sub) + (ld.j & ((1 << sub) - 1)) * (SK ? BK * BN : BN) + (SK ? ch * KC : ch * KC * (BN << sub));
            return SK ? S + (int64_t)ld.j * BN * p.s_ld + k : S + (int64_t)k * p.s_ld + (int64_t)ld.j * BN;
        };
        auto issue = [&](uint32_t at) {   // the stage under the cursor into the slot at byte offset `at`
            const uint32_t to = lds0 + at;
            const T* Dm = D + (DK ? (int64_t)ld.m0 * p.d_ld : (int64_t)ld.m0);
            if constexpr (PAIR) {
                const int k_a = (int)(ent_a & 0xffff) * BK, k_b = (int)(ent_b & 0xffff) * BK;
                if constexpr (DK) {
#pragma unroll
                    for (int q = 0; q < ND; ++q)
                        lds_direct_load16_at(Dm, d_off[q] + (uint32_t)((d_upper >> q) & 1 ? k_b : k_a) * ES, to + q * 1024);
                } else {
#pragma unroll
                    for (int q = 0; q < ND; ++q)
                        lds_direct_load16_at(Dm + (int64_t)(q < ND / 2 ? k_a : k_b) * p.d_ld, d_off[q], to + q * 1024);
                }
                const T *s_a = s_block(ent_a, 0), *s_b = s_block(ent_b, 0);
#pragma unroll
                for (int q = 0; q < NS; ++q) {
                    if constexpr (SK) {
                        const char* from = reinterpret_cast<const char*>((s_upper >> q) & 1 ? s_b : s_a);
                        lds_direct_load16(from + s_off[q], to + D_BYTES + q * 1024);
                    } else {
                        lds_direct_load16_at(q < NS / 2 ? s_a : s_b, s_off[q], to + D_BYTES + q * 1024);
                    }
                }
            } else {
                const int ch = ld_st % SPB * 2;
                const int k = (int)(ent_a & 0xffff) * BK + ch * KC;
                const T* Dk = Dm + (DK ? (int64_t)k : k * p.d_ld);
                const T* sb = s_block(ent_a, ch);
#pragma unroll
                for (int q = 0; q < ND; ++q) lds_direct_load16_at(Dk, d_off[q], to + q * 1024);
#pragma unroll
                for (int q = 0; q < NS; ++q) lds_direct_load16_at(sb, s_off[q], to + D_BYTES + q * 1024);
            }
            ++ld_st;
        };
        seek();
        int ahead = 0;                  // stages in flight
#pragma unroll
        for (int s = 0; s < NB - 1; ++s)
            if (ld_round < n_rounds) {
                issue(s * STAGE);
                seek();
                ++ahead;
            }
        uint32_t fill = (NB - 1) * STAGE;
        for (int r = 0; r < n_rounds; ++r) {
            Tile cur;
            if (!tile_at(r, cur)) continue;
            const int n_bar = GROUPS > 1 ? cur.n_bar : cur.n_st;
            for (int st = 0; st < n_bar; ++st) {
                // the stage has landed; the ones behind it may still be on their way
                if (NB == 4 && ahead == 3) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NL) : "memory");
                else if (ahead == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NL) : "memory");
                else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __syncthreads();
                if (ld_round < n_rounds) {
                    issue(fill);
                    seek();
                } else {
                    --ahead;
                }
                fill = fill + STAGE == NB * STAGE ? 0 : fill + STAGE;
            }
            if (n_bar == 0) __syncthreads();
            if constexpr (GROUPS > 1) {
                __syncthreads();
                __syncthreads();
            }
            __syncthreads();
        }
        return;
    }

    // ---- the four multiplying wavefronts: no loads of operands, so they never wait for their stores -----
    const int r16 = lane & 15, g4 = lane >> 4;
    const T* biasT = p.bias ? reinterpret_cast<const T*>(p.bias) + b * p.bias_batch : nullptr;
    T* out = reinterpret_cast<T*>(p.out) + b * p.o_batch;
    T* const tileT = reinterpret_cast<T*>(smem + TILE);
    f32x4 acc[MT][NT][CHAINS];
    struct Half {
        Frag a[MT], b[NT];
    };
    auto fetch = [&](const char* buf, int half, Half& h) {
#pragma unroll
        for (int i = 0; i < MT; ++i) h.a[i] = ring_frag<T, TM, DK, Frag>(buf, wave * (TM / 4) + i * 16, half, r16, g4);
#pragma unroll
        for (int t = 0; t < NT; ++t) h.b[t] = ring_frag<T, BN, SK, Frag>(buf + D_BYTES, t * 16, half, r16, g4);
    };
    auto multiply = [&](const Half& h, auto half) {
        if constexpr (CHAINS == 4) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    f32x4& c = acc[i][0][half * 2 + (j & 1)];
                    c = SWAP ? __builtin_amdgcn_mfma_f32_16x16x4f32(h.b[0][j], h.a[i][j], c, 0, 0, 0)
                             : __builtin_amdgcn_mfma_f32_16x16x4f32(h.a[i][j], h.b[0][j], c, 0, 0, 0);
                }
        } else {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[i][t][0] = SWAP ? MMA::mma(h.b[t], h.a[i], acc[i][t][0]) : MMA::mma(h.a[i], h.b[t], acc[i][t][0]);
        }
    };
    uint32_t at = 0;
    for (int r = 0; r < n_rounds; ++r) {
        Tile cur;
        if (!tile_at(r, cur)) continue;
        // bias values fetched together, ahead of the walk
        float bias_m[MT][4], bias_n[NT][4];
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) bias_m[i][q] = 0.f;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int q = 0; q < 4; ++q) bias_n[t][q] = 0.f;
        if (biasT) {
            if (p.bias_on_m) {
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const int m = cur.m0 + wave * (TM / 4) + i * 16 + (SWAP ? r16 : g4 * 4 + q);
                        bias_m[i][q] = Elem<T>::to_float(biasT[m < p.Mc ? m : 0]);
                    }
            } else {
#pragma unroll
                for (int t = 0; t < NT; ++t)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        bias_n[t][q] = Elem<T>::to_float(biasT[cur.j * BN + t * 16 + (SWAP ? g4 * 4 + q : r16)]);
            }
        }
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int c = 0; c < CHAINS; ++c) acc[i][t][c] = f32x4{0.f, 0.f, 0.f, 0.f};
        const int n_bar = GROUPS > 1 ? cur.n_bar : cur.n_st;
        for (int st = 0; st < n_bar; ++st) {
            __syncthreads();
            if (GROUPS > 1 && st >= cur.n_st) continue;
            Half h0, h1;
            fetch(ring + at, 0, h0);
            fetch(ring + at, 1, h1);
            multiply(h0, std::integral_constant<int, 0>());
            if (!PAIR || 2 * st + 1 < cur.n_blk) multiply(h1, std::integral_constant<int, 1>());
            at = at + STAGE == NB * STAGE ? 0 : at + STAGE;
        }
        // ---- epilogue: the tile meets in LDS in the orientation of the output and leaves as whole 16-byte
        // vectors of contiguous rows, past the last-level cache or (ring_results_through) through to it
        if (n_bar == 0) __syncthreads();
        if constexpr (GROUPS > 1) {
            __syncthreads();   // the rings have been read: their space carries the sums of the other groups
            f32x4* const part = reinterpret_cast<f32x4*>(smem) + wave * (NT * 64) + lane;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                f32x4& sum = acc[0][t][0];
                if constexpr (CHAINS == 4) {
                    sum = (sum + acc[0][t][1]) + (acc[0][t][2] + acc[0][t][3]);
                    acc[0][t][1] = acc[0][t][2] = acc[0][t][3] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
                if (group > 0) part[((group - 1) * 4 * NT + t) * 64] = sum;
            }
            __syncthreads();
            if (group == 0) {
#pragma unroll
                for (int g = 0; g < GROUPS - 1; ++g)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[0][t][0] += part[(g * 4 * NT + t) * 64];
            } else {
                __syncthreads();
                return;
            }
        }
        constexpr int ROWS = LDS.rows, LDE = LDS.pitch;
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int m = wave * (TM / 4) + i * 16 + (SWAP ? r16 : g4 * 4);
                const int n = t * 16 + (SWAP ? g4 * 4 : r16);
                f32x4 sum = acc[i][t][0];
                if constexpr (CHAINS == 4) sum = (sum + acc[i][t][1]) + (acc[i][t][2] + acc[i][t][3]);
                T vals[4];
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    vals[q] = Elem<T>::from_float(epilogue_act(sum[q] + bias_m[i][q] + bias_n[t][q], p.relu));
                T* dst = tileT + (SWAP ? m * LDE + n : n * LDE + m);
                if constexpr (sizeof(T) == 2) *reinterpret_cast<uint64_t*>(dst) = *reinterpret_cast<const uint64_t*>(vals);
                else *reinterpret_cast<vec16*>(dst) = *reinterpret_cast<const vec16*>(vals);
            }
        __syncthreads();
        constexpr int CPR = LDS.cols / E16;   // 16-byte vectors per row
        constexpr bool THROUGH = ES == 2 && BN == 32 && SWAP && DK && SK;
        const bool through = THROUGH && p.relu && ring_results_through(p.Mc, p.K, p.Nc, l.parts_log2);
#pragma unroll
        for (int v0 = 0; v0 < ROWS * CPR; v0 += 256) {
            const int v = v0 + threadIdx.x;
            const int row = v / CPR, c = v % CPR * E16;
            const bool in = (ROWS * CPR % 256 == 0 || v < ROWS * CPR) && cur.m0 + (SWAP ? row : c) < p.Mc;
            T* dst = SWAP ? out + (int64_t)(cur.m0 + row) * p.o_ld + (int64_t)cur.j * BN + c
                          : out + ((int64_t)cur.j * BN + row) * p.o_ld + cur.m0 + c;
            if (!in) continue;
            const vec16 piece = *reinterpret_cast<const vec16*>(tileT + row * LDE + c);
            if constexpr (THROUGH) {
                if (through) {
                    store16_through(dst, piece);
                    continue;
                }
            }
            store16_stream(dst, piece);
        }
    }
}

template <typename T, int TM, int BN, int BK, bool DK, bool SK, bool SWAP>
static int launch_spmm_ring_inst(const SpmmParams& p, int batch, hipStream_t st) {
    constexpr int ES = (int)sizeof(T);
    constexpr RingLds LDS = ring_lds(ES, TM, BN, SWAP);
    constexpr int most = LDS.list + kRingListMax * (int)sizeof(RingTile);
    static_assert(most <= kRingLdsOfCu && ring_stages(ES) * LDS.stage >= (2 * kRingTableMax + 1) * 4, "fits a CU, and the tables the ring");
    if ((int64_t)((p.Mc + TM - 1) / TM) * (p.Nc / BN) > 0x7fffff00) return fail(SPX_E_SHAPE, "problem too large for one launch");
    const RingLaunch launch = ring_launch(ES, TM, BN, SWAP, p.Mc, p.K, p.Nc, batch);
    const int n_pos = launch.n_pos, smem = launch.smem;
    const RingList& l = launch.list;
    // One tile to a workgroup, where 64-row tiles belong: an instance without the code for more of them, which is mostly
    // start-up (32 x 64 blocks: 9 x 768 -> 1920 bf16 4.0 -> 3.55 us, 375 x 1152 -> 896 fp16 3.5 -> 3.0, 52 x 576 -> 768 fp32 with
    // 16 x 16 blocks 6.1 -> 5.2; the general code's list of tiles alone cost these 0.2).
    if constexpr (TM == 64) {
        if (n_pos == launch.n_list) {
            SpmmParams q = p;
            if (n_pos * batch <= 32) q.sched = nullptr;   // one to a CU: the order is of no account, a trip to memory less
            const int64_t columns = p.Nc / (BN << p.sub_log2);
            const int64_t blocks = spmm_live_blocks(p.counted, p.s_batch / (BK * BN << p.sub_log2), columns * (p.K / BK));
            const int groups = ring_groups(ES, BN, SWAP, n_pos * batch, (double)blocks * BK * ES / (columns * 128));
            const int lds = smem + (groups - 1) * ring_stages(ES) * LDS.stage;
            constexpr bool cut = BN < 64 && (ES == 4 || BN == 32);   // what ring_sub_log2 makes
#define SPX_RING_GROUPS(cut, n)                                                                                                             \
    if (groups == n) {                                                                                                                      \
        SPX_GRANT_LDS((spmm_ring_kernel<T, TM, BN, BK, DK, SK, SWAP, true, cut, n>), kRingLdsOfCu, "spmm_ring_kernel");                     \
        hipLaunchKernelGGL((spmm_ring_kernel<T, TM, BN, BK, DK, SK, SWAP, true, cut, n>), dim3(8 * n_pos, batch, 1), dim3(n * kRingThreads), lds, st, q, l); \
        SPX_LAUNCH_CHECK("spmm_ring_kernel");                                                                                               \
        return 0;                                                                                                                           \
    }
            if (p.sub_log2 == 0) {
                SPX_RING_GROUPS(false, 1)
            }
            SPX_RING_GROUPS(cut, 1)
            if constexpr (ring_most_groups(ES, BN) == 3) {
                SPX_RING_GROUPS(cut, 2) SPX_RING_GROUPS(cut, 3)
            }
#undef SPX_RING_GROUPS
        }
    }
    SPX_GRANT_LDS((spmm_ring_kernel<T, TM, BN, BK, DK, SK, SWAP, false>), most, "spmm_ring_kernel");
    hipLaunchKernelGGL((spmm_ring_kernel<T, TM, BN, BK, DK, SK, SWAP, false>), dim3(8 * n_pos, batch, 1), dim3(kRingThreads), smem, st, p, l);
    SPX_LAUNCH_CHECK("spmm_ring_kernel");
    return 0;
}

template <typename T, int TM>
int launch_spmm_ring_tile(const SpmmParams& p0, int BN, int batch, hipStream_t st) {
    SpmmParams p = p0;
    p.sub_log2 = 0;
    if constexpr (TM == 64) {
        p.sub_log2 = ring_sub_log2((int)sizeof(T), BN, p.out_ncontig != 0, p.Mc, p.K, p.Nc, batch);
        BN >>= p.sub_log2;
    }
#define SPX_RING_LAYOUT(bn, bk, dk, sk)                                                                     \
    if ((p.d_kcontig != 0) == dk && (p.s_kcontig != 0) == sk)                                               \
        return p.out_ncontig ? launch_spmm_ring_inst<T, TM, bn, bk, dk, sk, true>(p, batch, st)             \
                             : launch_spmm_ring_inst<T, TM, bn, bk, dk, sk, false>(p, batch, st);
#define SPX_RING_CASE(bn, bk)                                                                               \
    if (BN == bn && p.BK == bk) {                                                                           \
        if constexpr (bk % (64 / (int)sizeof(T)) == 0) {                                                    \
            SPX_RING_LAYOUT(bn, bk, true, true) SPX_RING_LAYOUT(bn, bk, true, false)                        \
            SPX_RING_LAYOUT(bn, bk, false, true) SPX_RING_LAYOUT(bn, bk, false, false)                      \
        }                                                                                                   \
    }
    SPX_RING_CASE(16, 16) SPX_RING_CASE(16, 32) SPX_RING_CASE(16, 64)
    SPX_RING_CASE(32, 16) SPX_RING_CASE(32, 32) SPX_RING_CASE(32, 64)
    SPX_RING_CASE(64, 16) SPX_RING_CASE(64, 32) SPX_RING_CASE(64, 64)
#undef SPX_RING_CASE
#undef SPX_RING_LAYOUT
    return fail(SPX_E_CONFIG, "block (%d,%d) not supported by the LDS-ring kernel", p.BK, BN);
}

// rows: 64 or 128 rows of the dense operand per tile.
template <typename T>
int launch_spmm_ring(const SpmmParams& p, int BN, int batch, int rows, hipStream_t st);

}  // namespace spx
