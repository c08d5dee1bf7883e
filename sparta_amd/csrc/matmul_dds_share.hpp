// Sparse-output matmul, up to four live blocks of a block-row to a workgroup.
//
// A live block on its own needs BM + BN elements for BM x BN multiply-adds at every k: 8 flops to a byte for 32 x 32 fp32 blocks,
// more bytes than the L1s take in at the rate of the matrix cores.  Here four blocks (a wavefront each) or two (two wavefronts
// each) that are neighbours in the index share the rows of A: 12.8 or 10.7 flops to a byte, and up to twice the MFMAs to a byte
// read from LDS.  Stages of 128 bytes of k go global -> LDS directly through two buffers.  Operands both
// k-contiguous (scores of attention) or both k-major (weight gradient); any K, slices of k and column sums as in
// matmul_dds_split.hpp.  Slices of blocks of 32 rows and more are summed in the same order as there:
// the results are the same to the bit.
//
// What bounds it: the MFMAs, and how evenly the blocks come out on the CUs.  Weight gradient of 4096 x 3072 -> 768 fp32 at 20 %
// (461 blocks of 32 x 32, eight slices: 3.97 workgroups to a CU) 55.6 -> 44.7 us, the MFMAs of it 28 at the clock the chip
// holds; without loads 43, without loads, fragment reads and barriers 40.  Scores of 4096 x 3072 x 768 fp32 at 20 % (2458 blocks) 51 ->
// 43.5 us with two blocks to a workgroup (4.9 to a CU), 47 with four (2.7 to a CU, so three).
#pragma once
#include "matmul_dds_split.hpp"
#include "matmul_spmm_ring.hpp"

namespace spx {

// G: most blocks of a workgroup, 4 (a wavefront each) or 2 (a wavefront to half of the rows of one).
template <typename T, int BM, int BN, bool KC, int G>
__global__ __launch_bounds__(256, 2) void dds_share_kernel(DdsParams p, DdsSplit s) {
    typedef typename PanelMma<T>::M MMA;
    typedef typename MMA::frag Frag;
    constexpr int ES = (int)sizeof(T), HK = 64 / ES, KT = 2 * HK;   // k of a half and of a stage: rows of 128 bytes
    constexpr int WPB = 4 / G, MT = BM / 16 / WPB, NT = BN / 16;   // wavefronts to a block
    constexpr int A_BYTES = BM * 128, B_BYTES = BN * 128, STAGE = A_BYTES + G * B_BYTES;
    constexpr int NA = (BM / 8 + 3) / 4, NB = BN / 8 / WPB;         // load instructions of a wavefront and stage
    extern __shared__ __align__(16) char smem[];

    const int L = blockIdx.x;
    if (L >= s.n_product) {
        dds_colsum_range<T>(p, s, L - s.n_product, reinterpret_cast<float*>(smem));
        return;
    }
    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t b = blockIdx.y;

    // ---- which blocks, which range of k: a slice has 8 / slices XCDs of its own, which take consecutive groups ----------------
    const int n_rows = p.M / BM;
    auto groups_of = [&](int r) { return r < n_rows ? (p.row_ptr[r + 1] - p.row_ptr[r] + G - 1) / G : 0; };
    int g = L >> 3, slice = L & 7;
    if (s.slices < 8) {
        const int share = 8 / s.slices;
        int total = 0;
        for (int r0 = 0; r0 < n_rows; r0 += 64) total += __builtin_amdgcn_readlane(wave_inclusive_scan(groups_of(r0 + lane)), 63);
        const int chunk = (total + share - 1) / share;
        if (g >= chunk) return;
        g += (slice & (share - 1)) * chunk;
        slice /= share;
    }
    int bi = -1, e_first = 0, n_blocks = 0;
    for (int r0 = 0, before = 0; r0 < n_rows; r0 += 64) {
        const int n = groups_of(r0 + lane), upto = before + wave_inclusive_scan(n);
        const uint64_t past = __builtin_amdgcn_ballot_w64(upto > g);
        if (past != 0) {
            const int at = __builtin_ctzll(past);
            bi = r0 + at;
            const int in_row = g - __builtin_amdgcn_readlane(upto - n, at);
            e_first = p.row_ptr[bi] + in_row * G;
            n_blocks = min(G, p.row_ptr[bi + 1] - e_first);
            break;
        }
        before = __builtin_amdgcn_readlane(upto, 63);
    }
    if (bi < 0) return;
    e_first = __builtin_amdgcn_readfirstlane(e_first);
    n_blocks = __builtin_amdgcn_readfirstlane(n_blocks);
    const int own = wave / WPB, part = wave % WPB;   // its block, and its part of the rows (and of the loads)
    const int e = e_first + own;
    const bool mine = own < n_blocks;
    const int bj = mine ? __builtin_amdgcn_readfirstlane(p.idx[e] & 0xffff) : 0;
    const int k_begin = slice * s.k_slice;
    const int k_end = k_begin + s.k_slice < p.K ? k_begin + s.k_slice : p.K;
    const int n_st = (k_end - k_begin + KT - 1) / KT;   // 0 or less: an empty slice at the end
    // unsliced: the XCDs start at staggered depths (see dds_split_kernel)
    const int rot = s.slices > 1 ? 0 : (int)(((int64_t)(L & 7) * n_st) >> 3);
    auto stage_k = [&](int st) {
        const int t = st + rot;
        return k_begin + (t >= n_st ? t - n_st : t) * KT;
    };

    // ---- loads: rows as in the ring kernel.  `valid`: k of the stage that exist; others are read from its first ones ---------------
    const T* const A = reinterpret_cast<const T*>(p.A) + b * p.a_batch + (int64_t)bi * BM * (KC ? p.a_ld : 1);
    const T* const B = reinterpret_cast<const T*>(p.B) + b * p.b_batch + (int64_t)bj * BN * (KC ? p.b_ld : 1);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    auto offset = [&](auto rows, int q, uint32_t ld, int valid) -> uint32_t {   // bytes from the panel's first element of the stage
        if constexpr (KC) {
            const int row = q * 8 + (lane >> 3);
            const int k = ((lane & 7) ^ ((row >> 1) & 7)) * (16 / ES);
            return ((uint32_t)row * ld + (k < valid ? k : 0)) * ES;
        } else {
            constexpr int PITCH = rows * ES, IPH = rows / 16, USH = ES == 2 ? 5 : 6;
            const int o = (q % IPH) * 1024 + lane * 16;
            const int k = o / PITCH + q / IPH * HK, at = o % PITCH;
            const int col = ((((at >> USH) ^ ring_row_swizzle<T, PITCH>(o / PITCH)) << USH) + (at & ((1 << USH) - 1))) / ES;
            return ((uint32_t)(k < valid ? k : 0) * ld + col) * ES;
        }
    };
    const std::integral_constant<int, BM> a_rows;
    const std::integral_constant<int, BN> b_rows;
    uint32_t a_off[NA], b_off[NB];
#pragma unroll
    for (int q = 0; q < NA; ++q) a_off[q] = offset(a_rows, wave * NA + q, (uint32_t)p.a_ld, KT);
#pragma unroll
    for (int q = 0; q < NB; ++q) b_off[q] = offset(b_rows, part * NB + q, (uint32_t)p.b_ld, KT);
    const bool a_mine = wave * NA < BM / 8;
    auto issue = [&](int st, int slot) __attribute__((always_inline)) {
        const int k0 = stage_k(st), valid = k_end - k0;
        const uint32_t to = lds0 + slot * STAGE;
        const T* const Ak = A + (int64_t)k0 * (KC ? 1 : p.a_ld);
        const T* const Bk = B + (int64_t)k0 * (KC ? 1 : p.b_ld);
        if (valid >= KT) {
            if (a_mine) {
#pragma unroll
                for (int q = 0; q < NA; ++q) lds_direct_load16_at(Ak, a_off[q], to + (wave * NA + q) * 1024);
            }
            if (mine) {
#pragma unroll
                for (int q = 0; q < NB; ++q) lds_direct_load16_at(Bk, b_off[q], to + A_BYTES + own * B_BYTES + (part * NB + q) * 1024);
            }
        } else {
            if (a_mine) {
#pragma unroll
                for (int q = 0; q < NA; ++q) lds_direct_load16_at(Ak, offset(a_rows, wave * NA + q, (uint32_t)p.a_ld, valid), to + (wave * NA + q) * 1024);
            }
            if (mine) {
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    lds_direct_load16_at(Bk, offset(b_rows, part * NB + q, (uint32_t)p.b_ld, valid), to + A_BYTES + own * B_BYTES + (part * NB + q) * 1024);
            }
        }
    };

    // ---- products: lane holds C[m = 16 x + r16][n = 16 y + 4 g4 + q] in acc[x][y][q] -------------------------------
    const int r16 = lane & 15, g4 = lane >> 4;
    // A single tile is summed in four chains, as long as where four wavefronts share its k (and MFMAs do not wait for each other)
    constexpr bool CHAINS = MT * NT == 1;
    f32x4 acc[MT][NT], chain[CHAINS ? 4 : 1];
#pragma unroll
    for (int x = 0; x < MT; ++x)
#pragma unroll
        for (int y = 0; y < NT; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < (CHAINS ? 4 : 1); ++i) chain[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    struct Half {
        Frag a[MT], b[NT];
    };
    auto fetch = [&](int slot, int half, Half& h) __attribute__((always_inline)) {
        const char* buf = smem + slot * STAGE;
#pragma unroll
        for (int x = 0; x < MT; ++x) h.a[x] = ring_frag<T, BM, KC, Frag>(buf, (part * MT + x) * 16, half, r16, g4);
#pragma unroll
        for (int y = 0; y < NT; ++y) h.b[y] = ring_frag<T, BN, KC, Frag>(buf + A_BYTES + own * B_BYTES, y * 16, half, r16, g4);
    };
    auto multiply = [&](Half& h, auto half, int valid) __attribute__((always_inline)) {   // valid: k of this half and behind it that exist
        if (valid <= 0) return;
        if constexpr (ES == 2) {
            if (valid < HK && g4 * 8 >= valid) {   // both operands: 0 times what was read there need not be 0
#pragma unroll
                for (int x = 0; x < MT; ++x) h.a[x] = Frag{};
#pragma unroll
                for (int y = 0; y < NT; ++y) h.b[y] = Frag{};
            }
        }
        if constexpr (CHAINS) {
            static_assert(ES == 4, "16 x 16 blocks of fp32");
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                f32x4& c = chain[half * 2 + (j & 1)];
                c = __builtin_amdgcn_mfma_f32_16x16x4f32(h.b[0][j], h.a[0][j], c, 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int x = 0; x < MT; ++x)
#pragma unroll
                for (int y = 0; y < NT; ++y) acc[x][y] = MMA::mma(h.b[y], h.a[x], acc[x][y]);
        }
    };
    if (n_st > 0) {
        issue(0, 0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (n_st > 1) issue(1, 1);
        __syncthreads();
        // The barrier that hands a stage over stands between the halves of the stage before it, when all of that has been read
        auto walk = [&](auto act) __attribute__((always_inline)) {
            Half h0, h1;
            if constexpr (act) fetch(0, 0, h0);
            int slot = 0;
            for (int st = 0; st < n_st; ++st) {
                const int valid = k_end - stage_k(st);
                if constexpr (act) {
                    fetch(slot, 1, h1);
                    __builtin_amdgcn_sched_barrier(0);
                    multiply(h0, std::integral_constant<int, 0>(), valid);
                }
                if (st + 1 < n_st) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next stage has landed
                    __syncthreads();
                    if constexpr (act) fetch(slot ^ 1, 0, h0);
                    if (st + 2 < n_st) issue(st + 2, slot);
                    __builtin_amdgcn_sched_barrier(0);
                }
                if constexpr (act) multiply(h1, std::integral_constant<int, 1>(), valid - HK);
                slot ^= 1;
            }
        };
        if (mine) walk(std::true_type{}); else walk(std::false_type{});
    }
    if (!mine) return;
    if constexpr (CHAINS) acc[0][0] = (chain[0] + chain[1]) + (chain[2] + chain[3]);

    // ---- the block, or its part of it: 16-byte pieces, 64 bytes of a row to a store --------------------------------
    if (s.slices > 1) {
        float* const to = s.partial + ((b * s.slices + slice) * s.nnz + e) * (int64_t)(BM * BN);
#pragma unroll
        for (int x = 0; x < MT; ++x)
#pragma unroll
            for (int y = 0; y < NT; ++y) store16_through(to + ((part * MT + x) * 16 + r16) * BN + y * 16 + g4 * 4, __builtin_bit_cast(vec16, acc[x][y]));
        return;
    }
    T* const C = reinterpret_cast<T*>(p.C) + b * p.c_batch + (p.compressed ? (int64_t)e * (BM * BN) : (int64_t)bi * BM * p.N + (int64_t)bj * BN);
    const int64_t ld = p.compressed ? BN : p.N;
    if constexpr (ES == 4) {
#pragma unroll
        for (int x = 0; x < MT; ++x)
#pragma unroll
            for (int y = 0; y < NT; ++y)
                store16_stream(C + ((part * MT + x) * 16 + r16) * ld + y * 16 + g4 * 4, __builtin_bit_cast(vec16, acc[x][y]));
    } else {
        // lane groups 0 and 1 (2 and 3) swap halves: 8 columns of tile y to the even one, of tile y + 1 to the odd one
        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
        for (int x = 0; x < MT; ++x)
#pragma unroll
            for (int y = 0; y < NT; y += 2) {
                u32x2 half[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    T vals[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(acc[x][y + i][q]);
                    half[i] = *reinterpret_cast<const u32x2*>(vals);
                }
                const auto lo = __builtin_amdgcn_permlane16_swap(half[0][0], half[1][0], false, false);
                const auto hi = __builtin_amdgcn_permlane16_swap(half[0][1], half[1][1], false, false);
                store16_stream(C + ((part * MT + x) * 16 + r16) * ld + (y + (g4 & 1)) * 16 + (g4 >> 1) * 8, vec16{lo[0], hi[0], lo[1], hi[1]});
            }
    }
}

template <typename T, int BM, int BN, bool KC, int G>
static int launch_dds_share_inst(const DdsParams& p, DdsSplit s, void* colsum, int batch, hipStream_t st) {
    constexpr int KT = 128 / (int)sizeof(T), VE = 16 / (int)sizeof(T);
    constexpr int stages = 2 * (BM + G * BN) * 128, sums_lds = 32 * (8 * VE + 4) * (int)sizeof(float);
    constexpr int smem = stages > sums_lds ? stages : sums_lds;
    const bool sums = s.colsum || s.colsum_out;
    constexpr int whole = DdsSplitCfg<T, BM, BN>::KT;   // a slice is what it is where every block has a workgroup
    static_assert(whole % KT == 0, "whole stages");
    s.k_slice = (int)round_up((p.K + s.slices - 1) / s.slices, whole);
    const int share = 8 / s.slices;
    const int64_t rows = p.M / BM < s.nnz ? p.M / BM : s.nnz;
    const int64_t groups = ((int64_t)s.nnz + (G - 1) * rows) / G;   // at most
    const int64_t n_product = (groups + share - 1) / share * 8;
    const int64_t cs_groups = sums ? (int64_t)(p.M + 8 * VE - 1) / (8 * VE) * (s.colsum_out ? 1 : kColsumSlices) : 0;
    if (n_product + cs_groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)(n_product + cs_groups));
    if (n_product + cs_groups == 0) return 0;
    s.n_product = (int)n_product;
    SPX_GRANT_LDS((dds_share_kernel<T, BM, BN, KC, G>), smem, "dds_share_kernel");
    hipLaunchKernelGGL((dds_share_kernel<T, BM, BN, KC, G>), dim3((unsigned)(n_product + cs_groups), batch, 1), dim3(256), smem, st, p, s);
    SPX_LAUNCH_CHECK("dds_share_kernel");
    return launch_dds_split_reduce<T>(p, s, colsum, BM, BN, batch, st);
}

template <typename T>
int launch_dds_share_impl(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st) {
    const bool kcontig = p.a_kcontig && p.b_kcontig;
#define SPX_DDS_SHARE_CASE(bm, bn, kc, g) \
    if (BM == bm && BN == bn && kcontig == kc && s.share == g) return launch_dds_share_inst<T, bm, bn, kc, g>(p, s, colsum, batch, st);
    if constexpr (sizeof(T) == 4) {   // what dds_share_plan names
        SPX_DDS_SHARE_CASE(16, 16, false, 4) SPX_DDS_SHARE_CASE(32, 32, false, 2) SPX_DDS_SHARE_CASE(32, 32, false, 4)
        SPX_DDS_SHARE_CASE(32, 64, false, 2) SPX_DDS_SHARE_CASE(32, 32, true, 2)
    } else {
        SPX_DDS_SHARE_CASE(32, 32, false, 4) SPX_DDS_SHARE_CASE(32, 64, false, 2) SPX_DDS_SHARE_CASE(64, 64, false, 2)
    }
#undef SPX_DDS_SHARE_CASE
    return fail(SPX_E_CONFIG, "output block (%d,%d) not supported by the kernel whose blocks share A", BM, BN);
}

}  // namespace spx
