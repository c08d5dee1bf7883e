// Gathered GEMM of the mixture of experts: 256 x 256 tiles by workgroups that stay on their CU.
#include <type_traits>
#include "moe.hpp"
#include "moe_plan.hpp"

namespace spx {

// One workgroup of eight wavefronts (2 x 4, 128 x 64 each) to a CU, and to each a list of tiles.  The tiles of a list are one
// stream of stages (64 k of 256 token rows and 256 weight columns, 64 KB) through two LDS buffers: the loads run two
// stages ahead across tile boundaries, so that only the first tile has a prologue.
// The barrier that hands a stage over stands ahead of the last k-step of the stage before it: the MFMAs of that step run
// over the first fragment reads of the next stage (of the next tile as well), and the buffer that has just been read is
// refilled at once, the token rows in that k-step and the weights in the next one.  What is left after the whole
// rounds goes out as halves or quarters of a tile, one
// to each workgroup.  The output leaves straight from the registers: lane swaps give every lane 16 bytes of a row, a store
// instruction writes 64-byte pieces.
//
// What bounds it: the loads (L2 -> L1, 64 KB to 2048 clocks of MFMAs) and the MFMAs at the clock the chip holds, which overlap
// but for a third.  16384 x 1024 -> 4096 over 8 experts fp16, whole call: 145 us, without the loads 130, without the MFMAs 113,
// without the fragment reads 141.  A launch of 256 x 256 tiles by sixteen wavefronts and one of 128 x 128 tiles for what the
// whole rounds left took 166; this kernel with sixteen wavefronts of 64 x 64 156, eight 150, four of 128 x 128 157, all loads
// in the boundary's k-step + 1; column by column over all rows, as the other kernels go, + 3 (and 13838 x 2048 -> 2048 over 32
// bf16 186 with the two launches, 168 column by column, 158 in strips).
constexpr int kStrip = 4;   // row tiles; 2 and 8: up to 2 % behind

// A value that the compiler does not carry from place to place: what is derived from it is worked out where it is used.
__device__ __forceinline__ int here(int v) {
    asm volatile("" : "+v"(v));
    return v;
}

template <typename T, bool BKN>
__global__ __launch_bounds__(kPersistThreads, 2) void moe_persist_kernel(MoeParams p) {
    static_assert(sizeof(T) == 2, "16-bit types");
    constexpr int KT = 64, WGM = kPersistThreads / 256, RSTEP = kPersistThreads / 8, Q = 256 / RSTEP;   // wavefronts along the rows, rows to a load, loads of 256 rows
    typedef typename MmaW<T>::frag Frag;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) char smem[];
    int* const s_tok = reinterpret_cast<int*>(smem + kPersistTok);
    PersistTile* const list = reinterpret_cast<PersistTile*>(smem + kPersistList);

    const int lane = here(threadIdx.x) & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n_wg = gridDim.x, w = blockIdx.x;
    const int col_tiles = (p.N + 255) / 256;

    // ---- the tiles of this workgroup, a wavefront each ---------------------------------------------------
    int row_tiles = 0;
    for (int e0 = 0; e0 <= p.n_exp; e0 += 64) {
        const int e = e0 + lane;
        int cnt = 0;
        if (e <= p.n_exp) cnt = (e < p.n_exp ? p.expert_offset[e + 1] : p.n_tok) - p.expert_offset[e];
        row_tiles += __builtin_amdgcn_readlane(wave_inclusive_scan((cnt + 255) >> 8), 63);
    }
    // The list goes strip by strip of kStrip row tiles, column by column inside a strip, and a round gives each XCD (workgroup
    // w runs on XCD w % 8) consecutive places: 4 row tiles x 8 column tiles, so that its L2 fetches 12 panels for 32 tiles.
    const int places = row_tiles * col_tiles;
    const int n_whole = places / n_wg, rest = places - n_whole * n_wg;
    const int rest_xcd = (rest + 7) >> 3, wg_xcd = n_wg >> 3;
    const int cut = rest_xcd * 4 <= wg_xcd ? 2 : rest_xcd * 2 <= wg_xcd ? 1 : 0;   // log2 of the pieces of a tile in the last round
    for (int r = wave; r <= n_whole; r += kPersistThreads / 64) {
        const int xcd = w & 7, i = w >> 3;
        int L = r * n_wg + xcd * wg_xcd + i, piece = 0;
        bool exists = true;
        if (r == n_whole) {
            const int in = xcd * rest_xcd + (i >> cut);
            piece = i & ((1 << cut) - 1);
            exists = (i >> cut) < rest_xcd && in < rest;
            L = n_whole * n_wg + in;
        }
        const int strip = L / (kStrip * col_tiles), in = L - strip * (kStrip * col_tiles);
        const int height = min(kStrip, row_tiles - strip * kStrip);
        const int x = exists ? in / height : 0, y = strip * kStrip + in - x * height;
        PersistTile t = {-1, 0, 0, 0};
        if (exists) moe_find_tile<256>(p, y, lane, t.expert, t.row0, t.rows);
        t.n0 = x * 256;
        if (r == n_whole && cut > 0) {   // pieces of 128 rows, in quarters of 128 columns too
            t.row0 += (piece & 1) * 128;
            t.rows = min(t.rows - (piece & 1) * 128, 128);
            t.n0 += (piece >> 1) * 128;
            if (t.rows <= 0 || t.n0 >= p.N) t.expert = -1;
        }
        if (lane == 0) list[r] = t;
    }
    __syncthreads();

    struct Tile {
        int expert, row0, rows, n0, kind;   // kind: 0: 256 x 256, 1: 128 x 256, 2: 128 x 128, -1: none
    };
    int at = -1;
    auto next = [&]() -> Tile {   // zeroes the rows of tokens without an expert on its way
        while (++at <= n_whole) {
            const PersistTile t = list[at];
            Tile n = {__builtin_amdgcn_readfirstlane(t.expert), __builtin_amdgcn_readfirstlane(t.row0),
                      __builtin_amdgcn_readfirstlane(t.rows), __builtin_amdgcn_readfirstlane(t.n0), at < n_whole ? 0 : cut};
            if (n.expert < 0) continue;
            if (n.expert < p.n_exp) return n;
            moe_zero_tile<T>(p, n.row0, n.rows, n.n0, n.kind == 2 ? 128 : 256, kPersistThreads);
        }
        return {-1, 0, 0, 0, -1};
    };

    // ---- loads ---------------------------------------------------------------------------------------------
    // LDS: rows of 128 bytes, 16-byte chunk c of row r at c ^ ((r >> 1) & 7); weights stored [K, N] as k-rows, their 32-byte
    // units XORed by twice the low two bits of the k-row (as in moe_gemm_direct_kernel)
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * 1024;
    uint32_t a_off[Q], b_off[Q];     // bytes from the tokens, and from the weights of the expert
    const T* w_base = nullptr;
    auto set_loads = [&](const Tile& t, int tok_slot) {
        const int tid = here(threadIdx.x);
        const int srow = tid >> 3, schunk = (tid & 7) ^ ((srow >> 1) & 7);
        w_base = reinterpret_cast<const T*>(p.weight) + (int64_t)t.expert * p.K * p.N;
        if constexpr (!BKN) w_base += (int64_t)t.n0 * p.K;
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            a_off[q] = (uint32_t)s_tok[tok_slot * 256 + (srow + RSTEP * q)] * (uint32_t)(p.K * 2) + schunk * 16;
            if constexpr (BKN) {
                const int units = t.kind == 2 ? 4 : 5;   // log2 of the 16-byte pieces of a k-row
                const int slot = q * kPersistThreads + tid;
                const int kr = slot >> units, c = slot & ((1 << units) - 1);
                int n = t.n0 + ((((c >> 1) ^ ((kr & 3) << 1)) << 1) | (c & 1)) * 8;
                if (n + 8 > p.N) n = p.N - 8;            // columns past the end re-read valid ones; never stored
                b_off[q] = ((uint32_t)kr * (uint32_t)p.N + n) * 2;
            } else {
                const int n = srow + RSTEP * q;
                b_off[q] = (uint32_t)(t.n0 + n < p.N ? n : p.N - 1 - t.n0) * (uint32_t)(p.K * 2) + schunk * 16;
            }
        }
    };
    auto issue_a = [&](int kind, int s, int slot) __attribute__((always_inline)) {
        const uint32_t to = lds0 + slot * kPersistSlot;
        const T* a = reinterpret_cast<const T*>(p.tokens) + s * KT;
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (q < Q / 2 || kind == 0) lds_direct_load16_at(a, a_off[q], to + q * (RSTEP * 128));
    };
    auto issue_b = [&](int kind, int s, int slot) __attribute__((always_inline)) {
        const uint32_t to_b = lds0 + slot * kPersistSlot + (kind == 0 ? 256 : 128) * 128;
        const T* b = w_base + (BKN ? (int64_t)s * KT * p.N : (int64_t)s * KT);
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (q < Q / 2 || kind != 2) lds_direct_load16_at(b, b_off[q], to_b + q * (RSTEP * 128));
    };
    auto token_of = [&](const Tile& t) {   // threads 0 .. 255: rows past the end repeat the last one
        return p.token_perm[t.row0 + min((int)threadIdx.x, t.rows - 1)];
    };

    // ---- products ------------------------------------------------------------------------------------------
    const int wm = wave >> 2, wn = wave & 3;
    f32x16 acc[8 / WGM][2];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < 8 / WGM; ++i)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 16; ++j) acc[i][t][j] = 0.f;
    };
    // Where this lane's fragments are in a buffer: tokens: k-step c at a_at ^ (c * 32), 32 rows on 4096 bytes further; weights as k-rows:
    // k-step c 16 rows further, 32 columns on at b_at ^ 64, k + 4 four rows further; weights as rows: like the tokens
    auto a_place = [&](int kind) {
        const int lane = here(threadIdx.x) & 63, l32 = lane & 31, h2 = lane >> 5;
        const int row = wm * ((kind == 0 ? 256 : 128) / WGM) + l32;
        return row * 128 + ((h2 ^ ((row >> 1) & 7)) << 4);
    };
    auto b_place = [&](int kind) {
        const int lane = here(threadIdx.x) & 63, l32 = lane & 31, h2 = lane >> 5, r16 = lane & 15;
        const int at = (kind == 0 ? 256 : 128) * 128, col = wn * (kind == 2 ? 32 : 64);
        if constexpr (BKN) {
            const int kr = 8 * h2 + (r16 >> 2), unit = (col + 16 * ((lane >> 4) & 1)) >> 4;
            return at + kr * (kind == 2 ? 256 : 512) + ((unit ^ ((kr & 3) << 1)) << 5) + ((r16 & 3) << 3);
        } else {
            const int row = col + l32;
            return at + row * 128 + ((h2 ^ ((row >> 1) & 7)) << 4);
        }
    };
    int a_at = 0, b_at = 0;
    Frag af[2][8 / WGM], bf[2][2];   // two k-steps of 16
    auto read_frags = [&](auto kind, const char* buf, int c, int to) __attribute__((always_inline)) {
        constexpr int RB = kind == 2 ? 256 : 512;
#pragma unroll
        for (int i = 0; i < (kind == 0 ? 8 : 4) / WGM; ++i)
            af[to][i] = *reinterpret_cast<const Frag*>(buf + (a_at ^ (c * 32)) + i * 4096);
#pragma unroll
        for (int t = 0; t < (kind == 2 ? 1 : 2); ++t) {
            if constexpr (BKN) {
                const char* from = buf + (b_at ^ (t * 64)) + c * 16 * RB;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(from));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(from + 4 * RB));
                bf[to][t] = __builtin_bit_cast(Frag, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            } else {
                bf[to][t] = *reinterpret_cast<const Frag*>(buf + (b_at ^ (c * 32)) + t * 4096);
            }
        }
    };
    auto read_first = [&](int kind, const char* buf) {   // of the next tile, whose kind is known now only
        a_at = a_place(kind);
        b_at = b_place(kind);
        if (kind == 0) read_frags(std::integral_constant<int, 0>(), buf, 0, 0);
        else if (kind == 1) read_frags(std::integral_constant<int, 1>(), buf, 0, 0);
        else read_frags(std::integral_constant<int, 2>(), buf, 0, 0);
    };

    const int n_st = p.K / KT;
    Tile cur = next();
    if (cur.kind < 0) return;
    if (threadIdx.x < 256) s_tok[threadIdx.x] = token_of(cur);
    __syncthreads();
    set_loads(cur, 0);
    issue_a(cur.kind, 0, 0);
    issue_b(cur.kind, 0, 0);
    issue_a(cur.kind, 1, 1);
    clear();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    read_first(cur.kind, smem);
    int slot = 0, tok_slot = 0;
    Tile nxt;
    int tok_next = 0;

    // A stage.  `where`: 0: the first of a tile, 1: in between, 2: the last but one, 3: the last.  At the first k-step's
    // start its fragments are in registers; the loads of the next stage are on their way.
    auto stage = [&](auto kind, auto act, auto where, int s) __attribute__((always_inline)) {
        constexpr int MTW = (kind == 0 ? 8 : 4) / WGM, NTW = kind == 2 ? 1 : 2;
        const char* buf = smem + slot * kPersistSlot;
        const char* other = smem + (slot ^ 1) * kPersistSlot;
        a_at = here(a_at);
        b_at = here(b_at);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c < 3) {
                if constexpr (act) read_frags(kind, buf, c + 1, (c + 1) & 1);
                if (c == 0) {
                    if constexpr (where < 3) issue_b(kind, s + 1, slot ^ 1);
                    else if (nxt.kind >= 0) issue_b(nxt.kind, 0, slot ^ 1);
                }
            } else if (where < 3 || nxt.kind >= 0) {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next stage has landed
                if constexpr (where == 0) asm volatile("" : "+v"(tok_next));
                __syncthreads();                                   // everybody's part of it, and this one has been read
                if constexpr (where == 3) read_first(nxt.kind, other);
                else if constexpr (act) read_frags(kind, other, 0, 0);
                if constexpr (where < 2) {
                    issue_a(kind, s + 2, slot);
                } else {
                    if (where == 2 && nxt.kind >= 0) set_loads(nxt, tok_slot ^ 1);
                    if (nxt.kind >= 0) issue_a(nxt.kind, where - 2, slot);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (act) {
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int i = 0; i < MTW; ++i)
#pragma unroll
                    for (int t = 0; t < NTW; ++t) acc[i][t] = MmaW<T>::mma(bf[c & 1][t], af[c & 1][i], acc[i][t]);
                __builtin_amdgcn_s_setprio(0);
            }
        }
        slot ^= 1;
    };
    auto walk = [&](auto kind, auto act) __attribute__((always_inline)) {
        stage(kind, act, std::integral_constant<int, 0>(), 0);
        if (nxt.kind >= 0 && threadIdx.x < 256) s_tok[(tok_slot ^ 1) * 256 + threadIdx.x] = tok_next;
        for (int s = 1; s < n_st - 2; ++s) stage(kind, act, std::integral_constant<int, 1>(), s);
        stage(kind, act, std::integral_constant<int, 2>(), n_st - 2);
        stage(kind, act, std::integral_constant<int, 3>(), n_st - 1);
    };
    // lane holds out[m = i*32 + l32][n = t*32 + 8*jj + 4*h2 + q] in acc[i][t][4*jj + q]
    auto store = [&](auto kind, auto through) __attribute__((always_inline)) {
        constexpr int TM = kind == 0 ? 256 : 128, TN = kind == 2 ? 128 : 256;
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        const int lane = here(threadIdx.x) & 63, r16 = lane & 15;
        const int chunk = ((lane >> 3) & 2) | (lane >> 5);   // of the lane's row of sixteen: 0, 2, 1, 3
#pragma unroll
        for (int i = 0; i < TM / 32 / WGM; ++i) {
            const int row = wm * (TM / WGM) + i * 32 + r16;
            const int tok[2] = {s_tok[tok_slot * 256 + row], s_tok[tok_slot * 256 + row + 16]};
#pragma unroll
            for (int t = 0; t < TN / 128; ++t) {
                uint32_t d[4][2];
#pragma unroll
                for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const f32x2 v = {acc[i][t][4 * jj + 2 * h], acc[i][t][4 * jj + 2 * h + 1]};
                        if constexpr (std::is_same<T, _Float16>::value) {
                            typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
                            d[jj][h] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
                        } else {
                            typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
                            d[jj][h] = __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
                        }
                    }
                // the halves of a wavefront hold the halves of a 16-byte piece, its even and odd rows of sixteen different rows
                u32x4 out[2];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const auto lo = __builtin_amdgcn_permlane32_swap(d[0][h], d[1][h], false, false);
                    const auto hi = __builtin_amdgcn_permlane32_swap(d[2][h], d[3][h], false, false);
#pragma unroll
                    for (int x = 0; x < 2; ++x) {
                        const auto both = __builtin_amdgcn_permlane16_swap(lo[x], hi[x], false, false);
                        out[0][2 * x + h] = both[0];
                        out[1][2 * x + h] = both[1];
                    }
                }
                const int n = cur.n0 + wn * (TN / 4) + t * 32 + chunk * 8;
#pragma unroll
                for (int x = 0; x < 2; ++x)
                    if (row + 16 * x < cur.rows && n < p.N) {
                        T* const to = reinterpret_cast<T*>(p.out) + (int64_t)tok[x] * p.N + n;
                        if constexpr (through) store16_through(to, __builtin_bit_cast(vec16, out[x]));
                        else *reinterpret_cast<u32x4*>(to) = out[x];
                    }
            }
        }
    };
    auto tile = [&](auto kind) __attribute__((always_inline)) {
        // a partly filled tile: wavefronts whose rows are all past its end bring their share of the stages only
        if (wm * ((kind == 0 ? 256 : 128) / WGM) < cur.rows) {
            walk(kind, std::true_type{});
            if (nxt.kind < 0 && n_whole < 2) store(kind, std::true_type{});
            else store(kind, std::false_type{});
            clear();
        } else {
            walk(kind, std::false_type{});
        }
    };
    while (true) {
        nxt = next();
        if (nxt.kind >= 0 && threadIdx.x < 256) tok_next = token_of(nxt);
        if (cur.kind == 0) tile(std::integral_constant<int, 0>());
        else if (cur.kind == 1) tile(std::integral_constant<int, 1>());
        else tile(std::integral_constant<int, 2>());
        if (nxt.kind < 0) return;
        cur = nxt;
        tok_slot ^= 1;
    }
}

template <typename T, bool BKN>
static int launch_moe_persist_inst(const MoeParams& p, int n_wg, hipStream_t st) {
    const int smem = kPersistList + (int)persist_rounds(p.n_tok, p.N, p.n_exp, n_wg) * (int)sizeof(PersistTile);
    SPX_GRANT_LDS((moe_persist_kernel<T, BKN>), kPersistLds, "moe_persist_kernel");
    hipLaunchKernelGGL((moe_persist_kernel<T, BKN>), dim3(n_wg), dim3(kPersistThreads), smem, st, p);
    SPX_LAUNCH_CHECK("moe_persist_kernel");
    return 0;
}

template <typename T>
int launch_moe_persist(const MoeParams& p, int n_cu, hipStream_t st) {
    const int n_wg = persist_workgroups(n_cu);
    return p.w_kcontig ? launch_moe_persist_inst<T, false>(p, n_wg, st) : launch_moe_persist_inst<T, true>(p, n_wg, st);
}
template int launch_moe_persist<_Float16>(const MoeParams&, int, hipStream_t);
template int launch_moe_persist<bf16_t>(const MoeParams&, int, hipStream_t);

}  // namespace spx
