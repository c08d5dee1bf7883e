// Sparse-operand matmul, rows of the dense operand kept in LDS:
//     out[m, n] = sum_k D[m, k] S[k, n]   (canonical problem of matmul_spmm.hpp; 16-bit types, compressed blocks of 32 x 32, both
//     operands k-contiguous, results with n contiguous).
//
// A workgroup copies 64 whole rows of D into LDS (128 bytes for every k) and then owns all block-columns of its share
// of the result: its sixteen wavefronts take them one by one from a counter, read the live blocks of S from L2 into registers,
// two blocks ahead and across block-columns, and store a finished tile from their registers.  No barrier after the copy.
//
// What bounds it: a live block costs a CU its 2 KB of S, as fragments of 32 rows each (32 lines to a load), where the ring and the
// 256-row kernels bring 4 KB of D and more beside them and hand both over at a barrier; with few blocks to a column, the output.
// us, before / now: 8192 x 1024 -> 1024 fp16 at 40 % 26.6 / 16.1, 4464 x 1088 -> 3072 at 40 % 45.6 / 25.5, 16291 x 704 -> 3072 at 37 % 74 - 80 / 46,
// 15736 x 960 -> 3520 at 32 % 97 / 57.  On the first: stores without the non-temporal hint 18.4 against 17.1, block-columns handed out in twos
// 17.1, fragments turned in LDS out of loads of whole lines 25.8, 32 rows to a workgroup 20.6; eight wavefronts on the second 29.3.
// Blocks of depth 64 stay where they are: their fragments are four loads over the same 32 lines (8192 x 768 -> 3072 at 10 %
// 20.9 / 20.2, at 20 % 25.2 / 25.8, 2992 rows 10.5 / 17.0).
#pragma once
#include "matmul_spmm.hpp"

namespace spx {

constexpr int kRowsTile = 64, kRowsWaves = 16, kRowsLds = 160 * 1024, kRowsCus = 256;

struct RowsPlan {
    int parts, cols;                            // shares of the block-columns, and block-columns of one
    int start, entries, bias, counter, bytes;   // LDS, behind the rows
};

template <typename T>
__global__ __launch_bounds__(kRowsWaves * 64, kRowsWaves / 4) void spmm_rows_kernel(SpmmParams p, RowsPlan l) {
    static_assert(sizeof(T) == 2, "16-bit types");
    constexpr int BN = 32, BK = 32, KS = BK / 16, WAVES = kRowsWaves;   // KS: k-steps of a block
    typedef typename MmaW<T>::frag Frag;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    extern __shared__ __align__(16) char smem[];
    int* const s_start = reinterpret_cast<int*>(smem + l.start);
    uint2* const s_entry = reinterpret_cast<uint2*>(smem + l.entries);
    T* const s_bias = reinterpret_cast<T*>(smem + l.bias);
    int* const s_next = reinterpret_cast<int*>(smem + l.counter);

    // the shares of a panel run on one XCD (workgroup L runs on XCD L % 8), whose L2 then fetches its rows once
    const int i_xcd = blockIdx.x >> 3;
    const int panel = i_xcd / l.parts * 8 + (blockIdx.x & 7), part = i_xcd % l.parts;
    const int m0 = panel * kRowsTile, nb = p.Nc / BN;
    const int c0 = part * l.cols, n_cols = min(l.cols, nb - c0);
    if (m0 >= p.Mc || n_cols <= 0) return;
    const int64_t b = blockIdx.z;
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const T* const D = reinterpret_cast<const T*>(p.D) + b * p.d_batch + (int64_t)m0 * p.d_ld;
    const T* const S = reinterpret_cast<const T*>(p.S) + b * p.s_batch;
    const T* const bias = p.bias ? reinterpret_cast<const T*>(p.bias) + b * p.bias_batch + (int64_t)c0 * BN : nullptr;
    T* const out = reinterpret_cast<T*>(p.out) + b * p.o_batch;
    const int rows = min(p.Mc - m0, kRowsTile);

    // ---- rows: 64 k of all of them at a time, 128 bytes each, 16-byte chunk c of row r at c ^ ((r >> 1) & 7) -----------------
    {
        const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
        const int n_load = p.K / 64 * (kRowsTile / 8);
        for (int q = wave; q < n_load; q += WAVES) {
            const int r = (q % (kRowsTile / 8)) * 8 + (lane >> 3), chunk = (lane & 7) ^ ((r >> 1) & 7);
            lds_direct_load16_at(D, (uint32_t)min(r, rows - 1) * (uint32_t)(p.d_ld * 2) + (q / (kRowsTile / 8)) * 128 + chunk * 16, lds0 + q * 1024);
        }
    }
    // ---- index of the share -----------------------------------------------------------------------------------------------
    const int first = p.ptr[c0], n_entry = p.ptr[c0 + n_cols] - first;
    for (int i = threadIdx.x; i <= n_cols; i += WAVES * 64) s_start[i] = p.ptr[c0 + i] - first;
    for (int i = threadIdx.x; i < n_entry; i += WAVES * 64)   // (k-contiguous blocks of a dsd product come with a BCSR index)
        s_entry[i] = make_uint2((uint32_t)reinterpret_cast<const int32_t*>(p.idx)[first + i] & 0xffffu, (uint32_t)(first + i));
    if (bias)
        for (int i = threadIdx.x; i < n_cols * BN; i += WAVES * 64) s_bias[i] = bias[i];
    if (threadIdx.x == 0) *s_next = 0;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    // ---- walk ---------------------------------------------------------------------------------------------------------------
    const int l32 = lane & 31, h2 = lane >> 5;
    const int a_at = l32 * 128 + ((h2 ^ ((l32 >> 1) & 7)) << 4);
    // A block-column without a live block re-reads some block, a share without any its first row of D: every step has the
    // same loads, and the compiler can wait for the oldest ones only
    const uint32_t s_at = n_entry > 0 ? l32 * BK + h2 * 8 : 0;
    struct Item {
        int col, e, e_end, kb;   // col < 0: no more; e == e_end: a block-column without a live block
    };
    auto open = [&](Item& it) {
        it.e = __builtin_amdgcn_readfirstlane(s_start[it.col]);
        it.e_end = __builtin_amdgcn_readfirstlane(s_start[it.col + 1]);
    };
    auto take = [&](Item& it) {   // the next block-column
        int at = 0;
        if (lane == 0) at = atomicAdd(s_next, 1);
        at = __builtin_amdgcn_readfirstlane(at);
        it.col = at < n_cols ? at : -1;
        if (it.col >= 0) open(it);
    };
    auto advance = [&](const Item& from) -> Item {
        Item it = from;
        if (it.col < 0) return it;
        if (it.e + 1 < it.e_end) {
            ++it.e;
        } else {
            take(it);
        }
        return it;
    };
    auto fetch = [&](Item& it, Frag (&f)[KS]) __attribute__((always_inline)) {
        const uint2 entry = s_entry[max(min(it.e, n_entry - 1), 0)];
        it.kb = __builtin_amdgcn_readfirstlane(entry.x);
        const int64_t slot = (uint32_t)__builtin_amdgcn_readfirstlane(entry.y);
        const T* from = n_entry > 0 ? S + slot * (BK * BN) : D;
#pragma unroll
        for (int c = 0; c < KS; ++c) f[c] = *reinterpret_cast<const Frag*>(from + s_at + c * 16);
    };
    f32x16 acc[2];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[i][j] = 0.f;
    };
    // lane holds out[m = i * 32 + l32][n = 8 * jj + 4 * h2 + q] in acc[i][4 * jj + q]
    auto store = [&](int col) __attribute__((always_inline)) {
        const int r16 = lane & 15;
        const int chunk = ((lane >> 3) & 2) | (lane >> 5);   // of the lane's row of sixteen: 0, 2, 1, 3
        float add[16];
        if (bias) {
#pragma unroll
            for (int j = 0; j < 16; ++j) add[j] = Elem<T>::to_float(s_bias[col * BN + 8 * (j >> 2) + 4 * h2 + (j & 3)]);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            uint32_t d[4][2];
#pragma unroll
            for (int jj = 0; jj < 4; ++jj)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    T pair[2];
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        const int j = 4 * jj + 2 * h + q;
                        pair[q] = Elem<T>::from_float(epilogue_act(bias ? acc[i][j] + add[j] : acc[i][j], p.relu));
                    }
                    d[jj][h] = *reinterpret_cast<const uint32_t*>(pair);
                }
            // the halves of a wavefront hold the halves of a 16-byte piece, its even and odd rows of sixteen different rows
            u32x4 piece[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const auto lo = __builtin_amdgcn_permlane32_swap(d[0][h], d[1][h], false, false);
                const auto hi = __builtin_amdgcn_permlane32_swap(d[2][h], d[3][h], false, false);
#pragma unroll
                for (int x = 0; x < 2; ++x) {
                    const auto both = __builtin_amdgcn_permlane16_swap(lo[x], hi[x], false, false);
                    piece[0][2 * x + h] = both[0];
                    piece[1][2 * x + h] = both[1];
                }
            }
            T* const to = out + (int64_t)(m0 + i * 32 + r16) * p.o_ld + (int64_t)(c0 + col) * BN + chunk * 8;
#pragma unroll
            for (int x = 0; x < 2; ++x)
                if (i * 32 + r16 + 16 * x < rows) store16_stream(to + (int64_t)16 * x * p.o_ld, __builtin_bit_cast(vec16, piece[x]));
        }
    };
    auto multiply = [&](const Item& it, const Frag (&f)[KS]) __attribute__((always_inline)) {
        if (it.e >= it.e_end) return;
        const char* buf = smem + (it.kb >> 1) * (kRowsTile * 128);
        const int at = a_at ^ ((it.kb & 1) * 64);
#pragma unroll
        for (int c = 0; c < KS; ++c)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const Frag a = *reinterpret_cast<const Frag*>(buf + (at ^ (c * 32)) + i * 4096);
                acc[i] = MmaW<T>::mma(f[c], a, acc[i]);
            }
    };
    // Blocks are read two ahead: the loads of the next one are older than the stores of the last tile
    Item it = {0, 0, 0, 0};
    take(it);
    Frag f0[KS], f1[KS], f2[KS];
    fetch(it, f0);
    Item nxt = advance(it);
    fetch(nxt, f1);
    clear();
    auto step = [&](Frag (&now)[KS], Frag (&then)[KS]) __attribute__((always_inline)) {
        Item far = advance(nxt);
        fetch(far, then);
        multiply(it, now);
        if (nxt.col != it.col) {
            store(it.col);
            clear();
        }
        it = nxt;
        nxt = far;
    };
    while (true) {
        if (it.col < 0) break;
        step(f0, f2);
        if (it.col < 0) break;
        step(f1, f0);
        if (it.col < 0) break;
        step(f2, f1);
    }
}

// Shares of the block-columns: a round takes a workgroup's rows (about K / 96 block-columns' worth of time) and its
// block-columns, sixteen at a time.
inline bool spmm_rows_plan(const SpmmParams& p, int BN, int batch, RowsPlan* plan, double* filled) {
    const int nb = p.Nc / BN, per_col = p.K / p.BK;
    const int64_t panels = ((int64_t)p.Mc + kRowsTile - 1) / kRowsTile * batch;
    double best = 0;
    plan->parts = 0;
    for (int parts = 1; parts <= 16 && parts * 2 <= nb + 1; ++parts) {
        const int cols = (nb + parts - 1) / parts;
        const int64_t start = (int64_t)p.K * kRowsTile * 2, entries = start + (cols + 2) / 2 * 8, bias = entries + (int64_t)cols * per_col * 8;
        const int64_t counter = bias + cols * BN * 2, bytes = counter + 16;
        if (bytes > kRowsLds) continue;
        const int64_t rounds = (panels * parts + kRowsCus - 1) / kRowsCus;
        const double time = (double)rounds * (p.K / 96.0 + (cols + kRowsWaves - 1) / kRowsWaves * kRowsWaves);
        if (plan->parts == 0 || time < best) {
            best = time;
            *plan = {parts, cols, (int)start, (int)entries, (int)bias, (int)counter, (int)bytes};
            *filled = (double)(panels * parts) / (double)(rounds * kRowsCus);
        }
    }
    return plan->parts > 0;
}

template <typename T>
int launch_spmm_rows_impl(const SpmmParams& p, int BN, int batch, hipStream_t st) {
    if (!(BN == 32 && p.BK == 32 && p.compressed && p.s_batch > 0 && p.d_kcontig && p.s_kcontig && p.out_ncontig &&
          p.K % 64 == 0 && p.d_ld % 8 == 0 && p.o_ld % 8 == 0 && p.d_ld < (1 << 24) && p.Mc >= 2200 && p.Mc < (1 << 24)))
        return kSpmmRowsNot;
    // Enough live blocks to a column that its walk counts, and rounds of workgroups that at least half fill the chip.  170 problems
    // of 1800 to 16384 rows, other kernels / this one, us: from two blocks to a column on and K of 768 to 1152, or four, this one
    // takes 0.52 - 0.97 of the time (8179 x 960 -> 3008 with 2.4 blocks 22.7 / 20.1, 12200 x 960 -> 1984 with 3.3 26.1 / 22.4, 4627 x 832 -> 1088 with
    // 5.7 14.4 / 8.3, 8276 x 768 -> 2048 with 5.0 25.2 / 23.1); fewer blocks 7879 x 768 -> 3200 with 0.9 14.5 / 17.3, 5131 x 896 -> 1536 with 1.8 9.4 / 11.4;
    // longer rows 8614 x 1216 -> 2752 with 2.8 26.4 / 30.6, 4351 x 1216 -> 832 with 3.3 7.4 / 8.0; shorter ones 5402 x 704 -> 2176 with 3.5 15.5 / 16.8, but 4845 x 704 -> 2176 with 3.4 16.7 / 12.5; less than half full 2484 x 704 -> 704
    // 6.1 / 7.8, 2298 x 1088 -> 1216 level; 2011 x 576 -> 1856 with 5.0 9.1 / 9.4.
    const int nb = p.Nc / BN;
    const int64_t stored = p.s_batch / (p.BK * BN);
    RowsPlan plan;
    double filled = 0;
    if (stored < (p.K >= 768 && p.K <= 1152 ? 2 : 4) * (int64_t)nb || !spmm_rows_plan(p, BN, batch, &plan, &filled) || filled < 0.5) return kSpmmRowsNot;
    const int64_t panels = (p.Mc + kRowsTile - 1) / kRowsTile, groups = (panels + 7) / 8 * 8 * plan.parts;
    SPX_GRANT_LDS((spmm_rows_kernel<T>), kRowsLds, "spmm_rows_kernel");
    hipLaunchKernelGGL((spmm_rows_kernel<T>), dim3((unsigned)groups, 1, batch), dim3(kRowsWaves * 64), plan.bytes, st, p, plan);
    SPX_LAUNCH_CHECK("spmm_rows_kernel");
    return 0;
}

}  // namespace spx
