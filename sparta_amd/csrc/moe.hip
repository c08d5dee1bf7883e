// MoE sparse forward: out[t,:] = tokens[t,:] . W[exp_ids[t]].
//
//  spx_moe_index   stable counting sort of the tokens by expert, no atomics on
//                  global memory, no per-expert capacity, no host round trip:
//                  (1) per-chunk histograms, (2) an exclusive scan of them in
//                  (expert, chunk) order, (3) every chunk places its tokens in
//                  ascending order behind its scanned base.  A table of at most
//                  1024 (chunk, expert) counts is scanned by every placement
//                  workgroup itself (two launches); larger ones get a scan
//                  launch of their own.  Up to 20480 tokens over 63 experts
//                  one launch does all three.
//  spx_moe_forward one gathered GEMM over a flattened (expert, row tile) list (moe_persist.hip: large
//                  problems): a workgroup looks its tile up in the prefix of per-expert tile
//                  counts, gathers its token rows through token_perm, and walks
//                  K in 64-wide stages through LDS ([row][k], XOR-swizzled 16-byte
//                  chunks) into 16x16 MFMAs; rows are scattered back on store.
// Replaces convert_sparse_index / BATCH_BLOCK_SPARSE_MATMUL[_FP16] of the
// reference (csrc/moe_sparse_forward_kernel.cu.j2:58-71,120-325,363-483), whose
// grid is sized by the largest expert and whose fp16 path accumulates in fp16.
#include <type_traits>
#include "moe.hpp"
#include "moe_plan.hpp"

namespace spx {

constexpr int MOE_CHUNK = 1024;   // most tokens per workgroup in the index kernels (a multiple of 256)
constexpr int MOE_FUSED_TABLE = 1024;  // (chunk, expert) counts a placement workgroup scans itself
// Tokens up to which the placement workgroups count the experts themselves, a launch less: 1100 tokens 4.5 -> 3.5 us,
// 4000 5.1 -> 4.8; 6000 5.0 against 5.5, 8000 5.0 against 7.5 (with up to 63 experts moe_index_kernel takes over).
constexpr int MOE_SELF_COUNT = 4096;
constexpr int MOE_MAX_EXP = 2048; // LDS table capacity of the placement kernel
constexpr int MOE_MAX_ROW_TILES = 65535;   // the y extent of a grid

// ---- index -------------------------------------------------------------------
__global__ __launch_bounds__(256) void moe_hist_kernel(const int32_t* exp_ids, int n_tok, int n_exp, int chunk,
                                                       int32_t* partial /* [n_chunk][n_exp] */) {
    // n_exp here counts the pseudo expert that collects the tokens whose id is out of range
    extern __shared__ int hist[];
    for (int e = threadIdx.x; e < n_exp; e += 256) hist[e] = 0;
    __syncthreads();
    const int base = blockIdx.x * chunk;
    for (int i = threadIdx.x; i < chunk; i += 256) {
        const int t = base + i;
        if (t < n_tok) {
            int e = exp_ids[t];
            if (e < 0 || e >= n_exp - 1) e = n_exp - 1;
            atomicAdd(&hist[e], 1);
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < n_exp; e += 256) partial[(int64_t)blockIdx.x * n_exp + e] = hist[e];
}

// Wavefront e: exclusive prefix of expert e's counts over the chunks, in place, and the
// expert's total.  Every lane takes a run of consecutive chunks (sums it, then rewrites it
// from the lane's offset), so the serial part is 1/64 of the chunks.  n_exp counts the
// pseudo expert of out-of-range ids.
__global__ __launch_bounds__(256) void moe_colscan_kernel(int32_t* partial, int n_chunk, int n_exp, int32_t* totals) {
    const int lane = lane_id();
    const int e = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (e >= n_exp) return;
    const int per = (n_chunk + 63) / 64;
    const int c0 = lane * per < n_chunk ? lane * per : n_chunk;
    const int c1 = c0 + per < n_chunk ? c0 + per : n_chunk;
    int sum = 0;
    for (int c = c0; c < c1; ++c) sum += partial[(int64_t)c * n_exp + e];
    const int inc = wave_inclusive_scan(sum);
    int run = inc - sum;
    for (int c = c0; c < c1; ++c) {
        const int v = partial[(int64_t)c * n_exp + e];
        partial[(int64_t)c * n_exp + e] = run;
        run += v;
    }
    if (lane == 63) totals[e] = inc;
}

__global__ __launch_bounds__(256) void moe_zero_index_kernel(int n_exp, int32_t* expert_count, int32_t* expert_offset) {
    const int e = blockIdx.x * 256 + threadIdx.x;
    if (e < n_exp) expert_count[e] = 0;
    if (e <= n_exp) expert_offset[e] = 0;
}

// Stable placement of one chunk.  Waves take 64 tokens at a time; inside a wave the
// rank among equal experts comes from ballots, between waves from a small table.
// FUSED: `counts` holds the raw per-chunk histograms (at most MOE_FUSED_TABLE of them), or is null
// (at most MOE_SELF_COUNT tokens: counting them again in every workgroup is cheaper than the launch that would);
// every workgroup scans them in (expert, chunk) order itself and workgroup 0 also writes
// expert_offset and expert_count.  Otherwise `counts` holds every expert's prefix over the
// chunks (moe_colscan_kernel) and `totals` the experts' token counts, which every workgroup
// turns into the experts' offsets itself (at most MOE_MAX_EXP + 1 of them).
template <bool FUSED>
__global__ __launch_bounds__(256) void moe_place_kernel(const int32_t* exp_ids, int n_tok, int n_exp, int chunk,
                                                        const int32_t* counts, const int32_t* totals, int32_t* token_perm,
                                                        int32_t* expert_count, int32_t* expert_offset) {
    extern __shared__ int sm[];
    int* running = sm;               // [n_exp] tokens of expert e already placed by this chunk
    int* wavecnt = sm + n_exp;       // [4][n_exp] tokens of expert e in the current pass, per wave
    int* ebase = sm + 5 * n_exp;     // [n_exp] first position of expert e (not FUSED)
    __shared__ int tab[FUSED ? MOE_FUSED_TABLE : 1];
    __shared__ int wave_total[4];
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < 5 * n_exp; i += 256) sm[i] = 0;
    if constexpr (FUSED) {
        // entries 4 tid .. 4 tid + 3 of the (expert, chunk) order
        const int n_chunk = gridDim.x;
        const int n = n_chunk * n_exp;
        if (counts == nullptr) {   // few tokens: every workgroup counts all of them itself
            for (int i = threadIdx.x; i < n; i += 256) tab[i] = 0;
            __syncthreads();
            constexpr int BATCH = 8;   // loads in flight to a thread
            for (int t0 = threadIdx.x; t0 < n_tok; t0 += 256 * BATCH) {
                int id[BATCH];
#pragma unroll
                for (int j = 0; j < BATCH; ++j) id[j] = t0 + j * 256 < n_tok ? exp_ids[t0 + j * 256] : -1;
#pragma unroll
                for (int j = 0; j < BATCH; ++j) {
                    const int t = t0 + j * 256, c = __builtin_amdgcn_readfirstlane(t >> 8) / (chunk >> 8);   // chunks are whole 256s
                    const int e = id[j] < 0 || id[j] >= n_exp - 1 ? n_exp - 1 : id[j];
                    if (t < n_tok) atomicAdd(&tab[e * n_chunk + c], 1);
                }
            }
            __syncthreads();
        }
        int v[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = threadIdx.x * 4 + j;
            v[j] = 0;
            if (i < n) {
                const int e = i / n_chunk, c = i - e * n_chunk;
                v[j] = counts ? counts[c * n_exp + e] : tab[i];
            }
            sum += v[j];
        }
        const int inc = wave_inclusive_scan(sum);
        if (lane == 63) wave_total[wave] = inc;
        __syncthreads();
        int excl = inc - sum;
        for (int w = 0; w < wave; ++w) excl += wave_total[w];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = threadIdx.x * 4 + j;
            if (i < n) tab[i] = excl;
            excl += v[j];
        }
        __syncthreads();
        if (blockIdx.x == 0) {
            for (int e = threadIdx.x; e < n_exp; e += 256) {
                expert_offset[e] = tab[e * n_chunk];
                if (e + 1 < n_exp) expert_count[e] = tab[(e + 1) * n_chunk] - tab[e * n_chunk];
            }
        }
    }
    if constexpr (!FUSED) {
        // experts per * tid .. per * tid + per - 1: exclusive scan of their totals
        const int per = (n_exp + 255) / 256;
        int sum = 0;
        for (int j = 0; j < per; ++j) {
            const int e = threadIdx.x * per + j;
            if (e < n_exp) sum += totals[e];
        }
        const int inc = wave_inclusive_scan(sum);
        if (lane == 63) wave_total[wave] = inc;
        __syncthreads();
        int excl = inc - sum;
        for (int w = 0; w < wave; ++w) excl += wave_total[w];
        for (int j = 0; j < per; ++j) {
            const int e = threadIdx.x * per + j;
            if (e < n_exp) {
                const int t = totals[e];
                ebase[e] = excl;
                if (blockIdx.x == 0) {
                    expert_offset[e] = excl;
                    if (e + 1 < n_exp) expert_count[e] = t;
                }
                excl += t;
            }
        }
    }
    __syncthreads();
    const int chunk0 = blockIdx.x * chunk;
    const unsigned long long lt_mask = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int pass = 0; pass < chunk; pass += 256) {
        const int t = chunk0 + pass + threadIdx.x;
        int e = -1;
        if (t < n_tok) {
            e = exp_ids[t];
            if (e < 0 || e >= n_exp - 1) e = n_exp - 1;  // out of range: the pseudo expert
        }
        // intra-wave rank and per-wave count of my expert
        // (a ballot per bit of the expert; with one per expert in the wavefront 700 tokens over 32 experts took 5.6 and not
        // 3.6 us, 16384 over 32 13.4 and not 6.9, over 4 5.3 and 5.1)
        unsigned long long same = __ballot(e >= 0);
        for (int bit = 31 - __builtin_clz(n_exp | 1); bit >= 0; --bit) {
            const unsigned long long ones = __ballot((e >> bit) & 1);
            same &= (e >> bit) & 1 ? ones : ~ones;
        }
        const int rank = __popcll(same & lt_mask), cnt = __popcll(same);
        const bool leader = e >= 0 && rank == 0;
        if (leader) wavecnt[wave * n_exp + e] = cnt;
        __syncthreads();
        if (e >= 0) {
            int before = running[e];
            for (int w = 0; w < wave; ++w) before += wavecnt[w * n_exp + e];
            const int base = FUSED ? tab[e * gridDim.x + blockIdx.x] : ebase[e] + counts[(int64_t)blockIdx.x * n_exp + e];
            token_perm[base + before + rank] = t;
        }
        __syncthreads();
        if (leader) {
            atomicAdd(&running[e], cnt);
            wavecnt[wave * n_exp + e] = 0;
        }
        __syncthreads();
    }
}

// The whole index in one launch, from 4097 to 20480 tokens over at most 63 experts: a workgroup places 1024 tokens, 64 to a
// wavefront, and counts all of them itself before, those ahead of its own apart.  The counters of an expert are sixteen
// copies side by side, one for every sixteenth lane, so that a crowded expert does not queue up a wavefront's additions.
// What bounds it: the launch and the additions (a 64 KB list of 16384 tokens is counted in a microsecond).  Counting and placing
// launch against this one (kernels alone): 4100 tokens over 8 6.1 -> 3.9 us, 8192 over 32 8.7 -> 4.7, 16384 over 8 8.4 -> 5.5;
// whole passes 5000 x 256 -> 512 over 4 13.6 -> 12.1, 8192 x 768 -> 768 over 8 24.6 -> 23.6.  A workgroup's count grows with
// the tokens: 24000 over 4 6.2 against 6.1 us, 32768 over 4 6.2 against 7.0 (over 32 10.1 against 7.2): 20480 is the line.
constexpr int MOE_ONE_TOKENS = 20480, MOE_ONE_EXPERTS = 63, MOE_ONE_THREADS = 1024;
__global__ __launch_bounds__(MOE_ONE_THREADS) void moe_index_kernel(const int32_t* exp_ids, int n_tok, int n_exp, int32_t* token_perm,
                                                                    int32_t* expert_count, int32_t* expert_offset) {
    constexpr int COPIES = 16, MOST = MOE_ONE_EXPERTS + 1, WAVES = MOE_ONE_THREADS / 64;
    __shared__ int counts[2][MOST * COPIES];   // [ahead of this workgroup's tokens / from them on][expert, copy]
    __shared__ int base[MOST], wave_count[WAVES][MOST];
    const int lane = lane_id(), wave = threadIdx.x >> 6;
    const int own = blockIdx.x * MOE_ONE_THREADS;
    for (int i = threadIdx.x; i < 2 * MOST * COPIES; i += MOE_ONE_THREADS) (&counts[0][0])[i] = 0;
    for (int i = threadIdx.x; i < WAVES * MOST; i += MOE_ONE_THREADS) (&wave_count[0][0])[i] = 0;
    auto expert_of = [&](int t) {   // n_exp counts the pseudo expert of ids that are out of range, the last one
        const int e = t < n_tok ? exp_ids[t] : 0;
        return e < 0 || e >= n_exp - 1 ? n_exp - 1 : e;
    };
    const int mine = own + threadIdx.x;
    const int e = mine < n_tok ? expert_of(mine) : -1;
    __syncthreads();
    constexpr int BATCH = 8;   // loads in flight to a thread
    for (int t0 = threadIdx.x; t0 < n_tok; t0 += MOE_ONE_THREADS * BATCH) {
        int id[BATCH];
#pragma unroll
        for (int j = 0; j < BATCH; ++j) id[j] = expert_of(t0 + j * MOE_ONE_THREADS);
#pragma unroll
        for (int j = 0; j < BATCH; ++j) {
            const int t = t0 + j * MOE_ONE_THREADS;   // (the own tokens are one j of the loop)
            if (t < n_tok) atomicAdd(&counts[t < own ? 0 : 1][id[j] * COPIES + (lane & (COPIES - 1))], 1);
        }
    }
    // intra-wave rank and count of my expert, as in moe_place_kernel
    unsigned long long same = __ballot(e >= 0);
    for (int bit = 31 - __builtin_clz(n_exp | 1); bit >= 0; --bit) {
        const unsigned long long ones = __ballot((e >> bit) & 1);
        same &= (e >> bit) & 1 ? ones : ~ones;
    }
    const int rank = __popcll(same & (lane == 0 ? 0ull : (~0ull >> (64 - lane))));
    if (e >= 0 && rank == 0) wave_count[wave][e] = __popcll(same);
    __syncthreads();
    if (wave == 0) {   // a lane to an expert
        int ahead = 0, total = 0;
        if (lane < n_exp)
            for (int c = 0; c < COPIES; ++c) {   // (the copies in turn: lanes are sixteen words apart)
                const int at = lane * COPIES + ((c + lane) & (COPIES - 1));
                ahead += counts[0][at];
                total += counts[1][at];
            }
        total += ahead;
        const int first = wave_inclusive_scan(total) - total;
        if (lane < n_exp) {
            base[lane] = first + ahead;
            if (blockIdx.x == 0) {
                expert_offset[lane] = first;
                if (lane + 1 < n_exp) expert_count[lane] = total;
            }
        }
    }
    __syncthreads();
    if (e >= 0) {
        int at = base[e] + rank;
        for (int w = 0; w < wave; ++w) at += wave_count[w][e];
        token_perm[at] = mine;
    }
}

// ---- gathered GEMM -------------------------------------------------------------
constexpr int MOE_TM = 128, MOE_TN = 128;
// k per LDS stage: 128 bytes per row for every element type
template <typename T> struct MoeKt { static constexpr int value = 128 / (int)sizeof(T); };

// LDS tile: rows of 128 bytes = 8 chunks of 16 bytes; chunk c of row r is stored at
// chunk position c ^ (r & 7).
template <typename T>
__device__ __forceinline__ int moe_lds_off(int row, int chunk) {
    return (row * 8 + (chunk ^ (row & 7))) * 16;
}

template <typename T>
__global__ __launch_bounds__(256) void moe_gemm_kernel(MoeParams p) {
    constexpr int VE = 16 / (int)sizeof(T);
    constexpr int MOE_KT = MoeKt<T>::value;
    constexpr int CPR = MOE_KT / VE;                 // 16-byte chunks per LDS row (8)
    constexpr int TILE_BYTES = MOE_TM * MOE_KT * (int)sizeof(T);
    extern __shared__ __align__(16) char smem[];
    char* As = smem;
    char* Bs = smem + TILE_BYTES;
    __shared__ int s_expert, s_row0, s_rows;

    // ---- which (expert, row tile) is mine ------------------------------------------
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        int found_e, found_row0, found_rows;
        moe_find_tile<MOE_TM>(p, blockIdx.y, lane, found_e, found_row0, found_rows);
        if (lane == 0) { s_expert = found_e; s_row0 = found_row0; s_rows = found_rows; }
    }
    __syncthreads();
    const int expert = s_expert;
    if (expert < 0) return;  // uniform: this tile index is past the last tile
    const int row0 = s_row0, rows = s_rows;
    const int n0 = blockIdx.x * MOE_TN;
    if (expert == p.n_exp) {  // tokens without a valid expert id: zero rows
        moe_zero_tile<T>(p, row0, rows, n0, MOE_TN, 256);
        return;
    }

    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const int wm = wave >> 1, wn = wave & 1;  // 2 x 2 waves, each 64 x 64

    const T* X = reinterpret_cast<const T*>(p.tokens);
    const T* W = reinterpret_cast<const T*>(p.weight) + (int64_t)expert * p.K * p.N;

    // staging map: thread -> (row, 16-byte chunk) pairs; 128 rows x CPR chunks per tile
    constexpr int LOADS = MOE_TM * CPR / 256;
    int a_tok[LOADS];
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
        const int v = q * 256 + threadIdx.x;
        const int r = v / CPR;
        a_tok[q] = p.token_perm[row0 + (r < rows ? r : rows - 1)];
    }

    // 2-byte types: 2 x 2 tiles of 32 x 32 (accw); fp32: 4 x 4 tiles of 16 x 16 (acc)
    constexpr bool WIDE = HasMma32<T>::value;
    f32x4 acc[WIDE ? 1 : 4][WIDE ? 1 : 4];
    f32x16 accw[WIDE ? 2 : 1][WIDE ? 2 : 1];
#pragma unroll
    for (int i = 0; i < (WIDE ? 1 : 4); ++i)
#pragma unroll
        for (int t = 0; t < (WIDE ? 1 : 4); ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < (WIDE ? 2 : 1); ++i)
#pragma unroll
        for (int t = 0; t < (WIDE ? 2 : 1); ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j) accw[i][t][j] = 0.f;
    const int l32 = lane & 31, h2 = lane >> 5;

    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    for (int k0 = 0; k0 < p.K; k0 += MOE_KT) {
        // ---- stage A (gathered token rows) and B (weight rows n0..n0+127) ---------------
#pragma unroll
        for (int q = 0; q < LOADS; ++q) {
            const int v = q * 256 + threadIdx.x;
            const int r = v / CPR, c = v % CPR;
            const u32x4 val = *reinterpret_cast<const u32x4*>(X + (int64_t)a_tok[q] * p.K + k0 + c * VE);
            *reinterpret_cast<u32x4*>(As + moe_lds_off<T>(r, c)) = val;
        }
        if (p.w_kcontig) {
#pragma unroll
            for (int q = 0; q < LOADS; ++q) {
                const int v = q * 256 + threadIdx.x;
                const int r = v / CPR, c = v % CPR;
                const int n = n0 + r < p.N ? n0 + r : p.N - 1;
                const u32x4 val = *reinterpret_cast<const u32x4*>(W + (int64_t)n * p.K + k0 + c * VE);
                *reinterpret_cast<u32x4*>(Bs + moe_lds_off<T>(r, c)) = val;
            }
        } else {
            // weight stored [K, N]: 16-byte loads along n, transposed into [n][k]
            constexpr int NV = MOE_TN / VE;  // vectors per k row
            for (int v = threadIdx.x; v < MOE_KT * NV; v += 256) {
                const int k = v / NV, nv = v % NV;
                union { u32x4 v4; T e[VE]; } u;
                const int n = n0 + nv * VE;
                if (n + VE <= p.N) {
                    u.v4 = *reinterpret_cast<const u32x4*>(W + (int64_t)(k0 + k) * p.N + n);
                } else {
#pragma unroll
                    for (int i = 0; i < VE; ++i) u.e[i] = W[(int64_t)(k0 + k) * p.N + (n + i < p.N ? n + i : p.N - 1)];
                }
#pragma unroll
                for (int i = 0; i < VE; ++i) {
                    const int r = nv * VE + i;
                    reinterpret_cast<T*>(Bs + moe_lds_off<T>(r, k / VE))[k % VE] = u.e[i];
                }
            }
        }
        __syncthreads();
        // ---- MFMA over the stage -----------------------------------------------------------
        if constexpr (WIDE) {
#pragma unroll
            for (int kc = 0; kc < MOE_KT; kc += 16) {
                typename MmaW<T>::frag af[2], bf[2];
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    af[i] = *reinterpret_cast<const typename MmaW<T>::frag*>(As + moe_lds_off<T>(wm * 64 + i * 32 + l32, kc / VE + h2));
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    bf[t] = *reinterpret_cast<const typename MmaW<T>::frag*>(Bs + moe_lds_off<T>(wn * 64 + t * 32 + l32, kc / VE + h2));
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int t = 0; t < 2; ++t) accw[i][t] = MmaW<T>::mma(bf[t], af[i], accw[i][t]);
            }
        } else {
#pragma unroll
            for (int kc = 0; kc < MOE_KT; kc += 16) {
                typename Mma16<T>::frag af[4], bf[4];
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    af[i] = *reinterpret_cast<const typename Mma16<T>::frag*>(As + moe_lds_off<T>(wm * 64 + i * 16 + r16, kc / VE + g4));
#pragma unroll
                for (int t = 0; t < 4; ++t)
                    bf[t] = *reinterpret_cast<const typename Mma16<T>::frag*>(Bs + moe_lds_off<T>(wn * 64 + t * 16 + r16, kc / VE + g4));
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int t = 0; t < 4; ++t) acc[i][t] = Mma16<T>::mma(bf[t], af[i], acc[i][t]);
            }
        }
        __syncthreads();
    }

    // ---- scatter the rows back (fp32: lane holds out[m = i*16 + r16][n = t*16 + g4*4 .. +3]) ----
    T* out = reinterpret_cast<T*>(p.out);
    if constexpr (sizeof(T) == 2) {
        // 16-bit outputs leave through LDS (free after the last barrier): the wavefront's
        // 64 x 64 tile is laid out as 64 rows of 128 bytes (chunks XOR-swizzled by the
        // row), then every store instruction writes eight complete 128-byte row segments
        // instead of sixteen 32-byte pieces.
        // lane holds out[m = i*32 + lane%32][n = t*32 + 8*jj + 4*(lane/32) + q] in accw[i][t][4*jj + q]
        char* ep = smem + wave * (64 * 128);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    T vals[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(accw[i][t][4 * jj + q]);
                    const int row = i * 32 + l32;
                    const int chunk = t * 4 + jj;
                    *reinterpret_cast<uint64_t*>(ep + row * 128 + ((chunk ^ (row & 7)) << 4) + h2 * 8) =
                        *reinterpret_cast<const uint64_t*>(vals);
                }
        // LDS operations of one wavefront complete in order: no barrier needed
        const int c = lane & 7;
        const int n = n0 + wn * 64 + c * 8;
        // the tokens of the lane's rows, fetched together ahead of the stores (a load between
        // two stores waits for the store before it as well)
        int toks[8];
#pragma unroll
        for (int pass = 0; pass < 8; ++pass) {
            const int r = wm * 64 + pass * 8 + (lane >> 3);
            toks[pass] = r < rows ? p.token_perm[row0 + r] : -1;
        }
#pragma unroll
        for (int pass = 0; pass < 8; ++pass) {
            const int row = pass * 8 + (lane >> 3);
            const u32x4 v = *reinterpret_cast<const u32x4*>(ep + row * 128 + ((c ^ (row & 7)) << 4));
            if (toks[pass] >= 0 && n < p.N) store16_through(out + (int64_t)toks[pass] * p.N + n, __builtin_bit_cast(vec16, v));
        }
    } else {
    int toks[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = wm * 64 + i * 16 + r16;
        toks[i] = r < rows ? p.token_perm[row0 + r] : -1;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (toks[i] < 0) continue;
        const int tok = toks[i];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int n = n0 + wn * 64 + t * 16 + g4 * 4;
            T vals[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(acc[i][t][q]);
            T* dst = out + (int64_t)tok * p.N + n;
            if (n + 4 <= p.N) {
                if constexpr (sizeof(T) == 2) *reinterpret_cast<uint64_t*>(dst) = *reinterpret_cast<const uint64_t*>(vals);
                else *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(vals);
            } else {
                for (int q = 0; q < 4; ++q)
                    if (n + q < p.N) dst[q] = vals[q];
            }
        }
    }
    }
}

// Workgroup L (column tiles fastest) runs on XCD L % 8.  With a multiple of eight column tiles every XCD
// keeps the same columns for all row tiles, and its weight panels stay in its L2.  With other
// counts the columns of an XCD would change from row tile to row tile, and every XCD would read all weights:
// there the column tiles are cut into col_groups = 4, 2 or 1 groups, an XCD stays in one of them, and the row
// tiles go round the 8 / col_groups XCDs of a group.  fp16, before / after: 16384 x 2048 -> 768 over 32 experts
// 94.5 / 73.8 us (6 column tiles), 10007 x 768 -> 3072 over 32 bf16 82 / 76 us (12), 8192 x 768 -> 768 over 16 22.8 / 20.1 us,
// 16384 x 768 -> 768 over 8 29.3 / 28.2 us (3); 16384 x 1024 -> 768 and -> 3072 the same.  With a multiple of eight
// columns (16384 x 1024 -> 4096) no cut measured a difference, and with fewer than 256 rows per expert there is
// little to share (4096 x 2048 -> 768 over 32, whole call: 51.0 in launch order, 52.8 cut).
__device__ __forceinline__ void moe_tile_of_workgroup(const MoeParams& p, int& x, int& y) {
    if (p.col_groups == 0) { x = blockIdx.x; y = blockIdx.y; return; }
    const int L = blockIdx.y * gridDim.x + blockIdx.x;
    const int xcd = L & 7, j = L >> 3;
    const int cols = gridDim.x / p.col_groups;
    x = (xcd % p.col_groups) * cols + j % cols;
    y = (j / cols) * (8 / p.col_groups) + xcd / p.col_groups;
}

// ---- gathered GEMM with LDS-direct loads ------------------------------------------------
// Same tile lookup and LDS layout as moe_gemm_kernel (k-contiguous weights only); the
// workgroup tile is TM x TN with WAVES wavefronts (WGM of them along the rows), and the
// operands go from global memory straight into LDS (global_load_lds_dwordx4: each
// wavefront instruction writes 64 x 16 bytes to consecutive LDS addresses starting at
// M0), so no registers or LDS-store instructions are spent on staging.  NBUF LDS buffers hold stages s .. s + NBUF - 1; one barrier per
// stage.  The loads are issued through inline assembly, which keeps the compiler from
// serialising them against the fragment reads of the other buffers.

template <typename T, int TM, int TN, int WAVES, int WGM, int NBUF, int KTB, bool BKN, bool XS>
__global__ __launch_bounds__(64 * WAVES, (TM + TN) * NBUF * KTB > 80 * 1024 ? 1 : 2) void moe_gemm_direct_kernel(MoeParams p) {
    static_assert(!BKN || sizeof(T) == 2, "the [K, N] weight layout is read with 16-bit LDS transpose loads");
    static_assert(!XS || (HasMma32<T>::value && NBUF >= 3 && NBUF <= 4 && (KTB / (int)sizeof(T) / 16) % 2 == 0),
                  "the cross-stage pipeline needs 32x32 MFMAs, three or four buffers and an even number of k-steps per stage");
    constexpr int NTH = 64 * WAVES;
    constexpr int WGN = WAVES / WGM;
    constexpr int MT = TM / WGM / 16;   // 16-row tiles per wave
    constexpr int NTT = TN / WGN / 16;  // 16-column tiles per wave
    constexpr int VE = 16 / (int)sizeof(T);
    constexpr int KT = KTB / (int)sizeof(T);  // k per row and stage (KTB = 64 or 128 bytes)
    constexpr int CPR = KTB / 16;             // 16-byte chunks per LDS row
    constexpr int A_LOADS = TM * CPR / NTH;
    constexpr int B_LOADS = TN * CPR / NTH;
    constexpr int RSTEP = NTH / CPR;          // tile rows between a thread's vectors
    constexpr int A_BYTES = TM * KTB;
    constexpr int BUF = (TM + TN) * KTB;
    // chunk c of row r sits at position c ^ swz(r): rows of 128 bytes use the low three bits
    // of the row, rows of 64 bytes bits 2..3 (sixteen lanes of a 16-byte read then touch
    // sixteen different 16-byte bank groups)
    auto swz = [](int row) { return KTB == 128 ? ((row >> 1) & 7) : ((row >> 2) & 3); };
    auto lds_off = [&](int row, int chunk) { return (row * CPR + (chunk ^ swz(row))) * 16; };
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) char smem[];
    __shared__ int s_expert, s_row0, s_rows;

    int tile_x, tile_y;
    moe_tile_of_workgroup(p, tile_x, tile_y);
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        int found_e, found_row0, found_rows;
        moe_find_tile<TM>(p, tile_y, lane, found_e, found_row0, found_rows);
        if (lane == 0) { s_expert = found_e; s_row0 = found_row0; s_rows = found_rows; }
    }
    __syncthreads();
    const int expert = s_expert;
    if (expert < 0) return;
    const int row0 = s_row0, rows = s_rows;
    const int n0 = tile_x * TN;
    if (expert == p.n_exp) {  // tokens without a valid expert id: zero rows
        moe_zero_tile<T>(p, row0, rows, n0, TN, NTH);
        return;
    }

    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const int wm = wave / WGN, wn = wave % WGN;
    const int wrow = wm * (TM / WGM), wcol = wn * (TN / WGN);
    // a partly filled tile: wavefronts whose rows are all past its end load their share of the
    // stages and meet the barriers, but read no fragments, issue no MFMAs and store nothing
    const bool active = __builtin_amdgcn_readfirstlane(wrow) < rows;

    const T* X = reinterpret_cast<const T*>(p.tokens);
    const T* W = reinterpret_cast<const T*>(p.weight) + (int64_t)expert * p.K * p.N;

    // staging map: every wavefront instruction fills 1 KB of consecutive LDS rows (8 or 16);
    // lane l lands at position l % CPR of row l / CPR, so it fetches the chunk that the
    // swizzle keeps at that position
    const int srow = threadIdx.x / CPR;
    const int chunk = (threadIdx.x % CPR) ^ swz(srow);
    const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
    const uint32_t st_dst = __builtin_amdgcn_readfirstlane(lds_base + wave * 1024);
    const T* a_src[A_LOADS];
#pragma unroll
    for (int q = 0; q < A_LOADS; ++q) {
        const int r = srow + RSTEP * q;
        const int tok = p.token_perm[row0 + (r < rows ? r : rows - 1)];
        a_src[q] = X + (int64_t)tok * p.K + chunk * VE;
    }
    // Weight tile.  [N, K] storage (k contiguous): rows of KTB bytes like the token tile.
    // [K, N] storage (BKN, the stacked weight.T of the reference): the stage is kept as
    // KT k-rows of TN * 2 bytes; a wavefront instruction fills 1 KB of them linearly, the
    // 32-byte units of a k-row are XOR-swizzled by twice its low two bits (the source
    // address carries the swizzle; the two 16-lane groups that read neighbouring units of
    // the same four k-rows then cover eight different units), and the k-contiguous MFMA fragments come out of LDS transpose
    // reads, sixteen lanes fetching four k-rows of sixteen columns at a time.
    constexpr int RB = TN * (int)sizeof(T);   // BKN: bytes of a k-row in LDS
    constexpr int CB = RB / 16;               // BKN: 16-byte slots of a k-row
    const T* b_src[B_LOADS];
#pragma unroll
    for (int q = 0; q < B_LOADS; ++q) {
        if constexpr (BKN) {
            const int slot = q * NTH + (int)threadIdx.x;
            const int kr = slot / CB, c = slot % CB;
            int n = n0 + ((((c >> 1) ^ ((kr & 3) << 1)) << 1) | (c & 1)) * VE;
            if (n + VE > p.N) n = p.N - VE;   // columns past the end re-read valid data; never stored
            b_src[q] = W + (int64_t)kr * p.N + n;
        } else {
            const int r = srow + RSTEP * q;
            const int n = n0 + r < p.N ? n0 + r : p.N - 1;
            b_src[q] = W + (int64_t)n * p.K + chunk * VE;
        }
    }
    // load q of stage s (q < A_LOADS: token rows, else weight rows)
    auto issue_one = [&](int s, int q) {
        const uint32_t dst = st_dst + (uint32_t)((s % NBUF) * BUF);
        const int k = s * KT;
        if (q < A_LOADS) lds_direct_load16(a_src[q] + k, dst + q * RSTEP * KTB);
        else if constexpr (BKN) lds_direct_load16(b_src[q - A_LOADS] + (int64_t)k * p.N, dst + A_BYTES + (q - A_LOADS) * NTH * 16);
        else lds_direct_load16(b_src[q - A_LOADS] + k, dst + A_BYTES + (q - A_LOADS) * RSTEP * KTB);
    };
    auto issue_stage = [&](int s) {
#pragma unroll
        for (int q = 0; q < A_LOADS + B_LOADS; ++q) issue_one(s, q);
    };

    // 2-byte types: 32 x 32 x 16 MFMAs (half of the fragment reads of the 16 x 16 x 32 ones, at the same rate)
    constexpr bool WIDE = HasMma32<T>::value;
    constexpr int MTW = TM / WGM / 32, NTW = TN / WGN / 32;
    const int l32 = lane & 31, h2 = lane >> 5;
    f32x4 acc[WIDE ? 1 : MT][WIDE ? 1 : NTT];
    f32x16 accw[WIDE ? MTW : 1][WIDE ? NTW : 1];
#pragma unroll
    for (int i = 0; i < (WIDE ? 1 : MT); ++i)
#pragma unroll
        for (int t = 0; t < (WIDE ? 1 : NTT); ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < (WIDE ? MTW : 1); ++i)
#pragma unroll
        for (int t = 0; t < (WIDE ? NTW : 1); ++t)
#pragma unroll
            for (int j = 0; j < 16; ++j) accw[i][t][j] = 0.f;

    const int n_st = p.K / KT;
    constexpr int L = A_LOADS + B_LOADS;   // loads per thread and stage
#pragma unroll
    for (int s0 = 0; s0 < NBUF - 1; ++s0)
        if (s0 < n_st) issue_stage(s0);

    // wait until at most `newer` stages of this thread's loads are still in flight
    auto wait_stages = [&](int newer) {
        if (NBUF > 3 && newer >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * L) : "memory");
        else if (NBUF > 2 && newer == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    };

    if constexpr (XS) {
        // Cross-stage pipeline: shallow stages (KTB bytes of k) in a ring of NBUF buffers, and the
        // barrier that publishes stage s + 1 sits ahead of the LAST k-step of stage s, whose MFMAs
        // then run over the first fragment reads of stage s + 1.  The wait for the loads, the
        // barrier and the LDS latency of a stage's first fragments - about 800 clocks that a
        // barrier at the top of the stage leaves the matrix cores idle - are covered by MFMAs
        // that are already queued.  Loads run NBUF - 1 stages ahead, so the wait is short.
        constexpr int KSTEPS = KT / 16;
        typename MmaW<T>::frag af[2][MTW], bf[2][NTW];
        auto read_frags = [&](const char* As, const char* Bs, int c, int slot) {
#pragma unroll
            for (int i = 0; i < MTW; ++i)
                af[slot][i] = *reinterpret_cast<const typename MmaW<T>::frag*>(As + lds_off(wrow + i * 32 + l32, c * 2 + h2));
#pragma unroll
            for (int t = 0; t < NTW; ++t) {
                if constexpr (BKN) {
                    typedef short s16x8_t __attribute__((ext_vector_type(8)));
                    typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;
                    const int kr = c * 16 + 8 * h2 + (r16 >> 2);             // and kr + 4
                    const int unit = (wcol + t * 32 + 16 * ((lane >> 4) & 1)) >> 4;
                    const char* at = Bs + kr * RB + ((unit ^ ((kr & 3) << 1)) << 5) + ((r16 & 3) << 3);
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(at));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(at + 4 * RB));
                    bf[slot][t] = __builtin_bit_cast(typename MmaW<T>::frag,
                                                     (s16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                } else {
                    bf[slot][t] = *reinterpret_cast<const typename MmaW<T>::frag*>(Bs + lds_off(wcol + t * 32 + l32, c * 2 + h2));
                }
            }
        };
        // The walk exists twice, with and without the fragment reads and MFMAs, chosen once per
        // wavefront: a test of `active` inside the k-steps splits them into basic blocks, and the
        // compiler then waits for ALL fragment reads in flight ahead of a step's MFMAs instead of
        // the older ones only - the reads of step c + 1 no longer run under the MFMAs of step c.
        auto walk = [&](auto act) {
        constexpr bool ACT = decltype(act)::value;
        wait_stages(n_st - 1 < NBUF - 2 ? n_st - 1 : NBUF - 2);
        __syncthreads();
        if constexpr (ACT) read_frags(smem, smem + A_BYTES, 0, 0);
        for (int s = 0; s < n_st; ++s) {
            const char* cur = smem + (s % NBUF) * BUF;
            const char* nxt = smem + ((s + 1) % NBUF) * BUF;
            const bool more = s + NBUF - 1 < n_st;
#pragma unroll
            for (int c = 0; c < KSTEPS; ++c) {
                if (c + 1 < KSTEPS) {
                    if constexpr (ACT) read_frags(cur, cur + A_BYTES, c + 1, (c + 1) & 1);
                } else if (s + 1 < n_st) {
                    // stage s + 1 has landed once only the stages after it are in flight; every
                    // fragment read of stage s has been issued by now, and is complete before
                    // the barrier lets anyone's loads into that buffer
                    const int last = s + NBUF - 1 < n_st - 1 ? s + NBUF - 1 : n_st - 1;
                    wait_stages(last - (s + 1));
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __syncthreads();
                    if constexpr (ACT) read_frags(nxt, nxt + A_BYTES, 0, 0);
                }
                // the loads of stage s + NBUF - 1 reuse the buffer of stage s - 1, which the
                // barrier inside stage s - 1 has freed
                // (all of them in the first k-step, so that the wait above counts whole stages)
                if (more && c == 0) issue_stage(s + NBUF - 1);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (ACT) {
#pragma unroll
                    for (int i = 0; i < MTW; ++i)
#pragma unroll
                        for (int t = 0; t < NTW; ++t) accw[i][t] = MmaW<T>::mma(bf[c & 1][t], af[c & 1][i], accw[i][t]);
                }
            }
        }
        };
        if (active) walk(std::true_type{}); else walk(std::false_type{});
    } else {
    // (two copies of the walk, as above)
    auto walk = [&](auto act) {
    constexpr bool ACT = decltype(act)::value;
    for (int s = 0; s < n_st; ++s) {
        // stage s has landed once at most the loads of the stages after it are outstanding
        // (NBUF - 2 of them, fewer at the end of the walk)
        const int newer = n_st - 1 - s < NBUF - 2 ? n_st - 1 - s : NBUF - 2;
        if (NBUF > 3 && newer == 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * L) : "memory");
        else if (NBUF > 2 && newer == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();   // everyone's part of stage s is in LDS; the buffer of stage s - 1 is free
        // The loads of stage s + NBUF - 1 go out a few at a time between the MFMA groups of
        // this stage (16-bit types): issued in one burst right after the barrier, the
        // sixteen wavefronts queue up behind the address unit (one 1 KB instruction per 16
        // clocks) with the matrix cores idle.
        const bool more = s + NBUF - 1 < n_st;
        if (!WIDE && more) issue_stage(s + NBUF - 1);
        const char* cur = smem + (s % NBUF) * BUF;
        const char* As = cur;
        const char* Bs = cur + A_BYTES;
        if constexpr (WIDE) {
            // fragments of k-step c + 1 are read while the MFMAs of step c run
            constexpr int KSTEPS = KT / 16;
            typename MmaW<T>::frag af[2][MTW], bf[2][NTW];
            auto read_frags = [&](int c, int slot) {
#pragma unroll
                for (int i = 0; i < MTW; ++i)
                    af[slot][i] = *reinterpret_cast<const typename MmaW<T>::frag*>(As + lds_off(wrow + i * 32 + l32, c * 2 + h2));
#pragma unroll
                for (int t = 0; t < NTW; ++t) {
                    if constexpr (BKN) {
                        typedef short s16x8_t __attribute__((ext_vector_type(8)));
                        typedef __attribute__((address_space(3))) s16x4 lds_s16x4_t;
                        const int kr = c * 16 + 8 * h2 + (r16 >> 2);             // and kr + 4
                        const int unit = (wcol + t * 32 + 16 * ((lane >> 4) & 1)) >> 4;
                        const char* at = Bs + kr * RB + ((unit ^ ((kr & 3) << 1)) << 5) + ((r16 & 3) << 3);
                        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(at));
                        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t*)(at + 4 * RB));
                        bf[slot][t] = __builtin_bit_cast(typename MmaW<T>::frag,
                                                         (s16x8_t)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                    } else {
                        bf[slot][t] = *reinterpret_cast<const typename MmaW<T>::frag*>(Bs + lds_off(wcol + t * 32 + l32, c * 2 + h2));
                    }
                }
            };
            constexpr int LPS = (L + KSTEPS - 1) / KSTEPS;  // loads per k-step
            if constexpr (ACT) read_frags(0, 0);
#pragma unroll
            for (int c = 0; c < KSTEPS; ++c) {
                if constexpr (ACT) if (c + 1 < KSTEPS) read_frags(c + 1, (c + 1) & 1);
                if (more) {
#pragma unroll
                    for (int q = c * LPS; q < (c + 1) * LPS && q < L; ++q) issue_one(s + NBUF - 1, q);
                }
                __builtin_amdgcn_sched_barrier(0);   // the reads stay ahead of this step's MFMAs
                if constexpr (ACT) {
#pragma unroll
                    for (int i = 0; i < MTW; ++i)
#pragma unroll
                        for (int t = 0; t < NTW; ++t) accw[i][t] = MmaW<T>::mma(bf[c & 1][t], af[c & 1][i], accw[i][t]);
                }
            }
        } else if constexpr (ACT) {
#pragma unroll
            for (int kc = 0; kc < KT; kc += 16) {
                typename Mma16<T>::frag af[MT], bf[NTT];
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    af[i] = *reinterpret_cast<const typename Mma16<T>::frag*>(As + lds_off(wrow + i * 16 + r16, kc / VE + g4));
#pragma unroll
                for (int t = 0; t < NTT; ++t)
                    bf[t] = *reinterpret_cast<const typename Mma16<T>::frag*>(Bs + lds_off(wcol + t * 16 + r16, kc / VE + g4));
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int t = 0; t < NTT; ++t) acc[i][t] = Mma16<T>::mma(bf[t], af[i], acc[i][t]);
            }
        }
    }
    };
    if (active) walk(std::true_type{}); else walk(std::false_type{});
    }
    __syncthreads();   // the epilogue reuses the LDS buffers
    if (!active) return;   // no barrier follows

    T* out = reinterpret_cast<T*>(p.out);
    if constexpr (WIDE) {
        // the wavefront's (TM / WGM) x 64 tile leaves through LDS (free after the last
        // barrier) as rows of 128 bytes, chunks XOR-swizzled by the row; every store
        // instruction then writes eight complete 128-byte row segments.
        // lane holds out[m = i*32 + lane%32][n = t*32 + 8*jj + 4*(lane/32) + q] in accw[i][t][4*jj + q]
        static_assert(!WIDE || TN / WGN == 64, "epilogue assumes 64 output columns per wavefront");
        constexpr int WR = TM / WGM;
        char* ep = smem + wave * (WR * 128);
#pragma unroll
        for (int i = 0; i < MTW; ++i)
#pragma unroll
            for (int t = 0; t < NTW; ++t)
#pragma unroll
                for (int jj = 0; jj < 4; ++jj) {
                    T vals[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(accw[i][t][4 * jj + q]);
                    const int row = i * 32 + l32;
                    const int ch = t * 4 + jj;
                    *reinterpret_cast<uint64_t*>(ep + row * 128 + ((ch ^ (row & 7)) << 4) + h2 * 8) =
                        *reinterpret_cast<const uint64_t*>(vals);
                }
        const int c = lane & 7;
        const int n = n0 + wcol + c * 8;
        // The token of every row this lane stores, fetched together ahead of the stores: a
        // load placed between the stores waits for the store before it as well (one counter,
        // in order), i.e. for a write to memory and a read from it per pass.
        int toks[WR / 8];
#pragma unroll
        for (int pass = 0; pass < WR / 8; ++pass) {
            const int r = wrow + pass * 8 + (lane >> 3);
            toks[pass] = r < rows ? p.token_perm[row0 + r] : -1;
        }
#pragma unroll
        for (int pass = 0; pass < WR / 8; ++pass) {
            const int row = pass * 8 + (lane >> 3);
            const u32x4 v = *reinterpret_cast<const u32x4*>(ep + row * 128 + ((c ^ (row & 7)) << 4));
            if (toks[pass] >= 0 && n < p.N) store16_through(out + (int64_t)toks[pass] * p.N + n, __builtin_bit_cast(vec16, v));
        }
    } else {
    int toks[MT];   // fetched together ahead of the stores, as above
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int r = wrow + i * 16 + r16;
        toks[i] = r < rows ? p.token_perm[row0 + r] : -1;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        if (toks[i] < 0) continue;
        const int tok = toks[i];
#pragma unroll
        for (int t = 0; t < NTT; ++t) {
            const int n = n0 + wcol + t * 16 + g4 * 4;
            T vals[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(acc[i][t][q]);
            T* dst = out + (int64_t)tok * p.N + n;
            if (n + 4 <= p.N) {
                *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(vals);
            } else {
                for (int q = 0; q < 4; ++q)
                    if (n + q < p.N) dst[q] = vals[q];
            }
        }
    }
    }
}

template <typename T, int TM, int TN, int WAVES, int WGM, int NBUF, int KTB, bool BKN, bool XS>
static int launch_moe_direct_inst(const MoeParams& p, hipStream_t st) {
    int tiles = (p.n_tok + TM - 1) / TM + p.n_exp + 1;
    if (tiles > MOE_MAX_ROW_TILES) return fail(SPX_E_SHAPE, "too many row tiles for one launch");
    const int ntn = (p.N + TN - 1) / TN;
    MoeParams q = p;
    q.col_groups = ntn % 8 == 0 || p.n_tok < (int64_t)256 * p.n_exp ? 0 : ntn % 4 == 0 ? 4 : ntn % 2 == 0 ? 2 : 1;
    if (q.col_groups && round_up(tiles, 8 / q.col_groups) > MOE_MAX_ROW_TILES) q.col_groups = 0;
    if (q.col_groups) tiles = (int)round_up(tiles, 8 / q.col_groups);
    // the epilogue stages every wavefront's (TM / WGM) x 64 output tile as rows of 128 bytes
    const int epi = sizeof(T) == 2 ? WAVES * (TM / WGM) * 128 : 0;
    const int smem = NBUF * (TM + TN) * KTB > epi ? NBUF * (TM + TN) * KTB : epi;
    SPX_GRANT_LDS((moe_gemm_direct_kernel<T, TM, TN, WAVES, WGM, NBUF, KTB, BKN, XS>), smem, "moe_gemm_direct_kernel");
    hipLaunchKernelGGL((moe_gemm_direct_kernel<T, TM, TN, WAVES, WGM, NBUF, KTB, BKN, XS>), dim3(ntn, tiles, 1), dim3(64 * WAVES), smem, st, q);
    SPX_LAUNCH_CHECK("moe_gemm_direct_kernel");
    return 0;
}

template <typename T, int TM, int TN, int WAVES, int WGM, int NBUF, int KTB, bool XS = false>
static int launch_moe_direct(const MoeParams& p, hipStream_t st) {
    if constexpr (XS && sizeof(T) != 2) {
        return fail(SPX_E_CONFIG, "the cross-stage pipelined tile configurations take 16-bit types");
    } else {
        if (p.w_kcontig) return launch_moe_direct_inst<T, TM, TN, WAVES, WGM, NBUF, KTB, false, XS>(p, st);
        if constexpr (sizeof(T) == 2) return launch_moe_direct_inst<T, TM, TN, WAVES, WGM, NBUF, KTB, true, XS>(p, st);
        else return fail(SPX_E_CONFIG, "fp32 weights stored [E, in, out] run through tile config 1");
    }
}

// ---- few rows per expert --------------------------------------------------------------------
// With a handful of tokens to an expert the product is the reading of the weights, and a 128-row tile reads
// them in one serial chain per (expert, 128 columns): 8 experts of 2048 x 768 kept 48 of 256 CUs busy for 22 us.
// Here a workgroup takes 32 rows x 128 columns and each of its four wavefronts a quarter of k, through a ring of
// its own (two stages of 32 k, filled global -> LDS directly: 8 KB of weights, 2 KB of tokens), so that no
// barrier stands between a load and its use; the wavefronts add up through LDS once.  22.8 -> 11.5 us there (25 MB
// of weights: 2.2 TB/s, bound by the loads a CU keeps in flight on 48 CUs); ranges of k over several
// workgroups, added up by a second kernel, cost more than they gave (2 ranges 10.3 us, but 16.0 -> 19.5 for
// 1000 x 2048 -> 768, 8.0 -> 11.1 for 64 x 1024 -> 4096 over 4).  [E, in, out] weights, 16-bit types.
constexpr int MOE_ROWS_TM = 32, MOE_ROWS_TN = 128, MOE_ROWS_KT = 32;
constexpr int MOE_ROWS_STAGE = (MOE_ROWS_TM + MOE_ROWS_TN) * MOE_ROWS_KT * 2;   // bytes
constexpr int MOE_ROWS_PITCH = MOE_ROWS_TN + 4;                                // floats per row of a wavefront's partial tile
constexpr int MOE_ROWS_WAVE = 2 * MOE_ROWS_STAGE;                              // LDS of a wavefront
static_assert(MOE_ROWS_TM * MOE_ROWS_PITCH * 4 <= MOE_ROWS_WAVE, "the partial tile reuses the ring");

template <typename T>
__global__ __launch_bounds__(256, 2) void moe_rows_kernel(MoeParams p) {
    constexpr int TM = MOE_ROWS_TM, TN = MOE_ROWS_TN, KT = MOE_ROWS_KT, NT = TN / 32;
    constexpr int W_BYTES = KT * TN * 2;
    constexpr int W_LOADS = W_BYTES / 1024, LOADS = MOE_ROWS_STAGE / 1024;
    typedef typename MmaW<T>::frag Frag;
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    extern __shared__ __align__(16) char smem[];

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int expert, row0, rows;
    moe_find_tile<TM>(p, blockIdx.y, lane, expert, row0, rows);
    expert = __builtin_amdgcn_readfirstlane(expert);
    row0 = __builtin_amdgcn_readfirstlane(row0);
    rows = __builtin_amdgcn_readfirstlane(rows);
    if (expert < 0) return;
    const int n0 = blockIdx.x * TN;

    f32x16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[t][j] = 0.f;
    char* ring = smem + wave * MOE_ROWS_WAVE;
    if (expert < p.n_exp) {   // the pseudo expert's rows stay zero
        const int n_st = p.K / KT;
        const int s_begin = n_st * wave / 4, s_end = n_st * (wave + 1) / 4;
        const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * MOE_ROWS_WAVE;
        // weights: a load instruction fills four k-rows of 256 bytes, their 32-byte units XORed by twice the
        // low two bits of the row (as in moe_gemm_direct_kernel); columns past the end re-read valid ones
        const int kr = lane >> 4, c = lane & 15;
        int n = n0 + ((((c >> 1) ^ (kr << 1)) << 1) | (c & 1)) * 8;
        if (n + 8 > p.N) n = p.N - 8;
        const T* w_src = reinterpret_cast<const T*>(p.weight) + (int64_t)expert * p.K * p.N + (int64_t)kr * p.N + n;
        // tokens: sixteen rows of 64 bytes, chunks XORed by bits 2 and 3 of the row; rows past the end re-read the last one
        const T* a_src[2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int r = q * 16 + (lane >> 2);
            a_src[q] = reinterpret_cast<const T*>(p.tokens) + (int64_t)p.token_perm[row0 + (r < rows ? r : rows - 1)] * p.K +
                       ((lane & 3) ^ ((r >> 2) & 3)) * 8;
        }
        auto issue = [&](int s) {
            const uint32_t to = lds + (uint32_t)((s - s_begin) & 1) * MOE_ROWS_STAGE;
#pragma unroll
            for (int q = 0; q < W_LOADS; ++q) lds_direct_load16(w_src + (int64_t)(s * KT + q * 4) * p.N, to + q * 1024);
#pragma unroll
            for (int q = 0; q < 2; ++q) lds_direct_load16(a_src[q] + s * KT, to + W_BYTES + q * 1024);
        };
        const int l32 = lane & 31, h2 = lane >> 5, r16 = lane & 15;
        if (s_begin < s_end) issue(s_begin);
        if (s_begin + 1 < s_end) issue(s_begin + 1);
        for (int s = s_begin; s < s_end; ++s) {
            if (s + 1 < s_end) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            const char* W = ring + ((s - s_begin) & 1) * MOE_ROWS_STAGE;
            const char* A = W + W_BYTES;
            Frag af[KT / 16], wf[KT / 16][NT];
#pragma unroll
            for (int k = 0; k < KT / 16; ++k) {
                af[k] = *reinterpret_cast<const Frag*>(A + l32 * 64 + (((k * 2 + h2) ^ ((l32 >> 2) & 3)) << 4));
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int row = k * 16 + 8 * h2 + (r16 >> 2);   // and row + 4: the same low two bits
                    const int unit = t * 2 + ((lane >> 4) & 1);
                    const char* at = W + row * (TN * 2) + ((unit ^ ((row & 3) << 1)) << 5) + ((r16 & 3) << 3);
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 4 * TN * 2));
                    wf[k][t] = __builtin_bit_cast(Frag, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the fragments are out of the buffer that is refilled now
            if (s + 2 < s_end) issue(s + 2);
#pragma unroll
            for (int k = 0; k < KT / 16; ++k)
#pragma unroll
                for (int t = 0; t < NT; ++t) acc[t] = MmaW<T>::mma(wf[k][t], af[k], acc[t]);
        }
    }

    // lane holds D[n = t*32 + 8*jj + 4*(lane/32) + q][m = lane % 32] in acc[t][4*jj + q]
    float* mine = reinterpret_cast<float*>(ring);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
            *reinterpret_cast<f32x4*>(mine + (lane & 31) * MOE_ROWS_PITCH + t * 32 + 8 * jj + 4 * (lane >> 5)) =
                f32x4{acc[t][4 * jj], acc[t][4 * jj + 1], acc[t][4 * jj + 2], acc[t][4 * jj + 3]};
    __syncthreads();
    for (int i = threadIdx.x; i < rows * (TN / 4); i += 256) {
        const int row = i / (TN / 4), col = (i % (TN / 4)) * 4;
        if (n0 + col >= p.N) continue;
        f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < 4; ++w)
            sum += *reinterpret_cast<const f32x4*>(smem + w * MOE_ROWS_WAVE + (row * MOE_ROWS_PITCH + col) * 4);
        const int tok = p.token_perm[row0 + row];
        T vals[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(sum[q]);
        *reinterpret_cast<uint64_t*>(reinterpret_cast<T*>(p.out) + (int64_t)tok * p.N + n0 + col) = *reinterpret_cast<const uint64_t*>(vals);
    }
}

template <typename T>
static int launch_moe_rows(const MoeParams& p, hipStream_t st) {
    const int tiles = (p.n_tok + MOE_ROWS_TM - 1) / MOE_ROWS_TM + p.n_exp + 1;
    if (tiles > MOE_MAX_ROW_TILES) return fail(SPX_E_SHAPE, "too many row tiles for one launch");
    constexpr int smem = 4 * MOE_ROWS_WAVE;
    SPX_GRANT_LDS((moe_rows_kernel<T>), smem, "moe_rows_kernel");
    hipLaunchKernelGGL((moe_rows_kernel<T>), dim3((p.N + MOE_ROWS_TN - 1) / MOE_ROWS_TN, tiles, 1), dim3(256), smem, st, p);
    SPX_LAUNCH_CHECK("moe_rows_kernel");
    return 0;
}

// Tokens per workgroup of the index kernels: the smallest multiple of 256 (up to MOE_CHUNK)
// whose table of (chunk, expert) counts the placement workgroups can scan themselves;
// else 256 (more beyond 262144 tokens, so that a launch has at most 1024 chunks)
// with a launch in between that scans every expert's column of the table.
static int moe_index_chunk(int n_tok, int n_exp, bool* fused) {
    for (int chunk = 256; chunk <= MOE_CHUNK; chunk += 256) {
        const int64_t n_chunk = (n_tok + chunk - 1) / chunk;
        if (n_chunk * (n_exp + 1) <= MOE_FUSED_TABLE) { *fused = true; return chunk; }
    }
    *fused = false;
    int chunk = 256;
    while ((n_tok + chunk - 1) / chunk > 1024) chunk += 256;
    return chunk;
}

// [n_chunk][n_exp + 1] counts, then the n_exp + 1 totals of the experts
static size_t moe_index_table_bytes(int n_tok, int n_exp) {
    bool fused;
    const int chunk = moe_index_chunk(n_tok, n_exp, &fused);
    const int n_chunk = (n_tok + chunk - 1) / chunk;
    return round_up((size_t)(n_chunk > 0 ? n_chunk : 1) * (n_exp + 1) * sizeof(int32_t), 256);
}

static size_t moe_index_ws(int n_tok, int n_exp) {
    return moe_index_table_bytes(n_tok, n_exp) + round_up((size_t)(n_exp + 1) * sizeof(int32_t), 256);
}

}  // namespace spx

extern "C" size_t spx_moe_index_workspace_bytes(int n_tok, int n_exp) {
    if (n_tok < 0 || n_exp <= 0 || n_exp > spx::MOE_MAX_EXP) return 0;
    return spx::moe_index_ws(n_tok, n_exp);
}

extern "C" int spx_moe_index(const int32_t* exp_ids, int n_tok, int n_exp,
                             int32_t* expert_count, int32_t* expert_offset, int32_t* token_perm,
                             void* workspace, size_t workspace_bytes, spx_stream_t stream) {
    using namespace spx;
    SPX_REQUIRE(n_tok >= 0, SPX_E_SHAPE, "negative token count");
    SPX_REQUIRE(n_exp > 0 && n_exp <= MOE_MAX_EXP, SPX_E_SHAPE, "n_exp=%d must be in [1,%d]", n_exp, MOE_MAX_EXP);
    SPX_REQUIRE(expert_count && expert_offset && workspace, SPX_E_NULL, "expert_count, expert_offset and workspace are required");
    SPX_REQUIRE((exp_ids && token_perm) || n_tok == 0, SPX_E_NULL, "exp_ids and token_perm are required");
    SPX_REQUIRE(workspace_bytes >= moe_index_ws(n_tok, n_exp), SPX_E_WORKSPACE,
                "workspace of %zu bytes is smaller than the %zu required", workspace_bytes, moe_index_ws(n_tok, n_exp));
    SPX_REQUIRE(aligned(workspace, 256), SPX_E_ALIGN, "workspace must be 256-byte aligned");
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    int32_t* partial = reinterpret_cast<int32_t*>(workspace);
    if (n_tok > MOE_SELF_COUNT && n_tok <= MOE_ONE_TOKENS && n_exp <= MOE_ONE_EXPERTS) {
        hipLaunchKernelGGL(moe_index_kernel, dim3((n_tok + MOE_ONE_THREADS - 1) / MOE_ONE_THREADS), dim3(MOE_ONE_THREADS), 0, st, exp_ids, n_tok,
                           n_exp + 1, token_perm, expert_count, expert_offset);
        SPX_LAUNCH_CHECK("moe_index_kernel");
        return 0;
    }
    bool fused;
    const int chunk = moe_index_chunk(n_tok, n_exp, &fused);
    const int n_chunk = (n_tok + chunk - 1) / chunk;
    const bool self_count = fused && n_tok <= MOE_SELF_COUNT;
    if (n_chunk > 0 && !self_count) {
        hipLaunchKernelGGL(moe_hist_kernel, dim3(n_chunk), dim3(256), (n_exp + 1) * sizeof(int), st, exp_ids, n_tok, n_exp + 1, chunk, partial);
        SPX_LAUNCH_CHECK("moe_hist_kernel");
    }
    int32_t* totals = reinterpret_cast<int32_t*>(reinterpret_cast<char*>(workspace) + moe_index_table_bytes(n_tok, n_exp));
    if (n_chunk == 0) {   // no tokens: all offsets and counts are zero (a kernel, so that the call can be captured)
        hipLaunchKernelGGL(moe_zero_index_kernel, dim3((n_exp + 1 + 255) / 256), dim3(256), 0, st, n_exp, expert_count, expert_offset);
        SPX_LAUNCH_CHECK("moe_zero_index_kernel");
        return 0;
    }
    if (!fused) {
        hipLaunchKernelGGL(moe_colscan_kernel, dim3((n_exp + 1 + 3) / 4), dim3(256), 0, st, partial, n_chunk, n_exp + 1, totals);
        SPX_LAUNCH_CHECK("moe_colscan_kernel");
    }
    const size_t smem = 6 * (n_exp + 1) * sizeof(int);
    if (fused)
        hipLaunchKernelGGL(moe_place_kernel<true>, dim3(n_chunk), dim3(256), smem, st, exp_ids, n_tok, n_exp + 1, chunk,
                           self_count ? nullptr : partial,
                           totals, token_perm, expert_count, expert_offset);
    else
        hipLaunchKernelGGL(moe_place_kernel<false>, dim3(n_chunk), dim3(256), smem, st, exp_ids, n_tok, n_exp + 1, chunk, partial,
                           totals, token_perm, expert_count, expert_offset);
    SPX_LAUNCH_CHECK("moe_place_kernel");
    return 0;
}

extern "C" int spx_moe_forward(int dtype, const void* tokens, const void* weight, int weight_layout, void* out,
                               const int32_t* expert_offset, const int32_t* token_perm,
                               int n_tok, int in_dim, int out_dim, int n_exp,
                               int tile_cfg, spx_stream_t stream) {
    using namespace spx;
    SPX_REQUIRE(tile_cfg >= 0 && tile_cfg <= 7, SPX_E_CONFIG, "unknown tile config %d", tile_cfg);
    SPX_REQUIRE(dtype == SPX_F32 || dtype == SPX_F16 || dtype == SPX_BF16, SPX_E_DTYPE, "unknown dtype %d", dtype);
    SPX_REQUIRE(n_tok >= 0 && in_dim > 0 && out_dim > 0 && n_exp > 0, SPX_E_SHAPE, "bad sizes");
    SPX_REQUIRE(weight_layout == 0 || weight_layout == 1, SPX_E_CONFIG, "weight_layout must be 0 ([E,in,out]) or 1 ([E,out,in])");
    const int es = dtype_bytes(dtype);
    SPX_REQUIRE(in_dim % (128 / es) == 0, SPX_E_SHAPE, "in_dim=%d must be a multiple of %d", in_dim, 128 / es);
    SPX_REQUIRE(out_dim % (16 / es) == 0, SPX_E_SHAPE, "out_dim=%d must be a multiple of %d", out_dim, 16 / es);
    if (n_tok == 0) return 0;
    SPX_REQUIRE(tokens && weight && out && expert_offset && token_perm, SPX_E_NULL, "a required buffer is NULL");
    SPX_REQUIRE(aligned(tokens, 16) && aligned(weight, 16) && aligned(out, 16), SPX_E_ALIGN, "buffers must be 16-byte aligned");
    MoeParams p;
    p.tokens = tokens; p.weight = weight; p.out = out;
    p.expert_offset = expert_offset; p.token_perm = token_perm;
    p.n_tok = n_tok; p.K = in_dim; p.N = out_dim; p.n_exp = n_exp;
    p.w_kcontig = weight_layout == 1;
    p.col_groups = 0;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // tile_cfg 1: 128x128 tiles staged through registers (any dtype and weight layout);
    // 2 / 3 / 4: tiles filled by LDS-direct loads - 128x128 with four wavefronts (two
    // workgroups per CU; eight for 16-bit [E, in, out] weights: 700 x 2048 -> 2048 over 16 bf16 40.4 -> 37.8 us,
    // 2113 x 2048 -> 2048 over 8 fp16 44.5 -> 38.7, 1342 x 1024 -> 4096 over 8 30.1 -> 27.5), 256x256 with eight wavefronts of
    // 128x64, 256x256 with sixteen wavefronts of 64x64 - for 16-bit types in either weight layout and fp32 with
    // k-contiguous weights.  256x256 tiles move half the bytes from L2 to the CUs, which is
    // what bounds the 128x128 kernel.  5: 256x256 tiles by workgroups that stay on their CU (moe_persist.hip; 4 where it
    // does not take the type or the sizes).  7: 32-row
    // tiles for few rows per expert (16-bit, [E, in, out] weights).  0 picks between 7, 5, 4, 2 and, for 16-bit
    // [E, in, out] weights, 64 x 128 tiles of two or three stages that have no number of their own, by the number of
    // tiles and of rows per expert (below); fp32 [E, in, out] weights take 1.
    const bool direct_ok = p.w_kcontig || es == 2;
    static int n_cu = 0;
    if (n_cu == 0) {
        int dev = 0;
        hipDeviceProp_t prop;
        if (hipGetDevice(&dev) == hipSuccess && hipGetDeviceProperties(&prop, dev) == hipSuccess) n_cu = prop.multiProcessorCount;
        if (n_cu <= 0) n_cu = 256;
    }
    const bool persist_ok = es == 2 && persist_fits(n_tok, in_dim, out_dim, n_exp, p.w_kcontig != 0, n_cu);
    int stages64 = 0;   // 64 x 128 tiles with that many stages
    if (tile_cfg == 0) {
        // 16-bit types: 256x256 tiles by persistent workgroups (5) from 224 of them on; with experts of many rows, whose last
        // tiles waste little, from fewer on, and the fewer the longer the walk over k.  us of the best other choice below /
        // persistent: 3346 x 1024 -> 4096 over 16 (224 tiles) 62.5 / 53.1, 2670 x 768 -> 4096 over 16 (176, 166 rows each) 45.4 / 41.0,
        // 3569 x 768 -> 3072 over 8 (168) 34.0 / 31.4, 4564 x 1024 -> 2048 over 4 (144) 35.7 / 34.2, 9889 x 2048 -> 768 over 4 (117)
        // 46.1 / 41.0, 6673 x 2048 -> 768 over 8 (81) 42.7 / 38.4; but 3640 x 2048 -> 2048 over 4 (120) 45.8 / 49.3, 10529 x 768 -> 768 over 4 (126) 27.3 / 28.5, 2911 x 1024 -> 3072
        // over 16 (144, 181 rows each) 41.6 / 46.7, 3254 x 1024 -> 3072 over 32 (156, 101 rows each) level, 1994 x 2048 -> 768 over 8
        // (24) 25.3 / 29.5.  256x256 tiles of one workgroup each (4) where k is too short for the pipeline (16384 x 64 -> 4096 over 8 43.3 us,
        // with a second launch of 128-row tiles for what whole rounds leave 45.4; k of 192 64.6 / 63.8, 40000 tokens over 32 158 / 152): from 128 on when
        // all of them, the partly filled ones at the expert boundaries included, run in a
        // single round (ten mid-size problems measured 10 - 25 % ahead of the 128x128
        // tiles there, and behind them as soon as a second round starts); else 128x128
        const int64_t row_tiles = (n_tok + 255) / 256, col_tiles = (out_dim + 255) / 256;
        const int64_t big_tiles = row_tiles * col_tiles;
        // 32-row tiles whose wavefronts split k, while tiles of 128 rows (one at least to every expert with tokens) leave
        // CUs idle and hold few rows each.  fp16 us, 128-row tiles / these: 64 x 1024 -> 4096 over 4 13.5 / 8.0,
        // 100 x 2048 -> 3072 over 8 26.5 / 18.8, 333 x 1024 -> 768 over 16 14.8 / 9.0, 1000 x 2048 -> 768 over 8 26 / 16,
        // 39 x 2048 -> 768 over 32 27 / 12.6, 1000 x 768 -> 768 over 32 (240 tiles) 14.4 / 12.7; with 384 - 446 tiles
        // 16.0 / 16.2 (500 x 768 -> 4096 over 8), 21.0 / 24.5 (333 x 1024 -> 3072 over 16), at 256 rows per expert
        // 15.7 / 15.9 (2048 x 1024 -> 768 over 8).
        const int64_t tiles128 = ((n_tok + 127) / 128 + (int64_t)(n_tok < n_exp ? n_tok : n_exp)) * ((out_dim + 127) / 128);
        const bool few_rows = es == 2 && !p.w_kcontig && tiles128 <= 256 && n_tok <= (int64_t)128 * n_exp;
        const bool many_rows = n_tok >= (int64_t)256 * n_exp;
        // long walks: where tiles of 256 rows go out as halves, or tiles of 128 rows are more than two to a CU (half a tile
        // of every expert is unused, give or take)
        const bool long_walk = in_dim >= 2048 && big_tiles >= 64 &&
                               ((row_tiles + n_exp / 2) * col_tiles <= n_cu / 2 ||
                                ((n_tok + 127) / 128 + n_exp / 2) * ((out_dim + 127) / 128) > 2 * n_cu);
        const bool persist = persist_ok &&
                             (big_tiles >= 224 || (big_tiles >= 160 && n_tok >= (int64_t)128 * n_exp) ||
                              (many_rows && (big_tiles >= 130 || long_walk)));
        if (!direct_ok) tile_cfg = 1;
        else if (few_rows) tile_cfg = 7;
        else if (persist) tile_cfg = 5;
        else if (es == 2 && big_tiles >= 256) tile_cfg = 4;
        else if (es == 2 && big_tiles >= 128 && (row_tiles + n_exp) * col_tiles <= n_cu) tile_cfg = 4;
        // experts of more than a 256-row tile leave half a tile unused each, give or take: also where that many fit a round
        // (16108 x 768 -> 768 over 32 fp16 47.0 / 40.3 us with 128- and 256-row tiles, 4718 x 768 -> 2048 over 16 40.9 / 36.8;
        // 1592 x 1024 -> 4096 over 16, fewer rows, 42.4 / 46.1; 10421 x 768 -> 768 over 8, 123 tiles, 26.0 / 31.2)
        else if (es == 2 && big_tiles >= 150 && n_tok >= (int64_t)256 * n_exp && (row_tiles + n_exp * 5 / 8) * col_tiles <= n_cu) tile_cfg = 4;
        else {
            tile_cfg = 2;
            // 64-row tiles, three stages deep where the workgroups are few (51 x 2048 -> 2048 over 16 bf16 33.1 / 23.4 us,
            // 1976 x 768 -> 768 over 8 21.8 / 18.0, 3821 x 2048 -> 768 over 4 35.9 / 31.3; 375 x 2048 -> 2048 over 16, 304 tiles,
            // 31.9 with two / 35.9), two where the experts have few rows (375 x 2048 -> 2048 over 16 40.3 / 31.9,
            // 1130 x 1024 -> 2048 over 32 44.2 / 36.0, 68 x 768 -> 3072 over 32 34.9 / 26.9; 2110 x 1024 -> 4096 over 32, 65 rows
            // each, 76 / 80; 139 x 768 -> 4096 over 32, 1088 tiles, 38.6 / 40.6)
            if (es == 2 && !p.w_kcontig) {
                if (tiles128 <= (n_tok <= (int64_t)64 * n_exp ? 288 : 224)) stages64 = 3;
                else if (n_tok <= (int64_t)48 * n_exp && tiles128 <= 1024) stages64 = 2;
            }
        }
    }
    if (tile_cfg == 7) {
        SPX_REQUIRE(es == 2 && !p.w_kcontig, SPX_E_CONFIG, "tile config 7 takes 16-bit types and weights stored [E, in, out]");
        return dtype == SPX_F16 ? launch_moe_rows<_Float16>(p, st) : launch_moe_rows<bf16_t>(p, st);
    }
    if (tile_cfg >= 2) {
        SPX_REQUIRE(direct_ok, SPX_E_CONFIG, "tile config %d takes fp32 weights in layout 1 only", tile_cfg);
        if (tile_cfg == 5 && !persist_ok) tile_cfg = 4;
#define SPX_MOE_DIRECT(T)                                                                  \
        if constexpr (sizeof(T) == 2)                                                      \
            if (tile_cfg == 5) return launch_moe_persist<T>(p, n_cu, st);                  \
        if (tile_cfg == 6) return launch_moe_direct<T, 256, 256, 16, 4, 4, 64, true>(p, st); \
        if constexpr (sizeof(T) == 2) {                                                    \
            if (stages64 == 2) return launch_moe_direct_inst<T, 64, 128, 4, 2, 2, 128, true, false>(p, st); \
            if (stages64 == 3) return launch_moe_direct_inst<T, 64, 128, 4, 2, 3, 128, true, false>(p, st); \
            if (tile_cfg == 2 && !p.w_kcontig) return launch_moe_direct_inst<T, 128, 128, 8, 4, 2, 128, true, false>(p, st); \
        }                                                                                  \
        if (tile_cfg == 2) return launch_moe_direct<T, 128, 128, 4, 2, 2, 128>(p, st);     \
        if (tile_cfg == 3) return launch_moe_direct<T, 256, 256, 8, 2, 2, 128>(p, st);     \
        return launch_moe_direct<T, 256, 256, 16, 4, 2, 128>(p, st);
        switch (dtype) {
            case SPX_F32: SPX_MOE_DIRECT(float)
            case SPX_F16: SPX_MOE_DIRECT(_Float16)
            default: SPX_MOE_DIRECT(bf16_t)
        }
#undef SPX_MOE_DIRECT
    }
    const int max_tiles = (n_tok + MOE_TM - 1) / MOE_TM + n_exp + 1;
    SPX_REQUIRE(max_tiles <= MOE_MAX_ROW_TILES, SPX_E_SHAPE, "too many row tiles for one launch");
    dim3 grid((out_dim + MOE_TN - 1) / MOE_TN, max_tiles, 1);
    const size_t smem = 2 * (size_t)MOE_TM * 128;
    switch (dtype) {
        case SPX_F32: hipLaunchKernelGGL(moe_gemm_kernel<float>, grid, dim3(256), smem, st, p); break;
        case SPX_F16: hipLaunchKernelGGL(moe_gemm_kernel<_Float16>, grid, dim3(256), smem, st, p); break;
        default: hipLaunchKernelGGL(moe_gemm_kernel<bf16_t>, grid, dim3(256), smem, st, p); break;
    }
    SPX_LAUNCH_CHECK("moe_gemm_kernel");
    return 0;
}
