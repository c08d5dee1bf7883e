// Fused block-sparse and sequence-length attention forward with 32 queries per wavefront.
#include "attention.hpp"

namespace spx {

// ---- wide variant: 32 queries per wavefront, 32 x 32 x 16 MFMAs ---------------------------
//   S^T[key][query] (A = K rows from LDS, B = Q from registers): lane l holds, for query
//   l % 32, the keys 8a + 4(l / 32) + b (a, b = 0..3) of a 32-key tile in s[4a + b];
//   O^T[e][query] += V^T P^T in 16-key steps: k-slot i of half h = l / 32 is key
//   16u + 8(i / 4) + 4h + i % 4, which is s[8(u % 2) + i] of tile u / 2 - the probabilities go
//   from the accumulator straight into the B operand - and for V^T two LDS transpose reads
//   (keys 16u + 4h .. +3 and 16u + 8 + 4h .. +3 of column e).
//   Row sums of the rounded probabilities: 4 x 4 x 4 MFMAs against ones.  Their B operand is a
//   column per lane with its four k in the lane's registers, so every lane sums its own values
//   (two lanes per query, joined at the end) and no query meets another one's NaN.
// K and V tiles go global -> LDS directly, two buffers, one barrier per step: no staging
// registers, so the 32-query accumulators fit 128 registers at head dim 64 and four wavefronts
// share a SIMD.  Per wavefront and 32 x 64 scores: 16 MFMAs of 32 clocks (+ 8 small ones), 32 quarter-rate
// exponentials of 16 clocks and about 85 other vector instructions of 4: vector issue bounds the kernel
// (850 against 580 clocks), 26 us at 32 x 12 x 1024 x 64 with mixed lengths, which takes 56 us (64 before the work was ordered; 610 TFLOP/s).
// Measured and left out: one 32-key tile at a time, exponentials under the next tile's MFMAs (+3 %).  Both tiles keep rows of E elements without padding; the 16-byte chunks of a row
// are XORed by a function of the row (k_swizzle, v_swizzle) for which the 16 lanes of a
// fragment read and the 32 lanes of a transpose read cover all 64 banks.
template <int E> __device__ __forceinline__ int attn_k_swizzle(int row) { return E == 64 ? (row >> 1) & 7 : row & 15; }
template <int E> __device__ __forceinline__ int attn_v_swizzle(int row) { return E == 64 ? (row & 2) << 1 : (row & 3) << 2; }

// two buffers of K and V tiles; the same space carries the output rows at the end (16 bytes of padding each)
constexpr int attn_wide_smem(int BW, int E, int waves) {
    const int tiles = 2 * BW * E * 4, rows = waves * 32 * (E * 2 + 16);
    return tiles > rows ? tiles : rows;
}

// Sequence-length mode: what work item `slot` of XCD `xcd` is.  The (entry, head) pairs are dealt out to the XCDs longest
// entry first, and an XCD walks the query blocks that hold positions of its pairs before the ones that only get zeros:
// those are over in no time, and between the others they kept a third of the slots from work (32 x 12 x 1024 with mixed
// lengths: 2300 of 3650 wavefronts were at it half way through the launch).  Groups of 64 entries at a time, their
// lengths in the lanes of the wavefront.
struct SeqWork {
    int64_t b;      // entry * heads + head
    int br, len;    // query block; br * ROWS >= len: rows of zeros
};
template <int ROWS>
__device__ __forceinline__ bool seqlen_work(const AttnParams& p, int entries, int nbr, int slot, int xcd, SeqWork& w) {
    const int per_group = 8 * p.heads * nbr;   // 64 entries: 64 * heads / 8 pairs on an XCD
    const int first = slot / per_group * 64;
    int t = slot % per_group;
    const int n = entries - first < 64 ? entries - first : 64;
    const int lane = lane_id();
    int mine = -1;
    if (lane < n) {
        mine = p.seqlens[first + lane];
        mine = mine < 0 ? 0 : mine > p.Ns ? p.Ns : mine;
    }
    int rank = 0;   // lanes without an entry stay behind all others
    for (int j = 0; j < n; ++j) {
        const int other = __builtin_amdgcn_readlane(mine, j);
        rank += (other > mine || (other == mine && j < lane)) ? 1 : 0;
    }
    if (lane >= n) rank = lane;
    // from here on lane r holds the r-th longest entry
    const int len = __builtin_amdgcn_ds_permute(rank * 4, mine), id = __builtin_amdgcn_ds_permute(rank * 4, lane);
    const int busy = len > 0 ? (len + ROWS - 1) / ROWS : 0;
    const int pair0 = (first + lane) * p.heads;
    const int lo = (pair0 - xcd + 7) >> 3, hi = (pair0 + p.heads - xcd + 7) >> 3;   // its pairs 8 k + xcd
    const int pairs = lane < n ? hi - lo : 0;
    int share = pairs * busy, upto = wave_inclusive_scan(share), blocks = busy, skip = 0;
    const int total = __builtin_amdgcn_readlane(upto, 63);
    if (t >= total) {
        t -= total;
        blocks = nbr - busy;
        skip = busy;
        share = pairs * blocks;
        upto = wave_inclusive_scan(share);
    }
    const uint64_t past = __builtin_amdgcn_ballot_w64(upto > t);
    if (past == 0) return false;
    const int r = __builtin_ctzll(past);
    t -= __builtin_amdgcn_readlane(upto - share, r);
    const int of = __builtin_amdgcn_readlane(blocks, r);
    const int pair = 8 * (__builtin_amdgcn_readlane(lo, r) + t / of) + xcd;
    w.b = (int64_t)(first + __builtin_amdgcn_readlane(id, r)) * p.heads + pair % p.heads;
    w.br = __builtin_amdgcn_readlane(skip, r) + t % of;
    w.len = __builtin_amdgcn_readlane(len, r);
    return true;
}

template <typename T, int BW, int E, int WAVES, bool HAS_MASK, bool SEQ = false>
__global__ __launch_bounds__(64 * WAVES, E == 64 && BW <= 64 ? (HAS_MASK ? 3 : 4) : 2) void attention_wide_kernel(AttnParams p, int nbr, int batch) {
    static_assert(!SEQ || !HAS_MASK, "sequence-length mode: no mask bytes");
    constexpr int NT = 64 * WAVES;
    constexpr int KT = BW / 32, EC = E / 16, ET = E / 32, KS = BW / 16;
    constexpr int ROW = E * 2;                // bytes of a K / V row
    constexpr int VT = BW * ROW;              // byte offset of the V tile
    constexpr int TILE = 2 * VT;
    constexpr int VPR = E / 8;                // 16-byte chunks per row
    constexpr int NV = BW * VPR / NT;         // chunks per thread and tile
    constexpr int RSTEP = NT / VPR;           // rows between a thread's chunks
    static_assert(BW * VPR % NT == 0 && NT % VPR == 0 && NV >= 1 && NV <= 8, "tile does not split over the workgroup");
    typedef typename MmaW<T>::frag Frag;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    extern __shared__ __align__(16) char smem[];

    // workgroup L runs on XCD L % 8: give each XCD whole batch*head entries
    const int L = blockIdx.x;
    const int slot = L >> 3;
    int64_t b;
    int br, seq_len = 0;
    if constexpr (SEQ) {
        SeqWork w;
        if (!seqlen_work<32 * WAVES>(p, batch / p.heads, nbr, slot, L & 7, w)) return;
        b = w.b;
        br = w.br;
        seq_len = w.len;
        if (br * (32 * WAVES) >= seq_len) {   // rows of zeros
            const int rows = p.Nt - br * (32 * WAVES) < 32 * WAVES ? p.Nt - br * (32 * WAVES) : 32 * WAVES;
            char* dst = reinterpret_cast<char*>(reinterpret_cast<T*>(p.out) + (b * p.Nt + br * (32 * WAVES)) * E);
            for (int v = threadIdx.x; v < rows * VPR; v += NT)
                __builtin_nontemporal_store(u32x4{0u, 0u, 0u, 0u}, reinterpret_cast<u32x4*>(dst + v * 16));
            return;
        }
    } else {
        b = (slot / nbr) * 8 + (L & 7);
        br = slot % nbr;
        if (b >= batch) return;
    }

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l32 = lane & 31, h2 = lane >> 5;

    const T* Q = reinterpret_cast<const T*>(p.q) + b * (int64_t)p.Nt * E;
    const T* Kg = reinterpret_cast<const T*>(p.k) + b * (int64_t)p.Ns * E;
    const T* Vg = reinterpret_cast<const T*>(p.v) + b * (int64_t)p.Ns * E;
    T* O = reinterpret_cast<T*>(p.out) + b * (int64_t)p.Nt * E;

    const int row0 = br * (32 * WAVES) + wave * 32;   // first query of this wavefront
    const int qrow = row0 + l32;
    const bool rows_exist = !SEQ || row0 < p.Nt;      // Nt is a multiple of 32: a wavefront is inside or outside
    Frag qf[EC];
#pragma unroll
    for (int c = 0; c < EC; ++c)
        qf[c] = *reinterpret_cast<const Frag*>(Q + (int64_t)(rows_exist ? qrow : 0) * E + c * 16 + h2 * 8);

    f32x16 oacc[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) oacc[t][j] = 0.f;
    f32x4 lacc = f32x4{0.f, 0.f, 0.f, 0.f};
    // m: reference point of this lane's query; set to the row maximum by the first block with a
    // live entry, later moved only when a maximum outgrows it by more than 2^RESCALE_LOG2
    float c2 = p.inv_t * 1.4426950408889634f;
    if (!SEQ && c2 <= 0.f) {
        // The maximum is taken ahead of the scaling and a dead score is -inf: both want a positive factor.  The
        // sign of a negative one goes into the queries; with zero every live entry weighs the same.
        const uint32_t keep = c2 < 0.f ? 0xffffffffu : 0u, flip = c2 < 0.f ? 0x80008000u : 0u;
#pragma unroll
        for (int c = 0; c < EC; ++c) qf[c] = __builtin_bit_cast(Frag, (__builtin_bit_cast(u32x4, qf[c]) & keep) ^ flip);
        c2 = c2 < 0.f ? -c2 : 1.f;
    }
    float m_run = 0.f;
    bool fresh = true;
    constexpr float RESCALE_LOG2 = 6.f;
    constexpr float DEAD = -__builtin_inff();

    // staging map: chunk v = tid + i * NT of a tile lands at LDS offset 16 v, i.e. in place
    // v % VPR of row v / VPR, and is the row's chunk (v % VPR) ^ swizzle(row)
    const int st_row = threadIdx.x / VPR, st_slot = threadIdx.x % VPR;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem + wave * 1024;
    // fragment bases
    const int k_src = l32 * ROW;
    const int k_sw = attn_k_swizzle<E>(l32);
    const int v_key = h2 * 4 + ((lane & 15) >> 2);
    const int v_sw = attn_v_swizzle<E>(v_key);        // unchanged by the multiples of 8 that are added to the key
    const int v_chunk = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
    const int v_src = VT + v_key * ROW + (lane & 1) * 8;

    const int e_begin = SEQ ? 0 : p.row_ptr[br];
    const int n_blk = (SEQ ? (seq_len + BW - 1) / BW : p.row_ptr[br + 1]) - e_begin;
    const bool idle = SEQ && row0 >= seq_len;   // this wavefront only brings tiles: its rows are zeros
    int bc_vec = 0;
    if constexpr (!SEQ) {
        if (lane < n_blk) bc_vec = p.bcsr_idx[e_begin + lane] & 0xffff;
    }
    auto col_at = [&](int i) {
        if constexpr (SEQ) return i;
        else return i < 64 ? __builtin_amdgcn_readlane(bc_vec, i) : __builtin_amdgcn_readfirstlane(p.bcsr_idx[e_begin + i] & 0xffff);
    };
    auto issue = [&](int i) {
        const int key0 = col_at(i) * BW;
        const uint32_t to = lds0 + (i & 1) * TILE;
        // the last tile of a sequence may reach past the tensor: rows from there on are read from its last row
        const int last = SEQ ? p.Ns - 1 - key0 : BW;
#pragma unroll
        for (int i2 = 0; i2 < NV; ++i2) {
            const int row = st_row + i2 * RSTEP;
            const int from = (SEQ && row > last ? last : row) * ROW;
            lds_direct_load16_at(Kg + (int64_t)key0 * E, from + (st_slot ^ attn_k_swizzle<E>(row)) * 16, to + i2 * NT * 16);
            lds_direct_load16_at(Vg + (int64_t)key0 * E, from + (st_slot ^ attn_v_swizzle<E>(row)) * 16, to + VT + i2 * NT * 16);
        }
    };
    unsigned live[KT][4] = {};
    auto fetch_mask = [&](int i) {
        const uint8_t* m = p.mask + (int64_t)qrow * p.Ns + col_at(i) * BW + h2 * 4;
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int a = 0; a < 4; ++a) live[kt][a] = *reinterpret_cast<const uint32_t*>(m + kt * 32 + a * 8);
    };
    if (n_blk > 0) {
        issue(0);
        if constexpr (HAS_MASK) fetch_mask(0);
    }
    for (int i = 0; i < n_blk; ++i) {
        char* buf = smem + (i & 1) * TILE;
        __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wavefront's chunks of tile i are in LDS
        asm volatile("" ::: "memory");
        __syncthreads();                      // everybody's are, and tile i - 1 is consumed
        if (i + 1 < n_blk) issue(i + 1);
        const int left = SEQ ? seq_len - i * BW : BW;   // live keys of this tile
        if (SEQ && left < BW) {
            // value rows past the length: their probabilities are 0, and 0 times what padding may hold is not
            for (int v = threadIdx.x; v < (BW - left) * VPR; v += NT)
                *reinterpret_cast<u32x4*>(buf + VT + left * ROW + v * 16) = u32x4{0u, 0u, 0u, 0u};
            __syncthreads();
        }

        if (idle) continue;
        // ---- S^T tiles: 32 keys x this wave's 32 queries ------------------------------------
        f32x16 s[KT];
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
#pragma unroll
            for (int j = 0; j < 16; ++j) s[kt][j] = 0.f;
#pragma unroll
            for (int c = 0; c < EC; ++c) {
                const Frag kf = *reinterpret_cast<const Frag*>(buf + k_src + kt * 32 * ROW + (((c * 2 + h2) ^ k_sw) * 16));
                s[kt] = MmaW<T>::mma(kf, qf[c], s[kt]);
            }
        }
        if constexpr (HAS_MASK) {
            unsigned all = 0x01010101u;
#pragma unroll
            for (int kt = 0; kt < KT; ++kt) all &= live[kt][0] & live[kt][1] & live[kt][2] & live[kt][3];
            if (__builtin_amdgcn_ballot_w64(all != 0x01010101u) != 0) {
#pragma unroll
                for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                    for (int j = 0; j < 16; ++j) s[kt][j] = ((live[kt][j >> 2] >> (8 * (j & 3))) & 0xffu) ? s[kt][j] : DEAD;
            }
            if (i + 1 < n_blk) fetch_mask(i + 1);
        }
        if (SEQ && left < BW) {
#pragma unroll
            for (int kt = 0; kt < KT; ++kt)
#pragma unroll
                for (int j = 0; j < 16; ++j) s[kt][j] = kt * 32 + 8 * (j >> 2) + 4 * h2 + (j & 3) < left ? s[kt][j] : DEAD;
        }
        // three-way maxima throughout: two lanes of two chains per tile, joined with what is left over
        float top[KT * 2];
#pragma unroll
        for (int c = 0; c < KT * 2; ++c) {
            const f32x16& t = s[c >> 1];
            const int j = 8 * (c & 1);
            top[c] = max3f(max3f(max3f(t[j], t[j + 1], t[j + 2]), t[j + 3], t[j + 4]), t[j + 5], t[j + 6]);
        }
        float tmax = max3f(top[0], top[1], s[0][7]);
#pragma unroll
        for (int kt = 1; kt < KT; ++kt) tmax = max3f(max3f(tmax, top[2 * kt], top[2 * kt + 1]), s[kt - 1][15], s[kt][7]);
        tmax = xor32_max(fmaxf(tmax, s[KT - 1][15]));
        const bool any_live = tmax > -1e29f;
        if (__builtin_amdgcn_ballot_w64(any_live && (fresh || (tmax - m_run) * c2 > RESCALE_LOG2)) != 0) {
            const float m_new = any_live ? (fresh ? tmax : fmaxf(m_run, tmax)) : m_run;
            const float alpha = fresh ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * c2);   // nothing summed yet while fresh
            m_run = m_new;
            lacc *= alpha;
#pragma unroll
            for (int t = 0; t < ET; ++t) oacc[t] *= alpha;
        }
        fresh = fresh && !any_live;
        const float mc = -m_run * c2;
        Frag pf[KS];
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            f32x8 pv;
#pragma unroll
            for (int j = 0; j < 8; ++j) pv[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u >> 1][8 * (u & 1) + j], c2, mc));
            pf[u] = AttnPack<T>::pack(pv);
            lacc = AttnPack<T>::add_lane8(pf[u], lacc);
        }
        // ---- O^T[e][query] += V^T P^T ------------------------------------------------------
#pragma unroll
        for (int u = 0; u < KS; ++u) {
#pragma unroll
            for (int t = 0; t < ET; ++t) {
                const char* at = buf + v_src + u * 16 * ROW + ((t * 4 + v_chunk) ^ v_sw) * 16;
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at));
                const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 8 * ROW));
                const s16x8 both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                oacc[t] = MmaW<T>::mma(__builtin_bit_cast(Frag, both), pf[u], oacc[t]);
            }
        }
    }

    // lane holds O^T[e = t*32 + 8a + 4*h2 + q][query l32]; rows with no live entry give 0
    const float l_run = xor32_sum(lacc[0]);
    const float inv_l = l_run > 0.f ? 1.f / l_run : 0.f;
    constexpr int PP = ROW + 16;
    __syncthreads();   // the K / V tiles are dead: their space carries the output tiles
    char* tile = smem + wave * (32 * PP);
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f32x8 vals = {};
#pragma unroll
            for (int q = 0; q < 4; ++q) vals[q] = SEQ && qrow >= seq_len ? 0.f : oacc[t][4 * a + q] * inv_l;
            const uint64_t piece = __builtin_bit_cast(u64x2, AttnPack<T>::pack(vals))[0];
            *reinterpret_cast<uint64_t*>(tile + l32 * PP + (t * 32 + a * 8 + h2 * 4) * 2) = piece;
        }
    if (rows_exist) {
        char* dst = reinterpret_cast<char*>(O + (int64_t)row0 * E);
#pragma unroll
        for (int i = 0; i < 32 * VPR / 64; ++i) {
            const int c = i * 64 + lane;
            __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(tile + (c / VPR) * PP + (c % VPR) * 16),
                                        reinterpret_cast<u32x4*>(dst + c * 16));
        }
    }
}

template <typename T, int BW, int E, int WAVES>
static int launch_attention_wide_inst(const AttnParams& p, int batch, hipStream_t st) {
    constexpr size_t smem = attn_wide_smem(BW, E, WAVES);
    const int nbr = p.Nt / p.BH;
    const int64_t groups = ((int64_t)batch + 7) / 8 * 8 * nbr;
    if (groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)groups);
    if (p.mask) {
        SPX_GRANT_LDS((attention_wide_kernel<T, BW, E, WAVES, true>), smem, "attention_wide_kernel");
        hipLaunchKernelGGL((attention_wide_kernel<T, BW, E, WAVES, true>), dim3((unsigned)groups), dim3(64 * WAVES), smem, st, p, nbr, batch);
    } else {
        SPX_GRANT_LDS((attention_wide_kernel<T, BW, E, WAVES, false>), smem, "attention_wide_kernel");
        hipLaunchKernelGGL((attention_wide_kernel<T, BW, E, WAVES, false>), dim3((unsigned)groups), dim3(64 * WAVES), smem, st, p, nbr, batch);
    }
    SPX_LAUNCH_CHECK("attention_wide_kernel");
    return 0;
}

// Sequence-length mode: key tiles of 64, 128 queries per workgroup, any N that is a multiple of 32.
// (64 queries per workgroup: 63 -> 84 us at 32 x 12 x 1024 x 64 fp16, the L1s fetch every tile twice as
// often; 256 queries: 72 us, eight wavefronts meet at a barrier.)
template <typename T, int E>
static int launch_attention_wide_seq_inst(const AttnParams& p, int batch, hipStream_t st) {
    constexpr int WAVES = 4;
    constexpr size_t smem = attn_wide_smem(64, E, WAVES);
    const int nbr = (p.Nt + 32 * WAVES - 1) / (32 * WAVES);
    const int64_t groups = ((int64_t)batch + 7) / 8 * 8 * nbr;
    if (groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)groups);
    SPX_GRANT_LDS((attention_wide_kernel<T, 64, E, WAVES, false, true>), smem, "attention_wide_kernel");
    hipLaunchKernelGGL((attention_wide_kernel<T, 64, E, WAVES, false, true>), dim3((unsigned)groups), dim3(64 * WAVES), smem, st, p, nbr, batch);
    SPX_LAUNCH_CHECK("attention_wide_kernel (sequence lengths)");
    return 0;
}

template <typename T>
static int launch_attention_wide_seq_typed(const AttnParams& p, int batch, int E, hipStream_t st) {
    if (E == 64) return launch_attention_wide_seq_inst<T, 64>(p, batch, st);
    if (E == 128) return launch_attention_wide_seq_inst<T, 128>(p, batch, st);
    return fail(SPX_E_CONFIG, "the wide sequence-length kernel takes head dims 64 / 128 (got %d)", E);
}

// The wide-MFMA kernel covers query blocks of 32 / 64 / 128 (one wavefront per 32 queries),
// key blocks of 32 / 64 / 128 and head dimensions 64 / 128, as long as a thread stages one
// to eight 16-byte vectors of each tile: the combinations listed here.
template <typename T>
static int launch_attention_wide_typed(const AttnParams& p, int batch, int BW, int E, hipStream_t st) {
#define SPX_ATTN3_CASE(bh, bw, e) \
    if (p.BH == bh && BW == bw && E == e) return launch_attention_wide_inst<T, bw, e, bh / 32>(p, batch, st);
    SPX_ATTN3_CASE(32, 32, 64) SPX_ATTN3_CASE(32, 64, 64) SPX_ATTN3_CASE(32, 32, 128)
    SPX_ATTN3_CASE(64, 32, 64) SPX_ATTN3_CASE(64, 64, 64) SPX_ATTN3_CASE(64, 128, 64)
    SPX_ATTN3_CASE(64, 32, 128) SPX_ATTN3_CASE(64, 64, 128)
    SPX_ATTN3_CASE(128, 32, 64) SPX_ATTN3_CASE(128, 64, 64) SPX_ATTN3_CASE(128, 128, 64)
    SPX_ATTN3_CASE(128, 32, 128) SPX_ATTN3_CASE(128, 64, 128) SPX_ATTN3_CASE(128, 128, 128)
#undef SPX_ATTN3_CASE
    return fail(SPX_E_CONFIG, "the wide-MFMA attention kernel does not cover blocks (%d,%d) with head dim %d", p.BH, BW, E);
}

int launch_attention_wide(int dtype, const AttnParams& p, int batch, int BW, int E, hipStream_t st) {
    if (dtype == SPX_F16) return launch_attention_wide_typed<_Float16>(p, batch, BW, E, st);
    return launch_attention_wide_typed<bf16_t>(p, batch, BW, E, st);
}

int launch_attention_wide_seq(int dtype, const AttnParams& p, int batch, int E, hipStream_t st) {
    if (dtype == SPX_F16) return launch_attention_wide_seq_typed<_Float16>(p, batch, E, st);
    return launch_attention_wide_seq_typed<bf16_t>(p, batch, E, st);
}

}  // namespace spx
