// Fused block-sparse and sequence-length attention forward with 32 queries per wavefront.
#include <type_traits>
#include "attention.hpp"

namespace spx {

// ---- wide variant: 32 queries per wavefront, 32 x 32 x 16 MFMAs ---------------------------
//   S^T[key][query] (A = K rows from LDS, B = Q from registers): lane l holds, for query
//   l % 32, the keys 8a + 4(l / 32) + b (a, b = 0..3) of a 32-key tile in s[4a + b];
//   O^T[e][query] += V^T P^T in 16-key steps: k-slot i of half h = l / 32 is key
//   16u + 8(i / 4) + 4h + i % 4, which is s[8u + i] - the probabilities go
//   from the accumulator straight into the B operand - and for V^T two LDS transpose reads
//   (keys 16u + 4h .. +3 and 16u + 8 + 4h .. +3 of column e).
//   Row sums of the rounded probabilities: 4 x 4 x 4 MFMAs against ones.  Their B operand is a
//   column per lane with its four k in the lane's registers, so every lane sums its own values
//   (two lanes per query, joined at the end) and no query meets another one's NaN.
// K and V tiles of 32 KT keys go global -> LDS directly, two stages, one barrier per stage; the slots of
// the ring are constants (the walk is unrolled), so LDS addresses cost no arithmetic.  Over an index KT is 1: with 16 KB of
// LDS to two wavefronts sixteen of them share a CU, which is worth more than the barrier of every 64 keys (96 x 4096 x 64,
// 392 blocks of 64 x 64: bf16 62.8 us against 70.4 with tiles of 64 keys, fp16 65.9 against 74.2).  Over sequence lengths
// KT is 2: four wavefronts meet at a barrier (16.7 us against 18.5 at 4 x 12 x 1024, level at 32 x 12 x 1024); 4 where two
// wavefronts share the keys of 32 queries, the head dim is 64 and all workgroups are on the chip at once.
//
// What bounds it.  Per wavefront and 32 x 32 scores: 8 MFMAs of 32 clocks and 4 of 8, 16 exponentials of 8, about 45 other
// vector instructions of 3 - 4 clocks; in the steady part of a launch a SIMD takes 480 clocks for them, i.e. MFMAs and
// vector instructions overlap by a third.  Over an index 40 % of the launch is beginning and end: the chain index -> tiles
// of every workgroup (4000 clocks) and a last generation that does not fill the chip; all forms tried (wavefronts of 64 queries
// without any barrier, 2 - 4 stages, scores one tile ahead of the softmax) end between 63 and 76 us, and without tile loads
// at 60.  32 x 12 x 1024 x 64 with mixed lengths 64 -> 56 us (34 GFLOP), head dim 128 at 32 x 12 x 512 43.5 -> 35.7.
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
    int first = 0, t = slot;
    if (entries > 64) {
        const int per_group = 8 * p.heads * nbr;   // 64 entries: 64 * heads / 8 pairs on an XCD
        first = slot / per_group * 64;
        t = slot % per_group;
    }
    const int n = entries - first < 64 ? entries - first : 64;
    const int lane = lane_id();
    int mine = -1;
    if (lane < n) {
        mine = p.seqlens[first + lane];
        mine = mine < 0 ? 0 : mine > p.Ns ? p.Ns : mine;
    }
    // rank of this lane's entry by its tiles of 32 keys: one ballot per bit, from the highest (with a comparison with every
    // other entry and scratch for what the end needs, 16.0 -> 14.2 us at 19 x 8 x 576 bf16)
    const uint64_t all = n == 64 ? ~(uint64_t)0 : ((uint64_t)1 << n) - 1;
    const int key = (mine + 31) >> 5;
    uint64_t equal = all;   // entries like mine in the bits so far
    int rank = 0;           // and the ones that are ahead
    for (int bit = 31 - __builtin_clz(((p.Ns + 31) >> 5) | 1); bit >= 0; --bit) {
        const uint64_t ones = __builtin_amdgcn_ballot_w64((key >> bit) & 1) & all;
        const bool one = (key >> bit) & 1;
        rank += one ? 0 : __popcll(equal & ones);
        equal &= one ? ones : ~ones;
    }
    rank += __popcll(equal & (((uint64_t)1 << lane) - 1));
    if (lane >= n) rank = lane;
    // from here on lane r holds the r-th longest entry
    const int both = __builtin_amdgcn_ds_permute(rank * 4, (mine << 6) | lane);
    const int len = both >> 6, id = both & 63;
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
    // t / of, one comparison a lane for the first 64 pairs
    const int k = t < 64 * of ? __popcll(__builtin_amdgcn_ballot_w64(lane * of <= t)) - 1 : t / of;
    const int pair = 8 * (__builtin_amdgcn_readlane(lo, r) + k) + xcd;
    w.b = (int64_t)(first + __builtin_amdgcn_readlane(id, r)) * p.heads + pair - (first + r) * p.heads;
    w.br = __builtin_amdgcn_readlane(skip, r) + t - k * of;
    w.len = __builtin_amdgcn_readlane(len, r);
    return true;
}

constexpr int kWideStages = 2;
template <int E, int KT, int WAVES, bool HAS_MASK, int SPLIT = 1> struct WideLds {
    static constexpr int V = KT * AttnTile<E>::BYTES;
    static constexpr int MASK = 2 * V;                  // 32 x 32 bytes per wavefront
    static constexpr int STAGE = MASK + (HAS_MASK ? WAVES * 1024 : 0);
    // in the same space afterwards: what the wavefronts but those of the first share of the keys hold, and the output rows
    static constexpr int PART = E / 32 * 4096 + 512, OUT = (WAVES - WAVES / SPLIT) * PART;
    static constexpr int END = OUT + WAVES / SPLIT * 32 * (E * 2 + 16);
    static constexpr int TOTAL = kWideStages * STAGE > END ? kWideStages * STAGE : END;
};

// SPLIT: wavefronts to 32 queries; each takes KT / SPLIT of a stage's tiles, and the first one adds up what they hold.
template <typename T, int E, int KT, int WAVES, bool HAS_MASK, bool SEQ, int SPLIT>
__global__ __launch_bounds__(64 * WAVES, SPLIT > 1 ? 2 : E == 64 ? 4 : KT == 1 ? 3 : 2) void attention_wide_kernel(AttnParams p, int nbr, int log_sub, int batch) {
    static_assert(KT == 1 || (SEQ && !HAS_MASK), "an index is walked in tiles of 32 keys, and sequence-length mode has no mask bytes");
    static_assert(SPLIT == 1 || SEQ, "the keys of an index are not shared out");
    typedef AttnTile<E> Tile;
    typedef WideLds<E, KT, WAVES, HAS_MASK, SPLIT> Lds;
    constexpr int EC = Tile::EC, ET = Tile::ET, NB = kWideStages;
    constexpr int LPT = 2 * Tile::LOADS / WAVES;   // loads of a wavefront and 32 keys
    constexpr int QW = WAVES / SPLIT, KW = KT / SPLIT;   // wavefronts with queries of their own; tiles of a wavefront and stage
    constexpr int ROWS = 32 * QW, KEYS = 32 * KT;
    typedef typename MmaW<T>::frag Frag;
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    extern __shared__ __align__(16) char smem[];

    // workgroup L runs on XCD L % 8: give each XCD whole batch*head entries
    const int L = blockIdx.x;
    const int slot = L >> 3;
    int64_t b;
    int br, seq_len = 0;
    if constexpr (SEQ) {
        SeqWork w;
        // the first four workgroups of each CU go there and back along the list, which evens their sums out (the dispatcher
        // deals the 32 CUs of an XCD one after the other): 22 x 16 x 640 bf16 23.9 -> 23.5 us, 6 x 8 x 1696 29.3 -> 27.9
        const bool back = (slot & 32) != 0 && slot < 128 && (slot | 31) < (int)(gridDim.x >> 3);
        if (!seqlen_work<ROWS>(p, batch / p.heads, nbr, back ? slot ^ 31 : slot, L & 7, w)) return;
        b = w.b;
        br = w.br;
        seq_len = w.len;
        if (br * ROWS >= seq_len) {   // rows of zeros
            const int rows = p.Nt - br * ROWS < ROWS ? p.Nt - br * ROWS : ROWS;
            char* dst = reinterpret_cast<char*>(reinterpret_cast<T*>(p.out) + (b * p.Nt + br * ROWS) * E);
            for (int v = threadIdx.x; v < rows * (E / 8); v += 64 * WAVES)
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
    const Tile tile(lane);
    const int l32 = tile.l32, h2 = tile.h2;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)smem;

    const int qw = SPLIT > 1 ? wave % QW : wave, kw = SPLIT > 1 ? wave / QW : 0;   // its queries, its share of the keys
    const int row0 = br * ROWS + qw * 32;         // first query of this wavefront
    // sequence lengths: Nt is a multiple of 32, so a wavefront is inside or outside; one whose rows are all past the
    // length only brings tiles
    const bool rows_exist = !SEQ || row0 < p.Nt, idle = SEQ && row0 >= seq_len;
    const T* Kg = reinterpret_cast<const T*>(p.k) + b * (int64_t)p.Ns * E;
    const T* Vg = reinterpret_cast<const T*>(p.v) + b * (int64_t)p.Ns * E;
    Frag qf[EC];
#pragma unroll
    for (int c = 0; c < EC; ++c)
        qf[c] = *reinterpret_cast<const Frag*>(reinterpret_cast<const T*>(p.q) + (b * p.Nt + (rows_exist ? row0 + l32 : 0)) * E + c * 16 + h2 * 8);

    const int e_begin = SEQ ? 0 : p.row_ptr[br];
    const int n_ent = SEQ ? 0 : p.row_ptr[br + 1] - e_begin;
    const int n = SEQ ? (seq_len + KEYS - 1) / KEYS : n_ent << log_sub;
    int bc_vec = 0;
    if constexpr (!SEQ) {
        if (lane < n_ent) bc_vec = p.bcsr_idx[e_begin + lane] & 0xffff;
    }
    auto key0_at = [&](int i) {
        const int e = i >> log_sub;
        const int col = e < 64 ? __builtin_amdgcn_readlane(bc_vec, e) : __builtin_amdgcn_readfirstlane(p.bcsr_idx[e_begin + e] & 0xffff);
        return ((col << log_sub) + (i & ((1 << log_sub) - 1))) * 32;
    };
    auto issue = [&](int i, int at) {
#pragma unroll
        for (int kt = 0; kt < KT; ++kt) {
            int key0 = SEQ ? i * KEYS + kt * 32 : key0_at(i);
            if (kt > 0 && key0 >= p.Ns) key0 = p.Ns - 32;   // past the tensor and the length: any rows
            const uint32_t to = lds0 + at + kt * Tile::BYTES;
            if constexpr (WAVES == 1) {
                tile.template request<LPT / 2>(Kg + (int64_t)key0 * E, 0, to);
                tile.template request<LPT / 2>(Vg + (int64_t)key0 * E, 0, to + Lds::V);
            } else {   // the first half of the wavefronts brings K, the others V
                const T* from = wave < WAVES / 2 ? Kg : Vg;
                tile.template request<LPT>(from + (int64_t)key0 * E, (wave & (WAVES / 2 - 1)) * LPT, to + (wave < WAVES / 2 ? 0 : Lds::V));
            }
            if constexpr (HAS_MASK)
                lds_direct_load16_at(p.mask + (int64_t)row0 * p.Ns + key0, (lane >> 1) * p.Ns + (lane & 1) * 16, to + Lds::MASK + wave * 1024);
        }
    };
    if (n > 0) issue(0, 0);

    f32x16 oacc[ET];
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) oacc[t][j] = 0.f;
    f32x4 lacc = f32x4{0.f, 0.f, 0.f, 0.f};
    // m: reference point of this lane's query; set to the row maximum by the first tile with a
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

    auto step = [&](int i, auto slot) {
        constexpr int at = slot * Lds::STAGE, fill = (slot + NB - 1) % NB * Lds::STAGE;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's part of stage i is in LDS
        __syncthreads();                                   // everybody's is, and stage i - 1 has been read
        if (i + 1 < n) issue(i + 1, fill);
        const int left = SEQ ? seq_len - i * KEYS : KEYS;   // live keys of this stage
        if (SEQ && left < KEYS) {
            // value rows past the length: their probabilities are 0, and 0 times what padding may hold is not
            for (int v = threadIdx.x; v < (KEYS - left) * (E / 8); v += 64 * WAVES)
                *reinterpret_cast<u32x4*>(smem + at + Lds::V + left * Tile::ROW + v * 16) = u32x4{0u, 0u, 0u, 0u};
            __syncthreads();
        }
        const int mine = left - kw * KW * 32;               // of the ones that are this wavefront's
        if (idle || (SPLIT > 1 && mine <= 0)) return;
        const char* ks = smem + at + kw * KW * Tile::BYTES;
        const char* vs = ks + Lds::V;
        // ---- S^T: 32 keys x this wavefront's 32 queries at a time ----------------------------
        f32x16 s[KW];
#pragma unroll
        for (int kt = 0; kt < KW; ++kt) {
#pragma unroll
            for (int j = 0; j < 16; ++j) s[kt][j] = 0.f;
#pragma unroll
            for (int c = 0; c < EC; ++c) s[kt] = MmaW<T>::mma(tile.template row_frag<Frag>(ks + kt * Tile::BYTES, c), qf[c], s[kt]);
        }
        if constexpr (HAS_MASK) {
            unsigned live[4];
            const char* m = ks + Lds::MASK + wave * 1024 + l32 * 32 + h2 * 4;
#pragma unroll
            for (int a = 0; a < 4; ++a) live[a] = *reinterpret_cast<const uint32_t*>(m + a * 8);
            if (__builtin_amdgcn_ballot_w64((live[0] & live[1] & live[2] & live[3]) != 0x01010101u) != 0) {
#pragma unroll
                for (int j = 0; j < 16; ++j) s[0][j] = ((live[j >> 2] >> (8 * (j & 3))) & 0xffu) ? s[0][j] : DEAD;
            }
        }
        if (SEQ && mine < 32 * KW) {
#pragma unroll
            for (int kt = 0; kt < KW; ++kt)
#pragma unroll
                for (int j = 0; j < 16; ++j) s[kt][j] = kt * 32 + 8 * (j >> 2) + 4 * h2 + (j & 3) < mine ? s[kt][j] : DEAD;
        }
        // three-way maxima, two chains to 32 keys
        float tmax = DEAD;
#pragma unroll
        for (int kt = 0; kt < KW; ++kt) {
            const f32x16& x = s[kt];
            const float a0 = max3f(max3f(max3f(x[0], x[1], x[2]), x[3], x[4]), x[5], x[6]);
            const float a1 = max3f(max3f(max3f(x[8], x[9], x[10]), x[11], x[12]), x[13], x[14]);
            tmax = max3f(max3f(tmax, a0, a1), x[7], x[15]);
        }
        tmax = xor32_max(tmax);
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
        Frag pf[KW][2];
#pragma unroll
        for (int kt = 0; kt < KW; ++kt)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                f32x8 pv;
#pragma unroll
                for (int j = 0; j < 8; ++j) pv[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][8 * u + j], c2, mc));
                pf[kt][u] = AttnPack<T>::pack(pv);
                lacc = AttnPack<T>::add_lane8(pf[kt][u], lacc);
            }
        // ---- O^T[e][query] += V^T P^T ------------------------------------------------------
#pragma unroll
        for (int kt = 0; kt < KW; ++kt)
#pragma unroll
            for (int u = 0; u < 2; ++u)
#pragma unroll
                for (int t = 0; t < ET; ++t)
                    oacc[t] = MmaW<T>::mma(tile.template tr_frag<Frag>(vs + kt * Tile::BYTES, t, u), pf[kt][u], oacc[t]);
    };
    for (int i = 0; i < n; i += NB) {
        step(i, std::integral_constant<int, 0>());
        if (i + 1 < n) step(i + 1, std::integral_constant<int, 1>());
    }

    // lane holds O^T[e = t*32 + 8a + 4*h2 + q][query l32]; rows with no live entry give 0
    float l_run = xor32_sum(lacc[0]);
    if constexpr (SPLIT > 1) {
        __syncthreads();   // the K / V tiles are dead
        if (kw > 0) {
            char* to = smem + (wave - QW) * Lds::PART;
#pragma unroll
            for (int t = 0; t < ET; ++t)
#pragma unroll
                for (int a = 0; a < 4; ++a)
                    *reinterpret_cast<f32x4*>(to + ((t * 4 + a) * 64 + lane) * 16) =
                        f32x4{oacc[t][4 * a], oacc[t][4 * a + 1], oacc[t][4 * a + 2], oacc[t][4 * a + 3]};
            reinterpret_cast<float*>(to + ET * 4096)[lane] = h2 ? l_run : m_run;
        }
        __syncthreads();
        if (kw > 0) return;
        // their reference points differ; one that has seen no live key has a sum of 0 and none (a NaN counts as a sum)
        float m[SPLIT], l[SPLIT];
        m[0] = m_run;
        l[0] = l_run;
#pragma unroll
        for (int g = 1; g < SPLIT; ++g) {
            const float* from = reinterpret_cast<const float*>(smem + ((g - 1) * QW + qw) * Lds::PART + ET * 4096);
            m[g] = from[l32];
            l[g] = from[32 + l32];
        }
        float top = DEAD;
#pragma unroll
        for (int g = 0; g < SPLIT; ++g) top = l[g] == 0.f ? top : fmaxf(top, m[g]);
        l_run = 0.f;
#pragma unroll
        for (int g = 0; g < SPLIT; ++g) {
            const float weight = l[g] == 0.f ? 0.f : __builtin_amdgcn_exp2f((m[g] - top) * c2);
            l_run = __builtin_fmaf(weight, l[g], l_run);
            const char* from = smem + ((g - 1) * QW + qw) * Lds::PART;
#pragma unroll
            for (int t = 0; t < ET; ++t)
#pragma unroll
                for (int a = 0; a < 4; ++a) {
                    f32x4 part;
                    if (g > 0) part = *reinterpret_cast<const f32x4*>(from + ((t * 4 + a) * 64 + lane) * 16);
#pragma unroll
                    for (int x = 0; x < 4; ++x)
                        oacc[t][4 * a + x] = g == 0 ? oacc[t][4 * a + x] * weight : __builtin_fmaf(weight, part[x], oacc[t][4 * a + x]);
                }
        }
    }
    int out_lane = lane;   // made anew: what the stores derive from the lane would be kept through the walk, in scratch
    if constexpr (SEQ) asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(out_lane));
    const bool past = SEQ && row0 + (out_lane & 31) >= seq_len;
    const float inv_l = l_run > 0.f ? 1.f / l_run : 0.f;
    if (!SEQ && p.row_lse && h2 == 0)
        p.row_lse[b * p.Nt + row0 + l32] = l_run > 0.f ? __builtin_fmaf(m_run, c2, __builtin_amdgcn_logf(l_run)) : __builtin_inff();
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) oacc[t][j] = past ? 0.f : oacc[t][j] * inv_l;
    if constexpr (SPLIT == 1) __syncthreads();   // the K / V tiles are dead: their space carries the output rows
    if (rows_exist)
        store_rows32<T, E>(smem + Lds::OUT + qw * (32 * (E * 2 + 16)), reinterpret_cast<T*>(p.out) + (b * p.Nt + row0) * E, oacc, out_lane);
}

template <typename T, int E, int KT, int WAVES, bool HAS_MASK, bool SEQ, int SPLIT = 1>
static int launch_attention_wide_inst(const AttnParams& p, int nbr, int batch, int BW, hipStream_t st) {
    constexpr int smem = WideLds<E, KT, WAVES, HAS_MASK, SPLIT>::TOTAL;
    const int64_t groups = ((int64_t)batch + 7) / 8 * 8 * nbr;
    if (groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)groups);
    SPX_GRANT_LDS((attention_wide_kernel<T, E, KT, WAVES, HAS_MASK, SEQ, SPLIT>), smem, "attention_wide_kernel");
    hipLaunchKernelGGL((attention_wide_kernel<T, E, KT, WAVES, HAS_MASK, SEQ, SPLIT>), dim3((unsigned)groups), dim3(64 * WAVES), smem, st, p, nbr, ilog2(BW / 32), batch);
    SPX_LAUNCH_CHECK("attention_wide_kernel");
    return 0;
}

// Sequence-length mode, any N that is a multiple of 32.  With enough work 128 queries per workgroup.
// (64 queries per workgroup: 63 -> 84 us at 32 x 12 x 1024 x 64 fp16, the L1s fetch every tile twice as
// often; 256 queries: 72 us, eight wavefronts meet at a barrier.)  Below that a launch is as long as the walk over the
// longest sequence: 64 queries, and two wavefronts to 32 of them that share the keys out, stages of 128 keys for as long as
// all workgroups are on the chip at once (64 KB of LDS each, head dim 64).  fp16 us, 128 queries / shared keys and stages of
// 64 / and of 128:
//   head dim 64   3 x 16 x 640 12.3 / 9.7 / 9.4, 1 x 16 x 2048 18.6 / 13.5 / 11.9, 6 x 8 x 1024 18.0 / 13.4 / 12.6,
//                 5 x 12 x 1152 19.8 / 17.6 / 19.3, 8 x 12 x 1024 18.9 / 17.6 / 22.9, 9 x 16 x 1024 23.4 / 27.3 / 30.1
//                 (up to 1024 workgroups of 128 queries where N is 768 and more: 8 x 16 x 1024 22.3 / 20.8, 4 x 16 x 1984 33.6 / 33.0,
//                 but 32 x 16 x 256 11.1 / 13.2)
//   head dim 128  2 x 12 x 1024 19.8 / 15.0, 8 x 8 x 768 20.5 / 16.7, 4 x 16 x 1024 23.4 / 20.8, 11 x 16 x 448 16.6 / 21.6
static bool seqlen_shares_keys(int64_t entries, int N, int E) {
    return entries * ((N + 127) / 128) <= (E == 64 ? (N >= 768 ? 1024 : 768) : 512);
}

// Whether this kernel takes the call and not the 16-query one, whose wavefronts start sooner: N from 192 on; with few
// workgroups long sequences or 384 of 64 queries.  fp16 us, 16-query kernel / shared keys: 2 x 12 x 512 x 64 6.8 / 7.0,
// 4 x 12 x 512 9.3 / 8.1, 8 x 12 x 256 6.7 / 6.4, 6 x 12 x 320 6.6 / 7.3, 1 x 8 x 640 6.0 / 7.0, 1 x 12 x 768 6.8 / 6.9,
// 1 x 16 x 1024 8.4 / 8.0, 2 x 8 x 2048 19.5 / 15.5; head dim 128 2 x 16 x 256 6.5 / 7.6, 8 x 16 x 256 9.7 / 9.6,
// 14 x 12 x 192 8.3 / 9.5, 1 x 8 x 800 10.5 / 10.9, 1 x 8 x 1024 12.0 / 11.7.  16-query kernel / 128 queries: 32 x 16 x 192 x 64 9.6 / 9.0, 24 x 12 x 160 x
// 64 6.6 / 6.9, 20 x 16 x 192 x 128 11.6 / 11.2.
bool attention_wide_seq_wins(int64_t entries, int N, int E) {
    if (N < 192) return false;
    if (!seqlen_shares_keys(entries, N, E)) return true;
    return N >= (E == 64 ? 768 : 896) || (entries * ((N + 63) / 64) >= 384 && N >= (E == 64 ? 192 : 256));
}

template <typename T>
static int launch_attention_wide_seq_typed(const AttnParams& p, int batch, int E, hipStream_t st) {
    if (E != 64 && E != 128) return fail(SPX_E_CONFIG, "the wide sequence-length kernel takes head dims 64 / 128 (got %d)", E);
    if (seqlen_shares_keys(batch, p.Nt, E)) {
        const int nbr = (p.Nt + 63) / 64;
        if (E == 128) return launch_attention_wide_inst<T, 128, 2, 4, false, true, 2>(p, nbr, batch, 32, st);
        return (int64_t)batch * nbr <= 512 ? launch_attention_wide_inst<T, 64, 4, 4, false, true, 2>(p, nbr, batch, 32, st)
                                           : launch_attention_wide_inst<T, 64, 2, 4, false, true, 2>(p, nbr, batch, 32, st);
    }
    const int nbr = (p.Nt + 127) / 128;
    return E == 64 ? launch_attention_wide_inst<T, 64, 2, 4, false, true>(p, nbr, batch, 32, st)
                   : launch_attention_wide_inst<T, 128, 2, 4, false, true>(p, nbr, batch, 32, st);
}

template <typename T>
static int launch_attention_wide_typed(const AttnParams& p, int batch, int BW, int E, hipStream_t st) {
    if (!attention_wide_supported(p.BH, BW, E))
        return fail(SPX_E_CONFIG, "the wide-MFMA attention kernel does not cover blocks (%d,%d) with head dim %d", p.BH, BW, E);
    const int nbr = p.Nt / p.BH;
#define SPX_ATTN3_CASE(bh, e)                                                                           \
    if (p.BH == bh && E == e)                                                                           \
        return p.mask ? launch_attention_wide_inst<T, e, 1, bh / 32, true, false>(p, nbr, batch, BW, st)   \
                      : launch_attention_wide_inst<T, e, 1, bh / 32, false, false>(p, nbr, batch, BW, st);
    SPX_ATTN3_CASE(32, 64) SPX_ATTN3_CASE(64, 64) SPX_ATTN3_CASE(128, 64)
    SPX_ATTN3_CASE(32, 128) SPX_ATTN3_CASE(64, 128) SPX_ATTN3_CASE(128, 128)
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
