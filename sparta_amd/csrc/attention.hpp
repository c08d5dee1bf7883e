// What the fused attention translation units share: launch parameters, the packing of
// probabilities into MFMA operands, and the launchers of the wide kernel.
#pragma once
#include "common.hpp"
#include "mma.hpp"

namespace spx {

struct AttnParams {
    const void* q;
    const void* k;
    const void* v;
    void* out;
    const int32_t* row_ptr;
    const int32_t* bcsr_idx;
    const uint8_t* mask;  // [Nt, Ns] or NULL
    int mask_blocks;      // wide backward kernels: 1: mask holds the live blocks in BCSR order, [BH, BW] each
    float inv_t;
    int Nt, Ns, BH;
    void* probs;          // training kernels: compressed probabilities, block e at e * BH * BW
    int64_t probs_batch;  // elements between batch entries of probs (and of grad_scores)
    const void* grad_out; // backward kernel: gradient of the output
    void* grad_scores;    // backward kernel: compressed gradient of the scores (layout of probs)
    void* grad_q;         // backward kernel: gradient of the queries
    float* row_dot;       // backward kernels: D[b, i] / T = sum_e grad_out o out / T per query
    const int32_t* col_ptr;   // column-side backward kernel: BCSC index
    const void* bcsc_idx;
    int bcsc_wide;        // 1: int64 entries (bcsr_pos << 32 | col << 16 | row), 0: int32 (col << 16 | row)
    void* grad_k;
    void* grad_v;
    const int32_t* seqlens;   // sequence-length mode of the pipelined kernel: one length per `heads` entries
    int heads;
    float* row_lse;       // log2-domain log-sum-exp per query: written by the forward kernel, read by the recomputing backward kernels
};

template <typename T> struct AttnPack;
template <> struct AttnPack<_Float16> {
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    __device__ static f16x8 pack(f32x8 v) { return __builtin_convertvector(v, f16x8); }
    // sum of the lane's own eight values, added to every element of acc
    __device__ static f32x4 add_lane8(f16x8 v, f32x4 acc) {
        const f16x4 ones = {(_Float16)1.f, (_Float16)1.f, (_Float16)1.f, (_Float16)1.f};
        acc = __builtin_amdgcn_mfma_f32_4x4x4f16(ones, __builtin_shufflevector(v, v, 0, 1, 2, 3), acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_4x4x4f16(ones, __builtin_shufflevector(v, v, 4, 5, 6, 7), acc, 0, 0, 0);
    }
};
template <> struct AttnPack<bf16_t> {
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    // in pairs: one v_cvt_pk_bf16_f32 each (the eight-wide conversion became eight single ones and four merges)
    __device__ static bf16x8 pack(f32x8 v) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        typedef float f32x2 __attribute__((ext_vector_type(2)));
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        u32x4 bits;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            bits[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{v[2 * i], v[2 * i + 1]}, bf16x2));
        return __builtin_bit_cast(bf16x8, bits);
    }
    __device__ static f32x4 add_lane8(bf16x8 v, f32x4 acc) {
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        const s16x8 bits = __builtin_bit_cast(s16x8, v);
        const s16x4 ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
        acc = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_shufflevector(bits, bits, 0, 1, 2, 3), acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_shufflevector(bits, bits, 4, 5, 6, 7), acc, 0, 0, 0);
    }
};

// ---- tiles of 32 rows in LDS, for the kernels with 32 queries or keys per wavefront ----------------
// A tile keeps the rows of 32 queries or keys as they are in memory, 2 E bytes each; the 16-byte chunks of a row
// are XORed by `swizzle(row)`.  Both ways a tile is read then cover all 64 banks: the 16 rows of a pass of fragment
// reads (a chunk per row) and the four rows of a pass of transpose reads (64 bytes of each).
template <int E> struct AttnTile {
    static constexpr int ROW = E * 2;
    static constexpr int BYTES = 32 * ROW;
    static constexpr int LOADS = BYTES / 1024;    // direct loads of 64 x 16 bytes
    static constexpr int EC = E / 16, ET = E / 32;
    __device__ static int swizzle(int row) {
        return E == 64 ? ((row & 2) << 1) | ((row >> 2) & 3) : ((row & 3) << 2) | ((row >> 2) & 3);
    }
    int l32, h2;
    uint32_t fill;      // source offset of load 0; load i: XORed by fill_xor(i) and 1 KB further
    int row;            // row l32, chunk h2: fragment c (16 columns) is at row ^ (c * 32)
    int tr[2];          // transpose reads: k-rows h2 * 4 .. + 3, and 8 further; column tile t at tr ^ (t * 64)
    __device__ explicit AttnTile(int lane) {
        l32 = lane & 31;
        h2 = lane >> 5;
        const int r = lane / (ROW / 16);
        fill = r * ROW + (((lane % (ROW / 16)) ^ swizzle(r)) * 16);
        row = l32 * ROW + ((h2 ^ swizzle(l32)) * 16);
        const int k = h2 * 4 + ((lane & 15) >> 2), chunk = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
#pragma unroll
        for (int hi = 0; hi < 2; ++hi)
            tr[hi] = (k + 8 * hi) * ROW + ((chunk ^ swizzle(k + 8 * hi)) * 16) + (lane & 1) * 8;
    }
    __device__ static constexpr uint32_t fill_xor(int i) { return E == 64 ? (i & 1) * 32 : (i & 3) * 16; }
    // loads first .. first + N - 1 of the 32 rows at `rows` into the tile at LDS address `to`
    template <int N> __device__ __forceinline__ void request(const void* rows, int first, uint32_t to) const {
#pragma unroll
        for (int i = 0; i < N; ++i)
            lds_direct_load16_at(reinterpret_cast<const char*>(rows) + (first + i) * 1024, fill ^ fill_xor(first + i), to + (first + i) * 1024);
    }
    template <typename Frag> __device__ __forceinline__ Frag row_frag(const char* tile, int c) const {
        return *reinterpret_cast<const Frag*>(tile + (row ^ (c * 32)));
    }
    template <typename Frag> __device__ __forceinline__ Frag tr_frag(const char* tile, int t, int u) const {
        typedef short s16x8 __attribute__((ext_vector_type(8)));
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + (tr[0] ^ (t * 64)) + u * 16 * ROW));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(tile + (tr[1] ^ (t * 64)) + u * 16 * ROW));
        return __builtin_bit_cast(Frag, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
};

// 32 rows x 32 columns of an accumulated transpose (lane: row l32 of the result, registers: columns) to memory:
// through LDS to whole 16-byte vectors.
template <typename T, int E>
__device__ __forceinline__ void store_rows32(char* tile, T* dst, const f32x16 (&acc)[E / 32], int lane) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
    typedef float f32x8 __attribute__((ext_vector_type(8)));
    constexpr int PP = E * 2 + 16, VPR = E / 8;
    const int l32 = lane & 31, h2 = lane >> 5;
#pragma unroll
    for (int t = 0; t < E / 32; ++t)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            f32x8 v = {};
#pragma unroll
            for (int x = 0; x < 4; ++x) v[x] = acc[t][4 * a + x];
            *reinterpret_cast<uint64_t*>(tile + l32 * PP + (t * 32 + a * 8 + h2 * 4) * 2) = __builtin_bit_cast(u64x2, AttnPack<T>::pack(v))[0];
        }
#pragma unroll
    for (int i = 0; i < 32 * VPR / 64; ++i) {
        const int c = i * 64 + lane;
        __builtin_nontemporal_store(*reinterpret_cast<const u32x4*>(tile + (c / VPR) * PP + (c % VPR) * 16),
                                    reinterpret_cast<u32x4*>(reinterpret_cast<char*>(dst) + c * 16));
    }
}

// attention_wide.hip: the kernel with 32 queries per wavefront, over an index (query blocks p.BH)
// or over sequence lengths (128 queries per workgroup, or 64 where wavefronts share their keys)
// The index form covers query blocks of 32 / 64 / 128 (one wavefront per 32 queries), key blocks of 32 / 64 / 128 and head
// dimensions 64 / 128.
constexpr bool attention_wide_supported(int BH, int BW, int E) {
    return (BH == 32 || BH == 64 || BH == 128) && (BW == 32 || BW == 64 || BW == 128) && (E == 64 || E == 128) && BW * E <= 128 * BH;
}
int launch_attention_wide(int dtype, const AttnParams& p, int batch, int BW, int E, hipStream_t st);
bool attention_wide_seq_wins(int64_t entries, int N, int E);
int launch_attention_wide_seq(int dtype, const AttnParams& p, int batch, int E, hipStream_t st);

// attention_bwd_wide.hip: backward kernels that recompute the probabilities, 32 queries or keys per wavefront, with
// element masks; query and key blocks of 32 / 64, head dim 64 (on the row side also 128)
// (fp32_scores: what the row statistic is of, see attention.hip; always with an element mask)
int launch_attention_bwd_row_wide(int dtype, const AttnParams& p, int batch, int BW, int E, bool fp32_scores, hipStream_t st);
int launch_attention_bwd_col_wide(int dtype, const AttnParams& p, int batch, int BW, hipStream_t st);

}  // namespace spx
