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

// attention_wide.hip: the kernel with 32 queries per wavefront, over an index (query blocks p.BH)
// or over sequence lengths (128 queries per workgroup)
int launch_attention_wide(int dtype, const AttnParams& p, int batch, int BW, int E, hipStream_t st);
int launch_attention_wide_seq(int dtype, const AttnParams& p, int batch, int E, hipStream_t st);

// attention_bwd_wide.hip: backward kernels that recompute the probabilities, 32 queries or keys per wavefront, with
// element masks; query and key blocks of 32 / 64, head dim 64
int launch_attention_bwd_row_wide(int dtype, const AttnParams& p, int batch, int BW, hipStream_t st);
int launch_attention_bwd_col_wide(int dtype, const AttnParams& p, int batch, int BW, hipStream_t st);

}  // namespace spx
