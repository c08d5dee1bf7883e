// Sparse-operand matmul (the reference's 'sdd' and 'dsd' modes) in one canonical
// form:   out[m, n] = sum_k D[m, k] * S[k, n] (+ bias)
// where S is block-sparse with (BK x BN) blocks listed per block-column n, and D,
// out are dense with arbitrary (row- or column-major) layout.  'dsd' maps
// directly (D = A, S = B); 'sdd' is the transposed problem (D = B^T, S = A^T,
// out = C^T), so both modes, every transpose flag and the compressed /
// uncompressed storage of S differ only in strides.
//
// One workgroup (4 wavefronts) owns a (64*WM) x BN output tile and walks the
// live blocks of its block-column: each live block stages the D panel and the S
// block through LDS as [row][k] and feeds 16x16 MFMAs; the tile leaves through
// LDS so HBM sees full-width row segments.
#pragma once
#include <cmath>
#include "common.hpp"
#include "mma.hpp"
#include "matmul_spmm_ring_plan.hpp"

namespace spx {

struct SpmmParams {
    const void* D;
    const void* S;
    const void* bias;
    void* out;
    const int32_t* ptr;
    const void* idx;
    const int32_t* sched;  // optional launch order of the block-columns (longest first)
    int idx_kind;
    int Mc, K, Nc;       // canonical sizes (Mc: dense rows, Nc: sparse-side cols)
    int BK, log_bk;
    int d_kcontig;       // D[m*d_ld + k] if set, else D[k*d_ld + m]
    int counted;         // s_batch is the size of the live blocks (compressed, and not kept at the capacity of the index)
    int64_t d_ld;
    int s_kcontig;       // block element (k, n): n*s_ld + k if set, else k*s_ld + n
    int compressed;      // S blocks at slot*BK*BN, else inside the dense matrix
    int64_t s_ld;        // leading dimension of the stored S (block-local if compressed)
    int out_ncontig;     // out[m*o_ld + n] if set, else out[n*o_ld + m]
    int64_t o_ld;
    int bias_on_m;       // bias indexed by canonical m instead of n
    int64_t d_batch, s_batch, o_batch, bias_batch;
    int relu;           // epilogue: negative results (after the bias) become zero
    int sub_log2;       // ring kernel, one tile to a workgroup: log2 of the tiles side by side in a block-column
};

// Optional activation of the epilogue; NaN stays NaN (as torch.relu keeps it).
__device__ __forceinline__ float epilogue_act(float v, int relu) { return (relu && v < 0.f) ? 0.f : v; }

template <typename T, int BN, int WM>
__global__ __launch_bounds__(256) void spmm_kernel(SpmmParams p) {
    constexpr int TM = 64 * WM;
    constexpr int NT = BN / 16;
    constexpr int VE = 16 / (int)sizeof(T);
    extern __shared__ __align__(16) char smem[];

    const int ldk = p.BK + VE;  // 16 bytes of padding per row
    T* Ds = reinterpret_cast<T*>(smem);
    T* Ss = Ds + TM * ldk;

    const int j = blockIdx.x;
    const int m0 = blockIdx.y * TM;
    const int64_t b = blockIdx.z;
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int r16 = lane & 15;
    const int g4 = lane >> 4;

    const T* D = reinterpret_cast<const T*>(p.D) + b * p.d_batch;
    const T* S = reinterpret_cast<const T*>(p.S) + b * p.s_batch;
    const int rows_valid = p.Mc - m0;  // > 0 by grid construction

    f32x4 acc[WM][NT];
#pragma unroll
    for (int i = 0; i < WM; ++i)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int e_begin = p.ptr[j];
    const int e_end = p.ptr[j + 1];
    for (int e = e_begin; e < e_end; ++e) {
        int kb;
        int64_t slot;
        if (p.idx_kind == SPX_IDX_BCSC_I64) {
            const long long v = reinterpret_cast<const long long*>(p.idx)[e];
            kb = (int)(v & 0xffff);
            slot = v >> 32;
        } else {
            kb = reinterpret_cast<const int32_t*>(p.idx)[e] & 0xffff;
            slot = e;
        }
        const int64_t k0 = (int64_t)kb * p.BK;
        const T* dsrc = p.d_kcontig ? D + (int64_t)m0 * p.d_ld + k0 : D + k0 * p.d_ld + m0;
        const T* ssrc;
        if (p.compressed) ssrc = S + slot * (int64_t)(p.BK * BN);
        else ssrc = p.s_kcontig ? S + (int64_t)j * BN * p.s_ld + k0 : S + k0 * p.s_ld + (int64_t)j * BN;

        stage_tile<T, TM, 256>(Ds, ldk, p.BK, p.log_bk, dsrc, p.d_ld, p.d_kcontig != 0, rows_valid);
        stage_tile<T, BN, 256>(Ss, ldk, p.BK, p.log_bk, ssrc, p.s_ld, p.s_kcontig != 0, BN);
        __syncthreads();

        const T* a_base = Ds + (wave * 16 * WM + r16) * ldk;
        const T* b_base = Ss + r16 * ldk;
        bool done = false;
        if constexpr (HasMma32<T>::value) {
            if ((p.BK & 31) == 0) {
                for (int kc = 0; kc < p.BK; kc += 32) {
                    typename Mma32<T>::frag af[WM], bf[NT];
#pragma unroll
                    for (int i = 0; i < WM; ++i) af[i] = Mma32<T>::load(a_base + i * 16 * ldk + kc + g4 * 8);
#pragma unroll
                    for (int t = 0; t < NT; ++t) bf[t] = Mma32<T>::load(b_base + t * 16 * ldk + kc + g4 * 8);
#pragma unroll
                    for (int i = 0; i < WM; ++i)
#pragma unroll
                        for (int t = 0; t < NT; ++t) acc[i][t] = Mma32<T>::mma(af[i], bf[t], acc[i][t]);
                }
                done = true;
            }
        }
        if (!done) {
            for (int kc = 0; kc < p.BK; kc += 16) {
                typename Mma16<T>::frag af[WM], bf[NT];
#pragma unroll
                for (int i = 0; i < WM; ++i) af[i] = Mma16<T>::load(a_base + i * 16 * ldk + kc + g4 * 4);
#pragma unroll
                for (int t = 0; t < NT; ++t) bf[t] = Mma16<T>::load(b_base + t * 16 * ldk + kc + g4 * 4);
#pragma unroll
                for (int i = 0; i < WM; ++i)
#pragma unroll
                    for (int t = 0; t < NT; ++t) acc[i][t] = Mma16<T>::mma(af[i], bf[t], acc[i][t]);
            }
        }
        __syncthreads();
    }

    // ---- epilogue: registers -> LDS (output orientation) -> HBM -----------------
    T* Es = reinterpret_cast<T*>(smem);
    const T* biasT = p.bias ? reinterpret_cast<const T*>(p.bias) + b * p.bias_batch : nullptr;
    T* out = reinterpret_cast<T*>(p.out) + b * p.o_batch;
    if (p.out_ncontig) {
        constexpr int LDE = BN + VE;
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int m = wave * 16 * WM + i * 16 + g4 * 4 + q;
                    const int n = t * 16 + r16;
                    float v = acc[i][t][q];
                    if (biasT) {
                        const int bi = p.bias_on_m ? (m0 + m < p.Mc ? m0 + m : 0) : j * BN + n;
                        v += Elem<T>::to_float(biasT[bi]);
                    }
                    Es[m * LDE + n] = Elem<T>::from_float(epilogue_act(v, p.relu));
                }
        __syncthreads();
        constexpr int VPR = BN / VE;
        for (int v = threadIdx.x; v < TM * VPR; v += 256) {
            const int m = v / VPR;
            const int nv = v - m * VPR;
            if (m < rows_valid)
                *reinterpret_cast<vec16*>(out + (int64_t)(m0 + m) * p.o_ld + (int64_t)j * BN + nv * VE) =
                    *reinterpret_cast<const vec16*>(Es + m * LDE + nv * VE);
        }
    } else {
        constexpr int LDE = TM + VE;
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int m = wave * 16 * WM + i * 16 + g4 * 4 + q;
                    const int n = t * 16 + r16;
                    float v = acc[i][t][q];
                    if (biasT) {
                        const int bi = p.bias_on_m ? (m0 + m < p.Mc ? m0 + m : 0) : j * BN + n;
                        v += Elem<T>::to_float(biasT[bi]);
                    }
                    Es[n * LDE + m] = Elem<T>::from_float(epilogue_act(v, p.relu));
                }
        __syncthreads();
        constexpr int VPR = TM / VE;
        for (int v = threadIdx.x; v < BN * VPR; v += 256) {
            const int n = v / VPR;
            const int mv = v - n * VPR;
            if (mv * VE < rows_valid)
                *reinterpret_cast<vec16*>(out + ((int64_t)j * BN + n) * p.o_ld + m0 + mv * VE) =
                    *reinterpret_cast<const vec16*>(Es + n * LDE + mv * VE);
        }
    }
}

template <typename T>
int launch_spmm(const SpmmParams& p, int BN, int batch, int tile_cfg, hipStream_t st);

template <typename T, int BN, int WM>
static int launch_spmm_inst(const SpmmParams& p, int batch, hipStream_t st) {
    constexpr int TM = 64 * WM;
    constexpr int VE = 16 / (int)sizeof(T);
    const int ldk = p.BK + VE;
    size_t main_bytes = (size_t)(TM + BN) * ldk * sizeof(T);
    size_t epi_a = (size_t)TM * (BN + VE) * sizeof(T);
    size_t epi_b = (size_t)BN * (TM + VE) * sizeof(T);
    size_t smem = main_bytes;
    if (epi_a > smem) smem = epi_a;
    if (epi_b > smem) smem = epi_b;
    dim3 grid(p.Nc / BN, (p.Mc + TM - 1) / TM, batch);
    hipLaunchKernelGGL((spmm_kernel<T, BN, WM>), grid, dim3(256), smem, st, p);
    SPX_LAUNCH_CHECK("spmm_kernel");
    return 0;
}

template <typename T>
int launch_spmm_direct(const SpmmParams& p, int BN, int batch, int wm, hipStream_t st);
template <typename T>
int launch_spmm_panel(const SpmmParams& p, int BN, int batch, int nst, hipStream_t st);
template <typename T>
int launch_spmm_stream(const SpmmParams& p, int BN, int batch, hipStream_t st);
template <typename T>
int launch_spmm_ksplit(const SpmmParams& p, int BN, int batch, hipStream_t st);
template <typename T>
int launch_spmm_ring(const SpmmParams& p, int BN, int batch, int rows, hipStream_t st);
// What the LDS-ring kernel takes: 64-byte block rows, and a dense operand that can be read in 16-byte pieces.
template <typename T>
bool spmm_ring_supported(const SpmmParams& p, int BN) {
    constexpr int VE = 16 / (int)sizeof(T);
    return (p.BK * (int)sizeof(T)) % 64 == 0 && (BN == 16 || BN == 32 || BN == 64) &&
           (p.d_kcontig || (p.Mc % VE == 0 && p.d_ld % VE == 0)) && (p.out_ncontig || p.Mc % VE == 0) &&
           p.d_ld * 128 + p.K < (int64_t)1 << 29 && (p.compressed || p.s_ld * 64 + p.K < (int64_t)1 << 29);   // byte offsets in 32 bits
}
// Rows of the dense operand kept in LDS (matmul_spmm_rows.hpp), where that is ahead; kSpmmRowsNot: it is not.
constexpr int kSpmmRowsNot = -1000;   // (no status of the interface)
template <typename T>
int launch_spmm_rows(const SpmmParams& p, int BN, int batch, hipStream_t st);
template <typename T>
bool spmm_thin_supported(const SpmmParams& p, int BN);
template <typename T>
int launch_spmm_thin(const SpmmParams& p, int batch, hipStream_t st);

// fp32 blocks of 16 x 16, both operands k-contiguous: whether 64-row tiles of the ring kernel are ahead of split columns (`split`)
// or of 256-row tiles.  Estimates in us, fitted to 1300 random problems of 700 to 6000 rows and 2 - 40 % live blocks (root mean square off by
// 5 - 8 %).  What counts: the rounds of workgroups (the second one takes as long as the first, however few tiles it has), the dense
// rows that every XCD reads anew where panels are dealt out by columns, and the panels that leave XCDs idle in the other two.
// Other kernel / ring: 1024^3 at 35 % (one round) 17.5 / 15.0, 774 x 784 x 3584 at 25 % 28.6 / 23.8, 877 x 896 x 1728 at 20 % 16.2 / 13.7,
// 1044 x 1328 x 3648 at 10 % 30.3 / 22.2, 2285 x 576 x 1024 at 8 % 15.2 / 10.2, 4577 x 576 x 512 at 14 % 19.8 / 13.2, but 512 x 1024 x
// 1024 at 35 % 9.8 / 12.3, 1809 x 1056 x 704 at 31 % 18.5 / 27.4, 1966 x 784 x 576 at 14 % 10.6 / 17.3, 985 x 1120 x 768 at 40 % 14.3 / 15.7,
// 1848 x 1040 x 1920 at 38 % 43.4 / 51.5, 2855 x 656 x 832 at 18 % 17.7 / 22.3, 5998 x 752 x 1024 at 3 % 11.2 / 14.5.
inline bool spmm_ring_ahead_of_16(const SpmmParams& p, int64_t stored, bool split) {
    const int nb = p.Nc / 16, panels64 = (p.Mc + 63) / 64, panels256 = (p.Mc + 255) / 256;
    const double per = (double)stored / nb, out = (double)p.Mc * p.Nc * 1e-6;   // blocks to a column, millions of results
    const RingLaunch l = ring_launch(4, 64, 16, p.out_ncontig != 0, p.Mc, p.K, p.Nc, 1);
    const int rounds = ring_rounds(l.n_list, l.n_pos);
    const double tiles = l.n_list / 32.0, dense = (double)p.Mc * p.K * 4e-6 * (1 << l.list.parts_log2);   // tiles to a CU; MB
    const double ring = rounds == 1 ? 4.41 + per * (0.244 + 0.052 * tiles) + 0.149 * out + 0.006 * dense
                                    : 4.09 + per * (0.195 * rounds + 0.067 * tiles) + 0.51 * out + 0.065 * dense;
    const double tiles64 = (panels64 + 7) / 8 * nb / 32.0, tiles256 = (panels256 + 7) / 8 * nb / 32.0;   // of the XCD that has most, to a CU
    const double other = split ? 4.85 + tiles64 * (0.409 + 0.076 * per) + 0.045 * std::ceil(tiles64 / 5) * per + 0.84 * out
                               : 7.25 + per * (0.252 * std::ceil(tiles256) + 0.169 * std::ceil(tiles256 / 3) + 0.042 * tiles256) + 0.37 * out;
    return ring < other;
}

// tile_cfg: 0 = pick by layout and size;
//   1 / 2  LDS-staged kernel, 64 / 128-row workgroup tiles (any layout);
//   3 / 4  register-direct kernel, 64 / 256-row workgroup tiles (k-contiguous operands);
//   5 / 6  panel kernel, 256-row workgroup tiles, 2 / 3 load stages (k-contiguous
//          operands, block depth a multiple of 64 bytes);
//   8      K-split panel kernel: 64-row workgroup tiles, the four wavefronts split the
//          live blocks of a block-column (k-contiguous operands, BN <= 32): few rows.
//   7      panel kernel whose four wavefronts share the sparse block through LDS (the
//          sparse operand may be stored with n contiguous: it is transposed on the way).
//   9      thin dense operand (64 or 128 values of m, stored with m contiguous; 16-bit
//          types, 64-wide k-contiguous sparse blocks): one workgroup per block-column.
//   10     persistent form of 7 for a k-contiguous dense operand: a workgroup walks the
//          tiles of its XCD as one stream of steps (matmul_spmm_stream.hpp).
//   11 / 12  ring of LDS stages filled by a loader wavefront, 64 / 128-row tiles, any layout with
//          64-byte block rows (matmul_spmm_ring.hpp).
template <typename T>
int launch_spmm_impl(const SpmmParams& p, int BN, int batch, int tile_cfg, hipStream_t st) {
    const bool kcontig = p.d_kcontig && p.s_kcontig;
    const bool panel_ok = kcontig && (p.BK * (int)sizeof(T)) % 64 == 0;
    // the shared-S panel variant transposes an n-contiguous sparse block while staging it
    // ... and reads a dense operand stored with m contiguous through LDS transpose reads
    const bool panel7_ok = (p.BK * (int)sizeof(T)) % 64 == 0 &&
                           (p.d_kcontig || (p.Mc % (16 / (int)sizeof(T)) == 0 && p.d_ld % (16 / (int)sizeof(T)) == 0));
    if (tile_cfg < 0 || tile_cfg > 12) return fail(SPX_E_CONFIG, "unknown tile config %d", tile_cfg);
    const bool stream_ok = p.d_kcontig && (p.BK * (int)sizeof(T)) % 64 == 0 && p.d_ld * 256 + 64 < (int64_t)0x7fffffff / (int)sizeof(T);
    const bool ksplit_ok = panel_ok && BN <= 32;
    const bool thin_ok = spmm_thin_supported<T>(p, BN);
    // one workgroup per block-column only where every one of them has a long walk over a sparse operand
    // that streams from HBM (96 x 4096 x 4096: 82 us against 106 through the ring); below, the ring kernel
    // is ahead (1 x 3072 x 4096 x 64 at 20 %: 15.3 / 9.3, 48 x 1024 x 1024 x 64 at 10 %: 8.2 / 7.8)
    if (tile_cfg == 0 && thin_ok && (int64_t)batch * p.K * p.Nc >= 500000000) tile_cfg = 9;
    if (tile_cfg == 9) {
        if (!thin_ok) return fail(SPX_E_CONFIG, "tile config 9 needs a 16-bit dense operand with 64 or 128 contiguous m and 64-wide k-contiguous blocks of depth 32 / 64");
        return launch_spmm_thin<T>(p, batch, st);
    }
    const bool ring_ok = spmm_ring_supported<T>(p, BN);
    if constexpr (sizeof(T) == 2)
        if (tile_cfg == 0) {   // (the rule stands beside the kernel)
            const int rc = launch_spmm_rows<T>(p, BN, batch, st);
            if (rc != kSpmmRowsNot) return rc;
        }
    if (tile_cfg == 0) {
        // 256-row tiles only when they still give every CU a few workgroups; small
        // problems are latency-bound and want more, shorter workgroups.
        const int nb = p.Nc / BN, cols = p.K / p.BK;
        const int64_t big_tiles = (int64_t)((p.Mc + 255) / 256) * nb * batch;
        const int64_t tiles128 = (int64_t)((p.Mc + 127) / 128) * nb * batch;
        const bool fill = big_tiles >= 512;
        const int64_t tiles64 = (int64_t)((p.Mc + 63) / 64) * nb * batch;
        // 128-row tiles halve the traffic of the sparse blocks.  fp32 spends long on a tile and wants many of them; 16-bit
        // types take the tiles that need fewer rounds of the workgroups that fit the chip (64 / 128 rows, us): 32 x 64 blocks
        // 6993 x 768 -> 704 (2 rounds each) 7.4 / 10.6, 5639 x 704 -> 1152 (3) 10.4 / 15.8, 1036 x 2688 -> 2560 (2 and 1) 20.9 / 15.9,
        // 1911 x 1600 -> 3648 (3) 15.9 / 17.1, 4674 x 2432 -> 2496 (5 and 4) 47.9 / 43.9, 15667 x 896 -> 2304 (14 and 12) 34.3 / 31.1; blocks of depth 32
        // have shorter walks: 3917 x 2880 -> 704 (2 and 1) 20.7 / 18.2, but 6319 x 1792 -> 1792 (5 and 4) 13.9 / 17.2, 5350 x 3008 -> 1728
        // (4 and 3) 33.4 / 38.4; 64 x 64 blocks 3870 x 576 -> 896 (2 and 1) 9.7 / 7.6, 2748 x 1728 -> 1280 (2 and 1) 7.0 / 5.6
        int ring = tiles128 >= (sizeof(T) == 4 ? 2048 : 1024) ? 12 : 11;
        // (rounds over all batch entries together, which the launch deals out one by one)
        const int slots64 = ring_slots((int)sizeof(T), 64, BN, p.out_ncontig != 0), slots128 = ring_slots((int)sizeof(T), 128, BN, p.out_ncontig != 0);
        const int64_t rounds64 = (tiles64 + slots64 - 1) / slots64, rounds128 = (tiles128 + slots128 - 1) / slots128;
        if (sizeof(T) == 2) {
            if (BN != 64) ring = rounds128 < rounds64 && (p.BK == 64 || rounds64 <= 2) ? 12 : 11;
            else if (rounds64 == 2 && rounds128 == 1) ring = 12;
        }
        // The ring kernel, where it was measured ahead (rows x K x N; us of the best other kernel / ring):
        //   * operands that are not both k-contiguous: sdd 4096 x 3072 x 768 fp32 at 20 % 110 / 38, fp16 26 / 14,
        //     dsd 400 x 3072 x 768 fp32 at 15 % 38 / 10, bf16 14 / 10 - but for large fp32 problems in blocks
        //     of depth 16, whose stages hold two blocks each (4096 x 768 x 3072: 46 / 55);
        //   * k-contiguous fp32 and 16-bit blocks of depth 64: 4096 x 3072 x 768 fp32 at 10 % 33 / 22, bf16
        //     64 x 64 at 20 % 25 / 14, 200 x 768 x 3072 7 / 5;
        //   * 16-bit blocks of depth 32 (two to a stage) while the result is narrow: 8192 x 1024 x 1024
        //     at 10 % 16.5 / 13.5; wide results (tiles of one or two stages) stay with the 256-row
        //     kernels: 8192 x 768 x 3072 at 10 % 23 / 28, 4096^3 at 5 % 25.5 / 31.
        //     Up to 1024 rows the 256-row kernels have too few workgroups for long block-columns, also where
        //     the result is wide: 1024 x 4096 x 4096 at 35 % 61 / 43, 1024^2 x 4096 at 35 % 19.8 / 14.7, at 10 %
        //     9.8 / 9.2.  Against the column-split kernel (config 8) it is ahead from about 700 64-row tiles on:
        //     634 x 1152 x 3008 at 38 % 17.0 / 10.0, 580 x 3840 x 2496 at 37 % 30.8 / 23.5, 549 x 2176 x 4096 42 / 17, 1500 x 1024 x 2048 15.0 / 11.9; with 512 to
        //     700 tiles up to 20 live blocks to a column: 693 x 1280 x 1792 at 27 % 12.3 / 8.9, 605 x 1920 x 1792 at 28 % 13.9 / 10.4, 1151 x
        //     1856 x 1152 at 31 % 13.3 / 11.1, 944 x 1024 x 1152 at 2 % 5.7 / 4.0, but with more 13.5 / 18.7 (935 x 2880 x 1152 at 35 %),
        //     15.0 / 17.5 (392 x 3072 x 3072 at 37 %), 16.3 / 18.5 (1163 x 3072 x 1024 at 32 %).
        const bool two_blocks = p.BK * (int)sizeof(T) == 64;
        // stored blocks in all block-columns together (all places where it is not known), and the live ones as the later rules count on them
        const int64_t stored = p.compressed && p.s_batch > 0 ? p.s_batch / ((int64_t)p.BK * BN) : (int64_t)cols * nb;
        const int64_t live = spmm_live_blocks(p.counted, stored, (int64_t)cols * nb);
        // fp32 blocks of depth 16, long block-columns: four wavefronts that split a column and meet once keep
        // more loads in flight than 256-row tiles when those are few.  256-row kernel / split columns:
        // up to 1024 rows 512 x 4096 x 4096 at 35 % 259 / 85 us, at 5 % 45 / 20, 1024 x 2048 x 2048 74 / 45 and
        // 16.4 / 14.4; narrow results 8192 x 2048 x 512 91 / 76 and (5 %) 28.1 / 25.9, 4096 x 2048 x 512 54 / 42,
        // 4096 x 1024 x 512 32 / 28, 4380 x 1408 x 960 54 / 41, 4096 x 2048 x 1024 79 / 75, but 12.3 / 12.7 with four live blocks to a column and 158 / 148, 30 / 38 at
        // 16384 rows; wide ones with more rows are mixed (2048^3 at 35 % 74 / 77, 4096 x 512 x 2048 44 / 51).
        const bool split_columns = sizeof(T) == 4 && two_blocks && BN == 16 && ksplit_ok && cols > 48 &&
                                   p.Mc > 256 && (p.Mc <= 1024 || (p.Mc <= 8192 && nb <= 32 && stored >= 6 * nb) ||
                                                    (p.Mc <= 4608 && nb <= 64 && stored >= 12 * nb));
        bool use_ring = ring_ok;
        if (two_blocks && sizeof(T) == 4) {
            use_ring = ring_ok && (!kcontig || cols <= 48) && !(p.Mc >= 2048 && fill);
            // blocks of 16 x 16, where the number of blocks is known: by estimates (of wide results with more rows, 2719 x 640 x 2624, and
            // of less than two blocks to a column, 2187 x 544 x 1984, they are too good for the ring)
            if (kcontig && BN == 16 && ring_ok && batch == 1 && p.compressed && p.s_batch > 0 && p.Mc >= 700 && p.Mc <= 6000 &&
                (p.Mc < 2048 ? cols > 48 && cols <= 88 : cols <= 48 && fill && nb <= 96 && stored >= 2 * (int64_t)nb && stored <= 8 * (int64_t)nb) &&
                spmm_ring_ahead_of_16(p, stored, split_columns || !fill)) {
                use_ring = true;
                ring = 11;
            }
        } else if (two_blocks && kcontig) {
            const bool few_rows = p.Mc > 256 && p.Mc < 2048 && cols >= 32 && BN == 32 &&
                                  (tiles64 >= 700 || (tiles64 >= 512 && stored <= 20 * (int64_t)nb));
            // wide results of 2048 to 3072 rows: 256-row tiles do not come out even (256-row kernel / ring 2474 x
            // 1408 x 3328 at 28 % 31.0 / 23.3, 2518 x 1088 x 3776 28.7 / 21.9, 2579 x 2624 x 2048 37.9 / 30.4, 2520 x 2112 x 2240 at 13 % 18.9 / 15.7)
            // ... and neither do five and six of them over eight XCDs (256-row kernel / ring, us: 1256 x 3200 x 3488 at 21 % 33.8 / 22.9, 1503 x 1280 x
            // 3392 16.9 / 12.6, 1220 x 2496 x 3424 with 4.1 blocks to a column 10.6 / 8.9; seven 1606 x 2880 x 2688 15.0 / 17.3, shorter walks 1537 x
            // 896 x 3616 7.5 / 8.1; where the live blocks are not counted, dense storage with one, two, four and eight to a column: 1500 x 1024 x 3072
            // 6.9 / 6.9, 7.7 / 7.3, 9.9 / 8.9, 13.6 / 12.6, 1256 x 2048 x 3424 6.6 / 6.9, 8.5 / 7.3, 11.1 / 9.5, 16.7 / 13.5)
            const bool mid_rows = sizeof(T) == 2 && BN == 32 && p.Nc >= 2048 &&
                                  ((p.Mc > 2048 && p.Mc <= 3072) || (p.Mc > 1024 && p.Mc <= 1536 && live >= 4 * (int64_t)nb));
            if (mid_rows) ring = rounds128 < rounds64 ? 12 : 11;   // (4 and 3 rounds 29.3 / 23.3; 3 each 41 / 51, 2626 x 3584 x 2688 at 24 %)
            if (fill) use_ring = ring_ok && cols >= 32 && (p.Nc < 2048 || mid_rows || (few_rows && p.Mc <= 1024));
            else use_ring = ring_ok && p.Mc > 256 && (p.Mc >= 2048 || cols < 32 || few_rows);
        }
        // 16-bit blocks of depth 64, a block or less to a block-column: next to no walk, the time is the output's, and the
        // 256-row kernels write it faster.  Ring / 256-row: 32 x 64 blocks 16384 x 512 x 2048 at 5 % 27.7 / 15.4 us, 8192 x
        // 768 x 3072 at 10 % 20.8 / 18.5 and at 5 % 19.0 / 14.2, 4096 x 1024 x 4096 at 5 % 14.4 / 12.3; 64 x 64 blocks at 10 %
        // 29.0 / 24.5 and 23.2 / 20.9.  With 1.6 blocks to a column 16.1 / 17.4 (4096 x 1024 x 4096), with three 29 / 36
        // (8192 x 768 x 3072); at 2048 rows 6.9 / 7.3.
        // Between 2048 and 4096 rows the two cross (bf16, 32 x 64 blocks, 0.6 / 1.2 blocks to a column): 2560 x 768 x 3072 10.1 / 9.8
        // and 10.2 / 12.4, 2992 rows 10.6 / 9.7 and 11.4 / 12.4, 3584 rows 12.7 / 10.0 and 13.9 / 12.6; 2992 x 1024 x 4096 12.8 / 13.2
        // and 14.1 / 16.6, 3584 rows 14.5 / 13.3 and 16.2 / 16.8; the line lies at the end of that stretch.
        const bool short_columns = sizeof(T) == 2 && panel_ok && !two_blocks && p.Mc >= 4096 && fill && stored * 4 <= (int64_t)nb * 5;
        // the persistent form when its 8 * (N / BN) slots fill the device four times over, every
        // slot walks at least two 256-row tiles and the block-columns are long: 28.4 - 28.7 us
        // against 29.9 - 30.0 us for 7 on the 4096^3 problem (alternating runs on three
        // machines); with fewer slots or tiles it loses (C4 layers: 28 / 34 against 20 / 21 us)
        if (stream_ok && panel_ok && batch == 1 && 8 * nb >= 1024 && p.Mc >= 16 * 256 && cols >= 32 && two_blocks &&
            sizeof(T) == 2 && (BN == 16 || BN == 32 || BN == 64))
            tile_cfg = 10;
        else if (short_columns) tile_cfg = BN == 64 ? 7 : 5;
        else if (use_ring) tile_cfg = ring;
        else if (split_columns) tile_cfg = 8;
        else if (panel_ok && p.Mc >= 512 && fill) tile_cfg = p.Mc >= 1024 ? 7 : 5;
        // 16-bit blocks of 32 x 32, tiles that have a workgroup each: the ring kernel shares a walk out over more wavefronts than split
        // columns do and brings it through LDS stages ahead.  Split columns / ring, us: 320 x 1024 -> 1472 at 16 % 6.7 / 4.5, 80 x 1792 ->
        // 1856 5.9 / 4.4, 592 x 2880 -> 1536 at 27 % 15.0 / 10.6, 401 x 1152 -> 1344 at 26 % 7.1 / 5.9; longer walks in more tiles 368 x 2496 ->
        // 1472 at 36 % 8.9 / 10.1, 832 x 3136 -> 896 at 40 % 12.8 / 14.9.  No split (below) / ring: 192 x 896 -> 1408 at 26 % 5.7 / 4.5, 64 x 704 -> 1856
        // 5.3 / 4.5, but 28 x 960 -> 2816 4.2 / 4.5, 3 x 3328 -> 1728 3.9 / 5.7 and five blocks to a column 87 x 576 -> 3136 4.4 / 5.2.
        // The lines: split columns are ahead where a walk has too few stages for several groups, four blocks to a column up to 256 tiles
        // (ring / split 1.13 over 80 problems of 64 to 592 rows, with five 0.98, six 0.96, eight to twenty 1.00 - 1.03; above 256 tiles 0.94, 0.80, 0.81, 0.84 - 0.89).  No
        // split is ahead up to 48 rows below twelve blocks (33 x 704 -> 1856 with six, eight and twelve 4.2 / 4.6, 4.5 / 5.0, 5.2 / 5.2; 48 rows 4.5 / 4.7,
        // 4.7 / 5.0, 5.5 / 5.4; 64 rows 4.8 / 4.6, 5.1 / 4.7, 6.0 / 5.3).
        // Where the live blocks are not counted: from the places on that several groups of wavefronts share a walk (five blocks, 40 places), and
        // where the others have more tiles than CUs.  Dense storage, one, three and eight live blocks to a column, split columns / ring: 300 x 1280 -> 1024 (40
        // places) 4.2 / 4.0, 4.4 / 4.0, 5.1 / 4.8, but 300 x 1184 -> 1024 (37) 4.2 / 4.0, 4.4 / 4.6, 5.1 / 6.5; 300 x 1088 -> 2048 (320 tiles) 4.9 / 4.1,
        // 5.7 / 5.2, 6.8 / 6.8, 800 x 1024 -> 1024 (416) 5.2 / 4.6, 5.9 / 5.1, 7.2 / 7.4, 600 x 2048 -> 1024 (320) with 8, 16 and 26 7.3 / 5.7, 8.9 / 7.0, 11.1 / 8.7.  No
        // split / ring: one, two, four and ten: 128 x 512 -> 1536 (96 tiles) 3.7 / 3.9, 4.2 / 4.5, 5.0 / 5.1, 7.0 / 6.7, 64 x 768 -> 3072 3.5 / 3.8, 4.2 / 4.4,
        // 5.4 / 5.4, 7.4 / 7.2, but 256 x 768 -> 3072 (384) 4.7 / 4.6, 5.3 / 4.8, 7.3 / 5.8, 11.1 / 7.6.  Up to 64 places to a column (277 x 3840 -> 960 at 24 % 8.8 / 10.0).
        else if (sizeof(T) == 2 && ring_ok && kcontig && two_blocks && BN == 32 && !fill && p.Mc > 32 && tiles64 <= 512 &&
                 (tiles64 <= 256 || live <= 26 * (int64_t)nb) &&
                 (!p.counted                     ? cols >= 8 && cols <= 64 && (tiles64 > 256 || live >= 5 * (int64_t)nb)
                  : p.Mc <= 256 && cols <= 32    ? live >= (p.Mc <= 48 ? 12 : 6) * (int64_t)nb
                                                 : cols >= 8 && live >= (tiles64 > 256 ? 4 : 5) * (int64_t)nb))
            tile_cfg = 11;
        // few rows and short columns: no barrier and no shared block pays (64 x 768 x 3072 bf16: 3.9 us
        // against 4.4 with the columns split and 5.2 through the ring)
        else if (kcontig && (p.Mc <= 16 ? cols <= 128 : p.Mc <= 256 && cols <= 32)) tile_cfg = 3;
        else if (ksplit_ok && !fill && cols >= 8) tile_cfg = 8;  // few tiles, long block-columns
        else if (panel7_ok && p.Mc >= 512 && fill) tile_cfg = 7;
        else if (kcontig) tile_cfg = p.Mc >= 1024 && fill ? 4 : 3;
        else tile_cfg = p.Mc >= 1024 && fill ? 2 : 1;
    }
    if (tile_cfg >= 11) {
        if (!ring_ok) return fail(SPX_E_CONFIG, "tile config %d needs 64-byte block rows and 16-byte pieces of the dense operand", tile_cfg);
        return launch_spmm_ring<T>(p, BN, batch, tile_cfg == 11 ? 64 : 128, st);
    }
    if (tile_cfg == 10) {
        if (!stream_ok) return fail(SPX_E_CONFIG, "tile config 10 needs a k-contiguous dense operand and 64-byte block rows");
        return launch_spmm_stream<T>(p, BN, batch, st);
    }
    if (tile_cfg == 8) {
        if (!ksplit_ok) return fail(SPX_E_CONFIG, "tile config 8 needs k-contiguous operands, 64-byte block rows and BN <= 32");
        return launch_spmm_ksplit<T>(p, BN, batch, st);
    }
    if (tile_cfg >= 5) {
        if (!(tile_cfg == 7 ? panel7_ok : panel_ok))
            return fail(SPX_E_CONFIG, "tile config %d needs k-contiguous operands and 64-byte block rows", tile_cfg);
        return launch_spmm_panel<T>(p, BN, batch, tile_cfg == 6 ? 3 : tile_cfg == 7 ? 12 : 2, st);
    }
    if (tile_cfg >= 3) {
        if (!kcontig) return fail(SPX_E_CONFIG, "tile config %d needs k-contiguous operands", tile_cfg);
        return launch_spmm_direct<T>(p, BN, batch, tile_cfg == 4 ? 4 : 1, st);
    }
    const int wm = tile_cfg == 2 ? 2 : 1;
    if (wm == 2) {
        switch (BN) {
            case 16: return launch_spmm_inst<T, 16, 2>(p, batch, st);
            case 32: return launch_spmm_inst<T, 32, 2>(p, batch, st);
            case 64: return launch_spmm_inst<T, 64, 2>(p, batch, st);
        }
    } else {
        switch (BN) {
            case 16: return launch_spmm_inst<T, 16, 1>(p, batch, st);
            case 32: return launch_spmm_inst<T, 32, 1>(p, batch, st);
            case 64: return launch_spmm_inst<T, 64, 1>(p, batch, st);
        }
    }
    return fail(SPX_E_CONFIG, "sparse block width %d not in {16,32,64}", BN);
}

}  // namespace spx
