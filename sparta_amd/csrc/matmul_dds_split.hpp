// Sparse-output matmul for operands that are not both k-contiguous - the weight gradient
// grad_W = grad_y^T x (A stored [K, M], B stored [K, N], K = tokens) above all - with the
// reduction over k optionally split over several workgroups.
//
// What bounds it.  A live block is a skinny product: every k brings BM + BN elements for
// BM x BN multiply-adds, so the operand bytes through the L1s are the floor (a CU takes in
// 23 - 28 bytes per clock), and with one workgroup per block a pruned layer has too few
// workgroups to reach it: a 3072 x 768 weight with 115 live 32 x 64 blocks kept 115 of 256 CUs
// busy with one chain of dependent stages each.  Therefore:
//   * k is cut into 1, 2, 4 or 8 slices and a slice of all blocks runs on the 8 / slices XCDs of
//     its own: with eight of them an XCD reads its token range of both operands once into its own
//     L2, where a band of block rows per XCD (the unsliced launch) reads most of the other
//     operand eight times.  The fp32 partial blocks go to a workspace and a second kernel
//     adds them in slice order (no atomics, bit-identical from run to run).
//   * a stage is 64 k deep, half of the k-contiguous kernel's for 16-bit types, so that four or five
//     workgroups with two LDS buffers fit a CU.
//   * any K (a multiple of 16 as for every kernel of this family) runs here: the rows of a short
//     last stage are fetched from a valid address and written to LDS as zeros.  Before, a token
//     count that was no multiple of 128 fell to the kernel without a pipeline.
//   * the column sums of A over k - the bias gradient - ride along: extra workgroups at the
//     end of the launch add up all tokens, or where k is sliced 32 ranges of them, which the
//     second kernel finishes.
//
// AT / BT: the operand is stored [K, M] / [K, N]; otherwise it is k-contiguous.  LDS layouts and
// fragment reads: a stage keeps the rows as they are in memory; [k][m] rows give the
// k-contiguous fragments through the LDS transpose read (16-bit types: lane i of a 16-lane
// group addresses four entries of k-row i / 4, lane j receives column j of the four rows) or
// four 4-byte reads (fp32).
#pragma once
#include <cmath>
#include "matmul_dds.hpp"

namespace spx {

constexpr int kColsumSlices = 32;
constexpr int64_t kSplitPartialBytes = (int64_t)1 << 30;   // most that a chosen split takes for its partial blocks

constexpr int kColsumWholeK = 4096, kColsumWholeKEmpty = 2560;

// Whether a workgroup adds up its columns over all of k.  An unsliced product walks k just as far itself and hides
// that, and the call is one launch: without column ranges, their workspace and the second kernel the weight gradient
// with its bias gradient takes 3.1 instead of 6.2 us (115 blocks of 32 x 64 over 64 tokens fp16), 9.8 instead of 12.6
// (1024 tokens), 42 instead of 45 (1300 blocks over 2048), 88.6 instead of 93.6 (4096).  Without a block there is nothing
// that hides the walk.  fp32 columns, whose groups are twice as many, gain all the same (768, 3072 and 4096 of them at 4096
// tokens 6.8, 12.3 and 12.7 us against 5.7, 14.1 and 19.9 in ranges), 16-bit ones up to 2560 tokens (6.7, 6.8 and 6.8 against 5.7,
// 6.9 and 7.4; at 3072 7.5, 7.6 and 7.6 against 5.6, 7.1 and 7.7, at 4096 9.2, 9.3 and 11.1 against 5.8, 7.4 and 9.8).
inline bool dds_colsum_whole(int elem_bytes, int slices, int nnz, int K) {
    return slices == 1 && K <= (nnz > 0 || elem_bytes == 4 ? kColsumWholeK : kColsumWholeKEmpty);
}

struct DdsSplit {
    int slices;         // 1, 2, 4 or 8; 1: every block is one workgroup and writes C itself
    int k_slice;        // k per slice (a multiple of the stage depth)
    int nnz;            // live blocks (the bound, where nnz_dev gives the number)
    int n_product;      // workgroups of the product; the ones behind them sum columns
    float* partial;     // [batch][slices][nnz][BM * BN]
    float* colsum;      // [batch][kColsumSlices][M], NULL: not wanted, or:
    void* colsum_out;   // [batch][M] of the operand type: a workgroup adds up all of k and writes the sums themselves
    int share;          // blocks of a block-row to a workgroup (matmul_dds_share.hpp), 0: one each
};

template <typename T, int BM, int BN> struct DdsSplitCfg {
    // the 16 x 16 block splits a stage over its four wavefronts and needs 32 (16) k for each
    static constexpr int KT = sizeof(T) == 2 ? (BM + BN <= 32 ? 128 : 64) : (BM + BN <= 64 ? 64 : 32);
    static constexpr int NST = 2;
};

// Column sums of A over one of kColsumSlices ranges of k, or over all of it: eight lanes side by side
// (16 bytes of m each), 32 rows of k at a time.
template <typename T>
__device__ __forceinline__ void dds_colsum_range(const DdsParams& p, const DdsSplit& s, int id, float* lds) {
    constexpr int VE = 16 / (int)sizeof(T);
    constexpr int COLS = 8 * VE;
    const int64_t b = blockIdx.y;
    const bool whole = s.colsum_out != nullptr;
    const int sl = whole ? 0 : (id & 7) * (kColsumSlices / 8) + ((id >> 3) & (kColsumSlices / 8 - 1));  // XCD x reads what its slices read
    const int group = whole ? id : id / kColsumSlices;
    const int c = group * COLS + (threadIdx.x & 7) * VE;
    const int rl = threadIdx.x >> 3;
    const int k0 = (int)((int64_t)sl * p.K / kColsumSlices);
    const int k1 = whole ? p.K : (int)((int64_t)(sl + 1) * p.K / kColsumSlices);
    const T* A = reinterpret_cast<const T*>(p.A) + b * p.a_batch;
    float v[VE];
#pragma unroll
    for (int e = 0; e < VE; ++e) v[e] = 0.f;
    if (c < p.M) {
        // in runs of 1024 rows, 32 to a thread: the sums of all of k take no longer chains of additions than those of the ranges
        for (int kr = k0; kr < k1; kr += 1024) {
            const int end = kr + 1024 < k1 ? kr + 1024 : k1;
            float run[VE];
#pragma unroll
            for (int e = 0; e < VE; ++e) run[e] = 0.f;
#pragma unroll 8
            for (int k = kr + rl; k < end; k += 32) {
                union { vec16 q; T t[VE]; } u;
                u.q = *reinterpret_cast<const vec16*>(A + (int64_t)k * p.a_ld + c);
#pragma unroll
                for (int e = 0; e < VE; ++e) run[e] += Elem<T>::to_float(u.t[e]);
            }
#pragma unroll
            for (int e = 0; e < VE; ++e) v[e] += run[e];
        }
    }
    constexpr int LD = COLS + 4;
#pragma unroll
    for (int e = 0; e < VE; ++e) lds[rl * LD + (threadIdx.x & 7) * VE + e] = v[e];
    __syncthreads();
    const int col = group * COLS + threadIdx.x;
    if (threadIdx.x < COLS && col < p.M) {
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < 32; ++r) sum += lds[r * LD + threadIdx.x];
        if (whole) reinterpret_cast<T*>(s.colsum_out)[b * p.M + col] = Elem<T>::from_float(sum);
        else s.colsum[(b * kColsumSlices + sl) * p.M + col] = sum;
    }
}

template <typename T, int BM, int BN, bool AT, bool BT>
__global__ __launch_bounds__(256) void dds_split_kernel(DdsParams p, DdsSplit s) {
    constexpr int MT = BM / 16, NT = BN / 16;
    typedef DdsWaveGrid<MT, NT> W;
    constexpr int ES = (int)sizeof(T);
    constexpr int VE = 16 / ES;
    constexpr int KT = DdsSplitCfg<T, BM, BN>::KT, NST = DdsSplitCfg<T, BM, BN>::NST;
    constexpr int KW = KT / W::KS;
    constexpr int LDA = (AT ? BM : KT) + VE, LDB = (BT ? BN : KT) + VE;   // row pitches (elements)
    constexpr int A_ROWS = AT ? KT : BM, B_ROWS = BT ? KT : BN;           // LDS rows of a panel's stage
    constexpr int A_BYTES = A_ROWS * LDA * ES, B_BYTES = B_ROWS * LDB * ES;
    constexpr int BUF = A_BYTES + B_BYTES;
    constexpr int CA = (AT ? BM : KT) / VE, CB = (BT ? BN : KT) / VE;     // 16-byte chunks per row
    constexpr int NA = A_ROWS * CA, NB = B_ROWS * CB;
    constexpr int NVA = (NA + 255) / 256, NVB = (NB + 255) / 256;         // chunks per thread
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    extern __shared__ __align__(16) char smem[];

    const int L = blockIdx.x;
    if (L >= s.n_product) {
        dds_colsum_range<T>(p, s, L - s.n_product, reinterpret_cast<float*>(smem));
        return;
    }
    // which block, which range of k: a slice has 8 / slices XCDs of its own, which take contiguous
    // ranges of the BCSR order (bands of block rows: an A panel is read by one of them)
    const int nnz = p.nnz_dev ? p.nnz_dev[0] : s.nnz;
    int i, slice;
    {
        const int x = L & 7, t = L >> 3;
        if (s.slices == 8) {
            i = t;
            slice = x;
        } else {
            const int share = 8 / s.slices;
            const int chunk = (nnz + share - 1) / share;
            if (t >= chunk) return;
            i = (x & (share - 1)) * chunk + t;
            slice = x / share;
        }
    }
    if (i >= nnz) return;
    const int k_begin = slice * s.k_slice;
    const int k_end = k_begin + s.k_slice < p.K ? k_begin + s.k_slice : p.K;
    const int64_t b = blockIdx.y;
    const int lane = lane_id();
    const int wave = threadIdx.x >> 6;
    const int r16 = lane & 15;
    const int g4 = lane >> 4;
    const int wt = wave % (W::WGM * W::WGN);
    const int kpart = wave / (W::WGM * W::WGN);
    const int wgm = wt / W::WGN;
    const int wgn = wt % W::WGN;

    // staging map: chunk v = tid + 256 u of a panel's stage is (row, 16-byte piece)
    int a_kofs[NVA], a_dst[NVA], b_kofs[NVB], b_dst[NVB];   // first k inside the stage (KT and more: no chunk), LDS place
    int64_t a_src[NVA], b_src[NVB];                         // elements from the panel's origin
#pragma unroll
    for (int u = 0; u < NVA; ++u) {
        const int v = threadIdx.x + 256 * u, w = v < NA ? v : 0;
        const int r = w / CA, c = w % CA;
        a_src[u] = (int64_t)r * p.a_ld + c * VE;
        a_kofs[u] = v < NA ? (AT ? r : c * VE) : (1 << 30);
        a_dst[u] = (r * LDA + c * VE) * ES;
    }
#pragma unroll
    for (int u = 0; u < NVB; ++u) {
        const int v = threadIdx.x + 256 * u, w = v < NB ? v : 0;
        const int r = w / CB, c = w % CB;
        b_src[u] = (int64_t)r * p.b_ld + c * VE;
        b_kofs[u] = v < NB ? (BT ? r : c * VE) : (1 << 30);
        b_dst[u] = A_BYTES + (r * LDB + c * VE) * ES;
    }
    // fragment bases inside a buffer (bytes)
    const int a_tr = ((g4 * 8 + (r16 >> 2)) * LDA + (wgm * W::WTM * 16 + (r16 & 3) * 4)) * ES;
    const int b_tr = A_BYTES + ((g4 * 8 + (r16 >> 2)) * LDB + (wgn * W::WTN * 16 + (r16 & 3) * 4)) * ES;
    const int a_f32 = ((g4 * 4) * LDA + wgm * W::WTM * 16 + r16) * ES;
    const int b_f32 = A_BYTES + ((g4 * 4) * LDB + wgn * W::WTN * 16 + r16) * ES;
    // k-contiguous parts: row r16 of the wavefront's first tile, element 0 of the row
    const int a_row = ((wgm * W::WTM * 16 + r16) * LDA) * ES;
    const int b_row = A_BYTES + ((wgn * W::WTN * 16 + r16) * LDB) * ES;
    const int n_st = (k_end - k_begin + KT - 1) / KT;   // 0 or less: an empty slice at the end
    // unsliced: the XCDs start at staggered depths (rows are often a power of two apart, and
    // eight XCDs walking in step would keep hitting the same memory channels)
    const int rot = s.slices > 1 ? 0 : (int)(((int64_t)(L & 7) * n_st) >> 3);
    auto stage_k = [&](int st) {   // first k of the st-th stage of the walk (clamped past the end)
        int t = (st < n_st ? st : n_st - 1) + rot;
        t = t >= n_st ? t - n_st : t;
        return k_begin + t * KT;
    };

    const int code = p.idx[i];
    const int bi = (code >> 16) & 0xffff;
    const int bj = code & 0xffff;
    const T* A = reinterpret_cast<const T*>(p.A) + b * p.a_batch + (int64_t)bi * BM * (AT ? 1 : p.a_ld);
    const T* B = reinterpret_cast<const T*>(p.B) + b * p.b_batch + (int64_t)bj * BN * (BT ? 1 : p.b_ld);

    f32x4 acc[W::WTM][W::WTN];
#pragma unroll
    for (int x = 0; x < W::WTM; ++x)
#pragma unroll
        for (int y = 0; y < W::WTN; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};

    u32x4 ring_a[NST][NVA], ring_b[NST][NVB];
    auto load = [&](int k0, u32x4 (&ra)[NVA], u32x4 (&rb)[NVB]) {
        const bool whole = k0 + KT <= k_end;
        const int64_t ak = (int64_t)k0 * (AT ? p.a_ld : 1), bk = (int64_t)k0 * (BT ? p.b_ld : 1);
        // a chunk past the end of the range re-reads the panel's first bytes
#pragma unroll
        for (int u = 0; u < NVA; ++u) {
            const bool in = a_kofs[u] < KT && (whole || k0 + a_kofs[u] < k_end);
            ra[u] = *reinterpret_cast<const u32x4*>(A + (in ? ak + a_src[u] : 0));
        }
#pragma unroll
        for (int u = 0; u < NVB; ++u) {
            const bool in = b_kofs[u] < KT && (whole || k0 + b_kofs[u] < k_end);
            rb[u] = *reinterpret_cast<const u32x4*>(B + (in ? bk + b_src[u] : 0));
        }
    };
    if (n_st > 0) {
#pragma unroll
        for (int r = 0; r < NST; ++r) load(stage_k(r), ring_a[r], ring_b[r]);
    }
    for (int it = 0; it < n_st; it += NST) {
#pragma unroll
        for (int r = 0; r < NST; ++r) {
            const int st = it + r;
            char* buf = smem + (st & 1) * BUF;
            if (st < n_st) {
                const int k0 = stage_k(st);
                if (k0 + KT > k_end) {   // the short last stage: zeros past the end
#pragma unroll
                    for (int u = 0; u < NVA; ++u)
                        if (k0 + a_kofs[u] >= k_end) ring_a[r][u] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                    for (int u = 0; u < NVB; ++u)
                        if (k0 + b_kofs[u] >= k_end) ring_b[r][u] = u32x4{0u, 0u, 0u, 0u};
                }
#pragma unroll
                for (int u = 0; u < NVA; ++u)
                    if (NA % 256 == 0 || a_kofs[u] < KT) *reinterpret_cast<u32x4*>(buf + a_dst[u]) = ring_a[r][u];
#pragma unroll
                for (int u = 0; u < NVB; ++u)
                    if (NB % 256 == 0 || b_kofs[u] < KT) *reinterpret_cast<u32x4*>(buf + b_dst[u]) = ring_b[r][u];
            }
            // refill the slot; nothing past the end (with copies there instead a slice of eight stages read a fifth too much:
            // 62.5 against 61.1 us on the weight gradient of 4096 x 3072 -> 768 fp32 at 20 %)
            if (st + NST < n_st) load(stage_k(st + NST), ring_a[r], ring_b[r]);
            if (st < n_st) {
                __syncthreads();
                if constexpr (HasMma32<T>::value) {
                    typedef typename Mma32<T>::frag Frag;
                    auto frag_tr = [&](const char* at, int pitch) {
                        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at));
                        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at + 4 * pitch));
                        return __builtin_bit_cast(Frag, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                    };
#pragma unroll
                    for (int kc = 0; kc < KW; kc += 32) {
                        const int kb = kpart * KW + kc;
                        Frag af[W::WTM], bf[W::WTN];
#pragma unroll
                        for (int x = 0; x < W::WTM; ++x)
                            af[x] = AT ? frag_tr(buf + a_tr + (kb * LDA + x * 16) * ES, LDA * ES)
                                       : Mma32<T>::load(reinterpret_cast<const T*>(buf + a_row) + x * 16 * LDA + kb + g4 * 8);
#pragma unroll
                        for (int y = 0; y < W::WTN; ++y)
                            bf[y] = BT ? frag_tr(buf + b_tr + (kb * LDB + y * 16) * ES, LDB * ES)
                                       : Mma32<T>::load(reinterpret_cast<const T*>(buf + b_row) + y * 16 * LDB + kb + g4 * 8);
#pragma unroll
                        for (int x = 0; x < W::WTM; ++x)
#pragma unroll
                            for (int y = 0; y < W::WTN; ++y) acc[x][y] = Mma32<T>::mma(af[x], bf[y], acc[x][y]);
                    }
                } else {
                    typedef typename Mma16<T>::frag Frag;
                    auto frag_rows = [&](const char* at, int pitch) {
                        Frag f;
#pragma unroll
                        for (int j = 0; j < 4; ++j) f[j] = *reinterpret_cast<const float*>(at + j * pitch);
                        return f;
                    };
#pragma unroll
                    for (int kc = 0; kc < KW; kc += 16) {
                        const int kb = kpart * KW + kc;
                        Frag af[W::WTM], bf[W::WTN];
#pragma unroll
                        for (int x = 0; x < W::WTM; ++x)
                            af[x] = AT ? frag_rows(buf + a_f32 + (kb * LDA + x * 16) * ES, LDA * ES)
                                       : Mma16<T>::load(reinterpret_cast<const T*>(buf + a_row) + x * 16 * LDA + kb + g4 * 4);
#pragma unroll
                        for (int y = 0; y < W::WTN; ++y)
                            bf[y] = BT ? frag_rows(buf + b_f32 + (kb * LDB + y * 16) * ES, LDB * ES)
                                       : Mma16<T>::load(reinterpret_cast<const T*>(buf + b_row) + y * 16 * LDB + kb + g4 * 4);
#pragma unroll
                        for (int x = 0; x < W::WTM; ++x)
#pragma unroll
                            for (int y = 0; y < W::WTN; ++y) acc[x][y] = Mma16<T>::mma(af[x], bf[y], acc[x][y]);
                    }
                }
            }
        }
    }
    __syncthreads();  // all fragments are consumed before the buffers are reused
    float* Ef = reinterpret_cast<float*>(smem);
    if (s.slices == 1) {
        dds_epilogue<T, BM, BN>(p, acc, Ef, i, bi, bj, b, wgm, wgn, kpart, r16, g4);
        return;
    }
    // partial block: through LDS (one copy per k part) to whole 16-byte vectors
    constexpr int LDE = BN + 4;
#pragma unroll
    for (int x = 0; x < W::WTM; ++x)
#pragma unroll
        for (int y = 0; y < W::WTN; ++y)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                Ef[(kpart * BM + (wgm * W::WTM + x) * 16 + g4 * 4 + q) * LDE + (wgn * W::WTN + y) * 16 + r16] = acc[x][y][q];
    __syncthreads();
    float* dstp = s.partial + ((b * s.slices + slice) * s.nnz + i) * (int64_t)(BM * BN);
    for (int v = threadIdx.x; v < BM * BN / 4; v += 256) {
        const int m = v / (BN / 4), n = v % (BN / 4) * 4;
        f32x4 sum = *reinterpret_cast<const f32x4*>(Ef + m * LDE + n);
#pragma unroll
        for (int kp = 1; kp < W::KS; ++kp) sum += *reinterpret_cast<const f32x4*>(Ef + (kp * BM + m) * LDE + n);
        store16_through(dstp + v * 4, __builtin_bit_cast(vec16, sum));
    }
}

// Adds the partial blocks in slice order, and the column sums of A in range order.
template <typename T>
__global__ __launch_bounds__(256) void dds_split_reduce_kernel(DdsParams p, DdsSplit s, T* colsum, int BM, int BN, int n_product) {
    const int64_t b = blockIdx.y;
    if ((int)blockIdx.x >= n_product) {
        const int col = ((int)blockIdx.x - n_product) * 256 + threadIdx.x;
        if (col >= p.M) return;
        float sum = 0.f;
#pragma unroll 8
        for (int r = 0; r < kColsumSlices; ++r) sum += s.colsum[(b * kColsumSlices + r) * p.M + col];
        colsum[b * p.M + col] = Elem<T>::from_float(sum);
        return;
    }
    const int64_t total = (int64_t)s.nnz * BM * BN;
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (at >= total) return;
    const float* src = s.partial + b * s.slices * total + at;
    f32x4 sum = *reinterpret_cast<const f32x4*>(src);
#pragma unroll 7
    for (int r = 1; r < s.slices; ++r) sum += *reinterpret_cast<const f32x4*>(src + r * total);
    int64_t off = at;
    if (!p.compressed) {
        const int i = (int)(at / (BM * BN)), in = (int)(at % (BM * BN));
        const int code = p.idx[i];
        off = ((int64_t)((code >> 16) & 0xffff) * BM + in / BN) * p.N + (int64_t)(code & 0xffff) * BN + in % BN;
    }
    T vals[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) vals[q] = Elem<T>::from_float(sum[q]);
    T* dst = reinterpret_cast<T*>(p.C) + b * p.c_batch + off;
    if constexpr (sizeof(T) == 2) *reinterpret_cast<uint64_t*>(dst) = *reinterpret_cast<const uint64_t*>(vals);
    else *reinterpret_cast<vec16*>(dst) = *reinterpret_cast<const vec16*>(vals);
}

// Depth of a stage for a block shape.
inline int dds_split_stage(int elem_bytes, int BM, int BN) {
    return elem_bytes == 2 ? (BM + BN <= 32 ? 128 : 64) : (BM + BN <= 64 ? 64 : 32);
}

// How many slices.  The estimate (microseconds) follows what was measured on weights of 512 x 768 to
// 4096 x 4096 with 77 to 4915 live blocks and 80 to 8192 tokens:
//   * operand traffic, nnz * K * (BM + BN) elements.  The more slices, the fewer XCDs read the same
//     bytes; k-contiguous operands and panel rows of 128 bytes fill the cache lines they touch:
//     the rates of the table below;
//   * or the walk over the stages, 0.5 us each and 1.5 us around them, times the generations of
//     five workgroups per CU;
//   * a split adds a launch (2.5 us) and writes and reads the partial blocks at 4 TB/s.
//   * the partial blocks of a call take at most 1 GB.  That bounds what a training step needs beyond its tensors
//     (without a bound it grows to 16 times the 16-bit gradient), and only very large weights meet it: 26221 blocks of
//     32 x 64 over 8192 tokens fp16 6214 / 5129 / 3910 / 3744 us with 1 / 2 / 4 / 8 slices, which take 0 / 0.4 / 0.9 /
//     1.7 GB; 26151 of 32 x 32 keep eight slices (2741 us and 0.86 GB against 3318 with four).
// e.g. 115 blocks of 32 x 64 over 2992 tokens 25.0 / 16.7 / 13.3 / 14.6 us with 1 / 2 / 4 / 8 slices;
// 819 of 32 x 32 over 4096 57 / 57 / 50 / 47 us; 248 of 32 x 32 over 704 6.7 / 8.7 / 9.9 / 12.4 us.
inline int dds_split_slices(int elem_bytes, bool kcontig, int nnz, int batch, int K, int BM, int BN) {
    const double blocks = (double)nnz * batch;
    const int stage = dds_split_stage(elem_bytes, BM, BN);
    const double traffic = blocks * K * (BM + BN) * elem_bytes;
    static const double rates[3][4] = {{7.2e6, 8.6e6, 10.2e6, 12.2e6},      // bytes per us: half-line rows
                                       {8.4e6, 13.0e6, 14.0e6, 17.0e6},     // rows of 128 bytes and more
                                       {11.5e6, 14.0e6, 17.5e6, 23.0e6}};   // k-contiguous
    const double* rate = rates[kcontig ? 2 : (BM * elem_bytes >= 128 && BN * elem_bytes >= 128 ? 1 : 0)];
    int best = 1;
    double best_us = 0;
    for (int l = 0; l < 4; ++l) {
        const int S = 1 << l;
        if (S > 1 && S * blocks * BM * BN * sizeof(float) > (double)kSplitPartialBytes) break;
        const double move = traffic / rate[l];
        const double stages = (double)((K + S * stage - 1) / (S * stage));
        const double generations = blocks * S <= 1280 ? 1.0 : blocks * S / 1280;
        const double walk = (stages * 0.5 + 1.5) * generations;
        const double us = (move > walk ? move : walk) + (S > 1 ? 2.5 + S * blocks * BM * BN * 8 / 4e6 : 0.0);
        if (l == 0 || us < best_us) { best = S; best_us = l == 0 ? 0.95 * us : us; }
    }
    return best;
}

// The second launch: partial blocks and ranges of the column sums, where there are any.
template <typename T>
static int launch_dds_split_reduce(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st) {
    const int n_blocks = s.slices > 1 ? (int)(((int64_t)s.nnz * BM * BN / 4 + 255) / 256) : 0;
    const int n_cols = s.colsum ? (p.M + 255) / 256 : 0;
    if (n_blocks + n_cols == 0) return 0;
    hipLaunchKernelGGL((dds_split_reduce_kernel<T>), dim3(n_blocks + n_cols, batch, 1), dim3(256), 0, st, p, s,
                       reinterpret_cast<T*>(colsum), BM, BN, n_blocks);
    SPX_LAUNCH_CHECK("dds_split_reduce_kernel");
    return 0;
}

template <typename T, int BM, int BN, bool AT, bool BT>
static int launch_dds_split_inst(const DdsParams& p, DdsSplit s, void* colsum, int batch, hipStream_t st) {
    constexpr int VE = 16 / (int)sizeof(T);
    constexpr int KT = DdsSplitCfg<T, BM, BN>::KT;
    typedef DdsWaveGrid<BM / 16, BN / 16> W;
    constexpr size_t a_part = AT ? (size_t)KT * (BM + VE) : (size_t)BM * (KT + VE);
    constexpr size_t b_part = BT ? (size_t)KT * (BN + VE) : (size_t)BN * (KT + VE);
    constexpr size_t stages = 2 * (a_part + b_part) * sizeof(T);
    constexpr size_t epi = (size_t)W::KS * BM * (BN + 4) * sizeof(float);
    constexpr size_t cs = 32 * (8 * VE + 4) * sizeof(float);   // the column sums
    constexpr size_t product = epi > stages ? epi : stages, most = cs > product ? cs : product;
    const bool sums = s.colsum || s.colsum_out;
    const size_t smem = sums ? most : product;
    s.k_slice = (int)round_up((p.K + s.slices - 1) / s.slices, KT);
    const int share = 8 / s.slices;
    const int64_t n_product = ((int64_t)s.nnz + share - 1) / share * 8;
    const int64_t cs_groups = sums ? (int64_t)(p.M + 8 * VE - 1) / (8 * VE) * (s.colsum_out ? 1 : kColsumSlices) : 0;
    if (n_product + cs_groups > 0x7fffffff) return fail(SPX_E_SHAPE, "too many workgroups (%lld)", (long long)(n_product + cs_groups));
    if (n_product + cs_groups == 0) return 0;
    s.n_product = (int)n_product;
    SPX_GRANT_LDS((dds_split_kernel<T, BM, BN, AT, BT>), most, "dds_split_kernel");
    hipLaunchKernelGGL((dds_split_kernel<T, BM, BN, AT, BT>), dim3((unsigned)(n_product + cs_groups), batch, 1), dim3(256), smem, st, p, s);
    SPX_LAUNCH_CHECK("dds_split_kernel");
    return launch_dds_split_reduce<T>(p, s, colsum, BM, BN, batch, st);
}

// Blocks of a block-row to a workgroup, which then share their rows of A (0: one block to a workgroup), and the slices of k.
struct DdsShare {
    int blocks, slices;
};

// Scores (both operands k-contiguous), fp32 32 x 32: two blocks to a workgroup from 1000 of them on, in the slices that one block
// to a workgroup has (2458 blocks over 1536 in four 97.9 / 82.5 us, over 3072 in eight 186 / 153 with a relative error of
// 3.5e-7; unsliced and shared 70.6 and 136, but 7.0e-7 and 9.9e-7), where that saves rounds: the workgroups that are on a CU together
// take as long as their number says, a pair of blocks 1.33 times a single one and a little at the start.  us over 768, one block
// / shared: 1024 blocks (four and three rounds) 20.8 / 24.5, 1100 (five, three) 25.1 / 24.5, 1400 (six, three) 28.5 / 24.8,
// 1536 (six, four) 28.9 / 30.5, 1700 (seven, four) 32.6 / 30.9, 2048 (eight, five) 37.3 / 36.9, 2458 51 / 43.5, 2700 (eleven, six) 49.2 / 42.0;
// over 256 the pair is ahead sooner: 1536 14.5 / 13.5, but 1024 10.2 / 10.9.  Many short block-rows, whose last group is not full,
// count as they are launched: 4 x 300 blocks in 96 block-rows each (five, four) 26.3 / 31.0.  Fewer blocks: 388 over 768 14.5 / 15.7.
// 64 x 64: 396 over 768 34.3 / 33.2.
inline bool dds_scores_share(int elem_bytes, int nnz, int batch, int M, int K, int BM, int BN, int slices) {
    if (elem_bytes != 4 || BM != 32 || BN != 32 || (int64_t)nnz * batch < 1000) return false;
    const int64_t rows = M / BM < nnz ? M / BM : nnz, groups = (nnz + rows) / 2;   // as launch_dds_share_inst launches them
    const int64_t one = ((int64_t)nnz * batch * slices + 255) / 256, shared = (groups * batch * slices + 255) / 256;
    return 4 * shared + (K > 512 ? 3 : 2) <= 3 * one;
}

// Weight gradients (both operands k-major).  Estimates in us of product and second kernel, fitted to 1000 random problems of 512 to
// 4096 rows and columns, 256 to 8192 tokens and 2 - 40 % live blocks (root mean square off by 2 - 8 %):
//   start + sliced ? second + partial * (bytes of the partial blocks, written and read, at 4 TB/s) : 0
//         + thousands of tokens in a slice * (depth + rounds * ceil(W) + work * W + generation * ceil(W / fit))
// W: workgroups to a CU, fit: that are there together.
struct DdsEstimate {
    int elem_bytes, BM, BN, blocks, fit;   // blocks to a workgroup
    double start, second, partial, depth, rounds, work, generation;
};
inline double dds_estimate(const DdsEstimate& e, double blocks, double rows, int K, int slices) {
    // a block-row's last group is half full, give or take
    const double groups = (blocks + rows * (e.blocks - 1) * 0.5) / e.blocks, per_cu = groups * slices / 256;
    const double part = slices > 1 ? e.second + e.partial * slices * blocks * e.BM * e.BN * 8 / 4e6 : 0.0;
    return e.start + part + (double)K / slices * 1e-3 * (e.depth + e.rounds * std::ceil(per_cu) + e.work * per_cu + e.generation * std::ceil(per_cu / e.fit));
}

// From how many blocks times tokens on they are looked at (below, the many short chains of one block each are ahead), and what
// is taken then.  us with one block to a workgroup / with four or two, at the slices that the estimates choose:
//   16-bit 32 x 32  653 blocks over 1152 11.9 / 14.4 (in four slices, as all of them once were, 16.6), but 450 over 2416 21.1 / 15.7;
//                   fewer than 100 level or behind (71 over 7888 13.9 / 14.8)
//   16-bit 32 x 64  1077 over 1280 24.2 / 19.8 (four slices 30.9), 410 over 4096 33.6 / 28.5, but 64 over 2480 10.5 / 10.7
//   16-bit 64 x 64  691 over 1360 21.6 / 19.4 (four slices 33.1), but 126 over 5552 21.9 / 24.7
//   fp32 32 x 32    504 over 4736 70.2 / 64.9 (four blocks 84.5), 898 over 4144 125 / 96, but 253 over 2096 25.0 / 26.5
//   fp32 32 x 64    210 over 2544 39.9 / 36.3, but 128 over 6032 43.5 / 50.4
//   fp32 16 x 16    1270 over 5328 80.8 / 59.4, 1980 over 1856 50.0 / 38.2, 3074 over 336 (unsliced) 16.6 / 14.6, but 1229 over 768 14.9 /
//                   16.4, 31 over 4000 9.1 / 13.2: a line, without estimates
// Slices: for 16-bit types no fewer than one block to a workgroup has, so that no chain of fp32 additions is longer.  fp32 keeps
// four or eight, whose sums are the more exact ones, also where one block in fewer slices would be ahead (2462 blocks over 1056 in
// eight 92 us, in two 79).
inline DdsShare dds_share_plan(int elem_bytes, bool a_kcontig, bool b_kcontig, int nnz, int batch, int M, int K, int BM, int BN) {
    static const DdsEstimate estimates[] = {
        {2, 32, 32, 1, 5, 4.71, 2.42, 0.56, 0.42, 0.71, 1.10, 2.48}, {2, 32, 32, 4, 4, 7.06, 0.00, 0.72, 1.49, 1.71, 1.98, 2.57},
        {2, 32, 64, 1, 5, 5.20, 2.15, 0.53, 1.62, 1.38, 0.93, 1.80}, {2, 32, 64, 2, 4, 4.71, 2.25, 0.65, 0.75, 1.25, 1.53, 4.19},
        {2, 64, 64, 1, 5, 4.50, 2.09, 0.52, 2.44, 2.90, 0.51, 0.35}, {2, 64, 64, 2, 3, 5.36, 2.20, 0.65, 1.05, 0.66, 2.39, 5.35},
        {4, 32, 32, 1, 5, 6.49, 0.00, 1.05, 3.48, 3.89, 1.55, 0.00}, {4, 32, 32, 2, 6, 7.69, 0.00, 0.76, 0.00, 6.91, 0.69, 6.08},
        {4, 32, 32, 4, 4, 7.24, 0.00, 0.88, 0.00, 11.77, 2.38, 9.50},
        {4, 32, 64, 1, 5, 6.06, 0.00, 0.63, 6.51, 9.38, 0.33, 0.50}, {4, 32, 64, 2, 4, 8.07, 0.00, 0.59, 0.37, 12.51, 2.33, 8.01}};
    DdsShare plan = {0, dds_split_slices(elem_bytes, a_kcontig && b_kcontig, nnz, batch, K, BM, BN)};
    if (a_kcontig != b_kcontig) return plan;
    if (a_kcontig) {
        if (dds_scores_share(elem_bytes, nnz, batch, M, K, BM, BN, plan.slices)) plan.blocks = 2;
        return plan;
    }
    const int64_t blocks = (int64_t)nnz * batch, work = blocks * K;
    const auto fits = [&](int slices) { return slices * (double)blocks * BM * BN * sizeof(float) <= (double)kSplitPartialBytes; };
    int least = plan.slices;
    if (elem_bytes == 4 && BM == 16 && BN == 16) {
        if (work < 1000000) return plan;
        least = K < 1024 ? 1 : blocks <= 2048 ? 8 : 4;
    } else if (elem_bytes == 4 && BM == 32 && BN == 32) {
        if (K < 1024 || work < 800000) return plan;
        least = work < 1500000 ? 4 : 8;
    } else if (elem_bytes == 4 && BM == 32 && BN == 64) {
        if (K < 1024 || work < 500000) return plan;
        least = 4;
    } else if (!(elem_bytes == 2 && ((BM == 32 && BN == 32 && K >= 1024 && work >= 400000 && blocks >= 100) || (BM == 32 && BN == 64 && K >= 1024 && work >= 800000) ||
                                     (BM == 64 && BN == 64 && work >= 600000)))) {
        return plan;
    }
    if (least < plan.slices) least = plan.slices;
    while (least > 1 && !fits(least)) least /= 2;
    if (BM == 16) return {4, least};
    const double rows = (double)(M / BM < nnz ? M / BM : nnz) * batch;
    double best = 0;
    plan.blocks = -1;
    for (const DdsEstimate& e : estimates)
        if (e.elem_bytes == elem_bytes && e.BM == BM && e.BN == BN)
            for (int slices = least; slices <= 8 && (slices == least || fits(slices)); slices *= 2) {
                const double us = dds_estimate(e, (double)blocks, rows, K, slices);
                if (plan.blocks < 0 || us < best) {
                    best = us;
                    plan = {e.blocks == 1 ? 0 : e.blocks, slices};
                }
            }
    return plan;
}

template <typename T>
int launch_dds_share(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st);
template <typename T>
bool dds_share_takes(const DdsParams& p) {   // (byte offsets of 64 rows in 32 bits)
    return p.row_ptr && !p.bias && p.a_ld < (1 << 23) && p.b_ld < (1 << 23);
}
// Blocks to a workgroup of an unsliced product of spx_matmul, 0: one each.  (Several long scores outgrow the L2s side by side: 4 x 550
// blocks over 2048 103 / 123 us, 4 x 450 91 / 103, but 1536 of a single product 69 / 72 and 2048 of one 90 / 88.  Weight gradients that the
// plan does not slice come here where no column sums are wanted: 2409 16-bit blocks of 32 x 32 over 2048 51 / 36.)
template <typename T>
int dds_shared_blocks(const DdsParams& p, int BM, int BN, int nnz_bound, int batch) {
    if (p.a_kcontig != p.b_kcontig || !dds_share_takes<T>(p)) return 0;
    if (p.a_kcontig) return (batch == 1 || p.K <= 1024) && dds_scores_share((int)sizeof(T), nnz_bound, batch, p.M, p.K, BM, BN, 1) ? 2 : 0;
    const DdsShare plan = dds_share_plan((int)sizeof(T), false, false, nnz_bound, batch, p.M, p.K, BM, BN);
    return plan.slices == 1 ? plan.blocks : 0;
}

template <typename T>
int launch_dds_split_impl(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st) {
    if (s.share && dds_share_takes<T>(p)) return launch_dds_share<T>(p, s, colsum, BM, BN, batch, st);
#define SPX_DDS_SPLIT_CASE(bm, bn)                                                                                  \
    if (BM == bm && BN == bn)                                                                                       \
        return !p.a_kcontig && !p.b_kcontig ? launch_dds_split_inst<T, bm, bn, true, true>(p, s, colsum, batch, st) \
             : p.a_kcontig && !p.b_kcontig  ? launch_dds_split_inst<T, bm, bn, false, true>(p, s, colsum, batch, st) \
             : !p.a_kcontig                 ? launch_dds_split_inst<T, bm, bn, true, false>(p, s, colsum, batch, st) \
                                            : launch_dds_split_inst<T, bm, bn, false, false>(p, s, colsum, batch, st);
    SPX_DDS_SPLIT_CASE(16, 16) SPX_DDS_SPLIT_CASE(16, 32) SPX_DDS_SPLIT_CASE(16, 64)
    SPX_DDS_SPLIT_CASE(32, 16) SPX_DDS_SPLIT_CASE(32, 32) SPX_DDS_SPLIT_CASE(32, 64)
    SPX_DDS_SPLIT_CASE(64, 16) SPX_DDS_SPLIT_CASE(64, 32) SPX_DDS_SPLIT_CASE(64, 64)
#undef SPX_DDS_SPLIT_CASE
    return fail(SPX_E_CONFIG, "output block (%d,%d) not in {16,32,64}^2", BM, BN);
}

template <typename T>
int launch_dds_split(const DdsParams& p, const DdsSplit& s, void* colsum, int BM, int BN, int batch, hipStream_t st);

}  // namespace spx
