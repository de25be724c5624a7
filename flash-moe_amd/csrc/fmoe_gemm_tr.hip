// Products of the backward passes whose operands do not lie K-contiguous, for gfx950:
//   NN   C[M,N] = A[M,K] B[K,N]          (dh = dy Wd, dx = [da | db] [Wg; Wu], dq = d Wr)
//   TN   C[M,N] = A[K,M]^T B[K,N]        (the weight gradients)
// They run on the LDS pipeline of the forward's products (fmoe_gemm.h): a turned operand is brought into the LDS as it lies, k-row by
// k-row, and turned on the way to the matrix cores, in the 16-bit types by the LDS itself (ds_read_b64_tr_b16), in fp32 because a
// lane reads its k values one by one.  Operands that are not whole 16-byte packets go to the library.
//
// What bounds it is what bounds the forward's products: what a compute unit receives on small tiles, the matrix pipes on 256 x 256
// (fmoe_gemm256.h),
// and, with few tiles and a long k loop, the length of one chain, which slices of k cut (their sums are added by a second launch, in
// slice order).  A kernel that turned the operands in registers reached 600 TFLOP/s in bf16 where these reach 1000 to 1300.
//
// Against the library's kernels (rocBLAS), us:
//   bf16  2048 tokens, 4096 -> 16384: dh 187 for 203, dx 414 for 502, dWd 213 for 258, dWg and dWu 418 for 512; 4096 tokens, 1024 -> 4096:
//         31 for 33, 71 for 79, 39 for 45, 62 for 69; 615 tokens, 776 -> 2072: 8 for 17, 20 for 36, 7 for 17, 11 for 18; 32768 tokens, 2048
//         -> 8192: 871 for 871, 1501 for 1648, 783 for 944, 1613 for 1891.  Before the waves of a 256 x 256 tile worked in two groups
//         (fmoe_gemm256.h): 2048 tokens 206, 442, 221, 438; 8192 tokens of 2048 -> 8192 223, 406, 199, 428 for 198, 370, 193, 409 now.
//   fp32  383 tokens, 1880 -> 7520: dh 97 for 88, dx 200 for 828, dWd 100 for 105, dWg and dWu 191 for 218; 1000 tokens, 1024 -> 4096: 71
//         for 64, 136 for 120, 69 for 71, 125 for 152; 4096 tokens, 1024 -> 4096: 257 for 242, 520 for 460, 260 for 231, 479 for 455; 5000
//         tokens, 2048 -> 5464: 897 for 812, 1791 for 2426, 867 for 1094, 1746 for 1913; 16384 tokens, 512 -> 2048: 258 for 246, 488 for
//         913, 259 for 235, 516 for 788.  At 120 to 143 TFLOP/s these kernels are 5 to 15 % behind the library's best and far ahead of what
//         it takes at other extents; over the backward passes of 16 extents 21.0 ms for 25.0, the worst of them 9 % longer (4096 tokens).
//         Products of less than a round of tiles take up to 3 us longer (dq of 600 tokens, 256 -> 256: 7.6 for 6.1).
#include "fmoe_common.h"
#include "fmoe_gemm.h"
#include "fmoe_gemm256.h"
#include "fmoe_vec.h"

namespace fmoe {
namespace {

// SLICED: each XCD takes a run of slice * tiles + tile, so that it fetches its slices' part of the operands only, sums to plane `slice` of C
// (fp32).  dx of 615 tokens, 2072 -> 776 in six slices of 35 tiles 17.5 -> 14 us with both operands far from the compute units.
template <typename T, bool TA, int BM, int BN, int WAVES_N, int NSTAGE, bool SLICED>
__global__ __launch_bounds__(2 * WAVES_N * kWave) void gemm_turned_kernel(
    const T* __restrict__ A, int lda, const T* __restrict__ B0, const T* __restrict__ B1, int ldb, T* __restrict__ C, int M, int N, int K,
    int segments, int tiles_m, int tiles_n, int xcds, int slices) {
    const int tiles = tiles_m * tiles_n, block = SLICED ? xcd_run((int)blockIdx.x, (int)gridDim.x, xcds) : (int)blockIdx.x;
    gemm_dma_tiles<T, BM, BN, 2, WAVES_N, kStageK<T>, NSTAGE, SLICED ? kEpiPart : kEpiPlain, kSmallAhead<T>, kFragRows<T>, true, SLICED,
                   TA, true>(A, B0, B1, C, nullptr, M, N, K, tiles_m, tiles_n, SLICED ? 1 : xcds, SLICED ? block % tiles : block,
                             SLICED ? tiles : (int)gridDim.x, SLICED ? block / tiles : 0, slices, lda, ldb, segments);
}

template <typename T, bool TA, bool SLICED, bool RAGGED>
__global__ __launch_bounds__(kWideThreads, 2) void gemm_wide_turned_kernel(
    const T* __restrict__ A, int lda, const T* __restrict__ B0, const T* __restrict__ B1, int ldb, T* __restrict__ C, int M, int N, int K,
    int segments, int tiles_m, int tiles_n, int xcds, int slices) {
    const int tiles = tiles_m * tiles_n, block = SLICED ? xcd_run((int)blockIdx.x, (int)gridDim.x, xcds) : (int)blockIdx.x;
    gemm_wide_tiles<T, SLICED ? kEpiPart : kEpiPlain, RAGGED, SLICED, TA, true>(
        A, B0, B1, C, nullptr, M, N, K, tiles_m, tiles_n, SLICED ? 1 : xcds, SLICED ? block % tiles : block, SLICED ? tiles : (int)gridDim.x,
        SLICED ? block / tiles : 0, slices, lda, ldb, segments);
}

// C = sum over the slices, in order; one packet of C per thread
template <typename T>
__global__ __launch_bounds__(256) void gemm_turned_add_kernel(const float* __restrict__ planes, T* __restrict__ C, int64_t packets, int slices) {
    constexpr int V = Elem<T>::kVec;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= packets) return;
    float v[V];
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = 0.0f;
    for (int s = 0; s < slices; ++s)
#pragma unroll
        for (int h = 0; h < V; h += 4) {
            const f32x4_t p = *reinterpret_cast<const f32x4_t*>(planes + (s * packets + i) * V + h);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[h + e] += p[e];
        }
    reinterpret_cast<u32x4_t*>(C)[i] = pack16<T>(v);
}

// Tile shape and slices of k by price (us): a round of tiles costs what the forward's rule says, 2.3 ns per received row and k-tile,
// plus the stores of its tiles, which nothing hides on 256 x 256 (7 us; the smaller tiles overlap them with other workgroups);
// slices, as long as they are one round, add a launch of 5 us (fp32 4) and their planes, written and read at 6 TB/s.
// fp32 tiles are bound by the matrix pipes, which two workgroups of a compute unit keep a tenth busier than one (a k-tile of 128 x 128
// 2.0 us for 2.25), so slices of 64 x 64 tiles may be two rounds: dx of 1000 tokens, 1024 -> 4096 156 -> 138 in two slices.  64 x 128 has
// the faults of both its neighbours there and is left out (dx of 2048 tokens 279 for 268 on 64 x 64).
// These prices against 186 products timed in every shape and number of slices (bf16): 2.3 % over the best on average, 3.6 with the
// 256 x 256 tiles at the rate of the forward's and their stores at 8.5; us: dh of 1819 tokens, 1792 -> 4776 52 -> 39, of 4681, 1136 -> 4544
// 74 -> 58, dWd of 19470 tokens, 1704 -> 640 90 -> 60, dx of 1819 tokens, 4776 -> 1792 90 -> 75; the worst, 1536 x 3072 of 2760, 36 -> 45.
template <typename T> SlicePlan plan_turned(int M, int N, int K, int segments) {
    const int cus = chip_info().cus, k_tiles = (K + kStageK<T> - 1) / kStageK<T> * segments;
    SlicePlan best = {kTile64, 1};
    double best_time = 0.0;
    for (int i = sizeof(T) == 4 ? kTile128 : kTile256; i <= kTile64; ++i) {
        int64_t n = 0;
        if (sizeof(T) == 4 && i == kTile64x128) continue;
        const double row = tile_cost<T, kEpiPlain>(i, M, N, n) * 2.3e-3, stores = i == kTile256 ? 7.0 : 1.0;
        const int64_t most = sizeof(T) == 4 && i == kTile64 ? 2 * cus : cus;
        for (int s = 1; s <= kMaxSlices && (s == 1 || (n * s <= most && 2 * s <= k_tiles)); ++s) {
            const int share = (k_tiles + s - 1) / s;
            if ((s - 1) * share >= k_tiles) continue;                 // a slice would have no k-tile
            const double shared = sizeof(T) == 4 && n * s > cus ? 0.9 : 1.0;
            const double time = (double)((n * s + cus - 1) / cus) * (shared * row * share + stores) + (s > 1 ? (sizeof(T) == 4 ? 4.0 : 5.0) + 8.0e-6 * s * (double)M * N / 6.0 : 0.0);
            if (best_time == 0.0 || time < best_time) {
                best = {i, s};
                best_time = time;
            }
        }
    }
    return best;
}

template <typename T, bool TA>
void launch_turned(const void* A, int lda, const void* B0, const void* B1, int ldb, void* C, int M, int N, int K, int segments, SlicePlan p,
                   float* planes, hipStream_t stream) {
    const int xcds = chip_info().xcds, cus = chip_info().cus;
    const int tm = (M + kTileRows[p.shape] - 1) / kTileRows[p.shape], tn = (N + kTileCols[p.shape] - 1) / kTileCols[p.shape];
    const int64_t n = (int64_t)tm * tn;
    // PER: workgroups of a compute unit
#define FMOE_WHOLE(BM, BN, WAVES_N, NSTAGE, PER)                                                                                          \
    hipLaunchKernelGGL((gemm_turned_kernel<T, TA, BM, BN, WAVES_N, NSTAGE, false>), dim3((unsigned)(n < (PER) * cus ? n : (PER) * cus)), \
                       dim3(128 * WAVES_N), 0, stream, (const T*)A, lda, (const T*)B0, (const T*)B1, ldb, (T*)C, M, N, K, segments, tm,  \
                       tn, xcds, 1)
#define FMOE_SLICED(BM, BN, WAVES_N, NSTAGE)                                                                                          \
    hipLaunchKernelGGL((gemm_turned_kernel<T, TA, BM, BN, WAVES_N, NSTAGE, true>), dim3((unsigned)(n * p.slices)), dim3(128 * WAVES_N), \
                       0, stream, (const T*)A, lda, (const T*)B0, (const T*)B1, ldb, (T*)planes, M, N, K, segments, tm, tn, xcds, p.slices)
    if (p.slices > 1) {
        switch (p.shape) {
            case kTile256:
                if constexpr (sizeof(T) == 2)
                    hipLaunchKernelGGL((gemm_wide_turned_kernel<T, TA, true, true>), dim3((unsigned)(n * p.slices)), dim3(kWideThreads), 0, stream, (const T*)A,
                                       lda, (const T*)B0, (const T*)B1, ldb, (T*)planes, M, N, K, segments, tm, tn, xcds, p.slices);
                break;
            case kTile128: FMOE_SLICED(128, 128, 2, 4); break;
            case kTile64x128: if constexpr (sizeof(T) == 2) FMOE_SLICED(64, 128, 2, 4); break;
            default: FMOE_SLICED(64, 64, 2, 4); break;
        }
        const int64_t packets = (int64_t)M * N / Elem<T>::kVec;
        hipLaunchKernelGGL((gemm_turned_add_kernel<T>), dim3((unsigned)((packets + 255) / 256)), dim3(256), 0, stream, (const float*)planes,
                           (T*)C, packets, p.slices);
        return;
    }
    switch (p.shape) {
        case kTile256:
            if constexpr (sizeof(T) == 2) {
                const dim3 grid((unsigned)(n < cus ? n : cus));
                const bool whole = M % kWide == 0 && N % kWide == 0 && K % kWideK == 0 && (K / kWideK * segments) % 2 == 0;
#define FMOE_WIDE(RAGGED)                                                                                                               \
    hipLaunchKernelGGL((gemm_wide_turned_kernel<T, TA, false, RAGGED>), grid, dim3(kWideThreads), 0, stream, (const T*)A, lda, (const T*)B0, \
                       (const T*)B1, ldb, (T*)C, M, N, K, segments, tm, tn, xcds, 1)
                if (whole) FMOE_WIDE(false);
                else FMOE_WIDE(true);
#undef FMOE_WIDE
            }
            break;
        case kTile128:
            if (n <= cus) FMOE_WHOLE(128, 128, 2, 4, 1);
            else FMOE_WHOLE(128, 128, 2, 2, 2);
            break;
        case kTile64x128: if constexpr (sizeof(T) == 2) FMOE_WHOLE(64, 128, 2, 4, 1); break;
        default: FMOE_WHOLE(64, 64, 2, 4, 2); break;
    }
#undef FMOE_SLICED
#undef FMOE_WHOLE
}

}  // namespace

size_t gemm_backward_workspace_bytes(int M, int N, int K, int segments, int dtype) {
    const int slices = (dtype == FMOE_F32 ? plan_turned<float>(M, N, K, segments) : plan_turned<bf16_t>(M, N, K, segments)).slices;
    return slices > 1 ? (size_t)slices * M * N * sizeof(float) : 0;
}

int gemm_backward(int layout, int M, int N, int K, const void* A, int lda, const void* B0, const void* B1, int ldb, void* C, int dtype,
                  void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const int segments = B1 != nullptr ? 2 : 1;
    // whole packets: where M (TN) or K (NN) is none, the rows of A are padded with zeros up to lda
    const int a_cols = layout == kBlasTN ? M : K * segments, vec = dtype == FMOE_F32 ? 4 : 8;
    const bool packets = lda % vec == 0 && ldb % vec == 0 && N % vec == 0 && (a_cols + vec - 1) / vec * vec <= lda &&
                         (segments == 1 || K % vec == 0) && aligned16(A) && aligned16(B0) && aligned16(B1) && aligned16(C);
    // 32-bit byte offsets inside a descriptor
    const double most = dtype == FMOE_F32 ? 5.0e8 : 1.0e9;
    const bool reach = (double)K * ldb < most && (layout == kBlasTN ? (double)K * lda < most : 256.0 * lda < most);
    if (packets && reach) {
        SlicePlan p = dtype == FMOE_F32 ? plan_turned<float>(M, N, K, segments) : plan_turned<bf16_t>(M, N, K, segments);
        if ((size_t)p.slices * M * N * sizeof(float) > workspace_bytes) p.slices = 1;
        float* planes = (float*)workspace;
#define FMOE_TURNED(TT)                                                                                                       \
    do {                                                                                                                      \
        if (layout == kBlasTN) launch_turned<TT, true>(A, lda, B0, B1, ldb, C, M, N, K, segments, p, planes, stream);         \
        else launch_turned<TT, false>(A, lda, B0, B1, ldb, C, M, N, K, segments, p, planes, stream);                          \
    } while (0)
        switch (dtype) {
            case FMOE_F32: FMOE_TURNED(float); break;
            case FMOE_BF16: FMOE_TURNED(bf16_t); break;
            default: FMOE_TURNED(f16_t); break;
        }
#undef FMOE_TURNED
        FMOE_CHECK_LAUNCH("backward product");
        return FMOE_OK;
    }
    if (int rc = blas_gemm(layout, M, N, K, A, lda, B0, ldb, C, N, 0.0f, dtype, stream)) return rc;
    if (B1 == nullptr) return FMOE_OK;
    return blas_gemm(layout, M, N, K, (const char*)A + (size_t)K * dtype_size(dtype), lda, B1, ldb, C, N, 1.0f, dtype, stream);
}

}  // namespace fmoe
