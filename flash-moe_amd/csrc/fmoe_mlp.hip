// Shared SwiGLU MLP for gfx950:  out = (silu(x Wg^T) * (x Wu^T)) Wd^T [+ residual]
//
// Two launches of one MFMA GEMM  C[M,N] = A[M,K] * B[N,K]^T  (both operands K-contiguous, which is how x, the
// nn.Linear weights and the [T,I] activation are laid out, so a lane's 8 consecutive k values for one matrix
// instruction are one 16-byte LDS read):
//   1. gate/up: the B tile holds BN/2 rows of Wg and the same BN/2 rows of Wu, so each wave owns matching gate
//      and up accumulators and the epilogue writes silu(gate)*up, rounded once, to the [T,I] workspace.  The gate
//      and up products never go to memory.
//   2. down: plain epilogue, optional residual add (the routed-expert output in the block).
//
// 256 x 256 tiles of the 16-bit types are gemm_wide_kernel's (fmoe_gemm256.h), 128 x 128 ones that have a compute unit each
// gemm_solo_kernel's (fmoe_gemm128.h).  The other tiles (gemm_dma_kernel; they and those of
// gemm_splitk_kernel are in fmoe_gemm.h) go global -> LDS
// directly (global_load_lds_dwordx4, no staging registers) into NSTAGE LDS stages, issued NSTAGE-1 k-tiles
// ahead of their use; one workgroup barrier per k-tile; MFMA fragments (v_mfma_f32_16x16x32 for the 16-bit types) are
// read with 16-byte ds_reads.  An LDS row is one k-tile of one matrix row; its 16-byte chunks are XOR-swizzled with a key built
// from the row index so that the 16 lanes the 256-byte-per-clock LDS serves per cycle hit 64 different banks.
// Because a DMA load writes 64 consecutive chunks, the swizzle is applied on the global side: each lane fetches
// the chunk that belongs at its LDS position.  Workgroup ids are remapped so that each XCD (ids are dealt
// round-robin over the 8 XCDs) works on a compact patch of the tile grid and shares A/B tiles in its own L2.
//
// fp32 runs the same kernel on v_mfma_f32_32x32x2_f32: an LDS row is again 128 bytes (32 values), a fragment again one
// 16-byte read, and four matrix instructions use it.
//
// Extents that are no multiples of the tile run the same kernel with range-checked buffer loads (RAGGED); few output tiles take
// gemm_splitk_kernel; fp32 whose rows are no multiples of 16 bytes takes a plain FMA kernel.
#include "fmoe_common.h"
#include "fmoe_gemm.h"
#include "fmoe_gemm128.h"
#include "fmoe_gemm256.h"

namespace fmoe {
namespace {

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int BKT, int NSTAGE, int EPI, int PF, int FR, bool RAGGED>
__global__ __launch_bounds__(WAVES_M* WAVES_N * 64) void gemm_dma_kernel(
    const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1, T* __restrict__ C,
    const T* __restrict__ R, int M, int N, int K, int tiles_m, int tiles_n, int xcds) {
    gemm_dma_tiles<T, BM, BN, WAVES_M, WAVES_N, BKT, NSTAGE, EPI, PF, FR, RAGGED>(A, B0, B1, C, R, M, N, K, tiles_m, tiles_n, xcds,
                                                                                         (int)blockIdx.x, (int)gridDim.x);
}

template <typename T, int MT, int NT, int EPI>
__global__ __launch_bounds__(kSplitWaves * 64) void gemm_splitk_kernel(
    const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1, T* __restrict__ C,
    const T* __restrict__ R, int M, int N, int K, int tiles_m, int tiles, int xcds) {
    __shared__ __attribute__((aligned(16))) char lds[kSplitLds<MT, NT, EPI>];
    gemm_splitk_tile<T, MT, NT, EPI>(A, B0, B1, C, R, M, N, K, tiles_m, tiles, xcds, (int)blockIdx.x, (int)gridDim.x, lds);
}

template <typename T, int EPI, bool RAGGED>
__global__ __launch_bounds__(kWideThreads, 2) void gemm_wide_kernel(const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1,
                                                                 T* __restrict__ C, const T* __restrict__ R, int M, int N, int K,
                                                                 int tiles_m, int tiles_n, int xcds) {
    gemm_wide_tiles<T, EPI, RAGGED>(A, B0, B1, C, R, M, N, K, tiles_m, tiles_n, xcds, (int)blockIdx.x, (int)gridDim.x);
}

template <typename T>
__global__ __launch_bounds__(kWideThreads, 2) void gemm_wide_sliced_kernel(const T* __restrict__ A, const T* __restrict__ B, float* __restrict__ planes, int M,
                                                                        int N, int K, int tiles_m, int tiles_n, int xcds, int slices) {
    const int tiles = tiles_m * tiles_n, at = xcd_run((int)blockIdx.x, (int)gridDim.x, xcds);
    gemm_wide_tiles<T, kEpiPart, true, true>(A, B, nullptr, reinterpret_cast<T*>(planes), nullptr, M, N, K, tiles_m, tiles_n, 1, at % tiles,
                                             tiles, at / tiles, slices);
}

// tiles_m * tiles_n workgroups
template <typename T>
__global__ __launch_bounds__(256, 1) void gemm_solo_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, const T* __restrict__ R, int M,
                                                           int N, int K, int tiles_m, int tiles_n, int xcds) {
    __shared__ __attribute__((aligned(1024))) T lds[4 * kSoloStage];
    gemm_solo_tile<T>(A, B, C, R, M, N, K, tiles_m, tiles_n, xcds, (int)blockIdx.x, lds);
}

template <typename T, int BM, int BN, int WAVES_N, int NSTAGE>
__global__ __launch_bounds__(2 * WAVES_N * 64) void gemm_sliced_kernel(const T* __restrict__ A, const T* __restrict__ B, float* __restrict__ planes, int M,
                                                          int N, int K, int tiles_m, int tiles_n, int xcds, int slices) {
    const int tiles = tiles_m * tiles_n, at = xcd_run((int)blockIdx.x, (int)gridDim.x, xcds);
    gemm_dma_tiles<T, BM, BN, 2, WAVES_N, kStageK<T>, NSTAGE, kEpiPart, kSmallAhead<T>, kFragRows<T>, true, true>(
        A, B, nullptr, reinterpret_cast<T*>(planes), nullptr, M, N, K, tiles_m, tiles_n, 1, at % tiles, tiles, at / tiles, slices);
}

// C = sum of the planes in slice order [+ R]; four elements per thread.
template <typename T>
__global__ __launch_bounds__(256) void add_slices_kernel(const float* __restrict__ planes, const T* __restrict__ R, T* __restrict__ C,
                                                         int64_t elements, int slices) {
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (at >= elements) return;
    const bool whole = at + 4 <= elements && elements % 4 == 0;      // planes of a size that keeps 16-byte alignment
    if (whole) {
        f32x4_t sum = *reinterpret_cast<const f32x4_t*>(planes + at);
        for (int s = 1; s < slices; ++s) sum += *reinterpret_cast<const f32x4_t*>(planes + s * elements + at);
        for (int i = 0; i < 4; ++i) C[at + i] = Elem<T>::from_f32(R != nullptr ? sum[i] + Elem<T>::to_f32(R[at + i]) : sum[i]);
    } else {
        for (int64_t e = at; e < at + 4 && e < elements; ++e) {
            float sum = planes[e];
            for (int s = 1; s < slices; ++s) sum += planes[s * elements + e];
            C[e] = Elem<T>::from_f32(R != nullptr ? sum + Elem<T>::to_f32(R[e]) : sum);
        }
    }
}

// fp32 with ragged extents or unaligned tensors (not a tuned kernel): 64x64 tile, 16-deep LDS slabs, 4x4 outputs
// per thread, plain FMA.
template <int EPI>
__global__ __launch_bounds__(256) void sgemm_nt_kernel(const float* __restrict__ A, const float* __restrict__ B0,
                                                       const float* __restrict__ B1, float* __restrict__ C,
                                                       const float* __restrict__ R, int M, int N, int K) {
    constexpr int TS = 64, KS = 16;
    __shared__ float As[KS][TS + 1];
    __shared__ float Bg[KS][TS + 1];
    __shared__ float Bu[(EPI == kEpiSwiGLU) ? KS : 1][TS + 1];
    const int m0 = blockIdx.y * TS, n0 = blockIdx.x * TS;
    const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;
    float accg[4][4] = {}, accu[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += KS) {
        for (int q = threadIdx.x; q < TS * KS; q += 256) {
            const int r = q / KS, kk = q % KS;
            const int gk = k0 + kk;
            As[kk][r] = (m0 + r < M && gk < K) ? A[(int64_t)(m0 + r) * K + gk] : 0.0f;
            Bg[kk][r] = (n0 + r < N && gk < K) ? B0[(int64_t)(n0 + r) * K + gk] : 0.0f;
            if (EPI == kEpiSwiGLU) Bu[kk][r] = (n0 + r < N && gk < K) ? B1[(int64_t)(n0 + r) * K + gk] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            float a[4], g[4], u[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[j] = Bg[kk][tx * 4 + j];
                u[j] = (EPI == kEpiSwiGLU) ? Bu[kk][tx * 4 + j] : 0.0f;
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    accg[i][j] = __builtin_fmaf(a[i], g[j], accg[i][j]);
                    if (EPI == kEpiSwiGLU) accu[i][j] = __builtin_fmaf(a[i], u[j], accu[i][j]);
                }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int row = m0 + ty * 4 + i, col = n0 + tx * 4 + j;
            if (row < M && col < N) {
                float r = (EPI == kEpiSwiGLU) ? silu_f32(accg[i][j]) * accu[i][j] : accg[i][j];
                if (EPI == kEpiPlain && R != nullptr) r += R[(int64_t)row * N + col];
                if (EPI == kEpiSwiGLU && R != nullptr) {
                    const_cast<float*>(R)[(int64_t)row * N + col] = accg[i][j];
                    const_cast<float*>(R)[((int64_t)M + row) * N + col] = accu[i][j];
                }
                C[(int64_t)row * N + col] = r;
            }
        }
}

template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int BKT, int NSTAGE, int EPI, int PF, int FR = 32, bool RAGGED = false>
void launch_gemm_dma(const T* A, const T* B0, const T* B1, T* C, const T* R, int M, int N, int K, hipStream_t stream) {
    constexpr int BN_OUT = (EPI == kEpiSwiGLU) ? BN / 2 : BN;
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN_OUT - 1) / BN_OUT;      // without RAGGED only a ragged last row of tiles is allowed
    // persistent workgroups: as many as are resident at once (LDS-limited), a multiple of 8 so that the XCD patches hold
    constexpr int kStageBytes = (BM + BN) * BKT * (int)sizeof(T) * NSTAGE;
    constexpr int kPerCu = (160 * 1024 / kStageBytes) < 1 ? 1 : ((160 * 1024 / kStageBytes) > 2 ? 2 : (160 * 1024 / kStageBytes));
    const int total = tiles_m * tiles_n;
    const ChipInfo& chip = chip_info();
    const int resident = chip.cus * kPerCu;
    const int grid = total < resident ? total : resident;
    hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, WAVES_M, WAVES_N, BKT, NSTAGE, EPI, PF, FR, RAGGED>), dim3((unsigned)grid),
                       dim3(WAVES_M * WAVES_N * 64), 0, stream, A, B0, B1, C, R, M, N, K, tiles_m, tiles_n, chip.xcds);
}

template <typename T, int EPI>
void launch_gemm_wide(const T* A, const T* B0, const T* B1, T* C, const T* R, int M, int N, int K, hipStream_t stream) {
    constexpr int BN_OUT = EPI == kEpiSwiGLU ? kWide / 2 : kWide;
    const int tiles_m = (M + kWide - 1) / kWide, tiles_n = (N + BN_OUT - 1) / BN_OUT, total = tiles_m * tiles_n;
    const ChipInfo& chip = chip_info();
    const dim3 grid((unsigned)(total < chip.cus ? total : chip.cus));
    if (M % kWide == 0 && N % BN_OUT == 0 && K % (2 * kWideK) == 0)
        hipLaunchKernelGGL((gemm_wide_kernel<T, EPI, false>), grid, dim3(kWideThreads), 0, stream, A, B0, B1, C, R, M, N, K, tiles_m, tiles_n, chip.xcds);
    else
        hipLaunchKernelGGL((gemm_wide_kernel<T, EPI, true>), grid, dim3(kWideThreads), 0, stream, A, B0, B1, C, R, M, N, K, tiles_m, tiles_n, chip.xcds);
}

template <typename T, int MT, int NT, int EPI>
void launch_gemm_splitk(const T* A, const T* B0, const T* B1, T* C, const T* R, int M, int N, int K, hipStream_t stream) {
    const int tiles_m = (M + 16 * MT - 1) / (16 * MT), tiles_n = (N + 16 * NT - 1) / (16 * NT);
    const int tiles = tiles_m * tiles_n, xcds = chip_info().xcds;
    hipLaunchKernelGGL((gemm_splitk_kernel<T, MT, NT, EPI>), dim3((unsigned)((tiles + xcds - 1) / xcds * xcds)), dim3(kSplitWaves * 64),
                       0, stream, A, B0, B1, C, R, M, N, K, tiles_m, tiles, xcds);
}

// 128 x 128 and smaller tiles: 4 waves that read half a k-tile of fragments ahead (a whole one in fp32), one workgroup per CU
// with four stages in flight, or (128 x 128) two per CU with two stages when there are more tiles than CUs; 128 x 128 tiles of a long k
// loop that all have a CU to themselves: fmoe_gemm128.h.
template <typename T, int EPI, bool RAGGED>
void launch_tiles(const T* A, const T* B0, const T* B1, T* C, const T* R, int M, int N, int K, hipStream_t stream) {
    constexpr int KT = kStageK<T>, PF = kSmallAhead<T>, FR = kFragRows<T>;
    int tiles = 0;
    TileShape shape = choose_tile<T, EPI>(M, N, tiles);
    if (sizeof(T) == 2 && shape == kTile256 && !(aligned16(C) && aligned16(R))) {          // its results and residual move in 16-byte pieces
        shape = kTile128;
        tiles = ((M + 127) / 128) * ((N + kTileCols[kTile128] / (EPI == kEpiSwiGLU ? 2 : 1) - 1) / (kTileCols[kTile128] / (EPI == kEpiSwiGLU ? 2 : 1)));
    }
    switch (shape) {
        case kTile256:
            if constexpr (sizeof(T) == 2) launch_gemm_wide<T, EPI>(A, B0, B1, C, R, M, N, K, stream);
            else launch_gemm_dma<T, 256, 256, 2, 4, KT, 2, EPI, 1, FR, RAGGED>(A, B0, B1, C, R, M, N, K, stream);
            break;
        case kTile128:
            if constexpr (sizeof(T) == 2 && EPI == kEpiPlain) {
                if (tiles <= chip_info().cus && K > (kSoloTiles - 1) * 64 && aligned16(C) && aligned16(R)) {
                    hipLaunchKernelGGL((gemm_solo_kernel<T>), dim3((unsigned)tiles), dim3(256), 0, stream, A, B0, C, R, M, N, K, (M + 127) / 128,
                                       (N + 127) / 128, chip_info().xcds);
                    break;
                }
            }
            if (tiles <= chip_info().cus) launch_gemm_dma<T, 128, 128, 2, 2, KT, 4, EPI, PF, FR, RAGGED>(A, B0, B1, C, R, M, N, K, stream);
            else launch_gemm_dma<T, 128, 128, 2, 2, KT, 2, EPI, PF, FR, RAGGED>(A, B0, B1, C, R, M, N, K, stream);
            break;
        case kSplit32: launch_gemm_splitk<T, 2, 2, EPI>(A, B0, B1, C, R, M, N, K, stream); break;
        case kSplit16x32: launch_gemm_splitk<T, 1, 2, EPI>(A, B0, B1, C, R, M, N, K, stream); break;
        case kSplit16: launch_gemm_splitk<T, 1, 1, EPI>(A, B0, B1, C, R, M, N, K, stream); break;
        case kTile64x128: launch_gemm_dma<T, 64, 128, 2, 2, KT, 4, EPI, PF, FR, RAGGED>(A, B0, B1, C, R, M, N, K, stream); break;
        default: launch_gemm_dma<T, 64, 64, 2, 2, KT, 4, EPI, kTileAhead<T, 64, EPI>, kTileFrag<T, 64, EPI>, RAGGED>(A, B0, B1, C, R, M, N, K, stream);
    }
}

template <typename T, int EPI>
void launch_product(const T* A, const T* B0, const T* B1, T* C, const T* R, int M, int N, int K, hipStream_t stream) {
    // the DMA kernel moves 16-byte pieces of rows; fp32 callers need not align their tensors or rows
    if (sizeof(T) == 4 && !(K % 4 == 0 && aligned16(A) && aligned16(B0) && aligned16(B1))) {
        if constexpr (sizeof(T) == 4)
            hipLaunchKernelGGL((sgemm_nt_kernel<EPI>), dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, stream, A, B0, B1, C, R, M, N, K);
        return;
    }
    if (K % kStageK<T> == 0 && N % (EPI == kEpiSwiGLU ? 128 : 256) == 0) launch_tiles<T, EPI, false>(A, B0, B1, C, R, M, N, K, stream);
    else launch_tiles<T, EPI, true>(A, B0, B1, C, R, M, N, K, stream);
}

template <typename T>
int gate_up_tiled(const void* x, const void* wg, const void* wu, int M, int H, int I, void* h, void* saved, hipStream_t stream) {
    launch_product<T, kEpiSwiGLU>((const T*)x, (const T*)wg, (const T*)wu, (T*)h, (const T*)saved, M, I, H, stream);
    FMOE_CHECK_LAUNCH("fmoe_mlp(gate/up)");
    return FMOE_OK;
}

template <typename T>
void launch_sliced(const T* A, const T* B, T* C, const T* R, int M, int N, int K, const SlicePlan& p, float* planes, hipStream_t stream) {
    const int tiles_m = (M + kTileRows[p.shape] - 1) / kTileRows[p.shape], tiles_n = (N + kTileCols[p.shape] - 1) / kTileCols[p.shape];
    const dim3 grid((unsigned)(tiles_m * tiles_n * p.slices));
#define FMOE_GO(BM, BN, WAVES_N, NSTAGE)                                                                                            \
    hipLaunchKernelGGL((gemm_sliced_kernel<T, BM, BN, WAVES_N, NSTAGE>), grid, dim3(128 * WAVES_N), 0, stream, A, B, planes, M, N, K, \
                       tiles_m, tiles_n, chip_info().xcds, p.slices)
    switch (p.shape) {
        case kTile256:
            if constexpr (sizeof(T) == 2)
                hipLaunchKernelGGL((gemm_wide_sliced_kernel<T>), grid, dim3(kWideThreads), 0, stream, A, B, planes, M, N, K, tiles_m, tiles_n, chip_info().xcds,
                                   p.slices);
            break;
        case kTile128: FMOE_GO(128, 128, 2, 4); break;
        case kTile64x128: FMOE_GO(64, 128, 2, 4); break;
        default: FMOE_GO(64, 64, 2, 4); break;
    }
#undef FMOE_GO
    const int64_t elements = (int64_t)M * N;
    hipLaunchKernelGGL((add_slices_kernel<T>), dim3((unsigned)((elements + 1023) / 1024)), dim3(256), 0, stream, (const float*)planes, R, C,
                       elements, p.slices);
}

// planes: room for the fp32 sums of a product cut into slices of k (NULL: it is not cut)
template <typename T>
int down_tiled(const void* h, const void* wd, int M, int H, int I, const void* residual, void* out, float* planes, hipStream_t stream) {
    if (planes != nullptr && (sizeof(T) == 2 || (aligned16(h) && aligned16(wd)))) {
        const SlicePlan p = plan_slices_of_k<T>(M, H, I);
        if (p.slices > 1) {
            launch_sliced<T>((const T*)h, (const T*)wd, (T*)out, (const T*)residual, M, H, I, p, planes, stream);
            FMOE_CHECK_LAUNCH("fmoe_mlp(down)");
            return FMOE_OK;
        }
    }
    launch_product<T, kEpiPlain>((const T*)h, (const T*)wd, nullptr, (T*)out, (const T*)residual, M, H, I, stream);
    FMOE_CHECK_LAUNCH("fmoe_mlp(down)");
    return FMOE_OK;
}

}  // namespace

// C[M,N] = A[M,K] * B[N,K]^T in the 16-bit dtype and in fp32 (the same sums before rounding), on 256 x 256 tiles of the
// DMA kernel: for products large enough to give every compute unit a tile (the router's gate product for tens of thousands
// of tokens).  The k order of the sums is that of every other kernel here: ascending, 16 values per matrix instruction.
bool gemm_nt_dual_usable(int64_t M, int N, int K) {
    return M > 0 && M < (1ll << 31) && N % 256 == 0 && K % 64 == 0 && ((M + 255) / 256) * (int64_t)(N / 256) >= chip_info().cus;
}
int gemm_nt_dual(const void* A, const void* B, void* C, float* C32, int M, int N, int K, int dtype, hipStream_t stream) {
    if (dtype == FMOE_BF16)
        launch_gemm_dma<bf16_t, 256, 256, 2, 4, 64, 2, kEpiDual, 1>((const bf16_t*)A, (const bf16_t*)B, nullptr, (bf16_t*)C,
                                                                    (const bf16_t*)C32, M, N, K, stream);
    else
        launch_gemm_dma<f16_t, 256, 256, 2, 4, 64, 2, kEpiDual, 1>((const f16_t*)A, (const f16_t*)B, nullptr, (f16_t*)C,
                                                                   (const f16_t*)C32, M, N, K, stream);
    FMOE_CHECK_LAUNCH("gate product (tiled)");
    return FMOE_OK;
}

namespace {

int check_mlp_shape(const char* who, int64_t T_, int H, int I, int dtype) {
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "%s: unknown dtype %d", who, dtype);
    FMOE_REQUIRE(T_ >= 0 && H > 0 && I > 0, FMOE_ERR_BAD_SHAPE, "%s: bad shape T=%lld H=%d I=%d", who, (long long)T_, H, I);
    FMOE_REQUIRE(T_ < (1ll << 31), FMOE_ERR_UNSUPPORTED, "%s: T=%lld >= 2^31", who, (long long)T_);
    if (dtype != FMOE_F32)
        FMOE_REQUIRE(H % 8 == 0 && I % 8 == 0, FMOE_ERR_ALIGNMENT,
                     "%s: hidden=%d and intermediate=%d must be multiples of 8 (16-byte rows)", who, H, I);
    return FMOE_OK;
}

}  // namespace
}  // namespace fmoe

extern "C" size_t fmoe_mlp_workspace_bytes(int64_t num_tokens, int hidden, int intermediate, int dtype) {
    if (num_tokens <= 0 || intermediate <= 0 || !fmoe::dtype_ok(dtype)) return 0;
    return fmoe::round_up((size_t)num_tokens * (size_t)intermediate * fmoe::dtype_size(dtype), 256) +
           fmoe_mlp_down_workspace_bytes(num_tokens, hidden, intermediate, dtype);
}

namespace fmoe {
namespace {
int mlp_gate_up_impl(const char* who, const void* x, const void* gate_w, const void* up_w, int64_t num_tokens, int hidden,
                     int intermediate, int dtype, void* act, void* saved, void* stream) {
    clear_error();
    if (int rc = check_mlp_shape(who, num_tokens, hidden, intermediate, dtype)) return rc;
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(x && gate_w && up_w && act, FMOE_ERR_NULL_POINTER, "%s: null tensor pointer", who);
    FMOE_REQUIRE(dtype == FMOE_F32 || (aligned16(x) && aligned16(gate_w) && aligned16(up_w) && aligned16(act) && aligned16(saved)),
                 FMOE_ERR_ALIGNMENT, "%s: tensor pointers must be 16-byte aligned", who);
    hipStream_t s = (hipStream_t)stream;
    const int M = (int)num_tokens;
    switch (dtype) {
        case FMOE_F32: return gate_up_tiled<float>(x, gate_w, up_w, M, hidden, intermediate, act, saved, s);
        case FMOE_BF16: return gate_up_tiled<bf16_t>(x, gate_w, up_w, M, hidden, intermediate, act, saved, s);
        default: return gate_up_tiled<f16_t>(x, gate_w, up_w, M, hidden, intermediate, act, saved, s);
    }
}
}  // namespace
}  // namespace fmoe

extern "C" int fmoe_mlp_gate_up(const void* x, const void* gate_w, const void* up_w, int64_t num_tokens, int hidden,
                                int intermediate, int dtype, void* act, void* stream) {
    return fmoe::mlp_gate_up_impl("fmoe_mlp_gate_up", x, gate_w, up_w, num_tokens, hidden, intermediate, dtype, act, nullptr, stream);
}

extern "C" int fmoe_mlp_gate_up_save(const void* x, const void* gate_w, const void* up_w, int64_t num_tokens, int hidden,
                                     int intermediate, int dtype, void* act, void* saved, void* stream) {
    using namespace fmoe;
    if (saved == nullptr && num_tokens > 0) {
        clear_error();
        set_error("fmoe_mlp_gate_up_save: null buffer for the gate and up products");
        return FMOE_ERR_NULL_POINTER;
    }
    return mlp_gate_up_impl("fmoe_mlp_gate_up_save", x, gate_w, up_w, num_tokens, hidden, intermediate, dtype, act, saved, stream);
}

namespace fmoe {
namespace {
int mlp_down_impl(const char* who, const void* act, const void* down_w, int64_t num_tokens, int hidden, int intermediate, int dtype,
                  const void* residual, void* out, float* planes, void* stream) {
    clear_error();
    if (int rc = check_mlp_shape(who, num_tokens, hidden, intermediate, dtype)) return rc;
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(act && down_w && out, FMOE_ERR_NULL_POINTER, "%s: null tensor pointer", who);
    FMOE_REQUIRE(dtype == FMOE_F32 || (aligned16(act) && aligned16(down_w)), FMOE_ERR_ALIGNMENT,
                 "%s: tensor pointers must be 16-byte aligned", who);
    hipStream_t s = (hipStream_t)stream;
    const int M = (int)num_tokens;
    switch (dtype) {
        case FMOE_F32: return down_tiled<float>(act, down_w, M, hidden, intermediate, residual, out, planes, s);
        case FMOE_BF16: return down_tiled<bf16_t>(act, down_w, M, hidden, intermediate, residual, out, planes, s);
        default: return down_tiled<f16_t>(act, down_w, M, hidden, intermediate, residual, out, planes, s);
    }
}
}  // namespace
}  // namespace fmoe

extern "C" int fmoe_mlp_down(const void* act, const void* down_w, int64_t num_tokens, int hidden, int intermediate,
                             int dtype, const void* residual, void* out, void* stream) {
    return fmoe::mlp_down_impl("fmoe_mlp_down", act, down_w, num_tokens, hidden, intermediate, dtype, residual, out, nullptr, stream);
}

extern "C" size_t fmoe_mlp_down_workspace_bytes(int64_t num_tokens, int hidden, int intermediate, int dtype) {
    using namespace fmoe;
    if (num_tokens <= 0 || num_tokens >= (1ll << 31) || hidden <= 0 || intermediate <= 0 || !dtype_ok(dtype)) return 0;
    const SlicePlan p = dtype == FMOE_F32 ? plan_slices_of_k<float>((int)num_tokens, hidden, intermediate)
                                          : plan_slices_of_k<bf16_t>((int)num_tokens, hidden, intermediate);
    return p.slices > 1 ? round_up((size_t)p.slices * (size_t)num_tokens * (size_t)hidden * 4, 256) : 0;
}

extern "C" int fmoe_mlp_down_ws(const void* act, const void* down_w, int64_t num_tokens, int hidden, int intermediate, int dtype,
                                const void* residual, void* out, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace fmoe;
    const size_t need = fmoe_mlp_down_workspace_bytes(num_tokens, hidden, intermediate, dtype);
    if (need > 0 && (workspace == nullptr || workspace_bytes < need || !aligned16(workspace))) {
        clear_error();
        set_error("fmoe_mlp_down_ws: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
        return FMOE_ERR_WORKSPACE;
    }
    return mlp_down_impl("fmoe_mlp_down_ws", act, down_w, num_tokens, hidden, intermediate, dtype, residual, out,
                         need > 0 ? (float*)workspace : nullptr, stream);
}

extern "C" int fmoe_mlp_forward(const void* x, const void* gate_w, const void* up_w, const void* down_w,
                                int64_t num_tokens, int hidden, int intermediate, int dtype, const void* residual,
                                void* out, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace fmoe;
    clear_error();
    if (int rc = check_mlp_shape("fmoe_mlp_forward", num_tokens, hidden, intermediate, dtype)) return rc;
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(x && gate_w && up_w && down_w && out, FMOE_ERR_NULL_POINTER, "fmoe_mlp_forward: null tensor pointer");
    const size_t need = fmoe_mlp_workspace_bytes(num_tokens, hidden, intermediate, dtype);
    FMOE_REQUIRE(workspace && workspace_bytes >= need, FMOE_ERR_WORKSPACE,
                 "fmoe_mlp_forward: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    if (int rc = fmoe_mlp_gate_up(x, gate_w, up_w, num_tokens, hidden, intermediate, dtype, workspace, stream)) return rc;
    const size_t planes = fmoe_mlp_down_workspace_bytes(num_tokens, hidden, intermediate, dtype);
    return fmoe_mlp_down_ws(workspace, down_w, num_tokens, hidden, intermediate, dtype, residual, out, (char*)workspace + (need - planes),
                            planes, stream);
}
