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
// The MLP's backward forms dWd, dx, dWg and dWu in one launch (gemm_group_kernel): none of them alone is whole rounds of tiles, and two
// workgroups of different products share a compute unit as well as two of one.
//
// Against the library's kernels (rocBLAS), each product alone, us:
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

// dh = dy Wd and the SwiGLU gradient of it (kEpiGradient): dh makes no way through memory, and is not rounded on it.  us, two launches and
// one (bf16): 615 tokens, 776 -> 2072 14.6 and 11.5; 4096 tokens, 1024 -> 4096 63 and 54; 300 tokens, 512 -> 1360 9.0 and 6.1; 8000 tokens, 320
// -> 848 27 and 17.  da, db and h against 64 bits: 1.66e-3 of them, 2.34e-3 with dh rounded.  Bound by the planes, read and written at
// 6 TB/s, on few columns, by what the L2s deliver to 128 x 128 tiles on many.
template <typename T, int BM, int BN>
__global__ __launch_bounds__(256, 2) void gemm_gradient_kernel(const T* __restrict__ dy, const T* __restrict__ wd, const GradientPlanes<T> grad, int M, int N, int K,
                                                               int tiles_m, int tiles_n, int xcds) {
    gemm_dma_tiles<T, BM, BN, 2, 2, kStageK<T>, 2, kEpiGradient, kSmallAhead<T>, kFragRows<T>, true, false, false, true>(
        dy, wd, nullptr, nullptr, nullptr, M, N, K, tiles_m, tiles_n, xcds, (int)blockIdx.x, (int)gridDim.x, 0, 1, K, N, 1, grad);
}

// Several products in one launch: the workgroups of member i are first .. first + tiles * slices - 1 (first a multiple of the XCDs; ids
// past the last are spare), one tile or slice of k each, which the dispatcher hands to compute units as they fall free, longest first.
// us, dWd, dx, dWg and dWu one after the other and together, repeated alone, bf16: 4096 tokens, 1024 -> 4096 190 -> 152 (161 to 177 in a
// training step, behind what moves its operands out of the L2s); 615 tokens, 776 -> 2072 35.5 ->
// 23.6; 1000 tokens, 1024 -> 4096 63 -> 49; 130 tokens, 408 -> 1088 17.8 -> 9.4; 5616 tokens, 608 -> 2432 123 -> 82; fp32: 691 tokens, 1056
// -> 2112 177 -> 133; 103 tokens, 768 -> 1536 33 -> 22.  What is left is what the L2s deliver on 128 x 128 tiles, two to a compute unit
// (69 GB/s each), and the matrix pipes in fp32.
struct GroupMember {
    const void *A, *B0, *B1;
    void* out;                   // C, or the planes of its slices
    int lda, ldb, M, N, K, segments, tiles_m, tiles_n, slices, first, a_turned;
};
struct Group { GroupMember m[kGroupMost]; };

template <typename T, int SHAPE, bool TA, bool SLICED>
__device__ __forceinline__ void group_tile(const GroupMember& m, int at) {
    const int tiles = m.tiles_m * m.tiles_n, tile = at % tiles, slice = at / tiles;
    const T *A = (const T*)m.A, *B0 = (const T*)m.B0, *B1 = (const T*)m.B1;
    constexpr int EPI = SLICED ? kEpiPart : kEpiPlain;
    if constexpr (SHAPE == kTile256)
        gemm_wide_tiles<T, EPI, true, SLICED, TA, true>(A, B0, B1, (T*)m.out, nullptr, m.M, m.N, m.K, m.tiles_m, m.tiles_n, 1, tile, tiles, slice,
                                                        m.slices, m.lda, m.ldb, m.segments);
    else
        gemm_dma_tiles<T, kTileRows[SHAPE], kTileCols[SHAPE], 2, 2, kStageK<T>, 2, EPI, kSmallAhead<T>, kFragRows<T>, true, SLICED, TA, true>(
            A, B0, B1, (T*)m.out, nullptr, m.M, m.N, m.K, m.tiles_m, m.tiles_n, 1, tile, tiles, slice, m.slices, m.lda, m.ldb, m.segments);
}

template <typename T, int SHAPE>
__global__ __launch_bounds__(SHAPE == kTile256 ? kWideThreads : 256, 2) void gemm_group_kernel(const Group g, int members, int xcds) {
    const int block = (int)blockIdx.x;
    int i = 0;
    while (i + 1 < members && block >= g.m[i + 1].first) ++i;
    const GroupMember& m = g.m[i];
    const int items = m.tiles_m * m.tiles_n * m.slices, local = block - m.first;
    if (local >= items) return;
    const int at = xcd_run(local, items, xcds);
    if (m.slices > 1) {
        if (m.a_turned) group_tile<T, SHAPE, true, true>(m, at);
        else group_tile<T, SHAPE, false, true>(m, at);
    } else {
        if (m.a_turned) group_tile<T, SHAPE, true, false>(m, at);
        else group_tile<T, SHAPE, false, false>(m, at);
    }
}

// C = sum over the slices, in order, of one or several products; one packet of C per thread
struct SumMember { const float* planes; void* C; int64_t packets; int slices, first; };
struct Sums { SumMember m[kGroupMost]; };
template <typename T>
__global__ __launch_bounds__(256) void gemm_turned_add_kernel(const Sums g, int members) {
    constexpr int V = Elem<T>::kVec;
    int k = 0;
    while (k + 1 < members && (int)blockIdx.x >= g.m[k + 1].first) ++k;
    const SumMember& m = g.m[k];
    const int64_t i = (int64_t)((int)blockIdx.x - m.first) * blockDim.x + threadIdx.x;
    if (i >= m.packets) return;
    float v[V];
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = 0.0f;
    for (int s = 0; s < m.slices; ++s)
#pragma unroll
        for (int h = 0; h < V; h += 4) {
            const f32x4_t p = *reinterpret_cast<const f32x4_t*>(m.planes + (s * m.packets + i) * V + h);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[h + e] += p[e];
        }
    reinterpret_cast<u32x4_t*>(m.C)[i] = pack16<T>(v);
}
template <typename T> void launch_sums(Sums& g, int members, hipStream_t stream) {
    int blocks = 0;
    for (int i = 0; i < members; ++i) {
        g.m[i].first = blocks;
        blocks += (int)((g.m[i].packets + 255) / 256);
    }
    hipLaunchKernelGGL((gemm_turned_add_kernel<T>), dim3((unsigned)blocks), dim3(256), 0, stream, g, members);
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
template <typename T> SlicePlan plan_turned(int M, int N, int K, int segments, double* price = nullptr) {
    const int cus = chip_info().cus, k_tiles = (K + kStageK<T> - 1) / kStageK<T> * segments;
    SlicePlan best = {kTile64, 1};
    double best_time = 0.0;
    for (int i = sizeof(T) == 4 ? kTile128 : kTile256; i <= kTile64; ++i) {
        int64_t n = 0;
        if (sizeof(T) == 4 && i == kTile64x128) continue;
        const double row = tile_cost<T, kEpiPlain>(i, M, N, cus, n) * 2.3e-3, stores = i == kTile256 ? 7.0 : 1.0;
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
    if (price != nullptr) *price = best_time;
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
        Sums g = {};
        g.m[0] = {planes, C, (int64_t)M * N / Elem<T>::kVec, p.slices, 0};
        launch_sums<T>(g, 1, stream);
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

// Time of `kinds` lots of items (n[i] of time t[i], longest first) on `slots` that take the next item as they fall free.
inline double time_of_items(const int64_t* n, const double* t, int kinds, int slots) {
    struct Free { double at; int64_t slots; } f[2 * kGroupMost + 2] = {{0.0, slots}};
    int lots = 1;
    double end = 0.0;
    for (int i = 0; i < kinds; ++i)
        for (int64_t left = n[i]; left > 0;) {
            int e = 0;
            for (int j = 1; j < lots; ++j)
                if (f[j].at < f[e].at) e = j;
            const double done = f[e].at + t[i];
            int64_t take = left < f[e].slots ? left : f[e].slots;
            if (lots == 1 && take == f[e].slots) {                  // whole rounds at once
                const int64_t rounds = left / f[e].slots;
                f[e].at += (double)rounds * t[i];
                end = f[e].at > end ? f[e].at : end;
                left -= rounds * f[e].slots;
                continue;
            }
            left -= take;
            f[e].slots -= take;
            if (f[e].slots == 0) f[e] = f[--lots];
            int j = 0;
            while (j < lots && f[j].at != done) ++j;
            if (j < lots) f[j].slots += take;
            else if (lots < 2 * kGroupMost + 2) f[lots++] = {done, take};
            else f[lots - 1].slots += take;
            end = done > end ? done : end;
        }
    return end;
}

// Tile shape of dh = dy Wd with its SwiGLU gradient in one launch, or -1: two launches.  Prices (us): k-tiles at the rate of a full
// compute unit or of one tile alone, an epilogue's five values of 2 bytes at what a unit gets of 6.6 TB/s; two launches: the product at
// its own price and six planes at 6.3 TB/s.  Over 83 products timed all ways (16 to 8192 tokens, 256 to 4096 columns) the choice is 1 % behind
// the best on average; two launches take 20 % more.  Planes beyond 100 MB come from memory, no longer from the cache in front of it, and an
// epilogue waits for them where a launch that does nothing else streams them (4096 tokens, 1024 -> 4096 67 us in two, 72 to 74 in one,
// also on 256 x 256 tiles; 59 with the planes at hand).
int plan_gradient(int M, int N, int K) {
    const int cus = chip_info().cus, k_tiles = (K + 63) / 64;
    if ((double)M * N > 1.0e7) return -1;
    double best_time = 0.0;
    plan_turned<bf16_t>(M, N, K, 1, &best_time);
    const double planes = 12.0e-6 * (double)M * N / 6.3 + 2.0;
    best_time += (planes > 3.8 ? planes : 3.8) + 0.9;
    int best = -1;
    for (int shape : {kTile128, kTile64}) {
        const bool large = shape == kTile128;
        const int rows = kTileRows[shape], cols = kTileCols[shape], per = large ? 2 : 4;
        const int64_t n = (int64_t)((M + rows - 1) / rows) * ((N + cols - 1) / cols);
        const double share = 6550.0 / (n < cus ? n : cus), rate = large && share > 26.0 ? 26.0 : share;     // GB/s of a compute unit
        const double stores = 10.0e-3 * rows * cols / rate, item = k_tiles * (large ? 0.59 : 0.19) + stores;
        const double rounds = (double)((n + per * cus - 1) / (per * cus)) * item * per, blend = large ? 0.32 : 0.4;
        const double alone = k_tiles * (large ? 0.68 : 0.44) + 0.66 * stores, full = n > cus ? blend * rounds + (1.0 - blend) * (double)n * item / cus : 0.0;
        const double time = (full > alone ? full : alone) + 2.2;
        if (time < best_time) {
            best_time = time;
            best = shape;
        }
    }
    return best;
}

// Price (us) of a group on tiles of a shape: half (0.4 to 1) of what its items take on slots that hold two workgroups of 128 x 128 (four of
// 64 x 64) to a compute unit, the rest what they take if the tail were filled, at least the longest chain; per sliced product 4 us and
// its planes written and read at 6 TB/s.  The rates of a k-tile, with the compute unit full and alone, and the 3.4 % (fp32 2.3) by which the
// choice misses the best of 72 cuts on average come from 105 backward passes in bf16 (64 to 8192 tokens, 256 to 2048 columns) and 44 in fp32 (there up to
// 16384, best on 128 x 128 tiles from about 4000 tokens on: 4096 tokens, 1024 -> 4096 1258 us one by one, 1238 on 64 x 64, 1176; 5000, 2048
// -> 5464 4392, 4291, 4176).  64 x 128 tiles would gain half a percent.  Products over tokens (the weight gradients)
// are sliced from 2048 tokens on.
// A group must be cheaper than its products one by one, whose price is plan_turned's and a launch of 4 us for each but the first (fp32,
// whose prices fit less well: a fifth more, and 4 us each).  Few tiles over many tokens are not: alone, a product may be cut into 16 slices.
// Where groups were formed at any price, 32768 tokens, 256 columns, 24 keys, us: two launches 76, one 125, fp32 114 and 214; MLP, 65536
// tokens, 128 -> 344 171 and 247.  Of 316 such calls (256 to 65536 tokens) the choice is 0.1 % behind the better way on average, 8 % at most.
// 16-bit, beyond four rounds of 256 x 256 tiles: each product fills the chip and its persistent workgroups start a tile's loads under the last
// one's stores: 2048 tokens, 4096 -> 16384 1057 us one by one, 1087 together; 6000 tokens, 1800 -> 7200, three and a half rounds, 734 and 731.
template <typename T> GroupPlan plan_group(const BackwardProduct* p, int count) {
    GroupPlan best = {-1, {1, 1, 1, 1}};
    if (count < 2 || count > kGroupMost) return best;
    constexpr bool kSingle = sizeof(T) == 4;      // fp32
    const int cus = chip_info().cus;
    int64_t wide = 0;
    int token_cuts = 1;
    for (int i = 0; i < count; ++i) {
        if (p[i].layout == kBlasTN && p[i].K >= 2048) token_cuts = 3;
        wide += (int64_t)((p[i].M + 255) / 256) * ((p[i].N + 255) / 256);
    }
    if (!kSingle && wide > 4 * (int64_t)cus) return best;
    constexpr int kShapes[3] = {kTile256, kTile128, kTile64}, kPer[3] = {1, 2, 4};
    constexpr double kFull[3] = {1.5, kSingle ? 1.75 : 0.47, kSingle ? 0.475 : 0.225}, kAlone[3] = {1.3, kSingle ? 2.2 : 0.75, kSingle ? 0.6 : 0.3};
    constexpr double kStores[3] = {6.0, kSingle ? 2.0 : 0.65, kSingle ? 0.2 : 0.1}, kRounds[3] = {0.5, kSingle ? 1.0 : 0.4, kSingle ? 0.5 : 0.4};
    constexpr int kOver[6] = {1, 2, 3, 4, 6, 8}, kTokens[3] = {1, 2, 4};
    double best_time = kSingle ? 4.0 * count : 4.0 * (count - 1);          // one by one
    for (int i = 0; i < count; ++i) {
        double alone = 0.0;
        plan_turned<T>(p[i].M, p[i].N, p[i].K, p[i].segments, &alone);
        best_time += (kSingle ? 1.2 : 1.0) * alone;
    }
    for (int z = kSingle ? 1 : 0; z < 3; ++z) {
        const int shape = kShapes[z];
        int64_t tiles[kGroupMost];
        int k_tiles[kGroupMost];
        for (int i = 0; i < count; ++i) {
            tiles[i] = (int64_t)((p[i].M + kTileRows[shape] - 1) / kTileRows[shape]) * ((p[i].N + kTileCols[shape] - 1) / kTileCols[shape]);
            k_tiles[i] = (p[i].K + kStageK<T> - 1) / kStageK<T> * p[i].segments;
        }
        for (int over : kOver)
            for (int cut = 0; cut < token_cuts; ++cut)
                for (int cut_rest = 0; cut_rest <= cut; ++cut_rest) {
                    const int first = kTokens[cut], rest = kTokens[cut_rest];
                    GroupPlan g = {shape, {1, 1, 1, 1}};
                    int64_t n[kGroupMost];
                    double t[kGroupMost], work = 0.0, longest = 0.0, planes = 0.0;
                    bool usable = true, seen = false;
                    for (int i = 0; i < count && usable; ++i) {
                        const bool turned = p[i].layout == kBlasTN;
                        const int s = turned ? (seen ? rest : first) : over, share = (k_tiles[i] + s - 1) / s;
                        seen = seen || turned;
                        usable = s == 1 || ((!turned || p[i].K >= 2048) && k_tiles[i] >= 2 * s && (s - 1) * share < k_tiles[i]);
                        g.slices[i] = s;
                        int at = i;                                              // longest first
                        const double item = share * kFull[z] + kStores[z];
                        while (at > 0 && t[at - 1] < item) {
                            t[at] = t[at - 1];
                            n[at] = n[at - 1];
                            --at;
                        }
                        t[at] = item;
                        n[at] = tiles[i] * s;
                        work += (double)n[at] * item / cus;
                        if (share * kAlone[z] > longest) longest = share * kAlone[z];
                        if (s > 1) planes += 4.0 + 8.0e-6 * s * (double)p[i].M * p[i].N / 6.0;
                    }
                    if (!usable || (work > longest ? work : longest) + planes >= best_time) continue;
                    for (int i = 0; i < count; ++i) t[i] *= kPer[z];
                    const double mixed = kRounds[z] * time_of_items(n, t, count, kPer[z] * cus) + (1.0 - kRounds[z]) * work;
                    const double time = (mixed > longest ? mixed : longest) + planes;
                    if (time < best_time) {
                        best = g;
                        best_time = time;
                    }
                }
    }
    return best;
}

size_t group_planes_bytes(const BackwardProduct* p, int count, const GroupPlan& g) {
    size_t bytes = 0;
    for (int i = 0; i < count; ++i)
        if (g.slices[i] > 1) bytes += round_up((size_t)g.slices[i] * p[i].M * p[i].N * sizeof(float), 256);
    return bytes;
}

// Whether the kernels here can address a product: whole packets (where M (TN) or K (NN) is none, the rows of A are padded with zeros up to
// lda) and 32-bit byte offsets inside a descriptor.
bool addressable(const BackwardProduct& p, int dtype) {
    const int a_cols = p.layout == kBlasTN ? p.M : p.K * p.segments, vec = dtype == FMOE_F32 ? 4 : 8;
    const bool packets = p.lda % vec == 0 && p.ldb % vec == 0 && p.N % vec == 0 && (a_cols + vec - 1) / vec * vec <= p.lda &&
                         (p.segments == 1 || p.K % vec == 0) && aligned16(p.A) && aligned16(p.B0) && aligned16(p.B1) && aligned16(p.C);
    const double most = dtype == FMOE_F32 ? 5.0e8 : 1.0e9;
    return packets && (double)p.K * p.ldb < most && (p.layout == kBlasTN ? (double)p.K * p.lda < most : 256.0 * p.lda < most);
}

// Whether a product's result lies on what another one reads or writes: a caller may ask for gradients in the place of tensors that only
// earlier products need (dx in that of dy, a weight's gradient in that of the weight), which one launch would write while others read.
bool in_place(const BackwardProduct* p, int count, int dtype) {
    const int64_t elt = (int64_t)dtype_size(dtype);
    struct Span { const char* at; int64_t bytes; };
    auto rows = [&](const void* base, int64_t n, int64_t ld, int64_t cols) { return Span{(const char*)base, ((n - 1) * ld + cols) * elt}; };
    for (int i = 0; i < count; ++i) {
        const Span c = rows(p[i].C, p[i].M, p[i].N, p[i].N);
        for (int j = 0; j < count; ++j) {
            if (j == i) continue;
            const BackwardProduct& q = p[j];
            const Span other[4] = {q.layout == kBlasTN ? rows(q.A, q.K, q.lda, q.M) : rows(q.A, q.M, q.lda, (int64_t)q.K * q.segments),
                                   rows(q.B0, q.K, q.ldb, q.N), rows(q.segments > 1 ? q.B1 : q.B0, q.K, q.ldb, q.N), rows(q.C, q.M, q.N, q.N)};
            for (const Span& o : other)
                if (c.at < o.at + o.bytes && o.at < c.at + c.bytes) return true;
        }
    }
    return false;
}

template <typename T>
void launch_group(const BackwardProduct* p, int count, const GroupPlan& plan, void* workspace, hipStream_t stream, KeptPlanes* keep) {
    const int xcds = chip_info().xcds, rows = kTileRows[plan.shape], cols = kTileCols[plan.shape];
    Group g = {};
    Sums sums = {};
    int sliced = 0, blocks = 0, order[kGroupMost];
    auto share = [&](int i) { return ((p[i].K + kStageK<T> - 1) / kStageK<T> * p[i].segments + plan.slices[i] - 1) / plan.slices[i]; };
    for (int i = 0; i < count; ++i) {                    // longest first
        int at = i;
        while (at > 0 && share(order[at - 1]) < share(i)) {
            order[at] = order[at - 1];
            --at;
        }
        order[at] = i;
    }
    char* planes = (char*)workspace;
    for (int k = 0; k < count; ++k) {
        const int i = order[k];
        const BackwardProduct& q = p[i];
        g.m[k] = {q.A, q.B0, q.segments > 1 ? q.B1 : q.B0, q.C, q.lda, q.ldb, q.M, q.N, q.K, q.segments, (q.M + rows - 1) / rows, (q.N + cols - 1) / cols,
                  plan.slices[i], blocks, q.layout == kBlasTN};
        if (plan.slices[i] > 1) {
            g.m[k].out = planes;
            if (keep != nullptr && keep->product == i) {
                keep->planes = (const float*)planes;
                keep->slices = plan.slices[i];
            } else {
                sums.m[sliced++] = {(const float*)planes, q.C, (int64_t)q.M * q.N / Elem<T>::kVec, plan.slices[i], 0};
            }
            planes += round_up((size_t)plan.slices[i] * q.M * q.N * sizeof(float), 256);
        }
        blocks += (g.m[k].tiles_m * g.m[k].tiles_n * plan.slices[i] + xcds - 1) / xcds * xcds;
    }
#define FMOE_GO(SHAPE) \
    hipLaunchKernelGGL((gemm_group_kernel<T, SHAPE>), dim3((unsigned)blocks), dim3((SHAPE) == kTile256 ? kWideThreads : 256), 0, stream, g, count, xcds)
    if (plan.shape == kTile64) FMOE_GO(kTile64);
    else if (plan.shape == kTile128) FMOE_GO(kTile128);
    else if constexpr (sizeof(T) == 2) FMOE_GO(kTile256);
#undef FMOE_GO
    if (sliced > 0) launch_sums<T>(sums, sliced, stream);
}

}  // namespace

size_t gemm_backward_workspace_bytes(int M, int N, int K, int segments, int dtype) {
    const int slices = (dtype == FMOE_F32 ? plan_turned<float>(M, N, K, segments) : plan_turned<bf16_t>(M, N, K, segments)).slices;
    return slices > 1 ? (size_t)slices * M * N * sizeof(float) : 0;
}

template <typename T>
void launch_gradient(const void* dy, const void* wd, const GradientPlanes<T>& grad, int M, int N, int K, int shape, hipStream_t stream) {
    const int rows = kTileRows[shape], cols = kTileCols[shape], tm = (M + rows - 1) / rows, tn = (N + cols - 1) / cols;
    const int64_t n = (int64_t)tm * tn, resident = (int64_t)chip_info().cus * (shape == kTile128 ? 2 : 4);
    const dim3 grid((unsigned)(n < resident ? n : resident));
#define FMOE_GO(TILE) \
    hipLaunchKernelGGL((gemm_gradient_kernel<T, TILE, TILE>), grid, dim3(256), 0, stream, (const T*)dy, (const T*)wd, grad, M, N, K, tm, tn, chip_info().xcds)
    if (shape == kTile64) FMOE_GO(64);
    else FMOE_GO(128);
#undef FMOE_GO
}

bool swiglu_gradient_together(const void* dy, const void* wd, const void* a, const void* b, void* da, void* db, void* h, int M, int N, int K, int ld,
                              int dtype, hipStream_t stream) {
    if (dtype == FMOE_F32 || ld > 1 << 21 || !addressable({kBlasNN, M, N, K, 1, dy, K, wd, nullptr, N, h}, dtype) || !aligned16(a) || !aligned16(b) ||
        !aligned16(da) || !aligned16(db) || ld % 8 != 0)
        return false;
    const int shape = plan_gradient(M, N, K);
    if (shape < 0) return false;
    if (dtype == FMOE_BF16)
        launch_gradient<bf16_t>(dy, wd, {(const bf16_t*)a, (const bf16_t*)b, (bf16_t*)da, (bf16_t*)db, (bf16_t*)h, ld}, M, N, K, shape, stream);
    else
        launch_gradient<f16_t>(dy, wd, {(const f16_t*)a, (const f16_t*)b, (f16_t*)da, (f16_t*)db, (f16_t*)h, ld}, M, N, K, shape, stream);
    return true;
}

int gemm_backward(const BackwardProduct& q, int dtype, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    if (addressable(q, dtype)) {
        SlicePlan p = dtype == FMOE_F32 ? plan_turned<float>(q.M, q.N, q.K, q.segments) : plan_turned<bf16_t>(q.M, q.N, q.K, q.segments);
        if ((size_t)p.slices * q.M * q.N * sizeof(float) > workspace_bytes) p.slices = 1;
        float* planes = (float*)workspace;
#define FMOE_TURNED(TT)                                                                                                                         \
    do {                                                                                                                                        \
        if (q.layout == kBlasTN) launch_turned<TT, true>(q.A, q.lda, q.B0, q.B1, q.ldb, q.C, q.M, q.N, q.K, q.segments, p, planes, stream);     \
        else launch_turned<TT, false>(q.A, q.lda, q.B0, q.B1, q.ldb, q.C, q.M, q.N, q.K, q.segments, p, planes, stream);                        \
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
    if (int rc = blas_gemm(q.layout, q.M, q.N, q.K, q.A, q.lda, q.B0, q.ldb, q.C, q.N, 0.0f, dtype, stream)) return rc;
    if (q.segments == 1) return FMOE_OK;
    return blas_gemm(q.layout, q.M, q.N, q.K, (const char*)q.A + (size_t)q.K * dtype_size(dtype), q.lda, q.B1, q.ldb, q.C, q.N, 1.0f, dtype, stream);
}

GroupPlan plan_products(const BackwardProduct* p, int count, int dtype) {
    return dtype == FMOE_F32 ? plan_group<float>(p, count) : plan_group<bf16_t>(p, count);
}

size_t gemm_backward_workspace_bytes(const BackwardProduct* p, int count, const GroupPlan& plan, int dtype) {
    if (plan.shape >= 0) return group_planes_bytes(p, count, plan);
    size_t most = 0;
    for (int i = 0; i < count; ++i) {
        const size_t alone = gemm_backward_workspace_bytes(p[i].M, p[i].N, p[i].K, p[i].segments, dtype);
        if (alone > most) most = alone;
    }
    return most;
}

int gemm_backward(const BackwardProduct* p, int count, const GroupPlan& plan, int dtype, void* workspace, size_t workspace_bytes, hipStream_t stream,
                  KeptPlanes* keep) {
    bool together = plan.shape >= 0 && group_planes_bytes(p, count, plan) <= workspace_bytes;
    for (int i = 0; i < count; ++i) together = together && addressable(p[i], dtype);
    together = together && !in_place(p, count, dtype);
    if (together) {
        switch (dtype) {
            case FMOE_F32: launch_group<float>(p, count, plan, workspace, stream, keep); break;
            case FMOE_BF16: launch_group<bf16_t>(p, count, plan, workspace, stream, keep); break;
            default: launch_group<f16_t>(p, count, plan, workspace, stream, keep); break;
        }
        FMOE_CHECK_LAUNCH("backward products");
        return FMOE_OK;
    }
    for (int i = 0; i < count; ++i)
        if (int rc = gemm_backward(p[i], dtype, workspace, workspace_bytes, stream)) return rc;
    return FMOE_OK;
}

}  // namespace fmoe
