// Products of the backward passes whose operands do not lie K-contiguous, for gfx950:
//   NN   C[M,N] = A[M,K] B[K,N]          (dh = dy Wd, dx = [da | db] [Wg; Wu], dq = d Wr)
//   TN   C[M,N] = A[K,M]^T B[K,N]        (the weight gradients)
// A matrix instruction wants consecutive k values of one row in a lane, so operands stored k-row by k-row are transposed between
// the global load and the LDS: a thread loads an 8 x 8 block (one 16-byte packet from each of 8 consecutive k rows), turns it in
// registers (one v_perm per result register) and writes 8 packets of 8 consecutive k values, so that the LDS tile and the multiply loop are those of K-contiguous operands.
//
// What bounds it: the chain of one k-tile (barrier, LDS reads, LDS writes: 0.85 us per 128 k values at 64 x 64 tiles) and what a CU
// receives (about 50 GB/s), with the loads of kRing k-tiles in flight; so k is split over workgroups until every CU has a share
// of some tile, and a second launch adds the fp32 sums, always in the same order.  Measured against the library's kernels for one
// training step of 615 tokens (H = 776, I = 2072, bf16): dh 12 against 19 us, dWd 11 against 17, dx 20 against 28 + 10, the two
// gate / up gradients 17 against 21; a library call also takes 17 us of host time where a launch takes 3.  fp32 goes to the library (6 to 9 us for such products).  Keeping the operands
// out of LDS (fragments straight from global memory, turned in registers) was as fast for long k and slower for short.
#include "fmoe_common.h"
#include "fmoe_mfma.h"
#include "fmoe_vec.h"

namespace fmoe {
namespace {

constexpr uint32_t kOutOfRange = 0x80000000u;    // beyond every descriptor here: such loads give zeros
constexpr int kRing = 3;                          // k-tiles whose loads are in flight

// Tile BR x BR of C, k-tiles of KCH 16-byte packets per row; BR * KCH = 1024 packets per operand and k-tile: waves 0 and 1 bring A,
// waves 2 and 3 bring B, 8 packets per thread.  Packet c of LDS row r sits at c ^ (r ^ r / 8): both the 16 rows a fragment read
// touches and the rows V apart that a transposing write touches then lie in different banks.
// KG: groups of four waves; group g multiplies k-tiles g, g + KG, ... of the workgroup's share into accumulators of its own, which
// are added in group order through LDS at the end (two k loops side by side on a CU that has one tile).
// k runs over `segments` ranges of K values each: range s multiplies columns s*K.. of A (NN) with B0 or B1.  Workgroup: k share
// `split` of a tile; splits > 1: its sums go to partial[split] ([M][N] fp32) instead of C.
template <typename T, bool TA, int BR, int KCH, int KG>
__global__ __launch_bounds__(256 * KG) void gemm_tr_kernel(const T* __restrict__ A, int lda, const T* __restrict__ B0, const T* __restrict__ B1,
                                                      int ldb, T* __restrict__ C, int ldc, float* __restrict__ partial, int M, int N,
                                                      int K, int segments, int tiles_m, int tiles_n, int splits, int xcds) {
    constexpr int V = Elem<T>::kVec, E = (int)sizeof(T), KT = KCH * V;
    constexpr int W = BR / 2, F = W / 16;                    // wave tile and its fragments per side
    constexpr int NB = BR / V;                               // V-column blocks of a transposed operand
    static_assert(BR * KCH == 1024 && V == 8, "eight packets of eight elements per thread");
    __shared__ __attribute__((aligned(16))) u32x4_t lds_all[KG][2][2][BR * KCH];
    const int split = (int)blockIdx.y;
    int tm, tn;
    tile_of_block(tiles_m, tiles_n, xcds, tm, tn);
    const int m0 = tm * BR, n0 = tn * BR;
    const int grp = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane((int)threadIdx.x / 256);
    const int tid = (int)threadIdx.x % 256, lane = tid & 63;
    auto& lds = lds_all[grp];
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool for_b = wave >= 2;
    const int t = tid & 127;
    auto slot = [](int row, int ch) { return row * KCH + (ch ^ ((row ^ (row >> 3)) & (KCH - 1))); };

    const int tiles_k = (K + KT - 1) / KT, tiles_all = tiles_k * segments;
    const int share = (tiles_all + splits - 1) / splits, begin = split * share;
    const int end = begin + share < tiles_all ? begin + share : tiles_all;
    const int steps = (end - begin + KG - 1) / KG;           // every group runs every step; a step beyond the share multiplies zeros
    u32x4_t ring[kRing][8];
    auto bounded = [](const T* base, int64_t rows, int ld, int cols) {
        const int64_t bytes = ((rows - 1) * ld + cols) * (int64_t)E;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    auto whole = [](int cols) { return (cols + V - 1) / V * V; };      // a padded row's last packet
    // The loads of a k-tile are the same straight line for every wave - descriptor, eight lane offsets, one scalar offset that
    // advances with k - so that the compiler counts them and a wait for the oldest tile leaves the younger ones in flight.
    const bool turned = for_b || TA;                         // this wave's operand is stored k-row by k-row
    const __amdgpu_buffer_rsrc_t r0 = for_b ? bounded(B0, K, ldb, N)
                                            : (TA ? bounded(A, K, lda, whole(M)) : bounded(A + (int64_t)m0 * lda, M - m0, lda, whole(K * segments)));
    const __amdgpu_buffer_rsrc_t r1 = for_b && segments > 1 ? bounded(B1, K, ldb, N) : r0;
    const int ld = for_b ? ldb : lda, x0 = for_b ? n0 : m0, X = for_b ? N : M;
    const int k_bytes = turned ? ld * E : E;                 // bytes per k value
    const int seg_bytes = turned ? 0 : K * E;                // second range: further along A's rows, or in B1
    const int k_first = turned ? 0 : (t % KCH) * V;          // k of this lane's packets inside a tile, for the k tail of a row
    uint32_t off[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int nb = t % NB, kb = t / NB, qr = t + i * 128;
        const uint32_t block = x0 + nb * V < X ? (uint32_t)((kb * V + i) * ld + x0 + nb * V) * (uint32_t)E : kOutOfRange;
        off[i] = turned ? block : (uint32_t)((qr / KCH) * lda + k_first) * (uint32_t)E;
    }
    auto load = [&](int step, u32x4_t (&reg)[8]) {
        const int kt = begin + step * KG + grp;
        const int seg = kt >= tiles_k ? 1 : 0, k0 = (kt - seg * tiles_k) * KT;
        const bool drop = kt >= end || k0 + k_first >= K;
        const __amdgpu_buffer_rsrc_t r = seg ? r1 : r0;
        const int at = kt >= end ? 0 : k0 * k_bytes + seg * seg_bytes;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            reg[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(drop ? kOutOfRange : off[i]), at, 0));
    };
    auto store = [&](u32x4_t (&reg)[8], u32x4_t* tile_mem) {
        if (turned) {
            const int nb = t % NB, kb = t / NB;
#pragma unroll
            for (int j = 0; j < V; ++j) {
                u32x4_t out;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    out[r] = __builtin_amdgcn_perm(reg[2 * r + 1][j / 2], reg[2 * r][j / 2], (j & 1) ? 0x07060302u : 0x05040100u);
                tile_mem[slot(nb * V + j, kb)] = out;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int q = t + i * 128;
                tile_mem[slot(q / KCH, q % KCH)] = reg[i];
            }
        }
    };

    f32x4_t acc[F][F];
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int wm = wave >> 1, wn = wave & 1, frow = lane & 15, piece = lane >> 4;
#pragma unroll
    for (int d = 0; d < kRing; ++d) load(d, ring[d]);
    store(ring[0], lds[0][for_b]);
    load(kRing, ring[0]);
    __syncthreads();
    // step s multiplies from lds[s % 2] while the tile of step s + 1 leaves its registers for the other half; unrolled so that the
    // ring position is a compile-time index
    for (int s0 = 0; s0 < steps; s0 += 2 * kRing) {
#pragma unroll
        for (int d = 0; d < 2 * kRing; ++d) {
            const int s = s0 + d;
            if (s >= steps) break;
            const u32x4_t *as = lds[d % 2][0], *bs = lds[d % 2][1];
#pragma unroll
            for (int ks = 0; ks < KCH / 4; ++ks) {
                u32x4_t fa[F], fb[F];
#pragma unroll
                for (int i = 0; i < F; ++i) fa[i] = as[slot(wm * W + i * 16 + frow, ks * 4 + piece)];
#pragma unroll
                for (int j = 0; j < F; ++j) fb[j] = bs[slot(wn * W + j * 16 + frow, ks * 4 + piece)];
#pragma unroll
                for (int i = 0; i < F; ++i)
#pragma unroll
                    for (int j = 0; j < F; ++j) acc[i][j] = mfma16_packet<T>(fa[i], fb[j], acc[i][j]);
            }
            store(ring[(d + 1) % kRing], lds[(d + 1) % 2][for_b]);      // after the last step: zeros nobody reads
            load(s + 1 + kRing, ring[(d + 1) % kRing]);
            __syncthreads();
        }
    }
    if constexpr (KG > 1) {
        f32x4_t* sums = reinterpret_cast<f32x4_t*>(&lds_all[0][0][0][0]);      // the loop's last barrier has passed: free
        static_assert((KG - 1) * 4 * F * F * 64 <= KG * 2 * 2 * BR * KCH, "the groups' sums fit the tiles' memory");
        if (grp > 0) {
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int j = 0; j < F; ++j) sums[(((grp - 1) * 4 + wave) * F * F + i * F + j) * 64 + lane] = acc[i][j];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 1; g < KG; ++g)
#pragma unroll
            for (int i = 0; i < F; ++i)
#pragma unroll
                for (int j = 0; j < F; ++j) acc[i][j] += sums[(((g - 1) * 4 + wave) * F * F + i * F + j) * 64 + lane];
    }
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < F; ++j) {
            const int col = n0 + wn * W + j * 16 + frow;
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = m0 + wm * W + i * 16 + 4 * piece + v;
                if (row >= M || col >= N) continue;
                if (splits > 1) partial[((int64_t)split * M + row) * N + col] = acc[i][j][v];
                else C[(int64_t)row * ldc + col] = Elem<T>::from_f32(acc[i][j][v]);
            }
        }
}

// C = sum over the splits, in order; one packet of C per thread
template <typename T>
__global__ __launch_bounds__(256) void gemm_tr_add_kernel(const float* __restrict__ partial, T* __restrict__ C, int ldc, int64_t packets,
                                                          int packets_per_row, int64_t plane, int splits) {
    constexpr int V = Elem<T>::kVec;
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= packets) return;
    float v[V];
#pragma unroll
    for (int e = 0; e < V; ++e) v[e] = 0.0f;
    for (int s = 0; s < splits; ++s)
#pragma unroll
        for (int h = 0; h < V; h += 4) {
            const f32x4_t p = *reinterpret_cast<const f32x4_t*>(partial + s * plane + i * V + h);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[h + e] += p[e];
        }
    *reinterpret_cast<u32x4_t*>(C + i / packets_per_row * ldc + i % packets_per_row * V) = pack16<T>(v);
}

// Tile side: 128 x 128 once they give every CU one, 64 x 64 (with twice the k depth per k-tile) for fewer.  With at most one
// 64 x 64 tile per CU and a long k loop (1024 values and more) two k groups; with at most one per four CUs the k range is split
// over workgroups (a second launch adds their sums) as long as each keeps eight k-tiles.
struct TrPlan { int rows, groups, splits; };
TrPlan plan_tr(int layout, int M, int N, int K, int segments) {
    const int cus = chip_info().cus;
    auto tiles = [&](int rows) { return (int64_t)((M + rows - 1) / rows) * ((N + rows - 1) / rows); };
    TrPlan p = {tiles(128) >= cus ? 128 : 64, 1, 1};
    if (p.rows == 64) {
        const int64_t by_chip = cus / tiles(64), by_k = (int64_t)segments * ((K + 127) / 128) / 8;
        const int64_t s = by_chip < by_k ? by_chip : by_k;
        if (by_chip >= 4) p.splits = (int)(s < 1 ? 1 : (s > 16 ? 16 : s));
        else if (by_chip >= 1 && layout == kBlasNN && (int64_t)K * segments >= 1024) p.groups = 2;
    }
    return p;
}

template <typename T, bool TA>
void launch_gemm_tr(const void* A, int lda, const void* B0, const void* B1, int ldb, void* C, int ldc, int M, int N, int K, int segments,
                    TrPlan p, float* partial, hipStream_t stream) {
    const int xcds = chip_info().xcds;
    const int tm = (M + p.rows - 1) / p.rows, tn = (N + p.rows - 1) / p.rows;
    const dim3 grid((unsigned)(tm * tn), (unsigned)p.splits);
#define FMOE_LAUNCH_TR(BR, KCH, KG)                                                                                              \
    hipLaunchKernelGGL((gemm_tr_kernel<T, TA, BR, KCH, KG>), grid, dim3(256 * (KG)), 0, stream, (const T*)A, lda, (const T*)B0,    \
                       (const T*)B1, ldb, (T*)C, ldc, partial, M, N, K, segments, tm, tn, p.splits, xcds)
    if (p.rows == 128) FMOE_LAUNCH_TR(128, 8, 1);
    else if (p.groups == 2) FMOE_LAUNCH_TR(64, 16, 2);
    else FMOE_LAUNCH_TR(64, 16, 1);
#undef FMOE_LAUNCH_TR
    if (p.splits > 1) {
        const int64_t packets = (int64_t)M * N / Elem<T>::kVec;
        hipLaunchKernelGGL((gemm_tr_add_kernel<T>), dim3((unsigned)((packets + 255) / 256)), dim3(256), 0, stream, (const float*)partial, (T*)C,
                           ldc, packets, N / Elem<T>::kVec, (int64_t)M * N, p.splits);
    }
}

// Up to here the products are short enough for this kernel to be the faster one (8.6 GFLOP: 21 to 23 us against the library's 18).
constexpr double kOwnGemmFlops = 5e9;
bool own_kernel_pays(int M, int N, int K, int segments, int dtype) {
    return dtype != FMOE_F32 && 2.0 * M * N * (double)K * segments <= kOwnGemmFlops;
}

}  // namespace

size_t gemm_backward_workspace_bytes(int layout, int M, int N, int K, int segments, int dtype) {
    if (!own_kernel_pays(M, N, K, segments, dtype)) return 0;
    const int splits = plan_tr(layout, M, N, K, segments).splits;
    return splits > 1 ? (size_t)splits * M * N * sizeof(float) : 0;
}

bool gemm_backward_own(int M, int N, int K, int dtype) { return own_kernel_pays(M, N, K, 1, dtype); }

int gemm_backward(int layout, int M, int N, int K, const void* A, int lda, const void* B0, const void* B1, int ldb, void* C, int ldc,
                  int dtype, void* workspace, size_t workspace_bytes, hipStream_t stream) {
    const int segments = B1 != nullptr ? 2 : 1;
    // whole packets: where M (TN) or K (NN) is none, the rows of A are padded with zeros up to lda
    const int a_cols = layout == kBlasTN ? M : K * segments;
    const bool packets = lda % 8 == 0 && ldb % 8 == 0 && ldc % 8 == 0 && N % 8 == 0 && (a_cols + 7) / 8 * 8 <= lda && (segments == 1 || K % 8 == 0) &&
                         aligned16(A) && aligned16(B0) && aligned16(B1) && aligned16(C);
    // 32-bit byte offsets inside a descriptor
    const bool reach = (double)K * ldb < 1.0e9 && (layout == kBlasTN ? (double)K * lda < 1.0e9 : 256.0 * lda < 1.0e9);
    if (packets && reach && own_kernel_pays(M, N, K, segments, dtype)) {
        TrPlan p = plan_tr(layout, M, N, K, segments);
        if ((size_t)p.splits * M * N * sizeof(float) > workspace_bytes) p.splits = 1;
        float* partial = (float*)workspace;
#define FMOE_TR(TT, TA) launch_gemm_tr<TT, TA>(A, lda, B0, B1, ldb, C, ldc, M, N, K, segments, p, partial, stream)
        if (layout == kBlasTN) {
            if (dtype == FMOE_BF16) FMOE_TR(bf16_t, true);
            else FMOE_TR(f16_t, true);
        } else {
            if (dtype == FMOE_BF16) FMOE_TR(bf16_t, false);
            else FMOE_TR(f16_t, false);
        }
#undef FMOE_TR
        FMOE_CHECK_LAUNCH("backward product");
        return FMOE_OK;
    }
    if (int rc = blas_gemm(layout, M, N, K, A, lda, B0, ldb, C, ldc, 0.0f, dtype, stream)) return rc;
    if (B1 == nullptr) return FMOE_OK;
    return blas_gemm(layout, M, N, K, (const char*)A + (size_t)K * dtype_size(dtype), lda, B1, ldb, C, ldc, 1.0f, dtype, stream);
}

}  // namespace fmoe
