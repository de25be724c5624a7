// Tiles of C[M,N] = A[M,K] * B[N,K]^T on the matrix cores (gfx950), the parts of kernels that form such products: the shared MLP
// (fmoe_mlp.hip) and the launches that put a product beside other work (fmoe_small.hip).  `block` of `blocks` workgroups; lds: kSplitLds bytes
// of the kernel's memory.
#pragma once

#include "fmoe_common.h"
#include "fmoe_mfma.h"
#include "fmoe_vec.h"

namespace fmoe {
namespace {

enum Epilogue { kEpiSwiGLU = 0, kEpiPlain = 1, kEpiDual = 2, kEpiPart = 3, kEpiGradient = 4 };   // Dual: the product in T and, through R, in fp32
// kEpiGradient: the product is dh = dy Wd and is not stored; with the forward's products a = x Wg^T and b = x Wu^T it becomes the
// gradients da and db (rows ld apart) and h = silu(a) * b, all [M,N].
template <typename T> struct GradientPlanes {
    const T *a, *b;
    T *da, *db, *h;
    int ld;
};
template <bool B> struct Flag { static constexpr bool value = B; };
constexpr uint32_t kOutOfRange = 0x80000000u;    // beyond every buffer descriptor here: loads give zeros, stores are dropped

// The stages of a kernel's pipeline tiles.  The memory is reached by this function, not through a pointer handed down: with a pointer
// the compiler schedules the address arithmetic of the 256 x 256 tiles differently, which costs the large products 1 to 2 %.
template <typename T, int N> struct DmaLds {
    __device__ __forceinline__ static T* at() {
        __shared__ __attribute__((aligned(1024))) T stages[N];
        return stages;
    }
};
// The hardware reciprocal (1 ulp) instead of a division: the results are rounded to 16 bits.
__device__ __forceinline__ void swiglu_gradient(float dc, float a, float b, float& da, float& db, float& h) {
    const float sig = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(a * -1.44269504088896340736f)), silu = a * sig;
    db = dc * silu;
    da = dc * (silu * (1.0f - sig) + sig) * b;
    h = silu * b;
}
// Position of item t of n in the order the XCDs walk: XCD x (workgroup id mod xcds) takes a contiguous run, so that what its items share
// passes into its L2 once.  A permutation of [0, n) for every n.
__host__ __device__ __forceinline__ int xcd_run(int t, int n, int xcds) {
    const uint32_t x = (uint32_t)t % (uint32_t)xcds, each = (uint32_t)n / (uint32_t)xcds, more = (uint32_t)n % (uint32_t)xcds;
    return (int)(x * each + (x < more ? x : more) + (uint32_t)t / (uint32_t)xcds);
}

// Products whose number of tiles is no multiple of the XCDs, neither operand turned: runs where the operands are larger than this, two and
// a half times an XCD's L2, else the order as it is.  What every XCD fetches bounds the large ones: 816 tokens, 1320 -> 2640 (gate, up
// and down, bf16 or fp16) 51.7 -> 39.4 us, 337 tokens, 2192 -> 8768 76 -> 59, 1819 tokens, 1792 -> 4776 140 -> 118, 8000 tokens,
// 320 -> 848 32.4 -> 29.8; over 71 extents 2 % less, the worst 3 % more, as much as code that takes the same order differs by.  The
// small ones lie in every L2 in any order and took up to 10 % longer in runs: 1154 tokens, 392 -> 784 12.6 -> 13.9, 1500 tokens,
// 640 -> 1704 23.7 -> 24.9.
constexpr int64_t kRunBytes = 10 << 20;

constexpr int kSplitWaves = 8;
template <int MT, int NT, int EPI> constexpr int kSplitLds = kSplitWaves * MT * NT * (EPI == kEpiSwiGLU ? 2 : 1) * 64 * 16;

// ------------------------------------------------------------------------------------------------------------
// LDS-DMA pipelined kernel.  WAVES_M x WAVES_N waves, each (BM/WAVES_M) x (BN/WAVES_N); BKT = k extent of a stage.
// ------------------------------------------------------------------------------------------------------------
// FR: fragment shape (32: v_mfma_f32_32x32x16 / 32x32x2; 16: v_mfma_f32_16x16x32).
template <typename T, int BM, int BN, int WAVES_M, int WAVES_N, int BKT, int NSTAGE, int EPI, int PF, int FR, bool RAGGED, bool SLICED = false,
          bool TA = false, bool TB = false>
__device__ __forceinline__ void gemm_dma_tiles(
    const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1, T* __restrict__ C,
    const T* __restrict__ R, int M, int N, int K, int tiles_m, int tiles_n, int xcds, int block, int blocks, int slice = 0, int slices = 1,
    int lda = 0, int ldb = 0, int segments = 1, const GradientPlanes<T>& grad = {}) {
    using Shape = MfmaShape<T, FR>;
    using Frag = typename Shape::Frag;
    using Acc = typename Shape::Acc;
    constexpr int NV = Shape::kAccRegs;
    constexpr int NWAVES = WAVES_M * WAVES_N;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, MF = WM / FR, NF = WN / FR;
    constexpr int EPC = 16 / (int)sizeof(T);        // elements per 16-byte chunk
    constexpr int CPR = BKT / EPC;                  // 16-byte chunks per LDS row
    constexpr int RPI = 64 / CPR;                   // rows one wave-wide DMA load covers
    constexpr int ROWS_PER_IT = NWAVES * RPI;       // rows all waves cover per DMA round
    constexpr int STAGE = (BM + BN) * BKT;          // elements per stage
    constexpr int KSTEPS = BKT / (Shape::kChunks * EPC);   // a k-step is kChunks 16-byte pieces of a row: one per lane group
    static_assert(WM % FR == 0 && WN % FR == 0, "fragments tile the wave tile");
    constexpr int ROW_SHIFT = (CPR == 8) ? 1 : 2;   // log2(rows per 256 bytes)
    constexpr int BN_OUT = (EPI == kEpiSwiGLU) ? BN / 2 : BN;
    constexpr int A_ROUNDS = BM / ROWS_PER_IT, B_ROUNDS = BN / ROWS_PER_IT;
    constexpr int DMA_PER_TILE = A_ROUNDS + B_ROUNDS;
    // Turned operands (TA, TB) lie k-row by k-row: a stage holds them as they lie, BKT rows of BM (BN) values.  16-bit: a lane's 8 k
    // values come from two transposing LDS reads (lane l of 16 addresses piece l % 4 of row l / 4, and receives column l of the four
    // rows); fp32: from four plain ones, one per k value.  The 16-byte chunks of a row are XOR-ed with a key of the row number, so
    // that the rows a wave-wide read touches lie in different banks.  NN (TB only) may have a second range of K values, in A
    // further along the rows and in B1.
    constexpr bool kTurned = TA || TB;
    static_assert(!kTurned || (RAGGED && ((sizeof(T) == 2 && FR == 16 && BKT == 64) || (sizeof(T) == 4 && FR == 32 && BKT == 32)) &&
                               EPI != kEpiSwiGLU && EPI != kEpiDual), "turned operands");
    constexpr int CHA = BM / EPC, CHB = BN / EPC;    // 16-byte chunks of a k-row
    auto row_key = [](int k, int chunks) {
        if (sizeof(T) == 4) return ((k >> 2) & 1) << 3;
        return chunks >= 16 ? ((k & 3) | ((k >> 3) & 1) << 2) << 1 : (((k >> 1) & 1) | ((k >> 3) & 1) << 1) << 1;
    };
    static_assert(CPR == 4 || CPR == 8, "stage depth: LDS rows of 64 or 128 bytes");
    static_assert(ROWS_PER_IT % 16 == 0 && BM % ROWS_PER_IT == 0 && BN % ROWS_PER_IT == 0, "DMA rounds");
    static_assert(EPI != kEpiSwiGLU || ((BN / 2) % ROWS_PER_IT == 0 && NF % 2 == 0), "gate/up split");
    static_assert((NSTAGE - 2) * DMA_PER_TILE < 64, "vmcnt range");

    using Lds = DmaLds<T, NSTAGE * STAGE>;

    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const int num_tiles = tiles_m * tiles_n;

    // DMA: the lane's LDS position is row (round*ROWS_PER_IT + wave*RPI + lrow), physical chunk lp; it holds the
    // logical chunk lp ^ key(row), key(row) = (row >> ROW_SHIFT) & (CPR-1).  ROWS_PER_IT is a multiple of 16, so the
    // key does not depend on the round and one element offset per lane serves every load.
    const int lrow = lane / CPR, lp = lane % CPR;
    const int key_dma = ((wave * RPI + lrow) >> ROW_SHIFT) & (CPR - 1);
    const uint32_t lane_off = (uint32_t)(lrow * K + (lp ^ key_dma) * EPC) * (uint32_t)sizeof(T);   // bytes
    // turned: the lane's row of the round and logical chunk; rounds cover a multiple of 16 rows (8 in fp32), so the key is the same in all
    const int ta_row = wave * (64 / CHA) + lane / CHA, tb_row = wave * (64 / CHB) + lane / CHB;
    const uint32_t ta_off = (uint32_t)(ta_row * lda + ((lane % CHA) ^ row_key(ta_row, CHA)) * EPC) * (uint32_t)sizeof(T);
    const uint32_t tb_off = (uint32_t)(tb_row * ldb + ((lane % CHB) ^ row_key(tb_row, CHB)) * EPC) * (uint32_t)sizeof(T);
    // A rows beyond M (a ragged last tile row) are read from row M-1 instead: one byte offset per DMA round, set per
    // tile.  What the MFMAs make of those rows is never stored (the epilogue's buffer stores are bounds-checked).
    uint32_t a_lane_off[A_ROUNDS];
    const T *a_src, *b_src0, *b_src1 = nullptr;
    // RAGGED: rows and the k tail are cut off by the range check of buffer descriptors over the rest of each matrix
    __amdgpu_buffer_rsrc_t a_rsrc, b_rsrc0, b_rsrc1;
    int m0, n0;
    // SLICED: k-tiles [k_first, k_first + k_tiles) of the product (every slice has some), one tile per workgroup
    static_assert(!SLICED || (RAGGED && EPI == kEpiPart), "slices of k leave partial sums");
    const int k_range = (K + BKT - 1) / BKT;                     // k-tiles of a range of K values
    const int k_all = kTurned ? k_range * segments : k_range, k_share = SLICED ? (k_all + slices - 1) / slices : k_all, k_first = SLICED ? slice * k_share : 0;
    const int k_tiles = SLICED ? (k_all - k_first < k_share ? k_all - k_first : k_share) : (kTurned ? k_all : (K + BKT - 1) / BKT);
    if (SLICED && kTurned) C = reinterpret_cast<T*>(reinterpret_cast<float*>(C) + (int64_t)slice * M * N);
    if (SLICED && !kTurned) {
        A += k_first * BKT;
        B0 += k_first * BKT;
        C = reinterpret_cast<T*>(reinterpret_cast<float*>(C) + (int64_t)slice * M * N);
    }
    const bool lane_in_tail = kTurned ? (k_range - 1) * BKT + (lp ^ key_dma) * EPC < K : (k_first + k_tiles - 1) * BKT + (lp ^ key_dma) * EPC < K;      // the lane's chunk of the last k-tile exists
    auto rest_of = [&](const T* base, int64_t rows) {                              // descriptor from `base` to the end of its matrix
        const int64_t bytes = SLICED ? (rows * K - k_first * BKT) * (int64_t)sizeof(T) : rows * K * (int64_t)sizeof(T);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    auto rest_of_rows = [&](const T* base, int64_t rows, int ld, int cols) {        // turned launches: rows of `cols` values, ld apart
        const int64_t bytes = rows > 0 ? ((rows - 1) * ld + cols) * (int64_t)sizeof(T) : 0;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    // The workgroup is persistent: it takes tiles t, t + blocks, ...  Each XCD (workgroup id mod 8) gets a contiguous
    // run of the tile order, walked 8 tile-rows at a time so that a compact patch shares A and B tiles in the XCD's L2.
    // Turned products take runs whatever their number of tiles: backward passes of 777 tokens, 2048 -> 5464 252 -> 236 us, 8000 tokens,
    // 320 -> 848 125 -> 112, 546 tokens, 1304 -> 2608 106 -> 97, none slower.
    const bool runs = kTurned || (uint32_t)num_tiles % (uint32_t)xcds == 0 || ((int64_t)M + (EPI == kEpiSwiGLU ? 2 : 1) * (int64_t)N) * K * (int64_t)sizeof(T) > kRunBytes;
    auto set_tile = [&](int t) {
        if (runs) t = xcd_run(t, num_tiles, xcds);
        constexpr int GM = 8;
        const int width = GM * tiles_n, group = t / width, first_m = group * GM;
        const int gsz = (tiles_m - first_m) < GM ? (tiles_m - first_m) : GM;
        m0 = (first_m + (t % width) % gsz) * BM;
        n0 = ((t % width) / gsz) * BN_OUT;
        a_src = A + (int64_t)m0 * K;                     // wave-uniform; the lane's part is the 32-bit a_lane_off[r]
#pragma unroll
        for (int r = 0; r < A_ROUNDS; ++r) {
            int row = r * ROWS_PER_IT + wave * RPI + lrow;
            if (!RAGGED) row = m0 + row < M ? row : M - 1 - m0;
            a_lane_off[r] = (uint32_t)(row * (kTurned ? lda : K) + (lp ^ key_dma) * EPC) * (uint32_t)sizeof(T);
        }
        if constexpr (kTurned) {
            auto packets = [](int cols) { return (cols + EPC - 1) / EPC * EPC; };      // A's rows are padded to whole chunks
            a_rsrc = TA ? rest_of_rows(A + m0, K, lda, packets(M - m0)) : rest_of_rows(A + (int64_t)m0 * lda, M - m0, lda, packets(K * segments));
            static_assert(TB, "B is turned wherever A may be");
            b_rsrc0 = rest_of_rows(B0 + n0, K, ldb, N - n0);
            b_rsrc1 = segments > 1 ? rest_of_rows(B1 + n0, K, ldb, N - n0) : b_rsrc0;
            return;
        }
        b_src0 = B0 + (int64_t)(n0 + wave * RPI) * K;
        if (EPI == kEpiSwiGLU) b_src1 = B1 + (int64_t)(n0 + wave * RPI) * K;
        if constexpr (RAGGED) {
            a_rsrc = rest_of(a_src, M - m0);
            b_rsrc0 = rest_of(B0 + (int64_t)n0 * K, N - n0);
            if (EPI == kEpiSwiGLU) b_rsrc1 = rest_of(B1 + (int64_t)n0 * K, N - n0);
        }
    };
    auto issue = [&](int kt, T* stage) {
        const int k0 = kt * BKT;
        if constexpr (kTurned) {
            const int at = k_first + kt, seg = at >= k_range ? 1 : 0, kr = at - seg * k_range;
            const bool drop = kr + 1 == k_range && !lane_in_tail;
#pragma unroll
            for (int r = 0; r < A_ROUNDS; ++r)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    a_rsrc, (__attribute__((address_space(3))) void*)(stage + (r * ROWS_PER_IT + wave * RPI) * BKT), 16,
                    (int)(TA ? ta_off : (drop ? kOutOfRange : a_lane_off[r])),
                    TA ? (kr * BKT + r * (BKT / A_ROUNDS)) * lda * (int)sizeof(T) : (seg * K + kr * BKT) * (int)sizeof(T), 0, 0);
            const __amdgpu_buffer_rsrc_t b = seg ? b_rsrc1 : b_rsrc0;
#pragma unroll
            for (int r = 0; r < B_ROUNDS; ++r)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    b, (__attribute__((address_space(3))) void*)(stage + BM * BKT + (r * ROWS_PER_IT + wave * RPI) * BKT), 16, (int)tb_off,
                    (kr * BKT + r * (BKT / B_ROUNDS)) * ldb * (int)sizeof(T), 0, 0);
            return;
        }
        if constexpr (RAGGED) {
            const bool drop = kt + 1 == k_tiles && !lane_in_tail;
#pragma unroll
            for (int r = 0; r < A_ROUNDS; ++r)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    a_rsrc, (__attribute__((address_space(3))) void*)(stage + (r * ROWS_PER_IT + wave * RPI) * BKT), 16,
                    (int)(drop ? kOutOfRange : a_lane_off[r]), k0 * (int)sizeof(T), 0, 0);
#pragma unroll
            for (int r = 0; r < B_ROUNDS; ++r) {
                const bool second = EPI == kEpiSwiGLU && r >= B_ROUNDS / 2;
                const uint32_t off = (uint32_t)(((second ? r - B_ROUNDS / 2 : r) * ROWS_PER_IT + wave * RPI) * K) * (uint32_t)sizeof(T) + lane_off;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    second ? b_rsrc1 : b_rsrc0,
                    (__attribute__((address_space(3))) void*)(stage + BM * BKT + (r * ROWS_PER_IT + wave * RPI) * BKT), 16,
                    (int)(drop ? kOutOfRange : off), k0 * (int)sizeof(T), 0, 0);
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < A_ROUNDS; ++r)
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)((const char*)(a_src + k0) + a_lane_off[r]),
                (__attribute__((address_space(3))) void*)(stage + (r * ROWS_PER_IT + wave * RPI) * BKT), 16, 0, 0);
#pragma unroll
        for (int r = 0; r < B_ROUNDS; ++r) {
            const T* src;
            if (EPI == kEpiSwiGLU && r >= B_ROUNDS / 2) src = b_src1 + (int64_t)(r - B_ROUNDS / 2) * ROWS_PER_IT * K + k0;
            else src = b_src0 + (int64_t)r * ROWS_PER_IT * K + k0;
            __builtin_amdgcn_global_load_lds(
                (const __attribute__((address_space(1))) void*)((const char*)src + lane_off),
                (__attribute__((address_space(3))) void*)(stage + BM * BKT + (r * ROWS_PER_IT + wave * RPI) * BKT), 16, 0, 0);
        }
    };

    // Fragment rows of a lane are (multiple of FR) + frow: the swizzle key is the same for all of them, so the
    // address is (row base + one per-k-step offset) + an immediate per fragment.
    const int frow = lane % FR, fhalf = lane / FR;       // fhalf: which 16-byte piece of a k-step the lane supplies
    const int key_f = (frow >> ROW_SHIFT) & (CPR - 1);
    const int a_row_bytes = (wm * WM + frow) * BKT * (int)sizeof(T);
    int b_row_bytes[NF];
#pragma unroll
    for (int j = 0; j < NF; ++j) {
        int row;
        if (EPI == kEpiSwiGLU) row = (j < NF / 2) ? wn * (WN / 2) + j * FR : BN / 2 + wn * (WN / 2) + (j - NF / 2) * FR;
        else row = wn * WN + j * FR;
        b_row_bytes[j] = (BM + row + frow) * BKT * (int)sizeof(T);
    }
    int pc[KSTEPS];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) pc[ks] = ((ks * Shape::kChunks + fhalf) ^ key_f) << 4;

    // turned: byte address of the lane's piece in fragment 0's place; bits 5 to 7 (7 in fp32) of it are XOR-ed per fragment
    const int t_row = sizeof(T) == 4 ? fhalf * 4 : fhalf * 8 + frow / 4, t_piece = sizeof(T) == 4 ? frow * 4 : (frow % 4) * 8;
    const int ta_lane = t_row * BM * (int)sizeof(T) + (row_key(t_row, CHA) * 16 ^ t_piece);
    const int tb_lane = BM * BKT * (int)sizeof(T) + t_row * BN * (int)sizeof(T) + (row_key(t_row, CHB) * 16 ^ t_piece);
    auto turned_frag = [&](const char* stage, int lane_at, int piece, int ks, int cols) {
        constexpr int kBytes = FR * (int)sizeof(T), kInKey = 256 / kBytes;       // bytes of a fragment's columns in a k-row
        const char* at = stage + (lane_at ^ ((piece % kInKey) * kBytes)) + (piece / kInKey) * 256 + ks * (BKT / KSTEPS) * cols * (int)sizeof(T);
        if constexpr (sizeof(T) == 4) {
            Frag f;
#pragma unroll
            for (int q = 0; q < 4; ++q) f[q] = *reinterpret_cast<const float*>(at + q * cols * 4);
            return f;
        } else {
            typedef short i16x4_t __attribute__((__vector_size__(8)));
            typedef short i16x8_t __attribute__((__vector_size__(16)));
            typedef __attribute__((address_space(3))) i16x4_t* tr_ptr;
            const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at);
            const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 4 * cols * (int)sizeof(T)));
            const i16x8_t both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            return __builtin_bit_cast(Frag, both);
        }
    };

    int tile = block;
    if (tile >= num_tiles) return;
    set_tile(tile);
#pragma unroll
    for (int s = 0; s < NSTAGE - 1; ++s)
        if (s < k_tiles) issue(s, Lds::at() + s * STAGE);

    // Fragments of k-step q+PF are read from LDS while the MFMAs of k-step q run (PF+1 register buffers); the read-ahead crosses k-tile boundaries, so the barrier
    // that publishes the next stage sits PF steps before the end of a k-tile and the matrix pipe always has work queued
    // while a wave waits.
    constexpr int RING = PF + 1;
    static_assert(KSTEPS % RING == 0 && PF >= 1 && PF < KSTEPS + 1, "fragment buffers rotate with period RING");
    Frag fa[RING][MF], fb[RING][NF];
    auto read_frags = [&](const char* stage, int ks, Frag (&a)[MF], Frag (&b)[NF]) {
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            if constexpr (TA) a[i] = turned_frag(stage, ta_lane, wm * (WM / FR) + i, ks, BM);
            else a[i] = *reinterpret_cast<const Frag*>(stage + a_row_bytes + pc[ks] + i * FR * BKT * (int)sizeof(T));
        }
#pragma unroll
        for (int j = 0; j < NF; ++j) {
            if constexpr (TB) b[j] = turned_frag(stage, tb_lane, wn * (WN / FR) + j, ks, BN);
            else b[j] = *reinterpret_cast<const Frag*>(stage + b_row_bytes[j] + pc[ks]);
        }
    };
    // Entering k-tile kt (kt = 0: from the tile prologue): my share of its stage has landed once at most the loads of
    // the NSTAGE-2 younger k-tiles are outstanding; my reads of the stage that is overwritten next are complete (all
    // reads of k-tile kt-1 have been issued by then); after the barrier both hold for every wave, so the load of k-tile
    // kt+NSTAGE-1 can go into the stage kt-1 used.
    auto enter_k_tile = [&](int kt) {
        constexpr int kKeep = (NSTAGE - 2) * DMA_PER_TILE;
        if (kt + NSTAGE - 2 < k_tiles) __builtin_amdgcn_s_waitcnt(0x0070 | (kKeep & 0xF) | ((kKeep >> 4) << 14));
        else __builtin_amdgcn_s_waitcnt(0x0070);
        __builtin_amdgcn_s_barrier();
        if (kt + NSTAGE - 1 < k_tiles) issue(kt + NSTAGE - 1, Lds::at() + ((kt + NSTAGE - 1) % NSTAGE) * STAGE);
    };
    while (true) {
        Acc acc[MF][NF];
#pragma unroll
        for (int i = 0; i < MF; ++i)
#pragma unroll
            for (int j = 0; j < NF; ++j)
#pragma unroll
                for (int v = 0; v < NV; ++v) acc[i][j][v] = 0.0f;

        enter_k_tile(0);
#pragma unroll
        for (int s = 0; s < PF; ++s) read_frags(reinterpret_cast<const char*>(Lds::at()), s, fa[s % RING], fb[s % RING]);
        // the last k-tile has no successor to read ahead into: it is a separate copy of the body, so that no branch
        // merges a path with reads in flight into the MFMA sequence
        auto k_tile_body = [&](int kt, auto last_tag) {
            constexpr bool kLast = decltype(last_tag)::value;
            const char* stage = reinterpret_cast<const char*>(Lds::at() + (kt % NSTAGE) * STAGE);
            const char* next_stage = reinterpret_cast<const char*>(Lds::at() + ((kt + 1) % NSTAGE) * STAGE);
#pragma unroll
            for (int q = 0; q < KSTEPS; ++q) {
                const int nxt = q + PF;
                constexpr int kMfmas = MF * NF;     // runs of Shape::kInstr instructions
                const bool reads = nxt < KSTEPS || !kLast;
                constexpr int RT = sizeof(T) == 4 ? 4 : 2, RA = TA ? RT : 1, RB = TB ? RT : 1;       // LDS reads per fragment
                constexpr int n_reads = RA * MF + RB * NF;
                __builtin_amdgcn_sched_barrier(0);
                if (nxt < KSTEPS) {
                    read_frags(stage, nxt, fa[nxt % RING], fb[nxt % RING]);
                } else if (!kLast) {
                    if (nxt == KSTEPS) {
                        enter_k_tile(kt + 1);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    read_frags(next_stage, nxt - KSTEPS, fa[nxt % RING], fb[nxt % RING]);
                }
#pragma unroll
                for (int i = 0; i < MF; ++i)
#pragma unroll
                    for (int j = 0; j < NF; ++j) {
                        // exchanged, a lane receives four successive columns of C instead of four rows
                        if constexpr (EPI == kEpiGradient) acc[i][j] = Shape::run(fb[q % RING][j], fa[q % RING][i], acc[i][j]);
                        else acc[i][j] = Shape::run(fa[q % RING][i], fb[q % RING][j], acc[i][j]);
                    }
                // issue order: the LDS reads spread evenly behind the MFMAs
                constexpr int kPer = (n_reads + kMfmas - 1) / kMfmas;
#pragma unroll
                for (int m = 0; m < kMfmas; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x008, Shape::kInstr, 0);
                    if (reads && m * kPer < n_reads) __builtin_amdgcn_sched_group_barrier(0x100, kPer, 0);
                }
            }
        };
        for (int kt = 0; kt + 1 < k_tiles; ++kt) k_tile_body(kt, Flag<false>{});
        k_tile_body(k_tiles - 1, Flag<true>{});
        __builtin_amdgcn_sched_barrier(0);

        // start the next tile's first stages before this tile's epilogue, so that its global-load latency is covered
        const int out_m0 = m0, out_n0 = n0;
        const int next = tile + blocks;
        if (next < num_tiles) {
            set_tile(next);
            __builtin_amdgcn_s_barrier();     // every wave has consumed its reads of the last stage
#pragma unroll
            for (int s = 0; s < NSTAGE - 1; ++s)
                if (s < k_tiles) issue(s, Lds::at() + s * STAGE);
        }

        if constexpr (EPI == kEpiGradient) {
            // Lane l has row l % 16 and columns 4 (l / 16) .. + 3 of every fragment; rows of 16 lanes swap words between two fragments so
            // that loads and stores are of 16 bytes (a lane's eight successive columns of one of them), the arithmetic in the lanes'
            // own layout.  Offsets in the vector register alone: see fmoe_gemm256.h.
            static_assert(sizeof(T) == 2 && FR == 16 && TB && !TA && NF % 2 == 0, "gradient epilogue");
            const int row0 = out_m0 + wm * WM, col0 = out_n0 + wn * WN + (fhalf & 1) * 16 + (fhalf >> 1) * 8;
            const int rows = M - row0;
            auto plane = [&](const T* base, int ld) {
                const int64_t span = rows > 0 ? ((int64_t)(rows - 1) * ld + N) * 2 : 0;
                return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base + (int64_t)row0 * ld), 0, (int)(span < 0x7FFFFFFFll ? span : 0x7FFFFFFFll), 0x00020000);
            };
            const auto a_plane = plane(grad.a, N), b_plane = plane(grad.b, N), h_plane = plane(grad.h, N);
            const auto da_plane = plane(grad.da, grad.ld), db_plane = plane(grad.db, grad.ld);
            auto swap_rows = [](u32x4_t& w) {
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const auto swapped = __builtin_amdgcn_permlane16_swap(w[e], w[2 + e], false, false);
                    w[e] = swapped[0];
                    w[2 + e] = swapped[1];
                }
            };
            auto at = [&](int i, int j, int ld) {
                const int col = col0 + j * FR;
                return col < N ? ((i * FR + frow) * ld + col) * 2 : (int)kOutOfRange;
            };
            u32x4_t ra[MF][NF / 2], rb[MF][NF / 2];
            auto load = [&](int i) {
#pragma unroll
                for (int p = 0; p < NF / 2; ++p) {
                    ra[i][p] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(a_plane, at(i, 2 * p, N), 0, 0));
                    rb[i][p] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(b_plane, at(i, 2 * p, N), 0, 0));
                }
            };
#pragma unroll
            for (int i = 0; i < MF; ++i) load(i);            // all of a and b at once: one memory round trip
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MF; ++i) {
#pragma unroll
                for (int p = 0; p < NF / 2; ++p) {
                    float av[8], bv[8], dav[8], dbv[8], hv[8];
                    swap_rows(ra[i][p]);
                    swap_rows(rb[i][p]);
                    unpack16<T>(ra[i][p], av);
                    unpack16<T>(rb[i][p], bv);
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float dc = acc[i][2 * p + e / 4][e % 4];
                        swiglu_gradient(dc, av[e], bv[e], dav[e], dbv[e], hv[e]);
                    }
                    u32x4_t out[3] = {pack16<T>(dav), pack16<T>(dbv), pack16<T>(hv)};
#pragma unroll
                    for (int k = 0; k < 3; ++k) swap_rows(out[k]);
                    __builtin_amdgcn_raw_buffer_store_b128(out[0], da_plane, at(i, 2 * p, grad.ld), 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b128(out[1], db_plane, at(i, 2 * p, grad.ld), 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b128(out[2], h_plane, at(i, 2 * p, N), 0, 0);
                }
            }
            if (next >= num_tiles) break;
            tile = next;
            continue;
        }
        // D fragment layout (both shapes): lane l, register v holds
        //   row = 8*(v/4) + 4*(l/FR) + (v%4)   (A / M index),   col = l%FR   (B / N index)
        // Buffer addressing: a wave-uniform descriptor of the rows from the wave's first one on, a scalar byte offset
        // per (fragment, register) and one 32-bit byte offset per lane - no vector address arithmetic per element.
        const int lane_bytes0 = ((4 * fhalf) * N + frow) * (int)sizeof(T);
        const int64_t wave_off = (int64_t)(out_m0 + wm * WM) * N + out_n0 + wn * ((EPI == kEpiSwiGLU) ? WN / 2 : WN);
        const int64_t span = ((int64_t)M * N - wave_off) * (int64_t)sizeof(T);
        // a wave whose rows all lie beyond M gets an empty descriptor: every access of it is dropped
        const int span32 = (int)(span < 0 ? 0 : (span < 0x7FFFFFFFll ? span : 0x7FFFFFFFll));
        auto c_rsrc = __builtin_amdgcn_make_buffer_rsrc(C + wave_off, 0, span32, 0x00020000);
        // RAGGED: a lane whose column of fragment column j lies beyond N takes an offset no descriptor covers
        auto lane_at = [&](int j, int in_range) {
            if (!RAGGED) return in_range;
            const int col = out_n0 + wn * ((EPI == kEpiSwiGLU) ? WN / 2 : WN) + j * FR + frow;
            return col < N ? in_range : (int)kOutOfRange;
        };
        auto store_to = [&](auto rsrc, int lane_bytes, int uni_bytes, float value) {
            if constexpr (sizeof(T) == 4) {
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, value), rsrc, lane_bytes, uni_bytes, 0);
            } else {
                const T t = Elem<T>::from_f32(value);
                __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(short, t), rsrc, lane_bytes, uni_bytes, 0);
            }
        };
        // 16-bit outputs round once, so the fast reciprocal's last-bit error is invisible; fp32 divides
        auto silu = [](float v) { return sizeof(T) == 4 ? silu_f32(v) : silu_fast_f32(v); };
        // element offset of (fragment i, fragment column j, register v) from the wave's first output element
        auto elem_at = [&](int i, int j, int v) { return (i * FR + 8 * (v / 4) + (v % 4)) * N + j * FR; };
        if (EPI == kEpiSwiGLU) {
            if (R != nullptr) {
                // keep the gate and up products for a backward pass: planes [0] and [1] of a [2, M, N] buffer
                T* planes = const_cast<T*>(R);
                auto g_rsrc = __builtin_amdgcn_make_buffer_rsrc(planes + wave_off, 0, span32, 0x00020000);
                auto u_rsrc = __builtin_amdgcn_make_buffer_rsrc(planes + (int64_t)M * N + wave_off, 0, span32, 0x00020000);
#pragma unroll
                for (int i = 0; i < MF; ++i)
#pragma unroll
                    for (int j = 0; j < NF / 2; ++j)
#pragma unroll
                        for (int v = 0; v < NV; ++v) {
                            const int uni = elem_at(i, j, v) * (int)sizeof(T);
                            store_to(g_rsrc, lane_at(j, lane_bytes0), uni, acc[i][j][v]);
                            store_to(u_rsrc, lane_at(j, lane_bytes0), uni, acc[i][j + NF / 2][v]);
                        }
            }
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int j = 0; j < NF / 2; ++j)
#pragma unroll
                    for (int v = 0; v < NV; ++v)
                        store_to(c_rsrc, lane_at(j, lane_bytes0), elem_at(i, j, v) * (int)sizeof(T), silu(acc[i][j][v]) * acc[i][j + NF / 2][v]);
        } else if (EPI == kEpiPart) {
            // the unrounded sums, C being an fp32 [M, N] buffer
            const int64_t span_f = ((int64_t)M * N - wave_off) * 4;
            const int span32_f = (int)(span_f < 0 ? 0 : (span_f < 0x7FFFFFFFll ? span_f : 0x7FFFFFFFll));
            auto f_rsrc = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<float*>(C) + wave_off, 0, span32_f, 0x00020000);
            const int lane_bytes_f = ((4 * fhalf) * N + frow) * 4;
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int j = 0; j < NF; ++j)
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const float sum = acc[i][j][v];
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, sum), f_rsrc, lane_at(j, lane_bytes_f), elem_at(i, j, v) * 4, 0);
                    }
        } else if (EPI == kEpiDual) {
            // R points at an fp32 [M, N] buffer that receives the unrounded sums next to the rounded ones in C
            float* out32 = reinterpret_cast<float*>(const_cast<T*>(R));
            const int64_t span_f = ((int64_t)M * N - wave_off) * 4;
            const int span32_f = (int)(span_f < 0 ? 0 : (span_f < 0x7FFFFFFFll ? span_f : 0x7FFFFFFFll));
            auto f_rsrc = __builtin_amdgcn_make_buffer_rsrc(out32 + wave_off, 0, span32_f, 0x00020000);
            const int lane_bytes_f = ((4 * fhalf) * N + frow) * 4;
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int j = 0; j < NF; ++j)
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const int at = elem_at(i, j, v);
                        const float sum = acc[i][j][v];      // a scalar copy: the bit cast below must not see a vector element
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(int, sum), f_rsrc, lane_at(j, lane_bytes_f), at * 4, 0);
                        store_to(c_rsrc, lane_at(j, lane_bytes0), at * (int)sizeof(T), sum);
                    }
        } else if (kTurned) {
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int j = 0; j < NF; ++j)
#pragma unroll
                    for (int v = 0; v < NV; ++v) store_to(c_rsrc, lane_at(j, lane_bytes0), elem_at(i, j, v) * (int)sizeof(T), acc[i][j][v]);
        } else {
            auto r_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(R != nullptr ? R + wave_off : C), 0,
                                                            R != nullptr ? span32 : 0, 0x00020000);   // no residual: reads give 0
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int j = 0; j < NF; ++j) {
                    float res[NV];
                    const int lane_bytes = lane_at(j, lane_bytes0);
#pragma unroll
                    for (int v = 0; v < NV; ++v) {
                        const int uni = elem_at(i, j, v) * (int)sizeof(T);
                        if constexpr (sizeof(T) == 4) {
                            res[v] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r_rsrc, lane_bytes, uni, 0));
                        } else {
                            const short raw = __builtin_amdgcn_raw_buffer_load_b16(r_rsrc, lane_bytes, uni, 0);
                            res[v] = Elem<T>::to_f32(__builtin_bit_cast(T, raw));
                        }
                    }
#pragma unroll
                    for (int v = 0; v < NV; ++v) store_to(c_rsrc, lane_bytes, elem_at(i, j, v) * (int)sizeof(T), acc[i][j][v] + res[v]);
                }
        }
        if (next >= num_tiles) break;
        tile = next;
    }
}

// ------------------------------------------------------------------------------------------------------------
// Few output tiles: the waves of a workgroup share one small tile and split k.  Every wave takes its fragments straight from
// global memory (a fragment is 16 rows of 64 bytes: lane l reads 16-byte piece l / 16 of row l % 16), kAhead k-steps ahead and
// without a barrier; the waves' sums meet in LDS, added in wave order.  Rows beyond M or N and the k tail read as zeros (range
// check of the descriptors).  fp32: a 16-byte piece is four k values, one per v_mfma_f32_16x16x4.
// Bound by latency (about 4 us for a launch of one short wave per SIMD) and by what the L2s deliver (about 13 TB/s over the
// chip): the 1024 x 4096 down product takes 7.4 us for one token and 11 us for 64 where 64 x 64 tiles with the whole k loop in
// one chain take 14.3 us; from about 128 tokens on the larger tiles' smaller traffic wins.  Loads of whole lines (8 rows of 128
// bytes, fragments rebuilt with lane rotations) were no faster.
// kEpiPart: slice `slice` of `slices` of k, its sums in fp32 to plane `slice` of C.
// ------------------------------------------------------------------------------------------------------------
template <typename T, int MT, int NT, int EPI>
__device__ __forceinline__ void gemm_splitk_tile(
    const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1, T* __restrict__ C,
    const T* __restrict__ R, int M, int N, int K, int tiles_m, int tiles, int xcds, int block, int blocks, void* lds,
    int slice = 0, int slices = 1) {
    constexpr int BM = 16 * MT, BN = 16 * NT;
    constexpr int NB = EPI == kEpiSwiGLU ? 2 * NT : NT;          // B fragments: gate rows, then the same up rows
    constexpr int F = MT * NB;
    constexpr int kAhead = MT + NB <= 3 ? 8 : 4;
    constexpr int kStep = 64 / (int)sizeof(T);                   // k values of a step
    f32x4_t(*sums)[F][64] = reinterpret_cast<f32x4_t(*)[F][64]>(lds);      // [kSplitWaves]
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // XCD b % xcds takes a contiguous run of the tiles, all rows of a column first: its L2 holds B's part of the run only
    const int tile = (block % xcds) * (blocks / xcds) + block / xcds;
    if (tile >= tiles) return;
    const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
    auto rest_of = [&](const T* base, int64_t rows) {
        const int64_t bytes = rows * K * (int64_t)sizeof(T);
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ar = rest_of(A + (int64_t)m0 * K, M - m0), br = rest_of(B0 + (int64_t)n0 * K, N - n0);
    const __amdgpu_buffer_rsrc_t br1 = EPI == kEpiSwiGLU ? rest_of(B1 + (int64_t)n0 * K, N - n0) : br;
    const int frow = lane & 15, piece = lane >> 4;
    uint32_t row_off[MT > NT ? MT : NT];
#pragma unroll
    for (int i = 0; i < (MT > NT ? MT : NT); ++i) row_off[i] = (uint32_t)((i * 16 + frow) * K) * (uint32_t)sizeof(T) + (uint32_t)piece * 16u;
    const int steps = (K + kStep - 1) / kStep;
    const int parts = kSplitWaves * slices;
    const int share = ((steps + 2 * parts - 1) / (2 * parts)) * 2;                   // two steps are one 128-byte line of a row
    const int first = (slice * kSplitWaves + wave) * share, last = first + share < steps ? first + share : steps;
    const bool in_tail = (steps - 1) * kStep + piece * (16 / (int)sizeof(T)) < K;
    u32x4_t fa[kAhead][MT], fb[kAhead][NB];
    auto load = [&](int step, u32x4_t (&a)[MT], u32x4_t (&b)[NB]) {
        const bool drop = step >= last || (step + 1 == steps && !in_tail);
        const int at = step * 64;
#pragma unroll
        for (int i = 0; i < MT; ++i) a[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ar, (int)(drop ? kOutOfRange : row_off[i]), at, 0));
#pragma unroll
        for (int j = 0; j < NB; ++j)
            b[j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(j < NT ? br : br1, (int)(drop ? kOutOfRange : row_off[j % NT]), at, 0));
    };
    f32x4_t acc[MT][NB];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < kAhead; ++u) load(first + u, fa[u], fb[u]);
    for (int s0 = first; s0 < last; s0 += kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j) acc[i][j] = mfma16_packet<T>(fa[u][i], fb[u][j], acc[i][j]);
            load(s0 + u + kAhead, fa[u], fb[u]);
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) sums[wave][i * NB + j][lane] = acc[i][j];
    __syncthreads();
    // four rows of one column per (fragment, lane)
    for (int q = tid; q < MT * NT * 64; q += kSplitWaves * 64) {
        const int f = q >> 6, l = q & 63, i = f / NT, j = f % NT;
        f32x4_t g = sums[0][i * NB + j][l], u = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int w = 1; w < kSplitWaves; ++w) g += sums[w][i * NB + j][l];
        if (EPI == kEpiSwiGLU) {
            u = sums[0][i * NB + NT + j][l];
            for (int w = 1; w < kSplitWaves; ++w) u += sums[w][i * NB + NT + j][l];
        }
        const int col = n0 + j * 16 + (l & 15);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int row = m0 + i * 16 + 4 * (l >> 4) + v;
            if (row >= M || col >= N) continue;
            const int64_t at = (int64_t)row * N + col;
            if (EPI == kEpiPart) {
                reinterpret_cast<float*>(C)[(int64_t)slice * M * N + at] = g[v];
            } else if (EPI == kEpiSwiGLU) {
                const float act = sizeof(T) == 4 ? silu_f32(g[v]) : silu_fast_f32(g[v]);
                C[at] = Elem<T>::from_f32(act * u[v]);
                if (R != nullptr) {      // planes [0] and [1] of a [2, M, N] buffer keep the two products
                    const_cast<T*>(R)[at] = Elem<T>::from_f32(g[v]);
                    const_cast<T*>(R)[(int64_t)M * N + at] = Elem<T>::from_f32(u[v]);
                }
            } else {
                C[at] = Elem<T>::from_f32(R != nullptr ? g[v] + Elem<T>::to_f32(R[at]) : g[v]);
            }
        }
    }
}

// k extent of one LDS stage of the DMA kernel: 128 bytes of a row for every element type
template <typename T> constexpr int kStageK = 128 / (int)sizeof(T);
// 16-bit products run on v_mfma_f32_16x16x32 (more multiply-adds per joule than 32x32x16, which is what bounds these
// kernels); a k-step is then half a stage, so the read-ahead is one step.  Their 256 x 256 tiles are in fmoe_gemm256.h.  fp32 keeps
// 32x32x2.
template <typename T> constexpr int kFragRows = sizeof(T) == 2 ? 16 : 32;
template <typename T> constexpr int kSmallAhead = sizeof(T) == 2 ? 1 : 3;
// Gate/up tiles of 64 x 64 hold 32 columns of either, a wave 16 of them: fragments of 16 rows in fp32 too.
template <typename T, int BN, int EPI> constexpr bool kNarrowPair = sizeof(T) == 4 && BN == 64 && EPI == kEpiSwiGLU;
template <typename T, int BN, int EPI> constexpr int kTileFrag = kNarrowPair<T, BN, EPI> ? 16 : kFragRows<T>;
template <typename T, int BN, int EPI> constexpr int kTileAhead = kNarrowPair<T, BN, EPI> ? 1 : kSmallAhead<T>;

// Tile choice.  A workgroup's time per k-tile is the larger of what its CU receives from the L2 ((BM + BN) rows of 128 bytes, at 40
// to 70 GB/s per CU) and what its matrix pipes take (BM * BN), in units of one received row BM * BN / 95: with every CU busy a
// k-tile of 256 x 256 takes 1.65 us where 128 x 128 takes 0.6, 64 x 128 0.45 and 64 x 64 0.25.  The launch lasts as many rounds as
// the busiest CU has tiles.  The rule picks the shape with the smallest rounds * time: 256 x 256 (8 waves, two per SIMD) once that
// means fewer rounds, smaller ones so that every CU has a tile, whatever the extents.  (Pricing 256 x 256 at / 66 gave 1675 tokens
// of 2904 -> 7744 seven rounds of 128 x 128, 227 us; two of 256 x 256 take 157.)
// Its two groups of waves keep the pipes busier: BM * BN / 108 for the plain products (us: 22464 tokens, 3232 -> 808 147 -> 128; 15029
// tokens, 3408 -> 1280 166 -> 147); gate/up products, of which half are short in k, gain and lose about alike and stay at / 95.
// fp32 rows of 128 bytes hold half as many values for matrix pipes an eighth as fast: BM * BN / 15, gate/up pairs of 32 columns / 13 (the
// block, us, on the best of the other tiles and on these: 400 tokens, 512 -> 1024 43.1 -> 35.9; 300, 256 -> 1024 28.1 -> 24.5; 512, 256 -> 1024
// 33.1 -> 31.6; at / 15 1900 tokens, 640 -> 1704 would take them too, 159 -> 163).  The k-splitting kernel
// costs more per received row, and more so the more CUs receive at once (measured from 64 to 224 workgroups), but its tiles are
// small enough for a few rows of A.
enum TileShape { kTile256, kTile128, kTile64x128, kTile64, kSplit32, kSplit16x32, kSplit16 };
constexpr int kTileRows[7] = {256, 128, 64, 64, 32, 16, 16}, kTileCols[7] = {256, 128, 128, 64, 32, 32, 16};

// Workgroups of tile i, and the time of a round of them per k-tile.
template <typename T, int EPI> double tile_cost(int i, int M, int N, int cus, int64_t& n) {
    const bool split_k = i >= kSplit32;
    const int out_cols = EPI == kEpiSwiGLU && !split_k ? kTileCols[i] / 2 : kTileCols[i];
    const int cols = EPI == kEpiSwiGLU ? 2 * out_cols : out_cols;
    n = (int64_t)((M + kTileRows[i] - 1) / kTileRows[i]) * ((N + out_cols - 1) / out_cols);
    const double occupied = n < cus ? (double)n / cus : 1.0;
    const double received = (kTileRows[i] + cols) * (split_k ? 1.45 * (1.0 + occupied) : 1.0);
    const double rate = sizeof(T) == 4 ? (i == kTile64 && EPI == kEpiSwiGLU ? 13.0 : 15.0) : (i == kTile256 && EPI == kEpiPlain ? 108.0 : 95.0);
    const double multiplied = kTileRows[i] * (double)cols / rate;
    return received > multiplied ? received : multiplied;
}
template <typename T, int EPI> TileShape choose_tile(int M, int N, int& tiles, double* cost_out = nullptr) {
    const int cus = chip_info().cus;
    TileShape best = kTile128;
    double best_cost = 0.0;
    for (int i = 0; i < 7; ++i) {
        int64_t n = 0;
        const double round = tile_cost<T, EPI>(i, M, N, cus, n), cost = (double)((n + cus - 1) / cus) * round;
        if (i == 0 || cost < best_cost) {
            best = (TileShape)i;
            best_cost = cost;
            tiles = (int)(n < (1 << 30) ? n : (1 << 30));
        }
    }
    if (cost_out != nullptr) *cost_out = best_cost;
    return best;
}

// A long k loop on few tiles: slices of k to workgroups of their own, which leave fp32 sums in planes [slices][M][N] that one more
// launch adds.  The rule prices both ways, a received row and k-tile at 2.3 ns, that launch at 4 us and the planes written and read
// at 6 TB/s, and wants the slices to gain a tenth; against the k-splitting tiles, which this price makes too dear when they are
// short, 8.5 us and a fifth.  Down products, us: 47 tokens, 15360 -> 3840 49.6 -> 25.4; 128 tokens, 8192 -> 2048 29 -> 15.6; 300
// tokens, 10920 -> 4096 69 -> 51; 479 tokens, 13216 -> 3304 77 -> 61; fp32, 803 tokens, 5632 -> 1408 195 -> 130.
struct SlicePlan { int shape, slices; };
constexpr int kMaxSlices = 16;
template <typename T> SlicePlan plan_slices_of_k(int M, int N, int K) {
    SlicePlan best = {-1, 1};
    int tiles = 0;
    double whole = 0.0;
    const TileShape shape = choose_tile<T, kEpiPlain>(M, N, tiles, &whole);
    const bool split_k = shape >= kSplit32;
    const int cus = chip_info().cus, k_tiles = (K + kStageK<T> - 1) / kStageK<T>;
    const double kRow = 2.3e-3, launch = split_k ? 8.5 : 4.0;
    double best_time = (split_k ? 0.8 : 0.9) * whole * k_tiles * kRow;
    // Two 128 x 128 tiles to a compute unit hide each other's latency, by how much depends on the extents in ways the price does not
    // see.  Of 90 down products in bf16 that the price alone would cut, 0.85 cuts 46, of which 37 gain (0.91 of the time on average, at best
    // 2510 tokens, 5416 -> 2032: 102 us whole, 71 in slices) and 9 lose (at most 2685 tokens, 4160 -> 1560: 47 whole, 54); of the 44 it keeps
    // whole 27 would gain (2708 tokens, 4968 -> 1864: 90 whole, 70) and 17 lose, up to a fifth.  No fp32 product comes near.
    if (shape == kTile128 && tiles > cus) best_time *= 0.85;
    if (sizeof(T) == 4 && K % 4 != 0) return best;
    for (int i = sizeof(T) == 2 ? kTile256 : kTile128; i <= kTile64; ++i) {
        int64_t n = 0;
        const double round = tile_cost<T, kEpiPlain>(i, M, N, cus, n);
        for (int s = 2; s <= kMaxSlices && n * s <= cus && s * 4 <= k_tiles; ++s) {
            const int share = (k_tiles + s - 1) / s;
            if ((s - 1) * share >= k_tiles) continue;           // a slice would have no k-tile
            const double time = round * share * kRow + launch + (i == kTile256 ? 5.0 : 0.0) + 8.0e-6 * s * (double)M * N / 6.0;
            if (time < best_time) {
                best = {i, s};
                best_time = time;
            }
        }
    }
    return best;
}

}  // namespace
}  // namespace fmoe
