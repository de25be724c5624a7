// 128 x 128 tiles of C[M,N] = A[M,K] * B[N,K]^T (+ R) in the 16-bit types for products of at most one such tile per compute unit
// (gfx950): every wave has the whole tile and a quarter of the k-tiles.
//
// With one workgroup to a CU, four waves of 64 x 64 that share every k-tile meet at a barrier per k-tile with nothing else to run: 0.48 to
// 0.6 us per k-tile of 64, where the fetch of its 32 KB takes 0.31 (256 CUs fetching alone, in pieces of 128 or 256 bytes of a row
// alike) and its matrix instructions 0.22.  Here wave w takes k-tiles w, w + 4, ... into a stage of its own and waits for nobody: once
// its stage has landed it reads all of it into registers (128 of them, beside 256 sums) and requests its next k-tile into the same
// stage between the matrix instructions of this one, one load of 1 KB every second instruction, so that neither waits for the other: 0.41 us
// per k-tile.  The waves' sums meet in LDS at the end.  Two halves of the waves with half the tile's columns each would read the stages
// half as often, but share them.  Requests in one go before the matrix instructions cost 1 % on average, one every fourth instruction
// 4 %; requesting A's rows while B's are still read gained nothing, nor did this way for slices of k, or for more tiles than CUs (two
// workgroups of shared tiles to a CU hide each other's waits: 8192 tokens, 4096 -> 1024 65 us, 74 this way).
// us, down products in bf16, repeated alone, before | now (in the README block, behind the gate/up product, 48.8 | 43): 4096 tokens, 4096 -> 1024 37.1 | 34.7; 2048 tokens, 8192 -> 2048 67.1 | 62.2; 3000 tokens,
// 2664 -> 1000 34.7 | 31.3; 2500 tokens, 3736 -> 1400 45.3 | 40.9; error against float64 as before.
#pragma once

#include "fmoe_gemm.h"

namespace fmoe {
namespace {

constexpr int kSoloStage = 256 * 64;                 // elements of a wave's stage: 128 rows of A and 128 of B, a k-tile of 64
// The first requests and the meeting of the sums take about 8 us, half a microsecond more than in the shared tiles: us, 4096 x 1024 tiles,
// before | here: K = 1024 14.8 | 15.2, 1536 19.9 | 19.7, 2048 23.5 | 23.1, 3072 31.3 | 29.6.
constexpr int kSoloTiles = 24;

// C and R: 8-byte pieces of rows.  lds: four stages.
template <typename T>
__device__ __forceinline__ void gemm_solo_tile(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, const T* __restrict__ R, int M, int N,
                                               int K, int tiles_m, int tiles_n, int xcds, int block, T* lds) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    const int lane = (int)threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int t = xcd_run(block, tiles_m * tiles_n, xcds);
    constexpr int GM = 8;
    const int width = GM * tiles_n, first_m = t / width * GM, gsz = tiles_m - first_m < GM ? tiles_m - first_m : GM;
    const int m0 = (first_m + (t % width) % gsz) * 128, n0 = ((t % width) / gsz) * 128;
    auto rest_of = [&](const T* base, int64_t elements) {                          // rows beyond the ends read zeros, stores there are dropped
        const int64_t bytes = elements * 2;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ar = rest_of(A + (int64_t)m0 * K, (int64_t)(M - m0) * K), br = rest_of(B + (int64_t)n0 * K, (int64_t)(N - n0) * K);
    const int k_tiles = (K + 63) / 64;
    // A load covers 8 rows of 128 bytes; 16-byte chunk c of a row lies at c ^ (row / 2 % 8), so that fragment reads meet no bank twice.
    const int lrow = lane >> 3, chunk = (lane & 7) ^ (lrow >> 1);
    const uint32_t row_bytes = (uint32_t)K * 2u;
    T* stage = lds + wave * kSoloStage;
    auto issue = [&](int kt, int r) {                                             // load r of 32 of k-tile kt
        const int c = r & 1 ? chunk ^ 4 : chunk;
        const uint32_t at = (uint32_t)((r & 15) * 8 + lrow) * row_bytes + (uint32_t)c * 16u;
        // past the last k-tile the scalar offset is 0: with one row of A left it would pass the descriptor's end by itself
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r < 16 ? ar : br, (__attribute__((address_space(3))) void*)(stage + r * 512), 16,
                                                 (int)(kt * 64 + c * 8 < K ? at : kOutOfRange), kt < k_tiles ? kt * 128 : 0, 0, 0);
    };
    const int frow = lane & 15, fhalf = lane >> 4;
    const char* from = reinterpret_cast<const char*>(stage) + frow * 128;
    const int piece[2] = {(fhalf ^ (frow >> 1)) * 16, ((4 + fhalf) ^ (frow >> 1)) * 16};
    f32x4_t acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int r = 0; r < 32; ++r) issue(wave, r);                                  // beyond the last k-tile: zeros
    for (int kt = wave; kt < k_tiles; kt += 4) {
        __builtin_amdgcn_s_waitcnt(0x0F70);                                       // vmcnt(0): the stage has landed
        __builtin_amdgcn_sched_barrier(0);
        u32x4_t fa[2][8], fb[2][8];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                fa[s][i] = *reinterpret_cast<const u32x4_t*>(from + i * 2048 + piece[s]);
                fb[s][i] = *reinterpret_cast<const u32x4_t*>(from + 16384 + i * 2048 + piece[s]);
            }
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xC07F);                                       // lgkmcnt(0): and is in registers, it may be overwritten
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int q = s * 64 + i * 8 + j;
                    if (q % 2 == 0 && q < 64) {
                        __builtin_amdgcn_sched_barrier(0);
                        issue(kt + 4, q / 2);
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    acc[i][j] = mfma16_packet<T>(fb[s][j], fa[s][i], acc[i][j]);  // register v of a lane: row lane % 16, column 4 (lane / 16) + v
                }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);                                           // nothing lands in the stage any more
    // The four waves' sums meet in the stages, (0 + 2) + (1 + 3), half of the rows at a time; of each half wave w adds up and stores
    // fragment row w.
    const __amdgpu_buffer_rsrc_t cr = rest_of(C + (int64_t)m0 * N, (int64_t)(M - m0) * N);
    const __amdgpu_buffer_rsrc_t rr = rest_of(R != nullptr ? R + (int64_t)m0 * N : C, R != nullptr ? (int64_t)(M - m0) * N : 0);      // none: zeros
    uint32_t at[8];
    u32x2_t raw[2][8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const int col = n0 + j * 16 + fhalf * 4;                                  // N is a multiple of 8
        at[j] = col < N ? (uint32_t)((wave * 16 + frow) * N + col) * 2u : kOutOfRange;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            raw[h][j] = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(rr, (int)(at[j] + (uint32_t)(h * 128 * N)), 0, 0));
    }
    f32x4_t* mine = reinterpret_cast<f32x4_t*>(stage) + lane;
    const f32x4_t* sums = reinterpret_cast<const f32x4_t*>(lds) + wave * 512 + lane;
    constexpr int kNext = kSoloStage * 2 / 16;                                    // from a wave's sums to the next wave's
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if (h == 1) __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 8; ++j) mine[(i * 8 + j) * 64] = acc[h * 4 + i][j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const f32x4_t sum = (sums[j * 64] + sums[2 * kNext + j * 64]) + (sums[kNext + j * 64] + sums[3 * kNext + j * 64]);
            u32x2_t both;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const T lo = Elem<T>::from_f32(sum[2 * p] + Elem<T>::to_f32(__builtin_bit_cast(T, (uint16_t)(raw[h][j][p] & 0xffffu))));
                const T hi = Elem<T>::from_f32(sum[2 * p + 1] + Elem<T>::to_f32(__builtin_bit_cast(T, (uint16_t)(raw[h][j][p] >> 16))));
                both[p] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | (uint32_t)__builtin_bit_cast(uint16_t, hi) << 16;
            }
            __builtin_amdgcn_raw_buffer_store_b64(both, cr, (int)(at[j] + (uint32_t)(h * 128 * N)), 0, 0);
        }
    }
}

}  // namespace
}  // namespace fmoe
