// The router's gate product with its batch-norm prologue on small tiles, k split over the waves of a workgroup (gfx950): parts of the
// kernels in fmoe_router_prologue.hip and fmoe_small.hip.
#pragma once

#include "fmoe_common.h"
#include "fmoe_mfma.h"
#include "fmoe_vec.h"

namespace fmoe {
namespace {

constexpr int kFoldMaxRowBlocks = 16;     // row blocks of the statistics that a gate workgroup combines itself

// Running statistics live in any of the three dtypes; the gate kernel is not instantiated per statistics dtype.
__device__ inline float load_stat_rt(const void* p, int i, int dtype) {
    switch (dtype) {
        case FMOE_F32: return ((const float*)p)[i];
        case FMOE_BF16: return Elem<bf16_t>::to_f32(((const bf16_t*)p)[i]);
        default: return Elem<f16_t>::to_f32(((const f16_t*)p)[i]);
    }
}
__device__ inline void store_stat_rt(void* p, int i, float v, int dtype) {
    switch (dtype) {
        case FMOE_F32: ((float*)p)[i] = v; break;
        case FMOE_BF16: ((bf16_t*)p)[i] = Elem<bf16_t>::from_f32(v); break;
        default: ((f16_t*)p)[i] = Elem<f16_t>::from_f32(v); break;
    }
}

// What the gate kernel's prologue needs to turn block statistics (or running statistics) into mean and 1/std.
struct GateStats {
    const float* partial;          // [row_blocks][2][H] from bn_block_stats_kernel (training)
    int row_blocks, rows_per_block;
    int64_t num_tokens;
    int training, stats_dtype;
    int ready;                     // mean_rstd already holds the statistics (a finalize launch ran): just stage them
    float momentum, eps;
    void* running_mean;
    void* running_var;
    int64_t* num_batches_tracked;
    float* mean_rstd;              // [2][H]: kept for a backward pass
};

// q = round_T((x - mean) * rstd) for one 16-byte packet
template <typename T> __device__ inline u32x4_t normalise16(u32x4_t raw, const float* mean, const float* rstd);
template <> __device__ inline u32x4_t normalise16<bf16_t>(u32x4_t raw, const float* mean, const float* rstd) {
    float v[8];
    unpack16<bf16_t>(raw, v);
    u32x4_t out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bf16x2_t p = {(bf16_t)((v[2 * i] - mean[2 * i]) * rstd[2 * i]), (bf16_t)((v[2 * i + 1] - mean[2 * i + 1]) * rstd[2 * i + 1])};
        out[i] = __builtin_bit_cast(uint32_t, p);
    }
    return out;
}
template <> __device__ inline u32x4_t normalise16<f16_t>(u32x4_t raw, const float* mean, const float* rstd) {
    float v[8];
    unpack16<f16_t>(raw, v);
    u32x4_t out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const f16x2_t p = {(f16_t)((v[2 * i] - mean[2 * i]) * rstd[2 * i]), (f16_t)((v[2 * i + 1] - mean[2 * i + 1]) * rstd[2 * i + 1])};
        out[i] = __builtin_bit_cast(uint32_t, p);
    }
    return out;
}

template <> __device__ inline u32x4_t normalise16<float>(u32x4_t raw, const float* mean, const float* rstd) {
    u32x4_t out;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t r = raw[i];
        out[i] = __float_as_uint((__uint_as_float(r) - mean[i]) * rstd[i]);
    }
    return out;
}

// mean and 1/std of columns [k_off, k_off + K) into LDS (zeros up to kpad), by all threads of a workgroup.  keeper: the one column of
// tiles per k range that also stores them (for a backward pass) and updates the running statistics: its tile row (i / 64) mod
// tiles_m takes column i, so every column is written by exactly one workgroup.  CPT columns per thread and round: all their
// block statistics are loaded together, one memory round trip per round.
template <int CPT>
__device__ inline void stage_stats(const GateStats& st, float* stats, int kpad, int K, int K_full, int k_off, bool keeper, int tm, int tiles_m, bool first) {
    const int threads = (int)blockDim.x, tid = (int)threadIdx.x;
    if (first && tid == 0 && st.training && !st.ready && st.num_batches_tracked != nullptr) *st.num_batches_tracked += 1;
    const float n = (float)st.num_tokens;
    const float full = (float)st.rows_per_block;
    const float last = (float)(st.num_tokens - (int64_t)(st.row_blocks - 1) * st.rows_per_block);
    for (int i0 = tid; st.ready && i0 < kpad; i0 += threads) {
        stats[i0] = i0 < K ? st.mean_rstd[k_off + i0] : 0.0f;
        stats[kpad + i0] = i0 < K ? st.mean_rstd[K_full + k_off + i0] : 0.0f;
    }
    for (int i0 = tid; !st.ready && i0 < kpad; i0 += threads * CPT) {
        float mean[CPT], var[CPT], m2[CPT];
        if (st.training) {
            float mb[CPT][kFoldMaxRowBlocks], m2b[CPT][kFoldMaxRowBlocks];
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                const int i = i0 + u * threads;
                const float* pc = st.partial + k_off + (i < K ? i : 0);
#pragma unroll
                for (int b = 0; b < kFoldMaxRowBlocks; ++b) {
                    const bool ok = b < st.row_blocks;
                    mb[u][b] = ok ? pc[(int64_t)b * 2 * K_full] : 0.0f;
                    m2b[u][b] = ok ? pc[(int64_t)b * 2 * K_full + K_full] : 0.0f;
                }
            }
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                float snm = 0.0f;
#pragma unroll
                for (int b = 0; b < kFoldMaxRowBlocks; ++b) {
                    const float nb = b + 1 < st.row_blocks ? full : (b + 1 == st.row_blocks ? last : 0.0f);
                    snm = __builtin_fmaf(nb, mb[u][b], snm);
                }
                mean[u] = snm / n;
                float acc2 = 0.0f;
#pragma unroll
                for (int b = 0; b < kFoldMaxRowBlocks; ++b) {
                    const float nb = b + 1 < st.row_blocks ? full : (b + 1 == st.row_blocks ? last : 0.0f);
                    const float d = mb[u][b] - mean[u];
                    acc2 += __builtin_fmaf(nb * d, d, m2b[u][b]);
                }
                m2[u] = acc2;
                var[u] = acc2 / n;                              // biased: what normalises the batch
            }
        } else {
#pragma unroll
            for (int u = 0; u < CPT; ++u) {
                const int i = i0 + u * threads;
                const int c = k_off + (i < K ? i : 0);
                mean[u] = load_stat_rt(st.running_mean, c, st.stats_dtype);
                var[u] = load_stat_rt(st.running_var, c, st.stats_dtype);
                m2[u] = 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < CPT; ++u) {
            const int i = i0 + u * threads;
            if (i >= kpad) continue;
            const int c = k_off + i;
            const float rstd = 1.0f / sqrtf(var[u] + st.eps);
            if (i < K && keeper && tm == (i / 64) % tiles_m) {
                if (st.training && st.running_mean != nullptr && st.running_var != nullptr) {
                    const float unbiased = n > 1.0f ? m2[u] / (n - 1.0f) : var[u];
                    store_stat_rt(st.running_mean, c, (1.0f - st.momentum) * load_stat_rt(st.running_mean, c, st.stats_dtype) + st.momentum * mean[u], st.stats_dtype);
                    store_stat_rt(st.running_var, c, (1.0f - st.momentum) * load_stat_rt(st.running_var, c, st.stats_dtype) + st.momentum * unbiased, st.stats_dtype);
                }
                st.mean_rstd[c] = mean[u];
                st.mean_rstd[K_full + c] = rstd;
            }
            stats[i] = i < K ? mean[u] : 0.0f;
            stats[kpad + i] = i < K ? rstd : 0.0f;
        }
    }
}

// logits[M, N] = normalise(x)[M, K] * W[N, K]^T while there are few tiles: the waves of a workgroup share one tile of 16 MT rows and 16
// NT columns and split k, line l (128 bytes of k) to wave l mod kGateWaves.  Every wave takes its fragments straight from global
// memory (lane l reads 16-byte piece l / 16 of row l % 16), kAhead steps of 64 bytes ahead and without a barrier, and normalises
// the activations in registers; the waves' sums meet in LDS and are added in wave order, so the result depends neither on the
// tile shape nor, the zero blocks of a block-diagonal gate adding nothing, on split.
// STAGED: mean and 1/std of the tile's k range are made (or copied) in LDS first, overlapping the first loads; otherwise
// st.ready, and they are read from mean_rstd as the operands are.  stats: 8 bytes of LDS per column (STAGED).
constexpr int kGateWaves = 8;
constexpr int kGateStagedK = 4096;       // 8 bytes of LDS per column
constexpr uint32_t kGateOutOfRange = 0x80000000u;

// lds: kGateLds bytes.
template <int MT, int NT> constexpr int kGateLds = kGateWaves * (MT * NT < 8 ? MT * NT : 8) * kWave * 16;
// WAVES of the kernel: with half of kGateWaves each takes the lines of two, one after the other - the same sums.
template <typename T, int MT, int NT, bool STAGED, int WAVES = kGateWaves>
__device__ __forceinline__ void router_gate_splitk_tile(
    const T* __restrict__ x, const T* __restrict__ w, const GateStats& st, float* __restrict__ logits32, T* __restrict__ logits, int M, int N,
    int K_full, int tiles_m, int tiles_n, int split, int xcds, void* lds, float* stats, int block, int blocks) {
    constexpr int BM = 16 * MT, BN = 16 * NT, F = MT * NT, V = Elem<T>::kVec;
    constexpr int kStep = 64 / (int)sizeof(T);                   // k values of a step; two steps are a line
    constexpr int kAhead = MT + NT <= 3 ? 8 : 4;
    constexpr int kRound = F < 8 ? F : 8;                        // fragments exchanged at a time
    f32x4_t(*sums)[kRound][kWave] = reinterpret_cast<f32x4_t(*)[kRound][kWave]>(lds);      // [kGateWaves]
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // XCD b % xcds takes a contiguous run of the tiles, all columns of a row first: its L2 holds the run's part of x only
    const int tile = (block % xcds) * (blocks / xcds) + block / xcds;
    if (tile >= tiles_m * tiles_n) return;
    const int tm = tile / tiles_n, tn = tile % tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    // the k range of this tile: all of it, or the half of the activations its columns score (tiles do not straddle halves)
    const int K = split ? K_full / 2 : K_full;
    const int k_off = (split && n0 >= N / 2) ? K : 0;
    auto rsrc = [&](const void* base, int64_t bytes) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t ar = rsrc(x + (int64_t)m0 * K_full + k_off, ((int64_t)(M - m0) * K_full - k_off) * (int64_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t br = rsrc(w + (int64_t)n0 * K, (int64_t)(N - n0) * K * (int64_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t sr = rsrc(st.mean_rstd + k_off, ((int64_t)2 * K_full - k_off) * 4);
    const int frow = lane & 15, piece = lane >> 4;
    uint32_t a_off[MT], b_off[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i) a_off[i] = (uint32_t)((i * 16 + frow) * K_full) * (uint32_t)sizeof(T) + (uint32_t)piece * 16u;
#pragma unroll
    for (int j = 0; j < NT; ++j) b_off[j] = (uint32_t)((j * 16 + frow) * K) * (uint32_t)sizeof(T) + (uint32_t)piece * 16u;
    const int lines = (K + 2 * kStep - 1) / (2 * kStep);
    // step u of part `part` of k: half u % 2 of its line u / 2; lines are numbered over all of k, whichever half the tile scores
    int first_line = 0, steps = 0;
    auto set_part = [&](int part) {
        first_line = (part + kGateWaves - (k_off / (2 * kStep)) % kGateWaves) % kGateWaves;
        steps = first_line < lines ? 2 * ((lines - first_line + kGateWaves - 1) / kGateWaves) : 0;
    };
    set_part(wave);
    u32x4_t fa[kAhead][MT], fb[kAhead][NT];
    auto k_of = [&](int u) { return ((first_line + (u >> 1) * kGateWaves) * 2 + (u & 1)) * kStep; };
    auto load = [&](int u, u32x4_t (&a)[MT], u32x4_t (&b)[NT]) {
        const int k0 = k_of(u);
        const bool drop = u >= steps || k0 + piece * V >= K;
#pragma unroll
        for (int i = 0; i < MT; ++i)
            a[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(ar, (int)(drop ? kGateOutOfRange : a_off[i]), k0 * (int)sizeof(T), 0));
#pragma unroll
        for (int j = 0; j < NT; ++j)
            b[j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(br, (int)(drop ? kGateOutOfRange : b_off[j]), k0 * (int)sizeof(T), 0));
    };
#pragma unroll
    for (int u = 0; u < kAhead; ++u) load(u, fa[u], fb[u]);
    const int kpad = (K + 2 * kStep - 1) / (2 * kStep) * (2 * kStep);
    if constexpr (STAGED) {
        stage_stats<1>(st, stats, kpad, K, K_full, k_off, tn == (k_off ? tiles_n / 2 : 0), tm, tiles_m, tile == 0);
        __syncthreads();
    }
    f32x4_t acc[MT][NT];
    auto multiply = [&]() {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        for (int u0 = 0; u0 < steps; u0 += kAhead) {
#pragma unroll
            for (int d = 0; d < kAhead; ++d) {
                const int u = u0 + d;
                // Steps and pieces past the end multiply zeros.  Their q has to be zero as well as their weights: their statistics are
                // other columns' (staged ones are zero beyond K), whose (0 - mean) * rstd may be infinite in T.
                const int k0 = u < steps ? k_of(u) : 0;
                const uint32_t keep = u < steps && (STAGED || k0 + piece * V < K) ? ~0u : 0u;
                float mean[V], rstd[V];
#pragma unroll
                for (int c = 0; c < V / 4; ++c) {
                    u32x4_t mv, rv;
                    if constexpr (STAGED) {
                        mv = *reinterpret_cast<const u32x4_t*>(stats + k0 + piece * V + c * 4);
                        rv = *reinterpret_cast<const u32x4_t*>(stats + kpad + k0 + piece * V + c * 4);
                    } else {
                        const int at = (piece * V + c * 4) * 4;
                        mv = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(sr, at, k0 * 4, 0));
                        rv = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(sr, at, (K_full + k0) * 4, 0));
                    }
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const uint32_t mw = mv[v], rw = rv[v];
                        mean[c * 4 + v] = __uint_as_float(mw);
                        rstd[c * 4 + v] = __uint_as_float(rw);
                    }
                }
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const u32x4_t q = normalise16<T>(fa[d][i], mean, rstd) & keep;
#pragma unroll
                    for (int j = 0; j < NT; ++j) acc[i][j] = mfma16_packet<T>(q, fb[d][j], acc[i][j]);
                }
                load(u + kAhead, fa[d], fb[d]);
            }
        }
    };
    multiply();
    static_assert(WAVES == kGateWaves || F <= kRound, "one exchange");
#pragma unroll
    for (int part = WAVES; part < kGateWaves; part += WAVES) {
#pragma unroll
        for (int f = 0; f < F; ++f) sums[part - WAVES + wave][f][lane] = acc[f / NT][f % NT];
        set_part(part + wave);
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load(u, fa[u], fb[u]);
        multiply();
    }
#pragma unroll
    for (int f0 = 0; f0 < F; f0 += kRound) {
        if (f0 > 0) __syncthreads();
#pragma unroll
        for (int f = f0; f < f0 + kRound; ++f) sums[kGateWaves - WAVES + wave][f - f0][lane] = acc[f / NT][f % NT];
        __syncthreads();
        // four rows of one column per (fragment, lane)
        for (int q = tid; q < kRound * kWave; q += WAVES * kWave) {
            const int f = f0 + (q >> 6), l = q & 63;
            f32x4_t g = sums[0][q >> 6][l];
#pragma unroll
            for (int v = 1; v < kGateWaves; ++v) g += sums[v][q >> 6][l];
            const int col = n0 + (f % NT) * 16 + (l & 15);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = m0 + (f / NT) * 16 + 4 * (l >> 4) + v;
                if (row >= M || col >= N) continue;
                const float sum = g[v];
                logits32[(int64_t)row * N + col] = sum;
                logits[(int64_t)row * N + col] = Elem<T>::from_f32(sum);
            }
        }
    }
}

// Tiles of a launch with 16 mt x 16 nt outputs each.
inline int64_t gate_tiles(int M, int N, int mt, int nt) { return (int64_t)((M + 16 * mt - 1) / (16 * mt)) * ((N + 16 * nt - 1) / (16 * nt)); }

// Whether the gate product of these extents is the k-splitting kernel's, for the router alone and inside the block: the two have to
// agree to the last bit, so one rule decides for both.  16-bit products beyond a round of 32 x 64 tiles are left to router_gate_kernel,
// whose waves share the operands through LDS (4096 tokens, 1024 columns, 256 outputs: 20.6 us against 22.4 on 64 x 64 tiles here; 1024
// tokens 18.2 there against 14.7 here); fp32 is bound by its matrix rate (2048 tokens: 25 us where a kernel of plain FMAs took 196;
// 207 tokens, 1232 columns, 436 outputs: 13 for 194).
inline bool gate_splitk_pays(int M, int N, int dtype) { return dtype == FMOE_F32 || gate_tiles(M, N, 2, 4) <= chip_info().cus; }

}  // namespace
}  // namespace fmoe
