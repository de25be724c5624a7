// Router prologue of the FlashMoE block for gfx950, fused with the product-key top-k:
//   q = BatchNorm1d(x)  (affine=False; batch statistics in training mode, running statistics otherwise)
//   logits = q Wr^T     [T, 2*nk]
//   log-softmax per half, top-k over the pair sums, exp / renormalise   (router_topk_kernel, logits-input mode)
//
// Launches (three in training mode, two in evaluation mode):
//   bn_block_stats_kernel  per (row block, 128-byte column strip): shifted sums -> (mean, M2) of the block   [training]
//   router_gate_splitk_kernel   few tiles and fp32: MFMA product, the waves of a workgroup split k; or
//   router_gate_kernel     MFMA product on 64 x 64 tiles, operands shared through LDS.  With at most one tile per compute unit (4096
//                          tokens) a workgroup is 16 waves: four groups that each take every fourth k-tile and add their
//                          accumulators at the end.
//                          Either combines the (at most 16) row blocks per column (Chan's parallel formula) into mean and
//                          1/sqrt(var+eps) - or takes the running statistics - for the columns it multiplies, and a few workgroups
//                          also store them and update the running statistics (momentum, unbiased variance) and the batch counter.
//                          (x - mean) * rstd is rounded to the activation dtype exactly as a stand-alone batch-norm would emit
//                          it, then multiplied with the gate weights with fp32 accumulation; writes the logits in fp32 (for the
//                          routing) and in the activation dtype (the tensor the module returns).
//   router_select_kernel   (fmoe_router.hip)
// With many tiles the statistics are combined once instead: bn_partial_kernel per (row block, column strip), bn_finalize_kernel per
// column.
#include <math.h>

#include <mutex>

#include "fmoe_common.h"
#include "fmoe_gate.h"
#include "fmoe_mfma.h"
#include "fmoe_vec.h"

// Scratch of fmoe_router_forward_noalloc: the batch-norm partials and the mean / 1/std vectors of one call, for hidden sizes
// up to kNoAllocMaxHidden.  Every GPU the library runs on holds its own copy at its own address for the life of the
// process; host code reaches it only through the address hipGetSymbolAddress returns for the current device.
#define FMOE_NOALLOC_MAX_HIDDEN 2048
#define FMOE_NOALLOC_SCRATCH_BYTES (256 * 3 * FMOE_NOALLOC_MAX_HIDDEN * 4 + 2 * FMOE_NOALLOC_MAX_HIDDEN * 4)
static __device__ __align__(256) unsigned char scratch[FMOE_NOALLOC_SCRATCH_BYTES];

namespace fmoe {
namespace {

constexpr int kStatsThreads = 256;
constexpr int kMaxRowBlocks = 256;
static_assert(kMaxRowBlocks * 3 * FMOE_NOALLOC_MAX_HIDDEN * 4 % 256 == 0, "the static scratch holds the largest plan exactly");

// Device address of `scratch` on the current device, looked up once per device.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxDevices] = {};

int static_scratch(void** out) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
        set_error("fmoe_router_forward_noalloc: no usable current device (%s)", hipGetErrorString(e));
        return e != hipSuccess ? (int)e : FMOE_ERR_UNSUPPORTED;
    }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (g_scratch_ptr[dev] == nullptr) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) {
            set_error("fmoe_router_forward_noalloc: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
            return e != hipSuccess ? (int)e : FMOE_ERR_UNSUPPORTED;
        }
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return FMOE_OK;
}

// Block (rb, strip): rows [rb*rows_per_block, ...), columns strip*64*V + lane*V .. +V; the 4 waves take rows 4 apart.
// Sums are taken relative to the block's first row (pivot) so that var = E[d^2] - E[d]^2 does not cancel.
// partial: [row_blocks][3][H] = (mean, M2, n).
template <typename T>
__global__ __launch_bounds__(kStatsThreads) void bn_partial_kernel(const T* __restrict__ x, int64_t num_tokens, int hidden,
                                                                  int rows_per_block, float* __restrict__ partial) {
    constexpr int V = Elem<T>::kVec;
    __shared__ float red[3][2][kWave * V];   // waves 1..3 -> wave 0
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    const int col = ((int)blockIdx.y * kWave + lane) * V;
    const bool col_ok = col < hidden;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < num_tokens ? r0 + rows_per_block : num_tokens;
    float pivot[V], s1[V], s2[V];
    {
        u32x4_t raw = {0u, 0u, 0u, 0u};
        if (col_ok) raw = *reinterpret_cast<const u32x4_t*>(x + r0 * hidden + col);
        unpack16<T>(raw, pivot);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) s1[v] = s2[v] = 0.0f;
    if (col_ok) {
        // rows in batches of kBatch loads issued together (one memory round trip per batch); rows past the end are
        // read from the last row and left out of the sums
        constexpr int kBatch = 8;
        for (int64_t rb = r0 + wave; rb < r1; rb += 4 * kBatch) {
            u32x4_t raw[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int64_t r = rb + 4 * i;
                raw[i] = *reinterpret_cast<const u32x4_t*>(x + (r < r1 ? r : r1 - 1) * hidden + col);
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                if (rb + 4 * i < r1) {
                    float xv[V];
                    unpack16<T>(raw[i], xv);
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const float d = xv[v] - pivot[v];
                        s1[v] += d;
                        s2[v] = __builtin_fmaf(d, d, s2[v]);
                    }
                }
            }
        }
    }
    // waves 1..3 hand their sums (same pivot) to wave 0 through LDS
    if (wave > 0) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            red[wave - 1][0][lane * V + v] = s1[v];
            red[wave - 1][1][lane * V + v] = s2[v];
        }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                s1[v] += red[w][0][lane * V + v];
                s2[v] += red[w][1][lane * V + v];
            }
    }
    if (wave == 0 && col_ok) {
        const float n = (float)(r1 - r0);
        float* out = partial + (int64_t)blockIdx.x * 3 * hidden;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float m = s1[v] / n;
            out[col + v] = pivot[v] + m;
            out[hidden + col + v] = fmaxf(s2[v] - s1[v] * m, 0.0f);
            out[2 * hidden + col + v] = n;
        }
    }
}

// Statistics for the gate kernel's own prologue: few, tall row blocks, so that a gate workgroup can combine them itself.
// Block (rb, strip): rows [rb*rows_per_block, ...), 8*V columns (one 128-byte line per row for 16-bit elements).  A wave's
// load covers 8 rows (lanes 8 apart hold the same columns); the 4 waves take rows 8 apart.  Sums are relative to the
// block's first row, as in bn_partial_kernel.  partial: [row_blocks][2][H] = (mean, M2); the row count of a block follows
// from the geometry.
template <typename T>
__global__ __launch_bounds__(kStatsThreads) void bn_block_stats_kernel(const T* __restrict__ x, int64_t num_tokens, int hidden,
                                                                      int rows_per_block, float* __restrict__ partial) {
    constexpr int V = Elem<T>::kVec;
    __shared__ float red[3][2][8 * V];
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    const int sub = lane >> 3;                                   // which of the 8 rows of a load
    const int col = ((int)blockIdx.y * 8 + (lane & 7)) * V;
    const bool col_ok = col < hidden;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < num_tokens ? r0 + rows_per_block : num_tokens;
    float pivot[V], s1[V], s2[V];
    {
        u32x4_t raw = {0u, 0u, 0u, 0u};
        if (col_ok) raw = *reinterpret_cast<const u32x4_t*>(x + r0 * hidden + col);
        unpack16<T>(raw, pivot);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) s1[v] = s2[v] = 0.0f;
    if (col_ok) {
        constexpr int kBatch = 8;                                // loads issued together: one memory round trip per batch
        for (int64_t rb = r0 + wave * 8 + sub; rb < r1; rb += 32 * kBatch) {
            u32x4_t raw[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int64_t r = rb + 32 * i;
                raw[i] = *reinterpret_cast<const u32x4_t*>(x + (r < r1 ? r : r1 - 1) * hidden + col);
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                if (rb + 32 * i < r1) {
                    float xv[V];
                    unpack16<T>(raw[i], xv);
#pragma unroll
                    for (int v = 0; v < V; ++v) {
                        const float d = xv[v] - pivot[v];
                        s1[v] += d;
                        s2[v] = __builtin_fmaf(d, d, s2[v]);
                    }
                }
            }
        }
    }
    // the 8 row lanes of a wave (lane distance 8, 16, 32), then waves 1..3 -> wave 0 through LDS; fixed order
#pragma unroll
    for (int v = 0; v < V; ++v) {
#pragma unroll
        for (int m = 8; m < kWave; m <<= 1) {
            s1[v] += __shfl_xor(s1[v], m, kWave);
            s2[v] += __shfl_xor(s2[v], m, kWave);
        }
    }
    if (wave > 0 && lane < 8) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            red[wave - 1][0][lane * V + v] = s1[v];
            red[wave - 1][1][lane * V + v] = s2[v];
        }
    }
    __syncthreads();
    if (wave == 0 && lane < 8 && col_ok) {
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                s1[v] += red[w][0][lane * V + v];
                s2[v] += red[w][1][lane * V + v];
            }
        const float n = (float)(r1 - r0);
        float* out = partial + (int64_t)blockIdx.x * 2 * hidden;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            const float m = s1[v] / n;
            out[col + v] = pivot[v] + m;
            out[hidden + col + v] = fmaxf(s2[v] - s1[v] * m, 0.0f);
        }
    }
}

template <typename TS> __device__ inline float load_stat(const void* p, int i) { return Elem<TS>::to_f32(((const TS*)p)[i]); }
template <typename TS> __device__ inline void store_stat(void* p, int i, float v) { ((TS*)p)[i] = Elem<TS>::from_f32(v); }

// 64 columns per block, 16 waves: wave w takes row-block partials w, w+16, ... (at most kMaxRowBlocks/16 = 16, all
// loaded before any is used so that one memory round trip covers them).  Two passes: N = sum n_b and
// mean = sum n_b*mean_b / N, then M2 = sum [M2_b + n_b*(mean_b - mean)^2].
// training: batch statistics; else the running statistics.  mean_rstd: [2][H] fp32.
constexpr int kFinalizeWaves = 16;
template <typename TS>
__global__ __launch_bounds__(kFinalizeWaves* kWave) void bn_finalize_kernel(
    const float* __restrict__ partial, int row_blocks, int hidden, int training, float momentum, float eps,
    void* running_mean, void* running_var, int64_t* num_batches_tracked, float* __restrict__ mean_rstd) {
    constexpr int PER = kMaxRowBlocks / kFinalizeWaves;
    __shared__ float red[kFinalizeWaves][2][kWave];
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    const int h = (int)blockIdx.x * kWave + lane;
    if (blockIdx.x == 0 && threadIdx.x == 0 && training && num_batches_tracked != nullptr) *num_batches_tracked += 1;
    const bool h_ok = h < hidden;
    float mean = 0.0f, m2 = 0.0f, n = 0.0f;
    if (training) {
        float mb[PER], m2b[PER], nb[PER];
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int b = wave + i * kFinalizeWaves;
            const bool ok = h_ok && b < row_blocks;
            const float* p = partial + (int64_t)(ok ? b : 0) * 3 * hidden + (h_ok ? h : 0);
            mb[i] = ok ? p[0] : 0.0f;
            m2b[i] = ok ? p[hidden] : 0.0f;
            nb[i] = ok ? p[2 * hidden] : 0.0f;
        }
        float sn = 0.0f, snm = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            sn += nb[i];
            snm = __builtin_fmaf(nb[i], mb[i], snm);
        }
        red[wave][0][lane] = sn;
        red[wave][1][lane] = snm;
        __syncthreads();
        float tn = 0.0f, tnm = 0.0f;
#pragma unroll
        for (int w = 0; w < kFinalizeWaves; ++w) {
            tn += red[w][0][lane];
            tnm += red[w][1][lane];
        }
        n = tn;
        mean = tnm / fmaxf(tn, 1.0f);
        __syncthreads();
        float sm2 = 0.0f;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const float d = mb[i] - mean;
            sm2 += __builtin_fmaf(nb[i] * d, d, m2b[i]);
        }
        red[wave][0][lane] = sm2;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < kFinalizeWaves; ++w) m2 += red[w][0][lane];
    }
    if (wave != 0 || !h_ok) return;
    float var;
    if (training) {
        var = m2 / n;                                   // biased: what normalises the batch
        if (running_mean != nullptr && running_var != nullptr) {
            const float unbiased = n > 1.0f ? m2 / (n - 1.0f) : var;
            store_stat<TS>(running_mean, h, (1.0f - momentum) * load_stat<TS>(running_mean, h) + momentum * mean);
            store_stat<TS>(running_var, h, (1.0f - momentum) * load_stat<TS>(running_var, h) + momentum * unbiased);
        }
    } else {
        mean = load_stat<TS>(running_mean, h);
        var = load_stat<TS>(running_var, h);
    }
    mean_rstd[h] = mean;
    mean_rstd[hidden + h] = 1.0f / sqrtf(var + eps);
}

// logits[M, N] = normalise(x)[M, K] * W[N, K]^T for 16-bit activations: 64x64 tiles (256 of them at T=4096, 2*nk=256),
// 4 waves of one 32x32 MFMA tile each, register-staged LDS tiles (the A tile is normalised between the global load and
// the LDS store).  With one such workgroup per CU nothing else hides the global-load latency, so the packets of the
// next kGatePrefetch k-tiles are kept in flight in registers.
constexpr int kGatePrefetch = 3;
constexpr int kGateMaxK = 8192;     // mean / rstd of all k are staged in LDS once: 2 * 4 * K bytes

// split != 0: half h of the outputs (columns [h*N/2, (h+1)*N/2)) scores only half h of the normalised activations,
// w is [N, K/2]: the product-key form in which each sub-key table sees its own half of the query (a block-diagonal gate).
// KG > 1: the k-tiles are dealt to KG groups of four waves (group g takes k-tiles g, g + KG, ...), each with LDS tiles
// and an accumulator of its own, and the groups' accumulators are added in group order through LDS at the end.  With
// 256 tiles for 256 compute units a tile's k loop is a chain of global-load latencies; KG = 4 runs four of them side by
// side on the same compute unit.  The result depends on KG (another summation order), not on anything else.
template <typename T, int KG>
__global__ __launch_bounds__(256 * KG) __attribute__((amdgpu_waves_per_eu(4, 4))) void router_gate_kernel(const T* __restrict__ x, const T* __restrict__ w, GateStats st,
                                                          float* __restrict__ logits32, T* __restrict__ logits, int M, int N,
                                                          int K_full, int tiles_m, int tiles_n, int split, int xcds) {
    using Frag = typename Mfma32<T>::Frag;
    constexpr int BM = 64, BN = 64, CH = 2;   // CH = 16-byte packets per thread per tile and operand
    constexpr int D = KG > 1 ? 4 : kGatePrefetch;
    __shared__ __attribute__((aligned(16))) T tiles[KG][2][BM * kTileK];
    extern __shared__ __attribute__((aligned(16))) float stats[];   // [2][Kpad]: mean, rstd
    int tm, tn;
    tile_of_block(tiles_m, tiles_n, xcds, tm, tn);
    const int m0 = tm * BM, n0 = tn * BN;
    const int tid_all = (int)threadIdx.x;
    const int grp = __builtin_amdgcn_readfirstlane(tid_all / 256);
    const int tid = tid_all % 256, lane = tid & 63, wave = tid >> 6;
    T* As = tiles[grp][0];
    T* Bs = tiles[grp][1];
    const int wm = wave >> 1, wn = wave & 1;
    const int ch = tid % kTileChunks;          // this thread's packet column inside a k-tile: the same for all its packets
    const int row0 = tid / kTileChunks;        // rows row0 and row0 + 32
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};
    // the k range of this tile: all of it, or the half of the activations its columns score (tiles do not straddle halves)
    const int K = split ? K_full / 2 : K_full;
    const int k_off = (split && n0 >= N / 2) ? K : 0;
    const int k_tiles = (K + kTileK - 1) / kTileK;
    const int kpad = k_tiles * kTileK;
    const int steps = (k_tiles + KG - 1) / KG;         // k-tile of step s in this group: grp + s * KG
    u32x4_t ra[D][CH], rb[D][CH];

    auto load_global = [&](int step, int slot) {
        const int kt = grp + step * KG;
        const int gk = kt * kTileK + ch * 8;
        const bool k_ok = kt < k_tiles && gk < K;
#pragma unroll
        for (int it = 0; it < CH; ++it) {
            const int gm = m0 + row0 + it * 32, gn = n0 + row0 + it * 32;
            ra[slot][it] = (gm < M && k_ok) ? *reinterpret_cast<const u32x4_t*>(x + (int64_t)gm * K_full + k_off + gk) : zero4;
            rb[slot][it] = (gn < N && k_ok) ? *reinterpret_cast<const u32x4_t*>(w + (int64_t)gn * K + gk) : zero4;
        }
    };
    auto store_lds = [&](int step, int slot) {
        const int kt = grp + step * KG;
        const float* mu = stats + (kt < k_tiles ? kt : 0) * kTileK + ch * 8;     // a step beyond the range multiplies zeros
        const float* rs = mu + kpad;
        float m8[8], r8[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            m8[i] = mu[i];
            r8[i] = rs[i];
        }
#pragma unroll
        for (int it = 0; it < CH; ++it) {
            *reinterpret_cast<u32x4_t*>(&As[swizzled_offset(row0 + it * 32, ch)]) =
                kt < k_tiles ? normalise16<T>(ra[slot][it], m8, r8) : zero4;
            *reinterpret_cast<u32x4_t*>(&Bs[swizzled_offset(row0 + it * 32, ch)]) = rb[slot][it];
        }
    };
    f32x16_t acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    const int frow = lane & 31, fhalf = lane >> 5;
    // with k groups the operands of the first steps are requested before the statistics are combined: the two latencies overlap
    // (of the first two steps: the block statistics need the other registers)
    if (KG > 1) {
#pragma unroll
        for (int d = 0; d < 2; ++d) load_global(d, d);
    }
    stage_stats<KG == 1 ? 2 : 1>(st, stats, kpad, K, K_full, k_off, tn == (k_off ? tiles_n / 2 : 0), tm, tiles_m, blockIdx.x == 0);   // before the other loads claim its registers
#pragma unroll
    for (int d = KG > 1 ? 2 : 0; d < D; ++d) load_global(d, d);
    __syncthreads();               // stats[] visible
    // the step loop is unrolled by D so that the register slot of a tile is a compile-time index; every group runs every
    // step (a step beyond its k-tiles multiplies zeros), so the barriers are reached by all waves
    for (int s0 = 0; s0 < steps; s0 += D) {
#pragma unroll
        for (int d = 0; d < D; ++d) {
            const int step = s0 + d;
            if (step < steps) {
                store_lds(step, d);
                load_global(step + D, d);        // slot d is free again
                __syncthreads();
#pragma unroll
                for (int ks = 0; ks < kTileK / 16; ++ks) {
                    const int chunk = ks * 2 + fhalf;
                    const Frag fa = *reinterpret_cast<const Frag*>(&As[swizzled_offset(wm * 32 + frow, chunk)]);
                    const Frag fb = *reinterpret_cast<const Frag*>(&Bs[swizzled_offset(wn * 32 + frow, chunk)]);
                    acc = Mfma32<T>::run(fa, fb, acc);
                }
                __syncthreads();
            }
        }
    }
    if (KG > 1) {
        // groups 1 .. KG-1 hand their accumulators over through the tile memory; group 0 adds them in group order
        float* red = reinterpret_cast<float*>(&tiles[0][0][0]);
        static_assert(KG == 1 || (KG - 1) * BM * BN * sizeof(float) <= sizeof(tiles), "reduction fits the tile memory");
        if (grp > 0) {
#pragma unroll
            for (int v = 0; v < 16; ++v) red[(grp - 1) * BM * BN + (wave * 16 + v) * kWave + lane] = acc[v];
        }
        __syncthreads();
        if (grp > 0) return;
#pragma unroll
        for (int g = 1; g < KG; ++g)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] += red[(g - 1) * BM * BN + (wave * 16 + v) * kWave + lane];
    }
    const int col = n0 + wn * 32 + frow;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = m0 + wm * 32 + 8 * (v / 4) + 4 * fhalf + (v % 4);
        if (row < M && col < N) {
            logits32[(int64_t)row * N + col] = acc[v];
            logits[(int64_t)row * N + col] = Elem<T>::from_f32(acc[v]);
        }
    }
}

template <typename T, int MT, int NT, bool STAGED>
__global__ __launch_bounds__(kGateWaves* kWave) void router_gate_splitk_kernel(
    const T* __restrict__ x, const T* __restrict__ w, GateStats st, float* __restrict__ logits32, T* __restrict__ logits, int M, int N,
    int K_full, int tiles_m, int tiles_n, int split, int xcds) {
    extern __shared__ __attribute__((aligned(16))) float stats[];
    __shared__ __attribute__((aligned(16))) char lds[kGateLds<MT, NT>];
    router_gate_splitk_tile<T, MT, NT, STAGED>(x, w, st, logits32, logits, M, N, K_full, tiles_m, tiles_n, split, xcds, lds, stats,
                                               (int)blockIdx.x, (int)gridDim.x);
}

// q = round_T((x - mean) * rstd), 16 bytes per thread: the normalised activations as a stand-alone batch-norm emits them,
// for the gate product on the shared MLP's tiled kernel (many tokens).  mean_rstd: [2][hidden].
template <typename T>
__global__ __launch_bounds__(256) void bn_apply_kernel(const u32x4_t* __restrict__ x, const float* __restrict__ mean_rstd,
                                                       u32x4_t* __restrict__ q, int64_t packets, int hidden) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= packets) return;
    const int col = (int)(i % (hidden / 8)) * 8;
    float m8[8], r8[8];
#pragma unroll
    for (int v = 0; v < 8; ++v) {
        m8[v] = mean_rstd[col + v];
        r8[v] = mean_rstd[hidden + col + v];
    }
    q[i] = normalise16<T>(x[i], m8, r8);
}

struct ProloguePlan {
    int row_blocks, rows_per_block;
    size_t off_partial, off_mean_rstd, off_q, base_bytes, bytes;
    bool tiled_gate;     // enough tokens for the gate product to run on 256 x 256 tiles from a normalised copy of x
};

ProloguePlan plan_prologue(int64_t T_, int H, int nk) {
    ProloguePlan p;
    int64_t rb = (T_ + 31) / 32;
    p.row_blocks = (int)(rb < 1 ? 1 : (rb > kMaxRowBlocks ? kMaxRowBlocks : rb));
    p.rows_per_block = (int)((T_ + p.row_blocks - 1) / p.row_blocks);
    p.row_blocks = (int)((T_ + p.rows_per_block - 1) / p.rows_per_block);
    p.off_partial = 0;
    p.off_mean_rstd = round_up((size_t)kMaxRowBlocks * 3 * (size_t)H * 4, 256);
    p.base_bytes = round_up(p.off_mean_rstd + 2 * (size_t)H * 4, 256);
    // the normalised copy (16-bit activations; callers whose workspace stops at base_bytes keep the 64 x 64 gate kernel)
    p.tiled_gate = gemm_nt_dual_usable(T_, 2 * nk, H);
    p.off_q = p.base_bytes;
    p.bytes = p.base_bytes + (p.tiled_gate ? round_up((size_t)T_ * (size_t)H * 2, 256) : 0);
    return p;
}

// Row blocks of the statistics the gate kernel combines itself: at most kFoldMaxRowBlocks, at least 128 rows each.
struct BlockStatsPlan { int row_blocks, rows_per_block; };
BlockStatsPlan plan_block_stats(int64_t T_) {
    BlockStatsPlan p;
    int64_t rb = (T_ + 127) / 128;
    rb = rb < 1 ? 1 : (rb > kFoldMaxRowBlocks ? kFoldMaxRowBlocks : rb);
    p.rows_per_block = (int)((T_ + rb - 1) / rb);
    p.row_blocks = (int)((T_ + p.rows_per_block - 1) / p.rows_per_block);
    return p;
}

template <typename T>
void launch_block_stats(const void* x, int64_t T_, int H, const BlockStatsPlan& p, float* partial, hipStream_t stream) {
    constexpr int V = Elem<T>::kVec;
    const int strips = (H + 8 * V - 1) / (8 * V);
    hipLaunchKernelGGL((bn_block_stats_kernel<T>), dim3((unsigned)p.row_blocks, (unsigned)strips), dim3(kStatsThreads), 0, stream,
                       (const T*)x, T_, H, p.rows_per_block, partial);
}

template <typename T>
void launch_stats(const void* x, int64_t T_, int H, const ProloguePlan& p, float* partial, hipStream_t stream) {
    constexpr int V = Elem<T>::kVec;
    const int strips = (H + kWave * V - 1) / (kWave * V);
    hipLaunchKernelGGL((bn_partial_kernel<T>), dim3((unsigned)p.row_blocks, (unsigned)strips), dim3(kStatsThreads), 0, stream,
                       (const T*)x, T_, H, p.rows_per_block, partial);
}

template <typename TS>
void launch_finalize(const float* partial, const ProloguePlan& p, int H, int training, float momentum, float eps,
                     void* rm, void* rv, int64_t* nbt, float* mean_rstd, hipStream_t stream) {
    hipLaunchKernelGGL((bn_finalize_kernel<TS>), dim3((unsigned)((H + kWave - 1) / kWave)), dim3(kFinalizeWaves * kWave), 0, stream, partial,
                       p.row_blocks, H, training, momentum, eps, rm, rv, nbt, mean_rstd);
}

// The smallest tiles that still are one round of workgroups: 1024 tokens, 1024 columns, 256 outputs in bf16 take 14.7 us with the
// statistics launch on 32 x 32 tiles (256 of them), 23 on 16 x 32 and 17 on 32 x 64.  fp32 beyond a round goes on with 64 x 64 tiles.
template <typename T>
void launch_gate_splitk(const void* x, const void* w, const GateStats& st, float* logits32, void* logits, int M, int N, int K, int split,
                        hipStream_t stream) {
    const int cus = chip_info().cus, xcds = chip_info().xcds;
    const bool staged = K <= kGateStagedK;
    const int k_pad = (K + 63) / 64 * 64;
#define FMOE_GATE_GO(MT, NT, STAGED)                                                                                            \
    do {                                                                                                                        \
        const int tiles_m = (M + 16 * MT - 1) / (16 * MT), tiles_n = (N + 16 * NT - 1) / (16 * NT);                             \
        const int grid = (tiles_m * tiles_n + xcds - 1) / xcds * xcds;                                                          \
        hipLaunchKernelGGL((router_gate_splitk_kernel<T, MT, NT, STAGED>), dim3((unsigned)grid), dim3(kGateWaves * kWave),      \
                           STAGED ? (size_t)k_pad * 8 : 0, stream, (const T*)x, (const T*)w, st, logits32, (T*)logits, M, N, K, \
                           tiles_m, tiles_n, split, xcds);                                                                      \
    } while (0)
#define FMOE_GATE_TILE(MT, NT)                     \
    do {                                           \
        if (staged) FMOE_GATE_GO(MT, NT, true);    \
        else FMOE_GATE_GO(MT, NT, false);          \
    } while (0)
    if (gate_tiles(M, N, 1, 1) <= cus) FMOE_GATE_TILE(1, 1);
    else if (gate_tiles(M, N, 1, 2) <= cus) FMOE_GATE_TILE(1, 2);
    else if (gate_tiles(M, N, 2, 2) <= cus) FMOE_GATE_TILE(2, 2);
    else if (sizeof(T) == 2 || gate_tiles(M, N, 2, 4) <= cus) FMOE_GATE_TILE(2, 4);
    else FMOE_GATE_TILE(4, 4);
#undef FMOE_GATE_TILE
#undef FMOE_GATE_GO
}

// ------------------------------------------------------------------------------------------------------------
// Backward of the prologue (batch norm + gate product), for the differentiable composition of the block.
//   d   = dlogits (fp32) rounded to the activation dtype          q = round((x - mean) * rstd)     [recomputed]
//   dWr = d^T q,  dq = d Wr                                        (gemm_backward)
//   dx  = rstd * (dq - mean_t(dq) - xhat * mean_t(dq * xhat))      (training; xhat unrounded)   |   rstd * dq  (evaluation)
// ------------------------------------------------------------------------------------------------------------
// Workgroup b: row b / col_blocks of q (and of d), packets (b % col_blocks) * 256 + thread of that row.
template <typename T>
__global__ __launch_bounds__(256) void prologue_bwd_prepare_kernel(const float* __restrict__ dlogits, const T* __restrict__ x,
                                                                  const float* __restrict__ mean_rstd, T* __restrict__ d16,
                                                                  T* __restrict__ q, int hidden, int n_out, int n_pad, int col_blocks) {
    constexpr int V = Elem<T>::kVec;
    const uint32_t row = blockIdx.x / (uint32_t)col_blocks;
    const int pc = (int)(blockIdx.x % (uint32_t)col_blocks) * 256 + (int)threadIdx.x;
    const int col = pc * V;
    if (col < hidden) {
        const int64_t at = (int64_t)row * hidden + col;
        float xv[V], qv[V];
        unpack16<T>(*reinterpret_cast<const u32x4_t*>(x + at), xv);
#pragma unroll
        for (int h = 0; h < V / 4; ++h) {
            const f32x4_t m = *reinterpret_cast<const f32x4_t*>(mean_rstd + col + 4 * h);
            const f32x4_t r = *reinterpret_cast<const f32x4_t*>(mean_rstd + hidden + col + 4 * h);
#pragma unroll
            for (int j = 0; j < 4; ++j) qv[4 * h + j] = (xv[4 * h + j] - m[j]) * r[j];
        }
        *reinterpret_cast<u32x4_t*>(q + at) = pack16<T>(qv);
    }
    if (col < n_pad) {
        // rows of d are padded with zeros to a whole number of packets
        const int64_t at = (int64_t)row * n_out + col;
        float dv[V];
        if (n_out % V == 0) {
#pragma unroll
            for (int h = 0; h < V / 4; ++h) {
                const f32x4_t g = *reinterpret_cast<const f32x4_t*>(dlogits + at + 4 * h);
#pragma unroll
                for (int j = 0; j < 4; ++j) dv[4 * h + j] = g[j];
            }
        } else {
#pragma unroll
            for (int j = 0; j < V; ++j) dv[j] = col + j < n_out ? dlogits[at + j] : 0.0f;
        }
        *reinterpret_cast<u32x4_t*>(d16 + (int64_t)row * n_pad + col) = pack16<T>(dv);
    }
}

// partial: [row_blocks][2][H] = (sum dq, sum dq * xhat) over the block's rows.  A workgroup takes a strip of 2^lane_bits packets, a wave 64
// lanes of its rows, rows 256 >> lane_bits apart.
template <typename T>
__global__ __launch_bounds__(kStatsThreads) void bn_bwd_partial_kernel(const T* __restrict__ x, const T* __restrict__ dq,
                                                                      const float* __restrict__ mean_rstd, int64_t num_tokens,
                                                                      int hidden, int rows_per_block, int lane_bits, float* __restrict__ partial) {
    constexpr int V = Elem<T>::kVec;
    __shared__ float red[3][2][kWave * V];
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    const int width = 1 << lane_bits, wave_rows = kWave >> lane_bits, step = 4 * wave_rows;
    const int col = ((int)blockIdx.y * width + (lane & (width - 1))) * V;
    const bool col_ok = col < hidden;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < num_tokens ? r0 + rows_per_block : num_tokens;
    float mean[V], rstd[V], s1[V], s2[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        mean[v] = col_ok ? mean_rstd[col + v] : 0.0f;
        rstd[v] = col_ok ? mean_rstd[hidden + col + v] : 0.0f;
        s1[v] = s2[v] = 0.0f;
    }
    if (col_ok) {
        constexpr int kBatch = 4;                                // rows of x and dq issued together: one memory round trip per batch
        for (int64_t rb = r0 + wave * wave_rows + (lane >> lane_bits); rb < r1; rb += step * kBatch) {
            u32x4_t raw[kBatch], raw_dq[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int64_t r = rb + step * i < r1 ? rb + step * i : r1 - 1;
                raw[i] = *reinterpret_cast<const u32x4_t*>(x + r * hidden + col);
                raw_dq[i] = *reinterpret_cast<const u32x4_t*>(dq + r * hidden + col);
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                if (rb + step * i >= r1) continue;
                float xv[V], gv[V];
                unpack16<T>(raw[i], xv);
                unpack16<T>(raw_dq[i], gv);
#pragma unroll
                for (int v = 0; v < V; ++v) {
                    s1[v] += gv[v];
                    s2[v] = __builtin_fmaf(gv[v], (xv[v] - mean[v]) * rstd[v], s2[v]);
                }
            }
        }
    }
    // the row lanes of a wave, then waves 1..3 -> wave 0 through LDS; fixed order
    for (int m = width; m < kWave; m <<= 1)
#pragma unroll
        for (int v = 0; v < V; ++v) {
            s1[v] += __shfl_xor(s1[v], m, kWave);
            s2[v] += __shfl_xor(s2[v], m, kWave);
        }
    if (wave > 0 && lane < width) {
#pragma unroll
        for (int v = 0; v < V; ++v) {
            red[wave - 1][0][lane * V + v] = s1[v];
            red[wave - 1][1][lane * V + v] = s2[v];
        }
    }
    __syncthreads();
    if (wave == 0 && lane < width && col_ok) {
#pragma unroll
        for (int w = 0; w < 3; ++w)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                s1[v] += red[w][0][lane * V + v];
                s2[v] += red[w][1][lane * V + v];
            }
        float* out = partial + (int64_t)blockIdx.x * 2 * hidden;
#pragma unroll
        for (int v = 0; v < V; ++v) {
            out[col + v] = s1[v];
            out[hidden + col + v] = s2[v];
        }
    }
}

// The row blocks' column sums added, 32 columns to a workgroup, eight threads to a column: [2][H] after the row blocks.
__global__ __launch_bounds__(256) void bn_bwd_fold_kernel(const float* __restrict__ partial, int row_blocks, int hidden, float* __restrict__ sums) {
    __shared__ float red[8][32];
    const int c = (int)(blockIdx.x * 32 + (threadIdx.x & 31)), group = (int)(threadIdx.x >> 5);
    const bool col_ok = c < 2 * hidden;
    float acc[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) acc[u] = 0.0f;
    for (int b0 = group; b0 < row_blocks; b0 += 64) {
        float got[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int b = b0 + 8 * u < row_blocks ? b0 + 8 * u : row_blocks - 1;      // clamped: every load is unconditional
            got[u] = partial[(int64_t)b * 2 * hidden + (col_ok ? c : 0)];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc[u] += b0 + 8 * u < row_blocks ? got[u] : 0.0f;
    }
    float a = 0.0f;
#pragma unroll
    for (int u = 0; u < 8; ++u) a += acc[u];
    red[group][threadIdx.x & 31] = a;
    __syncthreads();
    if (group != 0 || !col_ok) return;
#pragma unroll
    for (int g = 1; g < 8; ++g) a += red[g][threadIdx.x];
    sums[c] = a;
}

// dx, and the block's other token gradients added in fp32: addend0 and addend1 (either may be NULL, or dx itself: a thread reads its
// packet before it writes), and fp32 planes of slices of k (of the MLP's dx, whose sum nobody else needs).
// A workgroup takes a strip of 2^lane_bits packets (64, or what a shorter row has) and rows_per_block rows, its waves 64 lanes of them, the
// four steps apart.  training: it first adds the blocks'
// column sums to the two means of the formula, a quarter of the blocks to a wave.  Where a launch of its own had formed the means: 4096
// tokens, 1024 columns 22.8 us in three launches, 18.7 in two; 615 tokens, 776 columns, with four planes that another launch had
// added, 17.6 in four and 10.7 in two.
template <typename T>
__global__ __launch_bounds__(256) void bn_bwd_apply_kernel(const T* __restrict__ x, const T* __restrict__ dq,
                                                           const float* __restrict__ mean_rstd, const float* __restrict__ partial,
                                                           int row_blocks, float inv_tokens, const T* addend0, const T* addend1,
                                                           const float* __restrict__ planes, int slices, T* dx, int64_t num_tokens,
                                                           int hidden, int rows_per_block, int lane_bits) {
    constexpr int V = Elem<T>::kVec, kShare = kFoldMaxRowBlocks / 4;
    __shared__ __attribute__((aligned(16))) float shared_sums[4][2][kWave * V];
    const int lane = lane_id(), wave = (int)(threadIdx.x >> 6);
    const int wave_rows = kWave >> lane_bits, step = 4 * wave_rows;
    const int col = ((int)blockIdx.y * kWave + (lane & ((1 << lane_bits) - 1))) * V;
    const bool col_ok = col < hidden;
    const int at_col = col_ok ? col : 0;
    // a wave's next row is asked for before the current one is worked on, the first before the means
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = r0 + rows_per_block < num_tokens ? r0 + rows_per_block : num_tokens;
    const T* const rows[4] = {x, dq, addend0 != nullptr ? addend0 : x, addend1 != nullptr ? addend1 : x};
    u32x4_t raw[4];
    auto load = [&](int64_t r) {
        const int64_t at = (r < r1 ? r : r1 - 1) * hidden + at_col;
#pragma unroll
        for (int i = 0; i < 4; ++i) raw[i] = *reinterpret_cast<const u32x4_t*>(rows[i] + at);
    };
    const int64_t first = r0 + wave * wave_rows + (lane >> lane_bits);
    load(first);
    float mean[V], rstd[V], m1[V], m2[V];
#pragma unroll
    for (int v = 0; v < V; v += 4) {
        const f32x4_t a = *reinterpret_cast<const f32x4_t*>(mean_rstd + at_col + v);
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(mean_rstd + hidden + at_col + v);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            mean[v + j] = a[j];
            rstd[v + j] = b[j];
            m1[v + j] = m2[v + j] = 0.0f;            // evaluation mode: the formula reduces to rstd * dq
        }
    }
    if (partial != nullptr) {
        f32x4_t got[kShare][2][V / 4];
#pragma unroll
        for (int u = 0; u < kShare; ++u) {
            const int b = wave * kShare + u < row_blocks ? wave * kShare + u : 0;      // clamped: every load is unconditional
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int v = 0; v < V; v += 4) got[u][h][v / 4] = *reinterpret_cast<const f32x4_t*>(partial + (int64_t)(2 * b + h) * hidden + at_col + v);
        }
#pragma unroll
        for (int u = 0; u < kShare; ++u) {
            if (wave * kShare + u >= row_blocks) continue;
#pragma unroll
            for (int v = 0; v < V; ++v) {
                m1[v] += got[u][0][v / 4][v % 4];
                m2[v] += got[u][1][v / 4][v % 4];
            }
        }
#pragma unroll
        for (int v = 0; v < V; v += 4) {
            *reinterpret_cast<f32x4_t*>(&shared_sums[wave][0][lane * V + v]) = f32x4_t{m1[v], m1[v + 1], m1[v + 2], m1[v + 3]};
            *reinterpret_cast<f32x4_t*>(&shared_sums[wave][1][lane * V + v]) = f32x4_t{m2[v], m2[v + 1], m2[v + 2], m2[v + 3]};
        }
        __syncthreads();
#pragma unroll
        for (int v = 0; v < V; v += 4) {
            f32x4_t a = *reinterpret_cast<const f32x4_t*>(&shared_sums[0][0][lane * V + v]);
            f32x4_t b = *reinterpret_cast<const f32x4_t*>(&shared_sums[0][1][lane * V + v]);
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                a += *reinterpret_cast<const f32x4_t*>(&shared_sums[w][0][lane * V + v]);
                b += *reinterpret_cast<const f32x4_t*>(&shared_sums[w][1][lane * V + v]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                m1[v + j] = a[j] * inv_tokens;
                m2[v + j] = b[j] * inv_tokens;
            }
        }
    }
    if (!col_ok) return;
    for (int64_t r = first; r < r1; r += step) {
        const int64_t at = r * hidden + col;
        float xv[V], gv[V], ov[V], more[2][V];
        unpack16<T>(raw[0], xv);
        unpack16<T>(raw[1], gv);
        unpack16<T>(raw[2], more[0]);
        unpack16<T>(raw[3], more[1]);
        if (r + step < r1) load(r + step);             // never this row, which may be written in place
#pragma unroll
        for (int v = 0; v < V; ++v) ov[v] = rstd[v] * (gv[v] - m1[v] - (xv[v] - mean[v]) * rstd[v] * m2[v]);
        if (planes != nullptr) {
            float sum[V];
#pragma unroll
            for (int v = 0; v < V; ++v) sum[v] = 0.0f;
            for (int s = 0; s < slices; ++s)
#pragma unroll
                for (int v = 0; v < V; v += 4) {
                    const f32x4_t p = *reinterpret_cast<const f32x4_t*>(planes + ((int64_t)s * num_tokens + r) * hidden + col + v);
#pragma unroll
                    for (int j = 0; j < 4; ++j) sum[v + j] += p[j];
                }
#pragma unroll
            for (int v = 0; v < V; ++v) ov[v] += sum[v];
        }
#pragma unroll
        for (int v = 0; v < V; ++v) {
            if (addend0 != nullptr) ov[v] += more[0][v];
            if (addend1 != nullptr) ov[v] += more[1][v];
        }
        *reinterpret_cast<u32x4_t*>(dx + at) = pack16<T>(ov);
    }
}

// Packets of a row that a wave's lanes have side by side: 64, or what a shorter row has.
int row_lane_bits(int packets) {
    int bits = 6;
    while (bits > 0 && packets <= 1 << (bits - 1)) --bits;
    return bits;
}

// Row blocks of the batch-norm gradient's column sums.  Few tokens: at most kFoldMaxRowBlocks of them on strips of 8 packets, which the last
// launch adds.  From 16384 on that leaves rows of few strips on few compute units and reads each row in pieces of 128 bytes: as many row
// blocks as fill the chip on strips of a wave's width, added by a launch of their own.  The router prologue's backward in bf16, 32 keys, two
// launches | three: 12000 tokens, 512 columns 51.2 | 53.5, 64 columns 39.6 | 38.2; 8192, 512 46.0 | 48.5; 16384, 64 58 | 45; 32768, 512 102 | 88.
constexpr int64_t kThreeLaunches = 16384;
struct ColumnSumsPlan { int row_blocks, rows_per_block, lane_bits; bool folded; };
ColumnSumsPlan plan_column_sums(int64_t T_, int packets) {
    const BlockStatsPlan few = plan_block_stats(T_);
    if (T_ < kThreeLaunches) return {few.row_blocks, few.rows_per_block, 3, false};
    const int bits = row_lane_bits(packets);
    const int64_t strips = (packets + (1 << bits) - 1) >> bits, wanted = 2 * chip_info().cus / strips + 1, most = (T_ + 31) / 32;
    int64_t rb = wanted < most ? wanted : most;
    if (rb > kMaxRowBlocks) rb = kMaxRowBlocks;
    const int rows = (int)((T_ + rb - 1) / rb);
    return {(int)((T_ + rows - 1) / rows), rows, bits, true};
}

// The two products, extents only.
void prologue_products(int T_, int H, int N, int n_pad, BackwardProduct (&q)[2]) {
    q[0] = {kBlasTN, N, H, T_, 1, nullptr, n_pad, nullptr, nullptr, H, nullptr};      // dWr = d^T q
    q[1] = {kBlasNN, T_, H, N, 1, nullptr, n_pad, nullptr, nullptr, H, nullptr};      // dq = d Wr
}

int check_prologue_backward(int64_t num_tokens, int hidden, int num_keys, int dtype) {
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "fmoe_router_prologue_backward: unknown dtype %d", dtype);
    FMOE_REQUIRE(num_tokens > 0 && hidden > 0 && num_keys > 0 && num_tokens < (1ll << 24), FMOE_ERR_BAD_SHAPE,
                 "fmoe_router_prologue_backward: bad shape T=%lld H=%d nk=%d", (long long)num_tokens, hidden, num_keys);
    const int vec = (int)(16 / dtype_size(dtype));
    FMOE_REQUIRE(hidden % vec == 0, FMOE_ERR_ALIGNMENT,
                 "fmoe_router_prologue_backward: hidden=%d must be a multiple of %d", hidden, vec);
    return FMOE_OK;
}

}  // namespace

PrologueBackwardPlan plan_prologue_backward(int64_t T_, int H, int nk, int dtype) {
    PrologueBackwardPlan p;
    const size_t elt = dtype_size(dtype);
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o = round_up(o + n, 256); return at; };
    const int vec = (int)(16 / elt), t = (int)T_;
    p.n_pad = (2 * nk + vec - 1) / vec * vec;
    p.off_d16 = take((size_t)T_ * p.n_pad * elt);
    p.off_q = take((size_t)T_ * H * elt);
    p.off_dq = take((size_t)T_ * H * elt);
    const ColumnSumsPlan sums = plan_column_sums(T_, (H + vec - 1) / vec);
    p.row_blocks = sums.row_blocks;
    p.rows_per_block = sums.rows_per_block;
    p.lane_bits = sums.lane_bits;
    p.folded = sums.folded;
    p.off_partial = take((size_t)(p.row_blocks + 1) * 2 * H * 4);
    BackwardProduct products[2];
    prologue_products(t, H, 2 * nk, p.n_pad, products);
    p.products = plan_products(products, 2, dtype);
    p.part_bytes = gemm_backward_workspace_bytes(products, 2, p.products, dtype);
    p.off_part = take(p.part_bytes);
    p.bytes = o;
    return p;
}

namespace {

template <typename T>
int launch_prologue_backward(const float* dlogits, const void* x, const void* gate_w, const float* mean_rstd, int training,
                             int64_t T_, int H, int nk, int dtype, void* dx, void* dgate_w, const TokenGradients& more, const PrologueBackwardPlan& p,
                             void* workspace, hipStream_t s, bool operands_ready) {
    constexpr int V = Elem<T>::kVec;
    char* ws = (char*)workspace;
    T *d16 = (T*)(ws + p.off_d16), *q = (T*)(ws + p.off_q), *dq = (T*)(ws + p.off_dq);
    float* partial = (float*)(ws + p.off_partial);
    const int N = 2 * nk;
    const int widest = H > p.n_pad ? H : p.n_pad;
    void* part = ws + p.off_part;
    const int col_blocks = ((widest + V - 1) / V + 255) / 256;
    if (!operands_ready) {
        hipLaunchKernelGGL((prologue_bwd_prepare_kernel<T>), dim3((unsigned)(T_ * col_blocks)), dim3(256), 0, s, dlogits,
                           (const T*)x, mean_rstd, d16, q, H, N, p.n_pad, col_blocks);
        FMOE_CHECK_LAUNCH("fmoe_router_prologue_backward(prepare)");
    }
    BackwardProduct products[2];
    prologue_products((int)T_, H, N, p.n_pad, products);
    products[0].A = products[1].A = d16;
    products[0].B0 = q, products[0].C = dgate_w;
    products[1].B0 = gate_w, products[1].C = dq;
    if (int rc = gemm_backward(products, 2, p.products, dtype, part, p.part_bytes, s)) return rc;
    if (training) {
        const int strips = (H / V + (1 << p.lane_bits) - 1) >> p.lane_bits;
        hipLaunchKernelGGL((bn_bwd_partial_kernel<T>), dim3((unsigned)p.row_blocks, (unsigned)strips), dim3(kStatsThreads), 0, s,
                           (const T*)x, (const T*)dq, mean_rstd, T_, H, p.rows_per_block, p.lane_bits, partial);
        FMOE_CHECK_LAUNCH("fmoe_router_prologue_backward(column sums)");
    }
    int row_blocks = p.row_blocks;
    if (training && p.folded) {
        float* sums = partial + (size_t)row_blocks * 2 * H;
        hipLaunchKernelGGL(bn_bwd_fold_kernel, dim3((unsigned)((2 * H + 31) / 32)), dim3(256), 0, s, (const float*)partial, row_blocks, H, sums);
        FMOE_CHECK_LAUNCH("fmoe_router_prologue_backward(row blocks)");
        partial = sums;
        row_blocks = 1;
    }
    // about two workgroups to a compute unit
    const int packets = H / V, lane_bits = row_lane_bits(packets);
    const int64_t strips = (packets + kWave - 1) / kWave, wanted = 2 * chip_info().cus / strips + 1, step = 4 * (kWave >> lane_bits);
    const int apply_rows = (int)((T_ + wanted * step - 1) / (wanted * step) * step);
    hipLaunchKernelGGL((bn_bwd_apply_kernel<T>), dim3((unsigned)((T_ + apply_rows - 1) / apply_rows), (unsigned)strips), dim3(256), 0, s, (const T*)x,
                       (const T*)dq, mean_rstd, training ? (const float*)partial : nullptr, row_blocks, 1.0f / (float)T_, (const T*)more.addend0,
                       (const T*)more.addend1, more.planes, more.slices, (T*)dx, T_, H, apply_rows, lane_bits);
    FMOE_CHECK_LAUNCH("fmoe_router_prologue_backward(apply)");
    return FMOE_OK;
}

}  // namespace
}  // namespace fmoe

extern "C" size_t fmoe_router_workspace_bytes(int64_t num_tokens, int hidden, int num_keys) {
    if (num_tokens <= 0 || hidden <= 0 || num_keys <= 0) return 0;
    return fmoe::plan_prologue(num_tokens, hidden, num_keys).bytes;
}

extern "C" int fmoe_router_forward(const void* x, const void* gate_w, void* running_mean, void* running_var,
                                   int64_t* num_batches_tracked, int stats_dtype, int training, float momentum,
                                   float eps, int64_t num_tokens, int hidden, int num_keys, int top_k, int dtype,
                                   int norm_topk_prob, void* router_logits, float* logits_fp32, float* scores,
                                   int64_t* indices, void* gates, void* workspace, size_t workspace_bytes, void* stream) {
    fmoe::clear_error();
    return fmoe::router_forward_impl(x, gate_w, running_mean, running_var, num_batches_tracked, stats_dtype, training,
                                     momentum, eps, num_tokens, hidden, num_keys, top_k, dtype, norm_topk_prob,
                                     router_logits, logits_fp32, scores, indices, gates, nullptr, 0u, workspace,
                                     workspace_bytes, (hipStream_t)stream);
}

extern "C" int fmoe_router_forward_split(const void* x, const void* sub_keys, void* running_mean, void* running_var,
                                         int64_t* num_batches_tracked, int stats_dtype, int training, float momentum,
                                         float eps, int64_t num_tokens, int hidden, int num_keys, int top_k, int dtype,
                                         int norm_topk_prob, void* router_logits, float* logits_fp32, float* scores,
                                         int64_t* indices, void* gates, void* workspace, size_t workspace_bytes, void* stream) {
    fmoe::clear_error();
    return fmoe::router_forward_impl(x, sub_keys, running_mean, running_var, num_batches_tracked, stats_dtype, training,
                                     momentum, eps, num_tokens, hidden, num_keys, top_k, dtype, norm_topk_prob,
                                     router_logits, logits_fp32, scores, indices, gates, nullptr, 0u, workspace,
                                     workspace_bytes, (hipStream_t)stream, 1);
}

extern "C" int fmoe_router_forward_noalloc(const void* x, const void* gate_w, void* running_mean, void* running_var,
                                           int64_t* num_batches_tracked, int stats_dtype, int training, float momentum,
                                           float eps, int64_t num_tokens, int hidden, int num_keys, int top_k, int dtype,
                                           int norm_topk_prob, void* router_logits, float* logits_fp32, float* scores,
                                           int64_t* indices, void* gates, void* stream) {
    using namespace fmoe;
    clear_error();
    FMOE_REQUIRE(hidden <= FMOE_NOALLOC_MAX_HIDDEN, FMOE_ERR_UNSUPPORTED,
                 "fmoe_router_forward_noalloc: hidden=%d exceeds the %d columns its static scratch is sized for; use "
                 "fmoe_router_forward with a workspace", hidden, FMOE_NOALLOC_MAX_HIDDEN);
    if (num_tokens <= 0 || hidden <= 0 || num_keys <= 0)   // rejected (or empty) below, before any scratch is needed
        return router_forward_impl(x, gate_w, running_mean, running_var, num_batches_tracked, stats_dtype, training, momentum,
                                   eps, num_tokens, hidden, num_keys, top_k, dtype, norm_topk_prob, router_logits, logits_fp32,
                                   scores, indices, gates, nullptr, 0u, nullptr, 0, (hipStream_t)stream);
    void* ws = nullptr;
    if (int rc = static_scratch(&ws)) return rc;
    return router_forward_impl(x, gate_w, running_mean, running_var, num_batches_tracked, stats_dtype, training, momentum,
                               eps, num_tokens, hidden, num_keys, top_k, dtype, norm_topk_prob, router_logits, logits_fp32,
                               scores, indices, gates, nullptr, 0u, ws, (size_t)FMOE_NOALLOC_SCRATCH_BYTES, (hipStream_t)stream, 0, 1);
}

// Statistics of the batch per row block, for a gate product that combines them itself: what to pass it.
size_t fmoe::router_block_stats_bytes(int hidden) { return (size_t)kFoldMaxRowBlocks * 2 * (size_t)hidden * 4; }
int fmoe::router_block_stats(const void* x, int64_t num_tokens, int hidden, int dtype, float* partial, int* row_blocks, int* rows_per_block,
                             hipStream_t s) {
    const BlockStatsPlan bp = plan_block_stats(num_tokens);
    *row_blocks = bp.row_blocks;
    *rows_per_block = bp.rows_per_block;
    switch (dtype) {
        case FMOE_F32: launch_block_stats<float>(x, num_tokens, hidden, bp, partial, s); break;
        case FMOE_BF16: launch_block_stats<bf16_t>(x, num_tokens, hidden, bp, partial, s); break;
        default: launch_block_stats<f16_t>(x, num_tokens, hidden, bp, partial, s); break;
    }
    FMOE_CHECK_LAUNCH("fmoe_block(batch statistics)");
    return FMOE_OK;
}

int fmoe::router_forward_impl(const void* x, const void* gate_w, void* running_mean, void* running_var,
                              int64_t* num_batches_tracked, int stats_dtype, int training, float momentum, float eps,
                              int64_t num_tokens, int hidden, int num_keys, int top_k, int dtype, int norm_topk_prob,
                              void* router_logits, float* logits_fp32, float* scores, int64_t* indices, void* gates,
                              uint32_t* row_offsets, uint32_t row_bytes, void* workspace, size_t workspace_bytes,
                              hipStream_t s, int split_query, int fixed_scratch, float* mean_rstd_out) {
    using namespace fmoe;
    FMOE_REQUIRE(!split_query || (num_keys % 64 == 0 && hidden % 2 == 0), FMOE_ERR_UNSUPPORTED,
                 "fmoe_router_forward_split: num_keys=%d must be a multiple of 64 and hidden=%d even", num_keys, hidden);
    FMOE_REQUIRE(dtype_ok(dtype) && dtype_ok(stats_dtype), FMOE_ERR_BAD_DTYPE,
                 "fmoe_router_forward: unknown dtype %d / statistics dtype %d", dtype, stats_dtype);
    FMOE_REQUIRE(num_tokens >= 0 && hidden > 0 && num_keys > 0, FMOE_ERR_BAD_SHAPE,
                 "fmoe_router_forward: bad shape T=%lld H=%d nk=%d", (long long)num_tokens, hidden, num_keys);
    FMOE_REQUIRE(top_k >= 0 && top_k <= num_keys, FMOE_ERR_TOPK_RANGE,
                 "num_experts_per_tok should be in [0, %d], but got %d", num_keys, top_k);
    FMOE_REQUIRE(dtype == FMOE_F32 || hidden <= kGateMaxK, FMOE_ERR_UNSUPPORTED,
                 "fmoe_router_forward: hidden=%d > %d for 16-bit activations", hidden, kGateMaxK);
    FMOE_REQUIRE(num_keys <= 32767 && router_topk_supported(num_keys, top_k) && num_tokens < (1ll << 31), FMOE_ERR_UNSUPPORTED,
                 "fmoe_router_forward: nk=%d top_k=%d T=%lld beyond what the kernels are built for", num_keys, top_k,
                 (long long)num_tokens);
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(!(training && num_tokens == 1), FMOE_ERR_BAD_SHAPE,
                 "Expected more than 1 value per channel when training, got input size [1, %d]", hidden);
    FMOE_REQUIRE(x && gate_w && router_logits && logits_fp32 && workspace, FMOE_ERR_NULL_POINTER,
                 "fmoe_router_forward: null tensor pointer");
    FMOE_REQUIRE(top_k == 0 || (scores && indices), FMOE_ERR_NULL_POINTER, "fmoe_router_forward: null scores/indices");
    FMOE_REQUIRE(training || (running_mean && running_var), FMOE_ERR_NULL_POINTER,
                 "fmoe_router_forward: evaluation mode needs running statistics");
    const int vec = (int)(16 / dtype_size(dtype));
    FMOE_REQUIRE(hidden % (split_query ? 2 * vec : vec) == 0 && aligned16(x) && aligned16(gate_w), FMOE_ERR_ALIGNMENT,
                 "fmoe_router_forward: hidden=%d must be a multiple of %d and tensors 16-byte aligned", hidden,
                 split_query ? 2 * vec : vec);
    const ProloguePlan p = plan_prologue(num_tokens, hidden, num_keys);
    // a workspace without room for the normalised copy (the fixed scratch of the no-allocation entry point) takes the
    // 64 x 64 gate kernel: the same sums in the same order
    const bool tiled_gate = p.tiled_gate && dtype != FMOE_F32 && !split_query && !fixed_scratch;
    const size_t need = fixed_scratch ? p.base_bytes : p.bytes;
    FMOE_REQUIRE(workspace_bytes >= need && aligned16(workspace), FMOE_ERR_WORKSPACE,
                 "fmoe_router_forward: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    char* ws = (char*)workspace;
    float* partial = (float*)(ws + p.off_partial);
    float* mean_rstd = mean_rstd_out ? mean_rstd_out : (float*)(ws + p.off_mean_rstd);
    float* logits32 = logits_fp32;

    const int M = (int)num_tokens, N = 2 * num_keys;
    const BlockStatsPlan bp = plan_block_stats(num_tokens);
    const int64_t tiles64 = (int64_t)((M + 63) / 64) * ((N + 63) / 64);
    // Every gate workgroup combining the block statistics itself saves a launch, but repeats the combination per tile: with more
    // than a couple of tiles per CU one finalize launch is cheaper.
    const bool splitk = gate_splitk_pays(M, N, dtype);
    const bool fold = tiles64 <= 2 * (int64_t)chip_info().cus && hidden <= (splitk ? kGateStagedK : kGateMaxK);
    if (training) {
        if (fold) {
            switch (dtype) {
                case FMOE_F32: launch_block_stats<float>(x, num_tokens, hidden, bp, partial, s); break;
                case FMOE_BF16: launch_block_stats<bf16_t>(x, num_tokens, hidden, bp, partial, s); break;
                default: launch_block_stats<f16_t>(x, num_tokens, hidden, bp, partial, s); break;
            }
        } else {
            switch (dtype) {
                case FMOE_F32: launch_stats<float>(x, num_tokens, hidden, p, partial, s); break;
                case FMOE_BF16: launch_stats<bf16_t>(x, num_tokens, hidden, p, partial, s); break;
                default: launch_stats<f16_t>(x, num_tokens, hidden, p, partial, s); break;
            }
        }
        FMOE_CHECK_LAUNCH("fmoe_router_forward(batch statistics)");
    }
    if (!fold) {
        switch (stats_dtype) {
            case FMOE_F32: launch_finalize<float>(partial, p, hidden, training, momentum, eps, running_mean, running_var, num_batches_tracked, mean_rstd, s); break;
            case FMOE_BF16: launch_finalize<bf16_t>(partial, p, hidden, training, momentum, eps, running_mean, running_var, num_batches_tracked, mean_rstd, s); break;
            default: launch_finalize<f16_t>(partial, p, hidden, training, momentum, eps, running_mean, running_var, num_batches_tracked, mean_rstd, s); break;
        }
        FMOE_CHECK_LAUNCH("fmoe_router_forward(finalize)");
    }
    if (tiled_gate) {
        // fold is false here (at least one 256 x 256 tile per compute unit): mean and 1/std are in the workspace
        void* q = ws + p.off_q;
        const int64_t packets = num_tokens * (int64_t)(hidden / 8);
        if (dtype == FMOE_BF16)
            hipLaunchKernelGGL((bn_apply_kernel<bf16_t>), dim3((unsigned)((packets + 255) / 256)), dim3(256), 0, s,
                               (const u32x4_t*)x, (const float*)mean_rstd, (u32x4_t*)q, packets, hidden);
        else
            hipLaunchKernelGGL((bn_apply_kernel<f16_t>), dim3((unsigned)((packets + 255) / 256)), dim3(256), 0, s,
                               (const u32x4_t*)x, (const float*)mean_rstd, (u32x4_t*)q, packets, hidden);
        FMOE_CHECK_LAUNCH("fmoe_router_forward(normalise)");
        if (int rc = gemm_nt_dual(q, gate_w, router_logits, logits32, M, N, hidden, dtype, s)) return rc;
    } else {
        GateStats st;
        st.ready = fold ? 0 : 1;
        st.partial = partial;
        st.row_blocks = bp.row_blocks;
        st.rows_per_block = bp.rows_per_block;
        st.num_tokens = num_tokens;
        st.training = training;
        st.stats_dtype = stats_dtype;
        st.momentum = momentum;
        st.eps = eps;
        st.running_mean = running_mean;
        st.running_var = running_var;
        st.num_batches_tracked = num_batches_tracked;
        st.mean_rstd = mean_rstd;
        if (splitk) {
            switch (dtype) {
                case FMOE_F32: launch_gate_splitk<float>(x, gate_w, st, logits32, router_logits, M, N, hidden, split_query, s); break;
                case FMOE_BF16: launch_gate_splitk<bf16_t>(x, gate_w, st, logits32, router_logits, M, N, hidden, split_query, s); break;
                default: launch_gate_splitk<f16_t>(x, gate_w, st, logits32, router_logits, M, N, hidden, split_query, s); break;
            }
        } else {
            const int tiles_m = (M + 63) / 64, tiles_n = (N + 63) / 64;
            const size_t stats_bytes = (size_t)((hidden + kTileK - 1) / kTileK) * kTileK * 2 * sizeof(float);
            // few tiles with a long k loop: four k groups per workgroup, two for up to two tiles per compute unit; many tiles
            // already fill the chip
            const bool long_k = (split_query ? hidden / 2 : hidden) >= 8 * kTileK;
            const int groups = !long_k || tiles64 > 2 * chip_info().cus ? 1 : (tiles64 > chip_info().cus ? 2 : 4);
#define FMOE_LAUNCH_GATE(TT, KG)                                                                                            \
    hipLaunchKernelGGL((router_gate_kernel<TT, KG>), dim3((unsigned)(tiles_m * tiles_n)), dim3(256 * KG), stats_bytes, s,  \
                       (const TT*)x, (const TT*)gate_w, st, logits32, (TT*)router_logits, M, N, hidden, tiles_m, tiles_n,   \
                       split_query, chip_info().xcds)
            if (dtype == FMOE_BF16) {
                if (groups == 4) FMOE_LAUNCH_GATE(bf16_t, 4);
                else if (groups == 2) FMOE_LAUNCH_GATE(bf16_t, 2);
                else FMOE_LAUNCH_GATE(bf16_t, 1);
            } else {
                if (groups == 4) FMOE_LAUNCH_GATE(f16_t, 4);
                else if (groups == 2) FMOE_LAUNCH_GATE(f16_t, 2);
                else FMOE_LAUNCH_GATE(f16_t, 1);
            }
#undef FMOE_LAUNCH_GATE
        }
    }
    FMOE_CHECK_LAUNCH("fmoe_router_forward(gate)");
    if (top_k == 0) return FMOE_OK;
    return launch_router_from_logits(logits32, num_tokens, num_keys, top_k, scores, indices, gates, dtype, norm_topk_prob,
                                     row_offsets, row_bytes, s);
}

extern "C" size_t fmoe_router_workspace_stats_offset(int64_t num_tokens, int hidden, int num_keys) {
    if (num_tokens <= 0 || hidden <= 0 || num_keys <= 0) return 0;
    return fmoe::plan_prologue(num_tokens, hidden, num_keys).off_mean_rstd;
}

extern "C" size_t fmoe_router_prologue_backward_workspace_bytes(int64_t num_tokens, int hidden, int num_keys, int dtype) {
    if (num_tokens <= 0 || hidden <= 0 || num_keys <= 0 || !fmoe::dtype_ok(dtype)) return 0;
    return fmoe::plan_prologue_backward(num_tokens, hidden, num_keys, dtype).bytes;
}

extern "C" int fmoe_router_prologue_backward(const float* dlogits_fp32, const void* x, const void* gate_w, const float* mean_rstd,
                                             int training, int64_t num_tokens, int hidden, int num_keys, int dtype, void* dx,
                                             void* dgate_w, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace fmoe;
    clear_error();
    if (int rc = check_prologue_backward(num_tokens, hidden, num_keys, dtype)) return rc;
    return router_prologue_backward_impl(dlogits_fp32, x, gate_w, mean_rstd, training, num_tokens, hidden, num_keys, dtype, dx, dgate_w, {},
                                         plan_prologue_backward(num_tokens, hidden, num_keys, dtype), workspace, workspace_bytes, (hipStream_t)stream);
}

fmoe::PrologueOperands fmoe::prologue_operands(const void* x, const float* mean_rstd, int hidden, const PrologueBackwardPlan& p, void* workspace) {
    return {(char*)workspace + p.off_d16, (char*)workspace + p.off_q, p.n_pad, hidden, x, mean_rstd};
}

int fmoe::router_prologue_backward_impl(const float* dlogits_fp32, const void* x, const void* gate_w, const float* mean_rstd,
                                        int training, int64_t num_tokens, int hidden, int num_keys, int dtype, void* dx,
                                        void* dgate_w, const TokenGradients& more, const PrologueBackwardPlan& p, void* workspace, size_t workspace_bytes,
                                        hipStream_t s, bool operands_ready) {
    using namespace fmoe;
    if (int rc = check_prologue_backward(num_tokens, hidden, num_keys, dtype)) return rc;
    FMOE_REQUIRE((dlogits_fp32 || operands_ready) && x && gate_w && mean_rstd && dx && dgate_w, FMOE_ERR_NULL_POINTER,
                 "fmoe_router_prologue_backward: null tensor pointer");
    FMOE_REQUIRE(aligned16(x) && aligned16(dx) && aligned16(dlogits_fp32) && aligned16(mean_rstd), FMOE_ERR_ALIGNMENT,
                 "fmoe_router_prologue_backward: tensor pointers must be 16-byte aligned");
    FMOE_REQUIRE(workspace && workspace_bytes >= p.bytes && aligned16(workspace), FMOE_ERR_WORKSPACE,
                 "fmoe_router_prologue_backward: workspace of %zu bytes needed, %zu given", p.bytes, workspace_bytes);
    switch (dtype) {
        case FMOE_F32: return launch_prologue_backward<float>(dlogits_fp32, x, gate_w, mean_rstd, training, num_tokens, hidden, num_keys, dtype, dx, dgate_w, more, p, workspace, s, operands_ready);
        case FMOE_BF16: return launch_prologue_backward<bf16_t>(dlogits_fp32, x, gate_w, mean_rstd, training, num_tokens, hidden, num_keys, dtype, dx, dgate_w, more, p, workspace, s, operands_ready);
        default: return launch_prologue_backward<f16_t>(dlogits_fp32, x, gate_w, mean_rstd, training, num_tokens, hidden, num_keys, dtype, dx, dgate_w, more, p, workspace, s, operands_ready);
    }
}
