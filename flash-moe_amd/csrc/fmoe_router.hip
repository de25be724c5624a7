// Product-key router for gfx950: per token, the K largest sums a[i] + b[j] over two score vectors
// of nk entries each, without materialising the nk*nk sums.
//
// Exact pruning.  Order each half by (score descending, key index ascending) and call the rank of
// an entry in that order r.  A pair of ranks (ri, rj) is dominated by the (ri+1)*(rj+1)-1 pairs whose
// ranks are component-wise <=, because fp32 addition is monotone in each operand.  So only pairs with
// (ri+1)*(rj+1) <= K can be among the K best: sum_i floor(K/i) candidates (280 for K=64, 645 for
// K=128) instead of nk*nk (16384 / 262144).  The returned scores are therefore exactly the K largest
// sums; where sums tie exactly at the cut the chosen index may differ from an exhaustive scan.
//
// One wavefront handles one token.  All selection is done with 64-bit keys
//   (order-preserving bits of the fp32 score) << 32 | ~index
// so that "larger key" means "larger score, then smaller index".  top-K of a long list is computed in
// groups of KP = max(64, next_pow2(K)) keys: each group is bitonic-sorted across the wave (RK = KP/64
// keys per lane), odd groups in ascending order so that max(best[p], group[p]) is the bitonic sequence
// holding the K best of both, which one bitonic merge re-sorts.
#include <math.h>

#include "fmoe_common.h"
#include "fmoe_select.h"

namespace fmoe {
namespace {

constexpr int kRouterWaves = 4;
constexpr int kMaxTopK = 256;
constexpr int kMaxCand = 2048;   // >= sum_{i=1..256} floor(256/i) = 1546

// Fold groups of KP keys into the running sorted-descending top-KP.  can_stop(g, kth) may end the scan before group
// g >= 1 when no key of groups g, g+1, ... can exceed `kth`, the key now at position `cut` (the last one kept).
template <int RK, typename Gen, typename Stop>
__device__ inline void topk_groups(uint64_t (&best)[RK], int lane, int num_groups, Gen gen, int cut, Stop can_stop) {
    {
        uint64_t cur[RK];
#pragma unroll
        for (int r = 0; r < RK; ++r) cur[r] = gen(0, r);
        bitonic_sort<RK, true>(cur, lane);
#pragma unroll
        for (int r = 0; r < RK; ++r) best[r] = cur[r];
    }
    for (int g = 1; g < num_groups; ++g) {
        if (can_stop(g, key_at<RK>(best, cut))) break;
        uint64_t cur[RK];
#pragma unroll
        for (int r = 0; r < RK; ++r) cur[r] = gen(g, r);
        bitonic_sort<RK, false>(cur, lane);
#pragma unroll
        for (int r = 0; r < RK; ++r) best[r] = best[r] > cur[r] ? best[r] : cur[r];
        bitonic_merge_desc<RK>(best, lane);
    }
}

// T: element type of the input and of `scores`; TG: element type of `gates`.  FROM_LOGITS: the input is the raw gate
// output [num_tokens, 2*nk] (both halves of a token side by side) and the per-half log-softmax is computed here, as
// torch does it: (v - max) - log(sum(exp(v - max))) in fp32; otherwise the input is [2, num_tokens, nk] scores.
template <typename T, typename TG, int RK, bool FROM_LOGITS>
__global__ __launch_bounds__(kRouterWaves* kWave) __attribute__((amdgpu_waves_per_eu(1, RK >= 4 ? 5 : 8))) void router_topk_kernel(
    const T* __restrict__ lp, int64_t num_tokens, int nk, int top_k, int num_cand, T* __restrict__ scores,
    int64_t* __restrict__ indices, TG* __restrict__ gates, int norm_topk_prob, uint32_t* __restrict__ row_offsets,
    uint32_t row_bytes) {
    constexpr int KP = RK * kWave;
    __shared__ uint16_t cand[kMaxCand];
    __shared__ float half_score[kRouterWaves][2][KP];
    __shared__ uint32_t half_index[kRouterWaves][2][KP];

    // candidate table: all (i, j) with (i+1)*(j+1) <= K, packed i | j << 8, listed by i then j.  Row i has
    // K/(i+1) entries; the row starts are a running sum over the row lengths (kept in half_index until the table is
    // built: one division per thread, then additions only).
    {
        uint32_t* row_len = &half_index[0][0][0];
        for (int i = threadIdx.x; i < top_k; i += blockDim.x) row_len[i] = (uint32_t)(top_k / (i + 1));
        __syncthreads();
        for (int i = threadIdx.x; i < top_k; i += blockDim.x) {
            int off = 0;
            for (int q = 0; q < i; ++q) off += (int)row_len[q];
            const int n = (int)row_len[i];
            for (int j = 0; j < n; ++j) cand[off + j] = (uint16_t)(i | (j << 8));
        }
        __syncthreads();
    }

    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t waves_total = (int64_t)gridDim.x * kRouterWaves;
    const int64_t rounds = (num_tokens + waves_total - 1) / waves_total;
    const int half_groups = (nk + KP - 1) / KP;
    const int cand_groups = (num_cand + KP - 1) / KP;

    for (int64_t round = 0; round < rounds; ++round) {
        const int64_t token = round * waves_total + (int64_t)blockIdx.x * kRouterWaves + wave;
        const bool active = token < num_tokens;
        if (active) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const T* row = FROM_LOGITS ? lp + (token * 2 + h) * nk : lp + ((int64_t)h * num_tokens + token) * nk;
                float shift = 0.0f, lse = 0.0f;
                if (FROM_LOGITS) {
                    float mx = -INFINITY;
                    for (int p = lane; p < nk; p += kWave) mx = fmaxf(mx, Elem<T>::to_f32(row[p]));
                    mx = wave_max(mx);
                    float se = 0.0f;
                    for (int p = lane; p < nk; p += kWave) se += expf(Elem<T>::to_f32(row[p]) - mx);
                    shift = mx;
                    lse = logf(wave_sum(se));
                }
                uint64_t best[RK];
                topk_groups<RK>(best, lane, half_groups, [&](int g, int r) -> uint64_t {
                    const int p = g * KP + lane * RK + r;
                    if (p >= nk) return 0ull;
                    const float v = Elem<T>::to_f32(row[p]);
                    return make_key(FROM_LOGITS ? (v - shift) - lse : v, (uint32_t)p);
                }, KP - 1, [](int, uint64_t) { return false; });
#pragma unroll
                for (int r = 0; r < RK; ++r) {
                    half_score[wave][h][lane * RK + r] = key_score(best[r]);
                    half_index[wave][h][lane * RK + r] = key_index(best[r]);
                }
            }
        }
        __syncthreads();
        if (active) {
            uint64_t best[RK];
            topk_groups<RK>(best, lane, cand_groups, [&](int g, int r) -> uint64_t {
                const int c = g * KP + lane * RK + r;
                if (c >= num_cand) return 0ull;
                const int ij = cand[c];
                const int i = ij & 0xff, j = ij >> 8;
                const float s = round_through<T>(half_score[wave][0][i] + half_score[wave][1][j]);
                const uint32_t flat = half_index[wave][0][i] * (uint32_t)nk + half_index[wave][1][j];
                return make_key(s, flat);
            }, top_k - 1, [&](int g, uint64_t kth) {
                // candidates are listed by ascending rank i in half 0, so every sum from group g on is at most
                // half_score[0][i of the group's first entry] + half_score[1][0]; rounding to T is monotone
                const int i_first = cand[g * KP] & 0xff;
                const float bound = round_through<T>(half_score[wave][0][i_first] + half_score[wave][1][0]);
                return bound < key_score(kth);
            });
            float e[RK];
            float total = 0.0f;
#pragma unroll
            for (int r = 0; r < RK; ++r) {
                const int p = lane * RK + r;
                e[r] = p < top_k ? expf(key_score(best[r])) : 0.0f;
                total += e[r];
            }
            if (gates != nullptr && norm_topk_prob) total = wave_sum(total);
#pragma unroll
            for (int r = 0; r < RK; ++r) {
                const int p = lane * RK + r;
                if (p < top_k) {
                    const int64_t o = token * top_k + p;
                    scores[o] = Elem<T>::from_f32(key_score(best[r]));
                    indices[o] = (int64_t)key_index(best[r]);
                    if (row_offsets != nullptr) row_offsets[o] = key_index(best[r]) * row_bytes;
                    if (gates != nullptr) gates[o] = Elem<TG>::from_f32(norm_topk_prob ? e[r] / total : e[r]);
                }
            }
        }
        __syncthreads();
    }
}

// OCC: waves per SIMD the register allocation must leave room for.  With more than four tokens per SIMD eight resident
// waves (at most 64 registers, a few of them spilled for the larger lists) finish sooner than seven, whose eighth token
// per SIMD would wait for a second round; with at most four tokens per SIMD the unconstrained allocation is faster.
template <typename T, typename TG, int RK, int RH, int RC, bool FROM_LOGITS, int OCC, bool SMALL, int TOK, bool REUSE>
__global__ __launch_bounds__(kRouterWaves* kWave, OCC) void router_select_kernel(
    const T* __restrict__ lp, int64_t num_tokens, int nk, int top_k, int num_cand, T* __restrict__ scores,
    int64_t* __restrict__ indices, TG* __restrict__ gates, int norm_topk_prob, uint32_t* __restrict__ row_offsets,
    uint32_t row_bytes, const CandidateTable table) {
    __shared__ SelectLds<RK, RC, kRouterWaves, false, TOK> lds;
    router_select_tokens<T, TG, RK, RH, RC, FROM_LOGITS, SMALL, kRouterWaves, false, TOK, REUSE>(
        lp, num_tokens, nk, top_k, num_cand, scores, indices, gates, norm_topk_prob, row_offsets, row_bytes, table, lds, (int)blockIdx.x,
        (int)gridDim.x);
}

// ------------------------------------------------------------------------------------------------------------
// top_k beyond 256 (up to 1024, with num_keys up to 8192): one workgroup per token, every ordering is a bitonic sort of
// the 64-bit keys in LDS.  Same pruning, same keys and therefore the same result as the kernels above; an order of
// magnitude slower per token, for shapes none of the reference's configurations use.
// ------------------------------------------------------------------------------------------------------------
constexpr int kBigThreads = 1024;
constexpr int kBigMaxKeys = 8192;      // 64 KiB of keys
constexpr int kBigMaxTopK = 1024;      // sum_{i<=1024} floor(1024/i) = 7689 candidates <= kBigMaxKeys

// descending bitonic sort of keys[0..m), m a power of two, by the whole workgroup
__device__ inline void block_sort_desc(uint64_t* keys, int m) {
    for (int k = 2; k <= m; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int i = (int)threadIdx.x; i < m / 2; i += (int)blockDim.x) {
                const int lo = ((i & ~(j - 1)) << 1) | (i & (j - 1)), hi = lo | j;
                const uint64_t a = keys[lo], b = keys[hi];
                if ((a < b) == ((lo & k) == 0)) {
                    keys[lo] = b;
                    keys[hi] = a;
                }
            }
            __syncthreads();
        }
}

template <typename T, typename TG, bool FROM_LOGITS>
__global__ __launch_bounds__(kBigThreads) void router_topk_big_kernel(
    const T* __restrict__ lp, int64_t num_tokens, int nk, int top_k, int num_cand, T* __restrict__ scores,
    int64_t* __restrict__ indices, TG* __restrict__ gates, int norm_topk_prob, uint32_t* __restrict__ row_offsets,
    uint32_t row_bytes) {
    __shared__ uint64_t keys[kBigMaxKeys];
    __shared__ float half_score[2][kBigMaxTopK];
    __shared__ uint32_t half_index[2][kBigMaxTopK];
    __shared__ uint32_t row_start[kBigMaxTopK + 1];    // candidates of rank i in half 0 start here; row i has top_k/(i+1)
    __shared__ float stat[2];
    const int tid = (int)threadIdx.x, lane = lane_id();
    for (int i = tid; i <= top_k; i += kBigThreads) {
        uint32_t off = 0;
        for (int q = 0; q < i; ++q) off += (uint32_t)(top_k / (q + 1));
        row_start[i] = off;
    }
    int m_half = 64, m_cand = 64;
    while (m_half < nk) m_half <<= 1;
    while (m_cand < num_cand) m_cand <<= 1;
    const int kept = top_k < nk ? top_k : nk;           // ranks of a half the candidates can name
    __syncthreads();

    for (int64_t token = blockIdx.x; token < num_tokens; token += gridDim.x) {
        for (int h = 0; h < 2; ++h) {
            const T* row = FROM_LOGITS ? lp + (token * 2 + h) * nk : lp + ((int64_t)h * num_tokens + token) * nk;
            if (FROM_LOGITS) {
                // by one wave, in the order the one-wave-per-token kernels use: identical log-probabilities
                if (tid < kWave) {
                    float mx = -INFINITY;
                    for (int p = lane; p < nk; p += kWave) mx = fmaxf(mx, Elem<T>::to_f32(row[p]));
                    mx = wave_max(mx);
                    float se = 0.0f;
                    for (int p = lane; p < nk; p += kWave) se += expf(Elem<T>::to_f32(row[p]) - mx);
                    const float lse = logf(wave_sum(se));
                    if (lane == 0) {
                        stat[0] = mx;
                        stat[1] = lse;
                    }
                }
                __syncthreads();
            }
            const float shift = FROM_LOGITS ? stat[0] : 0.0f, lse = FROM_LOGITS ? stat[1] : 0.0f;
            for (int p = tid; p < m_half; p += kBigThreads) {
                uint64_t key = 0ull;
                if (p < nk) {
                    const float v = Elem<T>::to_f32(row[p]);
                    key = make_key(FROM_LOGITS ? (v - shift) - lse : v, (uint32_t)p);
                }
                keys[p] = key;
            }
            __syncthreads();
            block_sort_desc(keys, m_half);
            for (int r = tid; r < kept; r += kBigThreads) {
                half_score[h][r] = key_score(keys[r]);
                half_index[h][r] = key_index(keys[r]);
            }
            __syncthreads();
        }
        for (int c = tid; c < m_cand; c += kBigThreads) keys[c] = 0ull;
        __syncthreads();
        for (int i = tid; i < kept; i += kBigThreads) {
            const uint32_t at = row_start[i];
            int n = (int)(row_start[i + 1] - at);
            n = n < kept ? n : kept;                                    // half 1 has only `kept` ranks
            const float si = half_score[0][i];
            const uint32_t base = half_index[0][i] * (uint32_t)nk;
            for (int j = 0; j < n; ++j)
                keys[at + j] = make_key(round_through<T>(si + half_score[1][j]), base + half_index[1][j]);
        }
        __syncthreads();
        block_sort_desc(keys, m_cand);
        if (tid < kWave) {
            float total = 0.0f;
            if (gates != nullptr && norm_topk_prob) {
                for (int p = lane; p < top_k; p += kWave) total += expf(key_score(keys[p]));
                total = wave_sum(total);
            }
            stat[0] = total;
        }
        __syncthreads();
        const float total = stat[0];
        for (int p = tid; p < top_k; p += kBigThreads) {
            const uint64_t key = keys[p];
            const int64_t o = token * top_k + p;
            scores[o] = Elem<T>::from_f32(key_score(key));
            indices[o] = (int64_t)key_index(key);
            if (row_offsets != nullptr) row_offsets[o] = key_index(key) * row_bytes;
            if (gates != nullptr) {
                const float e = expf(key_score(key));
                gates[o] = Elem<TG>::from_f32(norm_topk_prob ? e / total : e);
            }
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------------------------------------------------
// top_k up to 4096 with any num_keys (what the kernel above cannot hold in LDS): one workgroup per token.  Neither a half
// (up to 65535 keys) nor the candidate list (sum_i floor(K/i), 35 000 for K = 4096) is stored: the K-th largest 64-bit key of
// a list is found by radix selection (eight passes over the list, a 256-bin histogram in LDS per pass; the list is
// regenerated from global memory or from the sorted halves each time), the K keys at or above it are collected and
// bitonic-sorted in LDS.  Same pruning, same keys (unique: they carry the index), so the same result as the other
// kernels, ties to the lowest flat index.  A completeness path: milliseconds for thousands of tokens.
// ------------------------------------------------------------------------------------------------------------
constexpr int kRadixMaxTopK = 4096;

// K-th largest of the keys `each(f)` feeds to f (every thread its share; the same keys on every call), by the whole
// workgroup.  hist: 256 counters; pick: two words.
template <typename Each>
__device__ inline uint64_t block_kth_largest(Each each, int want, uint32_t* hist, uint64_t* pick) {
    uint64_t prefix = 0ull;
    int remaining = want;
    for (int d = 7; d >= 0; --d) {
        for (int i = (int)threadIdx.x; i < 256; i += (int)blockDim.x) hist[i] = 0u;
        __syncthreads();
        each([&](uint64_t key) {
            if (d == 7 || (key >> (8 * (d + 1))) == prefix) atomicAdd(&hist[(uint32_t)(key >> (8 * d)) & 255u], 1u);
        });
        __syncthreads();
        if (threadIdx.x == 0) {
            int above = 0, digit = 0;
            for (int bin = 255; bin >= 0; --bin) {
                const int n = (int)hist[bin];
                if (above + n >= remaining) {
                    digit = bin;
                    break;
                }
                above += n;
            }
            pick[0] = prefix << 8 | (uint64_t)digit;
            pick[1] = (uint64_t)(remaining - above);
        }
        __syncthreads();
        prefix = pick[0];
        remaining = (int)pick[1];
    }
    return prefix;
}

template <typename T, typename TG, bool FROM_LOGITS>
__global__ __launch_bounds__(kBigThreads) void router_topk_radix_kernel(
    const T* __restrict__ lp, int64_t num_tokens, int nk, int top_k, T* __restrict__ scores, int64_t* __restrict__ indices,
    TG* __restrict__ gates, int norm_topk_prob, uint32_t* __restrict__ row_offsets, uint32_t row_bytes) {
    __shared__ uint64_t keys[kRadixMaxTopK];
    __shared__ float half_score[2][kRadixMaxTopK];
    __shared__ uint32_t half_index[2][kRadixMaxTopK];
    __shared__ uint32_t hist[256];
    __shared__ uint64_t pick[2];
    __shared__ float stat[2];
    __shared__ int filled;
    const int tid = (int)threadIdx.x, lane = lane_id(), wave = tid >> 6;
    int m = 64;
    while (m < top_k) m <<= 1;
    // keys at or above `tau` into keys[0..top_k), the rest of keys[0..m) zero, sorted descending
    auto collect_and_sort = [&](auto each, uint64_t tau) {
        for (int i = tid; i < m; i += kBigThreads) keys[i] = 0ull;
        if (tid == 0) filled = 0;
        __syncthreads();
        each([&](uint64_t key) {
            if (key >= tau) {
                const int at = atomicAdd(&filled, 1);
                if (at < top_k) keys[at] = key;
            }
        });
        __syncthreads();
        block_sort_desc(keys, m);
    };
    for (int64_t token = blockIdx.x; token < num_tokens; token += gridDim.x) {
        for (int h = 0; h < 2; ++h) {
            const T* row = FROM_LOGITS ? lp + (token * 2 + h) * nk : lp + ((int64_t)h * num_tokens + token) * nk;
            if (FROM_LOGITS) {
                // by one wave, in the order the one-wave-per-token kernels use: identical log-probabilities
                if (tid < kWave) {
                    float mx = -INFINITY;
                    for (int p = lane; p < nk; p += kWave) mx = fmaxf(mx, Elem<T>::to_f32(row[p]));
                    mx = wave_max(mx);
                    float se = 0.0f;
                    for (int p = lane; p < nk; p += kWave) se += expf(Elem<T>::to_f32(row[p]) - mx);
                    const float lse = logf(wave_sum(se));
                    if (lane == 0) {
                        stat[0] = mx;
                        stat[1] = lse;
                    }
                }
                __syncthreads();
            }
            const float shift = FROM_LOGITS ? stat[0] : 0.0f, lse = FROM_LOGITS ? stat[1] : 0.0f;
            auto each_key = [&](auto f) {
                for (int p = tid; p < nk; p += kBigThreads) {
                    const float v = Elem<T>::to_f32(row[p]);
                    f(make_key(FROM_LOGITS ? (v - shift) - lse : v, (uint32_t)p));
                }
            };
            const uint64_t tau = block_kth_largest(each_key, top_k, hist, pick);
            collect_and_sort(each_key, tau);
            for (int r = tid; r < top_k; r += kBigThreads) {
                half_score[h][r] = key_score(keys[r]);
                half_index[h][r] = key_index(keys[r]);
            }
            __syncthreads();
        }
        // candidates: rank i of half 0 with ranks 0 .. top_k/(i+1)-1 of half 1; a wave per row, lanes along the row
        auto each_candidate = [&](auto f) {
            for (int i = wave; i < top_k; i += kBigThreads / kWave) {
                const int n = top_k / (i + 1);
                const float si = half_score[0][i];
                const uint32_t base = half_index[0][i] * (uint32_t)nk;
                for (int j = lane; j < n; j += kWave) f(make_key(round_through<T>(si + half_score[1][j]), base + half_index[1][j]));
            }
        };
        const uint64_t tau = block_kth_largest(each_candidate, top_k, hist, pick);
        collect_and_sort(each_candidate, tau);
        if (tid < kWave) {
            float total = 0.0f;
            if (gates != nullptr && norm_topk_prob) {
                for (int p = lane; p < top_k; p += kWave) total += expf(key_score(keys[p]));
                total = wave_sum(total);
            }
            stat[0] = total;
        }
        __syncthreads();
        const float total = stat[0];
        for (int p = tid; p < top_k; p += kBigThreads) {
            const uint64_t key = keys[p];
            const int64_t o = token * top_k + p;
            scores[o] = Elem<T>::from_f32(key_score(key));
            indices[o] = (int64_t)key_index(key);
            if (row_offsets != nullptr) row_offsets[o] = key_index(key) * row_bytes;
            if (gates != nullptr) {
                const float e = expf(key_score(key));
                gates[o] = Elem<TG>::from_f32(norm_topk_prob ? e / total : e);
            }
        }
        __syncthreads();
    }
}

int count_candidates(int top_k) {
    int n = 0;
    for (int i = 1; i <= top_k; ++i) n += top_k / i;
    return n;
}

template <typename T, typename TG, bool FROM_LOGITS>
int launch_router(const void* lp, int64_t T_, int nk, int K, void* scores, int64_t* indices, void* gates,
                  int norm, uint32_t* row_offsets, uint32_t row_bytes, hipStream_t stream) {
    const int num_cand = count_candidates(K);
    auto blocks_of = [&](int tokens_of_a_wave) {
        const int64_t needed = (T_ + kRouterWaves * tokens_of_a_wave - 1) / (kRouterWaves * tokens_of_a_wave);
        const int64_t most = (int64_t)chip_info().cus * 8;     // a few resident blocks per CU; the kernel loops over tokens
        return needed < most ? needed : most;
    };
    const dim3 grid((unsigned)blocks_of(1));
    const dim3 block(kRouterWaves * kWave);
    if (K > kMaxTopK) {      // the workgroup-per-token kernels; their limits are checked by the callers
        const int64_t big_blocks = T_ < (int64_t)chip_info().cus * 2 ? T_ : (int64_t)chip_info().cus * 2;
        if (K > kBigMaxTopK || nk > kBigMaxKeys) {
            const int64_t radix_blocks = T_ < (int64_t)chip_info().cus ? T_ : (int64_t)chip_info().cus;
            hipLaunchKernelGGL((router_topk_radix_kernel<T, TG, FROM_LOGITS>), dim3((unsigned)radix_blocks), dim3(kBigThreads), 0,
                               stream, (const T*)lp, T_, nk, K, (T*)scores, indices, (TG*)gates, norm, row_offsets, row_bytes);
            FMOE_CHECK_LAUNCH("fmoe_router_topk");
            return FMOE_OK;
        }
        hipLaunchKernelGGL((router_topk_big_kernel<T, TG, FROM_LOGITS>), dim3((unsigned)big_blocks), dim3(kBigThreads), 0, stream,
                           (const T*)lp, T_, nk, K, num_cand, (T*)scores, indices, (TG*)gates, norm, row_offsets, row_bytes);
        FMOE_CHECK_LAUNCH("fmoe_router_topk");
        return FMOE_OK;
    }
    // lists that fit the registers of a wave take the threshold selection
    const bool crowded = T_ > (int64_t)chip_info().cus * 4 * kRouterWaves;      // more than four tokens per SIMD
    const bool in_pairs = T_ >= (int64_t)chip_info().cus * 16 * kRouterWaves;     // sixteen or more
#define FMOE_LAUNCH_SELECT_OCC(RK_, RH_, RC_, OCC_, SMALL_, TOK_, REUSE_)                                                     \
    hipLaunchKernelGGL((router_select_kernel<T, TG, RK_, RH_, RC_, FROM_LOGITS, OCC_, SMALL_, TOK_, REUSE_>),                 \
                       dim3((unsigned)blocks_of(TOK_)), block, 0, stream, (const T*)lp, T_, nk, K, num_cand, (T*)scores, indices, (TG*)gates, norm, row_offsets, row_bytes, table)
// Many tokens: one key per lane lets the kernel run in the registers of eight waves per SIMD at no or little spilling (K = 16, nk =
// 128, 32768 tokens: 36 us against 40 at five waves when it was chosen); the instances of two keys per lane would spill 25 to 59
// registers (nk = 512, K = 128: 165 us against 138 without the bound).  Few tokens are one latency chain, spills would lengthen it.
// Two tokens to a wave save a third of the sorting once every wave has two (us, 128 keys, 16 experts, without REUSE: 32768 tokens 29.4
// -> 28.0, 16384 16.2 -> 15.6, but 12288 11.9 -> 12.9 and 8192 9.6 -> 10.5).
// Lists start from the score that served the wave's previous list (REUSE) where a wave has several and at least four slots beyond
// K are left, eight of 64, so that it often serves again (us with the sorts on integers, 32768 tokens, without | with, 128 keys: K = 16
// 28.0 | 22.4, 24 27.5 | 25.5, 28 29.7 | 28.8, 32 35.6 | 36.6, 40 39.1 | 36.7, 50 41.8 | 40.2, 58 44.2 | 44.4, 64 52.2 | 53.9; 512 keys:
// K = 16 44.1 | 35.1, 24 50.4 | 44.7, 30 56.9 | 56.9, 40 59.7 | 51.0; 10000 tokens, K = 16: 10.5 | 9.75, 6000 8.0 | 7.9).  Two keys per
// lane gain 0 to 4 % and are left as they are.
#define FMOE_LAUNCH_SELECT(RK_, RH_, RC_)                                                          \
    do {                                                                                           \
        if (crowded && RK_ == 1 && K <= 56) FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 8, false, 1, true); \
        else if (crowded && RK_ == 1) FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 8, false, 1, false);     \
        else FMOE_LAUNCH_SELECT_OCC(RK_, RH_, RC_, 1, false, 1, false);                            \
    } while (0)
#define FMOE_LAUNCH_SELECT_SMALL(RH_, RC_)                                                         \
    do {                                                                                           \
        constexpr bool all_reuse = RC_ == 1;              /* at most 19 experts */                 \
        if (in_pairs && (all_reuse || K <= 28)) FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 8, true, 2, true);      \
        else if (in_pairs) FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 8, true, 2, all_reuse);             \
        else if (crowded && (all_reuse || K <= 28)) FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 8, true, 1, true);  \
        else if (crowded) FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 8, true, 1, all_reuse);              \
        else FMOE_LAUNCH_SELECT_OCC(1, RH_, RC_, 1, true, 1, false);                               \
    } while (0)
    if (K <= 128 && nk <= 512) {
        CandidateTable table;
        candidate_table(K, table);
        if (K <= 32 && num_cand <= kWave) {          // up to 19 experts: the candidates are one key per lane
            if (nk <= 128) FMOE_LAUNCH_SELECT_SMALL(2, 1);
            else FMOE_LAUNCH_SELECT_SMALL(8, 1);
        } else if (K <= 32) {
            if (nk <= 128) FMOE_LAUNCH_SELECT_SMALL(2, 2);
            else FMOE_LAUNCH_SELECT_SMALL(8, 2);
        } else if (K <= 64) {
            if (nk <= 128) FMOE_LAUNCH_SELECT(1, 2, 5);
            else if (nk <= 256) FMOE_LAUNCH_SELECT(1, 4, 5);
            else FMOE_LAUNCH_SELECT(1, 8, 5);
        } else {
            if (nk <= 128) FMOE_LAUNCH_SELECT(2, 2, 11);
            else FMOE_LAUNCH_SELECT(2, 8, 11);
        }
        FMOE_CHECK_LAUNCH("fmoe_router_topk");
        return FMOE_OK;
    }
#undef FMOE_LAUNCH_SELECT_OCC
#undef FMOE_LAUNCH_SELECT
#undef FMOE_LAUNCH_SELECT_SMALL
#define FMOE_LAUNCH_ROUTER(R)                                                                                      \
    hipLaunchKernelGGL((router_topk_kernel<T, TG, R, FROM_LOGITS>), grid, block, 0, stream, (const T*)lp, T_, nk, K, \
                       num_cand, (T*)scores, indices, (TG*)gates, norm, row_offsets, row_bytes)
    if (K <= 64) FMOE_LAUNCH_ROUTER(1);
    else if (K <= 128) FMOE_LAUNCH_ROUTER(2);
    else FMOE_LAUNCH_ROUTER(4);
#undef FMOE_LAUNCH_ROUTER
    FMOE_CHECK_LAUNCH("fmoe_router_topk");
    return FMOE_OK;
}

}  // namespace

bool router_topk_supported(int num_keys, int top_k) {
    return top_k <= kRadixMaxTopK;       // <= 256: a wave per token; beyond: a workgroup per token
}

int launch_router_from_logits(const float* logits, int64_t num_tokens, int num_keys, int top_k, float* scores,
                              int64_t* indices, void* gates, int gate_dtype, int norm_topk_prob, uint32_t* row_offsets,
                              uint32_t row_bytes, hipStream_t stream) {
    switch (gate_dtype) {
        case FMOE_F32: return launch_router<float, float, true>(logits, num_tokens, num_keys, top_k, scores, indices, gates, norm_topk_prob, row_offsets, row_bytes, stream);
        case FMOE_BF16: return launch_router<float, bf16_t, true>(logits, num_tokens, num_keys, top_k, scores, indices, gates, norm_topk_prob, row_offsets, row_bytes, stream);
        default: return launch_router<float, f16_t, true>(logits, num_tokens, num_keys, top_k, scores, indices, gates, norm_topk_prob, row_offsets, row_bytes, stream);
    }
}

}  // namespace fmoe

extern "C" int fmoe_router_topk(const void* log_probs, int64_t num_tokens, int num_keys, int top_k, int dtype,
                                void* scores, int64_t* indices, void* gates, int norm_topk_prob, void* stream) {
    using namespace fmoe;
    clear_error();
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "fmoe_router_topk: unknown dtype %d", dtype);
    FMOE_REQUIRE(num_tokens >= 0 && num_keys > 0, FMOE_ERR_BAD_SHAPE, "fmoe_router_topk: bad shape T=%lld nk=%d",
                 (long long)num_tokens, num_keys);
    FMOE_REQUIRE(top_k >= 0 && top_k <= num_keys, FMOE_ERR_TOPK_RANGE,
                 "num_experts_per_tok should be in [0, %d], but got %d", num_keys, top_k);
    FMOE_REQUIRE(num_keys <= 65535, FMOE_ERR_UNSUPPORTED, "fmoe_router_topk: num_keys=%d > 65535", num_keys);
    FMOE_REQUIRE(router_topk_supported(num_keys, top_k), FMOE_ERR_UNSUPPORTED,
                 "fmoe_router_topk: top_k=%d > %d (num_keys=%d)", top_k, kRadixMaxTopK, num_keys);
    if (num_tokens == 0 || top_k == 0) return FMOE_OK;
    FMOE_REQUIRE(log_probs && scores && indices, FMOE_ERR_NULL_POINTER, "fmoe_router_topk: null tensor pointer");
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case FMOE_F32: return launch_router<float, float, false>(log_probs, num_tokens, num_keys, top_k, scores, indices, gates, norm_topk_prob, nullptr, 0u, s);
        case FMOE_BF16: return launch_router<bf16_t, bf16_t, false>(log_probs, num_tokens, num_keys, top_k, scores, indices, gates, norm_topk_prob, nullptr, 0u, s);
        default: return launch_router<f16_t, f16_t, false>(log_probs, num_tokens, num_keys, top_k, scores, indices, gates, norm_topk_prob, nullptr, 0u, s);
    }
}
