// Backward passes of the router op, the SwiGLU gate and the routed-expert op for gfx950.
//
//   router  : drouter_logits[0,t,i] = sum_{k : idx[t,k] / nk == i} dscores[t,k],  [1,t,j] likewise with idx % nk
//   route   : gates = exp(top-k sums of the per-half log-softmax), renormalised or not -> gradient of the gate logits
//   swiglu  : c = silu(a) * b  ->  da = dc * (silu(a) * (1 - sigmoid(a)) + sigmoid(a)) * b,  db = dc * silu(a)
//   experts : out[t] = sum_k silu(s) * g * up[e],  s = <x[t], down[e]>,  e = idx[t,k]:
//               da_p   = <dout[t], up[e]>                 dg_p = da_p * silu(s)
//               ds_p   = da_p * g * sigmoid(s) * (1 + s * (1 - sigmoid(s)))
//               dx[t]  = sum_k ds_p * down[e]
//               ddown[e] = sum_{p -> e} ds_p * x[t_p]     dup[e] = sum_{p -> e} silu(s_p) * g_p * dout[t_p]
//
// No floating-point atomics on global memory: every output element is written once and sums run in a fixed order
// (pairs of an expert in ascending pair index), so gradients are reproducible bit for bit.  The per-token part of the
// expert backward is one wave per token with the token's rows of x and dout in registers (the layout of the forward
// row kernel).  The per-expert part needs the pairs grouped by expert: group_pairs (fmoe_bucket.hip) gives each expert one segment
// listing its pairs in ascending pair index, and the wave that owns the expert walks it in that order.
#include <type_traits>

#include "fmoe_common.h"
#include "fmoe_vec.h"

namespace fmoe {
namespace {

constexpr int kBwdWaves = 4;

// ------------------------------------------------------------------------------------------------------------
// router
// ------------------------------------------------------------------------------------------------------------
// A wave takes `n` successive tokens, so that their pairs fill its lanes (four tokens of 16 pairs) and their gradient rows, which
// follow each other in each half, leave in 16-byte stores (WIDE: whole packets, aligned).  Bound by those rows (a fill of as much
// takes 7.0 us) and, with few keys per pair, by the adds in LDS (about three clocks each): 32768 tokens in fp32, us, against a wave
// per token with 4-byte stores and 64-bit divisions: 128 keys and 16 pairs 12.9 -> 12.1, 64 and 8 8.6 -> 7.9, 40 and 4 8.1 -> 5.4.
template <typename T, bool WIDE>
__global__ __launch_bounds__(kBwdWaves* kWave) void router_backward_kernel(const T* __restrict__ dscores,
                                                                           const int64_t* __restrict__ indices,
                                                                           T* __restrict__ dlogits, int64_t num_tokens,
                                                                           int nk, int top_k, int waves_per_block, int chunk, int n) {
    extern __shared__ __align__(16) float acc_all[];   // [waves_per_block][2][n][chunk], private to each wave
    constexpr int V = WIDE ? Elem<T>::kVec : 1;
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t token = ((int64_t)blockIdx.x * waves_per_block + wave) * n;
    if (wave >= waves_per_block || token >= num_tokens) return;   // whole waves leave; nobody waits on them
    const int mine = num_tokens - token < n ? (int)(num_tokens - token) : n;
    float* acc = acc_all + (size_t)wave * 2 * n * chunk;
    const int64_t num_pairs = (int64_t)nk * nk;                   // below 2^32
    // The gradient rows are built `chunk` keys at a time (chunk = nk when a row pair fits the LDS, else n = 1): per chunk the
    // pairs are scanned again and only the keys inside it are added.
    for (int c0 = 0; c0 < nk; c0 += chunk) {
        const int cn = nk - c0 < chunk ? nk - c0 : chunk;
        for (int p = lane * V; p < 2 * n * chunk; p += kWave * V)
#pragma unroll
            for (int e = 0; e < V; ++e) acc[p + e] = 0.0f;
        __builtin_amdgcn_wave_barrier();
        // LDS adds of one instruction that hit the same address are applied one after the other by the LDS unit, and the
        // instructions of a wave execute in order, so the sum has a fixed order for given inputs
        for (int q = lane; q < mine * top_k; q += kWave) {
            const int64_t id = indices[token * top_k + q];
            if (id >= 0 && id < num_pairs) {
                const float d = Elem<T>::to_f32(dscores[token * top_k + q]);
                float* row = acc + (uint32_t)q / (uint32_t)top_k * chunk;
                const uint32_t first = (uint32_t)id / (uint32_t)nk;
                const int i = (int)first - c0, j = (int)((uint32_t)id - first * (uint32_t)nk) - c0;
                if (i >= 0 && i < cn) __hip_atomic_fetch_add(&row[i], d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                if (j >= 0 && j < cn) __hip_atomic_fetch_add(&row[n * chunk + j], d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float* from = acc + h * n * chunk;
            T* to = dlogits + (h * num_tokens + token) * nk + c0;
            for (int p = lane * V; p < mine * cn; p += kWave * V) {
                if constexpr (WIDE) {
                    float v[V];
#pragma unroll
                    for (int e = 0; e < V; ++e) v[e] = from[p + e];
                    *reinterpret_cast<u32x4_t*>(to + p) = pack16<T>(v);
                } else {
                    to[p] = Elem<T>::from_f32(from[p]);
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// Keys of a half whose gradient row is held in LDS at a time: the whole half up to 8192 keys (64 KiB for the pair of
// rows), 4096 beyond.
inline int backward_key_chunk(int nk) { return nk <= 8192 ? nk : 4096; }

template <typename T>
int launch_router_backward(const void* dscores, const int64_t* indices, void* dlogits, int64_t T_, int nk, int K,
                           hipStream_t stream) {
    const int chunk = backward_key_chunk(nk);
    // tokens per wave: what fills the lanes, as long as four waves are left for every SIMD and four waves' rows take 32 KiB
    int64_t n = T_ / (chip_info().cus * 16);
    const int lanes = kWave / (K < 1 ? 1 : K), rows = 1024 / nk, most = rows < lanes ? rows : lanes;
    n = n > most ? most : n;
    n = n < 1 ? 1 : n;
    const size_t per_wave = (size_t)2 * n * chunk * sizeof(float);
    int waves = (int)((48 * 1024) / per_wave);
    waves = waves < 1 ? 1 : (waves > kBwdWaves ? kBwdWaves : waves);
    const unsigned grid = (unsigned)((T_ + waves * n - 1) / (waves * n));
    const bool wide = nk % Elem<T>::kVec == 0 && (uintptr_t)dlogits % 16 == 0;
#define FMOE_LAUNCH_ROUTE(WIDE_)                                                                                                    \
    hipLaunchKernelGGL((router_backward_kernel<T, WIDE_>), dim3(grid), dim3(kBwdWaves * kWave), waves * per_wave, stream,           \
                       (const T*)dscores, indices, (T*)dlogits, T_, nk, K, waves, chunk, (int)n)
    if (wide) FMOE_LAUNCH_ROUTE(true);
    else FMOE_LAUNCH_ROUTE(false);
#undef FMOE_LAUNCH_ROUTE
    FMOE_CHECK_LAUNCH("fmoe_router_topk_backward");
    return FMOE_OK;
}

// Routing stage between the gate logits and the gates, backward in one launch: exp / renormalisation, the scatter of the
// score gradients onto the two key rows, and the per-half log-softmax.  One wave per token; the log-probabilities are
// recomputed from the fp32 logits exactly as the forward computes them ((v - max) - log(sum exp(v - max))).
//   s_k = lp0[i_k] + lp1[j_k],  e_k = exp(s_k),  g_k = e_k  or  e_k / sum_m e_m
//   ds_k = dg_k * e_k                       (no renormalisation)
//   ds_k = g_k * (dg_k - sum_m dg_m g_m)    (renormalised)
//   dlp[h][i] = sum of ds_k over the pairs that use key i of half h
//   dlogits[h][i] = dlp[h][i] - softmax(logits[h])[i] * sum_i dlp[h][i]   (+ the gradient of the returned logits)
template <typename T>
__global__ __launch_bounds__(kBwdWaves* kWave) void route_backward_kernel(
    const T* __restrict__ dgates, const int64_t* __restrict__ indices, const float* __restrict__ logits,
    const T* __restrict__ dlogits_extra, int64_t extra_token, int64_t extra_half, float* __restrict__ dlogits,
    int64_t num_tokens, int nk, int top_k, int norm_topk_prob, int waves_per_block, int chunk) {
    extern __shared__ float acc_all[];   // [waves_per_block][2 * chunk], one private row pair per wave
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t token = (int64_t)blockIdx.x * waves_per_block + wave;
    if (wave >= waves_per_block || token >= num_tokens) return;   // whole waves leave; nobody waits on them
    float* acc = acc_all + (size_t)wave * 2 * chunk;
    const float* row = logits + token * 2 * nk;
    float shift[2], lse[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float mx = -INFINITY;
        for (int p = lane; p < nk; p += kWave) mx = fmaxf(mx, row[h * nk + p]);
        mx = wave_max(mx);
        float se = 0.0f;
        for (int p = lane; p < nk; p += kWave) se += expf(row[h * nk + p] - mx);
        shift[h] = mx;
        lse[h] = logf(wave_sum(se));
    }
    const int64_t num_pairs = (int64_t)nk * nk;
    // first pass (renormalised gates only): sum_m e_m and sum_m dg_m e_m
    float total = 1.0f, dot = 0.0f;
    if (norm_topk_prob) {
        float te = 0.0f, td = 0.0f;
        for (int k = lane; k < top_k; k += kWave) {
            const int64_t id = indices[token * top_k + k];
            if (id >= 0 && id < num_pairs) {
                const int i = (int)((uint32_t)id / (uint32_t)nk), j = (int)((uint32_t)id % (uint32_t)nk);      // at most 32767 keys
                const float e = expf(((row[i] - shift[0]) - lse[0]) + ((row[nk + j] - shift[1]) - lse[1]));
                te += e;
                td = __builtin_fmaf(Elem<T>::to_f32(dgates[token * top_k + k]), e, td);
            }
        }
        total = wave_sum(te);
        dot = wave_sum(td) / total;          // sum_m dg_m g_m
    }
    // The two gradient rows are built `chunk` keys at a time (chunk = nk when a row pair fits the LDS): per chunk the
    // pairs are scanned again and only the keys inside it are added.  With several chunks the row totals, which every
    // key's result needs, are the sum of the pair gradients themselves (each valid pair adds to one key of either half).
    const bool chunked = chunk < nk;
    float sum_all = 0.0f;
    if (chunked) {
        float part = 0.0f;
        for (int k = lane; k < top_k; k += kWave) {
            const int64_t id = indices[token * top_k + k];
            if (id >= 0 && id < num_pairs) {
                const int i = (int)((uint32_t)id / (uint32_t)nk), j = (int)((uint32_t)id % (uint32_t)nk);      // at most 32767 keys
                const float e = expf(((row[i] - shift[0]) - lse[0]) + ((row[nk + j] - shift[1]) - lse[1]));
                const float dg = Elem<T>::to_f32(dgates[token * top_k + k]);
                part += norm_topk_prob ? (e / total) * (dg - dot) : dg * e;
            }
        }
        sum_all = wave_sum(part);
    }
    for (int c0 = 0; c0 < nk; c0 += chunk) {
        const int cn = nk - c0 < chunk ? nk - c0 : chunk;
        for (int p = lane; p < 2 * chunk; p += kWave) acc[p] = 0.0f;
        __builtin_amdgcn_wave_barrier();
        // LDS adds of one instruction that hit the same address are applied one after the other by the LDS unit, and the
        // instructions of a wave execute in order, so the sum has a fixed order for given inputs
        for (int k = lane; k < top_k; k += kWave) {
            const int64_t id = indices[token * top_k + k];
            if (id >= 0 && id < num_pairs) {
                const int i = (int)((uint32_t)id / (uint32_t)nk), j = (int)((uint32_t)id % (uint32_t)nk);      // at most 32767 keys
                const float e = expf(((row[i] - shift[0]) - lse[0]) + ((row[nk + j] - shift[1]) - lse[1]));
                const float dg = Elem<T>::to_f32(dgates[token * top_k + k]);
                const float ds = norm_topk_prob ? (e / total) * (dg - dot) : dg * e;
                if (i >= c0 && i < c0 + cn) __hip_atomic_fetch_add(&acc[i - c0], ds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                if (j >= c0 && j < c0 + cn) __hip_atomic_fetch_add(&acc[chunk + j - c0], ds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            }
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float sum = sum_all;
            if (!chunked) {
                sum = 0.0f;
                for (int p = lane; p < nk; p += kWave) sum += acc[h * chunk + p];
                sum = wave_sum(sum);
            }
            for (int p = lane; p < cn; p += kWave) {
                const int64_t at = token * 2 * nk + h * nk + c0 + p;
                float d = acc[h * chunk + p] - expf((row[h * nk + c0 + p] - shift[h]) - lse[h]) * sum;
                if (dlogits_extra != nullptr) d += Elem<T>::to_f32(dlogits_extra[token * extra_token + h * extra_half + c0 + p]);
                dlogits[at] = d;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// The same for at most 64 R keys and 64 P pairs, held in registers: everything a wave reads but the pairs' logits is asked for at once, each
// pair is worked out once.  Bound by the latency of a wave's chain, which was four reductions on loads of their own and a 64-bit
// division for every pair and pass: 4096 tokens of 128 keys and 64 pairs 15.4 -> 10.6 us, 615 tokens
// of 64 keys and 17 pairs 6.3 -> 4.4.  The sums are those of the other kernel in its order.
// PREPARE: inside the block nobody reads the gradients in fp32: they leave as the prologue's products take them, and with them the token's
// row of q, whose loads hide in the chain: 4096 tokens, 1024 columns 16.3 us in two launches, 13.6 so; 615 tokens, 776 columns 6.9 -> 5.0.
template <typename T, int R, int P, bool PREPARE>
__global__ __launch_bounds__(kBwdWaves* kWave) void route_backward_small_kernel(
    const T* __restrict__ dgates, const int64_t* __restrict__ indices, const float* __restrict__ logits,
    const T* __restrict__ dlogits_extra, int64_t extra_token, int64_t extra_half, float* __restrict__ dlogits,
    int64_t num_tokens, int nk, int top_k, int norm_topk_prob, int waves_per_block, const PrologueOperands to) {
    extern __shared__ float acc_all[];   // [waves_per_block][2 * nk], one private row pair per wave
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t token = (int64_t)blockIdx.x * waves_per_block + wave;
    if (wave >= waves_per_block || token >= num_tokens) return;   // whole waves leave; nobody waits on them
    float* acc = acc_all + (size_t)wave * 2 * nk;
    const float* row = logits + token * 2 * nk;
    int64_t id[P];
    float dg[P], v[2][R], extra[2][R];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const int k = u * kWave + lane;
        id[u] = k < top_k ? indices[token * top_k + k] : -1;
        dg[u] = k < top_k ? Elem<T>::to_f32(dgates[token * top_k + k]) : 0.0f;
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int p = r * kWave + lane;
            v[h][r] = p < nk ? row[h * nk + p] : -INFINITY;
            extra[h][r] = dlogits_extra != nullptr && p < nk ? Elem<T>::to_f32(dlogits_extra[token * extra_token + h * extra_half + p]) : 0.0f;
        }
    int first[P], second[P];
    float a[P], b[P];
#pragma unroll
    for (int u = 0; u < P; ++u) {
        const bool valid = id[u] >= 0 && id[u] < (int64_t)nk * nk;
        const uint32_t at = valid ? (uint32_t)id[u] : 0u;
        first[u] = valid ? (int)(at / (uint32_t)nk) : -1;
        second[u] = (int)(at % (uint32_t)nk);
        a[u] = row[valid ? first[u] : 0];
        b[u] = row[nk + second[u]];
    }
    for (int p = lane; p < 2 * nk; p += kWave) acc[p] = 0.0f;
    float shift[2], lse[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float mx = v[h][0];
#pragma unroll
        for (int r = 1; r < R; ++r) mx = fmaxf(mx, v[h][r]);
        shift[h] = wave_max(mx);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        float se = 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) se += r * kWave + lane < nk ? expf(v[h][r] - shift[h]) : 0.0f;
        lse[h] = logf(wave_sum(se));
    }
    float e[P], total = 1.0f, dot = 0.0f;
#pragma unroll
    for (int u = 0; u < P; ++u) e[u] = expf(((a[u] - shift[0]) - lse[0]) + ((b[u] - shift[1]) - lse[1]));
    if (norm_topk_prob) {
        float te = 0.0f, td = 0.0f;
#pragma unroll
        for (int u = 0; u < P; ++u)
            if (first[u] >= 0) {
                te += e[u];
                td = __builtin_fmaf(dg[u], e[u], td);
            }
        total = wave_sum(te);
        dot = wave_sum(td) / total;          // sum_m dg_m g_m
    }
    __builtin_amdgcn_wave_barrier();
    // adds to one address: in a fixed order, as in the other kernel
#pragma unroll
    for (int u = 0; u < P; ++u)
        if (first[u] >= 0) {
            const float ds = norm_topk_prob ? (e[u] / total) * (dg[u] - dot) : dg[u] * e[u];
            __hip_atomic_fetch_add(&acc[first[u]], ds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            __hip_atomic_fetch_add(&acc[nk + second[u]], ds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
    __builtin_amdgcn_wave_barrier();
    float got[2][R], sum[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        sum[h] = 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int p = r * kWave + lane;
            got[h][r] = p < nk ? acc[h * nk + p] : 0.0f;
            sum[h] += got[h][r];
        }
        sum[h] = wave_sum(sum[h]);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int p = r * kWave + lane;
            if (p >= nk) continue;
            float d = got[h][r] - expf((v[h][r] - shift[h]) - lse[h]) * sum[h];
            if (dlogits_extra != nullptr) d += extra[h][r];
            if constexpr (PREPARE) reinterpret_cast<T*>(to.d)[token * to.n_pad + h * nk + p] = Elem<T>::from_f32(d);
            else dlogits[token * 2 * nk + h * nk + p] = d;
        }
    if constexpr (PREPARE) {
        constexpr int V = Elem<T>::kVec;
        if (2 * nk + lane < to.n_pad) reinterpret_cast<T*>(to.d)[token * to.n_pad + 2 * nk + lane] = Elem<T>::from_f32(0.0f);
        for (int c = lane; c < to.hidden / V; c += kWave) {
            float xv[V], qv[V];
            unpack16<T>(reinterpret_cast<const u32x4_t*>((const T*)to.x + token * to.hidden)[c], xv);
#pragma unroll
            for (int v = 0; v < V; v += 4) {
                const f32x4_t m = *reinterpret_cast<const f32x4_t*>(to.mean_rstd + c * V + v);
                const f32x4_t rs = *reinterpret_cast<const f32x4_t*>(to.mean_rstd + to.hidden + c * V + v);
#pragma unroll
                for (int j = 0; j < 4; ++j) qv[v + j] = (xv[v + j] - m[j]) * rs[j];
            }
            reinterpret_cast<u32x4_t*>((T*)to.q + token * to.hidden)[c] = pack16<T>(qv);
        }
    }
}

template <typename T>
int launch_route_backward(const void* dgates, const int64_t* indices, const float* logits, const void* dlogits_extra,
                          int64_t extra_token, int64_t extra_half, float* dlogits, int64_t T_, int nk, int K, int norm, hipStream_t stream,
                          const PrologueOperands* operands) {
    const int chunk = backward_key_chunk(nk);
    const size_t per_wave = (size_t)2 * chunk * sizeof(float);
    int waves = (int)((48 * 1024) / per_wave);
    waves = waves < 1 ? 1 : (waves > kBwdWaves ? kBwdWaves : waves);
    const unsigned grid = (unsigned)((T_ + waves - 1) / waves);
    const PrologueOperands to = operands != nullptr ? *operands : PrologueOperands{};
#define FMOE_LAUNCH_SMALL(R, P, PREPARE)                                                                                                    \
    hipLaunchKernelGGL((route_backward_small_kernel<T, R, P, PREPARE>), dim3(grid), dim3(kBwdWaves * kWave), waves * per_wave, stream,      \
                       (const T*)dgates, indices, logits, (const T*)dlogits_extra, extra_token, extra_half, dlogits, T_, nk, K, norm, waves, to)
    // what a lane's registers hold; up to 256 keys a row pair also lies in LDS whole, for four waves
    if (nk <= 2 * kWave && K <= kWave) {
        if (operands != nullptr) FMOE_LAUNCH_SMALL(2, 1, true);
        else FMOE_LAUNCH_SMALL(2, 1, false);
    } else if (route_backward_prepares(nk, K)) {
        if (operands != nullptr) FMOE_LAUNCH_SMALL(4, 2, true);
        else FMOE_LAUNCH_SMALL(4, 2, false);
    } else
        hipLaunchKernelGGL((route_backward_kernel<T>), dim3(grid), dim3(kBwdWaves * kWave), waves * per_wave, stream,
                           (const T*)dgates, indices, logits, (const T*)dlogits_extra, extra_token, extra_half, dlogits, T_, nk, K, norm, waves,
                           chunk);
#undef FMOE_LAUNCH_SMALL
    FMOE_CHECK_LAUNCH("fmoe_route_backward");
    return FMOE_OK;
}

// ------------------------------------------------------------------------------------------------------------
// SwiGLU
// ------------------------------------------------------------------------------------------------------------
// One 16-byte packet per thread; workgroup b works on row b / col_blocks.  Row strides (elements) let da / db / h live
// side by side in wider buffers.  h may be dc: a thread reads its packet of dc before it writes h.
template <typename T>
__global__ __launch_bounds__(256) void swiglu_backward_kernel(const T* dc, const T* __restrict__ a,
                                                              const T* __restrict__ b, T* __restrict__ da,
                                                              T* __restrict__ db, T* h, int col_blocks,
                                                              int cols, int64_t da_stride, int64_t db_stride) {
    constexpr int V = Elem<T>::kVec;
    const uint32_t row = blockIdx.x / (uint32_t)col_blocks;
    const int col = ((int)(blockIdx.x % (uint32_t)col_blocks) * 256 + (int)threadIdx.x) * V;
    if (col >= cols) return;
    const int64_t at = (int64_t)row * cols + col;
    float dcv[V], av[V], bv[V], dav[V], dbv[V], hv[V];
    unpack16<T>(*reinterpret_cast<const u32x4_t*>(dc + at), dcv);
    unpack16<T>(*reinterpret_cast<const u32x4_t*>(a + at), av);
    unpack16<T>(*reinterpret_cast<const u32x4_t*>(b + at), bv);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const float sig = 1.0f / (1.0f + __expf(-av[v]));
        const float silu = av[v] * sig;
        dbv[v] = dcv[v] * silu;
        dav[v] = dcv[v] * (silu * (1.0f - sig) + sig) * bv[v];
        hv[v] = silu * bv[v];
    }
    *reinterpret_cast<u32x4_t*>(da + row * da_stride + col) = pack16<T>(dav);
    *reinterpret_cast<u32x4_t*>(db + row * db_stride + col) = pack16<T>(dbv);
    if (h != nullptr) *reinterpret_cast<u32x4_t*>(h + at) = pack16<T>(hv);
}

// ------------------------------------------------------------------------------------------------------------
// routed experts, per-token part: dx, dgates and the two coefficients of every pair
// ------------------------------------------------------------------------------------------------------------
// WAVES = 1: a wave per token.  WAVES > 1 (few tokens): the workgroup's waves share one token as in the forward, their partial rows of
// dx are added in wave order through LDS.
template <typename T, int NCH, int WAVES>
__global__ __launch_bounds__((WAVES > 1 ? WAVES : kBwdWaves) * kWave) void expert_backward_token_kernel(
    const T* __restrict__ dout, const T* __restrict__ x, const T* __restrict__ down, const T* __restrict__ up,
    const int64_t* __restrict__ indices, const T* __restrict__ gates, T* __restrict__ dx, T* __restrict__ dgates,
    float2* __restrict__ coef, int64_t num_tokens,
    int hidden, int64_t num_experts, int top_k) {
    constexpr int V = Elem<T>::kVec;
    constexpr int PIF = NCH >= 8 ? 1 : (NCH >= 4 ? 2 : 4);   // (down, up) row pairs requested ahead
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int64_t token = WAVES > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * kBwdWaves + wave;
    if (token >= num_tokens) return;
    constexpr int ROW = NCH * V * kWave;
    __shared__ __attribute__((aligned(16))) float partial_rows[WAVES > 1 ? WAVES * ROW : 4];

    const int packets = hidden / V;
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};
    u32x4_t xr[NCH], gr[NCH];
    bool live[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int p = c * kWave + lane;
        live[c] = p < packets;
        xr[c] = live[c] ? reinterpret_cast<const u32x4_t*>(x + token * hidden)[p] : zero4;
        gr[c] = live[c] ? reinterpret_cast<const u32x4_t*>(dout + token * hidden)[p] : zero4;
    }
    float acc[NCH][V];
#pragma unroll
    for (int c = 0; c < NCH; ++c)
#pragma unroll
        for (int v = 0; v < V; ++v) acc[c][v] = 0.0f;

    for (int k0 = WAVES > 1 ? wave * PIF : 0; k0 < top_k; k0 += WAVES * PIF) {
        u32x4_t dn[PIF][NCH], uq[PIF][NCH];
        float gate[PIF];
        bool valid[PIF];
#pragma unroll
        for (int u = 0; u < PIF; ++u) {
            const int k = k0 + u;
            int64_t e = -1;
            gate[u] = 0.0f;
            if (k < top_k) {
                e = indices[token * top_k + k];
                gate[u] = Elem<T>::to_f32(gates[token * top_k + k]);
            }
            const uint32_t elo = __builtin_amdgcn_readfirstlane((uint32_t)(e & 0xffffffff));
            const uint32_t ehi = __builtin_amdgcn_readfirstlane((uint32_t)((uint64_t)e >> 32));
            e = (int64_t)(((uint64_t)ehi << 32) | elo);
            valid[u] = e >= 0 && e < num_experts;
            const u32x4_t* drow = reinterpret_cast<const u32x4_t*>(down + (valid[u] ? e : 0) * hidden);
            const u32x4_t* urow = reinterpret_cast<const u32x4_t*>(up + (valid[u] ? e : 0) * hidden);
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const int p = c * kWave + lane;
                dn[u][c] = (valid[u] && live[c]) ? drow[p] : zero4;
                uq[u][c] = (valid[u] && live[c]) ? urow[p] : zero4;
            }
        }
        float s[PIF], da[PIF];
#pragma unroll
        for (int u = 0; u < PIF; ++u) {
            float ps = 0.0f, pa = 0.0f;
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                ps = dot16<T>(xr[c], dn[u][c], ps);
                pa = dot16<T>(gr[c], uq[u][c], pa);
            }
            s[u] = ps;
            da[u] = pa;
        }
#pragma unroll
        for (int u = 0; u < PIF; ++u) {
            s[u] = wave_sum(s[u]);
            da[u] = wave_sum(da[u]);
        }
#pragma unroll
        for (int u = 0; u < PIF; ++u) {
            const int k = k0 + u;
            const float sig = 1.0f / (1.0f + __expf(-s[u]));
            const float act = s[u] * sig;
            const float ds = valid[u] ? da[u] * gate[u] * (sig * (1.0f + s[u] * (1.0f - sig))) : 0.0f;
#pragma unroll
            for (int c = 0; c < NCH; ++c) axpy16<T>(ds, dn[u][c], acc[c]);
            if (lane == 0 && k < top_k) {
                const int64_t p = token * top_k + k;
                coef[p] = float2{valid[u] ? act * gate[u] : 0.0f, ds};
                dgates[p] = Elem<T>::from_f32(valid[u] ? da[u] * act : 0.0f);
            }
        }
    }
    if constexpr (WAVES > 1) {
#pragma unroll
        for (int c = 0; c < NCH; ++c)
#pragma unroll
            for (int v = 0; v < V; v += 4)
                *reinterpret_cast<f32x4_t*>(&partial_rows[wave * ROW + (c * kWave + lane) * V + v]) =
                    f32x4_t{acc[c][v], acc[c][v + 1], acc[c][v + 2], acc[c][v + 3]};
        __syncthreads();
        for (int p = (int)threadIdx.x; p < packets; p += WAVES * kWave) {
            float sum[V];
#pragma unroll
            for (int v = 0; v < V; ++v) sum[v] = partial_rows[p * V + v];
#pragma unroll
            for (int w = 1; w < WAVES; ++w)
#pragma unroll
                for (int v = 0; v < V; ++v) sum[v] += partial_rows[w * ROW + p * V + v];
            reinterpret_cast<u32x4_t*>(dx + token * hidden)[p] = pack16<T>(sum);
        }
        return;
    }
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int p = c * kWave + lane;
        if (live[c]) reinterpret_cast<u32x4_t*>(dx + token * hidden)[p] = pack16<T>(acc[c]);
    }
}

// Column-slice schedule of the per-token part (same kernels as the forward, fmoe_expert.hip): the partial dot products
// s = <x, down[e]> and u = <dout, up[e]> come per slice; this kernel sums them (or takes the scores the forward kept) and forms
// every pair's coefficients and gate gradient; dx is then the forward's `states` pass over `down` with
// coef_list, the coefficients of `down` in list order.  place: NULL (list order is pair order), or the (token, k) position of every list
// position.
template <typename T>
__global__ __launch_bounds__(256) void expert_backward_gate_kernel(
    const float* __restrict__ spart_s, const float* __restrict__ scores, const float* __restrict__ spart_u,
    const T* __restrict__ gates, const uint32_t* __restrict__ off32, const uint16_t* __restrict__ place,
    T* __restrict__ dgates, float2* __restrict__ coef, float* __restrict__ coef_list, int64_t pairs,
    int num_slices, int top_k) {
    const int64_t at = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (at >= pairs) return;
    const int64_t p = place == nullptr ? at : at / top_k * top_k + place[at];
    float s = 0.0f, u = 0.0f;
    for (int sl = 0; sl < num_slices; ++sl) {
        if (scores == nullptr) s += spart_s[(int64_t)sl * pairs + at];
        u += spart_u[(int64_t)sl * pairs + at];
    }
    if (scores != nullptr) s = scores[p];
    const bool valid = off32[at] != kExpertBadOffset;
    const float gate = Elem<T>::to_f32(gates[p]);
    const float sig = 1.0f / (1.0f + __expf(-s));
    const float act = s * sig;
    const float cd = valid ? u * gate * (sig * (1.0f + s * (1.0f - sig))) : 0.0f;
    coef[p] = float2{valid ? act * gate : 0.0f, cd};
    coef_list[at] = cd;
    dgates[p] = Elem<T>::from_f32(valid ? u * act : 0.0f);
}

// A wave takes `span` consecutive experts (lane l holds the end of the l-th one's segment) and a chunk of the columns (NCH * 1024 bytes):
// their pieces of ddown and dup, each summed over its pairs in ascending pair index.  The segments follow each other, so the wave walks
// one list, 64 pairs per round, with the pieces of the next pairs in flight whether or not an expert ends between them.
// Bound by what the caches deliver (x and dout, 4 KB per pair at 1024 columns), so the work is ordered chunk by chunk and every XCD
// gets a run of it: its L2 holds a chunk of x and dout instead of their whole rows.  Weight gradients, us: 4096 tokens x 64 pairs,
// 16384 experts, 1024 columns 90 -> 70; 1024 x 512, 102400 experts 172 -> 145; 1024 x 64, 2048 columns 90 -> 60.
// Where x and dout fit the L2 whole, chunks of two packets per lane save walking the lists twice.
template <typename T, int NCH>
__global__ __launch_bounds__(kBwdWaves* kWave) void expert_backward_weight_kernel(
    const T* __restrict__ dout, const T* __restrict__ x, const float2* __restrict__ coef, const uint32_t* __restrict__ pairs, const int32_t* __restrict__ offsets,
    T* __restrict__ ddown, T* __restrict__ dup, int hidden, int64_t num_experts, int top_k, int span, int units, int chunks, int xcds) {
    constexpr int V = Elem<T>::kVec, PIF = 8 / NCH;
    const int lane = lane_id();
    const int item = ((int)blockIdx.x % xcds) * ((int)gridDim.x / xcds) + (int)blockIdx.x / xcds;      // chunk-major
    if (item >= units * chunks) return;
    const int64_t e0 = ((int64_t)(item % units) * kBwdWaves + (threadIdx.x >> 6)) * span;
    if (e0 >= num_experts) return;
    const int count = num_experts - e0 < span ? (int)(num_experts - e0) : span;
    bool live[NCH];
    int at[NCH];                                              // lanes past the row read its first packet and store nothing
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int packet = (item / units * NCH + c) * kWave + lane;
        live[c] = packet < hidden / V;
        at[c] = live[c] ? packet : 0;
    }
    float acc_d[NCH][V], acc_u[NCH][V];
    auto clear = [&]() {
#pragma unroll
        for (int c = 0; c < NCH; ++c)
#pragma unroll
            for (int v = 0; v < V; ++v) acc_d[c][v] = acc_u[c][v] = 0.0f;
    };
    clear();

    // list positions are unsigned: a round may end past the 2^31 - 1 pairs that a call may have
    const int ends = offsets[e0 + (lane < count ? lane + 1 : count)];
    const uint32_t begin = (uint32_t)__builtin_amdgcn_readfirstlane(offsets[e0]), end = (uint32_t)__builtin_amdgcn_readlane(ends, count - 1);
    int cur = 0;
    uint32_t cur_end = (uint32_t)__builtin_amdgcn_readlane(ends, 0);
    // rows of the experts whose segments end at list position `pos`
    auto flush = [&](uint32_t pos) {
        while (cur < count && cur_end == pos) {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                if (live[c]) {
                    reinterpret_cast<u32x4_t*>(ddown + (e0 + cur) * hidden)[at[c]] = pack16<T>(acc_d[c]);
                    reinterpret_cast<u32x4_t*>(dup + (e0 + cur) * hidden)[at[c]] = pack16<T>(acc_u[c]);
                }
            }
            clear();
            ++cur;
            cur_end = (uint32_t)__builtin_amdgcn_readlane(ends, cur < count ? cur : count - 1);
        }
    };
    flush(begin);
    for (uint32_t done = begin; done < end; done += kWave) {
        const int n = end - done < (uint32_t)kWave ? (int)(end - done) : kWave;
        const uint32_t mine = pairs[done + (lane < n ? lane : n - 1)];
        const uint32_t tok = mine / (uint32_t)top_k;
        const float2 both = coef[mine];
        const float cu = both.x, cd = both.y;
        u32x4_t xq[PIF][NCH], gq[PIF][NCH];
        auto load = [&](int j, u32x4_t (&xr)[NCH], u32x4_t (&gr)[NCH]) {
            const int64_t t = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)tok, j < n ? j : n - 1);
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                xr[c] = reinterpret_cast<const u32x4_t*>(x + t * hidden)[at[c]];
                gr[c] = reinterpret_cast<const u32x4_t*>(dout + t * hidden)[at[c]];
            }
        };
#pragma unroll
        for (int u = 0; u < PIF; ++u) load(u, xq[u], gq[u]);
        for (int j0 = 0; j0 < n; j0 += PIF) {
#pragma unroll
            for (int u = 0; u < PIF; ++u) {
                const int j = j0 + u;
                if (j < n) {
                    const float sd = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cd), j));
                    const float su = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cu), j));
#pragma unroll
                    for (int c = 0; c < NCH; ++c) {
                        axpy16<T>(sd, xq[u][c], acc_d[c]);
                        axpy16<T>(su, gq[u][c], acc_u[c]);
                    }
                    flush(done + (uint32_t)j + 1u);
                }
                load(j + PIF, xq[u], gq[u]);
            }
        }
    }
}

// ---- the same where 1-KB chunks of x and dout do not fit an L2 -------------------------------------------------------------------
// A wave's quarters of 16 lanes take spans of experts of their own and 256 bytes of the columns, so that an XCD's chunk of x and dout is a
// quarter as large.  With four times the chunks the lists are walked as often, so pair_entries_kernel first puts what a pair needs in
// list order: the byte offset of its token's rows and its two coefficients.  A round is 16 pairs of each quarter, the next rounds' entries
// and PIF pairs' pieces are requested ahead.  Sums run in ascending pair index here too: the gradients are the same bit for bit.
// Bound by what the L2s deliver (1 KB chunks: a third of the lines missed at 4096 tokens).  Expert forward and backward, us, 1-KB chunks |
// quarters, ids uniform and of a product-key router: 4096 tokens x 64 pairs, 16384 experts, 1024 columns 252 | 212 and 220 | 212; 16384 x
// 64 1047 | 865 and 746 | 744; 8192 x 64, 65536 experts, 512 columns, router 367 | 352.  Where the chunks do fit, quarters only walk the
// lists more often: 2048 x 32, 2048 columns 165 | 166 and 161 | 170.  8 pairs ahead instead of 4, or five waves per SIMD instead of four,
// were slower (214 to 220), as were entries that every lane loads, for which no wait stands at the end of a round (214; 16384 tokens 891).
// One expert that every token names, 4096 tokens x 8 of 8192: 690 | 491, its list a chain of additions for either.  Which calls take them:
// quarter_waves.
// Unsigned: the last workgroup's threads may lie past the 2^31 - 1 pairs that a call may have.
__host__ __device__ constexpr auto list_position(uint32_t block, uint32_t thread) { return block * 256u + thread; }
static_assert(list_position(0x7fffffffu / 256u, 255u) > 0x7ffffffeu && list_position(0x7fffffffu / 256u, 255u) < 0xffffffffu, "the last list position");

__global__ __launch_bounds__(256) void pair_entries_kernel(const float2* __restrict__ coef, const uint32_t* __restrict__ pairs,
                                                          const int32_t* __restrict__ offsets, int64_t num_experts, uint32_t top_k,
                                                          uint32_t row_bytes, u32x4_t* __restrict__ entries) {
    const uint32_t at = list_position(blockIdx.x, threadIdx.x);
    if (at >= (uint32_t)offsets[num_experts]) return;
    const uint32_t pair = pairs[at];
    const float2 c = coef[pair];
    entries[at] = u32x4_t{pair / top_k * row_bytes, __float_as_uint(c.x), __float_as_uint(c.y), 0u};
}

template <int J> __device__ inline uint32_t row_lane(uint32_t v) {          // lane J's value in each row of 16 lanes (row_newbcast)
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + J, 0xF, 0xF, true);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// span <= 16; num_tokens * hidden values of x are below 2 GB.
template <typename T>
__global__ __launch_bounds__(kBwdWaves* kWave) void expert_backward_weight_quarters_kernel(
    const T* __restrict__ dout, const T* __restrict__ x, const u32x4_t* __restrict__ entries, const int32_t* __restrict__ offsets,
    T* __restrict__ ddown, T* __restrict__ dup, int64_t num_tokens, int hidden, int64_t num_experts, int span, int units, int chunks, int xcds) {
    constexpr int V = Elem<T>::kVec, PIF = 4;
    const int lane = lane_id(), quarter = lane & 48, ql = lane & 15;
    const int item = ((int)blockIdx.x % xcds) * ((int)gridDim.x / xcds) + (int)blockIdx.x / xcds;      // chunk-major
    if (item >= units * chunks) return;
    const int64_t e0 = (((int64_t)(item % units) * kBwdWaves + (threadIdx.x >> 6)) * 4 + (lane >> 4)) * span;
    const int count = num_experts - e0 < span ? (num_experts > e0 ? (int)(num_experts - e0) : 0) : span;
    const int packet = item / units * 16 + ql;
    const bool live = packet < hidden / V;                    // lanes past the row read its first packet and store nothing
    const uint32_t column = (uint32_t)(live ? packet : 0) * 16u;
    const int bytes = (int)(num_tokens * hidden * (int64_t)sizeof(T));
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(x), 0, bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t gr = __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(dout), 0, bytes, 0x00020000);
    float acc_d[V], acc_u[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc_d[v] = acc_u[v] = 0.0f;

    // Positions count from the quarter's first pair, unsigned: the wave walks on to the end of its longest list.
    const uint32_t begin = count > 0 ? (uint32_t)offsets[e0] : 0u, length = count > 0 ? (uint32_t)offsets[e0 + count] - begin : 0u;
    const uint32_t ends = count > 0 ? (uint32_t)offsets[e0 + (ql < count ? ql + 1 : count)] - begin : 0u;      // lane ql of a quarter: of its ql-th expert
    uint32_t longest = 0u;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t n = (uint32_t)__builtin_amdgcn_readlane((int)length, q * 16);
        longest = n > longest ? n : longest;
    }
    constexpr uint32_t kNone = 0xffffffffu;                   // every row of the quarter has left
    const uint32_t first_end = (uint32_t)__shfl((int)ends, quarter);
    int cur = 0;
    uint32_t cur_end = count > 0 ? first_end : kNone;
    // Rows of the experts whose segments end at position `pos`.  The sums are cleared by a select, not under a branch of some lanes: with
    // that the compiler kept a second copy of them at every position, 34 of 90 vector instructions.
    auto flush = [&](uint32_t pos) {
        bool ends_here = cur_end == pos;
        if (__builtin_amdgcn_ballot_w64(ends_here) == 0ull) return;
        do {
            if (ends_here && live) {
                reinterpret_cast<u32x4_t*>(ddown + (e0 + cur) * hidden)[packet] = pack16<T>(acc_d);
                reinterpret_cast<u32x4_t*>(dup + (e0 + cur) * hidden)[packet] = pack16<T>(acc_u);
            }
#pragma unroll
            for (int v = 0; v < V; ++v) {
                acc_d[v] = ends_here ? 0.0f : acc_d[v];
                acc_u[v] = ends_here ? 0.0f : acc_u[v];
            }
            cur += ends_here ? 1 : 0;
            const uint32_t next = (uint32_t)__shfl((int)ends, quarter + (cur < 15 ? cur : 15));
            cur_end = cur < count ? next : kNone;
            ends_here = cur_end == pos;
        } while (__builtin_amdgcn_ballot_w64(ends_here) != 0ull);
    };
    flush(0u);
    auto round_at = [&](uint32_t first) {                     // entries past the quarter's list: nothing is fetched, zeros are added
        const uint32_t at = first + (uint32_t)ql;
        return at < length ? entries[begin + at] : u32x4_t{0x80000000u, 0u, 0u, 0u};
    };
    u32x4_t now = round_at(0u), next = round_at(16u), xq[PIF], gq[PIF];
    auto load = [&](auto j, const u32x4_t& of, u32x4_t& xv, u32x4_t& gv) {
        const int at = (int)(row_lane<decltype(j)::value>(of[0]) + column);
        xv = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(xr, at, 0, 0));
        gv = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(gr, at, 0, 0));
    };
    static_for<PIF>([&](auto j) { load(j, now, xq[j], gq[j]); });
    for (uint32_t done = 0u; done < longest; done += 16u) {
        const u32x4_t after = round_at(done + 32u);
        static_for<16>([&](auto j) {
            constexpr int J = decltype(j)::value, S = J % PIF;
            axpy16<T>(__uint_as_float(row_lane<J>(now[2])), xq[S], acc_d);
            axpy16<T>(__uint_as_float(row_lane<J>(now[1])), gq[S], acc_u);
            flush(done + (uint32_t)J + 1u);
            load(std::integral_constant<int, (J + PIF) % 16>{}, J + PIF < 16 ? now : next, xq[S], gq[S]);
        });
        now = next;
        next = after;
    }
}

struct ExpertBwdPlan {
    bool slices, ordered;      // slices: column slices of the tables, on ordered lists or not
    bool quarters;             // weight gradients by quarter waves
    int num_slices;
    size_t off_coef, off_entries, off_pairs, off_group, off_offsets, off_off32, off_place, off_coef_list, off_spart_s, off_spart_u, bytes;
};

// Weight gradients by quarter waves: 1-KB chunks of x and dout exceed an L2, and what that saves is more than the entries' launch and the
// shorter reads cost.  Expert backward, us, whole waves | quarters, over 425 sizes (2100 to 20000 tokens, 64 to 524288 experts, 4 to 64 per
// token; the rule is 0.3 % behind the better of the two on average, quarters everywhere 2.7 %, nowhere 7.2 %):
//   64 pairs to an expert and more, few waves that walk long lists: 3000 tokens x 32, 512 experts, 1024 columns 102 | 94; 64 experts 334 | 254;
//   rows of 256 bytes and less, of which a whole wave has idle lanes: 20000 x 16 of 4096, 64 columns 97 | 81;
//   else where the chunks exceed an L2 by two fifths (2868 tokens of 1 KB), for 48 K pairs and one and a half to an expert: 16384 x 16 of 16384,
//   1024 columns 317 | 268.  Below them: 2100 x 32 of 8192, 512 columns 66 | 69; x 4 25 | 31; 16384 x 16 of 262144, 1024 columns 565 | 630.
inline bool quarter_waves(int64_t tokens, int64_t row, int64_t experts, int64_t pairs) {
    const int64_t chunks = 2 * tokens * (row < 1024 ? row : 1024), l2 = chip_info().l2_bytes;
    if (pairs == 0 || chunks <= l2 || tokens * row >= (1ll << 31)) return false;
    return pairs / 64 >= experts || row <= 256 || (5 * chunks >= 7 * l2 && pairs >= 3 << 14 && 2 * pairs >= 3 * experts);
}

ExpertBwdPlan plan_expert_backward(int64_t T_, int H, int64_t E, int K, int dtype) {
    ExpertBwdPlan p;
    const size_t pairs = (size_t)T_ * K;
    size_t o = 0;
    auto take = [&](size_t n) { const size_t at = o; o = round_up(o + n, 256); return at; };
    p.off_coef = take(pairs * 8);
    p.quarters = quarter_waves(T_, (int64_t)H * (int64_t)dtype_size(dtype), E, (int64_t)pairs);
    p.off_entries = take(p.quarters ? pairs * 16 : 0);
    p.off_pairs = take(pairs * 4);
    p.off_group = take(group_pairs_workspace_bytes((int64_t)pairs, E));
    p.off_offsets = take((size_t)(E + 1) * 4);
    const ExpertSavedPlan kept = expert_saved_plan(T_, H, E, K, dtype);
    p.slices = kept.kept;
    p.ordered = kept.ordered;
    p.num_slices = p.slices ? expert_slice_count(T_, H, E, K, dtype, p.ordered) : 0;
    p.off_off32 = p.off_place = p.off_coef_list = p.off_spart_s = p.off_spart_u = o;
    if (p.slices) {
        p.off_coef_list = take(pairs * 4);
        p.off_off32 = take(pairs * 4);
        p.off_place = take(p.ordered ? pairs * 2 : 0);
        p.off_spart_s = take((size_t)p.num_slices * pairs * 4);
        p.off_spart_u = take((size_t)p.num_slices * pairs * 4);
    }
    p.bytes = o;
    return p;
}

template <typename T>
int launch_expert_backward(const void* dout, const void* x, const void* down, const void* up, const int64_t* indices,
                           const void* gates, int64_t T_, int H, int64_t E, int K, int dtype, void* dx, void* ddown, void* dup,
                           void* dgates, const void* saved, void* workspace, hipStream_t stream) {
    constexpr int V = Elem<T>::kVec;
    const ExpertBwdPlan p = plan_expert_backward(T_, H, E, K, dtype);
    char* ws = (char*)workspace;
    float2* coef = (float2*)(ws + p.off_coef);          // of every pair: of its row of dup, of its row of ddown
    uint32_t* pairs_by_expert = (uint32_t*)(ws + p.off_pairs);
    int32_t* offsets = (int32_t*)(ws + p.off_offsets);
    const int64_t pairs = T_ * K;
    const int nch = (H / V + kWave - 1) / kWave;
    const dim3 block(kBwdWaves * kWave);
    if (p.slices) {
        uint32_t* off32 = (uint32_t*)(ws + p.off_off32);
        uint16_t* place = p.ordered ? (uint16_t*)(ws + p.off_place) : nullptr;
        float* spart_s = (float*)(ws + p.off_spart_s);
        float* spart_u = (float*)(ws + p.off_spart_u);
        float* coef_list = (float*)(ws + p.off_coef_list);
        const float* scores = nullptr;
        if (saved != nullptr) {
            const ExpertSaved kept = expert_saved_plan(T_, H, E, K, dtype).at(saved);
            off32 = kept.off32;
            if (p.ordered) place = kept.place;
            scores = kept.scores;
        } else {
            if (int rc = p.ordered ? expert_order(indices, off32, place, T_, H, E, K, dtype, stream)
                                   : expert_slice_prepare(indices, off32, pairs, H, E, dtype, stream))
                return rc;
            if (int rc = expert_slice_scores(x, down, off32, spart_s, T_, H, E, K, dtype, p.ordered, stream)) return rc;
        }
        if (int rc = expert_slice_scores(dout, up, off32, spart_u, T_, H, E, K, dtype, p.ordered, stream)) return rc;
        hipLaunchKernelGGL((expert_backward_gate_kernel<T>), dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, stream,
                           (const float*)spart_s, scores, (const float*)spart_u, (const T*)gates, (const uint32_t*)off32,
                           (const uint16_t*)place, (T*)dgates, coef, coef_list, pairs, p.num_slices, K);
        FMOE_CHECK_LAUNCH("fmoe_expert_backward(coefficients)");
        if (int rc = expert_slice_states(coef_list, down, off32, dx, T_, H, E, K, dtype, p.ordered, stream)) return rc;
    } else {
        // waves per token: as the forward's rows; sixteen fit their registers up to two packets per lane
        const int waves = K <= 4 || T_ > 2048 ? 1 : (T_ > chip_info().cus ? 4 : (nch > 2 ? 8 : 16));
#define FMOE_LAUNCH_TOKEN(N, W)                                                                                                       \
        hipLaunchKernelGGL((expert_backward_token_kernel<T, N, W>), dim3((unsigned)(W > 1 ? T_ : (T_ + kBwdWaves - 1) / kBwdWaves)), \
                           dim3((W > 1 ? W : kBwdWaves) * kWave), 0, stream, (const T*)dout, (const T*)x, (const T*)down,            \
                           (const T*)up, indices, (const T*)gates, (T*)dx, (T*)dgates, coef, T_, H, E, K)
#define FMOE_LAUNCH_TOKENS(N, MOST)                                      \
        do {                                                             \
            if (waves >= 8) FMOE_LAUNCH_TOKEN(N, MOST);                  \
            else if (waves == 4) FMOE_LAUNCH_TOKEN(N, 4);                \
            else FMOE_LAUNCH_TOKEN(N, 1);                                \
        } while (0)
        if (nch <= 1) FMOE_LAUNCH_TOKENS(1, 16);
        else if (nch <= 2) FMOE_LAUNCH_TOKENS(2, 16);
        else if (nch <= 4) FMOE_LAUNCH_TOKENS(4, 8);
        else FMOE_LAUNCH_TOKENS(8, 8);
#undef FMOE_LAUNCH_TOKENS
#undef FMOE_LAUNCH_TOKEN
        FMOE_CHECK_LAUNCH("fmoe_expert_backward(tokens)");
    }

    // offsets and segments, each in ascending pair index
    if (int rc = group_pairs(indices, ws + p.off_group, pairs, E, K, offsets, (int32_t*)pairs_by_expert, stream)) return rc;

    // experts per wave: about a round of 64 pairs, as long as every SIMD keeps four waves
    const int xcds = chip_info().xcds;
    const bool resident = 2 * T_ * H * (int64_t)sizeof(T) < chip_info().l2_bytes;
    const int chunks = resident ? (nch + 1) / 2 : nch;
    int64_t span = pairs > 0 ? 64 * E / pairs : 32;
    const int64_t most = E * chunks / (chip_info().cus * 16);
    if (span > most) span = most;
    span = span < 1 ? 1 : (span > 32 ? 32 : span);
    const int64_t units = (E + span * kBwdWaves - 1) / (span * kBwdWaves);
#define FMOE_LAUNCH_WEIGHT(N)                                                                                                             \
    hipLaunchKernelGGL((expert_backward_weight_kernel<T, N>), dim3((unsigned)((units * chunks + xcds - 1) / xcds * xcds)), block, 0, stream, \
                       (const T*)dout, (const T*)x, (const float2*)coef, (const uint32_t*)pairs_by_expert,     \
                       (const int32_t*)offsets, (T*)ddown, (T*)dup, H, E, K, (int)span, (int)units, chunks, xcds)
    if (p.quarters) {
        const int quarters = (H / V + 15) / 16;
        u32x4_t* entries = (u32x4_t*)(ws + p.off_entries);
        hipLaunchKernelGGL(pair_entries_kernel, dim3((unsigned)((pairs + 255) / 256)), dim3(256), 0, stream, (const float2*)coef,
                           (const uint32_t*)pairs_by_expert, (const int32_t*)offsets, E, (uint32_t)K, (uint32_t)(H * sizeof(T)), entries);
        FMOE_CHECK_LAUNCH("fmoe_expert_backward(entries)");
        span = pairs > 0 ? 64 * E / pairs : 16;
        const int64_t most_q = E * quarters / (chip_info().cus * 64);
        if (span > most_q) span = most_q;
        span = span < 1 ? 1 : (span > 16 ? 16 : span);
        const int64_t units_q = (E + span * kBwdWaves * 4 - 1) / (span * kBwdWaves * 4);
        hipLaunchKernelGGL((expert_backward_weight_quarters_kernel<T>), dim3((unsigned)((units_q * quarters + xcds - 1) / xcds * xcds)), block, 0,
                           stream, (const T*)dout, (const T*)x, (const u32x4_t*)entries, (const int32_t*)offsets, (T*)ddown, (T*)dup, T_, H, E,
                           (int)span, (int)units_q, quarters, xcds);
    } else if (resident && nch > 1) {
        FMOE_LAUNCH_WEIGHT(2);
    } else {
        FMOE_LAUNCH_WEIGHT(1);
    }
#undef FMOE_LAUNCH_WEIGHT
    FMOE_CHECK_LAUNCH("fmoe_expert_backward(weights)");
    return FMOE_OK;
}

}  // namespace

__global__ void zero_fill_kernel(u32x4_t* __restrict__ p, size_t packets) {
    const u32x4_t zero4 = {0u, 0u, 0u, 0u};
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < packets; i += (size_t)gridDim.x * blockDim.x) p[i] = zero4;
}

// Used by the MLP backward (fmoe_mlp_backward.hip).
int launch_swiglu_backward(const void* dc, const void* a, const void* b, void* da, void* db, void* h, int64_t rows, int cols,
                           int64_t da_stride, int64_t db_stride, int dtype, hipStream_t stream) {
    const int vec = (int)(16 / dtype_size(dtype));
    if (rows == 0) return FMOE_OK;
    const int col_blocks = (cols / vec + 255) / 256;
    FMOE_REQUIRE(rows * col_blocks < (1ll << 31), FMOE_ERR_UNSUPPORTED, "fmoe_swiglu_backward: %lld rows of %d columns exceed the grid",
                 (long long)rows, cols);
    const dim3 grid((unsigned)(rows * col_blocks)), block(256);
    switch (dtype) {
        case FMOE_F32:
            hipLaunchKernelGGL((swiglu_backward_kernel<float>), grid, block, 0, stream, (const float*)dc, (const float*)a,
                               (const float*)b, (float*)da, (float*)db, (float*)h, col_blocks, cols, da_stride, db_stride);
            break;
        case FMOE_BF16:
            hipLaunchKernelGGL((swiglu_backward_kernel<bf16_t>), grid, block, 0, stream, (const bf16_t*)dc, (const bf16_t*)a,
                               (const bf16_t*)b, (bf16_t*)da, (bf16_t*)db, (bf16_t*)h, col_blocks, cols, da_stride, db_stride);
            break;
        default:
            hipLaunchKernelGGL((swiglu_backward_kernel<f16_t>), grid, block, 0, stream, (const f16_t*)dc, (const f16_t*)a,
                               (const f16_t*)b, (f16_t*)da, (f16_t*)db, (f16_t*)h, col_blocks, cols, da_stride, db_stride);
    }
    FMOE_CHECK_LAUNCH("fmoe_swiglu_backward");
    return FMOE_OK;
}

}  // namespace fmoe

extern "C" int fmoe_router_topk_backward(const void* dscores, const int64_t* indices, int64_t num_tokens, int num_keys,
                                         int top_k, int dtype, void* drouter_logits, void* stream) {
    using namespace fmoe;
    clear_error();
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "fmoe_router_topk_backward: unknown dtype %d", dtype);
    FMOE_REQUIRE(num_tokens >= 0 && num_keys > 0 && top_k >= 0, FMOE_ERR_BAD_SHAPE,
                 "fmoe_router_topk_backward: bad shape T=%lld nk=%d K=%d", (long long)num_tokens, num_keys, top_k);
    FMOE_REQUIRE(num_keys <= 65535, FMOE_ERR_UNSUPPORTED, "fmoe_router_topk_backward: num_keys=%d > 65535", num_keys);
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(drouter_logits && (top_k == 0 || (dscores && indices)), FMOE_ERR_NULL_POINTER,
                 "fmoe_router_topk_backward: null tensor pointer");
    hipStream_t s = (hipStream_t)stream;
    switch (dtype) {
        case FMOE_F32: return launch_router_backward<float>(dscores, indices, drouter_logits, num_tokens, num_keys, top_k, s);
        case FMOE_BF16: return launch_router_backward<bf16_t>(dscores, indices, drouter_logits, num_tokens, num_keys, top_k, s);
        default: return launch_router_backward<f16_t>(dscores, indices, drouter_logits, num_tokens, num_keys, top_k, s);
    }
}

extern "C" int fmoe_route_backward(const void* dgates, const int64_t* indices, const float* logits_fp32, const void* dlogits_extra,
                                   int64_t num_tokens, int num_keys, int top_k, int dtype, int norm_topk_prob,
                                   float* dlogits_fp32, void* stream) {
    fmoe::clear_error();
    return fmoe::route_backward_impl(dgates, indices, logits_fp32, dlogits_extra, 2 * (int64_t)num_keys, num_keys, num_tokens, num_keys,
                                     top_k, dtype, norm_topk_prob, dlogits_fp32, (hipStream_t)stream);
}

bool fmoe::route_backward_prepares(int num_keys, int top_k) { return num_keys <= 4 * kWave && top_k <= 2 * kWave; }

int fmoe::route_backward_impl(const void* dgates, const int64_t* indices, const float* logits_fp32, const void* dlogits_extra,
                              int64_t extra_token, int64_t extra_half, int64_t num_tokens, int num_keys, int top_k, int dtype,
                              int norm_topk_prob, float* dlogits_fp32, hipStream_t s, const PrologueOperands* operands) {
    using namespace fmoe;
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "fmoe_route_backward: unknown dtype %d", dtype);
    FMOE_REQUIRE(num_tokens >= 0 && num_keys > 0 && top_k >= 0, FMOE_ERR_BAD_SHAPE,
                 "fmoe_route_backward: bad shape T=%lld nk=%d K=%d", (long long)num_tokens, num_keys, top_k);
    FMOE_REQUIRE(num_keys <= 32767, FMOE_ERR_UNSUPPORTED, "fmoe_route_backward: num_keys=%d > 32767", num_keys);
    if (num_tokens == 0) return FMOE_OK;
    FMOE_REQUIRE(logits_fp32 && (dlogits_fp32 || operands) && (top_k == 0 || (dgates && indices)), FMOE_ERR_NULL_POINTER,
                 "fmoe_route_backward: null tensor pointer");
    switch (dtype) {
        case FMOE_F32: return launch_route_backward<float>(dgates, indices, logits_fp32, dlogits_extra, extra_token, extra_half, dlogits_fp32, num_tokens, num_keys, top_k, norm_topk_prob, s, operands);
        case FMOE_BF16: return launch_route_backward<bf16_t>(dgates, indices, logits_fp32, dlogits_extra, extra_token, extra_half, dlogits_fp32, num_tokens, num_keys, top_k, norm_topk_prob, s, operands);
        default: return launch_route_backward<f16_t>(dgates, indices, logits_fp32, dlogits_extra, extra_token, extra_half, dlogits_fp32, num_tokens, num_keys, top_k, norm_topk_prob, s, operands);
    }
}

extern "C" int fmoe_swiglu_backward(const void* dc, const void* a, const void* b, int64_t rows, int cols, int dtype, void* da,
                                    void* db, void* stream) {
    using namespace fmoe;
    clear_error();
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "fmoe_swiglu_backward: unknown dtype %d", dtype);
    FMOE_REQUIRE(rows >= 0 && cols > 0, FMOE_ERR_BAD_SHAPE, "fmoe_swiglu_backward: bad shape rows=%lld cols=%d", (long long)rows, cols);
    if (rows == 0) return FMOE_OK;
    FMOE_REQUIRE(dc && a && b && da && db, FMOE_ERR_NULL_POINTER, "fmoe_swiglu_backward: null tensor pointer");
    const int vec = (int)(16 / dtype_size(dtype));
    FMOE_REQUIRE(cols % vec == 0 && aligned16(dc) && aligned16(a) && aligned16(b) && aligned16(da) && aligned16(db), FMOE_ERR_ALIGNMENT,
                 "fmoe_swiglu_backward: cols=%d must be a multiple of %d and tensors 16-byte aligned", cols, vec);
    return launch_swiglu_backward(dc, a, b, da, db, nullptr, rows, cols, cols, cols, dtype, (hipStream_t)stream);
}

extern "C" size_t fmoe_expert_backward_workspace_bytes(int64_t num_tokens, int hidden, int64_t num_experts, int top_k, int dtype) {
    if (num_tokens <= 0 || hidden <= 0 || num_experts <= 0 || top_k <= 0 || !fmoe::dtype_ok(dtype)) return 0;
    return fmoe::plan_expert_backward(num_tokens, hidden, num_experts, top_k, dtype).bytes;
}

extern "C" int fmoe_expert_backward(const void* dout, const void* x, const void* down, const void* up, const int64_t* indices,
                                    const void* gates, int64_t num_tokens, int hidden, int64_t num_experts, int top_k, int dtype,
                                    void* dx, void* ddown, void* dup, void* dgates, void* workspace, size_t workspace_bytes,
                                    void* stream) {
    return fmoe_expert_backward_saved(dout, x, down, up, indices, gates, nullptr, num_tokens, hidden, num_experts, top_k, dtype, dx, ddown,
                                      dup, dgates, workspace, workspace_bytes, stream);
}

extern "C" int fmoe_expert_backward_saved(const void* dout, const void* x, const void* down, const void* up, const int64_t* indices,
                                          const void* gates, const void* saved, int64_t num_tokens, int hidden, int64_t num_experts,
                                          int top_k, int dtype, void* dx, void* ddown, void* dup, void* dgates, void* workspace,
                                          size_t workspace_bytes, void* stream) {
    using namespace fmoe;
    clear_error();
    FMOE_REQUIRE(dtype_ok(dtype), FMOE_ERR_BAD_DTYPE, "fmoe_expert_backward: unknown dtype %d", dtype);
    FMOE_REQUIRE(num_tokens >= 0 && hidden > 0 && num_experts > 0 && top_k >= 0, FMOE_ERR_BAD_SHAPE,
                 "fmoe_expert_backward: bad shape T=%lld H=%d E=%lld K=%d", (long long)num_tokens, hidden, (long long)num_experts, top_k);
    const int vec = (int)(16 / dtype_size(dtype));
    FMOE_REQUIRE(hidden % vec == 0, FMOE_ERR_ALIGNMENT, "fmoe_expert_backward: hidden=%d must be a multiple of %d (16-byte rows)", hidden, vec);
    // rows too long for the per-token row kernel take the column-slice kernels, which need 32-bit row offsets
    FMOE_REQUIRE(hidden <= 8 * kWave * vec || num_tokens == 0 || top_k == 0 || expert_saved_plan(num_tokens, hidden, num_experts, top_k, dtype).kept,
                 FMOE_ERR_UNSUPPORTED, "fmoe_expert_backward: rows of more than %d elements need tables below 4 GiB (hidden=%d, E=%lld)",
                 8 * kWave * vec, hidden, (long long)num_experts);
    FMOE_REQUIRE(num_experts < (1ll << 31) - 1 && (int64_t)num_tokens * top_k < (1ll << 31), FMOE_ERR_UNSUPPORTED,
                 "fmoe_expert_backward: E=%lld or T*K=%lld >= 2^31", (long long)num_experts, (long long)num_tokens * top_k);
    FMOE_REQUIRE(ddown && dup && down && up && (num_tokens == 0 || (dx && x && dout)), FMOE_ERR_NULL_POINTER,
                 "fmoe_expert_backward: null tensor pointer");
    FMOE_REQUIRE(aligned16(dx) && aligned16(ddown) && aligned16(dup) && aligned16(x) && aligned16(dout) && aligned16(down) && aligned16(up),
                 FMOE_ERR_ALIGNMENT, "fmoe_expert_backward: tensor pointers must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    const size_t elt = dtype_size(dtype);
    if (num_tokens == 0 || top_k == 0) {   // no pairs: every gradient is zero (a fill kernel, safe under graph capture)
        const size_t table_packets = (size_t)num_experts * hidden * elt / 16, x_packets = (size_t)num_tokens * hidden * elt / 16;
        hipLaunchKernelGGL(zero_fill_kernel, dim3(1024), dim3(256), 0, s, (u32x4_t*)ddown, table_packets);
        hipLaunchKernelGGL(zero_fill_kernel, dim3(1024), dim3(256), 0, s, (u32x4_t*)dup, table_packets);
        if (x_packets) hipLaunchKernelGGL(zero_fill_kernel, dim3(1024), dim3(256), 0, s, (u32x4_t*)dx, x_packets);
        FMOE_CHECK_LAUNCH("fmoe_expert_backward(clear)");
        return FMOE_OK;
    }
    FMOE_REQUIRE(indices && gates && dgates, FMOE_ERR_NULL_POINTER, "fmoe_expert_backward: null indices/gates with top_k=%d", top_k);
    const size_t need = plan_expert_backward(num_tokens, hidden, num_experts, top_k, dtype).bytes;
    FMOE_REQUIRE(workspace && workspace_bytes >= need && aligned16(workspace), FMOE_ERR_WORKSPACE,
                 "fmoe_expert_backward: workspace of %zu bytes needed, %zu given", need, workspace_bytes);
    switch (dtype) {
        case FMOE_F32: return launch_expert_backward<float>(dout, x, down, up, indices, gates, num_tokens, hidden, num_experts, top_k, dtype, dx, ddown, dup, dgates, saved, workspace, s);
        case FMOE_BF16: return launch_expert_backward<bf16_t>(dout, x, down, up, indices, gates, num_tokens, hidden, num_experts, top_k, dtype, dx, ddown, dup, dgates, saved, workspace, s);
        default: return launch_expert_backward<f16_t>(dout, x, down, up, indices, gates, num_tokens, hidden, num_experts, top_k, dtype, dx, ddown, dup, dgates, saved, workspace, s);
    }
}
