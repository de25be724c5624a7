// Product-key selection on one wave per token, for lists that fit the wave's registers (gfx950): the keys and sorting networks all
// selections share, and the selection by threshold of the kernels in fmoe_router.hip and fmoe_small.hip.
#pragma once

#include <math.h>

#include "fmoe_common.h"

namespace fmoe {
namespace {

__device__ inline uint32_t order_bits(float f) {
    const uint32_t u = __float_as_uint(f);
    return u ^ ((u >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ inline float order_value(uint32_t o) {
    return __uint_as_float(o ^ ((o >> 31) ? 0x80000000u : 0xffffffffu));
}
__device__ inline uint64_t make_key(float score, uint32_t index) {
    return ((uint64_t)order_bits(score) << 32) | (uint64_t)(~index);
}
__device__ inline float key_score(uint64_t k) { return order_value((uint32_t)(k >> 32)); }
__device__ inline uint32_t key_index(uint64_t k) { return ~(uint32_t)(k & 0xffffffffu); }

// Value of lane (lane ^ mask) for the masks of a sorting network, a power of two or one less than that; `mask` must be a compile-time
// constant after inlining.  Distances 1, 2 and 8 and mirrors within a row are single DPP moves.  The others would cost 2-4 vector
// instructions each on the DPP / permlane path; the kernel is bound by instruction issue, so they go through the LDS crossbar
// (ds_swizzle / ds_bpermute: no LDS memory is touched, no vector-ALU slot is used, other waves cover the latency).
__device__ inline uint32_t xor_lane_u32(uint32_t v, int mask, int lane) {
    const int iv = (int)v;
    switch (mask) {
        case 1: return (uint32_t)__builtin_amdgcn_update_dpp(0, iv, 0xB1, 0xF, 0xF, true);    // quad_perm [1,0,3,2]
        case 2: return (uint32_t)__builtin_amdgcn_update_dpp(0, iv, 0x4E, 0xF, 0xF, true);    // quad_perm [2,3,0,1]
        case 3: return (uint32_t)__builtin_amdgcn_update_dpp(0, iv, 0x1B, 0xF, 0xF, true);    // quad_perm [3,2,1,0]
        case 4: return (uint32_t)__builtin_amdgcn_ds_swizzle(iv, (4 << 10) | 0x1F);          // bit mode: lane ^ 4
        case 7: return (uint32_t)__builtin_amdgcn_update_dpp(0, iv, 0x141, 0xF, 0xF, true);   // row_half_mirror
        case 8: return (uint32_t)__builtin_amdgcn_update_dpp(0, iv, 0x128, 0xF, 0xF, true);   // row_ror:8
        case 15: return (uint32_t)__builtin_amdgcn_update_dpp(0, iv, 0x140, 0xF, 0xF, true);  // row_mirror
        case 16: return (uint32_t)__builtin_amdgcn_ds_swizzle(iv, (16 << 10) | 0x1F);        // bit mode: lane ^ 16
        case 31: return (uint32_t)__builtin_amdgcn_ds_swizzle(iv, (31 << 10) | 0x1F);        // bit mode: lane ^ 31
        default: return (uint32_t)__builtin_amdgcn_ds_bpermute((lane ^ mask) << 2, iv);
    }
}
__device__ inline uint64_t xor_lane_u64(uint64_t v, int mask, int lane) {
    const uint32_t lo = xor_lane_u32((uint32_t)v, mask, lane);
    const uint32_t hi = xor_lane_u32((uint32_t)(v >> 32), mask, lane);
    return ((uint64_t)hi << 32) | lo;
}

// Position of a key in the wave-wide sequence: p = lane*RK + r.
// One compare-exchange layer: a key and the one at p ^ X, X = J or (the first layer of a stage) 2J - 1, the mirror of its block.  The key
// with bit J of its position clear keeps the larger one (DESC).  With the mirror every block of a stage runs in one direction, so
// which lanes keep the larger key takes only six 64-bit constants over all layers; they stay in scalar registers and reach the selects
// as a lane mask (inverse ballot).  With blocks of alternating direction each layer had a constant of its own: 15 layers of 32 lanes
// took 45 scalar instructions for 15 now, and the scalar unit was the busiest of the kernel.
constexpr uint64_t lanes_with_clear(int bit) {
    uint64_t m = 0;
    for (int l = 0; l < kWave; ++l) m |= (uint64_t)((l & bit) == 0) << l;
    return m;
}
template <int RK, bool DESC, int J, int X>
__device__ inline void exchange_layer(uint64_t (&v)[RK], int lane) {
    if constexpr (X < RK) {
#pragma unroll
        for (int r = 0; r < RK; ++r) {
            if ((r & J) == 0) {
                const uint64_t a = v[r], b = v[r ^ X];
                const bool swap = DESC ? a < b : a > b;
                v[r] = swap ? b : a;
                v[r ^ X] = swap ? a : b;
            }
        }
    } else {
        constexpr uint64_t first = lanes_with_clear(J / RK);         // J is at least RK here
        const bool keep_max = __builtin_amdgcn_inverse_ballot_w64(DESC ? first : ~first);
        uint64_t w[RK];
#pragma unroll
        for (int r = 0; r < RK; ++r) {
            const uint64_t other = xor_lane_u64(v[r ^ (X % RK)], X / RK, lane);
            // keep my key if it is the larger one and I keep the max, or the smaller one and I keep the min
            w[r] = ((v[r] > other) == keep_max) ? v[r] : other;
        }
#pragma unroll
        for (int r = 0; r < RK; ++r) v[r] = w[r];
    }
}

// layers J, J/2, ..., 1: sorts blocks of 2J keys that hold a bitonic sequence each
template <int RK, bool DESC, int J>
__device__ inline void bitonic_layers(uint64_t (&v)[RK], int lane) {
    exchange_layer<RK, DESC, J, J>(v, lane);
    if constexpr (J > 1) bitonic_layers<RK, DESC, J / 2>(v, lane);
}
// sorted blocks of K keys out of sorted blocks of K / 2, up to blocks of N
template <int RK, bool DESC, int N, int K = 2>
__device__ inline void sort_blocks(uint64_t (&v)[RK], int lane) {
    exchange_layer<RK, DESC, K / 2, K - 1>(v, lane);
    if constexpr (K > 2) bitonic_layers<RK, DESC, K / 4>(v, lane);
    if constexpr (K < N) sort_blocks<RK, DESC, N, 2 * K>(v, lane);
}

template <int RK, bool DESC>
__device__ inline void bitonic_sort(uint64_t (&v)[RK], int lane) {
    sort_blocks<RK, DESC, RK * kWave>(v, lane);
}

// v holds a bitonic sequence of N keys; sort it descending.
template <int RK>
__device__ inline void bitonic_merge_desc(uint64_t (&v)[RK], int lane) {
    bitonic_layers<RK, true, RK * kWave / 2>(v, lane);
}

// Key at position `pos` of the wave-wide sequence (wave-uniform `pos`).
template <int RK>
__device__ inline uint64_t key_at(const uint64_t (&v)[RK], int pos) {
    uint64_t k = v[0];
#pragma unroll
    for (int r = 1; r < RK; ++r) k = (pos % RK == r) ? v[r] : k;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)k, pos / RK);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(k >> 32), pos / RK);
    return ((uint64_t)hi << 32) | lo;
}

// ------------------------------------------------------------------------------------------------------------
// Selection by threshold (num_keys <= 64*RH, candidates <= 64*RC): the same result as the group scan above, for the
// sizes where a whole list fits the wave's registers (R keys per lane).
//   1. a score tau that at least K and at most CAP keys reach (CAP: the slots that are sorted), found bit by bit from the top (per
//      bit one compare per register, the counts come from the ballots on the scalar unit): any such tau will do, so the search
//      ends after 3 to 9 of the 32 bits, where the exact K-th largest score would take about 22.  REUSE: the score that served
//      the wave's last list of this kind is tried first; lists of a batch resemble each other, and with slots to spare (CAP = 32,
//      K = 16) it serves nine lists of ten.  Whichever score is found, the result is the same;
//   2. the keys at or above tau go to slots in LDS (positions from ballot prefix counts);
//   3. one bitonic sort of the slots (num_keys is at most 512: pairs have 18 bits); the first K are the result.
// List order is key index order for a half (position p = r*64 + lane), so ties at the cut go to the lowest index there; among
// candidate sums tied at the cut the earlier candidate (lower rank in half 0) is taken: where the sorted keys show such a tie, or
// more than CAP keys tie with the K-th, the keys above that score and then the equal ones in list order are taken again.
// Up to 32 experts per token (SMALL) CAP is 32 and one sort orders both halves, 32 lanes each.
// Bound by instruction issue, the scalar unit (searches, lane masks) hardly less than the vector units: 32768 tokens, 128 keys, 16
// experts take 20.3 us, 22.4 with sorts on integers, 28 also without REUSE (323 scalar and 294 vector instructions per token: each unit
// busy two thirds of the time), 32 with a constant per layer of the sorts and the search on the vector unit (332 and 472), 92 with the
// exact search and three 64-lane sorts; 64 experts 46.6 for 57.  128 tokens or fewer, 32 experts: 10.3 -> 7.1 with the threshold, 4096
// tokens, 64 experts: 16 -> 12.5, 11.0 and now 9.9.
// ------------------------------------------------------------------------------------------------------------
template <int CTRL> __device__ inline uint32_t dpp_max_step(uint32_t v) {      // lanes without a source read 0
    const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, true);
    return v > o ? v : o;
}
// The largest a and the largest b of the wave: folded onto one half of the lanes each, then reduced together.
__device__ inline void wave_max_two_u32(uint32_t& a, uint32_t& b) {
    const auto folded = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    uint32_t v = folded[0] > folded[1] ? folded[0] : folded[1];
    v = dpp_max_step<0xB1>(v);       // lane ^ 1
    v = dpp_max_step<0x4E>(v);       // lane ^ 2
    v = dpp_max_step<0x141>(v);      // mirrored in 8 lanes
    v = dpp_max_step<0x140>(v);      // mirrored in 16 lanes
    v = dpp_max_step<0x142>(v);      // lane 15 of a row into the next row: rows 1 and 3 hold the maxima
    a = (uint32_t)__builtin_amdgcn_readlane((int)v, 31);
    b = (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
// RK = registers whose 64 * RK entries cover at least k: their smallest score bounds the K-th largest from below (k entries are at
// least that large), the largest score of the list bounds it from above, and tau shares the leading bits the two bounds
// share - the search starts below them.  A padding entry (key 0) among those registers just gives the bound 0.
// Ends at the first tau that at most `cap` keys reach, or at the exact K-th largest score.  LOW: low bits that every score of the
// list shares with its sign (those a 16-bit type does not have); ties are common there and would run the search through them.
template <int R, int RK, int LOW>
__device__ inline uint32_t selecting_score(const uint64_t (&key)[R], int k, int cap) {
    uint32_t hi = 0u, lo_inv = 0u;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t s = (uint32_t)(key[r] >> 32);
        hi = hi > s ? hi : s;
        if (r < RK) lo_inv = lo_inv > ~s ? lo_inv : ~s;        // max of the complements = complement of the min
    }
    wave_max_two_u32(hi, lo_inv);
    const uint32_t lo = ~lo_inv;
    const int bits = 32 - __builtin_clz((hi ^ lo) | 1u);         // low bits in which the bounds may differ
    uint32_t tau = bits >= 32 ? 0u : (hi >> bits) << bits;
    uint32_t step = 1u << (bits - 1);
    while (step >= 1u << LOW) {
        // on the scalar unit but for a compare per register, one branch per step
        const uint32_t trial = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tau | step));
        int count = 0;
#pragma unroll
        for (int r = 0; r < R; ++r)
            count += __builtin_popcountll(__builtin_amdgcn_ballot_w64((uint32_t)(key[r] >> 32) >= trial));
        tau = count >= k ? trial : tau;
        step = (uint32_t)(count - k) <= (uint32_t)(cap - k) ? 0u : step >> 1;
        asm("" : "+s"(step));                                    // one exit: the two conditions cost six instructions apart
    }
    if constexpr (LOW > 0) {                                     // make tau a score: the low bits of a negative one are ones
        if (!(tau >> 31)) tau |= (1u << LOW) - 1u;
    }
    return tau;
}

__device__ inline int lanes_below(uint64_t mask) {
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// The keys above tau, then those equal to it in list order, until k are taken.
template <int R>
__device__ inline void collect_exactly(const uint64_t (&key)[R], uint32_t tau, int k, int cap, uint64_t* slots, int lane) {
    int base = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool above = (uint32_t)(key[r] >> 32) > tau;
        const uint64_t m = __builtin_amdgcn_ballot_w64(above);
        if (above) slots[base + lanes_below(m)] = key[r];
        base += __builtin_popcountll(m);
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const bool equal = (uint32_t)(key[r] >> 32) == tau;
        const uint64_t m = __builtin_amdgcn_ballot_w64(equal);
        const int pos = base + lanes_below(m);
        if (equal && pos < k) slots[pos] = key[r];
        base += __builtin_popcountll(m);
    }
    for (int p = k + lane; p < cap; p += kWave) slots[p] = 0ull;
}

// The registers' lanes whose score reaches tau, and how many they are.
template <int R>
__device__ inline int lanes_reaching(const uint64_t (&key)[R], uint32_t tau, uint64_t (&m)[R]) {
    int total = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        m[r] = __builtin_amdgcn_ballot_w64((uint32_t)(key[r] >> 32) >= tau);
        total += __builtin_popcountll(m[r]);
    }
    return total;
}

// At least k of the list's keys, all that reach a common score (or exactly k of them), into slots[0 .. cap), the rest of them 0;
// cap wave-private LDS entries.  n: keys in the list; unused entries hold key 0 (below every score).
// REUSE: seen is a score that selected from a list of this kind before (0: none yet; 1 where n <= cap), replaced when another had
// to be searched for.  It stays in a vector register: the scalar registers of eight waves are all taken, and on them it cost 2 us of 25.
template <int R, int RK, int LOW, bool REUSE>
__device__ inline void collect_top(const uint64_t (&key)[R], int n, int k, int cap, uint64_t* slots, int lane, uint32_t& seen) {
    uint64_t m[R];
    uint32_t tau;
    int total;
    if constexpr (REUSE) {
        tau = seen;
        total = lanes_reaching<R>(key, tau, m);
        if (n > cap && (uint32_t)(total - k) > (uint32_t)(cap - k)) {
            tau = selecting_score<R, RK, LOW>(key, k, cap);
            total = lanes_reaching<R>(key, tau, m);
            seen = tau;
            asm("" : "+v"(seen));
        }
    } else {
        tau = n <= cap ? 1u : selecting_score<R, RK, LOW>(key, k, cap);
        total = lanes_reaching<R>(key, tau, m);
    }
    if (total > cap) {                    // more ties with the k-th score than there are slots
        collect_exactly<R>(key, tau, k, cap, slots, lane);
        return;
    }
    int base = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        if ((uint32_t)(key[r] >> 32) >= tau) slots[base + lanes_below(m[r])] = key[r];
        base += __builtin_popcountll(m[r]);
    }
    for (int p = base + lane; p < cap; p += kWave) slots[p] = 0ull;
}

// The network for lists whose indexes fit 20 bits: a key is the score's 32 bits and those 20 as the mantissa of a positive normal
// double, (hi, lo).  In a layer the lanes that keep the smaller key hold theirs with the sign set; then both lanes of a pair keep
// max(mine, -other): one v_max_f64 and one XOR of the signs into the next layer's, where 64-bit integers take a compare, a scalar XOR
// with the lane mask and two selects that wait for it.  us, integers | doubles: 32768 tokens, 128 keys, K = 16 22.4 | 20.3, 64 52.3 |
// 46.6, 512 keys, K = 16 35.0 | 33.7, 100 107 | 95.5, 128 138 | 126; 4096 tokens, 128 keys, K = 64 10.9 | 9.9.
template <int RK> constexpr int sign_bit(int J) {           // lane bit whose set lanes hold negated keys in layer J; -1: none
    int b = -1;
    for (int l = J / RK; l > 0; l >>= 1) ++b;
    return b;
}
template <int FROM, int TO> __device__ inline void turn_sign(uint32_t& hi, int lane) {
    if constexpr (FROM != TO) {
        uint32_t m = 0u;
        if constexpr (FROM >= 0) m ^= (uint32_t)lane << (31 - FROM);
        if constexpr (TO >= 0) m ^= (uint32_t)lane << (31 - TO);
        hi ^= m & 0x80000000u;
    }
}
template <int RK, int J, int X, int FROM>
__device__ inline void signed_layer(uint32_t (&hi)[RK], uint32_t (&lo)[RK], int lane) {
    constexpr int TO = sign_bit<RK>(J);
#pragma unroll
    for (int r = 0; r < RK; ++r) turn_sign<FROM, TO>(hi[r], lane);
    auto value = [&](uint32_t h, uint32_t l) { return __builtin_bit_cast(double, ((uint64_t)h << 32) | l); };
    double w[RK];
#pragma unroll
    for (int r = 0; r < RK; ++r) {
        const double a = value(hi[r], lo[r]);
        if constexpr (X < RK) {
            const double b = value(hi[r ^ X], lo[r ^ X]);
            if ((r & J) == 0) asm("v_max_f64 %0, %1, %2" : "=v"(w[r]) : "v"(a), "v"(b));
            else asm("v_min_f64 %0, %1, %2" : "=v"(w[r]) : "v"(a), "v"(b));
        } else {
            const double b = value(xor_lane_u32(hi[r ^ (X % RK)], X / RK, lane), xor_lane_u32(lo[r ^ (X % RK)], X / RK, lane));
            asm("v_max_f64 %0, %1, -%2" : "=v"(w[r]) : "v"(a), "v"(b));
        }
    }
#pragma unroll
    for (int r = 0; r < RK; ++r) {
        const uint64_t u = __builtin_bit_cast(uint64_t, w[r]);
        hi[r] = (uint32_t)(u >> 32);
        lo[r] = (uint32_t)u;
    }
}
template <int RK, int J>
__device__ inline void signed_layers(uint32_t (&hi)[RK], uint32_t (&lo)[RK], int lane) {
    signed_layer<RK, J, J, sign_bit<RK>(2 * J)>(hi, lo, lane);
    if constexpr (J > 1) signed_layers<RK, J / 2>(hi, lo, lane);
}
template <int RK, int N, int K = 2>
__device__ inline void signed_blocks(uint32_t (&hi)[RK], uint32_t (&lo)[RK], int lane) {
    signed_layer<RK, K / 2, K - 1, K == 2 ? -1 : sign_bit<RK>(1)>(hi, lo, lane);
    if constexpr (K > 2) signed_layers<RK, K / 4>(hi, lo, lane);
    if constexpr (K < N) signed_blocks<RK, N, 2 * K>(hi, lo, lane);
    else
#pragma unroll
        for (int r = 0; r < RK; ++r) turn_sign<sign_bit<RK>(1), -1>(hi[r], lane);
}

// Indexes below 2^20.
template <int RK, bool SMALL>
__device__ inline void sort_slots(const uint64_t* slots, uint64_t (&best)[RK], int lane) {
    __builtin_amdgcn_wave_barrier();      // LDS operations of one wave complete in order; keep the compiler from moving them
#pragma unroll
    for (int r = 0; r < RK; ++r) best[r] = slots[lane * RK + r];
    __builtin_amdgcn_wave_barrier();
    uint32_t hi[RK], lo[RK];
#pragma unroll
    for (int r = 0; r < RK; ++r) {
        const uint32_t score = (uint32_t)(best[r] >> 32);
        hi[r] = __builtin_amdgcn_alignbit(0x400u, score, 12);
        lo[r] = (score << 20) | ((uint32_t)best[r] & 0xfffffu);
    }
    signed_blocks<RK, SMALL ? kWave / 2 : RK * kWave>(hi, lo, lane);
#pragma unroll
    for (int r = 0; r < RK; ++r) best[r] = ((uint64_t)__builtin_amdgcn_alignbit(hi[r], lo[r], 20) << 32) | (lo[r] | 0xfff00000u);
}

// The candidate pairs (rank in half 0) | (rank in half 1) << 8, listed by rank in half 0: the list depends on top_k only,
// so the host writes it and it travels as a kernel argument (at most 64 * 11 entries for top_k <= 128).
constexpr int kSelectMaxCand = 11 * kWave;
struct CandidateTable { uint16_t pair[kSelectMaxCand]; };

// ... and what a launch needs with it: top_k <= 128.
inline int candidate_table(int top_k, CandidateTable& table) {
    int c = 0;
    for (int i = 0; i < top_k; ++i)
        for (int j = 0; j < top_k / (i + 1); ++j) table.pair[c++] = (uint16_t)(i | (j << 8));
    const int used = c;
    for (; c < kSelectMaxCand; ++c) table.pair[c] = 0;
    return used;
}

template <int RK, int RC, int WAVES, bool PAIRED, int TOK = 1> struct SelectLds {
    static constexpr int kTokens = PAIRED ? WAVES / 2 : WAVES * TOK;
    uint64_t slot[WAVES][RK * kWave];
    float half_score[kTokens][2][RK * kWave];
    uint32_t half_index[kTokens][2][RK * kWave];
    uint16_t cand[RC * kWave];
};

// WAVES waves per workgroup, a token each; PAIRED: two waves per token (one launch round of few tokens), one per half, the first of
// them going on with the candidates.  TOK = 2 (SMALL): two tokens per wave, whose candidates one sort orders, 32 lanes each.
template <typename T, typename TG, int RK, int RH, int RC, bool FROM_LOGITS, bool SMALL, int WAVES, bool PAIRED, int TOK = 1, bool REUSE = false>
__device__ __forceinline__ void router_select_tokens(
    const T* __restrict__ lp, int64_t num_tokens, int nk, int top_k, int num_cand, T* __restrict__ scores,
    int64_t* __restrict__ indices, TG* __restrict__ gates, int norm_topk_prob, uint32_t* __restrict__ row_offsets,
    uint32_t row_bytes, const CandidateTable& table, SelectLds<RK, RC, WAVES, PAIRED, TOK>& lds, int block, int blocks) {
    constexpr int KP = RK * kWave;
    constexpr int LOW = sizeof(T) == 4 ? 0 : __is_same(T, bf16_t) ? 16 : 13;      // fp32 bits below the type's mantissa
    constexpr int CAP = SMALL ? kWave / 2 : KP;
    static_assert(RC * kWave <= kSelectMaxCand, "candidate table");
    static_assert(!SMALL || RK == 1, "one key per lane");
    static_assert(TOK == 1 || (TOK == 2 && SMALL && !PAIRED), "32 lanes per token");
    constexpr int TOKENS = SelectLds<RK, RC, WAVES, PAIRED, TOK>::kTokens;
    auto& cand = lds.cand;
    auto& half_score = lds.half_score;
    auto& half_index = lds.half_index;
    auto& slot = lds.slot;

    for (int i = (int)threadIdx.x; i < RC * kWave; i += (int)blockDim.x) cand[i] = table.pair[i];
    __syncthreads();
    const int lane = lane_id();
    const int wave = (int)(threadIdx.x >> 6);
    const int mine = PAIRED ? wave >> 1 : wave * TOK;    // the wave's (first) token of the workgroup
    const int64_t tokens_total = (int64_t)blocks * TOKENS;
    uint32_t seen[3] = {nk <= CAP ? 1u : 0u, nk <= CAP ? 1u : 0u, num_cand <= CAP ? 1u : 0u};   // half 0, half 1, candidates
    if constexpr (REUSE) asm("" : "+v"(seen[0]), "+v"(seen[1]), "+v"(seen[2]));

    // PAIRED: one round; else nothing below synchronises across waves
    for (int64_t first = (int64_t)block * TOKENS + mine; PAIRED || first < num_tokens; first += tokens_total) {
        const bool both = TOK == 2 && first + 1 < num_tokens;
#pragma unroll
        for (int t = 0; t < TOK; ++t) {
            const int64_t token = first + t;
            if (t == 1 && !both) break;
#pragma unroll
            for (int h = PAIRED ? __builtin_amdgcn_readfirstlane(wave & 1) : 0; h < 2; ++h) {
                if (PAIRED && token >= num_tokens) break;
                const T* row = FROM_LOGITS ? lp + (token * 2 + h) * nk : lp + ((int64_t)h * num_tokens + token) * nk;
                float v[RH];
#pragma unroll
                for (int r = 0; r < RH; ++r) {
                    const int p = r * kWave + lane;
                    v[r] = p < nk ? Elem<T>::to_f32(row[p]) : 0.0f;
                }
                float shift = 0.0f, lse = 0.0f;
                if (FROM_LOGITS) {
                    float mx = -INFINITY;
#pragma unroll
                    for (int r = 0; r < RH; ++r)
                        if (r * kWave + lane < nk) mx = fmaxf(mx, v[r]);
                    mx = wave_max(mx);
                    float se = 0.0f;
#pragma unroll
                    for (int r = 0; r < RH; ++r)
                        if (r * kWave + lane < nk) se += expf(v[r] - mx);
                    shift = mx;
                    lse = logf(wave_sum(se));
                }
                uint64_t key[RH];
#pragma unroll
                for (int r = 0; r < RH; ++r) {
                    const int p = r * kWave + lane;
                    key[r] = p < nk ? make_key(FROM_LOGITS ? (v[r] - shift) - lse : v[r], (uint32_t)p) : 0ull;
                }
                // the candidates look up ranks below top_k (entries past nk stay key 0)
                collect_top<RH, RK, FROM_LOGITS ? 0 : LOW, REUSE>(key, nk, top_k < nk ? top_k : nk, CAP, slot[wave] + (SMALL && !PAIRED ? h * CAP : 0), lane, seen[h]);
                if (REUSE && h == 0 && seen[1] == 0u) seen[1] = seen[0];
                if (!SMALL || PAIRED || h == 1) {
                    uint64_t best[RK];
                    sort_slots<RK, SMALL>(slot[wave], best, lane);
#pragma unroll
                    for (int r = 0; r < RK; ++r) {
                        const int which = SMALL && !PAIRED ? lane / CAP : h, rank = SMALL && !PAIRED ? lane % CAP : lane * RK + r;
                        half_score[mine + t][which][rank] = key_score(best[r]);
                        half_index[mine + t][which][rank] = key_index(best[r]);
                    }
                }
                if (PAIRED) break;
            }
        }
        if (PAIRED) {
            __syncthreads();
            if ((wave & 1) != 0 || first >= num_tokens) return;
        }
        __builtin_amdgcn_wave_barrier();
        uint64_t ckey[TOK][RC];
        if (SMALL && !both && lane >= CAP) slot[wave][lane] = 0ull;        // the sort's other block
#pragma unroll
        for (int t = 0; t < TOK; ++t) {
            if (t == 1 && !both) break;
#pragma unroll
            for (int r = 0; r < RC; ++r) {
                const int c = r * kWave + lane;
                ckey[t][r] = 0ull;
                if (c < num_cand) {
                    const int ij = cand[c];
                    const int i = ij & 0xff, j = ij >> 8;
                    const float s = round_through<T>(half_score[mine + t][0][i] + half_score[mine + t][1][j]);
                    const uint32_t flat = half_index[mine + t][0][i] * (uint32_t)nk + half_index[mine + t][1][j];
                    ckey[t][r] = make_key(s, flat);
                }
            }
            collect_top<RC, RK, LOW, REUSE>(ckey[t], num_cand, top_k, CAP, slot[wave] + t * CAP, lane, seen[2]);
        }
        uint64_t best[RK];
        sort_slots<RK, SMALL>(slot[wave], best, lane);
#pragma unroll
        for (int t = 0; t < TOK; ++t) {
            if (t == 1 && !both) break;
            // a tie across the cut: the first candidates in list order among the equal sums are the ones to keep
            const uint32_t cut = (uint32_t)(key_at<RK>(best, t * CAP + top_k - 1) >> 32);
            if (top_k < CAP && cut == (uint32_t)(key_at<RK>(best, t * CAP + top_k) >> 32)) {
                collect_exactly<RC>(ckey[t], cut, top_k, CAP, slot[wave] + t * CAP, lane);
                sort_slots<RK, SMALL>(slot[wave], best, lane);
            }
        }
        const int64_t token = TOK == 2 ? first + lane / CAP : first;
        const int rank = TOK == 2 ? lane % CAP : lane * RK;
        const int kept = TOK == 2 && lane >= CAP && !both ? 0 : top_k;
        float e[RK];
        float total = 0.0f;
#pragma unroll
        for (int r = 0; r < RK; ++r) {
            e[r] = rank + r < kept ? expf(key_score(best[r])) : 0.0f;
            total += e[r];
        }
        if (gates != nullptr && norm_topk_prob) total = TOK == 2 ? half_wave_sum(total) : wave_sum(total);
#pragma unroll
        for (int r = 0; r < RK; ++r) {
            const int p = rank + r;
            if (p < kept) {
                const int64_t o = token * top_k + p;
                scores[o] = Elem<T>::from_f32(key_score(best[r]));
                indices[o] = (int64_t)key_index(best[r]);
                if (row_offsets != nullptr) row_offsets[o] = key_index(best[r]) * row_bytes;
                if (gates != nullptr) gates[o] = Elem<TG>::from_f32(norm_topk_prob ? e[r] / total : e[r]);
            }
        }
        if (PAIRED) break;
    }
}

}  // namespace
}  // namespace fmoe
