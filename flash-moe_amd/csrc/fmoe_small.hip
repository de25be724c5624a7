// The FlashMoE block for a few tokens in evaluation mode (a generation step), gfx950: three launches instead of five.
//   1. gate_and_up_kernel   logits = BatchNorm(x) Wr^T   beside   act = silu(x Wg^T) * (x Wu^T)
//   2. select_and_down_kernel   product-key selection and gates   beside   the fp32 sums of act Wd^T, k split over workgroups
//   3. expert_token_kernel (fmoe_expert.hip)   the routed experts, plus those sums -> out
// Each of the five is bound by its own latency (4 to 9 us for work that the memory would deliver in 1 to 4) and leaves most of
// the chip idle, so the two that do not depend on each other share a launch, the larger grid first.  README block in bf16: 8 tokens
// 39.0 -> 22.1 us, 64 tokens 42.6 -> 25.6, 256 tokens 53 -> 47; fp32, 64 tokens of 1024 columns 48 -> 32.
#include "fmoe_common.h"
#include "fmoe_gate.h"
#include "fmoe_gemm.h"
#include "fmoe_select.h"

namespace fmoe {
namespace {

static_assert(kGateWaves == kSplitWaves, "one workgroup size");
constexpr int kSmallThreads = kSplitWaves * kWave;

// How the gate/up product is cut: the k-splitting tiles, or the 64 x 64 tiles of the LDS pipeline (four of the waves; 16-bit).
enum UpTile { kUpSplit16, kUpSplit32, kUpDma64, kUpDma64Ragged };

template <typename T, int UP>
__global__ __launch_bounds__(kSmallThreads) void gate_and_up_kernel(
    const T* __restrict__ x, const T* __restrict__ gate_w, GateStats st, float* __restrict__ logits32, T* __restrict__ logits, int M, int N,
    int H, int gate_tiles_m, int gate_tiles_n, const T* __restrict__ wg, const T* __restrict__ wu, T* __restrict__ act, int I,
    int up_tiles_m, int up_tiles_n, int up_blocks, int xcds) {
    extern __shared__ __attribute__((aligned(16))) float stats[];
    const int block = (int)blockIdx.x;
    if (block >= up_blocks) {
        router_gate_splitk_tile<T, 1, 1, true>(x, gate_w, st, logits32, logits, M, N, H, gate_tiles_m, gate_tiles_n, 0, xcds, stats,
                                               block - up_blocks, (int)gridDim.x - up_blocks);
    } else if constexpr (UP == kUpSplit16 || UP == kUpSplit32) {
        constexpr int MT = UP == kUpSplit32 ? 2 : 1;
        gemm_splitk_tile<T, MT, MT, kEpiSwiGLU>(x, wg, wu, act, nullptr, M, I, H, up_tiles_m, up_tiles_m * up_tiles_n, xcds, block, up_blocks);
    } else if constexpr (sizeof(T) == 2) {
        if (threadIdx.x >= 256) return;          // whole waves; the barriers of the tile count those that are left
        gemm_dma_tiles<T, 64, 64, 2, 2, kStageK<T>, 4, kEpiSwiGLU, kSmallAhead<T>, kFragRows<T>, 1, UP == kUpDma64Ragged>(
            x, wg, wu, act, nullptr, M, I, H, up_tiles_m, up_tiles_n, xcds, block, up_blocks);
    }
}

template <typename T, int RH, int RC, bool SMALL, int MT>
__global__ __launch_bounds__(kSmallThreads) void select_and_down_kernel(
    const float* __restrict__ logits32, int64_t num_tokens, int nk, int top_k, int num_cand, float* __restrict__ scores,
    int64_t* __restrict__ indices, T* __restrict__ gates, int norm_topk_prob, const T* __restrict__ act, const T* __restrict__ wd,
    float* __restrict__ sums, int M, int H, int I, int tiles_m, int tiles, int slice_blocks, int slices, int xcds,
    const CandidateTable table) {
    const int block = (int)blockIdx.x, down_blocks = slice_blocks * slices;
    if (block >= down_blocks)
        router_select_tokens<float, T, 1, RH, RC, true, SMALL, kSplitWaves, true>(
            logits32, num_tokens, nk, top_k, num_cand, scores, indices, gates, norm_topk_prob, nullptr, 0u, table, block - down_blocks,
            (int)gridDim.x - down_blocks);
    else
        gemm_splitk_tile<T, MT, MT, kEpiPart>(act, wd, nullptr, reinterpret_cast<T*>(sums), nullptr, M, H, I, tiles_m, tiles, xcds,
                                              block % slice_blocks, slice_blocks, block / slice_blocks, slices);
}

struct DownPlan { int mt, tiles_m, tiles, slices; };
// 16 x 16 tiles while they leave compute units free, else 32 x 32.  A compute unit receives about 60 GB/s, so a workgroup that
// would read more than 256 KB leaves parts of k to others as long as there are compute units without a tile.
DownPlan plan_down(int64_t T_, int H, int I, int dtype) {
    DownPlan p;
    const int cus = chip_info().cus;
    p.mt = ((T_ + 15) / 16) * ((H + 15) / 16) < cus ? 1 : 2;
    const int b = 16 * p.mt;
    p.tiles_m = (int)((T_ + b - 1) / b);
    p.tiles = p.tiles_m * ((H + b - 1) / b);
    const int64_t bytes = 2 * b * (int64_t)I * (int64_t)dtype_size(dtype);
    const int64_t wanted = (bytes + (256 << 10) - 1) / (256 << 10), room = cus / p.tiles;
    p.slices = (int)(wanted < room ? wanted : room);
    if (p.slices > kSmallMaxSlices) p.slices = kSmallMaxSlices;
    if (p.slices < 1) p.slices = 1;
    return p;
}

inline int whole(int blocks, int xcds) { return (blocks + xcds - 1) / xcds * xcds; }

template <typename T>
int gate_and_up(const void* x, const void* gate_w, const GateStats& st, float* logits32, void* logits, int M, int N, int H, const void* wg,
                const void* wu, void* act, int I, hipStream_t stream) {
    const int xcds = chip_info().xcds;
    int tiles = 0;
    const TileShape shape = choose_tile<T, kEpiSwiGLU>(M, I, tiles);
    // fp32: 32 x 32 tiles where the rule would go beyond 16 rows; 16-bit: the pipeline's 64 x 64 tiles
    const UpTile up = shape == kSplit16 || (sizeof(T) == 4 && M <= 16) ? kUpSplit16
                      : sizeof(T) == 4                                 ? kUpSplit32
                      : H % kStageK<T> == 0 && I % 128 == 0            ? kUpDma64
                                                                       : kUpDma64Ragged;
    const int rows = up == kUpSplit16 ? 16 : (up == kUpSplit32 ? 32 : 64), cols = up == kUpSplit16 ? 16 : 32;
    const int up_m = (M + rows - 1) / rows, up_n = (I + cols - 1) / cols, up_blocks = whole(up_m * up_n, xcds);
    const int gm = (M + 15) / 16, gn = (N + 15) / 16;
    const dim3 grid((unsigned)(up_blocks + whole(gm * gn, xcds))), block(kSmallThreads);
    const size_t lds = (size_t)((H + 63) / 64) * 64 * 8;
#define FMOE_GO(UP)                                                                                                              \
    hipLaunchKernelGGL((gate_and_up_kernel<T, UP>), grid, block, lds, stream, (const T*)x, (const T*)gate_w, st, logits32, (T*)logits, \
                       M, N, H, gm, gn, (const T*)wg, (const T*)wu, (T*)act, I, up_m, up_n, up_blocks, xcds)
    switch (up) {
        case kUpSplit16: FMOE_GO(kUpSplit16); break;
        case kUpSplit32: if constexpr (sizeof(T) == 4) FMOE_GO(kUpSplit32); break;
        case kUpDma64: if constexpr (sizeof(T) == 2) FMOE_GO(kUpDma64); break;
        default: if constexpr (sizeof(T) == 2) FMOE_GO(kUpDma64Ragged); break;
    }
#undef FMOE_GO
    FMOE_CHECK_LAUNCH("fmoe_block(gate and up)");
    return FMOE_OK;
}

template <typename T>
int select_and_down(const float* logits32, int T_, int nk, int K, float* scores, int64_t* indices, void* gates, int norm, const void* act,
                    const void* wd, float* sums, int H, int I, const DownPlan& p, hipStream_t stream) {
    const int xcds = chip_info().xcds;
    CandidateTable table;
    const int num_cand = candidate_table(K, table);
    const int slice_blocks = whole(p.tiles, xcds), select_blocks = (T_ + kSplitWaves / 2 - 1) / (kSplitWaves / 2);
    const dim3 grid((unsigned)(slice_blocks * p.slices + select_blocks)), block(kSmallThreads);
#define FMOE_GO(RH, RC, SMALL)                                                                                                         \
    do {                                                                                                                               \
        if (p.mt == 1)                                                                                                                 \
            hipLaunchKernelGGL((select_and_down_kernel<T, RH, RC, SMALL, 1>), grid, block, 0, stream, logits32, T_, nk, K, num_cand,   \
                               scores, indices, (T*)gates, norm, (const T*)act, (const T*)wd, sums, T_, H, I, p.tiles_m, p.tiles,      \
                               slice_blocks, p.slices, xcds, table);                                                                   \
        else                                                                                                                           \
            hipLaunchKernelGGL((select_and_down_kernel<T, RH, RC, SMALL, 2>), grid, block, 0, stream, logits32, T_, nk, K, num_cand,   \
                               scores, indices, (T*)gates, norm, (const T*)act, (const T*)wd, sums, T_, H, I, p.tiles_m, p.tiles,      \
                               slice_blocks, p.slices, xcds, table);                                                                   \
    } while (0)
    if (K <= 32) {
        if (nk <= 128) FMOE_GO(2, 2, true);
        else FMOE_GO(8, 2, true);
    } else {
        if (nk <= 128) FMOE_GO(2, 5, false);
        else FMOE_GO(8, 5, false);
    }
#undef FMOE_GO
    FMOE_CHECK_LAUNCH("fmoe_block(select and down)");
    return FMOE_OK;
}

}  // namespace

// While every token has a compute unit for its experts and the down product is about one round of 32 x 32 tiles (128 tokens of 2048
// columns: 69 us for 71 as five launches; 200 tokens would take 89 for 83).
bool block_small_usable(int64_t T_, int H, int I, int nk, int64_t E, int K, int dtype) {
    return T_ <= kSmallMaxTokens && H <= 2048 && (int64_t)I * H < (1ll << 31) && (dtype != FMOE_F32 || I % 4 == 0) && K > 0 && K <= 64 &&
           nk <= 512 && 2 * ((T_ + 31) / 32) * ((H + 31) / 32) <= 3 * (int64_t)chip_info().cus && expert_rows_chosen(T_, H, E, K, dtype);
}

size_t block_small_sums_bytes(int64_t T_, int H, int I, int dtype) { return (size_t)plan_down(T_, H, I, dtype).slices * (size_t)T_ * (size_t)H * 4; }

int block_small_forward(const void* x, const void* gate_proj_w, const void* up_proj_w, const void* down_proj_w, const void* router_gate_w,
                        const void* down_embed, const void* up_embed, void* running_mean, void* running_var, int stats_dtype, float eps,
                        int64_t num_tokens, int H, int I, int64_t E, int nk, int K, int dtype, int norm_topk_prob, void* out,
                        void* router_logits, float* logits32, float* scores, int64_t* indices, void* gates, void* act, float* mean_rstd,
                        float* sums, hipStream_t s) {
    const int T_ = (int)num_tokens;
    GateStats st = {};
    st.num_tokens = num_tokens;
    st.stats_dtype = stats_dtype;
    st.eps = eps;
    st.running_mean = running_mean;
    st.running_var = running_var;
    st.mean_rstd = mean_rstd;
    const DownPlan p = plan_down(num_tokens, H, I, dtype);
    int rc;
    switch (dtype) {
        case FMOE_F32: rc = gate_and_up<float>(x, router_gate_w, st, logits32, router_logits, T_, 2 * nk, H, gate_proj_w, up_proj_w, act, I, s); break;
        case FMOE_BF16: rc = gate_and_up<bf16_t>(x, router_gate_w, st, logits32, router_logits, T_, 2 * nk, H, gate_proj_w, up_proj_w, act, I, s); break;
        default: rc = gate_and_up<f16_t>(x, router_gate_w, st, logits32, router_logits, T_, 2 * nk, H, gate_proj_w, up_proj_w, act, I, s); break;
    }
    if (rc) return rc;
    switch (dtype) {
        case FMOE_F32: rc = select_and_down<float>(logits32, T_, nk, K, scores, indices, gates, norm_topk_prob, act, down_proj_w, sums, H, I, p, s); break;
        case FMOE_BF16: rc = select_and_down<bf16_t>(logits32, T_, nk, K, scores, indices, gates, norm_topk_prob, act, down_proj_w, sums, H, I, p, s); break;
        default: rc = select_and_down<f16_t>(logits32, T_, nk, K, scores, indices, gates, norm_topk_prob, act, down_proj_w, sums, H, I, p, s); break;
    }
    if (rc) return rc;
    return expert_rows_added(x, down_embed, up_embed, indices, gates, num_tokens, H, E, K, dtype, sums, p.slices, out, s);
}

}  // namespace fmoe
