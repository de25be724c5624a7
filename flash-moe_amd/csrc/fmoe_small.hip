// The FlashMoE block for a few tokens (a generation step, a short prompt), gfx950: stages that do not depend on each other share a
// launch, because each of them is bound by its own latency (4 to 9 us for work that the memory would deliver in 1 to 4) or leaves compute
// units idle.  The MLP's product is dispatched first, but for fp32 down products on the k-splitting tiles, which the selections precede
// (kSelectFirst).
//   gate_and_up_kernel       logits = BatchNorm(x) Wr^T   beside   act = silu(x Wg^T) * (x Wu^T)
//   select_and_down_kernel   product-key selection and gates   beside   the fp32 sums of act Wd^T
//   expert_token_kernel (fmoe_expert.hip)   the routed experts, plus those sums -> out
// README block in bf16, evaluation mode: 8 tokens 39.0 -> 23.6 us, 64 tokens 42.6 -> 25.6.
#include "fmoe_common.h"
#include "fmoe_gate.h"
#include "fmoe_gemm.h"
#include "fmoe_gemm256.h"
#include "fmoe_select.h"

namespace fmoe {
namespace {

static_assert(kGateWaves == kSplitWaves, "one workgroup size");

// How a product is cut into workgroups: the k-splitting tiles (16 x 16, 32 x 32), or tiles of the LDS pipeline on four waves
// instead of eight, with as many stages as let two workgroups share a compute unit (all workgroups of a launch hold the same LDS).
enum Cut { kCutSplit16, kCutSplit32, kCut64, kCut64x128, kCut128, kCut256, kCutNone };
template <int CUT> struct CutShape {
    static constexpr bool kDma = CUT >= kCut64;
    static constexpr int BM = CUT == kCut256 ? 256 : (CUT == kCut128 ? 128 : 64), BN = CUT == kCut256 ? 256 : (CUT == kCut64 ? 64 : 128);
    static constexpr int kStages = CUT >= kCut128 ? 2 : (CUT == kCut64x128 ? 3 : 4), kWavesN = CUT == kCut256 ? 4 : 2;
    static constexpr int MT = CUT == kCutSplit32 ? 2 : 1;
};
// The memory of a launch: the stages of its pipeline tiles, or what the larger of its two kinds of work exchanges sums in.
template <typename T, int CUT, int EPI, int BESIDE> __device__ __forceinline__ char* launch_lds() {
    using S = CutShape<CUT>;
    if constexpr (S::kDma) {
        constexpr int kElems = (S::BM + S::BN) * kStageK<T> * S::kStages;
        static_assert(BESIDE <= kElems * (int)sizeof(T), "the stages have room for it");
        return reinterpret_cast<char*>(DmaLds<T, kElems>::at());
    } else {
        constexpr int kProduct = kSplitLds<S::MT, S::MT, EPI>;
        __shared__ __attribute__((aligned(16))) char memory[kProduct > BESIDE ? kProduct : BESIDE];
        return memory;
    }
}

// Waves of a workgroup.  The pipeline's tiles use four.  With few gate tiles, or in fp32 (whose gate product is bound by the matrix
// pipes), the gate's eight matter more, and the tile's other four end at once; else, and with the registers of a 128 x 128 tile, the
// four more would keep a second tile off the compute unit.
template <typename T, int CUT, int GT> constexpr int kGateUpWaves = (CutShape<CUT>::kDma && CUT != kCut256 && GT == 2 && sizeof(T) == 2) || CUT == kCut128 ? 4 : kSplitWaves;
template <int CUT> constexpr int kSelectDownWaves = CutShape<CUT>::kDma ? 4 : kSplitWaves;

struct Product { int cut, tiles_m, tiles_n, blocks, slices; };     // blocks: workgroups of a slice of k, whole rounds of XCDs

template <typename T, int CUT, int EPI>
__device__ __forceinline__ void product_tiles(const T* A, const T* B0, const T* B1, T* C, const T* R, int M, int N, int K, const Product& p,
                                              int xcds, int block, char* lds) {
    using S = CutShape<CUT>;
    if constexpr (S::kDma) {
        if (threadIdx.x >= 2 * S::kWavesN * kWave) return;          // whole waves; the barriers of the tile count those that are left
        if constexpr (CUT == kCut256 && sizeof(T) == 2 && EPI == kEpiSwiGLU)
            gemm_wide_tiles<T, EPI, true>(A, B0, B1, C, R, M, N, K, p.tiles_m, p.tiles_n, xcds, block, p.blocks);
        else
            gemm_dma_tiles<T, S::BM, S::BN, 2, S::kWavesN, kStageK<T>, S::kStages, EPI, kTileAhead<T, S::BN, EPI>, kTileFrag<T, S::BN, EPI>, true>(
                A, B0, B1, C, R, M, N, K, p.tiles_m, p.tiles_n, xcds, block, p.blocks);
    } else {
        gemm_splitk_tile<T, S::MT, S::MT, EPI>(A, B0, B1, C, R, M, N, K, p.tiles_m, p.tiles_m * p.tiles_n, xcds, block % p.blocks, p.blocks,
                                               lds, block / p.blocks, p.slices);
    }
}

template <typename T, int CUT, int GT>
__global__ __launch_bounds__((kGateUpWaves<T, CUT, GT> * kWave)) void gate_and_up_kernel(
    const T* __restrict__ x, const T* __restrict__ gate_w, GateStats st, float* __restrict__ logits32, T* __restrict__ logits, int M, int N,
    int H, int gate_tiles_m, int gate_tiles_n, const T* __restrict__ wg, const T* __restrict__ wu, T* __restrict__ act,
    const T* __restrict__ products, int I, const Product up, int xcds) {
    char* lds = launch_lds<T, CUT, kEpiSwiGLU, kGateLds<GT, GT>>();
    extern __shared__ __attribute__((aligned(16))) float stats[];
    const int block = (int)blockIdx.x;
    if (block >= up.blocks)
        router_gate_splitk_tile<T, GT, GT, true, kGateUpWaves<T, CUT, GT>>(x, gate_w, st, logits32, logits, M, N, H, gate_tiles_m, gate_tiles_n, 0, xcds, lds, stats,
                                                 block - up.blocks, (int)gridDim.x - up.blocks);
    else
        product_tiles<T, CUT, kEpiSwiGLU>(x, wg, wu, act, products, M, I, H, up, xcds, block, lds);
}

template <typename T, int CUT, int RH, int RC, bool SMALL>
__global__ __launch_bounds__(kSelectDownWaves<CUT> * kWave) void select_and_down_kernel(
    const float* __restrict__ logits32, int64_t num_tokens, int nk, int top_k, int num_cand, float* __restrict__ scores,
    int64_t* __restrict__ indices, T* __restrict__ gates, int norm_topk_prob, const T* __restrict__ act, const T* __restrict__ wd,
    float* __restrict__ sums, int M, int H, int I, const Product down, int xcds, const CandidateTable table) {
    constexpr int kWaves = kSelectDownWaves<CUT>;
    using Lds = SelectLds<1, RC, kWaves, true>;
    char* lds = launch_lds<T, CUT, kEpiPart, (int)sizeof(Lds)>();
    // fp32 products on the k-splitting tiles keep their compute unit's matrix pipes busy for the whole launch: the selections, chains of
    // latency, start before them and end beside them.  The block, us, product | selections first: 512 tokens, 256 -> 1024 31.4 | 29.1;
    // 1000, 256 -> 1024 35.7 | 33.4; 400, 512 -> 1024 34.6 | 32.7.  On larger tiles, more of which wait for a place, and in 16 bits the
    // product goes first: fp32, 1500 tokens, 512 -> 1360 90.8 | 110.7; fp16, 999 tokens, 1000 -> 2664 57.8 | 62.1.
    constexpr bool kSelectFirst = sizeof(T) == 4 && CUT < kCut64;
    const int down_blocks = down.blocks * down.slices, select_blocks = (int)gridDim.x - down_blocks;
    const int block = (int)blockIdx.x - (kSelectFirst ? select_blocks : 0);         // of the product; the others are selections
    if (block < 0 || block >= down_blocks)
        router_select_tokens<float, T, 1, RH, RC, true, SMALL, kWaves, true>(
            logits32, num_tokens, nk, top_k, num_cand, scores, indices, gates, norm_topk_prob, nullptr, 0u, table,
            *reinterpret_cast<Lds*>(lds), kSelectFirst ? (int)blockIdx.x : block - down_blocks, select_blocks);
    else
        product_tiles<T, CUT, kEpiPart>(act, wd, nullptr, reinterpret_cast<T*>(sums), nullptr, M, H, I, down, xcds, block, lds);
}

inline int whole(int64_t blocks, int xcds) { return (int)((blocks + xcds - 1) / xcds * xcds); }

// The tile the product would take on its own (choose_tile), as far as it leaves registers for a second kind of work.
template <typename T, int EPI> Product plan_product(int M, int N) {
    int tiles = 0;
    const int cus = chip_info().cus;
    Product p = {kCutNone, 0, 0, 0, 1};
    const TileShape shape = choose_tile<T, EPI>(M, N, tiles);
    switch (shape) {
        case kSplit16: p.cut = kCutSplit16; break;
        case kSplit16x32: p.cut = M <= 16 ? kCutSplit16 : kCutSplit32; break;
        case kSplit32: p.cut = kCutSplit32; break;
        case kTile64: p.cut = kCut64; break;
        case kTile64x128: p.cut = kCut64x128; break;
        case kTile128:
            if (EPI == kEpiPart) return p;      // gains nothing: without four stages of its own it is slower by what the selection takes
            p.cut = kCut128;
            break;
        default:
            // a 256 x 256 tile fills its compute unit: only those without one in the last round have room for the gate
            if (EPI == kEpiPart || sizeof(T) == 4 || (cus - tiles % cus) % cus < cus / 4) return p;
            p.cut = kCut256;
    }
    if (EPI == kEpiSwiGLU && sizeof(T) == 4 && M <= 256 && p.cut > kCutSplit32) p.cut = M <= 16 ? kCutSplit16 : kCutSplit32;
    const int rows = p.cut == kCutSplit16 ? 16 : (p.cut == kCutSplit32 ? 32 : (p.cut == kCut256 ? 256 : (p.cut == kCut128 ? 128 : 64)));
    const int cols = p.cut == kCutSplit16 ? 16 : (p.cut == kCutSplit32 ? 32 : (p.cut == kCut64 ? 64 : (p.cut == kCut256 ? 256 : 128)) / (EPI == kEpiSwiGLU ? 2 : 1));
    p.tiles_m = (M + rows - 1) / rows;
    p.tiles_n = (N + cols - 1) / cols;
    const int64_t n = (int64_t)p.tiles_m * p.tiles_n, resident = p.cut == kCut256 ? cus : 2 * cus;
    p.blocks = whole(p.cut >= kCut64 && n > resident ? resident : n, chip_info().xcds);
    return p;
}

// Few tokens: 16 x 16 tiles while they leave compute units free, else 32 x 32.  A compute unit receives about 60 GB/s, so a
// workgroup that would read more than 256 KB leaves parts of k to others as long as there are compute units without a tile; fp32, whose
// matrix pipes take as long, from 128 KB on beyond 256 tokens (300 tokens, 1024 -> 256: the block 24.5 -> 21.1 us; 8 tokens, 4096 -> 1024
// would take 33.3 -> 35.4).
template <typename T> Product plan_down(int M, int H, int I) {
    if (M > 256) {
        const Product whole = plan_product<T, kEpiPart>(M, H);
        if (sizeof(T) == 2 || whole.cut > kCutSplit32) return whole;
    }
    const int cus = chip_info().cus;
    Product p;
    p.cut = ((M + 15) / 16) * ((H + 15) / 16) < cus ? kCutSplit16 : kCutSplit32;
    const int b = p.cut == kCutSplit16 ? 16 : 32;
    p.tiles_m = (M + b - 1) / b;
    p.tiles_n = (H + b - 1) / b;
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n, bytes = 2 * b * (int64_t)I * (int64_t)sizeof(T);
    const int64_t most = M > 256 ? 128 << 10 : 256 << 10, wanted = (bytes + most - 1) / most, room = cus / tiles;
    p.slices = (int)(wanted < room ? wanted : room);
    if (p.slices > kSmallMaxSlices) p.slices = kSmallMaxSlices;
    if (p.slices < 1) p.slices = 1;
    p.blocks = whole(tiles, chip_info().xcds);
    return p;
}

template <typename T>
int gate_and_up(const void* x, const void* gate_w, const GateStats& st, float* logits32, void* logits, int M, int N, int H, const void* wg,
                const void* wu, void* act, const void* products, int I, hipStream_t stream) {
    const int xcds = chip_info().xcds;
    const Product up = plan_product<T, kEpiSwiGLU>(M, I);
    const int gt = gate_tiles(M, N, 1, 1) <= chip_info().cus ? 1 : 2;
    const int gm = (M + 16 * gt - 1) / (16 * gt), gn = (N + 16 * gt - 1) / (16 * gt);
    const dim3 grid((unsigned)(up.blocks + whole((int64_t)gm * gn, xcds)));
    const size_t lds = (size_t)((H + 63) / 64) * 64 * 8;
#define FMOE_GO(CUT)                                                                                                                   \
    do {                                                                                                                               \
        if (gt == 1)                                                                                                                   \
            hipLaunchKernelGGL((gate_and_up_kernel<T, CUT, 1>), grid, dim3(kGateUpWaves<T, CUT, 1> * kWave), lds, stream, (const T*)x, (const T*)gate_w, st, logits32, \
                               (T*)logits, M, N, H, gm, gn, (const T*)wg, (const T*)wu, (T*)act, (const T*)products, I, up, xcds);     \
        else                                                                                                                           \
            hipLaunchKernelGGL((gate_and_up_kernel<T, CUT, 2>), grid, dim3(kGateUpWaves<T, CUT, 2> * kWave), lds, stream, (const T*)x, (const T*)gate_w, st, logits32, \
                               (T*)logits, M, N, H, gm, gn, (const T*)wg, (const T*)wu, (T*)act, (const T*)products, I, up, xcds);     \
    } while (0)
    switch (up.cut) {
        case kCutSplit16: FMOE_GO(kCutSplit16); break;
        case kCutSplit32: FMOE_GO(kCutSplit32); break;
        case kCut64: FMOE_GO(kCut64); break;
        case kCut64x128: FMOE_GO(kCut64x128); break;
        case kCut128: FMOE_GO(kCut128); break;
        default: if constexpr (sizeof(T) == 2) FMOE_GO(kCut256); break;
    }
#undef FMOE_GO
    FMOE_CHECK_LAUNCH("fmoe_block(gate and up)");
    return FMOE_OK;
}

template <typename T>
int select_and_down(const float* logits32, int T_, int nk, int K, float* scores, int64_t* indices, void* gates, int norm, const void* act,
                    const void* wd, float* sums, int H, int I, const Product& down, hipStream_t stream) {
    const int xcds = chip_info().xcds;
    CandidateTable table;
    const int num_cand = candidate_table(K, table);
    const int per_block = down.cut >= kCut64 ? 2 : 4;        // tokens: two waves each
    const dim3 grid((unsigned)(down.blocks * down.slices + (T_ + per_block - 1) / per_block)), block(down.cut >= kCut64 ? 256 : 512);
#define FMOE_GO(CUT, RH, RC, SMALL)                                                                                                    \
    hipLaunchKernelGGL((select_and_down_kernel<T, CUT, RH, RC, SMALL>), grid, block, 0, stream, logits32, T_, nk, K, num_cand, scores,  \
                       indices, (T*)gates, norm, (const T*)act, (const T*)wd, sums, T_, H, I, down, xcds, table)
#define FMOE_FEW(CUT)                                \
    do {                                             \
        if (K <= 32) {                               \
            if (nk <= 128) FMOE_GO(CUT, 2, 2, true); \
            else FMOE_GO(CUT, 8, 2, true);           \
        } else {                                     \
            if (nk <= 128) FMOE_GO(CUT, 2, 5, false); \
            else FMOE_GO(CUT, 8, 5, false);          \
        }                                            \
    } while (0)
#define FMOE_MORE(CUT)                          \
    do {                                        \
        if (K <= 32) FMOE_GO(CUT, 4, 2, true);  \
        else FMOE_GO(CUT, 4, 5, false);         \
    } while (0)
    switch (down.cut) {
        case kCutSplit16: FMOE_FEW(kCutSplit16); break;
        case kCutSplit32: FMOE_FEW(kCutSplit32); break;
        case kCut64: FMOE_MORE(kCut64); break;
        default: FMOE_MORE(kCut64x128); break;
    }
#undef FMOE_MORE
#undef FMOE_FEW
#undef FMOE_GO
    FMOE_CHECK_LAUNCH("fmoe_block(select and down)");
    return FMOE_OK;
}

bool gate_beside_up(int64_t T_, int H, int I, int nk, int dtype) {
    if (T_ > kSmallMaxTokens || H > kGateStagedK || (dtype == FMOE_F32 && I % 4 != 0) || nk > 32767) return false;
    if (gate_tiles((int)T_, 2 * nk, 2, 2) > 2 * chip_info().cus || !gate_splitk_pays((int)T_, 2 * nk, dtype)) return false;
    switch (dtype) {
        case FMOE_F32: return plan_product<float, kEpiSwiGLU>((int)T_, I).cut != kCutNone;
        default: return plan_product<bf16_t, kEpiSwiGLU>((int)T_, I).cut != kCutNone;
    }
}

Product down_plan(int64_t T_, int H, int I, int dtype) { return dtype == FMOE_F32 ? plan_down<float>((int)T_, H, I) : plan_down<bf16_t>((int)T_, H, I); }

bool select_beside_down(int64_t T_, int H, int I, int nk, int64_t E, int K, int dtype) {
    if (T_ > kSmallMaxTokens || H > 2048 || (dtype == FMOE_F32 && I % 4 != 0) || K <= 0 || K > 64 || nk > 512) return false;
    // up to 256 tokens the down product is about one round of 32 x 32 tiles (128 tokens of 2048 columns: 69 us for 71 as five
    // launches; 200 tokens would take 89 for 83)
    if (T_ <= 256 && 2 * ((T_ + 31) / 32) * ((H + 31) / 32) > 3 * (int64_t)chip_info().cus) return false;
    const Product down = down_plan(T_, H, I, dtype);
    return down.cut != kCutNone && nk <= (down.cut >= kCut64 ? 256 : 512) && expert_rows_chosen(T_, H, E, K, dtype);
}

}  // namespace

SmallPlan plan_small(int64_t T_, int H, int I, int nk, int64_t E, int K, int dtype) {
    SmallPlan p;
    p.gate_and_up = gate_beside_up(T_, H, I, nk, dtype) && router_topk_supported(nk, K);
    p.select_and_down = select_beside_down(T_, H, I, nk, E, K, dtype);
    p.sums_bytes = p.select_and_down ? (size_t)down_plan(T_, H, I, dtype).slices * (size_t)T_ * (size_t)H * 4 : 0;
    return p;
}

int small_gate_and_up(const void* x, const void* gate_proj_w, const void* up_proj_w, const void* router_gate_w, void* running_mean,
                      void* running_var, int64_t* num_batches_tracked, int stats_dtype, int training, float momentum, float eps,
                      int64_t num_tokens, int H, int I, int nk, int dtype, void* router_logits, float* logits32, void* act, void* products,
                      float* scratch, float* mean_rstd, hipStream_t s) {
    const int M = (int)num_tokens, N = 2 * nk;
    GateStats st = {};
    st.num_tokens = num_tokens;
    st.training = training;
    st.stats_dtype = stats_dtype;
    st.momentum = momentum;
    st.eps = eps;
    st.running_mean = running_mean;
    st.running_var = running_var;
    st.num_batches_tracked = num_batches_tracked;
    st.mean_rstd = mean_rstd;
    st.partial = scratch;
    if (training)
        if (int rc = router_block_stats(x, num_tokens, H, dtype, scratch, &st.row_blocks, &st.rows_per_block, s)) return rc;
    switch (dtype) {
        case FMOE_F32: return gate_and_up<float>(x, router_gate_w, st, logits32, router_logits, M, N, H, gate_proj_w, up_proj_w, act, products, I, s);
        case FMOE_BF16: return gate_and_up<bf16_t>(x, router_gate_w, st, logits32, router_logits, M, N, H, gate_proj_w, up_proj_w, act, products, I, s);
        default: return gate_and_up<f16_t>(x, router_gate_w, st, logits32, router_logits, M, N, H, gate_proj_w, up_proj_w, act, products, I, s);
    }
}

int small_select_down_experts(const void* x, const void* down_proj_w, const void* down_embed, const void* up_embed, int64_t num_tokens, int H,
                              int I, int64_t E, int nk, int K, int dtype, int norm_topk_prob, void* out, const float* logits32,
                              float* scores, int64_t* indices, void* gates, const void* act, float* sums, hipStream_t s) {
    const int T_ = (int)num_tokens;
    const Product down = down_plan(num_tokens, H, I, dtype);
    int rc;
    switch (dtype) {
        case FMOE_F32: rc = select_and_down<float>(logits32, T_, nk, K, scores, indices, gates, norm_topk_prob, act, down_proj_w, sums, H, I, down, s); break;
        case FMOE_BF16: rc = select_and_down<bf16_t>(logits32, T_, nk, K, scores, indices, gates, norm_topk_prob, act, down_proj_w, sums, H, I, down, s); break;
        default: rc = select_and_down<f16_t>(logits32, T_, nk, K, scores, indices, gates, norm_topk_prob, act, down_proj_w, sums, H, I, down, s); break;
    }
    if (rc) return rc;
    return expert_rows_added(x, down_embed, up_embed, indices, gates, num_tokens, H, E, K, dtype, sums, down.slices, out, s);
}

}  // namespace fmoe
