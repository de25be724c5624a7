// 256 x 256 tiles of C[M,N] = A B^T (and of the backward's A B and A^T B) in the 16-bit types for gfx950: eight waves in two groups of
// four that alternate, one group multiplying while the other fetches.
//
// What bounds such a tile: a compute unit's matrix pipes need 2048 cycles for a k-tile of 64, its LDS 1500 for the fragments.  With all
// eight waves doing the same thing at the same time (gemm_dma_tiles) the two add up in part: every wave waits for its first fragments
// while the pipes run dry, 2740 cycles per k-tile.  Here waves w and w + 4 share a SIMD and are half a step apart, held there by a
// barrier at each end of a step: one issues 16 matrix instructions (256 cycles of its SIMD) while the other reads six fragments and
// sends two DMA loads, and has them before the roles change.  A k-tile is four such steps, the four 64 x 32 quarters of a wave's tile.
// The quarters lie in LDS apart (four regions of 16 KB in each of two buffers), so a region is refilled as soon as both groups have read
// it, six to seven steps, almost two k-tiles, before its next use.  Operands are exchanged in the matrix instructions, which gives a
// lane consecutive columns: results leave in 16-byte stores where the 2-byte ones took 4 us per tile.
//
// us before and after, gate/up and down with residual, bf16: 4096 tokens of 1024 -> 4096 61.5 -> 54.7; 2048 of 4096 -> 16384 417 -> 369;
// 32768 of 2048 -> 8192 1683 -> 1517 and 894 -> 746; 8192 of 2048 -> 8192 414 -> 370 and 210 -> 187 (1.45 to 1.5 PFLOP/s, the library's
// plain products 1.45 to 1.6).  Measured and not taken: the first k-tile apart from the loop instead of zeroed accumulators (2 to 5 %
// longer), DMA loads ahead of the fragment reads (3 %), no wave priorities (within 1 %), groups half a step apart over the stores too
// (1 % shorter with 16 k-tiles, 1 % longer with 32 and more).
#pragma once

#include "fmoe_common.h"
#include "fmoe_gemm.h"
#include "fmoe_vec.h"

namespace fmoe {
namespace {

template <int N> struct Number { static constexpr int value = N; };
constexpr int kWide = 256, kWideK = 64, kWideThreads = 512;      // tile, k extent of a k-tile
constexpr int kWideLdsElements = 65536;                          // two buffers of four regions, 16-bit elements

// Position of tile t in the order each XCD walks: XCD x (workgroup id mod xcds) takes a contiguous run, eight tile-rows at a time.
__device__ __forceinline__ void wide_tile_at(int t, int num_tiles, int tiles_m, int tiles_n, int xcds, int& tm, int& tn) {
    t = xcd_run(t, num_tiles, xcds);
    constexpr int GM = 8;
    const int width = GM * tiles_n, group = t / width, first_m = group * GM;
    const int gsz = (tiles_m - first_m) < GM ? (tiles_m - first_m) : GM;
    tm = first_m + (t % width) % gsz;
    tn = (t % width) / gsz;
}

// TA, TB: the operand lies k-row by k-row (lda, ldb values apart).  segments: a second range of K values, in A further along the rows and
// in B1 (TB only).  SLICED: slice `slice` of `slices` of k, one tile per workgroup, its sums in fp32 to plane `slice` of C (kEpiPart).
// RAGGED: extents that are no multiples of the tile, of 64 k values or with an odd number of k-tiles; the rest of the operands arrives as
// zeros, by the descriptors' range checks or by an offset beyond all of them.  A scalar offset never reaches the end of its
// descriptor: the hardware subtracts it from the extent before it compares.
template <typename T, int EPI, bool RAGGED, bool SLICED = false, bool TA = false, bool TB = false>
__device__ __forceinline__ void gemm_wide_tiles(const T* __restrict__ A, const T* __restrict__ B0, const T* __restrict__ B1, T* __restrict__ C,
                                                const T* __restrict__ R, int M, int N, int K, int tiles_m, int tiles_n, int xcds, int block,
                                                int blocks, int slice = 0, int slices = 1, int lda = 0, int ldb = 0, int segments = 1) {
    static_assert(sizeof(T) == 2, "16-bit types");
    static_assert(EPI == kEpiSwiGLU || EPI == kEpiPlain || EPI == kEpiPart, "epilogues");
    static_assert(SLICED == (EPI == kEpiPart) && (!(TA || TB) || (TB && EPI != kEpiSwiGLU)) && (!SLICED || RAGGED), "combinations in use");
    using Shape = MfmaShape<T, 16>;
    using Frag = typename Shape::Frag;
    using Lds = DmaLds<T, kWideLdsElements>;
    constexpr bool kTurned = TA || TB;
    constexpr int BN_OUT = EPI == kEpiSwiGLU ? 128 : 256;
    constexpr int kRegion = 16384, kBuffer = 65536;               // bytes
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 2, wn = wave & 3;                      // the two groups are the two halves of the rows
    const int frow = lane & 15, q = lane >> 4;
    const int num_tiles = tiles_m * tiles_n;
    if (block >= num_tiles) return;
    if (!kTurned) lda = ldb = K;

    // k-tiles of this workgroup, and their number made even: a step of the loop is two
    const int k_range = (K + kWideK - 1) / kWideK, k_all = k_range * segments;
    const int k_share = SLICED ? (k_all + slices - 1) / slices : k_all, k_first = SLICED ? slice * k_share : 0;
    const int k_tiles = SLICED ? (k_all - k_first < k_share ? k_all - k_first : k_share) : k_all;
    const int k_steps = RAGGED ? (k_tiles + 1) & ~1 : k_tiles;
    if (SLICED) C = reinterpret_cast<T*>(reinterpret_cast<float*>(C) + (int64_t)slice * M * N);

    // DMA.  A region holds 128 rows of A or B with 64 k values each (128 bytes), or, turned, 64 k-rows of 128 columns (256 bytes); its
    // 16-byte chunks are XOR-ed with a key of their row so that the rows a fragment read touches lie in different banks.  A wave
    // brings 1 KB pieces 2w and 2w + 1 of a region; a lane fetches the chunk that belongs at its place.
    // Keys: A's fragments are 16 successive rows; B's are rows 8 (l / 4) + l % 4, so that the four rows of D a lane receives from two of
    // them are eight successive columns of C.
    auto a_key = [](int row) { return (row >> 1) & 7; };
    auto b_key = [](int row) { return ((row >> 1) & 1) | ((row >> 3) & 3) << 1; };
    auto t_key = [](int k) { return ((k & 3) | ((k >> 3) & 1) << 2) << 1; };
    uint32_t a_off[2], b_off[2];
    bool a_tail[2], b_tail[2];           // the lane's chunk of a range's last k-tile exists
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int piece = 2 * wave + r, row = piece * 8 + lane / 8, k_row = piece * 4 + lane / 16;
        const int ca = (lane % 8) ^ a_key(row), cb = (lane % 8) ^ b_key(row), ct = (lane % 16) ^ t_key(k_row);
        a_off[r] = (uint32_t)(TA ? k_row * lda + ct * 8 : row * lda + ca * 8) * 2u;
        b_off[r] = (uint32_t)(TB ? k_row * ldb + ct * 8 : row * ldb + cb * 8) * 2u;
        a_tail[r] = TA || (k_range - 1) * kWideK + ca * 8 < K;
        b_tail[r] = TB || (k_range - 1) * kWideK + cb * 8 < K;
    }
    auto descriptor = [](const T* base, int64_t rows, int64_t ld, int64_t cols) {
        const int64_t bytes = rows > 0 ? ((rows - 1) * ld + cols) * 2 : 0;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<T*>(base), 0, (int)(bytes < 0x7FFFFFFFll ? bytes : 0x7FFFFFFFll), 0x00020000);
    };
    // the tile and k-tile the next DMA loads belong to, two k-tiles ahead of the products
    __amdgpu_buffer_rsrc_t a_rsrc, b_rsrc0, b_rsrc1;
    int p_tile = block, p_kt = 0;
    auto set_tile = [&]() {
        if (p_tile >= num_tiles) return;       // nothing follows: the offsets drop, the descriptors stay
        int tm, tn;
        wide_tile_at(p_tile, num_tiles, tiles_m, tiles_n, xcds, tm, tn);
        const int m0 = tm * kWide, n0 = tn * BN_OUT;
        const int cols_a = (M - m0 + 7) / 8 * 8;                  // A's rows are padded to whole chunks
        a_rsrc = TA ? descriptor(A + m0, K, lda, cols_a) : descriptor(A + (int64_t)m0 * lda, M - m0, lda, kTurned ? (K * segments + 7) / 8 * 8 : K);
        b_rsrc0 = TB ? descriptor(B0 + n0, K, ldb, N - n0) : descriptor(B0 + (int64_t)n0 * ldb, N - n0, ldb, K);
        if (EPI == kEpiSwiGLU) b_rsrc1 = descriptor(B1 + (int64_t)n0 * ldb, N - n0, ldb, K);
        else b_rsrc1 = TB && segments > 1 ? descriptor(B1 + n0, K, ldb, N - n0) : b_rsrc0;
    };
    auto advance = [&]() {
        if (++p_kt == k_steps) {
            p_kt = 0;
            p_tile += blocks;
            set_tile();
        }
    };
    auto dma = [&](int buffer, auto region_tag) {       // regions: halves 0 and 1 of A, then of B
        constexpr int region = decltype(region_tag)::value, half = region & 1;
        constexpr bool of_a = region < 2, turned = of_a ? TA : TB;
        const int at = k_first + p_kt, seg = kTurned && at >= k_range ? 1 : 0, kr = at - seg * k_range;
        const bool gone = p_tile >= num_tiles || (RAGGED && p_kt >= k_tiles), last = RAGGED && kr + 1 == k_range;
        const int ld = of_a ? lda : ldb;
        // gate and up rows are the halves of B
        const int half_off = (EPI == kEpiSwiGLU && !of_a) ? 0 : half * (turned ? 256 : 128 * ld * 2);
        const int k_off = turned ? kr * kWideK * ld * 2 : ((of_a && kTurned ? seg * K : 0) + kr * kWideK) * 2;
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t off = (of_a ? a_off[r] : b_off[r]) + (RAGGED ? (uint32_t)half_off : 0u);
            const bool drop = gone || (last && !(of_a ? a_tail[r] : b_tail[r]));
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                of_a ? a_rsrc : ((EPI == kEpiSwiGLU ? half : seg) ? b_rsrc1 : b_rsrc0),
                (__attribute__((address_space(3))) void*)(reinterpret_cast<char*>(Lds::at()) + buffer * kBuffer + region * kRegion + (2 * wave + r) * 1024), 16,
                (int)(drop ? kOutOfRange : off), gone ? 0 : k_off + (RAGGED ? 0 : half_off), 0, 0);
        }
    };

    // Fragments.  Normal operands: one 16-byte read, piece q of a 32-value k-step; turned ones: two transposing reads of 4 k-rows each
    // (lane l of 16 addresses piece l % 4 of row l / 4 and receives column l).
    int a_at[4], b_at[2];
    if (TA) {
        const int k = q * 8 + frow / 4, p = frow % 4;
#pragma unroll
        for (int i = 0; i < 4; ++i) a_at[i] = k * 256 + (((wm * 8 + 2 * i + p / 2) ^ t_key(k)) << 4) + (p & 1) * 8;
    } else {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) a_at[ks] = (wm * 64 + frow) * 128 + (((ks * 4 + q) ^ a_key(frow)) << 4);
        a_at[2] = a_at[3] = 0;
    }
    if (TB) {
        const int k = q * 8 + frow / 4, p = frow % 4;
#pragma unroll
        for (int j = 0; j < 2; ++j) b_at[j] = k * 256 + (((wn * 4 + 2 * j + p / 2) ^ t_key(k)) << 4) + (p & 1) * 8;
    } else {
        const int row = (frow >> 2) * 8 + (frow & 3);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) b_at[ks] = (wn * 32 + row) * 128 + (((ks * 4 + q) ^ b_key(row)) << 4);
    }
    auto turned_frag = [&](const char* at) {
        typedef short i16x4_t __attribute__((__vector_size__(8)));
        typedef short i16x8_t __attribute__((__vector_size__(16)));
        typedef __attribute__((address_space(3))) i16x4_t* tr_ptr;
        const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)at);
        const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(at + 4 * 256));
        const i16x8_t both = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
        return __builtin_bit_cast(Frag, both);
    };
    auto a_frag = [&](int buffer, int half, int ks, int i) {
        const char* at = reinterpret_cast<const char*>(Lds::at()) + buffer * kBuffer + half * kRegion;
        if constexpr (TA) return turned_frag(at + a_at[i] + ks * 8192);
        else return *reinterpret_cast<const Frag*>(at + a_at[ks] + i * 2048);
    };
    auto b_frag = [&](int buffer, int half, int ks, int j) {
        const char* at = reinterpret_cast<const char*>(Lds::at()) + buffer * kBuffer + (2 + half) * kRegion;
        if constexpr (TB) return turned_frag(at + b_at[j] + ks * 8192);
        else return *reinterpret_cast<const Frag*>(at + b_at[ks] + j * 512);
    };
    // a: the half of A in use; ahead: the first two fragments of the next one, read a step early so that every step reads six; b0 of the
    // next k-tile is read while this one's is still needed
    Frag a[2][4], ahead[2], b0[2][2][2], b1[2][2];
    auto read_ahead = [&](int buffer, int half) {
#pragma unroll
        for (int i = 0; i < 2; ++i) ahead[i] = a_frag(buffer, half, 0, i);
    };
    auto take_ahead = [&]() {
#pragma unroll
        for (int i = 0; i < 2; ++i) a[0][i] = ahead[i];
    };
    auto read_a = [&](int buffer, int half) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (ks > 0 || i >= 2) a[ks][i] = a_frag(buffer, half, ks, i);
    };
    auto read_b = [&](int buffer, int half, Frag (&b)[2][2]) {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int j = 0; j < 2; ++j) b[ks][j] = b_frag(buffer, half, ks, j);
    };
    f32x4_t acc[8][4];
    auto multiply = [&](int ha, int hb, const Frag (&b)[2][2]) {
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) acc[ha * 4 + i][hb * 2 + j] = Shape::run(b[ks][j], a[ks][i], acc[ha * 4 + i][hb * 2 + j]);
        __builtin_amdgcn_s_setprio(0);
    };
    // End of a wave's fetching half step: its fragments are there, and of its DMA loads all but the ten of the last five regions, so
    // that after the barrier everyone's loads of the region read next have landed.
    auto fetched = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070 | 10);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    auto multiplied = [&]() {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
    };
    using A0 = Number<0>;
    using A1 = Number<1>;
    using B0r = Number<2>;
    using B1r = Number<3>;

    set_tile();
    for (int buffer = 0; buffer < 2; ++buffer) {
        dma(buffer, B0r{});
        dma(buffer, A0{});
        dma(buffer, B1r{});
        dma(buffer, A1{});
        advance();
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0x0F70 | 12);       // the first two regions
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    read_b(0, 0, b0[0]);
    read_ahead(0, 0);
    take_ahead();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xC07F);            // the first DMA of the loop overwrites what these reads took
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    for (int tile = block;; ) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if (wm == 1) __builtin_amdgcn_s_barrier();       // the second group starts half a step later
        __builtin_amdgcn_sched_barrier(0);
        for (int kt = 0; kt < k_steps; kt += 2) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                read_a(b, 0);
                dma(b, B0r{});
                fetched();
                multiply(0, 0, b0[b]);
                multiplied();
                read_b(b, 1, b1);
                read_ahead(b, 1);
                dma(b, A0{});
                fetched();
                multiply(0, 1, b1);
                take_ahead();
                multiplied();
                read_a(b, 1);
                dma(b, B1r{});
                fetched();
                multiply(1, 1, b1);
                multiplied();
                read_b(b ^ 1, 0, b0[b ^ 1]);
                read_ahead(b ^ 1, 0);
                dma(b, A1{});
                advance();
                fetched();
                multiply(1, 0, b0[b]);
                take_ahead();
                multiplied();
            }
        }

        // Lane l holds row l % 16 of every fragment of A, and of B's half h columns 8 (l / 16) .. + 7.  With B turned it holds columns
        // 4 (l / 16) .. + 3 of either fragment of 16; rows of 16 lanes swap, so that the even ones have eight successive columns of
        // the first fragment and the odd ones of the second (stores of 8 bytes took 1 to 4 % longer).  Offsets sit in the vector register alone: with a scalar offset too the compiler leaves out the wait that a store
        // of more than 8 bytes needs before its registers are written again (seen as wrong values in lanes 12 to 15).
        int tm, tn;
        wide_tile_at(tile, num_tiles, tiles_m, tiles_n, xcds, tm, tn);
        const int row0 = tm * kWide + wm * 64, col0 = tn * BN_OUT + wn * 32 + (TB ? (EPI == kEpiPart ? q * 4 : (q & 1) * 16 + (q >> 1) * 8) : q * 8);
        constexpr int kSize = EPI == kEpiPart ? 4 : 2;
        auto plane = [&](const void* base) {
            const int64_t span = base != nullptr ? ((int64_t)M - row0) * N * kSize : 0;
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>((const char*)base + (base != nullptr ? (int64_t)row0 * N * kSize : 0)), 0,
                                                     (int)(span < 0 ? 0 : (span < 0x7FFFFFFFll ? span : 0x7FFFFFFFll)), 0x00020000);
        };
        auto place = [&](int f, int hb, int part) {
            const int col = col0 + hb * 128 + part * 16;
            const int off = (((f >> 2) * 128 + (f & 3) * 16 + frow) * N + col) * kSize;
            return !RAGGED || col < N ? off : (int)kOutOfRange;
        };
        auto values = [&](int f, int hb, float (&v)[8]) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) v[j * 4 + e] = acc[f][hb * 2 + j][e];
        };
        auto store8 = [&](auto rsrc, int f, int hb, const float (&v)[8]) {
            u32x4_t packed = pack16<T>(v);
            if constexpr (TB) {
#pragma unroll
                for (int w = 0; w < 2; ++w) {
                    const auto swapped = __builtin_amdgcn_permlane16_swap(packed[w], packed[2 + w], false, false);
                    packed[w] = swapped[0];
                    packed[2 + w] = swapped[1];
                }
            }
            __builtin_amdgcn_raw_buffer_store_b128(packed, rsrc, place(f, hb, 0), 0, 0);
        };
        const auto c_rsrc = plane(C);
        if constexpr (EPI == kEpiSwiGLU) {
            if (wm == 0) __builtin_amdgcn_s_barrier();
            if (R != nullptr) {            // keep the gate and up products for a backward pass: planes [0] and [1] of a [2, M, N] buffer
                const auto g_rsrc = plane(R), u_rsrc = plane(R + (int64_t)M * N);
#pragma unroll
                for (int f = 0; f < 8; ++f) {
                    float v[8];
                    values(f, 0, v);
                    store8(g_rsrc, f, 0, v);
                    values(f, 1, v);
                    store8(u_rsrc, f, 0, v);
                }
            }
#pragma unroll
            for (int f = 0; f < 8; ++f) {
                float g[8], u[8];
                values(f, 0, g);
                values(f, 1, u);
#pragma unroll
                for (int e = 0; e < 8; ++e) g[e] = silu_fast_f32(g[e]) * u[e];
                store8(c_rsrc, f, 0, g);
            }
        } else if constexpr (EPI == kEpiPart) {
            if (wm == 0) __builtin_amdgcn_s_barrier();
#pragma unroll
            for (int f = 0; f < 8; ++f)
#pragma unroll
                for (int hb = 0; hb < 2; ++hb)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[f][hb * 2 + j]), c_rsrc,
                                                               place(f, hb, TB ? j : 0) + (TB ? 0 : j * 16), 0, 0);
        } else if constexpr (kTurned) {
            if (wm == 0) __builtin_amdgcn_s_barrier();
#pragma unroll
            for (int f = 0; f < 8; ++f)
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) {
                    float v[8];
                    values(f, hb, v);
                    store8(c_rsrc, f, hb, v);
                }
        } else {
            const auto r_rsrc = plane(R);       // no residual: reads give 0
            u32x4_t res[4][2];
            auto load_residual = [&](int f) {
#pragma unroll
                for (int hb = 0; hb < 2; ++hb)
                    res[f & 3][hb] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(r_rsrc, place(f, hb, 0), 0, 0));
            };
#pragma unroll
            for (int f = 0; f < 4; ++f) load_residual(f);
            __builtin_amdgcn_sched_barrier(0);
            if (wm == 0) __builtin_amdgcn_s_barrier();
#pragma unroll
            for (int f = 0; f < 8; ++f) {
#pragma unroll
                for (int hb = 0; hb < 2; ++hb) {
                    float v[8], r[8];
                    values(f, hb, v);
                    unpack16<T>(res[f & 3][hb], r);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] += r[e];
                    store8(c_rsrc, f, hb, v);
                }
                if (f < 4) load_residual(f + 4);
            }
        }
        tile += blocks;
        if (tile >= num_tiles) break;
    }
    __builtin_amdgcn_s_waitcnt(0x0070);      // no load into the LDS is left when the workgroup ends
}

}  // namespace
}  // namespace fmoe
