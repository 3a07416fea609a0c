// The experts' products for few rows an expert, bfloat16, with W laid out in panels (moe_tile.h).
//
// An item is 16 result columns of a tile of up to 16 pairs of one expert: a panel of W, or one of gate and one of up rows. All items
// stand in a row and every workgroup has an equal share of them, across tiles. Wave w has an eighth of K: its part of an item
// comes straight into MFMA operands, 1 KB a load, and a register is asked for again for the next item as soon as its MFMA has been
// issued, so that a workgroup has a whole item, 64 K bytes gated and 32 K not, always on its way (of one workgroup a CU, up to K of
// 2,048 of two: 256 KB a CU at K of 2,048 and 4,096 gated, 32 KB at K of 512 not gated); its part of the tile's rows of x stays in registers. The waves'
// results are added through LDS in wave order; the barrier for that waits for no load.
//
// Bound by the reading of W, which goes past the caches (nontemporal). Measured, gate-up and down of 32 experts, four a token, with rows
// of W through LDS (moe_sweep.hip; caches / past them) / this kernel, us: of 6,144 x 4,096, 1 token 41 + 20, 37 + 22 / 34 + 19, 8
// tokens 194 + 102, 169 + 90 / 167 + 87 (6.6 TB/s).
#include "moe_tile.h"

typedef __bf16 mq_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float mq_float4_t __attribute__((ext_vector_type(4)));

#define MQ_WAVES 8

// A barrier that waits for the wave's own LDS accesses and for none of its loads from memory.
#define MQ_BARRIER()                                      \
    do {                                                  \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); \
        __builtin_amdgcn_s_barrier();                     \
        asm volatile("" ::: "memory");                    \
    } while (0)

// KW: steps of 64 columns of K a wave has at most (K <= 512 KW).
template <bool GATED, int KW>
__global__ __launch_bounds__(64 * MQ_WAVES) __attribute__((amdgpu_waves_per_eu(KW > 4 ? 2 : 4))) void moe_panel_sweep_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ meta, int x_rows, int N, int K, int top_div, const MoeAct act) {
    constexpr int NP = GATED ? 2 : 1;                          // panels of an item: 16 result columns
    __shared__ float red_both[2][MQ_WAVES * NP * 16 * 17];
    __shared__ int pair_both[2][16];
    __shared__ float scale_both[GATED ? 2 : 1][16];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int items = N >> 4, nk = K >> 6, w_bytes = NP * N * K * 2, kstep = NP * N * 128, x_bytes = x_rows * K * 2;
    const int k0 = wave * nk / MQ_WAVES, k_n = (wave + 1) * nk / MQ_WAVES - k0;
    const long long total = (long long)meta[0] * items;
    // Of fewer items than workgroups every eighth share, say, has one, and as workgroups go to the XCDs in turn, all of them would be
    // on one XCD (the 64 items of gate-up of 8 experts of 1,024 x 2,048, 2 pairs: both products and the plan 19.5 us, with the shares
    // in an XCD's order 17.2). With more items plain order is up to 5 % the faster one.
    const int G = gridDim.x, b = total < G && G % 8 == 0 ? (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3) : blockIdx.x;
    long long at = total * b / G;
    const long long end = total * (b + 1) / G;
    if (at >= end) return;                                     // (the same in every thread)
    int tile = (int)(at / items), item = (int)(at - (long long)tile * items);
    mq_bf16x8_t wf[KW][2][NP], xf[KW][2];
    const size_t w_size = (size_t)NP * N * K;
    const bf16* wt = w + (size_t)tiles[3 * tile] * w_size;     // W of the tile that is read from
    // (the first tile's pairs are asked for before its W: loads come back in order, and the rows of x that they name would wait for all
    // of W: 0.3 to 0.5 us a product where a workgroup has an item or two)
    auto pairs_of = [&](int t) { return order[tiles[3 * t + 1] + (n < tiles[3 * t + 2] ? n : 0)]; };
    int pair = pairs_of(tile);
    __builtin_amdgcn_sched_barrier(0);
    // (steps that the wave does not have, and what lies behind the last item, are read from buffers of no length: zeros)
    auto fetch = [&](int j, int h, int i, bool in) {
        const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc((void*)wt, 0, in && j < k_n ? w_bytes : 0, 0x00020000);
#pragma unroll
        for (int a = 0; a < NP; ++a)
            wf[j][h][a] = __builtin_bit_cast(mq_bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
                res, lane * 16 + a * 2048 + h * 1024, (k0 + j) * kstep + i * (NP * 2048), 2));
    };
#pragma unroll
    for (int j = 0; j < KW; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            fetch(j, h, item, true);
            __builtin_amdgcn_sched_barrier(0);                 // (waits count on the order of the loads)
        }
    int have = -1, n_rows = 0, turn = 0, pairs_in = 1;
    for (; at < end; ++at, turn ^= 1) {
        if (tile != have) {
            // lane (n, g) holds x[row n][64 (k0 + j) + 32 h + 8 g ..]; lanes of rows that the tile does not have hold its first
            // row, whose results are not used
            if (have >= 0) pair = pairs_of(tile);
            have = tile;
            n_rows = tiles[3 * tile + 2];
            const int row = pair / top_div;
            pairs_in ^= 1;                                     // (the tile before: its last results may still be read)
            if (tid < 16) {
                pair_both[pairs_in][tid] = pair;
                // (read here: a load behind those of W would wait for all of them)
                if constexpr (GATED) scale_both[pairs_in][tid] = act.in_scale != nullptr ? act.in_scale[pair] : 1.0f;
            }
#pragma unroll
            for (int j = 0; j < KW; ++j)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    xf[j][h] = __builtin_bit_cast(mq_bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(
                        __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, j < k_n ? x_bytes : 0, 0x00020000), (row * K + k0 * 64 + 8 * g) * 2,
                        (64 * j + 32 * h) * 2, 0));
            // (they have come here, so that the items behind wait for W alone)
#pragma unroll
            for (int j = 0; j < KW; ++j) asm volatile("" : "+v"(xf[j][0]), "+v"(xf[j][1]));
        }
        int next_tile = tile, next_item = item + 1;
        const bool more = at + 1 < end;
        if (next_item == items) {
            next_item = 0;
            if (more) wt = w + (size_t)tiles[3 * ++next_tile] * w_size;
        }
        mq_float4_t c[NP];
#pragma unroll
        for (int a = 0; a < NP; ++a) c[a] = mq_float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < KW; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
#pragma unroll
                for (int a = 0; a < NP; ++a) c[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][h][a], xf[j][h], c[a], 0, 0, 0);
                fetch(j, h, next_item, more);
                __builtin_amdgcn_sched_barrier(0);
            }
        MFMA_SETTLE();
        // c[a][i]: the wave's part of y[row n][panel a's row 4 g + i]. Two buffers in turn: one is written again two items on, which
        // is after the next item's barrier, and that its readers reach only when they have read
        float* red = red_both[turn];
#pragma unroll
        for (int a = 0; a < NP; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i) red[((wave * NP + a) * 16 + 4 * g + i) * 17 + n] = c[a][i];
        MQ_BARRIER();
        if (tid < 16 * n_rows) {
            const int m = tid >> 4, r = tid & 15, p = pair_both[pairs_in][m];
            float s = 0.f;
#pragma unroll
            for (int v = 0; v < MQ_WAVES; ++v) s += red[(v * NP * 16 + r) * 17 + m];
            if constexpr (GATED) {
                float up = 0.f;
#pragma unroll
                for (int v = 0; v < MQ_WAVES; ++v) up += red[(v * NP * 16 + 16 + r) * 17 + m];
                s = moe_gate<bf16>(s, up, act, scale_both[pairs_in][m]);
            }
            y[(size_t)p * N + item * 16 + r] = from_f<bf16>(s);
        }
        tile = next_tile;
        item = next_item;
    }
}

int moe_panel_sweep_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                           const int* meta, int x_rows, int N, int K, int top_div, bool gated, const MoeAct& act) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
#define MQ_LAUNCH(G_, KW_)                                                                                                       \
    hipLaunchKernelGGL((moe_panel_sweep_kernel<G_, KW_>), dim3(cus * (KW_ > 4 ? 1 : 2)), dim3(64 * MQ_WAVES), 0, st, x, w, y, order, \
                       tiles, meta, x_rows, N, K, top_div, act)
#define MQ_GO(KW_)                                                      \
    case KW_:                                                           \
        if (gated) MQ_LAUNCH(true, KW_); else MQ_LAUNCH(false, KW_);    \
        break
    switch ((K + 511) / 512) {
        MQ_GO(1); MQ_GO(2); MQ_GO(3); MQ_GO(4); MQ_GO(5); MQ_GO(6); MQ_GO(7); MQ_GO(8);
        default: return RA_ERR_ARG;
    }
#undef MQ_GO
#undef MQ_LAUNCH
    return ra_launch_status();
}
