// The experts' products for few rows an expert, bfloat16: W read in whole runs of 1 KB, as the sweeping product for small
// batches reads it (gemm_sweep.hip).
//
// A plan's tile is up to 16 pairs of one expert. Workgroups are dealt out to the tiles (each tile has as many as divide
// the grid evenly), and a tile's workgroups share its result columns in runs. Wave w has columns 512 w ... 512 w + 511 of K:
// a row of W is one load of 1 KB a wave, the sixteen rows of an item (16 result columns, or 8 gate and the 8 up rows of
// 8 columns) are on their way per lane while the item before is multiplied, a row of the next item asked for as soon as the
// same row of this one has arrived. An item goes through a part of LDS that is the wave's own, from where it is read back
// as A operands of MFMA 16x16x32 (rows padded by 16 bytes); the wave's columns of the tile's rows of x are B operands that
// stay in registers for all of the workgroup's items (one expert: x is gathered once). The waves' partial results are
// added through LDS in wave order.
//
// Why: with operands straight from memory a wave read 16 rows of W by 64 bytes at a time and the experts of a decode step
// came at 3.9 to 4.1 TB/s. Measured, gate-up and down of 32 experts, four a token: of 6,144 x 4,096, 1 token 61 us (65
// before), 8 tokens 296 (391; 1.5 GB at 5.1 TB/s), 16 tokens 369 (408); of 4,096 x 2,048, 1 token 23 us (38), 8 tokens 108
// (153), 64 tokens 155 (213).
// W is read past the caches: 8 tokens of 6,144 x 4,096 194 -> 169 us, 16 tokens 271 -> 239.
#include "moe_tile.h"

typedef __bf16 ms_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float ms_float4_t __attribute__((ext_vector_type(4)));

#define MS_KW 512                         // columns of K per wave
#define MS_STRIDE (MS_KW + 8)             // row stride of a wave's item in LDS (elements)
#define MS_STEPS (MS_KW / 32)

// order between the LDS accesses of one wave: LDS serves a wave in order, the compiler must too
#define MS_WAVE_SYNC()                                           \
    do {                                                         \
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   \
        __builtin_amdgcn_wave_barrier();                         \
    } while (0)

template <bool GATED>
__global__ __launch_bounds__(512) void moe_sweep_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ meta, int N, int K, int top_div, const MoeAct act) {
    constexpr int COLS = GATED ? 8 : 16;                        // result columns of an item
    extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4, waves = blockDim.x >> 6;
    uint16_t* stage = reinterpret_cast<uint16_t*>(lds_raw) + (size_t)wave * 16 * MS_STRIDE;
    float* red_both = reinterpret_cast<float*>(lds_raw + (size_t)waves * 16 * MS_STRIDE * 2);       // [2][wave][16 rows][17]
    int* pair_s = reinterpret_cast<int*>(red_both + 2 * waves * 16 * 17);                           // [16]
    const int n_tiles = meta[0], G = gridDim.x, b = blockIdx.x, items = (N + COLS - 1) / COLS;
    const size_t w_rows = GATED ? 2 * (size_t)N : (size_t)N;
    const int kb = wave * MS_KW;
    const bool k_in = kb + lane * 8 < K;                        // K % 8 == 0: a lane's 8 columns are in or out together
    const ms_bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};

    // (more tiles than workgroups: whole tiles in turn; else the workgroups of tile t are those from ceil(t G / n) on)
    for (int t = n_tiles > G ? b : (int)((long long)b * n_tiles / G); t < n_tiles; t += G) {
        int first = 0, last = items;
        if (n_tiles <= G) {
            const int from = (int)(((long long)t * G + n_tiles - 1) / n_tiles), to = (int)(((long long)(t + 1) * G + n_tiles - 1) / n_tiles);
            first = (int)((long long)items * (b - from) / (to - from));
            last = (int)((long long)items * (b - from + 1) / (to - from));
        }
        if (first >= last) continue;                            // (the same in every thread)
        const int e = tiles[3 * t], at = tiles[3 * t + 1], n_rows = tiles[3 * t + 2];
        const bf16* we = w + (size_t)e * w_rows * K + kb + lane * 8;
        ms_bf16x8_t wreg[16];
        auto fetch_row = [&](int item, int i) {
            const int col = item * COLS + (GATED ? (i & 7) : i);
            const size_t row = (GATED && i >= 8) ? (size_t)N + col : (size_t)col;
            wreg[i] = (k_in && col < N) ? __builtin_nontemporal_load(reinterpret_cast<const ms_bf16x8_t*>(we + row * K)) : zero;
        };
#pragma unroll
        for (int i = 0; i < 16; ++i) fetch_row(first, i);
        // the wave's columns of the tile's rows of x: lane (n, g) holds x[n][kb + 32 j + 8 g ..], rows beyond the tile's as zeros
        const int pair = n < n_rows ? order[at + n] : -1;
        __syncthreads();                                        // (a tile before: its last results have read pair_s)
        if (tid < 16) pair_s[tid] = pair;
        const bf16* xr = x + (size_t)(pair >= 0 ? pair / top_div : 0) * K;
        ms_bf16x8_t bx[MS_STEPS];
#pragma unroll
        for (int j = 0; j < MS_STEPS; ++j) {
            const int k = kb + 32 * j + 8 * g;
            bx[j] = (pair >= 0 && k < K) ? *reinterpret_cast<const ms_bf16x8_t*>(xr + k) : zero;
        }
        for (int item = first; item < last; ++item) {
            MS_WAVE_SYNC();                                     // the item before has been read out of the wave's LDS
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                *reinterpret_cast<ms_bf16x8_t*>(&stage[i * MS_STRIDE + lane * 8]) = wreg[i];
                if (item + 1 < last) fetch_row(item + 1, i);
            }
            MS_WAVE_SYNC();                                     // the item is complete in LDS
            ms_float4_t c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < MS_STEPS; ++j) {
                const ms_bf16x8_t a = *reinterpret_cast<const ms_bf16x8_t*>(&stage[n * MS_STRIDE + 32 * j + 8 * g]);
                c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bx[j], c, 0, 0, 0);
            }
            MFMA_SETTLE();
            // c[i] = partial y[row n][item's row 4 g + i]. Two buffers in turn: one is written again two items on, which is
            // after the next item's barrier, and that its readers reach only when they have read
            float* red = red_both + ((item - first) & 1) * (waves * 16 * 17);
#pragma unroll
            for (int i = 0; i < 4; ++i) red[(wave * 16 + 4 * g + i) * 17 + n] = c[i];
            __syncthreads();
            for (int i = tid; i < 16 * COLS; i += blockDim.x) {
                const int m = i / COLS, r = i % COLS, col = item * COLS + r;
                if (m >= n_rows || col >= N) continue;
                float s = 0.f;
                for (int v = 0; v < waves; ++v) s += red[(v * 16 + r) * 17 + m];
                const int p = pair_s[m];
                if constexpr (GATED) {
                    float up = 0.f;
                    for (int v = 0; v < waves; ++v) up += red[(v * 16 + 8 + r) * 17 + m];
                    s = moe_gate<bf16>(s, up, act, act.in_scale != nullptr ? act.in_scale[p] : 1.0f);
                }
                y[(size_t)p * N + col] = from_f<bf16>(s);
            }
        }
        if (n_tiles <= G) break;
    }
}

bool moe_sweep_fits(int K) { return K % 8 == 0 && K <= 8 * MS_KW; }

int moe_sweep_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                     const int* meta, int N, int K, int top_div, bool gated, const MoeAct& act) {
    const int waves = (K + MS_KW - 1) / MS_KW;
    const size_t lds = (size_t)waves * 16 * MS_STRIDE * 2 + sizeof(float) * 2 * waves * 16 * 17 + 64;
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    const dim3 grid(cus * (waves > 4 ? 1 : waves > 2 ? 2 : 4)), block(64 * waves);
    const void* kernel = gated ? (const void*)moe_sweep_kernel<true> : (const void*)moe_sweep_kernel<false>;
    if (lds > 64 * 1024 && hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
        return RA_ERR_LAUNCH;
    if (gated)
        hipLaunchKernelGGL(moe_sweep_kernel<true>, grid, block, lds, st, x, w, y, order, tiles, meta, N, K, top_div, act);
    else
        hipLaunchKernelGGL(moe_sweep_kernel<false>, grid, block, lds, st, x, w, y, order, tiles, meta, N, K, top_div, act);
    return ra_launch_status();
}
