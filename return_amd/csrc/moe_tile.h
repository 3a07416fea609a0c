// The experts' products for many rows an expert (moe_tile.hip) and for few (moe_sweep.hip), and what moe.hip shares with them.
#pragma once
#include "common.h"

// What a gated product makes of its halves. Kind 0: silu(g) * u. Kind 1: with g <- min(g, limit)
// and u <- clamp(u, -limit, limit): g * sigmoid(slope * g) * (u + 1).
struct MoeAct {
    int kind;
    float limit, slope;
    const float* in_scale;      // a factor on a pair's input row (null: none)
};
// both halves of pair p from their 32-bit sums: scaled, rounded to what a product kernel would have stored, activated
template <typename T>
__device__ __forceinline__ float moe_gate(float g, float u, const MoeAct act, float in_scale) {
    g = round_to<T>(g * in_scale);
    u = round_to<T>(u * in_scale);
    if (act.kind == 1) {
        g = fminf(g, act.limit);
        u = fminf(fmaxf(u, -act.limit), act.limit);
        return g / (1.0f + expf(-act.slope * g)) * (u + 1.0f);
    }
    return g / (1.0f + expf(-g)) * u;
}

#define MOE_TILE_ROWS 256
// Whether the kernel takes an expert's matrix of n_rows rows and n_pairs rows of x, all of K elements.
static inline bool moe_tile_fits(long long n_pairs, long long n_rows, int K) {
    return K % 32 == 0 && n_pairs * K * 2 < 0x7fffff00ll && n_rows * K * 2 < 0x7fffff00ll;
}
int moe_tile_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                    const int* meta, int max_tiles, int x_rows, int N, int K, int top_div, bool gated, const MoeAct& act);

// Few rows an expert: tiles of up to 16 rows.
bool moe_sweep_fits(int K);
int moe_sweep_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                     const int* meta, int N, int K, int top_div, bool gated, const MoeAct& act);

// Experts' matrices laid out in panels when they are loaded, for sizes that allow it (bfloat16, rows % 16 == 0, K % 64 == 0 and at most
// 4,096, for which the sweep over panels has a wave's eight steps in registers; the tiles have no such limit):
// [step of 64 columns][panel of 16 rows][half of the step][lane][8 elements], lane (n, g) of a half with row n, columns
// 8 g ... 8 g + 7: what a lane of MFMA 16x16x32 takes, so that a wave reads an operand as 1 KB in a row, and needs no LDS for it.
// Gated matrices have a panel of gate rows and the one of the up rows of the same columns side by side.
#define MOE_PANEL_ROWS 320                        // rows of a tile at most
#define MOE_PANEL_K 4096
int moe_panel_tile_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                          const int* meta, int max_tiles, int x_rows, int N, int K, int top_div, bool gated, const MoeAct& act);
int moe_panel_sweep_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                           const int* meta, int x_rows, int N, int K, int top_div, bool gated, const MoeAct& act);
