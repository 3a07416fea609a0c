// y = x W^T for more than 64 rows, bfloat16 in, 32-bit sums: tiles of 64 to 256 rows of x by 128 or 256 rows of W, chosen by size.
// Plain results in bfloat16, gated ones (silu(gate) * up of W = [gate; up], both rounded to bfloat16 first, as a stored product would
// be) in bfloat16, or 32-bit shares of a sum over pieces of K. Layout of the reference's F.linear
// (rollout/monkey_patch/qwen3.py:21): x [M, K], W [N, K], y [M, N].
//
// Why tiles of many sizes: at some hundred rows a product is one or two rounds of tiles over 256 CUs, and its time is the rounds'
// number times a tile's time; the twelve tiles (and pieces of K, where a later kernel adds shares) let block_plan() fill the rounds.
//
// A workgroup has eight waves, 2 x 4 or 4 x 2 over the tile. Both operands are copied into LDS (buffer_load ... lds) in steps of 64
// columns, whole 128-byte lines of a row; a row's 16-byte pieces lie at piece ^ (row / 2) % 8, so that operand reads
// (ds_read_b128) meet no bank conflict (measured: none). x has 2 to 5 stages and W 3 to 6: W comes from memory, x from L2. A step is
// two halves of 32 columns: a half's operands are read between the matrix instructions of the half before. One barrier a step, between
// the halves: before it a wave has read all of this step's stage and its copies of the next have landed, behind it the stage is
// refilled, the copies spread over the rest of this step and the first half of the next (x first, which is needed sooner). With the
// copies in one burst behind the barrier and W in two stages the largest tile lost 5 % (2,048 x 24,576 x 4,096: 328 -> 313 us).
//
// Bound by the matrix units and, below them, by what copies cost: 2,048 x 24,576 x 4,096 307 to 323 us (1.28 to 1.34 PFLOP/s, matrix units
// busy 68 % at 1.9 GHz; without the copies 245, without the barrier 295, with operands in LDS from the start and no reads 235). Waves that copy in
// turn, rows of K begun at different columns, priorities of 0: no faster. Microseconds with W from memory, the library
// (gated: and its SiLU-mul, residual: and the norm that takes the result) / this kernel: 536 rows of 19,456 x 2,560 gated 64 / 56, 6,144 x 2,560
// 29.3 / 24.8, 2,560 x 9,728 residual 49.3 / 42.6, 2,560 x 4,096 residual 30.7 / 27.2; 2,804 rows of 24,576 x 4,096 gated 504 / 449; 256 rows of
// 6,144 x 4,096 40.4 / 30.8.
#include "common.h"

typedef __bf16 blk_b8 __attribute__((ext_vector_type(8)));
typedef float blk_f4 __attribute__((ext_vector_type(4)));
typedef unsigned blk_u2 __attribute__((ext_vector_type(2)));
typedef unsigned blk_u4 __attribute__((ext_vector_type(4)));

enum { BLK_PLAIN = 0, BLK_GATED = 1, BLK_SHARES = 2 };

// What a kernel behind the product would make of its results, which are rounded to bfloat16 first, bit for bit: bias added (gated: N
// of them, gate and up halves; null: none); plain: act 2 max(y, 0)^2; gated: act 0 silu(g) u, 1 g sigmoid(slope g) (u + 1) with g = min(gate, limit),
// u = clamp(up, -limit, limit). 2,048 rows of 12,288 squared by a kernel of their own 17 us, 2,333 of 8,192 columns biased and gated 30.
struct BlockAct {
    int kind;
    float limit, slope;
    const float* bias;
};

// Waits until at most COPIES of the wave's copies are on their way, and for its LDS reads.
template <int COPIES>
__device__ __forceinline__ void blk_wait() {
    static_assert(COPIES >= 0 && COPIES < 64, "field of s_waitcnt");
    __builtin_amdgcn_s_waitcnt(0x0070 | (COPIES & 15) | ((COPIES >> 4) << 14));
}

template <int BM_, int BN_, int WM_, int WN_, int SX_, int SW_>
struct BlockTile {
    static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, SX = SX_, SW = SW_;       // stages of x and of W
    static constexpr int NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16, XB = BM / 8, WB = BN / 8;
    // copies of a refill, of 8 rows each, go round the waves, x first; the last of them that may be of x, plus one
    static constexpr int C = (XB + WB + NW - 1) / NW, CX = (XB + NW - 1) / NW;
    static constexpr bool PAD = C * NW != XB + WB;                                         // (what is over lands in a place of its own)
    static constexpr int LDS = (SX * BM + SW * BN) * 128 + (PAD ? 1024 : 0);
    // beside which group of operands of (a step's second half, the next one's first half) a copy is asked for
    static constexpr int slot(int c) { return c * 2 * TM / C; }
    static constexpr int late() {
        int k = 0;
        for (int i = 0; i < C; ++i) k += slot(i) >= TM;
        return k;
    }
    static constexpr int BEHIND = SW > SX ? C - CX : 0;                                    // copies of a refill behind its last of x
    static_assert(NW == 8 && SW >= SX && SX >= 2 && LDS <= 163840, "sizes of a tile");
};

// A workgroup's tile: workgroups go to the 8 XCDs round-robin, an XCD gets a run of neighbouring items, rows of x fastest (all of them
// up to 8 tiles, else 4), so that what its tiles share is read out of one L2.
template <typename T, int MODE>
__device__ __forceinline__ void block_tile(const bf16* __restrict__ X, const bf16* __restrict__ W, void* __restrict__ C, int M, int N, int K,
                                           int tiles_m, int tiles_n, int k_piece, const BlockAct& act) {
    constexpr int NW = T::NW, TM = T::TM, TN = T::TN, SX = T::SX, SW = T::SW, XS = T::BM * 128, WS = T::BN * 128;
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int wm = wave / T::WN, wn = wave % T::WN;
    int item;
    {
        const int total = gridDim.x, xcd = blockIdx.x & 7, q = total >> 3, r = total & 7;
        item = xcd * q + min(xcd, r) + (blockIdx.x >> 3);
    }
    const int piece = item / (tiles_m * tiles_n), t = item - piece * (tiles_m * tiles_n);
    int mt, nt;
    {
        const int run = tiles_m <= 8 ? tiles_m : 4, grp = t / (run * tiles_n), first = grp * run;
        const int rows = min(tiles_m - first, run), in = t - first * tiles_n;
        mt = first + in % rows;
        nt = in / rows;
    }
    const int m0 = mt * T::BM, n0 = nt * T::BN;
    const int kbeg = piece * k_piece, nk = (min(K, kbeg + k_piece) - kbeg) >> 6;
    const int xbytes = (int)((size_t)M * K * 2), wbytes = (int)((size_t)N * K * 2);
    // lane l of a copy writes piece l & 7 of row l >> 3 and reads what belongs there; rows that are not there are read beyond the
    // buffer's end, which gives zeros
    int off[T::C];
#pragma unroll
    for (int i = 0; i < T::C; ++i) {
        const int blk = wave + NW * i;
        const bool isx = blk < T::XB;
        const int row = 8 * (isx ? blk : blk - T::XB) + (lane >> 3), pc = (lane & 7) ^ ((row >> 1) & 7);
        if (isx) {
            off[i] = m0 + row < M ? (int)(((size_t)(m0 + row) * K + kbeg + pc * 8) * 2) : xbytes;
        } else {
            int wr = n0 + row;
            if constexpr (MODE == BLK_GATED) {               // 16 gate rows and the 16 up rows of the same columns in turn
                const int col = (n0 >> 1) + (row >> 5) * 16 + (row & 15);
                wr = col < (N >> 1) ? col + ((row >> 4) & 1) * (N >> 1) : N;
            }
            off[i] = wr < N && blk < T::XB + T::WB ? (int)(((size_t)wr * K + kbeg + pc * 8) * 2) : wbytes;
        }
    }
    // copy i of the refill behind step's half: x of step + SX into stage px, W of step + SW into stage pw (steps beyond K: nothing, zeros)
    auto copy = [&](int step, int px, int pw, int i) {
        const int blk = wave + NW * i;
        const bool allx = NW * (i + 1) <= T::XB, allw = NW * i >= T::XB, isx = allx || (!allw && blk < T::XB);
        const int kk = step + (isx ? SX : SW);
        const __amdgpu_buffer_rsrc_t res =
            __builtin_amdgcn_make_buffer_rsrc(isx ? (void*)X : (void*)W, 0, kk < nk ? (isx ? xbytes : wbytes) : 0, 0x00020000);
        unsigned at = isx ? px * XS + blk * 1024 : SX * XS + pw * WS + (blk - T::XB) * 1024;
        if (T::PAD && NW * (i + 1) > T::XB + T::WB) at = blk < T::XB + T::WB ? at : (unsigned)(SX * XS + SW * WS);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (void __attribute__((address_space(3)))*)(lds + at), 16, off[i], kk * 128, 0, 0);
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    uint32_t xr[2], wr[2];                                   // operand reads: lane (n, g) has row n, piece 4 h + g
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int at = ((4 * h + g) ^ ((n >> 1) & 7)) * 16 + n * 128;
        xr[h] = lds0 + wm * TM * 2048 + at;
        wr[h] = lds0 + SX * XS + wn * TN * 2048 + at;
    }
    typedef const blk_b8 __attribute__((address_space(3)))* frag_t;
    struct Half { blk_b8 w[TN], x[TM]; };
    Half f[2];
    blk_f4 acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = blk_f4{0.f, 0.f, 0.f, 0.f};

    // what the loop would have asked for before step 0, in its order; the last refill's late part is left to step 0
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = -SW; s < 0; ++s) {
#pragma unroll
        for (int i = 0; i < T::C; ++i) {
            if (s == -1 && T::slot(i) >= TM) continue;
            if (s >= -SX || NW * i >= T::XB) copy(s, s + SX, s + SW, i);
            else if (NW * (i + 1) > T::XB) {                 // a copy of x by some waves and W by others, at a step that x has not
                if (wave + NW * i >= T::XB) copy(s, 0, s + SW, i);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    blk_wait<T::BEHIND + (SX - 1) * T::C - T::late()>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int a = 0; a < TN; ++a) f[0].w[a] = *(frag_t)(uintptr_t)(wr[0] + a * 2048);
#pragma unroll
    for (int b = 0; b < TM; ++b) f[0].x[b] = *(frag_t)(uintptr_t)(xr[0] + b * 2048);

    int sx = 0, sw = 0, px = SX - 1, pw = SW - 1;            // stages of this step and of the one before
    // a half: its products group by group, the operands of the half that follows read in all groups but the last, and the copies
    auto half = [&](Half& now, Half& then, uint32_t xa, uint32_t wa, int step, int cx, int cw, int slot0) {
        constexpr int READS = TM + TN, GROUPS = TM > 1 ? TM - 1 : 1;
#pragma unroll
        for (int b = 0; b < TM; ++b) {
#pragma unroll
            for (int r = 0; r < READS; ++r)
                if (r * GROUPS / READS == b) {
                    if (r < TN) then.w[r] = *(frag_t)(uintptr_t)(wa + r * 2048);
                    else then.x[r - TN] = *(frag_t)(uintptr_t)(xa + (r - TN) * 2048);
                }
#pragma unroll
            for (int c = 0; c < T::C; ++c)
                if (T::slot(c) == slot0 + b) copy(step, cx, cw, c);
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int a = 0; a < TN; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(now.w[a], now.x[b], acc[a][b], 0, 0, 0);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    for (int it = 0; it < nk; ++it) {
        half(f[0], f[1], xr[1] + sx * XS, wr[1] + sw * WS, it - 1, px, pw, TM);
        // the next step's stages have landed for everyone, this step's have been read by everyone
        blk_wait<T::BEHIND + (SX - 2) * T::C>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const int nx = sx + 1 == SX ? 0 : sx + 1, nw = sw + 1 == SW ? 0 : sw + 1;
        half(f[1], f[0], xr[0] + nx * XS, wr[0] + nw * WS, it, sx, sw, 0);
        px = sx;
        pw = sw;
        sx = nx;
        sw = nw;
    }
    blk_wait<0>();
    MFMA_SETTLE();

    // acc[a][b][e]: row 16 b + n of the wave's rows, row 16 a + 4 g + e of its rows of W
    const int row0 = m0 + wm * TM * 16;
    if constexpr (MODE == BLK_SHARES) {
        float* out = (float*)C + (size_t)piece * M * N;
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            const int m = row0 + 16 * b + n;
            if (m >= M) continue;
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                const int col = n0 + (wn * TN + a) * 16 + 4 * g;
                if (col < N) *reinterpret_cast<blk_f4*>(out + (size_t)m * N + col) = acc[a][b];
            }
        }
    } else {
        // 16 rows at a time through the wave's own places in LDS, so that a row's results are stored side by side (1 us of 26 and of 60)
        constexpr int COLS = MODE == BLK_GATED ? TN * 8 : TN * 16, ROW = COLS * 2 + 16, PER = COLS / 8, ROWS = 64 / PER < 16 ? 64 / PER : 16;
        const int NO = MODE == BLK_GATED ? N >> 1 : N, c0 = (MODE == BLK_GATED ? n0 >> 1 : n0) + wn * COLS;
        __syncthreads();                                     // (everyone's copies have landed)
        const uint32_t mine = lds0 + wave * (2 * 16 * ROW);
        blk_f4 bias[TN];                                     // of the wave's rows of W
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            const int col = c0 + (MODE == BLK_GATED ? a / 2 : a) * 16 + 4 * g;
            bias[a] = blk_f4{0.f, 0.f, 0.f, 0.f};
            if (act.bias != nullptr && col < NO) bias[a] = *reinterpret_cast<const blk_f4*>(act.bias + (MODE == BLK_GATED && (a & 1) ? NO : 0) + col);
        }
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            const uint32_t buf = mine + (b & 1) * 16 * ROW;
#pragma unroll
            for (int a = 0; a < TN; a += MODE == BLK_GATED ? 2 : 1) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (MODE == BLK_GATED) {
                        float gate = round_to<bf16>(acc[a][b][e]), up = round_to<bf16>(acc[a + 1][b][e]);
                        if (act.bias != nullptr) {
                            gate += bias[a][e];
                            up += bias[a + 1][e];
                        }
                        if (act.kind == 1) {
                            const float x = fminf(gate, act.limit), u = fminf(fmaxf(up, -act.limit), act.limit);
                            v[e] = x / (1.0f + expf(-act.slope * x)) * (u + 1.0f);
                        } else {
                            v[e] = gate / (1.0f + expf(-gate)) * up;
                        }
                    } else {
                        v[e] = round_to<bf16>(acc[a][b][e]);
                        if (act.bias != nullptr) v[e] += bias[a][e];
                        if (act.kind == 2) {
                            v[e] = fmaxf(v[e], 0.f);
                            v[e] *= v[e];
                        }
                    }
                }
                *(blk_u2 __attribute__((address_space(3)))*)(uintptr_t)(buf + n * ROW + (MODE == BLK_GATED ? a / 2 : a) * 32 + g * 8) =
                    blk_u2{(uint32_t)f2bf_bits(v[0]) | ((uint32_t)f2bf_bits(v[1]) << 16), (uint32_t)f2bf_bits(v[2]) | ((uint32_t)f2bf_bits(v[3]) << 16)};
            }
            __builtin_amdgcn_wave_barrier();                 // (a wave's LDS operations are carried out in their order)
            if (lane < ROWS * PER) {
#pragma unroll
                for (int r = 0; r < 16; r += ROWS) {
                    const int rr = r + lane / PER, pc = lane % PER, m = row0 + 16 * b + rr, col = c0 + pc * 8;
                    const blk_u4 o = *(const blk_u4 __attribute__((address_space(3)))*)(uintptr_t)(buf + rr * ROW + pc * 16);
                    if (m < M && col < NO) *reinterpret_cast<blk_u4*>((bf16*)C + (size_t)m * NO + col) = o;
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
}

template <typename T, int MODE>
__global__ __launch_bounds__(512, 1) void gemm_block_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W, void* __restrict__ C, int M, int N,
                                                            int K, int tiles_m, int tiles_n, int k_piece, const BlockAct act) {
    block_tile<T, MODE>(X, W, C, M, N, K, tiles_m, tiles_n, k_piece, act);
}

// The tiles: rows of x, rows of W, microseconds a step of 64 columns and what start and end of a tile take, fitted to 4,700 measurements
// (72 to 4,096 rows, fifteen shapes of 2,048 to 24,576 rows and 2,048 to 12,288 columns of W, W from memory): 7 % apart from them, and the
// tile it chooses 0.7 % slower than the best one on average, 10 % at most.
#define BLK_TILES(F)                                                                                                                  \
    F(0, 256, 256, 2, 4, 2, 3, 1.382, 4.6) F(1, 224, 256, 2, 4, 2, 3, 1.232, 4.6) F(2, 192, 256, 2, 4, 2, 3, 1.054, 4.1)              \
    F(3, 160, 256, 2, 4, 2, 3, 0.993, 3.6) F(4, 128, 256, 2, 4, 2, 4, 0.875, 3.2) F(5, 96, 256, 2, 4, 3, 3, 0.755, 2.1)               \
    F(6, 256, 128, 4, 2, 3, 4, 0.757, 2.8) F(7, 192, 128, 4, 2, 3, 4, 0.632, 2.3) F(8, 160, 128, 2, 4, 3, 4, 0.587, 2.4)              \
    F(9, 128, 128, 2, 4, 4, 5, 0.514, 1.8) F(10, 96, 128, 2, 4, 4, 6, 0.452, 2.2) F(11, 64, 128, 2, 4, 5, 6, 0.366, 1.3)
struct BlockCost {
    int bm, bn;
    float step, ends;
};
#define BLK_COST(ID, BM, BN, WM, WN, SX, SW, STEP, ENDS) {BM, BN, STEP, ENDS},
static const BlockCost block_costs[] = {BLK_TILES(BLK_COST)};
#define BLK_PIECES 8

// The tile and the pieces of K (`least` to `most`) with the least time by the figures above: rounds of tiles over the CUs, a part-filled one
// at 0.83 to 1 of a full one; several shares cost the kernel that adds them 0.64 us a million values each, written and read. One, two, four or
// eight pieces: for these that kernel reads whole 16-byte pieces of all shares at once, other numbers go by one that reads 4 bytes after 4 (with the norm,
// three pieces / the best of these, 1,200 rows of 4,096 x 12,288 129 / 120 us, 2,048 x 6,144 49 / 45; five / these 66 rows of 5,120 x 5,120 28.1 / 25.2, but
// 256 rows of 5,120 x 25,600 98 / 107).
// Returns tile + 16 pieces and the time, or -1 for what the kernel does not take.
static int block_plan(int M, int N, int K, bool gated, int least, int most, int cus, int* workgroups, float* us) {
    if (M <= 0 || N <= 0 || K <= 0 || K % 64 != 0 || N % (gated ? 16 : 8) != 0 || cus <= 0) return -1;
    if ((size_t)M * K * 2 > 0x7fffff00ull || (size_t)N * K * 2 > 0x7fffff00ull) return -1;
    int best = -1;
    for (int c = 0; c < (int)(sizeof(block_costs) / sizeof(block_costs[0])); ++c) {
        const BlockCost& k = block_costs[c];
        const long long tiles = (long long)((M + k.bm - 1) / k.bm) * ((N + k.bn - 1) / k.bn);
        for (int p = least; p <= most; ++p) {
            if ((p & (p - 1)) != 0 || K % (64 * p) != 0 || tiles * p > 0x7ffffff) continue;
            const long long full = tiles * p / cus, rest = tiles * p % cus;
            const float rounds = (float)full + (rest ? 0.83f + 0.17f * (float)rest / (float)cus : 0.0f);
            const float t = 5.0f + rounds * ((float)(K / 64 / p) * k.step + k.ends) + (p > 1 ? 0.64e-6f * (2 * p - 1) * (float)M * (float)N : 0.0f);
            if (best < 0 || t < *us) {
                best = c + 16 * p;
                *workgroups = (int)(tiles * p);
                *us = t;
            }
        }
    }
    return best;
}

// The choice for a product of these sizes: tile + 16 pieces, -1 where the kernel does not take it; its workgroups and its time as it is
// reckoned (either may be null). pieces: of K, at most so many, or exactly so many where it is negative (none but powers of two have a plan).
extern "C" int ra_gemm_block_plan(int M, int N, int K, int gated, int pieces, int cus, int* workgroups, float* us) {
    float t = 0.0f;
    int n = 0;
    if (pieces == 0 || pieces > BLK_PIECES || pieces < -BLK_PIECES) return -1;
    const int plan = block_plan(M, N, K, gated != 0, pieces < 0 ? -pieces : 1, pieces < 0 ? -pieces : pieces, cus, &n, &t);
    if (workgroups != nullptr) *workgroups = n;
    if (us != nullptr) *us = t;
    return plan;
}

template <typename T>
static int block_go(hipStream_t st, const void* X, const void* W, void* C, int M, int N, int K, int mode, int pieces, const BlockAct& act) {
    const int tm = (M + T::BM - 1) / T::BM, tn = (N + T::BN - 1) / T::BN;
    const dim3 grid((unsigned)((long long)tm * tn * pieces)), block(512);
    auto go = [&](auto kernel) {
        if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS) != hipSuccess) return RA_ERR_LAUNCH;
        hipLaunchKernelGGL(kernel, grid, block, T::LDS, st, (const bf16*)X, (const bf16*)W, C, M, N, K, tm, tn, K / pieces, act);
        return ra_launch_status();
    };
    return mode == BLK_PLAIN ? go(gemm_block_kernel<T, BLK_PLAIN>) : mode == BLK_GATED ? go(gemm_block_kernel<T, BLK_GATED>)
                                                                                       : go(gemm_block_kernel<T, BLK_SHARES>);
}

// plan: what ra_gemm_block_plan gave for these sizes. gated: N rows of W are gate and up halves, C [M, N / 2] bfloat16. Else C [M, N]
// bfloat16 (one piece) or 32-bit [pieces, M, N]. x, W, C and bias 16-byte aligned. act, limit, slope, bias: BlockAct, for bfloat16 results.
extern "C" int ra_gemm_block_bf16(const void* X, const void* W, void* C, int M, int N, int K, int gated, int plan, int out_dtype, int act, float limit,
                                  float slope, const float* bias, void* stream) {
    const int tile = plan & 15, pieces = plan >> 4;
    if (plan < 0 || M <= 0 || N <= 0 || K <= 0 || pieces < 1 || pieces > BLK_PIECES || K % (64 * pieces) != 0 || N % (gated ? 16 : 8) != 0)
        return RA_ERR_ARG;
    if ((size_t)M * K * 2 > 0x7fffff00ull || (size_t)N * K * 2 > 0x7fffff00ull || (((uintptr_t)X | (uintptr_t)W | (uintptr_t)C) & 15) != 0)
        return RA_ERR_ARG;
    if ((gated || out_dtype != RA_DTYPE_F32) && (pieces != 1 || out_dtype != RA_DTYPE_BF16)) return RA_ERR_ARG;
    if ((long long)((M + 63) / 64) * ((N + 127) / 128) * pieces > 0x7fffffff) return RA_ERR_ARG;
    if (act < 0 || act > 2 || (act == 2 && gated) || (act == 1 && (!gated || !(limit > 0.f))) || ((uintptr_t)bias & 15) != 0) return RA_ERR_ARG;
    if (out_dtype == RA_DTYPE_F32 && (act != 0 || bias != nullptr)) return RA_ERR_ARG;
    const BlockAct with = {act, limit, slope, bias};
    const int mode = gated ? BLK_GATED : out_dtype == RA_DTYPE_F32 ? BLK_SHARES : BLK_PLAIN;
    hipStream_t st = (hipStream_t)stream;
    switch (tile) {
#define BLK_CASE(ID, BM, BN, WM, WN, SX, SW, STEP, ENDS) \
    case ID: return block_go<BlockTile<BM, BN, WM, WN, SX, SW>>(st, X, W, C, M, N, K, mode, pieces, with);
        BLK_TILES(BLK_CASE)
    }
    return RA_ERR_ARG;
}
