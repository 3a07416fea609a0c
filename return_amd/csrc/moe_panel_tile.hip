// The experts' products for many rows an expert, bfloat16, with W laid out in panels (moe_tile.h): tiles of up to 320 rows of one
// expert by 256 rows of its W.
//
// Eight waves, each with all of the tile's rows and two panels (32 rows) of W. W comes straight from memory into the operand
// registers, three steps of 64 columns ahead, and never goes through LDS; x, which all waves need, is copied into LDS
// (buffer_load ... lds), four stages, and read a few operands ahead of their MFMAs. So all of the LDS is there for x and a tile can
// have 320 rows, the bytes on their way into a CU are twice those of the form that holds both operands in LDS (moe_tile.hip), and the
// groups of 16 rows need not come in pairs: the loop is compiled for each count of them. One barrier a step: before it a wave has
// finished its reads of the step before, whose stage is refilled behind it. Everything is straight-line code of four steps
// (register and stage numbers are constants); steps beyond K read zeros from buffers of no length.
//
// The panels of a step lie side by side ([step][panel]), so that a workgroup reads 32 KB in a row: with [panel][step], runs a power of
// two apart, gate-up of 32 experts of 6,144 x 4,096 took 697 instead of 658 us at 12,432 pairs. Measured there, W in rows through LDS /
// this kernel, us: 256 pairs 298 / 231 (7.0 TB/s), 4,000 pairs 326 / 283, 8,000 pairs 489 / 376 (1.07 PFLOP/s), 12,432 pairs 629 /
// 550, uneven counts (147 to 742) 695 / 592, 32,768 pairs 1,486 / 1,285 (1.28 PFLOP/s); down (4,096 x 3,072) 8,000 pairs 281 / 193,
// 12,432 pairs 325 / 279; gate-up of 4,096 x 2,048, 256 pairs 130 / 82, 8,448 pairs 226 / 150. Bound, up to 100 rows an expert, by
// the reading of W, beyond that by LDS as much as by the matrix cores: all eight waves read all of x, 320 KB a step of 320 rows beside the
// 40 KB that are copied in, 2,880 clocks at 128 bytes a clock where the step's MFMAs take 2,560. MFMAs alone take 0.6 to 0.7 of the
// time. MFMA 32x32x16 instead of 16x16x32: 712 instead of 598 us at 12,432 pairs (before the copies of x were spread).
#include "moe_tile.h"
#include <type_traits>

typedef __bf16 mp_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float mp_float4_t __attribute__((ext_vector_type(4)));

#define MP_BK 64
#define MP_LDS (4 * MOE_PANEL_ROWS * MP_BK * 2)  // four stages of x (160 KB)
#define MP_RS 260                                // floats a row of results in LDS

// Waits until at most COPIES of the wave's last copies and loads are on their way.
template <int COPIES>
__device__ __forceinline__ void mp_wait() {
    static_assert(COPIES < 64, "field of s_waitcnt");
    __builtin_amdgcn_s_waitcnt(0x0f70 | (COPIES & 15) | ((COPIES >> 4) << 14));
}

// A tile of 16 NG rows at most. xoff, woff: where this lane's rows of x and its part of the wave's two panels begin (bytes).
template <bool GATED, int NG>
__device__ __forceinline__ void mp_tile(unsigned char* lds, const bf16* __restrict__ x, int x_bytes, const bf16* __restrict__ w_e,
                                        int w_bytes, const int (&xoff)[5], int woff, int K, int wave, int lane, bf16* __restrict__ y,
                                        const int* __restrict__ pairs, int n_rows, int n0, int N, const MoeAct& act) {
    constexpr int NX = (NG + 3) / 4;                           // copies of x a wave and stage (8 rows each)
    constexpr int STAGE = (NG > 16 ? MOE_PANEL_ROWS : 256) * MP_BK * 2;                // bytes of a stage of x
    // operands of a stage, places of the ring that they go through (4 ALL % R == 0: four steps leave it as it was), how far ahead they
    // are read (above 16 groups the sums leave registers for no more)
    constexpr int ALL = 2 * NG, R = NG > 16 ? 4 : 8, MOST = NG > 16 ? 3 : 5, D = ALL < MOST ? ALL : MOST;
    constexpr int AHEAD = NG > 16 ? 2 : 3;                     // steps that W is asked for ahead (likewise)
    // Large tiles spread the copies of x over a step, into the stage of two steps before: all at once behind the barrier they hold up the
    // operand reads of all waves (32,768 pairs 1,352 -> 1,285 us, 10,240 even ones 482 -> 439). Small ones, whose steps are short, ask
    // one step further ahead, behind the barrier.
    constexpr bool SPREAD = NG >= 10;
    const int n = lane & 15, g = lane >> 4, nk = K / MP_BK, kstep = w_bytes / nk;
    // (a step beyond K reads from buffers of no length, which gives zeros: the loop has no branches)
    auto copy_x = [&](int kk, int stage, int from, int to) {
        const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, kk < nk ? x_bytes : 0, 0x00020000);
        unsigned char* base = lds + stage * STAGE;
#pragma unroll
        for (int i = from; i < to; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (void __attribute__((address_space(3)))*)(base + (wave + 8 * i) * 1024), 16,
                                                     xoff[i], kk * (MP_BK * 2), 0, 0);
    };
    struct W { mp_bf16x8_t f[2][2]; };                          // [panel][half of the step]
    W w[4];
    auto load_w = [&](W& to, int kk) {
        const __amdgpu_buffer_rsrc_t res = __builtin_amdgcn_make_buffer_rsrc((void*)w_e, 0, kk < nk ? w_bytes : 0, 0x00020000);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int a = 0; a < 2; ++a)
                // (of tiles of 320 rows one of up to nine groups is its expert's only one, as the plan has it: W, which nothing shares then, is read
                // past the caches. 64 tokens 258 -> 231 us, 7.0 TB/s; with W that tiles share 605 -> 626. Shorter tiles, of steps that would leave
                // CUs idle, share it and read it so all the same: their matrices are small)
                to.f[a][h] = __builtin_bit_cast(mp_bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(res, woff + a * 2048 + h * 1024, kk * kstep, NG <= 9 ? 2 : 0));
    };
    // Piece c of row r of a stage lies at piece c ^ ((r >> 1) & 7); lane (n, g) reads row n of a group, piece 4 h + g
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds);
    // [pair of stages][h]. The instruction's offset has 16 bits: up to 16 groups a pair's reads end at 63,488; beyond, a stage is 40 KB and
    // those of an odd one from group 12 on lie further, an addition each (32 beside the 320 MFMAs of four steps of 20 groups)
    uint32_t rd[2][2];
#pragma unroll
    for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int h = 0; h < 2; ++h) rd[v][h] = lds0 + v * 2 * STAGE + n * 128 + (((4 * h + g) ^ (n >> 1)) * 16);
    asm volatile("" : "+v"(rd[0][0]), "+v"(rd[0][1]), "+v"(rd[1][0]), "+v"(rd[1][1]));
    typedef const mp_bf16x8_t __attribute__((address_space(3)))* frag_t;
    auto read_x = [&](auto stage_c, int i) {                   // operand i of the stage, in the order they are used
        constexpr int s = decltype(stage_c)::value;
        return *(frag_t)(uintptr_t)(rd[s >> 1][i / NG] + (s & 1) * STAGE + (i % NG) * 2048);
    };
    mp_float4_t acc[2][NG];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < NG; ++b) acc[a][b] = mp_float4_t{0.f, 0.f, 0.f, 0.f};
    using std::integral_constant;
    // (the waits count what was asked for in this order: nothing is moved across)
    __builtin_amdgcn_sched_barrier(0);
    load_w(w[0], 0);
    __builtin_amdgcn_sched_barrier(0);
    copy_x(0, 0, 0, NX);
    __builtin_amdgcn_sched_barrier(0);
    load_w(w[1], 1);
    __builtin_amdgcn_sched_barrier(0);
    copy_x(1, 1, 0, NX);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (AHEAD > 2) load_w(w[2], 2);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!SPREAD) copy_x(2, 2, 0, NX);
    __builtin_amdgcn_sched_barrier(0);
    mp_wait<4 * (AHEAD - 1) + (SPREAD ? 1 : 2) * NX>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    mp_bf16x8_t xf[R];
#pragma unroll
    for (int i = 0; i < D; ++i) xf[i] = read_x(integral_constant<int, 0>{}, i);

    auto step = [&](int it, auto slot_c) {
        constexpr int slot = decltype(slot_c)::value;          // it % 4, of W and of x
        constexpr integral_constant<int, (slot + 1) & 3> next{};
        constexpr integral_constant<int, (slot + 3) & 3> refill{};
        constexpr int at = slot * ALL;                         // place of this step's first operand in the ring
        load_w(w[(slot + AHEAD) & 3], it + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < ALL; ++i) {
            if (i == ALL - D) {
                // the next step's x has landed for everyone; everyone has read the step before this one, whose stage is refilled
                mp_wait<(SPREAD ? 4 : 8) + NX>();
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (!SPREAD) copy_x(it + 3, refill.value, 0, NX);
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (SPREAD) {
                constexpr int EACH = (ALL - D) / NX;           // operands between two copies
                if (i % EACH == EACH - 1 && i / EACH < NX) {
                    copy_x(it + 2, (slot + 2) & 3, i / EACH, i / EACH + 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            xf[(at + i + D) % R] = i + D < ALL ? read_x(slot_c, i + D) : read_x(next, i + D - ALL);
#pragma unroll
            for (int a = 0; a < 2; ++a)
                acc[a][i % NG] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[slot].f[a][i / NG], xf[(at + i) % R], acc[a][i % NG], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int it = 0;
    do {                                                       // (nk > 0)
        step(it, integral_constant<int, 0>{});
        step(it + 1, integral_constant<int, 1>{});
        step(it + 2, integral_constant<int, 2>{});
        step(it + 3, integral_constant<int, 3>{});
        it += 4;
    } while (it < nk);
    mp_wait<0>();                                              // (what was asked for beyond K has come)
    MFMA_SETTLE();

    // acc[a][b][c]: row 16 b + n of the tile, row 4 g + c of the wave's panel a. Results go through LDS, 64 rows at a time in two
    // buffers in turn, so that what forms and stores them is a loop and stores whole rows.
    __syncthreads();
    const int tid = wave * 64 + lane;
    constexpr int PER = GATED ? 16 : 32;                       // pieces of eight result columns a row
    const int r0 = tid / PER, c = (tid % PER) * 8;
    typedef mp_float4_t __attribute__((address_space(3)))* put_t;
    typedef const mp_float4_t __attribute__((address_space(3)))* get_t;
#pragma unroll 1
    for (int q = 0; q < (NG + 3) / 4; ++q) {
        const uint32_t buf = lds0 + (q & 1) * (64 * MP_RS * 4);
#pragma unroll
        for (int v = 0; v < (NG + 3) / 4; ++v)
            if (v == q) {
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    if (4 * v + b < NG)
#pragma unroll
                        for (int a = 0; a < 2; ++a)
                            *(put_t)(uintptr_t)(buf + ((16 * b + n) * MP_RS + 32 * wave + 16 * a + 4 * g) * 4) = acc[a][4 * v + b];
            }
        __syncthreads();
        if (n0 + c < N) {
#pragma unroll 1
            for (int r = r0; r < 64; r += 512 / PER) {
                const int m = 64 * q + r;
                if (m >= n_rows) break;
                const int p = pairs[m];
                const uint32_t from = buf + (r * MP_RS + (GATED ? (c >> 4) * 32 + (c & 15) : c)) * 4;
                const mp_float4_t g0 = *(get_t)(uintptr_t)from, g1 = *(get_t)(uintptr_t)(from + 16);
                float v[8];
                if constexpr (GATED) {
                    const mp_float4_t u0 = *(get_t)(uintptr_t)(from + 64), u1 = *(get_t)(uintptr_t)(from + 80);
                    const float scale = act.in_scale != nullptr ? act.in_scale[p] : 1.0f;
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = moe_gate<bf16>(k < 4 ? g0[k] : g1[k - 4], k < 4 ? u0[k] : u1[k - 4], act, scale);
                } else {
#pragma unroll
                    for (int k = 0; k < 8; ++k) v[k] = k < 4 ? g0[k] : g1[k - 4];
                }
                uint32_t o[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) o[k] = (uint32_t)f2bf_bits(v[2 * k]) | ((uint32_t)f2bf_bits(v[2 * k + 1]) << 16);
                *reinterpret_cast<uint4*>(y + (size_t)p * N + n0 + c) = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
    }
}

template <bool GATED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void moe_panel_tile_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ meta, int x_rows, int N, int K, int top_div,
    int tiles_n, const MoeAct act) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // Items are pairs of a row tile and a column tile; workgroups go to the XCDs round-robin. Of every eight row tiles in the plan's
    // order an XCD has an eighth of the items, of what is left too: runs of columns, for all of the tiles of an expert that stand
    // together, so that these share W in L2. As the plan has the large tiles first, the XCDs have about the same work and end
    // with small tiles: uneven counts (147 to 742), 12,432 pairs, gate-up 609 us (592 now); an eighth of all items in a row for each
    // XCD 676, of all work 631, items taken from a counter of the XCD's 633 and 50 us more for a small product.
    const int tiles_m = meta[0], xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, whole = tiles_m >> 3, rest = (tiles_m & 7) * tiles_n;
    int item;
    if (slot < whole * tiles_n) {
        item = (slot / tiles_n * 8 + xcd) * tiles_n + slot % tiles_n;
    } else {
        const int at = slot - whole * tiles_n + rest * xcd / 8;
        if (at >= rest * (xcd + 1) / 8) return;
        item = whole * 8 * tiles_n + at;
    }
    const int tl = item / tiles_n, run = tiles[3 * tl + 2] >> 16;                       // (tiles that stand together) * 16 + place among them
    const int first = tl - (run & 15), in = item - first * tiles_n, mt = first + in % (run >> 4), nt = in / (run >> 4);
    const int x_bytes = x_rows * K * 2;
    const size_t w_rows = GATED ? 2 * (size_t)N : (size_t)N;
    const int e = tiles[3 * mt], at = tiles[3 * mt + 1], n_rows = tiles[3 * mt + 2] & 0xffff;
    // a copy brings 8 rows: lane l writes piece l & 7 of row l >> 3, and reads the piece that belongs there; a row that the tile
    // does not have is read beyond the buffer's end, which reads nothing
    int xoff[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const int row = 8 * (wave + 8 * i) + (lane >> 3);
        xoff[i] = row < n_rows ? (int)(((size_t)(order[at + row] / top_div) * K + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2) : x_bytes;
    }
    // (a wave whose panels W does not have reads beyond the buffer's end too)
    const int w_bytes = (int)(w_rows * K * 2), panel = 2 * (8 * nt + wave);
    const int woff = (panel * 16 < (int)w_rows ? panel * 2048 : w_bytes) + lane * 16;
    const int groups = (n_rows + 15) >> 4;
#define MP_GO(NG_) case NG_: mp_tile<GATED, NG_>(lds, x, x_bytes, w + (size_t)e * w_rows * K, w_bytes, xoff, woff, K, wave, lane, y, order + at, n_rows, nt * (GATED ? 128 : 256), N, act); break
    switch (groups) {
        MP_GO(1); MP_GO(2); MP_GO(3); MP_GO(4); MP_GO(5); MP_GO(6); MP_GO(7); MP_GO(8); MP_GO(9); MP_GO(10);
        MP_GO(11); MP_GO(12); MP_GO(13); MP_GO(14); MP_GO(15); MP_GO(16); MP_GO(17); MP_GO(18); MP_GO(19); MP_GO(20);
    }
}

int moe_panel_tile_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles, const int* meta,
                          int max_tiles, int x_rows, int N, int K, int top_div, bool gated, const MoeAct& act) {
    const int tiles_n = (N + (gated ? 127 : 255)) / (gated ? 128 : 256);
    const long long total = (long long)max_tiles * tiles_n;
    if (total > 0x7ffffff8 || max_tiles > 0x7fff) return RA_ERR_ARG;
    const void* kernel = gated ? (const void*)moe_panel_tile_kernel<true> : (const void*)moe_panel_tile_kernel<false>;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MP_LDS) != hipSuccess) return RA_ERR_LAUNCH;
    const dim3 grid((unsigned)((total + 7) / 8 * 8));
    if (gated)
        hipLaunchKernelGGL(moe_panel_tile_kernel<true>, grid, dim3(512), MP_LDS, st, x, w, y, order, tiles, meta, x_rows, N, K, top_div,
                           tiles_n, act);
    else
        hipLaunchKernelGGL(moe_panel_tile_kernel<false>, grid, dim3(512), MP_LDS, st, x, w, y, order, tiles, meta, x_rows, N, K, top_div,
                           tiles_n, act);
    return ra_launch_status();
}
