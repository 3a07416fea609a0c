// The experts' products for many rows an expert, bfloat16: tiles of up to 256 rows of one expert by 256 rows of its W.
//
// Steps of 64 columns of K, so that a copy asks for whole 128-byte lines (with steps of 32 every line went into the CU's cache
// twice); eight waves as 2 x 4; operands copied straight into LDS (buffer_load ... lds), W three stages deep and x two: all of
// the 160 KB. W comes from memory and needs the longer way ahead, x is read by every column tile of an XCD and comes out of its
// L2. 16-byte pieces of a row are rotated by the copying lane's choice of address so that the reads meet no bank conflict, and
// the operands of the next 32 columns are read between the MFMAs of these. One barrier a step: in front of it a wave has
// finished its reads of the step's stage, behind it the copies refill that stage, and the next stage is read. Rows of x are
// gathered by pair; W comes from the tile's expert; gated, of a wave's four tiles of W rows the first two are gate rows and the
// last two the up rows of the same columns, so that a lane holds both halves of a result; and a tile has as many groups of 16
// rows as its expert left it (the plan cuts an expert's rows into even tiles). Wave row wm takes the groups wm, wm + 2, ...; the
// loop is compiled for each count of groups a wave, so that a tile of 100 rows issues the MFMAs and copies of 128 rows.
//
// Workgroups go to the XCDs round-robin: an XCD gets a run of consecutive (row tile, column tile) pairs, two row tiles
// (mostly of one expert, whose W they then share in L2) at a time through all columns.
//
// Bound by the bytes on their way into a CU: x waits in order behind W's misses. Without the MFMAs the kernel takes 561 of its
// 615 us at 12,432 pairs, with the copies of W alone 410, of x alone 322. Measured, gate-up of 32 experts of 6,144 x 4,096, four
// a token, steps of 32 in four stages / now: 8,000 pairs 558 / 490 us (0.82 PFLOP/s), 12,432 pairs 705 / 610 (1.03), 32,000 pairs
// 1,740 / 1,510 (1.07); down (4,096 x 3,072) at 12,432 pairs 371 / 320. At 2,800 pairs and fewer the time is the reading of W:
// 313 us for 1.6 GB. What is lost at 8,000 pairs is the last round of tiles: half of the experts have a few rows more than 256
// and so two tiles of 140.
#include "moe_tile.h"
#include <type_traits>

typedef __bf16 mt_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float mt_float4_t __attribute__((ext_vector_type(4)));

#define MB_BK 64
#define MB_UNIT (256 * MB_BK * 2)                // bytes of one operand's tile in a stage (32 KB)
#define MB_W 0                                   // three stages of W
#define MB_X (3 * MB_UNIT)                       // and two of x
#define MB_LDS (5 * MB_UNIT)                     // 160 KB

// Waits until at most COPIES of the wave's copies and READS of its LDS reads are on their way (the last ones: both finish in
// their order). A barrier waits for neither.
template <int COPIES, int READS>
__device__ __forceinline__ void mb_wait() {
    static_assert(COPIES < 16 && READS < 16, "fields of s_waitcnt");
    __builtin_amdgcn_s_waitcnt(0x0070 | COPIES | (READS << 8));        // (expcnt at its maximum)
}

// order between the LDS accesses of one wave: LDS serves a wave in order, the compiler must too
#define MB_WAVE_SYNC()                                           \
    do {                                                         \
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   \
        __builtin_amdgcn_wave_barrier();                         \
    } while (0)

// The results of up to four groups of 16 rows of a wave, group, group + 2, ... of the tile, from LDS ([row][64 columns], rows of
// MB_RS floats) to memory, in runs of 16 bytes.
#define MB_RS 68
typedef const mt_float4_t __attribute__((address_space(3)))* mb_lds_t;
template <bool GATED>
__device__ __forceinline__ void mb_store(uint32_t own, int lane, int group, int groups, int n_rows, const int* __restrict__ pairs,
                                         bf16* __restrict__ y, int N, int col0, const MoeAct& act) {
    constexpr int PER = GATED ? 4 : 8;                         // pieces of eight columns a row
    const int r0 = lane / PER, c = (lane % PER) * 8;
    if (col0 + c >= N) return;
#pragma unroll 1
    for (int r = r0; r < 16 * groups; r += 64 / PER) {
        const int m = 16 * (group + 2 * (r >> 4)) + (r & 15);
        if (m >= n_rows) continue;
        const int p = pairs[m];
        const uint32_t at = own + (r * MB_RS + c) * 4;
        const mt_float4_t g0 = *(mb_lds_t)(uintptr_t)at, g1 = *(mb_lds_t)(uintptr_t)(at + 16);
        float v[8];
        if constexpr (GATED) {
            const mt_float4_t u0 = *(mb_lds_t)(uintptr_t)(at + 128), u1 = *(mb_lds_t)(uintptr_t)(at + 144);
            const float scale = act.in_scale != nullptr ? act.in_scale[p] : 1.0f;
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = moe_gate<bf16>(k < 4 ? g0[k] : g1[k - 4], k < 4 ? u0[k] : u1[k - 4], act, scale);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) v[k] = k < 4 ? g0[k] : g1[k - 4];
        }
        bf16* dst = y + (size_t)p * N + col0 + c;
        if (((N & 7) | ((uintptr_t)y & 15)) == 0) {
            uint32_t w[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) w[k] = (uint32_t)f2bf_bits(v[2 * k]) | ((uint32_t)f2bf_bits(v[2 * k + 1]) << 16);
            *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (col0 + c + k < N) dst[k] = from_f<bf16>(v[k]);
        }
    }
}

// A tile of 32 NB rows at most. xoff, woff: where this lane's rows begin (bytes), one for each of its copies.
template <bool GATED, int NB>
__device__ __forceinline__ void mb_tile(unsigned char* lds, const __amdgpu_buffer_rsrc_t xres, const __amdgpu_buffer_rsrc_t wres,
                                        const int (&xoff)[4], const int (&woff)[4], int K, int wave, int lane, bf16* __restrict__ y,
                                        const int* __restrict__ pairs, int n_rows, int n0, int N, const MoeAct& act) {
    constexpr int NX = (NB + 1) / 2;                           // copies of x a wave and stage (8 rows each; of W: 4)
    const int n = lane & 15, g = lane >> 4, wm = wave >> 2, wn = wave & 3;
    const int nk = (K + MB_BK - 1) / MB_BK;
    auto copy_x = [&](int kk) {
        unsigned char* base = lds + MB_X + (kk & 1) * MB_UNIT;
#pragma unroll
        for (int i = 0; i < NX; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (void __attribute__((address_space(3)))*)(base + (wave + 8 * i) * 1024), 16,
                                                     xoff[i], kk * (MB_BK * 2), 0, 0);
    };
    auto copy_w = [&](int kk, int ring) {
        unsigned char* base = lds + MB_W + ring * MB_UNIT;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, (void __attribute__((address_space(3)))*)(base + (4 * wave + i) * 1024), 16,
                                                     woff[i], kk * (MB_BK * 2), 0, 0);
    };
    // lane (n, g) reads row n of a group, piece 4 s + g of the stage's eight, which lies at that piece ^ (n >> 1)
    const int rd0 = n * 128 + ((g ^ (n >> 1)) * 16), rd1 = n * 128 + (((4 + g) ^ (n >> 1)) * 16);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lds);
    const uint32_t x0 = lds0 + MB_X + wm * 2048, w0 = lds0 + MB_W + wn * 8192;
    typedef const mt_bf16x8_t __attribute__((address_space(3)))* frag_t;
    mt_float4_t acc[4][NB];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = mt_float4_t{0.f, 0.f, 0.f, 0.f};
    struct Frags { mt_bf16x8_t w[4], x[NB]; };
    Frags fa, fb;
    auto read = [&](Frags& f, uint32_t wb, uint32_t xb) {
#pragma unroll
        for (int a = 0; a < 4; ++a) f.w[a] = *(frag_t)(uintptr_t)(wb + a * 2048);
#pragma unroll
        for (int b = 0; b < NB; ++b) f.x[b] = *(frag_t)(uintptr_t)(xb + b * 4096);
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int a = 0; a < 4; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f.w[a], f.x[b], acc[a][b], 0, 0, 0);
    };

    copy_x(0);
    copy_w(0, 0);
    if (nk > 1) {
        copy_x(1);
        copy_w(1, 1);
    }
    if (nk > 2) copy_w(2, 2);
    if (nk > 2) mb_wait<NX + 8, 15>(); else mb_wait<0, 15>();
    mb_wait<15, 0>();                                          // (no reads are; the compiled branches of two sizes meet here)
    __builtin_amdgcn_s_barrier();
    read(fa, w0 + rd0, x0 + rd0);

    int ring = 0;                                              // it % 3
    auto step = [&](int it, auto steady_c) {
        constexpr bool steady = decltype(steady_c)::value;
        const uint32_t wb = w0 + ring * MB_UNIT, xb = x0 + (it & 1) * MB_UNIT;
        const int next = ring == 2 ? 0 : ring + 1;
        read(fb, wb + rd1, xb + rd1);
        multiply(fa);
        if constexpr (steady) {
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (steady) mb_wait<4, 0>(); else mb_wait<0, 0>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (steady || it + 2 < nk) copy_x(it + 2);
        if (steady || it + 3 < nk) copy_w(it + 3, ring);
        if (steady || it + 1 < nk) read(fa, w0 + next * MB_UNIT + rd0, x0 + ((it + 1) & 1) * MB_UNIT + rd0);
        if (steady || it + 1 < nk || K % MB_BK == 0) multiply(fb);
        if constexpr (steady) {
            __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (b == 0 && NX + 4 > NB) __builtin_amdgcn_sched_group_barrier(0x020, NX + 4 > NB ? NX + 4 - NB : 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        }
        ring = next;
    };
    using std::integral_constant;
    int it = 0;
    for (; it + 3 < nk; ++it) step(it, integral_constant<bool, true>{});
    for (; it < nk; ++it) step(it, integral_constant<bool, false>{});
    MFMA_SETTLE();

    // acc[a][b][c]: row 16 (wm + 2 b) + n of the tile, W row 64 wn + 16 a + 4 g + c of the workgroup's 256. A wave's results go through
    // a part of LDS that is its own, four groups of rows at a time, so that what forms and stores them is a loop, and what is stored
    // runs of 64 or 128 bytes. (Written out for all of a lane's results it was up to 30 KB of instructions for each count of groups,
    // and a tile waited for them: 32 experts, 12,432 pairs, routed by a model, gate-up 764 -> 739 us, 8,000 pairs, down 288 -> 276.)
    __syncthreads();                                           // every wave has read the last stage
    const uint32_t own = lds0 + wave * (64 * MB_RS * 4);
    typedef mt_float4_t __attribute__((address_space(3)))* put_t;
#pragma unroll
    for (int b0 = 0; b0 < NB; b0 += 4) {
        constexpr int MOST = NB < 4 ? NB : 4;
        const int groups = b0 + MOST < NB ? MOST : NB - b0;
#pragma unroll
        for (int b = 0; b < MOST; ++b)
            if (b0 + b < NB)
#pragma unroll
                for (int a = 0; a < 4; ++a) *(put_t)(uintptr_t)(own + ((b * 16 + n) * MB_RS + 16 * a + 4 * g) * 4) = acc[a][b0 + b];
        MB_WAVE_SYNC();
        mb_store<GATED>(own, lane, wm + 2 * b0, groups, n_rows, pairs, y, N, GATED ? n0 + wn * 32 : n0 + wn * 64, act);
        MB_WAVE_SYNC();
    }
}

template <bool GATED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void moe_tile_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ meta, int x_rows, int N, int K, int top_div, int tiles_n, const MoeAct act) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int tiles_m = meta[0], total = tiles_m * tiles_n;
    int item;
    {
        const int id = blockIdx.x, xcd = id & 7, slot = id >> 3, q = total >> 3, r = total & 7;
        if (slot >= q + (xcd < r ? 1 : 0)) return;
        item = xcd * q + min(xcd, r) + slot;
    }
    const int span = 2 * tiles_n, grp = item / span, in = item - grp * span, gsize = min(tiles_m - 2 * grp, 2);
    const int mt = 2 * grp + in % gsize, nt = in / gsize;
    const int e = tiles[3 * mt], at = tiles[3 * mt + 1], n_rows = tiles[3 * mt + 2];
    constexpr int CN = GATED ? 128 : 256;                      // result columns of the workgroup
    const int n0 = nt * CN;

    const size_t w_rows = GATED ? 2 * (size_t)N : (size_t)N;
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, x_rows * K * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t wres =
        __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)e * w_rows * K), 0, (int)(w_rows * K * 2), 0x00020000);
    // a copy brings 8 rows: lane l writes piece l & 7 of row l >> 3, and reads the piece that belongs there
    const int r8 = lane >> 3;
    int xoff[4], woff[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int xr = 8 * (wave + 8 * i) + r8, row = 32 * wave + 8 * i + r8;
        const int p = order[at + min(xr, n_rows - 1)];
        xoff[i] = (int)(((size_t)(p / top_div) * K + ((lane & 7) ^ ((xr >> 1) & 7)) * 8) * 2);
        size_t wr;
        if constexpr (GATED) {
            const int t4 = (row >> 4) & 3, col = n0 + (row >> 6) * 32 + (t4 & 1) * 16 + (row & 15);
            wr = (size_t)(t4 >> 1) * N + min(col, N - 1);
        } else {
            wr = min(n0 + row, N - 1);
        }
        woff[i] = (int)((wr * K + ((lane & 7) ^ ((row >> 1) & 7)) * 8) * 2);
    }
    const int groups = (n_rows + 15) >> 4;
#define MB_GO(NB_) mb_tile<GATED, NB_>(lds, xres, wres, xoff, woff, K, wave, lane, y, order + at, n_rows, n0, N, act)
    if (groups <= 2) MB_GO(1);
    else if (groups <= 4) MB_GO(2);
    else if (groups <= 8) MB_GO(4);
    else if (groups <= 10) MB_GO(5);
    else if (groups <= 12) MB_GO(6);
    else if (groups <= 14) MB_GO(7);
    else MB_GO(8);
#undef MB_GO
}

int moe_tile_launch(hipStream_t st, const bf16* x, const bf16* w, bf16* y, const int* order, const int* tiles,
                    const int* meta, int max_tiles, int x_rows, int N, int K, int top_div, bool gated, const MoeAct& act) {
    const int tiles_n = (N + (gated ? 127 : 255)) / (gated ? 128 : 256);
    const long long total = (long long)max_tiles * tiles_n;
    if (total > 0x7fffffff || K % 32) return RA_ERR_ARG;
    const void* kernel = gated ? (const void*)moe_tile_kernel<true> : (const void*)moe_tile_kernel<false>;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MB_LDS) != hipSuccess) return RA_ERR_LAUNCH;
    if (gated)
        hipLaunchKernelGGL(moe_tile_kernel<true>, dim3((unsigned)total), dim3(512), MB_LDS, st, x, w, y, order, tiles, meta, x_rows, N, K,
                           top_div, tiles_n, act);
    else
        hipLaunchKernelGGL(moe_tile_kernel<false>, dim3((unsigned)total), dim3(512), MB_LDS, st, x, w, y, order, tiles, meta, x_rows, N, K,
                           top_div, tiles_n, act);
    return ra_launch_status();
}
