// The experts' products for many rows an expert, bfloat16: tiles of up to 256 rows of one expert by 256 rows of its W.
//
// The scheme is that of the tiled product for many rows (gemm_tile.hip): k-steps of 32, eight waves as 2 x 4, operands
// copied straight into LDS (buffer_load ... lds) four stages deep, 16-byte pieces of a row rotated by the copying lane's
// choice of address so that the reads meet no bank conflict, the next step's operands read between this step's MFMAs.
// What differs: rows of x are gathered by pair; W comes from the tile's expert; gated, of a wave's four tiles of W rows
// the first two are gate rows and the last two the up rows of the same columns, so that a lane holds both halves of a
// result; and a tile has as many groups of 16 rows as its expert left it (the plan cuts an expert's rows into even tiles).
// Wave row wm takes the groups wm, wm + 2, ...; the loop is compiled for each count of groups a wave, so that a tile of
// 100 rows issues the MFMAs and copies of 128 rows and not of 256.
//
// Workgroups go to the XCDs round-robin: an XCD gets a run of consecutive (row tile, column tile) pairs, two row tiles
// (mostly of one expert, whose W they then share in L2) at a time through all columns.
//
// Why: with tiles of 128 x 128 staged through registers (what this replaces for K % 32 == 0) every k-step moved 16 KB
// for 64 MFMAs of a workgroup; here it is 24 to 32 KB for 160 to 256. Measured, gate-up of 32 experts
// of 6,144 x 4,096, four a token: 8,192 pairs 638 us (0.65 PFLOP/s) where the smaller tiles took 1,150, 12,432 pairs 731 (0.86)
// against 1,409, 32,000 pairs 1,802 (0.89) against 3,192. At 2,000 pairs and fewer the time is the reading of W: 300 to 345 us for
// 1.6 GB (5.4 TB/s at 480 pairs), where operands straight from memory took 415 to 790. What is lost at 8,192 pairs is the last
// rounds of tiles: half of the experts have a few rows more than 256 and so two tiles of 140.
#include "moe_tile.h"
#include <type_traits>

typedef __bf16 mt_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float mt_float4_t __attribute__((ext_vector_type(4)));

#define MB_BK 32
#define MB_HALF (256 * MB_BK * 2)                // bytes of one operand's tile in a stage (16 KB)
#define MB_STAGE (2 * MB_HALF)
#define MB_LDS (4 * MB_STAGE)                    // 128 KB

// Waits until at most COPIES of the wave's copies and READS of its LDS reads are on their way (the last ones: both finish in
// their order). A barrier waits for neither.
template <int COPIES, int READS>
__device__ __forceinline__ void mb_wait() {
    static_assert(COPIES < 16 && READS < 16, "fields of s_waitcnt");
    __builtin_amdgcn_s_waitcnt(0x0070 | COPIES | (READS << 8));        // (expcnt at its maximum)
}

// A tile of 32 NB rows at most. xoff: where this lane's rows of x begin (bytes), one for each of its copies.
template <bool GATED, int NB>
__device__ __forceinline__ void mb_tile(unsigned char* lds, const __amdgpu_buffer_rsrc_t xres, const __amdgpu_buffer_rsrc_t wres,
                                        const int (&xoff)[2], const int (&woff)[2], int nk, int wave, int lane, bf16* __restrict__ y,
                                        const int* __restrict__ pairs, int n_rows, int n0, int N, const MoeAct& act) {
    constexpr int NX = NB > 4 ? 2 : 1, PER = 2 + NX;           // copies of x, and of both, a wave and stage
    const int n = lane & 15, g = lane >> 4, wm = wave >> 2, wn = wave & 3;
    auto copy_stage = [&](int s, int kk) {
        unsigned char* base = lds + s * MB_STAGE;
        const int soff = kk * (MB_BK * 2);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, (void __attribute__((address_space(3)))*)(base + MB_HALF + (2 * wave + i) * 1024),
                                                     16, woff[i], soff, 0, 0);
#pragma unroll
        for (int i = 0; i < NX; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (void __attribute__((address_space(3)))*)(base + (wave + 8 * i) * 1024), 16,
                                                     xoff[i], soff, 0, 0);
    };
    // lane (n, g) reads row n of a group, piece g of the k-step, which lies at piece g ^ (n >> 2); a wave's groups of x
    // are wm, wm + 2, ... (two bases each, 64 KB apart: a read's offset fits the instruction's 16 bits)
    const int rd = n * 64 + ((g ^ ((n >> 2) & 3)) * 16);
    uint32_t xrd_lo = (uint32_t)(uintptr_t)(lds) + wm * 1024 + rd, xrd_hi = xrd_lo + 2 * MB_STAGE;
    uint32_t wrd_lo = (uint32_t)(uintptr_t)(lds) + MB_HALF + (wn * 64) * 64 + rd, wrd_hi = wrd_lo + 2 * MB_STAGE;
    asm volatile("" : "+v"(xrd_lo), "+v"(xrd_hi), "+v"(wrd_lo), "+v"(wrd_hi));
    typedef const mt_bf16x8_t __attribute__((address_space(3)))* frag_t;
    auto read_x = [&](int s, int b) { return *(frag_t)(uintptr_t)((s < 2 ? xrd_lo : xrd_hi) + (s & 1) * MB_STAGE + b * 2048); };
    auto read_w = [&](int s, int a) { return *(frag_t)(uintptr_t)((s < 2 ? wrd_lo : wrd_hi) + (s & 1) * MB_STAGE + a * 1024); };

    mt_float4_t acc[4][NB];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = mt_float4_t{0.f, 0.f, 0.f, 0.f};

    copy_stage(0, 0);
    if (nk > 1) copy_stage(1, 1);
    if (nk > 2) copy_stage(2, 2);
    if (nk > 2) mb_wait<PER, 15>(); else mb_wait<0, 15>();
    mb_wait<15, 0>();                                          // (no reads are; the compiled branches of two sizes meet here)
    __builtin_amdgcn_s_barrier();
    mt_bf16x8_t fwA[4], fxA[NB], fwB[4], fxB[NB];
#pragma unroll
    for (int a = 0; a < 4; ++a) fwA[a] = read_w(0, a);
#pragma unroll
    for (int b = 0; b < NB; ++b) fxA[b] = read_x(0, b);

    // Step it's operands are in registers, stage it + 1 is in LDS and is read meanwhile, stages it + 2 and it + 3 are on their
    // way. A step refills the stage of step it - 1, which was read in step it - 2: every wave has to have finished those reads
    // when it passes the barrier behind step it - 1, so at a step's end a wave waits until only that step's own reads are on
    // their way. (Two stages asked for in every other step, the halves of the same 128-byte lines, would refill a stage behind
    // the very barrier before which it was read: the wait for the reads cost that form 2 to 6 % at 2,000 to 12,000 pairs.)
    auto step = [&](int it, auto stage_c, auto steady_c, mt_bf16x8_t (&fw_c)[4], mt_bf16x8_t (&fx_c)[NB], mt_bf16x8_t (&fw_n)[4],
                    mt_bf16x8_t (&fx_n)[NB]) {
        constexpr int stage = decltype(stage_c)::value;
        constexpr bool steady = decltype(steady_c)::value;
        constexpr int nxt = (stage + 1) & 3;
        const bool more = steady || it + 1 < nk;
        if (steady || it + 3 < nk) copy_stage((stage + 3) & 3, it + 3);
        if (more) {
#pragma unroll
            for (int a = 0; a < 4; ++a) fw_n[a] = read_w(nxt, a);
            fx_n[0] = read_x(nxt, 0);
            if constexpr (NB > 1) fx_n[NB > 1] = read_x(nxt, 1);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int a = 0; a < 4; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw_c[a], fx_c[b], acc[a][b], 0, 0, 0);
            if (more && b + 2 < NB) fx_n[b + 2] = read_x(nxt, b + 2);
        }
        if constexpr (steady) {
            __builtin_amdgcn_sched_group_barrier(0x100, NB > 1 ? 6 : 5, 0);
#pragma unroll
            for (int b = 0; b + 2 < NB; ++b) {
                __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                if (b < PER) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        }
        if constexpr (steady) mb_wait<PER, 4 + NB>();
        else mb_wait<0, 0>();
        __builtin_amdgcn_s_barrier();
    };
    using std::integral_constant;
    constexpr integral_constant<bool, true> yes{};
    constexpr integral_constant<bool, false> no{};
    int it = 0;
    for (; it + 6 < nk; it += 4) {
        step(it, integral_constant<int, 0>{}, yes, fwA, fxA, fwB, fxB);
        step(it + 1, integral_constant<int, 1>{}, yes, fwB, fxB, fwA, fxA);
        step(it + 2, integral_constant<int, 2>{}, yes, fwA, fxA, fwB, fxB);
        step(it + 3, integral_constant<int, 3>{}, yes, fwB, fxB, fwA, fxA);
    }
    for (; it < nk; it += 4) {
        step(it, integral_constant<int, 0>{}, no, fwA, fxA, fwB, fxB);
        if (it + 1 < nk) step(it + 1, integral_constant<int, 1>{}, no, fwB, fxB, fwA, fxA);
        if (it + 2 < nk) step(it + 2, integral_constant<int, 2>{}, no, fwA, fxA, fwB, fxB);
        if (it + 3 < nk) step(it + 3, integral_constant<int, 3>{}, no, fwB, fxB, fwA, fxA);
    }
    MFMA_SETTLE();

    // acc[a][b][c]: row 16 (wm + 2 b) + n of the tile, W row 64 wn + 16 a + 4 g + c of the workgroup's 256
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const int m = 16 * (wm + 2 * b) + n;
        if (m >= n_rows) continue;
        const int p = pairs[m];
        bf16* yr = y + (size_t)p * N;
        const float scale = GATED && act.in_scale != nullptr ? act.in_scale[p] : 1.0f;
#pragma unroll
        for (int a = 0; a < (GATED ? 2 : 4); ++a) {
            const int col = GATED ? n0 + wn * 32 + a * 16 + 4 * g : n0 + wn * 64 + a * 16 + 4 * g;
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                v[c] = acc[a][b][c];
                if constexpr (GATED) v[c] = moe_gate<bf16>(acc[a][b][c], acc[a + 2][b][c], act, scale);
            }
            if (col + 3 < N && (N & 3) == 0) {
                uint2 pk;
                pk.x = (uint32_t)f2bf_bits(v[0]) | ((uint32_t)f2bf_bits(v[1]) << 16);
                pk.y = (uint32_t)f2bf_bits(v[2]) | ((uint32_t)f2bf_bits(v[3]) << 16);
                *reinterpret_cast<uint2*>(yr + col) = pk;
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (col + c < N) yr[col + c] = from_f<bf16>(v[c]);
            }
        }
    }
}

template <bool GATED>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void moe_tile_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ meta, int N, int K, int top_div, int tiles_n, const MoeAct act) {
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
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)x, 0, 0x7fffff00, 0x00020000);
    const __amdgpu_buffer_rsrc_t wres =
        __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)e * w_rows * K), 0, (int)(w_rows * K * 2), 0x00020000);
    // a copy brings 16 rows: lane l writes piece l & 3 of row l >> 2, and reads the piece that belongs there
    const int r16 = lane >> 2, pc = (lane & 3) ^ ((r16 >> 2) & 3);
    int xoff[2], woff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int p = order[at + min(16 * (wave + 8 * i) + r16, n_rows - 1)];
        xoff[i] = (int)(((size_t)(p / top_div) * K + pc * 8) * 2);
        const int row = 32 * wave + 16 * i + r16;
        size_t wr;
        if constexpr (GATED) {
            const int t4 = (row >> 4) & 3, col = n0 + (row >> 6) * 32 + (t4 & 1) * 16 + (row & 15);
            wr = (size_t)(t4 >> 1) * N + min(col, N - 1);
        } else {
            wr = min(n0 + row, N - 1);
        }
        woff[i] = (int)((wr * K + pc * 8) * 2);
    }
    const int nk = K / MB_BK, groups = (n_rows + 15) >> 4;
#define MB_GO(NB_) mb_tile<GATED, NB_>(lds, xres, wres, xoff, woff, nk, wave, lane, y, order + at, n_rows, n0, N, act)
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
                    const int* meta, int max_tiles, int N, int K, int top_div, bool gated, const MoeAct& act) {
    const int tiles_n = (N + (gated ? 127 : 255)) / (gated ? 128 : 256);
    const long long total = (long long)max_tiles * tiles_n;
    if (total > 0x7fffffff || K % MB_BK) return RA_ERR_ARG;
    const void* kernel = gated ? (const void*)moe_tile_kernel<true> : (const void*)moe_tile_kernel<false>;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MB_LDS) != hipSuccess) return RA_ERR_LAUNCH;
    if (gated)
        hipLaunchKernelGGL(moe_tile_kernel<true>, dim3((unsigned)total), dim3(512), MB_LDS, st, x, w, y, order, tiles, meta, N, K,
                           top_div, tiles_n, act);
    else
        hipLaunchKernelGGL(moe_tile_kernel<false>, dim3((unsigned)total), dim3(512), MB_LDS, st, x, w, y, order, tiles, meta, N, K,
                           top_div, tiles_n, act);
    return ra_launch_status();
}
