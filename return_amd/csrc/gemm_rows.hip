// y = x W^T for 17 to 64 rows of x, bfloat16 in, 32-bit sums: the products of a decode step of many requests, which are bound
// by reading W once. Layout of the reference's F.linear (rollout/monkey_patch/qwen3.py:21): x [M, K], W [N, K], y [M, N].
//
// A workgroup of four waves has 16 G rows of W (16 G result columns, or the gate and up rows of 8 G) and all rows of x. Steps of
// 128 columns of K go straight from memory into LDS (buffer_load ... lds), into as many stages as LDS has room for, so that
// 60 to 100 KB of a CU's loads are on their way at any time. A step's four runs of 32 columns belong to one wave each: every
// wave multiplies all rows by all columns of its run, so that LDS is read once, and the four sums are added through LDS at the
// end, in the order of the waves. A row of a stage is 256 bytes, whose 16-byte pieces lie at the piece's number xor the row's, so that
// neither the copies nor the reads meet a bank twice; one barrier a step, in front of which a wave has read all it asked for.
//
// A workgroup begins with a step of its own and goes once round K from there: if all began at column 0, the rows of W, which lie a
// power of two apart on most shapes, would be asked of the same few memory channels at the same time. Neighbours on an XCD begin one
// step apart. Gate-up of 12,288 columns of 4,096 at 64 rows 44.3 -> 39.0 us with that (W at 5.2 TB/s, launch and end included; the
// library's product and the SiLU-mul behind it 55), at 32 rows 44.9 -> 37.1; head of 151,936 x 4,096 280 -> 241 (library 273);
// down 4,096 x 12,288 in four pieces of K 24 -> 23 (library 27), o 4,096 x 4,096 in four 10.6 (13.6). With few columns a CU
// (q/k/v 6,144 x 4,096: 24) x is most of what a CU takes in, and the library's product is as fast (18.5 / 17.6).
// From 16 MB on W is read past the caches: gate-up 39.0 -> 36.9, head 243 -> 233.
#include "common.h"
#include <type_traits>

typedef __bf16 gr_b8 __attribute__((ext_vector_type(8)));
typedef float gr_f4 __attribute__((ext_vector_type(4)));

#define GR_KSTEP 128
#define GR_ROW 256                        // bytes of a row in a stage
#define GR_LDS 163840

// stages of LDS for NB blocks of 16 rows of x and G of W
static constexpr int gr_stages(int nb, int g) {
    const int s = GR_LDS / ((nb + g) * 16 * GR_ROW);
    return s < 8 ? s : 8;
}

// Waits until at most COPIES of the wave's copies are on their way, and none of its LDS reads. (A barrier waits for neither.)
template <int COPIES>
__device__ __forceinline__ void gr_wait() {
    static_assert(COPIES < 64, "field of s_waitcnt");
    __builtin_amdgcn_s_waitcnt(0x0070 | (COPIES & 15) | ((COPIES >> 4) << 14));        // (expcnt at its maximum)
}

template <int NB, int G, bool GATED, bool AWAY, typename TO>
__device__ __forceinline__ void gr_tile(unsigned char* lds, const bf16* __restrict__ X, const bf16* __restrict__ W, TO* __restrict__ C,
                                        int M, int N, int K, int tiles, int k_steps) {
    constexpr int S = gr_stages(NB, G), STAGE = (NB + G) * 16 * GR_ROW, NC = NB + G;      // (copies a wave and step: NC)
    constexpr int H = GATED ? G / 2 : G;                                                  // blocks of result columns
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
    const int z = blockIdx.x / tiles, n0 = (blockIdx.x - z * tiles) * 16 * H;
    const int first = z * k_steps, nk = min(k_steps, K / GR_KSTEP - first), begin = (int)((blockIdx.x >> 3) % nk);
    const size_t rb = (size_t)K * 2;
    const int w_rows = min(16 * H, N - n0);
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)X, 0, (int)(M * rb), 0x00020000);
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc((void*)(W + (size_t)n0 * K), 0, (int)(w_rows * rb), 0x00020000);
    const __amdgpu_buffer_rsrc_t ures =
        __builtin_amdgcn_make_buffer_rsrc((void*)(W + (size_t)(n0 + (GATED ? N : 0)) * K), 0, (int)(w_rows * rb), 0x00020000);
    // copy i brings rows 16 i + 4 wave .. + 3 of a stage (x first, then W's): lane l writes piece l & 15 of row l >> 4 of them and
    // reads the piece that belongs there. Rows beyond the last are the last one again.
    const int r16 = 4 * wave + (lane >> 4), piece = (lane & 15) ^ r16;
    int off[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int r = i < NB ? min(16 * i + r16, M - 1) : min(16 * ((i - NB) % H) + r16, w_rows - 1);
        off[i] = (int)(r * rb) + first * GR_ROW + piece * 16;
    }
    auto copy = [&](int step, int stage) {
        int at = step + begin;
        at = (at >= nk ? at - nk : at) * GR_ROW;
#pragma unroll
        for (int j = 0; j < NC; ++j) {
            const int i = NC - 1 - j;                          // W first: it comes from further away
            void __attribute__((address_space(3)))* to =
                (void __attribute__((address_space(3)))*)(lds + stage * STAGE + (16 * i + 4 * wave) * GR_ROW);
            if (i < NB) __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, to, 16, off[i], at, 0, 0);
            else if (i < NB + H) __builtin_amdgcn_raw_ptr_buffer_load_lds(wres, to, 16, off[i], at, 0, AWAY ? 2 : 0);
            else __builtin_amdgcn_raw_ptr_buffer_load_lds(ures, to, 16, off[i], at, 0, AWAY ? 2 : 0);
        }
    };
    gr_f4 acc[G][NB];
#pragma unroll
    for (int a = 0; a < G; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = gr_f4{0.f, 0.f, 0.f, 0.f};
    // lane (n, g) reads row n of a block, piece 4 wave + g
    const uint32_t rd = (uint32_t)(uintptr_t)lds + n * GR_ROW + (((4 * wave + g) ^ n) * 16);
    typedef const gr_b8 __attribute__((address_space(3)))* frag_t;
#pragma unroll
    for (int s = 0; s < S - 1; ++s)
        if (s < nk) copy(s, s);
    int stage = 0;
    auto step = [&](int it, auto steady_c) {
        constexpr bool steady = decltype(steady_c)::value;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (steady) gr_wait<(S - 2) * NC>(); else gr_wait<0>();      // the step's copies have landed
        __builtin_amdgcn_s_barrier();                                          // everyone's, and the step before is read
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (steady) copy(it + S - 1, stage == 0 ? S - 1 : stage - 1);
        const uint32_t at = rd + stage * STAGE;
        gr_b8 x[NB], w[G];
#pragma unroll
        for (int b = 0; b < NB; ++b) x[b] = *(frag_t)(uintptr_t)(at + b * 16 * GR_ROW);
#pragma unroll
        for (int a = 0; a < G; ++a) w[a] = *(frag_t)(uintptr_t)(at + (NB + a) * 16 * GR_ROW);
#pragma unroll
        for (int a = 0; a < G; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[a], x[b], acc[a][b], 0, 0, 0);
        stage = stage + 1 == S ? 0 : stage + 1;
    };
    int it = 0;
    for (; it + S - 1 < nk; ++it) step(it, std::integral_constant<bool, true>{});
    for (; it < nk; ++it) step(it, std::integral_constant<bool, false>{});
    MFMA_SETTLE();

    // acc[a][b][c] of a wave: its share of row 16 b + n, row 16 a + 4 g + c of the workgroup's rows of W
    static_assert(G * NB * 4096 <= S * STAGE, "the waves' sums lie where the stages lay");
    gr_f4* sums = reinterpret_cast<gr_f4*>(lds);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < G * NB; ++p) sums[(p * 4 + wave) * 64 + lane] = acc[p / NB][p % NB];
    __syncthreads();
    auto total = [&](int a, int b) {
        const gr_f4* s = sums + (a * NB + b) * 256 + lane;
        return ((s[0] + s[64]) + s[128]) + s[192];
    };
    TO* out = C + (size_t)z * M * N;
    for (int q = wave; q < H * NB; q += 4) {
        const int a = q / NB, b = q % NB, m = 16 * b + n, col = n0 + 16 * a + 4 * g;
        gr_f4 v = total(a, b);
        if constexpr (GATED) {
            const gr_f4 up = total(a + H, b);
#pragma unroll
            for (int c = 0; c < 4; ++c) v[c] = v[c] / (1.0f + expf(-v[c])) * up[c];     // gate and up stay 32-bit until here
        }
        if (m >= M) continue;
        TO* dst = out + (size_t)m * N + col;
        if (col + 3 < N && (N & 3) == 0) {
            if constexpr (sizeof(TO) == 4) {
                *reinterpret_cast<gr_f4*>(dst) = v;
            } else {
                uint2 pk;
                pk.x = (uint32_t)f2bf_bits(v[0]) | ((uint32_t)f2bf_bits(v[1]) << 16);
                pk.y = (uint32_t)f2bf_bits(v[2]) | ((uint32_t)f2bf_bits(v[3]) << 16);
                *reinterpret_cast<uint2*>(dst) = pk;
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (col + c < N) dst[c] = from_f<TO>(v[c]);
        }
    }
}

template <int NB, int G, bool GATED, bool AWAY, typename TO>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const bf16* __restrict__ X, const bf16* __restrict__ W, TO* __restrict__ C, int M,
                                                        int N, int K, int tiles, int k_steps) {
    extern __shared__ __attribute__((aligned(1024))) unsigned char lds[];
    gr_tile<NB, G, GATED, AWAY, TO>(lds, X, W, C, M, N, K, tiles, k_steps);
}

// What the kernel takes: operands 16-byte aligned.
extern "C" int ra_gemm_rows_fits(int M, int N, int K) {
    return M > 16 && M <= 64 && N > 0 && K > 0 && K % GR_KSTEP == 0 && (long long)K * 256 <= 0x7fffffffll;
}

// C [M, N] (bf16 or fp32), gated: W is [2N, K], C = silu(x Wg^T) * (x Wu^T) in bfloat16. pieces > 1: C fp32 [pieces, M, N], share
// i from the i-th run of K's steps (every run has at least one).
extern "C" int ra_gemm_rows_bf16(const void* X, const void* W, void* C, int M, int N, int K, int gated, int pieces, int out_dtype, int cus,
                                 void* stream) {
    if (!ra_gemm_rows_fits(M, N, K) || pieces < 1 || cus < 1 || (((uintptr_t)X | (uintptr_t)W | (uintptr_t)C) & 15) != 0) return RA_ERR_ARG;
    if (out_dtype != RA_DTYPE_F32 && out_dtype != RA_DTYPE_BF16) return RA_ERR_ARG;
    if ((gated || pieces > 1) && (out_dtype == RA_DTYPE_F32) == (gated != 0)) return RA_ERR_ARG;
    if (gated && pieces > 1) return RA_ERR_ARG;
    const int all = K / GR_KSTEP, k_steps = (all + pieces - 1) / pieces;
    if ((all + k_steps - 1) / k_steps != pieces) return RA_ERR_ARG;
    const int nb = (M + 15) / 16;
    // Columns of a workgroup: those with which the rounds over the CUs take the least, a round as its blocks of W and one and a half
    // more (gate-up as above, G 4 / 6 / 8: 49 / 39 / 42 us in 2 / 1 / 1 rounds).
    int G = 2;
    long long tiles = 0;
    double best = 0;
    for (int c = 2; c <= 8; c += 2) {
        const int cols = gated ? 8 * c : 16 * c;
        const long long t = ((long long)N + cols - 1) / cols;
        const double cost = (double)((t * pieces + cus - 1) / cus) * (c + 1.5);
        if (c == 2 || cost < best) {
            best = cost;
            G = c;
            tiles = t;
        }
    }
    if (tiles * pieces > 0x7fffffff) return RA_ERR_ARG;
    const dim3 grid((unsigned)(tiles * pieces)), block(256);
    const int lds = gr_stages(nb, G) * (nb + G) * 16 * GR_ROW;
    hipStream_t st = (hipStream_t)stream;
    // (a small W may well lie in the caches from the step before, and stays there: 1,024 x 512 at 64 rows 4.1 us, read past them 4.6)
    const bool away = 2ll * N * K * (gated ? 2 : 1) >= 16ll << 20;
#define GR_GO(NB_, G_, GATED_, T_)                                                                                                      \
    do {                                                                                                                                \
        const auto kern = away ? gemm_rows_kernel<NB_, G_, GATED_, true, T_> : gemm_rows_kernel<NB_, G_, GATED_, false, T_>;            \
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)    \
            return RA_ERR_LAUNCH;                                                                                                       \
        hipLaunchKernelGGL(kern, grid, block, lds, st, (const bf16*)X, (const bf16*)W, (T_*)C, M, N, K, (int)tiles, k_steps);           \
    } while (0)
#define GR_G(NB_, GATED_, T_)                      \
    do {                                           \
        if (G == 2) GR_GO(NB_, 2, GATED_, T_);     \
        else if (G == 4) GR_GO(NB_, 4, GATED_, T_); \
        else if (G == 6) GR_GO(NB_, 6, GATED_, T_); \
        else GR_GO(NB_, 8, GATED_, T_);            \
    } while (0)
#define GR_NB(GATED_, T_)                   \
    do {                                    \
        if (nb == 2) GR_G(2, GATED_, T_);   \
        else if (nb == 3) GR_G(3, GATED_, T_); \
        else GR_G(4, GATED_, T_);           \
    } while (0)
    if (gated) GR_NB(true, bf16);
    else if (out_dtype == RA_DTYPE_F32) GR_NB(false, float);
    else GR_NB(false, bf16);
#undef GR_NB
#undef GR_G
#undef GR_GO
    return ra_launch_status();
}
