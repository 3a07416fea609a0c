// y = x W^T in float32 for many rows, on the bfloat16 matrix units: every float32 operand is taken apart into three bfloat16
// parts, exactly (a float32 has 24 significant bits, a bfloat16 8; the first part is the value cut off after 8 bits, the second
// what is left cut off after 8, the third the rest), and a product is the six products of parts that reach above 2^-24 of it:
// hi hi in one accumulator, lo hi + hi lo + mid mid + mid hi + hi mid in another. The first accumulator is rounded once in 16
// columns of K, where a 32-bit matrix instruction rounds once in 2 or 4, the second is 2^-8 as large. Errors against 64 bits,
// 2-norm of the difference over 2-norm of the result, this kernel / the library's float32 product on normal inputs:
// K 256 1.1e-7 / 2.9e-7, 4,096 1.6e-7 / 1.15e-6, 12,288 2.5e-7 / 2.0e-6; on positive inputs 1e-7 / 2.3e-7 to 1.7e-6. A value
// that comes out as no number or as infinite is formed again by 32-bit FMAs over the operands themselves (an infinite operand
// has no parts), and so is one below 2^-64 that is not zero: the matrix units take a part below 2^-126 as zero, which is 2^-126
// times the other operand, and no more than 2^-24 of a larger sum while K times the largest operand is below 2^38.
//
// Bound by the matrix units: six 32x32x16 products where there is one in bfloat16. x is taken apart once, by a kernel of its
// own, into blocks of [rows of a tile][16 columns] that lie in memory as LDS holds them; W is taken apart on its way into LDS
// (44 vector instructions a thread beside 24 matrix instructions), since its parts would be 1.5 times its size to write and read.
// A workgroup has four waves and a tile of 64 MB x 128, a wave 32 MB x 64 of it (MB blocks by 2 of 32 x 32 results, in two
// accumulators); two workgroups a CU, so that one's barriers and copies run beside the other's products. LDS holds two steps of
// 16 columns, [side][part][half of the columns][row], 8 columns (16 bytes) an entry: a wave's operand is 64 entries side by
// side. The second half lies 64 bytes on, so that the two lanes that write one row of W meet different banks. Operands come from
// memory 32 columns (a 128-byte line of a row of W) at a time, asked for one such block ahead.
#include "common.h"

typedef __bf16 sp_b8 __attribute__((ext_vector_type(8)));
typedef float sp_f16 __attribute__((ext_vector_type(16)));
typedef float sp_f4 __attribute__((ext_vector_type(4)));
typedef unsigned sp_u4 __attribute__((ext_vector_type(4)));

#define SP_BN 128                                         // columns of a tile
#define SP_KB 32                                          // columns of K that are asked for at a time

// the three parts of eight floats: the upper halves of each pair side by side
__device__ __forceinline__ void sp_parts(sp_f4 a, sp_f4 b, sp_u4 (&p)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float u = i < 2 ? a[2 * i] : b[2 * i - 4], v = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
        const unsigned ub = __float_as_uint(u), vb = __float_as_uint(v);
        p[0][i] = __builtin_amdgcn_perm(vb, ub, 0x07060302);
        const float u1 = u - __uint_as_float(ub & 0xffff0000u), v1 = v - __uint_as_float(vb & 0xffff0000u);
        const unsigned u1b = __float_as_uint(u1), v1b = __float_as_uint(v1);
        p[1][i] = __builtin_amdgcn_perm(v1b, u1b, 0x07060302);
        p[2][i] = __builtin_amdgcn_perm(__float_as_uint(v1 - __uint_as_float(v1b & 0xffff0000u)),
                                        __float_as_uint(u1 - __uint_as_float(u1b & 0xffff0000u)), 0x07060302);
    }
}

// x [M, K] -> its parts, [tile of BM rows][16 columns][part][half][row][8], rows from M on zeros. A wave takes 16 rows x 32
// columns: 128-byte lines in, 256-byte runs out.
template <int BM>
__global__ __launch_bounds__(256) void split_rows_kernel(const float* __restrict__ x, sp_u4* __restrict__ parts, int M, int K) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row = blockIdx.y * 16 + (lane & 15);
    const int k = (blockIdx.x * 4 + wave) * 32 + 8 * (lane >> 4);
    if (k >= K) return;
    sp_u4 p[3];
    sp_f4 a = {0.f, 0.f, 0.f, 0.f}, b = a;
    if (row < M) {
        const sp_f4* src = reinterpret_cast<const sp_f4*>(x + (size_t)row * K + k);
        a = src[0];
        b = src[1];
    }
    sp_parts(a, b, p);
    const int t = row / BM, r = row - t * BM;
    sp_u4* dst = parts + (((size_t)t * (K / 16) + k / 16) * 3 * 2 + ((k >> 3) & 1)) * BM + r;
#pragma unroll
    for (int j = 0; j < 3; ++j) dst[(size_t)j * 2 * BM] = p[j];
}

template <int MB>
struct SplitTile {
    static constexpr int BM = 64 * MB;
    static constexpr int A_HALF = BM * 16 + 64, W_HALF = SP_BN * 16 + 64;      // bytes
    static constexpr int A_SIDE = 6 * A_HALF, W_SIDE = 6 * W_HALF;
    static constexpr int STEP = A_SIDE + W_SIDE;
};

// parts: as split_rows_kernel leaves them; y [slabs, M, N]: slab s holds the sum over columns [s kb, (s + 1) kb) x 32 of K.
// A workgroup's place: its XCD (workgroups go round the eight) takes a run of neighbouring tiles, rows of x fastest, so that
// the tiles that read the same rows of W read them out of one L2.
template <int MB>
__global__ __launch_bounds__(256, 2) void gemm_split_kernel(const sp_u4* __restrict__ parts, const float* __restrict__ x,
                                                            const float* __restrict__ W, float* __restrict__ y, int M, int N,
                                                            int K, int kb, int m_tiles, int n_tiles, int units) {
    typedef SplitTile<MB> T;
    __shared__ __attribute__((aligned(16))) unsigned char lds[2 * T::STEP];
    const int per = (units + 7) >> 3, u = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || u >= units) return;
    const int mt = u % m_tiles, nt = (u / m_tiles) % n_tiles, slab = u / (m_tiles * n_tiles);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
    const int b0 = slab * kb, b1 = min(b0 + kb, K / SP_KB);                    // blocks of 32 columns

    // where this thread's pieces come from: parts of x 16 bytes at a time, of W half of 16 columns of one row
    constexpr int AP = 6 * T::BM / 256;                                        // pieces of x a thread and step: 3 or 1.5
    const int w_row = tid >> 1, w_half = tid & 1;
    const float* wp = W + (size_t)min(nt * SP_BN + w_row, N - 1) * K + 8 * w_half;
    const sp_u4* ap = parts + (size_t)mt * (K / 16) * 6 * T::BM;
    constexpr int A_LAST = 6 * T::BM - 256 * AP;                               // threads that have one piece more
    sp_u4 a_in[2][AP + 1];
    sp_f4 w_in[2][2];
    auto ask = [&](int b) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const sp_u4* from = ap + (size_t)(2 * b + s) * 6 * T::BM;
#pragma unroll
            for (int j = 0; j < AP; ++j) a_in[s][j] = from[tid + 256 * j];
            if (A_LAST > 0 && tid < A_LAST) a_in[s][AP] = from[tid + 256 * AP];
            const sp_f4* w = reinterpret_cast<const sp_f4*>(wp + (size_t)b * SP_KB + 16 * s);
            w_in[s][0] = w[0];
            w_in[s][1] = w[1];
        }
    };
    auto put = [&](int s) {
        unsigned char* at = lds + s * T::STEP;
#pragma unroll
        for (int j = 0; j <= AP; ++j) {
            const int e = tid + 256 * j;                                       // [part][half][row]
            if (j < AP || (A_LAST > 0 && tid < A_LAST))
                *reinterpret_cast<sp_u4*>(at + (e / T::BM) * T::A_HALF + (e % T::BM) * 16) = a_in[s][j];
        }
        sp_u4 p[3];
        sp_parts(w_in[s][0], w_in[s][1], p);
        at += T::A_SIDE + w_half * T::W_HALF + w_row * 16;
#pragma unroll
        for (int j = 0; j < 3; ++j) *reinterpret_cast<sp_u4*>(at + j * 2 * T::W_HALF) = p[j];
    };
    sp_f16 main[MB][2], rest[MB][2];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) main[i][j][r] = rest[i][j][r] = 0.f;
    const int a_at = (lane >> 5) * T::A_HALF + (wm * 32 * MB + (lane & 31)) * 16;
    const int w_at = T::A_SIDE + (lane >> 5) * T::W_HALF + (wn * 64 + (lane & 31)) * 16;
    auto multiply = [&](int s) {
        const unsigned char* at = lds + s * T::STEP;
        sp_b8 a[3][MB], w[3][2];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int i = 0; i < MB; ++i) a[p][i] = *reinterpret_cast<const sp_b8*>(at + a_at + p * 2 * T::A_HALF + i * 512);
#pragma unroll
            for (int j = 0; j < 2; ++j) w[p][j] = *reinterpret_cast<const sp_b8*>(at + w_at + p * 2 * T::W_HALF + j * 512);
        }
        auto add = [&](sp_f16 (&to)[MB][2], int p, int q) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) to[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[p][i], w[q][j], to[i][j], 0, 0, 0);
        };
        __builtin_amdgcn_s_setprio(1);                     // a wave at its products goes before one at its copies: 6 %
        add(main, 0, 0);
        add(rest, 0, 1);
        add(rest, 1, 0);
        add(rest, 1, 1);
        add(rest, 0, 2);
        add(rest, 2, 0);
        __builtin_amdgcn_s_setprio(0);
    };

    ask(b0);
    put(0);
    put(1);
    __syncthreads();
    for (int b = b0; b < b1; ++b) {
        const bool more = b + 1 < b1;
        if (more) ask(b + 1);
        multiply(0);
        __syncthreads();                                  // the first step is read, the second written
        multiply(1);
        if (more) put(0);
        __syncthreads();                                  // the second step is read, the first written
        if (more) put(1);
    }
    MFMA_SETTLE();

    float* out = y + (size_t)slab * M * N;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = nt * SP_BN + wn * 64 + 32 * j + (lane & 31);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = mt * T::BM + wm * 32 * MB + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m >= M || n >= N) continue;
                float v = main[i][j][r] + rest[i][j][r];
                if (!(fabsf(v) < INFINITY) || (v != 0.f && fabsf(v) < 0x1p-64f)) {
                    v = 0.f;
                    for (int k = b0 * SP_KB; k < b1 * SP_KB; ++k) v = fmaf(x[(size_t)m * K + k], W[(size_t)n * K + k], v);
                }
                out[(size_t)m * N + n] = v;
            }
        }
}

// y = the sum of the slabs, in their order; n4 groups of four values each
__global__ __launch_bounds__(256) void add_slabs_kernel(const sp_f4* __restrict__ slabs, sp_f4* __restrict__ y, int count, long long n4) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    sp_f4 v = slabs[i];
    for (int s = 1; s < count; ++s) v += slabs[(long long)s * n4 + i];
    y[i] = v;
}

// Rows of a tile for M rows, and into how many slabs K is cut: as many as make the tiles come to the fewest rounds over the
// places there are (two workgroups a CU), where a slab costs its writing and reading.
static void split_plan(int M, int N, int K, int cus, int* mb, int* slabs) {
    *mb = M <= 64 ? 1 : 2;
    const int bm = 64 * *mb, blocks = K / SP_KB, slots = 2 * cus;
    const long long tiles = (long long)((M + bm - 1) / bm) * ((N + SP_BN - 1) / SP_BN);
    *slabs = 1;
    double best = 0;
    for (int s = 1; s <= 8 && s <= blocks / 8; ++s) {
        const int kb = (blocks + s - 1) / s;
        if ((blocks + kb - 1) / kb != s) continue;
        const double rounds = (double)((tiles * s + slots - 1) / slots);
        const double t = rounds * (kb + 6) * (*mb == 2 ? 1.0 : 0.6) + (s > 1 ? 4e-7 * (double)M * N * (2 * s + 1) : 0.0);
        if (s == 1 || t < 0.95 * best) {
            best = t;
            *slabs = s;
        }
    }
}

static int split_cus() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
        cus = 256;
    return cus;
}

// bytes of device memory that ra_gemm_split_f32 needs beside its operands, or -1 where it does not take them
extern "C" long long ra_gemm_split_scratch(int M, int N, int K) {
    if (M <= 0 || N <= 0 || K <= 0 || K % SP_KB != 0 || N % 4 != 0 || (long long)M * N >= (1LL << 31)) return -1;
    int mb, slabs;
    split_plan(M, N, K, split_cus(), &mb, &slabs);
    const long long rows = (long long)(M + 64 * mb - 1) / (64 * mb) * (64 * mb);
    if ((long long)(rows / 16) > 65535) return -1;
    return rows * K * 6 + (slabs > 1 ? (long long)slabs * M * N * 4 : 0);
}

// y [M, N] = x [M, K] W [N, K]^T, all float32 and 16-byte aligned; scratch: ra_gemm_split_scratch bytes, 16-byte aligned
extern "C" int ra_gemm_split_f32(const void* x, const void* W, void* y, int M, int N, int K, void* scratch, long long scratch_bytes,
                                 void* stream) {
    if (M <= 0 || N <= 0) return RA_OK;
    const long long need = ra_gemm_split_scratch(M, N, K);
    if (need < 0 || scratch_bytes < need) return RA_ERR_ARG;
    if ((((uintptr_t)x | (uintptr_t)W | (uintptr_t)y | (uintptr_t)scratch) & 15) != 0) return RA_ERR_ARG;
    int mb, slabs;
    split_plan(M, N, K, split_cus(), &mb, &slabs);
    const int bm = 64 * mb, m_tiles = (M + bm - 1) / bm, n_tiles = (N + SP_BN - 1) / SP_BN;
    const int kb = (K / SP_KB + slabs - 1) / slabs, units = m_tiles * n_tiles * slabs;
    hipStream_t st = (hipStream_t)stream;
    const dim3 block(256), sgrid((K / 32 + 3) / 4, m_tiles * bm / 16), grid((units + 7) / 8 * 8);
    sp_u4* parts = (sp_u4*)scratch;
    float* out = slabs > 1 ? (float*)((char*)scratch + (size_t)m_tiles * bm * K * 6) : (float*)y;
    if (mb == 1) {
        hipLaunchKernelGGL(split_rows_kernel<64>, sgrid, block, 0, st, (const float*)x, parts, M, K);
        hipLaunchKernelGGL(gemm_split_kernel<1>, grid, block, 0, st, parts, (const float*)x, (const float*)W, out, M, N, K, kb, m_tiles, n_tiles, units);
    } else {
        hipLaunchKernelGGL(split_rows_kernel<128>, sgrid, block, 0, st, (const float*)x, parts, M, K);
        hipLaunchKernelGGL(gemm_split_kernel<2>, grid, block, 0, st, parts, (const float*)x, (const float*)W, out, M, N, K, kb, m_tiles, n_tiles, units);
    }
    if (slabs > 1) {
        const long long n4 = (long long)M * N / 4;
        hipLaunchKernelGGL(add_slabs_kernel, dim3((unsigned)((n4 + 255) / 256)), block, 0, st, (const sp_f4*)out, (sp_f4*)y, slabs, n4);
    }
    return ra_launch_status();
}
