// out[b][m][:] = a[b][m][:] w[b], a batch of products of few rows, bfloat16 in and out, 32-bit sums: what moves the query of a
// single token over the latents of its head, and the result back (w [B, K, N] row-major: rows of N neighbouring elements).
//
// Bound by the way to W, which is read once: 32 heads of 128 x 512 are 4 MB. A workgroup of four waves has CN columns of one
// batch and up to eight rows of a; a thread has eight columns (16 bytes of a row of W) and every 2,048 / CN-th row of W, the loads of
// eight rows asked for at once; a sits in LDS in 32-bit. The threads' sums are added over the lanes of a wave that have the same columns,
// then over the waves through LDS, in a fixed order. CN is as wide as leaves 128 workgroups.
// Heads of 512 x 128 (a result over the latents back to values), microseconds at 1 / 2 / 4 / 8 rows, 32 heads 4.8 / 5.6 / 7.3 / 10.2 (the
// library's batched product 12.4), 16 heads 4.5 / 5.4 / 7.1 / 10.1 (12.2); where K is the shorter side, 128 x 512, it is no faster than the
// library from two rows on (4.3 / 5.0 / 6.2 / 8.5 against 5.1).
#include "common.h"

typedef float gh_f4 __attribute__((ext_vector_type(4)));
#define GH_ROWS 8
#define GH_MAX_K 1024

template <int M, int CN>
__global__ __launch_bounds__(256) void gemm_heads_kernel(const bf16* __restrict__ a, long long a_batch, long long a_row,
                                                         const bf16* __restrict__ w, bf16* __restrict__ out, long long o_batch,
                                                         long long o_row, int rows, int N, int K) {
    constexpr int TPR = CN / 8, GROUPS = 256 / TPR;            // threads to a row of W, rows of W at a time
    extern __shared__ __attribute__((aligned(16))) float gh_s[];                  // a [K][M], then the waves' sums [4][M][CN]
    const int tid = threadIdx.x, b = blockIdx.x, c0 = blockIdx.y * CN;
    const int here = min(rows, M);
    const int c = c0 + (tid % TPR) * 8, g = tid / TPR;
    const bf16* wb = w + (size_t)b * K * N + min(c, N - 8);
    constexpr int U = 8;
    uint4 wv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) wv[u] = *reinterpret_cast<const uint4*>(wb + (size_t)min(g + u * GROUPS, K - 1) * N);
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const bf16* ar = a + b * a_batch + (size_t)min(m, here - 1) * a_row;       // (a row beyond the last is it again, and not stored)
        for (int k = tid * 8; k < K; k += 2048) {
            const uint4 v = *reinterpret_cast<const uint4*>(ar + k);
            const uint32_t p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                gh_s[(k + 2 * e) * M + m] = __uint_as_float(p[e] << 16);
                gh_s[(k + 2 * e + 1) * M + m] = __uint_as_float(p[e] & 0xffff0000u);
            }
        }
    }
    __syncthreads();
    float acc[M][8];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[m][e] = 0.f;
    for (int k0 = g; k0 < K; k0 += U * GROUPS) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u * GROUPS;
            const uint32_t p[4] = {wv[u].x, wv[u].y, wv[u].z, wv[u].w};
            if (k0 + U * GROUPS < K) wv[u] = *reinterpret_cast<const uint4*>(wb + (size_t)min(k + U * GROUPS, K - 1) * N);
            if (k < K) {
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    const float x = M >= 4 ? reinterpret_cast<const gh_f4*>(gh_s)[(k * M + m) / 4][m % 4] : gh_s[k * M + m];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        acc[m][2 * e] = fmaf(x, __uint_as_float(p[e] << 16), acc[m][2 * e]);
                        acc[m][2 * e + 1] = fmaf(x, __uint_as_float(p[e] & 0xffff0000u), acc[m][2 * e + 1]);
                    }
                }
            }
        }
    }
    // over the lanes of the wave with the same columns
#pragma unroll
    for (int o = TPR; o < 64; o <<= 1)
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[m][e] += __shfl_xor(acc[m][e], o, 64);
    __syncthreads();
    const int wave = tid >> 6;
    if ((tid & 63) < TPR) {
#pragma unroll
        for (int m = 0; m < M; ++m)
#pragma unroll
            for (int e = 0; e < 8; ++e) gh_s[(wave * M + m) * CN + (tid % TPR) * 8 + e] = acc[m][e];
    }
    __syncthreads();
    for (int i = tid; i < here * CN; i += 256) {
        const int m = i / CN, cc = i - m * CN;
        if (c0 + cc >= N) continue;
        const float* s = gh_s + m * CN + cc;
        out[b * o_batch + m * o_row + c0 + cc] = from_f<bf16>(((s[0] + s[M * CN]) + s[2 * M * CN]) + s[3 * M * CN]);
    }
}

extern "C" int ra_gemm_heads_fits(int B, int M, int N, int K) {
    return B >= 1 && B <= 65535 && M >= 1 && M <= GH_ROWS && N >= 8 && N % 8 == 0 && K >= 8 && K % 8 == 0 && K <= GH_MAX_K && (long long)N / 32 < 65535;
}

// a: elements of a row side by side, rows a_row and batches a_batch elements apart, all whole 16-byte pieces; w [B, K, N]; out: rows
// and batches o_row and o_batch elements apart.
extern "C" int ra_gemm_heads_bf16(const void* a, long long a_batch, long long a_row, const void* w, void* out, long long o_batch,
                                  long long o_row, int B, int M, int N, int K, void* stream) {
    if (!ra_gemm_heads_fits(B, M, N, K) || (((uintptr_t)w | (uintptr_t)a) & 15) != 0 || a_batch % 8 != 0 || a_row % 8 != 0 || a_batch < 0 || a_row < 0 || o_batch < 0 || o_row < 0) return RA_ERR_ARG;
    const int cn = (long long)B * ((N + 127) / 128) >= 128 ? 128 : (long long)B * ((N + 63) / 64) >= 128 ? 64 : 32;
    const int m = M > 4 ? 8 : M > 2 ? 4 : M;
    const dim3 grid(B, (N + cn - 1) / cn), block(256);
    const size_t lds = sizeof(float) * m * (size_t)(K > 4 * cn ? K : 4 * cn);
    if (lds > 65536) return RA_ERR_ARG;
    hipStream_t st = (hipStream_t)stream;
#define GH_GO(M_, CN_)                                                                                                       \
    hipLaunchKernelGGL((gemm_heads_kernel<M_, CN_>), grid, block, lds, st, (const bf16*)a, a_batch, a_row, (const bf16*)w, (bf16*)out, \
                       o_batch, o_row, M, N, K)
#define GH_M(CN_)                     \
    do {                              \
        if (m == 1) GH_GO(1, CN_);    \
        else if (m == 2) GH_GO(2, CN_); \
        else if (m == 4) GH_GO(4, CN_); \
        else GH_GO(8, CN_);           \
    } while (0)
    if (cn == 128) GH_M(128); else if (cn == 64) GH_M(64); else GH_M(32);
#undef GH_M
#undef GH_GO
    return ra_launch_status();
}
