// Per-layer token input: a second, narrow embedding of the token, gated by the residual stream,
// projected up and added to the stream through an RMS norm of its own. For row t with token id:
//     h_t += delta_t                              (the pending output of the part before, if any)
//     a[r] = sum_c gate[r][c] * h_t[c]            r < S
//     g[r] = gelu_tanh(a[r]) * table[id][off + r]
//     y[c] = sum_r proj[c][r] * g[r]
//     h_t[c] += y[c] / sqrt(mean_c y[c]^2 + eps) * w[c]
// gelu_tanh(x) = 0.5 x (1 + tanh(sqrt(2/pi) (x + 0.044715 x^3))). Sums, the norm and the stream are
// 32-bit; gate [S, H], proj [H, S] and the table [vocab, ld_table] are in the storage type.
// One workgroup per row: every thread sums its columns' share of the gate products (SB of them a pass), the
// shares are added over the workgroup through LDS, then every thread forms its columns of y.
#include "common.h"

#define TS_MAX_S 512
#define TS_THREADS 256
#define TS_MAX_CPT 32        // columns per thread: H <= 256 * 32

template <typename T, int SB>
__global__ __launch_bounds__(TS_THREADS) void token_side_kernel(
    float* __restrict__ h, const T* __restrict__ delta, const int* __restrict__ ids, const T* __restrict__ table,
    long long ld_table, int off, const T* __restrict__ gate, const T* __restrict__ proj, const float* __restrict__ w,
    float eps, int H, int S) {
    __shared__ float part[TS_THREADS / 64][SB];
    __shared__ float g_s[TS_MAX_S];
    __shared__ float red[16];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float* hr = h + (size_t)t * H;
    for (int r0 = 0; r0 < S; r0 += SB) {                 // SB gate rows a pass; the first pass adds delta into the stream
        float a[SB];
#pragma unroll
        for (int r = 0; r < SB; ++r) a[r] = 0.f;
        for (int c = tid; c < H; c += TS_THREADS) {
            float v = hr[c];
            if (r0 == 0 && delta != nullptr) {
                v += to_f(delta[(size_t)t * H + c]);
                hr[c] = v;                               // (read again by this thread only)
            }
#pragma unroll
            for (int r = 0; r < SB; ++r)
                if (r0 + r < S) a[r] = fmaf(to_f(gate[(size_t)(r0 + r) * H + c]), v, a[r]);
        }
#pragma unroll
        for (int r = 0; r < SB; ++r) {
            const float v = wave_sum(a[r]);
            if (lane == 0) part[wave][r] = v;
        }
        __syncthreads();
        if (tid < SB && r0 + tid < S) {
            float x = 0.f;
            for (int wv = 0; wv < TS_THREADS / 64; ++wv) x += part[wv][tid];
            const float inner = 0.7978845608028654f * (x + 0.044715f * x * x * x);
            const float e = to_f(table[(size_t)ids[t] * ld_table + off + r0 + tid]);
            g_s[r0 + tid] = 0.5f * x * (1.f + tanhf(inner)) * e;
        }
        __syncthreads();
    }
    float y[TS_MAX_CPT];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < TS_MAX_CPT; ++i) {
        const int c = tid + i * TS_THREADS;
        y[i] = 0.f;
        if (c < H) {
            float v = 0.f;
            for (int r = 0; r < S; ++r) v = fmaf(to_f(proj[(size_t)c * S + r]), g_s[r], v);
            y[i] = v;
            ss = fmaf(v, v, ss);
        }
    }
    ss = block_sum(ss, red);
    const float rstd = 1.0f / sqrtf(ss / (float)H + eps);
#pragma unroll
    for (int i = 0; i < TS_MAX_CPT; ++i) {
        const int c = tid + i * TS_THREADS;
        if (c < H) hr[c] += y[i] * rstd * w[c];
    }
}

// The same for bfloat16 with 16-byte loads (H % 8 == 0, S % 8 == 0, S <= TS_MAX_S), R rows of the stream
// a workgroup: the rows (with delta added) sit in LDS in 32-bit; a wave takes every fourth gate row and
// forms its product with all R stream rows, each lane eight columns at a time, so that all of a row's
// loads are on their way at once and a gate row is read once for R rows; then a thread forms its columns of
// y for all R rows from one read of the projection's row.
template <int R, int NTH>
__global__ __launch_bounds__(NTH) void token_side_bf16x8_kernel(
    float* __restrict__ h, const bf16* __restrict__ delta, const int* __restrict__ ids, const bf16* __restrict__ table,
    long long ld_table, int off, const bf16* __restrict__ gate, const bf16* __restrict__ proj,
    const float* __restrict__ w, float eps, int T_tokens, int H, int S) {
    extern __shared__ __attribute__((aligned(16))) float ts_smem[];
    float* x_s = ts_smem;                        // [R][H]
    float* g_s = x_s + (size_t)R * H;            // [R][S]
    float* red = g_s + R * S;                    // [R][waves]
    const int t0 = blockIdx.x * R, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rows = min(R, T_tokens - t0);
    for (int idx = tid * 4; idx < R * H; idx += NTH * 4) {
        const int rr = idx / H, c = idx - rr * H;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (rr < rows) {
            v = *reinterpret_cast<const float4*>(h + (size_t)(t0 + rr) * H + c);
            if (delta != nullptr) {
                const uint2 d = *reinterpret_cast<const uint2*>(delta + (size_t)(t0 + rr) * H + c);
                v.x += __uint_as_float(d.x << 16); v.y += __uint_as_float(d.x & 0xffff0000u);
                v.z += __uint_as_float(d.y << 16); v.w += __uint_as_float(d.y & 0xffff0000u);
            }
        }
        *reinterpret_cast<float4*>(x_s + idx) = v;
    }
    __syncthreads();
    for (int r = wave; r < S; r += (NTH / 64)) {
        float a[R];
#pragma unroll
        for (int rr = 0; rr < R; ++rr) a[rr] = 0.f;
        for (int c = lane * 8; c < H; c += 512) {
            const uint4 gw = *reinterpret_cast<const uint4*>(gate + (size_t)r * H + c);
            const float g8[8] = {__uint_as_float(gw.x << 16), __uint_as_float(gw.x & 0xffff0000u),
                                 __uint_as_float(gw.y << 16), __uint_as_float(gw.y & 0xffff0000u),
                                 __uint_as_float(gw.z << 16), __uint_as_float(gw.z & 0xffff0000u),
                                 __uint_as_float(gw.w << 16), __uint_as_float(gw.w & 0xffff0000u)};
#pragma unroll
            for (int rr = 0; rr < R; ++rr) {
                const float4 x0 = *reinterpret_cast<const float4*>(x_s + (size_t)rr * H + c);
                const float4 x1 = *reinterpret_cast<const float4*>(x_s + (size_t)rr * H + c + 4);
                a[rr] = fmaf(g8[0], x0.x, a[rr]); a[rr] = fmaf(g8[1], x0.y, a[rr]);
                a[rr] = fmaf(g8[2], x0.z, a[rr]); a[rr] = fmaf(g8[3], x0.w, a[rr]);
                a[rr] = fmaf(g8[4], x1.x, a[rr]); a[rr] = fmaf(g8[5], x1.y, a[rr]);
                a[rr] = fmaf(g8[6], x1.z, a[rr]); a[rr] = fmaf(g8[7], x1.w, a[rr]);
            }
        }
#pragma unroll
        for (int rr = 0; rr < R; ++rr) {
            const float x = wave_sum(a[rr]);
            if (lane == 0 && rr < rows) {
                const float inner = 0.7978845608028654f * (x + 0.044715f * x * x * x);
                const float e = to_f(table[(size_t)ids[t0 + rr] * ld_table + off + r]);
                g_s[rr * S + r] = 0.5f * x * (1.f + tanhf(inner)) * e;
            }
        }
    }
    __syncthreads();
    float y[R][(4096 / NTH)];                  // H <= 4096 in this form
    float ss[R];
#pragma unroll
    for (int rr = 0; rr < R; ++rr) ss[rr] = 0.f;
#pragma unroll
    for (int i = 0; i < (4096 / NTH); ++i) {
        const int c = tid + i * NTH;
#pragma unroll
        for (int rr = 0; rr < R; ++rr) y[rr][i] = 0.f;
        if (c < H) {
            for (int r8 = 0; r8 < S; r8 += 8) {
                const uint4 pw = *reinterpret_cast<const uint4*>(proj + (size_t)c * S + r8);
                const float p8[8] = {__uint_as_float(pw.x << 16), __uint_as_float(pw.x & 0xffff0000u),
                                     __uint_as_float(pw.y << 16), __uint_as_float(pw.y & 0xffff0000u),
                                     __uint_as_float(pw.z << 16), __uint_as_float(pw.z & 0xffff0000u),
                                     __uint_as_float(pw.w << 16), __uint_as_float(pw.w & 0xffff0000u)};
#pragma unroll
                for (int rr = 0; rr < R; ++rr)
#pragma unroll
                    for (int k = 0; k < 8; ++k) y[rr][i] = fmaf(p8[k], g_s[rr * S + r8 + k], y[rr][i]);
            }
#pragma unroll
            for (int rr = 0; rr < R; ++rr) ss[rr] = fmaf(y[rr][i], y[rr][i], ss[rr]);
        }
    }
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
        const float v = wave_sum(ss[rr]);
        if (lane == 0) red[rr * (NTH / 64) + wave] = v;
    }
    __syncthreads();
#pragma unroll
    for (int rr = 0; rr < R; ++rr) {
        if (rr >= rows) break;
        float tot = 0.f;
        for (int wv = 0; wv < NTH / 64; ++wv) tot += red[rr * (NTH / 64) + wv];      // (the same order in every thread)
        const float rstd = 1.0f / sqrtf(tot / (float)H + eps);
#pragma unroll
        for (int i = 0; i < (4096 / NTH); ++i) {
            const int c = tid + i * NTH;
            if (c < H) h[(size_t)(t0 + rr) * H + c] = x_s[(size_t)rr * H + c] + y[rr][i] * rstd * w[c];
        }
    }
}

// bfloat16 and S up to 32 (H, S as above): the same sums in the same order, with the reads asked for before what they wait behind.
// (A loop over a row's runs of 512 columns waits for one load after the other, 1 us each where the matrices come from memory.)
__device__ __forceinline__ void ts_unpack(const uint4& v, float (&f)[8]) {
    const uint32_t p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[2 * k] = __uint_as_float(p[k] << 16);
        f[2 * k + 1] = __uint_as_float(p[k] & 0xffff0000u);
    }
}
__device__ __forceinline__ float4 ts_row4(const float* h, const bf16* delta, size_t at) {
    float4 v = *reinterpret_cast<const float4*>(h + at);
    if (delta != nullptr) {
        const uint2 d = *reinterpret_cast<const uint2*>(delta + at);
        v.x += __uint_as_float(d.x << 16); v.y += __uint_as_float(d.x & 0xffff0000u);
        v.z += __uint_as_float(d.y << 16); v.w += __uint_as_float(d.y & 0xffff0000u);
    }
    return v;
}
__device__ __forceinline__ float ts_gelu(float x) {
    const float inner = 0.7978845608028654f * (x + 0.044715f * x * x * x);
    return 0.5f * x * (1.f + tanhf(inner));
}

// One row a workgroup: a wave's gate rows (32 over WAVES waves), half of the projection and the token's entries are asked for beside
// the row itself, the rest of the projection as the first half is used. RUNS: of 512 columns. H 4,096, S 32, matrices from memory:
// 22 -> 17 us, which is one CU's reading of 512 KB (from the caches 14 -> 11).
template <int RUNS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void token_side_row_kernel(
    float* __restrict__ h, const bf16* __restrict__ delta, const int* __restrict__ ids, const bf16* __restrict__ table,
    long long ld_table, int off, const bf16* __restrict__ gate, const bf16* __restrict__ proj,
    const float* __restrict__ w, float eps, int H, int S) {
    constexpr int NT = 64 * WAVES, GATES = 32 / WAVES, COLS = 512 * RUNS / NT, QUADS = (128 * RUNS + NT - 1) / NT;
    __shared__ __attribute__((aligned(16))) float x_s[512 * RUNS];
    __shared__ float g_s[32], red[WAVES];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t row = (size_t)t * H;
    const int id = ids[t];
    // (what lies beyond H or S is read again from the last place, and meets zeros in x_s or g_s)
    float4 xv[QUADS];
    uint2 dv[QUADS];
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
        const int c = min((tid + NT * i) * 4, H - 4);
        xv[i] = *reinterpret_cast<const float4*>(h + row + c);
        dv[i] = make_uint2(0u, 0u);
        if (delta != nullptr) dv[i] = *reinterpret_cast<const uint2*>(delta + row + c);
    }
    uint4 gv[GATES][RUNS];
#pragma unroll
    for (int k = 0; k < GATES; ++k)
#pragma unroll
        for (int q = 0; q < RUNS; ++q) {
            const int r = min(wave + WAVES * k, S - 1), c = min(lane * 8 + 512 * q, H - 8);
            gv[k][q] = *reinterpret_cast<const uint4*>(gate + (unsigned)(r * H + c));
        }
    uint4 pv[COLS / 2][4];
    auto ask = [&](int i, int half) {
        const int c = min(tid + NT * (half * (COLS / 2) + i), H - 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) pv[i][q] = *reinterpret_cast<const uint4*>(proj + (unsigned)(c * S + min(8 * q, S - 8)));
    };
#pragma unroll
    for (int i = 0; i < COLS / 2; ++i) ask(i, 0);
    float e[GATES];
#pragma unroll
    for (int k = 0; k < GATES; ++k) e[k] = to_f(table[(size_t)id * ld_table + off + min(wave + WAVES * k, S - 1)]);
#pragma unroll
    for (int i = 0; i < QUADS; ++i) {
        const int c = (tid + NT * i) * 4;
        xv[i].x += __uint_as_float(dv[i].x << 16); xv[i].y += __uint_as_float(dv[i].x & 0xffff0000u);
        xv[i].z += __uint_as_float(dv[i].y << 16); xv[i].w += __uint_as_float(dv[i].y & 0xffff0000u);
        if (c < 512 * RUNS) *reinterpret_cast<float4*>(x_s + c) = c < H ? xv[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __syncthreads();
    float a[GATES];
#pragma unroll
    for (int k = 0; k < GATES; ++k) a[k] = 0.f;
#pragma unroll
    for (int q = 0; q < RUNS; ++q) {
        const int c = lane * 8 + 512 * q;
        const float4 x0 = *reinterpret_cast<const float4*>(x_s + c), x1 = *reinterpret_cast<const float4*>(x_s + c + 4);
        const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int k = 0; k < GATES; ++k) {
            float g[8];
            ts_unpack(gv[k][q], g);
#pragma unroll
            for (int i = 0; i < 8; ++i) a[k] = fmaf(g[i], x[i], a[k]);
        }
    }
#pragma unroll
    for (int k = 0; k < GATES; ++k) {
        const float x = wave_sum(a[k]);
        const int r = wave + WAVES * k;
        if (lane == k) g_s[r] = r < S ? ts_gelu(x) * e[k] : 0.f;
    }
    float wv[COLS];
#pragma unroll
    for (int i = 0; i < COLS; ++i) wv[i] = w[min(tid + NT * i, H - 1)];
    __syncthreads();
    float y[COLS], ss = 0.f;
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < COLS / 2; ++i) {
            float v = 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float p[8];
                ts_unpack(pv[i][q], p);
#pragma unroll
                for (int k = 0; k < 8; ++k) v = fmaf(p[k], g_s[8 * q + k], v);
            }
            if (half == 0) ask(i, 1);
            y[half * (COLS / 2) + i] = v;
            ss = fmaf(v, tid + NT * (half * (COLS / 2) + i) < H ? v : 0.f, ss);
        }
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    float tot = 0.f;
#pragma unroll
    for (int v = 0; v < WAVES; ++v) tot += red[v];
    const float rstd = 1.0f / sqrtf(tot / (float)H + eps);
#pragma unroll
    for (int i = 0; i < COLS; ++i) {
        const int c = tid + NT * i;
        if (c < H) h[row + c] = x_s[c] + y[i] * rstd * wv[i];
    }
}

// Many rows, four a workgroup of four waves: a wave has the next two gate rows on their way while it multiplies two, by the rows
// of the stream in LDS (in 32-bit); then y takes the rows' place there, a column a turn, the next one's projection on its way, and
// the stream is read again at the end. Two workgroups a CU. H 4,096, S 32: 2,048 rows 91 -> 56 us.
#define TR_ROWS 4
// From three rounds of single rows over the CUs on (4,096 columns: 200 rows 12 us, 700 rows 34 either way).
#define TR_FROM 768
template <int RUNS>
__global__ __launch_bounds__(256, 2) void token_side_rows_kernel(
    float* __restrict__ h, const bf16* __restrict__ delta, const int* __restrict__ ids, const bf16* __restrict__ table,
    long long ld_table, int off, const bf16* __restrict__ gate, const bf16* __restrict__ proj,
    const float* __restrict__ w, float eps, int T_tokens, int H, int S) {
    constexpr int HS = 512 * RUNS;
    extern __shared__ __attribute__((aligned(16))) float x_s[];                       // [TR_ROWS][HS]: the stream, then y
    __shared__ float g_s[TR_ROWS][32], red[TR_ROWS][4];
    const int t0 = blockIdx.x * TR_ROWS, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rows = min(TR_ROWS, T_tokens - t0);
    // piece (r0, first run): four runs of gate rows r0 and r0 + 4
    uint4 next[2][4];
    auto ask = [&](int r0, int q0) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int r = min(r0 + 4 * k, S - 1), c = min(lane * 8 + 512 * (q0 + q), H - 8);
                next[k][q] = *reinterpret_cast<const uint4*>(gate + (unsigned)(r * H + c));
            }
    };
    ask(wave, 0);
#pragma unroll 4
    for (int c = tid * 4; c < TR_ROWS * HS; c += 1024) {
        const int rr = c / HS, cc = c - rr * HS;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (rr < rows && cc < H) v = ts_row4(h, delta, (size_t)(t0 + rr) * H + cc);
        *reinterpret_cast<float4*>(x_s + c) = v;
    }
    __syncthreads();
    float a[2][TR_ROWS];
#pragma unroll 1
    for (int r0 = wave, q0 = 0; r0 < 32;) {
        uint4 now[2][4];
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int q = 0; q < 4; ++q) now[k][q] = next[k][q];
        const bool ends = q0 + 4 >= RUNS;
        const int r1 = ends ? r0 + 8 : r0, q1 = ends ? 0 : q0 + 4;
        ask(r1, q1);
        if (q0 == 0) {
#pragma unroll
            for (int k = 0; k < 2; ++k)
#pragma unroll
                for (int rr = 0; rr < TR_ROWS; ++rr) a[k][rr] = 0.f;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float g[2][8];
            ts_unpack(now[0][q], g[0]);
            ts_unpack(now[1][q], g[1]);
#pragma unroll
            for (int rr = 0; rr < TR_ROWS; ++rr) {
                const float* xr = x_s + rr * HS + lane * 8 + 512 * (q0 + q);
                const float4 x0 = *reinterpret_cast<const float4*>(xr), x1 = *reinterpret_cast<const float4*>(xr + 4);
                const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
                for (int k = 0; k < 2; ++k)
#pragma unroll
                    for (int i = 0; i < 8; ++i) a[k][rr] = fmaf(g[k][i], x[i], a[k][rr]);
            }
        }
        if (ends) {
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                float mine = 0.f;                                                     // lane rr gets row rr's
#pragma unroll
                for (int rr = 0; rr < TR_ROWS; ++rr) {
                    const float x = wave_sum(a[k][rr]);
                    if (lane == rr) mine = x;
                }
                const int r = r0 + 4 * k;
                if (lane < TR_ROWS) {
                    const float e = r < S ? to_f(table[(size_t)ids[t0 + min(lane, rows - 1)] * ld_table + off + r]) : 0.f;
                    g_s[lane][r] = r < S ? ts_gelu(mine) * e : 0.f;
                }
            }
        }
        r0 = r1;
        q0 = q1;
    }
    __syncthreads();
    // y of column tid + 256 i of every row, in place of the stream
    float ss[TR_ROWS];
#pragma unroll
    for (int rr = 0; rr < TR_ROWS; ++rr) ss[rr] = 0.f;
    uint4 pn[4];
    auto column = [&](int c) {
#pragma unroll
        for (int q = 0; q < 4; ++q) pn[q] = *reinterpret_cast<const uint4*>(proj + (unsigned)(min(c, H - 1) * S + min(8 * q, S - 8)));
    };
    column(tid);
#pragma unroll 1
    for (int c = tid; c < H; c += 256) {
        uint4 p4[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) p4[q] = pn[q];
        column(c + 256);
        float y[TR_ROWS];
#pragma unroll
        for (int rr = 0; rr < TR_ROWS; ++rr) y[rr] = 0.f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            float p[8];
            ts_unpack(p4[q], p);
#pragma unroll
            for (int rr = 0; rr < TR_ROWS; ++rr)
#pragma unroll
                for (int k = 0; k < 8; ++k) y[rr] = fmaf(p[k], g_s[rr][8 * q + k], y[rr]);
        }
#pragma unroll
        for (int rr = 0; rr < TR_ROWS; ++rr) {
            ss[rr] = fmaf(y[rr], y[rr], ss[rr]);
            x_s[rr * HS + c] = y[rr];
        }
    }
#pragma unroll
    for (int rr = 0; rr < TR_ROWS; ++rr) {
        const float v = wave_sum(ss[rr]);
        if (lane == 0) red[rr][wave] = v;
    }
    __syncthreads();
#pragma unroll 4
    for (int c = tid * 4; c < TR_ROWS * HS; c += 1024) {
        const int rr = c / HS, cc = c - rr * HS;
        if (rr >= rows || cc >= H) continue;
        const size_t at = (size_t)(t0 + rr) * H + cc;
        const float4 x = ts_row4(h, delta, at), y = *reinterpret_cast<const float4*>(x_s + c), wv = *reinterpret_cast<const float4*>(w + cc);
        const float rstd = 1.0f / sqrtf((((red[rr][0] + red[rr][1]) + red[rr][2]) + red[rr][3]) / (float)H + eps);
        *reinterpret_cast<float4*>(h + at) =
            make_float4(x.x + y.x * rstd * wv.x, x.y + y.y * rstd * wv.y, x.z + y.z * rstd * wv.z, x.w + y.w * rstd * wv.w);
    }
}

template <int R, int NTH>
static int token_side_x8_launch(hipStream_t st, float* h, const void* delta, const int* ids, const void* table,
                                long long ld_table, int off, const void* gate, const void* proj, const float* w, float eps,
                                int T_tokens, int H, int S) {
    const size_t lds = sizeof(float) * ((size_t)R * H + (size_t)R * S + R * (NTH / 64));
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute((const void*)token_side_bf16x8_kernel<R, NTH>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds) != hipSuccess)
        return RA_ERR_LAUNCH;
    hipLaunchKernelGGL((token_side_bf16x8_kernel<R, NTH>), dim3((T_tokens + R - 1) / R), dim3(NTH), lds, st, h,
                       (const bf16*)delta, ids, (const bf16*)table, ld_table, off, (const bf16*)gate, (const bf16*)proj, w,
                       eps, T_tokens, H, S);
    return ra_launch_status();
}

extern "C" int ra_token_side(float* h, const void* delta, const int* ids, const void* table, long long ld_table, int off,
                             const void* gate, const void* proj, const float* w, float eps, int T_tokens, int H, int S,
                             int dtype, void* stream) {
    if (T_tokens <= 0) return RA_OK;
    if (S < 1 || S > TS_MAX_S || H < 1 || H > TS_THREADS * TS_MAX_CPT || off < 0 || ld_table < off + S) return RA_ERR_ARG;
    dim3 grid(T_tokens), block(TS_THREADS);
    hipStream_t st = (hipStream_t)stream;
    auto al = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    if (dtype == RA_DTYPE_BF16 && S <= 32 && S % 8 == 0 && H % 8 == 0 && H <= 4096 && al(h) && al(delta) && al(gate) && al(proj) && al(w)) {
#define TS_ROW(RUNS_, WAVES_)                                                                                                      \
    hipLaunchKernelGGL((token_side_row_kernel<RUNS_, WAVES_>), grid, dim3(64 * WAVES_), 0, st, h, (const bf16*)delta, ids, (const bf16*)table, ld_table, \
                       off, (const bf16*)gate, (const bf16*)proj, w, eps, H, S)
#define TS_ROWS(RUNS_)                                                                                                             \
    hipLaunchKernelGGL(token_side_rows_kernel<RUNS_>, dim3((T_tokens + TR_ROWS - 1) / TR_ROWS), block, TR_ROWS * 2048 * RUNS_, st, h, \
                       (const bf16*)delta, ids, (const bf16*)table, ld_table, off, (const bf16*)gate, (const bf16*)proj, w, eps, T_tokens, H, S)
        if (T_tokens < TR_FROM) {
            if (H <= 2048) TS_ROW(4, 16); else TS_ROW(8, 8);
        } else {
            if (H <= 2048) TS_ROWS(4); else TS_ROWS(8);
        }
#undef TS_ROW
#undef TS_ROWS
        return ra_launch_status();
    }
    if (dtype == RA_DTYPE_BF16 && H % 8 == 0 && S % 8 == 0 && H <= 4096) {
        // many rows: four a workgroup, so that the two matrices are read once for four rows
        if (T_tokens >= 256)
            return token_side_x8_launch<4, 256>(st, h, delta, ids, table, ld_table, off, gate, proj, w, eps, T_tokens, H, S);
        // few rows: sixteen waves a row, so that a row's loads are spread over four times the threads
        if (T_tokens <= 64)
            return token_side_x8_launch<1, 1024>(st, h, delta, ids, table, ld_table, off, gate, proj, w, eps, T_tokens, H, S);
        return token_side_x8_launch<1, 256>(st, h, delta, ids, table, ld_table, off, gate, proj, w, eps, T_tokens, H, S);
    }
#define TS_GO(T_, SB_)                                                                                         \
    hipLaunchKernelGGL((token_side_kernel<T_, SB_>), grid, block, 0, st, h, (const T_*)delta, ids, (const T_*)table, \
                       ld_table, off, (const T_*)gate, (const T_*)proj, w, eps, H, S)
    if (dtype == RA_DTYPE_F32) {
        if (S <= 16) TS_GO(float, 16); else if (S <= 32) TS_GO(float, 32); else TS_GO(float, 64);
    } else if (dtype == RA_DTYPE_BF16) {
        if (S <= 16) TS_GO(bf16, 16); else if (S <= 32) TS_GO(bf16, 32); else TS_GO(bf16, 64);
    } else {
        return RA_ERR_ARG;
    }
#undef TS_GO
    return ra_launch_status();
}
