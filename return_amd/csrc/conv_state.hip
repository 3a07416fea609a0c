// Causal convolution over time on each channel, for requests that arrive in pieces: the last
// taps-1 inputs of every request are kept between steps in a tail [slots + 1, taps-1, C], so a
// row's result does not depend on how the request was cut into steps.
//
//   y_t[c] = sum_j w[c][j] * x_(t - taps + 1 + j)[c] + b[c]    (w's last column is the current row's; zeros
//                                                          before the request's first row; b null: no bias)
//   out_t  = act(y_t)  or  act(x_t + y_t)                 (flags: 1 adds the input, 2 applies SiLU)
//
// With an input bias every input is x + in_bias, rounded to the storage type (what a stored x + in_bias would be), in
// the rows as in the tail; the zeros before the request's first row stay zeros.
//
// x: rows of ld_x elements of which C are read (a column slice of a wider projection is fine),
// out: rows of ld_out elements. Request s brings rows cu_q[s]..cu_q[s+1]-1 and owns tail row
// slot_ids[s]. All sums in 32-bit; the result and the tail are rounded to the storage type.
//
// Grid (segments of CONV_SEG rows, requests, chunks of 256 channels); a thread owns one channel
// and walks its segment's rows with the last taps-1 inputs in registers. Only a request's first
// segment reads the tail (CONV_SEG >= taps-1), and the same thread writes the new tail for its
// channel when it is done, so no other thread ever sees a tail half way.
#include "common.h"

#define CONV_SEG 16
#define CONV_MAX_TAPS 17       // taps - 1 inputs must fit one segment

// MT: the most taps of this instantiation (4, 8 or CONV_MAX_TAPS)
template <typename T, int MT>
__global__ __launch_bounds__(256) void causal_conv_kernel(
    const T* __restrict__ x, long long ld_x, const float* __restrict__ w, T* __restrict__ tail,
    const int* __restrict__ cu_q, const int* __restrict__ slot_ids, T* __restrict__ out, long long ld_out,
    int C, int taps, int flags, const float* __restrict__ bias, const float* __restrict__ in_bias) {
    const int s = blockIdx.y;
    const int base = cu_q[s];
    const int q_len = cu_q[s + 1] - base;
    const int first = blockIdx.x * CONV_SEG;
    if (first >= q_len) return;
    const int c = blockIdx.z * 256 + threadIdx.x;
    if (c >= C) return;
    const int last = min(first + CONV_SEG, q_len);
    const int back = taps - 1;
    T* my_tail = tail + ((size_t)slot_ids[s] * back) * C + c;

    const float b0 = bias != nullptr ? bias[c] : 0.f;
    const float bi = in_bias != nullptr ? in_bias[c] : 0.f;
    auto input = [&](int li) {
        const float v = to_f(x[(size_t)(base + li) * ld_x + c]);
        return in_bias != nullptr ? round_to<T>(v + bi) : v;
    };
    float wt[MT], win[MT], old[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        wt[j] = j < taps ? w[(size_t)c * taps + j] : 0.f;
        win[j] = old[j] = 0.f;
        if (j < back) {
            const int li = first - back + j;                 // the input that far back, among this step's rows or before
            win[j] = li >= 0 ? input(li) : to_f(my_tail[(size_t)(back + li) * C]);
            old[j] = win[j];
        }
    }
    for (int li = first; li < last; ++li) {
        const float cur = input(li);
        float y = b0;
#pragma unroll
        for (int j = 0; j < MT - 1; ++j)
            if (j < back) y = fmaf(wt[j], win[j], y);
#pragma unroll
        for (int j = 0; j < MT; ++j)
            if (j == back) y = fmaf(wt[j], cur, y);
        if (flags & 1) y += cur;
        if (flags & 2) y = y / (1.f + expf(-y));
        out[(size_t)(base + li) * ld_out + c] = from_f<T>(y);
#pragma unroll
        for (int j = 0; j < MT - 1; ++j)
            if (j + 1 < back) win[j] = win[j + 1];
#pragma unroll
        for (int j = 0; j < MT; ++j)
            if (j == back - 1) win[j] = cur;
    }
    if (first == 0) {
        // the new tail: the last taps-1 inputs of (old tail, this step's rows)
#pragma unroll
        for (int j = 0; j < MT - 1; ++j) {
            if (j < back) {
                const int li = q_len - back + j;
                float v = 0.f;
                if (li >= 0) v = input(li);
                else {
#pragma unroll
                    for (int k = 0; k < MT - 1; ++k)
                        if (k == back + li) v = old[k];
                }
                my_tail[(size_t)j * C] = from_f<T>(v);
            }
        }
    }
}

// The same for bfloat16, two to four taps and many rows: eight neighbouring channels a thread, a few rows asked for
// while the few before are worked on (C, the row strides and the addresses whole 16-byte pieces); the filters go through LDS, so
// that their reads are whole lines. The sums are formed in the same order: the same bits. The loop over the rows stays a loop: a
// segment written out was 27 KB of instructions, whose way into the CUs took longer than the rows'. Bound by reading and writing
// the rows once: 2,048 rows of 4,096 channels 33 -> 12 us; with SiLU, whose exponential and division
// are then most of it, 2,804 rows of 6,144 45 -> 40.
__device__ __forceinline__ void conv_unpack(const uint4& v, float (&f)[8]) {
    const uint32_t p[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        f[2 * k] = __uint_as_float(p[k] << 16);
        f[2 * k + 1] = __uint_as_float(p[k] & 0xffff0000u);
    }
}
typedef float conv_f2 __attribute__((ext_vector_type(2)));
typedef __bf16 conv_b2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 conv_pack(const float (&f)[8]) {
    uint32_t p[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) p[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector(conv_f2{f[2 * k], f[2 * k + 1]}, conv_b2));
    return make_uint4(p[0], p[1], p[2], p[3]);
}

#define CONV8_THREADS 128
template <int TAPS, bool ADD, bool SILU>
__global__ __launch_bounds__(CONV8_THREADS) void causal_conv_bf16x8_kernel(
    const bf16* __restrict__ x, long long ld_x, const float* __restrict__ w, bf16* __restrict__ tail,
    const int* __restrict__ cu_q, const int* __restrict__ slot_ids, bf16* __restrict__ out, long long ld_out,
    int C, const float* __restrict__ bias, const float* __restrict__ in_bias) {
    constexpr int BACK = TAPS - 1, CHANNELS = CONV8_THREADS * 8, U = SILU ? 2 : 4;
    __shared__ __attribute__((aligned(16))) float w_s[TAPS][CHANNELS];
    const int s = blockIdx.y;
    const int base = cu_q[s];
    const int q_len = cu_q[s + 1] - base;
    const int first = blockIdx.x * CONV_SEG;
    if (first >= q_len) return;                            // (the same in every thread)
    const int c0 = blockIdx.z * CHANNELS, c = c0 + threadIdx.x * 8;
    const bool in = c < C;
    const int last = min(first + CONV_SEG, q_len);
    bf16* my_tail = tail + ((size_t)slot_ids[s] * BACK) * C + c;
    const bf16* xs = x + (size_t)base * ld_x + c;
    bf16* os = out + (size_t)base * ld_out + c;
    auto ask = [&](int li) { return *reinterpret_cast<const uint4*>(xs + (size_t)li * ld_x); };
    uint4 next[U], before[BACK];
    if (in) {
#pragma unroll
        for (int j = 0; j < BACK; ++j) {
            const int li = first - BACK + j;
            before[j] = li >= 0 ? ask(li) : *reinterpret_cast<const uint4*>(my_tail + (size_t)(BACK + li) * C);
        }
#pragma unroll
        for (int r = 0; r < U; ++r) next[r] = ask(min(first + r, last - 1));
    }
#pragma unroll 8
    for (int k = threadIdx.x; k < TAPS * min(CHANNELS, C - c0); k += CONV8_THREADS) w_s[k % TAPS][k / TAPS] = w[(size_t)c0 * TAPS + k];
    __syncthreads();
    if (!in) return;
    float bi[8], b0[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) bi[e] = b0[e] = 0.f;
    if (in_bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 8; ++e) bi[e] = in_bias[c + e];
    }
    if (bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 8; ++e) b0[e] = bias[c + e];
    }
    auto take = [&](const uint4& v, float (&f)[8]) {
        conv_unpack(v, f);
        if (in_bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] += bi[e];
            conv_unpack(conv_pack(f), f);
        }
    };
    float wt[TAPS][8], win[BACK][8];
#pragma unroll
    for (int j = 0; j < BACK; ++j) {
        if (first - BACK + j >= 0) take(before[j], win[j]);
        else conv_unpack(before[j], win[j]);               // (the tail holds inputs as they were taken)
    }
#pragma unroll
    for (int j = 0; j < TAPS; ++j)
#pragma unroll
        for (int e = 0; e < 8; ++e) wt[j][e] = w_s[j][threadIdx.x * 8 + e];
#pragma unroll 1
    for (int l0 = first; l0 < last; l0 += U) {
        uint4 now[U];
#pragma unroll
        for (int r = 0; r < U; ++r) {
            now[r] = next[r];
            next[r] = ask(min(l0 + U + r, last - 1));
        }
#pragma unroll
        for (int r = 0; r < U; ++r) {
            if (l0 + r >= last) break;
            float cur[8], y[8];
            take(now[r], cur);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                y[e] = b0[e];
#pragma unroll
                for (int j = 0; j < BACK; ++j) y[e] = fmaf(wt[j][e], win[j][e], y[e]);
                y[e] = fmaf(wt[BACK][e], cur[e], y[e]);
                if constexpr (ADD) y[e] += cur[e];
                if constexpr (SILU) y[e] = y[e] / (1.f + expf(-y[e]));
#pragma unroll
                for (int j = 0; j + 1 < BACK; ++j) win[j][e] = win[j + 1][e];
                win[BACK - 1][e] = cur[e];
            }
            *reinterpret_cast<uint4*>(os + (size_t)(l0 + r) * ld_out) = conv_pack(y);
        }
    }
    if (first == 0) {
        // the new tail: the last taps-1 inputs of (old tail, this step's rows), the old tail being what `before` holds here
#pragma unroll
        for (int j = 0; j < BACK; ++j) {
            const int li = q_len - BACK + j;
            float v[8];
            if (li >= 0) {
                take(ask(li), v);
            } else {
                uint4 o = before[0];
#pragma unroll
                for (int k = 1; k < BACK; ++k)
                    if (k == BACK + li) o = before[k];
                conv_unpack(o, v);
            }
            *reinterpret_cast<uint4*>(my_tail + (size_t)j * C) = conv_pack(v);
        }
    }
}

// Whether the form of eight channels a thread (1) is taken, where the rest allows it. It has an eighth of the threads and a quarter of the
// workgroups, many of which are empty where one long request stands beside single tokens. So it wins from three workgroups of the other form a CU on;
// with SiLU, whose 128 exponentials and divisions a thread come one after another (12 us for any segment of 16 rows), where the rows
// are many or the empty workgroups are. Microseconds, a channel a thread / eight: no SiLU, 64 rows of 4,096 channels 6.4 / 6.6, 512
// rows of 12,288 11.7 / 9.3, 2,048 of 4,096 14.7 / 10.9, 63 tokens beside 512 rows of 4,096 54 / 21; SiLU, 300 rows of 4,096 7.8 / 12.4,
// 2,048 of 4,096 19.1 / 22.4, of 6,144 23.9 / 22.9, of 12,288 41 / 38, 63 tokens beside 64 rows of 6,144 17 / 34, beside 512 of 4,096 55 / 35.
extern "C" int ra_causal_conv_form(int T_tokens, int n_seqs, int max_q_len, int C, int flags) {
    if (max_q_len < 8) return 0;
    const long long segs = (long long)((max_q_len + CONV_SEG - 1) / CONV_SEG) * n_seqs, blocks = segs * ((C + 255) / 256);
    if ((flags & 2) == 0) return blocks >= 768;
    return (long long)T_tokens * C >= 12000000 || blocks >= 20480 || segs >= 2048;
}

// x [T rows], w fp32 [C, taps], tail [slots, taps-1, C], out [T rows]; max_q_len: the longest request of the step.
static int causal_conv_run(const void* x, long long ld_x, const float* in_bias, const float* w, const float* bias, void* tail, const int* cu_q,
                           const int* slot_ids, void* out, long long ld_out, int T_tokens, int n_seqs, int max_q_len,
                           int C, int taps, int flags, int dtype, void* stream) {
    if (n_seqs <= 0 || max_q_len <= 0) return RA_OK;
    if (taps < 1 || taps > CONV_MAX_TAPS || taps - 1 > CONV_SEG || C <= 0 || ld_x < C || ld_out < C) return RA_ERR_ARG;
    if (n_seqs > 65535 || (C + 255) / 256 > 65535) return RA_ERR_ARG;
    if (dtype != RA_DTYPE_F32 && dtype != RA_DTYPE_BF16) return RA_ERR_ARG;
    if (dtype == RA_DTYPE_BF16 && taps >= 2 && taps <= 4 && ra_causal_conv_form(T_tokens, n_seqs, max_q_len, C, flags) != 0 && C % 8 == 0 && ld_x % 8 == 0 && ld_out % 8 == 0 &&
        (((uintptr_t)x | (uintptr_t)out | (uintptr_t)tail) & 15) == 0) {
        const dim3 grid8((max_q_len + CONV_SEG - 1) / CONV_SEG, n_seqs, (C / 8 + CONV8_THREADS - 1) / CONV8_THREADS);
#define CONV8_GO(TAPS_, ADD_, SILU_)                                                                                           \
    hipLaunchKernelGGL((causal_conv_bf16x8_kernel<TAPS_, ADD_, SILU_>), grid8, dim3(CONV8_THREADS), 0, (hipStream_t)stream,   \
                       (const bf16*)x, ld_x, w, (bf16*)tail, cu_q, slot_ids, (bf16*)out, ld_out, C, bias, in_bias)
#define CONV8_ACT(TAPS_)                                         \
    do {                                                         \
        if ((flags & 3) == 3) CONV8_GO(TAPS_, true, true);       \
        else if (flags & 1) CONV8_GO(TAPS_, true, false);        \
        else if (flags & 2) CONV8_GO(TAPS_, false, true);        \
        else CONV8_GO(TAPS_, false, false);                      \
    } while (0)
        if (taps == 2) CONV8_ACT(2); else if (taps == 3) CONV8_ACT(3); else CONV8_ACT(4);
#undef CONV8_ACT
#undef CONV8_GO
        return ra_launch_status();
    }
    dim3 grid((max_q_len + CONV_SEG - 1) / CONV_SEG, n_seqs, (C + 255) / 256), block(256);
#define CONV_GO(T_, MT_)                                                                                                 \
    hipLaunchKernelGGL((causal_conv_kernel<T_, MT_>), grid, block, 0, (hipStream_t)stream, (const T_*)x, ld_x, w, (T_*)tail, \
                       cu_q, slot_ids, (T_*)out, ld_out, C, taps, flags, bias, in_bias)
#define CONV_TAPS(T_)                                                                                                    \
    do {                                                                                                                 \
        if (taps <= 4) CONV_GO(T_, 4); else if (taps <= 8) CONV_GO(T_, 8); else CONV_GO(T_, CONV_MAX_TAPS);              \
    } while (0)
    if (dtype == RA_DTYPE_F32) CONV_TAPS(float); else CONV_TAPS(bf16);
#undef CONV_TAPS
#undef CONV_GO
    return ra_launch_status();
}

extern "C" int ra_causal_conv(const void* x, long long ld_x, const float* w, void* tail, const int* cu_q,
                              const int* slot_ids, void* out, long long ld_out, int T_tokens, int n_seqs, int max_q_len,
                              int C, int taps, int flags, int dtype, void* stream) {
    return causal_conv_run(x, ld_x, nullptr, w, nullptr, tail, cu_q, slot_ids, out, ld_out, T_tokens, n_seqs, max_q_len, C, taps, flags,
                           dtype, stream);
}

// the same with a bias per channel (fp32 [C]) added to the filter's sum before the activation, and one added to the
// inputs (each may be null)
extern "C" int ra_causal_conv_bias(const void* x, long long ld_x, const float* in_bias, const float* w, const float* bias, void* tail,
                                   const int* cu_q, const int* slot_ids, void* out, long long ld_out, int T_tokens, int n_seqs,
                                   int max_q_len, int C, int taps, int flags, int dtype, void* stream) {
    return causal_conv_run(x, ld_x, in_bias, w, bias, tail, cu_q, slot_ids, out, ld_out, T_tokens, n_seqs, max_q_len, C, taps, flags,
                           dtype, stream);
}

// A pre-norm and the convolution behind it for steps in which every request brings one token, bfloat16: h += delta, x = h / rms(h) w rounded
// to bfloat16, out = x + filter(x), one workgroup a request, four channels a thread; bit for bit what the norm's kernel (its thread
// count, order of sums and rounding) and the one above give. Both are bound by their start and end (4.6 us each in a decode step); the tail and
// the filter are asked for before the norm's sum is formed. Four taps, two kernels / this in a graph: a row of 2,048 5.6 / 3.7 us, of 4,096
// 6.3 / 5.0, 64 rows of 4,096 7.5 / 5.6. Several tokens a request need the rows before a token's own normed, so they stay with two kernels.
template <int TAPS>
__global__ __launch_bounds__(1024) void norm_conv_one_kernel(float* __restrict__ h, const bf16* __restrict__ delta, const float* __restrict__ norm_w,
                                                             float eps, const float* __restrict__ w, bf16* __restrict__ tail,
                                                             const int* __restrict__ slot_ids, bf16* __restrict__ out, int H) {
    __shared__ float scratch[16];
    const int r = blockIdx.x, c = 4 * threadIdx.x;
    const bool in = c < H;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f), nw = v;
    float taps[4][TAPS], win[TAPS - 1][4], ss = 0.f;
    bf16* my_tail = tail + (size_t)slot_ids[r] * (TAPS - 1) * H + c;
    if (in) {
        float4* hr = reinterpret_cast<float4*>(h + (size_t)r * H + c);
        v = *hr;
        if (delta != nullptr) {
            const uint2 d = *reinterpret_cast<const uint2*>(delta + (size_t)r * H + c);
            v.x += __uint_as_float(d.x << 16);
            v.y += __uint_as_float(d.x & 0xffff0000u);
            v.z += __uint_as_float(d.y << 16);
            v.w += __uint_as_float(d.y & 0xffff0000u);
            *hr = v;
        }
        nw = *reinterpret_cast<const float4*>(norm_w + c);
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) {
            const uint2 t = *reinterpret_cast<const uint2*>(my_tail + (size_t)j * H);
            win[j][0] = __uint_as_float(t.x << 16);
            win[j][1] = __uint_as_float(t.x & 0xffff0000u);
            win[j][2] = __uint_as_float(t.y << 16);
            win[j][3] = __uint_as_float(t.y & 0xffff0000u);
        }
#pragma unroll
        for (int i = 0; i < TAPS; ++i) {                       // four channels' filters lie side by side
            const float4 t = reinterpret_cast<const float4*>(w + (size_t)c * TAPS)[i];
            const float f[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) taps[(4 * i + k) / TAPS][(4 * i + k) % TAPS] = f[k];
        }
        ss += v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w;
    }
    ss = block_sum(ss, scratch);
    const float rstd = 1.0f / sqrtf(ss / (float)H + eps);
    if (!in) return;
    const float x[4] = {round_to<bf16>(v.x * rstd * nw.x), round_to<bf16>(v.y * rstd * nw.y), round_to<bf16>(v.z * rstd * nw.z),
                        round_to<bf16>(v.w * rstd * nw.w)};
    float y[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        y[k] = 0.f;
#pragma unroll
        for (int j = 0; j < TAPS - 1; ++j) y[k] = fmaf(taps[k][j], win[j][k], y[k]);
        y[k] = fmaf(taps[k][TAPS - 1], x[k], y[k]);
        y[k] += x[k];
    }
    auto pack = [](const float (&f)[4]) {
        return make_uint2((uint32_t)f2bf_bits(f[0]) | ((uint32_t)f2bf_bits(f[1]) << 16), (uint32_t)f2bf_bits(f[2]) | ((uint32_t)f2bf_bits(f[3]) << 16));
    };
    *reinterpret_cast<uint2*>(out + (size_t)r * H + c) = pack(y);
#pragma unroll
    for (int j = 0; j + 1 < TAPS - 1; ++j) *reinterpret_cast<uint2*>(my_tail + (size_t)j * H) = pack(win[j + 1]);
    *reinterpret_cast<uint2*>(my_tail + (size_t)(TAPS - 2) * H) = pack(x);
}

extern "C" int ra_norm_conv_fits(int H, int taps) { return H > 0 && H % 4 == 0 && H <= 4096 && taps >= 2 && taps <= 4; }

// h fp32 [rows, H], delta (may be null) and out bfloat16 [rows, H], w [H, taps], tail [slots, taps - 1, H]; row r is request r's one token.
// h, norm_w and w 16-byte aligned, the others 8.
extern "C" int ra_norm_conv_one(float* h, const void* delta, const float* norm_w, float eps, const float* w, void* tail, const int* slot_ids, void* out,
                                int rows, int H, int taps, void* stream) {
    if (rows <= 0) return RA_OK;
    if (!ra_norm_conv_fits(H, taps) || (((uintptr_t)h | (uintptr_t)norm_w | (uintptr_t)w) & 15) != 0 ||
        (((uintptr_t)delta | (uintptr_t)tail | (uintptr_t)out) & 7) != 0)
        return RA_ERR_ARG;
    const dim3 block(H <= 1024 ? 256 : H <= 2048 ? 512 : 1024);
#define NORM_CONV(TAPS_)                                                                                                               \
    hipLaunchKernelGGL(norm_conv_one_kernel<TAPS_>, dim3(rows), block, 0, (hipStream_t)stream, h, (const bf16*)delta, norm_w, eps, w,  \
                       (bf16*)tail, slot_ids, (bf16*)out, H)
    if (taps == 2) NORM_CONV(2); else if (taps == 3) NORM_CONV(3); else NORM_CONV(4);
#undef NORM_CONV
    return ra_launch_status();
}
