// Attention in float32 over the paged cache for heads of 64 and 128: prompts by the 32-bit matrix instructions, single tokens
// with a pass's keys and values asked for at once. Tables, masks and options are those of attention_plain.hip (formulas:
// rollout/attention.py:126-139, head mapping 65); every product and sum is 32-bit here too, in another order.
//
// Prompts: a workgroup of four waves takes 64 query rows of one head (a wave 16), K and V of 64 keys at a time in LDS, the next
// 64 on their way into registers. Scores are S^T = K Q^T by 16x16x4 products: a lane reads four neighbouring elements of a
// key, and four products take one of them each, so the contraction runs over the head's elements in the order 16 i + 4 g + j
// (lane group g, product j). Lane (n, g) ends up with keys 4g..4g+3 of every 16 for query n, which is how P^T enters
// O^T += V^T P^T. Rows in LDS are 4 elements longer than a head: both reads meet no bank conflict. Bound by the matrix
// instructions (32 cycles each) and, on short prompts, by the few tiles in a row. Microseconds, the plain kernel / this one, 32
// heads over 8 of 128: 3 prompts of 211 tokens 309 / 52, one of 64 37 / 16, of 1,000 1,076 / 198, of 4,000 11.8 ms / 2.0 ms, 17
// tokens after 2,000 418 / 259; 8 heads over 2 of 64: 3 of 211 62 / 29, 17 after 2,000 177 / 173.
//
// Single tokens: a workgroup of eight waves per (request, head), chunk c of 16 positions with wave c % 8. The plain kernel
// takes 64 keys a wave with loads that wait for each other; here a wave has all loads of its chunk in flight, and the next
// chunk's row numbers. Microseconds, the plain kernel / this one, 32 heads over 8 of 128: 3 requests of 211 keys (cold) 60 / 9,
// 1 of 4,000 422 / 72, 8 of 2,000 221 / 43, 64 of 500 210 / 93. A request's head stays with one workgroup: few requests over
// long contexts leave CUs idle.
#include "common.h"

typedef float af_f4 __attribute__((ext_vector_type(4)));

#define AF_BM 64
#define AF_BN 64

template <int D16>
__global__ __launch_bounds__(256, 2) void attn_prefill_f32_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ k_pool, const float* __restrict__ v_pool,
    const int* __restrict__ page_table, const int* __restrict__ cu_pages, const int* __restrict__ kv_start,
    const int* __restrict__ cu_q, const int* __restrict__ q_start, const int* __restrict__ tiles, int Hq, int Hkv, int P,
    float scale, int window, const float* __restrict__ head_scale, float softcap, int keep_first, int sink,
    const float* __restrict__ sink_logit, float out_scale, long long ld_out) {
    constexpr int D = 16 * D16, S = D + 4;
    __shared__ __attribute__((aligned(16))) float k_s[AF_BN * S], v_s[AF_BN * S];
    const int seg = tiles[2 * blockIdx.x], q_off = tiles[2 * blockIdx.x + 1], head = blockIdx.y, kvh = head / (Hq / Hkv);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int q_len = cu_q[seg + 1] - cu_q[seg], start = kv_start[seg];
    const int* pt = page_table + cu_pages[seg];
    const int n_listed = cu_pages[seg + 1] - cu_pages[seg];
    const int local = q_off + 16 * wave + n, row = cu_q[seg] + local;
    const bool mine = local < q_len;
    const int pos = q_start[seg] + local;
    const int first = window > 0 ? max(start, pos - window + 1) : start;
    // keys that any row of the tile reads: [lo, hi], and those below keep_first
    const int lo = window > 0 ? max(start, q_start[seg] + q_off - window + 1) : start;
    const int hi = q_start[seg] + min(q_off + AF_BM, q_len) - 1;
    if (head_scale != nullptr) scale *= head_scale[head];
    const float inv_cap = softcap > 0.f ? 1.0f / softcap : 0.f;

    const af_f4 zero = {0.f, 0.f, 0.f, 0.f};
    af_f4 qv[D16];
#pragma unroll
    for (int i = 0; i < D16; ++i)
        qv[i] = mine ? *reinterpret_cast<const af_f4*>(q + ((size_t)row * Hq + head) * D + 16 * i + 4 * g) : zero;

    // this thread's key of a tile and its quarter of the pieces of the row
    const int key = tid >> 2, part = tid & 3;
    af_f4 kr[D16], vr[D16];
    auto ask = [&](int c) {
        const int idx = c * AF_BN + key - start, page = idx >= 0 ? idx / P : 0;
        const int p = c * AF_BN + key;
        const bool there = idx >= 0 && page < n_listed && p <= hi && (p >= lo || p < keep_first);
        const size_t at = there ? (((size_t)pt[page] * Hkv + kvh) * P + (idx - page * P)) * D : 0;
#pragma unroll
        for (int i = 0; i < D16; ++i) {
            kr[i] = there ? *reinterpret_cast<const af_f4*>(k_pool + at + 4 * (part + 4 * i)) : zero;
            vr[i] = there ? *reinterpret_cast<const af_f4*>(v_pool + at + 4 * (part + 4 * i)) : zero;
        }
    };
    auto put = [&]() {                                     // returns whether one of the values is no finite number
        bool odd = false;
#pragma unroll
        for (int i = 0; i < D16; ++i) {
            *reinterpret_cast<af_f4*>(&k_s[key * S + 4 * (part + 4 * i)]) = kr[i];
            *reinterpret_cast<af_f4*>(&v_s[key * S + 4 * (part + 4 * i)]) = vr[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) odd |= !(fabsf(vr[i][j]) < INFINITY);
        }
        return odd;
    };
    // the tiles of 64 positions that hold a key of the tile, in order (with kept first keys those from position 0 on)
    const int c_last = hi / AF_BN;
    auto next = [&](int c) {
        while (c <= c_last && c * AF_BN >= keep_first && (c + 1) * AF_BN <= lo) ++c;
        return c;
    };
    const int end = start + n_listed * P;
    auto sees = [&](int p) { return p <= pos && p >= start && p < end && (p >= first || p < keep_first); };
    af_f4 acc[D16];
#pragma unroll
    for (int i = 0; i < D16; ++i) acc[i] = zero;
    float m = -INFINITY, l = 0.f;
    int c = next(keep_first > 0 ? 0 : lo / AF_BN);
    if (c <= c_last) ask(c);
    while (c <= c_last) {
        __syncthreads();                                   // every wave has left the tile before
        const bool odd = __syncthreads_or(put());
        const int c_next = next(c + 1);
        if (c_next <= c_last) ask(c_next);
        af_f4 sc[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) sc[b] = zero;
#pragma unroll
        for (int i = 0; i < D16; ++i) {
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const af_f4 kk = *reinterpret_cast<const af_f4*>(&k_s[(16 * b + n) * S + 16 * i + 4 * g]);
#pragma unroll
                for (int j = 0; j < 4; ++j) sc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kk[j], qv[i][j], sc[b], 0, 0, 0);
            }
        }
        MFMA_SETTLE();
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = c * AF_BN + 16 * b + 4 * g + r;
                float d = sc[b][r] * scale;
                if (softcap > 0.f) d = softcap * tanhf(d * inv_cap);
                const bool ok = mine && sees(p);
                sc[b][r] = ok ? d : -INFINITY;
                mx = fmaxf(mx, sc[b][r]);
            }
        const float m_new = fmaxf(m, rows_max(mx));
        const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
        float sum = 0.f;
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[b][r] = sc[b][r] == -INFINITY ? 0.f : expf(sc[b][r] - m_new);
                sum += sc[b][r];
            }
        l = l * alpha + sum;                               // (of this lane's keys; the lanes' sums are added at the end)
        m = m_new;
#pragma unroll
        for (int i = 0; i < D16; ++i) acc[i] *= alpha;
        if (odd) {                                         // weight 0 times such a value is no zero: keys a row does not see are left out
            for (int e = 0; e < AF_BN; ++e) {
                const float mine_p = (e >> 4) == 0 ? sc[0][e & 3] : (e >> 4) == 1 ? sc[1][e & 3] : (e >> 4) == 2 ? sc[2][e & 3] : sc[3][e & 3];
                const float pe = __shfl(mine_p, n + 16 * ((e >> 2) & 3), 64);
                if (!mine || !sees(c * AF_BN + e)) continue;
#pragma unroll
                for (int i = 0; i < D16; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][r] = fmaf(pe, v_s[e * S + 16 * i + 4 * g + r], acc[i][r]);
            }
            c = c_next;
            continue;
        }
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < D16; ++i)
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(v_s[(16 * b + 4 * g + r) * S + 16 * i + n], sc[b][r], acc[i], 0, 0, 0);
        MFMA_SETTLE();
        c = c_next;
    }
    float den = rows_sum(l), factor = out_scale;
    if (sink && sink_logit == nullptr) {
        den += expf(-m);                                   // one more key of score 0 that has no value
    } else if (sink) {                                     // one with a score of its own, which may be far above the others
        const float sl = sink_logit[head], top = fmaxf(m, sl), ew = m == -INFINITY ? 0.f : expf(m - top);
        factor *= ew;
        den = fmaf(den, ew, expf(sl - top));
    }
    if (!mine) return;
#pragma unroll
    for (int i = 0; i < D16; ++i) {
        af_f4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = den > 0.f ? acc[i][r] / den * factor : 0.f;
        float* to = out + (size_t)row * ld_out + (size_t)head * D + 16 * i + 4 * g;
#pragma unroll
        for (int r = 0; r < 4; ++r) to[r] = v[r];
    }
}

// one token of each listed request; segs null: request i is i
template <int D16>
__global__ __launch_bounds__(512) void attn_decode_f32_kernel(
    const float* __restrict__ q, float* __restrict__ out, const float* __restrict__ k_pool, const float* __restrict__ v_pool,
    const int* __restrict__ page_table, const int* __restrict__ cu_pages, const int* __restrict__ kv_start,
    const int* __restrict__ cu_q, const int* __restrict__ q_start, const int* __restrict__ segs, int Hq, int Hkv, int P,
    float scale, int window, const float* __restrict__ head_scale, float softcap, int keep_first, int sink,
    const float* __restrict__ sink_logit, float out_scale, long long ld_out) {
    constexpr int D = 16 * D16, VW = D / 64, WAVES = 8, CH = 16;
    __shared__ float ml_s[WAVES][2], acc_s[WAVES][D];
    const int seg = segs ? segs[blockIdx.x] : blockIdx.x, head = blockIdx.y, kvh = head / (Hq / Hkv);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, part = lane & 3, sub = lane >> 2;
    const int row = cu_q[seg], start = kv_start[seg], pos = q_start[seg];
    const int* pt = page_table + cu_pages[seg];
    const int n_listed = cu_pages[seg + 1] - cu_pages[seg];
    const int first = window > 0 ? max(start, pos - window + 1) : start;
    if (head_scale != nullptr) scale *= head_scale[head];
    const float inv_cap = softcap > 0.f ? 1.0f / softcap : 0.f;
    af_f4 qv[D16];
#pragma unroll
    for (int i = 0; i < D16; ++i) qv[i] = *reinterpret_cast<const af_f4*>(q + ((size_t)row * Hq + head) * D + 4 * (part + 4 * i));
    // the cache row of this lane's key of chunk c, or -1
    auto row_of = [&](int c) {
        const int p = c * CH + sub, idx = p - start, page = idx >= 0 ? idx / P : 0;
        const bool there = p <= pos && idx >= 0 && page < n_listed && (p >= first || p < keep_first);
        return there ? (pt[page] * Hkv + kvh) * P + (idx - page * P) : -1;
    };
    const int c_last = pos / CH;
    auto next = [&](int c) {                               // the first chunk from c on, in steps of the waves, that holds a key
        while (c <= c_last && c * CH >= keep_first && (c + 1) * CH <= first) c += WAVES;
        return c;
    };
    float m = -INFINITY, l = 0.f, acc[VW];
#pragma unroll
    for (int i = 0; i < VW; ++i) acc[i] = 0.f;
    // (without kept keys the chunks in front of the first key are passed over at once)
    const int c0 = keep_first > 0 ? 0 : first / CH;
    int c = next(c0 + (wave - c0 % WAVES + WAVES) % WAVES);
    int mine = c <= c_last ? row_of(c) : -1;
    while (c <= c_last) {
        af_f4 kk[D16];
        float vv[CH][VW];
        const float* kp = k_pool + (size_t)max(mine, 0) * D + 4 * part;
#pragma unroll
        for (int i = 0; i < D16; ++i) kk[i] = *reinterpret_cast<const af_f4*>(kp + 16 * i);
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const float* vp = v_pool + (size_t)max(__builtin_amdgcn_readlane(mine, 4 * e), 0) * D + VW * lane;
#pragma unroll
            for (int i = 0; i < VW; ++i) vv[e][i] = vp[i];
        }
        const int c_next = next(c + WAVES), row_next = c_next <= c_last ? row_of(c_next) : -1;
        float d = 0.f;
#pragma unroll
        for (int i = 0; i < D16; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) d = fmaf(qv[i][j], kk[i][j], d);
        d += __shfl_xor(d, 1, 64);
        d += __shfl_xor(d, 2, 64);
        d *= scale;
        if (softcap > 0.f) d = softcap * tanhf(d * inv_cap);
        if (mine < 0) d = -INFINITY;
        const float m_new = fmaxf(m, wave_max(d));
        const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
        const float p = d == -INFINITY ? 0.f : expf(d - m_new);
        l = l * alpha + p;                                 // (of this lane's keys; four lanes count each)
        m = m_new;
#pragma unroll
        for (int i = 0; i < VW; ++i) acc[i] *= alpha;
#pragma unroll
        for (int e = 0; e < CH; ++e) {
            const float pe = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(p), 4 * e));
            // (a key that is not there has weight 0, and row 0 of the pool, which stood in for it, may hold anything)
            const bool there = __builtin_amdgcn_readlane(mine, 4 * e) >= 0;
#pragma unroll
            for (int i = 0; i < VW; ++i) acc[i] = there ? fmaf(pe, vv[e][i], acc[i]) : acc[i];
        }
        c = c_next;
        mine = row_next;
    }
    l = wave_sum(part == 0 ? l : 0.f);
    if (lane == 0) {
        ml_s[wave][0] = m;
        ml_s[wave][1] = l;
    }
#pragma unroll
    for (int i = 0; i < VW; ++i) acc_s[wave][VW * lane + i] = acc[i];
    __syncthreads();
    if (tid >= D) return;
    float mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) mm = fmaxf(mm, ml_s[w][0]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        const float mw = ml_s[w][0], ew = mw == -INFINITY ? 0.f : expf(mw - mm);
        num = fmaf(acc_s[w][tid], ew, num);
        den = fmaf(ml_s[w][1], ew, den);
    }
    if (sink && sink_logit == nullptr) {
        den += expf(-mm);
    } else if (sink) {
        const float sl = sink_logit[head], top = fmaxf(mm, sl), ew = mm == -INFINITY ? 0.f : expf(mm - top);
        num *= ew;
        den = fmaf(den, ew, expf(sl - top));
    }
    out[(size_t)row * ld_out + (size_t)head * D + tid] = den > 0.f ? num / den * out_scale : 0.f;
}

extern "C" int ra_attention_f32_fits(int D) { return D == 64 || D == 128; }

// q tiles of 64 rows: [n_tiles][2] of (request, first row among its new tokens)
extern "C" int ra_attention_prefill_f32(const void* q, void* out, const void* k_pool, const void* v_pool, const int* page_table,
                                        const int* cu_pages, const int* kv_start, const int* cu_q, const int* q_start,
                                        const int* tiles, int n_tiles, int Hq, int Hkv, int D, int P, float scale, int window,
                                        const float* head_scale, float softcap, int keep_first, int sink,
                                        const float* sink_logit, float out_scale, long long ld_out, void* stream) {
    if (n_tiles <= 0) return RA_OK;
    if (!ra_attention_f32_fits(D) || ld_out < (long long)Hq * D || Hkv <= 0 || Hq % Hkv != 0 || P <= 0 || Hq > 65535) return RA_ERR_ARG;
#define AF_PRE(D16_)                                                                                                       \
    hipLaunchKernelGGL((attn_prefill_f32_kernel<D16_>), dim3(n_tiles, Hq), dim3(256), 0, (hipStream_t)stream,              \
                       (const float*)q, (float*)out, (const float*)k_pool, (const float*)v_pool, page_table, cu_pages,     \
                       kv_start, cu_q, q_start, tiles, Hq, Hkv, P, scale, window, head_scale, softcap, keep_first, sink,   \
                       sink_logit, out_scale, ld_out)
    if (D == 64) AF_PRE(4); else AF_PRE(8);
#undef AF_PRE
    return ra_launch_status();
}

extern "C" int ra_attention_decode_f32(const void* q, void* out, const void* k_pool, const void* v_pool, const int* page_table,
                                       const int* cu_pages, const int* kv_start, const int* cu_q, const int* q_start,
                                       const int* segs, int n_dec, int Hq, int Hkv, int D, int P, float scale, int window,
                                       const float* head_scale, float softcap, int keep_first, int sink,
                                       const float* sink_logit, float out_scale, long long ld_out, void* stream) {
    if (n_dec <= 0) return RA_OK;
    if (!ra_attention_f32_fits(D) || ld_out < (long long)Hq * D || Hkv <= 0 || Hq % Hkv != 0 || P <= 0 || Hq > 65535) return RA_ERR_ARG;
#define AF_DEC(D16_)                                                                                                       \
    hipLaunchKernelGGL((attn_decode_f32_kernel<D16_>), dim3(n_dec, Hq), dim3(512), 0, (hipStream_t)stream, (const float*)q, \
                       (float*)out, (const float*)k_pool, (const float*)v_pool, page_table, cu_pages, kv_start, cu_q,      \
                       q_start, segs, Hq, Hkv, P, scale, window, head_scale, softcap, keep_first, sink, sink_logit,        \
                       out_scale, ld_out)
    if (D == 64) AF_DEC(4); else AF_DEC(8);
#undef AF_DEC
    return ra_launch_status();
}
