// Attention of whole prompts (every request's tokens from position 0 on, all of them in this step) over latent rows, bfloat16, with
// the keys and values of the heads formed: k_h = [W_uk,h c | kr], v_h = W_uv,h c, one product over the step's rows c. The kernels of
// attention_latent_mfma.hip read the latents themselves, which is right where cached rows are read by few queries: a score costs
// C + R products and its value C, 1,088 with latents of 512 and rotated parts of 64. A prompt's queries read each key as often as
// there are queries behind it, and here a score costs D + R and its value Dv: 320. The products with W_uk and W_uv cost the same on
// either side.
//
// Head sizes D = Dv = 128, R = 0 or 64. One workgroup of four waves per (q tile of 128 rows, head); a wave has two groups of 16
// rows, so that an operand that comes out of LDS serves two matrix instructions. Per pass a tile of BN keys sits in LDS, keys and values
// row-major with padded rows (two buffers; the next tile's rows are on their way into registers). The scheme of
// attention_prefill.hip: S^T = K Q^T with the keys as A operand, softmax in registers, O^T += V^T P^T through the transposing read,
// P as two bfloat16 halves (16 bits of mantissa), maximum and sums 32-bit. A query's rotated part is turned as it is loaded
// (element i with i + 32); the keys' comes out of the key pool, turned. The workgroups of a head go to one XCD, whose L2 then holds
// the head's keys and values. At the end the sink's term joins the denominator, and the result is multiplied by sigmoid(gate).
//
// Measured, latents of 512 and rotated parts of 64, over the latents / over formed keys and values (launch included): four prompts
// of 777 tokens, 32 heads 459 / 79 us, one of 2,333, 16 heads 435 / 129 (0.37 PFLOP/s with the second half of P counted: the
// causal tiles of few heads leave CUs idle at the end). Bound by the vector work of the softmax between the matrix instructions.
#include "common.h"

typedef __bf16 lp_b8 __attribute__((ext_vector_type(8)));
typedef __bf16 lp_b2 __attribute__((ext_vector_type(2)));
typedef short lp_s4 __attribute__((ext_vector_type(4)));
typedef short lp_s8 __attribute__((ext_vector_type(8)));
typedef float lp_f2 __attribute__((ext_vector_type(2)));
typedef float lp_f4 __attribute__((ext_vector_type(4)));
typedef uint32_t lp_u4 __attribute__((ext_vector_type(4)));
typedef lp_s4 __attribute__((address_space(3))) * lp_lds_s4;

#define LP_LOG2E 1.44269504088896340736f
#define LP_BM 128

__device__ __forceinline__ uint32_t lp_pack2(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(lp_f2{a, b}, lp_b2));
}

template <int R>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void attn_latent_prompt_kernel(
    const bf16* __restrict__ q, long long ld_q, const bf16* __restrict__ kx, const bf16* __restrict__ vx, long long ld_kv,
    const bf16* __restrict__ kr_pool, const int* __restrict__ slots, const float* __restrict__ cos_t, const float* __restrict__ sin_t,
    const int* __restrict__ cu_q, const int* __restrict__ tiles, int n_tiles, int H, float scale,
    const float* __restrict__ sink, const bf16* __restrict__ gate, long long ld_gate, bf16* __restrict__ out) {
    constexpr int D = 128, DK = D + R, NQ = DK / 32, BN = R ? 32 : 64, KS = DK + 8, VS = D + 16, TPK = 256 / BN, D16 = D / 16;
    constexpr int NK = DK / 8 / TPK, NV = D / 8 / TPK;         // pieces of a key and of a value that a thread moves
    static_assert(DK / 8 % TPK == 0 && D / 8 % TPK == 0, "pieces");
    constexpr int TILE = BN * KS + BN * VS;
    __shared__ __attribute__((aligned(16))) uint16_t tiles_s[2 * TILE];
    int head, tile;
    {
        const int wg = blockIdx.x;
        if (H % 8 == 0) {
            const int slot = wg >> 3, per = H >> 3;
            head = (slot % per) * 8 + (wg & 7);
            tile = slot / per;
        } else {
            head = wg % H;
            tile = wg / H;
        }
    }
    const int seg = tiles[2 * tile], q_off = tiles[2 * tile + 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = lane & 15, g = lane >> 4;
    const int row0 = cu_q[seg], q_len = cu_q[seg + 1] - row0;

    int pos_q[2];
    bool q_ok[2];
    lp_b8 bq[2][NQ];
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
        pos_q[qg] = q_off + (wave * 2 + qg) * 16 + n;
        q_ok[qg] = pos_q[qg] < q_len;
        const int at = min(pos_q[qg], q_len - 1);
        const bf16* qp = q + (size_t)(row0 + at) * ld_q + (size_t)head * DK + 8 * g;
#pragma unroll
        for (int j = 0; j < NQ; ++j) bq[qg][j] = *reinterpret_cast<const lp_b8*>(qp + 32 * j);
        if constexpr (R > 0) {
            if (cos_t != nullptr) {                            // (a request's tokens are its positions)
                const float* cs = cos_t + (size_t)at * 32 + 8 * g;
                const float* sn = sin_t + (size_t)at * 32 + 8 * g;
                const lp_u4 a = __builtin_bit_cast(lp_u4, bq[qg][NQ - 2]), b = __builtin_bit_cast(lp_u4, bq[qg][NQ - 1]);
                lp_u4 ra, rb;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float x0 = __uint_as_float(a[i] << 16), x1 = __uint_as_float(a[i] & 0xffff0000u);
                    const float y0 = __uint_as_float(b[i] << 16), y1 = __uint_as_float(b[i] & 0xffff0000u);
                    const float c0 = cs[2 * i], c1 = cs[2 * i + 1], s0 = sn[2 * i], s1 = sn[2 * i + 1];
                    ra[i] = lp_pack2(x0 * c0 - y0 * s0, x1 * c1 - y1 * s1);
                    rb[i] = lp_pack2(y0 * c0 + x0 * s0, y1 * c1 + x1 * s1);
                }
                bq[qg][NQ - 2] = __builtin_bit_cast(lp_b8, ra);
                bq[qg][NQ - 1] = __builtin_bit_cast(lp_b8, rb);
            }
        }
    }
    const int last = min(q_off + LP_BM, q_len) - 1;            // the tile's last position
    const int wave_first = q_off + wave * 32, wave_last = wave_first + 31;
    const float scale2 = scale * LP_LOG2E;
    float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.f, 0.f};      // (the maxima are raw scores, before the scale)
    lp_f4 acc[2][D16];
#pragma unroll
    for (int qg = 0; qg < 2; ++qg)
#pragma unroll
        for (int dt = 0; dt < D16; ++dt) acc[qg][dt] = lp_f4{0.f, 0.f, 0.f, 0.f};

    const int my_key = tid / TPK, my_sub = tid % TPK;
    lp_u4 kreg[NK], vreg[NV];
    auto token_of = [&](int kp) { return row0 + min(kp, last); };      // (so that every address is valid)
    auto slot_of = [&](int t) { return R > 0 ? slots[t] : 0; };
    auto fetch = [&](int t, int slot) {
        const bf16* kp = kx + (size_t)t * ld_kv + (size_t)head * D;
        const bf16* vp = vx + (size_t)t * ld_kv + (size_t)head * D;
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int pc = my_sub + TPK * i;
            kreg[i] = 8 * TPK * i < D ? *reinterpret_cast<const lp_u4*>(kp + 8 * pc)
                                      : *reinterpret_cast<const lp_u4*>(kr_pool + (size_t)slot * R + (8 * pc - D));
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) vreg[i] = *reinterpret_cast<const lp_u4*>(vp + 8 * (my_sub + TPK * i));
    };
    auto stage = [&](int buf) {
        uint16_t* k_s = tiles_s + buf * TILE + my_key * KS;
        uint16_t* v_s = tiles_s + buf * TILE + BN * KS + my_key * VS;
#pragma unroll
        for (int i = 0; i < NK; ++i) *reinterpret_cast<lp_u4*>(k_s + 8 * (my_sub + TPK * i)) = kreg[i];
#pragma unroll
        for (int i = 0; i < NV; ++i) *reinterpret_cast<lp_u4*>(v_s + 8 * (my_sub + TPK * i)) = vreg[i];
    };
    int t_next, slot_next;                                     // of this thread's key in the tile fetched next
    {
        const int t0 = token_of(my_key);
        t_next = token_of(BN + my_key);
        const int s0 = slot_of(t0);
        slot_next = slot_of(t_next);
        fetch(t0, s0);
        stage(0);
        fetch(t_next, slot_next);
        t_next = token_of(2 * BN + my_key);
        slot_next = slot_of(t_next);
    }
    __syncthreads();
    int cur = 0;
    for (int u = 0; u <= last; u += BN, cur ^= 1) {
        const uint16_t* k_cur = tiles_s + cur * TILE;
        const uint16_t* v_cur = k_cur + BN * KS;
        if (u + BN <= last) {
            stage(cur ^ 1);
            if (u + 2 * BN <= last) {
                fetch(t_next, slot_next);
                t_next = token_of(u + 3 * BN + my_key);
                slot_next = slot_of(t_next);
            }
        }
        if (u <= wave_last) {                                  // (a tile above every row of the wave has nothing for it)
            lp_f4 cs[2][BN / 16];
#pragma unroll
            for (int st = 0; st < BN / 16; ++st) {
                cs[0][st] = cs[1][st] = lp_f4{0.f, 0.f, 0.f, 0.f};
                const uint16_t* kr = &k_cur[(st * 16 + n) * KS + 8 * g];
#pragma unroll
                for (int j = 0; j < NQ; ++j) {
                    const lp_b8 a = *reinterpret_cast<const lp_b8*>(kr + 32 * j);
#pragma unroll
                    for (int qg = 0; qg < 2; ++qg) cs[qg][st] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bq[qg][j], cs[qg][st], 0, 0, 0);
                }
            }
            MFMA_SETTLE();
            const bool need_mask = u + BN - 1 > wave_first;
            lp_u4 pw[2][BN / 32], pl[2][BN / 32];              // the weights' upper and lower halves
#pragma unroll
            for (int qg = 0; qg < 2; ++qg) {
                float s[BN / 16][4], mx = -INFINITY;
#pragma unroll
                for (int st = 0; st < BN / 16; ++st)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        s[st][i] = cs[qg][st][i];
                        if (need_mask && u + st * 16 + 4 * g + i > pos_q[qg]) s[st][i] = -INFINITY;
                        mx = fmaxf(mx, s[st][i]);
                    }
                mx = rows_max(mx);
                const float m_new = fmaxf(m_run[qg], mx), m_use = m_new == -INFINITY ? 0.f : m_new, off = -m_use * scale2;
                float lsum = 0.f;
#pragma unroll
                for (int st = 0; st < BN / 16; ++st)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        s[st][i] = __builtin_amdgcn_exp2f(fmaf(s[st][i], scale2, off));
                        lsum += s[st][i];
                    }
                lsum = rows_sum(lsum);
                const float alpha = m_run[qg] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((m_run[qg] - m_use) * scale2);
                l_run[qg] = l_run[qg] * alpha + lsum;
                if (__any(m_new != m_run[qg])) {
#pragma unroll
                    for (int dt = 0; dt < D16; ++dt) acc[qg][dt] *= alpha;
                }
                m_run[qg] = m_new;
#pragma unroll
                for (int b = 0; b < BN / 32; ++b)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float x = s[2 * b + (j >> 1)][2 * (j & 1)], y = s[2 * b + (j >> 1)][2 * (j & 1) + 1];
                        const uint32_t hi = lp_pack2(x, y);
                        pw[qg][b][j] = hi;
                        pl[qg][b][j] = lp_pack2(x - __uint_as_float(hi << 16), y - __uint_as_float(hi & 0xffff0000u));
                    }
            }
#pragma unroll
            for (int b = 0; b < BN / 32; ++b) {
                const uint16_t* vr = &v_cur[(32 * b + 4 * g + (n >> 2)) * VS + 4 * (n & 3)];
#pragma unroll
                for (int dt = 0; dt < D16; ++dt) {
                    const lp_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_s4)(vr + dt * 16));
                    const lp_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lp_lds_s4)(vr + 16 * VS + dt * 16));
                    const lp_b8 v = __builtin_bit_cast(lp_b8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
#pragma unroll
                    for (int qg = 0; qg < 2; ++qg) {
                        acc[qg][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, __builtin_bit_cast(lp_b8, pw[qg][b]), acc[qg][dt], 0, 0, 0);
                        acc[qg][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, __builtin_bit_cast(lp_b8, pl[qg][b]), acc[qg][dt], 0, 0, 0);
                    }
                }
            }
        }
        __syncthreads();                                       // every wave is done with this tile, the next one is complete
    }
    MFMA_SETTLE();
#pragma unroll
    for (int qg = 0; qg < 2; ++qg) {
        if (!q_ok[qg]) continue;
        float inv = l_run[qg] > 0.f ? 1.0f / l_run[qg] : 0.f;
        if (sink != nullptr) {                                 // (its score may be far above the others)
            const float sl = sink[head] * LP_LOG2E, m2 = m_run[qg] * scale2, top = fmaxf(m2, sl);
            const float rescale = __builtin_amdgcn_exp2f(m2 - top), l = fmaf(l_run[qg], rescale, __builtin_amdgcn_exp2f(sl - top));
            inv = l > 0.f ? rescale / l : 0.f;
        }
        const size_t t = row0 + pos_q[qg];
        if (gate != nullptr) inv *= 1.0f / (1.0f + expf(-to_f(gate[t * ld_gate + head])));
        bf16* op = out + (t * H + head) * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < D16; ++dt) {
            uint2 w;
            w.x = lp_pack2(acc[qg][dt][0] * inv, acc[qg][dt][1] * inv);
            w.y = lp_pack2(acc[qg][dt][2] * inv, acc[qg][dt][3] * inv);
            *reinterpret_cast<uint2*>(op + dt * 16) = w;
        }
    }
}

// rows[i] = pool row slots[i], C elements each (C a multiple of 8)
__global__ __launch_bounds__(256) void latent_rows_kernel(const uint4* __restrict__ pool, const int* __restrict__ slots,
                                                          uint4* __restrict__ rows, int per_row, long long total) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= total) return;
    const long long t = i / per_row;
    rows[i] = pool[(long long)slots[t] * per_row + (i - t * per_row)];
}

extern "C" int ra_latent_rows(const void* pool, const int* slots, void* rows, int T_tokens, int C, void* stream) {
    if (T_tokens <= 0) return RA_OK;
    if (C < 8 || C % 8 != 0 || (((uintptr_t)pool | (uintptr_t)rows) & 15) != 0) return RA_ERR_ARG;
    const long long total = (long long)T_tokens * (C / 8);
    hipLaunchKernelGGL(latent_rows_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, (hipStream_t)stream, (const uint4*)pool, slots,
                       (uint4*)rows, C / 8, total);
    return ra_launch_status();
}

// Head sizes and ranks that the kernel takes; rotary: elements of R that turn (0 or all of them).
extern "C" int ra_attention_latent_prompt_fits(int H, int D, int R, int Dv, int rotary) {
    return H >= 1 && D == 128 && Dv == 128 && (R == 0 || R == 64) && (rotary == 0 || rotary == R);
}

// q [T, ld_q]: heads of D + R, the rotated parts not yet turned (cos_t, sin_t [positions, R / 2]; null: none turns); kv [T, ld_kv]:
// H D key elements, then H Dv value elements; kr_pool rows of R by slot, turned; tiles [n_tiles][2] of 128 rows; sink [H] (null:
// none); gate: H logits a token, rows ld_gate apart (null: none); out [T, H Dv]. Every request's rows begin at position 0.
extern "C" int ra_attention_latent_prompt(const void* q, long long ld_q, const void* kv, long long ld_kv, const void* kr_pool,
                                          const int* slots, const float* cos_t, const float* sin_t, const int* cu_q, const int* tiles,
                                          int n_tiles, int H, int D, int R, int Dv, float scale, const float* sink,
                                          const void* gate, long long ld_gate, void* out, void* stream) {
    if (n_tiles <= 0) return RA_OK;
    if (!ra_attention_latent_prompt_fits(H, D, R, Dv, cos_t != nullptr ? R : 0) || !(scale > 0.f) ||
        ld_q < (long long)H * (D + R) || ld_kv < (long long)H * (D + Dv) || ld_q % 8 != 0 || ld_kv % 8 != 0 ||
        (((uintptr_t)q | (uintptr_t)kv | (uintptr_t)kr_pool) & 15) != 0 || ((uintptr_t)out & 7) != 0 || (R > 0 && kr_pool == nullptr) ||
        (long long)n_tiles * H > 0x7fffffffLL)
        return RA_ERR_ARG;
    const dim3 grid(n_tiles * H), block(256);
    hipStream_t st = (hipStream_t)stream;
    const bf16* k = (const bf16*)kv;
#define LP_GO(R_)                                                                                                                   \
    hipLaunchKernelGGL(attn_latent_prompt_kernel<R_>, grid, block, 0, st, (const bf16*)q, ld_q, k, k + (size_t)H * D, ld_kv,         \
                       (const bf16*)kr_pool, slots, cos_t, sin_t, cu_q, tiles, n_tiles, H, scale, sink, (const bf16*)gate, \
                       ld_gate, (bf16*)out)
    if (R > 0) LP_GO(64); else LP_GO(0);
#undef LP_GO
    return ra_launch_status();
}
