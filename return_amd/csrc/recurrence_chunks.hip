// The gated recurrences of delta_rule.hip (same rules, same inputs, same state) by chunks of 32 rows.
//
// Walking the rows one after the other costs 0.6 us a row, whatever the width: the walk is a chain of dependent steps.
// Here only the carry from chunk to chunk is a chain. With a_t the decays of a row (one per key channel), P_i the
// products a_1 ... a_i inside a chunk and S the state before it,
//     o_i = sum_(j<=i) A_ij u_j + (q_i P_i) S,            A_ij = sum_d q_i[d] k_j[d] P_i[d] / P_j[d]
//     S  <- P_C S + sum_j (k_j P_C / P_j) u_j
// where u_j is the value (rules 1 and 2, times delta in the latter), or for the delta rules the solution of
//     u_i = beta_i (v_i - sum_(j<i) L_ij u_j - (k_i P_i) S),   L_ij = sum_d k_i[d] k_j[d] P_i[d] / P_j[d]
// that is, with T = (1 + diag(beta) L)^-1,  u = T beta v - (T beta k P) S = U - W S.
//
// Two kernels. The first (prepare), a workgroup per (chunk, head), forms A, U, W, q P, k P_C / P and P_C, which depend on
// no state: unit vectors and decays, products of decays along the rows, A and L by products of 16 x 16 tiles, T by
// substitution in its two diagonal tiles and one product between them, U and W by products with T. The second (carry), a
// workgroup per (request, head, 16 or 32 columns of S), goes through the chunks with its part of S in registers. All
// products are 32-bit matrix instructions (16x16x4), every sum is 32-bit.
//
// The quotients P_i / P_j never overflow: products of decays are formed from one row to the next, between the two halves
// of a chunk as (P_i from the later half's start) times (product from j to the earlier half's end), both at most one,
// and inside a half as (q_i P_i) (k_j / P_j) only where the half's whole product is at least RC_TINY in every channel
// and no key is beyond RC_LARGE; else the half's pairs are formed one by one with the products between them (recur_pairs).
//
// What the carry reads lies in scratch in the order of the matrix instructions' operands: an A operand of the 16x16x4
// product holds, lane (m + 16 g), the four columns 4 g .. 4 g + 3 of row m as one 16-byte load that serves four
// instructions (the k index may be taken in any order as long as both operands take the same), and a result tile, lane
// (n + 16 g), the rows 4 g .. 4 g + 3 of column n: the state's result tiles are the next product's B operands as they
// are, without a trip through LDS. The scratch of a step is cut into runs of chunks of about RC_SCRATCH floats.
//
// Digits. The walk rounds a state twice a row; here the roundings are fewer but fall on products that many rows share, so they
// are kept few: a decay near one is held as what it lacks to one, products of decays are formed as pairs of numbers, an
// operand is an input times one factor that was formed as a pair (rounded once), numbers of a row are formed in 64 bits, and
// every sum of products is several sums (a chain of 4 to 16 roundings). Errors against 64 bits, the walk's taken as 1, over the
// designs' decays, 24 / 64 / 250 / 2,048 rows: read-outs of rule 0 0.93 / 0.85 / 0.67 / 0.55, rule 1 0.82 / 0.63 / 0.33 / 0.12,
// rule 2 0.99 / 0.89 / 0.53 / 0.16, rule 3 1.00 / 0.91 / 0.74 / 0.46, states 0.79 and less; where a state forgets in a row or two,
// read-outs 1.02 and states up to 1.15 (of 6e-8). With products of decays as single numbers and one sum each it was 1.06 to 1.37
// and 1.0.
//
// Bounds and what it measured (bf16, one layer, recurrence without the output kernel): one request of 2,048 rows, 32 heads
// of 128 x 128, rule 0: 224 us (prepare 97, carry 127) where the walk took 1,408; rule 3 202 (1,155), rule 1 148 (1,211);
// four requests of 700 rows 295 (2,344), eight of 250 rows 208 (1,670); 64 heads of 128 x 64, rule 2, eight of 250 rows 172
// (1,116). The products are 11 GFLOP at 32 heads of 128 x 128, about 100 us at the 32-bit matrix rate; of the carry's 1.9 us
// a chunk 0.85 are its 56 products a wave, the rest the way of W S through LDS, which the state waits for. Asking for
// operands two chunks ahead instead of one changes nothing; 16 columns a workgroup in place of 32 when the chip is full
// anyway took 181 us in place of 149 (four of 700 rows). The digits cost 4 to 12 % of the time, the look for
// odd numbers 2 %.
//
// A row that is no number (infinite, NaN) reaches the rows behind it and no row before it, as in the walk; the carry goes through
// a request and head that has one without asking for operands ahead.
#include "common.h"
#include "recurrence_chunks.h"
#include <atomic>
#include <type_traits>

#define RC_C 32                       // rows of a chunk: two tiles of 16
#define RC_TINY 1e-20f
#define RC_LARGE 1e15f
#define RC_SCRATCH (48ll << 20)       // floats of scratch beyond which a step is cut into groups of requests and runs of chunks (192 MiB)
#define RC_GROUP 64                   // requests of one launch at most

typedef float rc_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ rc_f4 rc_mfma(float a, float b, rc_f4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// A product of two tiles as four sums, which rc_sum4 adds up: a chain of roundings is as long as four rows, not sixteen.
struct RcSums { rc_f4 s[4]; };
__device__ __forceinline__ RcSums rc_zero() {
    const rc_f4 z = {0.f, 0.f, 0.f, 0.f};
    return RcSums{{z, z, z, z}};
}
__device__ __forceinline__ RcSums rc_mul4(rc_f4 a, rc_f4 b, RcSums c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) c.s[r] = rc_mfma(a[r], b[r], c.s[r]);
    return c;
}
__device__ __forceinline__ rc_f4 rc_sum4(const RcSums& c) { return (c.s[0] + c.s[1]) + (c.s[2] + c.s[3]); }
// A and T have zeros behind the diagonal, and a product takes them times what stands in later rows: times an infinity or NaN
// that gives NaN in rows before it, which do not know of it. So where a lane of the wave holds such a number (rc_odd; or one so
// large that a sum of it may become one), the product with a diagonal tile is formed another way, and the carry goes through
// such a request and head with code of its own.
__device__ __forceinline__ bool rc_odd(rc_f4 x) {
    return __ballot(!(fabsf(x[0]) + fabsf(x[1]) + (fabsf(x[2]) + fabsf(x[3])) < 1e30f)) != 0ull;
}
// c and the product of two tiles over the rows j <= i alone, one by one (ROWS: i is the result's row, else its column)
template <bool ROWS>
__device__ __forceinline__ rc_f4 rc_lower(rc_f4 a, rc_f4 b, rc_f4 c) {
    const int lane = threadIdx.x & 63, m16 = lane & 15, g4 = (lane >> 4) * 4;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        const int from = 16 * (j >> 2);
        const float y = __shfl(b[j & 3], from + m16, 64);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float x = __shfl(a[j & 3], from + g4 + r, 64);
            if (j <= (ROWS ? g4 + r : m16)) c[r] = fmaf(x, y, c[r]);
        }
    }
    return c;
}
// The same on the matrix instructions, for a tile u whose columns are the result's: takes what is no number out of u and gives
// what the result lacks then, NaN for the rows from there on, zero for those before.
__device__ __forceinline__ rc_f4 rc_spoilt(rc_f4& u) {
    const int lane = threadIdx.x & 63;
    rc_f4 e;
    float run = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const bool odd = !(fabsf(u[r]) < INFINITY);
        run += odd ? NAN : 0.f;
        e[r] = run;
        u[r] = odd ? 0.f : u[r];
    }
    float before = 0.f;
#pragma unroll
    for (int g = 1; g < 4; ++g) {
        const float x = __shfl_up(run, 16 * g, 64);
        before += lane >= 16 * g ? x : 0.f;
    }
    return e + before;
}

// Floats per (chunk, head): W and q P [2][DT], k P_C / P [DT][2], U [VT][2], A [3] tiles of 256, P_C [16 DT], a word that says
// whether an odd number (rc_odd) is among them, and three to keep the next one's tiles at 16 bytes
__host__ __device__ static inline long long rc_stride(int DT, int VT, bool delta) {
    return (long long)((delta ? 6 : 4) * DT + 2 * VT + 3) * 256 + 16 * DT + 4;
}

// Numbers of a row (one or two a row and head) are formed in 64 bits: an error in them is in all of the row's elements alike.
__device__ __forceinline__ double rc_softplus(double x) { return x > 40.0 ? x : log1p(exp(x)); }

// e^x for x <= 20 to about one unit in the last place: the hardware's power of two, of a product with log2 e in two parts.
__device__ __forceinline__ float rc_exp(float x) {
    x = x < -150.f ? -150.f : x;
    const float y = x * 1.44269502f, rest = fmaf(x, 1.92596303e-8f, fmaf(x, 1.44269502f, -y));
    const float e = __builtin_amdgcn_exp2f(y);
    return fmaf(e * 0.693147182f, rest, e);
}
// log(1 + t) for t >= 0: what 1 + t rounds away goes in behind; near zero by the series
__device__ __forceinline__ float rc_log1p(float t) {
    const float u = 1.f + t;
    const float far = fmaf(__builtin_amdgcn_logf(u), 0.693147182f, (t - (u - 1.f)) * __builtin_amdgcn_rcpf(u));
    const float near = t * fmaf(t, fmaf(t, fmaf(t, fmaf(t, 0.2f, -0.25f), 0.333333343f), -0.5f), 1.f);
    return t < 0.015625f ? near : far;
}
// A decay e^g, g <= 0, in one word: near one as e^g - 1 with the sign set, which has the digits that e^g in 32 bits has
// not, else e^g itself.
#define RC_NEAR_ONE (-0.25f)
__device__ __forceinline__ float rc_decay(float g) {
    float e = fmaf(g, 1.f / 7.f, 1.f);
#pragma unroll
    for (int n = 6; n >= 2; --n) e = fmaf(g * e, 1.f / n, 1.f);
    return g > RC_NEAR_ONE ? -fabsf(g * e) : rc_exp(g);
}
__device__ __forceinline__ float rc_decay(double g) { return g > RC_NEAR_ONE ? -fabsf((float)expm1(g)) : (float)exp(g); }
// A number as the sum of two.
struct RcPair { float hi, lo; };
__device__ __forceinline__ RcPair rc_decay_pair(float word) {
    if (!(__float_as_uint(word) & 0x80000000u)) return {word, 0.f};
    const float hi = 1.f + word;
    return {hi, word - (hi - 1.f)};
}
__device__ __forceinline__ RcPair rc_times(RcPair p, RcPair a) {
    const float h = p.hi * a.hi, e = fmaf(p.lo, a.hi, fmaf(p.hi, a.lo, fmaf(p.hi, a.hi, -h))), hi = h + e;
    return {hi, e - (hi - h)};
}
__device__ __forceinline__ RcPair rc_one_over(RcPair p) {
    const float hi = __builtin_amdgcn_rcpf(p.hi);
    return {hi, hi * fmaf(-p.lo, hi, fmaf(-p.hi, hi, 1.f))};
}
__device__ __forceinline__ RcPair rc_pair(double x) { return {(float)x, (float)(x - (double)(float)x)}; }
// x times a pair, rounded once
__device__ __forceinline__ float rc_scaled(float x, RcPair p) { return fmaf(x, p.hi, x * p.lo); }
#define RC_DPP(v, ctrl) ((v) + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, (v)), ctrl, 0xF, 0xF, true)))
// sums over 8 and 16 neighbouring lanes, in every one of them
__device__ __forceinline__ float rc_sum8(float v) {
    v = RC_DPP(v, 0xB1);
    v = RC_DPP(v, 0x4E);
    return RC_DPP(v, 0x141);
}
__device__ __forceinline__ float rc_sum16(float v) {
    v = rc_sum8(v);
    return RC_DPP(v, 0x140);
}

// Chunks of request s that the run of `run` chunks from chunk `first` on holds. (min_rows comes from the rule in the kernel:
// not knowing that a request has at least 16 rows costs the carry 112 registers.)
__device__ __forceinline__ int rc_chunks(const int* cu_q, int s, int n_seqs, int first, int run, int min_rows) {
    if (s >= n_seqs) return 0;
    const int len = cu_q[s + 1] - cu_q[s];
    if (len < min_rows) return 0;
    return max(0, min(run, (len + RC_C - 1) / RC_C - first));
}

// ---------------------------------------------------------------------------------------------------- prepare
// Threads: rows x 8 while rows come in, one per (half, channel) for the products along the rows, then matrix tiles.
template <typename T, int DT>
__global__ __launch_bounds__(256, 2) void recur_prepare_kernel(
    const T* __restrict__ qkv, long long ld_qkv, const T* __restrict__ b, long long ld_b, const T* __restrict__ ag,
    long long ld_ag, const float* __restrict__ A_log, const float* __restrict__ dt_bias, const int* __restrict__ cu_q,
    float* __restrict__ ws, int n_seqs, int H, int G, int D, int V, int first, int run, int rule, float rate, int vec) {
    constexpr int DP = 16 * DT, LD = DP + 4, EP = DP / 8;
    constexpr int VW = 128, LV = VW + 4;                     // columns of v that are staged at a time
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float* qs = sm;                                          // [32][LD]  q as it comes, then unit q times P
    float* ks = qs + RC_C * LD;                              // [32][LD]  k as it comes, then unit k times P
    float* as = ks + RC_C * LD;                              // [32][LD]  decays (rc_decay's words), then k / P
    float* kt = as + RC_C * LD;                              // [16][LD]  first half: k times the decays behind it in the half
    // [32][LV] values: with heads of 128 in the place of k / P, once A and L are formed (two workgroups share a CU's LDS)
    float* vs = DT == 8 ? as : kt + 16 * LD;
    float* Ls = kt + 16 * LD + (DT == 8 ? 0 : RC_C * LV);    // [32][36]  beta L
    float* Ts = Ls + RC_C * 36;                              // [32][36]  T
    float* Ms = Ts + RC_C * 36;                              // [16][20]
    float* SA = Ms + 16 * 20;                                // [2][16][16] pairs of a half formed one by one
    float* SL = SA + 512;
    float* pt = SL + 512;                                    // [2][DP]   product of a half's decays
    float* beta_s = pt + 2 * DP;                             // [32]
    RcPair* nq_s = (RcPair*)(beta_s + RC_C);                 // [32] factors that make q and k of a row unit vectors, q times its scale
    RcPair* nk_s = nq_s + RC_C;                              // [32]
    int* slow = (int*)(nk_s + RC_C);                         // [2]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int h = blockIdx.x, kvh = h / (H / G);
    const bool delta = rule == 0 || rule == 3;

    // ---- which request's chunk
    int s = -1, c = 0;
    {
        int before = 0;
        const int want = blockIdx.y;
        for (int s0 = 0; s0 < n_seqs; s0 += 64) {
            const int n = rc_chunks(cu_q, s0 + lane, n_seqs, first, run, rc_min_rows(rule));
            int incl = n;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int x = __shfl_up(incl, o, 64);
                if (lane >= o) incl += x;
            }
            const int total = __shfl(incl, 63, 64);
            if (want < before + total) {
                const int at = __ffsll((unsigned long long)__ballot(before + incl > want)) - 1;
                s = s0 + at;
                c = want - before - (__shfl(incl, at, 64) - __shfl(n, at, 64));
                break;
            }
            before += total;
        }
    }
    if (s < 0) return;                                       // (the same in every thread)
    const int base = cu_q[s], q_len = cu_q[s + 1] - base;
    const int c0 = (first + c) * RC_C, nt = min(RC_C, q_len - c0);
    const int VT = (V + 15) / 16;
    float* out = ws + ((long long)blockIdx.y * H + h) * rc_stride(DT, VT, delta);
    float* oW = out;                                         // (rules without a correction have no W)
    float* oQ = oW + (delta ? 2 * DT * 256 : 0);
    float* oK = oQ + 2 * DT * 256;
    float* oU = oK + 2 * DT * 256;
    float* oA = oU + 2 * VT * 256;
    float* oP = oA + 3 * 256;
    int* odd = (int*)(oP + DP);
    if (tid == 0) *odd = 0;                                  // (waves that find one set it behind barriers)

    const double neg_a = rule == 1 ? -(double)rate : -exp((double)A_log[h]);
    const float neg_a32 = (float)neg_a;
    const float a_sign = rule == 1 ? -1.f : 1.f;
    const double q_scale = rule == 2 ? 1.0 : rsqrt((double)D);

    // ---- rows: 8 threads each, EP neighbouring elements a thread
    const int row = tid >> 3, e0 = (tid & 7) * EP;
    const bool live = row < nt;
    const T* qrow = qkv + (size_t)(base + c0 + (live ? row : 0)) * ld_qkv;
    const T* arow = ag + (size_t)(base + c0 + (live ? row : 0)) * ld_ag;
    float fq[EP], fk[EP], fa[EP], fv[VW / 8];
    // (`per` elements of a row from `from` on, as many as lie before `end`; whole 16-byte pieces where the rows allow it)
    auto take = [&](float* to, const T* src, int from, int end, int per) {
        if (vec) {
            constexpr int PER = 16 / sizeof(T);
#pragma unroll
            for (int e = 0; e < per; e += PER) {
                uint4 x = make_uint4(0, 0, 0, 0);
                if (live && from + e < end) x = *reinterpret_cast<const uint4*>(src + e);
                const T* p = reinterpret_cast<const T*>(&x);
#pragma unroll
                for (int i = 0; i < PER; ++i) to[e + i] = to_f(p[i]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < per; ++e) to[e] = live && from + e < end ? to_f(src[e]) : 0.f;
        }
    };
    take(fq, qrow + kvh * D + e0, e0, D, EP);
    take(fk, qrow + (size_t)G * D + kvh * D + e0, e0, D, EP);
    if (rule < 2) take(fa, arow + (size_t)h * D + e0, e0, D, EP);
    const T* vrow = qrow + (size_t)2 * G * D + (size_t)h * V;
    const int v0 = (tid & 7) * (VW / 8);
    take(fv, vrow + v0, v0, V, VW / 8);
    double sp = 0.0;                                         // rules 2 and 3: the row's step
    if (rule >= 2 && live) sp = rc_softplus((double)to_f(arow[h]) + dt_bias[h]);
    float bet = 0.f;
    if (live)
        bet = rule == 1 ? 1.f : rule == 2 ? (float)sp : (float)(1.0 / (1.0 + exp(-(double)to_f(b[(size_t)(base + c0 + row) * ld_b + h]))));
    if ((tid & 7) == 0) beta_s[row] = bet;
    if (tid < 2) slow[tid] = 0;
    double nk = 1.0, nq = q_scale;
    if (delta) {
        double sk = 0.0, sq = 0.0;
#pragma unroll
        for (int e = 0; e < EP; ++e) {
            sk = fma((double)fk[e], (double)fk[e], sk);
            sq = fma((double)fq[e], (double)fq[e], sq);
        }
        nk = rsqrt((double)rc_sum8((float)sk) + 1e-6);
        nq = q_scale * rsqrt((double)rc_sum8((float)sq) + 1e-6);
    }
    if ((tid & 7) == 0) {
        nq_s[row] = rc_pair(nq);
        nk_s[row] = rc_pair(nk);
    }
    const float one = -0.f;                                  // (rc_decay's word for it)
    const float row_decay = rule >= 2 && live ? rc_decay(neg_a * sp) : one;
#pragma unroll
    for (int e = 0; e < EP; ++e) {
        const bool in = live && e0 + e < D;
        if (rule < 2) {
            const float x = in ? a_sign * (fa[e] + dt_bias[h * D + e0 + e]) : 0.f;
            const float word = rc_decay(neg_a32 * (x > 20.f ? x : rc_log1p(rc_exp(x > 20.f ? 20.f : x))));
            fa[e] = in ? word : one;
        } else {
            fa[e] = in ? row_decay : one;
        }
        qs[row * LD + e0 + e] = fq[e];
        ks[row * LD + e0 + e] = fk[e];
        as[row * LD + e0 + e] = fa[e];
    }
    __syncthreads();

    // ---- products along the rows: a thread per (half, channel)
    const int hf = tid / DP, d = tid - hf * DP;
    const bool chan = hf < 2;
    float ak[16], aq[16], aa[16];
    RcPair pp[16];
    if (chan) {
        RcPair p = {1.f, 0.f};
        float top = 0.f;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int at = (hf * 16 + i) * LD + d;
            aq[i] = qs[at];
            ak[i] = ks[at];
            aa[i] = as[at];
            top = fmaxf(top, fabsf(ak[i]));
            p = rc_times(p, rc_decay_pair(aa[i]));
            pp[i] = p;
        }
        pt[hf * DP + d] = p.hi;
        if (!(p.hi >= RC_TINY) || !(top <= RC_LARGE)) slow[hf] = 1;
    }
    __syncthreads();
    // (a half whose decays go below RC_TINY or whose keys go beyond RC_LARGE: pairs one by one, 16 lanes to a column j, their channels' products carried
    // from row to row)
    const int slow0 = slow[0], slow1 = slow[1];
    if (slow0 | slow1) {
        const int j = tid >> 4, sl = tid & 15;
        for (int x = 0; x < 2; ++x) {
            if (!(x ? slow1 : slow0)) continue;
            float p[DT], kj[DT];
#pragma unroll
            for (int e = 0; e < DT; ++e) {
                p[e] = 1.f;
                kj[e] = rc_scaled(ks[(x * 16 + j) * LD + sl + 16 * e], nk_s[x * 16 + j]);
            }
            for (int i = 0; i < 16; ++i) {
                const RcPair fq_i = nq_s[x * 16 + i], fk_i = nk_s[x * 16 + i];
                float da = 0.f, dl = 0.f;
#pragma unroll
                for (int e = 0; e < DT; ++e) {
                    const int at = (x * 16 + i) * LD + sl + 16 * e;
                    if (i > j) p[e] *= rc_decay_pair(as[at]).hi;
                    const float kp = kj[e] * p[e];
                    da = fmaf(rc_scaled(qs[at], fq_i), kp, da);
                    dl = fmaf(rc_scaled(ks[at], fk_i), kp, dl);
                }
                da = rc_sum16(da);
                dl = rc_sum16(dl);
                if (sl == 0) {
                    SA[(x * 16 + i) * 16 + j] = da;
                    SL[(x * 16 + i) * 16 + j] = dl;
                }
            }
        }
        __syncthreads();
    }
    if (chan) {
        // k times the decays behind it in the half; times the second half's product it is k P_C / P
        const float other = hf == 0 ? pt[DP + d] : 1.f;
        RcPair p = {1.f, 0.f};
        float kend[16];
#pragma unroll
        for (int i = 15; i >= 0; --i) {
            kend[i] = rc_scaled(ak[i], rc_times(p, nk_s[hf * 16 + i]));
            p = rc_times(p, rc_decay_pair(aa[i]));
        }
        if (hf == 0) {
#pragma unroll
            for (int i = 0; i < 16; ++i) kt[i * LD + d] = kend[i];
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const rc_f4 x = {kend[4 * g] * other, kend[4 * g + 1] * other, kend[4 * g + 2] * other, kend[4 * g + 3] * other};
            *reinterpret_cast<rc_f4*>(oK + (((d >> 4) * 2 + hf) * 64 + g * 16 + (d & 15)) * 4) = x;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int at = (hf * 16 + i) * LD + d;
            const RcPair fk_i = nk_s[hf * 16 + i];
            qs[at] = rc_scaled(aq[i], rc_times(pp[i], nq_s[hf * 16 + i]));
            ks[at] = rc_scaled(ak[i], rc_times(pp[i], fk_i));
            as[at] = rc_scaled(ak[i], rc_times(rc_one_over(pp[i]), fk_i));
        }
    }
    __syncthreads();

    // ---- A and L: wave 0 and 1 the halves' own tiles, wave 2 the tile between them, wave 3 q P and P_C
    const int m16 = lane & 15, g4 = (lane >> 4) * 4;
    if (wave < 3) {
        const int bi = wave == 0 ? 0 : 1, bj = wave == 1 ? 1 : 0;
        const float* col = wave < 2 ? as + (bj * 16 + m16) * LD : kt + m16 * LD;
        const float* rq = qs + (bi * 16 + m16) * LD;
        const float* rk = ks + (bi * 16 + m16) * LD;
        // (sixteen sums each: short chains of roundings)
        RcSums pa[4] = {rc_zero(), rc_zero(), rc_zero(), rc_zero()}, pl[4] = {rc_zero(), rc_zero(), rc_zero(), rc_zero()};
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const rc_f4 x = *reinterpret_cast<const rc_f4*>(col + 16 * t + g4);
            const rc_f4 y = *reinterpret_cast<const rc_f4*>(rq + 16 * t + g4);
            pa[t & 3] = rc_mul4(x, y, pa[t & 3]);
            if (delta) pl[t & 3] = rc_mul4(x, *reinterpret_cast<const rc_f4*>(rk + 16 * t + g4), pl[t & 3]);
        }
        MFMA_SETTLE();
        rc_f4 ta = (rc_sum4(pa[0]) + rc_sum4(pa[1])) + (rc_sum4(pa[2]) + rc_sum4(pa[3]));
        rc_f4 tl = (rc_sum4(pl[0]) + rc_sum4(pl[1])) + (rc_sum4(pl[2]) + rc_sum4(pl[3]));
        // (lane m16 + 16 g: row i = m16, columns j = 4 g .. 4 g + 3)
        if (wave < 2) {
            if (wave ? slow1 : slow0) {
                ta = *reinterpret_cast<const rc_f4*>(SA + (wave * 16 + m16) * 16 + g4);
                tl = *reinterpret_cast<const rc_f4*>(SL + (wave * 16 + m16) * 16 + g4);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                if (g4 + r > m16) ta[r] = 0.f;
                if (g4 + r >= m16) tl[r] = 0.f;
            }
        }
        *reinterpret_cast<rc_f4*>(oA + ((wave == 0 ? 0 : wave == 1 ? 2 : 1) * 64 + lane) * 4) = ta;
        if (delta) {
            const float be = beta_s[bi * 16 + m16];
            const rc_f4 x = {tl[0] * be, tl[1] * be, tl[2] * be, tl[3] * be};
            *reinterpret_cast<rc_f4*>(Ls + (bi * 16 + m16) * 36 + bj * 16 + g4) = x;
        }
    } else {
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            const rc_f4 p0 = *reinterpret_cast<const rc_f4*>(pt + 16 * t + g4);
            *reinterpret_cast<rc_f4*>(oQ + (t * 64 + lane) * 4) = *reinterpret_cast<const rc_f4*>(qs + m16 * LD + 16 * t + g4);
            *reinterpret_cast<rc_f4*>(oQ + ((DT + t) * 64 + lane) * 4) =
                *reinterpret_cast<const rc_f4*>(qs + (16 + m16) * LD + 16 * t + g4) * p0;
        }
        for (int i = lane; i < DP; i += 64) oP[i] = pt[i] * pt[DP + i];
    }

    __syncthreads();
#pragma unroll
    for (int e = 0; e < VW / 8; ++e) vs[row * LV + v0 + e] = fv[e] * bet;
    if (delta) {
        // ---- T: the two diagonal tiles by substitution, a lane per column, then the tile between them
        if (tid < 32) {
            const int x = tid >> 4, cc = tid & 15;
            float t[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float v = i == cc ? 1.f : 0.f;
#pragma unroll
                for (int j = 0; j < i; ++j) v = fmaf(-Ls[(x * 16 + i) * 36 + x * 16 + j], t[j], v);
                t[i] = v;
                Ts[(x * 16 + i) * 36 + x * 16 + cc] = v;
            }
        }
        __syncthreads();
        const int ti = tid >> 4, tc = tid & 15;
        float v = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j) v = fmaf(Ls[(16 + ti) * 36 + j], Ts[j * 36 + tc], v);
        Ms[ti * 20 + tc] = v;
        __syncthreads();
        v = 0.f;
#pragma unroll
        for (int j = 0; j < 16; ++j)
            if (j <= ti) v = fmaf(-Ts[(16 + ti) * 36 + 16 + j], Ms[j * 20 + tc], v);
        Ts[(16 + ti) * 36 + tc] = v;
        __syncthreads();
        // ---- W^T = (beta k P)^T T^T: rows d, columns i
        const rc_f4 t00 = *reinterpret_cast<const rc_f4*>(Ts + m16 * 36 + g4);
        const rc_f4 t10 = *reinterpret_cast<const rc_f4*>(Ts + (16 + m16) * 36 + g4);
        const rc_f4 t11 = *reinterpret_cast<const rc_f4*>(Ts + (16 + m16) * 36 + 16 + g4);
#pragma unroll
        for (int tt = 0; tt < DT / 4; ++tt) {
            const int t = wave * (DT / 4) + tt;
            const float p0 = pt[16 * t + m16];
            rc_f4 x0, x1;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x0[r] = ks[(g4 + r) * LD + 16 * t + m16] * beta_s[g4 + r];
                x1[r] = ks[(16 + g4 + r) * LD + 16 * t + m16] * p0 * beta_s[16 + g4 + r];
            }
            const RcSums s0 = rc_mul4(x0, t00, rc_zero()), s10 = rc_mul4(x0, t10, rc_zero()), s1 = rc_mul4(x1, t11, s10);
            MFMA_SETTLE();
            rc_f4 w0 = rc_sum4(s0), w1 = rc_sum4(s1);
            if (rc_odd(w0) || rc_odd(w1)) {
                if (lane == 0) *odd = 1;
                w0 = rc_lower<false>(x0, t00, rc_f4{0.f, 0.f, 0.f, 0.f});
                w1 = rc_lower<false>(x1, t11, rc_sum4(s10));
            }
            *reinterpret_cast<rc_f4*>(oW + (t * 64 + lane) * 4) = w0;
            *reinterpret_cast<rc_f4*>(oW + ((DT + t) * 64 + lane) * 4) = w1;
        }
        // ---- U = T beta v, 128 columns of v at a time
        for (int vb = 0; vb < V; vb += VW) {
            if (vb) {
                __syncthreads();
                take(fv, vrow + vb + v0, vb + v0, V, VW / 8);
#pragma unroll
                for (int e = 0; e < VW / 8; ++e) vs[row * LV + v0 + e] = fv[e] * bet;
                __syncthreads();
            }
            const int tiles = min(VW, V - vb + 15) / 16;
            for (int n = wave; n < tiles; n += 4) {
                rc_f4 x0, x1;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    x0[r] = vs[(g4 + r) * LV + 16 * n + m16];
                    x1[r] = vs[(16 + g4 + r) * LV + 16 * n + m16];
                }
                const RcSums s0 = rc_mul4(t00, x0, rc_zero()), s10 = rc_mul4(t10, x0, rc_zero()), s1 = rc_mul4(t11, x1, s10);
                MFMA_SETTLE();
                rc_f4 u0 = rc_sum4(s0), u1 = rc_sum4(s1);
                if (rc_odd(u0) || rc_odd(u1)) {
                    if (lane == 0) *odd = 1;
                    u0 = rc_lower<true>(t00, x0, rc_f4{0.f, 0.f, 0.f, 0.f});
                    u1 = rc_lower<true>(t11, x1, rc_sum4(s10));
                }
                float* to = oU + (long long)(vb / 16 + n) * 512 + lane * 4;
                *reinterpret_cast<rc_f4*>(to) = u0;
                *reinterpret_cast<rc_f4*>(to + 256) = u1;
            }
        }
        return;
    }
    // ---- no correction: U is the values (times delta) themselves
    __syncthreads();
    for (int vb = 0; vb < V; vb += VW) {
        if (vb) {
            __syncthreads();
            take(fv, vrow + vb + v0, vb + v0, V, VW / 8);
#pragma unroll
            for (int e = 0; e < VW / 8; ++e) vs[row * LV + v0 + e] = fv[e] * bet;
            __syncthreads();
        }
        const int tiles = min(VW, V - vb + 15) / 16;
        for (int n = wave; n < tiles; n += 4) {
            rc_f4 x0, x1;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                x0[r] = vs[(g4 + r) * LV + 16 * n + m16];
                x1[r] = vs[(16 + g4 + r) * LV + 16 * n + m16];
            }
            if ((rc_odd(x0) || rc_odd(x1)) && lane == 0) *odd = 1;
            float* to = oU + (long long)(vb / 16 + n) * 512 + lane * 4;
            *reinterpret_cast<rc_f4*>(to) = x0;
            *reinterpret_cast<rc_f4*>(to + 256) = x1;
        }
    }
}

static size_t rc_prepare_lds(int DT) {
    const int LD = 16 * DT + 4;
    return sizeof(float) * ((size_t)(3 * RC_C + 16) * LD + (DT == 8 ? 0 : RC_C * 132) + 2 * RC_C * 36 + 16 * 20 + 1024 + 32 * DT + 5 * RC_C + 4);
}

// ---------------------------------------------------------------------------------------------------- carry
// What a wave needs of one chunk: its channels' parts of W, q P, k P_C / P and P_C, its tile of A, the workgroup's U.
template <int DPW, int NV, bool DELTA>
struct RcChunk {
    rc_f4 w[DELTA ? 2 : 1][DPW], q[2][DPW], k[DPW][2], p[DPW], u[NV][2], a[2];
};

// A wave holds 16 DPW rows of the workgroup's columns of S and takes part in every product with the state over its own
// rows; the four waves' shares of W S and q P S meet in LDS (two buffers, one barrier a chunk).
template <int DT, int NV, bool DELTA>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(DELTA ? 1 : 2, 2))) void recur_carry_kernel(
    const float* __restrict__ ws, float* __restrict__ S, const int* __restrict__ cu_q, const int* __restrict__ slot_ids,
    float* __restrict__ o_raw, int n_seqs, int H, int D, int V, int first, int run, int splits, int rule) {
    constexpr int DPW = DT / 4, PARTS = DELTA ? 4 : 2;
    __shared__ __attribute__((aligned(16))) float part[2][4][PARTS][NV][256];
    // the splits of one head lie eight workgroups apart, on one XCD, whose L2 then holds what they share
    const int unit = (blockIdx.x / (8 * splits)) * 8 + (blockIdx.x & 7), split = (blockIdx.x >> 3) % splits;
    const int s = unit / H, h = unit - s * H;
    if (s >= n_seqs) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, m16 = lane & 15, g4 = (lane >> 4) * 4;
    const int n_chunks = rc_chunks(cu_q, s, n_seqs, first, run, rc_min_rows(rule));
    if (n_chunks <= 0) return;
    int before = 0;
    for (int r = lane; r < s; r += 64) before += rc_chunks(cu_q, r, n_seqs, first, run, rc_min_rows(rule));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o, 64);
    const int base = cu_q[s], q_len = cu_q[s + 1] - base;
    const int VT = (V + 15) / 16;
    const long long stride = rc_stride(DT, VT, DELTA) * H;
    const float* at = ws + ((long long)before * H + h) * rc_stride(DT, VT, DELTA);
    const int oi = wave & 1, on = wave >> 1;                 // the tile of the read-out that this wave finishes

    // ---- the state: column n of a tile with lane n, rows 4 g .. 4 g + 3
    float* Sh = S + ((size_t)slot_ids[s] * H + h) * V * D;
    const bool svec = (D & 3) == 0;
    rc_f4 st[NV][DPW];
#pragma unroll
    for (int nv = 0; nv < NV; ++nv)
#pragma unroll
        for (int t = 0; t < DPW; ++t) {
            const int v = (split * NV + nv) * 16 + m16, d = (wave * DPW + t) * 16 + g4;
            st[nv][t] = rc_f4{0.f, 0.f, 0.f, 0.f};
            if (v < V) {
                const float* p = Sh + (size_t)v * D + d;
                if (svec) {
                    if (d < D) st[nv][t] = *reinterpret_cast<const rc_f4*>(p);
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (d + r < D) st[nv][t][r] = p[r];
                }
            }
        }

    typedef RcChunk<DPW, NV, DELTA> Chunk;
    auto load = [&](Chunk& x, const float* c) {
        const float* w = c;
        const float* q = w + (DELTA ? 2 * DT * 256 : 0);
        const float* k = q + 2 * DT * 256;
        const float* u = k + 2 * DT * 256;
        const float* a = u + 2 * VT * 256;
        const float* p = a + 3 * 256;
#pragma unroll
        for (int t = 0; t < DPW; ++t) {
            const int dt = wave * DPW + t;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if constexpr (DELTA) x.w[i][t] = *reinterpret_cast<const rc_f4*>(w + ((i * DT + dt) * 64 + lane) * 4);
                x.q[i][t] = *reinterpret_cast<const rc_f4*>(q + ((i * DT + dt) * 64 + lane) * 4);
                x.k[t][i] = *reinterpret_cast<const rc_f4*>(k + ((dt * 2 + i) * 64 + lane) * 4);
            }
            x.p[t] = *reinterpret_cast<const rc_f4*>(p + dt * 16 + g4);
        }
#pragma unroll
        for (int nv = 0; nv < NV; ++nv)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int n = min(split * NV + nv, VT - 1);
                x.u[nv][i] = *reinterpret_cast<const rc_f4*>(u + (long long)n * 512 + i * 256 + lane * 4);
            }
        // (rows of the first half read the first half only; the third tile is the second half's own)
        x.a[0] = *reinterpret_cast<const rc_f4*>(a + (oi * 64 + lane) * 4);
        x.a[1] = *reinterpret_cast<const rc_f4*>(a + (2 * 64 + lane) * 4);
    };

    auto go = [&](const Chunk& x, int ci, int buf, auto odd_c) {
        // (two sums each, as of S below: half the chain of roundings. W S first: the next chunk's state waits for it, q P S
        // only for the read-out. The reads of these results sit in the same basic block, where the compiler keeps the
        // distance by itself.)
        auto with_state = [&](const rc_f4 (&m)[2][DPW], int what, int nv) {
            rc_f4 s[2][2];
#pragma unroll
            for (int i = 0; i < 2; ++i) s[0][i] = s[1][i] = rc_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int t = 0; t < DPW; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
#pragma unroll
                    for (int i = 0; i < 2; ++i) s[r & 1][i] = rc_mfma(m[i][t][r], st[nv][t][r], s[r & 1][i]);
#pragma unroll
            for (int i = 0; i < 2; ++i) *reinterpret_cast<rc_f4*>(&part[buf][wave][what + i][nv][lane * 4]) = s[0][i] + s[1][i];
        };
        if constexpr (DELTA) {
#pragma unroll
            for (int nv = 0; nv < NV; ++nv) with_state(x.w, 2, nv);
        }
#pragma unroll
        for (int nv = 0; nv < NV; ++nv) with_state(x.q, 0, nv);
        __syncthreads();
        auto sum_waves = [&](int what, int nv) {
            rc_f4 w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const rc_f4*>(&part[buf][i][what][nv][lane * 4]);
            return (w[0] + w[1]) + (w[2] + w[3]);
        };
        rc_f4 u[NV][2];
#pragma unroll
        for (int nv = 0; nv < NV; ++nv)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                u[nv][i] = x.u[nv][i];
                if constexpr (DELTA) {
                    u[nv][i] -= sum_waves(2 + i, nv);
                }
            }
        auto move_on = [&]() {
#pragma unroll
            for (int nv = 0; nv < NV; ++nv) {
                rc_f4 ku[2][DPW];
#pragma unroll
                for (int t = 0; t < DPW; ++t) ku[0][t] = ku[1][t] = rc_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int t = 0; t < DPW; ++t) ku[r & 1][t] = rc_mfma(x.k[t][i][r], u[nv][i][r], ku[r & 1][t]);
#pragma unroll
                for (int t = 0; t < DPW; ++t) {
                    const rc_f4 add = ku[0][t] + ku[1][t];
#pragma unroll
                    for (int r = 0; r < 4; ++r) st[nv][t][r] = fmaf(st[nv][t][r], x.p[t][r], add[r]);
                }
            }
        };
        // (the delta rules' next chunk waits for S; without a correction nothing does, and the read-out first takes fewer registers)
        if constexpr (DELTA) move_on();
        if (on < NV) {
            rc_f4 o = sum_waves(oi, on);
            rc_f4 u0 = on ? u[NV - 1][0] : u[0][0], u1 = on ? u[NV - 1][1] : u[0][1];
            if constexpr (decltype(odd_c)::value) {          // (what meets A's diagonal tile)
                if (oi) o += rc_spoilt(u1);
                else o += rc_spoilt(u0);
            }
            constexpr int SUMS = DELTA || NV == 1 || DT < 8 ? 4 : 2;      // (what the registers of two workgroups a CU hold)
            rc_f4 au[SUMS];
#pragma unroll
            for (int r = 0; r < SUMS; ++r) au[r] = rc_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 4; ++r) au[r % SUMS] = rc_mfma(x.a[0][r], u0[r], au[r % SUMS]);
            if (oi) {
#pragma unroll
                for (int r = 0; r < 4; ++r) au[r % SUMS] = rc_mfma(x.a[1][r], u1[r], au[r % SUMS]);
            }
            MFMA_SETTLE();
            if constexpr (SUMS == 4) o += (au[0] + au[1]) + (au[2] + au[3]);
            else o += au[0] + au[1];
            const int v = (split * NV + on) * 16 + m16, c0 = (first + ci) * RC_C + oi * 16 + g4;
            if (v < V) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (c0 + r < q_len) o_raw[(size_t)(base + c0 + r) * H * V + (size_t)h * V + v] = o[r];
            }
        }
        if constexpr (!DELTA) {
            __builtin_amdgcn_sched_barrier(0);
            move_on();
        }
    };

    // (a chunk's operands are asked for while the one before it is worked on; the last chunk has code of its own, because
    // behind a branch around the loads the compiler waits for those of the next chunk too)
    constexpr std::integral_constant<bool, false> plain{};
    constexpr std::integral_constant<bool, true> odd{};
    int any_odd = 0;
    for (int c = lane; c < n_chunks; c += 64)
        any_odd |= reinterpret_cast<const int*>(at + (long long)c * stride)[rc_stride(DT, VT, DELTA) - 4];
    if (__ballot(any_odd != 0)) {                            // (the same in every wave)
        Chunk z;
        for (int c = 0; c < n_chunks; ++c) {
            load(z, at + (long long)c * stride);
            go(z, c, c & 1, odd);
        }
    } else {
        Chunk x, y;
        load(x, at);
        for (int c = 0;; c += 2) {
            if (c + 1 >= n_chunks) {
                go(x, c, 0, plain);
                break;
            }
            load(y, at + (long long)(c + 1) * stride);
            __builtin_amdgcn_sched_barrier(0);
            go(x, c, 0, plain);
            if (c + 2 >= n_chunks) {
                go(y, c + 1, 1, plain);
                break;
            }
            load(x, at + (long long)(c + 2) * stride);
            __builtin_amdgcn_sched_barrier(0);
            go(y, c + 1, 1, plain);
        }
    }
#pragma unroll
    for (int nv = 0; nv < NV; ++nv)
#pragma unroll
        for (int t = 0; t < DPW; ++t) {
            const int v = (split * NV + nv) * 16 + m16, d = (wave * DPW + t) * 16 + g4;
            if (v >= V) continue;
            float* p = Sh + (size_t)v * D + d;
            if (svec) {
                if (d < D) *reinterpret_cast<rc_f4*>(p) = st[nv][t];
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (d + r < D) p[r] = st[nv][t][r];
            }
        }
}

// ---------------------------------------------------------------------------------------------------- host
static int rc_tiles(int D) { return D <= 64 ? 4 : 8; }

// Requests that one launch takes at most: as many as have room for a chunk each in RC_SCRATCH (one that has not goes alone).
static int rc_group(int H, long long stride) {
    const long long fit = RC_SCRATCH / (stride * H);
    return fit < 1 ? 1 : fit > RC_GROUP ? RC_GROUP : (int)fit;
}

// Chunks of every request that a run takes at once, so that the scratch of a group of requests is at most RC_SCRATCH.
static int rc_run(const int* q_lens, int n, int H, long long stride, int min_rows, int* longest, long long* most) {
    int count = 0, top = 0;
    for (int i = 0; i < n; ++i)
        if (q_lens[i] >= min_rows) {
            ++count;
            top = top > (q_lens[i] + RC_C - 1) / RC_C ? top : (q_lens[i] + RC_C - 1) / RC_C;
        }
    *longest = top;
    *most = 0;
    if (!count) return 0;
    long long run = RC_SCRATCH / (stride * H * count);
    if (run < 1) run = 1;
    if (run > top) run = top;
    for (int i = 0; i < n; ++i)
        if (q_lens[i] >= min_rows) {
            const long long c = (q_lens[i] + RC_C - 1) / RC_C;
            *most += c < run ? c : run;
        }
    return (int)run;
}

long long recurrence_chunks_workspace(const int* q_lens, int n_seqs, int H, int D, int V, int rule) {
    if (q_lens == nullptr || n_seqs < 1 || H < 1 || D < 1 || D > 128 || V < 1 || V > 4096) return 0;
    const long long stride = rc_stride(rc_tiles(D), (V + 15) / 16, rule == 0 || rule == 3);
    const int group = rc_group(H, stride);
    long long need = 0;
    for (int r0 = 0; r0 < n_seqs; r0 += group) {
        int longest;
        long long most;
        rc_run(q_lens + r0, n_seqs - r0 < group ? n_seqs - r0 : group, H, stride, rc_min_rows(rule), &longest, &most);
        if (most * H * stride > need) need = most * H * stride;
    }
    return need;
}

template <typename T, int DT>
static int rc_launch(hipStream_t st, const T* qkv, long long ld_qkv, const T* b, long long ld_b, const T* ag, long long ld_ag,
                     const float* A_log, const float* dt_bias, float* S, const int* cu_q, const int* slot_ids, float* o_raw,
                     const int* q_lens, int n_seqs, int H, int G, int D, int V, int rule, float rate, float* ws) {
    const bool delta = rule == 0 || rule == 3;
    const int VT = (V + 15) / 16;
    const long long stride = rc_stride(DT, VT, delta);
    const size_t lds = rc_prepare_lds(DT);
    static std::atomic<unsigned long long> allowed{0};          // (devices on which the kernel may have so much LDS)
    int dev = 0;
    if (lds > 64 * 1024 && (hipGetDevice(&dev) != hipSuccess || dev > 63 || !(allowed.load() >> dev & 1))) {
        if (hipFuncSetAttribute((const void*)recur_prepare_kernel<T, DT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
            return RA_ERR_LAUNCH;
        if (dev <= 63) allowed |= 1ull << dev;
    }
    // 16-byte loads: a row's pieces and a head's begin at whole pieces
    const size_t per = 16 / sizeof(T);
    const bool vec = D % per == 0 && V % per == 0 && ld_qkv % per == 0 && ((size_t)qkv & 15) == 0 &&
                     (rule >= 2 || (ld_ag % per == 0 && ((size_t)ag & 15) == 0));
    const int group = rc_group(H, stride);
    for (int r0 = 0; r0 < n_seqs; r0 += group) {
        const int n = n_seqs - r0 < group ? n_seqs - r0 : group;
        int longest;
        long long most;
        const int run = rc_run(q_lens + r0, n, H, stride, rc_min_rows(rule), &longest, &most);
        for (int first = 0; first < longest; first += run) {
            long long chunks = 0;
            for (int i = 0; i < n; ++i) {
                const int len = q_lens[r0 + i];
                const long long c = len < rc_min_rows(rule) ? 0 : (len + RC_C - 1) / RC_C - first;
                chunks += c < 0 ? 0 : c < run ? c : run;
            }
            if (chunks > 65535) return RA_ERR_ARG;
            hipLaunchKernelGGL((recur_prepare_kernel<T, DT>), dim3(H, (unsigned)chunks), dim3(256), lds, st, qkv, ld_qkv, b, ld_b,
                               ag, ld_ag, A_log, dt_bias, cu_q + r0, ws, n, H, G, D, V, first, run, rule, rate, vec ? 1 : 0);
            // 32 columns a workgroup (what the chunks bring is read half as often) where that still fills the chip twice
            const bool wide = V > 16 && (long long)n * H * ((VT + 1) / 2) >= 512;
            const int splits = wide ? (VT + 1) / 2 : VT;
            const long long units = ((long long)n * H + 7) / 8 * 8;
            const dim3 grid((unsigned)(units * splits));
#define RC_CARRY(NV_, DE_)                                                                                                    \
    hipLaunchKernelGGL((recur_carry_kernel<DT, NV_, DE_>), grid, dim3(256), 0, st, ws, S, cu_q + r0, slot_ids + r0, o_raw, n, \
                       H, D, V, first, run, splits, rule)
            if (wide && delta) RC_CARRY(2, true);
            else if (wide) RC_CARRY(2, false);
            else if (delta) RC_CARRY(1, true);
            else RC_CARRY(1, false);
#undef RC_CARRY
        }
    }
    return ra_launch_status();
}

int recurrence_chunks_run(hipStream_t st, const void* qkv, long long ld_qkv, const void* b, long long ld_b, const void* ag,
                          long long ld_ag, const float* A_log, const float* dt_bias, float* S, const int* cu_q,
                          const int* slot_ids, float* o_raw, const int* q_lens, int n_seqs, int H, int G, int D, int V,
                          int rule, float rate, float* ws, long long ws_floats, int dtype) {
    const long long need = recurrence_chunks_workspace(q_lens, n_seqs, H, D, V, rule);
    if (need <= 0 || ws == nullptr || ws_floats < need) return RA_ERR_ARG;
#define RC_GO(T_, DT_)                                                                                                    \
    rc_launch<T_, DT_>(st, (const T_*)qkv, ld_qkv, (const T_*)b, ld_b, (const T_*)ag, ld_ag, A_log, dt_bias, S, cu_q, slot_ids, \
                       o_raw, q_lens, n_seqs, H, G, D, V, rule, rate, ws)
    if (dtype != RA_DTYPE_BF16) return RA_ERR_ARG;
    return rc_tiles(D) == 4 ? RC_GO(bf16, 4) : RC_GO(bf16, 8);
#undef RC_GO
}
