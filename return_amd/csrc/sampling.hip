// Token choice from fp32 logits: greedy, temperature, top-k, top-p; and the chosen token's
// log-probability under the raw logits. One block per row; several for few rows of a large vocabulary (sample_parts).
//
// What the reference samples with (rollout/model.py:15-61): temperature <= 0 is argmax;
// otherwise logits / temperature; keep the top_k largest; over the kept values in descending
// order drop every token before which more than top_p of the (top-k renormalised) mass
// already lies (the crossing token stays, the first always stays); draw from what is left.
// Logprob is log_softmax(raw logits)[token] (rollout/model.py:64-67).
//
// The draw uses a uniform number u in [0,1) that the host supplies per row: the token is the
// first, in vocabulary order, at which the running sum of kept probabilities exceeds u.
// Among tokens that tie at a boundary the earlier ones in the vocabulary stay, as a stable sort
// puts them first: exactly top_k tokens are kept (rollout/model.py:45-50 keeps topk(k)), and of the
// tokens that tie with the top-p boundary value those before which at most top_p of the mass lies.
//
// top-k and top-p need a threshold among the largest logits. The row's tokens within CAND_SPAN of
// the largest logit (in units of the temperature: every other token weighs less than e^-16 of the
// largest) are first collected into a list in LDS, in vocabulary order; if they fit, and if the
// thresholds lie among them (k is at most their number; their mass is more than top_p of the whole),
// the thresholds are searched and the token is drawn from the list alone, which takes microseconds.
// Otherwise (a flat row, a large k, top_p near 1) the searches go over the whole row, in two passes as a rule.
// Which way a row goes and which token it draws depends on that row alone, and not on the rows beside it: what decides either
// is a sum of whole numbers, or a sum in an order of its own. (The log-probability's sum of exponentials is formed in the order
// of the kernels that serve so many rows: its last bits depend on their number.)
// One block a row is bound by its chain of barriers and short sums (a peaked row of 16,384: 21 us, 6 of them for the
// maximum) and, flat, by one CU's arithmetic (32,000: 41 us; before the searches of two passes 54, and peaked 32).
#include "common.h"

#define SAMPLE_THREADS 1024
#define CAND_WAVES (SAMPLE_THREADS / 64)
#define CAND_PER_WAVE 512                                        // list entries of one wave's run of the row
#define CAND_OWN (CAND_WAVES * CAND_PER_WAVE / SAMPLE_THREADS)   // entries a thread looks after in a search: 8
#define CAND_SPAN 16.0f
#define WEIGHS_NOTHING 28.5f      // (max - x) / T from which to_fixed(exp(-that)) is 0: 2^-41 is exp(-28.42)
#define TOP_K_SPAN 32.0f          // logits: top-k beyond the list is searched closely so far from the largest
#define SAMPLE_BLOCKS 64                                         // blocks of 256 tokens in a wave's run whose masses are kept

__device__ __forceinline__ uint32_t order_key(float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);      // ascending float order -> ascending uint
}

__device__ __forceinline__ float key_value(uint32_t k) {      // the float whose order_key is k
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// f(i, v) for every element of the row, four at a time where the row allows 16-byte loads
template <typename F>
__device__ __forceinline__ void for_each_logit(const float* __restrict__ x, int V, int tid, F f) {
    if ((V & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0) {
        const float4* x4 = reinterpret_cast<const float4*>(x);
        const int n4 = V >> 2;
        int i = tid;
        for (; i + 7 * SAMPLE_THREADS < n4; i += 8 * SAMPLE_THREADS) {   // eight loads on their way per thread
            float4 a[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) a[j] = x4[i + j * SAMPLE_THREADS];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = 4 * (i + j * SAMPLE_THREADS);
                f(k, a[j].x); f(k + 1, a[j].y); f(k + 2, a[j].z); f(k + 3, a[j].w);
            }
        }
        for (; i < n4; i += SAMPLE_THREADS) {
            const float4 a = x4[i];
            f(4 * i, a.x); f(4 * i + 1, a.y); f(4 * i + 2, a.z); f(4 * i + 3, a.w);
        }
    } else {
        for (int i = tid; i < V; i += SAMPLE_THREADS) f(i, x[i]);
    }
}

// Measures are whole numbers: a token counts 2^40 (top-k), or weighs exp((x - gmax) / T) as a multiple of
// 2^-40 (top-p; what weighs less than 2^-41 of the largest token weighs nothing). Sums of whole numbers do
// not depend on the order in which they are formed, so they may be formed by atomics, by any number of
// threads, and come out the same in every run of the program.
typedef unsigned long long fixed_t;
#define FIXED_ONE_F 1099511627776.0f               // 2^40
__device__ __forceinline__ fixed_t to_fixed(float w) {          // 0 <= w <= 1
    const float t = w * 256.0f;
    const float hi = floorf(t);
    return ((fixed_t)(uint32_t)hi << 32) + (fixed_t)(uint32_t)((t - hi) * 4294967296.0f);
}

// What weighs less than e^-CAND_SPAN of the largest token, as a multiple of 2^-50 (sixteen of them fit 32 bits; and a sum of
// such in the unit above).
__device__ __forceinline__ uint32_t to_fixed_rest(float w) { return (uint32_t)(w * 1125899906842624.0f); }
__device__ __forceinline__ fixed_t fixed_of_rest(fixed_t rest) { return rest >> 10; }

// Sum of whole numbers over the block; every thread gets it. wsum: CAND_WAVES words of LDS.
__device__ __forceinline__ fixed_t block_sum_fixed(fixed_t v, fixed_t* wsum) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
    __syncthreads();
    fixed_t t = 0ull;
    for (int w = 0; w < CAND_WAVES; ++w) t += wsum[w];
    __syncthreads();
    return t;
}

// The smallest key t in [lo, hi] with measure{key > t} <= limit, given measure{key > hi} = 0. visit(lo, hi, f)
// calls f(key, measure) for every token with lo < key <= hi that this thread looks after (all threads
// together: every such token once).
// A pass cuts (lo, hi] into up to SEARCH_BUCKETS runs of equal width, adds the tokens' measures into the
// runs (fx, LDS atomics) and finds the highest run b with more than `limit` at and above it: t lies in it.
// A range of 2^32 keys takes three passes. wsum: CAND_WAVES words, sh_b, sh_above: one word each, all LDS.
#define SEARCH_BITS 11
#define SEARCH_BUCKETS (1 << SEARCH_BITS)
// above (may be nullptr) is told measure{key > t}; at (may be nullptr) measure{key == t} where the last pass has
// it (its run of the key range was the one key t), else FIXED_UNKNOWN (t is the lo it was given, whose tokens no
// pass visits).
#define FIXED_UNKNOWN (~0ull)
template <typename Visit>
__device__ __noinline__ uint32_t search_threshold(Visit visit, int tid, uint32_t lo, uint32_t hi, fixed_t limit, fixed_t* fx,
                                     fixed_t* wsum, int* sh_b, fixed_t* sh_above, fixed_t* above = nullptr,
                                     fixed_t* at = nullptr) {
    fixed_t at_t = FIXED_UNKNOWN;
    static_assert(SEARCH_BUCKETS == 2 * SAMPLE_THREADS, "a thread looks after two runs");
    const int wave = tid >> 6, lane = tid & 63;
    fixed_t above_hi = 0ull;
    while (lo < hi) {
        const uint32_t width = hi - lo;
        const int bits = 32 - __builtin_clz(width);
        const int sh = bits > SEARCH_BITS ? bits - SEARCH_BITS : 0;       // (width >> sh) < SEARCH_BUCKETS
        fx[2 * tid] = 0ull;
        fx[2 * tid + 1] = 0ull;
        if (tid == 0) *sh_b = 0;
        __syncthreads();
        visit(lo, hi, [&](uint32_t key, fixed_t m) { atomicAdd(&fx[(key - lo) >> sh], m); });
        __syncthreads();
        // at_and_above(b) = the measure of runs b and higher; this thread has runs 2 tid and 2 tid + 1
        const fixed_t f0 = fx[2 * tid], f1 = fx[2 * tid + 1];
        fixed_t from_here = f0 + f1;                                      // then: over this and the higher threads
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const fixed_t t = __shfl_down(from_here, o, 64);
            if (lane + o < 64) from_here += t;
        }
        if (lane == 0) wsum[wave] = from_here;
        __syncthreads();
        for (int w = wave + 1; w < CAND_WAVES; ++w) from_here += wsum[w];
        const fixed_t s0 = from_here, s1 = from_here - f0;               // at_and_above(2 tid), (2 tid + 1)
        // the highest run with more than `limit` at and above it (run 0 if there is none)
        const int mine = above_hi + s1 > limit ? 2 * tid + 1 : (above_hi + s0 > limit ? 2 * tid : 0);
        if (mine > 0) atomicMax(sh_b, mine);
        __syncthreads();
        const int b = *sh_b;
        // what lies above run b: at_and_above(b + 1)
        if (b + 1 == 2 * tid) *sh_above = above_hi + s0;
        if (b + 1 == 2 * tid + 1) *sh_above = above_hi + s1;
        if (b + 1 == SEARCH_BUCKETS && tid == 0) *sh_above = above_hi;
        __syncthreads();
        above_hi = *sh_above;
        // run b ends at key lo + ((b + 1) << sh) - 1
        const unsigned long long end = (unsigned long long)lo + (((unsigned long long)b + 1ull) << sh) - 1ull;
        const uint32_t new_hi = end < (unsigned long long)hi ? (uint32_t)end : hi;
        lo = b == 0 ? lo : lo + ((uint32_t)b << sh);
        hi = new_hi;
        if (lo == hi && b > 0) at_t = fx[b];           // the run was that one key: what was added into it is the key's
        __syncthreads();
    }
    if (above) *above = above_hi;
    if (at) *at = at_t;
    return lo;
}

// The same threshold among few tokens (OWN a thread), in one pass where the logits spread: run_of(key), 0 for the
// largest logits up to SEARCH_BUCKETS - 1, is a run of equal width in the logit, token(e, key) tells a token's key and
// gives its measure (0: no token), limit_of(sum) the limit for their sum. What falls into the boundary's run, a handful, every wave puts in order
// for itself. (By halving the keys' range, as above, 300 tokens took three passes, 14 us of a row's 31; the row takes 20 this way.)
// Gives whether there is a boundary among them; `key` is left alone if its run holds more than 64 tokens (many that tie):
// then found == FEW_CROWDED, and the caller searches as above. limit: what limit_of gave.
#define SEARCH_FEW 64
enum { FEW_NONE = 0, FEW_FOUND = 1, FEW_CROWDED = 2 };
struct FewLds { fixed_t mass[SEARCH_FEW], above; uint32_t key[SEARCH_FEW]; int run, n; };
// The masses of the runs are in fx: finds the run in which their sum, from run 0 on, passes the limit (few->run; -1:
// none), and the sum before it. Barriers before and after.
template <typename Limit>
__device__ __forceinline__ int crossing_run(Limit limit_of, int tid, const fixed_t* fx, fixed_t* wsum, FewLds* few,
                                            fixed_t& limit) {
    const int wave = tid >> 6, lane = tid & 63;
    __syncthreads();
    const fixed_t f0 = fx[2 * tid], f1 = fx[2 * tid + 1];
    fixed_t upto = f0 + f1;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const fixed_t t = __shfl_up(upto, o, 64);
        if (lane >= o) upto += t;
    }
    if (lane == 63) wsum[wave] = upto;
    __syncthreads();
    fixed_t sum = 0ull, before = 0ull;
#pragma unroll
    for (int w = 0; w < CAND_WAVES; ++w) {
        const fixed_t t = wsum[w];
        sum += t;
        before += w < wave ? t : 0ull;
    }
    limit = limit_of(sum);
    const fixed_t b1 = before + upto - f1, b0 = b1 - f0;              // measure before runs 2 tid + 1 and 2 tid
    if (b0 <= limit && b1 > limit) { few->run = 2 * tid; few->above = b0; }
    if (b1 <= limit && b1 + f1 > limit) { few->run = 2 * tid + 1; few->above = b1; }
    __syncthreads();
    return few->run;
}
__device__ __forceinline__ void clear_runs(int tid, fixed_t* fx, FewLds* few) {
    fx[2 * tid] = 0ull;
    fx[2 * tid + 1] = 0ull;
    if (tid == 0) { few->run = -1; few->n = 0; }
    __syncthreads();
}
template <int OWN, typename Run, typename Token, typename Limit>
__device__ __forceinline__ int search_few(Run run_of, Token token, Limit limit_of, int tid,
                                          fixed_t* fx, fixed_t* wsum, FewLds* few, uint32_t& key, fixed_t& limit,
                                          fixed_t& above, fixed_t& at) {
    const int lane = tid & 63;
    clear_runs(tid, fx, few);
#pragma unroll 4
    for (int e = 0; e < OWN; ++e) {
        uint32_t k;
        const fixed_t m = token(e, k);
        if (m) atomicAdd(&fx[run_of(k)], m);
    }
    const int run = crossing_run(limit_of, tid, fx, wsum, few, limit);
    if (run < 0) return FEW_NONE;
#pragma unroll 4
    for (int e = 0; e < OWN; ++e) {
        uint32_t k;
        const fixed_t m = token(e, k);
        if (m && run_of(k) == run) {
            const int i = atomicAdd(&few->n, 1);
            if (i < SEARCH_FEW) { few->key[i] = k; few->mass[i] = m; }
        }
    }
    __syncthreads();
    const int n = few->n;
    if (n > SEARCH_FEW) return FEW_CROWDED;
    const uint32_t mine = lane < n ? few->key[lane] : 0u;
    fixed_t over = few->above, same = 0ull;
    for (int j = 0; j < n; ++j) {
        const uint32_t k = few->key[j];
        const fixed_t m = few->mass[j];
        over += k > mine ? m : 0ull;
        same += k == mine ? m : 0ull;
    }
    uint32_t t = lane < n && over <= limit ? mine : 0xffffffffu;     // the smallest with at most the limit above it
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t = min(t, (uint32_t)__shfl_xor((int)t, o, 64));
    const int who = __ffsll((long long)__ballot(lane < n && mine == t)) - 1;
    key = t;
    above = __shfl(over, who, 64);
    at = __shfl(same, who, 64);
    return FEW_FOUND;
}

// Of the tokens that tie at a boundary, the first `stay` in vocabulary order stay: returns the index of the
// last of them (`upto` if all of them stay). count_ties(f) calls f(index) for every tying token of this thread
// with index <= upto. One pass counts them; only if they are more than may stay, the index is searched.
// (A function of its own, not inlined: it runs four times in the kernel, and inlined the kernel no longer
// fits the 128 registers that a block of 1,024 threads leaves a lane.)
// known: their number if the search has it already (then nothing is counted), else FIXED_UNKNOWN.
template <typename Ties>
__device__ __noinline__ int tie_cut(Ties ties, int tid, int V, unsigned long long stay, int upto, fixed_t known,
                       fixed_t* fx, fixed_t* wsum, int* sh_b, fixed_t* sh_above) {
    fixed_t n = known;
    if (known == FIXED_UNKNOWN) {
        fixed_t mine = 0ull;
        ties([&](int) { mine += 1ull; });
        n = block_sum_fixed(mine, wsum);
    }
    if (stay >= n) return upto;
    if (stay == 0ull) return -1;
    // the stay-th tie from the front: the smallest t with at most stay - 1 ties at keys V - 1 - index above it
    const uint32_t t = search_threshold(
        [=](uint32_t lo, uint32_t hi, auto add) {
            ties([&](int i) {
                const uint32_t key = (uint32_t)(V - 1 - i);
                if (key > lo && key <= hi) add(key, 1ull << 40);
            });
        },
        tid, 0u, (uint32_t)(V - 1), (fixed_t)(stay - 1ull) << 40, fx, wsum, sh_b, sh_above);
    return V - 1 - (int)t;
}

// The draw's first step: wmass[w] is the kept mass of wave w's run of tokens (runs in vocabulary order).
// Gives the wave in whose run the running sum passes u times the total (the last run with kept mass if it
// never does), the sum before that run and the target. Every thread computes the same.
__device__ __forceinline__ void pick_wave(const float* wmass, float u, int& owner, float& before, float& target) {
    float m[CAND_WAVES], total = 0.f;
#pragma unroll
    for (int w = 0; w < CAND_WAVES; ++w) m[w] = wmass[w];            // (all on their way at once)
#pragma unroll
    for (int w = 0; w < CAND_WAVES; ++w) total += m[w];
    target = u * total;
    float run = 0.f;
    owner = -1;
    before = 0.f;
    bool passed = false;
#pragma unroll
    for (int w = 0; w < CAND_WAVES; ++w) {
        if (!passed && m[w] > 0.f) {
            owner = w;
            before = run;
            passed = run + m[w] > target;
            run += m[w];
        }
    }
}

// Running sums over the lanes of a wave, lane by lane in lane order (inclusive).
__device__ __forceinline__ float wave_running_sum(float v, int lane) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const float t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    return v;
}

// ---- Large vocabularies, few rows: one block a row leaves the chip idle (a flat row of 151,936 takes it 111 us, all
// of it one CU's arithmetic over five passes; 45 this way), so kernels over CAND_WAVES * parts blocks a row find what the
// last one, sample_kernel, needs:
//   sample_top      largest logit, first index that holds it, smallest, sum of exp, of every part of the row
//   sample_span     marks (a bit a token) of those within CAND_SPAN of the largest, their number and mass; for top-p
//                   alone the masses of HIST runs of equal width in the logit, which hold every token that weighs anything
//   sample_gather   flat rows under top-p alone: the tokens of the run in which the boundary lies
//   sample_settle   the boundary itself, searched among those (one block a row)
//   sample_masses   the kept mass of every 256 tokens
// Whole numbers are added, so that thresholds are the ones that the passes over the row find, bit for bit, and the
// masses of 256 tokens are summed as the draw sums them. Rows that need none of a kernel leave it at once; what none
// of them settles (top-k beyond the list, a run with more than GATHER tokens, a largest logit that is no number) goes
// the way it goes without them.
#define HIST 512
#define GATHER 8192
#define PART_THREADS 256
#define MAX_PARTS 64

struct RowPart { float mx, se, mn; int arg, count; fixed_t rest, mass; };
struct RowState { uint32_t keep_key; int tie_limit, status, gathered; };
enum { ROW_OPEN = 0, ROW_SETTLED = 1 };
struct RowTop { float mx, se, mn; int arg; };

struct SampleWs {
    char* base;
    size_t row_bytes, marks_at, masses_at;
    static constexpr size_t HIST_AT = MAX_PARTS * sizeof(RowPart), STATE_AT = HIST_AT + HIST * sizeof(fixed_t),
                            LIST_AT = STATE_AT + sizeof(RowState);
    __device__ char* at(int row) const { return base + (size_t)row * row_bytes; }
    __device__ RowPart* parts(int row) const { return reinterpret_cast<RowPart*>(at(row)); }
    __device__ fixed_t* hist(int row) const { return reinterpret_cast<fixed_t*>(at(row) + HIST_AT); }
    __device__ RowState& state(int row) const { return *reinterpret_cast<RowState*>(at(row) + STATE_AT); }
    __device__ uint2* list(int row) const { return reinterpret_cast<uint2*>(at(row) + LIST_AT); }      // key, token
    __device__ fixed_t* marks(int row) const { return reinterpret_cast<fixed_t*>(at(row) + marks_at); } // four words per 256
    __device__ float* masses(int row) const { return reinterpret_cast<float*>(at(row) + masses_at); }
};

static SampleWs sample_ws(char* base, int V) {
    const size_t blocks = (size_t)(V + 255) / 256;
    SampleWs w{base, 0, SampleWs::LIST_AT + GATHER * sizeof(uint2), 0};
    w.masses_at = w.marks_at + blocks * 4 * sizeof(fixed_t);
    w.row_bytes = (w.masses_at + blocks * sizeof(float) + 255) / 256 * 256;
    return w;
}

__device__ __forceinline__ bool finite(float f) { return fabsf(f) < INFINITY; }

// One pass's maximum, first index that holds it and sum of exp(x - maximum). What is subtracted is never -inf, so that a
// token of logit -inf weighs nothing, in front of the first other one too (-inf less -inf would be NaN).
struct RunningTop {
    float mx = -INFINITY, ref = -3.402823466e38f, se = 0.f;
    int arg = 0x7fffffff;
    __device__ __forceinline__ void add(int i, float v) {
        if (v > mx) {
            se = se * __expf(mx - v) + 1.0f;              // mx = -inf: se is 0 and stays finite
            mx = ref = v;
            arg = i;
        } else {
            se += __expf(v - ref);
        }
    }
};

// merges (mx, se, arg) over the lanes of a wave: every lane gets the same
__device__ __forceinline__ void merge_top(float& mx, float& se, int& arg) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float m2 = __shfl_xor(mx, o, 64), s2 = __shfl_xor(se, o, 64);
        const int a2 = __shfl_xor(arg, o, 64);
        const float m = fmaxf(mx, m2);
        const float s1 = (mx == -INFINITY) ? 0.f : se * __expf(mx - m);
        const float s3 = (m2 == -INFINITY) ? 0.f : s2 * __expf(m2 - m);
        arg = (m2 > mx) ? a2 : ((m2 == mx) ? min(arg, a2) : arg);
        se = s1 + s3;                                 // the same two numbers in both lanes of a pair
        mx = m;
    }
}

// The whole row's from its parts' (n <= 64); every wave does it for itself.
__device__ __forceinline__ RowTop row_top(const RowPart* parts, int n) {
    const int lane = threadIdx.x & 63;
    RowTop t{-INFINITY, 0.f, INFINITY, 0x7fffffff};
    if (lane < n) t = RowTop{parts[lane].mx, parts[lane].se, parts[lane].mn, parts[lane].arg};
    merge_top(t.mx, t.se, t.arg);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t.mn = fminf(t.mn, __shfl_xor(t.mn, o, 64));
    return t;
}

// One part's tokens: run (part / parts) of the row, which is what one wave of sample_kernel has, cut into `parts`
// pieces of whole 256s. f(token of the lane's first, its four logits, -inf beyond the end; number of the 256).
struct PartRange { int beg, end; };
__device__ __forceinline__ PartRange part_range(int V, int part, int parts) {
    const int seg = ((V + CAND_WAVES - 1) / CAND_WAVES + 255) / 256 * 256;
    const int piece = (seg / 256 + parts - 1) / parts * 256;
    const int run = part / parts, k = part - run * parts;
    const int end = min(V, run * seg + min(seg, (k + 1) * piece));
    return {min(end, run * seg + k * piece), end};
}
template <typename F>
__device__ __forceinline__ void for_each_256(const float* __restrict__ x, int V, PartRange r, F f) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool vec = (V & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    constexpr int STEP = 256 * (PART_THREADS / 64), AHEAD = 4;
    for (int b0 = r.beg + 256 * wave; b0 < r.end; b0 += AHEAD * STEP) {
        float a[AHEAD][4];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            const int i = b0 + j * STEP + 4 * lane;
            if (vec) {
                float4 t = make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);
                if (i < r.end) t = *reinterpret_cast<const float4*>(x + i);
                a[j][0] = t.x; a[j][1] = t.y; a[j][2] = t.z; a[j][3] = t.w;
            } else {
#pragma unroll
                for (int c = 0; c < 4; ++c) a[j][c] = i + c < r.end ? x[i + c] : -INFINITY;
            }
        }
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (b0 + j * STEP < r.end) f(b0 + j * STEP + 4 * lane, a[j], (b0 + j * STEP) / 256);
    }
}

__global__ __launch_bounds__(PART_THREADS) void sample_top_kernel(const float* __restrict__ logits, int V, SampleWs ws,
                                                                  int parts) {
    const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x;
    for (int i = part * PART_THREADS + tid; i < HIST; i += gridDim.x * PART_THREADS) ws.hist(row)[i] = 0ull;
    if (part == 0 && tid == 0) ws.state(row).gathered = 0;
    const PartRange r = part_range(V, part, parts);
    RunningTop top;
    float mn = INFINITY;
    for_each_256(logits + (size_t)row * V, V, r, [&](int i, const float (&a)[4], int) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (i + c >= r.end) continue;
            mn = fminf(mn, a[c]);
            top.add(i + c, a[c]);
        }
    });
    float mx = top.mx, se = top.se;
    int arg = top.arg;
    merge_top(mx, se, arg);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mn = fminf(mn, __shfl_xor(mn, o, 64));
    __shared__ RowTop w[PART_THREADS / 64];
    if ((tid & 63) == 0) w[tid >> 6] = RowTop{mx, se, mn, arg};
    __syncthreads();
    if (tid != 0) return;
    for (int k = 1; k < PART_THREADS / 64; ++k) {
        const float m = fmaxf(mx, w[k].mx);
        const float s1 = (mx == -INFINITY) ? 0.f : se * __expf(mx - m);
        const float s2 = (w[k].mx == -INFINITY) ? 0.f : w[k].se * __expf(w[k].mx - m);
        if (w[k].mx > mx) arg = w[k].arg;
        else if (w[k].mx == mx) arg = min(arg, w[k].arg);
        mx = m;
        se = s1 + s2;
        mn = fminf(mn, w[k].mn);
    }
    RowPart& p = ws.parts(row)[part];
    p.mx = mx; p.se = se; p.mn = mn; p.arg = arg;
}

// The run of equal width in the logit that a token belongs to: 0 holds the largest. -1: it weighs nothing.
struct Runs {
    float mx, inv_t, scale;
    __device__ Runs(const RowTop& t, float temp) : mx(t.mx), inv_t(1.0f / temp) {
        scale = fminf((float)HIST / fminf(WEIGHS_NOTHING * temp, t.mx - t.mn), 1e30f);      // (one value only: 1e30, all in run 0)
    }
    __device__ int operator()(float v) const {
        return (mx - v) * inv_t < WEIGHS_NOTHING ? (int)fminf((mx - v) * scale, (float)(HIST - 1)) : -1;
    }
};

__global__ __launch_bounds__(PART_THREADS) void sample_span_kernel(
    const float* __restrict__ logits, int V, const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, SampleWs ws, int parts) {
    const int row = blockIdx.y, part = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const float temp = temperature[row];
    const int k = top_k[row];
    const bool want_k = k > 0 && k < V, want_p = top_p[row] < 1.0f;
    if (!(temp > 0.f) || !(want_k || want_p)) return;
    const RowTop top = row_top(ws.parts(row), gridDim.x);
    if (!finite(top.mx)) return;
    const bool masses = want_p && !want_k;
    const Runs run_of(top, temp);
    const float gmax = top.mx, inv_t = 1.0f / temp, cut = gmax - CAND_SPAN * temp;
    __shared__ fixed_t h[HIST];
    for (int i = tid; i < HIST; i += PART_THREADS) h[i] = 0ull;
    __syncthreads();
    int count = 0;
    fixed_t mass = 0ull, rest = 0ull;
    const PartRange r = part_range(V, part, parts);
    for_each_256(logits + (size_t)row * V, V, r, [&](int i, const float (&a)[4], int b) {
        uint32_t rest4 = 0u;
        fixed_t mark = 0ull;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const bool in = a[c] >= cut;
            const unsigned long long m = __ballot(in);
            count += __popcll(m);
            if (lane == c) mark = m;
            if (masses && i + c < r.end) {
                const float weight = __expf((a[c] - gmax) * inv_t);
                const int at = run_of(a[c]);
                if (at >= 0) {
                    const fixed_t f = to_fixed(weight);
                    atomicAdd(&h[at], f);
                    mass += in ? f : 0ull;
                }
                rest4 += in ? 0u : to_fixed_rest(weight);
            }
        }
        rest += rest4;
        if (lane < 4) ws.marks(row)[4 * (size_t)b + lane] = mark;
    });
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        rest += __shfl_xor(rest, o, 64);
        mass += __shfl_xor(mass, o, 64);
    }
    __shared__ int wc[PART_THREADS / 64];
    __shared__ fixed_t wr[PART_THREADS / 64], wm[PART_THREADS / 64];
    if (lane == 0) { wc[tid >> 6] = count; wr[tid >> 6] = rest; wm[tid >> 6] = mass; }
    __syncthreads();
    if (masses)
        for (int i = tid; i < HIST; i += PART_THREADS)
            if (h[i]) atomicAdd(&ws.hist(row)[i], h[i]);
    if (tid != 0) return;
    for (int w = 1; w < PART_THREADS / 64; ++w) { count += wc[w]; rest += wr[w]; mass += wm[w]; }
    RowPart& p = ws.parts(row)[part];
    p.count = count; p.rest = rest; p.mass = mass;
}

// Whether a row under top-p alone is one for the searches over the whole row: too many candidates for the list in
// one run, or less than top_p of the mass among them. Every wave finds it for itself.
__device__ __forceinline__ bool row_is_flat(const RowPart* all, int parts, float gmax, float temp, float top_p) {
    const int lane = threadIdx.x & 63;
    if (order_key(gmax - CAND_SPAN * temp) == 0u) return true;
    int count = 0;
    if (lane < CAND_WAVES)
        for (int j = 0; j < parts; ++j) count += all[lane * parts + j].count;
    if (__ballot(count > CAND_PER_WAVE)) return true;
    fixed_t mass = lane < CAND_WAVES * parts ? all[lane].mass : 0ull;
    fixed_t rest = lane < CAND_WAVES * parts ? all[lane].rest : 0ull;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        mass += __shfl_xor(mass, o, 64);
        rest += __shfl_xor(rest, o, 64);
    }
    const fixed_t z = mass + fixed_of_rest(rest);
    return mass <= (fixed_t)((double)top_p * (double)z);
}

// The run in which the top-p boundary lies, the mass of the runs before it, and what may lie above the boundary.
struct Boundary { int run; fixed_t above, limit; };
__device__ __forceinline__ Boundary boundary_run(const fixed_t* hist, float top_p) {
    const int lane = threadIdx.x & 63;
    constexpr int EACH = HIST / 64;
    fixed_t h[EACH], mine = 0ull;
#pragma unroll
    for (int e = 0; e < EACH; ++e) { h[e] = hist[lane * EACH + e]; mine += h[e]; }
    fixed_t upto = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const fixed_t t = __shfl_up(upto, o, 64);
        if (lane >= o) upto += t;
    }
    const fixed_t z = __shfl(upto, 63, 64);
    const fixed_t limit = (fixed_t)((double)top_p * (double)z);
    const unsigned long long past = __ballot(upto > limit);
    const int who = past ? __ffsll((long long)past) - 1 : 63;
    fixed_t above = upto - mine;
    int run = lane * EACH;
#pragma unroll
    for (int e = 0; e < EACH - 1; ++e)
        if (run == lane * EACH + e && above + h[e] <= limit) { above += h[e]; ++run; }
    return {__shfl(run, who, 64), __shfl(above, who, 64), limit};
}

__global__ __launch_bounds__(PART_THREADS) void sample_gather_kernel(
    const float* __restrict__ logits, int V, const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, SampleWs ws, int parts) {
    const int row = blockIdx.y, part = blockIdx.x, lane = threadIdx.x & 63;
    const float temp = temperature[row], p = top_p[row];
    const int k = top_k[row];
    if (!(temp > 0.f) || !(p < 1.0f) || (k > 0 && k < V)) return;
    const RowTop top = row_top(ws.parts(row), gridDim.x);
    if (!finite(top.mx) || !row_is_flat(ws.parts(row), parts, top.mx, temp, p)) return;
    const Boundary b = boundary_run(ws.hist(row), p);
    const Runs run_of(top, temp);
    const PartRange r = part_range(V, part, parts);
    for_each_256(logits + (size_t)row * V, V, r, [&](int i, const float (&a)[4], int) {
        int before = 0, all = 0;
        bool in[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            in[c] = i + c < r.end && run_of(a[c]) == b.run;
            const unsigned long long m = __ballot(in[c]);
            before += __popcll(m & ((1ull << lane) - 1ull));
            all += __popcll(m);
        }
        if (all == 0) return;
        int at = 0;
        if (lane == 0) at = atomicAdd(&ws.state(row).gathered, all);
        at = __shfl(at, 0, 64) + before;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (in[c]) {
                if (at < GATHER) ws.list(row)[at] = make_uint2(order_key(a[c]), (uint32_t)(i + c));
                ++at;
            }
    });
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_settle_kernel(
    int V, const float* __restrict__ temperature, const int* __restrict__ top_k, const float* __restrict__ top_p,
    SampleWs ws, int parts) {
    __shared__ fixed_t fx[SEARCH_BUCKETS], wsum[CAND_WAVES], sh_above;
    __shared__ int sh_b;
    __shared__ FewLds few;
    const int row = blockIdx.x, tid = threadIdx.x;
    const float temp = temperature[row], p = top_p[row];
    const int k = top_k[row];
    RowState& st = ws.state(row);
    const bool want_k = k > 0 && k < V, want_p = p < 1.0f;
    const RowTop top = row_top(ws.parts(row), CAND_WAVES * parts);
    if (!(temp > 0.f) || want_k || !finite(top.mx)) {
        if (tid == 0) st.status = ROW_OPEN;
        return;
    }
    if (!want_p) {                                     // all of it is kept
        if (tid == 0) { st.keep_key = 0u; st.tie_limit = 0x7fffffff; st.status = ROW_SETTLED; }
        return;
    }
    const int n = st.gathered;
    if (n > GATHER || n == 0 || !row_is_flat(ws.parts(row), parts, top.mx, temp, p)) {
        if (tid == 0) st.status = ROW_OPEN;
        return;
    }
    const Boundary b = boundary_run(ws.hist(row), p);
    const float inv_t = 1.0f / temp;
    constexpr int OWN = GATHER / SAMPLE_THREADS;
    const uint2* list = ws.list(row);
    auto entry = [list, tid, n](int e, uint32_t& key, int& i) {
        const int at = tid + e * SAMPLE_THREADS;
        const uint2 t = at < n ? list[at] : make_uint2(0u, 0u);
        key = t.x;
        i = (int)t.y;
        return at < n;
    };
    auto weighed = [=](int e, uint32_t& key) {
        int i;
        return entry(e, key, i) ? to_fixed(__expf((key_value(key) - top.mx) * inv_t)) : 0ull;
    };
    const Runs runs(top, temp);
    fixed_t above = 0ull, at = FIXED_UNKNOWN, limit_in;
    uint32_t keep = 0u;
    if (search_few<OWN>(
            [=](uint32_t key) {                        // the run's width, cut once more
                const float d = ((top.mx - key_value(key)) * runs.scale - (float)b.run) * (float)SEARCH_BUCKETS;
                return (int)fminf(fmaxf(d, 0.f), (float)(SEARCH_BUCKETS - 1));
            },
            weighed, [=](fixed_t) { return b.limit - b.above; }, tid, fx, wsum, &few, keep, limit_in, above, at) != FEW_FOUND) {
        __syncthreads();
        keep = search_threshold(
            [=](uint32_t lo, uint32_t hi, auto add) {
                for (int e = 0; e < OWN; ++e) {
                    uint32_t key;
                    const fixed_t m = weighed(e, key);
                    if (m && key > lo && key <= hi) add(key, m);
                }
            },
            tid, 0u, order_key(top.mx), b.limit - b.above, fx, wsum, &sh_b, &sh_above, &above, &at);
    }
    // of the tokens that tie with the boundary value, as in sample_kernel
    const fixed_t each = to_fixed(__expf((key_value(keep) - top.mx) * inv_t));
    const unsigned long long stay = each ? (b.limit - b.above - above) / each + 1ull : ~0ull;
    const int limit = tie_cut(
        [entry, keep](auto f) {
            for (int e = 0; e < OWN; ++e) {
                uint32_t key;
                int i;
                if (entry(e, key, i) && key == keep) f(i);
            }
        },
        tid, V, stay, 0x7fffffff, at != FIXED_UNKNOWN && each ? at / each : FIXED_UNKNOWN, fx, wsum, &sh_b, &sh_above);
    if (tid == 0) { st.keep_key = keep; st.tie_limit = limit; st.status = ROW_SETTLED; }
}

__global__ __launch_bounds__(PART_THREADS) void sample_masses_kernel(const float* __restrict__ logits, int V,
                                                                     const float* __restrict__ temperature, SampleWs ws,
                                                                     int parts) {
    const int row = blockIdx.y, lane = threadIdx.x & 63;
    const RowState st = ws.state(row);
    if (st.status != ROW_SETTLED) return;
    const float gmax = row_top(ws.parts(row), gridDim.x).mx, inv_t = 1.0f / temperature[row];
    const PartRange r = part_range(V, blockIdx.x, parts);
    for_each_256(logits + (size_t)row * V, V, r, [&](int i, const float (&a)[4], int b) {
        float m = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t key = order_key(a[c]);
            const bool kept = i + c < r.end && (key > st.keep_key || (key == st.keep_key && i + c <= st.tie_limit));
            m += kept ? __expf((a[c] - gmax) * inv_t) : 0.f;
        }
        m = wave_sum(m);
        if (lane == 0) ws.masses(row)[b] = m;
    });
}

// A wave's part of the list from the marks of its run of the row (n 256s, at most SAMPLE_BLOCKS = 64: one a lane), in
// vocabulary order: entry e is the e-th mark. Gives the number of marks; nothing is written if they are too many.
__device__ __forceinline__ int list_of_marks(const fixed_t* __restrict__ marks, int n, const float* __restrict__ x,
                                             int beg, int lane, float* cv, int* ci) {
    int mine = 0;
    if (lane < n)
#pragma unroll
        for (int c = 0; c < 4; ++c) mine += __popcll(marks[4 * lane + c]);
    int upto = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(upto, o, 64);
        if (lane >= o) upto += t;
    }
    const int all = __shfl(upto, 63, 64);
    if (all > CAND_PER_WAVE) return all;
    for (int e0 = 0; e0 < all; e0 += 64) {
        const int e = e0 + lane;
        int b = 0;                                     // the first 256 with more than e marks up to its end
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
            if (__shfl(upto, b + o - 1, 64) <= e) b += o;
        const int left = e - __shfl(upto - mine, b, 64);       // (all lanes take part in the shuffles)
        if (e < all) {
            fixed_t m[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) m[c] = marks[4 * b + c];
            int l = 0, below = 0;                      // the lane of the 256 that holds it: marks of the lanes before it <= left
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) {
                const unsigned long long mask = (1ull << (l + o)) - 1ull;
                int c2 = 0;
#pragma unroll
                for (int c = 0; c < 4; ++c) c2 += __popcll(m[c] & mask);
                if (c2 <= left) { l += o; below = c2; }
            }
            int want = left - below, c = 0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int bit = (int)((m[q] >> l) & 1ull);
                if (bit && want == 0) c = q;
                want -= bit;
            }
            const int token = beg + 256 * b + 4 * l + c;
            cv[e] = x[token];
            ci[e] = token;
        }
    }
    return all;
}

// PREPARED: the row's sums, candidates and block masses were found by the kernels above (ws); else this block finds
// them itself.
template <bool PREPARED>
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_kernel(
    const float* __restrict__ logits, int V, const float* __restrict__ temperature,
    const int* __restrict__ top_k, const float* __restrict__ top_p, const float* __restrict__ u,
    int* __restrict__ out, int* __restrict__ path, SampleWs ws_all, int parts) {
    extern __shared__ __attribute__((aligned(16))) float dyn[];           // the list (64 KB), then the search's runs (16 KB)
    __shared__ float scratch[16];
    __shared__ float wmass[CAND_WAVES];
    __shared__ fixed_t wsum[CAND_WAVES];
    __shared__ fixed_t sh_above;
    __shared__ int sh_b;
    __shared__ FewLds few;
    fixed_t* fx = reinterpret_cast<fixed_t*>(dyn + 2 * CAND_WAVES * CAND_PER_WAVE);
    const int row = blockIdx.x, tid = threadIdx.x;
    const float* x = logits + (size_t)row * V;

    float gmax, total_e = 0.f;
    int argmax;
    [[maybe_unused]] const int n_parts = CAND_WAVES * parts;
    if constexpr (PREPARED) {
        const RowTop t = row_top(ws_all.parts(row), n_parts);
        gmax = t.mx;
        argmax = t.arg;
        total_e = t.se;
    } else {
        // ---- one pass: running maximum, first index that holds it, sum of exp(x - maximum)
        RunningTop top;
        for_each_logit(x, V, tid, [&](int i, float v) { top.add(i, v); });
        float mx = top.mx, se = top.se;
        int arg = top.arg;
        merge_top(mx, se, arg);                           // over the wave; then over the waves in wave order
        __shared__ float wm[16], ws[16];
        __shared__ int wa[16];
        if ((tid & 63) == 0) { wm[tid >> 6] = mx; ws[tid >> 6] = se; wa[tid >> 6] = arg; }
        __syncthreads();
        gmax = wm[0];
        argmax = wa[0];
        for (int w = 1; w < SAMPLE_THREADS / 64; ++w) {
            if (wm[w] > gmax) { gmax = wm[w]; argmax = wa[w]; }
            else if (wm[w] == gmax) argmax = min(argmax, wa[w]);
        }
        for (int w = 0; w < SAMPLE_THREADS / 64; ++w)
            total_e += (wm[w] == -INFINITY) ? 0.f : ws[w] * __expf(wm[w] - gmax);
    }
    // a row with no value above -inf (all -inf, or NaN after an overflow upstream) never set an index:
    // token 0 then, so that nothing below reads beyond the row
    if ((unsigned)argmax >= (unsigned)V) argmax = 0;
    const float lse = gmax + logf(total_e);

    const float temp = temperature[row];
    if (!(temp > 0.f)) {
        if (tid == 0) {
            out[2 * row] = argmax;
            out[2 * row + 1] = __float_as_int(x[argmax] - lse);
            if (path) path[row] = 0;
        }
        return;
    }
    const float inv_t = 1.0f / temp;
    const uint32_t top_key = order_key(gmax);

    // Wave w's run of the row (a multiple of 256 tokens): a lane reads four consecutive tokens of every 256,
    // so that what a wave meets, load by load, lane by lane, is in vocabulary order.
    const int wave = tid >> 6, lane = tid & 63;
    const int seg = ((V + CAND_WAVES - 1) / CAND_WAVES + 255) / 256 * 256;
    const int beg = min(V, wave * seg), end = min(V, beg + seg);
    const bool vec = (V & 3) == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    auto load4 = [&](int i, float (&a)[4]) {           // tokens i .. i+3 of the run, -inf beyond its end
        if (vec) {
            if (i < end) {
                const float4 t = *reinterpret_cast<const float4*>(x + i);
                a[0] = t.x; a[1] = t.y; a[2] = t.z; a[3] = t.w;
            } else {
                a[0] = a[1] = a[2] = a[3] = -INFINITY;
            }
        } else {
#pragma unroll
            for (int c = 0; c < 4; ++c) a[c] = i + c < end ? x[i + c] : -INFINITY;
        }
    };

    const int k = top_k[row];
    const float p = top_p[row];
    const bool want_k = k > 0 && k < V, want_p = p < 1.0f;
    // what stays: tokens whose key is above keep_key, and of those whose key is keep_key the ones up to tie_limit
    uint32_t keep_key = 0u;
    int tie_limit = 0x7fffffff;
    auto kept = [&](uint32_t key, int i) { return key > keep_key || (key == keep_key && i <= tie_limit); };

    bool settled = false;                              // thresholds and block masses are there already
    if constexpr (PREPARED) {
        const RowState st = ws_all.state(row);
        if (st.status == ROW_SETTLED) {
            settled = true;
            keep_key = st.keep_key;
            tie_limit = st.tie_limit;
        }
    }
    if (!settled && (want_k || want_p)) {
        // ---- the list: wave w goes through its run of the row, 64 tokens a load, and appends the tokens
        // within CAND_SPAN of the largest to its part of the list, in their order
        float* cv = dyn;                                                   // [CAND_WAVES][CAND_PER_WAVE] logits
        int* ci = reinterpret_cast<int*>(dyn + CAND_WAVES * CAND_PER_WAVE);    // and their token numbers
        __shared__ int cnt[CAND_WAVES];
        __shared__ int sh_over;
        const float cut = gmax - CAND_SPAN * temp;
        const uint32_t cut_key = order_key(cut);
        const bool sum_rest = want_p && !want_k;       // top-p alone is over the mass of the whole row
        if (tid == 0) sh_over = 0;
        __syncthreads();
        {
            int have = 0;
            fixed_t rest = 0ull;
            [[maybe_unused]] bool marked = false;
            if constexpr (PREPARED) marked = finite(gmax);
            if (marked) {
                have = list_of_marks(ws_all.marks(row) + 4 * (beg / 256), (end - beg + 255) / 256, x, beg, lane,
                                     cv + wave * CAND_PER_WAVE, ci + wave * CAND_PER_WAVE);
                if (sum_rest && tid < n_parts) rest = ws_all.parts(row)[tid].rest;
            } else {
                const unsigned long long below = (1ull << lane) - 1ull;        // the lanes before this one
                for (int i0 = beg + 4 * lane; i0 - 4 * lane < end; i0 += 4 * 256) {      // four loads on their way
                    if (have > CAND_PER_WAVE) break;          // (a flat row: this run alone is too much for the list)
                    float v[4][4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) load4(i0 + 256 * j, v[j]);
                    uint32_t rest16 = 0u;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        int before = 0, all = 0;
                        bool in[4];
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            in[c] = v[j][c] >= cut;
                            const unsigned long long m = __ballot(in[c]);
                            before += __popcll(m & below);
                            all += __popcll(m);
                        }
                        if (all != 0) {
                            int at = have + before;
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                if (in[c]) {
                                    if (at < CAND_PER_WAVE) {
                                        cv[wave * CAND_PER_WAVE + at] = v[j][c];
                                        ci[wave * CAND_PER_WAVE + at] = i0 + 256 * j + c;
                                    }
                                    ++at;
                                }
                            }
                            have += all;
                        }
                        if (sum_rest) {
#pragma unroll
                            for (int c = 0; c < 4; ++c) rest16 += in[c] ? 0u : to_fixed_rest(__expf((v[j][c] - gmax) * inv_t));
                        }
                    }
                    rest += rest16;
                }
            }
            if (lane == 0) {
                cnt[wave] = min(have, CAND_PER_WAVE);
                if (have > CAND_PER_WAVE) sh_over = 1;
            }
            const fixed_t z_rest = sum_rest ? block_sum_fixed(rest, wsum) : 0ull;       // (with barriers of its own, or:)
            __syncthreads();
            int total = 0;
            for (int w = 0; w < CAND_WAVES; ++w) total += cnt[w];
            bool listed = sh_over == 0 && cut_key > 0u && (!want_k || k <= total);

            // a thread's entries for the searches: place (tid % CAND_PER_WAVE) of every other wave's part
            if (listed) {
                const int half = tid / CAND_PER_WAVE, off = tid - half * CAND_PER_WAVE;
                const int* held = cnt;
                auto entry = [cv, ci, held, half, off](int e, float& v, int& i) {
                    const int w = half + (SAMPLE_THREADS / CAND_PER_WAVE) * e;
                    v = cv[w * CAND_PER_WAVE + off];
                    i = ci[w * CAND_PER_WAVE + off];
                    return off < held[w];
                };
                // the entries that tie at key t, up to token `upto`
                auto ties_at = [entry](uint32_t t, int upto) {
                    return [entry, t, upto](auto f) {
#pragma unroll 4
                        for (int e = 0; e < CAND_OWN; ++e) {
                            float v;
                            int i;
                            if (entry(e, v, i) && order_key(v) == t && i <= upto) f(i);
                        }
                    };
                };
                const float scale = fminf((float)SEARCH_BUCKETS / (CAND_SPAN * temp), 1e30f);
                auto run_of = [=](uint32_t key) {
                    return (int)fminf(fmaxf((gmax - key_value(key)) * scale, 0.f), (float)(SEARCH_BUCKETS - 1));
                };
                // top-k: the k-th largest is on the list; below cut_key - 1 nothing of it lies
                if (want_k) {
                    auto one = [=](int e, uint32_t& key) {
                        float v;
                        int i;
                        const bool there = entry(e, v, i);
                        key = order_key(v);
                        return there ? 1ull << 40 : 0ull;
                    };
                    fixed_t above = 0ull, at = FIXED_UNKNOWN, limit;
                    if (search_few<CAND_OWN>(run_of, one, [=](fixed_t) { return (fixed_t)(k - 1) << 40; }, tid, fx, wsum, &few,
                                             keep_key, limit, above, at) != FEW_FOUND) {
                        __syncthreads();
                        keep_key = search_threshold(
                            [=](uint32_t lo, uint32_t hi, auto add) {
                                for (int e = 0; e < CAND_OWN; ++e) {
                                    uint32_t key;
                                    const fixed_t m = one(e, key);
                                    if (m && key > lo && key <= hi) add(key, m);
                                }
                            },
                            tid, cut_key - 1u, top_key, (fixed_t)(k - 1) << 40, fx, wsum, &sh_b, &sh_above, &above, &at);
                    }
                    // of the tokens that tie with the k-th value, as many stay as make k with those above them
                    tie_limit = tie_cut(ties_at(keep_key, 0x7fffffff), tid, V, (unsigned long long)k - (above >> 40),
                                        0x7fffffff, at == FIXED_UNKNOWN ? at : at >> 40, fx, wsum, &sh_b, &sh_above);
                    __syncthreads();
                }
                if (want_p) {
                    const uint32_t k_key = keep_key;         // what top-k left: the search goes over that
                    const int k_limit = tie_limit;
                    auto weighed = [=](int e, uint32_t& key) {
                        float v;
                        int i;
                        const bool there = entry(e, v, i);
                        key = order_key(v);
                        return there && (key > k_key || (key == k_key && i <= k_limit)) ? to_fixed(__expf((v - gmax) * inv_t))
                                                                                        : 0ull;
                    };
                    fixed_t above = 0ull, at = FIXED_UNKNOWN, limit, zc = 0ull;
                    const int found = search_few<CAND_OWN>(
                        run_of, weighed,
                        [&](fixed_t sum) {
                            zc = sum;
                            const fixed_t z = sum + fixed_of_rest(z_rest);
                            return (fixed_t)((double)p * (double)z);
                        },
                        tid, fx, wsum, &few, keep_key, limit, above, at);
                    // the boundary is on the list if the list's mass is more than p of the whole (always, after top-k)
                    if (want_k || zc > limit) {
                        if (found != FEW_FOUND) {
                            __syncthreads();
                            keep_key = search_threshold(
                                [=](uint32_t lo, uint32_t hi, auto add) {
                                    for (int e = 0; e < CAND_OWN; ++e) {
                                        uint32_t key;
                                        const fixed_t m = weighed(e, key);
                                        if (m && key > lo && key <= hi) add(key, m);
                                    }
                                },
                                tid, want_k ? k_key : cut_key - 1u, top_key, limit, fx, wsum, &sh_b, &sh_above, &above, &at);
                        }
                        // of the tokens that tie with the boundary value, the i-th in vocabulary order stays while
                        // what lies before it, the mass above them and i of their own, is at most top_p of the whole
                        const fixed_t each = to_fixed(__expf((key_value(keep_key) - gmax) * inv_t));
                        const unsigned long long stay = each ? (limit - above) / each + 1ull : ~0ull;
                        const int upto = keep_key == k_key ? k_limit : 0x7fffffff;
                        // (a boundary above top-k's: every token of that value was in the search, their mass is their number)
                        const fixed_t known = (at != FIXED_UNKNOWN && each && (!want_k || keep_key != k_key)) ? at / each : FIXED_UNKNOWN;
                        tie_limit = tie_cut(ties_at(keep_key, upto), tid, V, stay, upto, known, fx, wsum, &sh_b, &sh_above);
                    } else {
                        listed = false;
                    }
                }
            }
            if (listed) {
                // ---- the draw over the list, which is in vocabulary order: wave w has its own part,
                // a lane CAND_PER_WAVE / 64 consecutive entries of it
                constexpr int RUN = CAND_PER_WAVE / 64;
                float* cw = cv + wave * CAND_PER_WAVE;      // every entry's kept mass first, in the logit's place
                for (int o = lane; o < CAND_PER_WAVE; o += 64)
                    cw[o] = o < cnt[wave] && kept(order_key(cw[o]), ci[wave * CAND_PER_WAVE + o])
                                ? __expf((cw[o] - gmax) * inv_t) : 0.f;
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                float own[RUN], mine = 0.f;
#pragma unroll
                for (int o = 0; o < RUN; ++o) own[o] = cw[RUN * lane + o];
#pragma unroll
                for (int o = 0; o < RUN; ++o) mine += own[o];
                const float upto = wave_running_sum(mine, lane);
                __syncthreads();
                if (lane == 63) wmass[wave] = upto;
                __syncthreads();
                int owner;
                float before, target;
                pick_wave(wmass, u[row], owner, before, target);
                if (owner < 0) {                       // (nothing is kept: cannot be, the largest always is)
                    if (tid == 0) {
                        out[2 * row] = argmax;
                        out[2 * row + 1] = __float_as_int(x[argmax] - lse);
                        if (path) path[row] = 1;
                    }
                    return;
                }
                if (wave != owner) return;
                // the lane in whose entries the running sum passes the target, else the last one with kept mass
                const unsigned long long passed = __ballot(mine > 0.f && before + upto > target);
                const unsigned long long any = __ballot(mine > 0.f);
                const int who = passed ? __ffsll((long long)passed) - 1 : 63 - __builtin_clzll(any);
                if (lane == who) {
                    float run = before + (upto - mine);
                    int at = -1;                           // the last kept entry if the target is never passed
                    bool over = false;
#pragma unroll
                    for (int o = 0; o < RUN; ++o)
                        if (!over && own[o] > 0.f) {
                            at = o;
                            run += own[o];
                            over = run > target;
                        }
                    const int tok = at < 0 ? argmax : ci[wave * CAND_PER_WAVE + RUN * lane + at];
                    out[2 * row] = tok;
                    out[2 * row + 1] = __float_as_int(x[tok] - lse);
                    if (path) path[row] = 1;
                }
                return;
            }
        }
        __syncthreads();
        keep_key = 0u;
        tie_limit = 0x7fffffff;
        // the row's tokens that tie at key t, up to token `upto`
        auto ties_at = [&](uint32_t t, int upto) {
            return [x, V, tid, t, upto](auto f) {
                for_each_logit(x, V, tid, [&](int i, float v) {
                    if (order_key(v) == t && i <= upto) f(i);
                });
            };
        };

        // ---- over the whole row, in two passes: masses of runs of equal width in the logit (beyond `span` from the
        // largest all in the last one), then the tokens of the run in which the boundary lies, into the list's place. mass(i, v):
        // a token's measure. False (too many tokens in it): the keys' range is halved, pass by pass, instead.
        auto search_row = [&](float span, auto mass, auto limit_of, fixed_t& limit, fixed_t& above, fixed_t& at) {
            const float scale = fminf((float)SEARCH_BUCKETS / span, 1e30f);
            auto place = [=](float v) { return (gmax - v) * scale; };
            auto cut_to_runs = [](float d) { return (int)fminf(fmaxf(d, 0.f), (float)(SEARCH_BUCKETS - 1)); };
            clear_runs(tid, fx, &few);
            for_each_logit(x, V, tid, [&](int i, float v) {
                const fixed_t m = mass(i, v);
                if (m) atomicAdd(&fx[cut_to_runs(place(v))], m);
            });
            const int run = crossing_run(limit_of, tid, fx, wsum, &few, limit);
            if (run < 0) return false;
            const fixed_t before = few.above;
            for_each_logit(x, V, tid, [&](int i, float v) {
                if (cut_to_runs(place(v)) == run && mass(i, v)) {
                    const int at = atomicAdd(&few.n, 1);
                    if (at < CAND_WAVES * CAND_PER_WAVE) {
                        cv[at] = v;
                        ci[at] = i;
                    }
                }
            });
            __syncthreads();
            const int n = few.n;
            __syncthreads();
            if (n > CAND_WAVES * CAND_PER_WAVE) return false;
            fixed_t limit_in;
            const bool found = search_few<CAND_OWN>(
                [=](uint32_t key) { return cut_to_runs((place(key_value(key)) - (float)run) * (float)SEARCH_BUCKETS); },
                [=](int e, uint32_t& key) {
                    const int o = tid + e * SAMPLE_THREADS;
                    if (o >= n) return (fixed_t)0ull;
                    key = order_key(cv[o]);
                    return mass(ci[o], cv[o]);
                },
                [=](fixed_t) { return limit - before; }, tid, fx, wsum, &few, keep_key, limit_in, above, at) == FEW_FOUND;
            above += before;
            return found;
        };
        // top-k: the key of the k-th largest value is the smallest key with at most k - 1 tokens above it
        if (want_k) {
            fixed_t above = 0ull, at = FIXED_UNKNOWN, limit;
            if (!search_row(TOP_K_SPAN, [=](int, float v) { return v <= gmax ? 1ull << 40 : 0ull; },
                            [=](fixed_t) { return (fixed_t)(k - 1) << 40; }, limit, above, at)) {
                __syncthreads();
                at = FIXED_UNKNOWN;
                keep_key = search_threshold(
                    [=](uint32_t lo, uint32_t hi, auto add) {
                        for_each_logit(x, V, tid, [&](int, float v) {
                            const uint32_t key = order_key(v);
                            if (key > lo && key <= hi) add(key, 1ull << 40);
                        });
                    },
                    tid, 0u, top_key, (fixed_t)(k - 1) << 40, fx, wsum, &sh_b, &sh_above, &above, &at);
            }
            tie_limit = tie_cut(ties_at(keep_key, 0x7fffffff), tid, V, (unsigned long long)k - (above >> 40),
                                0x7fffffff, at == FIXED_UNKNOWN ? at : at >> 40, fx, wsum, &sh_b, &sh_above);
            __syncthreads();
        }
        // top-p: the smallest key with at most p of the kept mass above it
        if (want_p) {
            const uint32_t k_key = keep_key;             // what top-k left: the search goes over that
            const int k_limit = tie_limit;
            auto mass = [=](int i, float v) {
                const uint32_t key = order_key(v);
                return v <= gmax && (key > k_key || (key == k_key && i <= k_limit)) ? to_fixed(__expf((v - gmax) * inv_t)) : 0ull;
            };
            fixed_t above = 0ull, at = FIXED_UNKNOWN, limit;
            if (!search_row(WEIGHS_NOTHING * temp, mass, [=](fixed_t sum) { return (fixed_t)((double)p * (double)sum); }, limit,
                            above, at)) {
                __syncthreads();
                at = FIXED_UNKNOWN;
                keep_key = search_threshold(
                    [=](uint32_t lo, uint32_t hi, auto add) {
                        for_each_logit(x, V, tid, [&](int i, float v) {
                            const uint32_t key = order_key(v);
                            if (key > lo && key <= hi && (key > k_key || i <= k_limit))
                                add(key, to_fixed(__expf((v - gmax) * inv_t)));
                        });
                    },
                    tid, k_key, top_key, limit, fx, wsum, &sh_b, &sh_above, &above, &at);
            }
            const fixed_t each = to_fixed(__expf((key_value(keep_key) - gmax) * inv_t));
            const unsigned long long stay = each ? (limit - above) / each + 1ull : ~0ull;
            const int upto = keep_key == k_key ? k_limit : 0x7fffffff;
            const fixed_t known = (at != FIXED_UNKNOWN && each && (!want_k || keep_key != k_key)) ? at / each : FIXED_UNKNOWN;
            tie_limit = tie_cut(ties_at(keep_key, upto), tid, V, stay, upto, known, fx, wsum, &sh_b, &sh_above);
        }
    }

    // ---- the draw over the whole row, in vocabulary order. Wave w has a run of the row (a multiple of 256
    // tokens); a lane reads four consecutive tokens of every 256. First the kept mass of every block of 256
    // tokens, and with them every wave's; then the wave in whose run the running sum passes the target finds
    // the block in which it does, and goes through that block again, token by token.
    {
        auto kept_mass = [&](int i, float v) {             // (a token beyond the run's end has none: exp(-inf))
            return (i < end && kept(order_key(v), i)) ? __expf((v - gmax) * inv_t) : 0.f;
        };
        __shared__ float bmass[CAND_WAVES][SAMPLE_BLOCKS];
        const int n_it = (end - beg + 255) / 256;            // this wave's blocks
        const bool by_block = seg / 256 <= SAMPLE_BLOCKS;    // (a vocabulary beyond 262,144: the whole run is gone through again)
        float mine = 0.f;
        if (settled) {                                       // (at most SAMPLE_BLOCKS blocks: ra_sample_traced sees to it)
            const float m = lane < n_it ? ws_all.masses(row)[beg / 256 + lane] : 0.f;
            if (lane < n_it) bmass[wave][lane] = m;
            for (int it = 0; it < n_it; ++it) mine += __shfl(m, it, 64);
        } else for (int it0 = 0; it0 < n_it; it0 += 4) {     // four loads on their way
            float a[4][4];
#pragma unroll
            for (int j = 0; j < 4; ++j) load4(beg + 256 * (it0 + j) + 4 * lane, a[j]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int i = beg + 256 * (it0 + j) + 4 * lane;
                float m = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) m += kept_mass(i + c, a[j][c]);
                m = wave_sum(m);
                if (by_block && lane == 0 && it0 + j < n_it) bmass[wave][it0 + j] = m;
                mine += m;
            }
        }
        __syncthreads();
        if (lane == 0) wmass[wave] = mine;
        __syncthreads();
        int owner;
        float before, target;
        pick_wave(wmass, u[row], owner, before, target);
        if (owner < 0) owner = 0;
        if (wave != owner) return;
        float run = before;
        int it_lo = 0, it_hi = n_it;
        if (by_block) {                                      // the block, as pick_wave finds the wave
            int ob = -1;
            float r2 = before;
            for (int it = 0; it < n_it; ++it) {
                const float bm = bmass[wave][it];
                if (bm > 0.f) {
                    ob = it;
                    run = r2;
                    if (r2 + bm > target) break;
                    r2 += bm;
                }
            }
            it_lo = max(ob, 0);
            it_hi = ob < 0 ? 0 : ob + 1;
        }
        int last_kept = -1, tok = -1;
        constexpr int AHEAD = 4;                             // loads on their way
        float a[AHEAD][4];
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) load4(beg + 256 * (it_lo + j) + 4 * lane, a[j]);
        for (int it0 = it_lo; it0 < it_hi && tok < 0; it0 += AHEAD) {
#pragma unroll
            for (int j = 0; j < AHEAD; ++j) {
                const int i = it0 + j < it_hi ? beg + 256 * (it0 + j) + 4 * lane : end;      // (beyond the blocks asked for: nothing)
                float m[4], s[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) m[c] = kept_mass(i + c, a[j][c]);
                s[0] = m[0]; s[1] = s[0] + m[1]; s[2] = s[1] + m[2]; s[3] = s[2] + m[3];
                const float upto = wave_running_sum(s[3], lane);
                const float base = run + (upto - s[3]);
                int first = -1;
#pragma unroll
                for (int c = 3; c >= 0; --c) {
                    const bool is_kept = i + c < end && kept(order_key(a[j][c]), i + c);
                    if (is_kept && base + s[c] > target) first = c;
                    if (is_kept) last_kept = max(last_kept, i + c);
                }
                const unsigned long long passed = __ballot(first >= 0);
                if (passed && tok < 0) {
                    const int who = __ffsll((long long)passed) - 1;
                    tok = __shfl(i + max(first, 0), who, 64);
                }
                run += __shfl(upto, 63, 64);
                load4(beg + 256 * (it0 + j + AHEAD) + 4 * lane, a[j]);                 // (beyond the run's end: -inf)
            }
        }
        if (tok < 0) {                                       // never passed: the last kept token of the run
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) last_kept = max(last_kept, __shfl_xor(last_kept, o, 64));
            tok = last_kept < 0 ? argmax : last_kept;
        }
        if (lane == 0) {
            out[2 * row] = tok;
            out[2 * row + 1] = __float_as_int(x[tok] - lse);
            if (path) path[row] = (want_k || want_p) ? 2 : 0;
        }
    }
}

// How many pieces a wave's run of the row is cut into for the kernels over several blocks a row; 0: one block a row.
// The line, one block a row / several blocks, microseconds a call, logits near normal at T 0.7, greedy | top-p 0.9 with
// 300 large logits | top-p 0.9, flat:
//   vocabulary  65,536   1 row  10.5 / 13.1 | 30 / 32 |  56 / 37      32 rows 11.0 / 16.3 | 31 / 37 |  59 / 47
//              128,256   1      16.4 / 13.8 | 41 / 33 |  99 / 42      32      16.9 / 18.0 | 41 / 41 | 101 / 62
//              151,936   1      18.0 / 14.0 | 45 / 34 | 111 / 45      32      18.7 / 18.9 | 45 / 44 | 116 / 67
//              151,936  64      19.7 / 23.6 | 53 / 54 | 123 / 84
// so that from about 100,000 tokens and up to 32 rows no kind of row loses; beyond SAMPLE_BLOCKS 256s a run the masses
// have no room.
static int sample_parts(int M, int V) {
    if (V < 98304 || V > CAND_WAVES * 256 * SAMPLE_BLOCKS || M > 32) return 0;
    return M <= 8 ? 4 : (M <= 24 ? 2 : 1);
}

extern "C" long long ra_sample_scratch(int M, int V) {
    return M > 0 && sample_parts(M, V) ? (long long)M * (long long)sample_ws(nullptr, V).row_bytes : 0;
}

// path (may be nullptr): per row 0 = no threshold was needed, 1 = thresholds and draw from the list of the
// largest logits, 2 = by passes over the whole row. ws: ra_sample_scratch bytes, 16-byte aligned (nullptr: one block
// a row).
extern "C" int ra_sample_traced(const float* logits, int M, int V, const float* temperature,
                                const int* top_k, const float* top_p, const float* u, int* out, int* path,
                                char* ws, long long ws_bytes, void* stream) {
    if (M <= 0) return RA_OK;
    if (V <= 0) return RA_ERR_ARG;
    const size_t lds = (size_t)2 * CAND_WAVES * CAND_PER_WAVE * sizeof(float) + SEARCH_BUCKETS * sizeof(fixed_t);   // 80 KB
    static bool allowed = false;
    if (!allowed) {
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(sample_kernel<false>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds) != hipSuccess ||
            hipFuncSetAttribute(reinterpret_cast<const void*>(sample_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)lds) != hipSuccess)
            return RA_ERR_ARG;
        allowed = true;
    }
    hipStream_t s = (hipStream_t)stream;
    const SampleWs w = sample_ws(ws, V);
    const int parts = ws ? sample_parts(M, V) : 0;
    if (parts == 0) {
        hipLaunchKernelGGL(sample_kernel<false>, dim3(M), dim3(SAMPLE_THREADS), lds, s, logits, V, temperature, top_k, top_p,
                           u, out, path, w, 0);
        return ra_launch_status();
    }
    if (ws_bytes < (long long)M * (long long)w.row_bytes || (reinterpret_cast<uintptr_t>(ws) & 15) != 0) return RA_ERR_ARG;
    const dim3 grid(CAND_WAVES * parts, M), block(PART_THREADS);
    hipLaunchKernelGGL(sample_top_kernel, grid, block, 0, s, logits, V, w, parts);
    hipLaunchKernelGGL(sample_span_kernel, grid, block, 0, s, logits, V, temperature, top_k, top_p, w, parts);
    hipLaunchKernelGGL(sample_gather_kernel, grid, block, 0, s, logits, V, temperature, top_k, top_p, w, parts);
    hipLaunchKernelGGL(sample_settle_kernel, dim3(M), dim3(SAMPLE_THREADS), 0, s, V, temperature, top_k, top_p, w, parts);
    hipLaunchKernelGGL(sample_masses_kernel, grid, block, 0, s, logits, V, temperature, w, parts);
    hipLaunchKernelGGL(sample_kernel<true>, dim3(M), dim3(SAMPLE_THREADS), lds, s, logits, V, temperature, top_k, top_p,
                       u, out, path, w, parts);
    return ra_launch_status();
}

extern "C" int ra_sample(const float* logits, int M, int V, const float* temperature,
                         const int* top_k, const float* top_p, const float* u, int* out,
                         void* stream) {
    return ra_sample_traced(logits, M, V, temperature, top_k, top_p, u, out, nullptr, nullptr, 0, stream);
}
