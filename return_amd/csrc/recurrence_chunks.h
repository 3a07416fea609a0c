// The gated recurrences of delta_rule.hip for requests of several rows, by chunks of rows on the matrix cores.
#pragma once
#include <hip/hip_runtime.h>

// Requests of fewer rows stay with the kernels that walk the rows. Measured, walked / by chunks: rule 0, 32 heads of 128 x 128,
// four requests of 8 rows 25 / 31 us, one of 16 rows 20 / 24, eight of 16 rows 91 / 48; rule 1, 16 heads of 128 x 128, eight of 16
// rows 26 / 27. Rule 2 gains nothing before 24 rows (32 heads of 128 x 64, eight requests of 16 rows 33 / 32 us, of 24 rows
// 58 / 25), and up to there its read-outs are 5 % further from 64 bits by chunks.
__host__ __device__ static inline int rc_min_rows(int rule) { return rule == 2 ? 24 : 16; }

// Floats of scratch that recurrence_chunks_run wants for a step whose requests bring q_lens[0..n_seqs) rows (host
// memory); 0: no request is long enough, or the heads are beyond these kernels.
long long recurrence_chunks_workspace(const int* q_lens, int n_seqs, int H, int D, int V, int rule);

// The recurrence (o_raw and S) of all requests of rc_min_rows rows and more; arguments as in delta_rule_run.
int recurrence_chunks_run(hipStream_t st, const void* qkv, long long ld_qkv, const void* b, long long ld_b, const void* ag,
                          long long ld_ag, const float* A_log, const float* dt_bias, float* S, const int* cu_q,
                          const int* slot_ids, float* o_raw, const int* q_lens, int n_seqs, int H, int G, int D, int V,
                          int rule, float rate, float* ws, long long ws_floats, int dtype);
