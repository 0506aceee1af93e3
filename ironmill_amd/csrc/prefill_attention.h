// prefill_attention.h -- launch of the multi-token attention kernel (prefill_attention.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include "imh_internal.h"

namespace imh {

// Query rows are (token, head of the group) pairs of a kv head.  q: FP16 rows
// [batch][T][nh][128], or the four TurboQuant query planes of each row
// ([row][4][128]).  k / v: f16 rows or code bytes [batch][nkv][max_seq][128].
// Split z covers positions [z split_len, ...); with several splits the
// unnormalised partials go to part_o [row][splits][128], part_m (log2 units)
// and part_l.
struct PrefillAttention {
    const _Float16 *q;
    const uint8_t *k, *v;
    const float *k_scales, *k_rnorm, *v_scales;
    const float *k_codebook, *v_codebook, *signs;
    const int32_t *seq_lens;
    float *part_o, *part_m, *part_l;
    __half *out;
    int T, gqa, nh, nkv, max_seq, seq_len, split_len;
    float attn_scale;
};

// KV splits for `groups` (batch x kv heads x row tiles) over L positions
uint32_t prefill_splits(bool tq, uint32_t groups, uint32_t L, int cus);

// query rows per workgroup
int prefill_row_tile(bool tq);

int launch_prefill_attention(imh_stream *s, bool tq, uint32_t batch, uint32_t splits, const PrefillAttention &a);

// The TurboQuant query planes of `rows` query rows (f16 [row][128]): rotated
// (q) and projected onto the QJL matrix (s), each as f16 hi + lo, planes
// [row][q_hi, q_lo, s_hi, s_lo][128] in the k-slot order {0, 2, 1, 3, 4, 6, 5,
// 7} of the code-byte unpack.
int launch_tq_query_prep(imh_stream *s, const __half *q, size_t rows, const float *signs, const float *qjl_t,
                         _Float16 *planes);

// Merges the splits' partials of each row (maxima in log2 units), normalises
// and, for TurboQuant, rotates back.
int launch_prefill_combine(imh_stream *s, bool tq, size_t rows, uint32_t splits, const float *part_o,
                           const float *part_m, const float *part_l, const float *signs, __half *out);

}  // namespace imh
