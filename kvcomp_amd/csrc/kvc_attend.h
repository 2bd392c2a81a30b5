// kvc_attend.h -- decode attention of small caches, one launch for K and V (kvc_attend.hip).
#pragma once
#include "kvc_common.h"

// Workgroups (128-token groups x KV heads x batch entries) up to which the joint kernel is taken.  Beyond, the chip is full of
// waves either way, and the two kernels, whose waves hold fewer registers and no tables of both streams, are as fast or
// faster.  Two kernels against this one, head_dim 128: 1024 workgroups 26.9 / 20.9 us, 1536 29.6 / 26.4, 2048 33.6 / 34.4,
// 3072 43.6 / 45.0 (one query head per KV head; two and four alike); eight query heads: 1024 41.2 / 30.6, 1536 48.3 / 50.0.
constexpr int64_t KVC_ATTEND_MAX_WGS = 1536, KVC_ATTEND_MAX_WGS_8 = 1024;
constexpr int KVC_ATTEND_K_PAIR_BITS = 6;         // longest code for which K's table of two symbols per look-up is built

// Partials [groups, B * Hq, D] and their (maximum, sum of weights) of all whole groups of 128 tokens that V holds compressed,
// and the scores of the tokens that only K does.  *taken: false where the call is not one for it (nothing launched).
int kvc_attend_groups(const kvc_compressed_desc *k, const kvc_compressed_desc *v, const void *d_q_f16, float softmax_scale,
                      float *scores, int64_t scores_stride, float *part, float *ml, int64_t batch, int64_t kv_heads, int64_t q_heads,
                      int64_t head_dim, hipStream_t stream, bool *taken);
