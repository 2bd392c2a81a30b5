// kvc_attend.h -- decode attention with one launch for K and V: a workgroup per 128-token group of a head in small caches
// (kvc_attend.hip), a wave per group in those that fill the chip (kvc_attend_waves.hip).
#pragma once
#include "kvc_common.h"

// Workgroups (128-token groups x KV heads x batch entries) up to which the joint kernel is taken, by query heads per KV head.
// Beyond, the chip is full of waves either way, and the two kernels, whose waves hold fewer registers and no tables of both
// streams, are as fast or faster.  Two kernels against this one in us, head_dim 128 / 64:
//   1 query head    1024 workgroups 27.2 : 20.7 / 23.5 : 17.2    1536 29.8 : 30.0 / 24.8 : 24.0    2048 34.1 : 34.1 / 25.8 : 25.9
//   4 query heads   1536            36.8 : 34.8 / 30.4 : 28.6    2048 41.3 : 40.5 / 32.4 : 31.9    3072 58.5 : 58.0 / 41.2 : 45.4
//   8 query heads   2048            70.5 : 48.6 / 47.0 : 37.7    3072 81.8 : 72.0 / 54.8 : 53.8
constexpr int64_t kvc_attend_max_wgs(int64_t rep) { return rep <= 2 ? 1536 : rep == 4 ? 2048 : 3072; }
// ... and from which a wave takes a group by itself (head_dim 128, codes of 6 or 7 bits of symbols up to 16).  Two kernels, the joint
// kernel and this one in us, per decode attention call:
//   1 query head    1536 groups 28 : 29 : 30    2048 31.5 : 31.9 : 31.2    4096 49.7 : 55.6 : 43.1    8192  79 : 94 : 71
//   4 query heads   1536        34 : 33 : 34    2048 38.2 : 38.1 : 35.1    4096 61.1 : 65.8 : 48.9    8192  96 : 118 : 81
//   8 query heads   1536        46 : 42 : 42    2048 61.1 : 48.4 : 43.8    4096 98.2 : 85.1 : 71.9    8192 161 : 155 : 112
constexpr int64_t KVC_ATTEND_WAVES_MIN_WGS = 1536;
// ... and with how many of its workgroups on a compute unit: its LDS is as large as the longest streams of K and V ask for.  This kernel with
// four, three and two (eight query heads: three and two, by their registers) against what else the call would take, us:
//   1 query head    1792 groups 28, 28, 29 : 28   3008 32, 33 : 34       3200 36, 46 : 40       8192 67, 75, 95 : 68
//   2 query heads   1792        26, 27, 28 : 28   3008 32, 32 : 36       3200 37, 47 : 43       8192 66, 74, 96 : 74
//   4 query heads   1984        28, 29, 29 : 31   3008 35, 35, 49 : 46   4096 42, 51, 54 : 54   8192 74, 83, 103 : 87
//   8 query heads   1984        34, 34 : 40       2112 -, 58 : 47       4160 64, 86 : 95
// One less than the registers allow is enough while all waves fit at a time.
constexpr bool kvc_attend_waves_pays(int64_t rep, int64_t groups, int per_cu)
{
    const int enough = rep <= 2 ? 4 : 3;
    return per_cu >= enough || (per_cu == enough - 1 && (groups <= 1024 * per_cu || (rep == 8 && groups > kvc_attend_max_wgs(rep))));
}
constexpr int KVC_ATTEND_K_PAIR_BITS = 6;         // longest code for which K's table of two symbols per look-up is built

struct KvcFusedArgs;
struct KvcWavesPlan {
    int k_rows_lds, v_rows_lds, area_words, heads_per_wg;   // of KvcAttendWavesArgs
    int64_t group_wgs, k_only;   // workgroups of whole groups, K tiles behind the last group
    size_t lds;
    int per_cu;          // workgroups on a compute unit; 0: does not fit
};
KvcWavesPlan kvc_plan_attend_waves(const kvc_compressed_desc *k, const kvc_compressed_desc *v, int64_t rep, int64_t bh);
int kvc_attend_waves(const KvcFusedArgs &k, const KvcFusedArgs &v, const kvc_compressed_desc *kd, const kvc_compressed_desc *vd, const KvcWavesPlan &plan,
                     int64_t rep, hipStream_t stream);

// What takes the whole groups of 128 tokens that V holds compressed, and the K tiles behind them
enum KvcAttendRoute { KVC_ATTEND_SEPARATE = 0, KVC_ATTEND_JOINT = 1, KVC_ATTEND_WAVES = 2 };
KvcAttendRoute kvc_attend_route(const kvc_compressed_desc *k, const kvc_compressed_desc *v, int64_t batch, int64_t kv_heads, int64_t q_heads,
                                int64_t head_dim);
// Partials [groups, B * Hq, D] and their (maximum, sum of weights) of those groups, and the scores of the tokens that only K holds so.
// *taken: false where the call is not one for it (nothing launched).
int kvc_attend_groups(const kvc_compressed_desc *k, const kvc_compressed_desc *v, const void *d_q_f16, float softmax_scale,
                      float *scores, int64_t scores_stride, float *part, float *ml, int64_t batch, int64_t kv_heads, int64_t q_heads,
                      int64_t head_dim, hipStream_t stream, bool *taken);
