// kvc_v_small_heads.hip -- p.V for head sizes of which a tile of 64 channels can touch more than two heads (8, 16, 24, 40).
//
//   kvc_v_small_heads_kernel<REP, SOFTMAX>   <- v_huffman_decode_and_mat_vec_mul (kvcomp_cuda_extension/src/kernels.cu:778-861)
//
// The fused V kernels keep operand tables for the two heads a tile may straddle; with three and more they would multiply the
// rest by the wrong weights.  Here every lane owns a channel and looks its own head's weights up, so any head size is right.
// Heads this small are rare, so the kernel is plain: payload staged whole, symbols decoded with the two-step decoder's loops,
// weights read where they lie (a tile's few score rows stay in the first-level cache).  It is bound by the latency of those
// loads: batch 2 x 32 heads x 40 x 4096 tokens 24.0 us, x 16 21.7 us; 14.7 us for heads of 48 on the matrix-core kernel.
#include "kvc_fused_common.h"

// (softmax weights relative to the maximum of the 128-token group and query head, as in the other V kernels; the group's
// maximum and sum go to ml from the lane of the head's first channel)
template <int REP, bool SOFTMAX>
__global__ void __launch_bounds__(KVC_WG) kvc_v_small_heads_kernel(KvcFusedArgs a)
{
    __shared__ uint32_t s_lut[KVC_LUT_NARROW_OFFSET];
    __shared__ __align__(16) uint32_t s_stage[KVC_WAVES_PER_WG][KVC_STAGE_WORDS];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row = blockIdx.y, col = blockIdx.x * KVC_WAVES_PER_WG + wave;
    const int64_t cb = a.s.rows_per_codebook ? row / a.s.rows_per_codebook : 0;
    kvc_load_lut(a.s.luts + cb * KVC_LUT_WORDS, s_lut, tid);
    __syncthreads();
    if (col >= a.s.cols) return;
    uint32_t *stage = s_stage[wave];
    uint32_t pos = kvc_stage_tile(a.s, (int64_t)row * a.s.cols + col, stage, lane);
    kvc_wave_sync();
    const int D = a.head_dim, c = col * KVC_WAVE + lane, bh = c / D, d = c - bh * D;
    const int b = bh / a.kv_heads, h = bh - b * a.kv_heads;
    const int64_t t0 = (int64_t)row * KVC_V_TOKENS, hq0 = (int64_t)b * a.q_heads + (int64_t)h * REP;
    // group of (token, batch entry, head): token * per + own
    const int64_t per = a.quant_mask == KVC_MASK_V_TOKEN ? 1 : a.quant_mask == KVC_MASK_SIM_TOKEN ? a.batch : (int64_t)a.batch * a.kv_heads;
    const int64_t g0 = t0 * per + (a.quant_mask == KVC_MASK_V_TOKEN ? 0 : a.quant_mask == KVC_MASK_SIM_TOKEN ? b : bh);
    const float *scores[REP];
    const __half *weights[REP];
    float top[REP], sum[REP], acc[REP];
#pragma unroll
    for (int r = 0; r < REP; r++) {
        scores[r] = a.scores + (hq0 + r) * a.scores_stride + t0;
        weights[r] = a.x + (hq0 + r) * a.tokens + t0;
        top[r] = -INFINITY;
        sum[r] = acc[r] = 0.f;
        if (SOFTMAX)
            for (int i = 0; i < KVC_V_TOKENS; i++) top[r] = fmaxf(top[r], scores[r][i] * a.sm_scale);
    }
    auto emit = [&](int i, uint32_t sym) {
        const int64_t g = g0 + i * per;
        const __half scale = a.scale[g];
        const float value = a.rounded ? __half2float(__hmul(__float2half_rn((float)((int)sym + a.min_i8[g])), scale))
                                      : (float)((int)sym + a.min_i8[g]) * __half2float(scale);
#pragma unroll
        for (int r = 0; r < REP; r++) {
            const float w = SOFTMAX ? __expf(scores[r][i] * a.sm_scale - top[r]) : __half2float(weights[r][i]);
            if (SOFTMAX) sum[r] += w;
            acc[r] = fmaf(value, w, acc[r]);
        }
    };
    kvc_dispatch_group(s_lut, [&]<int G, bool S>() { kvc_decode_run<G, S>(stage, pos, s_lut, KVC_V_TOKENS, emit); });
#pragma unroll
    for (int r = 0; r < REP; r++) {
        const int64_t hq = (int64_t)row * a.batch * a.q_heads + hq0 + r, o = hq * D + d;
        if (a.out_f32) reinterpret_cast<float *>(a.out)[o] = acc[r];
        else reinterpret_cast<__half *>(a.out)[o] = __float2half_rn(acc[r]);
        if (SOFTMAX && d == 0) {
            a.ml[2 * hq] = top[r];
            a.ml[2 * hq + 1] = sum[r];
        }
    }
}

int kvc_launch_v_small_heads(int rep, const KvcFusedArgs &a, int64_t rows, hipStream_t stream)
{
    const dim3 grid((unsigned)((a.s.cols + KVC_WAVES_PER_WG - 1) / KVC_WAVES_PER_WG), (unsigned)rows);
#define KVC_LAUNCH(R, SM) hipLaunchKernelGGL((kvc_v_small_heads_kernel<R, SM>), grid, dim3(KVC_WG), 0, stream, a)
    if (a.scores) {
        switch (rep) {
            case 1: KVC_LAUNCH(1, true); break;
            case 2: KVC_LAUNCH(2, true); break;
            case 4: KVC_LAUNCH(4, true); break;
            default: KVC_LAUNCH(8, true); break;
        }
    } else {
        switch (rep) {
            case 1: KVC_LAUNCH(1, false); break;
            case 2: KVC_LAUNCH(2, false); break;
            case 4: KVC_LAUNCH(4, false); break;
            default: KVC_LAUNCH(8, false); break;
        }
    }
#undef KVC_LAUNCH
    return kvc_check_hip(hipGetLastError(), "kvc_v_small_heads_kernel launch");
}
