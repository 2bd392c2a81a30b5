// kvc_attend_waves.hip -- decode attention of caches that fill the chip: a 128-token group of a head by one wave (no counterpart
// in the reference, whose models decompress everything; models/cache/kvcomp_quant.py:74-75).
//
// With the short loop for codes of 6 or 7 bits (kvc_mfma_dot's BYTE) the two kernels wait for the LDS: a tile of 64 streams x 128
// symbols costs it some 1050 cycles (look-ups among 64 words 540, parameters 140, refills 110, operand columns 75, staging) and
// takes 890 vector instructions, and a wave spends as long on its tables, its first loads and its operands as on a tile.  Here a
// wave decodes two tiles at a time, a step of each in turn: the two K tiles of a group share q, its two V tiles share weights and
// parameters as well, so a group costs the LDS a fifth less; the wave's set-up serves four tiles; V's payload arrives while K is
// decoded; scores stay in the wave's LDS; and the two chains of look-ups cover each other's round trips, so four waves per
// SIMD, which may then hold 128 registers, keep as many look-ups going as eight did.
#include "kvc_attend.h"
#include "kvc_fused_mfma_impl.h"

constexpr int KVC_WAVES_TILES = 2;                 // tiles of K, and of V, in a group: head_dim 128
constexpr int KVC_WAVES_TAB_WORDS = (1 << KVC_LUT_ESC_BITS) / 2;

struct KvcAttendWavesArgs {
    KvcFusedArgs k, v;
    int k_bits, v_bits;      // longest codes, as the caller knows them
    int groups, group_wgs;   // a group per wave; workgroups behind those take K tiles behind the last group
    int heads_per_wg;        // 2: the waves take the groups of one head after the other, head by head; 1: a workgroup's are of one head
    int k_rows;
    int k_rows_lds, v_rows_lds;   // words of a stream that the LDS holds
    int area_words;          // LDS of a wave's payloads
};

// kvc_mfma_dot's BYTE loop over two tiles at a time.  ms_step: bytes between the tiles' parameters, 0 where they share them.
template <int NM>
__device__ __forceinline__ void kvc_mfma_dot_two(const uint32_t (&column)[2], uint32_t (&u)[2], uint32_t fe, uint32_t mask, int n,
                                                 uint32_t bptr, uint32_t msptr, uint32_t ms_step, kvc_f4 (&acc)[2][NM])
{
    asm volatile("" : "+v"(mask), "+v"(msptr));        // mask: in a vector register, mask and offset then are one instruction
#pragma unroll 1
    for (int i = 0; i < n; i += 8) {
        uint32_t lo[2], hi[2], R[2], es[2], e[2][8];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const kvc_lds_word *wp = (const kvc_lds_word *)(uintptr_t)kvc_column_address(column[t], u[t]);
            const uint32_t w0 = wp[0], w1 = wp[64], w2 = wp[128];
            lo[t] = __builtin_amdgcn_alignbit(w1, w0, u[t]);
            hi[t] = __builtin_amdgcn_alignbit(w2, w1, u[t]);
            R[t] = lo[t];
            es[t] = 0;
        }
        kvc_static_for<8>([&](auto g_) {
            constexpr int g = decltype(g_)::value;
#pragma unroll
            for (int t = 0; t < 2; t++) {
                if (g == 4) R[t] = __builtin_amdgcn_alignbit(hi[t], lo[t], es[t]);       // at most 28 bits so far
                e[t][g] = *(const kvc_lds_u16 *)(uintptr_t)((R[t] & mask) | fe);
            }
#pragma unroll
            for (int t = 0; t < 2; t++) {
                if (g != 3 && g != 7) R[t] = __builtin_amdgcn_alignbit(R[t], R[t], e[t][g]);
                es[t] += e[t][g];
            }
            if constexpr (g % 4 == 3) {
                constexpr int q = g / 4;
                kvc_w2 cols[NM];
#pragma unroll
                for (int s = 0; s < NM; s++) cols[s] = kvc_read_columns<true, true>(bptr + (q * NM + s) * 32, true);
                kvc_w4 ms = *(const kvc_lds_w4 *)(uintptr_t)(msptr + q * 16);
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    if (t == 1 && ms_step) ms = *(const kvc_lds_w4 *)(uintptr_t)(msptr + ms_step + q * 16);
                    const uint32_t a01 = kvc_dequant_pair(kvc_pack_byte1(e[t][g - 3], e[t][g - 2]), ms.x, ms.z);
                    const uint32_t a23 = kvc_dequant_pair(kvc_pack_byte1(e[t][g - 1], e[t][g]), ms.y, ms.w);
#pragma unroll
                    for (int s = 0; s < NM; s++) acc[t][s] = kvc_mfma4<true>(a01, a23, cols[s], acc[t][s]);
                }
            }
        });
        u[0] += es[0] & 0xffu;
        u[1] += es[1] & 0xffu;
        bptr += 2 * NM * 32;
        msptr += 32;
    }
}

// A tile's sums of one query head: register i of lane 4 b + j, j even, holds those of stream 4 b + i for query head 2 set + j / 2
__device__ __forceinline__ kvc_f4 kvc_waves_sums(kvc_f4 acc, bool lo_used)
{
    kvc_f4 res = acc;
    if (lo_used) {
#pragma unroll
        for (int i = 0; i < 4; i++) res[i] = fmaf(kvc_quad_next(acc[i]), 1.f / KVC_LO_SCALE, acc[i]);
    }
    return res;
}

template <int REP>
__global__ void __launch_bounds__(KVC_WG, REP == 8 ? 3 : 4) kvc_attend_waves_kernel(KvcAttendWavesArgs j)
{
    constexpr int NM = kvc_mfma_sets(REP), T = KVC_WAVES_TILES;
    constexpr int COLS = KvcMfmaTables<REP>::BTAB_SLOT_WORDS, MS = KvcMfmaTables<REP>::MSTAB_SLOT_WORDS;
    // dynamic LDS: K's table at offset 0, V's; per wave two payloads (then the scores [REP][128] in their place, then the columns of
    // V's weights before V's payloads); per wave the parameters of two tiles; q's columns (one head per workgroup)
    // (LDS by its byte addresses: pointers that pass through arrays or selects become generic ones, whose stores wait for the loads in
    // flight)
    extern __shared__ __align__(16) uint32_t smem[];
    uint32_t *vtab = smem + KVC_WAVES_TAB_WORDS;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t area = kvc_lds_addr(smem) + 4u * (2 * KVC_WAVES_TAB_WORDS + wave * j.area_words);
    uint32_t *ms = vtab + KVC_WAVES_TAB_WORDS + KVC_WAVES_PER_WG * j.area_words + wave * (T * MS);
    uint32_t *qcols = vtab + KVC_WAVES_TAB_WORDS + KVC_WAVES_PER_WG * (j.area_words + T * MS);
    const int heads = j.k.s.cols, D = KVC_WAVE * T;
    const bool whole = (int)blockIdx.x < j.group_wgs;
    // this wave's head and group; or (the second of the wave's two tiles is the first once more) K tiles behind the last group, row-major
    int bh, g, first_bh;
    if (!whole) {
        const int unit = ((int)blockIdx.x - j.group_wgs) * KVC_WAVES_PER_WG + wave;
        g = unit / heads;                                                    // (row behind the groups)
        bh = first_bh = unit - g * heads;
    } else if (j.heads_per_wg == 2) {
        const int unit = (int)blockIdx.x * KVC_WAVES_PER_WG;
        first_bh = unit / j.groups;
        g = unit - first_bh * j.groups + wave;
        bh = first_bh;
        if (g >= j.groups) g -= j.groups, bh++;                              // (at least three groups)
    } else {
        const int quad = (int)blockIdx.x / heads;
        bh = first_bh = (int)blockIdx.x - quad * heads;
        g = quad * KVC_WAVES_PER_WG + wave;
    }
    const int row0 = whole ? T * g : T * j.groups + g, row_step = whole ? 1 : 0;
    const bool active = whole ? g < j.groups && bh < heads : row0 < j.k_rows;
    if (bh >= heads) bh = heads - 1;
    // ---- everything whose address is known: block_infos, headers, one-symbol entries, q
    uint32_t k_off[T], k_bn[T], v_off[T], v_bn[T], k_ti[T], v_ti[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        k_off[t] = k_bn[t] = v_off[t] = v_bn[t] = k_ti[t] = v_ti[t] = 0;
        if (!active) continue;
        int64_t tile = (int64_t)(row0 + t * row_step) * heads + bh;
        const uint32_t *bi = reinterpret_cast<const uint32_t *>(j.k.s.block_infos + 8 * tile);
        k_off[t] = bi[0];
        k_bn[t] = bi[1];
        k_ti[t] = kvc_load_at<uint16_t>(j.k.s.thread_infos + tile * KVC_WAVE, 2u * (uint32_t)lane);
        if (!whole) continue;
        tile = (int64_t)g * j.v.s.cols + bh * T + t;
        bi = reinterpret_cast<const uint32_t *>(j.v.s.block_infos + 8 * tile);
        v_off[t] = bi[0];
        v_bn[t] = bi[1];
        v_ti[t] = kvc_load_at<uint16_t>(j.v.s.thread_infos + tile * KVC_WAVE, 2u * (uint32_t)lane);
    }
    const uint32_t *__restrict__ lut_k = j.k.s.luts, *__restrict__ lut_v = j.v.s.luts;
    const uint32_t kb = (uint32_t)j.k_bits, vb = (uint32_t)j.v_bits;                      // 1 .. 7
    {
        const uint32_t i = (uint32_t)tid & 127u, bits = tid < 128 ? kb : vb;
        const uint32_t *lut = tid < 128 ? lut_k : lut_v;
        if (i < (1u << bits)) {
            const uint32_t e = lut[KVC_LUT_FENTRY_OFFSET + i], len = (e & 0xffu) > bits ? bits : (e & 0xffu);
            reinterpret_cast<uint16_t *>(tid < 128 ? smem : vtab)[i] =
                (uint16_t)(__half_as_ushort(__float2half_rn(__uint_as_float(e & 0xffffff00u) - (float)KVC_BYTE_CENTRE)) | len);
        }
    }
    const bool k_fast = lut_k[0] == kb && lut_k[1] == kb && lut_k[2] == 0u && (lut_k[6] & KVC_LUT_WIDE_SYMBOLS) == 0u;
    const bool v_fast = lut_v[0] == vb && lut_v[1] == vb && lut_v[2] == 0u && (lut_v[6] & KVC_LUT_WIDE_SYMBOLS) == 0u;
    // q's columns: as loaded, high parts only, unless one of the weights is subnormal (kvc_mfma_stage_ops)
    const int b = bh / j.k.kv_heads, h = bh - b * j.k.kv_heads;
    bool q_lo;
    {
        uint32_t x[REP];
        bool subnormal = false;
#pragma unroll
        for (int r = 0; r < REP; r++) {
            x[r] = kvc_load_at<uint32_t>(j.k.x + ((int64_t)b * j.k.q_heads + h * REP + r) * D, 4u * (uint32_t)lane);
            const kvc_h2 w = __builtin_bit_cast(kvc_h2, x[r]);
            subnormal = subnormal | __builtin_amdgcn_classh(w.x, 0x90) | __builtin_amdgcn_classh(w.y, 0x90);
        }
        q_lo = __any(subnormal);
        // a head's first wave writes its columns (behind the groups every wave has a head of its own: they lie where its second payload
        // would)
        if (!whole) qcols = vtab + KVC_WAVES_TAB_WORDS + wave * j.area_words + 64 * j.k_rows_lds;
        else if (bh != first_bh) qcols += COLS;
        const bool mine = !whole || wave == 0 || (bh != first_bh && g == 0);
        uint32_t *bg = qcols + (lane >> 1) * (NM * 8) + (lane & 1);
#pragma unroll
        for (int r = 0; r < 2 * NM; r++) {                                                // (a column pair no query head owns: zeros)
            if (!mine) break;
            uint32_t hi = r < REP ? x[r < REP ? r : 0] : 0u, low = 0u;
            if (q_lo && r < REP) {
                float h0, l0, h1, l1;
                kvc_split_weight(kvc_half_bits_to_float(hi & 0xffffu), h0, l0);
                kvc_split_weight(kvc_half_bits_to_float(hi >> 16), h1, l1);
                hi = kvc_half_pair(h0, h1);
                low = kvc_half_pair(l0, l1);
            }
            bg[(((2 * r) >> 2) * 4 + ((2 * r) & 3)) * 2] = hi;
            bg[(((2 * r + 1) >> 2) * 4 + ((2 * r + 1) & 3)) * 2] = low;
        }
    }
    KvcRaw<REP, 1, 1> raw[T];
    KvcStreams st[T], st_v[T];
    KvcTilePos pos = {0, bh, b, h, 0};
    if (active) {
#pragma unroll
        for (int t = 0; t < T; t++) {
            pos.row = row0 + t * row_step;
            kvc_fetch_tile<REP, 0, 2, false, false>(j.k, pos, k_off[t], k_bn[t], lane, raw[t]);
            raw[t].ti_cur = k_ti[t];
            st[t] = kvc_fetch_streams(j.k, lane, j.k_rows_lds, 1u, raw[t]);
        }
    }
    __syncthreads();
    if (!active) return;
    // ---- K
    uint32_t column[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        column[t] = area + (whole ? 256u * t * j.k_rows_lds : 0u) + 4u * lane;
        kvc_stage_streams(j.k, lane, j.k_rows_lds, raw[t], st[t], column[t]);
        uint32_t mins, scales;
        kvc_mfma_min_scale_words(raw[t], 0, kvc_pair_mode<0>(j.k), mins, scales, KVC_BYTE_CENTRE);
        uint32_t *mg = ms + t * MS + (lane >> 1) * 4 + (lane & 1);
        mg[0] = mins;
        mg[2] = scales;
    }
    const bool k_loop = k_fast && st[0].fits && st[1].fits;
    if (!k_loop) {
#pragma unroll
        for (int t = 0; t < T; t++) kvc_stream_in_memory(j.k, lane, raw[t], st[t]);
    }
    if (whole) {                                                                          // V's loads fly while K is decoded
        int lane_f = lane;
        asm volatile("" : "+v"(lane_f));
#pragma unroll
        for (int t = 0; t < T; t++) {
            const KvcTilePos pv = {g, bh * T + t, b, h, t * KVC_WAVE};
            kvc_fetch_tile<REP, 1, 2, false, false>(j.v, pv, v_off[t], v_bn[t], lane_f, raw[t]);
            raw[t].ti_cur = v_ti[t];
            st_v[t] = kvc_fetch_streams(j.v, lane_f, j.v_rows_lds, 1u, raw[t]);
        }
    }
    kvc_wave_sync();
    const int rows4 = (lane >> 2) * 4, cj = lane & 3;
    kvc_f4 acc[T][NM];
    auto decode = [&](uint32_t fe, uint32_t bits, uint32_t cols, uint32_t ms_step) {
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int s = 0; s < NM; s++) acc[t][s] = kvc_f4{0.f, 0.f, 0.f, 0.f};
        uint32_t u[2] = {st[0].u0, st[1].u0};
        const uint32_t mask = ((1u << bits) - 1u) << 1, bptr = cols + cj * 8, msptr = kvc_lds_addr(ms);
        kvc_mfma_dot_two<NM>(column, u, fe, mask, 128, bptr, msptr, ms_step, acc);
    };
    // one symbol at a time: tables that are not what the caller said, tiles that do not fit the LDS
    auto decode_slow = [&](int t, const uint32_t *lut, const uint32_t *cols, const uint32_t *params) {
        return kvc_mfma_slow_tile<REP, true, true>(st[t].gwords, st[t].gnwords, st[t].gpos, lut, 128, cols, params, 0u, KVC_BYTE_CENTRE);
    };
    typedef __attribute__((address_space(3))) float lds_float;
    lds_float *const scores = (lds_float *)(uintptr_t)area;
    float *const out_scores = reinterpret_cast<float *>(j.k.out) + ((int64_t)b * j.k.q_heads + h * REP) * j.k.out_stride + (int64_t)row0 * KVC_WAVE;
    if (k_loop) {
        decode(0u, kb, kvc_lds_addr(qcols), MS * 4);
        kvc_wave_sync();                                                                  // scores take the place of what was decoded
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int s = 0; s < NM; s++) {
                const int r = 2 * s + (cj >> 1);
                const kvc_f4 res = kvc_waves_sums(acc[t][s], q_lo);
                if ((cj & 1) != 0 || r >= REP) continue;
                if (whole) *(__attribute__((address_space(3))) kvc_f4 *)(scores + r * KVC_V_TOKENS + t * KVC_WAVE + rows4) = res;
                else if (t == 0) *reinterpret_cast<kvc_f4 *>(out_scores + r * j.k.out_stride + rows4) = res;
            }
    } else {
        KvcVec<REP> res[T];
#pragma unroll
        for (int t = 0; t < T; t++) res[t] = decode_slow(t, lut_k, qcols, ms + t * MS);
        kvc_wave_sync();
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int r = 0; r < REP; r++) {
                if (whole) scores[r * KVC_V_TOKENS + t * KVC_WAVE + lane] = res[t].v[r];
                else if (t == 0) out_scores[r * j.k.out_stride + lane] = res[t].v[r];
            }
    }
    if (!whole) return;
    kvc_wave_sync();
    // ---- softmax weights of the group; lane: tokens 2 lane and 2 lane + 1
    float s0[REP], s1[REP];
#pragma unroll
    for (int r = 0; r < REP; r++) {
        s0[r] = scores[r * KVC_V_TOKENS + 2 * lane];
        s1[r] = scores[r * KVC_V_TOKENS + 2 * lane + 1];
    }
    kvc_wave_sync();
    kvc_lds_u32 *const cols = (kvc_lds_u32 *)(uintptr_t)area;
#pragma unroll
    for (int r = 0; r < 2 * NM; r++) {
        kvc_lds_u32 *bg = cols + (lane >> 1) * (NM * 8) + (lane & 1);
        uint32_t hi = 0u, low = 0u;
        if (r < REP) {
            const float a0 = s0[r < REP ? r : 0] * j.v.sm_scale, a1 = s1[r < REP ? r : 0] * j.v.sm_scale;
            const float m = kvc_wave_fmax_dpp(fmaxf(a0, a1));
            const float w0 = __expf(a0 - m), w1 = __expf(a1 - m);
            const float l = kvc_wave_sum_dpp(w0 + w1);
            if (lane == 0) *reinterpret_cast<float2 *>(j.v.ml + 2 * (((int64_t)g * heads + bh) * REP + r)) = make_float2(m, l);
            float h0, l0, h1, l1;
            kvc_split_weight(w0, h0, l0);
            kvc_split_weight(w1, h1, l1);
            hi = kvc_half_pair(h0, h1);
            low = kvc_half_pair(l0, l1);
        }
        bg[(((2 * r) >> 2) * 4 + ((2 * r) & 3)) * 2] = hi;
        bg[(((2 * r + 1) >> 2) * 4 + ((2 * r + 1) & 3)) * 2] = low;
    }
    // ---- V
    {
        int lane_s = lane;
        asm volatile("" : "+v"(lane_s));
        uint32_t mins, scales;
        kvc_mfma_min_scale_words(raw[0], 0, kvc_pair_mode<1>(j.v), mins, scales, KVC_BYTE_CENTRE);
        uint32_t *mg = ms + (lane_s >> 1) * 4 + (lane_s & 1);
        mg[0] = mins;
        mg[2] = scales;
#pragma unroll
        for (int t = 0; t < T; t++) {
            column[t] = area + 4u * COLS + 256u * t * j.v_rows_lds + 4u * lane_s;
            st[t] = st_v[t];
            kvc_stage_streams(j.v, lane_s, j.v_rows_lds, raw[t], st[t], column[t]);
        }
    }
    kvc_wave_sync();
    float *out = reinterpret_cast<float *>(j.v.out) + (((int64_t)g * j.v.batch + b) * j.v.q_heads + h * REP) * D;
    if (v_fast && st[0].fits && st[1].fits) {
        decode(kvc_lds_addr(vtab), vb, area, 0u);
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int s = 0; s < NM; s++) {
                const int r = 2 * s + (cj >> 1);
                const kvc_f4 res = kvc_waves_sums(acc[t][s], true);
                if ((cj & 1) == 0 && r < REP) *reinterpret_cast<kvc_f4 *>(out + r * D + t * KVC_WAVE + rows4) = res;
            }
    } else {
#pragma unroll
        for (int t = 0; t < T; t++) {
            kvc_stream_in_memory(j.v, lane, raw[t], st[t]);
            const KvcVec<REP> res = decode_slow(t, lut_v, smem + (area - kvc_lds_addr(smem)) / 4u, ms);
#pragma unroll
            for (int r = 0; r < REP; r++) out[r * D + t * KVC_WAVE + lane] = res.v[r];
        }
    }
}

KvcWavesPlan kvc_plan_attend_waves(const kvc_compressed_desc *k, const kvc_compressed_desc *v, int64_t rep, int64_t bh)
{
    KvcWavesPlan p = {};
    const int64_t groups = v->tokens / KVC_V_TOKENS, k_rows = k->tokens / KVC_WAVE;
    p.k_only = (k_rows - KVC_WAVES_TILES * groups) * bh;
    const int cols = KVC_MFMA_GROUPS * kvc_mfma_sets((int)rep) * 8, ms = KVC_MFMA_GROUPS * 4;
    p.k_rows_lds = kvc_stream_rows(k->max_stream_bytes, k->encoded_bytes, k_rows * bh);
    p.v_rows_lds = kvc_stream_rows(v->max_stream_bytes, v->encoded_bytes, groups * bh * KVC_WAVES_TILES);
    const int k_area = KVC_WAVES_TILES * 64 * p.k_rows_lds, v_area = cols + KVC_WAVES_TILES * 64 * p.v_rows_lds;
    p.area_words = k_area > v_area ? k_area : v_area;
    if (p.area_words < (int)rep * KVC_V_TOKENS) p.area_words = (int)rep * KVC_V_TOKENS;
    if (p.k_only > 0 && p.area_words < 64 * p.k_rows_lds + cols) p.area_words = 64 * p.k_rows_lds + cols;
    // the last wave's second payload, and what a corrupt one may lead to
    int least = 2 * KVC_WAVES_TAB_WORDS + (KVC_WAVES_PER_WG - 1) * p.area_words + 64 * KVC_COLUMN_REACH;
    least += cols + 64 * p.v_rows_lds > 64 * p.k_rows_lds ? cols + 64 * p.v_rows_lds : 64 * p.k_rows_lds;
    auto bytes = [&](int heads) {
        const int words = 2 * KVC_WAVES_TAB_WORDS + KVC_WAVES_PER_WG * (p.area_words + KVC_WAVES_TILES * ms) + heads * cols;
        return 4 * (size_t)(words < least ? least : words);
    };
    auto workgroups = [&](size_t lds) {
        const int n = lds > 65536 ? 0 : kvc_lds_workgroups(lds), most = rep == 8 ? 3 : 4;       // by their registers
        return n < most ? n : most;
    };
    // A workgroup across two heads leaves no wave without a group, and takes room for the columns of two: where the groups are no
    // multiple of four, unless it costs a compute unit a workgroup.  3 x 24 heads x 14 464 tokens (113 groups) 79.1 -> 71 us
    const bool two_heads = groups % KVC_WAVES_PER_WG != 0 && groups >= KVC_WAVES_PER_WG - 1 && workgroups(bytes(2)) == workgroups(bytes(1));
    p.heads_per_wg = two_heads ? 2 : 1;
    p.group_wgs = two_heads ? (groups * bh + KVC_WAVES_PER_WG - 1) / KVC_WAVES_PER_WG : (groups + KVC_WAVES_PER_WG - 1) / KVC_WAVES_PER_WG * bh;
    p.lds = bytes(p.heads_per_wg);
    p.per_cu = workgroups(p.lds);
    return p;
}

int kvc_attend_waves(const KvcFusedArgs &k, const KvcFusedArgs &v, const kvc_compressed_desc *kd, const kvc_compressed_desc *vd, const KvcWavesPlan &p,
                     int64_t rep, hipStream_t stream)
{
    KvcAttendWavesArgs j = {};
    j.k = k;
    j.v = v;
    j.k_bits = kvc_hint_bits(kd->max_code_bits);
    j.v_bits = kvc_hint_bits(vd->max_code_bits);
    j.groups = (int)(vd->tokens / KVC_V_TOKENS);
    j.k_rows = (int)(kd->tokens / KVC_WAVE);
    j.k_rows_lds = p.k_rows_lds;
    j.v_rows_lds = p.v_rows_lds;
    j.area_words = p.area_words;
    j.heads_per_wg = p.heads_per_wg;
    j.group_wgs = (int)p.group_wgs;
    const size_t lds = p.lds;
    const unsigned grid = (unsigned)(p.group_wgs + (p.k_only + KVC_WAVES_PER_WG - 1) / KVC_WAVES_PER_WG);
    static const bool trace_plan = getenv("KVCOMP_TRACE_PLAN") != nullptr;
    if (trace_plan)
        fprintf(stderr, "[kvcomp] attention by waves rep %d: %u workgroups (%d of whole groups), lds %zu B (codes %d / %d bits, rows %d / %d)\n",
                (int)rep, grid, j.group_wgs, lds, j.k_bits, j.v_bits, j.k_rows_lds, j.v_rows_lds);
    if (rep == 1) hipLaunchKernelGGL(kvc_attend_waves_kernel<1>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    else if (rep == 2) hipLaunchKernelGGL(kvc_attend_waves_kernel<2>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    else if (rep == 4) hipLaunchKernelGGL(kvc_attend_waves_kernel<4>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    else hipLaunchKernelGGL(kvc_attend_waves_kernel<8>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    KVC_HIP(hipGetLastError());
    return 0;
}
