// kvc_attend.hip -- decode attention of small caches: scores, softmax and weighted values of a 128-token group in one
// workgroup (no counterpart in the reference, whose models decompress everything; models/cache/kvcomp_quant.py:74-75).
//
// What bounds a small call is a chain, not a rate: a K kernel of one wave per tile (arguments, table, payload: three trips
// to memory; then 128 look-ups in a row, each an LDS round trip and two dependent instructions), and behind it a V kernel
// with the same chain that cannot start before K's scores are there.  Only the weights depend on the scores, though.  Here
// the workgroup of a (batch entry, head, group) decodes its two K tiles and its one or two V tiles at the same time, one
// wave each; the V waves keep their symbols as bytes in 32 registers until the K waves have left the scores in LDS, the four
// waves turn those into softmax weights, and the V waves then multiply: 32 groups of four tokens, one matrix instruction
// each.  Scores of these groups never go to memory.  Calls of (batch x KV heads x query heads per KV head x head_dim, tokens),
// two kernels -> this one, the merge of the groups included: 1 x 8 x 4 x 128, 1000: 28.0 -> 16.5 us; 1 x 32 x 1 x 128, 4096:
// 24.8 -> 18.2; 1 x 32 x 1 x 64, 4096: 21.0 -> 14.6; 1 x 8 x 8 x 128, 3000: 35.3 -> 19.4.
//
// Where a V wave's 21 600 cycles go (clock stamps, 1 x 32 heads x 128 x 1024 tokens, one workgroup per CU): arguments,
// one-symbol tables and the tile's loads 5000, tables, staging and operands 2000, 128 look-ups in a row 11 600 (K alike),
// scores to weights and two barriers 1300, the products 1700.  With four workgroups per CU (4096 tokens) the look-ups take
// 16 600: the waves then share the LDS.
// The operands of K's products and of V's are read by all lanes, without a branch, and V's some groups ahead: with the read
// under the branch that the larger launches use (it saves LDS time) each group of four waited for its own round trip: 1 x 8 x
// 4 x 128, 1000 tokens 19.2 -> 16.5 us.  Registers are given away for that: five waves per SIMD (four with four and eight
// query heads), which is what the LDS leaves room for.
//
// Two symbols per look-up where every pair of codes fits the table (K up to 6 bits, V up to 4): as many look-ups in a row again
// saved.  Tables that hold nearly all pairs of 7-bit codes, with a second look-up for the rest, gain nothing: waiting for
// every look-up's outcome and building 2048 entries cost what the look-ups saved (18.9 -> 19.0 us at 1024 workgroups).
// One symbol at a time, V's entries have two bytes, so that 128 of them are two words per LDS bank: 1024 workgroups 19.1 ->
// 18.2 us.  For K, whose two-byte entries take more instructions to join, it gains 0.3 us there and costs 0.3 to 0.5 below.
#include "kvc_attend.h"
#include "kvc_fused_mfma_impl.h"

typedef uint32_t kvc_w32 __attribute__((ext_vector_type(32)));

constexpr int KVC_ATTEND_VTAB_WORDS = 256;     // two V symbols per look-up for codes of at most 4 bits, else one
constexpr int KVC_ATTEND_V_PAIR_BITS = 4;
constexpr int KVC_ATTEND_TMP_WORDS = 256;      // the one-symbol tables of K and V
constexpr int KVC_ATTEND_K_TILES = KVC_V_TOKENS / KVC_WAVE;

struct KvcAttendArgs {
    KvcFusedArgs k, v;
    int ktab_words;          // a power of two, at least KVC_ATTEND_VTAB_WORDS
    int k_bits, v_bits;      // longest codes, as the caller knows them
    int group_wgs;           // workgroups of whole groups; those after them take K tiles behind the last group, one per wave
    int k_tiles;             // all K tiles
};

// -- V tiles as bytes ------------------------------------------------------------------------------------
// Table entries: {code length(s) | symbol << 8 [| second symbol << 16]}, two bytes each without the second symbol; register i of `vd` holds tokens 4 i .. 4 i + 3.
template <bool PAIRS>
__device__ __forceinline__ void kvc_decode_bytes(uint32_t sbase, uint32_t u, uint32_t fe, uint32_t mask, kvc_w32 &vd)
{
    asm volatile("" : "+v"(mask));                               // in a vector register: mask and offset in one instruction
    constexpr int N = PAIRS ? 4 : 8;                             // look-ups per refill: 8 symbols, half from each half window
#pragma unroll 1
    for (int i = 0; i < KVC_V_TOKENS / 8; i++) {
        const kvc_lds_word *wp = (const kvc_lds_word *)(uintptr_t)kvc_refill_address<false, true>(sbase, u);
        const uint32_t w0 = wp[0], w1 = wp[1], w2 = wp[2];
        const uint32_t lo = __builtin_amdgcn_alignbit(w1, w0, u), hi = __builtin_amdgcn_alignbit(w2, w1, u);
        uint32_t R = lo, es = 0;
        uint32_t e[N];
        kvc_static_for<N>([&](auto p_) {
            constexpr int p = decltype(p_)::value;
            if constexpr (p == N / 2) R = __builtin_amdgcn_alignbit(hi, lo, es);        // at most 28 bits so far
            if constexpr (PAIRS) e[p] = *(const kvc_lds_u32 *)(uintptr_t)((R & mask) | fe);
            else e[p] = *(const kvc_lds_u16 *)(uintptr_t)((R & mask) | fe);
            if constexpr (p != N / 2 - 1 && p != N - 1) R = __builtin_amdgcn_alignbit(R, R, e[p]);
            es += e[p];
        });
        u += es & 0xffu;
        if constexpr (PAIRS) {
            vd[2 * i] = __builtin_amdgcn_perm(e[1], e[0], 0x06050201u);
            vd[2 * i + 1] = __builtin_amdgcn_perm(e[3], e[2], 0x06050201u);
        } else {
            vd[2 * i] = __builtin_amdgcn_perm(e[1], e[0], 0x0c0c0501u) | __builtin_amdgcn_perm(e[3], e[2], 0x05010c0cu);
            vd[2 * i + 1] = __builtin_amdgcn_perm(e[5], e[4], 0x0c0c0501u) | __builtin_amdgcn_perm(e[7], e[6], 0x05010c0cu);
        }
    }
}

// The same one symbol at a time through the generic table and its list of long codes in global memory; words from LDS
// (staged, bit-reversed) or, where the tile did not fit, from global memory.
__device__ __forceinline__ void kvc_decode_bytes_slow(const uint32_t *words, uint32_t nwords, bool staged, uint32_t pos,
                                                      const uint32_t *__restrict__ lut_g, kvc_w32 &vd)
{
    const uint32_t lshift = 32u - lut_g[0], nlong = lut_g[2];
    const uint32_t *longs = lut_g + KVC_LUT_HEADER_WORDS, *entries = longs + KVC_LUT_LONG_WORDS;
#pragma unroll 1
    for (int i = 0; i < KVC_V_TOKENS / 4; i++) {
        uint32_t four = 0;
#pragma unroll 1
        for (int k = 0; k < 4; k++) {
            const uint32_t wi = pos >> 5;
            uint32_t w0 = wi < nwords ? words[wi] : 0u, w1 = wi + 1 < nwords ? words[wi + 1] : 0u;
            w0 = staged ? __brev(w0) : kvc_bswap(w0);
            w1 = staged ? __brev(w1) : kvc_bswap(w1);
            const uint32_t hi = (uint32_t)(((((uint64_t)w0) << 32 | w1) << (pos & 31u)) >> 32);
            const uint32_t e = entries[hi >> lshift];
            uint32_t len = e & 0xffu, sym = (e >> 8) & 0xffu;
            if (len == 0) {
                len = 1;
                sym = 0;
                for (uint32_t j = 0; j < nlong; j++) {
                    const uint32_t ls = longs[2 * j + 1], l = ls & 0xffu;
                    if (((hi ^ longs[2 * j]) >> (32u - l)) == 0u) {
                        len = l;
                        sym = (ls >> 8) & 0xffu;
                        break;
                    }
                }
            }
            four |= sym << (8 * k);
            pos += len;
        }
        vd[i] = four;
    }
}

template <int REP>
__global__ void __launch_bounds__(KVC_WG) __attribute__((amdgpu_waves_per_eu(REP <= 2 ? 5 : 4, REP <= 2 ? 5 : 4))) kvc_attend_group_kernel(KvcAttendArgs j)
{
    constexpr int NM = kvc_mfma_sets(REP);
    using T = KvcMfmaTables<REP>;
    constexpr int K_OPS = kvc_mfma_ops_words(1, REP, true);
    // dynamic LDS: K's table (at offset 0), V's table (both at multiples of their sizes, so that "window bits | offset" is an
    // entry's address), the one-symbol tables, the weights' columns, the group's scores, then the waves' areas
    extern __shared__ __align__(16) uint32_t smem[];
    uint32_t *ktab = smem, *vtab = smem + j.ktab_words, *tmp = vtab + KVC_ATTEND_VTAB_WORDS, *btab_v = tmp + KVC_ATTEND_TMP_WORDS;
    float *s_scores = reinterpret_cast<float *>(btab_v + T::BTAB_SLOT_WORDS);            // [REP][128]
    uint32_t *areas = btab_v + T::BTAB_SLOT_WORDS + REP * KVC_V_TOKENS;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int D = j.k.head_dim;
    const bool whole = (int)blockIdx.x < j.group_wgs;
    const bool is_k = !whole || wave < KVC_ATTEND_K_TILES;
    // ---- everything whose address is known: the wave's block_info, the codebooks' headers and one-symbol entries
    int row, col;
    bool active = true;
    if (whole) {
        const int g = blockIdx.x / j.k.s.cols, bh = blockIdx.x - g * j.k.s.cols, v_tiles = D / KVC_WAVE;
        row = is_k ? g * KVC_ATTEND_K_TILES + wave : g;
        col = is_k ? bh : bh * v_tiles + wave - KVC_ATTEND_K_TILES;
        active = is_k || wave - KVC_ATTEND_K_TILES < v_tiles;
    } else {
        const int t = j.group_wgs * KVC_ATTEND_K_TILES + ((int)blockIdx.x - j.group_wgs) * KVC_WAVES_PER_WG + wave;
        active = t < j.k_tiles;
        row = t / j.k.s.cols;
        col = t - row * j.k.s.cols;
    }
    const KvcStreamArgs &s = is_k ? j.k.s : j.v.s;
    uint32_t bi_off = 0, bi_bn = 0;
    if (active) {
        const uint32_t *bi = reinterpret_cast<const uint32_t *>(s.block_infos + 8 * ((int64_t)row * s.cols + col));
        bi_off = bi[0];
        bi_bn = bi[1];
    }
    const uint32_t *__restrict__ lut_k = j.k.s.luts, *__restrict__ lut_v = j.v.s.luts;
    const uint32_t kb = (uint32_t)j.k_bits, vb = (uint32_t)j.v_bits;                      // 1 .. 7
    {
        const uint32_t i = (uint32_t)tid & 127u;
        if (tid < 128) {
            if (i < (1u << kb)) {
                const uint32_t e = lut_k[KVC_LUT_FENTRY_OFFSET + i], len = (e & 0xffu) > kb ? kb : (e & 0xffu);
                tmp[i] = ((uint32_t)__half_as_ushort(__float2half_rn(__uint_as_float(e & 0xffffff00u))) << 16) | len;
            }
        } else if (i < (1u << vb)) {
            const uint32_t e = lut_v[KVC_LUT_FENTRY_OFFSET + i], len = (e & 0xffu) > vb ? vb : (e & 0xffu);
            tmp[128 + i] = (((uint32_t)__uint_as_float(e & 0xffffff00u) & 0xffu) << 8) | len;
        }
    }
    const bool k_fast = lut_k[0] == kb && lut_k[1] == kb && lut_k[2] == 0u, v_fast = lut_v[0] == vb && lut_v[1] == vb && lut_v[2] == 0u;
    const bool k_pairs = k_fast && (1 << (2 * kb)) <= j.ktab_words && (lut_k[6] & KVC_PAIR_LEN_MASK) == 0u;
    const bool v_pairs = vb <= (uint32_t)KVC_ATTEND_V_PAIR_BITS;
    const int k_area = K_OPS + j.k.pack_words, v_area = T::MSTAB_SLOT_WORDS + j.v.pack_words;
    uint32_t *area = areas + (is_k ? wave * k_area : KVC_ATTEND_K_TILES * k_area + (wave - KVC_ATTEND_K_TILES) * v_area);
    uint32_t *btab = area, *mstab = area + (is_k ? T::BTAB_SLOT_WORDS : 0), *pack = mstab + T::MSTAB_SLOT_WORDS;
    if (is_k) {
        for (int i = lane; i < T::BTAB_SLOT_WORDS; i += KVC_WAVE) btab[i] = 0;           // columns that no query head owns
    }
    for (int i = tid; i < T::BTAB_SLOT_WORDS; i += KVC_WG) btab_v[i] = 0;
    if (active && lane < KVC_PACK_LEAD) pack[lane] = 0;
    KvcRaw<REP, 1, 1> raw;
    KvcTilePos pos = {};
    if (active) {
        if (is_k) {
            pos = kvc_tile_pos<true>(j.k, row, col);
            kvc_fetch_tile<REP, 0>(j.k, pos, bi_off, bi_bn, lane, raw);
        } else {
            pos = kvc_tile_pos<false>(j.v, row, col);
            kvc_fetch_tile<REP, 1, 2>(j.v, pos, bi_off, bi_bn, lane, raw);                // payload and parameters, no weights
        }
    }
    __syncthreads();
    if (k_pairs) {
        const uint32_t m1 = (1u << kb) - 1u;
        for (uint32_t idx = tid; idx < (1u << (2 * kb)); idx += KVC_WG) {
            const uint32_t e0 = tmp[idx & m1], e1 = tmp[(idx >> (e0 & 0xffu)) & m1];
            ktab[idx] = (e1 & 0xffff0000u) | (e0 >> 16) | ((e0 & 0xffu) + (e1 & 0xffu));
        }
    } else if (tid < (1 << kb)) {
        ktab[tid] = tmp[tid];
    }
    if (v_pairs) {
        const uint32_t m1 = (1u << vb) - 1u;
        if (tid < (1 << (2 * vb))) {
            const uint32_t e0 = tmp[128 + (tid & m1)], e1 = tmp[128 + (((uint32_t)tid >> (e0 & 0xffu)) & m1)];
            vtab[tid] = ((e1 & 0xff00u) << 8) | (e0 & 0xff00u) | ((e0 & 0xffu) + (e1 & 0xffu));
        }
    } else if (tid < (1 << vb)) {
        reinterpret_cast<uint16_t *>(vtab)[tid] = (uint16_t)tmp[128 + tid];
    }
    const uint32_t lead_bits = is_k || v_pairs ? 2u : 1u;                                 // bits of the window below the table index
    KvcStaged st = {};
    KvcTableState tabs = {-1, -1, -1, 0, 0};
    if (active) {
        const KvcFusedArgs &a = is_k ? j.k : j.v;
        uint32_t first, longest;
        st = kvc_stage_payload<true>(a, lane, raw, pack, first, longest);
        if (st.fits) st.u0 = 32u * KVC_PACK_LEAD + first * 8u - lead_bits;               // one or two bits before the lane's first code
        if (is_k) {
            const KvcTablePlan plan = {0, 1, 0};
            float bias[REP], unscale;
            int sel;
            kvc_mfma_stage_ops<REP, 0, true>(j.k, pos, plan, lane, raw, btab, mstab, bias, unscale, sel, tabs);
        } else {
            // minima less the 1024 that a byte under 0x64 stands for as fp16 (sums of integers below 2048: exact)
            const kvc_h2 off = {(_Float16)-1024.f, (_Float16)-1024.f};
            uint32_t mins, scales;
            kvc_mfma_min_scale_words(raw, 0, kvc_pair_mode<1>(j.v), mins, scales);
            uint32_t *mg = mstab + (lane >> 1) * 4 + (lane & 1);
            mg[0] = __builtin_bit_cast(uint32_t, __builtin_bit_cast(kvc_h2, mins) + off);
            mg[2] = scales;
        }
    }
    __syncthreads();
    // ---- decode: K tiles to scores, V tiles to bytes
    kvc_w32 vd;
    const uint32_t sbase = kvc_lds_addr(pack), fe_k = kvc_lds_addr(smem), fe_v = kvc_lds_addr(vtab);
    const int rows4 = (lane >> 2) * 4, cj = lane & 3;
    if (active && is_k) {
        float *dst = s_scores + wave * KVC_WAVE;
        int64_t dst_step = KVC_V_TOKENS;
        if (!whole) {
            dst = reinterpret_cast<float *>(j.k.out) + ((int64_t)pos.b * j.k.q_heads + pos.h * REP) * j.k.out_stride + (int64_t)pos.row * KVC_WAVE;
            dst_step = j.k.out_stride;
        }
        if (k_fast && st.fits) {
            kvc_f4 acc[NM];
#pragma unroll
            for (int q = 0; q < NM; q++) acc[q] = kvc_f4{0.f, 0.f, 0.f, 0.f};
            uint32_t u = st.u0, bptr = kvc_lds_addr(btab) + cj * 8, msptr = kvc_lds_addr(mstab);
            const uint32_t mask = ((1u << (k_pairs ? 2 * kb : kb)) - 1u) << lead_bits;
            if (k_pairs) {
                // 30 bits of a half window hold three pairs of codes of up to 5 bits, two of 6
                int n_main = kb <= 5u ? D / 12 * 12 : 0;
                while ((D - n_main) % 8 != 0) n_main -= 12;
                if (n_main) kvc_mfma_pair_dot<3, KVC_PACKED_PLAIN, NM, true, true, true>(sbase, u, fe_k, mask, n_main, bptr, msptr, acc, true);
                kvc_mfma_pair_dot<2, KVC_PACKED_PLAIN, NM, true, true, true>(sbase, u, fe_k, mask, D - n_main, bptr, msptr, acc, true);
            } else {
                kvc_mfma_dot<4, KVC_PACKED_PLAIN, NM, true, true, KVC_ENTRY_WORD, true>(sbase, u, fe_k, mask, D, bptr, msptr, acc, true);
            }
#pragma unroll
            for (int q = 0; q < NM; q++) {
                const int r = 2 * q + (cj >> 1);
                float4 res = make_float4(acc[q][0], acc[q][1], acc[q][2], acc[q][3]);
                if (tabs.lo0) {
                    res.x = fmaf(kvc_quad_next(acc[q][0]), 1.f / KVC_LO_SCALE, res.x);
                    res.y = fmaf(kvc_quad_next(acc[q][1]), 1.f / KVC_LO_SCALE, res.y);
                    res.z = fmaf(kvc_quad_next(acc[q][2]), 1.f / KVC_LO_SCALE, res.z);
                    res.w = fmaf(kvc_quad_next(acc[q][3]), 1.f / KVC_LO_SCALE, res.w);
                }
                if ((cj & 1) == 0 && r < REP) *reinterpret_cast<float4 *>(dst + r * dst_step + rows4) = res;
            }
        } else {
            KvcVec<REP> res;
            if (st.fits) res = kvc_mfma_slow_tile<REP, false, true>(pack, (uint32_t)j.k.pack_logical, st.u0 + lead_bits, lut_k, D, btab, mstab, 0u);
            else res = kvc_mfma_slow_tile<REP, true, true>(st.gwords, st.gnwords, st.gpos, lut_k, D, btab, mstab, 0u);
#pragma unroll
            for (int r = 0; r < REP; r++) dst[r * dst_step + lane] = res.v[r];
        }
    } else if (active) {
        const uint32_t mask = ((1u << (v_pairs ? 2 * vb : vb)) - 1u) << lead_bits;
        if (!v_fast || !st.fits)
            kvc_decode_bytes_slow(st.fits ? pack : st.gwords, st.fits ? (uint32_t)j.v.pack_logical : st.gnwords, st.fits,
                                  st.fits ? st.u0 + lead_bits : st.gpos, lut_v, vd);
        else if (v_pairs) kvc_decode_bytes<true>(sbase, st.u0, fe_v, mask, vd);
        else kvc_decode_bytes<false>(sbase, st.u0, fe_v, mask, vd);
    }
    if (!whole) return;                                                                   // uniform over the workgroup
    __syncthreads();
    // ---- softmax weights of the group, one query head per wave at a time; lane: tokens 2 lane and 2 lane + 1
    const int g = blockIdx.x / j.k.s.cols;
    for (int r = wave; r < REP; r += KVC_WAVES_PER_WG) {
        const float2 sc = *reinterpret_cast<const float2 *>(s_scores + r * KVC_V_TOKENS + 2 * lane);
        const float s0 = sc.x * j.v.sm_scale, s1 = sc.y * j.v.sm_scale;
        const float m = kvc_wave_fmax_dpp(fmaxf(s0, s1));
        const float w0 = __expf(s0 - m), w1 = __expf(s1 - m);
        const float l = kvc_wave_sum_dpp(w0 + w1);
        if (lane == 0) {
            const int bh = blockIdx.x - g * j.k.s.cols;
            *reinterpret_cast<float2 *>(j.v.ml + 2 * (((int64_t)g * j.k.s.cols + bh) * REP + r)) = make_float2(m, l);
        }
        float h0, l0, h1, l1;
        kvc_split_weight(w0, h0, l0);
        kvc_split_weight(w1, h1, l1);
        uint32_t *bg = btab_v + (lane >> 1) * (NM * 8) + (lane & 1);
        bg[(((2 * r) >> 2) * 4 + ((2 * r) & 3)) * 2] = kvc_half_pair(h0, h1);
        bg[(((2 * r + 1) >> 2) * 4 + ((2 * r + 1) & 3)) * 2] = kvc_half_pair(l0, l1);
    }
    __syncthreads();
    if (is_k || !active) return;
    kvc_f4 acc[NM];
#pragma unroll
    for (int q = 0; q < NM; q++) acc[q] = kvc_f4{0.f, 0.f, 0.f, 0.f};
    const uint32_t bptr = kvc_lds_addr(btab_v) + cj * 8, msptr = kvc_lds_addr(mstab);
    // the operands of a few groups are asked for while the groups before them are multiplied (left to itself the compiler asks for
    // them right before their use: 32 groups, 48 LDS round trips)
    constexpr int AHEAD = NM <= 2 ? 4 : 2;
    kvc_w4 ms[2][AHEAD];
    kvc_w2 cols[2][AHEAD][NM];
    auto ask = [&](auto buf_, int i0) {
        constexpr int buf = decltype(buf_)::value;
#pragma unroll
        for (int k = 0; k < AHEAD; k++) {
            ms[buf][k] = *(const kvc_lds_w4 *)(uintptr_t)(msptr + (i0 + k) * 16);
#pragma unroll
            for (int q = 0; q < NM; q++) cols[buf][k][q] = kvc_read_columns<true, true>(bptr + ((i0 + k) * NM + q) * 32, true);
        }
    };
    ask(std::integral_constant<int, 0>{}, 0);
    kvc_static_for<KVC_MFMA_GROUPS / AHEAD>([&](auto s_) {
        constexpr int s = decltype(s_)::value, buf = s & 1;
        if constexpr ((s + 1) * AHEAD < KVC_MFMA_GROUPS) ask(std::integral_constant<int, buf ^ 1>{}, (s + 1) * AHEAD);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < AHEAD; k++) {
            const uint32_t four = vd[s * AHEAD + k];
            const uint32_t a01 = kvc_dequant_pair(__builtin_amdgcn_perm(0x64u, four, 0x04010400u), ms[buf][k].x, ms[buf][k].z);
            const uint32_t a23 = kvc_dequant_pair(__builtin_amdgcn_perm(0x64u, four, 0x04030402u), ms[buf][k].y, ms[buf][k].w);
#pragma unroll
            for (int q = 0; q < NM; q++) acc[q] = kvc_mfma4<true>(a01, a23, cols[buf][k][q], acc[q]);
        }
        __builtin_amdgcn_sched_barrier(0);
    });
    float *out = reinterpret_cast<float *>(j.v.out) + (((int64_t)pos.row * j.v.batch + pos.b) * j.v.q_heads + pos.h * REP) * D + pos.d0;
#pragma unroll
    for (int q = 0; q < NM; q++) {
        const int r = 2 * q + (cj >> 1);
        float4 res;
        res.x = fmaf(kvc_quad_next(acc[q][0]), 1.f / KVC_LO_SCALE, acc[q][0]);
        res.y = fmaf(kvc_quad_next(acc[q][1]), 1.f / KVC_LO_SCALE, acc[q][1]);
        res.z = fmaf(kvc_quad_next(acc[q][2]), 1.f / KVC_LO_SCALE, acc[q][2]);
        res.w = fmaf(kvc_quad_next(acc[q][3]), 1.f / KVC_LO_SCALE, acc[q][3]);
        if ((cj & 1) == 0 && r < REP) *reinterpret_cast<float4 *>(out + r * D + rows4) = res;
    }
}

// Payload words a wave of this stream needs in LDS: the largest tile where the encoder said it, else somewhat more than the
// mean (tiles that do not fit are decoded from global memory).
static int kvc_attend_pack_words(const kvc_compressed_desc *c, int64_t tiles)
{
    const int64_t mean = c->encoded_bytes / (tiles > 0 ? tiles : 1);
    int64_t bytes = c->max_tile_bytes > 0 ? c->max_tile_bytes : mean + mean / 4 + 256;
    if (bytes > KVC_MAX_TILE_BYTES) bytes = KVC_MAX_TILE_BYTES;
    return (int)(KVC_PACK_LEAD + ((bytes + 15 + 15) / 16) * 4 + 4);
}

static int kvc_attend_fill(KvcFusedArgs &a, const kvc_compressed_desc *c, int is_k, int64_t batch, int64_t kv_heads, int64_t q_heads,
                           int64_t head_dim)
{
    KVC_REQUIRE(((uintptr_t)c->d_quant_scales_f16 & 3) == 0 && ((uintptr_t)c->d_quant_min_ints & 1) == 0,
                "quant_scales must be 4-byte aligned and quant_min_ints 2-byte aligned");
    int64_t rows;
    if (int rc = kvc_fill_stream_args(a.s, c->d_encoded, c->encoded_bytes, c->d_block_infos, c->block_infos_bytes, c->d_thread_infos,
                                      c->thread_infos_bytes, (const uint32_t *)c->d_luts, is_k, c->tokens,
                                      batch * kv_heads * head_dim, head_dim, &rows))
        return rc;
    a.s.rows_per_codebook = 0;
    a.min_i8 = c->d_quant_min_ints;
    a.scale = reinterpret_cast<const __half *>(c->d_quant_scales_f16);
    a.quant_mask = (int)c->quant_mask;
    a.out_f32 = 1;
    a.tokens = c->tokens;
    a.batch = (int)batch;
    a.kv_heads = (int)kv_heads;
    a.q_heads = (int)q_heads;
    a.head_dim = (int)head_dim;
    a.rounded = 1;
    return 0;
}

// The joint kernel's LDS
struct KvcJointPlan {
    int k_pack_words, v_pack_words, ktab_words;
    size_t lds;          // more than 64 KiB: does not fit
};
static KvcJointPlan kvc_plan_joint(const kvc_compressed_desc *k, const kvc_compressed_desc *v, int64_t rep, int64_t bh, int64_t head_dim)
{
    KvcJointPlan p = {};
    const int kb = kvc_hint_bits(k->max_code_bits);
    const int64_t groups = v->tokens / KVC_V_TOKENS, k_tiles = k->tokens / KVC_WAVE * bh;
    p.k_pack_words = kvc_attend_pack_words(k, k_tiles);
    p.v_pack_words = kvc_attend_pack_words(v, groups * bh * (head_dim / KVC_WAVE));
    const int sets = kvc_mfma_sets((int)rep), btab = KVC_MFMA_GROUPS * sets * 8, mstab = KVC_MFMA_GROUPS * 4;
    const int k_area = btab + mstab + p.k_pack_words, v_area = mstab + p.v_pack_words;
    int waves = KVC_ATTEND_K_TILES * k_area + (int)(head_dim / KVC_WAVE) * v_area;
    if (k_tiles > groups * bh * KVC_ATTEND_K_TILES && waves < KVC_WAVES_PER_WG * k_area) waves = KVC_WAVES_PER_WG * k_area;
    const int fixed = KVC_ATTEND_VTAB_WORDS + KVC_ATTEND_TMP_WORDS + btab + (int)rep * KVC_V_TOKENS + waves + KVC_LDS_SLACK_WORDS;
    p.ktab_words = KVC_ATTEND_VTAB_WORDS;
    if (kb <= KVC_ATTEND_K_PAIR_BITS && (1 << (2 * kb)) > p.ktab_words) p.ktab_words = 1 << (2 * kb);
    if (4 * (p.ktab_words + fixed) > 65536) p.ktab_words = KVC_ATTEND_VTAB_WORDS;
    p.lds = 4 * (size_t)(p.ktab_words + fixed);
    return p;
}

KvcAttendRoute kvc_attend_route(const kvc_compressed_desc *k, const kvc_compressed_desc *v, int64_t batch, int64_t kv_heads, int64_t q_heads,
                                int64_t head_dim)
{
    const int want = kvc_option(KVC_OPT_ATTENTION_JOINT);
    const int64_t rep = q_heads / kv_heads, bh = batch * kv_heads;
    const int kb = kvc_hint_bits(k->max_code_bits), vb = kvc_hint_bits(v->max_code_bits);
    if (want == 0 || v->tokens == 0 || k->tokens < v->tokens || head_dim % KVC_WAVE != 0 || kb < 1 || kb > 7 || vb < 1 || vb > 7) return KVC_ATTEND_SEPARATE;
    if (k->rows_per_codebook != 0 || v->rows_per_codebook != 0 || !(rep == 1 || rep == 2 || rep == 4 || rep == 8)) return KVC_ATTEND_SEPARATE;
    if (!(k->quant_mask == KVC_MASK_K_BLOCK || k->quant_mask == KVC_MASK_CHANNEL)) return KVC_ATTEND_SEPARATE;
    if (!(v->quant_mask == KVC_MASK_V_TOKEN || v->quant_mask == KVC_MASK_SIM_TOKEN || v->quant_mask == KVC_MASK_VECTOR)) return KVC_ATTEND_SEPARATE;
    if (kvc_option(KVC_OPT_FUSED_ROUNDED) == 0 || kvc_option(KVC_OPT_FUSED_MFMA) == 0 || kvc_option(KVC_OPT_FUSED_ROWS) == 1) return KVC_ATTEND_SEPARATE;
    const int64_t wgs = v->tokens / KVC_V_TOKENS * bh;
    if (k->tokens / KVC_WAVE * bh > (int64_t)1 << 30) return KVC_ATTEND_SEPARATE;
    // a wave per group (kvc_attend_waves.hip) where both codebooks are its
    if (want != 1 && (want > 1 || wgs > KVC_ATTEND_WAVES_MIN_WGS) && head_dim == 2 * KVC_WAVE && kb >= 6 && vb >= 6 &&
        kvc_hint_byte_symbols(k->max_code_bits) && kvc_hint_byte_symbols(v->max_code_bits) && kvc_hint_pair_bits(v->max_code_bits) == 0 &&
        kvc_option(KVC_OPT_FUSED_HALF_TABLE) != 0) {
        const int per_cu = kvc_plan_attend_waves(k, v, rep, bh).per_cu;
        if (want > 1 ? per_cu > 0 : kvc_attend_waves_pays(rep, wgs, per_cu)) return KVC_ATTEND_WAVES;
    }
    if (want > 1 || (want < 0 && wgs > kvc_attend_max_wgs(rep))) return KVC_ATTEND_SEPARATE;
    return kvc_plan_joint(k, v, rep, bh, head_dim).lds <= 65536 ? KVC_ATTEND_JOINT : KVC_ATTEND_SEPARATE;
}

int kvc_attend_groups(const kvc_compressed_desc *k, const kvc_compressed_desc *v, const void *d_q_f16, float softmax_scale,
                      float *scores, int64_t scores_stride, float *part, float *ml, int64_t batch, int64_t kv_heads, int64_t q_heads,
                      int64_t head_dim, hipStream_t stream, bool *taken)
{
    const KvcAttendRoute route = kvc_attend_route(k, v, batch, kv_heads, q_heads, head_dim);
    *taken = false;
    if (route == KVC_ATTEND_SEPARATE) return 0;
    const int64_t rep = q_heads / kv_heads, bh = batch * kv_heads, wgs = v->tokens / KVC_V_TOKENS * bh;
    const int64_t k_tiles = k->tokens / KVC_WAVE * bh, k_rest = k_tiles - wgs * KVC_ATTEND_K_TILES;
    KvcAttendArgs j = {};
    if (int rc = kvc_attend_fill(j.k, k, 1, batch, kv_heads, q_heads, head_dim)) return rc;
    if (int rc = kvc_attend_fill(j.v, v, 0, batch, kv_heads, q_heads, head_dim)) return rc;
    j.k.x = reinterpret_cast<const __half *>(d_q_f16);
    j.k.out = scores;
    j.k.out_stride = scores_stride;
    j.v.out = part;
    j.v.ml = ml;
    j.v.sm_scale = softmax_scale;
    *taken = true;
    if (route == KVC_ATTEND_WAVES) return kvc_attend_waves(j.k, j.v, k, v, kvc_plan_attend_waves(k, v, rep, bh), rep, stream);
    const KvcJointPlan plan = kvc_plan_joint(k, v, rep, bh, head_dim);
    j.k.pack_words = j.k.pack_logical = plan.k_pack_words;
    j.v.pack_words = j.v.pack_logical = plan.v_pack_words;
    j.k_bits = kvc_hint_bits(k->max_code_bits);
    j.v_bits = kvc_hint_bits(v->max_code_bits);
    j.group_wgs = (int)wgs;
    j.k_tiles = (int)k_tiles;
    j.ktab_words = plan.ktab_words;
    const size_t lds = plan.lds;
    const unsigned grid = (unsigned)(wgs + (k_rest + KVC_WAVES_PER_WG - 1) / KVC_WAVES_PER_WG);
    static const bool trace_plan = getenv("KVCOMP_TRACE_PLAN") != nullptr;
    if (trace_plan)
        fprintf(stderr, "[kvcomp] joint attention rep %d: %u workgroups (%d of whole groups), lds %zu B (K table %d w, codes %d / %d bits, payload %d / %d w)\n",
                (int)rep, grid, (int)wgs, lds, j.ktab_words, j.k_bits, j.v_bits, j.k.pack_words, j.v.pack_words);
    if (rep == 1) hipLaunchKernelGGL(kvc_attend_group_kernel<1>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    else if (rep == 2) hipLaunchKernelGGL(kvc_attend_group_kernel<2>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    else if (rep == 4) hipLaunchKernelGGL(kvc_attend_group_kernel<4>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    else hipLaunchKernelGGL(kvc_attend_group_kernel<8>, dim3(grid), dim3(KVC_WG), lds, stream, j);
    KVC_HIP(hipGetLastError());
    return 0;
}
