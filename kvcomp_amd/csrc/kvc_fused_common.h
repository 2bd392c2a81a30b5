// kvc_fused_common.h -- pieces shared by the fused decode + matvec kernels (kvc_fused.hip: fp32 FMA loops and plain
// decode; kvc_fused_mfma_impl.h: matrix-core loops): launch arguments, the one-tile-ahead fetch, payload staging.
#pragma once
#include "kvc_tile.h"

#include <mutex>
#include <type_traits>

constexpr int KVC_SCHED_SEGMENTS = 4;

struct KvcFusedArgs {
    KvcStreamArgs s;
    const int8_t *min_i8;
    const __half *scale;
    int quant_mask;
    const __half *x;     // K: q [batch, q_heads, head_dim];  V: p [batch, q_heads, tokens]
    void *out;           // K: scores [batch, q_heads, tokens]; V: partial [tokens/128, batch, q_heads, head_dim]
    int out_f32;         // 0: fp16 (reference layout), 1: fp32
    int64_t out_stride;  // K: elements between the score rows of two query heads (>= tokens)
    // softmax kinds of the V kernel: instead of p it reads raw fp32 scores and forms, per 128-token group and
    // query head, m = max(score * sm_scale), w = exp(score * sm_scale - m), l = sum w; the partial is the
    // w-weighted sum and (m, l) go to ml[group][batch][q_head][2]
    const float *scores;
    int64_t scores_stride;
    float sm_scale;
    float *ml;
    int64_t tokens;
    int batch, kv_heads, q_heads, head_dim;
    int table_words;     // LDS words reserved for the fused table (>= 1 << lbits of every codebook used)
    int pack_words;      // LDS words per wave reserved for the packed tile payload (multiple of 4)
    int pack_logical;    // payload words (lead words included) that fit there; fewer than pack_words when skewed
    int skew;            // 0, or 2: every 32 payload words are followed by a copy of the next two (see kvc_skewed)
    int row_words;       // LDS words per lane stream (odd); 0 = decode from the packed payload
    int column_rows;     // payloads in columns: words of a stream that the LDS holds
    int pair_bits;       // index width of the two-symbol table the host made room for; 0 = none
    int narrow_pair_bits; // matrix-core V kernels: index bits of a two-symbol table that next to all pairs that occur fit; 0 = none
    int double_window;   // refill 64 stream bits at a time where the vector length allows
    int builtin_dpp;     // fp32-FMA kernels: lane permutes through the compiler's intrinsic instead of inline assembly
    int half_table;      // matrix-core kernels: two-byte table entries for codes of 6 or 7 bits
    // kvc_expand_kernel (plain decode, decode + dequantize): no x; the operand table holds {scale, min} per element
    // Rounded mode of the matvec kernels: every (sym + min) * scale is rounded to fp16 before it meets q / p, as the
    // reference's dequantizer does (models/cache/kvcomp_encode.py:146); the operand table then holds
    // {min, scale, weight of each query head} per element and nothing is folded into a constant term.
    int rounded;
    int expand;          // 0: matvec kernels; 1: symbols out (uint8); 2: dequantized values out (fp16)
    int out_words;       // LDS words per wave for the 32-element output slab
    // Matrix-core kernels, one codebook per stream: 1-D grid over the row-major tile sequence in sched_nseg segments
    // (0: the 2-D grid of kvc_grid).  Segment k = workgroups sched_wg[k] .. sched_wg[k + 1] - 1, whose waves take
    // sched_run[k] consecutive tiles each, starting at tile sched_tile[k]; sched_tile[sched_nseg] = number of tiles.
    int sched_nseg;
    int sched_run[KVC_SCHED_SEGMENTS];
    int sched_wg[KVC_SCHED_SEGMENTS + 1];
    int sched_tile[KVC_SCHED_SEGMENTS + 1];
};

// Workgroups per CU (= waves per SIMD) each matvec kernel is compiled for.  With one query head per KV head the
// decode loops wait on LDS round trips and every further wave pays, so those kernels get the most their register
// demand allows without spilling (kinds 2 - 4 carry a second operand table or the softmax).  With four query heads
// the four FMAs per symbol hide the round trip; measured, 4 and 5 waves tie and 6 or 7 are 6 - 8 % slower.
constexpr int kvc_fused_occupancy(int rep, int kind)
{
    const bool two_slots = kind == 2 || kind == 4;
    return rep == 1 ? (kind == 1 ? 8 : 7) : (rep == 2 || (rep == 4 && !two_slots)) ? 5 : 1;
}
#ifndef KVC_FUSED_OCC
#define KVC_FUSED_OCC(REP, KIND) kvc_fused_occupancy(REP, KIND)
#endif
#ifndef KVC_MFMA_OCC_K1
#define KVC_MFMA_OCC_K1 8
#endif
#ifndef KVC_MFMA_OCC_V1
#define KVC_MFMA_OCC_V1 6
#endif
constexpr int kvc_fused_mfma_occupancy(int rep, int kind)
{
    // (four query heads, K: the kernel needs 80 registers, which leave six waves; with a bound of five the register
    // allocator settles on 81 and the sixth wave is lost: 46 -> 49 us at batch 16 x 8 KV heads x 8192 tokens)
    // (one query head, V: seven waves.  Tiles of one head each -- head_dim a multiple of 64 --: 65 registers, 37.7 -> 36.4 us
    // at batch 8 x 32 heads x 128 x 4096 tokens; eight waves fit too, with 30 spilled scalars, and measured no better.
    // Tiles that may straddle two heads, softmax on the fly: 72 registers without a spill only in a translation unit of
    // its own, kvc_fused_mfma_v96.hip; 71.7 -> 68.4 us at batch 4 x 32 heads x 96 x 32 768 tokens.)
    return rep == 1 ? (kind == 0 ? KVC_MFMA_OCC_K1 : (kind == 1 || kind == 3 || kind == 4) ? KVC_MFMA_OCC_V1 + 1 : KVC_MFMA_OCC_V1)
                    : (rep == 4 && kind == 0) ? 6 : kvc_fused_occupancy(rep, kind);
}
// the same for codebooks with codes of more than 7 bits (kvc_fused_mfma_long.hip)
constexpr int kvc_fused_long_occupancy(int rep, int kind) { return rep == 1 ? (kind == 0 ? 7 : 6) : rep == 2 ? 5 : rep == 4 ? 4 : 1; }
// the same for codes of 6 or 7 bits (kvc_fused_mfma_mid.hip)
constexpr int kvc_fused_mid_occupancy(int rep, int kind)
{
    return rep == 1 ? (kind == 2 || kind == 4 ? 7 : 8) : rep == 4 && kind == 0 ? 6 : kvc_fused_occupancy(rep, kind);
}
constexpr int KVC_PRE_CHUNKS = 4;     // 16-byte chunks per lane fetched one tile ahead (4 KiB of payload)
constexpr int KVC_PACK_LEAD = 4;      // zero words in front of the packed payload: bit positions never drop below 2

// How the (scale, minimum) pairs of a lane's two elements (2 * lane and 2 * lane + 1) lie in memory: next to each
// other (one 4-byte and one 2-byte load fetch both), the same pair for both elements, or anywhere.
enum { KVC_PAIR_SEPARATE = 0, KVC_PAIR_ADJACENT = 1, KVC_PAIR_SAME = 2 };

// What a tile needs from global memory, fetched into registers one tile ahead of its use.
template <int REP, int SLOTS, int XW>
struct KvcRaw {
    uint4 pay[KVC_PRE_CHUNKS];        // payload chunks lane, lane + 64, ...
    uint32_t off, bn;                 // block_info, clamped to the payload buffer (wave-uniform)
    uint32_t ti_cur;                  // thread_info of this lane (the previous lane's comes through a lane shift)
    // operands of elements 2 * lane and 2 * lane + 1 (K: channels, V: tokens of the 128-token group), as loaded:
    uint32_t scw[SLOTS][2];           // quantization scales (fp16 bits): see scale_bits
    uint32_t mnw[SLOTS][2];           // quantization minima (int8): see min_int
    uint32_t x[SLOTS][REP][XW];       // per query head: q / p (two fp16 in one word), or two fp32 scores
    __device__ __forceinline__ uint32_t scale_bits(int s, int half, int mode) const
    {
        if (mode == KVC_PAIR_ADJACENT) return half ? scw[s][0] >> 16 : scw[s][0] & 0xffffu;
        if (mode == KVC_PAIR_SAME) return scw[s][0] & 0xffffu;
        return scw[s][half] & 0xffffu;
    }
    __device__ __forceinline__ int min_int(int s, int half, int mode) const
    {
        if (mode == KVC_PAIR_ADJACENT) return (int)(int8_t)(mnw[s][0] >> (8 * half));
        if (mode == KVC_PAIR_SAME) return (int)(int8_t)mnw[s][0];
        return (int)(int8_t)mnw[s][half];
    }
};
// Nothing in it is touched before the tile is staged: any arithmetic on a loaded value would make the wave
// wait for the load at that point and the fetch would no longer overlap the decode of the previous tile.

// LDS traffic between the lanes of one wave needs no barrier (a wave's LDS operations complete in order);
// this only keeps the compiler from moving accesses across the hand-over.
__device__ __forceinline__ void kvc_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// memory byte j of a word carries stream bits 8j .. 8j+7, most significant first: a byte swap followed by a
// full bit reversal leaves stream bit k of the word at bit k
__device__ __forceinline__ uint32_t kvc_stream_word(uint32_t raw) { return __brev(kvc_bswap(raw)); }

// Skewed packed payload.  Lane l starts about l mean-stream-lengths into the payload, so when a small
// multiple of that length is close to 32 words, every k-th lane reads the same bank at every refill.  With
// two spare words after every 32 (holding a copy of the two words that follow, so that the three-word read
// of a refill never has to jump), streams 32 words apart land two banks apart instead.
//   word w of the payload lives at w + skew * (w >> 5), skew = 2 (or 0: plain layout)
__device__ __forceinline__ uint32_t kvc_skewed(uint32_t w, uint32_t skew) { return __umul24(w >> 5, skew) + w; }

// Whether the lanes line up: a small multiple of the mean stream length is close to a multiple of the 32 banks.
static inline bool kvc_streams_resonate(int64_t encoded_bytes, int64_t tiles)
{
    const double mean_stream_words = (double)encoded_bytes / (double)(tiles > 0 ? tiles : 1) / KVC_WAVE / 4.0;
    bool resonant = false;
    for (int k = 1; k <= 4; k++) {
        const double x = k * mean_stream_words / 32.0;
        const double dist = (x - (double)(int64_t)(x + 0.5)) * 32.0;
        if (x >= 0.5 && dist > -1.0 && dist < 1.0) resonant = true;
    }
    return resonant;
}

// Byte address in LDS of payload word u >> 5 for a refill.  No clamp: a lane's position cannot pass its start
// by more than 128 symbols x 10 bits, and the workgroup's LDS ends with that much slack (KVC_LDS_SLACK_WORDS),
// so even a corrupt stream only ever reads this workgroup's own LDS.
typedef __attribute__((address_space(3))) uint32_t kvc_lds_word;
// WORD: left to itself the compiler makes "u >> 3 & ~3" of the word's address, an instruction more than shift and shifted add.  A percent at
// most either way, as measured in turn: attention of 1 x 8 x 4 heads x 128 x 1000 tokens 16.49 -> 16.44 us, but with codes of more than 7
// bits, whose loop asks in several places, 2 x 8 x 8 x 128 x 1905 tokens 40.6 -> 41.0.
template <bool SKEW, bool WORD = false>
__device__ __forceinline__ uint32_t kvc_refill_address(uint32_t stage_base, uint32_t u)
{
    uint32_t a = u >> 5;
    if (WORD) asm("" : "+v"(a));
    if (SKEW) return (a << 2) + (__umul24(u >> 10, 8u) + stage_base);     // + 2 words per 32
    return (a << 2) + stage_base;
}
constexpr int KVC_LDS_SLACK_WORDS = 48;
// what a lane can run further where codes of up to 32 bits are taken in the same loops
constexpr int KVC_LDS_LONG_SLACK_WORDS = 96;

// Rounded mode: RN16((sym + min) * scale) as the reference's dequantizer computes it (sym + min exactly, one
// rounding of the product).  Both steps are fp16 instructions: the sum of two small integers is exact in fp16
// and an fp16 multiplication rounds the exact product once.  `ms` = {min, scale} as two fp16 in one word.
__device__ __forceinline__ float kvc_rounded_value(__half sym, uint32_t ms)
{
    const __half mn = __ushort_as_half((unsigned short)(ms & 0xffffu)), sc = __ushort_as_half((unsigned short)(ms >> 16));
    return __half2float(__hmul(__hadd(sym, mn), sc));
}

typedef _Float16 kvc_h2 __attribute__((ext_vector_type(2)));
// {x.lo, x.hi} -> RN16((x + mn) * sc) per half: the sum of two small integers is exact in fp16, the product is
// rounded once
__device__ __forceinline__ uint32_t kvc_dequant_pair(uint32_t x, uint32_t mn, uint32_t sc)
{
    const kvc_h2 v = (__builtin_bit_cast(kvc_h2, x) + __builtin_bit_cast(kvc_h2, mn)) * __builtin_bit_cast(kvc_h2, sc);
    return __builtin_bit_cast(uint32_t, v);
}

// upper halves of two table entries side by side: {a >> 16, b >> 16 << 16}
__device__ __forceinline__ uint32_t kvc_pack_hi16(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

template <int REP>
struct KvcVec {
    float v[REP];
};

// LDS accessed by its byte offset: the table's offset is a multiple of its size, so "window bits | offset"
// is the entry's address.
typedef __attribute__((address_space(3))) uint32_t kvc_lds_u32;
typedef __attribute__((address_space(3))) uint16_t kvc_lds_u16;

// compile-time loop: body(std::integral_constant<int, 0>) ... body(std::integral_constant<int, N - 1>)
template <int N, int I = 0, class Body>
__device__ __forceinline__ void kvc_static_for(Body &&body)
{
    if constexpr (I < N) {
        body(std::integral_constant<int, I>{});
        kvc_static_for<N, I + 1>(body);
    }
}

// -- the narrow two-symbol table of V's kernels --------------------------------------------------------
// The table is as wide as the first store's symbols asked for.  Where later data are not like them, tiles meet pairs that do
// not fit and are decoded twice.  A tile that did is counted, and the kernel that closes the call (one wave of it) adds the
// counters up and turns the table off for this codebook where it costs more than it gives.  Everything here decides about
// speed alone: both loops give the same bits, whoever reads or writes these words in between.
// One tile in sixteen: V kernel in us with the table / one symbol per look-up, by the share of tiles decoded twice,
//   4 x 32 heads x 96 x 32 768 tokens   1 %: 72.7 / 90.1   6 %: 79.4 / 90.3   11 %: 84.8 / 89.9   24 %: 95.2 / 90.5
//   8 x 32 heads x 128 x 8192           1 %: 52.2 / 61.8   6 %: 57.0 / 61.8   11 %: 60.0 / 61.6   24 %: 68.4 / 61.7
//   4 x 32 heads x 128 x 8192           1 %: 35.5 / 37.5   6 %: 37.8 / 37.7   11 %: 39.8 / 37.6   24 %: 43.0 / 37.4
// (Counters in lines of their own: into one word, every atomic waits for the one before it, and the wave's next loads for
// it: 244 us instead of 95 in the first row.  The off bit lies in a word that is read anyway.)
constexpr int KVC_NARROW_TOO_MANY = 16;
__device__ __forceinline__ void kvc_narrow_miss(const uint32_t *lut, uint32_t block)
{
    // (lane number and constants are made here, where they are used: kept in registers across the decode loops they cost some
    // of the kernels a wave per SIMD)
    uint32_t id, one, at = block % KVC_NARROW_COUNTERS * (KVC_NARROW_LINE_WORDS * 4u) + KVC_LUT_NARROW_OFFSET * 4u;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(id));
    if (id != 0) return;
    asm volatile("v_mov_b32 %0, 1" : "=v"(one));
    asm volatile("" : "+v"(at));
    __hip_atomic_fetch_add(reinterpret_cast<uint32_t *>(reinterpret_cast<char *>(const_cast<uint32_t *>(lut)) + at), one,
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// One wave, all its lanes: a counter each.
__device__ __forceinline__ uint32_t *kvc_narrow_counter(uint32_t *lut, int lane)
{
    static_assert(KVC_NARROW_COUNTERS == KVC_WAVE, "a counter per lane");
    return lut + KVC_LUT_NARROW_OFFSET + KVC_NARROW_LINE_WORDS * lane;
}
__device__ __forceinline__ uint32_t kvc_narrow_missed(uint32_t *lut, int lane)
{
    return __hip_atomic_load(kvc_narrow_counter(lut, lane), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// `tiles`: how many the launch before this one decoded (with this table, if it was on); `missed`: kvc_narrow_missed
__device__ __forceinline__ void kvc_narrow_decide(uint32_t *lut, uint64_t tiles, int lane, uint32_t missed)
{
    if (!__any(missed != 0u)) return;
    uint32_t *mine = kvc_narrow_counter(lut, lane);
    __hip_atomic_store(mine, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) missed += __shfl_xor(missed, s);
    if (lane == 0 && missed * (uint64_t)KVC_NARROW_TOO_MANY > tiles)
        __hip_atomic_store(lut + KVC_LUT_NARROW_WORD, lut[KVC_LUT_NARROW_WORD] | KVC_LUT_NARROW_OFF, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// -- tile geometry ------------------------------------------------------------------------------------
// KIND 0: K tile (64 tokens x head_dim channels of one (batch, head); lane = token)
// KIND 1: V tile (128 tokens x 64 flat channels; lane = channel), head_dim a multiple of 64: one head per tile
// KIND 2: V tile with any other head_dim: the 64 channels may straddle two heads (two operand tables); the small ones of
//         which they may touch more go to kvc_v_small_heads.hip
// KIND 3, 4: as 1, 2 but with the softmax over the group's scores computed on the fly
// Whether a tile of 64 flat channels can touch more than two heads: tiles start at every multiple of gcd(head_dim, 64) inside
// a head, and behind the latest start the head has only that many channels left.
constexpr bool kvc_tile_spans_many_heads(int64_t head_dim)
{
    int64_t g = KVC_WAVE;
    while (head_dim % g != 0) g /= 2;
    return KVC_WAVE - g > head_dim;
}
static_assert(kvc_tile_spans_many_heads(40) && kvc_tile_spans_many_heads(24) && kvc_tile_spans_many_heads(16) && kvc_tile_spans_many_heads(8) &&
              !kvc_tile_spans_many_heads(32) && !kvc_tile_spans_many_heads(48) && !kvc_tile_spans_many_heads(56) && !kvc_tile_spans_many_heads(72),
              "the head sizes that take the kernel of their own");
int kvc_launch_v_small_heads(int rep, const KvcFusedArgs &a, int64_t rows, hipStream_t stream);

template <int KIND>
struct KvcGeom {
    static constexpr bool IS_K = KIND == 0;
    static constexpr int SLOTS = (KIND == 2 || KIND == 4) ? 2 : 1;
    static constexpr bool SOFTMAX = KIND >= 3;
    static constexpr int XW = SOFTMAX ? 2 : 1;
};

template <int KIND>
__device__ __forceinline__ int kvc_pair_mode(const KvcFusedArgs &a)
{
    if (KIND == 0) return a.quant_mask == KVC_MASK_CHANNEL ? KVC_PAIR_ADJACENT : KVC_PAIR_SAME;
    if (a.quant_mask == KVC_MASK_V_TOKEN) return KVC_PAIR_ADJACENT;
    if (a.quant_mask == KVC_MASK_SIM_TOKEN) return a.batch == 1 ? KVC_PAIR_ADJACENT : KVC_PAIR_SEPARATE;
    return a.batch * a.kv_heads == 1 ? KVC_PAIR_ADJACENT : KVC_PAIR_SEPARATE;           // KVC_MASK_VECTOR
}

// Loads relative to a wave-uniform base with a 32-bit per-lane byte offset: the base stays in scalar registers and
// the address costs no 64-bit vector arithmetic.
template <class T>
__device__ __forceinline__ T kvc_load_at(const void *uniform_base, uint32_t byte_offset)
{
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(uniform_base) + byte_offset);
}

// Where a tile lies: its row and column in the tile grid and what follows from the column -- the (batch entry, head)
// it belongs to and, for a V tile, the first of its 64 channels inside that head.  Working these out from the column
// takes integer divisions, for which the hardware has no scalar instruction (each becomes some fifteen vector
// instructions, wave-uniform or not); stepping to the next tile of the row-major sequence takes a few scalar additions.
struct KvcTilePos {
    int row, col;
    int b, h;       // K: the tile's (batch entry, kv head); V: those of the tile's first channel
    int d0;         // V: the first channel's index inside head h (K: 0)
};

template <bool IS_K>
__device__ __forceinline__ KvcTilePos kvc_tile_pos(const KvcFusedArgs &a, int row, int col)
{
    KvcTilePos p;
    p.row = row;
    p.col = col;
    if (IS_K) {
        p.b = col / a.kv_heads;
        p.h = col - p.b * a.kv_heads;
        p.d0 = 0;
    } else {
        const int c0 = col * KVC_WAVE, bh = c0 / a.head_dim;
        p.d0 = c0 - bh * a.head_dim;
        p.b = bh / a.kv_heads;
        p.h = bh - p.b * a.kv_heads;
    }
    return p;
}

template <bool IS_K>
__device__ __forceinline__ KvcTilePos kvc_tile_after(const KvcFusedArgs &a, KvcTilePos p)
{
    p.col++;
    if (p.col == a.s.cols) {                                // the rows' tiles cover all (batch entry, head) pairs exactly
        p.col = 0;
        p.row++;
        p.b = p.h = p.d0 = 0;
        return p;
    }
    if (IS_K) {
        p.h++;
    } else {
        p.d0 += KVC_WAVE;
        if (p.d0 < a.head_dim) return p;
        p.d0 -= a.head_dim;
        p.h++;
        while (p.d0 >= a.head_dim) {                        // heads narrower than a tile
            p.d0 -= a.head_dim;
            p.h++;
        }
    }
    while (p.h >= a.kv_heads) {
        p.h -= a.kv_heads;
        p.b++;
    }
    return p;
}

// (batch entry, head) of a V tile's second head (the one its channels past a head boundary belong to), clamped to the
// last pair: the tile that ends a row has no second head and must not make one up.
__device__ __forceinline__ void kvc_second_head(const KvcFusedArgs &a, const KvcTilePos &p, int &b, int &h)
{
    b = p.b;
    h = p.h + 1;
    if (h == a.kv_heads) {
        if (b + 1 < a.batch) b++, h = 0;
        else h = p.h;
    }
}

// Issue the global loads of tile (row, col).  bi_off / bi_bn: the tile's block_info words.
// Parameters of a V tile's two elements per lane where every token has groups of its own per batch entry (or per batch
// entry and head): two 2-byte and two 1-byte loads.
template <class Raw>
__device__ __forceinline__ void kvc_fetch_separate_params(const KvcFusedArgs &a, int row, int b, int h, int lane, int s, Raw &raw)
{
    const int64_t tk0 = (int64_t)row * KVC_V_TOKENS;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        // group of token tk0 + t: (tk0 + t) * batch + b, times kv_heads + h for per-vector groups
        const int64_t per = a.quant_mask == KVC_MASK_SIM_TOKEN ? a.batch : (int64_t)a.batch * a.kv_heads;
        const int64_t g0 = a.quant_mask == KVC_MASK_SIM_TOKEN ? tk0 * per + b : tk0 * per + (int64_t)b * a.kv_heads + h;
        const uint32_t t = 2u * (uint32_t)lane + half;
        raw.scw[s][half] = kvc_load_at<uint16_t>(a.scale + g0, 2u * t * (uint32_t)per);
        raw.mnw[s][half] = kvc_load_at<uint8_t>(a.min_i8 + g0, t * (uint32_t)per);
    }
}

// `skip_x`: bit s set = the weights of head slot s are not needed (the wave still has that head's operand table).
// LATE_SECOND: the separate-groups parameters of a tile's second head are left to the caller, who fetches them when the
// tile is staged (kvc_fetch_separate_params): four registers less to hold through the previous tile's decode loops.
// PAYLOAD = false: the operands only (the payload comes by kvc_fetch_streams).
template <int REP, int KIND, int EXPAND = 0, bool LATE_SECOND = false, bool PAYLOAD = true>
__device__ __forceinline__ void kvc_fetch_tile(const KvcFusedArgs &a, const KvcTilePos &pos, uint32_t bi_off, uint32_t bi_bn,
                                               int lane, KvcRaw<REP, KvcGeom<KIND>::SLOTS, KvcGeom<KIND>::XW> &raw, int skip_x = 0)
{
    constexpr int SLOTS = KvcGeom<KIND>::SLOTS;
    const int row = pos.row, col = pos.col;
    const int64_t tile = (int64_t)row * a.s.cols + col;                 // wave-uniform, like everything derived from it
    const int D = a.head_dim;
    // sizes are clamped so that corrupt metadata yields wrong symbols, never an out-of-bounds access
    uint32_t off = bi_off, bn = bi_bn & 0xffffu;
    if (bn > (uint32_t)KVC_MAX_TILE_BYTES) bn = KVC_MAX_TILE_BYTES;
    if ((int64_t)off >= a.s.enc_bytes) bn = 0;
    else if ((int64_t)off + bn > a.s.enc_bytes) bn = (uint32_t)(a.s.enc_bytes - off);
    raw.off = off;
    raw.bn = bn;
    if constexpr (PAYLOAD) raw.ti_cur = kvc_load_at<uint16_t>(a.s.thread_infos + tile * KVC_WAVE, 2u * (uint32_t)lane);
    // payload: whole aligned 16-byte chunks that each hold at least one payload byte (such reads never leave
    // the pages the payload lives in)
    const uint8_t *src = a.s.enc + off;
    const uint32_t head = (uint32_t)(reinterpret_cast<uintptr_t>(src) & 15u);
    const uint32_t nchunks = bn ? (head + bn + 15u) >> 4 : 0u;
    const uint8_t *g = src - head;
#pragma unroll
    for (int j = 0; j < (PAYLOAD ? KVC_PRE_CHUNKS : 0); j++) {
        const uint32_t c = (uint32_t)lane + 64u * j;
        if (c < nchunks) raw.pay[j] = kvc_load_at<uint4>(g, 16u * c);
    }
    // operands; lanes past the end of a short vector load the last pair (ignored when staged)
    const int mode = kvc_pair_mode<KIND>(a);
    if (KIND == 0) {
        const int b = pos.b, h = pos.h;
        const uint32_t e0 = (uint32_t)(2 * lane < D ? 2 * lane : D - 2);
        if (EXPAND != 1) {                                     // symbols out: no quantization parameters
            // per-channel pairs, or one pair per 64-token block (kernels.cu:771-772)
            if (mode == KVC_PAIR_ADJACENT) {
                raw.scw[0][0] = kvc_load_at<uint32_t>(a.scale + tile * D, 2u * e0);
                raw.mnw[0][0] = kvc_load_at<uint16_t>(a.min_i8 + tile * D, e0);
            } else {
                raw.scw[0][0] = kvc_load_at<uint16_t>(a.scale + row, 0u);
                raw.mnw[0][0] = kvc_load_at<uint8_t>(a.min_i8 + row, 0u);
            }
        }
        if (EXPAND == 0) {
#pragma unroll
            for (int r = 0; r < REP; r++)
                raw.x[0][r][0] = kvc_load_at<uint32_t>(a.x + ((int64_t)b * a.q_heads + h * REP + r) * D, 2u * e0);
        }
    } else {
        const int64_t tk0 = (int64_t)row * KVC_V_TOKENS;       // the group's first token; this lane's are tk0 + 2 lane (+ 1)
        const bool straddles = pos.d0 + KVC_WAVE > D;          // wave-uniform
#pragma unroll
        for (int s = 0; s < SLOTS; s++) {
            if (s == 1 && !straddles) continue;                // the second head's operands are not needed
            int b = pos.b, h = pos.h;
            if (s == 1) kvc_second_head(a, pos, b, h);         // (unused by a tile that ends the row)
            if (EXPAND != 1) {
                if (mode == KVC_PAIR_ADJACENT) {               // one group per token, whatever the batch entry and head:
                    if (s == 0) {                              // loaded once (also where the first head needs nothing)
                        raw.scw[0][0] = kvc_load_at<uint32_t>(a.scale + tk0, 4u * (uint32_t)lane);
                        raw.mnw[0][0] = kvc_load_at<uint16_t>(a.min_i8 + tk0, 2u * (uint32_t)lane);
                    } else {
                        raw.scw[s][0] = raw.scw[0][0];
                        raw.mnw[s][0] = raw.mnw[0][0];
                    }
                } else if (!((skip_x >> s) & 1) && (s == 0 || !LATE_SECOND)) {
                    kvc_fetch_separate_params(a, row, b, h, lane, s, raw);
                }
            }
#pragma unroll
            for (int r = 0; r < REP; r++) {
                if (EXPAND != 0 || ((skip_x >> s) & 1)) break;
                const int64_t xrow = (int64_t)b * a.q_heads + h * REP + r;
                if (KvcGeom<KIND>::SOFTMAX) {
                    const uint2 v = kvc_load_at<uint2>(a.scores + xrow * a.scores_stride + tk0, 8u * (uint32_t)lane);
                    raw.x[s][r][0] = v.x;
                    raw.x[s][r][KvcGeom<KIND>::XW - 1] = v.y;
                } else {
                    raw.x[s][r][0] = kvc_load_at<uint32_t>(a.x + xrow * a.tokens + tk0, 4u * (uint32_t)lane);
                }
            }
        }
    }
}

// The same for callers that know the tile by its row and column only.
template <int REP, int KIND, int EXPAND = 0>
__device__ __forceinline__ void kvc_fetch_tile(const KvcFusedArgs &a, int row, int col, uint32_t bi_off, uint32_t bi_bn,
                                               int lane, KvcRaw<REP, KvcGeom<KIND>::SLOTS, KvcGeom<KIND>::XW> &raw)
{
    kvc_fetch_tile<REP, KIND, EXPAND>(a, kvc_tile_pos<KIND == 0>(a, row, col), bi_off, bi_bn, lane, raw);
}

__device__ __forceinline__ float kvc_half_bits_to_float(uint32_t bits16)
{
    return __half2float(__ushort_as_half((unsigned short)bits16));
}

// Workgroups that a compute unit's LDS holds (160 KiB, handed out in pieces of 1280 bytes)
static inline int kvc_lds_workgroups(size_t lds) { return (int)(163840 / ((lds + 1279) / 1280 * 1280)); }

// What the decode step needs to know about a staged tile.
template <class Flag>
struct KvcStagedAs {
    Flag fits;            // staged in LDS (wave-uniform); otherwise decode from global memory
    uint32_t u0;          // fast-path start position (`lb` bits before the first code) in the lane's LDS words
    const uint32_t *gwords;   // the lane's stream in global memory, from the aligned word holding its first byte
    uint32_t gnwords, gpos;
};
// A bool is a bit per lane in scalar registers, an int a vector register; but copies of the struct with a bool, whose padding is copied
// too, would go through scratch memory: streams in columns are copied.
using KvcStaged = KvcStagedAs<bool>;
using KvcStreams = KvcStagedAs<int>;

// Move a fetched tile's payload into the wave's packed LDS area (least-significant-bit-first words, skewed if asked
// for) and work out where this lane's stream lies.  `first`: byte offset of the lane's stream in the packed area;
// `longest`: with per-lane rows, the longest lane stream of the tile in words.  The caller finishes st.u0.
// ALIGNED: the packed area starts at a multiple of 16 bytes; unskewed, a chunk is then one 16-byte write (two of 8 bytes, which
// leave every second pair of banks out, take twice as long).
template <bool ALIGNED = false, class Raw>
__device__ __forceinline__ KvcStaged kvc_stage_payload(const KvcFusedArgs &a, int lane, const Raw &raw, uint32_t *pack,
                                                       uint32_t &first_out, uint32_t &longest_out)
{
    KvcStaged st;
    const uint32_t bn = raw.bn;
    // the previous lane's thread_info: one lane shift over the whole wave (lane 0 starts the tile)
    const uint32_t ti_prev = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)raw.ti_cur, 0x138 /* wave_shr:1 */, 0xf, 0xf, false);
    uint32_t start = lane ? ti_prev >> 3 : 0u, end = raw.ti_cur >> 3;
    if (start > bn) start = bn;
    if (end > bn) end = bn;
    if (end < start) end = start;
    const uint8_t *src = a.s.enc + raw.off;
    const uint32_t head = (uint32_t)(reinterpret_cast<uintptr_t>(src) & 15u);
    const uint32_t nchunks = bn ? (head + bn + 15u) >> 4 : 0u;
    const uint32_t first = head + start;                                   // byte offset in the packed area
    const uint32_t nwords = end > start ? ((first & 3u) + (end - start) + 3u) >> 2 : 0u;
    {
        const uint8_t *lsrc = src + start;
        const uint32_t skew = (uint32_t)(reinterpret_cast<uintptr_t>(lsrc) & 3u);
        st.gwords = reinterpret_cast<const uint32_t *>(lsrc - skew);
        st.gnwords = nwords;
        st.gpos = skew * 8u;
    }
    // the packed area keeps row_words spare words at its end: the copy into rows moves the same
    // number of words for every lane, so the last lanes read past the payload
    bool fits = KVC_PACK_LEAD + 4u * nchunks + 3u + (uint32_t)a.row_words <= (uint32_t)a.pack_logical;
    uint32_t longest = 0;
    if (a.row_words) {
        longest = kvc_wave_max_dpp(nwords);
        fits = fits && longest + 3u <= (uint32_t)a.row_words;
    }
    st.fits = fits;
    st.u0 = 0;
    if (fits) {
        const uint32_t skew = (uint32_t)a.skew;
        // chunk c holds payload words 4c .. 4c + 3 (after the lead words); chunks never straddle a run of 32.
        // Chunk lane + 64 j lies a fixed number of words after chunk lane + 64 (j - 1), skewed or not, and whether
        // a chunk opens a run of 32 (and so is also the copy that ends the previous run) depends on the lane alone.
        const uint32_t w0 = KVC_PACK_LEAD + 4u * (uint32_t)lane;
        uint32_t *dst0 = pack + kvc_skewed(w0, skew);
        const uint32_t jstride = 256u + 8u * skew;
        const bool opens_run = skew && (w0 & 31u) == 0u;
        auto put = [&](uint32_t *dstw, uint4 v) {
            v.x = kvc_stream_word(v.x);
            v.y = kvc_stream_word(v.y);
            v.z = kvc_stream_word(v.z);
            v.w = kvc_stream_word(v.w);
            if (ALIGNED && !skew) {
                *reinterpret_cast<uint4 *>(dstw) = v;
                return;
            }
            uint2 *dst = reinterpret_cast<uint2 *>(dstw);                            // 8-byte aligned either way
            dst[0] = make_uint2(v.x, v.y);
            dst[1] = make_uint2(v.z, v.w);
            if (opens_run) dst[-1] = make_uint2(v.x, v.y);
        };
#pragma unroll
        for (int j = 0; j < KVC_PRE_CHUNKS; j++) {
            const uint32_t c = (uint32_t)lane + 64u * j;
            if (c < nchunks) put(dst0 + j * jstride, raw.pay[j]);
        }
        const uint8_t *g = src - head;
        for (uint32_t c = (uint32_t)lane + 64u * KVC_PRE_CHUNKS; c < nchunks; c += KVC_WAVE)            // tiles beyond 4 KiB
            put(dst0 + (c >> 6) * jstride, kvc_load_at<uint4>(g, 16u * c));
    }
    first_out = first;
    longest_out = longest;
    return st;
}

// -- payloads in columns ------------------------------------------------------------------------------
// A lane loads its own stream, sixteen bytes at a time, and puts word k of it in row k of an LDS area of 64 words a row.  A
// lane's words then lie in its own bank, wherever the other lanes are: the three words of a refill take the LDS 7.3 cycles, where
// lanes that read at their streams' places in the packed payload meet in the banks (19.5 cycles; streams of 52 bytes, positions
// within 6 words).  The loads' addresses are as far apart as the streams are long, which costs nothing: 65 536 tiles of 3360
// bytes in 33 us, as with whole lines in order.
// With them the attention kernels of 4 x 32 heads x 96 x 32 768 tokens (K six bits and skewed before, V two symbols per look-up) take 152 us
// for 161; such a kernel has no skewed variant of its loops and needs two to six registers less than the packed one.  Which calls
// take columns: kvc_columns_from, kvc_columns_workgroups.
struct KvcLane {
    const uint8_t *base;      // wave-uniform, a multiple of four
    uint32_t at;              // the stream's first word, in bytes from there
    uint32_t skip, bytes;     // bytes of that word before the stream, bytes from the word to the stream's end
};
// raw.off, raw.bn and raw.ti_cur are there
struct KvcTileBytes {
    uint32_t off, bn;         // block_info, clamped to the payload buffer (wave-uniform)
    uint32_t ti_cur;          // thread_info of this lane
};
template <class Raw>
__device__ __forceinline__ KvcLane kvc_lane_stream(const KvcFusedArgs &a, int lane, const Raw &raw)
{
    // the previous lane's thread_info: one lane shift over the whole wave (lane 0 starts the tile)
    const uint32_t ti_prev = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)raw.ti_cur, 0x138 /* wave_shr:1 */, 0xf, 0xf, true);
    uint32_t start = ti_prev >> 3, end = raw.ti_cur >> 3;
    if (start > raw.bn) start = raw.bn;
    if (end > raw.bn) end = raw.bn;
    if (end < start) end = start;
    const uint8_t *p = a.s.enc + raw.off;
    const uint32_t ahead = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 3u), from = ahead + start;
    return {p - ahead, from & ~3u, from & 3u, (from & 3u) + (end - start)};
}
// Word k of the lane's stream, whatever lies behind the payload's buffer: words that hold a byte of the stream, and zeros
__device__ __forceinline__ uint32_t kvc_lane_word(const KvcLane &l, uint32_t k)
{
    return l.bytes > l.skip && 4u * k < l.bytes ? kvc_load_at<uint32_t>(l.base, l.at + 4u * k) : 0u;
}
// Wave-uniform: the sixteen-byte loads of the tile's lanes stay inside the payload's buffer (all but a stream's last tiles)
template <class Raw>
__device__ __forceinline__ bool kvc_streams_inside(const KvcFusedArgs &a, const Raw &raw)
{
    return (int64_t)raw.off + raw.bn + 16 * KVC_PRE_CHUNKS <= a.s.enc_bytes;
}
// Loads of a tile's payload; rows: words of a stream that the LDS area holds.  Sets fits (wave-uniform: every stream is that short) and
// u0: `lead_bits` before the lane's first code, and a word on, so that it is never negative (kvc_column_address takes it off again).
template <class Raw>
__device__ __forceinline__ KvcStreams kvc_fetch_streams(const KvcFusedArgs &a, int lane, int rows, uint32_t lead_bits, Raw &raw)
{
    typedef uint32_t w4 __attribute__((ext_vector_type(4), aligned(4)));
    const KvcLane l = kvc_lane_stream(a, lane, raw);
    KvcStreams st;
    st.gwords = nullptr;
    st.gnwords = st.gpos = 0;
    st.fits = !__any((int)(l.bytes > 4u * (uint32_t)rows));
    st.u0 = l.skip * 8u + 32u - lead_bits;
    if (!kvc_streams_inside(a, raw)) return st;
#pragma unroll
    for (int j = 0; j < KVC_PRE_CHUNKS; j++) {
        if (4 * j >= rows) break;
        const w4 v = kvc_load_at<w4>(l.base, l.at + 16u * j);
        raw.pay[j] = make_uint4(v.x, v.y, v.z, v.w);
    }
    return st;
}
// ... into the columns.  column: LDS byte address of the lane's word in row 0.
template <class Raw>
__device__ __forceinline__ void kvc_stage_streams(const KvcFusedArgs &a, int lane, int rows, const Raw &raw, const KvcStreams &st, uint32_t column)
{
    if (!st.fits) return;
    kvc_lds_u32 *dst = (kvc_lds_u32 *)(uintptr_t)column;
    const bool inside = kvc_streams_inside(a, raw);
    if (inside) {
#pragma unroll
        for (int j = 0; j < KVC_PRE_CHUNKS; j++) {
            if (4 * j < rows) dst[64 * (4 * j)] = kvc_stream_word(raw.pay[j].x);
            if (4 * j + 1 < rows) dst[64 * (4 * j + 1)] = kvc_stream_word(raw.pay[j].y);
            if (4 * j + 2 < rows) dst[64 * (4 * j + 2)] = kvc_stream_word(raw.pay[j].z);
            if (4 * j + 3 < rows) dst[64 * (4 * j + 3)] = kvc_stream_word(raw.pay[j].w);
        }
        if (rows <= 4 * KVC_PRE_CHUNKS) return;
    }
    const KvcLane l = kvc_lane_stream(a, lane, raw);
#pragma unroll 1
    for (int k = inside ? 4 * KVC_PRE_CHUNKS : 0; k < rows; k++) dst[64 * k] = kvc_stream_word(kvc_lane_word(l, k));     // streams beyond 61 bytes
}
// What the one-symbol decoder needs to know of a lane's stream
template <class Raw>
__device__ __forceinline__ void kvc_stream_in_memory(const KvcFusedArgs &a, int lane, const Raw &raw, KvcStreams &st)
{
    const KvcLane l = kvc_lane_stream(a, lane, raw);
    st.gwords = reinterpret_cast<const uint32_t *>(l.base + l.at);
    st.gnwords = l.bytes > l.skip ? (l.bytes + 3u) >> 2 : 0u;
    st.gpos = l.skip * 8u;
}
// Byte address in LDS of row (u >> 5) - 1 of a lane's column; `column`: that of row 0.  A lane's position cannot pass its start by
// more than 128 codes of 7 bits, so even a corrupt stream stays within KVC_COLUMN_REACH rows; the row before the first is read too
// (bits before the first code, which nothing looks at).
constexpr int KVC_COLUMN_REACH = 34;
__device__ __forceinline__ uint32_t kvc_column_address(uint32_t column, uint32_t u)
{
    uint32_t row = u >> 5;
    asm("" : "+v"(row));                                                                  // (see kvc_refill_address)
    return (row << 8) + (column - 256u);
}
enum { KVC_BOOK_SHORT = 0, KVC_BOOK_MID = 1, KVC_BOOK_LONG = 2, KVC_BOOK_PACKED = 3 };       // of kvc_fused_mfma_kernel
// Which launches of the matrix-core kernels for codes of at most 7 bits take their payloads in columns (eight query heads: K's with one-byte
// entries only; the rest has no such kernels, V's took 41.3 us for 40.4 at 2 x 8 x 8 heads x 128 x 1905 tokens).  From `tiles` of a kind on: a
// wave of fewer waits for its one tile, which the lanes' own loads make longer, by how much depends on a stream's sixteen-byte loads.
// K with one-byte entries, whole attention calls over 4 x 8 KV heads with K packed, and what its columns add, us:
//   head_dim 128  1 query head  1024 tiles 23.1 +0.2   2048 24.2 +0.0   2560 26.1 -0.4      96  512 21.5 -0.3       72  256 20.2 -0.4
//                 2             1024       22.3 +0.8   2048 23.9 +0.5   2560 26.1 +0.0      96 1024 21.5 +0.4   2560 23.9 -0.2      72 2048 21.8 +0.1
//                 4             1024       26.6 +0.2   2048 28.0 +0.2   2560 30.5 -0.3      96 1024 25.7 +0.3   2560 28.5 -0.6      72 1024 24.3 -0.1
//                 8             1024       31.0 +0.5   2048 36.2 +0.2   2560 42.3 +0.0    3584 61.9 -6.1                        72 2048 34.3 +0.0
//   and the kernel alone at 32 768 tiles of 128, 1, 2, 4 and 8 query heads: 70, 73, 80 and 141 -> 61, 64, 72 and 118
// V with one-byte entries, the kernel with 1, 2 and 4 query heads: 512, 256 and 128 tiles 11.1 : 11.2, 10.5 : 10.7 and 12.4 : 12.0, 4096 tiles 16.0 :
// 14.2, 15.6 : 14.6 and 17.7 : 16.2.  Other codebooks (one query head; with two and four the same to 0.5 us):
//   K 2048 10.5 : 10.9   4096 13.2 : 13.3   8192 19.8 : 19.2      V 2048 9.4 : 10.1   3072 12.1 : 10.9   8192 20.7 : 19.8
// and products that are not rounded: K 2048 10.4 : 11.6   8192 21.5 : 23.3   16384 35.2 : 34.5    V 2048 11.0 : 11.6   4096 14.4 : 14.6   8192 23.8 : 22.4
constexpr int64_t kvc_columns_from(bool is_k, int rep, int head_dim, bool byte_entries, bool rounded)
{
    if (!rounded) return is_k ? 16384 : 4096;
    if (!byte_entries) return is_k ? 4096 : 3072;
    return !is_k || (rep == 1 && head_dim <= 96) || (rep == 4 && head_dim <= 72) ? 0 : 2560;
}
// ... and where the LDS still holds this many workgroups of a compute unit: columns are as long as the longest stream of the whole cache,
// packed payloads take their tile's bytes.  K of 4 x 32 heads x 96 x 32 768 tokens, packed 99 us: columns of 13, 17, 19, 21 and 29 words 84, 91,
// 96, 107 and 127 (eight, six, six, five and four workgroups); V (71): 6, 11 and 15 words 70, 73 and 80 (seven, six, five).  K and V of
// 8 x 8 heads x 128 x 8320, two query heads, 53: 17, 25 and 27 words 49, 51 and 60 (six, five, four); four query heads, 60: 17, 21 and 23 words 57,
// 58 and 74 (five, five, four), of head_dim 96 and 8192 tokens V (29.8): 12 and 19 words 27.9 and 28.5 (five, four; its registers allow four);
// eight, K and V 99: 21 and 23 words 95.8 and 99.1 (four, three).  K with wider entries of 7-bit codes, whose loop is longer: 8192 and 16 384 tiles of
// head_dim 128 (20 words, five) 25.9 and 41.2 -> 26.8 and 45.7 with two query heads, 28.3 and 50.1 -> 29.3 and 51.2 with four; of 72 (13
// words, eight and six) 16.6 and 27.0 -> 16.5 and 26.8, 19.6 and 30.8 -> 18.7 and 30.0.
constexpr int kvc_columns_workgroups(bool is_k, int rep, int slots, bool byte_entries)
{
    return rep == 1 || (is_k && !byte_entries) ? 6 : rep == 2 || (rep == 4 && slots == 1) ? 5 : 4;
}
enum { KVC_PACKED_PLAIN = 0, KVC_PACKED_SKEWED = 1, KVC_COLUMNS = 2 };
// The three words of a refill.  base: kvc_refill_address's, or the lane's column.
template <int LAYOUT, bool WORD = true>
__device__ __forceinline__ void kvc_refill(uint32_t base, uint32_t u, uint32_t &w0, uint32_t &w1, uint32_t &w2)
{
    constexpr int STEP = LAYOUT == KVC_COLUMNS ? KVC_WAVE : 1;
    const kvc_lds_word *wp = (const kvc_lds_word *)(uintptr_t)(LAYOUT == KVC_COLUMNS ? kvc_column_address(base, u) : kvc_refill_address<LAYOUT == KVC_PACKED_SKEWED, WORD>(base, u));
    w0 = wp[0];
    w1 = wp[STEP];
    w2 = wp[2 * STEP];
}

// Rows for the streams of a payload: the longest one where the encoder said it (it may start anywhere in its first word), else
// somewhat more than the mean
static inline int kvc_stream_rows(int64_t max_stream_bytes, int64_t encoded_bytes, int64_t tiles)
{
    const int64_t mean = encoded_bytes / (tiles > 0 ? tiles : 1) / KVC_WAVE;
    int64_t bytes = max_stream_bytes > 0 ? max_stream_bytes : mean + mean / 2 + 8;
    if (bytes > 112) bytes = 112;                                                         // 128 codes of 7 bits
    return (int)((bytes + 3 + 3) / 4);
}

// ---------------------------------------------------------------------------------------------------
// matrix-core variant (kvc_fused_mfma_impl.h)
// ---------------------------------------------------------------------------------------------------
// Columns of the operand matrix: every query head contributes a high and a low fp16 part of its weight, four
// columns per v_mfma_f32_4x4x4_16b_f16.
constexpr int kvc_mfma_sets(int rep) { return (2 * rep + 3) / 4; }
constexpr int KVC_MFMA_GROUPS = 32;       // groups of four elements per lane stream (128 / 4)
// LDS words per wave for the operand tables of one tile: per head slot 32 groups x sets x (4 columns x 4 fp16), and
// in rounded mode 32 groups x {two min pairs, two scale pairs}
constexpr int kvc_mfma_ops_words(int slots, int rep, bool rounded)
{
    return slots * (KVC_MFMA_GROUPS * kvc_mfma_sets(rep) * 8 + (rounded ? KVC_MFMA_GROUPS * 4 : 0));
}
// codes of more than 7 bits: 128 two-byte entries, then the list of those codes
constexpr int KVC_LONG_TABLE_WORDS = (1 << KVC_LUT_ESC_BITS) / 2 + 2 * KVC_LUT_ESC_MAX;
// rounded arithmetic only
void kvc_launch_fused_mid(int rep, int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream);
// kinds 0, 3 and 4, rounded arithmetic only
void kvc_launch_fused_long(int rep, int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream);
// payloads in columns: one, two or four query heads per KV head
void kvc_launch_fused_packed(int rep, int kind, bool rounded, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream);
void kvc_launch_fused_mfma(int rep, int kind, bool rounded, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream);
