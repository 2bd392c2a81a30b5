// kvc_common.h -- shared host/device definitions of libkvcomp_hip (gfx950, wave64).
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>
#include <stdarg.h>

#include "../../include/kvcomp_hip.h"

// ---------------------------------------------------------------------------------------------------
// geometry
// ---------------------------------------------------------------------------------------------------
constexpr int KVC_WAVE = 64;               // lanes per tile = vectors per tile (include/kernels.h:13,18)
#ifndef KVC_WAVES_PER_WG_VALUE
#define KVC_WAVES_PER_WG_VALUE 4
#endif
constexpr int KVC_WAVES_PER_WG = KVC_WAVES_PER_WG_VALUE;
constexpr int KVC_WG = KVC_WAVE * KVC_WAVES_PER_WG;
constexpr int KVC_V_TOKENS = 128;          // tokens per V vector (include/kernels.h:17)
constexpr int KVC_MAX_TILE_BYTES = 8191;   // thread_info is u16 = end_byte*8 + pad (include/kernels.h:30-32)

// Payload staging area of one wave in LDS: the tile payload plus the up-to-15 bytes that precede it
// in its first 16-byte chunk, rounded up, plus two guard words for the look-ahead of the last refill.
constexpr int KVC_STAGE_BYTES = ((KVC_MAX_TILE_BYTES + 15 + 15) / 16) * 16 + 16;   // 8224
constexpr int KVC_STAGE_WORDS = KVC_STAGE_BYTES / 4;

// ---------------------------------------------------------------------------------------------------
// decode look-up table (built on the device from the decode tree, see kvc_lut.hip)
//
//   header   {lbits, lmax, n_long, group, fused_group, fused_check, OR of the symbols' fp16 bit patterns, n_esc}
//   long[ ]  codes longer than lbits: {code left-aligned in 32 bits, len | sym << 8}
//   entry[ ] 1 << lbits words indexed by the next lbits stream bits: len | sym << 8, or 0 when the
//            code is longer than lbits (search long[]) or the bits match no code.
//   fentry[] for the fused kernels, indexed by the next lbits stream bits taken least-significant-bit first
//            (bit j of the index = j-th next stream bit): the symbol as an fp32 bit pattern with the code
//            length in its lowest mantissa byte (zero for any integer <= 255, so read as a float the entry
//            is the symbol to within 4e-6 relative, read as a shift count it is the length).  Indices
//            whose code is longer than lbits or that match no code hold "symbol 0, length 1".
//   narrow[] 64 counters behind esc[] and bit 31 of the header's word 6, see KVC_LUT_NARROW_OFFSET
//   esc[ ]   the n_esc codes longer than 7 bits (at most 64 are listed): {code, first stream bit in bit 0; len | sym << 8},
//            for the loops whose table index has 7 bits
//   group    how many symbols may be decoded from one 32-bit window: floor(32 / lmax), one of 8,4,2,1.
//   fused_group / fused_check
//            the same for the fused kernels, whose window has 30 usable bits: 8 if lmax <= 3, 4 if
//            lmax <= 7 (both guaranteed to fit); for longer codes 4 with fused_check = 1 when four symbols
//            are expected to stay well inside the window (mean code length, estimated from the code
//            lengths themselves as sum len * 2^-len, at most 5.5 bits), else 2.
// ---------------------------------------------------------------------------------------------------
constexpr int KVC_LUT_MAX_BITS = 10;
constexpr int KVC_LUT_MAX_LONG = 256;
constexpr int KVC_LUT_HEADER_WORDS = 8;
constexpr int KVC_LUT_LONG_WORDS = 2 * KVC_LUT_MAX_LONG;
constexpr int KVC_LUT_ENTRY_WORDS = 1 << KVC_LUT_MAX_BITS;
constexpr int KVC_LUT_FENTRY_OFFSET = KVC_LUT_HEADER_WORDS + KVC_LUT_LONG_WORDS + KVC_LUT_ENTRY_WORDS;
constexpr int KVC_LUT_ESC_OFFSET = KVC_LUT_FENTRY_OFFSET + KVC_LUT_ENTRY_WORDS;
constexpr int KVC_LUT_ESC_BITS = 7, KVC_LUT_ESC_MAX = 64;
// What V's kernels learn about the narrow two-symbol table (kvc_narrow_miss): counters behind the tables, each in a 64-byte
// line of its own, and a bit of the header word that holds the symbols' fp16 patterns, which turns the table off.
constexpr int KVC_LUT_NARROW_OFFSET = KVC_LUT_ESC_OFFSET + 2 * KVC_LUT_ESC_MAX;
constexpr int KVC_NARROW_LINE_WORDS = 16, KVC_NARROW_COUNTERS = 64;
constexpr int KVC_LUT_NARROW_WORD = 6;
// header word 6: some symbol is above 16 (see KVC_BYTE_CENTRE)
constexpr uint32_t KVC_LUT_WIDE_SYMBOLS = 0x10000u;
constexpr uint32_t KVC_LUT_NARROW_OFF = 0x80000000u;
constexpr int KVC_LUT_WORDS = KVC_LUT_NARROW_OFFSET + KVC_NARROW_LINE_WORDS * KVC_NARROW_COUNTERS;
constexpr int KVC_LUT_BYTES = KVC_LUT_WORDS * 4;          // 14880
static_assert(KVC_LUT_BYTES % 16 == 0, "decode tables of several codebooks lie one behind the other");
constexpr int KVC_TREE_MAX_NODES = 512;                   // 2 * 256 symbols - 2, rounded up

// ---------------------------------------------------------------------------------------------------
// host helpers (kvc_host.hip)
// ---------------------------------------------------------------------------------------------------
int kvc_fail(int code, const char *fmt, ...);
// Tuning knobs settable through kvc_set_option (or, before first use, KVCOMP_<NAME> in the environment).
enum KvcOption { KVC_OPT_FUSED_ROWS = 0, KVC_OPT_FUSED_TILES_PER_WAVE = 1, KVC_OPT_FUSED_PAIR_BITS = 2, KVC_OPT_FUSED_DOUBLE_WINDOW = 3, KVC_OPT_FUSED_SKEW = 4, KVC_OPT_DECODE_PIPELINED = 5, KVC_OPT_FUSED_ROUNDED = 6, KVC_OPT_ATTENTION_TAIL_IN_MERGE = 7, KVC_OPT_FUSED_MFMA = 8, KVC_OPT_FUSED_BUILTIN_DPP = 9, KVC_OPT_FUSED_SCHEDULE = 10, KVC_OPT_ENCODE_ONE_PASS = 11, KVC_OPT_FUSED_HALF_TABLE = 12, KVC_OPT_ENCODE_LOOKBACK_POLLS = 13, KVC_OPT_FUSED_SCHEDULE_V = 14, KVC_OPT_FUSED_TILES_PER_WAVE_V = 15, KVC_OPT_ATTENTION_JOINT = 16, KVC_OPT_COUNT };
int kvc_option(KvcOption which);
int kvc_check_hip(hipError_t e, const char *what);
// A slot of the per-device scratch ring (each slot holds KVC_WS_SLOT_BYTES); used for the LUT that the
// reference-signature entry points derive from the decode tree on every call.
constexpr size_t KVC_WS_SLOT_BYTES = 16384;
int kvc_workspace_slot(void **slot, void *stream);   // stream: the one the call launches on (a recorded call gets a slot of its own)
struct KvcCountsToHost {
    unsigned long long *host;      // pinned host memory: [256] counters, [256] the call's number, written last
    unsigned long long call;
    bool handed_over;              // by the quantizer; else the counters are on the device, for the caller to fetch and to clear
};
int kvc_quant_to_host(const void *d_x_f16, int64_t NB, int64_t BS, int64_t B, int64_t H, int64_t D, int quant_mask, float eb, uint8_t *d_sym,
                      bool packed, int8_t *d_min_i8, void *d_scale_f16, int64_t *d_counts, KvcCountsToHost *to_host, void *stream);
int kvc_quant_params(const void *d_x_f16, int64_t NB, int64_t BS, int64_t B, int64_t H, int64_t D, int quant_mask,
                     float eb, int8_t *d_min_i8, void *d_scale_f16, void *stream);
// What a caller that keeps its decode tables knows beyond the stream itself (all zero: nothing).
struct KvcDecodeHints {
    const uint32_t *luts;          // tables from kvc_build_lut; NULL: derived from the decode tree per call
    int64_t rows_per_codebook;
    int64_t max_tile_bytes, max_stream_bytes;
    int code_hint;                 // as kvc_compressed_desc::max_code_bits
};
// kvc_compressed_desc::max_code_bits: the longest code, whether every symbol is known to lie below 64, and
// kvc_codebook::pair_bits
static inline int kvc_hint_bits(int64_t hint) { return (int)(hint & 0xff); }
static inline int kvc_hint_pair_bits(int64_t hint) { return (int)(hint >> 12 & 7); }
static inline bool kvc_hint_byte_symbols(int64_t hint) { return (hint & 0x200) != 0; }      // none above 16
static inline bool kvc_hint_small_alphabet(int64_t hint) { return (hint & 0x100) != 0; }
int kvc_expand(int is_k, int deq, const uint8_t *d_decode_tree, int64_t decode_tree_bytes, int tree_format,
               const uint8_t *d_block_infos, int64_t block_infos_bytes, const uint8_t *d_thread_infos,
               int64_t thread_infos_bytes, const uint8_t *d_encoded, int64_t encoded_bytes, const int8_t *d_min,
               const void *d_scale, int quant_mask, void *d_out, int64_t tokens, int64_t batch, int64_t heads,
               int64_t head_dim, float *elapsed_ms, void *stream, const KvcDecodeHints &hints);
int kvc_launch_build_lut(const uint8_t *d_tree, int64_t tree_bytes, int tree_format, uint32_t *d_lut,
                         int n_codebooks, int64_t tree_stride_bytes, hipStream_t stream);

#define KVC_REQUIRE(cond, ...)                     \
    do {                                           \
        if (!(cond)) return kvc_fail(-1, __VA_ARGS__); \
    } while (0)
#define KVC_HIP(call)                              \
    do {                                           \
        int rc_ = kvc_check_hip((call), #call);    \
        if (rc_) return rc_;                       \
    } while (0)

// Optional event bracket implementing the reference's "returns elapsed milliseconds" contract
// (kvcomp_cuda_extension/src/kernels.cu:1026-1048).  The two events come from a small pool per device (kvc_host.hip):
// creating and destroying a pair costs a timed call more host time than recording it.
struct KvcEventPair {
    hipEvent_t a = nullptr, b = nullptr;
    int dev = -1;
};
KvcEventPair kvc_take_events();
void kvc_give_events(const KvcEventPair &p);
struct KvcTimer {
    KvcEventPair ev;
    hipStream_t s;
    float *out;
    KvcTimer(float *out_, hipStream_t s_) : s(s_), out(out_) {
        if (out) {
            ev = kvc_take_events();
            (void)hipEventRecord(ev.a, s);
        }
    }
    KvcTimer(const KvcTimer &) = delete;
    ~KvcTimer() { if (ev.a) kvc_give_events(ev); }
    int finish() {
        if (!out) return 0;
        hipError_t e = hipEventRecord(ev.b, s);
        if (e == hipSuccess) e = hipEventSynchronize(ev.b);
        if (e == hipSuccess) e = hipEventElapsedTime(out, ev.a, ev.b);
        return kvc_check_hip(e, "event timing");
    }
};

// ---------------------------------------------------------------------------------------------------
// device helpers
// ---------------------------------------------------------------------------------------------------
#ifdef __HIPCC__
// kvc_packed_symbols: symbols below 16 on their way from the quantizer to the encoder, two neighbouring channels to a byte, the
// even one in the low half.
//   V   [tokens][channels / 2], as the symbols themselves
//   K   a tile (64 tokens of one head) in 32 D bytes of its own, one tile behind the other; in it a token's D / 2 bytes in pieces
//       of 16 (4 where D is no multiple of 32), piece j of token t at (64 j + t) pieces: lane t of the encoder loads them in
//       whole lines, straight into the registers it packs from.
__device__ __forceinline__ constexpr uint32_t kvc_packed_k_chunk(uint32_t D) { return D % 32 == 0 ? 16u : 4u; }
// where in its tile the eight channels that channel c belongs to lie, four bytes
__device__ __forceinline__ constexpr uint32_t kvc_packed_k_place(uint32_t D, uint32_t c, uint32_t token)
{
    const uint32_t o = c >> 3;
    return D % 32 == 0 ? (o >> 2) * (16 * KVC_WAVE) + token * 16 + (o & 3) * 4 : o * (4 * KVC_WAVE) + token * 4;
}

__device__ __forceinline__ uint32_t kvc_bswap(uint32_t v) { return __builtin_bswap32(v); }

__device__ __forceinline__ float kvc_readlane(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

__device__ __forceinline__ float kvc_wave_sum(float v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

// Wave-wide reductions through the VALU's data-parallel lane permutes instead of LDS round trips; every lane
// of the wave must be active.  Six steps, each one instruction whose first operand is read through the
// permute: neighbours within quads (twice), quads within a row of 16 (rotate by 4, by 8: every lane of a row
// then holds the row's result), then the last lane of a row is combined into the following row (rows 1 and 3),
// and lane 31 into rows 2 and 3; lane 63 ends up with the total, which is read back as a scalar.  Rows that a
// step does not select keep their value.  A permuted read of a register needs two idle cycles after the
// instruction that wrote it, hence the s_nop between the steps (and in front: the input may have just been
// written).
#define KVC_DPP_REDUCE(op, v)                                                          \
    asm("s_nop 1\n\t" op " %0, %0, %0 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t" \
        "s_nop 1\n\t" op " %0, %0, %0 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n\t" \
        "s_nop 1\n\t" op " %0, %0, %0 row_ror:4 row_mask:0xf bank_mask:0xf\n\t"           \
        "s_nop 1\n\t" op " %0, %0, %0 row_ror:8 row_mask:0xf bank_mask:0xf\n\t"           \
        "s_nop 1\n\t" op " %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf\n\t"        \
        "s_nop 1\n\t" op " %0, %0, %0 row_bcast:31 row_mask:0xc bank_mask:0xf\n\t"        \
        "s_nop 1"                                                                          \
        : "+v"(v))

__device__ __forceinline__ float kvc_wave_sum_dpp(float v)
{
    KVC_DPP_REDUCE("v_add_f32_dpp", v);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ float kvc_wave_fmax_dpp(float v)
{
    KVC_DPP_REDUCE("v_max_f32_dpp", v);
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ uint32_t kvc_wave_max_dpp(uint32_t v)
{
    KVC_DPP_REDUCE("v_max_u32_dpp", v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// The kernel's argument block read again from the kernarg segment (scalar loads that hit the scalar cache): what a
// stretch of code needs of it is then live only where it is used, not in scalar registers through everything between
// (a kernel that needs more scalars than there are registers keeps the surplus in lanes of a vector register, and every
// access to those costs a vector instruction).
template <class T>
__device__ __forceinline__ const T &kvc_kernarg_again()
{
    auto p = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const T *)p;
}

// Sum over the 64 lanes, and inclusive prefix sum, the same way (every lane active).  The prefix sum adds lanes 1, 2, 4 and 8 to
// the left within rows of 16, then the rows' totals; as six shuffles through the LDS it took ten times as long.
__device__ __forceinline__ uint32_t kvc_wave_sum_dpp_u32(uint32_t v)
{
    KVC_DPP_REDUCE("v_add_u32_dpp", v);
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

__device__ __forceinline__ uint32_t kvc_wave_inclusive_scan(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);      // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);     // row_bcast:15 into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);     // row_bcast:31 into rows 2 and 3
    return v;
}
#endif
