// kvc_sim.hip -- the dense caches of the simulated-quantization backend (models/cache/kvcomp_quant.py:14-124).
//
//   kvc_append_dense   <- apply_rotary_pos_emb_single (utils/compute.py:25-33) and the two safe_cat(..., dim=2) of an
//                         update: keys rotated and values copied straight to their place in the [B, H, capacity, D] caches
//   kvc_quant_in_place <- quant_error (utils/compute.py:108-133) on a stretch of such a cache
//   kvc_append_quantized  both, for the first tokens of a cache
//
// Both are bound by HBM for a prompt and by launches for a token: one launch per update of a layer (the rotation and the
// two appends took eight), and one or two for blocks that leave the tail, where they lie, without the contiguous copies
// that a [B, H, T, D] stretch with the strides of its capacity needed before and behind the quantizer.
#include "kvc_common.h"
#include "kvc_quant_math.h"

// ---------------------------------------------------------------------------------------------------
// append
// ---------------------------------------------------------------------------------------------------
template <int VEC>
struct KvcHalves {
    _Float16 v[VEC];
};
template <int VEC>
__device__ __forceinline__ KvcHalves<VEC> kvc_load_halves(const _Float16 *p)
{
    KvcHalves<VEC> r;
    if constexpr (VEC == 8) r = __builtin_bit_cast(KvcHalves<VEC>, *reinterpret_cast<const uint4 *>(p));
    else if constexpr (VEC == 4) r = __builtin_bit_cast(KvcHalves<VEC>, *reinterpret_cast<const uint2 *>(p));
    else r.v[0] = *p;
    return r;
}
template <int VEC>
__device__ __forceinline__ void kvc_store_halves(_Float16 *p, const KvcHalves<VEC> &r)
{
    if constexpr (VEC == 8) *reinterpret_cast<uint4 *>(p) = __builtin_bit_cast(uint4, r);
    else if constexpr (VEC == 4) *reinterpret_cast<uint2 *>(p) = __builtin_bit_cast(uint2, r);
    else *p = r.v[0];
}

// VEC adjacent channels of a new key from channel c on, and the VEC that lie half a head further on, which the rotation pairs
// them with.  The rotation is the reference's: t * cos and rotate_half(t) * sin, each rounded to fp16, then their sum.
template <int VEC>
__device__ __forceinline__ void kvc_rotated_key(const kvc_append_job &a, int64_t b, int64_t h, int64_t t, int c, int half, KvcHalves<VEC> &lo,
                                                KvcHalves<VEC> &hi)
{
#pragma clang fp contract(off)
    const _Float16 *p = reinterpret_cast<const _Float16 *>(a.d_k) + b * a.k_stride_b + h * a.k_stride_h + t * a.k_stride_t + c;
    lo = kvc_load_halves<VEC>(p);
    hi = kvc_load_halves<VEC>(p + half);
    if (a.d_cos) {                                         // uniform
        const _Float16 *cp = reinterpret_cast<const _Float16 *>(a.d_cos) + b * a.cos_stride_b + t * a.cos_stride_t + c;
        const _Float16 *sp = reinterpret_cast<const _Float16 *>(a.d_sin) + b * a.sin_stride_b + t * a.sin_stride_t + c;
        const KvcHalves<VEC> cl = kvc_load_halves<VEC>(cp), ch = kvc_load_halves<VEC>(cp + half);
        const KvcHalves<VEC> sl = kvc_load_halves<VEC>(sp), sh = kvc_load_halves<VEC>(sp + half);
#pragma unroll
        for (int k = 0; k < VEC; k++) {
            const _Float16 x = lo.v[k], y = hi.v[k];
            const _Float16 xc = x * cl.v[k], ys = -y * sl.v[k], yc = y * ch.v[k], xs = x * sh.v[k];
            lo.v[k] = xc + ys;
            hi.v[k] = yc + xs;
        }
    }
}

// A thread takes VEC adjacent channels of a token and their partners.  Grid (items, 2): y = 0 the keys from token k_from on,
// 1 the values from v_from on.
template <int VEC>
__global__ void __launch_bounds__(KVC_WG) kvc_append_dense_kernel(kvc_append_job a, int64_t k_from, int64_t v_from)
{
    const int half = (int)a.head_dim / 2, per = half / VEC;
    const int64_t item = (int64_t)blockIdx.x * KVC_WG + threadIdx.x, from = blockIdx.y ? v_from : k_from, tokens = a.tokens - from;
    if (item >= a.batch * a.heads * tokens * per) return;
    int64_t r = item / per;
    const int c = (int)(item - r * per) * VEC;
    const int64_t bh = r / tokens, t = r - bh * tokens + from, b = bh / a.heads, h = bh - b * a.heads;
    const int64_t to = (bh * a.capacity + a.at + t) * a.head_dim + c;
    if (blockIdx.y == 1) {
        const _Float16 *p = reinterpret_cast<const _Float16 *>(a.d_v) + b * a.v_stride_b + h * a.v_stride_h + t * a.v_stride_t + c;
        _Float16 *o = reinterpret_cast<_Float16 *>(a.d_v_cache) + to;
        const KvcHalves<VEC> lo = kvc_load_halves<VEC>(p), hi = kvc_load_halves<VEC>(p + half);
        kvc_store_halves<VEC>(o, lo);
        kvc_store_halves<VEC>(o + half, hi);
        return;
    }
    _Float16 *o = reinterpret_cast<_Float16 *>(a.d_k_cache) + to;
    KvcHalves<VEC> lo, hi;
    kvc_rotated_key<VEC>(a, b, h, t, c, half, lo, hi);
    kvc_store_halves<VEC>(o, lo);
    kvc_store_halves<VEC>(o + half, hi);
}

static int kvc_append_check(const kvc_append_job *job, int *vec)
{
    KVC_REQUIRE(job != nullptr, "NULL argument");
    const kvc_append_job &a = *job;
    KVC_REQUIRE(a.batch > 0 && a.heads > 0 && a.head_dim > 0 && a.head_dim % 2 == 0 && a.tokens >= 0, "bad shape");
    KVC_REQUIRE(a.at >= 0 && a.at + a.tokens <= a.capacity, "the cache holds %lld tokens, %lld + %lld are to lie in it", (long long)a.capacity,
                (long long)a.at, (long long)a.tokens);
    *vec = 1;
    if (a.tokens == 0) return 0;
    KVC_REQUIRE(a.d_k && a.d_v && a.d_k_cache && a.d_v_cache && (!a.d_cos == !a.d_sin), "NULL argument");
    // the widest loads that every address allows
    const int64_t half = a.head_dim / 2;
    uint64_t bits = (uint64_t)(uintptr_t)a.d_k | (uintptr_t)a.d_v | (uintptr_t)a.d_k_cache | (uintptr_t)a.d_v_cache | (uintptr_t)a.d_cos | (uintptr_t)a.d_sin;
    for (int64_t s : {a.k_stride_b, a.k_stride_h, a.k_stride_t, a.v_stride_b, a.v_stride_h, a.v_stride_t, a.cos_stride_b, a.cos_stride_t,
                      a.sin_stride_b, a.sin_stride_t, half})
        bits |= (uint64_t)s * 2;
    KVC_REQUIRE((bits & 1) == 0, "fp16 buffers are misaligned");
    *vec = (bits & 15) == 0 ? 8 : (bits & 7) == 0 ? 4 : 1;
    const int64_t wgs = (a.batch * a.heads * a.tokens * (half / *vec) + KVC_WG - 1) / KVC_WG;
    KVC_REQUIRE(wgs < (1ll << 31), "too many tokens for one call");
    return 0;
}

static int kvc_append_launch(const kvc_append_job &a, int vec, int64_t k_from, int64_t v_from, hipStream_t stream)
{
    const int64_t most = a.tokens - (k_from < v_from ? k_from : v_from);
    if (most <= 0) return 0;
    const dim3 grid((unsigned)((a.batch * a.heads * most * (a.head_dim / 2 / vec) + KVC_WG - 1) / KVC_WG), 2);
    if (vec == 8) hipLaunchKernelGGL(kvc_append_dense_kernel<8>, grid, dim3(KVC_WG), 0, stream, a, k_from, v_from);
    else if (vec == 4) hipLaunchKernelGGL(kvc_append_dense_kernel<4>, grid, dim3(KVC_WG), 0, stream, a, k_from, v_from);
    else hipLaunchKernelGGL(kvc_append_dense_kernel<1>, grid, dim3(KVC_WG), 0, stream, a, k_from, v_from);
    return kvc_check_hip(hipGetLastError(), "kvc_append_dense_kernel launch");
}

extern "C" int kvc_append_dense(const kvc_append_job *job, void *stream)
{
    int vec;
    if (int rc = kvc_append_check(job, &vec)) return rc;
    return kvc_append_launch(*job, vec, 0, 0, (hipStream_t)stream);
}

// ---------------------------------------------------------------------------------------------------
// simulated quantization where the tokens lie
// ---------------------------------------------------------------------------------------------------
struct KvcInPlaceArgs {
    _Float16 *x;                  // first token of the stretch, batch entry 0, head 0
    int64_t stride_b, stride_h;   // elements; a token's row follows the one before it
    const _Float16 *from;         // where the tokens are read (x itself, unless they are appended by the same launch)
    int64_t from_b, from_h, from_t;
    int NB, BS, B, H, D;
    float eb;
    uint32_t *minmax;             // block groups: {ord(min), ord(max)} per (batch entry, block)
};

__device__ __forceinline__ kvc_half2 kvc_as_half2(uint32_t w) { return __builtin_bit_cast(kvc_half2, w); }

// what a group's elements become
struct KvcRequant {
    bool packed;
    KvcGroupParams g;
    KvcPackedParams pp;
    uint32_t min2, scale2;
    __device__ __forceinline__ KvcRequant(float lo, float hi, float eb)
    {
        g = kvc_group_params(lo, hi, eb);
        packed = kvc_packed_quantizer_applies(g, hi);      // else: quotients beyond the packed arithmetic's range, or a zero scale
        pp = kvc_packed_params(g, g);
        min2 = kvc_half_pair_bits(g.min_h, g.min_h);
        scale2 = kvc_half_pair_bits(g.scale_h, g.scale_h);
    }
    __device__ __forceinline__ uint32_t pair(uint32_t w) const
    {
        if (packed) return kvc_quant_error_pair(kvc_quant_pair_biased(w, pp), min2, scale2);
        return kvc_half_pair_bits(kvc_quant_error_one(kvc_half_lo(w), g), kvc_quant_error_one(kvc_half_hi(w), g));
    }
    __device__ __forceinline__ uint4 eight(const uint4 &v) const { return make_uint4(pair(v.x), pair(v.y), pair(v.z), pair(v.w)); }
};

// Per-channel groups: a thread owns two channels of one (batch entry, head, block).  Blocks of 64 tokens stay in registers.
template <bool ONCE>
__global__ void __launch_bounds__(KVC_WG) kvc_in_place_channel_kernel(KvcInPlaceArgs a)
{
    const int pairs = a.D >> 1;
    const int64_t gid = (int64_t)blockIdx.x * KVC_WG + threadIdx.x;
    if (gid >= (int64_t)a.B * a.H * a.NB * pairs) return;
    const int64_t r = gid / pairs;
    const int c = (int)(gid - r * pairs) * 2;
    const int64_t bh = r / a.NB, nb = r - bh * a.NB, b = bh / a.H, h = bh - b * a.H;
    _Float16 *p = a.x + b * a.stride_b + h * a.stride_h + nb * a.BS * a.D + c;
    kvc_half2 mn, mx;
    auto at = [&](int t) -> uint32_t & { return *reinterpret_cast<uint32_t *>(p + (int64_t)t * a.D); };
    uint32_t raw[ONCE ? KVC_WAVE : 1];
    if constexpr (ONCE) {
#pragma unroll
        for (int t = 0; t < KVC_WAVE; t++) raw[t] = at(t);
        mn = mx = kvc_as_half2(raw[0]);
#pragma unroll
        for (int t = 1; t < KVC_WAVE; t++) {
            mn = __builtin_elementwise_min(mn, kvc_as_half2(raw[t]));
            mx = __builtin_elementwise_max(mx, kvc_as_half2(raw[t]));
        }
    } else {
        mn = mx = kvc_as_half2(at(0));
        for (int t = 1; t < a.BS; t++) {
            const kvc_half2 x = kvc_as_half2(at(t));
            mn = __builtin_elementwise_min(mn, x);
            mx = __builtin_elementwise_max(mx, x);
        }
    }
    const uint32_t mnw = __builtin_bit_cast(uint32_t, mn), mxw = __builtin_bit_cast(uint32_t, mx);
    const KvcGroupParams g0 = kvc_group_params(kvc_half_lo(mnw), kvc_half_lo(mxw), a.eb);
    const KvcGroupParams g1 = kvc_group_params(kvc_half_hi(mnw), kvc_half_hi(mxw), a.eb);
    const bool packed = kvc_packed_quantizer_applies(g0, kvc_half_lo(mxw)) && kvc_packed_quantizer_applies(g1, kvc_half_hi(mxw));
    const KvcPackedParams pp = kvc_packed_params(g0, g1);
    const uint32_t min2 = kvc_half_pair_bits(g0.min_h, g1.min_h), scale2 = kvc_half_pair_bits(g0.scale_h, g1.scale_h);
    auto value = [&](uint32_t w) {
        if (packed) return kvc_quant_error_pair(kvc_quant_pair_biased(w, pp), min2, scale2);
        return kvc_half_pair_bits(kvc_quant_error_one(kvc_half_lo(w), g0), kvc_quant_error_one(kvc_half_hi(w), g1));
    };
    if constexpr (ONCE) {
#pragma unroll
        for (int t = 0; t < KVC_WAVE; t++) at(t) = value(raw[t]);
    } else {
        for (int t = 0; t < a.BS; t++) at(t) = value(at(t));
    }
}

// New keys with per-channel groups over blocks of 64 tokens, rotated, quantized and put in place by one launch (appended
// first and then quantized in place, a prompt's keys went over the bus twice more).  A workgroup takes a (batch entry, head,
// block): sixteen bytes of a token and their partners per load; the rotated block lies in LDS for the channels' minima and
// maxima, and stays in registers to be quantized.  Bound by HBM: K of 4 x 32 heads x 128 x 2048 tokens 35 us (134 MB), V, whose
// tokens are read where they come from, 26; appended first (43) and then quantized in place (28 and 29) the two took 99.  A cache update with
// that prompt and two more tokens: 110 -> 72 us; with 32 more the host's calls take longer than the prompt (576 -> 570).
template <int ITEMS>
__global__ void __launch_bounds__(KVC_WG) kvc_append_channel_kernel(kvc_append_job a, int NB, float eb)
{
    constexpr int BS = KVC_WAVE, PAIRS = KVC_K_VEC_LEN / 2;
    __shared__ __align__(16) uint32_t s_tile[BS * PAIRS];              // [token][channel pair]
    __shared__ __align__(16) uint2 s_minmax[KVC_WG];                   // {minima, maxima} of a pair's part of the block, then of the block
    __shared__ __align__(16) uint4 s_packed[PAIRS];
    __shared__ __align__(16) uint4 s_value[PAIRS];                     // {min2, scale2, whether the packed arithmetic applies}
    const int tid = threadIdx.x, D = (int)a.head_dim, half = D / 2, per = half / 8, pairs = D / 2;
    const int64_t bh = blockIdx.x / (unsigned)NB, nb = blockIdx.x - bh * NB, b = bh / a.heads, h = bh - b * a.heads;
    KvcHalves<8> lo[ITEMS], hi[ITEMS];
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const int item = tid + KVC_WG * j, t = item / per, c = (item - t * per) * 8;
        if (t < BS) kvc_rotated_key<8>(a, b, h, nb * BS + t, c, half, lo[j], hi[j]);
    }
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const int item = tid + KVC_WG * j, t = item / per, c = (item - t * per) * 8;
        if (t < BS) {
            *reinterpret_cast<uint4 *>(s_tile + t * pairs + c / 2) = __builtin_bit_cast(uint4, lo[j]);
            *reinterpret_cast<uint4 *>(s_tile + t * pairs + (c + half) / 2) = __builtin_bit_cast(uint4, hi[j]);
        }
    }
    __syncthreads();
    const int parts = KVC_WG / pairs, part = tid / pairs, pair = tid - part * pairs;
    if (part < parts) {
        kvc_half2 mn = kvc_as_half2(s_tile[part * pairs + pair]), mx = mn;
        for (int t = part + parts; t < BS; t += parts) {
            const kvc_half2 x = kvc_as_half2(s_tile[t * pairs + pair]);
            mn = __builtin_elementwise_min(mn, x);
            mx = __builtin_elementwise_max(mx, x);
        }
        s_minmax[tid] = make_uint2(__builtin_bit_cast(uint32_t, mn), __builtin_bit_cast(uint32_t, mx));
    }
    __syncthreads();
    if (tid < pairs) {
        kvc_half2 mn = kvc_as_half2(s_minmax[tid].x), mx = kvc_as_half2(s_minmax[tid].y);
        for (int q = 1; q < parts; q++) {
            mn = __builtin_elementwise_min(mn, kvc_as_half2(s_minmax[tid + q * pairs].x));
            mx = __builtin_elementwise_max(mx, kvc_as_half2(s_minmax[tid + q * pairs].y));
        }
        const uint32_t mnw = __builtin_bit_cast(uint32_t, mn), mxw = __builtin_bit_cast(uint32_t, mx);
        const KvcGroupParams g0 = kvc_group_params(kvc_half_lo(mnw), kvc_half_lo(mxw), eb), g1 = kvc_group_params(kvc_half_hi(mnw), kvc_half_hi(mxw), eb);
        const bool packed = kvc_packed_quantizer_applies(g0, kvc_half_lo(mxw)) && kvc_packed_quantizer_applies(g1, kvc_half_hi(mxw));
        const KvcPackedParams pp = kvc_packed_params(g0, g1);
        s_packed[tid] = make_uint4(pp.P2, pp.S2, pp.r2, pp.c2);
        s_value[tid] = make_uint4(kvc_half_pair_bits(g0.min_h, g1.min_h), kvc_half_pair_bits(g0.scale_h, g1.scale_h), packed ? 1u : 0u, 0u);
        s_minmax[tid] = make_uint2(mnw, mxw);
    }
    __syncthreads();
    auto value = [&](uint32_t w, int p) {
        const uint4 c = s_packed[p], v = s_value[p];
        if (v.z) return kvc_quant_error_pair(kvc_quant_pair_biased(w, KvcPackedParams{c.x, c.y, c.z, c.w}), v.x, v.y);
        const uint2 mm = s_minmax[p];
        const KvcGroupParams g0 = kvc_group_params(kvc_half_lo(mm.x), kvc_half_lo(mm.y), eb), g1 = kvc_group_params(kvc_half_hi(mm.x), kvc_half_hi(mm.y), eb);
        return kvc_half_pair_bits(kvc_quant_error_one(kvc_half_lo(w), g0), kvc_quant_error_one(kvc_half_hi(w), g1));
    };
#pragma unroll
    for (int j = 0; j < ITEMS; j++) {
        const int item = tid + KVC_WG * j, t = item / per, c = (item - t * per) * 8;
        if (t >= BS) continue;
        _Float16 *o = reinterpret_cast<_Float16 *>(a.d_k_cache) + (bh * a.capacity + a.at + nb * BS + t) * D + c;
        const uint4 x = __builtin_bit_cast(uint4, lo[j]), y = __builtin_bit_cast(uint4, hi[j]);
        const int p = c / 2, q = (c + half) / 2;
        *reinterpret_cast<uint4 *>(o) = make_uint4(value(x.x, p), value(x.y, p + 1), value(x.z, p + 2), value(x.w, p + 3));
        *reinterpret_cast<uint4 *>(o + half) = make_uint4(value(y.x, q), value(y.y, q + 1), value(y.z, q + 2), value(y.w, q + 3));
    }
}

// Per-vector groups: a group is one token's row of one head; 16 lanes take it, eight elements each.
__global__ void __launch_bounds__(KVC_WG) kvc_in_place_vector_kernel(KvcInPlaceArgs a)
{
    const int64_t tokens = (int64_t)a.NB * a.BS;
    const int64_t r = ((int64_t)blockIdx.x * KVC_WG + threadIdx.x) >> 4;
    const int c = 8 * (threadIdx.x & 15);
    const bool row = r < (int64_t)a.B * a.H * tokens, live = row && c < a.D;
    const int64_t bh = r / tokens, t = r - bh * tokens, b = bh / a.H, h = bh - b * a.H;
    uint4 *p = reinterpret_cast<uint4 *>(a.x + b * a.stride_b + h * a.stride_h + t * a.D + c);
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    float lo = INFINITY, hi = -INFINITY;
    if (live) {
        v = *reinterpret_cast<const uint4 *>(a.from + b * a.from_b + h * a.from_h + t * a.from_t + c);
        kvc_half2 mn = kvc_as_half2(v.x), mx = mn;
        for (uint32_t w : {v.y, v.z, v.w}) {
            mn = __builtin_elementwise_min(mn, kvc_as_half2(w));
            mx = __builtin_elementwise_max(mx, kvc_as_half2(w));
        }
        const uint32_t mnw = __builtin_bit_cast(uint32_t, mn), mxw = __builtin_bit_cast(uint32_t, mx);
        lo = fminf(kvc_half_lo(mnw), kvc_half_hi(mnw));
        hi = fmaxf(kvc_half_lo(mxw), kvc_half_hi(mxw));
    }
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) {
        lo = fminf(lo, __shfl_xor(lo, off, 64));
        hi = fmaxf(hi, __shfl_xor(hi, off, 64));
    }
    if (!live) return;
    const KvcRequant q(lo, hi, a.eb);
    *p = q.eight(v);
}

// Per-token groups: the H rows of one token of one batch entry, which lie a head's stretch apart.  WPR waves per token keep
// them in registers, NIT pieces of eight elements per lane.
template <int NIT, int WPR>
__global__ void __launch_bounds__(KVC_WG) kvc_in_place_token_kernel(KvcInPlaceArgs a)
{
    __shared__ float s_lo[KVC_WAVES_PER_WG], s_hi[KVC_WAVES_PER_WG];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t tokens = (int64_t)a.NB * a.BS;
    const int64_t g = WPR == 1 ? (int64_t)blockIdx.x * KVC_WAVES_PER_WG + wave : (int64_t)blockIdx.x;
    if (g >= a.B * tokens) return;                         // (uniform over the waves that share a token)
    const int64_t b = g / tokens, t = g - b * tokens;
    _Float16 *x = a.x + b * a.stride_b + t * a.D;
    const int at = WPR == 1 ? lane : (int)threadIdx.x, per = a.D >> 3, pieces = a.H * per;
    const _Float16 *from = a.from + b * a.from_b + t * a.from_t;
    auto where = [&](int j) {
        const int i = at + 64 * WPR * j, h = i / per;
        return reinterpret_cast<uint4 *>(x + h * a.stride_h + 8 * (i - h * per));
    };
    auto read = [&](int j) {
        const int i = at + 64 * WPR * j, h = i / per;
        return *reinterpret_cast<const uint4 *>(from + h * a.from_h + 8 * (i - h * per));
    };
    uint4 raw[NIT];
    kvc_half2 mn = {(_Float16)INFINITY, (_Float16)INFINITY}, mx = -mn;
#pragma unroll
    for (int j = 0; j < NIT; j++)
        if (at + 64 * WPR * j < pieces) raw[j] = read(j);
#pragma unroll
    for (int j = 0; j < NIT; j++) {
        if (at + 64 * WPR * j < pieces) {
            for (uint32_t w : {raw[j].x, raw[j].y, raw[j].z, raw[j].w}) {
                mn = __builtin_elementwise_min(mn, kvc_as_half2(w));
                mx = __builtin_elementwise_max(mx, kvc_as_half2(w));
            }
        }
    }
    const uint32_t mnw = __builtin_bit_cast(uint32_t, mn), mxw = __builtin_bit_cast(uint32_t, mx);
    float lo = kvc_wave_min(fminf(kvc_half_lo(mnw), kvc_half_hi(mnw)));
    float hi = kvc_wave_max(fmaxf(kvc_half_lo(mxw), kvc_half_hi(mxw)));
    if constexpr (WPR > 1) {
        if (lane == 0) {
            s_lo[wave] = lo;
            s_hi[wave] = hi;
        }
        __syncthreads();
#pragma unroll
        for (int w = 0; w < WPR; w++) {
            lo = fminf(lo, s_lo[w]);
            hi = fmaxf(hi, s_hi[w]);
        }
    }
    const KvcRequant q(lo, hi, a.eb);
#pragma unroll
    for (int j = 0; j < NIT; j++)
        if (at + 64 * WPR * j < pieces) *where(j) = q.eight(raw[j]);
}
constexpr int64_t KVC_IN_PLACE_TOKEN_MAX = 512 * KVC_WAVES_PER_WG * 32;

// Block groups: all heads and tokens of one block of one batch entry.  A wave takes the contiguous BS * D elements of one
// head: first their minimum and maximum, merged per group with atomics, then, in a second launch, their new values.
__global__ void __launch_bounds__(KVC_WG) kvc_in_place_block_init_kernel(uint32_t *minmax, int groups)
{
    const int g = blockIdx.x * KVC_WG + threadIdx.x;
    if (g < groups) {
        minmax[2 * g] = 0xffffffffu;
        minmax[2 * g + 1] = 0u;
    }
}
template <bool APPLY>
__global__ void __launch_bounds__(KVC_WG) kvc_in_place_block_kernel(KvcInPlaceArgs a)
{
    const int lane = threadIdx.x & 63;
    const int64_t r = (int64_t)blockIdx.x * KVC_WAVES_PER_WG + (threadIdx.x >> 6);
    if (r >= (int64_t)a.B * a.H * a.NB) return;
    const int64_t bh = r / a.NB, nb = r - bh * a.NB, b = bh / a.H, h = bh - b * a.H;
    uint4 *p = reinterpret_cast<uint4 *>(a.x + b * a.stride_b + h * a.stride_h + nb * a.BS * a.D);
    const int n = a.BS * a.D / 8;
    uint32_t *group = a.minmax + 2 * (b * a.NB + nb);
    if constexpr (APPLY) {
        const KvcRequant q(kvc_ord2f(group[0]), kvc_ord2f(group[1]), a.eb);
#pragma unroll 4
        for (int i = lane; i < n; i += KVC_WAVE) p[i] = q.eight(p[i]);
    } else {
        kvc_half2 mn = {(_Float16)INFINITY, (_Float16)INFINITY}, mx = -mn;
#pragma unroll 4
        for (int i = lane; i < n; i += KVC_WAVE) {
            const uint4 v = p[i];
            for (uint32_t w : {v.x, v.y, v.z, v.w}) {
                mn = __builtin_elementwise_min(mn, kvc_as_half2(w));
                mx = __builtin_elementwise_max(mx, kvc_as_half2(w));
            }
        }
        const uint32_t mnw = __builtin_bit_cast(uint32_t, mn), mxw = __builtin_bit_cast(uint32_t, mx);
        const float lo = kvc_wave_min(fminf(kvc_half_lo(mnw), kvc_half_hi(mnw)));
        const float hi = kvc_wave_max(fmaxf(kvc_half_lo(mxw), kvc_half_hi(mxw)));
        if (lane == 0) {
            atomicMin(&group[0], kvc_f2ord(lo));
            atomicMax(&group[1], kvc_f2ord(hi));
        }
    }
}

static dim3 kvc_wgs(int64_t threads) { return dim3((unsigned)((threads + KVC_WG - 1) / KVC_WG)); }

// groups of one token of one batch entry, or of one token of one head
static void kvc_launch_token_groups(const KvcInPlaceArgs &a, int quant_mask, hipStream_t stream)
{
    const int64_t tokens = (int64_t)a.NB * a.BS, row = (int64_t)a.H * a.D;
    if (quant_mask == KVC_MASK_VECTOR) {
        hipLaunchKernelGGL(kvc_in_place_vector_kernel, kvc_wgs(a.B * a.H * tokens * 16), dim3(KVC_WG), 0, stream, a);
        return;
    }
    constexpr int W = KVC_WAVES_PER_WG;
    const dim3 one = kvc_wgs(a.B * tokens * KVC_WAVE), all((unsigned)(a.B * tokens));
    if (row <= 512 * 4) hipLaunchKernelGGL((kvc_in_place_token_kernel<4, 1>), one, dim3(KVC_WG), 0, stream, a);
    else if (row <= 512 * 8) hipLaunchKernelGGL((kvc_in_place_token_kernel<8, 1>), one, dim3(KVC_WG), 0, stream, a);
    else if (row <= 512 * 16) hipLaunchKernelGGL((kvc_in_place_token_kernel<16, 1>), one, dim3(KVC_WG), 0, stream, a);
    else if (row <= 512 * W * 16) hipLaunchKernelGGL((kvc_in_place_token_kernel<16, W>), all, dim3(KVC_WG), 0, stream, a);
    else hipLaunchKernelGGL((kvc_in_place_token_kernel<32, W>), all, dim3(KVC_WG), 0, stream, a);
}

// 1: not a layout these kernels take
extern "C" int kvc_quant_in_place(void *d_x_f16, int64_t B, int64_t H, int64_t tokens, int64_t D, int64_t stride_b, int64_t stride_h,
                                  int64_t block_size, int quant_mask, float eb, void *stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    KVC_REQUIRE(B > 0 && H > 0 && D > 0 && tokens >= 0 && block_size > 0 && tokens % block_size == 0, "bad shape");
    KVC_REQUIRE(eb > 0.f, "error bound must be positive");
    if (tokens == 0) return 0;
    KVC_REQUIRE(d_x_f16 != nullptr, "NULL argument");
    if (D % 8 != 0 || ((uintptr_t)d_x_f16 & 15) != 0 || stride_b % 8 != 0 || stride_h % 8 != 0 || D > 128 || B * H * tokens >= (1ll << 31)) return 1;
    KvcInPlaceArgs a;
    a.x = reinterpret_cast<_Float16 *>(d_x_f16);
    a.stride_b = stride_b;
    a.stride_h = stride_h;
    a.NB = (int)(tokens / block_size);
    a.BS = (int)block_size;
    a.B = (int)B;
    a.H = (int)H;
    a.D = (int)D;
    a.eb = eb;
    a.minmax = nullptr;
    a.from = a.x;
    a.from_b = stride_b;
    a.from_h = stride_h;
    a.from_t = D;
    if (quant_mask == KVC_MASK_CHANNEL) {
        const dim3 grid = kvc_wgs(B * H * a.NB * (D / 2));
        if (block_size == KVC_WAVE) hipLaunchKernelGGL(kvc_in_place_channel_kernel<true>, grid, dim3(KVC_WG), 0, stream, a);
        else hipLaunchKernelGGL(kvc_in_place_channel_kernel<false>, grid, dim3(KVC_WG), 0, stream, a);
    } else if (quant_mask == KVC_MASK_VECTOR || quant_mask == KVC_MASK_SIM_TOKEN) {
        if (quant_mask == KVC_MASK_SIM_TOKEN && H * D > KVC_IN_PLACE_TOKEN_MAX) return 1;
        kvc_launch_token_groups(a, quant_mask, stream);
    } else if (quant_mask == KVC_MASK_SIM_BLOCK) {
        const int groups = (int)B * a.NB;
        if ((size_t)groups * 8 > KVC_WS_SLOT_BYTES) return 1;
        void *slot;
        if (int rc = kvc_workspace_slot(&slot, stream_)) return rc;
        a.minmax = reinterpret_cast<uint32_t *>(slot);
        const dim3 grid = kvc_wgs(B * H * a.NB * KVC_WAVE);
        hipLaunchKernelGGL(kvc_in_place_block_init_kernel, kvc_wgs(groups), dim3(KVC_WG), 0, stream, a.minmax, groups);
        hipLaunchKernelGGL(kvc_in_place_block_kernel<false>, grid, dim3(KVC_WG), 0, stream, a);
        hipLaunchKernelGGL(kvc_in_place_block_kernel<true>, grid, dim3(KVC_WG), 0, stream, a);
    } else {
        return kvc_fail(-1, "unsupported quantization group mask 0x%x", quant_mask);
    }
    return kvc_check_hip(hipGetLastError(), "in-place quantizer launch");
}

// ---------------------------------------------------------------------------------------------------
// both at once, for a prompt
// ---------------------------------------------------------------------------------------------------
// 1: not tensors or groups this takes
extern "C" int kvc_append_quantized(const kvc_append_job *job, int64_t k_tokens, int64_t k_block_size, int k_mask, float k_eb, int64_t v_tokens,
                                    int64_t v_block_size, int v_mask, float v_eb, void *stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    int vec;
    if (int rc = kvc_append_check(job, &vec)) return rc;
    const kvc_append_job &a = *job;
    KVC_REQUIRE(k_block_size > 0 && v_block_size > 0 && k_tokens >= 0 && v_tokens >= 0 && k_tokens <= a.tokens && v_tokens <= a.tokens &&
                    k_tokens % k_block_size == 0 && v_tokens % v_block_size == 0, "bad stretch");
    KVC_REQUIRE(k_eb > 0.f && v_eb > 0.f, "error bound must be positive");
    const int64_t D = a.head_dim, blocks = k_tokens / KVC_WAVE;
    if (vec != 8 || D % 16 != 0 || D > KVC_K_VEC_LEN || k_mask != KVC_MASK_CHANNEL || k_block_size != KVC_WAVE) return 1;
    if (!(v_mask == KVC_MASK_VECTOR || (v_mask == KVC_MASK_SIM_TOKEN && a.heads * D <= KVC_IN_PLACE_TOKEN_MAX))) return 1;
    if (a.batch * a.heads * a.tokens >= (1ll << 31)) return 1;
    if (blocks > 0) {
        const dim3 grid((unsigned)(a.batch * a.heads * blocks));
        if (D / 16 * KVC_WAVE <= KVC_WG) hipLaunchKernelGGL(kvc_append_channel_kernel<1>, grid, dim3(KVC_WG), 0, stream, a, (int)blocks, k_eb);
        else hipLaunchKernelGGL(kvc_append_channel_kernel<2>, grid, dim3(KVC_WG), 0, stream, a, (int)blocks, k_eb);
    }
    if (v_tokens > 0) {
        KvcInPlaceArgs v = {};
        v.x = reinterpret_cast<_Float16 *>(a.d_v_cache) + a.at * D;
        v.stride_b = a.heads * a.capacity * D;
        v.stride_h = a.capacity * D;
        v.from = reinterpret_cast<const _Float16 *>(a.d_v);
        v.from_b = a.v_stride_b;
        v.from_h = a.v_stride_h;
        v.from_t = a.v_stride_t;
        v.NB = (int)(v_tokens / v_block_size);
        v.BS = (int)v_block_size;
        v.B = (int)a.batch;
        v.H = (int)a.heads;
        v.D = (int)D;
        v.eb = v_eb;
        kvc_launch_token_groups(v, v_mask, stream);
    }
    if (int rc = kvc_append_launch(a, vec, k_tokens, v_tokens, stream)) return rc;
    return kvc_check_hip(hipGetLastError(), "append and quantize launch");
}
