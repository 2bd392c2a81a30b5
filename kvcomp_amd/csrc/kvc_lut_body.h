// kvc_lut_body.h -- decode tree to decode tables, by one workgroup: for kvc_lut.hip and for the launch behind a first store's
// encode (kvc_encode.hip).
//
// One 256-thread workgroup per codebook:
//   1. unpack the nodes into LDS (leaf flag, two children / the symbol);
//   2. record each node's parent and incoming bit, then every leaf walks up to the root: that gives its
//      code length, hence lmax, and the left-aligned code of every "long" code (length > lbits);
//   3. every table index walks down from the root along its own bits until it meets a leaf.
// All of it is waiting: for LDS, a read per step of a walk.  With a node in one word (leaf flag, then child: two reads after one
// another before) and one walk for both tables, 7.6 -> 7.1 us of the launch behind a large first store and 7.1 -> 6.3 behind a small one.
// A malformed tree (child index out of range, cycles) cannot hang or fault: walks are bounded by 32
// steps and indices are range-checked; the affected entries stay 0 (= "no code").
#pragma once
#include "kvc_common.h"

__device__ __forceinline__ void kvc_build_lut_body(const uint8_t *__restrict__ tree, int tree_bytes, int node_bytes, uint32_t *__restrict__ lut)
{
    // A step of a walk waits for one LDS read, so a node is one word: LEAF | symbol, or the two children, NONE where out of range; and so is
    // its way up: its parent, NONE at the root, and the bit that leads to it.
    constexpr uint32_t LEAF = 0x80000000u, NONE = 0x3ffu;
    static_assert(KVC_TREE_MAX_NODES <= (int)NONE, "node numbers of ten bits");
    __shared__ uint32_t s_node[KVC_TREE_MAX_NODES], s_up[KVC_TREE_MAX_NODES];
    __shared__ uint32_t s_lmax, s_nlong, s_nesc;
    __shared__ float s_avg;   // sum over leaves of len * 2^-len: the mean code length if the code is well matched
    __shared__ uint32_t s_symbits;   // OR over the symbols' fp16 patterns

    const int tid = threadIdx.x;
    int n_nodes = tree_bytes / node_bytes;
    if (n_nodes > KVC_TREE_MAX_NODES) n_nodes = KVC_TREE_MAX_NODES;

    if (tid == 0) { s_lmax = 0; s_nlong = 0; s_nesc = 0; s_avg = 0.f; s_symbits = 0; }
    for (int n = tid; n < KVC_TREE_MAX_NODES; n += KVC_WG) {
        int leaf = 0, a = -1, b = -1;
        if (n < n_nodes) {
            const uint8_t *p = tree + (int64_t)n * node_bytes;
            leaf = p[0] != 0;
            if (node_bytes == KVC_TREE_I8) {
                a = (int8_t)p[1];
                b = (int8_t)p[2];
            } else {
                a = (int16_t)(p[1] | (p[2] << 8));
                b = (int16_t)(p[3] | (p[4] << 8));
            }
            if (leaf) { a &= 0xff; b = a; }   // symbol value 0..255 (the int8 form stores it sign-wrapped)
        }
        auto child = [&](int c) { return c >= 0 && c < n_nodes ? (uint32_t)c : NONE; };
        s_node[n] = leaf ? LEAF | (uint32_t)a : child(a) | child(b) << 10;
        s_up[n] = NONE | (uint32_t)(n & 1) << 10;         // nodes 0 / 1 hang off the implicit root by bit 0 / 1
    }
    __syncthreads();
    for (int n = tid; n < n_nodes; n += KVC_WG) {
        const uint32_t node = s_node[n];
        if (node & LEAF) continue;
        for (int bit = 0; bit < 2; bit++) {
            const uint32_t c = (node >> (10 * bit)) & 0x3ffu;
            if (c >= 2u && c != NONE) s_up[c] = (uint32_t)n | (uint32_t)bit << 10;
        }
    }
    __syncthreads();
    // leaf -> root: length and code (bits arrive last-first)
    uint32_t my_len[KVC_TREE_MAX_NODES / KVC_WG], my_code[KVC_TREE_MAX_NODES / KVC_WG];
#pragma unroll
    for (int k = 0; k < KVC_TREE_MAX_NODES / KVC_WG; k++) {
        int n = tid + k * KVC_WG;
        my_len[k] = 0;
        my_code[k] = 0;
        if (n < n_nodes && (s_node[n] & LEAF)) {
            uint32_t len = 0, code = 0;
            int cur = n;
            while (len < 33) {
                const uint32_t up = s_up[cur];
                code |= (up >> 10) << (len & 31);
                len++;
                if ((up & 0x3ffu) == NONE) break;
                cur = (int)(up & 0x3ffu);
            }
            // a valid chain ends at node 0 or 1; anything else (orphan, over-long) is ignored
            if (len <= 32 && cur < 2) {
                my_len[k] = len;
                my_code[k] = code;
                atomicMax(&s_lmax, len);
                atomicAdd(&s_avg, (float)len * exp2f(-(float)len));
                const int sym = (int)(s_node[n] & 0xffu);
                atomicOr(&s_symbits, (uint32_t)__half_as_ushort(__float2half_rn((float)sym)) | (sym > 16 ? KVC_LUT_WIDE_SYMBOLS : 0u));
            }
        }
    }
    __syncthreads();
    const uint32_t lmax = s_lmax;
    const uint32_t lbits = lmax == 0 ? 1u : (lmax < (uint32_t)KVC_LUT_MAX_BITS ? lmax : (uint32_t)KVC_LUT_MAX_BITS);
#pragma unroll
    for (int k = 0; k < KVC_TREE_MAX_NODES / KVC_WG; k++) {
        if (my_len[k] > (uint32_t)KVC_LUT_ESC_BITS) {
            const uint32_t slot = atomicAdd(&s_nesc, 1u);
            if (slot < (uint32_t)KVC_LUT_ESC_MAX) {
                lut[KVC_LUT_ESC_OFFSET + 2 * slot] = __brev(my_code[k] << (32 - my_len[k]));
                lut[KVC_LUT_ESC_OFFSET + 2 * slot + 1] = my_len[k] | ((s_node[tid + k * KVC_WG] & 0xffu) << 8);
            }
        }
        if (my_len[k] > lbits) {
            uint32_t slot = atomicAdd(&s_nlong, 1u);
            if (slot < (uint32_t)KVC_LUT_MAX_LONG) {
                int n = tid + k * KVC_WG;
                lut[KVC_LUT_HEADER_WORDS + 2 * slot] = my_code[k] << (32 - my_len[k]);
                lut[KVC_LUT_HEADER_WORDS + 2 * slot + 1] = my_len[k] | ((s_node[n] & 0xffu) << 8);
            }
        }
    }
    // table entries: walk down along the index bits.  The fused kernels' entry is that of the reversed index: their index bits are the
    // stream bits in arrival order from bit 0 up (they keep their window least-significant-bit first).
    uint32_t *entries = lut + KVC_LUT_HEADER_WORDS + KVC_LUT_LONG_WORDS;
    for (uint32_t idx = tid; idx < (1u << lbits); idx += KVC_WG) {
        uint32_t e = 0, fused = 1u;            // no code / code longer than the index: none, and "symbol 0, length 1"
        uint32_t cur = (idx >> (lbits - 1)) & 1u;
        for (uint32_t depth = 1; depth <= lbits; depth++) {
            if (cur >= (uint32_t)n_nodes) break;
            const uint32_t node = s_node[cur];
            if (node & LEAF) {
                e = depth | (node & 0xffu) << 8;
                fused = __float_as_uint((float)(node & 0xffu)) | depth;
                break;
            }
            if (depth == lbits) break;
            cur = (node >> (10u * ((idx >> (lbits - 1 - depth)) & 1u))) & 0x3ffu;
        }
        entries[idx] = e;
        lut[KVC_LUT_FENTRY_OFFSET + (__brev(idx) >> (32u - lbits))] = fused;
    }
    for (int i = KVC_LUT_NARROW_OFFSET + tid; i < KVC_LUT_WORDS; i += KVC_WG) lut[i] = 0u;
    __syncthreads();
    if (tid == 0) {
        uint32_t nlong = s_nlong < (uint32_t)KVC_LUT_MAX_LONG ? s_nlong : (uint32_t)KVC_LUT_MAX_LONG;
        uint32_t group = lmax <= 4 ? 8u : lmax <= 8 ? 4u : lmax <= 16 ? 2u : 1u;
        lut[0] = lbits;
        lut[1] = lmax;
        lut[2] = nlong;
        lut[3] = group;
        const bool roomy = s_avg <= 5.5f;
        const bool roomy8 = lmax == 4 && s_avg <= 2.75f;
        // symbols that a 30-bit window is sure to hold (30 / lmax, at most 8); more where the average code is short
        // enough for the window to overflow rarely (lut[5] = 1: the kernel checks and falls back)
        lut[4] = (lmax <= 3 || roomy8) ? 8u : lmax <= 7 ? 30u / lmax : roomy ? 4u : 2u;
        lut[5] = (roomy8 || (lmax > 7 && roomy)) ? 1u : 0u;
        lut[6] = s_symbits;       // low bits clear in every symbol's fp16 pattern: room for lengths in a packed entry; KVC_LUT_WIDE_SYMBOLS
        lut[7] = s_nesc;
    }
}
