// kvc_lut.hip -- turns a decode tree (the reference's 3-byte node array, src/huffman.cpp:229-252, or
// the wide 5-byte variant) into the table-driven form the decoders use.
//
// One 256-thread workgroup per codebook (kvc_lut_body.h).
#include "kvc_common.h"
#include "kvc_lut_body.h"

#include <cstring>

__global__ void __launch_bounds__(KVC_WG)
kvc_build_lut_kernel(const uint8_t *__restrict__ trees, int64_t tree_stride, int tree_bytes, int node_bytes,
                     uint32_t *__restrict__ luts)
{
    kvc_build_lut_body(trees + (int64_t)blockIdx.x * tree_stride, tree_bytes, node_bytes, luts + (int64_t)blockIdx.x * KVC_LUT_WORDS);
}

static int kvc_check_tree(int64_t tree_bytes, int tree_format)
{
    KVC_REQUIRE(tree_format == KVC_TREE_I8 || tree_format == KVC_TREE_I16, "unknown tree format %d", tree_format);
    KVC_REQUIRE(tree_bytes >= 2 * tree_format && tree_bytes % tree_format == 0,
                "decode tree size %lld is not a whole number (>= 2) of %d-byte nodes", (long long)tree_bytes, tree_format);
    KVC_REQUIRE(tree_bytes / tree_format <= KVC_TREE_MAX_NODES, "decode tree has more than %d nodes", KVC_TREE_MAX_NODES);
    return 0;
}

// A codebook that the host has just built: its tables travel in the kernel's argument block (written by the host when it
// queues the launch; a copy from pageable memory would make the host wait for the stream), and the one workgroup that puts
// them where they belong derives the decode tables from them.
struct KvcPutCodebookArgs {
    uint32_t words[960];
    uint8_t *dst;
    uint32_t *lut;
    int bytes, tree_at, node_bytes;
};
__global__ void __launch_bounds__(KVC_WG) kvc_put_codebook_kernel(KvcPutCodebookArgs a)
{
    const uint8_t *src = reinterpret_cast<const uint8_t *>(a.words);
    for (int i = threadIdx.x; i < a.bytes; i += KVC_WG) a.dst[i] = src[i];
    kvc_build_lut_body(src + a.tree_at, a.bytes - a.tree_at, a.node_bytes, a.lut);
}

extern "C" int kvc_put_codebook(const kvc_codebook *book, void *d_tables, void *d_lut, void *stream_)
{
    KVC_REQUIRE(book != nullptr && d_tables != nullptr && d_lut != nullptr, "NULL argument");
    KVC_REQUIRE(((uintptr_t)d_lut & 15) == 0, "table buffer must be 16-byte aligned");
    KVC_REQUIRE(book->encode_bytes >= 0 && book->encode_bytes <= (int64_t)sizeof(book->encode_table) && book->decode_bytes >= 0 &&
                    book->decode_bytes <= (int64_t)sizeof(book->decode_tree), "bad codebook");
    const int64_t tree_at = (book->encode_bytes + 15) / 16 * 16, bytes = tree_at + book->decode_bytes;
    KvcPutCodebookArgs a;
    if (bytes > (int64_t)sizeof(a.words)) {                  // (more than about 170 symbols: fine error bounds)
        if (int rc = kvc_put_bytes(d_tables, book->encode_table, book->encode_bytes, stream_)) return rc;
        if (int rc = kvc_put_bytes((uint8_t *)d_tables + tree_at, book->decode_tree, book->decode_bytes, stream_)) return rc;
        return kvc_launch_build_lut((uint8_t *)d_tables + tree_at, book->decode_bytes, book->tree_format, (uint32_t *)d_lut, 1, 0, (hipStream_t)stream_);
    }
    if (int rc = kvc_check_tree(book->decode_bytes, book->tree_format)) return rc;
    std::memset(a.words, 0, (size_t)tree_at);
    std::memcpy(a.words, book->encode_table, (size_t)book->encode_bytes);
    std::memcpy(reinterpret_cast<uint8_t *>(a.words) + tree_at, book->decode_tree, (size_t)book->decode_bytes);
    a.dst = (uint8_t *)d_tables;
    a.lut = (uint32_t *)d_lut;
    a.bytes = (int)bytes;
    a.tree_at = (int)tree_at;
    a.node_bytes = book->tree_format;
    hipLaunchKernelGGL(kvc_put_codebook_kernel, dim3(1), dim3(KVC_WG), 0, (hipStream_t)stream_, a);
    return kvc_check_hip(hipGetLastError(), "kvc_put_codebook_kernel launch");
}

int kvc_launch_build_lut(const uint8_t *d_tree, int64_t tree_bytes, int tree_format, uint32_t *d_lut,
                         int n_codebooks, int64_t tree_stride_bytes, hipStream_t stream)
{
    if (int rc = kvc_check_tree(tree_bytes, tree_format)) return rc;
    hipLaunchKernelGGL(kvc_build_lut_kernel, dim3(n_codebooks), dim3(KVC_WG), 0, stream, d_tree, tree_stride_bytes,
                       (int)tree_bytes, tree_format, d_lut);
    return kvc_check_hip(hipGetLastError(), "kvc_build_lut_kernel launch");
}
