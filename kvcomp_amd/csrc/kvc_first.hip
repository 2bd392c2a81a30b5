// kvc_first.hip -- the first store of a context: quantize, learn the codebook, hand it to the device.
//
//   kvc_quant_codebook  <- quant + build_codebook of the first stored chunk (models/cache/kvcomp_encode.py:86-103,
//                          src/huffman.cpp:99-157); in two halves, kvc_quant_counted and kvc_counted_codebook, for callers
//                          with something to do while the quantizer runs
//   kvc_put_bytes          host bytes to device memory without a copy engine or a pinned buffer
//
// What a first store waits for is the histogram of its symbols: 256 numbers.  The quantizers count while they write
// (kvc_quant.hip) and the last workgroup stores the counters to pinned host memory (quantizers that do not count: a kernel of one
// workgroup behind the histogram), and the calling thread looks at that memory until they are there.  The host then builds the code in two or three microseconds; the tie-exact
// construction is one serial chain, which a lane of the GPU needed 65 us for (13 symbols).
// The device has nothing to do from the counts' arrival to the encoder's launch, so the host does only what needs the code
// in between: everything else (buffers, the encoder's status words and marks) is queued while the quantizer runs.  First
// stores of K and V with 32 heads x 128 channels, 8 x 4096 tokens: 579 -> 491 us; 8 heads x 777 tokens: 320 -> 241 us.
// (Today 346 and 205 us, 4 x 32 x 96 x 32 768 tokens 810: the encoder reads the codes from its argument block, so that the codebook need not
// be on the device before it, and the symbols go two to a byte; between the counts' arrival and the encoder the device idles 26 - 38 us.)
#include "kvc_common.h"

#include <atomic>
#include <chrono>
#include <cstring>
#include <mutex>
#include <new>
#include <thread>

namespace {
// Counters on the device (zero between calls: the kernel that hands them over clears them) and where the host reads
// them.  A call holds one block and returns it before it returns; at most KVC_COUNT_BLOCKS unused ones are kept per device.
struct CountBlock {
    unsigned long long *d_counts = nullptr;    // [256] counters, [256] workgroups that have added theirs
    unsigned long long *h_counts = nullptr;    // [256] counters, [256] number of the call that stored them
    unsigned long long calls = 0;
    int dev = -1;
};
constexpr int KVC_COUNT_BLOCKS = 4, KVC_COUNT_DEVICES = 16;
std::mutex g_count_mutex;
CountBlock g_count_blocks[KVC_COUNT_DEVICES][KVC_COUNT_BLOCKS];
int g_count_held[KVC_COUNT_DEVICES] = {};

void free_block(CountBlock &b)
{
    if (b.d_counts) (void)hipFree(b.d_counts);
    if (b.h_counts) (void)hipHostFree(b.h_counts);
    b = CountBlock();
}

int take_block(CountBlock &b)
{
    int dev = 0;
    KVC_HIP(hipGetDevice(&dev));
    KVC_REQUIRE(dev >= 0 && dev < KVC_COUNT_DEVICES, "device index %d out of range", dev);
    {
        std::lock_guard<std::mutex> lock(g_count_mutex);
        if (g_count_held[dev] > 0) {
            b = g_count_blocks[dev][--g_count_held[dev]];
            return 0;
        }
    }
    b.dev = dev;
    int rc = kvc_check_hip(hipMalloc((void **)&b.d_counts, 257 * 8), "hipMalloc");
    if (!rc) rc = kvc_check_hip(hipHostMalloc((void **)&b.h_counts, 257 * 8, hipHostMallocDefault), "hipHostMalloc");
    if (!rc) rc = kvc_check_hip(hipMemset(b.d_counts, 0, 257 * 8), "hipMemset");
    if (!rc) rc = kvc_check_hip(hipDeviceSynchronize(), "hipDeviceSynchronize");       // once per block: the call may be on any stream
    if (rc) {
        free_block(b);
        return rc;
    }
    b.h_counts[256] = 0;
    return 0;
}

void give_block(CountBlock &b)
{
    {
        std::lock_guard<std::mutex> lock(g_count_mutex);
        if (g_count_held[b.dev] < KVC_COUNT_BLOCKS) {
            g_count_blocks[b.dev][g_count_held[b.dev]++] = b;
            return;
        }
    }
    free_block(b);
}
}  // namespace

// 2 KB over the bus.  System-scope stores, then the call's number with release order: a reader that sees the number sees
// the counters.
__global__ void __launch_bounds__(256) kvc_counts_to_host_kernel(unsigned long long *__restrict__ counts, unsigned long long *host,
                                                                 unsigned long long call)
{
    const int t = threadIdx.x;
    __hip_atomic_store(&host[t], counts[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    counts[t] = 0;
    __threadfence_system();
    __syncthreads();
    if (t == 0) __hip_atomic_store(&host[256], call, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Looks for the call's number for at most 5 ms (a first store's quantizer takes 0.01 to 0.3 ms), then lets the runtime wait
// for the stream.
static int wait_for_counts(const CountBlock &b, hipStream_t stream)
{
    const auto began = std::chrono::steady_clock::now();
    for (;;) {
        for (int i = 0; i < 256; i++) {
            if (__atomic_load_n(&b.h_counts[256], __ATOMIC_ACQUIRE) == b.calls) return 0;
            __builtin_ia32_pause();
        }
        if (std::chrono::steady_clock::now() - began > std::chrono::milliseconds(5)) break;
    }
    KVC_HIP(hipStreamSynchronize(stream));
    KVC_REQUIRE(__atomic_load_n(&b.h_counts[256], __ATOMIC_ACQUIRE) == b.calls, "the symbol counts did not arrive");
    return 0;
}

// Whether everything on the stream that words 10 - 12 of an outcome name has run.  Nothing is asked of a stream that is being
// recorded (what was queued before that is still on its way), and a runtime that will not answer during a recording has not said yes.
static int outcome_stream_is_idle(const uint32_t *h_outcome, bool *idle)
{
    hipStream_t stream = (hipStream_t)(uintptr_t)(h_outcome[10] | (uint64_t)h_outcome[11] << 32);
    *idle = false;
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (stream) KVC_HIP(hipStreamIsCapturing(stream, &capturing));
    if (capturing != hipStreamCaptureStatusNone) return 0;
    int here = 0;
    KVC_HIP(hipGetDevice(&here));
    KVC_HIP(hipSetDevice((int)h_outcome[12]));             // (the default stream is the current device's)
    const hipError_t e = hipStreamQuery(stream);
    if (e != hipSuccess) (void)hipGetLastError();          // "not ready" is no error of anyone's
    KVC_HIP(hipSetDevice(here));
    *idle = e == hipSuccess;
    return e == hipErrorNotReady || e == hipErrorStreamCaptureImplicit || e == hipErrorStreamCaptureUnsupported ? 0 : kvc_check_hip(e, "hipStreamQuery");
}

// Looks at the words alone for two seconds (an encode takes 0.01 to 2 ms); from then on also at their stream, ten times a
// second, so that a number which never comes does not hold the caller.  Other streams are never waited for.
extern "C" int kvc_wait_outcome(const uint32_t *h_outcome, uint32_t outcome_number)
{
    KVC_REQUIRE(h_outcome != nullptr, "NULL argument");
    const auto began = std::chrono::steady_clock::now();
    auto ask = began + std::chrono::seconds(2);
    for (;;) {
        for (int i = 0; i < 256; i++) {
            if (__atomic_load_n(&h_outcome[9], __ATOMIC_ACQUIRE) == outcome_number) return 0;
            __builtin_ia32_pause();
        }
        const auto now = std::chrono::steady_clock::now();
        if (now > ask) {
            bool idle;
            if (int rc = outcome_stream_is_idle(h_outcome, &idle)) return rc;
            if (idle) return 0;
            ask = now + std::chrono::milliseconds(100);
        }
        if (now - began > std::chrono::milliseconds(5)) std::this_thread::sleep_for(std::chrono::microseconds(20));
    }
}

static int kvc_quant_counted_form(const void *d_x_f16, int64_t NB, int64_t BS, int64_t B, int64_t H, int64_t D, int quant_mask, float eb,
                                  uint8_t *d_sym, bool packed, int8_t *d_min_i8, void *d_scale_f16, void **counted, void *stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    KVC_REQUIRE(counted != nullptr, "NULL argument");
    *counted = nullptr;
    KVC_REQUIRE(NB > 0, "nothing to quantize");
    hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
    if (stream) KVC_HIP(hipStreamIsCapturing(stream, &capturing));
    KVC_REQUIRE(capturing == hipStreamCaptureStatusNone, "the first store of a context waits for its codebook and cannot be recorded into a graph");
    CountBlock *block = new (std::nothrow) CountBlock();
    KVC_REQUIRE(block != nullptr, "out of memory");
    if (int rc = take_block(*block)) {
        delete block;
        return rc;
    }
    block->calls++;
    KvcCountsToHost to_host = {block->h_counts, block->calls, false};
    int rc = kvc_quant_to_host(d_x_f16, NB, BS, B, H, D, quant_mask, eb, d_sym, packed, d_min_i8, d_scale_f16, (int64_t *)block->d_counts, &to_host, stream_);
    if (!rc && !to_host.handed_over) {
        hipLaunchKernelGGL(kvc_counts_to_host_kernel, dim3(1), dim3(256), 0, stream, block->d_counts, block->h_counts, block->calls);
        rc = kvc_check_hip(hipGetLastError(), "kvc_counts_to_host_kernel launch");
    }
    if (rc) {
        (void)hipStreamSynchronize(stream);                // whatever was queued may still write the block
        free_block(*block);
        delete block;
        return rc;
    }
    *counted = block;
    return 0;
}

extern "C" int kvc_quant_counted(const void *d_x_f16, int64_t NB, int64_t BS, int64_t B, int64_t H, int64_t D, int quant_mask,
                                 float eb, uint8_t *d_sym, int8_t *d_min_i8, void *d_scale_f16, void **counted, void *stream)
{
    return kvc_quant_counted_form(d_x_f16, NB, BS, B, H, D, quant_mask, eb, d_sym, false, d_min_i8, d_scale_f16, counted, stream);
}

extern "C" int kvc_quant_counted_packed(const void *d_x_f16, int64_t NB, int64_t BS, int64_t B, int64_t H, int64_t D, int quant_mask,
                                        float eb, uint8_t *d_packed, int8_t *d_min_i8, void *d_scale_f16, void **counted, void *stream)
{
    return kvc_quant_counted_form(d_x_f16, NB, BS, B, H, D, quant_mask, eb, d_packed, true, d_min_i8, d_scale_f16, counted, stream);
}

extern "C" int kvc_counted_codebook(void *counted, int smoothed_symbols, kvc_codebook *out, void *stream_)
{
    hipStream_t stream = (hipStream_t)stream_;
    KVC_REQUIRE(counted != nullptr, "NULL argument");
    CountBlock block = *(CountBlock *)counted;
    delete (CountBlock *)counted;
    if (int rc = wait_for_counts(block, stream)) {
        (void)hipStreamSynchronize(stream);
        free_block(block);
        return rc;
    }
    int64_t counts[256];
    for (int s = 0; s < 256; s++) counts[s] = (int64_t)block.h_counts[s];
    give_block(block);
    KVC_REQUIRE(out != nullptr, "NULL argument");
    KVC_REQUIRE(smoothed_symbols >= 0 && smoothed_symbols <= 256, "smoothed_symbols must be 0 .. 256");
    int64_t smoothed[256];
    for (int s = 0; s < 256; s++) smoothed[s] = counts[s] + (s < smoothed_symbols ? 1 : 0);
    // the reference's int8 tree where the code fits it, the int16 tree where it does not
    int shift = 0;
    out->tree_format = KVC_TREE_I8;
    int rc = kvc_build_codebook_host(smoothed, KVC_TREE_I8, &shift, out->encode_table, sizeof(out->encode_table), &out->encode_bytes,
                                     out->decode_tree, sizeof(out->decode_tree), &out->decode_bytes);
    if (rc) {
        out->tree_format = KVC_TREE_I16;
        if (int rc16 = kvc_build_codebook_host(smoothed, KVC_TREE_I16, &shift, out->encode_table, sizeof(out->encode_table), &out->encode_bytes,
                                               out->decode_tree, sizeof(out->decode_tree), &out->decode_bytes))
            return rc16;
    }
    KVC_REQUIRE(shift == 0, "shift must be 0");
    out->max_code_bits = 0;
    out->payload_bits = 0;
    int64_t by_length[33] = {}, total = 0;                 // symbols by code length
    const uint32_t *entry = reinterpret_cast<const uint32_t *>(out->encode_table);
    for (int64_t s = 0; s < out->encode_bytes / 8; s++) {
        const uint32_t length = entry[2 * s + 1];
        if ((int)length > out->max_code_bits) out->max_code_bits = (int)length;
        out->payload_bits += counts[s] * (int64_t)length;
        by_length[length <= 32 ? length : 32] += counts[s];
        total += counts[s];
    }
    // The narrowest index that next to all pairs of these symbols fit.  A tile that meets another pair is decoded twice: at one
    // pair in two hundred thousand that is a tile of 64 x 64 pairs in fifty, against a sixth gained on all of them.
    out->pair_bits = 0;
    int64_t longer[34] = {};                               // symbols with codes of more than l bits
    for (int l = 32; l >= 0; l--) longer[l] = (l < 32 ? longer[l + 1] + by_length[l + 1] : 0);
    for (int w = 7; w >= 2 && total > 0; w--) {
        double missed = 0;
        for (int l = 1; l <= 32; l++) missed += (double)by_length[l] / (double)total * ((double)longer[l < w ? w - l : 0] / (double)total);
        if (missed <= 5e-6) out->pair_bits = w;
    }
    return 0;
}

extern "C" int kvc_quant_codebook(const void *d_x_f16, int64_t NB, int64_t BS, int64_t B, int64_t H, int64_t D, int quant_mask,
                                  float eb, uint8_t *d_sym, int8_t *d_min_i8, void *d_scale_f16, int smoothed_symbols,
                                  kvc_codebook *out, void *stream)
{
    KVC_REQUIRE(out != nullptr, "NULL argument");
    KVC_REQUIRE(smoothed_symbols >= 0 && smoothed_symbols <= 256, "smoothed_symbols must be 0 .. 256");
    void *counted;
    if (int rc = kvc_quant_counted(d_x_f16, NB, BS, B, H, D, quant_mask, eb, d_sym, d_min_i8, d_scale_f16, &counted, stream)) return rc;
    return kvc_counted_codebook(counted, smoothed_symbols, out, stream);
}

// The bytes travel in the kernel's argument block (written by the host when it queues the launch).  A codebook's tables
// are some hundred bytes: one launch, where a copy from pageable memory makes the host wait for the stream.
struct KvcPutArgs {
    uint32_t words[960];
    uint8_t *dst;
    int bytes;
};
__global__ void __launch_bounds__(256) kvc_put_bytes_kernel(KvcPutArgs a)
{
    const uint8_t *src = reinterpret_cast<const uint8_t *>(a.words);
    for (int i = threadIdx.x; i < a.bytes; i += 256) a.dst[i] = src[i];
}

extern "C" int kvc_put_bytes(void *d_dst, const void *h_src, int64_t bytes, void *stream_)
{
    KVC_REQUIRE(bytes >= 0 && (bytes == 0 || (d_dst && h_src)), "NULL argument");
    KvcPutArgs a;
    for (int64_t at = 0; at < bytes; at += (int64_t)sizeof(a.words)) {
        const int64_t n = bytes - at < (int64_t)sizeof(a.words) ? bytes - at : (int64_t)sizeof(a.words);
        std::memcpy(a.words, (const uint8_t *)h_src + at, (size_t)n);
        a.dst = (uint8_t *)d_dst + at;
        a.bytes = (int)n;
        hipLaunchKernelGGL(kvc_put_bytes_kernel, dim3(1), dim3(256), 0, (hipStream_t)stream_, a);
    }
    return kvc_check_hip(hipGetLastError(), "kvc_put_bytes_kernel launch");
}
