// staging.cpp -- copies between pageable host buffers and device memory at
// close to link speed, and the small scratch of the calls that return sums.
//
// A copy from pageable memory goes through a single CPU copy into the
// runtime's own staging (17 to 27 GB/s measured here, the link 56).  Instead,
// 8 host threads share the copy of a chunk into one of two pinned buffers while
// the DMA of the other runs on a stream of the pool's own: 252 MiB in 5.1 ms up
// and 5.2 down (9.2 and 15.0 by hipMemcpy), 1080 MiB in 20.7 (54 GB/s).  Chunks
// are as large as the buffers, since each DMA leaves a gap behind it (4 threads
// with 4 MiB chunks of their own: 5.8 and 24 ms), except for uploads below 256
// MiB, which start their first DMA earlier with an eighth of the copy (16 MiB
// 0.55 -> 0.45 ms, 64 MiB 1.6 -> 1.5; downloads 0.56 -> 0.6, 1.6 -> 1.9).
//
// Each call is ordered after the work already queued on the null stream (the
// stage layer's launches) and returns when its copies are complete, so it
// replaces a synchronous hipMemcpy.  Buffers the runtime knows (pinned,
// managed) and short ones are left to hipMemcpy, as is everything while the
// pool cannot be made.  The pool of each device (64 MiB pinned, one stream, two
// events) is made on first use and kept until the process ends; calls on one
// device are serialised by its lock.
#include "tops_internal.hpp"

#include <string.h>

#include <algorithm>
#include <mutex>
#include <thread>

namespace tops {
namespace {

constexpr size_t kMinChunk = 4u << 20;
constexpr size_t kMaxChunk = 32u << 20;   // a pinned buffer
constexpr int kMaxDevices = 16;
constexpr int kThreads = 8;

struct Pool {
    std::mutex mu;
    bool ready = false;
    char* buf[2] = {nullptr, nullptr};
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipStream_t s = nullptr;
};

Pool g_pools[kMaxDevices];

// whether the runtime knows the memory: pinned, managed or device memory, not
// malloc'd, stack or mapped files
bool known(const void* h)
{
    hipPointerAttribute_t a;
    memset(&a, 0, sizeof(a));
    if (hipPointerGetAttributes(&a, h) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

// The pool's buffers, made on first use, and again after a device reset took
// them.  A pool that cannot be made is tried again by the next call.
bool pool_init(Pool& p)
{
    if (p.ready && known(p.buf[0])) return true;
    p.ready = false;
    p.s = nullptr;
    for (int k = 0; k < 2; k++) {
        p.buf[k] = nullptr;
        p.ev[k] = nullptr;
    }
    hipError_t e = hipStreamCreateWithFlags(&p.s, hipStreamNonBlocking);
    for (int k = 0; k < 2; k++) {
        if (e == hipSuccess) e = hipHostMalloc((void**)&p.buf[k], kMaxChunk, hipHostMallocDefault);
        if (e == hipSuccess) e = hipEventCreateWithFlags(&p.ev[k], hipEventDisableTiming);
    }
    p.ready = e == hipSuccess;
    if (!p.ready) {   // give back what was made, and forget the error
        for (int k = 0; k < 2; k++) {
            if (p.ev[k]) (void)hipEventDestroy(p.ev[k]);
            if (p.buf[k]) (void)hipHostFree(p.buf[k]);
        }
        if (p.s) (void)hipStreamDestroy(p.s);
        (void)hipGetLastError();
    }
    return p.ready;
}

// f(0) .. f(n - 1) on threads of their own, the first and those that no thread
// could be made for on this one; f must not throw
template <class F>
void on_threads(int n, F&& f)
{
    std::thread th[kThreads];
    int made = 1;
    try {
        for (; made < n; made++) th[made] = std::thread([&f, made] { f(made); });
    } catch (...) {
    }
    f(0);
    for (int i = made; i < n; i++) f(i);
    for (int i = 1; i < made; i++) th[i].join();
}

// dst <- src (n bytes of host memory), a share per thread
void parallel_copy(char* dst, const char* src, size_t n)
{
    const int t = (int)std::min<size_t>(kThreads, std::max<size_t>(1, n >> 20));
    const size_t piece = (n / t + 64) / 64 * 64;
    on_threads(t, [&](int i) {
        const size_t off = piece * i;
        if (off < n) memcpy(dst + off, src + off, std::min(piece, n - off));
    });
}

// One copy through the pool; false: nothing was copied, the pool is not there.
bool staged_copy(bool up, char* dev, char* host, size_t bytes, int* rc_out)
{
    int dev_id = 0;
    if (hipGetDevice(&dev_id) != hipSuccess || dev_id < 0 || dev_id >= kMaxDevices) return false;
    Pool& p = g_pools[dev_id];
    std::lock_guard<std::mutex> lock(p.mu);
    if (!pool_init(p)) return false;
    *rc_out = TOPS_OK;
    // the device buffer is written (or no longer used)
    hipError_t e0 = hipStreamSynchronize(nullptr);
    if (e0 != hipSuccess) {
        *rc_out = hip_fail(e0, "staged copy", __FILE__, __LINE__);
        return true;
    }
    const size_t chunk = up ? std::min(kMaxChunk, std::max(kMinChunk, bytes / 8)) : kMaxChunk;
    const size_t chunks = (bytes + chunk - 1) / chunk;
    hipError_t e = hipSuccess;
    auto size = [&](size_t c) { return std::min(chunk, bytes - c * chunk); };
    auto dma = [&](size_t c) {
        char* b = p.buf[c & 1];
        e = up ? hipMemcpyAsync(dev + c * chunk, b, size(c), hipMemcpyHostToDevice, p.s)
               : hipMemcpyAsync(b, dev + c * chunk, size(c), hipMemcpyDeviceToHost, p.s);
        if (e == hipSuccess) e = hipEventRecord(p.ev[c & 1], p.s);
    };
    if (!up) dma(0);
    for (size_t c = 0; c < chunks && e == hipSuccess; c++) {
        if (up) {
            // the buffer's copy of two chunks ago is through
            if (c >= 2) e = hipEventSynchronize(p.ev[c & 1]);
            if (e != hipSuccess) break;
            parallel_copy(p.buf[c & 1], host + c * chunk, size(c));
            dma(c);
        } else {
            // the next chunk goes into the other buffer, already copied out
            if (c + 1 < chunks) dma(c + 1);
            if (e == hipSuccess) e = hipEventSynchronize(p.ev[c & 1]);
            if (e == hipSuccess) parallel_copy(host + c * chunk, p.buf[c & 1], size(c));
        }
    }
    // every copy is through, also after an error
    const hipError_t es = hipStreamSynchronize(p.s);
    if (e == hipSuccess) e = es;
    if (e != hipSuccess) *rc_out = hip_fail(e, "staged copy", __FILE__, __LINE__);
    return true;
}

// ---- scratch -------------------------------------------------------------
constexpr size_t kKeepBytes = 8u << 20;   // larger device blocks are not kept
constexpr int kKeepBlocks = 4;            // idle blocks kept per device
constexpr size_t kPinnedBytes = 4096;

struct ScratchPool {
    std::mutex mu;
    CallScratch::Block idle[kKeepBlocks];
    int n = 0;

    CallScratch::Block remove(int i)
    {
        const CallScratch::Block b = idle[i];
        idle[i] = idle[--n];
        return b;
    }
    // the smallest idle block of at least that many bytes, or none
    CallScratch::Block best(size_t bytes)
    {
        int at = -1;
        for (int i = 0; i < n; i++)
            if (idle[i].bytes >= bytes && (at < 0 || idle[i].bytes < idle[at].bytes)) at = i;
        return at < 0 ? CallScratch::Block() : remove(at);
    }
    // keeps b, in the place of the smallest block when there is none free; the
    // block that is not kept (none: nothing)
    CallScratch::Block keep(const CallScratch::Block& b)
    {
        CallScratch::Block out;
        if (n == kKeepBlocks) {
            int at = 0;
            for (int i = 1; i < n; i++)
                if (idle[i].bytes < idle[at].bytes) at = i;
            if (idle[at].bytes >= b.bytes) return b;
            out = remove(at);
        }
        idle[n++] = b;
        return out;
    }
};
ScratchPool g_scratch[kMaxDevices];

// (waits for the device)
void free_block(const CallScratch::Block& b)
{
    if (b.dev) (void)hipFree(b.dev);
    if (b.host) (void)hipHostFree(b.host);
}

}  // namespace

int CallScratch::take(size_t dev_bytes, size_t host_bytes)
{
    if (hipGetDevice(&device_) != hipSuccess || device_ >= kMaxDevices) device_ = -1;
    if (device_ >= 0 && dev_bytes <= kKeepBytes && host_bytes <= kPinnedBytes) {
        ScratchPool& p = g_scratch[device_];
        std::lock_guard<std::mutex> lock(p.mu);
        // (a block that the runtime no longer knows went with a device reset)
        while ((b_ = p.best(dev_bytes)).dev)
            if (known(b_.host)) return TOPS_OK;
    }
    // a new block, rounded up so that calls of about one size share it; one too
    // large to be kept has no pinned part
    size_t n = 1u << 20;
    while (n < dev_bytes && n < kKeepBytes) n <<= 1;
    b_.bytes = std::max(n, dev_bytes);
    TOPS_HIP(hipMalloc(&b_.dev, b_.bytes));
    if (b_.bytes <= kKeepBytes && host_bytes <= kPinnedBytes &&
        hipHostMalloc(&b_.host, kPinnedBytes, 0) != hipSuccess) {
        b_.host = nullptr;
        (void)hipGetLastError();
    }
    return TOPS_OK;
}

CallScratch::~CallScratch()
{
    if (!b_.dev) return;
    if (device_ >= 0 && b_.host && idle_) {
        ScratchPool& p = g_scratch[device_];
        std::lock_guard<std::mutex> lock(p.mu);
        b_ = p.keep(b_);
    }
    free_block(b_);
}

void release_idle_scratch()
{
    for (ScratchPool& p : g_scratch) {
        std::lock_guard<std::mutex> lock(p.mu);
        for (CallScratch::Block b; (b = p.best(0)).dev;)
            if (known(b.host)) free_block(b);
    }
}

int staged_upload(void* d_dst, const void* h_src, size_t bytes)
{
    if (bytes == 0) return TOPS_OK;
    int rc = TOPS_OK;
    if (bytes > kMinChunk && !known(h_src) &&
        staged_copy(true, (char*)d_dst, (char*)const_cast<void*>(h_src), bytes, &rc))
        return rc;
    TOPS_HIP(hipMemcpy(d_dst, h_src, bytes, hipMemcpyHostToDevice));
    return TOPS_OK;
}

int staged_download(void* h_dst, const void* d_src, size_t bytes)
{
    if (bytes == 0) return TOPS_OK;
    int rc = TOPS_OK;
    if (bytes > kMinChunk && !known(h_dst) &&
        staged_copy(false, (char*)const_cast<void*>(d_src), (char*)h_dst, bytes, &rc))
        return rc;
    TOPS_HIP(hipMemcpy(h_dst, d_src, bytes, hipMemcpyDeviceToHost));
    return TOPS_OK;
}

}  // namespace tops
