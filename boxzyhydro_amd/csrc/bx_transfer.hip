// bx_transfer.hip -- host <-> device copies of large host arrays.
//
// A copy between pageable memory and the device by hipMemcpyAsync runs through
// one thread: 9.5 GB/s down into fresh pages (their first touch is the larger
// part) and 29 GB/s up at 256^3.  Here a few worker threads each own a pinned
// slot and take every kWorkers-th chunk: the device moves chunk after chunk on
// the caller's stream while the other workers copy theirs between the pinned
// slots and the caller's memory, so that the bus, not one core, is the limit.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>

#include "bx_internal.h"

namespace bx {

constexpr int kWorkers = 6;
constexpr size_t kSlotBytes = size_t(4) << 20;

size_t pipe_slot_bytes() { return kSlotBytes; }
size_t pipe_stage_bytes() { return kSlotBytes * kWorkers; }

// Pinned slots and events of one owner (a context or a batch), made on its
// first large transfer and freed with it.
struct HostPipe {
    int device = 0;
    char *pinned = nullptr;
    hipEvent_t done[kWorkers] = {};
};

void pipe_free(HostPipe *p)
{
    if (!p) return;
    for (hipEvent_t e : p->done)
        if (e) (void)hipEventDestroy(e);
    if (p->pinned) (void)hipHostFree(p->pinned);
    delete p;
}

// the owner's pipe, or null when it cannot be made (the caller then copies directly)
static HostPipe *pipe_of(HostPipe **slot, int device)
{
    if (*slot) return *slot;
    HostPipe *p = new (std::nothrow) HostPipe();
    if (!p) return nullptr;
    p->device = device;
    bool ok = hipHostMalloc((void **)&p->pinned, kSlotBytes * kWorkers, hipHostMallocDefault) == hipSuccess;
    for (int i = 0; i < kWorkers && ok; i++)
        ok = hipEventCreateWithFlags(&p->done[i], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        pipe_free(p);
        return nullptr;
    }
    return *slot = p;
}

// Runs one(chunk, worker) for every chunk, worker w taking w, w+kWorkers, ...
template <typename F>
static hipError_t each_chunk(int device, int64_t chunks, const F &one)
{
    std::atomic<int> err{(int)hipSuccess};
    auto work = [&](int w) {
        hipError_t e = hipSetDevice(device);
        for (int64_t c = w; c < chunks && e == hipSuccess && err.load() == (int)hipSuccess; c += kWorkers) e = one(c, w);
        if (e != hipSuccess) err.store((int)e);
    };
    std::thread th[kWorkers];
    const int n = (int)std::min<int64_t>(kWorkers, chunks);
    int started = 1;
    try {
        for (; started < n; started++) th[started] = std::thread(work, started);
    } catch (const std::exception &) {  // no more threads, or no memory for one: their chunks are taken here
    }
    work(0);
    for (int w = started; w < n; w++) work(w);
    for (int w = 1; w < started; w++) th[w].join();
    return (hipError_t)err.load();
}

static std::mutex g_issue;  // a chunk's kernel, copy and event are issued together

int pipe_download(HostPipe **slot, int device, hipStream_t stream, char *dst, size_t bytes, size_t unit,
                  const PipeChunk &chunk, void *self)
{
    HostPipe *p = bytes >= kPipeMin ? pipe_of(slot, device) : nullptr;
    const size_t step = p ? kSlotBytes / unit * unit : bytes;
    if (!p) {
        const void *src = nullptr;
        for (size_t off = 0, len; off < bytes; off += len) {
            len = std::min(bytes - off, chunk.stage_bytes ? chunk.stage_bytes / unit * unit : bytes);
            BX_HIP(chunk.get(self, off, len, 0, &src));
            BX_HIP(hipMemcpyAsync(dst + off, src, len, hipMemcpyDeviceToHost, stream));
        }
        BX_HIP(hipStreamSynchronize(stream));
        return BX_OK;
    }
    BX_HIP(each_chunk(device, (int64_t)((bytes + step - 1) / step), [&](int64_t c, int w) -> hipError_t {
        const size_t off = (size_t)c * step, len = std::min(step, bytes - off);
        char *pin = p->pinned + (size_t)w * kSlotBytes;
        hipError_t e;
        {
            std::lock_guard<std::mutex> lk(g_issue);
            const void *src = nullptr;
            if ((e = chunk.get(self, off, len, w, &src)) != hipSuccess) return e;
            if ((e = hipMemcpyAsync(pin, src, len, hipMemcpyDeviceToHost, stream)) != hipSuccess) return e;
            if ((e = hipEventRecord(p->done[w], stream)) != hipSuccess) return e;
        }
        if ((e = hipEventSynchronize(p->done[w])) != hipSuccess) return e;
        std::memcpy(dst + off, pin, len);
        return hipSuccess;
    }));
    return BX_OK;
}

int pipe_upload(HostPipe **slot, int device, hipStream_t stream, const char *src, size_t bytes, size_t unit,
                const PipeChunk &chunk, void *self)
{
    HostPipe *p = bytes >= kPipeMin ? pipe_of(slot, device) : nullptr;
    const size_t step = p ? kSlotBytes / unit * unit : bytes;
    if (!p) {
        void *to = nullptr;
        for (size_t off = 0, len; off < bytes; off += len) {
            len = std::min(bytes - off, chunk.stage_bytes ? chunk.stage_bytes / unit * unit : bytes);
            BX_HIP(chunk.room(self, off, len, 0, &to));
            BX_HIP(hipMemcpyAsync(to, src + off, len, hipMemcpyHostToDevice, stream));
            BX_HIP(chunk.put(self, off, len, 0));
        }
        BX_HIP(hipStreamSynchronize(stream));
        return BX_OK;
    }
    BX_HIP(each_chunk(device, (int64_t)((bytes + step - 1) / step), [&](int64_t c, int w) -> hipError_t {
        const size_t off = (size_t)c * step, len = std::min(step, bytes - off);
        char *pin = p->pinned + (size_t)w * kSlotBytes;
        std::memcpy(pin, src + off, len);
        hipError_t e;
        {
            std::lock_guard<std::mutex> lk(g_issue);
            void *to = nullptr;
            if ((e = chunk.room(self, off, len, w, &to)) != hipSuccess) return e;
            if ((e = hipMemcpyAsync(to, pin, len, hipMemcpyHostToDevice, stream)) != hipSuccess) return e;
            if ((e = chunk.put(self, off, len, w)) != hipSuccess) return e;
            if ((e = hipEventRecord(p->done[w], stream)) != hipSuccess) return e;
        }
        return hipEventSynchronize(p->done[w]);  // the slot is free again
    }));
    BX_HIP(hipStreamSynchronize(stream));
    return BX_OK;
}

}  // namespace bx
