// Reads of device arrays into the caller's host memory.
#include "cnd_ctx.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace cnd {

namespace {

// A pageable copy runs at the rate one thread touches the caller's pages, page
// faults included, well below the link.  From kStagedMin on the copy goes
// through kBuffers pinned chunks in turn, and kCopyThreads threads of the call
// move each chunk on, a huge page each, while the next ones arrive.  Into fresh
// arrays: 679 MB (257^3 points) 64.3 -> 14.3 ms, 86 MB 8.6 -> 2.7 ms, 36 MB
// 3.9 -> 1.35 ms (a context's first, with the pinned allocation, 4.3 -> 3.8
// ms).  Below 32 MB that first read would be the slower one.  Memory that is
// page-locked already takes the plain copy, which runs at the link's rate into
// it: 679 MB 11.9 ms against 12.9 through the chunks, 36 MB 0.65 against 0.87.
constexpr size_t kStagedMin = size_t(32) << 20, kChunk = size_t(16) << 20;
constexpr int kBuffers = 3, kCopyThreads = 8;

// Memory the runtime knows (page-locked, managed), which a copy reaches directly.
bool known(const void *p)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

bool staging(cnd_ctx *c)
{
    static_assert(sizeof(c->stage_ev) / sizeof(c->stage_ev[0]) == kBuffers);
    if (c->stage) return true;
    bool good = hipHostMalloc((void **)&c->stage, kBuffers * kChunk, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t &e : c->stage_ev) good = good && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (good) return true;
    (void)hipGetLastError();
    read_release(c);
    return false;
}

// The chunks' way through the staging memory; started is false where no
// thread could be started, and nothing is copied then.
int staged_copy(cnd_ctx *c, const std::vector<HostCopy> &chunks, bool &started)
{
    std::mutex m;
    std::condition_variable go, drained;
    size_t ready = 0;              // chunks that have arrived
    int left[kBuffers] = {};       // threads still to copy a buffer's chunk
    bool stop = false;
    std::vector<std::thread> threads;
    int T = 0;
    auto work = [&](int t) {
        for (size_t i = 0; i < chunks.size(); ++i) {
            {
                std::unique_lock<std::mutex> l(m);
                go.wait(l, [&] { return ready > i || stop; });
                if (ready <= i) return;
            }
            constexpr size_t page = 4096;
            const size_t n = chunks[i].bytes, per = ((n + T - 1) / T + page - 1) / page * page;
            const size_t lo = std::min(n, per * t), hi = std::min(n, lo + per);
            std::memcpy((char *)chunks[i].dst + lo, c->stage + (i % kBuffers) * kChunk + lo, hi - lo);
            std::lock_guard<std::mutex> l(m);
            if (--left[i % kBuffers] == 0) drained.notify_one();
        }
    };
    std::unique_lock<std::mutex> hold(m);   // the threads wait until T is known
    try {
        threads.reserve(kCopyThreads);
        for (int t = 0; t < kCopyThreads; ++t) threads.emplace_back(work, t);
    } catch (const std::exception &) {
    }
    T = int(threads.size());
    hold.unlock();
    started = T > 0;
    hipError_t e = hipSuccess;
    size_t queued = 0;
    for (size_t i = 0; started && e == hipSuccess && i < chunks.size(); ++i) {
        // every free buffer has a copy on its way before the oldest is waited for
        for (; e == hipSuccess && queued < chunks.size() && queued < i + kBuffers; ++queued) {
            const int b = int(queued % kBuffers);
            {
                std::unique_lock<std::mutex> l(m);
                // (only the next chunk's buffer is worth waiting for)
                if (queued > i && left[b] > 0) break;
                drained.wait(l, [&] { return left[b] == 0; });
                left[b] = T;
            }
            e = hipMemcpyAsync(c->stage + b * kChunk, chunks[queued].src, chunks[queued].bytes, hipMemcpyDeviceToHost, c->st);
            if (e == hipSuccess) e = hipEventRecord(c->stage_ev[b], c->st);
        }
        if (e == hipSuccess) e = hipEventSynchronize(c->stage_ev[i % kBuffers]);
        if (e != hipSuccess) break;
        std::lock_guard<std::mutex> l(m);
        ready = i + 1;
        go.notify_all();
    }
    {
        std::lock_guard<std::mutex> l(m);
        stop = true;   // (threads still finish what has arrived)
        go.notify_all();
    }
    for (std::thread &t : threads) t.join();
    if (e != hipSuccess) return fail(c, CND_EDEVICE, std::string("read: ") + hipGetErrorString(e));
    return CND_OK;
}

}  // namespace

int read_to_host(cnd_ctx *c, const HostCopy *copies, int n)
{
    size_t bytes = 0;
    for (int k = 0; k < n; ++k) bytes += copies[k].bytes;
    bool direct = bytes < kStagedMin;
    for (int k = 0; k < n && !direct; ++k)
        direct = known(copies[k].dst) || known((const char *)copies[k].dst + copies[k].bytes - 1);
    if (!direct && staging(c)) {
        std::vector<HostCopy> chunks;
        try {
            for (int k = 0; k < n; ++k)
                for (size_t o = 0; o < copies[k].bytes; o += kChunk)
                    chunks.push_back(HostCopy{(char *)copies[k].dst + o, (const char *)copies[k].src + o,
                                              std::min(kChunk, copies[k].bytes - o)});
        } catch (const std::exception &) {
            chunks.clear();
        }
        bool started = false;
        const int r = chunks.empty() ? CND_OK : staged_copy(c, chunks, started);
        if (started) return r;
    }
    for (int k = 0; k < n; ++k)
        HIPX(c, hipMemcpyAsync(copies[k].dst, copies[k].src, copies[k].bytes, hipMemcpyDeviceToHost, c->st));
    HIPX(c, hipStreamSynchronize(c->st));
    return CND_OK;
}

void read_release(cnd_ctx *c)
{
    if (c->stage) (void)hipHostFree(c->stage);
    c->stage = nullptr;
    for (hipEvent_t &e : c->stage_ev) {
        if (e) (void)hipEventDestroy(e);
        e = nullptr;
    }
}

}  // namespace cnd
