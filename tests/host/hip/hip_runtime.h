// A host double of the few runtime calls readback.hpp makes.  "Device" memory is
// host memory; a stream is a queue of copies that run when somebody waits for
// them, and waiting blocks while the stream's gate is closed, as it does while
// earlier work of the stream still runs.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2, hipMemoryTypeManaged = 3 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
struct hipPointerAttribute_t { hipMemoryType type; };

struct FakeStream {
    std::mutex mu;
    std::condition_variable cv;
    bool open = true;
    std::atomic<int> waiting{0}, copies{0};
    std::atomic<size_t> largest{0};
    struct Copy { void* d; const void* s; size_t n; };
    std::vector<Copy> queue;
    void wait()
    {
        std::unique_lock<std::mutex> l(mu);
        waiting++;
        cv.wait(l, [&] { return open; });
        waiting--;
        for (const Copy& c : queue) std::memcpy(c.d, c.s, c.n);
        queue.clear();
    }
    void gate(bool o)
    {
        std::lock_guard<std::mutex> l(mu);
        open = o;
        cv.notify_all();
    }
};
struct FakeEvent { FakeStream* st = nullptr; };
typedef FakeStream* hipStream_t;
typedef FakeEvent* hipEvent_t;

// what hipPointerGetAttributes reports, by default pageable memory
inline std::atomic<int> fake_type{hipMemoryTypeUnregistered};

inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned)
{
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipHostFree(void* p)
{
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = static_cast<FakeEvent*>(std::calloc(1, sizeof(FakeEvent)));
    return *e ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipEventDestroy(hipEvent_t e)
{
    std::free(e);
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    e->st = s;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    e->st->wait();
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s)
{
    s->wait();
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t st)
{
    std::lock_guard<std::mutex> l(st->mu);
    st->copies++;
    if (n > st->largest) st->largest = n;
    st->queue.push_back({d, s, n});
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void*)
{
    a->type = static_cast<hipMemoryType>(fake_type.load());
    return hipSuccess;
}
