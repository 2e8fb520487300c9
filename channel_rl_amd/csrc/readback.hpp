// readback.hpp -- device to host copies of whole fields into memory the caller
// owns.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>

namespace chan {

// The runtime copies into pageable memory through a staging buffer of its own
// on the calling thread, which also takes every page fault of a fresh array:
// 10 GB/s, where the link moves 57.  Large fields are therefore cut into
// chunks that a few threads fetch through pinned slots, each thread with one
// chunk in flight while it copies the one before (and faults its pages in).
//
// The slots are the process's, one set for all channels (a copy that finds them
// in use, or on another device than theirs, goes the runtime's way), allocated
// by the first large copy and freed with the last channel.
// U, V, W of 384x192x384 (695 MB): 66 -> 19 ms; 192x96x192 (89 MB) 6.9 -> 4.1.
// Four threads with 2 MB chunks: six or twelve gain nothing, 1 MB chunks take 23
// ms and 0.5 MB 32 (each copy costs some 20 us beside its bytes), 4 MB 18 for
// twice the pinned memory.  The first copy takes 1.5 ms more for the slots, which
// a field below 16 MB would not win back.
class Readback {
    static constexpr size_t CHUNK = 2 << 20;
    static constexpr size_t LEAST = 16 << 20;
    static constexpr int WORKERS = 4;

    struct Slots {
        int device = 0;
        char* mem = nullptr;  // WORKERS x 2 chunks
        hipEvent_t ev[WORKERS][2] = {};
        ~Slots()
        {
            for (auto& w : ev)
                for (hipEvent_t e : w)
                    if (e) (void)hipEventDestroy(e);
            if (mem) (void)hipHostFree(mem);
        }
        bool make(int dev)
        {
            device = dev;
            if (hipHostMalloc((void**)&mem, CHUNK * 2 * WORKERS, hipHostMallocDefault) != hipSuccess) {
                mem = nullptr;
                (void)hipGetLastError();
                return false;
            }
            for (auto& w : ev)
                for (hipEvent_t& e : w)
                    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
                        e = nullptr;
                        (void)hipGetLastError();
                        return false;
                    }
            return true;
        }
    };
    std::mutex use_;  // held by the copy that uses the slots, never for work before it
    std::unique_ptr<Slots> slots_;
    std::mutex count_;  // held to change the number of channels
    int channels_ = 0;

    // the slots for a copy from `device` (use_ held), made by the first one
    bool ready(int device)
    {
        if (!slots_) {
            std::unique_ptr<Slots> s(new (std::nothrow) Slots);
            if (s && s->make(device)) slots_ = std::move(s);
        }
        return slots_ && slots_->device == device;
    }

    // worker w's chunks w, w + n, ...: one in flight while the one before is copied
    static hipError_t work(Slots& s, int w, int n, char* dst, const char* src, size_t bytes, hipStream_t st)
    {
        hipError_t e = hipSetDevice(s.device);
        if (e != hipSuccess) return e;
        char* const mem = s.mem + (size_t)w * 2 * CHUNK;
        const size_t step = (size_t)n * CHUNK;
        auto len = [&](size_t at) { return std::min(CHUNK, bytes - at); };
        auto fetch = [&](size_t at, int b) {
            hipError_t r = hipMemcpyAsync(mem + b * CHUNK, src + at, len(at), hipMemcpyDeviceToHost, st);
            return r != hipSuccess ? r : hipEventRecord(s.ev[w][b], st);
        };
        size_t at = (size_t)w * CHUNK;
        if (at >= bytes) return hipSuccess;
        if ((e = fetch(at, 0)) != hipSuccess) return e;
        for (int b = 0; at < bytes; at += step, b ^= 1) {
            hipError_t next = hipSuccess;
            if (at + step < bytes) next = fetch(at + step, b ^ 1);
            if ((e = hipEventSynchronize(s.ev[w][b])) != hipSuccess) return e;
            std::memcpy(dst + at, mem + b * CHUNK, len(at));
            if (next != hipSuccess) return next;
        }
        return hipSuccess;
    }

public:
    static Readback& get()
    {
        // never destroyed: it outlives the runtime's own teardown
        alignas(Readback) static unsigned char mem[sizeof(Readback)];
        static Readback* const r = ::new (mem) Readback;
        return *r;
    }
    void add_channel()
    {
        std::lock_guard<std::mutex> l(count_);
        channels_++;
    }
    void remove_channel()
    {
        std::lock_guard<std::mutex> l(count_);
        if (--channels_ > 0) return;
        std::lock_guard<std::mutex> u(use_);  // free: a copy needs a channel
        slots_.reset();
    }
    // src (device memory of `device`, written by earlier work of st) to dst;
    // returns with the copy complete
    hipError_t copy(void* dst, const void* src, size_t bytes, int device, hipStream_t st)
    {
        if (bytes >= LEAST && pageable(dst)) {
            std::unique_lock<std::mutex> l(use_, std::try_to_lock);
            if (l.owns_lock()) {
                (void)ready(device);  // their allocation beside the stream's work
                l.unlock();
            }
            // the work before the copy is waited for by this thread alone and
            // without the slots, which other channels may want meanwhile
            const hipError_t e = hipStreamSynchronize(st);
            if (e != hipSuccess) return e;
            if (l.try_lock() && ready(device)) return shared(dst, src, bytes, st);
            if (l.owns_lock()) l.unlock();
        }
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
        return e != hipSuccess ? e : hipStreamSynchronize(st);
    }

private:
    // memory the runtime does not know; what it knows it copies to itself, at the
    // link's rate into pinned memory, and a device's the threads cannot write
    static bool pageable(const void* p)
    {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return true;
        }
        return a.type == hipMemoryTypeUnregistered;
    }
    hipError_t shared(void* dst, const void* src, size_t bytes, hipStream_t st)
    {
        const int n = (int)std::min<size_t>(WORKERS, (bytes + 2 * CHUNK - 1) / (2 * CHUNK));
        hipError_t res[WORKERS] = {};
        auto part = [&](int w) { res[w] = work(*slots_, w, n, (char*)dst, (const char*)src, bytes, st); };
        std::thread t[WORKERS];
        int made = 1;  // this thread takes part 0, and those that got no thread
        try {
            for (; made < n; made++) t[made] = std::thread(part, made);
        } catch (const std::exception&) {
        }
        part(0);
        for (int w = made; w < n; w++) part(w);
        for (int w = 1; w < made; w++) t[w].join();
        // nothing of this copy is left in flight when the slots go to the next
        hipError_t e = hipStreamSynchronize(st);
        for (int w = 0; w < n; w++)
            if (res[w] != hipSuccess) e = res[w];
        return e;
    }
};

}  // namespace chan
