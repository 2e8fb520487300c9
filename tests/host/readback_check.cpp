// The host logic of readback.hpp against a double of the runtime (hip/hip_runtime.h
// here): one check per argument, exit status 0 when it holds.
#include "readback.hpp"

#include <chrono>
#include <cstdio>
#include <future>
#include <new>
#include <string>

using chan::Readback;
using namespace std::chrono_literals;

// from here on this many allocations succeed and the rest fail (below 0: all succeed)
static std::atomic<int> fake_budget{-1};
static void* fake_new(size_t n)
{
    int b = fake_budget;
    while (b > 0 && !fake_budget.compare_exchange_weak(b, b - 1)) {}
    return b == 0 ? nullptr : std::malloc(n ? n : 1);
}
void* operator new(size_t n)
{
    if (void* p = fake_new(n)) return p;
    throw std::bad_alloc();
}
void* operator new(size_t n, const std::nothrow_t&) noexcept { return fake_new(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

static constexpr size_t BYTES = (37u << 20) + 12345;  // over the threaded copy's limit, a partial last chunk

static std::vector<char> pattern(int seed)
{
    std::vector<char> v(BYTES);
    for (size_t q = 0; q < BYTES; q++) v[q] = static_cast<char>((q * 2654435761u + seed) >> 13);
    return v;
}

// A copy behind unfinished work of its stream waits for it on one thread, and
// neither channels that come and go nor another channel's copy wait with it.
static int busy()
{
    Readback& r = Readback::get();
    r.add_channel();
    r.add_channel();
    const std::vector<char> src = pattern(1), src2 = pattern(2);
    std::vector<char> dst(BYTES), dst2(BYTES);
    FakeStream slow, idle;
    slow.gate(false);
    auto copy = std::async(std::launch::async, [&] { return r.copy(dst.data(), src.data(), BYTES, 0, &slow); });
    while (slow.waiting == 0) std::this_thread::sleep_for(1ms);
    std::this_thread::sleep_for(50ms);  // the copy's other threads, if it has any, get there too
    const int waiters = slow.waiting;
    auto others = std::async(std::launch::async, [&] {
        r.add_channel();
        r.remove_channel();
    });
    const bool free_to_go = others.wait_for(5s) == std::future_status::ready;
    const hipError_t e2 = r.copy(dst2.data(), src2.data(), BYTES, 0, &idle);
    const size_t largest2 = idle.largest;
    slow.gate(true);
    const hipError_t e = copy.get();
    others.get();
    r.remove_channel();
    r.remove_channel();
    std::printf("channels free %d, threads waiting %d, the other copy's pieces up to %zu bytes\n", free_to_go, waiters,
                largest2);
    return free_to_go && waiters == 1 && largest2 < BYTES && e == hipSuccess && e2 == hipSuccess && dst == src &&
                   dst2 == src2
               ? 0
               : 1;
}

// Memory that the runtime knows (the device's, managed, pinned) is copied by one
// call of the runtime: the copy's threads could not write the device's.
static int known()
{
    Readback& r = Readback::get();
    r.add_channel();
    const std::vector<char> src = pattern(3);
    int bad = 0;
    for (int type : {hipMemoryTypeDevice, hipMemoryTypeManaged, hipMemoryTypeHost}) {
        fake_type = type;
        std::vector<char> dst(BYTES);
        FakeStream s;
        const hipError_t e = r.copy(dst.data(), src.data(), BYTES, 0, &s);
        std::printf("type %d: %d copies, the largest of %zu bytes\n", type, s.copies.load(), s.largest.load());
        bad += e != hipSuccess || dst != src || s.copies != 1 || s.largest != BYTES;
    }
    r.remove_channel();
    return bad;
}

// No host memory for the slots or for any of the threads: the copy still
// arrives, and nothing is thrown (its caller is a C function).
static int memory()
{
    const std::vector<char> src = pattern(4);
    for (int budget = 0; budget < 8; budget++) {
        std::vector<char> dst(BYTES);
        FakeStream s;
        s.queue.reserve(64);  // the runtime's own memory is another matter
        hipError_t e = hipErrorOutOfMemory;
        fake_budget = budget;
        try {
            Readback::get().add_channel();
            e = Readback::get().copy(dst.data(), src.data(), BYTES, 0, &s);
            Readback::get().remove_channel();
        } catch (const std::bad_alloc&) {
            fake_budget = -1;
            std::printf("thrown with %d allocations left\n", budget);
            return 1;
        }
        fake_budget = -1;
        if (e != hipSuccess || dst != src) return 1;
    }
    return 0;
}

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "busy") return busy();
    if (what == "known") return known();
    if (what == "memory") return memory();
    return 2;
}
