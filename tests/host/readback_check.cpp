// The host logic of readback.hpp against a double of the runtime (hip/hip_runtime.h
// here): one check per argument, exit status 0 when it holds.
#include "readback.hpp"

#include <chrono>
#include <cstdio>
#include <future>
#include <string>

using chan::Readback;
using namespace std::chrono_literals;

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

int main(int argc, char** argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "busy") return busy();
    if (what == "known") return known();
    return 2;
}
