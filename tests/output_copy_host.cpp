// OutputCopy (csrc/output_copy.hpp) on the CPU: the runtime's calls are stood in for by a queue whose copies
// happen when an event after them, or the stream, is waited for. Exit status 0: every byte arrived.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

static std::atomic<long> g_countdown{-1};  // the allocation that fails, counted from where it is set
static bool g_no_pinned = false;

void* operator new(std::size_t n) {
    if (g_countdown.load() >= 0 && g_countdown.fetch_sub(1) == 0) throw std::bad_alloc();
    if (void* p = std::malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

struct Queued {
    void* dst;
    const void* src;
    std::size_t bytes;
};
static Queued g_queue[4096];
static int g_head = 0, g_tail = 0;
static int g_event[64], g_events = 0;

static void drain(int to) {
    for (; g_head < to; ++g_head) std::memcpy(g_queue[g_head].dst, g_queue[g_head].src, g_queue[g_head].bytes);
}

extern "C" {
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = nullptr;
    if (!g_no_pinned) *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    if (g_tail == 4096) return hipErrorOutOfMemory;
    g_queue[g_tail++] = {d, s, n};
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(&g_event[g_events++]);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    *reinterpret_cast<int*>(e) = g_tail;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    drain(*reinterpret_cast<int*>(e));
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    drain(g_tail);
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "stood in"; }
}

#include "output_copy.hpp"

int main(int argc, char** argv) {
    const long fail = argc > 1 ? std::atol(argv[1]) : -1;
    g_no_pinned = argc > 2 && std::atoi(argv[2]) != 0;
    cn::OutputCopy copy;
    const std::size_t mb = std::size_t{1} << 20;
    for (std::size_t bytes : {std::size_t{0}, std::size_t{5}, 4 * mb - 1, 4 * mb, 4 * mb + 1, 12 * mb, 13 * mb + 7, 40 * mb + 3}) {
        std::vector<unsigned char> src(bytes), dst(bytes + 16, 0xA5);
        for (std::size_t i = 0; i < bytes; ++i) src[i] = static_cast<unsigned char>((i * 2654435761u) >> 13);
        g_countdown = fail;
        copy.run(dst.data(), src.data(), bytes, nullptr);
        g_countdown = -1;
        if (std::memcmp(dst.data(), src.data(), bytes) != 0) return std::printf("wrong bytes of %zu\n", bytes), 1;
        for (std::size_t i = bytes; i < bytes + 16; ++i)
            if (dst[i] != 0xA5) return std::printf("past the end of %zu\n", bytes), 1;
    }
    return 0;
}
