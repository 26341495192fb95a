// The host's wait for results that kernels store into pinned memory
// (massivemds_amd/csrc/mds_host.hpp) over a stub stream: a word that arrives
// while later work keeps the stream busy ends the wait without a stream wait;
// an idle stream ends it, whatever the memory holds; a failed one raises.
// Exit status 0 = as stated.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <thread>

#include "mds_host.hpp"

static std::atomic<int> g_streamWaits{0}, g_queries{0};
static std::atomic<hipError_t> g_stream{hipErrorNotReady};
static thread_local hipError_t g_last = hipSuccess;

extern "C" {
hipError_t hipStreamSynchronize(hipStream_t) {
    ++g_streamWaits;
    return hipSuccess;
}
hipError_t hipStreamQuery(hipStream_t) {
    ++g_queries;
    g_last = g_stream;
    return g_stream;
}
hipError_t hipPeekAtLastError() { return g_last; }
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "stub"; }
hipError_t hipHostMalloc(void**, size_t, unsigned int) { return hipErrorOutOfMemory; }
hipError_t hipHostGetDevicePointer(void**, void*, unsigned int) { return hipErrorOutOfMemory; }
hipError_t hipHostFree(void*) { return hipSuccess; }
}

static int g_failed = 0;
static void expect(bool ok, const char* what) {
    if (!ok) {
        std::printf("failed: %s\n", what);
        g_failed = 1;
    }
}

int main() {
    using namespace mdship;
    const auto later = [](auto store, int ms) {
        return std::thread([=] {
            std::this_thread::sleep_for(std::chrono::milliseconds(ms));
            store();
        });
    };
    {
        uint32_t word = 6;
        const auto start = std::chrono::steady_clock::now();
        std::thread t = later([&] { __atomic_store_n(&word, 7u, __ATOMIC_RELEASE); }, 20);
        wait_words(nullptr, &word, 1, 7);
        const std::chrono::duration<double, std::milli> took = std::chrono::steady_clock::now() - start;
        t.join();
        expect(g_streamWaits == 0, "a word's arrival ends the wait, not the stream's end");
        expect(g_queries > 0 && g_queries <= took.count(), "the stream is asked about once a millisecond at most");
        expect(hipGetLastError() == hipSuccess, "no error is left behind");
    }
    {
        double v = 0.0;
        expect_values(&v, 1);
        std::thread t = later([&] { __atomic_store_n((uint64_t*)&v, 0x3ff0000000000000ull, __ATOMIC_RELEASE); }, 5);
        wait_values(nullptr, &v, 1);
        t.join();
        expect(v == 1.0 && g_streamWaits == 0, "a value's arrival ends the wait");
    }
    {
        uint32_t word = 6;
        std::thread t = later([&] { g_stream = hipSuccess; }, 5);
        wait_words(nullptr, &word, 1, 7);
        t.join();
        expect(word == 6, "an idle stream ends the wait");
    }
    {
        uint32_t word = 6;
        g_stream = hipErrorLaunchFailure;
        bool raised = false;
        try {
            wait_words(nullptr, &word, 1, 7);
        } catch (const Error& e) {
            raised = e.code == MDS_HIP_ERR_DEVICE;
        }
        expect(raised, "a failed stream raises");
    }
    return g_failed;
}
