// Host helpers shared by the single-instance engine and the batch: errors,
// a small thread pool loop, the tile list and the packing of observations
// into the kernels' tile layout.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <limits>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "mds_hip.h"
#include "mds_internal.hpp"

namespace mdship {

struct Error : std::runtime_error {
    int code;
    Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

inline void check(hipError_t e, const char* what) {
    if (e != hipSuccess) {
        throw Error(MDS_HIP_ERR_DEVICE, std::string(what) + ": " + hipGetErrorString(e));
    }
}

// Parts of one allocation of pinned, coherent host memory, each on cache lines
// of its own, with the parts' device addresses.
class PinnedParts {
    struct Part {
        void **host, **dev;
        size_t offset;
    };
    std::vector<Part> parts;
    size_t total = 0;

public:
    template <typename T>
    void add(T** host, T** dev, size_t bytes) {
        parts.push_back({(void**)host, (void**)dev, total});
        total += (bytes + 255) / 256 * 256;
    }
    template <typename T>
    void add(T** host, size_t bytes) {  // a part that no kernel reaches
        add(host, (T**)nullptr, bytes);
    }
    // Sets every part's addresses; the caller frees the result (hipHostFree).
    void* allocate() {
        void *host = nullptr, *dev = nullptr;
        check(hipHostMalloc(&host, total, hipHostMallocCoherent), "hipHostMalloc");
        const hipError_t st = hipHostGetDevicePointer(&dev, host, 0);
        if (st != hipSuccess) (void)hipHostFree(host);
        check(st, "hipHostGetDevicePointer");
        for (const Part& p : parts) {
            *p.host = (char*)host + p.offset;
            if (p.dev) *p.dev = (char*)dev + p.offset;
        }
        return host;
    }
};

// Results that kernels of `stream` store into pinned host memory are waited for
// by looking at that memory: a stream wait costs another packet and its
// completion signal after the kernel (with it a single-location move at N =
// 10,000 took 19.0 us, looking 12.2).  After kSpin the looks give the processor
// away in between and the stream is asked about once per kSpin: once it is idle
// (or has failed) the memory is final.  The stream is not waited for, as work
// queued after the awaited kernel may be on it (four passes of 0.84 ms before a
// staging buffer's upload and eight after it: waiting for the buffer took 9.7
// ms with a stream wait).
template <typename Arrived>
__attribute__((noinline)) void keep_looking(hipStream_t stream, Arrived& arrived) {
    using clock = std::chrono::steady_clock;
    constexpr auto kSpin = std::chrono::microseconds(1000);
    constexpr int kLooks = 64;  // per look at the clock
    auto until = clock::now() + kSpin;
    do {
        for (int k = 0; k < kLooks; ++k) {
            if (arrived()) return;
            __builtin_ia32_pause();
        }
    } while (clock::now() < until);
    for (;;) {
        const hipError_t st = hipStreamQuery(stream);
        if (st != hipErrorNotReady) {
            check(st, "hipStreamQuery");
            return;
        }
        if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();  // no error of a later launch's
        until = clock::now() + kSpin;
        do {
            if (arrived()) return;
            std::this_thread::yield();
        } while (clock::now() < until);
    }
}
template <typename Arrived>
inline void wait_host(hipStream_t stream, Arrived arrived) {
    if (!arrived()) keep_looking(stream, arrived);
}

// `count` words in which kernels of the stream store numbers that grow from
// launch to launch: each at `value` or past it.
inline void wait_words(hipStream_t stream, const uint32_t* words, int count, uint32_t value) {
    int k = 0;
    wait_host(stream, [&] {
        while (k < count && (int32_t)(__atomic_load_n(words + k, __ATOMIC_ACQUIRE) - value) >= 0) ++k;
        return k == count;
    });
}

// Doubles that kernels store, one 8-byte store each: set to kNotYet before the
// launch (a signalling NaN, which no arithmetic gives; were it stored all the
// same, the wait would only end with the stream's work).
constexpr uint64_t kNotYet = 0x7ff4a5a5c3c3965aull;
inline void expect_values(double* v, int count) {
    for (int k = 0; k < count; ++k) __atomic_store_n((uint64_t*)v + k, kNotYet, __ATOMIC_RELAXED);
}
inline void wait_values(hipStream_t stream, const double* v, int count) {
    int k = 0;
    wait_host(stream, [&] {
        while (k < count && __atomic_load_n((const uint64_t*)v + k, __ATOMIC_ACQUIRE) != kNotYet) ++k;
        return k == count;
    });
}

inline int host_threads() {
    const unsigned hc = std::thread::hardware_concurrency();
    return (int)std::max(1u, std::min(hc == 0 ? 1u : hc, 16u));
}

template <typename F>
inline void parallel_for(size_t n, F&& f) {
    const int nt = (int)std::min<size_t>((size_t)host_threads(), std::max<size_t>(n, 1));
    if (nt <= 1) {
        f(0, n);
        return;
    }
    std::vector<std::thread> pool;
    const size_t chunk = (n + nt - 1) / nt;
    for (int k = 0; k < nt; ++k) {
        const size_t a = std::min(n, k * chunk), b = std::min(n, a + chunk);
        pool.emplace_back([&f, a, b] { f(a, b); });
    }
    for (auto& th : pool) th.join();
}

// Locations (n x p, row-major FP64) as the kernels read them: [n][kdim] in the
// engine's real type, padding coordinates 0.
template <typename Real>
inline void stage_locations(const double* loc, int n, int p, int kdim, Real* out) {
    if (p == kdim) {
        std::copy(loc, loc + (size_t)n * p, out);
        return;
    }
    for (int r = 0; r < n; ++r, loc += p, out += kdim) {
        std::copy(loc, loc + p, out);
        std::fill(out + p, out + kdim, Real(0));
    }
}

// Tile order: off-diagonal tiles (I < J) row-major, then the diagonal tiles
// (half the pairs) last, so the heavier work is dispatched first.
inline std::vector<uint32_t> make_tiles(int nb) {
    std::vector<uint32_t> t;
    t.reserve((size_t)nb * (nb + 1) / 2);
    for (int I = 0; I < nb; ++I)
        for (int J = I + 1; J < nb; ++J) t.push_back(((uint32_t)I << 16) | (uint32_t)J);
    for (int I = 0; I < nb; ++I) t.push_back(((uint32_t)I << 16) | (uint32_t)I);
    return t;
}

template <typename Real>
inline bool same_value(Real a, Real b) {
    return (a != a && b != b) || std::memcmp(&a, &b, sizeof(Real)) == 0;
}

// Packs the row-major N x N matrix into 64 x 64 tiles of the upper block
// triangle in the kernels' skewed order: element k * 64 + l of tile (I, J)
// holds delta(64 I + l, 64 J + (l + k) mod 64) in plane 0 and the transposed
// entry delta(64 J + (l + k) mod 64, 64 I + l) in plane 1.  Entries outside
// the matrix are NaN (missing).  Returns whether the stored values are
// symmetric, in which case plane 1 is not needed.
template <typename Real>
inline bool pack_tiles(const double* src, int n, const std::vector<uint32_t>& tiles, Real* plane0,
                       Real* plane1) {
    std::atomic<bool> asym(false);
    const Real nan = std::numeric_limits<Real>::quiet_NaN();
    parallel_for(tiles.size(), [&](size_t t0, size_t t1) {
        bool local = false;
        for (size_t t = t0; t < t1; ++t) {
            const int I = (int)(tiles[t] >> 16), J = (int)(tiles[t] & 0xffffu);
            Real* a = plane0 + t * kTileElems;
            Real* b = plane1 + t * kTileElems;
            // plane 0: row i fixed, columns visited in order (contiguous reads)
            for (int l = 0; l < kTile; ++l) {
                const int64_t i = (int64_t)I * kTile + l;
                for (int k = 0; k < kTile; ++k) {
                    const int64_t j = (int64_t)J * kTile + ((l + k) & (kTile - 1));
                    a[k * kTile + l] = (i < n && j < n) ? (Real)src[i * n + j] : nan;
                }
            }
            // plane 1: source row j fixed, l varies (contiguous reads)
            for (int c = 0; c < kTile; ++c) {
                const int64_t j = (int64_t)J * kTile + c;
                for (int l = 0; l < kTile; ++l) {
                    const int64_t i = (int64_t)I * kTile + l;
                    const int k = (c - l) & (kTile - 1);
                    const Real v = (i < n && j < n) ? (Real)src[j * n + i] : nan;
                    b[k * kTile + l] = v;
                    if (i < j && !same_value(v, a[k * kTile + l])) local = true;
                }
            }
        }
        if (local) asym.store(true);
    });
    return !asym.load();
}

}  // namespace mdship
