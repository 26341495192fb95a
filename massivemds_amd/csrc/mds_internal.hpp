// Host-side declarations shared by the kernel launchers and the engine.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace mdship {

constexpr int kWave = 64;                 // CDNA wavefront width
constexpr int kTile = 64;                 // tile edge: 64 rows (one per lane) x 64 columns
constexpr int kTileElems = kTile * kTile;
constexpr int kWavesPerBlock = 4;
constexpr int kBlockThreads = kWave * kWavesPerBlock;

// Kernel embedding dimensions that are compiled; a location dimension P runs
// on the smallest of these >= P with zero-padded coordinates (padding adds 0
// to every distance and gradient).
constexpr int kKernelDims[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16};
constexpr int kMaxDim = 16;

inline int kernel_dim(int p) {
    for (int d : kKernelDims)
        if (d >= p) return d;
    return -1;
}

// Small instances are walked by several wavefronts per tile (the split walk);
// their FP64 additions take the groups those wavefronts walk (GroupSum)
// wherever they are evaluated, so that every launch gives the same bits.
// FP32 additions take groups at every size.
//
// The limit, in tiles: 1024 (N <= 2,816: no more tiles than the MI355X has
// SIMDs, so that a wavefront per tile would leave every SIMD waiting on one
// walk's latencies).  FP64 only: untruncated asymmetric data, two planes and
// little arithmetic, are bound by memory once they exceed the L2s (512 tiles,
// 32 MB): split they measured 13.4 -> 14.0-14.7 us at N = 2,500, P = 3; and
// P > 12 (over 200 registers, 67 KB of group sums per tile) fits two
// workgroups per CU, split beyond 768 tiles 32.3 -> 33.3 us at N = 2,800.
inline int split_tiles(bool fp32, int kdim, bool truncated, bool symmetric) {
    if (fp32) return 1024;
    if (!truncated && !symmetric) return 512;
    return kdim > 12 ? 768 : 1024;
}

inline bool grouped_order(bool fp32, int kdim, bool truncated, bool symmetric, int numTiles) {
    return fp32 || numTiles <= split_tiles(fp32, kdim, truncated, symmetric);
}

// One fused evaluation over the packed upper-triangle tiles.
struct TileLaunch {
    const void* delta;       // packed tiles, Real, [planes][numTiles][64 cols][64 rows]
    const void* x;           // Real [nb * 64][kdim], zero padded
    const uint32_t* tiles;   // (I << 16) | J for I <= J, one per tile
    int numTiles;
    int nb;                  // 64-row blocks
    int kdim;                // kernel dimension
    int64_t planeStride;     // elements between the two planes (asymmetric data)
    double tau;
    bool truncated;
    bool symmetric;
    bool gradient;
    double* tileSums;        // [numTiles]
    void* part;              // [nb][nb][kdim][64] gradient partials, Real
    const double* devTau = nullptr;  // if set, the precision is read from here
};

struct ReduceLaunch {
    const void* part;        // gradient partials in the engine's real type (fp32: float)
    bool fp32;
    const double* tileSums;
    int numTiles;
    int nb;
    int kdim;
    int n;
    int p;                   // output dimension (<= kdim)
    bool gradient;
    double* grad;            // [n][p]
    double* gradHost = nullptr;  // optional second copy of it (pinned host memory)
    double* sumOut;          // 1 double: (0.5 * sum of tile sums) * sumScale
    double* sumHost = nullptr;  // optional second copy of it (pinned host memory)
    double sumScale = 1.0;
    // With gradHost: each workgroup stores `pass` in its word here after its
    // rows, so that the host can see them arrive (nb words of coherent pinned
    // host memory).
    uint32_t* rowsDone = nullptr;
    uint32_t pass = 0;
    // Optional HMC kick of each gradient row right after it is written
    // (kickForm: a KickForm of the sampler, or -1 for none): the locations
    // (the engine's real type, [n][kdim]), the momenta [n][p] and the
    // sampler's parameter block.
    int kickForm = -1;
    void* kickX = nullptr;
    double* kickMom = nullptr;
    const double* kickParams = nullptr;
};

// Change of the raw sum of increments when one location row moves (O(N)):
// per block of kRowThreads locations j, the partial
// sum_j [term(delta_ij, d_new) - term(delta_ij, d_old) + the same for delta_ji]
// over observed entries, written to partial[block] (device-accessible; the
// engine passes coherent pinned host memory) -- the caller adds the
// partials in order and halves.
constexpr int kRowThreads = 256;

struct RowDeltaLaunch {
    const void* delta;       // packed tiles as in TileLaunch
    void* x;                 // Real [nb * 64][kdim]; row `row` holds the previous location,
                             // also after the launch
    double xNew[kMaxDim];    // the row's new location (the engine's real type, widened), P values
    int row;
    int carryRow;            // >= 0: a row whose location is xCarry, not what x holds; the
    double xCarry[kMaxDim];  // launch writes it into x
    int n;
    int nb;
    int kdim;
    int p;
    int64_t planeStride;
    double tau;
    bool truncated;
    bool symmetric;
    bool fp32;               // Real = float (else double)
    double* partial;         // [blocks(n)]
};

// Writes one location row (the engine's real type; padding dimensions stay 0).
struct RowWrite {
    void* x;
    double values[kMaxDim];
    int row, kdim, p;
    bool fp32;
};
hipError_t launch_row_write(const RowWrite& w, hipStream_t s);

// Pinned host memory into a device buffer (multiples of 16 bytes); each
// workgroup stores `pass` in its word of `read` (coherent pinned host memory)
// once it has read its part.
constexpr int kUploadThreads = 256, kUploadBlocks = 256;
inline int upload_blocks(size_t bytes) {
    const size_t want = (bytes / 16 + kUploadThreads - 1) / kUploadThreads;
    return want < (size_t)kUploadBlocks ? (int)want : kUploadBlocks;
}
hipError_t launch_upload(const void* src, void* dst, size_t bytes, uint32_t* read, uint32_t pass, hipStream_t s);

inline int row_delta_blocks(int n) { return (n + kRowThreads - 1) / kRowThreads; }

hipError_t launch_row_delta(const RowDeltaLaunch& a, hipStream_t s);
hipError_t launch_tiles_f64(const TileLaunch& a, hipStream_t s);
hipError_t launch_tiles_f32(const TileLaunch& a, hipStream_t s);
hipError_t launch_reduce(const ReduceLaunch& a, hipStream_t s);

}  // namespace mdship
