// gfx950 kernels for the pairwise truncated-normal MDS log-likelihood and its
// gradient.
//
// Work decomposition.  The N x N observation matrix is stored by the engine
// as packed 64 x 64 tiles of its upper block triangle (tile (I, J), I <= J),
// each tile in skewed order (step k, lane l) -> (row l, column (l + k) mod 64)
// so that one wavefront reads 64 consecutive values per step.  Symmetric data keep one plane; asymmetric
// data keep a second plane with the transposed tile (delta_ji), so the
// reference's row-wise semantics (row i uses delta_ij, row j uses delta_ji;
// src/NewMultiDimensionalScaling.hpp:421-461, 494-522) are reproduced while
// every transcendental is evaluated once per unordered pair.
//
// One wavefront owns one tile (small instances: several share it, see
// tile_kernel_split): lane l is row i = 64 I + l and visits the 64 columns in
// 64 steps (diagonal tiles: 32 steps, each unordered pair once).
// Row partials of the gradient stay in registers; column partials rotate
// across the wavefront with DPP; column locations are read from LDS (small
// P) or rotate with the partials.
// Each tile writes its likelihood partial and its two 64-row gradient
// partials to fixed slots; a second kernel adds them in a fixed order in
// FP64.  No atomics anywhere, so results are bitwise reproducible.
#include <algorithm>

#include "mds_hmc_device.hpp"
#include "mds_internal.hpp"
#include "mds_tile.hpp"

namespace mdship {

// Wavefronts per workgroup of the single-instance tile kernel.  FP64 with
// staged columns (P <= 2) runs eight, measured 2-4.5 % faster at
// N = 5,000-20,000: the 31 KB log Phi table is copied once per eight tiles
// instead of four.  The symmetric P = 2 walk's 76 VGPRs allow 6 wavefronts
// per SIMD, so three eight-wavefront workgroups per CU, as many as their
// 47 KB of LDS allow.  Everything else keeps four.
template <typename Real, int P>
constexpr int tile_block_waves() {
    return (sizeof(Real) == 8 && ColumnStage<Real, P>::kInLds) ? 2 * kWavesPerBlock : kWavesPerBlock;
}

// Single instance: one wavefront per tile of the upper block triangle.  The
// truncated forms copy the log Phi table into LDS and every wavefront stages
// its tile's column locations (small P); all wavefronts of the block take
// part in the barrier before any leaves.
template <typename Real, int P, bool TRUNC, bool SYM, bool GRAD, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void tile_kernel(
    const Real* __restrict__ delta, const Real* __restrict__ x,
    const uint32_t* __restrict__ tiles, int numTiles, int nb, int64_t planeStride,
    double tau, double* __restrict__ tileSums, Real* __restrict__ part, const double* __restrict__ devTau) {
    __shared__ __align__(16) Real lnPhiTab[TRUNC ? TableOf<Real>::kCount : 1];
    __shared__ __align__(16) Real colStage[WAVES][ColumnStage<Real, P>::kElems];
    const int t = __builtin_amdgcn_readfirstlane(blockIdx.x * WAVES + threadIdx.x / kWave);
    const uint32_t code = t < numTiles ? tiles[t] : 0u;
    Real* stage = colStage[threadIdx.x / kWave];
    if (t < numTiles) stage_columns<Real, P>(stage, x, (int)(code & 0xffffu));
    if constexpr (TRUNC) copy_lnphi_table(lnPhiTab);
    __syncthreads();
    if (t >= numTiles) return;
    const PairConst<Real> pc = make_pair_const<Real>(devTau ? *devTau : tau, lnPhiTab);
    tile_walk<Real, P, TRUNC, SYM, GRAD, kGroup, (sizeof(Real) == 4 ? kGroups : kPlain)>(
        delta + (int64_t)t * kTileElems, planeStride, x, stage, (int)(code >> 16), (int)(code & 0xffffu), nb, pc,
        tileSums + t, part);
}

// Small instances (split_tiles): kSegments wavefronts per tile.  A pass was
// one wavefront's walk of 64 steps, each waiting on its own latencies;
// several per tile put more wavefronts on a SIMD and shorten the walk (FP64
// P = 2, evaluation with its reduce: N = 372 untruncated 10.0 -> 7.0 us, N =
// 1,000 15.7 -> 8.9, 2,500 18.8 -> 13.3; two empty launches take 7.1; FP32 N =
// 1,000 12.3 -> 9.3).
//
// Tiles per workgroup: truncated P <= 6 share one copy of the log Phi table
// per CU while sixteen wavefronts (128 registers) hold the walk (N = 2,500,
// P = 5: 18.0 us against 19.0 with a tile each).  Others take a tile each:
// untruncated walks copy no table (N = 2,500, P = 2: 9.7 against 10.3 us), and
// from P = 8 on the registers, not the table, bound the wavefronts per CU (N =
// 2,000, P = 12: 21.9 against 27.0).
constexpr int kCUs = 256;

template <typename Real, int P, bool TRUNC>
constexpr int split_max_waves() {
    return !TRUNC || (sizeof(Real) == 8 && P > 6) ? kSegments<Real> : (sizeof(Real) == 8 ? 16 : 8);
}

template <typename Real, int P, bool TRUNC>
int split_block_tiles(int numTiles) {
    return std::min(split_max_waves<Real, P, TRUNC>() / kSegments<Real>, (numTiles + kCUs - 1) / kCUs);
}

template <typename Real, int P, bool TRUNC, bool GRAD>
constexpr size_t split_lds_bytes(int tiles) {
    const size_t table = TRUNC ? TableOf<Real>::kCount * sizeof(Real) : 0;
    const size_t stage = (size_t)tiles * ColumnStage<Real, P>::kElems * sizeof(Real);
    const size_t comb = (size_t)tiles * segment_elems<Real, P, GRAD>() * sizeof(Real);
    return table + stage > comb ? table + stage : comb;
}

template <typename Real, int P, bool TRUNC, bool SYM, bool GRAD>
__global__ __launch_bounds__((split_max_waves<Real, P, TRUNC>() * kWave)) void tile_kernel_split(
    const Real* __restrict__ delta, const Real* __restrict__ x, const uint32_t* __restrict__ tiles, int numTiles,
    int tilesPerBlock, int nb, int64_t planeStride, double tau, double* __restrict__ tileSums,
    Real* __restrict__ part, const double* __restrict__ devTau) {
    extern __shared__ __align__(16) unsigned char splitLds[];
    constexpr int kSegs = kSegments<Real>;
    Real* tab = (Real*)splitLds;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const int slot = wave / kSegs, seg = wave % kSegs;
    // wavefronts past the last tile walk it again and write nothing
    const int t = min((int)blockIdx.x * tilesPerBlock + slot, numTiles - 1);
    const uint32_t code = tiles[t];
    const int I = (int)(code >> 16), J = (int)(code & 0xffffu);
    Real* stage = tab + (TRUNC ? TableOf<Real>::kCount : 0) + slot * ColumnStage<Real, P>::kElems;
    Real* comb = (Real*)splitLds + slot * segment_elems<Real, P, GRAD>();
    segment_walk<Real, P, TRUNC, SYM, GRAD, kGroup>(delta + (int64_t)t * kTileElems, planeStride, x, stage, I, J, seg,
                                                    devTau ? *devTau : tau, tab, comb, [&] {
                                                        if (seg == 0) stage_columns<Real, P>(stage, x, J);
                                                        if constexpr (TRUNC) copy_lnphi_table(tab);
                                                        __syncthreads();
                                                    });
    __syncthreads();
    if (blockIdx.x * tilesPerBlock + slot >= numTiles) return;
    for (int a = seg; a < (GRAD ? P + 1 : 1); a += kSegs)
        combine_segments<Real, P, SYM, GRAD>(comb, a, I, J, nb, tileSums + t, part);
}

constexpr int kReduceWaves = 8;
constexpr int kReduceThreads = kReduceWaves * kWave;

// Block b + 1: gradient rows of row block b, 8 wavefronts splitting the
// column blocks J (J = w mod 8), combined through LDS in fixed order.
// Block 0: the likelihood, a fixed-order FP64 sum of the tile partials,
// halved as in src/NewMultiDimensionalScaling.hpp:556, then scaled by
// sumScale (1, or 0.5 tau for the untruncated value of :198-202), into
// sumOut and, when sumHost is set, also there (pinned host memory, which the
// host looks at: no copy command); likewise the gradient rows into grad and
// gradHost (rowsDone: see ReduceLaunch).
// Bound by the latency of the column blocks' loads: kAhead of them in flight,
// the rest one by one (groups of four or eight whose last re-read a slot, added
// or not, took N = 3,001, P = 10 from 5.8 to 7.1 us, P = 16 from 8.4 to 10.0, N =
// 500, P = 2 from 2.5 to 3.2); with a kick such groups, whose loop holds fewer
// registers beside the row's, are the faster (twenty iterations of ten steps,
// FP32 N = 1,000, P = 16: 9,050 us, one by one 9,430).  A wavefront adds and writes a coordinate; with
// gradHost a row block's values go through LDS into memory order, so that each
// store to the host link carries a wavefront's 64 neighbours (without it that
// costs 0.1-0.3 us and gives nothing).
// KICK >= 0: each row's thread then applies the sampler's kick of that form
// to its row (RowKick), so that a leapfrog step needs no kick launch of its
// own; the reduce blocks read no locations, so moving them here races with
// nothing.
template <typename PartT, int P, int KICK>
__global__ __launch_bounds__(kReduceThreads) void reduce_kernel(
    const PartT* __restrict__ part, const double* __restrict__ tileSums, int numTiles,
    int nb, int n, int pOut, double* __restrict__ grad, double* __restrict__ gradHost, double* __restrict__ sumOut,
    double* __restrict__ sumHost, double sumScale, uint32_t* __restrict__ rowsDone, uint32_t pass,
    PartT* __restrict__ kickX, double* __restrict__ kickMom, const double* __restrict__ kickParams) {
    __shared__ double red[kReduceThreads * (P > 1 ? P : 1)];
    const int tid = threadIdx.x;
    // Loads are issued kAhead iterations at a time and added in the same
    // order as a plain loop would (latency hidden, results unchanged).
    constexpr int kAhead = 4;
    if (blockIdx.x == 0) {
        double acc = 0.0;
        int k = tid;
        for (; k + (2 * kAhead - 1) * kReduceThreads < numTiles; k += 2 * kAhead * kReduceThreads) {
            double v[2 * kAhead];
#pragma unroll
            for (int u = 0; u < 2 * kAhead; ++u) v[u] = tileSums[k + u * kReduceThreads];
#pragma unroll
            for (int u = 0; u < 2 * kAhead; ++u) acc += v[u];
        }
        for (; k < numTiles; k += kReduceThreads) acc += tileSums[k];
        red[tid] = acc;
        __syncthreads();
        for (int s = kReduceThreads / 2; s > 0; s >>= 1) {
            if (tid < s) red[tid] += red[tid + s];
            __syncthreads();
        }
        if (tid == 0) {
            const double v = (0.5 * red[0]) * sumScale;  // x * 1.0 == x: the plain sum keeps its bits
            host_store(sumOut, v);  // device memory, or a sampler's pinned slot
            if (sumHost) host_store(sumHost, v);
        }
        return;
    }
    const int K = blockIdx.x - 1;
    const int wave = tid / kWave;
    const int lane = tid % kWave;
    const int row = K * kTile + lane;
    RowKick<PartT, P, KICK> kick;
    if constexpr (KICK >= 0) {
        if (wave == 0) kick.load(kickX, kickMom, kickParams, n, pOut, P, row);
    }
    double acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) acc[p] = 0.0;
    const PartT* base = part + (int64_t)K * nb * (P * kTile) + lane;
    if constexpr (KICK >= 0) {
        constexpr int kRowsAhead = P <= 4 ? 8 : kAhead;
        for (int J = wave; J < nb; J += kRowsAhead * kReduceWaves) {
            PartT v[kRowsAhead][P];
#pragma unroll
            for (int u = 0; u < kRowsAhead; ++u) {
                const PartT* slot = base + (int64_t)min(J + u * kReduceWaves, nb - 1) * (P * kTile);
#pragma unroll
                for (int p = 0; p < P; ++p) v[u][p] = slot[p * kTile];
            }
#pragma unroll
            for (int u = 0; u < kRowsAhead; ++u) {
                if (J + u * kReduceWaves < nb) {
#pragma unroll
                    for (int p = 0; p < P; ++p) acc[p] += (double)v[u][p];
                }
            }
        }
    } else {
        int J = wave;
        for (; J + (kAhead - 1) * kReduceWaves < nb; J += kAhead * kReduceWaves) {
            PartT v[kAhead][P];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                const PartT* slot = base + (int64_t)(J + u * kReduceWaves) * (P * kTile);
#pragma unroll
                for (int p = 0; p < P; ++p) v[u][p] = slot[p * kTile];
            }
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
#pragma unroll
                for (int p = 0; p < P; ++p) acc[p] += (double)v[u][p];
        }
        for (; J < nb; J += kReduceWaves) {
            const PartT* slot = base + (int64_t)J * (P * kTile);
#pragma unroll
            for (int p = 0; p < P; ++p) acc[p] += (double)slot[p * kTile];
        }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) red[(p * kReduceWaves + wave) * kWave + lane] = acc[p];
    __syncthreads();
    auto total = [&](int p, int l) {
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < kReduceWaves; ++w) v += red[(p * kReduceWaves + w) * kWave + l];
        return v;
    };
    if constexpr (KICK >= 0) {
        if (wave == 0) {
            double g[P];
#pragma unroll
            for (int p = 0; p < P; ++p) {
                g[p] = total(p, lane);
                if (row < n && p < pOut) grad[(int64_t)row * pOut + p] = g[p];
            }
            kick.apply(g, kickX, kickMom, kickParams, n, pOut, P, row);
        }
    } else if (!gradHost) {
        for (int p = wave; p < pOut; p += kReduceWaves) {
            const double v = total(p, lane);
            if (row < n) grad[(int64_t)row * pOut + p] = v;
        }
    } else {
        const int64_t first = (int64_t)K * kTile * pOut;
        const int count = min(kTile, n - K * kTile) * pOut;
        // a wavefront per coordinate adds (memory order would read one LDS bank P
        // times: 4.9 against 4.0 us at N = 3,000, P = 10), then red in memory order
        constexpr int kItems = (P * kTile + kReduceThreads - 1) / kReduceThreads;
        double v[kItems];
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int p = (tid + u * kReduceThreads) / kTile;
            v[u] = p < P ? total(p, lane) : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kItems; ++u) {
            const int p = (tid + u * kReduceThreads) / kTile;
            if (p < pOut) red[lane * pOut + p] = v[u];
        }
        __syncthreads();
        for (int o = tid; o < count; o += kReduceThreads) {
            grad[first + o] = red[o];
            host_store(gradHost + first + o, red[o]);
        }
        if (rowsDone) {
            host_stores_wait();
            __syncthreads();
            if (tid == 0) host_store(rowsDone + K, pass);
        }
    }
}

// See launch_upload.  Bound by the host link: 16 bytes per thread, all in
// flight at once (160 KB in 6.3 us, 1 KB in 3.6).  A copy command and its
// event in its place, which hand over to another engine and back, took about
// 5 us more per proposal at N = 372 (with the stream waits 36.9 us, with the
// copy gone and the waits looking at memory 22.6).
__global__ __launch_bounds__(kUploadThreads) void upload_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                                int count, uint32_t* read, uint32_t pass) {
    for (int k = blockIdx.x * kUploadThreads + threadIdx.x; k < count; k += gridDim.x * kUploadThreads)
        dst[k] = src[k];
    __syncthreads();  // every thread has stored, so read, its values
    if (threadIdx.x == 0) host_store(read + blockIdx.x, pass);
}

hipError_t launch_upload(const void* src, void* dst, size_t bytes, uint32_t* read, uint32_t pass, hipStream_t s) {
    if (!src || !dst || !read || bytes == 0 || bytes % 16 != 0) return hipErrorInvalidValue;
    hipLaunchKernelGGL(upload_kernel, dim3(upload_blocks(bytes)), dim3(kUploadThreads), 0, s, (const uint4*)src,
                       (uint4*)dst, (int)(bytes / 16), read, pass);
    return hipGetLastError();
}

template <typename Real, int P, bool TRUNC, bool SYM, bool GRAD, int WAVES>
static hipError_t go_whole(const TileLaunch& a, hipStream_t s) {
    const dim3 grid((a.numTiles + WAVES - 1) / WAVES);
    hipLaunchKernelGGL((tile_kernel<Real, P, TRUNC, SYM, GRAD, WAVES>), grid, dim3(WAVES * kWave), 0, s,
                       (const Real*)a.delta, (const Real*)a.x, a.tiles, a.numTiles, a.nb, a.planeStride, a.tau,
                       a.tileSums, (Real*)a.part, a.devTau);
    return hipGetLastError();
}

template <typename Real, int P, bool TRUNC, bool SYM, bool GRAD>
static hipError_t go(const TileLaunch& a, hipStream_t s) {
    if (a.numTiles <= split_tiles(sizeof(Real) == 4, P, TRUNC, SYM)) {
        const int tiles = split_block_tiles<Real, P, TRUNC>(a.numTiles);
        const dim3 grid((a.numTiles + tiles - 1) / tiles);
        hipLaunchKernelGGL((tile_kernel_split<Real, P, TRUNC, SYM, GRAD>), grid, dim3(tiles * kSegments<Real> * kWave),
                           (split_lds_bytes<Real, P, TRUNC, GRAD>(tiles)), s, (const Real*)a.delta, (const Real*)a.x,
                           a.tiles, a.numTiles, tiles, a.nb, a.planeStride, a.tau, a.tileSums, (Real*)a.part, a.devTau);
        return hipGetLastError();
    }
    constexpr int kWaves = tile_block_waves<Real, P>();
    if constexpr (kWaves != kWavesPerBlock && !TRUNC && !SYM) {
        // untruncated asymmetric data past their split limit: four wavefronts
        // per workgroup while these fit one per CU
        if (a.numTiles <= kWavesPerBlock * kCUs) return go_whole<Real, P, TRUNC, SYM, GRAD, kWavesPerBlock>(a, s);
    }
    return go_whole<Real, P, TRUNC, SYM, GRAD, kWaves>(a, s);
}

template <typename Real, int P>
static hipError_t dispatch_flags(const TileLaunch& a, hipStream_t s) {
    if (a.truncated) {
        if (a.symmetric)
            return a.gradient ? go<Real, P, true, true, true>(a, s) : go<Real, P, true, true, false>(a, s);
        return a.gradient ? go<Real, P, true, false, true>(a, s) : go<Real, P, true, false, false>(a, s);
    }
    if (a.symmetric)
        return a.gradient ? go<Real, P, false, true, true>(a, s) : go<Real, P, false, true, false>(a, s);
    return a.gradient ? go<Real, P, false, false, true>(a, s) : go<Real, P, false, false, false>(a, s);
}

template <typename Real>
static hipError_t dispatch_dim(const TileLaunch& a, hipStream_t s) {
    switch (a.kdim) {
        case 1: return dispatch_flags<Real, 1>(a, s);
        case 2: return dispatch_flags<Real, 2>(a, s);
        case 3: return dispatch_flags<Real, 3>(a, s);
        case 4: return dispatch_flags<Real, 4>(a, s);
        case 5: return dispatch_flags<Real, 5>(a, s);
        case 6: return dispatch_flags<Real, 6>(a, s);
        case 8: return dispatch_flags<Real, 8>(a, s);
        case 10: return dispatch_flags<Real, 10>(a, s);
        case 12: return dispatch_flags<Real, 12>(a, s);
        case 16: return dispatch_flags<Real, 16>(a, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_tiles_f64(const TileLaunch& a, hipStream_t s) { return dispatch_dim<double>(a, s); }
hipError_t launch_tiles_f32(const TileLaunch& a, hipStream_t s) { return dispatch_dim<float>(a, s); }

template <typename PartT, int P, int KICK>
static void reduce_go(const ReduceLaunch& a, hipStream_t s) {
    const dim3 grid(a.gradient ? a.nb + 1 : 1);
    hipLaunchKernelGGL((reduce_kernel<PartT, P, KICK>), grid, dim3(kReduceThreads), 0, s, (const PartT*)a.part,
                       a.tileSums, a.numTiles, a.nb, a.n, a.p, a.grad, a.gradHost, a.sumOut, a.sumHost, a.sumScale,
                       a.rowsDone, a.pass, (PartT*)a.kickX, a.kickMom, a.kickParams);
}

template <typename PartT, int P>
static hipError_t reduce_kick(const ReduceLaunch& a, hipStream_t s) {
    switch (a.kickForm) {
        case -1: reduce_go<PartT, P, -1>(a, s); break;
        case kKick: reduce_go<PartT, P, kKick>(a, s); break;
        case kKick2Drift: reduce_go<PartT, P, kKick2Drift>(a, s); break;
        default: return hipErrorInvalidValue;  // the kick that starts a trajectory has no gradient before it
    }
    return hipGetLastError();
}

template <int P>
static hipError_t reduce_p(const ReduceLaunch& a, hipStream_t s) {
    if (a.rowsDone && (!a.gradient || !a.gradHost || a.kickForm >= 0)) return hipErrorInvalidValue;
    if (a.kickForm >= 0 && (!a.gradient || !a.kickX || !a.kickMom || !a.kickParams)) return hipErrorInvalidValue;
    return a.fp32 ? reduce_kick<float, P>(a, s) : reduce_kick<double, P>(a, s);
}

hipError_t launch_reduce(const ReduceLaunch& a, hipStream_t s) {
    switch (a.kdim) {
        case 1: return reduce_p<1>(a, s);
        case 2: return reduce_p<2>(a, s);
        case 3: return reduce_p<3>(a, s);
        case 4: return reduce_p<4>(a, s);
        case 5: return reduce_p<5>(a, s);
        case 6: return reduce_p<6>(a, s);
        case 8: return reduce_p<8>(a, s);
        case 10: return reduce_p<10>(a, s);
        case 12: return reduce_p<12>(a, s);
        case 16: return reduce_p<16>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mdship
