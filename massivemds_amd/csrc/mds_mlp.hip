// Per-location MLP surrogate of the log-likelihood gradient rows (no
// counterpart in the reference): input (x_i centred and scaled, e_i) of
// P + 16 values padded to 32, two hidden layers of 256 with tanh, output the
// P gradient components (centred and scaled, padded to 16).  The centres are
// per location (the mean of x_i and of g_i over the training snapshots), the
// scales per dimension: the posterior moves each x_i by far less than the
// spread of the configuration, so a global centre would leave the network's
// BF16 inputs unable to resolve those moves.  Weights are kept in FP32 (Adam
// masters) and in BF16 copies for the MFMA matrix cores; products accumulate
// in FP32.
//
// Every product runs on v_mfma_f32_16x16x32_bf16 (lane l: A[m = l % 16][k =
// 8 (l / 16) + 0..7], B[k = 8 (l / 16) + 0..7][n = l % 16], C[row = 4 (l / 16) +
// j][col = l % 16]), each output element accumulated over k in steps of 32 from
// 0 upwards.  Weights and the operands of the weight gradients lie in memory in
// fragment order (frag_index): the 64 lanes' 8 values of one step are one
// contiguous kilobyte, so a wavefront reads an operand with one coalesced
// 16-byte load per lane.
//
// A training step is three launches: the rows (mlp_rows_kernel, forward and
// backward of 32 locations per workgroup with the activations in LDS and
// registers), the weight gradients (mlp_weights_kernel, split over kSplits
// slices of the rows) and the update (mlp_update_kernel: the slices' sums in a
// fixed order, Adam, BF16 copies).  Training is deterministic.
//
// Training step = one snapshot of all N locations, so each location's
// embedding row receives exactly one gradient row (no scatter, no atomics).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "mds_datagen.hpp"
#include "mds_engine.hpp"
#include "mds_host_store.hpp"
#include "mds_mlp.hpp"

namespace mdship {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

// Position of element (n, k) of an operand with K values of k per n, n < 16
// * groups: fragments of 16 n x 32 k, n group by n group, each in lane order.
__host__ __device__ inline int64_t frag_index(int n, int k, int K) {
    return ((int64_t)(n / 16) * (K / 32) + k / 32) * 512 + ((n % 16) + 16 * ((k % 32) / 8)) * 8 + k % 8;
}

// What the row kernel reads: BF16 weights as B operands (of W and, for the
// backward pass, of its transpose), biases, normalisation, embeddings.
struct MlpNet {
    const __bf16 *w1, *w2, *w3;     // forward: K = 32, 256, 256
    const __bf16 *w3b, *w2b, *w1b;  // backward: K = 32 (outputs, zero padded), 256, 256
    const float *b1, *b2, *b3;
    const float* norm;  // 1/sigma_x, 1/sigma_g, sigma_g (kMlpMaxP each)
    const float *xc, *gc;
    const float* emb;
    int n, p, rows;
};

// What a training pass writes: the operands of the weight gradients in
// fragment order (channels x rows), embedding gradients, row losses.
struct MlpTrainOut {
    const float* g;
    __bf16 *a0t, *h1t, *h2t, *dOutT, *dH2t, *dH1t;
    float* dEmb;
    float* lossPart;  // kMlpLoss: [gridDim.y][rows]
    int snapshots;    // kMlpLoss: of them gridDim.y, evenly spaced, are evaluated (x and g point to the first)
    // kMlpPredict: when set, the gradient goes to pinned host memory and each
    // workgroup stores `pass` in its word after its rows
    uint32_t* done;
    uint32_t pass;
};

enum MlpMode : int { kMlpPredict = 0, kMlpLoss = 1, kMlpTrain = 2 };

// Rows of one workgroup, and the LDS strides of its operands (values; padded
// so that the 16 rows a fragment read touches start four banks apart).
constexpr int kMlpRows = 32;
constexpr int kActStride = kMlpHidden + 8;
constexpr int kInStride = kMlpIn + 8;

__device__ __forceinline__ bf16x8 lds_frag(const __bf16* act, int stride, int m0, int k0) {
    const int lane = threadIdx.x % kWave;
    return *(const bf16x8*)(act + (m0 + lane % 16) * stride + k0 + (lane / 16) * 8);
}

// acc[t][q] = rows 16 t.. of act (K values) times the 16-column group q of
// the fragments from w on.
template <int KS, int NT>
__device__ __forceinline__ void rows_product(const __bf16* act, int stride, const __bf16* __restrict__ w,
                                             f32x4 (&acc)[2][NT]) {
    const bf16x8* frag = (const bf16x8*)w + threadIdx.x % kWave;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[t][q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        bf16x8 b[NT];
#pragma unroll
        for (int q = 0; q < NT; ++q) b[q] = frag[(q * KS + ks) * kWave];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const bf16x8 a = lds_frag(act, stride, 16 * t, 32 * ks);
#pragma unroll
            for (int q = 0; q < NT; ++q)
                acc[t][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[q], acc[t][q], 0, 0, 0);
        }
    }
}

// The four rows a lane holds of tile t of column group q0 + q: into LDS
// (row-major) and, with T, the fragment-order copy (columns x rows) in HBM.
__device__ __forceinline__ void put_rows(__bf16* act, __bf16* __restrict__ T, int rowBlock, int rowBlocks, int t,
                                         int group, bf16x4 v) {
    const int lane = threadIdx.x % kWave, g = lane / 16;
    __bf16* to = act + (16 * t + 4 * g) * kActStride + group * 16 + lane % 16;
#pragma unroll
    for (int j = 0; j < 4; ++j) to[j * kActStride] = v[j];
    if (T)
        *(bf16x4*)(T + ((int64_t)group * rowBlocks + rowBlock) * 512 + (lane % 16 + 16 * (2 * t + g / 2)) * 8 +
                   4 * (g % 2)) = v;
}

// 32 locations per workgroup, forward and (kMlpTrain) backward.  Four
// wavefronts, each with 64 of the 256 hidden columns of every row; the
// activations of one layer go through LDS to the next and stay in registers
// for the tanh derivatives.  The tanh evaluations bind the kernel (about 40
// VALU instructions each, 512 per location: 10 us at 20,000 locations); 32
// rows per workgroup keep the last round of workgroups short (64 rows would
// be 313 workgroups on 256 CUs).  At N = 20,000, P = 5, the same bits:
// prediction 81 us in five launches (one product each, operands and results
// through HBM) -> 19.6 us; a training step's 24 launches, 330 us -> 53 us, of
// them this kernel 30.  Three wavefronts per SIMD: the training form took 194
// registers by itself, so that 626 workgroups ran in two rounds of 512 (45 us);
// four spill nothing either but measured 33.
template <int MODE, typename XT>
__global__ __launch_bounds__(256, 3) void mlp_rows_kernel(MlpNet net, const XT* __restrict__ x, int xStride,
                                                       double* __restrict__ grad, MlpTrainOut o) {
    __shared__ __align__(16) __bf16 actA[kMlpRows * kActStride];
    __shared__ __align__(16) __bf16 actB[kMlpRows * kActStride];
    __shared__ __align__(16) __bf16 in[kMlpRows * kInStride];
    __shared__ float out[kMlpRows][kMlpOut + 1];
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    const int rowBlock = blockIdx.x, rowBlocks = net.rows / kMlpRows, row0 = rowBlock * kMlpRows;
    const int n = net.n, p = net.p;
    constexpr bool kTrain = MODE == kMlpTrain;
    if constexpr (MODE == kMlpLoss) {
        const int64_t at = ((int64_t)blockIdx.y * o.snapshots / gridDim.y) * n * p;
        x += at;
        o.g += at;
        o.lossPart += (int64_t)blockIdx.y * net.rows;
    }
    // The rows' locations, contiguous in x: read next to each other where they
    // may come over the host link.
    __shared__ float xs[MODE == kMlpPredict ? kMlpRows * kMlpMaxP : 1];
    if constexpr (MODE == kMlpPredict) {
        const int have = min(kMlpRows, n - row0) * xStride;
        for (int k = tid; k < have; k += 256) xs[k] = (float)x[(int64_t)row0 * xStride + k];
        __syncthreads();
    }

    // network inputs [ (x_i - xc_i) / sigma_x (P), e_i (16), 0 ... ]
    for (int k = tid; k < kMlpRows * kMlpIn; k += 256) {
        const int r = k / kMlpIn, c = k % kMlpIn, i = row0 + r;
        float v = 0.f;
        if (i < n) {
            if (c < p)
                v = ((MODE == kMlpPredict ? xs[r * xStride + c] : (float)x[(int64_t)i * xStride + c]) - net.xc[(int64_t)i * p + c]) * net.norm[c];
            else if (c < p + kMlpEmbed)
                v = net.emb[(int64_t)i * kMlpEmbed + (c - p)];
        }
        in[r * kInStride + c] = (__bf16)v;
    }
    __syncthreads();
    if (kTrain && tid < 2 * kWave) {  // fragment-order copy, 8 rows per thread
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = in[(8 * (lane / 16) + j) * kInStride + wave * 16 + lane % 16];
        *(bf16x8*)(o.a0t + ((int64_t)wave * rowBlocks + rowBlock) * 512 + lane * 8) = v;
    }

    f32x4 acc[2][4];
    bf16x4 h1[2][4], h2[2][4];
    const int group0 = wave * 4;  // this wavefront's first column group
    rows_product<1, 4>(in, kInStride, net.w1 + (int64_t)group0 * 512, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float bias = net.b1[(group0 + q) * 16 + lane % 16];
#pragma unroll
            for (int j = 0; j < 4; ++j) h1[t][q][j] = (__bf16)tanhf(acc[t][q][j] + bias);
            put_rows(actA, kTrain ? o.h1t : nullptr, rowBlock, rowBlocks, t, group0 + q, h1[t][q]);
        }
    __syncthreads();
    rows_product<8, 4>(actA, kActStride, net.w2 + (int64_t)group0 * 8 * 512, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float bias = net.b2[(group0 + q) * 16 + lane % 16];
#pragma unroll
            for (int j = 0; j < 4; ++j) h2[t][q][j] = (__bf16)tanhf(acc[t][q][j] + bias);
            put_rows(actB, kTrain ? o.h2t : nullptr, rowBlock, rowBlocks, t, group0 + q, h2[t][q]);
        }
    __syncthreads();
    if (wave < 2) {  // the 16 outputs: one row tile per wavefront
        const bf16x8* frag = (const bf16x8*)net.w3 + lane;
        f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < 8; ++ks)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(actB, kActStride, 16 * wave, 32 * ks),
                                                        frag[ks * kWave], c, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v = c[j];
            v += net.b3[lane % 16];
            out[16 * wave + 4 * (lane / 16) + j][lane % 16] = v;
        }
    }
    __syncthreads();
    if constexpr (MODE == kMlpPredict) {
        // gradient rows g_i = gc_i + out_i * sigma_g
        for (int k = tid; k < kMlpRows * p; k += 256) {
            const int r = k / p, c = k % p;
            const int64_t i = (int64_t)row0 * p + k;
            if (row0 + r < n) {
                const double v = (double)net.gc[i] + (double)out[r][c] * (double)net.norm[2 * kMlpMaxP + c];
                if (o.done)
                    host_store(grad + i, v);
                else
                    grad[i] = v;
            }
        }
        if (o.done) {
            host_stores_wait();
            __syncthreads();
            if (tid == 0) host_store(o.done + rowBlock, o.pass);
        }
        return;
    }
    // Loss gradient of the mean squared error over the p outputs:
    // dOut = 2 (out - t) / (n p) with t = (g - gc) / sigma_g, zero padded
    const float scale = 2.0f / ((float)n * (float)p);
    for (int k = tid; k < kMlpRows * kMlpIn; k += 256) {
        const int r = k / kMlpIn, c = k % kMlpIn, i = row0 + r;
        float d = 0.f, e = 0.f;
        if (i < n && c < p) {
            const float t = (o.g[(int64_t)i * p + c] - net.gc[(int64_t)i * p + c]) * net.norm[kMlpMaxP + c];
            e = out[r][c] - t;
            d = scale * e;
        }
        if (c < kMlpOut) out[r][c] = e;
        if (kTrain) in[r * kInStride + c] = (__bf16)d;
    }
    __syncthreads();
    if (tid < kMlpRows) {
        float l = 0.f;
        for (int c = 0; c < p; ++c) {
            const float e = out[tid][c];
            l += e * e;
        }
        o.lossPart[row0 + tid] = l;
    }
    if constexpr (!kTrain) return;
    if (tid >= 2 * kWave && tid < 3 * kWave) {
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = in[(8 * (lane / 16) + j) * kInStride + lane % 16];
        *(bf16x8*)(o.dOutT + (int64_t)rowBlock * 512 + lane * 8) = v;
    }
    // dH2 = (dOut W3^T) (1 - h2^2), dH1 = (dH2 W2^T) (1 - h1^2)
    rows_product<1, 4>(in, kInStride, net.w3b + (int64_t)group0 * 512, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bf16x4 d;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float h = (float)h2[t][q][j];
                d[j] = (__bf16)(acc[t][q][j] * (1.0f - h * h));
            }
            put_rows(actA, o.dH2t, rowBlock, rowBlocks, t, group0 + q, d);
        }
    __syncthreads();
    rows_product<8, 4>(actA, kActStride, net.w2b + (int64_t)group0 * 8 * 512, acc);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            bf16x4 d;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float h = (float)h1[t][q][j];
                d[j] = (__bf16)(acc[t][q][j] * (1.0f - h * h));
            }
            put_rows(actB, o.dH1t, rowBlock, rowBlocks, t, group0 + q, d);
        }
    __syncthreads();
    // input gradient dH1 W1^T, of which the embedding columns p .. p + 15 are used
    const int t = wave % 2, group = wave / 2;
    const bf16x8* frag = (const bf16x8*)net.w1b + (int64_t)group * 8 * kWave + lane;
    f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int ks = 0; ks < 8; ++ks)
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lds_frag(actB, kActStride, 16 * t, 32 * ks), frag[ks * kWave], c,
                                                    0, 0, 0);
    const int e = group * 16 + lane % 16 - p;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = row0 + 16 * t + 4 * (lane / 16) + j;
        if (i < n && e >= 0 && e < kMlpEmbed) o.dEmb[(int64_t)i * kMlpEmbed + e] = c[j];
    }
}

// One slice of a weight gradient dW (channels of aT x channels of yT), the
// sum over the slice's rows: 16 MT x 16 NT values per wavefront, operands
// loaded kAhead steps before their use.
template <int MT, int NT>
__device__ __forceinline__ void weight_slice(const __bf16* __restrict__ aT, const __bf16* __restrict__ yT, int m0,
                                             int n0, int firstStep, int steps, int rowBlocks, int ldc,
                                             float* __restrict__ part) {
    constexpr int kAhead = 4;
    const int lane = threadIdx.x % kWave;
    const bf16x8* a = (const bf16x8*)aT + ((int64_t)(m0 / 16) * rowBlocks + firstStep) * kWave + lane;
    const bf16x8* b = (const bf16x8*)yT + ((int64_t)(n0 / 16) * rowBlocks + firstStep) * kWave + lane;
    f32x4 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 av[kAhead][MT], bv[kAhead][NT];
    auto load = [&](int u, int step) {
        const int s = min(step, steps - 1);  // past the end: the last step again, not used
#pragma unroll
        for (int i = 0; i < MT; ++i) av[u][i] = a[((int64_t)i * rowBlocks + s) * kWave];
#pragma unroll
        for (int j = 0; j < NT; ++j) bv[u][j] = b[((int64_t)j * rowBlocks + s) * kWave];
    };
    if (steps > 0) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) load(u, u);
        for (int s0 = 0; s0 < steps; s0 += kAhead) {
#pragma unroll
            for (int u = 0; u < kAhead; ++u) {
                if (s0 + u < steps) {
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u][i], bv[u][j], acc[i][j], 0, 0, 0);
                }
                load(u, s0 + u + kAhead);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                part[(int64_t)(m0 + 16 * i + 4 * (lane / 16) + r) * ldc + n0 + 16 * j + lane % 16] = acc[i][j][r];
}

// Sums over the rows of channels c0 .. c0 + 7 of a fragment group of T: each
// (channel, row mod 256) sum in row order, then a fixed tree over the 256.
// Bound by the loads' latency and the serial additions: a thread holds 8 of
// the 256 x 8 sums and takes one 16-byte piece per 256 rows, kAhead in flight
// (N = 20,000, the whole launch: 10 us without these sums, 17 with them; 23
// with 16 channels per workgroup and a test per piece).
constexpr int kSumChannels = 8;
constexpr int kSumStride = 257;  // LDS floats per channel: a wavefront's writes on different banks

__device__ __forceinline__ void channel_sums(const __bf16* __restrict__ T, int c0, int rowBlocks,
                                             float* __restrict__ out, float* red) {
    constexpr int kChunk = 8;   // 32-row steps of 256 rows
    constexpr int kAhead = 20;
    const int step = threadIdx.x / 32, c = threadIdx.x % kSumChannels, q = (threadIdx.x / kSumChannels) % 4;
    const bf16x8* v = (const bf16x8*)T + c0 + c + 16 * q;
    float s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = 0.f;
    int at = step;
    for (; at + (kAhead - 1) * kChunk < rowBlocks; at += kAhead * kChunk) {
        bf16x8 w[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) w[u] = v[(int64_t)(at + u * kChunk) * kWave];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j) s[j] += (float)w[u][j];
    }
    if (at < rowBlocks) {  // fewer than kAhead pieces left
        bf16x8 w[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) w[u] = v[(int64_t)min(at + u * kChunk, rowBlocks - 1) * kWave];
#pragma unroll
        for (int u = 0; u < kAhead; ++u)
            if (at + u * kChunk < rowBlocks)
#pragma unroll
                for (int j = 0; j < 8; ++j) s[j] += (float)w[u][j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) red[c * kSumStride + step * 32 + q * 8 + j] = s[j];
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        for (int k = threadIdx.x; k < kSumChannels * w; k += 256) {
            const int to = (k / w) * kSumStride + k % w;
            red[to] += red[to + w];
        }
        __syncthreads();
    }
    if (threadIdx.x < kSumChannels) out[c0 + threadIdx.x] = red[threadIdx.x * kSumStride];
}

// The weight gradients' slices and the bias gradients.  Workgroups 0 ..
// kSplits * kWeightJobs - 1: slice = workgroup % kSplits (so that all readers
// of a slice's rows share an XCD's L2), job = workgroup / kSplits: 0..3 dW2
// (a 128 x 128 quarter, 64 x 64 per wavefront), 4 dW1 (32 x 64 each), 5 dW3
// (64 x 16 each).  The rest: kSumChannels channels of a bias gradient each.
constexpr int kWeightJobs = 6;
constexpr int kBiasGroups = (2 * kMlpHidden + kMlpOut) / kSumChannels;

struct MlpWeightGrads {
    const __bf16 *a0t, *h1t, *h2t, *dOutT, *dH2t, *dH1t;
    int rowBlocks, sliceSteps;
    float *part1, *part2, *part3;  // [kSplits][weights of the layer]
    float *db1, *db2, *db3;
};

__global__ __launch_bounds__(256) void mlp_weights_kernel(MlpWeightGrads a) {
    __shared__ float red[kSumChannels * kSumStride];
    const int wave = threadIdx.x / kWave;
    if (blockIdx.x >= kSplits * kWeightJobs) {
        const int channel = (blockIdx.x - kSplits * kWeightJobs) * kSumChannels;  // of dH1, dH2, dOut
        const int matrix = channel / kMlpHidden, group = channel % kMlpHidden / 16, c0 = channel % 16;
        const __bf16* T = matrix == 0 ? a.dH1t : matrix == 1 ? a.dH2t : a.dOutT;
        float* out = matrix == 0 ? a.db1 : matrix == 1 ? a.db2 : a.db3;
        channel_sums(T + (int64_t)group * a.rowBlocks * 512, c0, a.rowBlocks, out + group * 16, red);
        return;
    }
    const int slice = blockIdx.x % kSplits, job = blockIdx.x / kSplits;
    const int first = slice * a.sliceSteps;
    const int steps = max(0, min(a.sliceSteps, a.rowBlocks - first));
    if (job < 4)
        weight_slice<4, 4>(a.h1t, a.dH2t, (job / 2) * 128 + (wave / 2) * 64, (job % 2) * 128 + (wave % 2) * 64, first,
                           steps, a.rowBlocks, kMlpHidden, a.part2 + (int64_t)slice * kMlpHidden * kMlpHidden);
    else if (job == 4)
        weight_slice<2, 4>(a.a0t, a.dH1t, 0, wave * 64, first, steps, a.rowBlocks, kMlpHidden,
                           a.part1 + (int64_t)slice * kMlpIn * kMlpHidden);
    else
        weight_slice<4, 1>(a.h2t, a.dOutT, wave * 64, 0, first, steps, a.rowBlocks, kMlpOut,
                           a.part3 + (int64_t)slice * kMlpHidden * kMlpOut);
}

// Parameter i of layer matrices W1, W2, W3 (rows x cols, row-major) into its
// two BF16 copies: W as a B operand (n = column, k = row) and W^T.
__device__ __forceinline__ void pack_weight(const MlpPacked& w, int layer, int at, float value) {
    const __bf16 v = (__bf16)value;
    if (layer == 0) {
        const int r = at / kMlpHidden, c = at % kMlpHidden;
        w.w1[frag_index(c, r, kMlpIn)] = v;
        w.w1b[frag_index(r, c, kMlpHidden)] = v;
    } else if (layer == 1) {
        const int r = at / kMlpHidden, c = at % kMlpHidden;
        w.w2[frag_index(c, r, kMlpHidden)] = v;
        w.w2b[frag_index(r, c, kMlpHidden)] = v;
    } else {
        const int r = at / kMlpOut, c = at % kMlpOut;
        w.w3[frag_index(c, r, kMlpHidden)] = v;
        w.w3b[frag_index(r, c, 32)] = v;
    }
}

// Which layer's weights parameter i belongs to (-1: a bias or an embedding)
// and its index there, in the flat order W1, b1, W2, b2, W3, b3, embeddings.
__device__ __forceinline__ int weight_layer(int i, int& at) {
    constexpr int kW1 = kMlpIn * kMlpHidden, kW2 = kMlpHidden * kMlpHidden, kW3 = kMlpHidden * kMlpOut;
    constexpr int kAt2 = kW1 + kMlpHidden, kAt3 = kAt2 + kW2 + kMlpHidden;
    at = i;
    if (i < kW1) return 0;
    at = i - kAt2;
    if (at >= 0 && at < kW2) return 1;
    at = i - kAt3;
    if (at >= 0 && at < kW3) return 2;
    return -1;
}

__global__ void pack_weights_kernel(const float* __restrict__ params, int count, MlpPacked packed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    int at;
    if (i >= count) return;
    const int layer = weight_layer(i, at);
    if (layer >= 0) pack_weight(packed, layer, at, params[i]);
}

// Per parameter: the sum of its weight gradient's slices in order (weights;
// biases and embeddings have theirs already) into grad and, with ADAM, an
// Adam step (Kingma & Ba 2015) on the FP32 parameter and its BF16 copies.
template <bool ADAM>
__global__ __launch_bounds__(256) void mlp_update_kernel(float* __restrict__ w, float* __restrict__ grad,
                                                         float* __restrict__ m, float* __restrict__ v, int count,
                                                         const float* __restrict__ part1,
                                                         const float* __restrict__ part2,
                                                         const float* __restrict__ part3, MlpPacked packed, float lr,
                                                         float b1, float b2, float c1, float c2, float epsilon) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) return;
    int at;
    const int layer = weight_layer(i, at);
    float gi;
    if (layer >= 0) {
        const float* part = (layer == 0 ? part1 : layer == 1 ? part2 : part3) + at;
        const int size = layer == 0 ? kMlpIn * kMlpHidden : layer == 1 ? kMlpHidden * kMlpHidden : kMlpHidden * kMlpOut;
        float s = 0.f;
#pragma unroll
        for (int z = 0; z < kSplits; ++z) s += part[(int64_t)z * size];
        gi = s;
        grad[i] = gi;
    } else {
        gi = grad[i];
    }
    if constexpr (ADAM) {
        const float mi = b1 * m[i] + (1.f - b1) * gi;
        const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        const float wi = w[i] - lr * (mi * c1) / (sqrtf(vi * c2) + epsilon);
        w[i] = wi;
        if (layer >= 0) pack_weight(packed, layer, at, wi);
    }
}

// Per-element mean and sum of squared deviations over `count` snapshots of
// n p values each (two passes over the store, for the centres and scales);
// blockIdx.y = 0: of x, 1: of g.  The sums of squares go to pinned host memory,
// each workgroup's word after them: the host adds them in order.
__global__ __launch_bounds__(256) void snapshot_moments_kernel(const float* __restrict__ x, const float* __restrict__ g,
                                                               int count, int64_t np, float* __restrict__ mean,
                                                               float* __restrict__ ssdHost, uint32_t* done,
                                                               uint32_t pass) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const float* store = blockIdx.y ? g : x;
    if (i < np) {
        double s = 0.0;
        for (int k = 0; k < count; ++k) s += store[(int64_t)k * np + i];
        const double m = s / count;
        double q = 0.0;
        for (int k = 0; k < count; ++k) {
            const double d = store[(int64_t)k * np + i] - m;
            q += d * d;
        }
        mean[blockIdx.y * np + i] = (float)m;
        host_store(ssdHost + blockIdx.y * np + i, (float)q);
    }
    host_stores_wait();
    __syncthreads();
    if (threadIdx.x == 0) host_store(done + blockIdx.y * gridDim.x + blockIdx.x, pass);
}

// The mean over n p values of each slot's row losses, summed in FP64 (per
// thread in row order, then a fixed tree), into pinned host memory.
constexpr int kLossThreads = 1024;
__global__ __launch_bounds__(kLossThreads) void mlp_loss_kernel(const float* __restrict__ lossPart, int rows, int n,
                                                                int p, double* out) {
    __shared__ double red[kLossThreads];
    const int tid = threadIdx.x;
    const float* l = lossPart + (int64_t)blockIdx.x * rows;
    double s = 0.0;
    for (int i = tid; i < n; i += kLossThreads) s += l[i];
    red[tid] = s;
    __syncthreads();
    for (int w = kLossThreads / 2; w > 0; w >>= 1) {
        if (tid < w) red[tid] += red[tid + w];
        __syncthreads();
    }
    if (tid == 0) host_store(out + blockIdx.x, red[0] / ((double)n * p));
}

// Device memory to pinned host memory, kStageChunk doubles per workgroup, its
// word after them.
constexpr int kStageChunk = 2048;
__global__ __launch_bounds__(256) void stage_out_kernel(const double* __restrict__ src, double* __restrict__ dst,
                                                        int count, uint32_t* done, uint32_t pass) {
    const int first = blockIdx.x * kStageChunk, last = min(count, first + kStageChunk);
    for (int k = first + threadIdx.x; k < last; k += 256) host_store(dst + k, src[k]);
    host_stores_wait();
    __syncthreads();
    if (threadIdx.x == 0) host_store(done + blockIdx.x, pass);
}

// Snapshot collection: x (engine layout) and the FP64 gradient into FP32 slot
// `slot` of the store; the slot index is read from the device (advanced by
// snapshot_advance_kernel), so the step can be replayed from a graph.
template <typename XT>
__global__ void snapshot_kernel(const XT* __restrict__ x, int xStride, const double* __restrict__ grad, int n,
                                int p, float* __restrict__ sx, float* __restrict__ sg,
                                const double* __restrict__ slotPtr, int capacity) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int slot = (int)slotPtr[0];
    if (i >= n * p || slot < 0 || slot >= capacity) return;
    const int r = i / p, c = i % p;
    sx[(int64_t)slot * n * p + i] = (float)x[(int64_t)r * xStride + c];
    sg[(int64_t)slot * n * p + i] = (float)grad[i];
}

__global__ void snapshot_advance_kernel(double* __restrict__ slotPtr) {
    if (threadIdx.x == 0 && blockIdx.x == 0) slotPtr[0] += 1.0;
}

// ------------------------------------------------------------------ host

static inline int blocks_for(int64_t count, int threads = 256) { return (int)((count + threads - 1) / threads); }

Mlp::Mlp(int n_, int p_, int device_, uint64_t seed) : n(n_), p(p_), device(device_) {
    if (p < 1 || p > kMlpMaxP) throw Error(MDS_HIP_ERR_ARGUMENT, "surrogate dimension must be in [1, 16]");
    if (n < 1) throw Error(MDS_HIP_ERR_ARGUMENT, "location count must be >= 1");
    rows = (n + 63) / 64 * 64;
    check(hipSetDevice(device), "hipSetDevice");
    check(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate");
    // parameters: W1 32x256, b1 256, W2 256x256, b2 256, W3 256x16, b3 16, emb n x 16
    sizes = {kMlpIn * kMlpHidden, kMlpHidden, kMlpHidden * kMlpHidden, kMlpHidden, kMlpHidden * kMlpOut, kMlpOut,
             n * kMlpEmbed};
    offsets.resize(sizes.size());
    int total = 0;
    for (size_t k = 0; k < sizes.size(); ++k) {
        offsets[k] = total;
        total += sizes[k];
    }
    paramCount = total;
    // Glorot-uniform weights on the real fan-in / fan-out, zero biases, small
    // random embeddings; padded rows / columns stay zero
    std::vector<float> host(total, 0.f);
    mdsgen::Stream rng(seed, 31);
    auto uni = [&](float a) { return (float)((2.0 * rng.uniform() - 1.0) * a); };
    const int fanIn1 = p + kMlpEmbed;
    const float a1 = std::sqrt(6.f / (fanIn1 + kMlpHidden));
    for (int r = 0; r < fanIn1; ++r)
        for (int c = 0; c < kMlpHidden; ++c) host[offsets[0] + r * kMlpHidden + c] = uni(a1);
    const float a2 = std::sqrt(6.f / (2 * kMlpHidden));
    for (int i = 0; i < kMlpHidden * kMlpHidden; ++i) host[offsets[2] + i] = uni(a2);
    const float a3 = std::sqrt(6.f / (kMlpHidden + p));
    for (int r = 0; r < kMlpHidden; ++r)
        for (int c = 0; c < p; ++c) host[offsets[4] + r * kMlpOut + c] = uni(a3);
    for (int i = 0; i < n * kMlpEmbed; ++i) host[offsets[6] + i] = uni(0.1f);
    norm.assign(3 * kMlpMaxP, 1.f);
    try {
        check(hipMalloc((void**)&dParams, (size_t)total * sizeof(float)), "hipMalloc(mlp)");
        check(hipMalloc((void**)&dGrads, (size_t)total * sizeof(float)), "hipMalloc(mlp grads)");
        check(hipMalloc((void**)&dM, (size_t)total * sizeof(float)), "hipMalloc(adam m)");
        check(hipMalloc((void**)&dV, (size_t)total * sizeof(float)), "hipMalloc(adam v)");
        check(hipMemcpy(dParams, host.data(), (size_t)total * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        check(hipMemset(dM, 0, (size_t)total * sizeof(float)), "hipMemset");
        check(hipMemset(dV, 0, (size_t)total * sizeof(float)), "hipMemset");
        check(hipMemset(dGrads, 0, (size_t)total * sizeof(float)), "hipMemset");
        check(hipMalloc((void**)&dNorm, norm.size() * sizeof(float)), "hipMalloc(norm)");
        check(hipMemcpy(dNorm, norm.data(), norm.size() * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        check(hipMalloc((void**)&dCenter, 2 * (size_t)n * p * sizeof(float)), "hipMalloc(centres)");
        check(hipMemset(dCenter, 0, 2 * (size_t)n * p * sizeof(float)), "hipMemset");
        auto bf = [&](__bf16** ptr, size_t count) {
            check(hipMalloc((void**)ptr, count * sizeof(__bf16)), "hipMalloc(bf16)");
            check(hipMemset(*ptr, 0, count * sizeof(__bf16)), "hipMemset");
        };
        bf(&packed.w1, (size_t)kMlpIn * kMlpHidden);
        bf(&packed.w2, (size_t)kMlpHidden * kMlpHidden);
        bf(&packed.w3, (size_t)kMlpHidden * kMlpOut);
        bf(&packed.w3b, (size_t)32 * kMlpHidden);  // outputs 16..31 stay zero
        bf(&packed.w2b, (size_t)kMlpHidden * kMlpHidden);
        bf(&packed.w1b, (size_t)kMlpHidden * kMlpIn);
        bf(&a0t, (size_t)kMlpIn * rows);
        bf(&h1t, (size_t)kMlpHidden * rows);
        bf(&h2t, (size_t)kMlpHidden * rows);
        bf(&dOutT, (size_t)kMlpOut * rows);
        bf(&dH2t, (size_t)kMlpHidden * rows);
        bf(&dH1t, (size_t)kMlpHidden * rows);
        check(hipMalloc((void**)&lossPart, (size_t)kLossSlots * rows * sizeof(float)), "hipMalloc(loss)");
        check(hipMalloc((void**)&splitBuf,
                        (size_t)kSplits * (kMlpHidden * kMlpHidden + kMlpIn * kMlpHidden + kMlpHidden * kMlpOut) *
                            sizeof(float)),
              "hipMalloc(split-K)");
        const size_t np = (size_t)n * p;
        const size_t stage = std::max((size_t)total * sizeof(float), 2 * np * sizeof(double));
        const int words = std::max({rows / kMlpRows, 2 * blocks_for((int64_t)np), blocks_for(total / 2, kStageChunk)});
        PinnedParts parts;
        parts.add(&hLoss, &kLoss, kLossSlots * sizeof(double));
        parts.add(&hStage, &kStage, stage);
        parts.add(&hWords, &kWords, words * sizeof(uint32_t));
        hPinned = parts.allocate();
        std::memset(hWords, 0, words * sizeof(uint32_t));
        convertWeights();
        check(hipStreamSynchronize(stream), "hipStreamSynchronize");
    } catch (...) {
        release();
        throw;
    }
}

Mlp::~Mlp() { release(); }

void Mlp::release() {
    (void)hipSetDevice(device);
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* ptr : {(void*)dParams, (void*)dGrads, (void*)dM, (void*)dV, (void*)dNorm, (void*)dCenter,
                      (void*)packed.w1, (void*)packed.w2, (void*)packed.w3, (void*)packed.w3b, (void*)packed.w2b,
                      (void*)packed.w1b, (void*)a0t, (void*)h1t, (void*)h2t, (void*)dOutT, (void*)dH2t, (void*)dH1t,
                      (void*)lossPart, (void*)splitBuf})
        (void)hipFree(ptr);
    dParams = dGrads = dM = dV = dNorm = dCenter = lossPart = splitBuf = nullptr;
    packed = MlpPacked{};
    a0t = h1t = h2t = dOutT = dH2t = dH1t = nullptr;
    (void)hipHostFree(hPinned);
    hPinned = nullptr;
    if (stream) (void)hipStreamDestroy(stream);
    stream = nullptr;
}

void Mlp::convertWeights() {
    const int weights = offsets[5];  // everything before b3
    hipLaunchKernelGGL(pack_weights_kernel, dim3(blocks_for(weights)), dim3(256), 0, stream, dParams, weights, packed);
    check(hipGetLastError(), "pack weights");
}

MlpNet Mlp::net() const {
    MlpNet a{};
    a.w1 = packed.w1;
    a.w2 = packed.w2;
    a.w3 = packed.w3;
    a.w3b = packed.w3b;
    a.w2b = packed.w2b;
    a.w1b = packed.w1b;
    a.b1 = dParams + offsets[1];
    a.b2 = dParams + offsets[3];
    a.b3 = dParams + offsets[5];
    a.norm = dNorm;
    a.xc = dCenter;
    a.gc = dCenter + (size_t)n * p;
    a.emb = dParams + offsets[6];
    a.n = n;
    a.p = p;
    a.rows = rows;
    return a;
}

// Per-dimension scales sx, sg (p each); per-location centres xc, gc (n x p
// each, host or device pointers as `centresOnDevice` says).
void Mlp::setNormalisation(const float* xc, const float* gc, const float* sx, const float* sg,
                           bool centresOnDevice) {
    for (int c = 0; c < kMlpMaxP; ++c) {
        if (c < p && !(sx[c] > 0.f && sg[c] > 0.f)) throw Error(MDS_HIP_ERR_ARGUMENT, "scales must be > 0");
        norm[c] = c < p ? 1.f / sx[c] : 1.f;
        norm[kMlpMaxP + c] = c < p ? 1.f / sg[c] : 1.f;
        norm[2 * kMlpMaxP + c] = c < p ? sg[c] : 1.f;
    }
    check(hipMemcpyAsync(dNorm, norm.data(), norm.size() * sizeof(float), hipMemcpyHostToDevice, stream),
          "hipMemcpy(norm)");
    const size_t bytes = (size_t)n * p * sizeof(float);
    const hipMemcpyKind kind = centresOnDevice ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice;
    check(hipMemcpyAsync(dCenter, xc, bytes, kind, stream), "hipMemcpy(centres)");
    check(hipMemcpyAsync(dCenter + (size_t)n * p, gc, bytes, kind, stream), "hipMemcpy(centres)");
    // the caller's host memory has been read (device centres stay the caller's
    // until the stream has passed here)
    if (!centresOnDevice) check(hipStreamSynchronize(stream), "hipStreamSynchronize");
}

// Forward on `slots` of `snapshots` snapshots (x, g: the first, n x p FP32
// each, one after another), evenly spaced: the per-row losses into slots 0 ..
// of lossPart.  One launch: at N = 20,000, P = 5 eight snapshots take 86
// us (by themselves 17.4 each, 626 workgroups that fill the chip once).
void Mlp::lossOnly(const float* x, const float* g, int snapshots, int slots) {
    MlpTrainOut o{};
    o.g = g;
    o.lossPart = lossPart;
    o.snapshots = snapshots;
    hipLaunchKernelGGL((mlp_rows_kernel<kMlpLoss, float>), dim3(rows / kMlpRows, slots), dim3(256), 0, stream, net(), x,
                       p, nullptr, o);
    check(hipGetLastError(), "loss kernel");
}

// One forward + backward on a snapshot: the slices of the weight gradients,
// the bias and embedding gradients (in dGrads) and the per-row losses.
void Mlp::backpropagate(const float* x, const float* g) {
    MlpTrainOut o{};
    o.g = g;
    o.a0t = a0t;
    o.h1t = h1t;
    o.h2t = h2t;
    o.dOutT = dOutT;
    o.dH2t = dH2t;
    o.dH1t = dH1t;
    o.dEmb = dGrads + offsets[6];
    o.lossPart = lossPart;
    hipLaunchKernelGGL((mlp_rows_kernel<kMlpTrain, float>), dim3(rows / kMlpRows), dim3(256), 0, stream, net(), x, p,
                       nullptr, o);
    check(hipGetLastError(), "row kernel");
    MlpWeightGrads a{};
    a.a0t = a0t;
    a.h1t = h1t;
    a.h2t = h2t;
    a.dOutT = dOutT;
    a.dH2t = dH2t;
    a.dH1t = dH1t;
    a.rowBlocks = rows / 32;
    a.sliceSteps = (a.rowBlocks + kSplits - 1) / kSplits;  // trailing slices may be empty
    a.part2 = splitBuf;
    a.part1 = a.part2 + (size_t)kSplits * kMlpHidden * kMlpHidden;
    a.part3 = a.part1 + (size_t)kSplits * kMlpIn * kMlpHidden;
    a.db1 = dGrads + offsets[1];
    a.db2 = dGrads + offsets[3];
    a.db3 = dGrads + offsets[5];
    hipLaunchKernelGGL(mlp_weights_kernel, dim3(kSplits * kWeightJobs + kBiasGroups), dim3(256), 0, stream, a);
    check(hipGetLastError(), "weight gradient kernel");
}

// adam: also the parameter update at rate lr.
void Mlp::finishGradients(bool adam, float lr) {
    const float* part2 = splitBuf;
    const float* part1 = part2 + (size_t)kSplits * kMlpHidden * kMlpHidden;
    const float* part3 = part1 + (size_t)kSplits * kMlpIn * kMlpHidden;
    if (adam) {
        ++adamStep;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f / (1.f - std::pow(b1, (float)adamStep));
        const float c2 = 1.f / (1.f - std::pow(b2, (float)adamStep));
        hipLaunchKernelGGL(mlp_update_kernel<true>, dim3(blocks_for(paramCount)), dim3(256), 0, stream, dParams,
                           dGrads, dM, dV, paramCount, part1, part2, part3, packed, lr, b1, b2, c1, c2, 1e-8f);
    } else {
        const int weights = offsets[5];
        hipLaunchKernelGGL(mlp_update_kernel<false>, dim3(blocks_for(weights)), dim3(256), 0, stream, dParams, dGrads,
                           dM, dV, weights, part1, part2, part3, packed, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f);
    }
    check(hipGetLastError(), "update kernel");
}

// One forward + backward on a snapshot: fills the parameter gradients dGrads
// and the per-row losses.
void Mlp::lossAndGradient(const float* x, const float* g) {
    backpropagate(x, g);
    finishGradients(false, 0.f);
}

void Mlp::trainStep(const float* x, const float* g, float lr) {
    backpropagate(x, g);
    finishGradients(true, lr);
}

// The mean losses of the first `slots` slots of lossPart, one after another
// in out.
void Mlp::losses(int slots, double* out) {
    std::lock_guard<std::mutex> lock(stageLock);
    expect_values(hLoss, slots);
    hipLaunchKernelGGL(mlp_loss_kernel, dim3(slots), dim3(kLossThreads), 0, stream, lossPart, rows, n, p, kLoss);
    check(hipGetLastError(), "loss sum kernel");
    wait_values(stream, hLoss, slots);
    std::copy(hLoss, hLoss + slots, out);
}

// The sums over locations of the squared deviations from the snapshots' means,
// per dimension, of x and g; mean: x's (n x p), then g's.
void Mlp::moments(const float* x, const float* g, int count, float* mean, double* qx, double* qg) {
    std::lock_guard<std::mutex> lock(stageLock);
    const int64_t np = (int64_t)n * p;
    const int blocks = blocks_for(np);
    hipLaunchKernelGGL(snapshot_moments_kernel, dim3(blocks, 2), dim3(256), 0, stream, x, g, count, np, mean,
                       (float*)kStage, kWords, ++stagePass);
    check(hipGetLastError(), "snapshot moments");
    wait_words(stream, hWords, 2 * blocks, stagePass);
    const float *sx = (const float*)hStage, *sg = sx + np;
    std::fill(qx, qx + p, 0.0);
    std::fill(qg, qg + p, 0.0);
    for (int i = 0; i < n; ++i, sx += p, sg += p)
        for (int c = 0; c < p; ++c) {
            qx[c] += sx[c];
            qg[c] += sg[c];
        }
}

// The gradient rows at host locations (n x p): the row kernel reads the staged
// locations and writes the rows itself, and they are copied as they arrive
// (N = 20,000, P = 5, through the API: 88 us, 122 with two device buffers and a
// copy command each way).
void Mlp::predictHost(const double* x, double* grad) {
    std::lock_guard<std::mutex> lock(stageLock);
    const size_t np = (size_t)n * p;
    double *in = (double*)hStage, *out = in + np;
    std::copy(x, x + np, in);
    predictInto<double>((const double*)kStage, p, (double*)kStage + np, stream, kWords, ++stagePass);
    const size_t chunk = (size_t)kMlpRows * p;
    for (size_t k = 0; k * chunk < np; ++k) {
        wait_words(stream, hWords + k, 1, stagePass);
        std::memcpy(grad + k * chunk, out + k * chunk, std::min(chunk, np - k * chunk) * sizeof(double));
    }
}

void Mlp::parametersToHost(float* out) {
    static_assert(kMlpEmbed % 2 == 0 && kMlpHidden % 2 == 0 && kMlpOut % 2 == 0, "the parameters are whole doubles");
    std::lock_guard<std::mutex> lock(stageLock);
    const size_t count = (size_t)paramCount / 2;
    hipLaunchKernelGGL(stage_out_kernel, dim3(blocks_for((int64_t)count, kStageChunk)), dim3(256), 0, stream,
                       (const double*)dParams, (double*)kStage, (int)count, kWords, ++stagePass);
    check(hipGetLastError(), "parameter read-back kernel");
    for (size_t k = 0; k * kStageChunk < count; ++k) {
        const size_t at = k * kStageChunk, len = std::min<size_t>(kStageChunk, count - at);
        wait_words(stream, hWords + k, 1, stagePass);
        std::memcpy(out + 2 * at, (const double*)hStage + at, len * sizeof(double));
    }
}

template <typename XT>
void Mlp::predictInto(const XT* x, int xStride, double* grad, hipStream_t s, uint32_t* done, uint32_t pass) {
    MlpTrainOut o{};
    o.done = done;
    o.pass = pass;
    hipLaunchKernelGGL((mlp_rows_kernel<kMlpPredict, XT>), dim3(rows / kMlpRows), dim3(256), 0, s, net(), x, xStride,
                       grad, o);
    check(hipGetLastError(), "predict kernel");
}

template void Mlp::predictInto<double>(const double*, int, double*, hipStream_t, uint32_t*, uint32_t);
template void Mlp::predictInto<float>(const float*, int, double*, hipStream_t, uint32_t*, uint32_t);

void launch_snapshot(const Engine& e, const double* grad, float* sx, float* sg, const double* slotPtr,
                     int capacity, hipStream_t s) {
    const int count = e.N * e.P;
    if (e.fp32)
        hipLaunchKernelGGL((snapshot_kernel<float>), dim3(blocks_for(count)), dim3(256), 0, s,
                           (const float*)e.dX[e.cur], e.kdim, grad, e.N, e.P, sx, sg, slotPtr, capacity);
    else
        hipLaunchKernelGGL((snapshot_kernel<double>), dim3(blocks_for(count)), dim3(256), 0, s,
                           (const double*)e.dX[e.cur], e.kdim, grad, e.N, e.P, sx, sg, slotPtr, capacity);
    hipLaunchKernelGGL(snapshot_advance_kernel, dim3(1), dim3(64), 0, s, (double*)slotPtr);
    check(hipGetLastError(), "snapshot kernels");
}

SnapshotStore::SnapshotStore(int n_, int p_, int capacity_, int device_)
    : n(n_), p(p_), capacity(capacity_), device(device_) {
    if (capacity < 1) throw Error(MDS_HIP_ERR_ARGUMENT, "snapshot capacity must be >= 1");
    const size_t bytes = (size_t)capacity * n * p * sizeof(float);
    try {
        check(hipMalloc((void**)&sx, bytes), "hipMalloc(snapshots x)");
        check(hipMalloc((void**)&sg, bytes), "hipMalloc(snapshots g)");
        check(hipMalloc((void**)&dSlot, 2 * sizeof(double)), "hipMalloc(slot)");
        check(hipMemset(dSlot, 0, 2 * sizeof(double)), "hipMemset(slot)");
    } catch (...) {
        (void)hipFree(sx);
        (void)hipFree(sg);
        (void)hipFree(dSlot);
        throw;
    }
}

SnapshotStore::~SnapshotStore() {
    (void)hipSetDevice(device);
    (void)hipFree(sx);
    (void)hipFree(sg);
    (void)hipFree(dSlot);
}

int SnapshotStore::count() {
    double v = 0.0;
    check(hipDeviceSynchronize(), "hipDeviceSynchronize");
    check(hipMemcpy(&v, dSlot, sizeof(double), hipMemcpyDeviceToHost), "hipMemcpy(slot)");
    return std::min((int)v, capacity);
}

// Trains on every stored snapshot `epochs` times in a shuffled order, Adam
// with a cosine learning-rate decay to lr / 20.  Inputs and targets are
// centred per location on their means over all snapshots and scaled per
// dimension by the root mean square deviation.  Returns the mean squared
// error (normalised targets) over up to 32 snapshots after training.
double Surrogate::train(int epochs, double lr) {
    const int count = store.count();
    if (count < 1) throw Error(MDS_HIP_ERR_STATE, "no snapshots to train on");
    if (epochs < 1 || !(lr > 0)) throw Error(MDS_HIP_ERR_ARGUMENT, "epochs >= 1 and learning rate > 0 required");
    const int n = store.n, p = store.p;
    const size_t np = (size_t)n * p;
    if (!dMeans) check(hipMalloc((void**)&dMeans, 2 * np * sizeof(float)), "hipMalloc(means)");
    std::vector<double> qx(p), qg(p);
    mlp.moments(store.sx, store.sg, count, dMeans, qx.data(), qg.data());
    std::vector<float> sx(p), sg(p);
    for (int c = 0; c < p; ++c) {
        sx[c] = (float)std::sqrt(std::max(qx[c] / ((double)n * count), 1e-30));
        sg[c] = (float)std::sqrt(std::max(qg[c] / ((double)n * count), 1e-30));
    }
    mlp.setNormalisation(dMeans, dMeans + np, sx.data(), sg.data(), true);
    mdsgen::Stream rng(seed, 91);
    std::vector<int> order(count);
    const long long total = (long long)epochs * count;
    long long step = 0;
    for (int ep = 0; ep < epochs; ++ep) {
        for (int k = 0; k < count; ++k) order[k] = k;
        for (int k = count - 1; k > 0; --k) std::swap(order[k], order[(int)(rng.uniform() * (k + 1))]);
        for (int k = 0; k < count; ++k, ++step) {
            const double frac = (double)step / std::max(1LL, total - 1);
            const float rate = (float)(lr * (0.05 + 0.95 * 0.5 * (1.0 + std::cos(M_PI * frac))));
            mlp.trainStep(store.sx + (size_t)order[k] * np, store.sg + (size_t)order[k] * np, rate);
        }
    }
    double l = 0.0, each[kLossSlots];
    const int evals = std::min(count, kLossSlots);
    mlp.lossOnly(store.sx, store.sg, count, evals);
    mlp.losses(evals, each);
    for (int q = 0; q < evals; ++q) l += each[q];
    return l / evals;
}

}  // namespace mdship

static thread_local std::string g_surrogate_error = "no error";

template <typename F>
static int sguard(mds_hip_surrogate_handle h, F&& f) {
    if (!h || !h->s) {
        g_surrogate_error = "null handle";
        return MDS_HIP_ERR_ARGUMENT;
    }
    try {
        (void)hipSetDevice(h->s->mlp.device);
        f(*h->s);
        return MDS_HIP_OK;
    } catch (const mdship::Error& err) {
        h->s->lastError = err.what();
        return err.code;
    } catch (const std::exception& err) {
        h->s->lastError = err.what();
        return MDS_HIP_ERR_DEVICE;
    }
}

extern "C" {

int mds_hip_surrogate_create(int locationCount, int embeddingDimension, int snapshotCapacity,
                             unsigned long long seed, int device, mds_hip_surrogate_handle* out) {
    if (!out) {
        g_surrogate_error = "null output handle";
        return MDS_HIP_ERR_ARGUMENT;
    }
    *out = nullptr;
    try {
        int devices = 0;
        mdship::check(hipGetDeviceCount(&devices), "hipGetDeviceCount");
        if (devices <= 0) throw mdship::Error(MDS_HIP_ERR_DEVICE, "no HIP device");
        const int dev = (device < 0 || device >= devices) ? 0 : device;
        *out = new mds_hip_surrogate{
            new mdship::Surrogate(locationCount, embeddingDimension, snapshotCapacity, seed, dev)};
        return MDS_HIP_OK;
    } catch (const mdship::Error& err) {
        g_surrogate_error = err.what();
        return err.code;
    } catch (const std::exception& err) {
        g_surrogate_error = err.what();
        return MDS_HIP_ERR_DEVICE;
    }
}

int mds_hip_surrogate_destroy(mds_hip_surrogate_handle h) {
    if (!h) return MDS_HIP_ERR_ARGUMENT;
    delete h->s;
    delete h;
    return MDS_HIP_OK;
}

const char* mds_hip_surrogate_last_error(mds_hip_surrogate_handle h) {
    if (!h || !h->s) return g_surrogate_error.c_str();
    return h->s->lastError.c_str();
}

int mds_hip_surrogate_snapshot_count(mds_hip_surrogate_handle h, int* count) {
    return sguard(h, [&](mdship::Surrogate& s) {
        if (!count) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "null output pointer");
        *count = s.store.count();
    });
}

int mds_hip_surrogate_add_snapshot(mds_hip_surrogate_handle h, const double* x, const double* g, size_t length) {
    return sguard(h, [&](mdship::Surrogate& s) {
        const size_t np = (size_t)s.store.n * s.store.p;
        if (!x || !g || length != np) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "snapshot length must be N*P");
        const int slot = s.store.count();
        if (slot >= s.store.capacity) throw mdship::Error(MDS_HIP_ERR_STATE, "snapshot store full");
        std::vector<float> fx(np), fg(np);
        for (size_t k = 0; k < np; ++k) {
            fx[k] = (float)x[k];
            fg[k] = (float)g[k];
        }
        mdship::check(hipMemcpy(s.store.sx + (size_t)slot * np, fx.data(), np * sizeof(float), hipMemcpyHostToDevice),
                      "hipMemcpy");
        mdship::check(hipMemcpy(s.store.sg + (size_t)slot * np, fg.data(), np * sizeof(float), hipMemcpyHostToDevice),
                      "hipMemcpy");
        const double next = slot + 1;
        mdship::check(hipMemcpy(s.store.dSlot, &next, sizeof(double), hipMemcpyHostToDevice), "hipMemcpy");
    });
}

int mds_hip_surrogate_train(mds_hip_surrogate_handle h, int epochs, double learningRate, double* finalLoss) {
    return sguard(h, [&](mdship::Surrogate& s) {
        const double l = s.train(epochs, learningRate);
        if (finalLoss) *finalLoss = l;
    });
}

int mds_hip_surrogate_predict(mds_hip_surrogate_handle h, const double* x, size_t length, double* grad) {
    return sguard(h, [&](mdship::Surrogate& s) {
        const size_t np = (size_t)s.mlp.n * s.mlp.p;
        if (!x || !grad || length != np) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "length must be N*P");
        s.mlp.predictHost(x, grad);
    });
}

int mds_hip_surrogate_parameter_count(mds_hip_surrogate_handle h, long long* count) {
    return sguard(h, [&](mdship::Surrogate& s) {
        if (!count) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "null output pointer");
        *count = s.mlp.paramCount;
    });
}

int mds_hip_surrogate_get_parameters(mds_hip_surrogate_handle h, float* out, size_t count) {
    return sguard(h, [&](mdship::Surrogate& s) {
        if (!out || count != (size_t)s.mlp.paramCount) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "wrong length");
        s.mlp.parametersToHost(out);
    });
}

int mds_hip_surrogate_set_parameters(mds_hip_surrogate_handle h, const float* in, size_t count) {
    return sguard(h, [&](mdship::Surrogate& s) {
        if (!in || count != (size_t)s.mlp.paramCount) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "wrong length");
        mdship::check(hipMemcpy(s.mlp.dParams, in, count * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
        s.mlp.convertWeights();
        mdship::check(hipStreamSynchronize(s.mlp.stream), "hipStreamSynchronize");
    });
}

int mds_hip_surrogate_set_normalisation(mds_hip_surrogate_handle h, const float* xCentre, const float* gCentre,
                                        size_t centreLength, const float* sigmaX, const float* sigmaG,
                                        size_t scaleLength) {
    return sguard(h, [&](mdship::Surrogate& s) {
        if (!xCentre || !gCentre || !sigmaX || !sigmaG || centreLength != (size_t)s.mlp.n * s.mlp.p ||
            scaleLength != (size_t)s.mlp.p)
            throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "centres must hold N*P values and scales P");
        s.mlp.setNormalisation(xCentre, gCentre, sigmaX, sigmaG, false);
    });
}

int mds_hip_surrogate_loss_gradient(mds_hip_surrogate_handle h, const double* x, const double* g, size_t length,
                                    float* paramGrad, size_t count, double* loss) {
    return sguard(h, [&](mdship::Surrogate& s) {
        const size_t np = (size_t)s.mlp.n * s.mlp.p;
        if (!x || !g || length != np) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "length must be N*P");
        if (paramGrad && count != (size_t)s.mlp.paramCount) throw mdship::Error(MDS_HIP_ERR_ARGUMENT, "wrong length");
        std::vector<float> fx(np), fg(np);
        for (size_t k = 0; k < np; ++k) {
            fx[k] = (float)x[k];
            fg[k] = (float)g[k];
        }
        float *dx = nullptr, *dg = nullptr;
        try {
            mdship::check(hipMalloc((void**)&dx, np * sizeof(float)), "hipMalloc");
            mdship::check(hipMalloc((void**)&dg, np * sizeof(float)), "hipMalloc");
            mdship::check(hipMemcpy(dx, fx.data(), np * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
            mdship::check(hipMemcpy(dg, fg.data(), np * sizeof(float), hipMemcpyHostToDevice), "hipMemcpy");
            s.mlp.lossAndGradient(dx, dg);
            double l = 0.0;
            s.mlp.losses(1, &l);
            if (loss) *loss = l;
            if (paramGrad)
                mdship::check(hipMemcpy(paramGrad, s.mlp.dGrads, count * sizeof(float), hipMemcpyDeviceToHost),
                              "hipMemcpy");
        } catch (...) {
            (void)hipFree(dx);
            (void)hipFree(dg);
            throw;
        }
        (void)hipFree(dx);
        (void)hipFree(dg);
    });
}

}  // extern "C"
