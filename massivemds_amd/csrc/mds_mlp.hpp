// Per-location MLP surrogate of the gradient rows (see mds_mlp.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <mutex>
#include <vector>

#include "mds_engine.hpp"

namespace mdship {

constexpr int kMlpIn = 32;      // P + 16 embedding values, zero padded
constexpr int kMlpHidden = 256;
constexpr int kMlpOut = 16;     // P outputs, zero padded
constexpr int kMlpEmbed = 16;
constexpr int kMlpMaxP = 16;
constexpr int kSplits = 32;     // K slices of the weight-gradient products

constexpr int kLossSlots = 32;  // snapshots whose losses are evaluated after training

// BF16 copies of the weights as the row kernel reads them (see mds_mlp.hip).
struct MlpPacked {
    __bf16 *w1 = nullptr, *w2 = nullptr, *w3 = nullptr;     // forward
    __bf16 *w3b = nullptr, *w2b = nullptr, *w1b = nullptr;  // transposed, backward
};
struct MlpNet;

struct Mlp {
    int n = 0, p = 0, device = 0, rows = 0;
    hipStream_t stream = nullptr;
    std::vector<int> sizes, offsets;
    int paramCount = 0;
    long long adamStep = 0;
    float* dParams = nullptr;  // W1 (32x256), b1, W2 (256x256), b2, W3 (256x16), b3, embeddings (n x 16)
    float* dGrads = nullptr;
    float* dM = nullptr;
    float* dV = nullptr;
    std::vector<float> norm;   // 1/sigma_x, 1/sigma_g, sigma_g (kMlpMaxP each)
    float* dNorm = nullptr;
    float* dCenter = nullptr;  // per-location centres: x (n x p), then g (n x p)
    MlpPacked packed;
    // operands of the weight gradients of one training step (channels x rows)
    __bf16 *a0t = nullptr, *h1t = nullptr, *h2t = nullptr;
    __bf16 *dOutT = nullptr, *dH2t = nullptr, *dH1t = nullptr;
    float* lossPart = nullptr;  // [kLossSlots][rows]
    float* splitBuf = nullptr;  // slices of the weight gradients: W2, W1, W3
    // Pinned, coherent host memory (k*: device addresses): the mean losses,
    // and a stage for what one call at a time (stageLock) exchanges with the
    // device, whose kernels number their workgroups' words.
    std::mutex stageLock;
    void* hPinned = nullptr;
    double *hLoss = nullptr, *kLoss = nullptr;
    char *hStage = nullptr, *kStage = nullptr;
    uint32_t *hWords = nullptr, *kWords = nullptr;
    uint32_t stagePass = 0;

    Mlp(int n, int p, int device, uint64_t seed);
    ~Mlp();
    void release();
    void convertWeights();
    MlpNet net() const;
    void lossOnly(const float* x, const float* g, int snapshots, int slots);
    void backpropagate(const float* x, const float* g);
    void finishGradients(bool adam, float lr);
    void losses(int slots, double* out);
    void setNormalisation(const float* xc, const float* gc, const float* sx, const float* sg, bool centresOnDevice);
    void lossAndGradient(const float* x, const float* g);
    void trainStep(const float* x, const float* g, float lr);
    template <typename XT>
    void predictInto(const XT* x, int xStride, double* grad, hipStream_t s, uint32_t* done = nullptr,
                     uint32_t pass = 0);
    void predictHost(const double* x, double* grad);
    void moments(const float* x, const float* g, int count, float* mean, double* qx, double* qg);
    void parametersToHost(float* out);
};

// Device store of (x, gradient) snapshots in FP32, [capacity][n][p] each;
// the next slot index is kept on the device so that collection can run
// inside a captured graph.
struct SnapshotStore {
    int n = 0, p = 0, capacity = 0, device = 0;
    float* sx = nullptr;
    float* sg = nullptr;
    double* dSlot = nullptr;  // [0] next slot, [1] the value at the current trajectory's start
    SnapshotStore(int n, int p, int capacity, int device);
    ~SnapshotStore();
    int count();
};

struct Surrogate {
    Mlp mlp;
    SnapshotStore store;
    float* dMeans = nullptr;  // the snapshots' means, while train() takes them over
    uint64_t seed;
    std::string lastError;
    Surrogate(int n, int p, int capacity, uint64_t seed, int device)
        : mlp(n, p, device, seed), store(n, p, capacity, device), seed(seed) {}
    ~Surrogate() {
        (void)hipSetDevice(mlp.device);
        if (mlp.stream) (void)hipStreamSynchronize(mlp.stream);
        (void)hipFree(dMeans);
    }
    double train(int epochs, double lr);
};

void launch_snapshot(const Engine& e, const double* grad, float* sx, float* sg, const double* slotPtr,
                     int capacity, hipStream_t s);

}  // namespace mdship

struct mds_hip_surrogate {
    mdship::Surrogate* s;
};
