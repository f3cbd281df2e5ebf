// Device-side interface of the learned warm start: network shape and kernel launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "spg_vbd_learned.h"

namespace spgvbd {

constexpr int kMlpFeatures = 24;  // per-vertex input features
constexpr int kMlpIn = 32;        // features zero-padded to one MFMA K step
constexpr int kMlpHidden = 128;
constexpr int kMlpOut = 3;
constexpr int kMlpOutPad = 32;  // output rows of the last weight padded to one MFMA K step
constexpr int kMlpLayers = 4;

constexpr int kMlpPadded = kMlpHidden * (kMlpIn + 1) + 2 * kMlpHidden * (kMlpHidden + 1) + kMlpOutPad * (kMlpHidden + 1);

// The gradient of one batch: rows index[0 .. n) (0 .. n without an index) of a feature table (n x 24 FP32, standardised
// here) and its targets (n x 3), in `parts` workgroups that share the row blocks of mlpTrainBlocks(n); each leaves its
// sums in partial (kMlpPadded floats, padded master layout) and its squared error in lossPartial.
struct MlpTrainArgs {
    const float *features, *targets;
    const int32_t *index;
    const float *mean, *invStd;
    const float *params;  // padded master layout (the biases are read from it)
    const void *frag;
    int32_t n, rowBlocks;
    float *partial;
    double *lossPartial;
};
int mlpTrainBlocks(int64_t rows);
hipError_t launchMlpTrain(const MlpTrainArgs &a, int parts, hipStream_t stream);
// The sums over the parts: into grad, or (adam) an Adam step of the parameters, moments and fragments. Adds the batch's
// squared error to *loss.
struct MlpUpdateArgs {
    const float *partial;
    const double *lossPartial;
    int32_t parts;
    double *loss;
    float *grad;
    float *params, *m, *v;
    void *frag;
    float lr, b1, b2, eps, c1, c2;  // c1, c2: 1 - b1^t, 1 - b2^t
};
hipError_t launchMlpUpdate(const MlpUpdateArgs &a, bool adam, hipStream_t stream);

// The weights in the kernels' operand order, for inference and the gradient: rebuilt from the FP32 master parameters
// (padded layout) by launchMlpFrag, kept up to date by launchMlpUpdate.
size_t mlpFragBytes();
hipError_t launchMlpFrag(const float *params, void *frag, hipStream_t stream);
// Fused inference: all layers in registers, weights staged in LDS.
// y[row][0..2] = network(f[row]) for rows < n (f: n x 24 FP32, y stride ldy >= 3); at most maxBlocks
// persistent workgroups of 256 threads.
hipError_t launchMlpInfer(const float *f, int n, const float *mean, const float *invStd, const void *frag,
                          const float *b1, const float *b2, const float *b3, const float *b4, float *y, int ldy,
                          int maxBlocks, hipStream_t stream);

// Inputs of the feature kernel (warmstart_kernels.hip), slot numbering of a VBD context.
struct FeatureArgs {
    const float4 *xt = nullptr;    // inertial target (w: mass)
    const float4 *vel = nullptr;   // velocity after the substep's gravity kick
    const float4 *corr = nullptr;  // x* - x~ of the previous substep
    const int32_t *nbPtr = nullptr;
    const int32_t *nbIdx = nullptr;
    const float *nbRest = nullptr;  // rest length of each one-ring edge
    const float4 *stat = nullptr;   // (log10 Y, log10 k_bending, anchored, 0)
    int32_t n = 0;
    float h = 0.f, gx = 0.f, gy = 0.f, gz = 0.f;
    float invS = 0.f, invU = 0.f;  // 1 / (h^2 a_ref), 1 / (h a_ref)
    float *out = nullptr;          // n x kMlpFeatures
};

hipError_t launchFeatures(const FeatureArgs &a, hipStream_t stream);
// x = x~ + base + s y (base may be null: x~ + s y)
hipError_t launchApplyWarmStart(float4 *pos, const float4 *xt, const float4 *base, const float *y, int32_t ldy, float s,
                                int32_t n,
                                hipStream_t stream);
// y, out: n rows of 4 floats (the first three are the displacement)
hipError_t launchSmoothPrediction(const float *y, float *out, const int32_t *nbPtr, const int32_t *nbIdx, int32_t n,
                                  hipStream_t stream);
hipError_t launchGate(float4 *pos, const float4 *xt, const int32_t *objOfSlot, const int32_t *reject, int32_t n,
                      hipStream_t stream);

// Network inference on device-resident features (n x kMlpFeatures FP32) into y (n rows, stride
// ldy >= kMlpOut), ordered on `stream`, with the fused kernel. Throws VbdError. Defined with the
// network object.
void mlpInferDevice(spg_mlp *net, const float *features, int64_t n, float *y, int32_t ldy, hipStream_t stream);
// The same on the network's own stream, after `ready` (recorded by the caller); records `done`, which
// the caller waits on before it reads y.
void mlpInferAfter(spg_mlp *net, const float *features, int64_t n, float *y, int32_t ldy, hipEvent_t ready,
                   hipEvent_t done);
int mlpDevice(const spg_mlp *net);
int mlpHistoryBase(const spg_mlp *net);

}  // namespace spgvbd
