// dbx_mlp.h -- learned warm start for new contact points (host side).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "../../include/dbox_hip.h"
#include "dbx_device.h"
#include "dbx_mlp_dev.h"

namespace dbx {

struct MlpState {
    bool ready = false;     // parameters and normalisation loaded
    float *params = nullptr; // fp32 parameters (kMlpParams)
    float *grad = nullptr;
    float *adam1 = nullptr, *adam2 = nullptr;
    float *norm = nullptr;   // kMlpNorm
    bf16x8 *frag = nullptr;  // packed MFMA operands
    float *loss = nullptr;
    int adamStep = 0;
    std::vector<void *> allocs;
};

void mlp_release(MlpState &m);
hipError_t mlp_ensure(MlpState &m, hipStream_t s);
MlpDev mlp_dev(const MlpState &m);
// Uploads parameters and/or normalisation (either may be null) and repacks.
hipError_t mlp_upload(MlpState &m, const float *params, const float *norm, hipStream_t s);
// Predicted normal and tangent impulse y[2i], y[2i+1] of feature row i of x (rows of kMlpIn
// floats), both in pinned host memory (x readable to the next multiple of 16 bytes); then
// the signal.
hipError_t mlp_forward(MlpState &m, const float *x, int n, float *y, HostSignal sig, hipStream_t s);
// Accumulates into m.grad the gradient of the mean squared error over `batch` samples of
// X (rows of kMlpFeatStride) and T, and adds the loss to *dLoss (zeroed by the caller);
// samples are drawn with replacement by `seed`.
hipError_t mlp_gradients(MlpState &m, const float *dX, const float *dT, long long n, long long batch, uint64_t seed,
                         float *dLoss, hipStream_t s);
// The same over the n rows of x and t in pinned host memory (as mlp_forward's), weighted
// 1 / total, with the loss added to m.loss.
hipError_t mlp_gradients_rows(MlpState &m, const float *x, const float *t, long long n, long long total, hipStream_t s);
// m.grad and then m.loss to pinned host memory (kMlpParams + 1 floats) and cleared;
// then the signal.
hipError_t mlp_take(MlpState &m, float *out, HostSignal sig, hipStream_t s);
hipError_t mlp_fill(float *p, long long n, float v, hipStream_t s);
hipError_t mlp_adam_step(MlpState &m, float lr, hipStream_t s);
hipError_t mlp_clear_grad(MlpState &m, hipStream_t s);

} // namespace dbx
