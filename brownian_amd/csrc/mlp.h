// Surrogate network interface shared by the step (api.cpp) and the network
// kernels (mlp.hip).
#pragma once
#include <hip/hip_runtime.h>

struct bw_mlp;

namespace bw {

constexpr int MLP_IN = 144, MLP_INP = 160, MLP_H = 256, MLP_OUT = 12, MLP_OUTP = 32, MLP_T = 6;
constexpr int MLP_L = 4;

// activations of one forward/backward pass over up to `cap` rows
struct MlpBuf {
    int cap = 0;
    unsigned short *Xb = nullptr, *Hb[3] = {};
    float *Y = nullptr;
    // training only: pre-activations, output gradients, two layers' dZ in turn,
    // losses, partial sums of the parameter gradients
    unsigned short *dYb = nullptr, *dZb[2] = {};
    float *Z[3] = {}, *dY = nullptr, *dZ[2] = {}, *loss = nullptr, *part = nullptr;
};
int mlp_buf_alloc(MlpBuf &b, int rows, bool train = false);  // hipMalloc; 0 on success
void mlp_buf_free(MlpBuf &b);

// features x (n x 144 raw units, device) -> y_out (n x 12, device): impulse
// mean (6) and log-variance (6) in physical units; launches only, on `st`
void mlp_forward_device(bw_mlp *m, MlpBuf &b, const float *x, int n, float *y_out, hipStream_t st);

}  // namespace bw
