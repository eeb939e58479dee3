// mlp.h -- the stepping network (internal): sizes, device parameter views,
// launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hipdvr {

constexpr int kMlpIn = 16;       // brick/TF/octant features (zero padded)
constexpr int kMlpHidden = 64;
constexpr int kMlpOut = 2;       // skip logit, log2 step multiplier
constexpr int kMlpTargets = 3;   // skip label, log2 multiplier label, multiplier weight
constexpr int kMlpParams = kMlpIn * kMlpHidden + kMlpHidden + kMlpHidden * kMlpHidden + kMlpHidden +
                           kMlpHidden * kMlpOut + kMlpOut;

// BF16 weights and FP32 biases the kernels read.
struct MlpDevParams {
    short* w1;   // [16][64]
    short* w2;   // [64][64]
    short* w3;   // [64][16], columns >= 2 zero
    float* b;    // b1[64] b2[64] b3[2]
    // the weights once more in the order the gradient kernel's lanes hold them
    // as MFMA operands (pack_param)
    short* frag;   // [kMlpFrag]
};
constexpr int kMlpFrag = kMlpIn * kMlpHidden + 2 * kMlpHidden * kMlpHidden + kMlpHidden * kMlpOut;

// Gradient sums of one workgroup (kMlpParams, then the loss), and workgroups:
// one per compute unit (512 at 8192 rows: 14.7 us and 5.9 for the sums, 256:
// 14.2 and 4.7).
constexpr int kMlpPartial = (kMlpParams + 1 + 3) / 4 * 4;
constexpr uint32_t kMlpGradBlocks = 256;

void launch_mlp_pack(const float* master, const MlpDevParams& p, hipStream_t st);
void launch_mlp_forward(const MlpDevParams& p, const float* x, uint32_t rows, float* y, hipStream_t st);
// Gradient sums per workgroup into partial [kMlpGradBlocks][kMlpPartial];
// returns the number of workgroups (0 rows: none).
uint32_t launch_mlp_grad(const MlpDevParams& p, const float* x, const float* tgt, uint32_t rows, float* partial,
                         hipStream_t st);
// Sums the workgroups' gradients into grad and loss.
void launch_mlp_sum(const float* partial, uint32_t blocks, float* grad, float* loss, hipStream_t st);
// The same, with an Adam step on the master parameters and their packed copies.
void launch_mlp_update(const float* partial, uint32_t blocks, float* grad, float* loss, float* w, float* m, float* v,
                       const MlpDevParams& p, float lr, int step, hipStream_t st);

}  // namespace hipdvr
