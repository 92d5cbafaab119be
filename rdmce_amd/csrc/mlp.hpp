// Learned root-cost model: sizes and kernel launchers (mlp.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace rdmce {

constexpr int kFeat = 8;
constexpr int kH1 = 32;
constexpr int kH2 = 32;
// Trainable floats: W1, b1, W2, b2, W3, b3.
constexpr int kTrainFloats = kFeat * kH1 + kH1 + kH1 * kH2 + kH2 + kH2 + 1;
// Plus the input normalisation (mean, 1/std per feature).
constexpr int kParamFloats = kTrainFloats + 2 * kFeat;

hipError_t launch_features(const uint64_t *rowoff, const uint32_t *col, const uint32_t *core, float inv_degen,
                           const uint64_t *roots, uint64_t n_roots, float *out, hipStream_t s);
hipError_t launch_forward(const float *params, const float *X, uint64_t n, float *out, hipStream_t s);
uint32_t backward_blocks(uint64_t count);
// Adam settings of one step (bias corrections of step number `step`), the
// partial gradients it sums (`blocks` of them; 0: no update) and the state it
// reads and writes: m, v and the parameters go to other buffers than they are
// read from.
struct AdamStep {
  float lr, b1, b2, eps, bc1, bc2;
  uint32_t blocks;
  const float *partial, *loss_partial;
  const float *m_in, *v_in;
  float *m_out, *v_out, *p_out, *loss;
};
AdamStep adam_step(float lr, int step);
// Up to this many blocks a step's update is done by the next step's launch,
// which every block repeats; beyond, the repeated reads (5.5 KB per block and
// partial) outweigh the launch they save.
constexpr uint32_t kFusedBlocks = 32;
// Partial gradients of one step over samples idx[0, count) (nullptr: 0 ..),
// after the update `apply` of the parameters when it has blocks.
hipError_t launch_step(const float *params, const float *X, const float *Y, const uint32_t *idx, uint64_t count,
                       float *partial, float *loss_partial, const AdamStep &apply, hipStream_t s);
hipError_t launch_reduce(const float *partial, uint32_t blocks, float *grad, const float *loss_partial, float *loss,
                         hipStream_t s);
hipError_t launch_adam(const float *params, const AdamStep &apply, hipStream_t s);

}  // namespace rdmce
