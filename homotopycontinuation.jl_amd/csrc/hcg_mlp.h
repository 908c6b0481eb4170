// Learned step-size proposer: host interface of the hand-written HIP training kernels.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>

#include "hcg_mlp_work.h"
#include "hcgpu.h"

namespace hcg {

void mlp_work_free(MlpWork* w);
int mlp_forward_backward(MlpWork* w, hipStream_t s, const float* params, int32_t n, const float* x, const float* y,
                         const float* wt, float* out_pred, float* loss, float* grad, std::string* err);
int mlp_train(MlpWork* w, hipStream_t s, float* params, int32_t n, const float* x, const float* y, const float* wt,
              int32_t epochs, int32_t batch, float lr, uint64_t seed, float* final_loss, std::string* err);

}  // namespace hcg
