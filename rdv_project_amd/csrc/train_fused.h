// Host side of train_fused.hip for train.hip's step.
#ifndef RDV_TRAIN_FUSED_H
#define RDV_TRAIN_FUSED_H

#include "mlp_layout.h"
#include "rdv_common.h"

namespace rdv {

constexpr int kTrainFusedDepth = 5;  // hidden layers

// Whether one kernel runs the whole step of the (already checked) chain.
bool train_fused_ok(const rdv_mlp_desc& d);
// Blocks of that kernel, which each write one partial per gradient.
int train_fused_blocks(const rdv_mlp_desc& d, int64_t n, int cu);
int launch_train_fused(const rdv_mlp_desc& d, const MlpLayout& lay, const void* packed, const void* x,
                       const float* target, int64_t n, int blocks, float* loss_partial, float* const* dw,
                       float* const* db, hipStream_t stream);

}  // namespace rdv

#endif  // RDV_TRAIN_FUSED_H
