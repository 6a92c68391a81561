// rvk_volgrad.h -- the volume adjoint of a DRR plan (rvk_volgrad.hip).
#pragma once
#include "rvk_batch.h"

namespace rvk {

constexpr int kVgSlots = 64;        // where the launch's largest |coef| is collected,
constexpr int kVgSlotStride = 16;   // each on a line of its own
struct VolGradArgs {
  BatchArgs b;
  const float* img;
  const float* dldi;
  unsigned* slots;          // bits of the largest |coef| (+inf if one is not finite)
  unsigned long long* acc;  // fixed-point sums, one per voxel
  float* grad;              // dims x-fastest
};
int launch_volume_grad(const VolGradArgs& a, const rvk_volume* vol, int frame, hipStream_t s);

}  // namespace rvk
