// rvk_lanes.hip -- the DRR casters with several lanes of a wave on one ray,
// for launches whose rays do not fill the device (drr_march_lanes).
//
// A wave takes 64 >> ls pixels, a Morton-order block of a tile, and the lanes
// of one ray are neighbours, so their samples, consecutive on the ray, share
// cells within one load.
#include "rvk_lanes.h"

namespace rvk {

template <typename CV, bool SKIP, bool RUNS>
__global__ __launch_bounds__(256) void drr_lanes_kernel(DrrArgs a, int ls) {
  const int blk = a.deal ? xcd_deal(blockIdx.x, kDealLog2 + ls) : xcd_remap(blockIdx.x, gridDim.x);
  int x, y;
  lanes_pixel(blk, a.tiles_x, ls, x, y);
  if (x >= a.v.W || y >= a.v.H) return;
  const Ray r = form_ray(a.g, a.v, a.step_len, x, y);
  const float v = drr_march_lanes<CV, SKIP, RUNS>(cells_of<CV>(a.vol), a.g, a.m, r, x, y, ls);
  if ((threadIdx.x & ((1 << ls) - 1)) == 0) drr_store(a, x, y, v);
}

int launch_drr_lanes(const DrrArgs& a, const rvk_volume* vol, int frame, bool skip, int ls, int nblk, hipStream_t s) {
  const dim3 grid(a.deal ? deal_grid((long long)nblk << ls, kDealLog2 + ls) : (unsigned)nblk << ls);
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    const bool runs = a.m.ranges != nullptr;
    if (skip && runs) hipLaunchKernelGGL((drr_lanes_kernel<CV, true, true>), grid, dim3(256), 0, s, a, ls);
    else if (skip) hipLaunchKernelGGL((drr_lanes_kernel<CV, true, false>), grid, dim3(256), 0, s, a, ls);
    else if (runs) hipLaunchKernelGGL((drr_lanes_kernel<CV, false, true>), grid, dim3(256), 0, s, a, ls);
    else hipLaunchKernelGGL((drr_lanes_kernel<CV, false, false>), grid, dim3(256), 0, s, a, ls);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

// The wave's part of a work item of the plan's tile shape.
__device__ __forceinline__ void item_part_pixel(int shape, int tiles16_x, int local, int part, int ls, int& x, int& y) {
  const int macro = local >> 2, q = local & 3;
  const int p = (part << (6 - ls)) | ((int)(threadIdx.x & 63u) >> ls);  // pixel of the item
  if (shape == RVK_TILE_16X4) {
    x = p & 15;
    y = q * 4 + (p >> 4);
  } else if (shape == RVK_TILE_4X16) {
    x = q * 4 + (p & 3);
    y = p >> 2;
  } else {
    morton_pixel((q << 6) | p, x, y);
  }
  x += (macro % tiles16_x) * 16;
  y += (macro / tiles16_x) * 16;
}

__device__ __forceinline__ void group_sum(V3<float>& v, int S) {
  for (int o = 1; o < S; o <<= 1) {
    v.x += __shfl_xor(v.x, o, 64);
    v.y += __shfl_xor(v.y, o, 64);
    v.z += __shfl_xor(v.z, o, 64);
  }
}

// Part w mod 2^ls of work item w >> ls.
template <typename CV, bool SKIP, bool JAC>
__device__ __forceinline__ void lanes_part(const BatchArgs& a, int w, int ls) {
  const int2 vt = a.work[w >> ls];
  const BatchView& bv = a.views[__builtin_amdgcn_readfirstlane(vt.x)];
  int x, y;
  item_part_pixel(a.shape, bv.tiles16_x, __builtin_amdgcn_readfirstlane(vt.y), w & ((1 << ls) - 1), ls, x, y);
  if (x >= bv.v.W || y >= bv.v.H) return;
  const Ray r = form_ray(a.g, bv.v, a.step_len, x, y);
  const long long pi = bv.pix_off + (long long)y * bv.v.W + x;
  const bool lead = (threadIdx.x & ((1 << ls) - 1)) == 0;
  if (!JAC) {
    const float v = drr_march_lanes<CV, SKIP, true>(cells_of<CV>(a.vol), a.g, a.m, r, x, y, ls);
    if (lead) a.out[pi] = v;
    return;
  }
  V3<float> A{0, 0, 0}, B{0, 0, 0};
  PoseVisit visit{ray_offset(a.m.jitter, x, y), A, B};
  const float v = drr_march_lanes<CV, SKIP, true, true>(cells_of<CV>(a.vol), a.g, a.m, r, x, y, ls, visit);
  if (lead) a.out[pi] = v;
  // the lanes' sums added, lane s forms pose directions s, s + 2^ls, ...
  // (dL/dpose_i = A . dstart_i + B . dinc_i)
  const int S = 1 << ls;
  group_sum(A, S);
  group_sum(B, S);
  const bool any = A.x != 0.0f || A.y != 0.0f || A.z != 0.0f || B.x != 0.0f || B.y != 0.0f || B.z != 0.0f;
  if (any) pose_sums(ray_length(a.g, r.inc) * a.m.slope, A, B);
  for (int i = (int)(threadIdx.x & (S - 1)); i < 6; i += S) {
    float jv = 0.0f;
    if (any) {
      const RayTangent tg = form_ray_tangent(a.g, bv.v, bv.dm + 16 * i, a.step_len, x, y);
      jv = A.x * tg.dstart.x + A.y * tg.dstart.y + A.z * tg.dstart.z + B.x * tg.dinc.x + B.y * tg.dinc.y +
           B.z * tg.dinc.z;
    }
    a.jac[i * a.total + pi] = jv;
  }
}

template <typename CV, bool SKIP, bool JAC>
__global__ __launch_bounds__(256) void batch_lanes_kernel(BatchArgs a, int ls) {
  const int blk = a.deal ? xcd_deal(blockIdx.x, kDealLog2 + ls) : xcd_remap(blockIdx.x, gridDim.x);
  const int w = blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if ((w >> ls) >= a.n_items) return;
  lanes_part<CV, SKIP, JAC>(a, w, ls);
}

// The persistent schedule (batch_persistent_kernel), over the items' parts.
template <typename CV, bool SKIP, bool JAC>
__global__ __launch_bounds__(256) void batch_lanes_persistent_kernel(BatchArgs a, int ls) {
  const int home = blockIdx.x % kNumXcd;
  const long long parts = (long long)a.n_items << ls;
  for (int r = 0; r < kNumXcd; ++r) {
    const int c = (home + r) % kNumXcd;
    const int begin = (int)(parts * c / kNumXcd), end = (int)(parts * (c + 1) / kNumXcd);
    while (true) {
      int w = 0;
      if ((threadIdx.x & 63) == 0) w = (int)atomicAdd(&a.queues[c], 1u);
      w = begin + __builtin_amdgcn_readfirstlane(w);
      if (w >= end) break;
      lanes_part<CV, SKIP, JAC>(a, w, ls);
    }
  }
}

int launch_batch_lanes(const BatchArgs& a, const rvk_volume* vol, int frame, bool skip, bool jac, int ls,
                       unsigned persistent, hipStream_t s) {
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    auto go = [&](auto S, auto J) {
      constexpr bool kSkip = decltype(S)::value, kJac = decltype(J)::value;
      if (persistent)
        hipLaunchKernelGGL((batch_lanes_persistent_kernel<CV, kSkip, kJac>), dim3(persistent), dim3(256), 0, s, a, ls);
      else
        hipLaunchKernelGGL((batch_lanes_kernel<CV, kSkip, kJac>), dim3(batch_grid(a, ls)), dim3(256), 0, s, a, ls);
    };
    if (jac) skip ? go(std::true_type(), std::true_type()) : go(std::false_type(), std::true_type());
    else skip ? go(std::true_type(), std::false_type()) : go(std::false_type(), std::false_type());
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

}  // namespace rvk
