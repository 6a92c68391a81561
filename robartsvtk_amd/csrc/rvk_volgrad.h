// rvk_volgrad.h -- the volume adjoint of a DRR plan: by ray tiles
// (rvk_volgrad.hip) or by voxel bricks (rvk_volbrick.hip), the same sums.
#pragma once
#include "rvk_batch.h"

namespace rvk {

constexpr int kVgSlots = 64;        // where the launch's largest |coef| is collected,
constexpr int kVgSlotStride = 16;   // each on a line of its own
constexpr int kVgEdge = 8;          // voxels along a brick

// A ray as the bricks read it back.
struct alignas(16) RayRec {
  float p0x, p0y, p0z;  // start in cell coordinates (p0 + 0.5)
  float coef;           // d loss / d L_p * ds * slope
  float ix, iy, iz;     // step
  int n;                // samples
  float cs, ci;         // alpha = cs * value + ci
  float kw0, kw1;       // keyhole window: samples t in [kw0, kw1) are never accumulated
};
static_assert(sizeof(RayRec) == 48, "RayRec is three 16-byte vectors");

struct VolGradArgs {
  BatchArgs b;
  const float* img;
  const float* dldi;
  unsigned* slots;          // bits of the largest |coef| (+inf if one is not finite)
  unsigned long long* acc;  // fixed-point sums, one per voxel (tiles)
  RayRec* rays;             // packed like the images (bricks)
  float* grad;              // dims x-fastest
};
constexpr int kVgNonFinite = 1 << 30;

struct VgRay {
  V3<float> p0c, inc;
  int n;
  float coef, cs, ci, kw0, kw1;
};

// The ray of a pixel with the forward's samples, opacities and keyhole window.
__device__ __forceinline__ VgRay vg_ray(const VolGradArgs& a, const BatchView& bv, int x, int y) {
  const VolGeom& g = a.b.g;
  const Ray r = form_ray(g, bv.v, a.b.step_len, x, y);
  const float j = ray_offset(a.b.m.jitter, x, y);
  const long long pi = bv.pix_off + (long long)y * bv.v.W + x;
  const float I = a.img[pi];
  const float dLdI = a.dldi[pi];
  const float ds = ray_length(g, r.inc);
  VgRay q;
  q.p0c = V3<float>{(r.start.x + j * r.inc.x) + 0.5f, (r.start.y + j * r.inc.y) + 0.5f,
                    (r.start.z + j * r.inc.z) + 0.5f};
  q.inc = r.inc;
  q.n = step_count(r.num_steps - j);
  // the rays the precise forward march takes no samples of (drr_march)
  if (!samples_in_cells(g, q.p0c, q.inc, q.n)) q.n = 0;
  const int es = q.n - (int)ceilf(r.exclude_start), ee = q.n - (int)floorf(r.exclude_end);
  q.kw0 = (float)(q.n - es);
  q.kw1 = (float)(q.n - ee);
  q.ci = a.b.m.intercept * -ds;
  q.cs = a.b.m.slope * -ds;
  // d loss / d mu at a sample = (d loss / d L) * ds * slope, with dL/dI = -I for exp(-L)
  const float dLdL = (a.b.m.output == RVK_DRR_F32_EXP_NEG_L) ? -dLdI * I : dLdI;
  q.coef = dLdL * ds * a.b.m.slope;
  return q;
}

// The pixel of a thread in workgroup blk's tile: four 8x8 items.
__device__ __forceinline__ const BatchView& vg_pixel(const VolGradArgs& a, int blk, int& x, int& y) {
  const int2 vt = a.b.work[blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6)];
  const BatchView& bv = a.b.views[__builtin_amdgcn_readfirstlane(vt.x)];
  const int local = __builtin_amdgcn_readfirstlane(vt.y), macro = local >> 2, q = local & 3;
  const int lane = (int)(threadIdx.x & 63u);
  x = (macro % bv.tiles16_x) * 16 + (q & 1) * 8 + (lane & 7);
  y = (macro / bv.tiles16_x) * 16 + (q >> 1) * 8 + (lane >> 3);
  return bv;
}

// |coef| of a ray with samples; +inf if it is not finite (it poisons the call).
__device__ __forceinline__ float vg_magnitude(const VgRay& q) {
  return q.n > 0 ? (isfinite(q.coef) ? fabsf(q.coef) : __builtin_huge_valf()) : 0.0f;
}

__device__ __forceinline__ void vg_clear_slots(const VolGradArgs& a) {
  if (threadIdx.x < kVgSlots) a.slots[threadIdx.x * kVgSlotStride] = 0u;
}

// The largest m of a workgroup's threads, into one of the slots.
__device__ __forceinline__ void vg_collect(const VolGradArgs& a, float m) {
  __shared__ float s_m[4];
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((threadIdx.x & 63) == 0) s_m[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0)
    atomicMax(a.slots + (blockIdx.x % kVgSlots) * kVgSlotStride,
              __float_as_uint(fmaxf(fmaxf(s_m[0], s_m[1]), fmaxf(s_m[2], s_m[3]))));
}

// k = 30 - e for the largest |coef| = f 2^e (f in [0.5, 1)): every scaled
// contribution |coef w 2^k| (w <= 1) is below 2^30 and rounds into an int32.
__device__ __forceinline__ int vg_scale(const unsigned* slots) {
  float m = __uint_as_float(slots[(threadIdx.x & 63) * kVgSlotStride]);
  for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  int e = 0;
  if (m > 0.0f) frexpf(m, &e);
  return __builtin_amdgcn_readfirstlane(isfinite(m) ? 30 - e : kVgNonFinite);
}

__device__ __forceinline__ unsigned long long vg_fixed(float v) {
  return (unsigned long long)(long long)(int)__builtin_rintf(v);
}

// Launches on the frame; by tiles needs acc, by bricks rays.
int launch_volume_grad(const VolGradArgs& a, const rvk_volume* vol, int frame, hipStream_t s);
int launch_volume_grad_bricks(const VolGradArgs& a, const rvk_volume* vol, int frame, hipStream_t s);

}  // namespace rvk
