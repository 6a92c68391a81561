// rvk_batch.h -- a plan's device-side views and arguments, and the pieces its
// forward and adjoint kernels share.
#pragma once
#include "rvk_internal.h"
#include "rvk_march.h"

namespace rvk {

struct BatchView {
  ViewGeom v;
  float dm[96];      // d(view_to_voxels)/d pose_i, i = 0..5 (baked, row major)
  float inv[16];     // inverse of view_to_voxels: voxel position -> (vx, vy, z, 1) * w
  long long pix_off; // first pixel of this view in the packed image buffer
  int tiles16_x;
  int pad;
};

struct BatchArgs {
  VolGeom g;
  DrrMarchArgs m;
  float step_len;
  const void* vol;
  const BatchView* views;
  const int* item_begin;  // n_views + 1 prefix sums of 8x8 tiles
  int n_views;
  int n_items;
  float* out;
  float* jac;             // 6 x total pixels (SoA) d L_p / d pose_i, or NULL
  long long total;        // pixels in the packed images
  unsigned* queues;       // kNumXcd work-queue heads (persistent schedule)
  int shape;              // wave tile of the forward kernels (RVK_TILE_*)
  int deal;               // work dealt to the XCDs in runs (xcd_deal), or one band each
  const int2* work;       // forward work order: (view, tile of the view) per work item
};

// Workgroups of 4 waves for the items' 2^ls parts.
inline unsigned batch_grid(const BatchArgs& a, int ls) {
  const long long n = (((long long)a.n_items << ls) + 3) / 4;
  return a.deal ? deal_grid(n, kDealLog2 + ls) : (unsigned)n;
}

// Accumulates S = sum grad mu and T = sum (j+t) grad mu over the accumulated
// samples of one ray; A = ds*slope*S and B = ds*slope*T (see the pose adjoint
// below) are formed once per ray by pose_sums().
struct PoseVisit {
  static constexpr bool kFlatRuns = true;  // a zero gradient adds nothing
  float j;
  V3<float>& S;
  V3<float>& T;
  __device__ __forceinline__ void operator()(const V3<float>&, float t, float, const V3<float>& gr) const {
    const float w = j + t;
    S.x += gr.x; S.y += gr.y; S.z += gr.z;
    T.x = fmaf(w, gr.x, T.x); T.y = fmaf(w, gr.y, T.y); T.z = fmaf(w, gr.z, T.z);
  }
};
// Scales the sums by ncs = ds*slope; called only for rays that accumulated
// a sample (a ray that misses the volume can have a non-finite ds).
__device__ __forceinline__ void pose_sums(float ncs, V3<float>& A, V3<float>& B) {
  A.x *= ncs; A.y *= ncs; A.z *= ncs;
  B.x *= ncs; B.y *= ncs; B.z *= ncs;
}

__device__ __forceinline__ int find_view(const int* __restrict__ ib, int n, int item) {
  int lo = 0, hi = n;  // ib[lo] <= item < ib[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (ib[mid] <= item) lo = mid;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}
__device__ __forceinline__ float wave_sumf(float v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// d loss / d I_p = -( (T_p - mean_T) / sqrt(Saa Sbb) - ncc (I_p - mean_I) / Saa )
__device__ __forceinline__ float dloss_dimage(const double* st, float I, float T) {
  return (float)(-((double)T - st[1]) * st[2] + st[3] * ((double)I - st[0]));
}

// ---------------------------------------------------------------------------
// Pose adjoint.  For one pixel, L = sum_m ds*mu(p_m) over accumulated samples
// p_m = start + (j + t_m) inc, so
//   dL/dpose_i = A . dstart_i + B . dinc_i,
//   A = sum_m ds*slope*grad mu(p_m),   B = sum_m (j + t_m) ds*slope*grad mu(p_m),
// with (dstart_i, dinc_i) the forward-mode tangent of the ray set-up along
// d(view_to_voxels)/d pose_i.  The ray is re-marched (PRECISE positions) with
// the forward's control flow; nothing is stored per sample.
struct AdjArgs {
  BatchArgs b;
  const float* img;   // rendered images (packed)
  const float* dldi;  // d loss / d image, or NULL: formed from the NCC state
  const double* stats;
  const float* tgt;
  float* part;  // n_items x 6
};

__device__ __forceinline__ float dloss_at(const float* dldi, const double* stats, const float* img, const float* tgt,
                                          int v, long long pi) {
  return dldi ? dldi[pi] : dloss_dimage(stats + 8 * v, img[pi], tgt[pi]);
}

}  // namespace rvk
