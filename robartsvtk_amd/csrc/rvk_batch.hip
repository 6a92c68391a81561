// rvk_batch.hip -- batched multi-view DRR, NCC registration loss and the
// hand-written DRR adjoint (pose and volume gradients).
//
// No counterpart in the reference: it renders one view per Render() call and
// has no derivatives.  The forward march is the reference DRR caster
// (V/CUDA_vtkCudaDRRImageVolumeMapper_renderAlgo.cuh:11-117) shared with the
// single-view kernel through rvk_march.h.
//
// Work unit: an 8x8-pixel tile of one view, processed by one wave64.  Tiles
// are numbered view by view; inside a view, four consecutive tiles form a
// 16x16 block (same ray-offset phase as the single-view kernel).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <vector>

#include "rvk_lanes.h"
#include "rvk_volgrad.h"
#include "rvk_pose_math.h"

namespace rvk {

__device__ __forceinline__ void item_pixel(int tiles16_x, int local, int lane, int& x, int& y) {
  const int macro = local >> 2, q = local & 3;
  x = (macro % tiles16_x) * 16 + (q & 1) * 8 + (lane & 7);
  y = (macro / tiles16_x) * 16 + (q >> 1) * 8 + (lane >> 3);
}
// The forward kernels' wave tile (the autotuner's choice; the reductions
// keep the 8x8 mapping above, so their sums do not depend on it): the four
// items of a 16x16 block as 8x8 quadrants, 16x4 rows or 4x16 columns.
__device__ __forceinline__ void item_pixel_shaped(int shape, int tiles16_x, int local, int lane, int& x, int& y) {
  const int macro = local >> 2, q = local & 3;
  const int bx = (macro % tiles16_x) * 16, by = (macro / tiles16_x) * 16;
  if (shape == RVK_TILE_16X4) {
    x = bx + (lane & 15);
    y = by + q * 4 + (lane >> 4);
  } else if (shape == RVK_TILE_4X16) {
    x = bx + q * 4 + (lane & 3);
    y = by + (lane >> 2);
  } else {
    x = bx + (q & 1) * 8 + (lane & 7);
    y = by + (q >> 1) * 8 + (lane >> 3);
  }
}

// One pixel of one view.  With JAC the march also gathers trilinear gradients
// and the pixel's pose Jacobian dL/dpose_i = A . dstart_i + B . dinc_i is
// written next to the image (the registration step's single march).
template <typename CV, bool SKIP, bool PRECISE, bool JAC, bool TERM>
__device__ __forceinline__ void forward_item(const BatchArgs& a, int item, int lane) {
  // the forward writes only its own pixels, so it may take the tiles in any
  // order (the reductions keep the view-major one)
  const int2 vt = a.work[item];
  const int v = __builtin_amdgcn_readfirstlane(vt.x);
  const BatchView& bv = a.views[v];
  int x, y;
  item_pixel_shaped(a.shape, bv.tiles16_x, __builtin_amdgcn_readfirstlane(vt.y), lane, x, y);
  if (x >= bv.v.W || y >= bv.v.H) return;
  const Ray r = form_ray(a.g, bv.v, a.step_len, x, y);
  const long long pi = bv.pix_off + (long long)y * bv.v.W + x;
  if (!JAC) {
    a.out[pi] = drr_march<CV, SKIP, PRECISE, false, true, true, TERM>(cells_of<CV>(a.vol), a.g, a.m, r, x, y);
    return;
  }
  const float ds = sqrtf(r.inc.x * r.inc.x * a.g.sp[0] * a.g.sp[0] + r.inc.y * r.inc.y * a.g.sp[1] * a.g.sp[1] +
                         r.inc.z * r.inc.z * a.g.sp[2] * a.g.sp[2]);
  V3<float> A{0, 0, 0}, B{0, 0, 0};
  PoseVisit visit{ray_offset(a.m.jitter, x, y), A, B};
  a.out[pi] = drr_march<CV, SKIP, true, true, true, true, TERM>(cells_of<CV>(a.vol), a.g, a.m, r, x, y, visit);
  const bool any = A.x != 0.0f || A.y != 0.0f || A.z != 0.0f || B.x != 0.0f || B.y != 0.0f || B.z != 0.0f;
  if (any) pose_sums(ds * a.m.slope, A, B);
#pragma unroll 1
  for (int i = 0; i < 6; ++i) {
    float jv = 0.0f;
    if (any) {
      const RayTangent tg = form_ray_tangent(a.g, bv.v, bv.dm + 16 * i, a.step_len, x, y);
      jv = A.x * tg.dstart.x + A.y * tg.dstart.y + A.z * tg.dstart.z + B.x * tg.dinc.x + B.y * tg.dinc.y +
           B.z * tg.dinc.z;
    }
    a.jac[i * a.total + pi] = jv;
  }
}

// One wave per tile; workgroups XCD-remapped so neighbouring tiles share an L2.
template <typename CV, bool SKIP, bool PRECISE, bool JAC, bool TERM>
__global__ __launch_bounds__(256) void batch_grid_kernel(BatchArgs a) {
  const int blk = a.deal ? xcd_deal(blockIdx.x, kDealLog2) : xcd_remap(blockIdx.x, gridDim.x);
  const int item = blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= a.n_items) return;
  forward_item<CV, SKIP, PRECISE, JAC, TERM>(a, item, threadIdx.x & 63);
}

// Persistent: the tile range is cut into kNumXcd contiguous queues.  A wave
// drains the queue of the XCD its workgroup was dispatched to (blockIdx mod
// kNumXcd under round-robin dispatch), then the others in turn; every queue
// is finite, so every wave reaches the end.
template <typename CV, bool SKIP, bool PRECISE, bool JAC, bool TERM>
__global__ __launch_bounds__(256) void batch_persistent_kernel(BatchArgs a) {
  const int lane = threadIdx.x & 63;
  const int home = blockIdx.x % kNumXcd;
  for (int r = 0; r < kNumXcd; ++r) {
    const int c = (home + r) % kNumXcd;
    const int begin = (int)((long long)a.n_items * c / kNumXcd);
    const int end = (int)((long long)a.n_items * (c + 1) / kNumXcd);
    while (true) {
      int w = 0;
      if (lane == 0) w = (int)atomicAdd(&a.queues[c], 1u);
      w = __builtin_amdgcn_readfirstlane(w);
      const int item = begin + w;
      if (item >= end) break;
      forward_item<CV, SKIP, PRECISE, JAC, TERM>(a, item, lane);
    }
  }
}

// Queue heads are cleared by a kernel (not a memset node) so the sequence can
// live in a replayed hipGraph.
__global__ void reset_queues_kernel(unsigned* q) {
  if (threadIdx.x < kNumXcd) q[threadIdx.x] = 0u;
}

// ---------------------------------------------------------------------------
// NCC per view, zero-mean (Pearson) or the reference's uncentred
// sum(I T) / (sqrt(sum I^2) sqrt(sum T^2))
// (ImageProcessing/vtkRobartsRegistration/vtkImageNormalizedCrossCorrelation.cxx:116-128,203-218).
// Per tile: raw moments in double; per view: combine.
struct NccArgs {
  const BatchView* views;
  const int* item_begin;
  int n_views, n_items;
  int centred;
  const float* img;
  const float* tgt;
  double* part;    // n_items x 5
  double* stats;   // n_views x 8: mean_I, mean_T, inv_sqrt(Saa*Sbb), ncc/Saa, ncc, n, valid
  float* loss;     // n_views
  float* grad_img; // optional packed dloss/dI
};

__global__ __launch_bounds__(256) void ncc_partial_kernel(NccArgs a) {
  const int item = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= a.n_items) return;
  const int lane = threadIdx.x & 63;
  const int v = __builtin_amdgcn_readfirstlane(find_view(a.item_begin, a.n_views, item));
  const BatchView& bv = a.views[v];
  int x, y;
  item_pixel(bv.tiles16_x, item - a.item_begin[v], lane, x, y);
  double s[5] = {0, 0, 0, 0, 0};
  if (x < bv.v.W && y < bv.v.H) {
    const long long i = bv.pix_off + (long long)y * bv.v.W + x;
    const double I = a.img[i], T = a.tgt[i];
    s[0] = I; s[1] = T; s[2] = I * I; s[3] = T * T; s[4] = I * T;
  }
#pragma unroll
  for (int k = 0; k < 5; ++k) s[k] = wave_sum(s[k]);
  if (lane == 0)
#pragma unroll
    for (int k = 0; k < 5; ++k) a.part[(long long)item * 5 + k] = s[k];
}

// One workgroup per view; a fixed reduction order keeps results reproducible.
__global__ __launch_bounds__(256) void ncc_view_kernel(NccArgs a) {
  const int v = blockIdx.x;
  __shared__ double red[5][256];
  double s[5] = {0, 0, 0, 0, 0};
  for (int it = a.item_begin[v] + threadIdx.x; it < a.item_begin[v + 1]; it += blockDim.x)
#pragma unroll
    for (int k = 0; k < 5; ++k) s[k] += a.part[(long long)it * 5 + k];
#pragma unroll
  for (int k = 0; k < 5; ++k) red[k][threadIdx.x] = s[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int k = 0; k < 5; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const double n = (double)a.views[v].v.W * (double)a.views[v].v.H;
    // the uncentred form is the centred one with both means taken as 0
    const double mi = a.centred ? red[0][0] / n : 0.0, mt = a.centred ? red[1][0] / n : 0.0;
    const double saa = red[2][0] - n * mi * mi, sbb = red[3][0] - n * mt * mt, sab = red[4][0] - n * mi * mt;
    const bool ok = saa > 0.0 && sbb > 0.0;
    const double inv = !ok ? 0.0 : a.centred ? 1.0 / sqrt(saa * sbb) : 1.0 / (sqrt(saa) * sqrt(sbb));
    const double ncc = ok ? sab * inv : 0.0;
    double* st = a.stats + 8 * v;
    st[0] = mi; st[1] = mt; st[2] = inv; st[3] = ok ? ncc / saa : 0.0; st[4] = ncc; st[5] = n; st[6] = ok;
    a.loss[v] = (float)(1.0 - ncc);
  }
}

__global__ __launch_bounds__(256) void ncc_grad_image_kernel(NccArgs a) {
  const int item = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= a.n_items) return;
  const int lane = threadIdx.x & 63;
  const int v = __builtin_amdgcn_readfirstlane(find_view(a.item_begin, a.n_views, item));
  const BatchView& bv = a.views[v];
  int x, y;
  item_pixel(bv.tiles16_x, item - a.item_begin[v], lane, x, y);
  if (x >= bv.v.W || y >= bv.v.H) return;
  const long long i = bv.pix_off + (long long)y * bv.v.W + x;
  a.grad_img[i] = dloss_dimage(a.stats + 8 * v, a.img[i], a.tgt[i]);
}

template <typename CV, bool SKIP, bool TERM>
__global__ __launch_bounds__(256) void adjoint_pose_kernel(AdjArgs a) {
  const int blk = a.b.deal ? xcd_deal(blockIdx.x, kDealLog2) : xcd_remap(blockIdx.x, gridDim.x);
  const int item = blk * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= a.b.n_items) return;
  const int lane = threadIdx.x & 63;
  const int2 vt = a.b.work[item];
  const int v = __builtin_amdgcn_readfirstlane(vt.x), local = __builtin_amdgcn_readfirstlane(vt.y);
  const BatchView& bv = a.b.views[v];
  int x, y;
  item_pixel(bv.tiles16_x, local, lane, x, y);
  float c[6] = {0, 0, 0, 0, 0, 0};
  if (x < bv.v.W && y < bv.v.H) {
    const VolGeom& g = a.b.g;
    const Ray r = form_ray(g, bv.v, a.b.step_len, x, y);
    const float ds = sqrtf(r.inc.x * r.inc.x * g.sp[0] * g.sp[0] + r.inc.y * r.inc.y * g.sp[1] * g.sp[1] +
                           r.inc.z * r.inc.z * g.sp[2] * g.sp[2]);
    V3<float> A{0, 0, 0}, B{0, 0, 0};
    const float jt = ray_offset(a.b.m.jitter, x, y);
    PoseVisit visit{jt, A, B};
    const float I = drr_march<CV, SKIP, true, true, true, true, TERM>(cells_of<CV>(a.b.vol), g, a.b.m, r, x, y, visit);
    const long long pi = bv.pix_off + (long long)y * bv.v.W + x;
    const float dLdI = dloss_at(a.dldi, a.stats, a.img, a.tgt, v, pi);
    // dI/dL = -I for exp(-L) output, 1 for L output
    const float coef = (a.b.m.output == RVK_DRR_F32_EXP_NEG_L) ? -dLdI * I : dLdI;
    if (coef != 0.0f && (A.x != 0.0f || A.y != 0.0f || A.z != 0.0f)) {
      pose_sums(ds * a.b.m.slope, A, B);
#pragma unroll 1
      for (int i = 0; i < 6; ++i) {
        const RayTangent tg = form_ray_tangent(g, bv.v, bv.dm + 16 * i, a.b.step_len, x, y);
        c[i] = coef * (A.x * tg.dstart.x + A.y * tg.dstart.y + A.z * tg.dstart.z + B.x * tg.dinc.x +
                       B.y * tg.dinc.y + B.z * tg.dinc.z);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) c[i] = wave_sumf(c[i]);
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < 6; ++i) a.part[((long long)a.b.item_begin[v] + local) * 6 + i] = c[i];
}

__global__ __launch_bounds__(256) void pose_reduce_kernel(const int* item_begin, const float* part, float* grad) {
  const int v = blockIdx.x;
  __shared__ double red[6][256];
  double s[6] = {0, 0, 0, 0, 0, 0};
  for (int it = item_begin[v] + threadIdx.x; it < item_begin[v + 1]; it += blockDim.x)
#pragma unroll
    for (int k = 0; k < 6; ++k) s[k] += part[(long long)it * 6 + k];
#pragma unroll
  for (int k = 0; k < 6; ++k) red[k][threadIdx.x] = s[k];
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w)
#pragma unroll
      for (int k = 0; k < 6; ++k) red[k][threadIdx.x] += red[k][threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x < 6) grad[6 * v + threadIdx.x] = (float)red[threadIdx.x][0];
}

// d loss / d pose from the stored per-pixel Jacobians (registration step).
struct JacGradArgs {
  const BatchView* views;
  const int* item_begin;
  int n_views, n_items;
  const float* img;
  const float* tgt;
  const float* jac;
  long long total;
  const double* stats;
  int output;
  float* part;
};

__global__ __launch_bounds__(256) void jac_grad_kernel(JacGradArgs a) {
  const int item = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (item >= a.n_items) return;
  const int lane = threadIdx.x & 63;
  const int v = __builtin_amdgcn_readfirstlane(find_view(a.item_begin, a.n_views, item));
  const BatchView& bv = a.views[v];
  int x, y;
  item_pixel(bv.tiles16_x, item - a.item_begin[v], lane, x, y);
  float c[6] = {0, 0, 0, 0, 0, 0};
  if (x < bv.v.W && y < bv.v.H) {
    const long long pi = bv.pix_off + (long long)y * bv.v.W + x;
    const float I = a.img[pi];
    const float dLdI = dloss_dimage(a.stats + 8 * v, I, a.tgt[pi]);
    const float coef = (a.output == RVK_DRR_F32_EXP_NEG_L) ? -dLdI * I : dLdI;
#pragma unroll
    for (int i = 0; i < 6; ++i) c[i] = coef * a.jac[i * a.total + pi];
  }
#pragma unroll
  for (int i = 0; i < 6; ++i) c[i] = wave_sumf(c[i]);
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < 6; ++i) a.part[(long long)item * 6 + i] = c[i];
}

// ---------------------------------------------------------------------------
// Device-resident poses: the registration loop's pose update and the views'
// matrices recomputed from the poses, so that one replayed graph holds the
// whole iteration (render, NCC, pose gradient, update).
struct PoseGeom {
  double pv[16];      // the view's camera transform P V (its aspect)
  double vox[16];     // voxel -> world
  double center[3];   // rotation centre (world mm)
  int slot;           // which pose drives this view
  int pad;
};

__global__ __launch_bounds__(64) void pose_views_kernel(const PoseGeom* __restrict__ geo, const double* poses,
                                                        BatchView* views, int n_views) {
  const int v = blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= n_views) return;
  const PoseGeom& G = geo[v];
  float m[16], dm[96];
  // a singular posed matrix (no rigid pose gives one) leaves the view as it was
  if (!pose::posed_view(G.pv, G.vox, poses + 6 * G.slot, G.center, m, dm)) return;
  BatchView& b = views[v];
  for (int k = 0; k < 16; ++k) b.v.m[k] = m[k];
  for (int k = 0; k < 96; ++k) b.dm[k] = dm[k];
  pose::baked_inverse(m, b.inv);
}

struct PoseUpdateArgs {
  rvk_pose_optimizer o;
  int n_views, n_slots;
};

// One workgroup.  The gradient of slot s's pose is the sum of d loss / d pose
// over the views it drives (one view each with per-view poses).  state holds
// the Adam moments m[n_slots*6], v[n_slots*6] and the step count.
__global__ __launch_bounds__(256) void pose_update_kernel(PoseUpdateArgs a, const PoseGeom* __restrict__ geo,
                                                          const float* __restrict__ grad, double* poses,
                                                          double* state) {
  const int nd = a.n_slots * 6;
  const double t = state[2 * nd] + 1.0;
  for (int i = threadIdx.x; i < nd; i += blockDim.x) {
    const int slot = i / 6, d = i % 6;
    double g = 0.0;
    for (int v = 0; v < a.n_views; ++v)
      if (geo[v].slot == slot) g += (double)grad[6 * v + d];
    const double lr = d < 3 ? a.o.lr_rotation : a.o.lr_translation;
    if (a.o.kind == RVK_OPT_ADAM) {
      const double b1 = a.o.beta1, b2 = a.o.beta2;
      const double m = b1 * state[i] + (1.0 - b1) * g;
      const double s = b2 * state[nd + i] + (1.0 - b2) * g * g;
      state[i] = m;
      state[nd + i] = s;
      const double mh = m / (1.0 - pow(b1, t)), sh = s / (1.0 - pow(b2, t));
      poses[i] -= lr * mh / (sqrt(sh) + (double)a.o.eps);
    } else {
      poses[i] -= lr * g;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) state[2 * nd] = t;
}

}  // namespace rvk

using namespace rvk;

struct rvk_drr_plan {
  rvk_ctx* ctx = nullptr;
  const rvk_volume* vol = nullptr;
  int frame = 0;
  int n_views = 0;
  rvk_march_params march{};
  rvk_drr_params drr{};
  std::vector<int> item_begin;     // host copy
  std::vector<long long> pix_off;  // n_views + 1
  int n_items = 0;
  BatchView* d_views = nullptr;
  int* d_item_begin = nullptr;
  unsigned* d_queues = nullptr;
  double* d_part = nullptr;   // n_items x 5
  double* d_stats = nullptr;  // n_views x 8
  float* d_pose_part = nullptr;  // n_items x 6
  unsigned long long* d_vg_acc = nullptr;  // per voxel, the volume gradient's sums, allocated by its first call
  RayRec* d_vg_rays = nullptr;             // or per pixel, its ray records, by the first call that goes by bricks
  unsigned* d_vg_slots = nullptr;          // its largest |coef|
  double vg_tiles = 0.0;  // 16x16-pixel tiles whose central ray meets the volume
  double vg_span = 0.0;   // distance in voxels between neighbouring ones, mean across and down
  float* d_jac = nullptr;        // 6 x total pixels, allocated with the plan when it has pose derivatives
  int schedule = RVK_SCHED_GRID;
  int waves_per_simd = 4;
  int shape = RVK_TILE_8X8;       // wave tile of the render
  int jac_shape = RVK_TILE_8X8;   // and of the registration forward
  // forward work orders: view-major, or grouped by the volume region the
  // tile's central ray crosses (all views' tiles of one region together, so
  // an XCD's L2 serves one region's cells to every view)
  int2* d_work[2] = {nullptr, nullptr};
  int order = RVK_ORDER_REGIONS, jac_order = RVK_ORDER_REGIONS;
  // the fused registration forward (pose Jacobians) has its own schedule:
  // its per-wave work differs enough that the best choice can differ
  int jac_schedule = RVK_SCHED_GRID;
  int jac_waves_per_simd = 4;
  int n_cu = 256;
  hipStream_t cap_stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  // buffers the graph was captured with
  float* g_out = nullptr;
  const float* g_tgt = nullptr;
  float* g_loss = nullptr;
  float* g_grad = nullptr;
  int g_enc = 0;  // cell encoding of the frame when the graph was captured
  unsigned g_gen = 0;  // and the volume's generation (its cells' addresses and layout)
  bool g_step = false;  // the graph is a registration step with the pose update
  int ncc_mode = RVK_NCC_CENTERED;
  // device-resident poses (rvk_drr_plan_set_poses)
  PoseGeom* d_pose_geom = nullptr;  // per view
  double* d_poses = nullptr;        // n_slots x 6
  double* d_opt_state = nullptr;    // 2 x n_slots x 6 moments + the step count
  int n_slots = 0;
  rvk_pose_optimizer opt{};
};

namespace {

int fill_views(rvk_drr_plan* p, const rvk_view* views, const float* dview, std::vector<BatchView>& hv) {
  hv.resize(p->n_views);
  for (int v = 0; v < p->n_views; ++v) {
    int rc = check_view(&views[v]);
    if (rc) return rc;
    if (v < (int)p->pix_off.size() - 1 && p->item_begin.size() == (size_t)p->n_views + 1) {
      const long long npix = (long long)views[v].width * views[v].height;
      if (npix != p->pix_off[v + 1] - p->pix_off[v])
        return fail(RVK_ERR_INVALID_ARGUMENT, "view %d changed size", v);
    }
    BatchView& b = hv[v];
    std::memset(&b, 0, sizeof(b));
    b.v = view_geom(&views[v]);
    if (dview) std::memcpy(b.dm, dview + 96 * (size_t)v, sizeof(b.dm));
    // inverse of the baked matrix (Gauss-Jordan, partial pivoting)
    pose::baked_inverse(views[v].view_to_voxels, b.inv);
    b.tiles16_x = (views[v].width + 15) / 16;
  }
  return RVK_OK;
}

// Work orders of the forward.  Order 0 is view-major.  Order 1 sorts the
// 16x16 tiles (4 work items each, kept together) by the volume region their
// central ray crosses: the midpoint of the ray's chord through the volume
// box, on a 32^3 grid of regions in Morton order (c4 forward: 39.2 ms
// view-major, 35.3 ms on a 16^3 grid, 35.0 ms on 32^3, 36.3 ms on 8^3);
// tiles whose ray misses the volume go last.  Ties keep view-major order.
static uint32_t morton3(uint32_t x, uint32_t y, uint32_t z) {
  uint32_t k = 0;
  for (int b = 0; b < 5; ++b) k |= (((x >> b) & 1u) << (3 * b)) | (((y >> b) & 1u) << (3 * b + 1)) | (((z >> b) & 1u) << (3 * b + 2));
  return k;
}

// Also counts the tiles whose central ray meets the volume, and measures how
// far apart neighbouring ones lie across and down the views (vg_by_tiles).
static void work_orders(rvk_drr_plan* p, const rvk_view* views, std::vector<int2>& by_view,
                        std::vector<int2>& by_region) {
  by_view.resize(p->n_items);
  for (int v = 0; v < p->n_views; ++v)
    for (int i = p->item_begin[v]; i < p->item_begin[v + 1]; ++i) by_view[i] = make_int2(v, i - p->item_begin[v]);
  const int* dims = p->vol->dims;
  const double cell = std::max(1.0, std::max(dims[0], std::max(dims[1], dims[2])) / 32.0);
  struct Tile { uint32_t key; int v, macro; };
  std::vector<Tile> tiles;
  tiles.reserve(p->n_items / 4);
  double hit = 0.0, apart[2] = {0.0, 0.0}, pairs[2] = {0.0, 0.0};
  std::vector<std::array<double, 3>> mid;  // the chords' midpoints (NaN: none), of a view's tiles so far
  for (int v = 0; v < p->n_views; ++v) {
    mid.clear();
    const rvk_view& vw = views[v];
    const float* m = vw.view_to_voxels;
    const int tx = (vw.width + 15) / 16, n_macro = (p->item_begin[v + 1] - p->item_begin[v]) / 4;
    for (int mc = 0; mc < n_macro; ++mc) {
      const double x = std::min(vw.width - 1, (mc % tx) * 16 + 8), y = std::min(vw.height - 1, (mc / tx) * 16 + 8);
      const double vx = vw.flipped ? x / vw.width : 1.0 - x / vw.width, vy = y / vw.height;
      double pt[2][3];
      bool ok = true;
      for (int d = 0; d < 2; ++d) {
        const double w = vx * m[12] + vy * m[13] + d * m[14] + m[15];
        ok = ok && w != 0.0;
        for (int a = 0; a < 3; ++a) pt[d][a] = (vx * m[4 * a] + vy * m[4 * a + 1] + d * m[4 * a + 2] + m[4 * a + 3]) / (ok ? w : 1.0);
      }
      // the line's chord through the box [0, n - 1]^3 (slab clipping)
      double t0 = -1e300, t1 = 1e300;
      for (int a = 0; a < 3 && ok; ++a) {
        const double dir = pt[1][a] - pt[0][a];
        if (dir == 0.0) {
          ok = pt[0][a] >= 0.0 && pt[0][a] <= dims[a] - 1;
        } else {
          double ta = (0.0 - pt[0][a]) / dir, tb = (dims[a] - 1 - pt[0][a]) / dir;
          if (ta > tb) std::swap(ta, tb);
          t0 = std::max(t0, ta);
          t1 = std::min(t1, tb);
        }
      }
      uint32_t key = 0xffffffffu;
      mid.push_back({std::nan(""), 0.0, 0.0});
      if (ok && t0 <= t1) {
        const double tm = 0.5 * (t0 + t1);
        std::array<double, 3>& c = mid.back();
        uint32_t g[3];
        for (int a = 0; a < 3; ++a) {
          c[a] = pt[0][a] + tm * (pt[1][a] - pt[0][a]);
          g[a] = (uint32_t)std::min(31.0, std::max(0.0, std::floor(c[a] / cell)));
        }
        key = morton3(g[0], g[1], g[2]);
        hit += 1.0;
        for (int k = 0; k < 2; ++k) {
          if (k == 0 ? mc % tx == 0 : mc < tx) continue;
          const std::array<double, 3>& o = mid[mc - (k == 0 ? 1 : tx)];
          if (std::isnan(o[0])) continue;
          apart[k] += std::hypot(c[0] - o[0], c[1] - o[1], c[2] - o[2]);
          pairs[k] += 1.0;
        }
      }
      tiles.push_back(Tile{key, v, mc});
    }
  }
  p->vg_tiles = hit;
  p->vg_span = pairs[0] > 0.0 && pairs[1] > 0.0 ? std::sqrt(apart[0] / pairs[0] * (apart[1] / pairs[1])) : 1e30;
  std::stable_sort(tiles.begin(), tiles.end(), [](const Tile& a, const Tile& b) { return a.key < b.key; });
  by_region.resize(p->n_items);
  size_t i = 0;
  for (const Tile& tl : tiles)
    for (int q = 0; q < 4; ++q) by_region[i++] = make_int2(tl.v, 4 * tl.macro + q);
}

static int upload_work_orders(rvk_drr_plan* p, const rvk_view* views) {
  std::vector<int2> o[2];
  work_orders(p, views, o[0], o[1]);
  for (int k = 0; k < 2; ++k) {
    if (!p->d_work[k]) RVK_HIP(hipMalloc((void**)&p->d_work[k], sizeof(int2) * (size_t)p->n_items));
    RVK_HIP(hipMemcpy(p->d_work[k], o[k].data(), sizeof(int2) * (size_t)p->n_items, hipMemcpyHostToDevice));
  }
  return RVK_OK;
}

// The order the marches take the tiles in: view by view in a band per XCD, or by
// region (a new plan's) with the tiles dealt to the XCDs in runs of 8.  The
// regions cluster what the views share, and the deal evens out what the runs
// leave each XCD to do (us, forward / pose adjoint): 64 poses of a 512x512x400
// CT 25100 / 35250 view by view in bands, 21310 / 31790 so, 4 poses 2996 / 3443
// and 1706 / 2436; 16 x 512^2 half a circle around a 256^3 f32 volume
// 1683 / 1809 and 1590 / 1741.  Dealing the view-major order is slower there
// (2500 / 2800: the XCDs then share no view's cells).
void use_order(const rvk_drr_plan* p, BatchArgs& a, int order) {
  const bool regions = order == RVK_ORDER_REGIONS;
  a.work = p->d_work[regions ? 1 : 0];
  a.deal = regions;
}

BatchArgs batch_args(const rvk_drr_plan* p, float* out) {
  BatchArgs a;
  a.g = vol_geom(p->vol);
  a.m.intercept = p->drr.ct_intercept;
  a.m.slope = p->drr.ct_slope;
  a.m.offset = p->drr.ct_offset;
  a.m.output = p->drr.output;
  a.m.ranges = p->vol->ranges[p->frame];
  a.m.rbx = p->vol->nrb[0];
  a.m.rby = p->vol->nrb[1];
  a.m.groups = p->vol->range_groups(p->frame);
  a.m.rgx = p->vol->nrg(0);
  a.m.rgy = p->vol->nrg(1);
  a.m.ref_term = p->drr.ref_termination;
  a.m.jitter = p->march.jitter;
  a.step_len = min_spacing(p->vol) * p->march.step_scale;
  a.vol = p->vol->frames[p->frame];
  a.views = p->d_views;
  a.item_begin = p->d_item_begin;
  a.n_views = p->n_views;
  a.n_items = p->n_items;
  a.out = out;
  a.jac = p->d_jac;
  a.total = p->pix_off[p->n_views];
  a.queues = p->d_queues;
  a.shape = p->shape;
  use_order(p, a, p->order);
  return a;
}

// Whether the volume adjoint goes by ray tiles (rvk_volgrad.hip) or by voxel
// bricks (rvk_volbrick.hip): by tiles where these fill the device (6 workgroups
// on each of 256 CUs; or more of them than half the bricks, which fill it no
// better) and their rays are close enough for some layers of the box they
// share in LDS.  Tiles / bricks, us, f32: 16384 tiles 7.7 voxels apart in 256^3
// 4050 / 7860; 5184 at 15 1494 / 2315; 2704 at 21 1632 / 1375, in 200^3 at 17
// 850 / 1007; 1225 at 7.7 in 256^3 499 / 536; 625 at 10.7 455 / 398; 169 at 21
// 614 / 257; 784 at 39 3196 / 655; 64 at 63 1038 / 255; 1296 at 47 in 400^3
// 10320 / 2056, 2500 at 17 2156 / 2264; 324 at 7.6 in 64^3 82 / 117, 81 at 7.5
// 75 / 40; 658 at 16 in 400x64x64 494 / 165.
bool vg_by_tiles(const rvk_drr_plan* p) {
  const int* n = p->vol->dims;
  double bricks = 1.0;
  for (int a = 0; a < 3; ++a) bricks *= (n[a] + kVgEdge - 1) / kVgEdge;
  return p->vg_span <= 18.0 && p->vg_tiles >= std::min(1000.0, 0.5 * bricks);
}

// log2 of the lanes per ray of the plan's forward (grad: with Jacobians).  A
// march that may terminate takes one.
int plan_lanes(const rvk_drr_plan* p, bool grad) {
  if (p->drr.ref_termination) return 0;
  return batch_lanes(p->vol, p->pix_off[p->n_views], min_spacing(p->vol) * p->march.step_scale, grad);
}

int launch_forward(rvk_drr_plan* p, float* out, hipStream_t s, bool jac = false) {
  BatchArgs a = batch_args(p, out);
  a.shape = jac ? p->jac_shape : p->shape;
  use_order(p, a, jac ? p->jac_order : p->order);
  const bool skip = p->march.skip_rule != 0, pr = p->march.precise != 0;
  const bool persistent = (jac ? p->jac_schedule : p->schedule) == RVK_SCHED_PERSISTENT;
  const long long groups = (long long)p->n_cu * (jac ? p->jac_waves_per_simd : p->waves_per_simd);
  if (persistent) hipLaunchKernelGGL(reset_queues_kernel, dim3(1), dim3(64), 0, s, p->d_queues);
  if (pr || jac)
    if (const int ls = plan_lanes(p, jac)) {
      const long long n = (((long long)p->n_items << ls) + 3) / 4;
      return launch_batch_lanes(a, p->vol, p->frame, skip, jac, ls, persistent ? (unsigned)std::min(groups, n) : 0u, s);
    }
  return dispatch_frame(p->vol, p->frame, [&](auto tag) {
    using CV = decltype(tag);
    if (persistent) {
      const unsigned blocks = (unsigned)std::min(groups, ((long long)p->n_items + 3) / 4);
#define RVK_LP(S, P, J)                                                                                     \
  do {                                                                                                      \
    if (p->drr.ref_termination)                                                                             \
      hipLaunchKernelGGL((batch_persistent_kernel<CV, S, P, J, true>), dim3(blocks), dim3(256), 0, s, a);    \
    else                                                                                                    \
      hipLaunchKernelGGL((batch_persistent_kernel<CV, S, P, J, false>), dim3(blocks), dim3(256), 0, s, a);   \
  } while (0)
      if (jac) { if (skip) RVK_LP(true, true, true); else RVK_LP(false, true, true); }
      else if (skip) { if (pr) RVK_LP(true, true, false); else RVK_LP(true, false, false); }
      else { if (pr) RVK_LP(false, true, false); else RVK_LP(false, false, false); }
#undef RVK_LP
    } else {
      const unsigned blocks = batch_grid(a, 0);
#define RVK_LG(S, P, J)                                                                                     \
  do {                                                                                                      \
    if (p->drr.ref_termination)                                                                             \
      hipLaunchKernelGGL((batch_grid_kernel<CV, S, P, J, true>), dim3(blocks), dim3(256), 0, s, a);          \
    else                                                                                                    \
      hipLaunchKernelGGL((batch_grid_kernel<CV, S, P, J, false>), dim3(blocks), dim3(256), 0, s, a);         \
  } while (0)
      if (jac) { if (skip) RVK_LG(true, true, true); else RVK_LG(false, true, true); }
      else if (skip) { if (pr) RVK_LG(true, true, false); else RVK_LG(true, false, false); }
      else { if (pr) RVK_LG(false, true, false); else RVK_LG(false, false, false); }
#undef RVK_LG
    }
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

NccArgs ncc_args(const rvk_drr_plan* p, const float* img, const float* tgt, float* loss, float* grad_img) {
  NccArgs n;
  n.views = p->d_views;
  n.item_begin = p->d_item_begin;
  n.n_views = p->n_views;
  n.n_items = p->n_items;
  n.img = img;
  n.tgt = tgt;
  n.part = p->d_part;
  n.stats = p->d_stats;
  n.loss = loss;
  n.grad_img = grad_img;
  n.centred = p->ncc_mode == RVK_NCC_CENTERED;
  return n;
}

// The registration step: one march per pixel producing the image and its
// pose Jacobian, then NCC (tile moments, per-view statistics) and the
// Jacobian-weighted reduction to d loss / d pose.
int launch_register(rvk_drr_plan* p, float* out, const float* tgt, float* loss, float* grad, hipStream_t s) {
  if (!p->d_jac) return fail(RVK_ERR_NOT_READY, "the plan was created without pose derivatives (dview)");
  int rc = launch_forward(p, out, s, true);
  if (rc) return rc;
  const int blocks = (p->n_items + 3) / 4;
  NccArgs n = ncc_args(p, out, tgt, loss, nullptr);
  hipLaunchKernelGGL(ncc_partial_kernel, dim3(blocks), dim3(256), 0, s, n);
  hipLaunchKernelGGL(ncc_view_kernel, dim3(p->n_views), dim3(256), 0, s, n);
  JacGradArgs ja;
  ja.views = p->d_views;
  ja.item_begin = p->d_item_begin;
  ja.n_views = p->n_views;
  ja.n_items = p->n_items;
  ja.img = out;
  ja.tgt = tgt;
  ja.jac = p->d_jac;
  ja.total = p->pix_off[p->n_views];
  ja.stats = p->d_stats;
  ja.output = p->drr.output;
  ja.part = p->d_pose_part;
  hipLaunchKernelGGL(jac_grad_kernel, dim3(blocks), dim3(256), 0, s, ja);
  hipLaunchKernelGGL(pose_reduce_kernel, dim3(p->n_views), dim3(256), 0, s, p->d_item_begin, p->d_pose_part, grad);
  RVK_HIP(hipGetLastError());
  return RVK_OK;
}

// A captured graph holds the frame's cell pointer, encoding and layout as
// they were at capture: replayed only while all three are unchanged.
bool graph_current(const rvk_drr_plan* p) {
  return p->exec && p->g_enc == p->vol->enc[p->frame] && p->g_gen == p->vol->generation;
}

void drop_graph(rvk_drr_plan* p) {
  if (p->exec) hipGraphExecDestroy(p->exec);
  if (p->graph) hipGraphDestroy(p->graph);
  p->exec = nullptr;
  p->graph = nullptr;
  p->g_out = nullptr;
  p->g_tgt = nullptr;
  p->g_loss = nullptr;
  p->g_grad = nullptr;
  p->g_step = false;
}

// The pose update and the views' matrices from the new poses.
int launch_pose_update(rvk_drr_plan* p, const float* grad, hipStream_t s) {
  PoseUpdateArgs a;
  a.o = p->opt;
  a.n_views = p->n_views;
  a.n_slots = p->n_slots;
  hipLaunchKernelGGL(pose_update_kernel, dim3(1), dim3(256), 0, s, a, p->d_pose_geom, grad, p->d_poses,
                     p->d_opt_state);
  hipLaunchKernelGGL(pose_views_kernel, dim3((p->n_views + 63) / 64), dim3(64), 0, s, p->d_pose_geom, p->d_poses,
                     p->d_views, p->n_views);
  RVK_HIP(hipGetLastError());
  return RVK_OK;
}

int launch_step(rvk_drr_plan* p, float* out, const float* tgt, float* loss, float* grad, hipStream_t s) {
  int rc = launch_register(p, out, tgt, loss, grad, s);
  if (rc) return rc;
  return launch_pose_update(p, grad, s);
}

}  // namespace

extern "C" {

int rvk_drr_plan_create(rvk_ctx* ctx, const rvk_volume* vol, int frame, int n_views, const rvk_view* views,
                        const float* dview, const rvk_march_params* march, const rvk_drr_params* drr,
                        rvk_drr_plan** out) {
  if (!ctx || !views || !march || !drr || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *out = nullptr;
  int rc = check_frame(vol, frame);
  if (rc) return rc;
  if (n_views < 1 || n_views > 65536) return fail(RVK_ERR_INVALID_ARGUMENT, "n_views %d out of range", n_views);
  if (drr->output != RVK_DRR_F32_EXP_NEG_L && drr->output != RVK_DRR_F32_L)
    return fail(RVK_ERR_UNSUPPORTED, "batched DRR renders the float output modes only");
  if (!(march->step_scale > 0.0f) || !std::isfinite(march->step_scale))
    return fail(RVK_ERR_INVALID_ARGUMENT, "step_scale must be positive and finite");
  RVK_HIP(hipSetDevice(ctx->device));
  rvk_drr_plan* p = new rvk_drr_plan();
  p->ctx = ctx;
  p->vol = vol;
  p->frame = frame;
  p->n_views = n_views;
  p->march = *march;
  p->drr = *drr;
  p->item_begin.assign(n_views + 1, 0);
  p->pix_off.assign(n_views + 1, 0);
  long long items = 0;
  for (int v = 0; v < n_views; ++v) {
    p->item_begin[v] = (int)items;
    p->pix_off[v] = (v ? p->pix_off[v - 1] + (long long)views[v - 1].width * views[v - 1].height : 0);
    const long long t = 4LL * ((views[v].width + 15) / 16) * ((views[v].height + 15) / 16);
    items += t;
  }
  p->pix_off[n_views] = p->pix_off[n_views - 1] + (long long)views[n_views - 1].width * views[n_views - 1].height;
  if (items > (1LL << 30)) { delete p; return fail(RVK_ERR_INVALID_ARGUMENT, "too many pixels in one plan"); }
  p->item_begin[n_views] = (int)items;
  p->n_items = (int)items;
  std::vector<BatchView> hv;
  std::vector<long long> keep = p->pix_off;
  p->pix_off.clear();  // no size check on creation
  rc = fill_views(p, views, dview, hv);
  p->pix_off = keep;
  if (rc) { delete p; return rc; }
  for (int v = 0; v < n_views; ++v) hv[v].pix_off = p->pix_off[v];
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, ctx->device) == hipSuccess) p->n_cu = prop.multiProcessorCount;
  auto alloc = [&](void** d, size_t bytes) { return hipMalloc(d, bytes); };
  hipError_t e = alloc((void**)&p->d_views, sizeof(BatchView) * n_views);
  if (e == hipSuccess) e = alloc((void**)&p->d_item_begin, sizeof(int) * (n_views + 1));
  if (e == hipSuccess) e = alloc((void**)&p->d_queues, sizeof(unsigned) * kNumXcd);
  if (e == hipSuccess) e = alloc((void**)&p->d_part, sizeof(double) * 5 * (size_t)p->n_items);
  if (e == hipSuccess) e = alloc((void**)&p->d_stats, sizeof(double) * 8 * (size_t)n_views);
  if (e == hipSuccess) e = alloc((void**)&p->d_pose_part, sizeof(float) * 6 * (size_t)p->n_items);
  if (e == hipSuccess && dview) e = alloc((void**)&p->d_jac, sizeof(float) * 6 * (size_t)p->pix_off[n_views]);
  if (e == hipSuccess) e = hipMemcpy(p->d_views, hv.data(), sizeof(BatchView) * n_views, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(p->d_item_begin, p->item_begin.data(), sizeof(int) * (n_views + 1), hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&p->cap_stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    rvk_drr_plan_destroy(p);
    return hip_fail(e, "plan allocation");
  }
  rc = upload_work_orders(p, views);
  if (rc) {
    rvk_drr_plan_destroy(p);
    return rc;
  }
  *out = p;
  return RVK_OK;
}

int rvk_drr_plan_destroy(rvk_drr_plan* p) {
  if (!p) return RVK_OK;
  hipSetDevice(p->ctx->device);
  hipStreamSynchronize(p->ctx->stream);
  drop_graph(p);
  if (p->cap_stream) hipStreamDestroy(p->cap_stream);
  hipFree(p->d_views);
  hipFree(p->d_item_begin);
  hipFree(p->d_work[0]);
  hipFree(p->d_work[1]);
  hipFree(p->d_queues);
  hipFree(p->d_part);
  hipFree(p->d_stats);
  hipFree(p->d_pose_part);
  if (p->d_vg_acc) hipFree(p->d_vg_acc);
  if (p->d_vg_rays) hipFree(p->d_vg_rays);
  if (p->d_vg_slots) hipFree(p->d_vg_slots);
  if (p->d_jac) hipFree(p->d_jac);
  if (p->d_pose_geom) hipFree(p->d_pose_geom);
  if (p->d_poses) hipFree(p->d_poses);
  if (p->d_opt_state) hipFree(p->d_opt_state);
  delete p;
  return RVK_OK;
}

int rvk_drr_plan_update_views(rvk_drr_plan* p, const rvk_view* views, const float* dview) {
  if (!p || !views) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (p->d_jac && !dview) return fail(RVK_ERR_INVALID_ARGUMENT, "this plan carries pose derivatives: pass dview");
  std::vector<BatchView> hv;
  int rc = fill_views(p, views, dview, hv);
  if (rc) return rc;
  for (int v = 0; v < p->n_views; ++v) hv[v].pix_off = p->pix_off[v];
  RVK_HIP(hipSetDevice(p->ctx->device));
  RVK_HIP(hipMemcpyAsync(p->d_views, hv.data(), sizeof(BatchView) * p->n_views, hipMemcpyHostToDevice,
                         p->ctx->stream));
  RVK_HIP(hipStreamSynchronize(p->ctx->stream));
  // new views, new regions (a captured graph reads the arrays, not their contents)
  return upload_work_orders(p, views);
}

int rvk_drr_plan_offsets(const rvk_drr_plan* p, int64_t* offsets) {
  if (!p || !offsets) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  for (int v = 0; v <= p->n_views; ++v) offsets[v] = p->pix_off[v];
  return RVK_OK;
}

int rvk_drr_plan_set_schedule(rvk_drr_plan* p, int schedule, int wps) {
  if (!p) return fail(RVK_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (schedule != RVK_SCHED_GRID && schedule != RVK_SCHED_PERSISTENT)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown schedule %d", schedule);
  if (wps < 1 || wps > 8) return fail(RVK_ERR_INVALID_ARGUMENT, "waves_per_simd must be within 1..8");
  if (schedule != p->schedule || wps != p->waves_per_simd || schedule != p->jac_schedule ||
      wps != p->jac_waves_per_simd)
    drop_graph(p);
  p->schedule = p->jac_schedule = schedule;
  p->waves_per_simd = p->jac_waves_per_simd = wps;
  return RVK_OK;
}

int rvk_drr_plan_get_schedule(const rvk_drr_plan* p, int* schedule, int* wps) {
  if (!p) return fail(RVK_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (schedule) *schedule = p->schedule;
  if (wps) *wps = p->waves_per_simd;
  return RVK_OK;
}

int rvk_drr_plan_autotune(rvk_drr_plan* p, float* out, int reps, float* best_ms) {
  if (!p || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  reps = std::max(1, std::min(reps, 100));
  RVK_HIP(hipSetDevice(p->ctx->device));
  drop_graph(p);
  // schedule x waves per SIMD x wave tile x work order
  const int cand[][2] = {{RVK_SCHED_GRID, 4}, {RVK_SCHED_PERSISTENT, 2}, {RVK_SCHED_PERSISTENT, 4},
                         {RVK_SCHED_PERSISTENT, 8}};
  const int shapes[] = {RVK_TILE_8X8, RVK_TILE_16X4, RVK_TILE_4X16};
  hipEvent_t e0, e1;
  RVK_HIP(hipEventCreate(&e0));
  RVK_HIP(hipEventCreate(&e1));
  int rc = RVK_OK;
  // the plain render, and for plans with pose derivatives the registration
  // forward, each keep their fastest candidate
  for (int jac = 0; jac < ((p->d_jac && p->march.precise) ? 2 : 1) && !rc; ++jac) {
    int& sched = jac ? p->jac_schedule : p->schedule;
    int& wps = jac ? p->jac_waves_per_simd : p->waves_per_simd;
    int& shape = jac ? p->jac_shape : p->shape;
    int& order = jac ? p->jac_order : p->order;
    float best = 1e30f;
    int bs = sched, bw = wps, bsh = shape, bo = order;
    for (int oi = 0; oi < 2 * 3 && !rc; ++oi) {
      const int o = oi / 3, sh = shapes[oi % 3];
      for (const auto& c : cand) {
        sched = c[0];
        wps = c[1];
        shape = sh;
        order = o;
        rc = launch_forward(p, out, p->ctx->stream, jac);  // warm-up
        if (rc) break;
        hipEventRecord(e0, p->ctx->stream);
        for (int r = 0; r < reps && !rc; ++r) rc = launch_forward(p, out, p->ctx->stream, jac);
        hipEventRecord(e1, p->ctx->stream);
        hipEventSynchronize(e1);
        float ms = 0.0f;
        hipEventElapsedTime(&ms, e0, e1);
        ms /= reps;
        if (ms < best) { best = ms; bs = c[0]; bw = c[1]; bsh = sh; bo = o; }
      }
    }
    sched = bs;
    wps = bw;
    shape = bsh;
    order = bo;
    if (!jac && best_ms) *best_ms = best;
  }
  hipEventDestroy(e0);
  hipEventDestroy(e1);
  return rc;
}

int rvk_drr_plan_autotune_layout(rvk_drr_plan* p, rvk_volume* vol, float* out, int reps, float* best_ms,
                                 int* layout) {
  if (!p || !vol || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (vol != p->vol) return fail(RVK_ERR_INVALID_ARGUMENT, "vol is not the volume the plan renders");
  int rc = RVK_OK;
  struct Choice {
    int layout = -1, sched, wps, shape, order, jsched, jwps, jshape, jorder;
    float ms = 1e30f;
  } best;
  for (const int l : {RVK_CELLS_PLAIN, RVK_CELLS_BRICK4, RVK_CELLS_PAIR8}) {
    // a layout the volume does not fit (its address limits, or the device
    // memory for a second copy of its cells) is skipped; the volume keeps
    // its cells then
    if (rvk_volume_relayout(vol, l) != RVK_OK) continue;
    float ms = 0.0f;
    rc = rvk_drr_plan_autotune(p, out, reps, &ms);
    if (rc) return rc;
    if (ms < best.ms) {
      best.layout = l;
      best.ms = ms;
      best.sched = p->schedule;
      best.wps = p->waves_per_simd;
      best.shape = p->shape;
      best.order = p->order;
      best.jsched = p->jac_schedule;
      best.jwps = p->jac_waves_per_simd;
      best.jshape = p->jac_shape;
      best.jorder = p->jac_order;
    }
  }
  if (best.layout < 0) return fail(RVK_ERR_INVALID_ARGUMENT, "no cell layout fits the volume");
  rc = rvk_volume_relayout(vol, best.layout);
  if (rc) return rc;
  drop_graph(p);
  p->schedule = best.sched;
  p->waves_per_simd = best.wps;
  p->shape = best.shape;
  p->order = best.order;
  p->jac_schedule = best.jsched;
  p->jac_waves_per_simd = best.jwps;
  p->jac_shape = best.jshape;
  p->jac_order = best.jorder;
  if (best_ms) *best_ms = best.ms;
  if (layout) *layout = best.layout;
  return RVK_OK;
}

int rvk_drr_plan_set_work_order(rvk_drr_plan* p, int order) {
  if (!p) return fail(RVK_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (order != RVK_ORDER_VIEWS && order != RVK_ORDER_REGIONS)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown work order %d", order);
  if (order != p->order || order != p->jac_order) drop_graph(p);
  p->order = p->jac_order = order;
  return RVK_OK;
}

int rvk_drr_plan_get_work_order(const rvk_drr_plan* p, int* order) {
  if (!p || !order) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *order = p->order;
  return RVK_OK;
}

int rvk_drr_plan_set_tile_shape(rvk_drr_plan* p, int shape) {
  if (!p) return fail(RVK_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (shape != RVK_TILE_8X8 && shape != RVK_TILE_16X4 && shape != RVK_TILE_4X16)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown tile shape %d", shape);
  if (shape != p->shape || shape != p->jac_shape) drop_graph(p);
  p->shape = p->jac_shape = shape;
  return RVK_OK;
}

int rvk_drr_plan_get_tile_shape(const rvk_drr_plan* p, int* shape) {
  if (!p || !shape) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *shape = p->shape;
  return RVK_OK;
}

int rvk_drr_plan_render(rvk_drr_plan* p, float* out) {
  if (!p || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  RVK_HIP(hipSetDevice(p->ctx->device));
  if (graph_current(p) && !p->g_step && p->g_out == out && !p->g_tgt) {
    RVK_HIP(hipGraphLaunch(p->exec, p->ctx->stream));
    return RVK_OK;
  }
  return launch_forward(p, out, p->ctx->stream);
}

int rvk_drr_plan_capture(rvk_drr_plan* p, float* out, const float* tgt, float* loss, float* grad) {
  if (!p) return fail(RVK_ERR_INVALID_ARGUMENT, "plan is NULL");
  RVK_HIP(hipSetDevice(p->ctx->device));
  drop_graph(p);
  if (!out) return RVK_OK;
  if (tgt && (!loss || !grad)) return fail(RVK_ERR_INVALID_ARGUMENT, "registration capture needs loss and grad");
  if (tgt && !p->march.precise) return fail(RVK_ERR_UNSUPPORTED, "the adjoint differentiates the precise march");
  // Capture on the plan's own stream (the context may use the legacy default
  // stream, which cannot be captured); replays go to the context stream.
  RVK_HIP(hipStreamSynchronize(p->ctx->stream));
  RVK_HIP(hipStreamBeginCapture(p->cap_stream, hipStreamCaptureModeThreadLocal));
  int rc = tgt ? launch_register(p, out, tgt, loss, grad, p->cap_stream) : launch_forward(p, out, p->cap_stream);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(p->cap_stream, &g);
  if (rc) { if (g) hipGraphDestroy(g); return rc; }
  if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
  p->graph = g;
  e = hipGraphInstantiate(&p->exec, g, nullptr, nullptr, 0);
  if (e != hipSuccess) { drop_graph(p); return hip_fail(e, "hipGraphInstantiate"); }
  p->g_out = out;
  p->g_tgt = tgt;
  p->g_loss = loss;
  p->g_grad = grad;
  p->g_enc = p->vol->enc[p->frame];
  p->g_gen = p->vol->generation;
  return RVK_OK;
}

int rvk_drr_plan_register(rvk_drr_plan* p, float* out, const float* tgt, float* loss, float* grad) {
  if (!p || !out || !tgt || !loss || !grad) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (!p->march.precise) return fail(RVK_ERR_UNSUPPORTED, "the adjoint differentiates the precise march");
  RVK_HIP(hipSetDevice(p->ctx->device));
  if (graph_current(p) && !p->g_step && p->g_out == out && p->g_tgt == tgt && p->g_loss == loss &&
      p->g_grad == grad) {
    RVK_HIP(hipGraphLaunch(p->exec, p->ctx->stream));
    return RVK_OK;
  }
  return launch_register(p, out, tgt, loss, grad, p->ctx->stream);
}

int rvk_drr_plan_ncc(rvk_drr_plan* p, const float* images, const float* tgt, float* loss, float* dldi) {
  if (!p || !images || !tgt || !loss) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  RVK_HIP(hipSetDevice(p->ctx->device));
  const int blocks = (p->n_items + 3) / 4;
  NccArgs n = ncc_args(p, images, tgt, loss, dldi);
  hipLaunchKernelGGL(ncc_partial_kernel, dim3(blocks), dim3(256), 0, p->ctx->stream, n);
  hipLaunchKernelGGL(ncc_view_kernel, dim3(p->n_views), dim3(256), 0, p->ctx->stream, n);
  if (dldi) hipLaunchKernelGGL(ncc_grad_image_kernel, dim3(blocks), dim3(256), 0, p->ctx->stream, n);
  RVK_HIP(hipGetLastError());
  return RVK_OK;
}

int rvk_drr_plan_backward(rvk_drr_plan* p, const float* images, const float* dldi, float* grad_pose,
                          float* grad_vol) {
  if (!p || !images || !dldi) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (!p->march.precise) return fail(RVK_ERR_UNSUPPORTED, "the adjoint differentiates the precise march");
  // the pose tangents come from the plan's dview (d_jac exists exactly then)
  if (grad_pose && !p->d_jac) return fail(RVK_ERR_NOT_READY, "the plan was created without pose derivatives (dview)");
  RVK_HIP(hipSetDevice(p->ctx->device));
  hipStream_t s = p->ctx->stream;
  if (grad_pose) {
    AdjArgs aa;
    aa.b = batch_args(p, const_cast<float*>(images));
    aa.img = images;
    aa.dldi = dldi;
    aa.stats = nullptr;
    aa.tgt = nullptr;
    aa.part = p->d_pose_part;
    int rc = dispatch_frame(p->vol, p->frame, [&](auto tag) {
      using CV = decltype(tag);
#define RVK_LA(S)                                                                                            \
  do {                                                                                                       \
    if (p->drr.ref_termination)                                                                              \
      hipLaunchKernelGGL((adjoint_pose_kernel<CV, S, true>), dim3(blocks), dim3(256), 0, s, aa);             \
    else                                                                                                     \
      hipLaunchKernelGGL((adjoint_pose_kernel<CV, S, false>), dim3(blocks), dim3(256), 0, s, aa);            \
  } while (0)
      const unsigned blocks = batch_grid(aa.b, 0);
      if (p->march.skip_rule) RVK_LA(true);
      else RVK_LA(false);
#undef RVK_LA
      return (int)RVK_OK;
    });
    if (rc) return rc;
    hipLaunchKernelGGL(pose_reduce_kernel, dim3(p->n_views), dim3(256), 0, s, p->d_item_begin, p->d_pose_part,
                       grad_pose);
    RVK_HIP(hipGetLastError());
  }
  if (grad_vol) {
    if (p->march.skip_rule || p->drr.ref_termination)
      return fail(RVK_ERR_UNSUPPORTED, "the volume gradient needs the plain march (no skip rule, no termination)");
    // each buffer on its own, set only once allocated: after a failed
    // allocation the next call allocates what is still missing
    auto need = [](void* have, size_t bytes, void** out) -> hipError_t {
      if (have) return hipSuccess;
      void* q = nullptr;
      const hipError_t e = hipMalloc(&q, bytes);
      if (e == hipSuccess) *out = q;
      return e;
    };
    const int* d = p->vol->dims;
    RVK_HIP(need(p->d_vg_slots, sizeof(unsigned) * kVgSlots * kVgSlotStride, (void**)&p->d_vg_slots));
    bool tiles = vg_by_tiles(p);
    if (tiles) {
      const hipError_t e =
          need(p->d_vg_acc, sizeof(unsigned long long) * (size_t)d[0] * d[1] * d[2], (void**)&p->d_vg_acc);
      if (e != hipSuccess && e != hipErrorOutOfMemory) return hip_fail(e, "hipMalloc(volume gradient)");
      if (e != hipSuccess) (void)hipGetLastError();
      tiles = e == hipSuccess;  // a volume's sums that do not fit: the bricks need only the pixels' rays
    }
    if (!tiles)
      RVK_HIP(need(p->d_vg_rays, sizeof(RayRec) * (size_t)p->pix_off[p->n_views], (void**)&p->d_vg_rays));
    VolGradArgs va;
    va.b = batch_args(p, nullptr);
    va.img = images;
    va.dldi = dldi;
    va.slots = p->d_vg_slots;
    va.acc = p->d_vg_acc;
    va.rays = p->d_vg_rays;
    va.grad = grad_vol;
    const int rc = tiles ? launch_volume_grad(va, p->vol, p->frame, s)
                         : launch_volume_grad_bricks(va, p->vol, p->frame, s);
    if (rc) return rc;
  }
  return RVK_OK;
}

int rvk_drr_plan_set_ncc(rvk_drr_plan* p, int mode) {
  if (!p) return fail(RVK_ERR_INVALID_ARGUMENT, "plan is NULL");
  if (mode != RVK_NCC_CENTERED && mode != RVK_NCC_UNCENTERED)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown NCC mode %d", mode);
  if (mode != p->ncc_mode) drop_graph(p);
  p->ncc_mode = mode;
  return RVK_OK;
}

int rvk_drr_plan_set_poses(rvk_drr_plan* p, const rvk_camera* cameras, const double center[3], const double origin[3],
                           const double* poses, const rvk_pose_optimizer* opt) {
  if (!p || !cameras || !center || !poses || !opt) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (!p->d_jac) return fail(RVK_ERR_NOT_READY, "the plan was created without pose derivatives (dview)");
  if (!p->march.precise) return fail(RVK_ERR_UNSUPPORTED, "the adjoint differentiates the precise march");
  if (opt->kind != RVK_OPT_GD && opt->kind != RVK_OPT_ADAM)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown optimizer kind %d", opt->kind);
  if (!std::isfinite(opt->lr_rotation) || !std::isfinite(opt->lr_translation) || opt->lr_rotation < 0.0f ||
      opt->lr_translation < 0.0f)
    return fail(RVK_ERR_INVALID_ARGUMENT, "learning rates must be finite and >= 0");
  if (opt->kind == RVK_OPT_ADAM && !(opt->beta1 >= 0.0f && opt->beta1 < 1.0f && opt->beta2 >= 0.0f &&
                                     opt->beta2 < 1.0f && opt->eps > 0.0f))
    return fail(RVK_ERR_INVALID_ARGUMENT, "Adam needs beta1, beta2 in [0, 1) and eps > 0");
  const int n_slots = opt->shared_pose ? 1 : p->n_views;
  const double zero[3] = {0.0, 0.0, 0.0};
  std::vector<PoseGeom> geo(p->n_views);
  std::vector<BatchView> hv(p->n_views);
  RVK_HIP(hipSetDevice(p->ctx->device));
  RVK_HIP(hipStreamSynchronize(p->ctx->stream));
  RVK_HIP(hipMemcpy(hv.data(), p->d_views, sizeof(BatchView) * p->n_views, hipMemcpyDeviceToHost));
  for (int v = 0; v < p->n_views; ++v) {
    PoseGeom& g = geo[v];
    std::memset(&g, 0, sizeof(g));
    const double aspect = (double)hv[v].v.W / (double)hv[v].v.H;
    if (camera_pv(&cameras[v], aspect, g.pv)) return fail(RVK_ERR_INVALID_ARGUMENT, "camera %d is invalid", v);
    voxels_matrix(origin ? origin : zero, p->vol->spacing, g.vox);
    for (int a = 0; a < 3; ++a) g.center[a] = center[a];
    g.slot = opt->shared_pose ? 0 : v;
    float m[16];
    if (!pose::posed_view(g.pv, g.vox, poses + 6 * g.slot, g.center, m, nullptr))
      return fail(RVK_ERR_INVALID_ARGUMENT, "view %d: singular posed matrix", v);
  }
  if (n_slots != p->n_slots) {
    if (p->d_poses) hipFree(p->d_poses);
    if (p->d_opt_state) hipFree(p->d_opt_state);
    p->d_poses = nullptr;
    p->d_opt_state = nullptr;
    p->n_slots = 0;
    // both or neither: the plan never holds poses without their optimiser state
    void* dp = nullptr;
    void* ds = nullptr;
    hipError_t e = hipMalloc(&dp, sizeof(double) * 6 * n_slots);
    if (e == hipSuccess) e = hipMalloc(&ds, sizeof(double) * (12 * (size_t)n_slots + 1));
    if (e != hipSuccess) {
      if (dp) hipFree(dp);
      return hip_fail(e, "hipMalloc(device poses)");
    }
    p->d_poses = (double*)dp;
    p->d_opt_state = (double*)ds;
    p->n_slots = n_slots;
  }
  if (!p->d_pose_geom) {
    void* q = nullptr;
    RVK_HIP(hipMalloc(&q, sizeof(PoseGeom) * p->n_views));
    p->d_pose_geom = (PoseGeom*)q;
  }
  drop_graph(p);
  p->opt = *opt;
  const std::vector<double> state(12 * (size_t)n_slots + 1, 0.0);
  RVK_HIP(hipMemcpy(p->d_pose_geom, geo.data(), sizeof(PoseGeom) * p->n_views, hipMemcpyHostToDevice));
  RVK_HIP(hipMemcpy(p->d_poses, poses, sizeof(double) * 6 * n_slots, hipMemcpyHostToDevice));
  RVK_HIP(hipMemcpy(p->d_opt_state, state.data(), sizeof(double) * state.size(), hipMemcpyHostToDevice));
  hipLaunchKernelGGL(pose_views_kernel, dim3((p->n_views + 63) / 64), dim3(64), 0, p->ctx->stream, p->d_pose_geom,
                     p->d_poses, p->d_views, p->n_views);
  RVK_HIP(hipGetLastError());
  RVK_HIP(hipStreamSynchronize(p->ctx->stream));
  return RVK_OK;
}

int rvk_drr_plan_get_poses(rvk_drr_plan* p, double* poses) {
  if (!p || !poses) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (!p->d_poses) return fail(RVK_ERR_NOT_READY, "the plan has no device poses (rvk_drr_plan_set_poses)");
  RVK_HIP(hipSetDevice(p->ctx->device));
  RVK_HIP(hipMemcpyAsync(poses, p->d_poses, sizeof(double) * 6 * p->n_slots, hipMemcpyDeviceToHost, p->ctx->stream));
  RVK_HIP(hipStreamSynchronize(p->ctx->stream));
  return RVK_OK;
}

int rvk_drr_plan_step(rvk_drr_plan* p, float* out, const float* tgt, float* loss, float* grad) {
  if (!p || !out || !tgt || !loss || !grad) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (!p->d_poses) return fail(RVK_ERR_NOT_READY, "the plan has no device poses (rvk_drr_plan_set_poses)");
  RVK_HIP(hipSetDevice(p->ctx->device));
  if (graph_current(p) && p->g_step && p->g_out == out && p->g_tgt == tgt && p->g_loss == loss &&
      p->g_grad == grad) {
    RVK_HIP(hipGraphLaunch(p->exec, p->ctx->stream));
    return RVK_OK;
  }
  return launch_step(p, out, tgt, loss, grad, p->ctx->stream);
}

int rvk_drr_plan_capture_step(rvk_drr_plan* p, float* out, const float* tgt, float* loss, float* grad) {
  if (!p || !out || !tgt || !loss || !grad) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (!p->d_poses) return fail(RVK_ERR_NOT_READY, "the plan has no device poses (rvk_drr_plan_set_poses)");
  RVK_HIP(hipSetDevice(p->ctx->device));
  drop_graph(p);
  RVK_HIP(hipStreamSynchronize(p->ctx->stream));
  RVK_HIP(hipStreamBeginCapture(p->cap_stream, hipStreamCaptureModeThreadLocal));
  int rc = launch_step(p, out, tgt, loss, grad, p->cap_stream);
  hipGraph_t g = nullptr;
  hipError_t e = hipStreamEndCapture(p->cap_stream, &g);
  if (rc) { if (g) hipGraphDestroy(g); return rc; }
  if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
  p->graph = g;
  e = hipGraphInstantiate(&p->exec, g, nullptr, nullptr, 0);
  if (e != hipSuccess) { drop_graph(p); return hip_fail(e, "hipGraphInstantiate"); }
  p->g_out = out;
  p->g_tgt = tgt;
  p->g_loss = loss;
  p->g_grad = grad;
  p->g_enc = p->vol->enc[p->frame];
  p->g_gen = p->vol->generation;
  p->g_step = true;
  return RVK_OK;
}

}  // extern "C"
