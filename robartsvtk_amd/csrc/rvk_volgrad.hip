// rvk_volgrad.hip -- volume adjoint of the batched DRR (any voxel type, plain
// march).
//
// d loss / d v_ijk (v the stored voxel value, alpha = cs v + ci) =
// sum_views sum_pixels coef_p * sum_m [alpha(p_m) < 0] w_ijk(p_m), w the
// trilinear weight of voxel ijk at the sample and coef_p = d loss / d L_p *
// ds * slope.  The sums are 64-bit fixed point (contributions rounded to
// multiples of 2^-k, with 2^k set per call from the largest |coef| so that
// one stays below 2^30): integer sums do not depend on the order of the adds,
// so the result is the same on every call and LDS integer atomics are far
// cheaper than float ones.
//
// A workgroup takes a 16x16-pixel tile of one view and marches its rays
// through the volume slab by slab along the axis they mostly follow.  A slab's
// voxels that the tile can reach are a sheared box, which follows the tile
// from layer to layer, held in LDS; at the slab's end the sums go to the
// volume's by global atomics.  So each sample is gathered once, in the order
// of the rays, and passes over empty bricks as the forward does.  Bound by
// VALU issue (about 95 instructions a sample) and the wait for the gather.
// A tile whose rays lie far apart has room for few layers or none, and few
// tiles leave the device idle: such plans go brick by brick (rvk_volbrick.hip).
#include "rvk_volgrad.h"

#include <type_traits>

namespace rvk {

// Sums a workgroup holds (25 KiB: 6 workgroups per CU, as its registers allow)
// and the most layers of cells in a slab.  Volume gradient, us, with room for
// 1536 / 2560 / 3200 / 3840 / 5120 sums: 256^3 16 x 512^2 (a tile spans 8 voxels)
// 4180 / 4192 / 4179 / 4552 / 6273, 200^3 8 x 400^2 757 / 727 / 731 / 784 / 1028,
// 128x128x100 4 x 200^2 (20 voxels) 661 / 422 / 354 / 330 / 310.  Registers for 5, 7
// or 8 workgroups per CU 4572 / 4373 / 5168; slabs of 24 layers 4358, of 12 4192.
constexpr int kVgCap = 3200;
constexpr int kVgMaxLayers = 8;

__global__ __launch_bounds__(256) void vg_clear_kernel(VolGradArgs a, long long n) {
  const long long i = (long long)blockIdx.x * 512 + threadIdx.x;
  if (i < n) a.acc[i] = 0ull;
  if (i + 256 < n) a.acc[i + 256] = 0ull;
  if (blockIdx.x == 0) vg_clear_slots(a);
}

__global__ __launch_bounds__(256) void vg_coef_kernel(VolGradArgs a) {
  int x, y;
  const BatchView& bv = vg_pixel(a, blockIdx.x, x, y);
  float m = 0.0f;
  if (x < bv.v.W && y < bv.v.H) m = vg_magnitude(vg_ray(a, bv, x, y));
  vg_collect(a, m);
}

// The 8 corner contributions of the sample at q, corner voxel (i - 1 + dx,
// ...) of its cell i: add(dx, dy, dz, sum).
template <typename F>
__device__ __forceinline__ void vg_corners(const V3<float>& q, float coef, F&& add) {
  const float fx = __builtin_amdgcn_fractf(q.x), fy = __builtin_amdgcn_fractf(q.y), fz = __builtin_amdgcn_fractf(q.z);
  const float cz0 = coef * (1.0f - fz), cz1 = coef * fz;
  const float c00 = cz0 * (1.0f - fy), c10 = cz0 * fy, c01 = cz1 * (1.0f - fy), c11 = cz1 * fy;
  const float wx0 = 1.0f - fx;
  add(0, 0, 0, vg_fixed(c00 * wx0));
  add(1, 0, 0, vg_fixed(c00 * fx));
  add(0, 1, 0, vg_fixed(c10 * wx0));
  add(1, 1, 0, vg_fixed(c10 * fx));
  add(0, 0, 1, vg_fixed(c01 * wx0));
  add(1, 0, 1, vg_fixed(c01 * fx));
  add(0, 1, 1, vg_fixed(c11 * wx0));
  add(1, 1, 1, vg_fixed(c11 * fx));
}

// Adds to a voxel's sum; indices past a face are the face's voxel, as the edge
// cells hold them.
__device__ __forceinline__ void vg_global_add(const VolGradArgs& a, int x, int y, int z, unsigned long long v) {
  const VolGeom& g = a.b.g;
  const int i = min(max(x, 0), g.n[0] - 1), j = min(max(y, 0), g.n[1] - 1), k = min(max(z, 0), g.n[2] - 1);
  __hip_atomic_fetch_add(a.acc + ((size_t)k * g.n[1] + j) * g.n[0] + i, v, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ float vg_axis(const V3<float>& v, int d) { return d == 0 ? v.x : d == 1 ? v.y : v.z; }

template <typename CV>
__global__ __launch_bounds__(256, 6) void vg_scatter_kernel(VolGradArgs a) {
  __shared__ unsigned long long s_acc[kVgCap];
  __shared__ int s_base[kVgMaxLayers + 1], s_off1[kVgMaxLayers + 1], s_off2[kVgMaxLayers + 1];
  __shared__ float s_red[2][4][5];
  __shared__ int s_lead;
  __shared__ float s_slope[2];
  __shared__ int s_code;
  const int tid = threadIdx.x;
  const int blk = xcd_deal(blockIdx.x, kDealLog2);
  if (blk * 4 >= a.b.n_items) return;
  const int k = vg_scale(a.slots);
  if (k == kVgNonFinite) return;
  const VolGeom& g = a.b.g;
  const CV vol = cells_of<CV>(a.b.vol);
  int x, y;
  const BatchView& bv = vg_pixel(a, blk, x, y);
  VgRay r{};
  if (x < bv.v.W && y < bv.v.H) {
    r = vg_ray(a, bv, x, y);
    if (r.coef == 0.0f) r.n = 0;
  }
  // the axis most rays follow and their sense, from the first ray with samples
  if (tid == 0) s_lead = 256;
  for (int e = tid; e < kVgCap; e += 256) s_acc[e] = 0ull;
  __syncthreads();
  if (r.n > 0) atomicMin(&s_lead, tid);
  __syncthreads();
  if (s_lead == 256) return;
  if (tid == s_lead) {
    const float ax = fabsf(r.inc.x), ay = fabsf(r.inc.y), az = fabsf(r.inc.z);
    const int d = ax >= ay && ax >= az ? 0 : ay >= az ? 1 : 2;
    const float id = vg_axis(r.inc, d);
    s_code = 2 * d + (id < 0.0f ? 1 : 0);
    s_slope[0] = vg_axis(r.inc, d == 0 ? 1 : 0) / fabsf(id);
    s_slope[1] = vg_axis(r.inc, d == 2 ? 1 : 2) / fabsf(id);
  }
  __syncthreads();
  const int code = __builtin_amdgcn_readfirstlane(s_code), d = code >> 1;
  const bool down = code & 1;
  const int d1 = d == 0 ? 1 : 0, d2 = d == 2 ? 1 : 2;
  const float slope1 = s_slope[0], slope2 = s_slope[1];
  const float coef = ldexpf(r.coef, k);
  auto at = [&](float t) { return sample_pos<true>(r.p0c, r.p0c, r.inc, t); };
  // whether sample t counts (its alpha, as the forward has it)
  auto counts = [&](float t, const V3<float>& q) {
    // samples in the keyhole window are not accumulated by the forward
    if (bv.v.n_key && t >= r.kw0 && t < r.kw1) return false;
    return fmaf(r.cs, trilinear<false>(vol, g, q.x, q.y, q.z), r.ci) < 0.0f;
  };
  auto direct = [&](float t) {
    const V3<float> q = at(t);
    if (!counts(t, q)) return;
    vg_corners(q, coef, [&](int dx, int dy, int dz, unsigned long long v) {
      vg_global_add(a, (int)q.x - 1 + dx, (int)q.y - 1 + dy, (int)q.z - 1 + dz, v);
    });
  };
  // Layers count up along the march: cell index c on axis d is layer c, or -c
  // for rays that go down; a position is at depth p, or 1 - p, which for a
  // sample of layer L lies in [L, L + 1] either way.
  const float pd = vg_axis(r.p0c, d), id = vg_axis(r.inc, d);
  const float sid = down ? -id : id;
  float t = 0.0f, tend = (float)r.n;
  // a ray against the others' sense is scattered straight away
  if (r.n > 0 && !(sid > 0.0f)) {
    for (; t < tend; t += 1.0f) direct(t);
  }
  const RangeWalk w = range_walk(r.p0c, r.inc);
  const float rid = 1.0f / sid;
  auto depth = [&](const V3<float>& q) { return down ? 1.0f - vg_axis(q, d) : vg_axis(q, d); };
  auto layer = [&](float tt) {
    const int c = (int)fmaf(tt, id, pd);
    return down ? -c : c;
  };
  // The ray's next cnt samples into the box, whose rows are w1 long (axis d1
  // fastest: the corners of a sample then are four addresses and their
  // successors).  Each lane starts at its own sample (3 x its lane) and wraps
  // round: in step, a wave's rays would add to the same voxels in the same
  // instructions (LDS address conflicts).
  auto scatter = [&](auto axis, int cnt, int L0, int w1) {
    constexpr int D = decltype(axis)::value;
    const int top = kVgCap - 2 - w1;
    int mm = (int)(3 * (tid & 63)) % cnt;
    for (int i = 0; i < cnt; ++i, mm = mm + 1 == cnt ? 0 : mm + 1) {
      const float ts = t + (float)mm;
      const V3<float> q = at(ts);
      if (!counts(ts, q)) continue;
      const int cx = (int)q.x, cy = (int)q.y, cz = (int)q.z;
      const int cd = D == 0 ? cx : D == 1 ? cy : cz, c1 = D == 0 ? cy : cx, c2 = D == 2 ? cy : cz;
      const int j = (down ? -cd : cd) - L0;
      // the lower corner's address in the layers of the lower and upper voxel
      const int lat = (c1 - 1) + __mul24(c2 - 1, w1);
      const int b0 = s_base[j], b1 = s_base[j + 1];
      unsigned long long* const e0 = s_acc + min(max((down ? b1 : b0) + lat, 0), top);
      unsigned long long* const e1 = s_acc + min(max((down ? b0 : b1) + lat, 0), top);
      unsigned long long* const f0 = e0 + w1;
      unsigned long long* const f1 = e1 + w1;
      vg_corners(q, coef, [&](int dx, int dy, int dz, unsigned long long v) {
        const int hd = D == 0 ? dx : D == 1 ? dy : dz, h1 = D == 0 ? dy : dx, h2 = D == 2 ? dy : dz;
        __hip_atomic_fetch_add((hd ? (h2 ? f1 : e1) : (h2 ? f0 : e0)) + h1, v, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WORKGROUP);
      });
    }
  };
  int ref = 0;  // the first slab's first layer; the box's shear starts there
  for (int it = 0;; ++it) {
    // the ray's next sample that may count
    if (a.b.m.ranges) {
      while (t < tend) {
        const float m = empty_run(a.b.m, at(t), w, r.cs, r.ci, t, tend, 1.0f);
        if (!(m > 0.0f)) break;
        t += m;
      }
    }
    const bool active = t < tend;
    int L = 0x7fffff;
    float lo1 = 1e30f, hi1 = -1e30f, lo2 = 1e30f, hi2 = -1e30f;
    if (active) {
      L = layer(t);
      // sheared lateral positions at both ends of the longest stretch ahead
      const float te = fminf(tend - 1.0f, t + ceilf((float)(kVgMaxLayers + 1) * rid));
      const V3<float> q0 = at(t), q1 = at(te);
      const float u0 = depth(q0), u1 = depth(q1);
      const float a0 = vg_axis(q0, d1) - slope1 * u0, a1 = vg_axis(q1, d1) - slope1 * u1;
      const float b0 = vg_axis(q0, d2) - slope2 * u0, b1 = vg_axis(q1, d2) - slope2 * u1;
      lo1 = fminf(a0, a1); hi1 = fmaxf(a0, a1);
      lo2 = fminf(b0, b1); hi2 = fmaxf(b0, b1);
    }
    float fl = (float)L;  // layers are below 2^13: exact
    for (int o = 32; o > 0; o >>= 1) {
      fl = fminf(fl, __shfl_xor(fl, o, 64));
      lo1 = fminf(lo1, __shfl_xor(lo1, o, 64));
      hi1 = fmaxf(hi1, __shfl_xor(hi1, o, 64));
      lo2 = fminf(lo2, __shfl_xor(lo2, o, 64));
      hi2 = fmaxf(hi2, __shfl_xor(hi2, o, 64));
    }
    if ((tid & 63) == 0) {
      float* s = s_red[it & 1][tid >> 6];
      s[0] = fl; s[1] = lo1; s[2] = hi1; s[3] = lo2; s[4] = hi2;
    }
    __syncthreads();
    {
      const float(*s)[5] = s_red[it & 1];
      fl = fminf(fminf(s[0][0], s[1][0]), fminf(s[2][0], s[3][0]));
      lo1 = fminf(fminf(s[0][1], s[1][1]), fminf(s[2][1], s[3][1]));
      hi1 = fmaxf(fmaxf(s[0][2], s[1][2]), fmaxf(s[2][2], s[3][2]));
      lo2 = fminf(fminf(s[0][3], s[1][3]), fminf(s[2][3], s[3][3]));
      hi2 = fmaxf(fmaxf(s[0][4], s[1][4]), fmaxf(s[2][4], s[3][4]));
    }
    if (fl >= (float)0x7fffff) break;
    const int L0 = __builtin_amdgcn_readfirstlane((int)fl);
    if (it == 0) ref = L0;
    // Voxel V (a layer's lower or upper one) of a sample at depth u with
    // |u - V| <= 1: with off(V) = floor(slope (V - ref)) its lateral indices
    // less off lie within (s - |slope| - 2, s + |slope| + 1), s the sheared
    // position less slope * -ref; a margin for the rounding of both.
    const float eps = 0.02f;
    const float sh1 = slope1 * (float)ref, sh2 = slope2 * (float)ref;
    const int b1 = __builtin_amdgcn_readfirstlane((int)floorf(lo1 + sh1 - fabsf(slope1) - 2.0f - eps));
    const int b2 = __builtin_amdgcn_readfirstlane((int)floorf(lo2 + sh2 - fabsf(slope2) - 2.0f - eps));
    const int w1 = __builtin_amdgcn_readfirstlane((int)floorf(hi1 + sh1 + fabsf(slope1) + 1.0f + eps)) - b1 + 1;
    const int w2 = __builtin_amdgcn_readfirstlane((int)floorf(hi2 + sh2 + fabsf(slope2) + 1.0f + eps)) - b2 + 1;
    const bool fits = w1 <= kVgCap && w2 <= kVgCap && w1 * w2 * 2 <= kVgCap;
    const int T = fits ? min(kVgMaxLayers, kVgCap / (w1 * w2) - 1) : kVgMaxLayers;
    if (fits && tid <= T) {
      const float v = (float)(L0 + tid - ref);
      const int o1 = (int)floorf(slope1 * v), o2 = (int)floorf(slope2 * v);
      s_off1[tid] = o1;
      s_off2[tid] = o2;
      s_base[tid] = tid * w1 * w2 - (o1 + b1) - (o2 + b2) * w1;
    }
    __syncthreads();
    if (active && L < L0 + T) {
      // the ray's samples of the slab's layers: estimated, then exact
      const float rest = tend - t;
      float m = fminf(fmaxf(ceilf(((float)(L0 + T) - depth(at(t))) * rid), 1.0f), rest);
      while (m > 1.0f && layer(t + m - 1.0f) >= L0 + T) m -= 1.0f;
      while (m < rest && layer(t + m) < L0 + T) m += 1.0f;
      const int cnt = (int)m;
      if (fits) {
        if (d == 0) scatter(std::integral_constant<int, 0>{}, cnt, L0, w1);
        else if (d == 1) scatter(std::integral_constant<int, 1>{}, cnt, L0, w1);
        else scatter(std::integral_constant<int, 2>{}, cnt, L0, w1);
      } else {
        for (int i = 0; i < cnt; ++i) direct(t + (float)i);
      }
      t += m;
    }
    __syncthreads();
    if (!fits) continue;
    const int total = (T + 1) * w1 * w2;
    // x along the lanes: the axis of the layers when d is x
    const int r0 = d == 0 ? T + 1 : w1, r1 = d == 0 ? w1 : w2;
    const float i0 = 1.0f / (float)r0, i1r = 1.0f / (float)r1;
    for (int e = tid; e < total; e += 256) {
      // e / r0 and so on: e < 2^12, so half a unit keeps the floats exact
      const int g0 = (int)(((float)e + 0.5f) * i0), f0 = e - g0 * r0;
      const int f2 = (int)(((float)g0 + 0.5f) * i1r), f1 = g0 - f2 * r1;
      const int V = d == 0 ? f0 : f2, i1 = d == 0 ? f1 : f0, i2 = d == 0 ? f2 : f1;
      const int at_e = (V * w2 + i2) * w1 + i1;
      const unsigned long long v = s_acc[at_e];
      if (v == 0ull) continue;
      s_acc[at_e] = 0ull;
      // voxel on axis d: layer L's cell holds voxels L - 1 and L, layers
      // counted down -L - 1 and -L
      const int vd = down ? -(L0 + V) : L0 + V - 1;
      const int v1 = b1 + s_off1[V] + i1, v2 = b2 + s_off2[V] + i2;
      vg_global_add(a, d == 0 ? vd : v1, d == 0 ? v1 : d == 1 ? vd : v2, d == 2 ? vd : v2, v);
    }
    __syncthreads();
  }
}

// Sums to gradients, one workgroup per 8^3-voxel brick.  After a non-finite
// coefficient every voxel whose neighbourhood can contribute is NaN: with mu =
// value (slope > 0, intercept 0) a sample is accumulated exactly when its
// trilinear value is > 0, and the samples weighing in a brick interpolate
// voxels [8b - 1, 8b + 8], so a brick whose voxels there are all <= 0 stays 0.
// (A voxel is read as the trilinear value at its own cell corner, weights
// exactly 0, which is its value in every cell encoding.)
template <typename CV>
__global__ __launch_bounds__(256) void vg_finish_kernel(VolGradArgs a) {
  const VolGeom& g = a.b.g;
  const int nb[2] = {(g.n[0] + kVgEdge - 1) / kVgEdge, (g.n[1] + kVgEdge - 1) / kVgEdge};
  const int bid = blockIdx.x, tid = threadIdx.x;
  const int o[3] = {bid % nb[0] * kVgEdge, bid / nb[0] % nb[1] * kVgEdge, bid / (nb[0] * nb[1]) * kVgEdge};
  const int k = vg_scale(a.slots);
  bool live = true;
  if (k == kVgNonFinite && a.b.m.intercept == 0.0f && a.b.m.slope > 0.0f) {
    const CV vol = cells_of<CV>(a.b.vol);
    float mx = -1.0f;
    for (int e = tid; e < 1000; e += 256) {
      const int xi = min(max(o[0] - 1 + e % 10, 0), g.n[0] - 1);
      const int yi = min(max(o[1] - 1 + (e / 10) % 10, 0), g.n[1] - 1);
      const int zi = min(max(o[2] - 1 + e / 100, 0), g.n[2] - 1);
      mx = fmaxf(mx, trilinear<false>(vol, g, (float)(xi + 1), (float)(yi + 1), (float)(zi + 1)));
    }
    live = __syncthreads_or(mx > 0.0f);
  }
  for (int e = tid; e < kVgEdge * kVgEdge * kVgEdge; e += 256) {
    const int x = o[0] + e % kVgEdge, y = o[1] + e / kVgEdge % kVgEdge, z = o[2] + e / (kVgEdge * kVgEdge);
    if (x >= g.n[0] || y >= g.n[1] || z >= g.n[2]) continue;
    const size_t i = ((size_t)z * g.n[1] + y) * g.n[0] + x;
    a.grad[i] = k != kVgNonFinite ? (float)ldexp((double)(long long)a.acc[i], -k) : live ? __builtin_nanf("") : 0.0f;
  }
}

int launch_volume_grad(const VolGradArgs& a, const rvk_volume* vol, int frame, hipStream_t s) {
  const int* n = vol->dims;
  const long long voxels = (long long)n[0] * n[1] * n[2];
  const unsigned tiles = (unsigned)(a.b.n_items / 4);
  const unsigned bricks = (unsigned)(((n[0] + kVgEdge - 1) / kVgEdge) * ((n[1] + kVgEdge - 1) / kVgEdge) *
                                     ((n[2] + kVgEdge - 1) / kVgEdge));
  hipLaunchKernelGGL(vg_clear_kernel, dim3((unsigned)((voxels + 511) / 512)), dim3(256), 0, s, a, voxels);
  hipLaunchKernelGGL(vg_coef_kernel, dim3(tiles), dim3(256), 0, s, a);
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    hipLaunchKernelGGL((vg_scatter_kernel<CV>), dim3(deal_grid(tiles, kDealLog2)), dim3(256), 0, s, a);
    hipLaunchKernelGGL((vg_finish_kernel<CV>), dim3(bricks), dim3(256), 0, s, a);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

}  // namespace rvk
