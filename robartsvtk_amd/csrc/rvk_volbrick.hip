// rvk_volbrick.hip -- the volume adjoint (rvk_volgrad.hip) brick by brick: the
// same contributions into the same fixed-point sums, so the same bits.
//
// Per pixel a ray record; then one workgroup owns an 8^3-voxel brick and
// marches every ray that can meet the cells its voxels weigh in, over that
// stretch only, and adds each accumulated sample's 8 corner contributions to
// the brick's sums in LDS.  Every sample is gathered 1.4 times over and 55 % of
// the lanes are kept, but the launch is as wide as the volume, however few and
// far apart the rays are, and it needs 48 bytes per pixel instead of 8 per
// voxel.
#include "rvk_volgrad.h"

namespace rvk {

__global__ __launch_bounds__(kVgSlots) void vg_clear_slots_kernel(VolGradArgs a) { vg_clear_slots(a); }

__global__ __launch_bounds__(256) void vg_record_kernel(VolGradArgs a) {
  int x, y;
  const BatchView& bv = vg_pixel(a, blockIdx.x, x, y);
  float m = 0.0f;
  if (x < bv.v.W && y < bv.v.H) {
    const VgRay q = vg_ray(a, bv, x, y);
    a.rays[bv.pix_off + (long long)y * bv.v.W + x] =
        RayRec{q.p0c.x, q.p0c.y, q.p0c.z, q.coef, q.inc.x, q.inc.y, q.inc.z, q.n, q.cs, q.ci, q.kw0, q.kw1};
    m = vg_magnitude(q);
  }
  vg_collect(a, m);
}

// The LDS cube holds voxels [8b - 2, 8b + 9] per axis.  A sample's lower
// corner index, clamped into [0, 10], is the true one whenever either corner
// is a brick voxel; otherwise both land in the halo, which is dropped, except
// that at the volume's faces the clamped edge voxels are folded in (voxel -1
// holds voxel 0, voxels n and n + 1 hold voxel n - 1, as the edge cells do).
constexpr int kVgL = kVgEdge + 4;
constexpr int kVgCube = kVgL * kVgL * kVgL;
constexpr int kVgViews = 64;  // view boxes held in LDS at a time

__device__ __forceinline__ void vg_add(unsigned long long* s, float v) {
  __hip_atomic_fetch_add(s, vg_fixed(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

template <typename CV>
__global__ __launch_bounds__(256) void vg_brick_kernel(VolGradArgs a) {
  __shared__ unsigned long long s_acc[kVgCube];
  __shared__ int s_box[kVgViews][3];
  __shared__ long long s_pre[kVgViews + 1];  // box ray counts can pass 2^31 (whole images)
  const VolGeom& g = a.b.g;
  const int nb[3] = {(g.n[0] + kVgEdge - 1) / kVgEdge, (g.n[1] + kVgEdge - 1) / kVgEdge,
                     (g.n[2] + kVgEdge - 1) / kVgEdge};
  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int bi[3] = {bid % nb[0], (bid / nb[0]) % nb[1], bid / (nb[0] * nb[1])};
  const int o[3] = {bi[0] * kVgEdge, bi[1] * kVgEdge, bi[2] * kVgEdge};
  const int tid = threadIdx.x;
  const int k = vg_scale(a.slots);
  const CV vol = cells_of<CV>(a.b.vol);
  // With mu = value (slope > 0, intercept 0) a sample is accumulated exactly
  // when its trilinear value is > 0; the samples weighing in this brick
  // interpolate voxels [8b - 1, 8b + 8], so if all of those are <= 0 none is.
  // (A voxel is read as the trilinear value at its own cell corner, weights
  // exactly 0, which is its value in every cell encoding.)
  bool live = true;
  if (a.b.m.intercept == 0.0f && a.b.m.slope > 0.0f) {
    float mx = -1.0f;
    for (int e = tid; e < 1000; e += 256) {
      const int xi = min(max(o[0] - 1 + e % 10, 0), g.n[0] - 1);
      const int yi = min(max(o[1] - 1 + (e / 10) % 10, 0), g.n[1] - 1);
      const int zi = min(max(o[2] - 1 + e / 100, 0), g.n[2] - 1);
      mx = fmaxf(mx, trilinear<false>(vol, g, (float)(xi + 1), (float)(yi + 1), (float)(zi + 1)));
    }
    live = __syncthreads_or(mx > 0.0f);
  }
  if (live && k != kVgNonFinite) {
    for (int e = tid; e < kVgCube; e += 256) s_acc[e] = 0ull;
    // the cells whose samples weigh in the brick's voxels: (8b, 8b + 9) per
    // axis, reaching below c = 1 and above c = n at the faces
    float clo[3], chi[3];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      clo[ax] = bi[ax] == 0 ? -1.0f : (float)o[ax];
      chi[ax] = bi[ax] == nb[ax] - 1 ? (float)(g.n[ax] + 2) : (float)(o[ax] + kVgEdge + 1);
    }
    for (int v0 = 0; v0 < a.b.n_views; v0 += kVgViews) {
      const int nv = min(kVgViews, a.b.n_views - v0);
      __syncthreads();
      if (tid < nv) {
        // pixel box of the region's 8 corners (sample coordinates p = c -
        // 0.5), a pixel of margin beyond the rays that can meet it
        const BatchView& bv = a.b.views[v0 + tid];
        const int W = bv.v.W, H = bv.v.H;
        float xmin = 1e30f, xmax = -1e30f, ymin = 1e30f, ymax = -1e30f;
        bool behind = false;
        for (int c = 0; c < 8; ++c) {
          const float px = ((c & 1) ? chi[0] : clo[0]) - 0.5f, py = ((c & 2) ? chi[1] : clo[1]) - 0.5f;
          const float pz = ((c & 4) ? chi[2] : clo[2]) - 0.5f;
          const float* M = bv.inv;
          const float hx = M[0] * px + M[1] * py + M[2] * pz + M[3];
          const float hy = M[4] * px + M[5] * py + M[6] * pz + M[7];
          const float hw = M[12] * px + M[13] * py + M[14] * pz + M[15];
          if (!(hw > 0.0f)) { behind = true; break; }
          const float vx = hx / hw, vy = hy / hw;
          const float xp = bv.v.flipped ? vx * (float)W : (1.0f - vx) * (float)W;
          const float yp = vy * (float)H;
          xmin = fminf(xmin, xp); xmax = fmaxf(xmax, xp);
          ymin = fminf(ymin, yp); ymax = fmaxf(ymax, yp);
        }
        int x0 = 0, x1 = W - 1, y0 = 0, y1 = H - 1;
        if (!behind) {
          x0 = max(0, (int)floorf(xmin) - 1); x1 = min(W - 1, (int)ceilf(xmax) + 1);
          y0 = max(0, (int)floorf(ymin) - 1); y1 = min(H - 1, (int)ceilf(ymax) + 1);
        }
        const int w = max(0, x1 - x0 + 1), h = max(0, y1 - y0 + 1);
        s_box[tid][0] = x0;
        s_box[tid][1] = y0;
        s_box[tid][2] = w;
        s_pre[tid + 1] = (long long)w * h;
      }
      __syncthreads();
      if (tid == 0) {
        s_pre[0] = 0;
        for (int v = 0; v < nv; ++v) s_pre[v + 1] += s_pre[v];
      }
      __syncthreads();
      // the boxes' rays, view after view, one per thread
      const long long total = s_pre[nv];
      int cv = 0;
      for (long long r = tid; r < total; r += 256) {
        while (r >= s_pre[cv + 1]) ++cv;
        const int local = (int)(r - s_pre[cv]);
        const int bw = s_box[cv][2];
        const int ly = local / bw;
        const int px = s_box[cv][0] + (local - ly * bw), py = s_box[cv][1] + ly;
        const BatchView& bv = a.b.views[v0 + cv];
        const float4* rec = reinterpret_cast<const float4*>(a.rays + bv.pix_off);
        const long long q = 3 * ((long long)py * bv.v.W + px);
        const float4 A = rec[q], B = rec[q + 1], K = rec[q + 2];
        const int n = __float_as_int(B.w);
        if (n <= 0 || A.w == 0.0f) continue;
        // sample indices m with c0 + m inc inside the open region: the entry
        // and exit times from v_rcp_f32 reciprocals differ from the
        // quotients by a few ulp, far less than the one-sample margin each
        // side, and a sample outside adds only to the halo
        float tlo = 0.0f, thi = (float)(n - 1);
        const float p0[3] = {A.x, A.y, A.z}, in[3] = {B.x, B.y, B.z};
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          if (in[ax] != 0.0f) {
            const float rin = __builtin_amdgcn_rcpf(in[ax]);
            const float ta = (clo[ax] - p0[ax]) * rin, tb = (chi[ax] - p0[ax]) * rin;
            tlo = fmaxf(tlo, fminf(ta, tb));
            thi = fminf(thi, fmaxf(ta, tb));
          } else if (p0[ax] <= clo[ax] || p0[ax] >= chi[ax]) {
            thi = -1.0f;
          }
        }
        const int m0 = max(0, (int)floorf(tlo) - 1), m1 = min(n - 1, (int)ceilf(thi) + 1);
        const float coef = ldexpf(A.w, k);
        // each lane starts its stretch at its own sample (3 x its lane, mod
        // the length) and wraps round: a wave's rays enter the region
        // together, and marched in step they would add to the same voxels in
        // the same instructions (LDS address conflicts); the sum is the same
        // in any order
        const int cnt = m1 - m0 + 1;
        int mm = m0 + (cnt > 0 ? (int)(3 * (threadIdx.x & 63)) % cnt : 0);
        for (int i = 0; i < cnt; ++i, mm = (mm == m1) ? m0 : mm + 1) {
          const int m = mm;
          const float t = (float)m;
          // samples in the keyhole window are not accumulated by the forward
          if (t >= K.z && t < K.w) continue;
          const float qx = fmaf(t, B.x, A.x), qy = fmaf(t, B.y, A.y), qz = fmaf(t, B.z, A.z);
          // the forward's sample value (precise march: no clamp needed)
          const float alpha = fmaf(K.x, trilinear<false>(vol, g, qx, qy, qz), K.y);
          if (!(alpha < 0.0f)) continue;
          // corners ix - 1 (weight 1 - f) and ix (weight f) per axis
          const float fx = __builtin_amdgcn_fractf(qx), fy = __builtin_amdgcn_fractf(qy);
          const float fz = __builtin_amdgcn_fractf(qz);
          const int lx = min(max((int)qx - o[0] + 1, 0), kVgL - 2);
          const int ly2 = min(max((int)qy - o[1] + 1, 0), kVgL - 2);
          const int lz = min(max((int)qz - o[2] + 1, 0), kVgL - 2);
          const float cz0 = coef * (1.0f - fz), cz1 = coef * fz;
          const float c00 = cz0 * (1.0f - fy), c10 = cz0 * fy, c01 = cz1 * (1.0f - fy), c11 = cz1 * fy;
          const float wx0 = 1.0f - fx;
          unsigned long long* s = s_acc + (lz * kVgL + ly2) * kVgL + lx;
          vg_add(s, c00 * wx0);
          vg_add(s + 1, c00 * fx);
          vg_add(s + kVgL, c10 * wx0);
          vg_add(s + kVgL + 1, c10 * fx);
          vg_add(s + kVgL * kVgL, c01 * wx0);
          vg_add(s + kVgL * kVgL + 1, c01 * fx);
          vg_add(s + kVgL * kVgL + kVgL, c11 * wx0);
          vg_add(s + kVgL * kVgL + kVgL + 1, c11 * fx);
        }
      }
    }
    // fold the clamped edge voxels at the volume's faces, one axis at a time
    const int st[3] = {1, kVgL, kVgL * kVgL};
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
      __syncthreads();
      const int a1 = ax == 0 ? 1 : 0, a2 = ax == 2 ? 1 : 2;
      if (tid < kVgL * kVgL) {
        const int base = (tid % kVgL) * st[a1] + (tid / kVgL) * st[a2];
        if (bi[ax] == 0) s_acc[base + 2 * st[ax]] += s_acc[base + st[ax]];
        if (bi[ax] == nb[ax] - 1) {
          const int nl = g.n[ax] - o[ax] + 1;  // voxel n - 1
          s_acc[base + nl * st[ax]] += s_acc[base + (nl + 1) * st[ax]] + s_acc[base + (nl + 2) * st[ax]];
        }
      }
    }
    __syncthreads();
  }
  for (int e = tid; e < kVgEdge * kVgEdge * kVgEdge; e += 256) {
    const int lx = e % kVgEdge, ly = (e / kVgEdge) % kVgEdge, lz = e / (kVgEdge * kVgEdge);
    const int x = o[0] + lx, y = o[1] + ly, z = o[2] + lz;
    if (x >= g.n[0] || y >= g.n[1] || z >= g.n[2]) continue;
    float val = 0.0f;
    if (live) {
      val = k == kVgNonFinite ? __builtin_nanf("")
                              : (float)ldexp((double)(long long)s_acc[((lz + 2) * kVgL + ly + 2) * kVgL + lx + 2], -k);
    }
    a.grad[((long long)z * g.n[1] + y) * g.n[0] + x] = val;
  }
}

int launch_volume_grad_bricks(const VolGradArgs& a, const rvk_volume* vol, int frame, hipStream_t s) {
  const int* n = vol->dims;
  const unsigned bricks = (unsigned)(((n[0] + kVgEdge - 1) / kVgEdge) * ((n[1] + kVgEdge - 1) / kVgEdge) *
                                     ((n[2] + kVgEdge - 1) / kVgEdge));
  hipLaunchKernelGGL(vg_clear_slots_kernel, dim3(1), dim3(kVgSlots), 0, s, a);
  hipLaunchKernelGGL(vg_record_kernel, dim3((unsigned)(a.b.n_items / 4)), dim3(256), 0, s, a);
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    hipLaunchKernelGGL((vg_brick_kernel<CV>), dim3(bricks), dim3(256), 0, s, a);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

}  // namespace rvk
