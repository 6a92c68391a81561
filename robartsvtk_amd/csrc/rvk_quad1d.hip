// rvk_quad1d.hip -- cast1d_kernel with four lanes per ray.
#include "rvk_quad.h"

namespace rvk {

// A sample's gradient is taken one step on, where the reference's march
// stands when it shades (cast1d_kernel).
template <typename CV, bool SKIP, bool GRAD>
__global__ __launch_bounds__(256) void quad1d_kernel(Cast1dArgs a) {
  extern __shared__ float lds[];
  const int n = a.n;
  uint32_t* s_bits = reinterpret_cast<uint32_t*>(lds + 5 * n);  // entries with opacity
  int x, y;
  lanes_pixel(xcd_deal(blockIdx.x, kQuadDealLog2), a.tiles_x, 2, x, y);
  const bool inside = x < a.v.W && y < a.v.H;
  QuadSetup q{};
  int kst = 0;
  if (inside) {
    q = quad_setup(a.g, a.v, a.step_len, a.jitter, x, y);
    kst = step_count(q.r.num_steps - q.j);
  }
  if (__syncthreads_or(kst > 0)) {  // the tables only where a ray needs them
    for (int i = threadIdx.x; i < 5 * n; i += 256) lds[i] = a.tables[i];
    for (int i = threadIdx.x; i < ((n + 63) & ~63); i += 256) {
      const unsigned long long live = __ballot(i < n && a.tables[i] > 0.0f);
      if ((i & 63) == 0) {
        s_bits[i >> 5] = (uint32_t)live;
        s_bits[(i >> 5) + 1] = (uint32_t)(live >> 32);
      }
    }
    __syncthreads();
  }
  if (!inside) return;
  const float *t_alpha = lds, *t_galpha = lds + n, *t_r = lds + 2 * n, *t_g = lds + 3 * n, *t_b = lds + 4 * n;
  const CV vol = cells_of<CV>(a.vol);
  const VolGeom& g = a.g;
  const V3<float> inc = q.r.inc;
  const float lo = a.p.intensity_low, mult = a.p.intensity_multiplier;
  const float rlen = ray_length(g, inc);
  const bool use_galpha = isfinite(a.p.gradient_multiplier);
  float u = 0.0f, al = 0.0f;
  const QuadSkip skip = quad_skip(g, a.m, q, kst, s_bits, n, lo, mult, true);
  const QuadRay o = quad_march<SKIP, false>(
      kst, a.term_T,
      [&](float t) -> uint32_t {
        const V3<float> c = sample_pos<true>(q.p0c, q.p0c, inc, t);
        u = mult * (trilinear(vol, g, c.x, c.y, c.z) - lo);
        al = tf1d_lookup(t_alpha, n, u);
        return al > 0.0f ? 1u : 4u;
      },
      [&](float t, float& alpha, float& r, float& gg, float& b) {
        float shd = a.p.ambient, shs = 0.0f;
        alpha = al;
        if (GRAD) {
          const V3<float> gr = sample_gradient(vol, g, sample_pos<true>(q.p0c, q.p0c, inc, t + 1.0f));
          const float gm = sqrtf(gr.x * gr.x + gr.y * gr.y + gr.z * gr.z);
          alpha *= use_galpha ? tf1d_lookup(t_galpha, n, a.p.gradient_multiplier * (gm - a.p.gradient_low)) : 1.0f;
          const float pl =
              satf(fabsf(gr.x * inc.x * g.sp[0] + gr.y * inc.y * g.sp[1] + gr.z * inc.z * g.sp[2]) / (gm * rlen));
          shd = a.p.ambient + a.p.diffuse * pl;
          shs = a.p.specular * powf(pl, a.p.specular_power);
        }
        r = satf(shd * tf1d_lookup(t_r, n, u) + shs);
        gg = satf(shd * tf1d_lookup(t_g, n, u) + shs);
        b = satf(shd * tf1d_lookup(t_b, n, u) + shs);
      },
      [&](float t, float tend, float inv) { return quad_run(a.m, skip, q, t, tend, inv); });
  quad_store(a, x, y, q.r, pack_rgba(satf(o.r), satf(o.g), satf(o.b), 1.0f - o.Tr), o.t);
}

int launch_quad_1d(const Cast1dArgs& a, const rvk_volume* vol, int frame, bool skip, bool grad, size_t lds, int nblk,
                   hipStream_t s) {
  lds += sizeof(uint32_t) * 2 * (size_t)((a.n + 63) / 64);
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    const dim3 grid(deal_grid(nblk * 4, kQuadDealLog2)), block(256);
    if (skip && grad) hipLaunchKernelGGL((quad1d_kernel<CV, true, true>), grid, block, lds, s, a);
    else if (skip) hipLaunchKernelGGL((quad1d_kernel<CV, true, false>), grid, block, lds, s, a);
    else if (grad) hipLaunchKernelGGL((quad1d_kernel<CV, false, true>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((quad1d_kernel<CV, false, false>), grid, block, lds, s, a);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

}  // namespace rvk
