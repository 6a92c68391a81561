// rvk_quad2d.hip -- cast2d_kernel (no keyhole) with four lanes per ray.
#include "rvk_quad.h"

namespace rvk {

template <typename CV, bool SKIP, bool GMAG>
__global__ __launch_bounds__(256) void quad2d_kernel(Cast2dArgs a) {
  extern __shared__ uint32_t s_lds[];
  const int cw = a.col_words, n = a.n;
  uint32_t* s_occ = s_lds + cw;
  const bool use_occ = a.occ != nullptr;
  int x, y;
  lanes_pixel(xcd_deal(blockIdx.x, kQuadDealLog2), a.tiles_x, 2, x, y);
  const bool inside = x < a.v.W && y < a.v.H;
  QuadSetup q{};
  int kst = 0;
  if (inside) {
    q = quad_setup(a.g, a.v, a.step_len, a.jitter, x, y);
    kst = step_count(q.r.num_steps - q.j);
  }
  if (__syncthreads_or(kst > 0)) {  // the bitmaps only where a ray needs them
    for (int i = threadIdx.x; i < cw; i += 256) s_lds[i] = a.col[i];
    if (use_occ)
      for (int i = threadIdx.x; i < a.occ_words; i += 256) s_occ[i] = a.occ[i];
    __syncthreads();
  }
  if (!inside) return;
  const CV vol = cells_of<CV>(a.vol);
  const VolGeom& g = a.g;
  const V3<float> inc = q.r.inc;
  const float lo = a.p.intensity_low, mult = a.p.intensity_multiplier;
  const float glo = a.p.gradient_low, gmult = a.p.gradient_multiplier, goff = a.p.gradient_offset;
  const float rlen = ray_length(g, inc);
  float4 c0{};
  V3<float> gr{};
  float gmag = 0.0f;
  int ti = 0;
  const QuadRay o = quad_march<SKIP, false>(
      kst, a.term_T,
      [&](float t) -> uint32_t {
        const V3<float> c = sample_pos<true>(q.p0c, q.p0c, inc, t);
        const float u = mult * (trilinear(vol, g, c.x, c.y, c.z) - lo);
        if (!tf2d_column_live(s_lds, tf2d_axis(n, u))) return 4u;
        float gm2;
        if (GMAG) {
          gmag = trilinear(Cells<uint8_t, CV::kLog2>{a.gradmag}, g, c.x, c.y, c.z) * a.gradmag_scale;
          gm2 = gmag * gmag;
        } else {
          gr = sample_gradient(vol, g, c);
          gm2 = gr.x * gr.x + gr.y * gr.y + gr.z * gr.z;
          gmag = sqrtf(gm2);
        }
        ti = tf2d_index(n, u, gmult * (log2f(gm2 + goff) + glo));
        if (use_occ) return (s_occ[ti >> 5] >> (ti & 31)) & 1u;
        return (GMAG ? a.lit[ti].x : a.cells[ti].alpha) > 0.0f ? 1u : 0u;
      },
      [&](float, float& alpha, float& r, float& gg, float& b) {
        if (GMAG) {
          c0 = a.lit[ti];
          alpha = c0.x; r = c0.y; gg = c0.z; b = c0.w;
        } else {
          c0 = *(const float4*)&a.cells[ti].alpha;
          lit_cell(a.cells + ti, c0, g, gr, gmag, inc, rlen, alpha, r, gg, b);
        }
      },
      [](float, float, float) { return 0.0f; });
  quad_store(a, x, y, q.r, pack_rgba(o.r, o.g, o.b, 1.0f - o.Tr), o.t);
}

int launch_quad_2d(const Cast2dArgs& a, const rvk_volume* vol, int frame, bool skip, bool gradmag, size_t lds,
                   int nblk, hipStream_t s) {
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    const dim3 grid(deal_grid(nblk * 4, kQuadDealLog2)), block(256);
    if (skip && gradmag) hipLaunchKernelGGL((quad2d_kernel<CV, true, true>), grid, block, lds, s, a);
    else if (skip) hipLaunchKernelGGL((quad2d_kernel<CV, true, false>), grid, block, lds, s, a);
    else if (gradmag) hipLaunchKernelGGL((quad2d_kernel<CV, false, true>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((quad2d_kernel<CV, false, false>), grid, block, lds, s, a);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

}  // namespace rvk
