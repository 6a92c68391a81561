// rvk_quad_ext.hip -- inex_kernel and dual_kernel (no keyhole) with four lanes
// per ray.
#include <type_traits>

#include "rvk_quad.h"

namespace rvk {

template <typename CV, bool SKIP>
__global__ __launch_bounds__(256) void quad_inex_kernel(InExArgs a) {
  extern __shared__ uint32_t s_lds[];
  const int cw = a.col_words, n = a.n, w = a.occ_words;
  uint32_t* s_occ = s_lds + cw;
  const bool use_occ = a.occ != nullptr;
  int x, y;
  lanes_pixel(xcd_deal(blockIdx.x, kQuadDealLog2), a.tiles_x, 2, x, y);
  const bool inside = x < a.v.W && y < a.v.H;
  QuadSetup q{};
  int kst = 0;
  if (inside) {
    q = quad_setup(a.g, a.v, a.step_len, a.jitter, x, y);
    kst = step_count(q.r.num_steps);
  }
  if (__syncthreads_or(kst > 0)) {
    for (int i = threadIdx.x; i < cw; i += 256) s_lds[i] = a.col[i];
    if (use_occ)
      for (int i = threadIdx.x; i < 2 * w; i += 256) s_occ[i] = a.occ[i];
    __syncthreads();
  }
  if (!inside) return;
  const CV vol = cells_of<CV>(a.vol);
  const VolGeom& g = a.g;
  const V3<float> inc = q.r.inc;
  const float lo = a.p.intensity_low, mult = a.p.intensity_multiplier;
  const float glo = a.p.gradient_low, gmult = a.p.gradient_multiplier, goff = a.p.gradient_offset;
  const float rlen = ray_length(g, inc);
  const int es = kst - (int)ceilf(q.r.exclude_start);
  const int ee = kst - (int)floorf(q.r.exclude_end);
  V3<float> gr{};
  float gmag = 0.0f;
  int ti = 0;
  const QuadSkip skip = quad_skip(g, a.m, q, kst, s_lds, n, lo, mult, false);
  const QuadRay o = quad_march<SKIP, true>(
      kst, a.term_T,
      [&](float t) -> uint32_t {
        const V3<float> c = sample_pos<true>(q.p0c, q.p0c, inc, t);
        const float u = mult * (trilinear(vol, g, c.x, c.y, c.z) - lo);
        if (!tf2d_column_live(s_lds, tf2d_axis(n, u))) return 4u;
        gr = sample_gradient(vol, g, c);
        const float gm2 = gr.x * gr.x + gr.y * gr.y + gr.z * gr.z;
        gmag = sqrtf(gm2);
        ti = tf2d_index(n, u, gmult * (log2f(gm2 + goff) + glo));
        uint32_t fl;
        if (use_occ) {
          const uint32_t wi = (uint32_t)ti >> 5, b = (uint32_t)ti & 31u;
          fl = ((s_occ[wi] >> b) & 1u) | (((s_occ[w + wi] >> b) & 1u) << 1);
        } else {
          fl = a.flags[ti];
        }
        const int k = kst - 1 - (int)t;  // steps left when the sample is composited
        return (es >= k && ee <= k) ? fl & 1u : fl;
      },
      [&](float, float& alpha, float& r, float& gg, float& b) {
        const float4 c0 = *(const float4*)&a.cells[ti].alpha;
        lit_cell(a.cells + ti, c0, g, gr, gmag, inc, rlen, alpha, r, gg, b);
      },
      [&](float t, float tend, float inv) { return quad_run(a.m, skip, q, t, tend, inv); });
  const float A = (a.black_keyhole && o.special) ? 1.0f : 1.0f - o.Tr;
  // depth: (j + kst) - (kst - steps), as the one-lane caster forms it
  quad_store(a, x, y, q.r, pack_rgba(satf(o.r), satf(o.g), satf(o.b), satf(A)),
             (q.j + (float)kst) - (float)(kst - (int)o.t));
}

int launch_quad_inex(const InExArgs& a, const rvk_volume* vol, int frame, bool skip, size_t lds, int nblk,
                     hipStream_t s) {
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    const dim3 grid(deal_grid(nblk * 4, kQuadDealLog2)), block(256);
    if (skip) hipLaunchKernelGGL((quad_inex_kernel<CV, true>), grid, block, lds, s, a);
    else hipLaunchKernelGGL((quad_inex_kernel<CV, false>), grid, block, lds, s, a);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

template <typename CV, typename CV2, bool SKIP>
__global__ __launch_bounds__(256) void quad_dual_kernel(DualArgs a) {
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
    kst = dual_step_count(q.r.num_steps, q.j);
  }
  if (__syncthreads_or(kst > 0)) {
    for (int i = threadIdx.x; i < cw; i += 256) s_lds[i] = a.col[i];
    if (use_occ)
      for (int i = threadIdx.x; i < a.occ_words; i += 256) s_occ[i] = a.occ[i];
    __syncthreads();
  }
  if (!inside) return;
  const CV vol1 = cells_of<CV>(a.vol1);
  const CV2 vol2 = cells_of<CV2>(a.vol2);
  const VolGeom& g = a.g;
  const V3<float> inc = q.r.inc;
  const float lo1 = a.p.intensity1_low, m1 = a.p.intensity1_multiplier;
  const float lo2 = a.p.intensity2_low, m2 = a.p.intensity2_multiplier;
  const float rlen = ray_length(g, inc);
  int ti = 0;
  V3<float> c{};
  const QuadSkip skip = quad_skip(g, a.m, q, kst, s_lds, n, lo1, m1, false);
  const QuadRay o = quad_march<SKIP, false>(
      kst, a.term_T,
      [&](float t) -> uint32_t {
        c = sample_pos<true>(q.p0c, q.p0c, inc, t);
        const float u1 = m1 * (trilinear(vol1, g, c.x, c.y, c.z) - lo1);
        if (!tf2d_column_live(s_lds, tf2d_axis(n, u1))) return 4u;
        const float u2 = m2 * (trilinear(vol2, g, c.x, c.y, c.z) - lo2);
        ti = tf2d_index(n, u1, u2);
        if (use_occ) return (s_occ[ti >> 5] >> (ti & 31)) & 1u;
        return a.cells[ti].alpha > 0.0f ? 1u : 0u;
      },
      [&](float, float& alpha, float& r, float& gg, float& b) {
        // the gradient only shades: samples that composite alone need it
        const V3<float> gr = sample_gradient(vol1, g, c);
        const float gmag = sqrtf(gr.x * gr.x + gr.y * gr.y + gr.z * gr.z);
        const float4 c0 = *(const float4*)&a.cells[ti].alpha;
        lit_cell(a.cells + ti, c0, g, gr, gmag, inc, rlen, alpha, r, gg, b);
      },
      [&](float t, float tend, float inv) { return quad_run(a.m, skip, q, t, tend, inv); });
  quad_store(a, x, y, q.r, pack_rgba(o.r, o.g, o.b, 1.0f - o.Tr), o.t);
}

int launch_quad_dual(const DualArgs& a, const rvk_volume* vol1, const rvk_volume* vol2, int frame, bool skip,
                     size_t lds, int nblk, hipStream_t s) {
  return dispatch_frame<false>(vol1, frame, [&](auto tag1) {
    using CV = decltype(tag1);
    return dispatch_frame<false>(vol2, frame, [&](auto tag2) {
      using CV2 = decltype(tag2);
      if constexpr (std::is_same<typename CV::value_type, typename CV2::value_type>::value &&
                    CV::kLog2 == CV2::kLog2) {
        const dim3 grid(deal_grid(nblk * 4, kQuadDealLog2)), block(256);
        if (skip) hipLaunchKernelGGL((quad_dual_kernel<CV, CV2, true>), grid, block, lds, s, a);
        else hipLaunchKernelGGL((quad_dual_kernel<CV, CV2, false>), grid, block, lds, s, a);
        RVK_HIP(hipGetLastError());
        return (int)RVK_OK;
      } else {
        return fail(RVK_ERR_INVALID_ARGUMENT, "the two component volumes differ in type or cell layout");
      }
    });
  });
}

}  // namespace rvk
