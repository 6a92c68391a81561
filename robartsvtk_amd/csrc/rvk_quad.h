// rvk_quad.h -- the compositing march with four lanes of a wave on one ray.
//
// A quad takes four samples of its ray at once and composites them in order,
// so every ray accumulates the same samples in the same order with the same
// operations as the one-lane casters: the images are the same to the bit.
// The skip rule's chunks are speculative as in drr_march_lanes.
//
// Why four lanes: with one, a wave waits on one chain of load, table and
// gradient per sample (VALU 24 % busy for a 128^3 u8 volume at 512^2), and its
// 64 rays' gathers share few cells; a quad's four samples share most of
// theirs, the chain is a quarter as long, and the ordered compositing of a
// chunk, by quad broadcasts, costs about 33 VALU instructions per 64 samples
// of 60 to 250.  Now bound by VALU issue (73 to 95 % busy in the 2D casters).
// 16 blocks in a row go to one XCD, which are a strip of 64x16 pixels (four
// tiles of a super-tile's row), the strips dealt over the XCDs (runs of 4, 8,
// 16, 32 and 64 blocks measured within 3 %, a band per XCD 10 to 50 % slower: it
// leaves the XCDs of the image's rim idle).
//
// One lane in bands against this, us: 1D 128^3 u8 512^2 108 -> 90, 1024^2
// 267 -> 249, 128^2 120 -> 57; shaded 1D 250x250x181 int16 800x600 453 -> 282;
// 2D with gradient magnitude 512^3 u16 1920x1080 4555 -> 2872 (another scene
// 2549 -> 2068, at 3840x2160 8250 -> 6448), with gradients per sample
// 11636 -> 5353; shaded 2D 301x257x180 1280x720 1134 -> 871; in/ex 256x256x200
// 640x480 626 -> 281; dual 320x320x211 1024x768 1225 -> 516.  The one-lane
// casters take the views that these do not march (quad_ok) and those of many
// rays with few samples each (quad_pays).
#pragma once
#include "rvk_cast.h"

namespace rvk {

// Lane S of the quad's value in all its lanes (the quad is converged).
template <int S> __device__ __forceinline__ float quad_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), S * 0x55, 0xf, 0xf, true));
}
__device__ __forceinline__ uint32_t quad_bits(bool c) {
  return (uint32_t)(__ballot(c) >> (threadIdx.x & 60u)) & 15u;
}

struct QuadRay {
  float Tr, r, g, b;
  float t;       // steps taken
  bool special;  // in/ex: something was composited
};

// (1D, in/ex and dual casters: 5 to 10 % of their time; in the 2D caster runs
// were slower, 2872 -> 3212 us, its columns being live nearly everywhere.)
// Passes over samples whose value alone keeps them from compositing: the
// columns of the transfer function that the values of the range brick (or
// group of bricks) around a sample can reach have no opacity, so no sample in
// it counts.  `bits` are the columns with opacity; a range over more than two
// of their words counts as live.
struct QuadSkip {
  RangeWalk w;
  const float2* ranges;  // NULL: no skipping
  const uint32_t* bits;
  float lo, mult, scale, shift;  // column of a value v: floor(mult (v - lo) scale + shift)
  int n;
  bool pair;  // a sample reads its column and the next one

  __device__ __forceinline__ int column(float v) const {
    const float x = fminf(fmaxf(mult * (v - lo) * scale + shift, -1.0f), scale);
    return (int)floorf(x);
  }
  __device__ __forceinline__ bool dead(const float2& r) const {
    const int a = column(r.x), b = column(r.y);
    const int i0 = min(max(min(a, b), 0), n - 1), i1 = min(max(max(a, b) + (pair ? 1 : 0), 0), n - 1);
    const int w0 = i0 >> 5, w1 = i1 >> 5;
    const uint32_t m0 = ~0u << (i0 & 31), m1 = ~0u >> (31 - (i1 & 31));
    const uint32_t b0 = bits[w0], b1 = bits[w1];
    return w1 == w0 ? (b0 & m0 & m1) == 0u : (w1 == w0 + 1 && ((b0 & m0) | (b1 & m1)) == 0u);
  }
};

// The march of kst samples.  test(t) evaluates the sample t (never past the
// end) and says whether it counts: bit 0 it composites, bit 1 (EXCLUDES) it
// ends the ray when it would be the first composited, bit 2 its value alone
// keeps it from compositing.  shade(t, a, r, g, b) gives the opacity and
// colour of the sample tested last; run_at(t, tend, 1 / stride) how many of
// the samples t, t + stride, ... before tend do not composite, after a chunk
// of samples that could not by their value.  Needs term <= 1.
template <bool SKIP, bool EXCLUDES, typename Test, typename Shade, typename Run>
__device__ __forceinline__ QuadRay quad_march(int kst, float term, Test&& test, Shade&& shade, Run&& run_at) {
  QuadRay o{1.0f, 0.0f, 0.0f, 0.0f, 0.0f, false};
  const int s = (int)(threadIdx.x & 3u);
  const float fs = (float)s, tend = (float)kst;
  float t = 0.0f;
  bool two = false;      // looking at every other sample
  uint32_t stepped = 0;  // 1: the chunk's first sample is a step back
  while (t < tend) {
    const float ts = fmaf(fs, (SKIP && two) ? 2.0f : 1.0f, t);
    const bool in = ts < tend;
    const uint32_t fl = test(in ? ts : t);
    const bool c = in && (fl & 1u);
    const uint32_t bits = quad_bits(c);
    const bool dead = quad_bits(!in || (fl & 4u)) == 15u;
    if (SKIP && two) {
      const int run = __ffs(bits | 16u) - 1;
      if (run < 4) {
        t += (float)(2 * run - 1);
        two = false;
        stepped = 1u;
      } else {
        t = fminf(t + 8.0f, fmaf(2.0f, ceilf((tend - t) * 0.5f), t));
        if (dead && t < tend) t = fmaf(2.0f, run_at(t, tend, 0.5f), t);
      }
      continue;
    }
    const int run = SKIP ? __ffs(~(bits | stepped)) - 1 : 4;  // bits above 3 are clear: at most 4
    const uint32_t taken = SKIP ? bits & ((1u << run) - 1u) : bits;
    if (taken) {
      const int first = __ffs(taken) - 1;
      if (EXCLUDES && !o.special) {
        if ((quad_bits((fl & 2u) != 0u) >> first) & 1u) {
          o.t = t + (float)(first + 1);
          return o;
        }
        o.special = true;
      }
      float a = 0.0f, r = 0.0f, g = 0.0f, b = 0.0f;
      if ((taken >> s) & 1u) shade(ts, a, r, g, b);
      const float om = 1.0f - a;
      const float T1 = o.Tr * quad_bcast<0>(om), T2 = T1 * quad_bcast<1>(om);
      const float T3 = T2 * quad_bcast<2>(om), T4 = T3 * quad_bcast<3>(om);
      // the sample after which the ray's transmittance is below term
      const int stop = T1 < term ? 0 : T2 < term ? 1 : T3 < term ? 2 : T4 < term ? 3 : 4;
      const float Ts = s == 0 ? o.Tr : s == 1 ? T1 : s == 2 ? T2 : T3;
      const float wt = s <= stop ? Ts * a : 0.0f;
      r *= wt; g *= wt; b *= wt;
      if (s > stop) r = g = b = 0.0f;
      o.r += quad_bcast<0>(r); o.g += quad_bcast<0>(g); o.b += quad_bcast<0>(b);
      o.r += quad_bcast<1>(r); o.g += quad_bcast<1>(g); o.b += quad_bcast<1>(b);
      o.r += quad_bcast<2>(r); o.g += quad_bcast<2>(g); o.b += quad_bcast<2>(b);
      o.r += quad_bcast<3>(r); o.g += quad_bcast<3>(g); o.b += quad_bcast<3>(b);
      if (stop < 4) {
        o.Tr = 0.0f;
        o.t = t + (float)(stop + 1);
        return o;
      }
      o.Tr = T4;
    }
    if (SKIP) {
      // past the run the next sample is empty and the one after it unseen;
      // past the ray's last sample there is neither
      const float u = t + (float)run;
      two = run < 4;
      t = (two && u < tend) ? u + 2.0f : fminf(u, tend);
      stepped = 0u;
    } else {
      t = fminf(t + 4.0f, tend);
      if (dead && t < tend) t += run_at(t, tend, 1.0f);
    }
  }
  o.t = t;
  return o;
}

// A quad ray's set-up; samples are counted by the caster.
struct QuadSetup {
  Ray r;
  V3<float> p0c;
  float j;
};
__device__ __forceinline__ QuadSetup quad_setup(const VolGeom& g, const ViewGeom& v, float step_len, int jitter, int x,
                                                int y) {
  QuadSetup q;
  q.r = form_ray(g, v, step_len, x, y);
  q.j = ray_offset(jitter, x, y);
  q.p0c = cell_coord(V3<float>{q.r.start.x + q.j * q.r.inc.x, q.r.start.y + q.j * q.r.inc.y,
                               q.r.start.z + q.j * q.r.inc.z});
  return q;
}

// QuadSkip of a ray (only where every sample lies in the cells).
__device__ __forceinline__ QuadSkip quad_skip(const VolGeom& g, const DrrMarchArgs& m, const QuadSetup& q, int kst,
                                              const uint32_t* bits, int n, float lo, float mult, bool pair) {
  QuadSkip k;
  k.w = range_walk(q.p0c, q.r.inc);
  k.ranges = samples_in_cells(g, q.p0c, q.r.inc, kst) ? m.ranges : nullptr;
  k.bits = bits;
  k.lo = lo;
  k.mult = mult;
  k.scale = (float)n;
  k.shift = pair ? -0.5f : 0.0f;
  k.n = n;
  k.pair = pair;
  return k;
}
// The run of samples from t on (quad_march's run_at).
__device__ __forceinline__ float quad_run(const DrrMarchArgs& m, const QuadSkip& k, const QuadSetup& q, float t,
                                          float tend, float inv_stride) {
  if (!k.ranges) return 0.0f;
  RangeAt at;
  if (!range_at(m, sample_pos<true>(q.p0c, q.p0c, q.r.inc, t), at, [&](const float2& r) { return k.dead(r); }))
    return 0.0f;
  return run_length(at, k.w, t, tend, inv_stride);
}

// Central differences at q (V/...2D...cuh:263-271).
template <typename CV>
__device__ __forceinline__ V3<float> sample_gradient(CV vol, const VolGeom& g, const V3<float>& q) {
  V3<float> gr;
  gr.x = (trilinear(vol, g, q.x + 1.0f, q.y, q.z) - trilinear(vol, g, q.x - 1.0f, q.y, q.z)) * g.srecip[0];
  gr.y = (trilinear(vol, g, q.x, q.y + 1.0f, q.z) - trilinear(vol, g, q.x, q.y - 1.0f, q.z)) * g.srecip[1];
  gr.z = (trilinear(vol, g, q.x, q.y, q.z + 1.0f) - trilinear(vol, g, q.x, q.y, q.z - 1.0f)) * g.srecip[2];
  return gr;
}

// The Phong-lit colour of a table cell at a sample with gradient gr.
__device__ __forceinline__ void lit_cell(const Tf2dCell* cell, const float4& c0, const VolGeom& g, const V3<float>& gr,
                                         float gmag, const V3<float>& inc, float rlen, float& a, float& r, float& gg,
                                         float& b) {
  const float4 c1 = *(const float4*)&cell->spec_power;
  const float pl =
      satf(fabsf(gr.x * inc.x * g.sp[0] + gr.y * inc.y * g.sp[1] + gr.z * inc.z * g.sp[2]) / (gmag * rlen));
  const float shd = c0.y + c0.z * pl;
  const float shs = c0.w * powf(pl, c1.x);
  a = c0.x;
  r = satf(shd * c1.y + shs);
  gg = satf(shd * c1.z + shs);
  b = satf(shd * c1.w + shs);
}

template <typename A>
__device__ __forceinline__ void quad_store(const A& a, int x, int y, const Ray& r, uint32_t rgba, float depth) {
  if (threadIdx.x & 3u) return;
  const long idx = (long)y * a.v.W + x;
  a.out[idx] = rgba;
  if (a.depth) a.depth[idx] = depth;
  if (a.min_depth) a.min_depth[idx] = r.min_depth;
  if (a.max_depth) a.max_depth[idx] = r.max_depth;
}
__device__ __forceinline__ uint32_t pack_rgba(float r, float g, float b, float a) {
  return to_u8(255.0f * r) | (to_u8(255.0f * g) << 8) | (to_u8(255.0f * b) << 16) | (to_u8(255.0f * a) << 24);
}

}  // namespace rvk
