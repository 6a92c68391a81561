// rvk_march.h -- the DRR march and its shared pieces, used by the single-view
// caster and by the batched forward / adjoint kernels, so every path runs the
// same operations in the same order.
#pragma once
#include <type_traits>

#include "rvk_internal.h"

namespace rvk {

// The reference's 16x16 ray-offset table (V/vtkCudaVolumeMapper.cxx:59-93),
// indexed by (x mod 16) + 16 (y mod 16).  Parity depends on it bit for bit.
static __constant__ float kRayOffsets[256] = {
  0.70554f, 0.53342f, 0.57951f, 0.28956f, 0.30194f, 0.77474f, 0.01401f, 0.76072f,
  0.81449f, 0.70903f, 0.04535f, 0.41403f, 0.86261f, 0.79048f, 0.37353f, 0.96195f,
  0.87144f, 0.05623f, 0.94955f, 0.36401f, 0.52486f, 0.76711f, 0.0535f, 0.59245f,
  0.4687f, 0.29816f, 0.62269f, 0.64782f, 0.26379f, 0.27934f, 0.8298f, 0.8246f,
  0.58916f, 0.98609f, 0.91096f, 0.22686f, 0.69511f, 0.98f, 0.24393f, 0.53387f,
  0.10636f, 0.99941f, 0.67617f, 0.0157f, 0.57518f, 0.10005f, 0.10302f, 0.79888f,
  0.28448f, 0.04564f, 0.29577f, 0.38201f, 0.30097f, 0.94857f, 0.97982f, 0.40137f,
  0.27827f, 0.16044f, 0.16282f, 0.64658f, 0.41007f, 0.41276f, 0.71273f, 0.3262f,
  0.63317f, 0.20756f, 0.18601f, 0.58335f, 0.08071f, 0.45797f, 0.90572f, 0.26136f,
  0.78521f, 0.3789f, 0.28966f, 0.91937f, 0.63174f, 0.62764f, 0.42845f, 0.09797f,
  0.56104f, 0.69448f, 0.91371f, 0.83481f, 0.02262f, 0.54336f, 0.91616f, 0.43026f,
  0.67794f, 0.50245f, 0.51373f, 0.46298f, 0.35347f, 0.40483f, 0.26973f, 0.05559f,
  0.24384f, 0.97907f, 0.06091f, 0.39029f, 0.36499f, 0.48989f, 0.15566f, 0.47445f,
  0.25726f, 0.62875f, 0.54207f, 0.1563f, 0.93854f, 0.65449f, 0.50608f, 0.39047f,
  0.10737f, 0.78399f, 0.45964f, 0.75368f, 0.59609f, 0.83273f, 0.01875f, 0.21036f,
  0.07395f, 0.10545f, 0.33169f, 0.12824f, 0.00024f, 0.53679f, 0.65705f, 0.54401f,
  0.82741f, 0.08189f, 0.19192f, 0.67891f, 0.4542f, 0.35702f, 0.14998f, 0.70439f,
  0.92878f, 0.53021f, 0.08964f, 0.75772f, 0.40184f, 0.46187f, 0.49216f, 0.20762f,
  0.32973f, 0.09542f, 0.58979f, 0.16987f, 0.92761f, 0.09792f, 0.44386f, 0.27294f,
  0.87254f, 0.75068f, 0.27294f, 0.67364f, 0.25662f, 0.08989f, 0.03095f, 0.32271f,
  0.79012f, 0.29725f, 0.23528f, 0.48047f, 0.2546f, 0.3406f, 0.04493f, 0.48242f,
  0.20601f, 0.86453f, 0.58862f, 0.7549f, 0.92788f, 0.33101f, 0.54294f, 0.08069f,
  0.63437f, 0.41003f, 0.96042f, 0.11462f, 0.92344f, 0.6202f, 0.34772f, 0.14924f,
  0.47997f, 0.2194f, 0.99373f, 0.13042f, 0.02888f, 0.34539f, 0.54766f, 0.92295f,
  0.53824f, 0.40642f, 0.84724f, 0.82622f, 0.67242f, 0.72189f, 0.99677f, 0.3398f,
  0.49521f, 0.41296f, 0.69528f, 0.17908f, 0.42291f, 0.54317f, 0.81466f, 0.54091f,
  0.42753f, 0.50906f, 0.22778f, 0.61918f, 0.48983f, 0.68081f, 0.8866f, 0.37051f,
  0.30249f, 0.29286f, 0.15031f, 0.52982f, 0.22326f, 0.58452f, 0.36345f, 0.87597f,
  0.47801f, 0.19063f, 0.68406f, 0.74741f, 0.61393f, 0.78213f, 0.16174f, 0.80777f,
  0.20261f, 0.95676f, 0.06585f, 0.06152f, 0.79319f, 0.3796f, 0.46358f, 0.11954f,
  0.11547f, 0.17377f, 0.04811f, 0.71481f, 0.53302f, 0.561f, 0.21673f, 0.468f,
  0.74635f, 0.75231f, 0.39893f, 0.90309f, 0.746f, 0.08855f, 0.63457f, 0.71302f};

__device__ __forceinline__ float ray_offset(int jitter, int x, int y) {
  return jitter ? kRayOffsets[(x & 15) + 16 * (y & 15)] : 0.0f;
}

__device__ __forceinline__ float ray_length(const VolGeom& g, const V3<float>& inc) {
  return sqrtf(inc.x * inc.x * g.sp[0] * g.sp[0] + inc.y * inc.y * g.sp[1] * g.sp[1] +
               inc.z * inc.z * g.sp[2] * g.sp[2]);
}

__device__ __forceinline__ void step(V3<float>& p, const V3<float>& inc) {
  p.x += inc.x; p.y += inc.y; p.z += inc.z;
}

// Sample coordinate in cell units (c = p + 0.5, what trilinear() takes).
// Reference mode keeps the incrementally updated p (p += inc per step, as the
// CUDA kernels do) and adds 0.5; PRECISE derives it from the step index,
// c = (p0 + 0.5) + (k_start - k) inc with one rounding per axis, which removes
// the drift repeated FP32 additions build up.
template <bool PRECISE>
__device__ __forceinline__ V3<float> sample_pos(const V3<float>& p, const V3<float>& p0c, const V3<float>& inc,
                                                float t) {
  if (!PRECISE) return V3<float>{p.x + 0.5f, p.y + 0.5f, p.z + 0.5f};
  return V3<float>{fmaf(t, inc.x, p0c.x), fmaf(t, inc.y, p0c.y), fmaf(t, inc.z, p0c.z)};
}
template <bool PRECISE>
__device__ __forceinline__ V3<float> sample_pos(const V3<float>& p, const V3<float>& p0c, const V3<float>& inc, int kst,
                                                int k) {
  return sample_pos<PRECISE>(p, p0c, inc, (float)(kst - k));
}

__device__ __forceinline__ V3<float> cell_coord(const V3<float>& p) {
  return V3<float>{p.x + 0.5f, p.y + 0.5f, p.z + 0.5f};
}

// The precise DRR march samples at c = p0c + t inc for t in [0, kst - 1], one
// fma per axis, which is monotone in t.  So when c at t = 0 and at t = kst
// lies in the cell range [0, n + 1] on every axis, every sample does and
// trilinear() needs no clamp.  Rays that pass the volume clip have both ends
// within [0, n - 1] in voxels (V/CUDA_vtkCudaVolumeMapper_renderAlgo.cu:297-311),
// so their samples lie in [0.5, n - 0.5] and always pass; a ray that fails
// (a non-finite set-up) takes no samples, in the oracle as here.  (The
// compositing casters keep the clamp: their +-1 gradient taps reach
// [-0.5, n + 0.5].)
__device__ __forceinline__ bool samples_in_cells(const VolGeom& g, const V3<float>& p0c, const V3<float>& inc,
                                                 int kst) {
  const float t = (float)kst;
  const float s[3] = {p0c.x, p0c.y, p0c.z};
  const float e[3] = {fmaf(t, inc.x, p0c.x), fmaf(t, inc.y, p0c.y), fmaf(t, inc.z, p0c.z)};
  bool ok = true;
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    const float hi = (float)(g.n[a] + 1);
    ok = ok && s[a] >= 0.0f && s[a] <= hi && e[a] >= 0.0f && e[a] <= hi;
  }
  return ok;
}

// ===========================================================================
// DRR march (V/CUDA_vtkCudaDRRImageVolumeMapper_renderAlgo.cuh:11-117)
struct DrrMarchArgs {
  float intercept, slope, offset;
  int output, ref_term, jitter;
  const float2* ranges;  // per range brick (min, max) of the frame, or NULL
  int rbx, rby;          // range-brick grid extent in x and y
  const float2* groups;  // the same per 4^3 range bricks
  int rgx, rgy;
};

// One view of the single-view caster.
struct DrrArgs {
  VolGeom g;
  ViewGeom v;
  float step_len;
  DrrMarchArgs m;
  uint32_t tint;
  const void* vol;
  void* out;
  int tiles_x;
  int deal;  // tiles dealt to the XCDs in runs (xcd_deal), or one band each
};

// Run skipping of the precise march.  Each range brick (kRangeEdge^3 cells)
// has the (min, max) of every value its cells can interpolate, and each group
// of 4^3 bricks (32^3 cells) that of its bricks.  After a sample at cell
// coordinate q, with R the group that holds q, or else its brick:
//  - if no value of R can contribute (alpha = fma(cs, v, ci) >= 0 at the
//    bound that minimises it: alpha is monotone in v), the samples the march
//    takes next inside R do not contribute either;
//  - if R is constant (min == max: every corner equal, so every sample in it
//    interpolates that value exactly) and q contributed, the next samples
//    contribute the same alpha.
// Either way the march's state after such a run is known in closed form, so
// the run's gathers are skipped (a contributing run of m adds m alpha with
// one f64 rounding; with termination it adds one by one, testing each).
//
// The run ends kRunMargin voxels before R's far face, so that no rounding of
// the exit time or of a sample's position (below 0.0015 voxels for coordinates
// up to 4097) can count a sample outside R; positions are monotone in t.
constexpr float kRunMargin = 0.004f;
struct RangeWalk {
  V3<float> e, c;     // exit time of the brick with index b on an axis: b e + c
  V3<uint32_t> far;   // 3 on axes the ray goes up: a group's last brick is b | 3, else b & ~3
};
__device__ __forceinline__ RangeWalk range_walk(const V3<float>& p0c, const V3<float>& inc) {
  RangeWalk w;
  auto axis = [](float p, float i, float& e, float& c, uint32_t& far) {
    const float r = 1.0f / i;
    e = i != 0.0f ? (float)kRangeEdge * r : 0.0f;
    c = i != 0.0f ? ((i > 0.0f ? (float)kRangeEdge - kRunMargin : kRunMargin) - p) * r : __builtin_huge_valf();
    far = i > 0.0f ? 3u : 0u;
  };
  axis(p0c.x, inc.x, w.e.x, w.c.x, w.far.x);
  axis(p0c.y, inc.y, w.e.y, w.c.y, w.far.y);
  axis(p0c.z, inc.z, w.e.z, w.c.z, w.far.z);
  return w;
}

// The ranges around q and the brick index; group = whether `use` holds for
// the group's range, and the return whether for either.
struct RangeAt {
  uint32_t bx, by, bz;
  bool group;
};
template <typename U>
__device__ __forceinline__ bool range_at(const DrrMarchArgs& a, const V3<float>& q, RangeAt& at, U&& use) {
  at.bx = (uint32_t)(int)q.x >> kRangeLog2;
  at.by = (uint32_t)(int)q.y >> kRangeLog2;
  at.bz = (uint32_t)(int)q.z >> kRangeLog2;
  const float2 g = a.groups[((at.bz >> 2) * (uint32_t)a.rgy + (at.by >> 2)) * (uint32_t)a.rgx + (at.bx >> 2)];
  const float2 r = a.ranges[(at.bz * (uint32_t)a.rby + at.by) * (uint32_t)a.rbx + at.bx];
  at.group = use(g);
  return at.group || use(r);
}

// How many of the samples t1, t1 + stride, ... before lim (stride a power of
// two; t1 and lim integers) lie in the region, which holds the sample before.
__device__ __forceinline__ float run_length(const RangeAt& at, const RangeWalk& w, float t1, float lim,
                                            float inv_stride) {
  const uint32_t keep = at.group ? ~3u : ~0u, on = at.group ? 3u : 0u;
  const float tx = fmaf((float)((at.bx & keep) | (w.far.x & on)), w.e.x, w.c.x);
  const float ty = fmaf((float)((at.by & keep) | (w.far.y & on)), w.e.y, w.c.y);
  const float tz = fmaf((float)((at.bz & keep) | (w.far.z & on)), w.e.z, w.c.z);
  const float te = fminf(fminf(tx, ty), fminf(tz, lim));
  return fmaxf(ceilf((te - t1) * inv_stride), 0.0f);
}

// Non-contributing samples to pass over after the one at q (the next at t1).
__device__ __forceinline__ float empty_run(const DrrMarchArgs& a, const V3<float>& q, const RangeWalk& w, float cs,
                                           float ci, float t1, float lim, float inv_stride) {
  RangeAt at;
  if (!range_at(a, q, at, [&](const float2& r) { return fmaf(cs, cs <= 0.0f ? r.y : r.x, ci) >= 0.0f; }))
    return 0.0f;
  return run_length(at, w, t1, lim, inv_stride);
}

// Contributing run after the sample at q (alpha; next sample at t): adds the
// run's alphas to acc and advances t.  Returns true when acc reached stop_at
// inside the run (the march ends there, as it would have).
template <bool TERM, typename Acc>
__device__ __forceinline__ bool flat_run(const DrrMarchArgs& a, const V3<float>& q, const RangeWalk& w, float cs,
                                         float ci, float alpha, float& t, float lim, float stride, float inv_stride,
                                         Acc& acc, Acc stop_at) {
  RangeAt at;
  if (!range_at(a, q, at, [&](const float2& r) { return r.x == r.y && fmaf(cs, r.x, ci) == alpha; })) return false;
  const float m = run_length(at, w, t, lim, inv_stride);
  if (TERM) {
    for (int i = 0; i < (int)m; ++i) {
      acc += (Acc)alpha;
      if (acc <= stop_at) return true;
    }
  } else {
    acc = fma((Acc)m, (Acc)alpha, acc);
  }
  t = fmaf(m, stride, t);
  return false;
}

// Visitors declare whether a sample with a zero gradient may go unvisited
// (kFlatRuns): samples of constant bricks have gradient +0.
struct NoVisit {
  static constexpr bool kFlatRuns = true;
  __device__ __forceinline__ void operator()(const V3<float>&, float, float, const V3<float>&) const {}
};

// The output of a march that ended with accumulator L, by selects: written as
// a chain of uniform branches, hipcc's code for the L output skipped the
// negation in some of the kernels this is inlined into.
__device__ __forceinline__ float drr_value(const DrrMarchArgs& a, float L) {
  const float e = expf(L), o = 256.0f - e;
  const float ref = o < 0.0f ? 0.0f : o;
  const float v = a.output == RVK_DRR_F32_EXP_NEG_L ? e : -L;
  return a.output == RVK_DRR_RGBA8_REF ? ref : v;
}

// Line integral along one ray.  The accumulator starts at ln(256*offset) in
// the reference RGBA8 mode and at 0 in the float modes.  `visit(c, t, alpha,
// grad)` is called for every accumulated sample, with c its sample cell
// coordinate (c = p0 + 0.5 + t*inc in PRECISE mode); with VG the trilinear
// gradient at c comes from the same gathers as the value (the adjoint marches
// through this very control flow).  RUNS (precise mode only) takes the runs
// above when the volume frame has brick ranges (a.ranges): the same samples
// count, and a run's sum is rounded once instead of per sample.  Runs make the
// tiles through empty space cheap, so their launches deal the tiles to the
// XCDs instead of giving each a band (drr_ahead_kernel has both measured).
template <typename CV, bool SKIP, bool PRECISE, bool VG = false, bool RUNS = false, bool KEY = true,
          bool TERM = true, typename F = NoVisit>
__device__ __forceinline__ float drr_march(CV vol, const VolGeom& g, const DrrMarchArgs& a,
                                           const Ray& r, int x, int y, F&& visit = F()) {
  using FV = typename std::remove_reference<F>::type;
  const bool ref_mode = a.output == RVK_DRR_RGBA8_REF;
  const float lg = logf(256.0f * a.offset);
  // PRECISE sums the line integral in double: a converted f32 sample and one
  // f64 add cost less than a compensated f32 sum and carry more precision
  // (the f64 add runs at the f32 rate).  The reference mode sums in f32.
  using Acc = typename std::conditional<PRECISE, double, float>::type;
  Acc acc = ref_mode ? (Acc)lg : (Acc)0;
  // termination at acc <= stop_at only with ref_term (otherwise never)
  const Acc stop_at = !a.ref_term ? (Acc)-__builtin_huge_valf() : (ref_mode ? (Acc)0 : (Acc)-lg);
  const float j = ray_offset(a.jitter, x, y);
  V3<float> p{r.start.x + j * r.inc.x, r.start.y + j * r.inc.y, r.start.z + j * r.inc.z};
  const V3<float> inc = r.inc;
  const V3<float> p0c = cell_coord(p);
  int kst = step_count(r.num_steps - j);
  if (PRECISE && !samples_in_cells(g, p0c, inc, kst)) kst = 0;
  const float ds = ray_length(g, inc);
  const float ci = a.intercept * -ds;
  const float cs = a.slope * -ds;
  // The march counts in t = kst - k (k = steps left), exactly, as a float:
  // sample t sits at p0 + t inc, the ray ends at t = kst, and the keyhole
  // window es >= k > ee is t in [kst - es, kst - ee).
  const int es = kst - (int)ceilf(r.exclude_start);
  const int ee = kst - (int)floorf(r.exclude_end);
  const float tend = (float)kst, kw0 = (float)(kst - es), kw1 = (float)(kst - ee);
  float t = 0.0f;
  // skip-rule state z = sb - sa in {-1, 0, 1}: sa = the sample is a
  // back-step, sb = the last step skipped a sample (never both), so each arm
  // updates one float in place
  float z = 0.0f;
  const bool runs = RUNS && PRECISE && a.ranges != nullptr;
  const RangeWalk w = range_walk(p0c, inc);
  // a contributing run must end before the keyhole window
  const float flat_lim = fminf(kw0, tend);
  // a repeated alpha is the cheap hint of a constant brick
  float alpha_prev = __builtin_nanf("");
  while (t < tend) {
    // KEY = false: the view has no keyhole planes, so no ray has a window
    const bool in_key = KEY && (t >= kw0 && t < kw1);
    const V3<float> q = sample_pos<PRECISE>(p, p0c, inc, t);
    V3<float> gr{0.0f, 0.0f, 0.0f};
    const float alpha = fmaf(cs, VG ? trilinear_vg<!PRECISE>(vol, g, q.x, q.y, q.z, gr)
                                    : trilinear<!PRECISE>(vol, g, q.x, q.y, q.z), ci);
    const bool repeat = alpha == alpha_prev;
    alpha_prev = alpha;
    const float ts = t;
    if (SKIP) {
      // t stays an exact integer, so one add of +-1 or 2 equals the
      // reference's single steps; a back-stepped sample adds +0 (acc is
      // never -0), which leaves the sum unchanged without a select
      if (alpha < 0.0f && !in_key) {
        // sa' = sb, sb' = 0: z' = -sb = median(-z, -1, 0), and sa' = -z'
        z = __builtin_amdgcn_fmed3f(-z, -1.0f, 0.0f);
        if (!PRECISE) {
          if (z != 0.0f) { p.x = p.x - inc.x; p.y = p.y - inc.y; p.z = p.z - inc.z; }
          else { p.x = p.x + inc.x; p.y = p.y + inc.y; p.z = p.z + inc.z; }
        }
        t += fmaf(2.0f, z, 1.0f);  // 1 - 2 sa'
        if (VG && z == 0.0f) visit(q, ts, alpha, gr);
        // alpha - alpha * sa': alpha, or +0 for a back-stepped sample
        acc += (Acc)fmaf(alpha, z, alpha);
        if (TERM && acc <= stop_at) break;
        // each further sample of a contributing run steps 1 (sa = sb = 0)
        if (FV::kFlatRuns && runs && repeat && z == 0.0f) {
          if (flat_run<TERM>(a, q, w, cs, ci, alpha, t, t >= kw1 ? tend : flat_lim, 1.0f, 1.0f, acc, stop_at)) break;
        }
      } else {
        if (!PRECISE) {
          if (z >= 0.0f) step(p, inc);  // sa == 0
          step(p, inc);
        }
        // sa' = 0, sb' = 1 - sa = min(z + 1, 1) (z + 1 >= 0); the step is 2 - sa
        z = __builtin_amdgcn_fmed3f(z + 1.0f, 0.0f, 1.0f);
        t += 1.0f + z;
        // each further non-contributing sample steps 2 and leaves sb = 1
        if (runs) {
          const float m = empty_run(a, q, w, cs, ci, t, tend, 0.5f);
          if (m > 0.0f) {
            t += 2.0f * m;
            z = 1.0f;
          }
        }
      }
    } else {
      if (!PRECISE) step(p, inc);
      t += 1.0f;
      if (alpha < 0.0f && !in_key) {
        acc += (Acc)alpha;
        if (VG) visit(q, ts, alpha, gr);
        if (TERM && acc <= stop_at) break;
        if (FV::kFlatRuns && runs && repeat) {
          if (flat_run<TERM>(a, q, w, cs, ci, alpha, t, t >= kw1 ? tend : flat_lim, 1.0f, 1.0f, acc, stop_at)) break;
        }
      } else if (runs) {
        t += empty_run(a, q, w, cs, ci, t, tend, 1.0f);
      }
    }
  }
  return drr_value(a, (float)acc);
}

// A wave whose lanes found no run looks for none for a while: inside a body, or
// where values scatter about alpha = 0 (a scanner's air), bricks are neither
// empty nor constant, yet some lane asks nearly every time (256^3 CT with noise
// in the air at 1024^2, looking always / so: 1012 / 604 us, without the skip rule
// 793 / 418; in clean air, where the loop without lookups is the shorter,
// 323 / 232 and 326 / 217; rests of 8 and 16 iterations within 4 %).
constexpr int kRunRest = 16;    // iterations of drr_march_ahead
constexpr int kLanesRest = 24;  // samples of drr_march_lanes, in chunks of a ray's lanes

// The same line integral, the sample after the next gathered along with the
// next: where the march goes on as it did (sample by sample while samples
// contribute, two by two while they do not) that one is the next but one, and
// otherwise it is dropped, so the samples taken, their order and the sum are
// drr_march's to the bit.  For single views, whose last round of waves is
// nearly empty and waits on one gather at a time.  Where a quarter of a wave's
// lanes drop theirs (samples that contribute or not at random) it goes on one
// sample at a time for a while.  Precise march, no termination.
template <typename CV, bool SKIP, bool KEY>
__device__ __forceinline__ float drr_march_ahead(CV vol, const VolGeom& g, const DrrMarchArgs& a, const Ray& r, int x,
                                                 int y) {
  const float j = ray_offset(a.jitter, x, y);
  const V3<float> inc = r.inc;
  const V3<float> p0c = cell_coord(V3<float>{r.start.x + j * inc.x, r.start.y + j * inc.y, r.start.z + j * inc.z});
  int kst = step_count(r.num_steps - j);
  if (!samples_in_cells(g, p0c, inc, kst)) kst = 0;
  const float ds = ray_length(g, inc);
  const float ci = a.intercept * -ds;
  const float cs = a.slope * -ds;
  const int es = kst - (int)ceilf(r.exclude_start);
  const int ee = kst - (int)floorf(r.exclude_end);
  const float tend = (float)kst, kw0 = (float)(kst - es), kw1 = (float)(kst - ee);
  const float flat_lim = fminf(kw0, tend);
  const bool runs = a.ranges != nullptr;
  const RangeWalk w = range_walk(p0c, inc);
  double acc = a.output == RVK_DRR_RGBA8_REF ? (double)logf(256.0f * a.offset) : 0.0;
  float t = 0.0f;
  float z = 0.0f;  // the skip rule's state, as in drr_march
  float alpha_prev = 0.0f;
  // one sample; look: with the lookups
  auto take = [&](const V3<float>& q, float alpha, auto look) {
    constexpr bool LOOK = decltype(look)::value;
    const bool in_key = KEY && (t >= kw0 && t < kw1);
    const bool repeat = alpha == alpha_prev;
    alpha_prev = alpha;
    if (alpha < 0.0f && !in_key) {
      if (SKIP) {
        z = __builtin_amdgcn_fmed3f(-z, -1.0f, 0.0f);
        t += fmaf(2.0f, z, 1.0f);
        acc += (double)fmaf(alpha, z, alpha);
      } else {
        t += 1.0f;
        acc += (double)alpha;
      }
      if (LOOK && runs && repeat && z == 0.0f)
        flat_run<false>(a, q, w, cs, ci, alpha, t, t >= kw1 ? tend : flat_lim, 1.0f, 1.0f, acc, 0.0);
    } else if (SKIP) {
      z = __builtin_amdgcn_fmed3f(z + 1.0f, 0.0f, 1.0f);
      t += 1.0f + z;
      if (LOOK && runs) {
        const float m = empty_run(a, q, w, cs, ci, t, tend, 0.5f);
        if (m > 0.0f) {
          t += 2.0f * m;
          z = 1.0f;
        }
      }
    } else {
      t += 1.0f;
      if (LOOK && runs) t += empty_run(a, q, w, cs, ci, t, tend, 1.0f);
    }
  };
  // two samples; whether the second was dropped
  auto two = [&](auto look) {
    constexpr bool LOOK = decltype(look)::value;
    // the ray's end is in the cells too (samples_in_cells)
    const float t1 = fminf(SKIP ? t + 1.0f + fmaxf(z, 0.0f) : t + 1.0f, tend);
    const V3<float> q0 = sample_pos<true>(p0c, p0c, inc, t), q1 = sample_pos<true>(p0c, p0c, inc, t1);
    const float v0 = trilinear<false>(vol, g, q0.x, q0.y, q0.z), v1 = trilinear<false>(vol, g, q1.x, q1.y, q1.z);
    take(q0, fmaf(cs, v0, ci), look);
    const bool drop = t != t1;
    if (!SKIP && !LOOK) {
      // never dropped; without a branch, or hipcc sinks its gather into it
      const float alpha = fmaf(cs, v1, ci);
      const bool on = alpha < 0.0f && t < tend && !(KEY && (t >= kw0 && t < kw1));
      acc += on ? (double)alpha : 0.0;
      t += 1.0f;
    } else if (!drop && t < tend) {
      take(q1, fmaf(cs, v1, ci), look);
    }
    return drop;
  };
  while (t < tend) {
    const float t0 = t;
    alpha_prev = __builtin_nanf("");
    const bool drop = two(std::true_type());
    if (__ballot(t - t0 > 4.0f)) continue;  // a run moves a lane on by more than two steps
    if (SKIP && 4 * __popcll(__ballot(drop)) >= __popcll(__ballot(true))) {
#pragma unroll 1
      for (int i = 0; i < 4 * kRunRest && t < tend; ++i) {
        const V3<float> q = sample_pos<true>(p0c, p0c, inc, t);
        take(q, fmaf(cs, trilinear<false>(vol, g, q.x, q.y, q.z), ci), std::false_type());
      }
    } else {
#pragma unroll 1
      for (int i = 0; i < kRunRest && t < tend; ++i) two(std::false_type());
    }
  }
  return drr_value(a, (float)acc);
}

// The same line integral with 2^ls lanes of a wave on one ray, for launches
// with too few rays to fill the device (a wave then waits on one chain of
// dependent samples: 128^2 rays of ~100 samples took 63 us, 0.5 us a sample,
// with one wave on every fourth SIMD).  Lane s of the ray's 2^ls takes
// samples s, s + 2^ls, ...; the f64 partial sums are added at the end.
// Precise march, no termination (both tests are the caller's).
//
// The skip rule makes which samples count depend on the ones before, so its
// lanes take a chunk of samples at once, speculatively, and keep what the
// serial march would have: it runs either sample by sample (each one counts,
// until the first empty one at u: the next looked at is u + 2) or two by two
// (until the first contributing one at u: the march steps back to u - 1,
// which counts if it contributes, and goes on sample by sample from u).
// Either way the chunk's first change of run, found in the ballot of the
// samples' signs, says where the next chunk starts.
template <typename CV, bool SKIP, bool RUNS, bool VG = false, typename F = NoVisit>
__device__ __forceinline__ float drr_march_lanes(CV vol, const VolGeom& g, const DrrMarchArgs& a, const Ray& r, int x,
                                                 int y, int ls, F&& visit = F()) {
  const int S = 1 << ls, lane = (int)(threadIdx.x & 63u);
  const int s = lane & (S - 1), first = lane & ~(S - 1);
  const float j = ray_offset(a.jitter, x, y);
  const V3<float> p{r.start.x + j * r.inc.x, r.start.y + j * r.inc.y, r.start.z + j * r.inc.z};
  const V3<float> inc = r.inc, p0c = cell_coord(p);
  int kst = step_count(r.num_steps - j);
  if (!samples_in_cells(g, p0c, inc, kst)) kst = 0;
  const float ds = ray_length(g, inc);
  const float ci = a.intercept * -ds;
  const float cs = a.slope * -ds;
  const int es = kst - (int)ceilf(r.exclude_start);
  const int ee = kst - (int)floorf(r.exclude_end);
  const float tend = (float)kst, kw0 = (float)(kst - es), kw1 = (float)(kst - ee);
  const float fS = (float)S, fs = (float)s;
  double acc = 0.0;
  V3<float> gr{0.0f, 0.0f, 0.0f};
  auto sample = [&](float t) {
    const V3<float> q = sample_pos<true>(p, p0c, inc, t);
    return fmaf(cs, VG ? trilinear_vg<false>(vol, g, q.x, q.y, q.z, gr) : trilinear<false>(vol, g, q.x, q.y, q.z), ci);
  };
  const bool runs = a.ranges != nullptr;
  const RangeWalk w = range_walk(p0c, inc);
  const float flat_lim = fminf(kw0, tend);  // a contributing run ends before the keyhole window
  const int rest = kLanesRest >> ls;
  if (SKIP) {
    const uint32_t all = (1u << S) - 1u;
    float t = 0.0f;        // the chunk's first sample, the same in the ray's lanes
    bool two = false;      // running two by two
    uint32_t stepped = 0;  // 1: the chunk's first sample is a step back
    auto chunk = [&](bool look) {
      const float ts = fmaf(fs, two ? 2.0f : 1.0f, t);
      const bool in = ts < tend;
      const float tq = in ? ts : t;
      const float alpha = sample(tq);
      const bool c = in && alpha < 0.0f && !(tq >= kw0 && tq < kw1);
      const uint32_t bits = (uint32_t)(__ballot(c) >> first) & all;
      // two by two: samples before the first contributing one; one by one:
      // before the first empty one (a step back goes on from its successor)
      const int run = __ffs((two ? bits : ~(bits | stepped)) | (1u << S)) - 1;
      const bool whole = run == S;
      if (!two && s < run && c) {
        acc += (double)alpha;
        if (VG) visit(V3<float>{}, tq, alpha, gr);
      }
      t += two ? (whole ? 2.0f * fS : (float)(2 * run - 1)) : (whole ? fS : (float)(run + 2));
      stepped = (two && !whole) ? 1u : 0u;
      // a chunk that ended in its run: the run may go on through q's region
      // (samples one by one only when all alphas of the chunk were equal)
      if (look && whole && t < tend) {
        const bool flat = (((__ballot(alpha == __shfl(alpha, first, 64)) >> first) & all) == all);
        if (two || flat) {
          const V3<float> q = sample_pos<true>(p, p0c, inc, t);
          if (two) {
            t = fmaf(empty_run(a, q, w, cs, ci, t, tend, 0.5f), 2.0f, t);
          } else {
            double add = 0.0;
            flat_run<false>(a, q, w, cs, ci, alpha, t, t >= kw1 ? tend : flat_lim, 1.0f, 1.0f, add, 0.0);
            if (s == 0) acc += add;
          }
        }
      }
      two = two == whole;
    };
    if (!RUNS)
      while (t < tend) chunk(false);
    while (t < tend) {
      const float t0 = t;
      chunk(runs);
      if (__ballot(t - t0 > 2.0f * fS)) continue;  // a run moves a ray on by more than a chunk
#pragma unroll 1
      for (int i = 0; i < rest && t < tend; ++i) chunk(false);
    }
  } else {
    const float rS = 1.0f / fS;
    float alpha_prev = 0.0f;
    float t = fs;
    auto take = [&](bool look) {
      const V3<float> q = sample_pos<true>(p, p0c, inc, t);
      const float alpha = sample(t);
      const bool repeat = alpha == alpha_prev;
      alpha_prev = alpha;
      const float ts = t;
      t += fS;
      if (alpha < 0.0f && !(ts >= kw0 && ts < kw1)) {
        acc += (double)alpha;
        if (VG) visit(V3<float>{}, ts, alpha, gr);
        if (look && repeat) flat_run<false>(a, q, w, cs, ci, alpha, t, t >= kw1 ? tend : flat_lim, fS, rS, acc, 0.0);
      } else if (look) {
        t = fmaf(empty_run(a, q, w, cs, ci, t, tend, rS), fS, t);
      }
    };
    alpha_prev = __builtin_nanf("");
    if (!RUNS)
      while (t < tend) take(false);
    while (t < tend) {
      const float t0 = t;
      take(runs);
      if (__ballot(t - t0 > fS)) continue;
#pragma unroll 1
      for (int i = 0; i < rest && t < tend; ++i) take(false);
    }
  }
  for (int o = 1; o < S; o <<= 1) acc += __shfl_xor(acc, o, 64);
  return drr_value(a, (float)((a.output == RVK_DRR_RGBA8_REF ? (double)logf(256.0f * a.offset) : 0.0) + acc));
}

// Pixel of index i (0..255) of a 16x16 tile in Morton order: any aligned
// power-of-two run of indices is a compact block.
__device__ __forceinline__ void morton_pixel(int i, int& x, int& y) {
  x = (i & 1) | ((i >> 1) & 2) | ((i >> 2) & 4) | ((i >> 3) & 8);
  y = ((i >> 1) & 1) | ((i >> 2) & 2) | ((i >> 3) & 4) | ((i >> 4) & 8);
}

// Pixel of a lane when 2^ls lanes share a ray: workgroup `blk` takes part
// blk mod 2^ls of 16x16 tile blk >> ls (in the launch's super-tile order).
__device__ __forceinline__ void lanes_pixel(int blk, int stiles_x, int ls, int& x, int& y) {
  int tx, ty;
  tile_origin(blk >> ls, stiles_x, tx, ty);
  morton_pixel(((blk & ((1 << ls) - 1)) << (8 - ls)) | ((int)threadIdx.x >> ls), x, y);
  x += tx;
  y += ty;
}

// The DRR caster's pixel: exp(-L) or L, or the tinted RGBA8
// (V/...DRR...cuh:163-166).
__device__ __forceinline__ void drr_store(const DrrArgs& a, int x, int y, float v) {
  const long idx = (long)y * a.v.W + x;
  if (a.m.output == RVK_DRR_RGBA8_REF) {
    const float tw = (float)(a.tint >> 24);
    const float q = tw / (tw + v);
    const uint32_t A = to_u8(tw + (1.0f - tw / 255.0f) * v);
    const uint32_t R = to_u8(q * (float)(a.tint & 255u));
    const uint32_t G = to_u8(q * (float)((a.tint >> 8) & 255u));
    const uint32_t B = to_u8(q * (float)((a.tint >> 16) & 255u));
    ((uint32_t*)a.out)[idx] = R | (G << 8) | (B << 16) | (A << 24);
  } else {
    ((float*)a.out)[idx] = v;
  }
}

}  // namespace rvk
