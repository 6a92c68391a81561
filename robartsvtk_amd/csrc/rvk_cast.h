// rvk_cast.h -- arguments of the compositing casters.
#pragma once
#include <cmath>

#include "rvk_internal.h"
#include "rvk_march.h"

namespace rvk {

struct Cast1dArgs {
  VolGeom g;
  ViewGeom v;
  float step_len, term_T;
  int jitter;
  int n;
  rvk_tf1d_params p;
  const float* tables;
  const void* vol;
  uint32_t* out;
  float* depth;
  float* min_depth;
  float* max_depth;
  int tiles_x;
  DrrMarchArgs m;  // the frame's range bricks alone
};

struct Cast2dArgs {
  VolGeom g;
  ViewGeom v;
  float step_len, term_T;
  int jitter;
  int n;
  rvk_tf2d_params p;
  const Tf2dCell* cells;
  const Tf2dCell* kcells;
  const float4* lit;     // the cells lit with a Phong-Lambert factor of 1 (GMAG)
  const float4* klit;
  const uint32_t* occ;   // opacity bitmaps staged in LDS, or NULL
  const uint32_t* kocc;
  int occ_words;
  const uint32_t* col;   // column bitmaps (TF, then keyhole TF), staged in LDS
  int col_words;
  const void* vol;
  const uint8_t* gradmag;
  float gradmag_scale;
  uint32_t* out;
  float* depth;
  float* min_depth;
  float* max_depth;
  int tiles_x;
};

struct InExArgs {
  VolGeom g;
  ViewGeom v;
  float step_len, term_T;
  int jitter;
  int n;
  int black_keyhole;
  rvk_tf2d_params p;
  const Tf2dCell* cells;
  const uint8_t* flags;  // per cell: bit 0 composites, bit 1 excludes
  const uint32_t* occ;   // the same as two bitmaps (occ_words each), or NULL
  int occ_words;
  const uint32_t* col;   // column bitmap of bit 0 (col_words), staged in LDS
  int col_words;
  const void* vol;
  uint32_t* out;
  float* depth;
  float* min_depth;
  float* max_depth;
  int tiles_x;
  DrrMarchArgs m;  // the frame's range bricks alone
};

struct DualArgs {
  VolGeom g;
  ViewGeom v;
  float step_len, term_T;
  int jitter;
  int n;
  rvk_dual_params p;
  const Tf2dCell* cells;
  const Tf2dCell* kcells;
  const uint32_t* occ;  // opacity bitmaps staged in LDS, or NULL
  const uint32_t* kocc;
  int occ_words;
  const uint32_t* col;  // column bitmaps (TF, then keyhole TF), staged in LDS
  int col_words;
  const void* vol1;
  const void* vol2;
  uint32_t* out;
  float* depth;
  float* min_depth;
  float* max_depth;
  int tiles_x;
  DrrMarchArgs m;  // the frame's range bricks alone
};

// Ray samples of the dual caster: floor(numSteps) less the ray offset,
// truncated (V/...DualImage...cuh:66-67 store an int minus a float back in an
// int); rays the 2D caster would not march march nothing here either.
__device__ __forceinline__ int dual_step_count(float num_steps, float j) {
  if (!(num_steps > 0.0f && num_steps < 16777216.0f)) return 0;
  return (int)((float)(int)floorf(num_steps) - j);
}

inline void set_ranges(DrrMarchArgs& m, const rvk_volume* vol, int frame) {
  m.ranges = vol->ranges[frame];
  m.rbx = vol->nrb[0];
  m.rby = vol->nrb[1];
  m.groups = vol->range_groups(frame);
  m.rgx = vol->nrg(0);
  m.rgy = vol->nrg(1);
}

// What the four-lane casters do not march: the reference's incremental
// positions, a jump over a keyhole window, and a termination threshold above
// 1, which ends a ray on its first contributing sample, a step back included.
inline bool quad_ok(const rvk_view* v, const rvk_march_params* m) {
  return m->precise && m->term_T <= 1.0f && v->n_keyhole_planes == 0;
}

// Whether four lanes per ray pay.  A quad forms its ray four times over
// (about 0.055 ns a ray on the device) and takes samples in chunks of four; it
// gains on every gather, the more the further apart a one-lane wave's rays
// are.  So one lane wins where pixels are many per voxel column (rho) and
// rays composite few samples: at most k, ln(term) over ln(1 - the smallest
// opacity of the table).  Measured over 64^3 to 512^3 volumes, 256^2 to
// 3840x2160 views and opacities of 0.02 to 1 (one lane / four, us): tables of
// opacity 1, 128^3 at 1400x1100 (rho 94) 1D 135 / 263, unshaded 122 / 217, 2D
// 148 / 233, with gradient magnitude 135 / 190, dual 160 / 276, in/ex
// 164 / 302; 256^3 at 1280x1024 (rho 20, k 12) 1D 256 / 350, 2D 308 / 350;
// opacity 0.1 (k 39) at rho 94 1D 402 / 454, 2D 434 / 415; but ramps (k
// without bound) 128^3 at rho 94 1D 566 / 427, 2D 1670 / 1243, and 400^3 of
// opacity 1 at rho 10 524 / 476: the larger the cells beside the 256 MiB
// cache, the later.  At rho above 3.5 samples per ray (64^3 at 1400x1100) the
// set-up alone decides: 1D 252 / 258, gradient magnitude 216 / 259.  The
// unshaded 1D sample is the cheapest: for it also at above 40 N^2 rays of N
// samples (ramps, 64^3 of 64 samples at 400^2 31 / 36, 128^3 of 128 at 1024x768
// 102 / 121, of 256 176 / 159).  `share` is k / rho at the crossing, by caster.
inline bool quad_pays(const rvk_volume* v, const rvk_view* view, float step_len, float least, float term, float share,
                      bool unshaded = false) {
  const double rays = (double)view->width * view->height;
  const double bytes = 8.0 * (double)dtype_size(v->dtype) * (double)v->n_cells;
  const double rho = rays / std::pow((double)v->dims[0] * v->dims[1] * v->dims[2], 2.0 / 3.0);
  if (rays < 100000.0) return true;
  const double n = longest_ray(v, step_len);
  if (rho >= 3.5 * n || (unshaded && rays >= 40.0 * n * n)) return false;
  if (rho < 12.0 * std::max(1.0, bytes / (double)(256 << 20))) return true;
  const double k = least >= 1.0f ? 1.0 : term > 0.0f ? std::log((double)term) / std::log1p(-(double)least) : 1e30;
  return k > share * rho;
}
constexpr float kQuadShare1d = 1.5f, kQuadShareUnshaded = 8.0f, kQuadShareGradmag = 1.5f, kQuadShareGradient = 0.5f;

constexpr int kQuadDealLog2 = 4;  // workgroups of 8x8 pixels in runs of a 64x16 strip

// The same casters with four lanes per ray (rvk_quad.h); nblk is the launch's
// count of 16x16-pixel tiles.
int launch_quad_1d(const Cast1dArgs& a, const rvk_volume* vol, int frame, bool skip, bool grad, size_t lds, int nblk,
                   hipStream_t s);
int launch_quad_2d(const Cast2dArgs& a, const rvk_volume* vol, int frame, bool skip, bool gradmag, size_t lds,
                   int nblk, hipStream_t s);
int launch_quad_inex(const InExArgs& a, const rvk_volume* vol, int frame, bool skip, size_t lds, int nblk,
                     hipStream_t s);
int launch_quad_dual(const DualArgs& a, const rvk_volume* vol1, const rvk_volume* vol2, int frame, bool skip,
                     size_t lds, int nblk, hipStream_t s);

}  // namespace rvk
