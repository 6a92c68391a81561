// rvk_cast.h -- arguments of the compositing casters.
#pragma once
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

constexpr int kQuadDealLog2 = 4;  // workgroups of 8x8 pixels in runs of a 32x32 square

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
