// rvk_lanes.h -- how a DRR launch spreads its rays, and the kernels with
// several lanes on one ray (rvk_lanes.hip).
#pragma once
#include "rvk_batch.h"

namespace rvk {

// The schedule of a precise march without termination.
struct DrrSchedule {
  int lanes;  // log2 of the lanes per ray
  bool deal;  // tiles dealt to the XCDs in runs (xcd_deal), or one band each
  bool runs;  // pass over runs of empty and constant bricks
};

// One view of `rays` rays.  The device holds 8192 waves, and 64 rays are one
// wave: below that it waits on chains of dependent samples, which more lanes
// per ray shorten; the chunks' bookkeeping costs throughput above.  Measured
// with the skip rule on int16 CT, us.  1 / 2 / 4 / 8 / 16 lanes, 256^3 of
// 512-sample rays at 64^2 261 / 157 / 80 / 43 / 24, 128^2 265 / 159 / 83 / 48 / 38;
// 128^3 of 128-sample rays at 128^2 64 / 40 / 23 / 15 / 12.  Four lanes against
// drr_ahead_kernel's one, bodies in clean air / tissue throughout: 512-sample
// rays at 400^2 120 / 168 and 137 / 156, 480^2 147 / 268 and 142 / 177, 560^2
// 189 / 309 and 130 / 180; 256-sample rays at 300^2 54 / 76 and 85 / 98, 400^2
// 82 / 93 and 86 / 89; 800-sample rays at 520^2 311 / 521 and 338 / 803, 700^2
// 472 / 830 and 489 / 828: the longer the rays, the later they cross.
// Short rays have no runs worth finding (128^3 at 200^2 24 us without, 36 with)
// and share their cells within an XCD's band, and so does the smallest launch
// (256^3 at 64^2: 24 us without runs, 29 with); many of them are drr_kernel's
// (drr_kernel / drr_ahead_kernel in clean air and with noise, 128-sample rays
// at 430^2 56 / 41 and 59 / 60, 460^2 54 / 47 and 57 / 65, 64-sample rays at
// 460^2 20 / 24 and 22 / 29, 1024^2 56 / 59 and 59 / 73; drr_kernel / four lanes,
// 64-sample rays at 200^2 18 / 14 and 20 / 18, 300^2 18 / 19 and 20 / 28).
inline DrrSchedule drr_schedule(const rvk_volume* vol, long long rays, float step_len) {
  if (rays <= 24576) return {4, false, false};
  const float n = longest_ray(vol, step_len);
  if (n >= 192.0f) return {rays <= std::max(150000.0f, 400.0f * n) ? 2 : 0, true, true};
  if (rays <= (n >= 96.0f ? 100000 : 50000)) return {2, false, false};
  return {0, n >= 96.0f && rays <= 200000, true};
}

// log2 of the lanes per ray for a plan's forward of `rays` rays in all, always
// with runs; the plan's alone, so that its results do not depend on its tuned
// schedule, tile and order (the lanes set the order of a ray's sums).  grad: the
// march also sums gradients, and every lane forms the ray's set-up and shares
// its tangents, so more lanes pay less.  Measured (us, register on f32 / int16
// volumes, 1 / 2 / 4 / 8 / 16 lanes): 200^3 1 x 128^2 133 / 78 / 51 / 40 / 39, 2 x
// 128^2 139 / 82 / 57 / 53 / 63, 2 x 200^2 151 / 92 / 74 / 77 / 84, 8 x 200^2
// 266 / 198 / 195 / 218.  Above 400 thousand rays 1 / 2 / 4 lanes, int16 CT in clean
// air: render 128^3 of 128 samples 4 x 400^2 107 / 100 / 120, with the skip rule
// 105 / 108 / 128, 16 x 200^2 137 / 116 / 136 and 135 / 126 / 140, 200^3 4 x 400^2
// 168 / 151 / 197; register 189 / 189 / 228, 180 / 187 / 221, 214 / 208 / 245 and
// 205 / 205 / 235, 255 / 242 / 313; 256^3 of 512 samples, render
// 8 x 560^2 761 / 666 / 835 (skip rule 759 / 813 / 973), 40 x 512^2 2818 / 2603 / 3371;
// register 4 x 560^2 586 / 590 / 725, 6 x 560^2 824 / 883 / 1064.
inline int batch_lanes(const rvk_volume* vol, long long rays, float step_len, bool grad) {
  if (rays <= 24576) return 4;
  if (rays <= 49152) return 3;
  if (rays <= 400000) return 2;
  const bool is_long = longest_ray(vol, step_len) >= 256.0f;
  return rays <= (!is_long ? 700000 : grad ? 1500000 : 4500000) ? 1 : 0;
}

// One view; nblk is the launch's count of 16x16-pixel tiles (launch_grid).
int launch_drr_lanes(const DrrArgs& a, const rvk_volume* vol, int frame, bool skip, int ls, int nblk, hipStream_t s);
// One view, one lane per ray, tiles dealt (rvk_ahead.hip).
int launch_drr_ahead(const DrrArgs& a, const rvk_volume* vol, int frame, bool skip, int nblk, hipStream_t s);
// A plan's forward (jac: with the pose Jacobians); persistent: the workgroups
// of that schedule, whose queues are cleared, or 0.
int launch_batch_lanes(const BatchArgs& a, const rvk_volume* vol, int frame, bool skip, bool jac, int ls,
                       unsigned persistent, hipStream_t s);

}  // namespace rvk
