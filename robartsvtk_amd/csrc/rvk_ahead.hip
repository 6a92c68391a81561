// rvk_ahead.hip -- the DRR caster of one view with enough long rays to fill
// the device with one lane each (drr_march_ahead).
#include "rvk_lanes.h"

namespace rvk {

// A 16x16-pixel tile per workgroup, the tiles (of a super-tile of 4x4) dealt
// to the XCDs in runs of 8: the march passes over runs of empty and constant
// bricks, so a band of tiles per XCD would leave the XCDs of the bands
// through air idle (256^3 CT at 1024^2 387 us, 1400^2 698 us; deals of 1, 2,
// 4, 8, 16 and 32 tiles 375 / 365 / 361 / 360 / 382 / 488 us at 1024^2).
//
// Half of a launch's waves end at once in air, and the long rays of the rest
// make little more than one round of the 8192 the device holds, 3.9 waves per
// SIMD on average with the VALU 59 % busy: the second sample in flight fills
// that.  One sample at a time against two (us, int16 CT): 256^3 of 512-sample
// rays at 1024^2 319 / 290 and 386 / 355 (two scenes), without the skip rule
// 402 / 376, at 1400x1100 350 / 327, 400^3 at 900^2 461 / 389, 360^3 at
// 1400x1100 529 / 480; 256-sample rays at 900x800 169 / 155.  Rays of 128
// samples (128^3 at 1024^2) 107 / 112: they are left to drr_kernel.
template <typename CV, bool SKIP, bool KEY>
__global__ __launch_bounds__(256) void drr_ahead_kernel(DrrArgs a) {
  int x, y;
  tile_pixel(xcd_deal(blockIdx.x, kDealLog2), a.tiles_x, x, y);
  if (x >= a.v.W || y >= a.v.H) return;
  const Ray r = form_ray(a.g, a.v, a.step_len, x, y);
  drr_store(a, x, y, drr_march_ahead<CV, SKIP, KEY>(cells_of<CV>(a.vol), a.g, a.m, r, x, y));
}

int launch_drr_ahead(const DrrArgs& a, const rvk_volume* vol, int frame, bool skip, int nblk, hipStream_t s) {
  return dispatch_frame(vol, frame, [&](auto tag) {
    using CV = decltype(tag);
    const dim3 grid(deal_grid(nblk, kDealLog2)), block(256);
    const bool key = a.v.n_key != 0;
    if (skip && key) hipLaunchKernelGGL((drr_ahead_kernel<CV, true, true>), grid, block, 0, s, a);
    else if (skip) hipLaunchKernelGGL((drr_ahead_kernel<CV, true, false>), grid, block, 0, s, a);
    else if (key) hipLaunchKernelGGL((drr_ahead_kernel<CV, false, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((drr_ahead_kernel<CV, false, false>), grid, block, 0, s, a);
    RVK_HIP(hipGetLastError());
    return (int)RVK_OK;
  });
}

}  // namespace rvk
