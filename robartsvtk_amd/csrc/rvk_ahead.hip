// rvk_ahead.hip -- the DRR caster of one view with enough long rays to fill
// the device with one lane each (drr_march_ahead).
#include "rvk_lanes.h"

namespace rvk {

// A 16x16-pixel tile per workgroup, the tiles (of a super-tile of 4x4) dealt
// to the XCDs in runs of 8: the march passes over runs of empty and constant
// bricks, so a band of tiles per XCD would leave the XCDs of the bands
// through air idle (256^3 CT of 512-sample rays, us, in bands / dealt in runs of
// 1, 2, 4, 8, 16 and 32 tiles: at 1024^2 260 / 240 / 240 / 232 / 231 / 235 / 307,
// at 1400^2 472 / 372 / 368 / 366 / 364 / 364 / 362; 400^3 at 1024^2
// 669 / 556 / 553 / 554 / 568 / 596 / 822).
//
// Half of a launch's waves end at once in air, and the long rays of the rest
// make little more than one round of the 8192 the device holds: the second
// sample in flight fills the wait for the first.  Registers for 8 waves per
// SIMD (7 without the bound: 390 / 363 us at 1400^2).  drr_kernel against
// this, us, for three bodies -- CT in clean air, in air with noise (values that
// contribute or not at random), tissue filling the volume: 256^3 at 560^2
// 261 / 131, 392 / 348, 256 / 182; at 1024^2 453 / 232, 553 / 604, 451 / 444; at
// 1400^2 833 / 364, 869 / 861, 831 / 735; at 2048^2 1531 / 696, 1588 / 1657,
// 1547 / 1468; 400^3 at 1024^2 1684 / 568, 2069 / 2046, 1149 / 881.  Without the
// skip rule 256^3 at 1024^2 437 / 217, 434 / 418, 438 / 402.
template <typename CV, bool SKIP, bool KEY>
__global__ __launch_bounds__(256, 8) void drr_ahead_kernel(DrrArgs a) {
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
