// rvk_runtime.hip -- contexts, volumes, transfer functions and errors.
//
// Replaces, on HIP:
//   C/CudaObject.cxx:55-212 and C/vtkCudaDeviceManager.cxx:50-443 (device and
//     stream per object; here one rvk_ctx = one device + one stream);
//   V/CUDA_vtkCudaVolumeMapper_renderAlgo.cu:584-651 (CUDA_castBuffer: host
//     copy + widening to float) and the *_loadImageInfo 3D-array uploads
//     (e.g. V/CUDA_vtkCuda1DVolumeMapper_renderAlgo.cuh:409-443): volumes stay
//     in their native type and are relaid out on the device into cells that
//     hold each trilinear 2x2x2 footprint whole (8x the voxel bytes);
//   the TF loadTextures functions (V/CUDA_vtkCuda1DVolumeMapper_renderAlgo.cuh:324-372,
//     V/CUDA_vtkCuda2DVolumeMapper_renderAlgo.cuh:589-651).
#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <type_traits>
#include <vector>

#include "rvk_internal.h"

namespace rvk {

static thread_local std::string g_last_error;

int fail(int status, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return status;
}

int hip_fail(hipError_t e, const char* what) {
  const int st = (e == hipErrorOutOfMemory) ? RVK_ERR_OUT_OF_MEMORY
                 : (e == hipErrorNoDevice || e == hipErrorInvalidDevice) ? RVK_ERR_NO_DEVICE
                                                                          : RVK_ERR_HIP;
  return fail(st, "%s failed: %s", what, hipGetErrorString(e));
}

size_t dtype_size(int dtype) {
  switch (dtype) {
    case RVK_U8: case RVK_I8: return 1;
    case RVK_U16: case RVK_I16: return 2;
    case RVK_U32: case RVK_I32: case RVK_F32: return 4;
    default: return 0;
  }
}

// V/vtkCudaVolumeInformationHandler.cxx:80-108
VolGeom vol_geom(const rvk_volume* v) {
  VolGeom g;
  for (int a = 0; a < 3; ++a) {
    g.n[a] = v->dims[a];
    g.srecip[a] = (float)(0.5 / v->spacing[a]);
    g.sp[a] = (float)v->spacing[a];
    g.bounds[2 * a] = 0.0f;
    g.bounds[2 * a + 1] = (float)v->dims[a] - 1.0f;
  }
  if (v->layout == kCellLayoutPair8) {
    // x-pair bricks: the brick grid's row length and rows per slab
    g.cys = (uint32_t)v->ncb[0];
    g.crows = (uint32_t)v->ncb[1];
    g.czs = (uint32_t)v->ncb[0] * (uint32_t)v->ncb[1];
    return g;
  }
  const uint32_t bc = 1u << (3 * v->layout);  // cells per brick
  g.cys = bc * (uint32_t)v->ncb[0];
  g.czs = bc * (uint32_t)v->ncb[0] * (uint32_t)v->ncb[1];
  g.crows = (uint32_t)v->ncb[1];
  return g;
}

float min_spacing(const rvk_volume* v) {
  return (float)std::fmin(v->spacing[0], std::fmin(v->spacing[1], v->spacing[2]));
}

ViewGeom view_geom(const rvk_view* v) {
  ViewGeom g;
  std::memcpy(g.m, v->view_to_voxels, sizeof(g.m));
  g.W = v->width;
  g.H = v->height;
  g.flipped = v->flipped;
  g.n_clip = v->n_clip_planes;
  g.n_key = v->n_keyhole_planes;
  std::memcpy(g.clip, v->clip_planes, sizeof(g.clip));
  std::memcpy(g.key, v->keyhole_planes, sizeof(g.key));
  g.zbuf = v->zbuffer;
  g.zbw = v->zb_width;
  g.zbh = v->zb_height;
  return g;
}

int check_view(const rvk_view* v) {
  if (!v) return fail(RVK_ERR_INVALID_ARGUMENT, "view is NULL");
  if (v->width <= 0 || v->height <= 0 || v->width > 16384 || v->height > 16384)
    return fail(RVK_ERR_INVALID_ARGUMENT, "view size %dx%d out of range [1,16384]", v->width, v->height);
  if (v->n_clip_planes < 0 || v->n_clip_planes > 6 || v->n_keyhole_planes < 0 || v->n_keyhole_planes > 6)
    return fail(RVK_ERR_INVALID_ARGUMENT, "plane counts must be within 0..6");
  if (v->zbuffer && (v->zb_width <= 0 || v->zb_height <= 0))
    return fail(RVK_ERR_INVALID_ARGUMENT, "z-buffer given without a positive size");
  return RVK_OK;
}

int check_frame(const rvk_volume* v, int frame) {
  if (!v) return fail(RVK_ERR_INVALID_ARGUMENT, "volume is NULL");
  if (frame < 0 || frame >= v->n_frames)
    return fail(RVK_ERR_INVALID_ARGUMENT, "frame %d out of range [0,%d)", frame, v->n_frames);
  if (!v->frames[frame]) return fail(RVK_ERR_NOT_READY, "frame %d has no data", frame);
  return RVK_OK;
}

int ensure_scratch(rvk_ctx* ctx, size_t bytes) {
  if (ctx->scratch_bytes >= bytes) return RVK_OK;
  if (ctx->scratch) {
    RVK_HIP(hipStreamSynchronize(ctx->stream));
    RVK_HIP(hipFree(ctx->scratch));
    ctx->scratch = nullptr;
    ctx->scratch_bytes = 0;
  }
  RVK_HIP(hipMalloc(&ctx->scratch, bytes));
  ctx->scratch_bytes = bytes;
  return RVK_OK;
}

// ---------------------------------------------------------------------------
// Linear (x fastest) -> cells.  One thread per cell: it gathers the cell's 8
// clamped voxels and writes them as one vector.  Cells past [0, n+1] (brick
// padding) are never sampled; they repeat the nearest edge.
template <typename VT> struct CellVec;
template <> struct CellVec<uint8_t> { using T = uint2; };
template <> struct CellVec<int8_t> { using T = uint2; };
template <> struct CellVec<uint16_t> { using T = uint4; };
template <> struct CellVec<int16_t> { using T = uint4; };

// DIFF stores each x-pair (a, b) as (a, b - a): exactly, as a 16-bit two's
// complement difference (the frame's value range is below 32768) or, for
// float, as the rounded difference the trilinear lerp computes from (a, b).
// HALF (16-bit DIFF cells): 1 stores the bases as binary16, 2 the
// differences too (both exact for the frames given those encodings).
template <typename VT, int L, bool DIFF = false, int HALF = 0>
__global__ __launch_bounds__(256) void cell_relayout_kernel(const VT* __restrict__ src, VT* __restrict__ dst, int nx,
                                                            int ny, int nz, int ncbx, int ncby, long long n_cells) {
  using O = CellOrder<L>;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n_cells) return;
  const long long b = c / O::kCells;
  const int o = (int)(c % O::kCells);
  const int bx = (int)(b % ncbx);
  const int by = (int)((b / ncbx) % ncby);
  const int bz = (int)(b / ((long long)ncbx * ncby));
  const int m = O::kEdge - 1;
  const int cx = bx * O::kEdge + (o & m);
  const int cy = by * O::kEdge + ((o >> L) & m);
  const int cz = bz * O::kEdge + (o >> (2 * L));
  alignas(16) VT v[8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const int i = min(max(cx - 1 + (q & 1), 0), nx - 1);
    const int j = min(max(cy - 1 + ((q >> 1) & 1), 0), ny - 1);
    const int k = min(max(cz - 1 + (q >> 2), 0), nz - 1);
    v[q] = src[(long long)i + (long long)j * nx + (long long)k * nx * ny];
  }
  if (DIFF) {
#pragma unroll
    for (int q = 1; q < 8; q += 2) {
      if constexpr (sizeof(VT) == 2) v[q] = (VT)(uint16_t)((int)v[q] - (int)v[q - 1]);
      else v[q] = v[q] - v[q - 1];
    }
  }
  if constexpr (HALF > 0 && sizeof(VT) == 2) {
    // bases in [-2048, 2048]: exact as binary16
#pragma unroll
    for (int q = 0; q < 8; q += 2) v[q] = (VT)__builtin_bit_cast(uint16_t, (_Float16)(float)(int)v[q]);
    if constexpr (HALF > 1) {
#pragma unroll
      for (int q = 1; q < 8; q += 2)
        v[q] = (VT)__builtin_bit_cast(uint16_t, (_Float16)(float)(int)(int16_t)(uint16_t)v[q]);
    }
  }
  VT* out = dst + c * 8;
  if constexpr (sizeof(VT) == 4) {
    reinterpret_cast<uint4*>(out)[0] = *reinterpret_cast<const uint4*>(&v[0]);
    reinterpret_cast<uint4*>(out)[1] = *reinterpret_cast<const uint4*>(&v[4]);
  } else {
    *reinterpret_cast<typename CellVec<VT>::T*>(out) = *reinterpret_cast<const typename CellVec<VT>::T*>(&v[0]);
  }
}

// Linear -> x-pair bricks.  One thread per stored pair: brick (bx, by, bz),
// slab lz and row ly (voxel rows 8b - 1 + l, clamped) and pair lx, holding
// voxels x = 8 bx + lx - 1 and x + 1 (clamped), encoded like a cell's pairs.
template <typename VT, bool DIFF = false, int HALF = 0>
__global__ __launch_bounds__(256) void pair_relayout_kernel(const VT* __restrict__ src, VT* __restrict__ dst, int nx,
                                                            int ny, int nz, int nbx, int nby, long long n_pairs) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n_pairs) return;
  const long long b = p / kPairBrick;
  const int r = (int)(p % kPairBrick);
  const int lz = r / kPairSlab, ly = (r / kPairRow) % 9, lx = r % kPairRow;
  const int bx = (int)(b % nbx), by = (int)((b / nbx) % nby), bz = (int)(b / ((long long)nbx * nby));
  const int x = bx * 8 + lx - 1;
  const int j = min(max(by * 8 + ly - 1, 0), ny - 1);
  const int k = min(max(bz * 8 + lz - 1, 0), nz - 1);
  const long long row = (long long)j * nx + (long long)k * nx * ny;
  VT a = src[row + min(max(x, 0), nx - 1)];
  VT c = src[row + min(max(x + 1, 0), nx - 1)];
  if (DIFF) {
    if constexpr (sizeof(VT) == 2) c = (VT)(uint16_t)((int)c - (int)a);
    else c = c - a;
  }
  if constexpr (HALF > 0 && sizeof(VT) == 2) {
    a = (VT)__builtin_bit_cast(uint16_t, (_Float16)(float)(int)a);
    if constexpr (HALF > 1) c = (VT)__builtin_bit_cast(uint16_t, (_Float16)(float)(int)(int16_t)(uint16_t)c);
  }
  dst[2 * p] = a;
  dst[2 * p + 1] = c;
}

// Gradient magnitude by central differences at voxel centres, the value the
// reference's on-the-fly gradient takes there (tex3D at p +- 1 with clamp,
// times 0.5/spacing; V/CUDA_vtkCuda2DVolumeMapper_renderAlgo.cuh:263-271),
// quantised to u8 as round(|g| / scale), written x-fastest.
template <typename CV>
__global__ __launch_bounds__(256) void gradmag_kernel(CV vol, uint8_t* __restrict__ out, VolGeom g, float inv_scale,
                                                      long long total) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int i = (int)(e % g.n[0]);
  const int j = (int)((e / g.n[0]) % g.n[1]);
  const int k = (int)(e / ((long long)g.n[0] * g.n[1]));
  auto at = [&](int x, int y, int z) {
    x = min(max(x, 0), g.n[0] - 1);
    y = min(max(y, 0), g.n[1] - 1);
    z = min(max(z, 0), g.n[2] - 1);
    return load_voxel(vol, g, x, y, z);
  };
  const float gx = (at(i + 1, j, k) - at(i - 1, j, k)) * g.srecip[0];
  const float gy = (at(i, j + 1, k) - at(i, j - 1, k)) * g.srecip[1];
  const float gz = (at(i, j, k + 1) - at(i, j, k - 1)) * g.srecip[2];
  const float q = sqrtf(gx * gx + gy * gy + gz * gz) * inv_scale;
  out[e] = (uint8_t)fminf(rintf(q), 255.0f);
}

template <typename VT, int L, bool DIFF = false, int HALF = 0>
static int launch_relayout(rvk_volume* v, const void* dsrc, void* dst) {
  if constexpr (L == kCellLayoutPair8) {
    const long long total = (long long)v->n_cells * 4;  // pairs: 8 voxels per storage unit
    const int blocks = (int)((total + 255) / 256);
    hipLaunchKernelGGL((pair_relayout_kernel<VT, DIFF, HALF>), dim3(blocks), dim3(256), 0, v->ctx->stream,
                       (const VT*)dsrc, (VT*)dst, v->dims[0], v->dims[1], v->dims[2], v->ncb[0], v->ncb[1], total);
  } else {
    const long long total = (long long)v->n_cells;
    const int blocks = (int)((total + 255) / 256);
    hipLaunchKernelGGL((cell_relayout_kernel<VT, L, DIFF, HALF>), dim3(blocks), dim3(256), 0, v->ctx->stream,
                       (const VT*)dsrc, (VT*)dst, v->dims[0], v->dims[1], v->dims[2], v->ncb[0], v->ncb[1], total);
  }
  RVK_HIP(hipGetLastError());
  return RVK_OK;
}

// Value statistics of a frame in one pass over its native voxels.
//
// Ranges: (min, max) of the voxels each range brick's cells reach, i.e.
// voxels [8b - 1, 8b + 7] per axis, clamped into the volume.  The y and z
// lerps round the difference of their operands, so an interpolated value may
// leave the voxels' range by a few ulp of the largest magnitude: the bounds
// of a non-constant brick are widened by 2^-20 of it.  A constant brick
// interpolates its value exactly and keeps min == max.  A brick with a
// non-finite voxel gets (-inf, +inf): no run is ever taken through it.
//
// Encoding (16-bit frames, stats != NULL): the frame's value range and
// whether some x-neighbour difference is not exact in binary16 (|d| > 2048
// and odd; used only for frames within [-2048, 2048], whose differences are
// at most 4096) decide the cell encoding.
//
// One wave per 8 bricks of a brick row: lane l takes column x = 64 c + l
// through the bricks' 81 voxel rows and reads it with its left neighbour, so
// an aligned group of 8 lanes covers a brick's 9 columns; the loads of a row
// are one or two lines, 9 rows in flight (loaded into registers before any is
// used; with the compares between the loads 256^3 f32 took 79 us).  Bound by
// that load chain: 250 x 250 x 181 int16 11.9 us, 256^3 f32 21 us (3.2 TB/s).
// One thread per brick, reading 729 strided voxels, took 79 and 128 us, and
// the int16 totals, every wave's min and max on one pair of addresses
// (16384 waves), 380 us more.  The totals go to kStatSlots slots on lines of
// their own, the blocks dealt over them.
constexpr int kStatSlots = 64;
constexpr int kStatStride = 16;  // ints: a 64-byte line per slot
constexpr size_t kStatBytes = sizeof(int) * kStatSlots * kStatStride;

__global__ __launch_bounds__(kStatSlots) void stats_init_kernel(int* stats) {
  int* s = stats + threadIdx.x * kStatStride;
  s[0] = 0x7fffffff;
  s[1] = -0x7fffffff - 1;
  s[2] = 0;
}

template <typename VT>
__global__ __launch_bounds__(256) void frame_stats_kernel(const VT* __restrict__ src, int nx, int ny, int nz, int rbx,
                                                          int rby, int rbz, float2* __restrict__ out, int* stats) {
  constexpr bool kInt16 = sizeof(VT) == 2;
  const int lane = threadIdx.x & 63;
  const int chunks = (rbx + 7) / 8;
  const int task = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const float inf = __builtin_huge_valf();
  float lo = inf, hi = -inf;
  int finite = 1;
  int odd = 0;
  const bool has_task = task < chunks * rby * rbz;
  if (has_task) {
    const int c = task % chunks, by = (task / chunks) % rby, bz = task / (chunks * rby);
    const int col = c * 64 + lane;
    const int x = min(col, nx - 1), xl = min(max(col - 1, 0), nx - 1);
    for (int k = 0; k < 9; ++k) {
      const int z = min(max(bz * kRangeEdge - 1 + k, 0), nz - 1);
      const VT* slab = src + (size_t)z * ny * nx;
      VT rv[9], rl[9];  // the 9 rows' loads are issued together
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const VT* row = slab + (size_t)min(max(by * kRangeEdge - 1 + j, 0), ny - 1) * nx;
        rv[j] = row[x];
        rl[j] = row[xl];
      }
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const float v = (float)rv[j], l = (float)rl[j];
        if constexpr (std::is_same<VT, float>::value) finite = finite & (int)isfinite(v) & (int)isfinite(l);
        lo = fminf(lo, fminf(v, l));
        hi = fmaxf(hi, fmaxf(v, l));
        if constexpr (kInt16) {
          const int d = abs((int)rv[j] - (int)rl[j]);
          odd |= (int)(d > 2048 && (d & 1));
        }
      }
    }
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) {
      lo = fminf(lo, __shfl_xor(lo, o, 64));
      hi = fmaxf(hi, __shfl_xor(hi, o, 64));
    }
    const unsigned long long bad = __ballot(!finite);
    const int bx = c * 8 + (lane >> 3);
    if ((lane & 7) == 0 && bx < rbx) {
      const float w = hi > lo ? fmaxf(fabsf(lo), fabsf(hi)) * 0x1p-20f : 0.0f;
      const bool ok = ((bad >> lane) & 0xffull) == 0ull;
      out[((size_t)bz * rby + by) * rbx + bx] = ok ? make_float2(lo - w, hi + w) : make_float2(-inf, inf);
    }
  }
  if constexpr (kInt16) {
    // every voxel is in some brick: the bricks' extremes are the frame's
    __shared__ int s_lo[4], s_hi[4], s_odd[4];
#pragma unroll
    for (int o = 8; o < 64; o <<= 1) {
      lo = fminf(lo, __shfl_xor(lo, o, 64));
      hi = fmaxf(hi, __shfl_xor(hi, o, 64));
    }
    const bool any_odd = __ballot(odd) != 0ull;
    if (lane == 0) {
      const int w = threadIdx.x >> 6;
      s_lo[w] = has_task ? (int)lo : 0x7fffffff;
      s_hi[w] = has_task ? (int)hi : -0x7fffffff - 1;
      s_odd[w] = any_odd;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      int* s = stats + (blockIdx.x % kStatSlots) * kStatStride;
      atomicMin(s, min(min(s_lo[0], s_lo[1]), min(s_lo[2], s_lo[3])));
      atomicMax(s + 1, max(max(s_hi[0], s_hi[1]), max(s_hi[2], s_hi[3])));
      if (s_odd[0] | s_odd[1] | s_odd[2] | s_odd[3]) atomicMax(s + 2, 1);
    }
  }
}

// Ranges of the groups of 4^3 range bricks, one wave per group.  (Groups of
// constant bricks of one value are constant; a brick's widened bounds stay.)
__global__ __launch_bounds__(64) void range_groups_kernel(const float2* __restrict__ ranges, int rbx, int rby, int rbz,
                                                          int gx, int gy, float2* __restrict__ groups) {
  const int g = blockIdx.x, l = threadIdx.x;
  const int bx = min((g % gx) * 4 + (l & 3), rbx - 1), by = min((g / gx % gy) * 4 + ((l >> 2) & 3), rby - 1);
  const int bz = min(g / (gx * gy) * 4 + (l >> 4), rbz - 1);
  float2 r = ranges[((size_t)bz * rby + by) * rbx + bx];
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    r.x = fminf(r.x, __shfl_xor(r.x, o, 64));
    r.y = fmaxf(r.y, __shfl_xor(r.y, o, 64));
  }
  if (l == 0) groups[g] = r;
}

// Binary16 cells -> difference cells: each x-pair's base (and, for
// HalfPair cells, its difference) becomes the 16-bit integer it holds
// (exact); an int16 difference stays.
__global__ __launch_bounds__(256) void half_to_diff_kernel(uint32_t* __restrict__ w, long long n_words, int pair) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n_words) return;
  const uint32_t q = w[i];
  const int a = (int)(float)__builtin_bit_cast(_Float16, (uint16_t)(q & 0xffffu));
  const uint32_t d = pair ? (uint32_t)(int)(float)__builtin_bit_cast(_Float16, (uint16_t)(q >> 16)) << 16
                          : q & 0xffff0000u;
  w[i] = d | ((uint32_t)a & 0xffffu);
}

int frame_drop_half(const rvk_volume* cv, int frame, hipStream_t s) {
  if (cv->enc[frame] != kEncHalf && cv->enc[frame] != kEncHalfPair) return RVK_OK;
  rvk_volume* v = const_cast<rvk_volume*>(cv);
  const long long n = (long long)v->n_cells * 4;  // 8 x 16-bit per cell
  hipLaunchKernelGGL(half_to_diff_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s,
                     (uint32_t*)v->frames[frame], n, (int)(cv->enc[frame] == kEncHalfPair));
  RVK_HIP(hipGetLastError());
  v->enc[frame] = kEncDiff;
  return RVK_OK;
}

// The frame's range bricks from its native voxels on the device, and for
// 16-bit frames its value range and odd-difference flag (waits for them).
// The slots of the totals follow the frame's ranges in one allocation.
template <typename VT>
static int launch_stats(rvk_volume* v, int frame, const void* dsrc) {
  const int tasks = (v->nrb[0] + 7) / 8 * v->nrb[1] * v->nrb[2];
  hipStream_t s = v->ctx->stream;
  int* stats = v->frame_stats(frame);
  if (sizeof(VT) == 2) hipLaunchKernelGGL(stats_init_kernel, dim3(1), dim3(kStatSlots), 0, s, stats);
  hipLaunchKernelGGL((frame_stats_kernel<VT>), dim3((tasks + 3) / 4), dim3(256), 0, s, (const VT*)dsrc, v->dims[0],
                     v->dims[1], v->dims[2], v->nrb[0], v->nrb[1], v->nrb[2], v->ranges[frame], stats);
  hipLaunchKernelGGL(range_groups_kernel, dim3((unsigned)v->n_range_groups()), dim3(64), 0, s, v->ranges[frame],
                     v->nrb[0], v->nrb[1], v->nrb[2], v->nrg(0), v->nrg(1), v->range_groups(frame));
  RVK_HIP(hipGetLastError());
  return RVK_OK;
}

static int frame_stats(rvk_volume* v, int frame, const void* dsrc, int& lo, int& hi, bool& odd_diff) {
  if (!v->ranges[frame]) {
    void* q = nullptr;
    RVK_HIP(hipMalloc(&q, sizeof(float2) * (v->n_range_bricks() + v->n_range_groups()) + kStatBytes));
    v->ranges[frame] = (float2*)q;
  }
  int rc = RVK_OK;
  switch (v->dtype) {
    case RVK_U8: return launch_stats<uint8_t>(v, frame, dsrc);
    case RVK_I8: return launch_stats<int8_t>(v, frame, dsrc);
    case RVK_U32: return launch_stats<uint32_t>(v, frame, dsrc);
    case RVK_I32: return launch_stats<int32_t>(v, frame, dsrc);
    case RVK_F32: return launch_stats<float>(v, frame, dsrc);
    case RVK_U16: rc = launch_stats<uint16_t>(v, frame, dsrc); break;
    default: rc = launch_stats<int16_t>(v, frame, dsrc); break;
  }
  if (rc) return rc;
  int h[kStatSlots * kStatStride];
  RVK_HIP(hipMemcpyAsync(h, v->frame_stats(frame), sizeof(h), hipMemcpyDeviceToHost, v->ctx->stream));
  RVK_HIP(hipStreamSynchronize(v->ctx->stream));
  lo = h[0];
  hi = h[1];
  odd_diff = h[2] != 0;
  for (int i = 1; i < kStatSlots; ++i) {
    lo = std::min(lo, h[i * kStatStride]);
    hi = std::max(hi, h[i * kStatStride + 1]);
    odd_diff = odd_diff || h[i * kStatStride + 2] != 0;
  }
  return RVK_OK;
}

template <typename CV>
static int launch_gradmag(rvk_volume* v, int frame, float inv_scale, uint8_t* linear) {
  using VT = typename CV::value_type;
  const long long total = (long long)v->dims[0] * v->dims[1] * v->dims[2];
  const int blocks = (int)((total + 255) / 256);
  hipLaunchKernelGGL((gradmag_kernel<CV>), dim3(blocks), dim3(256), 0, v->ctx->stream,
                     CV{(const VT*)v->frames[frame]}, linear, vol_geom(v), inv_scale, total);
  RVK_HIP(hipGetLastError());
  return launch_relayout<uint8_t, CV::kLog2>(v, linear, v->gradmag[frame]);
}

// Cell grid and count of a volume in its cell order; fails when the cell
// addressing limits (slab < 2^24 cells, plain order: rows < 2^24, < 2^32
// cells) are exceeded.
static int size_cells(rvk_volume* v) {
  const int edge = 1 << v->layout;
  for (int a = 0; a < 3; ++a) v->ncb[a] = (v->dims[a] + 2 + edge - 1) / edge;
  for (int a = 0; a < 3; ++a) v->nrb[a] = (v->dims[a] + 2 + kRangeEdge - 1) / kRangeEdge;
  if (v->layout == kCellLayoutPair8) {
    // storage units of 8 voxels: a brick's 648 pairs are 162 of them
    const size_t nb = (size_t)v->ncb[0] * v->ncb[1] * v->ncb[2];
    v->n_cells = nb * (kPairBrick / 4);
    if (nb * kPairBrick > (size_t)0xffffffffu || (size_t)v->ncb[0] * v->ncb[1] >= ((size_t)1 << 24))
      return fail(RVK_ERR_INVALID_ARGUMENT, "volume too large for 32-bit x-pair indices");
    return RVK_OK;
  }
  const size_t bc = (size_t)1 << (3 * v->layout);
  v->n_cells = bc * v->ncb[0] * v->ncb[1] * v->ncb[2];
  const size_t slab = bc * v->ncb[0] * v->ncb[1];
  if (slab >= ((size_t)1 << 24))  // cell addressing multiplies with 24-bit operands
    return fail(RVK_ERR_INVALID_ARGUMENT, "volume x/y extent too large: %zu cells per z slab, limit 2^24 - 1", slab);
  if (v->layout == kCellLayoutPlain && (size_t)v->ncb[1] * v->ncb[2] >= ((size_t)1 << 24))
    return fail(RVK_ERR_INVALID_ARGUMENT, "volume y/z extent too large for x-fastest cells: %zu cell rows, limit 2^24 - 1",
                (size_t)v->ncb[1] * v->ncb[2]);
  if (v->n_cells > (size_t)0xffffffffu)
    return fail(RVK_ERR_INVALID_ARGUMENT, "volume too large: %zu cells exceed 32-bit cell indices", v->n_cells);
  return RVK_OK;
}

// Default cell order: bricks once the cell volume passes 1 GiB (large
// volumes, where the plain order's long strides across rows and slabs miss
// the caches), plain x-fastest order below.
static int default_layout(const int32_t dims[3], int dtype) {
  const double bytes = 8.0 * (double)dtype_size(dtype) * (dims[0] + 2.0) * (dims[1] + 2.0) * (dims[2] + 2.0);
  const double rows = (dims[1] + 2.0) * (dims[2] + 2.0);
  return (bytes > (double)(1ull << 30) || rows >= (double)(1 << 24)) ? kCellLayoutBrick4 : kCellLayoutPlain;
}

}  // namespace rvk

using namespace rvk;

// ---------------------------------------------------------------------------
// Cells -> x-fastest native voxels: voxel (i, j, k) is the first slot of
// cell (i+1, j+1, k+1) in every layout and encoding (the base of its x-pair,
// stored exactly; binary16 bases hold integers in [-2048, 2048]).
template <typename CV, typename VT>
__global__ __launch_bounds__(256) void extract_voxels_kernel(const void* cell_data, VolGeom g, VT* __restrict__ out,
                                                             long long total) {
  const CV cells = cells_of<CV>(cell_data);
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= total) return;
  const int i = (int)(e % g.n[0]);
  const int j = (int)((e / g.n[0]) % g.n[1]);
  const int k = (int)(e / ((long long)g.n[0] * g.n[1]));
  using T = typename CV::value_type;
  constexpr int L = CV::kLog2;
  const T raw = cells.d[(size_t)CellOrder<L>::index(g, i + 1, j + 1, k + 1) * CellStride<L>::k];
  if constexpr (std::is_same<T, Half16>::value || std::is_same<T, HalfPair>::value) out[e] = (VT)(int)(float)raw;
  else out[e] = (VT)raw;
}

// ---------------------------------------------------------------------------
// Streaming-read probe: every 16-byte word of a buffer read once, coalesced,
// with a grid that fills the device.  The loads feed an xor that is stored
// only on a match no real buffer produces, so they are not dropped.
namespace rvk {
__global__ __launch_bounds__(256) void stream_read_kernel(const uint4* __restrict__ p, size_t n, uint32_t* sink) {
  uint32_t acc = 0;
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (; i + 3 * stride < n; i += 4 * stride) {
    const uint4 a = p[i], b = p[i + stride], c = p[i + 2 * stride], d = p[i + 3 * stride];
    acc ^= a.x ^ a.y ^ a.z ^ a.w ^ b.x ^ b.y ^ b.z ^ b.w ^ c.x ^ c.y ^ c.z ^ c.w ^ d.x ^ d.y ^ d.z ^ d.w;
  }
  for (; i < n; i += stride) {
    const uint4 a = p[i];
    acc ^= a.x ^ a.y ^ a.z ^ a.w;
  }
  if (acc == 0x9e3779b9u && sink) sink[0] = acc;
}
}  // namespace rvk

extern "C" {

const char* rvk_last_error_string(void) { return g_last_error.c_str(); }

const char* rvk_status_string(int status) {
  switch (status) {
    case RVK_OK: return "ok";
    case RVK_ERR_INVALID_ARGUMENT: return "invalid argument";
    case RVK_ERR_NO_DEVICE: return "no device";
    case RVK_ERR_HIP: return "HIP runtime error";
    case RVK_ERR_OUT_OF_MEMORY: return "out of device memory";
    case RVK_ERR_NOT_READY: return "not ready";
    case RVK_ERR_UNSUPPORTED: return "unsupported";
    default: return "unknown status";
  }
}

int rvk_version(void) { return RVK_VERSION; }

int rvk_device_count(int* count) {
  if (!count) return fail(RVK_ERR_INVALID_ARGUMENT, "count is NULL");
  *count = 0;
  hipError_t e = hipGetDeviceCount(count);
  if (e == hipErrorNoDevice) { *count = 0; return RVK_OK; }
  RVK_HIP(e);
  return RVK_OK;
}

static int ctx_create(int device, bool borrow, void* stream, rvk_ctx** out) {
  if (!out) return fail(RVK_ERR_INVALID_ARGUMENT, "out is NULL");
  *out = nullptr;
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n == 0) return fail(RVK_ERR_NO_DEVICE, "no HIP device available");
  if (device < 0 || device >= n) return fail(RVK_ERR_NO_DEVICE, "device %d out of range [0,%d)", device, n);
  RVK_HIP(hipSetDevice(device));
  rvk_ctx* c = new rvk_ctx();
  c->device = device;
  if (borrow) {
    c->stream = (hipStream_t)stream;  // NULL is the device's default stream
  } else {
    e = hipStreamCreateWithFlags(&c->own_stream, hipStreamNonBlocking);
    if (e != hipSuccess) { delete c; return hip_fail(e, "hipStreamCreateWithFlags"); }
    c->stream = c->own_stream;
  }
  *out = c;
  return RVK_OK;
}

int rvk_ctx_create(int device, rvk_ctx** out) { return ctx_create(device, false, nullptr, out); }
int rvk_ctx_create_on_stream(int device, void* s, rvk_ctx** out) { return ctx_create(device, true, s, out); }

int rvk_ctx_destroy(rvk_ctx* ctx) {
  if (!ctx) return RVK_OK;
  hipSetDevice(ctx->device);
  hipStreamSynchronize(ctx->stream);
  if (ctx->scratch) hipFree(ctx->scratch);
  if (ctx->own_stream) hipStreamDestroy(ctx->own_stream);
  delete ctx;
  return RVK_OK;
}

int rvk_ctx_device(const rvk_ctx* ctx, int* device) {
  if (!ctx || !device) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *device = ctx->device;
  return RVK_OK;
}

int rvk_ctx_stream(const rvk_ctx* ctx, void** s) {
  if (!ctx || !s) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *s = (void*)ctx->stream;
  return RVK_OK;
}

int rvk_ctx_set_stream(rvk_ctx* ctx, void* s) {
  if (!ctx) return fail(RVK_ERR_INVALID_ARGUMENT, "ctx is NULL");
  if (!s && !ctx->own_stream) {
    RVK_HIP(hipSetDevice(ctx->device));
    RVK_HIP(hipStreamCreateWithFlags(&ctx->own_stream, hipStreamNonBlocking));
  }
  ctx->stream = s ? (hipStream_t)s : ctx->own_stream;
  return RVK_OK;
}

int rvk_ctx_sync(rvk_ctx* ctx) {
  if (!ctx) return fail(RVK_ERR_INVALID_ARGUMENT, "ctx is NULL");
  RVK_HIP(hipSetDevice(ctx->device));
  RVK_HIP(hipStreamSynchronize(ctx->stream));
  return RVK_OK;
}

int rvk_device_alloc(rvk_ctx* ctx, size_t bytes, void** out) {
  if (!ctx || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *out = nullptr;
  if (bytes == 0) return RVK_OK;
  RVK_HIP(hipSetDevice(ctx->device));
  RVK_HIP(hipMalloc(out, bytes));
  return RVK_OK;
}

int rvk_device_free(rvk_ctx* ctx, void* ptr) {
  if (!ctx) return fail(RVK_ERR_INVALID_ARGUMENT, "ctx is NULL");
  if (!ptr) return RVK_OK;
  RVK_HIP(hipSetDevice(ctx->device));
  RVK_HIP(hipStreamSynchronize(ctx->stream));
  RVK_HIP(hipFree(ptr));
  return RVK_OK;
}

int rvk_copy_to_device(rvk_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx || (bytes && (!dst || !src))) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  RVK_HIP(hipSetDevice(ctx->device));
  RVK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, ctx->stream));
  RVK_HIP(hipStreamSynchronize(ctx->stream));
  return RVK_OK;
}

int rvk_copy_to_host(rvk_ctx* ctx, void* dst, const void* src, size_t bytes) {
  if (!ctx || (bytes && (!dst || !src))) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  RVK_HIP(hipSetDevice(ctx->device));
  RVK_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, ctx->stream));
  RVK_HIP(hipStreamSynchronize(ctx->stream));
  return RVK_OK;
}

// ---- volumes ----------------------------------------------------------------
int rvk_volume_create(rvk_ctx* ctx, const int32_t dims[3], const double spacing[3], int dtype, int n_frames,
                      rvk_volume** out) {
  if (!ctx || !dims || !spacing || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *out = nullptr;
  if (dtype_size(dtype) == 0) return fail(RVK_ERR_INVALID_ARGUMENT, "unknown dtype %d", dtype);
  if (n_frames < 1 || n_frames > RVK_MAX_FRAMES)
    return fail(RVK_ERR_INVALID_ARGUMENT, "n_frames %d out of range [1,%d]", n_frames, RVK_MAX_FRAMES);
  for (int a = 0; a < 3; ++a) {
    if (dims[a] < 2 || dims[a] > 4096) return fail(RVK_ERR_INVALID_ARGUMENT, "dims[%d]=%d out of range [2,4096]", a, dims[a]);
    if (!(spacing[a] > 0.0) || !std::isfinite(spacing[a]))
      return fail(RVK_ERR_INVALID_ARGUMENT, "spacing[%d] must be positive and finite", a);
  }
  rvk_volume* v = new rvk_volume();
  v->ctx = ctx;
  v->dtype = dtype;
  v->n_frames = n_frames;
  for (int a = 0; a < 3; ++a) {
    v->dims[a] = dims[a];
    v->spacing[a] = spacing[a];
  }
  v->layout = default_layout(dims, dtype);
  const int rc = size_cells(v);
  if (rc != RVK_OK) {
    delete v;
    return rc;
  }
  *out = v;
  return RVK_OK;
}

int rvk_volume_set_layout(rvk_volume* v, int layout) {
  if (!v) return fail(RVK_ERR_INVALID_ARGUMENT, "volume is NULL");
  if (layout != RVK_CELLS_PLAIN && layout != RVK_CELLS_BRICK4 && layout != RVK_CELLS_PAIR8)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown cell layout %d", layout);
  for (int f = 0; f < RVK_MAX_FRAMES; ++f)
    if (v->frames[f]) return fail(RVK_ERR_INVALID_ARGUMENT, "the cell layout is fixed once a frame has data");
  const int old = v->layout;
  v->layout = layout == RVK_CELLS_BRICK4 ? kCellLayoutBrick4
              : layout == RVK_CELLS_PAIR8 ? kCellLayoutPair8
                                          : kCellLayoutPlain;
  const int rc = size_cells(v);
  if (rc != RVK_OK) {
    v->layout = old;
    size_cells(v);
  }
  return rc;
}

int rvk_volume_get_layout(const rvk_volume* v, int* layout) {
  if (!v || !layout) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *layout = v->layout == kCellLayoutBrick4 ? RVK_CELLS_BRICK4
            : v->layout == kCellLayoutPair8 ? RVK_CELLS_PAIR8
                                            : RVK_CELLS_PLAIN;
  return RVK_OK;
}

// Cells of one frame (in the volume's layout and the frame's encoding) from
// x-fastest native voxels on the device.
static int write_frame_cells(rvk_volume* v, int frame, const void* dsrc) {
  const int enc = v->enc[frame];
  // dispatched on the source voxel type: binary16 cells are written by the
  // difference relayout of their 16-bit source
  const bool half = enc == kEncHalf || enc == kEncHalfPair;
  return dispatch_cells<false>(v->dtype, v->layout, half ? kEncDiff : enc, [&](auto tag) {
    using CV = decltype(tag);
    using VT = typename CV::value_type;
    if constexpr (sizeof(VT) == 2 && CV::kDiff) {
      if (enc == kEncHalfPair) return launch_relayout<VT, CV::kLog2, true, 2>(v, dsrc, v->frames[frame]);
      if (enc == kEncHalf) return launch_relayout<VT, CV::kLog2, true, 1>(v, dsrc, v->frames[frame]);
      return launch_relayout<VT, CV::kLog2, true>(v, dsrc, v->frames[frame]);
    } else {
      return launch_relayout<VT, CV::kLog2, CV::kDiff>(v, dsrc, v->frames[frame]);
    }
  });
}

int rvk_volume_relayout(rvk_volume* v, int layout) {
  if (!v) return fail(RVK_ERR_INVALID_ARGUMENT, "volume is NULL");
  if (layout != RVK_CELLS_PLAIN && layout != RVK_CELLS_BRICK4 && layout != RVK_CELLS_PAIR8)
    return fail(RVK_ERR_INVALID_ARGUMENT, "unknown cell layout %d", layout);
  const int target = layout == RVK_CELLS_BRICK4 ? kCellLayoutBrick4
                     : layout == RVK_CELLS_PAIR8 ? kCellLayoutPair8
                                                 : kCellLayoutPlain;
  if (target == v->layout) return RVK_OK;
  bool any = false;
  for (int f = 0; f < RVK_MAX_FRAMES; ++f) any = any || v->frames[f];
  if (!any) return rvk_volume_set_layout(v, layout);
  {
    rvk_volume probe = *v;  // the new layout must fit its addressing limits
    probe.layout = target;
    const int rc = size_cells(&probe);
    if (rc) return rc;
  }
  RVK_HIP(hipSetDevice(v->ctx->device));
  RVK_HIP(hipStreamSynchronize(v->ctx->stream));
  const size_t n = (size_t)v->dims[0] * v->dims[1] * v->dims[2];
  const size_t es = dtype_size(v->dtype);
  const VolGeom g = vol_geom(v);
  const int blocks = (int)((n + 255) / 256);
  std::vector<void*> lin(RVK_MAX_FRAMES, nullptr), glin(RVK_MAX_FRAMES, nullptr);
  auto release = [&]() {
    for (void* q : lin) if (q) hipFree(q);
    for (void* q : glin) if (q) hipFree(q);
  };
  int rc = RVK_OK;
  // every frame (and gradient-magnitude volume) back to native voxels
  for (int f = 0; f < RVK_MAX_FRAMES && !rc; ++f) {
    if (!v->frames[f]) continue;
    if (hipMalloc(&lin[f], n * es) != hipSuccess) { rc = fail(RVK_ERR_OUT_OF_MEMORY, "relayout staging"); break; }
    rc = dispatch_frame(v, f, [&](auto tag) {
      using CV = decltype(tag);
      auto go = [&](auto vt) {
        using VT = decltype(vt);
        hipLaunchKernelGGL((extract_voxels_kernel<CV, VT>), dim3(blocks), dim3(256), 0, v->ctx->stream,
                           (const void*)v->frames[f], g, (VT*)lin[f], (long long)n);
        return (int)RVK_OK;
      };
      switch (v->dtype) {
        case RVK_U8: return go(uint8_t{});
        case RVK_I8: return go(int8_t{});
        case RVK_U16: return go(uint16_t{});
        case RVK_I16: return go(int16_t{});
        case RVK_U32: return go(uint32_t{});
        case RVK_I32: return go(int32_t{});
        default: return go(float{});
      }
    });
    if (!rc && v->gradmag[f]) {
      if (hipMalloc(&glin[f], n) != hipSuccess) { rc = fail(RVK_ERR_OUT_OF_MEMORY, "relayout staging"); break; }
      auto gm = [&](auto tagL) {
        constexpr int L = decltype(tagL)::value;
        hipLaunchKernelGGL((extract_voxels_kernel<Cells<uint8_t, L>, uint8_t>), dim3(blocks), dim3(256), 0,
                           v->ctx->stream, (const void*)v->gradmag[f], g, (uint8_t*)glin[f], (long long)n);
      };
      if (v->layout == kCellLayoutBrick4) gm(std::integral_constant<int, kCellLayoutBrick4>{});
      else if (v->layout == kCellLayoutPair8) gm(std::integral_constant<int, kCellLayoutPair8>{});
      else gm(std::integral_constant<int, kCellLayoutPlain>{});
    }
  }
  if (!rc) {
    const hipError_t e = hipStreamSynchronize(v->ctx->stream);
    if (e != hipSuccess) rc = hip_fail(e, "relayout extraction");
  }
  if (rc) { release(); return rc; }
  // the new cells are allocated before the old ones are released, so that a
  // failed allocation leaves the volume as it was
  rvk_volume probe = *v;
  probe.layout = target;
  size_cells(&probe);
  std::vector<void*> nf(RVK_MAX_FRAMES, nullptr);
  std::vector<uint8_t*> ng(RVK_MAX_FRAMES, nullptr);
  for (int f = 0; f < RVK_MAX_FRAMES && !rc; ++f) {
    if (lin[f] && hipMalloc(&nf[f], probe.n_cells * 8 * es) != hipSuccess) rc = RVK_ERR_OUT_OF_MEMORY;
    if (!rc && glin[f] && hipMalloc((void**)&ng[f], probe.n_cells * 8) != hipSuccess) rc = RVK_ERR_OUT_OF_MEMORY;
  }
  if (rc) {
    for (void* q : nf) if (q) hipFree(q);
    for (uint8_t* q : ng) if (q) hipFree(q);
    release();
    return fail(RVK_ERR_OUT_OF_MEMORY, "relayout: no device memory for the new cells (volume unchanged)");
  }
  // the new layout: cells rewritten from the native voxels, same encodings
  std::vector<void*> of(v->frames, v->frames + RVK_MAX_FRAMES);
  std::vector<uint8_t*> og(v->gradmag, v->gradmag + RVK_MAX_FRAMES);
  v->layout = target;
  size_cells(v);
  for (int f = 0; f < RVK_MAX_FRAMES; ++f) {
    v->frames[f] = nf[f];
    v->gradmag[f] = ng[f];
  }
  for (int f = 0; f < RVK_MAX_FRAMES && !rc; ++f) {
    if (!lin[f]) continue;
    rc = write_frame_cells(v, f, lin[f]);
    if (!rc && glin[f]) {
      if (v->layout == kCellLayoutBrick4) rc = launch_relayout<uint8_t, kCellLayoutBrick4>(v, glin[f], v->gradmag[f]);
      else if (v->layout == kCellLayoutPair8) rc = launch_relayout<uint8_t, kCellLayoutPair8>(v, glin[f], v->gradmag[f]);
      else rc = launch_relayout<uint8_t, kCellLayoutPlain>(v, glin[f], v->gradmag[f]);
    }
  }
  const hipError_t e = hipStreamSynchronize(v->ctx->stream);
  release();
  for (void* q : of) if (q) hipFree(q);
  for (uint8_t* q : og) if (q) hipFree(q);
  ++v->generation;
  if (!rc && e != hipSuccess) rc = hip_fail(e, "relayout");
  return rc;
}

int rvk_volume_set_frame(rvk_volume* v, int frame, const void* src, int src_on_device) {
  if (!v || !src) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  if (frame < 0 || frame >= v->n_frames)
    return fail(RVK_ERR_INVALID_ARGUMENT, "frame %d out of range [0,%d)", frame, v->n_frames);
  RVK_HIP(hipSetDevice(v->ctx->device));
  const size_t es = dtype_size(v->dtype);
  const size_t n = (size_t)v->dims[0] * v->dims[1] * v->dims[2];
  if (!v->frames[frame]) RVK_HIP(hipMalloc(&v->frames[frame], v->n_cells * 8 * es));
  const void* dsrc = src;
  void* staging = nullptr;
  if (!src_on_device) {
    RVK_HIP(hipMalloc(&staging, n * es));
    hipError_t e = hipMemcpyAsync(staging, src, n * es, hipMemcpyHostToDevice, v->ctx->stream);
    if (e != hipSuccess) { hipFree(staging); return hip_fail(e, "hipMemcpyAsync(volume)"); }
    dsrc = staging;
  }
  // float cells always store x-pair differences; 16-bit cells when the
  // frame's values span less than 32768 (then every difference fits), with
  // binary16 bases when they all lie in [-2048, 2048], and binary16
  // differences when these are exact too
  int enc = v->dtype == RVK_F32 ? kEncDiff : kEncPlain;
  int lo = 0, hi = 0;
  bool odd = false;
  int rc = frame_stats(v, frame, dsrc, lo, hi, odd);
  if (v->dtype == RVK_U16 || v->dtype == RVK_I16) {
    if (rc == RVK_OK && hi - lo <= 32767) {
      enc = kEncDiff;
      if (lo >= -2048 && hi <= 2048) enc = odd ? kEncHalf : kEncHalfPair;
    }
  }
  if (rc == RVK_OK) {
    v->enc[frame] = (uint8_t)enc;
    rc = write_frame_cells(v, frame, dsrc);
  }
  if (staging) {
    hipError_t e = hipStreamSynchronize(v->ctx->stream);
    hipFree(staging);
    if (rc == RVK_OK && e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
  }
  return rc;
}

int rvk_volume_compute_gradmag(rvk_volume* v, int frame, float max_gradient) {
  int rc = check_frame(v, frame);
  if (rc) return rc;
  if (!(max_gradient > 0.0f) || !std::isfinite(max_gradient))
    return fail(RVK_ERR_INVALID_ARGUMENT, "max_gradient must be positive and finite");
  RVK_HIP(hipSetDevice(v->ctx->device));
  if (!v->gradmag[frame]) RVK_HIP(hipMalloc((void**)&v->gradmag[frame], v->n_cells * 8));
  v->gradmag_scale[frame] = max_gradient / 255.0f;
  const float inv = 255.0f / max_gradient;
  uint8_t* linear = nullptr;
  RVK_HIP(hipMalloc((void**)&linear, (size_t)v->dims[0] * v->dims[1] * v->dims[2]));
  rc = dispatch_frame(v, frame, [&](auto tag) { return launch_gradmag<decltype(tag)>(v, frame, inv, linear); });
  const hipError_t e = hipStreamSynchronize(v->ctx->stream);
  hipFree(linear);
  if (rc == RVK_OK && e != hipSuccess) return hip_fail(e, "hipStreamSynchronize");
  return rc;
}

int rvk_volume_destroy(rvk_volume* v) {
  if (!v) return RVK_OK;
  hipSetDevice(v->ctx->device);
  hipStreamSynchronize(v->ctx->stream);
  for (int f = 0; f < RVK_MAX_FRAMES; ++f) {
    if (v->frames[f]) hipFree(v->frames[f]);
    if (v->gradmag[f]) hipFree(v->gradmag[f]);
    if (v->ranges[f]) hipFree(v->ranges[f]);
  }
  delete v;
  return RVK_OK;
}

int rvk_volume_dims(const rvk_volume* v, int32_t dims[3], double spacing[3], int* dtype, int* n_frames) {
  if (!v) return fail(RVK_ERR_INVALID_ARGUMENT, "volume is NULL");
  for (int a = 0; a < 3; ++a) {
    if (dims) dims[a] = v->dims[a];
    if (spacing) spacing[a] = v->spacing[a];
  }
  if (dtype) *dtype = v->dtype;
  if (n_frames) *n_frames = v->n_frames;
  return RVK_OK;
}

// ---- transfer functions -------------------------------------------------------
int rvk_tf1d_create(rvk_ctx* ctx, int n, const float* alpha, const float* galpha, const float* red,
                    const float* green, const float* blue, const rvk_tf1d_params* p, rvk_tf1d** out) {
  if (!ctx || !alpha || !red || !green || !blue || !p || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *out = nullptr;
  if (n < 1 || n > 2048) return fail(RVK_ERR_INVALID_ARGUMENT, "TF size %d out of range [1,2048]", n);
  std::vector<float> h((size_t)5 * n);
  std::memcpy(&h[0], alpha, sizeof(float) * n);
  for (int i = 0; i < n; ++i) h[(size_t)n + i] = galpha ? galpha[i] : 1.0f;
  std::memcpy(&h[(size_t)2 * n], red, sizeof(float) * n);
  std::memcpy(&h[(size_t)3 * n], green, sizeof(float) * n);
  std::memcpy(&h[(size_t)4 * n], blue, sizeof(float) * n);
  RVK_HIP(hipSetDevice(ctx->device));
  rvk_tf1d* t = new rvk_tf1d();
  t->ctx = ctx;
  t->n = n;
  t->p = *p;
  t->least = least_positive(alpha, n) * (std::isfinite(p->gradient_multiplier) ? least_positive(&h[n], n) : 1.0f);
  hipError_t e = hipMalloc((void**)&t->tables, h.size() * sizeof(float));
  if (e != hipSuccess) { delete t; return hip_fail(e, "hipMalloc(tf1d)"); }
  e = hipMemcpy(t->tables, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice);
  if (e != hipSuccess) { hipFree(t->tables); delete t; return hip_fail(e, "hipMemcpy(tf1d)"); }
  *out = t;
  return RVK_OK;
}

int rvk_tf1d_destroy(rvk_tf1d* t) {
  if (!t) return RVK_OK;
  hipSetDevice(t->ctx->device);
  hipStreamSynchronize(t->ctx->stream);
  if (t->tables) hipFree(t->tables);
  delete t;
  return RVK_OK;
}

static int upload_occupancy(int n, const float* alpha, uint32_t** dst) {
  const size_t nn = (size_t)n * n, words = (nn + 31) / 32;
  std::vector<uint32_t> bits(words, 0u);
  for (size_t c = 0; c < nn; ++c)
    if (alpha[c] > 0.0f) bits[c >> 5] |= 1u << (c & 31);
  RVK_HIP(hipMalloc((void**)dst, words * sizeof(uint32_t)));
  hipError_t e = hipMemcpy(*dst, bits.data(), words * sizeof(uint32_t), hipMemcpyHostToDevice);
  if (e != hipSuccess) { hipFree(*dst); *dst = nullptr; return hip_fail(e, "hipMemcpy(tf2d occupancy)"); }
  return RVK_OK;
}

// Column bitmaps of `count` n x n tables (index g*n + i): bit i of table t is
// set when some row has a value > 0 in column i.
static int upload_columns(int n, const float* const* tabs, int count, uint32_t** dst) {
  const size_t w = (size_t)(n + 31) / 32;
  std::vector<uint32_t> bits(w * count, 0u);
  for (int t = 0; t < count; ++t)
    for (int g = 0; g < n; ++g)
      for (int i = 0; i < n; ++i)
        if (tabs[t][(size_t)g * n + i] > 0.0f) bits[w * t + (i >> 5)] |= 1u << (i & 31);
  RVK_HIP(hipMalloc((void**)dst, bits.size() * sizeof(uint32_t)));
  hipError_t e = hipMemcpy(*dst, bits.data(), bits.size() * sizeof(uint32_t), hipMemcpyHostToDevice);
  if (e != hipSuccess) { hipFree(*dst); *dst = nullptr; return hip_fail(e, "hipMemcpy(tf2d columns)"); }
  return RVK_OK;
}

// A cell's contribution in the gradient-magnitude path (Phong-Lambert factor
// 1), with the operations cast2d_kernel would apply per sample.
__global__ __launch_bounds__(256) void tf2d_lit_kernel(const Tf2dCell* __restrict__ c, float4* __restrict__ lit,
                                                       long long nn) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nn) return;
  const Tf2dCell e = c[i];
  const float pl = 1.0f;
  const float shd = e.ambient + e.diffuse * pl;
  const float shs = e.specular * powf(pl, e.spec_power);
  lit[i] = make_float4(e.alpha, satf(shd * e.r + shs), satf(shd * e.g + shs), satf(shd * e.b + shs));
}

static int make_lit(rvk_ctx* ctx, int n, const Tf2dCell* cells, float4** dst) {
  const long long nn = (long long)n * n;
  RVK_HIP(hipMalloc((void**)dst, nn * sizeof(float4)));
  hipLaunchKernelGGL(tf2d_lit_kernel, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, ctx->stream, cells, *dst, nn);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) { hipFree(*dst); *dst = nullptr; return hip_fail(e, "tf2d lit cells"); }
  return RVK_OK;
}

static int upload_cells(int n, const float* const tables[8], Tf2dCell** dst) {
  for (int i = 0; i < 8; ++i)
    if (!tables[i]) return fail(RVK_ERR_INVALID_ARGUMENT, "2D TF table %d is NULL", i);
  const size_t nn = (size_t)n * n;
  std::vector<Tf2dCell> h(nn);
  for (size_t c = 0; c < nn; ++c) {
    h[c].alpha = tables[0][c];
    h[c].r = tables[1][c];
    h[c].g = tables[2][c];
    h[c].b = tables[3][c];
    h[c].ambient = tables[4][c];
    h[c].diffuse = tables[5][c];
    h[c].specular = tables[6][c];
    h[c].spec_power = tables[7][c];
  }
  RVK_HIP(hipMalloc((void**)dst, nn * sizeof(Tf2dCell)));
  hipError_t e = hipMemcpy(*dst, h.data(), nn * sizeof(Tf2dCell), hipMemcpyHostToDevice);
  if (e != hipSuccess) { hipFree(*dst); *dst = nullptr; return hip_fail(e, "hipMemcpy(tf2d)"); }
  return RVK_OK;
}

int rvk_tf2d_create(rvk_ctx* ctx, int n, const float* const tables[8], const float* const ktables[8],
                    const rvk_tf2d_params* p, rvk_tf2d** out) {
  if (!ctx || !tables || !p || !out) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  *out = nullptr;
  if (n < 1 || n > 2048) return fail(RVK_ERR_INVALID_ARGUMENT, "TF size %d out of range [1,2048]", n);
  RVK_HIP(hipSetDevice(ctx->device));
  rvk_tf2d* t = new rvk_tf2d();
  t->ctx = ctx;
  t->n = n;
  t->p = *p;
  int rc = upload_cells(n, tables, &t->cells);
  if (rc == RVK_OK && ktables) rc = upload_cells(n, ktables, &t->kcells);
  if (rc == RVK_OK) rc = make_lit(ctx, n, t->cells, &t->lit);
  if (rc == RVK_OK && ktables) rc = make_lit(ctx, n, t->kcells, &t->klit);
  if (rc == RVK_OK && n <= kTf2dOccMaxN) {
    t->occ_words = (int)(((size_t)n * n + 31) / 32);
    rc = upload_occupancy(n, tables[0], &t->occ);
    if (rc == RVK_OK && ktables) rc = upload_occupancy(n, ktables[0], &t->kocc);
  }
  if (rc == RVK_OK) {
    const float* alphas[2] = {tables[0], ktables ? ktables[0] : nullptr};
    t->col_words = (n + 31) / 32;
    rc = upload_columns(n, alphas, ktables ? 2 : 1, &t->col);
  }
  if (rc != RVK_OK) {
    if (t->cells) hipFree(t->cells);
    if (t->kcells) hipFree(t->kcells);
    if (t->lit) hipFree(t->lit);
    if (t->klit) hipFree(t->klit);
    if (t->occ) hipFree(t->occ);
    if (t->kocc) hipFree(t->kocc);
    if (t->col) hipFree(t->col);
    delete t;
    return rc;
  }
  t->alpha_host.assign(tables[0], tables[0] + (size_t)n * n);
  t->least = least_positive(tables[0], (size_t)n * n);
  *out = t;
  return RVK_OK;
}

// The In/Ex table reduced to the two comparisons the caster makes
// (V/CUDA_vtkCuda2DInExLogicVolumeMapper_renderAlgo.cuh:111,125-126):
// bit 0 = (inEx > 0 || alpha > 0), bit 1 = (inEx > 0.5).
int rvk_tf2d_set_inex(rvk_tf2d* t, const float* inex) {
  if (!t) return fail(RVK_ERR_INVALID_ARGUMENT, "NULL argument");
  RVK_HIP(hipSetDevice(t->ctx->device));
  RVK_HIP(hipStreamSynchronize(t->ctx->stream));
  if (t->inex_flags) { hipFree(t->inex_flags); t->inex_flags = nullptr; }
  if (t->inex_occ) { hipFree(t->inex_occ); t->inex_occ = nullptr; }
  if (t->inex_col) { hipFree(t->inex_col); t->inex_col = nullptr; }
  if (!inex) return RVK_OK;
  const size_t nn = (size_t)t->n * t->n;
  std::vector<uint8_t> flags(nn);
  for (size_t c = 0; c < nn; ++c)
    flags[c] = (uint8_t)(((inex[c] > 0.0f || t->alpha_host[c] > 0.0f) ? 1u : 0u) | (inex[c] > 0.5f ? 2u : 0u));
  // a marked cell without opacity composites nothing: no bound on the samples
  t->inex_least = least_positive(t->alpha_host.data(), nn);
  for (size_t c = 0; c < nn; ++c)
    if ((flags[c] & 1u) && !(t->alpha_host[c] > 0.0f)) t->inex_least = 0.0f;
  RVK_HIP(hipMalloc((void**)&t->inex_flags, nn));
  hipError_t e = hipMemcpy(t->inex_flags, flags.data(), nn, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    hipFree(t->inex_flags);
    t->inex_flags = nullptr;
    return hip_fail(e, "hipMemcpy(inex flags)");
  }
  {
    std::vector<float> live(nn);
    for (size_t c = 0; c < nn; ++c) live[c] = (flags[c] & 1u) ? 1.0f : 0.0f;
    const float* tabs[1] = {live.data()};
    const int rc = upload_columns(t->n, tabs, 1, &t->inex_col);
    if (rc != RVK_OK) {
      hipFree(t->inex_flags);
      t->inex_flags = nullptr;
      return rc;
    }
  }
  if (t->occ_words) {
    const size_t w = (size_t)t->occ_words;
    std::vector<uint32_t> bits(2 * w, 0u);
    for (size_t c = 0; c < nn; ++c) {
      if (flags[c] & 1u) bits[c >> 5] |= 1u << (c & 31);
      if (flags[c] & 2u) bits[w + (c >> 5)] |= 1u << (c & 31);
    }
    RVK_HIP(hipMalloc((void**)&t->inex_occ, 2 * w * sizeof(uint32_t)));
    e = hipMemcpy(t->inex_occ, bits.data(), 2 * w * sizeof(uint32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
      hipFree(t->inex_occ);
      t->inex_occ = nullptr;
      return hip_fail(e, "hipMemcpy(inex bitmaps)");
    }
  }
  return RVK_OK;
}

int rvk_tf2d_destroy(rvk_tf2d* t) {
  if (!t) return RVK_OK;
  hipSetDevice(t->ctx->device);
  hipStreamSynchronize(t->ctx->stream);
  if (t->cells) hipFree(t->cells);
  if (t->kcells) hipFree(t->kcells);
  if (t->lit) hipFree(t->lit);
  if (t->klit) hipFree(t->klit);
  if (t->occ) hipFree(t->occ);
  if (t->kocc) hipFree(t->kocc);
  if (t->inex_flags) hipFree(t->inex_flags);
  if (t->inex_occ) hipFree(t->inex_occ);
  if (t->inex_col) hipFree(t->inex_col);
  if (t->col) hipFree(t->col);
  delete t;
  return RVK_OK;
}

int rvk_stream_read(rvk_ctx* ctx, const void* buf, size_t bytes, uint32_t* sink) {
  if (!ctx || !buf || bytes < 16 || (bytes & 15) || ((uintptr_t)buf & 15))
    return fail(RVK_ERR_INVALID_ARGUMENT, "need a 16-byte aligned buffer of a multiple of 16 bytes");
  RVK_HIP(hipSetDevice(ctx->device));
  int n_cu = 256;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, ctx->device) == hipSuccess) n_cu = prop.multiProcessorCount;
  const size_t n = bytes / 16;
  const size_t want = (n + 255) / 256;
  const unsigned blocks = (unsigned)std::max<size_t>(1, std::min<size_t>(want, (size_t)n_cu * 8));
  hipLaunchKernelGGL(stream_read_kernel, dim3(blocks), dim3(256), 0, ctx->stream, (const uint4*)buf, n, sink);
  RVK_HIP(hipGetLastError());
  return RVK_OK;
}

}  // extern "C"
