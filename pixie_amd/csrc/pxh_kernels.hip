// pxh_kernels.hip -- HIP kernels for gfx950 (MI355X) and their launchers.
//
//   fill_rows_kernel   one fillShapes call (paths.nim:1593-1912): a wave per
//                      (canvas row, column window) runs the row program and the fused
//                      coverage -> paint -> blend -> write-back epilogue
//   composite_kernel   blendRect (images.nim:468-529), all 20 blend modes
//   opacity_kernel     applyOpacity (images.nim:261-277)
//
// Every kernel is memory-bound integer / float32 work: no MFMA.
#include <hip/hip_runtime.h>

#include "pxh_kernels.h"
#include "pxh_raster.h"

namespace pxh {

// ---------------------------------------------------------------------------
// fill: one wave (64 threads) per workgroup, grid-stride over (row, window)
// units
// ---------------------------------------------------------------------------
template <bool kA8>
__global__ void __launch_bounds__(64) fill_rows_kernel(FillArgs a) {
  extern __shared__ __align__(16) char smem[];
  const FillInfo& F = *a.F;
  const size_t fixedBytes = row_lds_fixed_bytes(a.ww);
  char* arr = a.capInLds ? smem + fixedBytes : a.gscratch + (size_t)blockIdx.x * row_cap_bytes(a.cap);
  RowLds L = row_lds_carve(smem, arr, a.cap, a.ww);
  for (int i = threadIdx.x; i < a.ww + 4; i += kWave) L.D[i] = 0;
  wave_sync();
  const bool mask = F.mode == kMask;
  const int32_t W = F.canvasW;
  const int32_t lo = mask ? 0 : F.xlo, hi = mask ? W : F.xhi;
  const int32_t x0 = lo & ~3;
  const int32_t nWin = hi > x0 ? (hi - x0 + a.ww - 1) / a.ww : 0;
  const int64_t nUnits = (int64_t)a.nRows * nWin;
  uint32_t ntouch = 0;
  // one work unit per (row, column window), grid-stride
  for (int64_t u = blockIdx.x; u < nUnits; u += gridDim.x) {
    const int32_t y = a.rowBase + (int32_t)(u / nWin);
    const int32_t wx = x0 + (int32_t)(u % nWin) * a.ww;
    RowCtx C;
    C.F = a.F;
    C.parts = a.parts;
    C.E = a.E;
    C.EW = a.EW;
    C.y = y;
    C.wx0 = wx;
    C.wx1 = wx + a.ww < hi ? wx + a.ww : hi;
    C.cx0 = lo;
    C.cx1 = hi;
    int32_t kind = row_program(C, L);
    if (kind < 0) {
      if (threadIdx.x == 0) atomicOr(a.err, 1);
      break;
    }
    if (kind == kRowNone) continue;
    if (kA8)
      ntouch += row_epilogue_a8(C, L, kind, (uint8_t*)a.canvas, W, F.rgbx, F.mode);
    else
      ntouch += row_epilogue(C, L, kind, (uint32_t*)a.canvas, W, F.rgbx, F.mode);
  }
  if (a.touched) {
    // wave reduction, one atomic per workgroup
    for (int o = 32; o > 0; o >>= 1) ntouch += __shfl_xor(ntouch, o, kWave);
    if (threadIdx.x == 0 && ntouch) atomicAdd(a.touched, (unsigned long long)ntouch);
  }
}

int launch_fill_rows(const FillArgs& a, int grid, size_t ldsBytes, bool a8, hipStream_t s) {
  if (a8)
    hipLaunchKernelGGL(fill_rows_kernel<true>, dim3(grid), dim3(64), ldsBytes, s, a);
  else
    hipLaunchKernelGGL(fill_rows_kernel<false>, dim3(grid), dim3(64), ldsBytes, s, a);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int set_fill_lds_limit(size_t bytes) {
  if (hipFuncSetAttribute((const void*)fill_rows_kernel<false>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
    return kErrDevice;
  if (hipFuncSetAttribute((const void*)fill_rows_kernel<true>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess)
    return kErrDevice;
  return 0;
}

// ---------------------------------------------------------------------------
// gradient paints (paints.nim:72-248) through fillPath's mask route
// (paths.nim:2115-2142), one pass: each pixel takes the path's coverage from
// the A8 mask, the gradient colour at its integer coordinates, masks the
// colour with the coverage as fill.draw(mask, MaskBlend) does, and blends it
// as image.draw(fill, blendMode) does.  Float math is pixie's float32 order.
// ---------------------------------------------------------------------------
// gradientColor (paints.nim:72-97), then Color -> ColorRGBX (round to 8 bits,
// premultiply with (c * a + 127) div 255)
__device__ uint32_t gradient_color(const PaintArgs& a, float t) {
  int index = -1;
  for (int i = 0; i < a.nstops; i++) {
    const float pos = a.stops[5 * i + 4];
    if (pos < t) index = i;
    if (pos > t) break;
  }
  float c[4];
  if (index == -1 || index + 1 >= a.nstops) {
    const int k = index == -1 ? 0 : index;
    for (int j = 0; j < 4; j++) c[j] = a.stops[5 * k + j];
  } else {
    const float* s1 = a.stops + 5 * index;
    const float* s2 = a.stops + 5 * (index + 1);
    const float v = (t - s1[4]) / (s2[4] - s1[4]);
    for (int j = 0; j < 4; j++) c[j] = s1[j] * (1.0f - v) + s2[j] * v;
  }
  const FColor f = {c[0], c[1], c[2], c[3]};
  return from_fcolor(f);
}

__device__ __forceinline__ float fix_angle_p(float x) {
  const float PI = 3.14159265358979323846f;
  while (x > PI) x -= PI * 2.0f;
  while (x < -PI) x += PI * 2.0f;
  return x;
}

// the gradient parameter t of pixel (x, y) (paints.nim:108-113, 199-209,
// 224-236)
__device__ float gradient_t(const PaintArgs& a, int32_t x, int32_t y) {
  const float fx = (float)x, fy = (float)y;
  if (a.kind == 3) {  // linear: toLineSpace
    const float dx = a.hx[2] - a.hx[0], dy = a.hx[3] - a.hx[1];
    const float det = dx * dx + dy * dy;
    return (dy * (fy - a.hx[1]) + dx * (fx - a.hx[0])) / det;
  }
  if (a.kind == 4) {  // radial: |inverse gradient matrix * xy|
    const float px = a.m[0] * fx + a.m[3] * fy + a.m[6];
    const float py = a.m[1] * fx + a.m[4] * fy + a.m[7];
    return sqrtf(px * px + py * py);
  }
  const float PI = 3.14159265358979323846f;  // angular
  const float vx = fx - a.hx[0], vy = fy - a.hx[1];
  const float l = sqrtf(vx * vx + vy * vy);
  const float angle = atan2f(vy / l, vx / l);
  return fix_angle_p(angle + a.ga + PI / 2.0f) / 2.0f / PI + 0.5f;
}

__global__ void __launch_bounds__(256) paint_kernel(PaintArgs a) {
  const int32_t y = blockIdx.y;
  const int32_t x = blockIdx.x * 256 + threadIdx.x;
  if (x >= a.w) return;
  const size_t i = (size_t)y * a.w + x;
  uint32_t m = a.mask[i];
  if (a.useOpacity) m = m * a.o255 / 255u;  // applyOpacity on the mask (images.nim:261-277)
  // image paints read the image drawn onto a transparent canvas
  const uint32_t g = a.kind <= 2 ? a.fill[i] : gradient_color(a, gradient_t(a, x, y));
  // fill.draw(mask, MaskBlend): every channel times the mask's alpha
  const uint32_t src = pack(ch_r(g) * m / 255u, ch_g(g) * m / 255u, ch_b(g) * m / 255u, ch_a(g) * m / 255u);
  // a transparent source leaves the backdrop of these modes bit for bit
  const int md = a.mode;
  const bool keepOnZero = md == kNormal || md == kDarken || md == kMultiply || md == kLighten ||
                          md == kScreen || md == kOverlay || md == kHardLight || md == kDifference ||
                          md == kExclusion;
  if (src == 0u && keepOnZero) return;
  a.dst[i] = blend(md, a.dst[i], src);
}

int launch_paint(const PaintArgs& a, hipStream_t s) {
  dim3 g((a.w + 255) / 256, a.h);
  hipLaunchKernelGGL(paint_kernel, g, dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// composite (blendRect): each thread handles 4 consecutive destination pixels
// ---------------------------------------------------------------------------
template <bool kSrcA8>
__global__ void __launch_bounds__(256) composite_kernel(CompositeArgs a) {
  const int32_t y = blockIdx.y;  // destination row
  const int32_t x0 = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (x0 >= a.aw) return;
  uint32_t* arow = a.dst + (size_t)y * a.aw;
  const bool mask = a.mode == kMask;
  const int32_t sy = y - a.py;
  const bool rowIn = sy >= a.yStart && sy < a.yEnd;
  const bool vec = ((a.aw & 3) == 0);
  uint32_t px[4];
  bool any = false;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    int32_t x = x0 + k;
    px[k] = 0;
    if (x >= a.aw) continue;
    int32_t sx = x - a.px;
    bool in = rowIn && sx >= a.xStart && sx < a.xEnd;
    if (in || mask) any = true;
  }
  if (!any) return;
  if (vec) {
    uint4 v = *(const uint4*)(arow + x0);
    px[0] = v.x; px[1] = v.y; px[2] = v.z; px[3] = v.w;
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) px[k] = (x0 + k < a.aw) ? arow[x0 + k] : 0u;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    int32_t x = x0 + k;
    if (x >= a.aw) continue;
    int32_t sx = x - a.px;
    bool in = rowIn && sx >= a.xStart && sx < a.xEnd;
    if (in) {
      uint32_t s;
      if (kSrcA8) {
        uint32_t v = ((const uint8_t*)a.src)[(size_t)sy * a.bw + sx];
        s = v * 0x01010101u;
      } else {
        s = ((const uint32_t*)a.src)[(size_t)sy * a.bw + sx];
      }
      px[k] = blend(a.mode, px[k], s);
    } else if (mask) {
      px[k] = 0;
    }
  }
  if (vec) {
    *(uint4*)(arow + x0) = make_uint4(px[0], px[1], px[2], px[3]);
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (x0 + k < a.aw) arow[x0 + k] = px[k];
  }
}

int launch_composite(const CompositeArgs& a, bool srcA8, hipStream_t s) {
  dim3 grid((a.aw + 1023) / 1024, a.ah);
  if (srcA8)
    hipLaunchKernelGGL(composite_kernel<true>, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(composite_kernel<false>, grid, dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// applyOpacity (images.nim:261-277), o = round(255*opacity) in (0, 255)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) opacity_kernel(uint32_t* img, int64_t n, uint32_t o) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uint32_t p = img[i];
  img[i] = pack((ch_r(p) * o) / 255u, (ch_g(p) * o) / 255u, (ch_b(p) * o) / 255u, (ch_a(p) * o) / 255u);
}

int launch_opacity(uint32_t* img, int64_t n, uint32_t o, hipStream_t s) {
  hipLaunchKernelGGL(opacity_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, img, n, o);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// blend test kernel: out[i] = blend(mode, b[i], s[i])
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) blend_pixels_kernel(const uint32_t* b, const uint32_t* src,
                                                           uint32_t* out, int64_t n, int32_t mode) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  out[i] = blend(mode, b[i], src[i]);
}

int launch_blend_pixels(const uint32_t* b, const uint32_t* s_, uint32_t* out, int64_t n, int32_t mode,
                        hipStream_t s) {
  hipLaunchKernelGGL(blend_pixels_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, b, s_,
                     out, n, mode);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

}  // namespace pxh
