// pxh_kernels.hip -- HIP kernels for gfx950 (MI355X) and their launchers.
//
//   fill_rows_kernel   one fillShapes call (paths.nim:1593-1912): a wave per
//                      (canvas row, column window) runs the row program and the fused
//                      coverage -> paint -> blend -> write-back epilogue
//   composite_kernel   blendRect (images.nim:468-529), all 20 blend modes
//   opacity_kernel     applyOpacity (images.nim:261-277)
//
// No kernel here is a contraction: integer and float32 arithmetic, no MFMA.
#include <hip/hip_runtime.h>

#include "pxh_kernels.h"
#include "pxh_raster.h"

namespace pxh {

// ---------------------------------------------------------------------------
// fill: one wave (64 threads) per workgroup, grid-stride over (row, window)
// units.  100 KB of code with the twenty blend modes and the row program's
// forms in line; at the 128 VGPRs of four waves a SIMD it spills 11 VGPRs and
// 194 SGPRs (48 B of scratch a lane).
// ---------------------------------------------------------------------------
template <bool kA8>
__global__ void __launch_bounds__(64, 4) fill_rows_kernel(FillArgs a) {
  extern __shared__ __align__(16) char smem[];
  // the same in every lane, and read once: through the pointer every use would
  // load it again behind the canvas's stores
  FillInfo F = *a.F;
  F.startX = uni(F.startX);
  F.startY = uni(F.startY);
  F.pathWidth = uni(F.pathWidth);
  F.pathHeight = uni(F.pathHeight);
  F.nParts = uni(F.nParts);
  F.bandH = uni(F.bandH);
  F.mode = uni(F.mode);
  F.rule = uni(F.rule);
  F.xlo = uni(F.xlo);
  F.xhi = uni(F.xhi);
  F.canvasW = uni(F.canvasW);
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
    C.F = &F;
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
    if (threadIdx.x == 0 && ntouch) atomicAdd(touched_slot(a.touched), (unsigned long long)ntouch);
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
// premultiply with (c * a + 127) div 255).  The search runs over all stops
// without leaving early, so that its lanes stay together.
struct StopTable {
  float4 color[kMaxStops];
  float pos[kMaxStops];
};
__device__ __forceinline__ uint32_t round_unit(float v) {  // unit_u8
  v = !(v > 0.0f) ? 0.0f : v > 1.0f ? 1.0f : v;
  v = v * 255.0f;
  const uint32_t n = (uint32_t)v;  // v - n is exact: halves go up, as roundf's
  return n + (v - (float)n >= 0.5f ? 1u : 0u);
}
__device__ __forceinline__ uint32_t gradient_color(const PaintArgs& a, const StopTable& S, float t) {
  int index = -1;
  bool on = true;
  for (int i = 0; i < a.nstops; i++) {
    const float pos = a.stops[5 * i + 4];
    if (on && pos < t) index = i;
    on = on && !(pos > t);
  }
  float4 c;
  if (index == -1 || index + 1 >= a.nstops) {
    c = S.color[index == -1 ? 0 : index];
  } else {
    const float4 s1 = S.color[index], s2 = S.color[index + 1];
    const float p1 = S.pos[index];
    const float v = (t - p1) / (S.pos[index + 1] - p1);
    c = make_float4(s1.x * (1.0f - v) + s2.x * v, s1.y * (1.0f - v) + s2.y * v, s1.z * (1.0f - v) + s2.z * v,
                    s1.w * (1.0f - v) + s2.w * v);
  }
  const uint32_t al = round_unit(c.w);
  const uint32_t p = pack(round_unit(c.x), round_unit(c.y), round_unit(c.z), 255u);
  // premultiply: 255 div-multiplied by al is al itself, and al = 0 gives 0
  return mul_div255(p, al, 127u);
}

__device__ __forceinline__ float fix_angle_p(float x) {
  const float PI = 3.14159265358979323846f;
  while (x > PI) x -= PI * 2.0f;
  while (x < -PI) x += PI * 2.0f;
  return x;
}

// the gradient parameter t of pixel (x, y) (paints.nim:108-113, 199-209,
// 224-236)
__device__ __forceinline__ float gradient_t(const PaintArgs& a, int32_t x, int32_t y) {
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

// Four pixels to a thread; bound by the arithmetic of the colour.  4,096 x
// 4,096, radial: 83 us by single pixels with the stops read from the arguments
// lane by lane, 55 us in this form.
template <int kKind>
__global__ void __launch_bounds__(256) paint_kernel(PaintArgs a) {
  __shared__ StopTable S;
  if (kKind != 0) {
    for (int i = threadIdx.x; i < a.nstops; i += 256) {
      const float* p = a.stops + 5 * i;
      S.color[i] = make_float4(p[0], p[1], p[2], p[3]);
      S.pos[i] = p[4];
    }
    __syncthreads();
  }
  a.kind = kKind;
  const int32_t y = blockIdx.y;
  const int32_t x0 = ((int32_t)blockIdx.x * 256 + (int32_t)threadIdx.x) * 4;
  if (x0 >= a.w) return;
  const size_t i = (size_t)y * a.w + x0;
  const int n = a.w - x0 < 4 ? a.w - x0 : 4;
  uint32_t m4 = 0;
  if (n == 4) {
    __builtin_memcpy(&m4, a.mask + i, 4);
  } else {
    for (int k = 0; k < n; k++) m4 |= (uint32_t)a.mask[i + k] << (8 * k);
  }
  // a transparent source leaves the backdrop of these modes bit for bit
  const int md = a.mode;
  const bool keepOnZero = md == kNormal || md == kDarken || md == kMultiply || md == kLighten ||
                          md == kScreen || md == kOverlay || md == kHardLight || md == kDifference ||
                          md == kExclusion;
  if (m4 == 0 && keepOnZero) return;
  u32x4 d, f = (u32x4){0, 0, 0, 0};
  if (n == 4) {
    d = *(const u32x4*)(a.dst + i);
    if (kKind == 0) f = *(const u32x4*)(a.fill + i);
  } else {
    for (int k = 0; k < 4; k++) {
      d[k] = k < n ? a.dst[i + k] : 0u;
      if (kKind == 0) f[k] = k < n ? a.fill[i + k] : 0u;
    }
  }
  u32x4 src, was;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    uint32_t m = (m4 >> (8 * k)) & 255u;
    if (a.useOpacity) m = div255(m * a.o255);  // applyOpacity on the mask (images.nim:261-277)
    // image paints read the image drawn onto a transparent canvas
    const uint32_t g = kKind == 0 ? f[k] : gradient_color(a, S, gradient_t(a, x0 + k, y));
    // fill.draw(mask, MaskBlend): every channel times the mask's alpha
    src[k] = mul_div255(g, m, 0u);
    was[k] = d[k];
  }
  blend4(md, &d, src);
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (src[k] == 0u && keepOnZero) d[k] = was[k];
  if (n == 4) {
    *(u32x4*)(a.dst + i) = d;
  } else {
    for (int k = 0; k < n; k++) a.dst[i + k] = d[k];
  }
}

int launch_paint(const PaintArgs& a, hipStream_t s) {
  dim3 g((a.w + 1023) / 1024, a.h);
  if (a.kind <= 2)
    hipLaunchKernelGGL(paint_kernel<0>, g, dim3(256), 0, s, a);
  else if (a.kind == 3)
    hipLaunchKernelGGL(paint_kernel<3>, g, dim3(256), 0, s, a);
  else if (a.kind == 4)
    hipLaunchKernelGGL(paint_kernel<4>, g, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(paint_kernel<5>, g, dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// composite (blendRect): a thread takes four destination pixels, of the
// rectangle the source covers (MaskBlend: of the whole destination, which it
// clears outside that).  Bound by memory: Normal, Mask and Overwrite, whose
// arithmetic is short, are compiled alone, sources are read four pixels at a
// time at any offset, and Overwrite does not read what it replaces.  4,096 x
// 4,096 onto itself in size: Overwrite 38 -> 20 us (6.8 TB/s), an A8 mask
// 40 -> 22 us, a mode chosen at run time 34 -> 29 us.
// ---------------------------------------------------------------------------
template <bool kSrcA8, int kMode>  // kMode -1: a.mode
__global__ void __launch_bounds__(256) composite_kernel(CompositeArgs a) {
  constexpr bool whole = kMode == kMask;
  const int32_t rx0 = whole ? 0 : a.px + a.xStart, rx1 = whole ? a.aw : a.px + a.xEnd;
  const int32_t y = (int32_t)blockIdx.y + (whole ? 0 : a.py + a.yStart);  // destination row
  const int32_t x0 = rx0 + ((int32_t)blockIdx.x * 256 + (int32_t)threadIdx.x) * 4;
  if (x0 >= rx1) return;
  uint32_t* dst = a.dst + (size_t)y * a.aw + x0;
  const int32_t sy = y - a.py, sx = x0 - a.px;
  const bool rowIn = sy >= a.yStart && sy < a.yEnd;
  const size_t at = rowIn ? (size_t)sy * a.bw : 0;
  if (x0 + 4 <= rx1 && (!whole || !rowIn || (sx >= a.xStart && sx + 4 <= a.xEnd))) {  // four pixels alike
    u32x4 d = (u32x4){0, 0, 0, 0};
    if (rowIn) {
      u32x4 s;
      if (kSrcA8) {
        uint32_t v;
        __builtin_memcpy(&v, (const uint8_t*)a.src + at + sx, 4);
        s = (u32x4){(v & 255u) * 0x01010101u, ((v >> 8) & 255u) * 0x01010101u, ((v >> 16) & 255u) * 0x01010101u,
                    (v >> 24) * 0x01010101u};
      } else {
        s = *(const u32x4*)((const uint32_t*)a.src + at + sx);
      }
      if (kMode != kOverwrite) d = *(const u32x4*)dst;
      blend4(kMode >= 0 ? kMode : a.mode, &d, s);
    }
    *(u32x4*)dst = d;
    return;
  }
  for (int k = 0; k < 4 && x0 + k < rx1; k++) {
    uint32_t d = 0;
    if (rowIn && sx + k >= a.xStart && sx + k < a.xEnd) {
      const uint32_t s = kSrcA8 ? ((const uint8_t*)a.src)[at + sx + k] * 0x01010101u : ((const uint32_t*)a.src)[at + sx + k];
      d = blend(kMode >= 0 ? kMode : a.mode, dst[k], s);
    }
    dst[k] = d;
  }
}

template <bool kSrcA8>
static void go_composite(const CompositeArgs& a, hipStream_t s) {
  if (a.mode == kMask) {
    const dim3 grid((a.aw + 1023) / 1024, a.ah);
    hipLaunchKernelGGL((composite_kernel<kSrcA8, kMask>), grid, dim3(256), 0, s, a);
    return;
  }
  const int32_t w = a.xEnd - a.xStart, h = a.yEnd - a.yStart;
  if (w <= 0 || h <= 0) return;
  const dim3 grid((w + 1023) / 1024, h);
  if (a.mode == kNormal)
    hipLaunchKernelGGL((composite_kernel<kSrcA8, kNormal>), grid, dim3(256), 0, s, a);
  else if (a.mode == kOverwrite)
    hipLaunchKernelGGL((composite_kernel<kSrcA8, kOverwrite>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((composite_kernel<kSrcA8, -1>), grid, dim3(256), 0, s, a);
}

int launch_composite(const CompositeArgs& a, bool srcA8, hipStream_t s) {
  if (srcA8)
    go_composite<true>(a, s);
  else
    go_composite<false>(a, s);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// applyOpacity (images.nim:261-277), o = round(255*opacity), neither 0 nor 255
// ---------------------------------------------------------------------------
// (an opacity above 1 gives a larger o, whose products leave 16 bits)
// 4,096 x 4,096: 28 us by single pixels, 20 us by fours.
__device__ __forceinline__ uint32_t scaled(uint32_t p, uint32_t o) {
  if (o < 256u) return mul_div255(p, o, 0u);
  return pack((ch_r(p) * o) / 255u, (ch_g(p) * o) / 255u, (ch_b(p) * o) / 255u, (ch_a(p) * o) / 255u);
}
__global__ void __launch_bounds__(256) opacity_kernel(uint32_t* img, int64_t n, uint32_t o) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) {
    u32x4 p = *(const u32x4*)(img + i);
#pragma unroll
    for (int k = 0; k < 4; k++) p[k] = scaled(p[k], o);
    *(u32x4*)(img + i) = p;
  } else {
    for (int64_t k = i; k < n; k++) img[k] = scaled(img[k], o);
  }
}

int launch_opacity(uint32_t* img, int64_t n, uint32_t o, hipStream_t s) {
  hipLaunchKernelGGL(opacity_kernel, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, img, n, o);
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
