// pxh_blur.hip -- blur, shadow and spread (images.nim:304-365, 700-776) for
// gfx950.
//
//   blur_table_kernel   a radius' taps as bytes for the matrix cores
//   blur_x / blur_y     the two passes of blur on RGBA8
//   spread_x / _y       the two passes of spread, through a plane of alpha bytes
//   shadow_blur_kernel  both passes of a shadow's blur on that plane, and its
//                       colour
//   shadow_color_kernel a shadow without blur: the plane's colour
//
// A blur pass is a product with a banded matrix: out[n] = sum over k of
// in[n - r + k] * tap[k], so it runs on the matrix cores as int8 products,
// exactly: v_mfma_i32_16x16x64_i8 takes 16 lines of 64 bytes of one channel
// and 16 outputs' weights.  Bytes are signed there, so a pixel p enters as
// p - 128 (128 * sum(tap) is in the accumulator's start), and a 16-bit tap as
// 256 * hi + lo with lo in [-128, 127]; a hi over 127 (the middle tap of
// radius 1 only) is split once more.  With L and H the lo and hi sums, pixie's
// (sum div 256) div 255 is q / 255, q = H + (L >> 8) < 2^16.
#include <hip/hip_runtime.h>

#include "pxh_kernels.h"
#include "pxh_pixel.h"

namespace pxh {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// weights
// ---------------------------------------------------------------------------
// Digit d (lo, hi, the rest of hi) of tap j stands at byte kTapPad + j of a
// line with zeros around it.  A lane reads dwords at any byte of it, so each
// line is there four times, copy s shifted by s bytes: byte x is read at
// x - s of copy s = x & 3.
constexpr int kTapPad = 64;
constexpr __host__ __device__ __forceinline__ int tap_line(int r) { return (2 * r + 224) & ~15; }  // bytes
int blur_table_dwords(int r) { return 3 * tap_line(r); }

__global__ void __launch_bounds__(256) blur_table_kernel(const uint32_t* lut, int r, int8_t* tab) {
  const int len = tap_line(r);
  for (int e = threadIdx.x; e < 12 * len; e += 256) {
    const int line = e / len, d = line / 4, j = e % len + (line & 3) - kTapPad;
    const int k = j >= 0 && j <= 2 * r ? (int)lut[j] : 0;
    const int lo = (int8_t)(k & 255), hi = (k - lo) / 256, h1 = hi < 127 ? hi : 127;
    tab[e] = (int8_t)(d == 0 ? lo : d == 1 ? h1 : hi - h1);
  }
}

int launch_blur_table(const uint32_t* lut, int r, uint32_t* wtab, hipStream_t s) {
  hipLaunchKernelGGL(blur_table_kernel, dim3(1), dim3(256), 0, s, lut, r, (int8_t*)wtab);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// One lane's operand of 16 outputs' weights for 64 inputs: the bytes x + p of
// the lines, for its 16 input positions p.  kQuads: position 4i + b of the
// lane is input 16i + 4g + b (g = lane / 16), else 16g + 4i + b.
struct Weights {
  v4i lo, hi, rest;
};
template <bool kQuads>
__device__ __forceinline__ Weights load_weights(const int8_t* tab, int len, int x, bool three) {
  x += (int)(threadIdx.x & 63) / 16 * (kQuads ? 4 : 16);
  const int s = x & 3;
  const int8_t* p = tab + s * len + (x - s);
  Weights w;
  w.rest = (v4i){0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int8_t* q = p + i * (kQuads ? 16 : 4);
    w.lo[i] = *(const int*)q;
    w.hi[i] = *(const int*)(q + 4 * len);
    if (three) w.rest[i] = *(const int*)(q + 8 * len);
  }
  return w;
}

struct Sums {
  v4i lo, hi;
};
// bias: 128 * sum(tap) + 256 (so that q + 1 comes out)
__device__ __forceinline__ Sums start_sums(int bias) {
  return Sums{(v4i){bias, bias, bias, bias}, (v4i){0, 0, 0, 0}};
}
// kWeightsA: the outputs run along the result's registers (four per lane),
// the lines along its lanes; else the other way round.
template <bool kWeightsA>
__device__ __forceinline__ void add_product(Sums& s, v4i px, const Weights& w, bool three) {
  if (kWeightsA) {
    s.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.lo, px, s.lo, 0, 0, 0);
    s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.hi, px, s.hi, 0, 0, 0);
    if (three) s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(w.rest, px, s.hi, 0, 0, 0);
  } else {
    s.lo = __builtin_amdgcn_mfma_i32_16x16x64_i8(px, w.lo, s.lo, 0, 0, 0);
    s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(px, w.hi, s.hi, 0, 0, 0);
    if (three) s.hi = __builtin_amdgcn_mfma_i32_16x16x64_i8(px, w.rest, s.hi, 0, 0, 0);
  }
}

// Two sums' q / 255, in the high bytes of the result's halves: with y = q + 1,
// q / 255 is (y + (y >> 8)) >> 8 for every q < 65280 (taps add up to 65304 at
// most, so q <= 65048).
__device__ __forceinline__ uint32_t div2(int l0, int h0, int l1, int h1) {
  const u16x2 y = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm((uint32_t)l1, (uint32_t)l0, 0x06050201u)) +
                  __builtin_bit_cast(u16x2, __builtin_amdgcn_perm((uint32_t)h1, (uint32_t)h0, 0x05040100u));
  return __builtin_bit_cast(uint32_t, (u16x2)(y + (y >> 8)));
}
__device__ __forceinline__ uint32_t high_bytes(uint32_t a, uint32_t b) {
  return __builtin_amdgcn_perm(b, a, 0x07050301u);
}
// pixel i of four channels' sums
__device__ __forceinline__ uint32_t pixel_of(const Sums* c, int i) {
  return high_bytes(div2(c[0].lo[i], c[0].hi[i], c[1].lo[i], c[1].hi[i]),
                    div2(c[2].lo[i], c[2].hi[i], c[3].lo[i], c[3].hi[i]));
}

// Four RGBA8 pixels -> four channel planes (plane c, byte i = channel c of
// pixel i), less 128.
__device__ __forceinline__ void planes4(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3, int* out) {
  const uint32_t t0 = __builtin_amdgcn_perm(p1, p0, 0x05010400u);  // r0 r1 g0 g1
  const uint32_t t1 = __builtin_amdgcn_perm(p1, p0, 0x07030602u);  // b0 b1 a0 a1
  const uint32_t t2 = __builtin_amdgcn_perm(p3, p2, 0x05010400u);  // r2 r3 g2 g3
  const uint32_t t3 = __builtin_amdgcn_perm(p3, p2, 0x07030602u);  // b2 b3 a2 a3
  out[0] = (int)(__builtin_amdgcn_perm(t2, t0, 0x05040100u) ^ 0x80808080u);
  out[1] = (int)(__builtin_amdgcn_perm(t2, t0, 0x07060302u) ^ 0x80808080u);
  out[2] = (int)(__builtin_amdgcn_perm(t3, t1, 0x05040100u) ^ 0x80808080u);
  out[3] = (int)(__builtin_amdgcn_perm(t3, t1, 0x07060302u) ^ 0x80808080u);
}

// ---------------------------------------------------------------------------
// blur of RGBA8.  Every wave works by itself on 64 inputs at a time: NT tiles
// of 16 outputs that share them.  kWhole: the inputs of all NT tiles are one
// 64-input block (16 NT + 2r <= 64: NT = 3 for r up to 8, 2 up to 16), whose
// sums are finished tile by tile; else the blocks are streamed past the sums
// of all tiles.  The weights are in LDS: read from memory by every wave they
// took more of the load unit's time than the pixels.
//
// Both passes are bound by memory: of 4,096 x 4,096 at r = 8, 134 MB each, the
// X pass takes 27 us and the Y pass 24 us (5.6 TB/s), where byte dot products
// over LDS tiles took 53 and 59 us, limited by 48 dot products per pixel and
// pass.  A Y pass of 64-byte pieces (NC = 1) takes 34 us and of 256-byte ones
// 26 us (224 registers); several pieces per wave are slower, 29 to 36 us.  The
// streamed form at r = 8 takes 37 and 34 us.
// ---------------------------------------------------------------------------
template <int NT, bool kWhole, bool kThree>
struct BlurWeights {
  const int8_t* lds;
  int len;
  // all lanes of the workgroup
  __device__ __forceinline__ void init(const BlurArgs& a, int8_t* mem) {
    lds = mem;
    len = tap_line(a.radius);
    const int8_t* line = (const int8_t*)a.wtab;
    if (kWhole) {  // the operands of each tile, digit by digit
      const int wave = (int)threadIdx.x >> 6, lane = threadIdx.x & 63;
      for (int t = wave; t < NT; t += 4) {
        const Weights w = load_weights<true>(line, len, kTapPad - (lane & 15) - 16 * t, kThree);
        v4i* p = (v4i*)mem + t * 192 + lane;
        p[0] = w.lo;
        p[64] = w.hi;
        if (kThree) p[128] = w.rest;
      }
    } else {  // the lines of two digits
      for (int i = threadIdx.x; i < len / 2; i += 256) ((u32x4*)mem)[i] = ((const u32x4*)line)[i];
    }
    __syncthreads();
  }
  __device__ __forceinline__ Weights get(int n, int j, int t) const {
    if (!kWhole) return load_weights<true>(lds, len, kTapPad - n + 64 * j - 16 * t, false);
    const v4i* p = (const v4i*)lds + t * 192 + (threadIdx.x & 63);
    Weights w;
    w.lo = p[0];
    w.hi = p[64];
    w.rest = (v4i){0, 0, 0, 0};
    if (kThree) w.rest = p[128];
    return w;
  }
};

// Lets the compiler know nothing of v: what depends on it stays where it is
// (the addresses of border reads would otherwise be kept through all steps).
__device__ __forceinline__ int unknown(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// X pass: 16 rows to a wave, 16 NT columns; lane (g, n) holds row n.
template <int NT, bool kWhole, bool kThree>
__global__ void __launch_bounds__(256, kWhole ? 5 : 2) blur_x_kernel(BlurArgs a) {
  extern __shared__ __align__(16) int8_t taps[];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int x0 = ((int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * (16 * NT);
  const int r = a.radius, s0 = x0 - r, nb = kWhole ? 1 : (16 * NT + 2 * r + 63) / 64;
  BlurWeights<NT, kWhole, kThree> W;
  W.init(a, taps);
  if (x0 >= a.w) return;
  const uint32_t at = (uint32_t)n * (uint32_t)a.w + 4u * (uint32_t)g;  // the lane's first pixel from the wave's
  const int yt = (int)blockIdx.y * 16;
  const bool rows = yt + 16 <= a.h;
  auto store = [&](const Sums* s, int t) {
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) o[i] = pixel_of(s, i);
    uint32_t* out = a.dst + (size_t)yt * a.w + (x0 + 16 * t);
    if (rows && x0 + 16 * t + 16 <= a.w) {
      *(u32x4*)(out + at) = (u32x4){o[0], o[1], o[2], o[3]};
    } else if (yt + n < a.h) {
      const int x = unknown(4 * g);
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (x0 + 16 * t + x + i < a.w) out[(size_t)n * a.w + x + i] = o[i];
    }
  };
  Sums s[kWhole ? 1 : NT][4];
  if (!kWhole) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int c = 0; c < 4; c++) s[t][c] = start_sums(a.bias);
  }
  for (int j = 0; j < nb; j++) {
    const int xs = s0 + 64 * j;
    u32x4 v[4];
    if (rows && xs >= 0 && xs + 64 <= a.w) {
      const uint32_t* in = a.src + (size_t)yt * a.w + xs;
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = *(const u32x4*)(in + at + 16 * i);
    } else {
      const int y = unknown(yt + n < a.h ? yt + n : a.h - 1), x = unknown(xs + 4 * g);
      const uint32_t* in = a.src + (size_t)y * a.w;
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int xx = x + 16 * i + k;
          const uint32_t p = in[xx < 0 ? 0 : xx < a.w ? xx : a.w - 1];
          v[i][k] = (uint32_t)xx < (uint32_t)a.w ? p : a.oob;
        }
    }
    v4i px[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      int pl[4];
      planes4(v[i][0], v[i][1], v[i][2], v[i][3], pl);
#pragma unroll
      for (int c = 0; c < 4; c++) px[c][i] = pl[c];
    }
#pragma unroll
    for (int t = 0; t < NT; t++) {
      if (!kWhole && (64 * j + 63 < 16 * t || 64 * j > 16 * t + 15 + 2 * r)) continue;  // no common input
      const Weights w = W.get(n, j, t);
      if (kWhole) {
#pragma unroll
        for (int c = 0; c < 4; c++) s[0][c] = start_sums(a.bias);
      }
#pragma unroll
      for (int c = 0; c < 4; c++) add_product<true>(s[kWhole ? 0 : t][c], px[c], w, kThree);
      if (kWhole) store(s[0], t);
    }
  }
  if (!kWhole) {
#pragma unroll
    for (int t = 0; t < NT; t++) store(s[kWhole ? 0 : t], t);
  }
}

// Y pass: NC columns to a lane (16 NC to a wave), 16 NT rows; lane (g, n)
// holds columns NC n .. NC n + NC - 1, so that rows are read and written in
// pieces of 64 NC bytes.
template <int NT, int NC, bool kWhole, bool kThree>
__global__ void __launch_bounds__(256, kWhole ? 3 : 2) blur_y_kernel(BlurArgs a) {
  extern __shared__ __align__(16) int8_t taps[];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int y0 = ((int)blockIdx.y * 4 + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * (16 * NT);
  const int r = a.radius, s0 = y0 - r, nb = kWhole ? 1 : (16 * NT + 2 * r + 63) / 64;
  typedef uint32_t vec __attribute__((ext_vector_type(NC), aligned(4)));
  BlurWeights<NT, kWhole, kThree> W;
  W.init(a, taps);
  if (y0 >= a.h) return;
  const uint32_t at = 4u * (uint32_t)g * (uint32_t)a.w + (uint32_t)(NC * n);  // the lane's first pixel from the wave's
  const int xt = (int)blockIdx.x * (16 * NC);
  const bool cols = xt + 16 * NC <= a.w;
  auto store = [&](const Sums(*s)[4], int t) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      vec v;
#pragma unroll
      for (int c = 0; c < NC; c++) v[c] = pixel_of(s[c], i);
      if (cols && y0 + 16 * t + 16 <= a.h) {
        *(vec*)(a.dst + (size_t)(y0 + 16 * t + i) * a.w + xt + at) = v;
      } else {
        const int y = unknown(y0 + 16 * t + i + 4 * g);
#pragma unroll
        for (int c = 0; c < NC; c++)
          if (y < a.h && xt + NC * n + c < a.w) a.dst[(size_t)y * a.w + xt + NC * n + c] = v[c];
      }
    }
  };
  Sums s[kWhole ? 1 : NT][NC][4];
  if (!kWhole) {
#pragma unroll
    for (int t = 0; t < NT; t++)
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) s[t][c][k] = start_sums(a.bias);
  }
  for (int j = 0; j < nb; j++) {
    const int ys = s0 + 64 * j;
    vec v[4][4];
    if (cols && ys >= 0 && ys + 64 <= a.h) {
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int b = 0; b < 4; b++) v[i][b] = *(const vec*)(a.src + (size_t)(ys + 16 * i + b) * a.w + xt + at);
    } else {
      const int y = unknown(ys + 4 * g), x = unknown(xt + NC * n);
#pragma unroll
      for (int i = 0; i < 4; i++)
#pragma unroll
        for (int b = 0; b < 4; b++) {
          const int yy = y + 16 * i + b;
          const uint32_t* in = a.src + (size_t)(yy < 0 ? 0 : yy < a.h ? yy : a.h - 1) * a.w;
#pragma unroll
          for (int c = 0; c < NC; c++) {
            const uint32_t p = in[x + c < a.w ? x + c : a.w - 1];
            v[i][b][c] = (uint32_t)yy < (uint32_t)a.h ? p : a.oob;
          }
        }
    }
    v4i px[NC][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int c = 0; c < NC; c++) {
        int pl[4];
        planes4(v[i][0][c], v[i][1][c], v[i][2][c], v[i][3][c], pl);
#pragma unroll
        for (int k = 0; k < 4; k++) px[c][k][i] = pl[k];
      }
#pragma unroll
    for (int t = 0; t < NT; t++) {
      if (!kWhole && (64 * j + 63 < 16 * t || 64 * j > 16 * t + 15 + 2 * r)) continue;  // no common input
      const Weights w = W.get(n, j, t);
      if (kWhole) {
#pragma unroll
        for (int c = 0; c < NC; c++)
#pragma unroll
          for (int k = 0; k < 4; k++) s[0][c][k] = start_sums(a.bias);
      }
#pragma unroll
      for (int c = 0; c < NC; c++)
#pragma unroll
        for (int k = 0; k < 4; k++) add_product<true>(s[kWhole ? 0 : t][c][k], px[c][k], w, kThree);
      if (kWhole) store(s[0], t);
    }
  }
  if (!kWhole) {
#pragma unroll
    for (int t = 0; t < NT; t++) store(s[kWhole ? 0 : t], t);
  }
}

// LDS that a workgroup asks for: the lines of two digits (streamed blocks), and
// a shadow's columns.
constexpr size_t blur_lds(int r) { return 8 * (size_t)tap_line(r); }
constexpr int shadow_blocks(int r) { return (16 + 2 * ((r + 15) & ~15) + 63) / 64; }
constexpr size_t shadow_lds(int r) { return 64 * (48 + 64 * (size_t)shadow_blocks(r)); }

template <int NT, bool kWhole, bool kThree = false>
static void go_x(const BlurArgs& a, hipStream_t s) {
  const dim3 grid((a.w + 64 * NT - 1) / (64 * NT), (a.h + 15) / 16);
  const size_t lds = kWhole ? NT * 3072 : blur_lds(a.radius);
  hipLaunchKernelGGL((blur_x_kernel<NT, kWhole, kThree>), grid, dim3(256), lds, s, a);
}
template <int NT, int NC, bool kWhole, bool kThree = false>
static void go_y(const BlurArgs& a, hipStream_t s) {
  const dim3 grid((a.w + 16 * NC - 1) / (16 * NC), (a.h + 64 * NT - 1) / (64 * NT));
  const size_t lds = kWhole ? NT * 3072 : blur_lds(a.radius);
  hipLaunchKernelGGL((blur_y_kernel<NT, NC, kWhole, kThree>), grid, dim3(256), lds, s, a);
}

int launch_blur(const BlurArgs& ax, const BlurArgs& ay, hipStream_t s) {
  const int r = ax.radius;
  if (r == 1) {
    go_x<3, true, true>(ax, s);
    go_y<3, 2, true, true>(ay, s);
  } else if (r <= 8) {
    go_x<3, true>(ax, s);
    go_y<3, 2, true>(ay, s);
  } else if (r <= 16) {
    go_x<2, true>(ax, s);
    go_y<2, 2, true>(ay, s);
  } else {
    go_x<4, false>(ax, s);
    go_y<2, 2, false>(ay, s);
  }
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// The radii that are accepted stay those of the form before the matrix
// products: 1,024-pixel row segments and 64 x 64 tiles of four channel planes,
// with their borders and weights, in a workgroup's LDS (276 at 160 KB).  All of
// them ask for less than the 64 KB that a launch gets without an attribute.
constexpr bool blur_radius_accepted(int r, size_t lds) {
  const size_t nd = (size_t)(2 * (int64_t)r + 10) / 4;
  return (256 + 3 * nd) * 16 <= lds && (15 + nd) * 1024 + nd * 32 <= lds;
}
constexpr int kMaxRadius = 276;
static_assert(blur_radius_accepted(kMaxRadius, 160 << 10) && !blur_radius_accepted(kMaxRadius + 1, 160 << 10),
              "the largest radius");
static_assert(blur_lds(kMaxRadius) <= 64 << 10 && shadow_lds(kMaxRadius) + 1024 <= 64 << 10, "no LDS attribute is set");
bool blur_radius_fits(int r, size_t lds) { return r <= kMaxRadius && blur_radius_accepted(r, lds); }

// Writes a Gaussian table passed by value into device memory (the
// allocation-free blur keeps its table in static device scratch).
__global__ void __launch_bounds__(256) lut_store_kernel(LutTaps t, uint32_t* dst) {
  for (int i = threadIdx.x; i < t.n; i += 256) dst[i] = t.v[i];
}

int launch_lut_store(const LutTaps& t, uint32_t* dst, hipStream_t s) {
  hipLaunchKernelGGL(lut_store_kernel, dim3(1), dim3(256), 0, s, t, dst);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// spread, on alpha bytes in a plane whose rows are padded with zeros to a
// multiple of 16.  The window is clamped to the image.  A negative spread
// takes the least of the window: the greatest of the complements.  Bytes are
// compared as the 16-bit halves of even and odd bytes.  Bound by latency at the
// sizes of layers, so each pass has several loads in flight.  1,921 x 1,081,
// both passes: 15 us at spread 4 and 29 at 20; a pixel to a thread 27 and 82.
// ---------------------------------------------------------------------------
struct MaxBytes {
  u16x2 even = {0, 0}, odd = {0, 0};
  __device__ __forceinline__ void add(uint32_t v) {
    const u16x2 e = __builtin_bit_cast(u16x2, v & 0x00ff00ffu), o = __builtin_bit_cast(u16x2, (v >> 8) & 0x00ff00ffu);
    even = __builtin_elementwise_max(even, e);
    odd = __builtin_elementwise_max(odd, o);
  }
  __device__ __forceinline__ uint32_t get() const {
    return __builtin_bit_cast(uint32_t, even) | (__builtin_bit_cast(uint32_t, odd) << 8);
  }
};

// Four pixels from x of a row of the translated source: loaded at once, or
// one by one at clamped addresses where they reach over a border (kSingles:
// always, so that lanes at a border and lanes inside take one way), so that
// several of these are in flight before the first is used.
struct Quad {
  u32x4 v;
  bool inside;
};
template <bool kSingles>
__device__ __forceinline__ Quad load_quad(const SpreadArgs& a, const uint32_t* row, int32_t x) {
  const int32_t sx = x - a.dx;
  Quad q;
  q.inside = x >= 0 && x + 4 <= a.w && row && sx >= 0 && sx + 4 <= a.w;
  if (!kSingles && q.inside) {
    q.v = *(const u32x4*)(row + sx);
  } else {
    const uint32_t* from = row ? row : a.src;
#pragma unroll
    for (int i = 0; i < 4; i++) q.v[i] = from[sx + i < 0 ? 0 : sx + i < a.w ? sx + i : a.w - 1];
  }
  return q;
}
// Their alphas, flipped by `flip` inside the image and 0 outside it.
__device__ __forceinline__ uint32_t alphas4(const SpreadArgs& a, const uint32_t* row, int32_t x, const Quad& q,
                                            uint32_t flip) {
  uint32_t out = __builtin_amdgcn_perm(q.v[1], q.v[0], 0x0c0c0703u) | __builtin_amdgcn_perm(q.v[3], q.v[2], 0x07030c0cu);
  if (!q.inside) {
    const int32_t sx = x - a.dx;
    uint32_t in = 0;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (!(row && sx + i >= 0 && sx + i < a.w)) out &= ~(255u << (8 * i));
      if (x + i >= 0 && x + i < a.w) in |= 255u << (8 * i);
    }
    return (out ^ flip) & in;
  }
  return out ^ flip;
}

// X pass, four pixels to a thread; s = 0 only takes the translated alphas.
template <bool kSingles>
__global__ void __launch_bounds__(256) spread_x_kernel(SpreadArgs a) {
  const int32_t y = blockIdx.y, x = ((int32_t)blockIdx.x * 256 + (int32_t)threadIdx.x) * 4;
  if (x >= a.pitch) return;
  const uint32_t flip = a.grow ? 0u : ~0u;
  const int64_t sy = (int64_t)y - a.dy;
  const uint32_t* row = sy >= 0 && sy < a.h ? a.src + (size_t)sy * a.w : nullptr;
  uint32_t out = 0;
  if (x < a.w) {
    const int32_t s = a.s;
    // dwords from x holding offsets -s .. s, and part of the image
    int32_t m0 = -((s + 3) / 4), m1 = s / 4;
    m0 = m0 < -x / 4 - 1 ? -x / 4 - 1 : m0;
    m1 = m1 > (a.w - 1 - x) / 4 ? (a.w - 1 - x) / 4 : m1;
    auto get = [&](int32_t m, const Quad& q) { return alphas4(a, row, x + 4 * m, q, flip); };
    Quad q0 = load_quad<kSingles>(a, row, x + 4 * m0);
    MaxBytes best;
    auto take = [&](int32_t m, uint32_t cur, uint32_t next) {
      if (4 * m >= -s) best.add(cur);
      if (4 * m + 1 >= -s && 4 * m + 1 <= s) best.add(__builtin_amdgcn_alignbyte(next, cur, 1));
      if (4 * m + 2 >= -s && 4 * m + 2 <= s) best.add(__builtin_amdgcn_alignbyte(next, cur, 2));
      if (4 * m + 3 >= -s && 4 * m + 3 <= s) best.add(__builtin_amdgcn_alignbyte(next, cur, 3));
    };
    if (s == 0) {
      best.add(get(0, q0));
    } else {
      uint32_t cur = 0;
      for (int32_t m = m0; m <= m1; m += 2) {
        const Quad q1 = load_quad<kSingles>(a, row, x + 4 * (m + 1)), q2 = load_quad<kSingles>(a, row, x + 4 * (m + 2));
        if (m == m0) cur = get(m, q0);
        const uint32_t n1 = get(m + 1, q1), n2 = get(m + 2, q2);
        take(m, cur, n1);
        if (m < m1) take(m + 1, n1, n2);
        cur = n2;
      }
    }
    out = best.get() ^ flip;
    if (x + 4 > a.w) out &= (1u << (8 * (a.w - x))) - 1u;
  }
  *(uint32_t*)(a.plane + (size_t)y * a.pitch + x) = out;
}

// Y pass, four pixels of kRows rows to a thread: into the second plane, or
// into an image of black with that alpha.
template <bool kImage, int kRows>
__global__ void __launch_bounds__(256) spread_y_kernel(SpreadArgs a) {
  const int32_t y0 = (int32_t)blockIdx.y * kRows, x = ((int32_t)blockIdx.x * 256 + (int32_t)threadIdx.x) * 4;
  if (x >= (kImage ? a.w : a.pitch)) return;
  const uint32_t flip = a.grow ? 0u : ~0u;
  const int32_t s = a.s;
  const int32_t lo = y0 - s > 0 ? y0 - s : 0, hi = (int64_t)y0 + kRows - 1 + s < a.h - 1 ? y0 + kRows - 1 + s : a.h - 1;
  MaxBytes best[kRows];
  // four rows in flight; past the end the last again
  auto four = [&](int32_t yb, bool clamp) {
    uint32_t v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
      v[u] = *(const uint32_t*)(a.plane + (size_t)(clamp && yb + u > hi ? hi : yb + u) * a.pitch + x) ^ flip;
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int i = 0; i < kRows; i++) {
        const int32_t d = (clamp && yb + u > hi ? hi : yb + u) - (y0 + i);
        if (d >= -s && d <= s) best[i].add(v[u]);
      }
  };
  int32_t yb = lo;
  for (; yb + 3 <= hi; yb += 4) four(yb, false);
  if (yb <= hi) four(yb, true);
#pragma unroll
  for (int i = 0; i < kRows; i++) {
    if (y0 + i >= a.h) break;
    const uint32_t v = best[i].get() ^ flip;
    if (!kImage) {
      *(uint32_t*)(a.plane2 + (size_t)(y0 + i) * a.pitch + x) = v;
      continue;
    }
    uint32_t* out = a.dst + (size_t)(y0 + i) * a.w + x;
    if (x + 3 < a.w) {
      *(u32x4*)out = (u32x4){v << 24, (v << 16) & 0xff000000u, (v << 8) & 0xff000000u, v & 0xff000000u};
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (x + k < a.w) out[k] = (v << (24 - 8 * k)) & 0xff000000u;
    }
  }
}

// A small image does not fill the chip with four rows to a thread, and each of
// its waves reaches over a border: its Y pass takes a row to a thread, its X
// pass loads single pixels.  257 x 199, spread 1 and 20: 5.9 and 12.1 us,
// 6.8 and 15.9 as larger images; 1,023 x 767 fills the chip either way.
constexpr int64_t kSmallPlane = 1 << 19;  // bytes
int launch_spread_x(const SpreadArgs& a, hipStream_t s) {
  const dim3 grid((a.pitch + 1023) / 1024, a.h);
  if ((int64_t)a.pitch * a.h <= kSmallPlane)
    hipLaunchKernelGGL(spread_x_kernel<true>, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(spread_x_kernel<false>, grid, dim3(256), 0, s, a);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}
template <int kRows>
static void go_spread_y(const SpreadArgs& a, bool image, hipStream_t s) {
  const dim3 grid((a.pitch + 1023) / 1024, (a.h + kRows - 1) / kRows);
  if (image)
    hipLaunchKernelGGL((spread_y_kernel<true, kRows>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((spread_y_kernel<false, kRows>), grid, dim3(256), 0, s, a);
}
int launch_spread_y(const SpreadArgs& a, bool image, hipStream_t s) {
  if ((int64_t)a.pitch * a.h <= kSmallPlane)
    go_spread_y<1>(a, image, s);
  else
    go_spread_y<4>(a, image, s);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

// ---------------------------------------------------------------------------
// a shadow's blur: its image holds black with alpha, so only the alpha plane
// is blurred, transparent outside.  A workgroup takes 64 x 64 outputs: the X
// pass of their rows and borders goes to LDS, transposed (byte y of line x),
// where the Y pass finds its 64 inputs in 16-byte reads.  Windows of
// 16 outputs start R before them, R the radius rounded up to a multiple of
// 16, so that reads are aligned.  fill(color).draw(mask, MaskBlend) is a table
// of 256 colours.  Bound by latency at the sizes of layers: 1,921 x 1,081 at
// r = 16 takes 8 us, where the two passes on RGBA8 took 15 and 20 us.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int shadow_border(int r) { return (r + 15) & ~15; }

__device__ __forceinline__ uint32_t bytes_of(const Sums& s) {
  return high_bytes(div2(s.lo[0], s.hi[0], s.lo[1], s.hi[1]), div2(s.lo[2], s.hi[2], s.lo[3], s.hi[3]));
}

__device__ __forceinline__ void store_colors(uint32_t* out, int32_t x, int32_t w, uint32_t v, const uint32_t* color) {
  if (x + 3 < w) {
    *(u32x4*)(out + x) = (u32x4){color[v & 255u], color[(v >> 8) & 255u], color[(v >> 16) & 255u], color[v >> 24]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (x + i < w) out[x + i] = color[(v >> (8 * i)) & 255u];
  }
}

template <bool kOneBlock>
__global__ void __launch_bounds__(256) shadow_blur_kernel(ShadowArgs a) {
  extern __shared__ __align__(16) uint8_t tcol[];  // 64 lines of `pitch` bytes
  __shared__ uint32_t color[256];
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int R = shadow_border(a.radius), len = tap_line(a.radius);
  const int nb = kOneBlock ? 1 : (16 + 2 * R + 63) / 64;
  const int pitch = 48 + 64 * nb;  // an odd multiple of 16: no bank is met twice
  const int x0 = (int)blockIdx.x * 64, y0 = (int)blockIdx.y * 64;
  const bool three = a.radius == 1;
  const int8_t* tab = (const int8_t*)a.wtab;
  const int first = kTapPad - n - (R - a.radius);
  color[threadIdx.x] = blend(kMask, a.color, (uint32_t)threadIdx.x << 24);
  Weights w = load_weights<false>(tab, len, first, three);
  // X pass: 16 rows by 16 columns at a time
  for (int u = wave; u < (64 + 2 * R) / 4; u += 4) {
    const int y = y0 - R + (u >> 2) * 16 + n, xs = x0 - R + (u & 3) * 16 + 16 * g;
    Sums s = start_sums(a.bias);
    for (int j = 0; j < nb; j++) {
      const int x = xs + 64 * j;
      v4i px = {0, 0, 0, 0};
      if (y >= 0 && y < a.h && x >= 0 && x < a.pitch) px = *(const v4i*)(a.plane + (size_t)y * a.pitch + x);
      px ^= (int)0x80808080;
      if (!kOneBlock) w = load_weights<false>(tab, len, first + 64 * j, three);
      add_product<false>(s, px, w, three);
    }
    *(uint32_t*)(tcol + ((u & 3) * 16 + n) * pitch + (u >> 2) * 16 + 4 * g) = bytes_of(s) ^ 0x80808080u;
  }
  __syncthreads();
  // Y pass: 16 columns by 16 rows at a time
  for (int u = wave; u < 16; u += 4) {
    const int xc = (u & 3) * 16, yr = (u >> 2) * 16;
    if (x0 + xc >= a.w || y0 + yr >= a.h) continue;
    Sums s = start_sums(a.bias);
    for (int j = 0; j < nb; j++) {
      const v4i px = *(const v4i*)(tcol + (xc + n) * pitch + yr + 16 * g + 64 * j);
      if (!kOneBlock) w = load_weights<false>(tab, len, first + 64 * j, three);
      add_product<false>(s, px, w, three);
    }
    const int y = y0 + yr + n;
    if (y < a.h) store_colors(a.dst + (size_t)y * a.w, x0 + xc + 4 * g, a.w, bytes_of(s), color);
  }
}

__global__ void __launch_bounds__(256) shadow_color_kernel(ShadowArgs a) {
  __shared__ uint32_t color[256];
  color[threadIdx.x] = blend(kMask, a.color, (uint32_t)threadIdx.x << 24);
  __syncthreads();
  const int32_t x = ((int32_t)blockIdx.x * 256 + (int32_t)threadIdx.x) * 4, y = blockIdx.y;
  if (x >= a.w) return;
  store_colors(a.dst + (size_t)y * a.w, x, a.w, *(const uint32_t*)(a.plane + (size_t)y * a.pitch + x), color);
}

int launch_shadow(const ShadowArgs& a, hipStream_t s) {
  const dim3 grid((a.w + 63) / 64, (a.h + 63) / 64);
  if (a.radius == 0) {
    hipLaunchKernelGGL(shadow_color_kernel, dim3((a.w + 1023) / 1024, a.h), dim3(256), 0, s, a);
  } else {
    const int nb = shadow_blocks(a.radius);
    const size_t lds = shadow_lds(a.radius);
    if (nb == 1)
      hipLaunchKernelGGL(shadow_blur_kernel<true>, grid, dim3(256), lds, s, a);
    else
      hipLaunchKernelGGL(shadow_blur_kernel<false>, grid, dim3(256), lds, s, a);
  }
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

}  // namespace pxh
