// pxh_raster.h -- the per-row raster program of fillShapes (paths.nim:1631-1908)
// as wave-level (64-lane) device code, and its fused scan -> paint -> blend ->
// write-back epilogue.  Included by the HIP translation units only.
//
// One wavefront owns one (fill, row, window) item.  The row program decides
// pixie's per-row path (two-spanning fill, trapezoid, 5-sample coverage or
// 1-sample fill), computes the row's pixel operations as runs of codes and
// adds them to a difference array D in LDS.  The epilogue prefix-scans D
// across the window (one wave scan per 256 pixels) and applies each pixel's
// operation to the canvas in HBM with 16-byte accesses.
//
// Pixel codes (prefix sums of D):
//   coverage rows: 0..255 = accumulated coverage; kClear = cleared (mask mode)
//   other rows:    0 = untouched, kFill = blend with paint, kArea = blend with
//                  paint * AX[x] (trapezoid sliver), kClear = cleared
#pragma once

#include <hip/hip_runtime.h>

#include "pxh_common.h"
#include "pxh_geom.h"
#include "pxh_pixel.h"

namespace pxh {

constexpr int kWave = 64;
constexpr int32_t kFill = 256;
constexpr int32_t kArea = 512;
constexpr int32_t kClear = 1024;

enum RowKind : int32_t { kRowNone = 0, kRowCoverage = 1, kRowOps = 2 };

// Per-wave row scratch.  cap = capacity (power of two >= 64) for selected
// entries / hits of one row; ww = window width in pixels (multiple of 256).
// D and AX always live in LDS; the cap-sized arrays live in LDS when they fit
// and otherwise in a per-wave global scratch slot (same code either way).
struct RowLds {
  int32_t* D;        // ww + 4: difference array of pixel codes
  uint32_t* AX;      // ww: coverage factor of trapezoid sliver pixels
  uint64_t* keys;    // cap: sort keys (value << 32 | position)
  int32_t* A;        // cap: selected entries (band-local indices)
  int32_t* B;        // cap: reordered selection / hit windings by position
  float* tx0;        // cap: trapezoid x at scanTop (by selection position)
  float* tx1;        // cap: trapezoid x at scanBottom
  int cap, ww;
  uint32_t* stage;   // LDS staging of the wide path's hit keys: AX, which
  int stageCap;      // coverage rows leave free
};

PXH_HD size_t row_lds_fixed_bytes(int ww) { return (size_t)(ww + 4) * 4 + (size_t)ww * 4; }
PXH_HD size_t row_cap_bytes(int cap) { return (size_t)cap * 24; }

// D/AX from `fixed` (LDS), cap arrays from `arr` (LDS or global).
__device__ __forceinline__ RowLds row_lds_carve(char* fixed, char* arr, int cap, int ww) {
  RowLds L;
  L.cap = cap;
  L.ww = ww;
  L.D = (int32_t*)fixed;
  L.AX = (uint32_t*)(L.D + ww + 4);
  L.keys = (uint64_t*)arr;
  L.A = (int32_t*)(L.keys + cap);
  L.B = L.A + cap;
  L.tx0 = (float*)(L.B + cap);
  L.tx1 = L.tx0 + cap;
  L.stage = L.AX;
  L.stageCap = ww;
  return L;
}

__device__ __forceinline__ int lane_id() { return threadIdx.x & (kWave - 1); }

__device__ __forceinline__ uint64_t ballot(bool p) { return __ballot(p); }

// Wave-wide scans with DPP lane moves (GFX9 row_shr / row_bcast): a
// Hillis-Steele scan inside each 16-lane row, then rows 1..3 pick up the
// totals of the rows before them.  Lanes a move has no source for keep the
// identity.  No LDS traffic, about two VALU operations per step.
constexpr int kDppRowShr1 = 0x111, kDppRowShr2 = 0x112, kDppRowShr4 = 0x114,
              kDppRowShr8 = 0x118, kDppRowBcast15 = 0x142, kDppRowBcast31 = 0x143,
              kDppWaveShr1 = 0x138, kDppWaveShl1 = 0x130;

// Where this workgroup adds the pixels it wrote: one of kTouchSlots counters,
// 64 bytes apart.  On one address the additions of thousands of workgroups
// wait for each other, 10 to 20 ns each: a fill of 8,192 workgroups took
// 118 us, and 46 us spread; the composition of a page of text 89 and 48 us.
__device__ __forceinline__ unsigned long long* touched_slot(unsigned long long* slots) {
  return slots + (size_t)(blockIdx.x % kTouchSlots) * 8;
}

// A value that is the same in every lane, moved to a scalar register.
__device__ __forceinline__ int32_t uni(int32_t v) { return __builtin_amdgcn_readfirstlane(v); }

__device__ __forceinline__ int32_t wave_incl_sum(int32_t v) {
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowShr1, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowShr2, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowShr4, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowShr8, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowBcast15, 0xa, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowBcast31, 0xc, 0xf, false);
  return v;
}

__device__ __forceinline__ int32_t imax(int32_t a, int32_t b) { return a > b ? a : b; }

__device__ __forceinline__ int32_t wave_incl_max(int32_t v) {
  const int32_t lo = INT32_MIN;
  v = imax(v, __builtin_amdgcn_update_dpp(lo, v, kDppRowShr1, 0xf, 0xf, false));
  v = imax(v, __builtin_amdgcn_update_dpp(lo, v, kDppRowShr2, 0xf, 0xf, false));
  v = imax(v, __builtin_amdgcn_update_dpp(lo, v, kDppRowShr4, 0xf, 0xf, false));
  v = imax(v, __builtin_amdgcn_update_dpp(lo, v, kDppRowShr8, 0xf, 0xf, false));
  v = imax(v, __builtin_amdgcn_update_dpp(lo, v, kDppRowBcast15, 0xa, 0xf, false));
  v = imax(v, __builtin_amdgcn_update_dpp(lo, v, kDppRowBcast31, 0xc, 0xf, false));
  return v;
}

// Exclusive prefix sum over the wave; *total receives the wave's sum.
__device__ __forceinline__ int32_t wave_excl_scan(int32_t v, int32_t* total) {
  int32_t x = wave_incl_sum(v);
  *total = __builtin_amdgcn_readlane(x, kWave - 1);
  return x - v;
}

// Exclusive prefix max (INT32_MIN in lane 0).
__device__ __forceinline__ int32_t wave_excl_max(int32_t v) {
  int32_t x = wave_incl_max(v);
  return __builtin_amdgcn_update_dpp(INT32_MIN, x, kDppWaveShr1, 0xf, 0xf, false);
}

__device__ __forceinline__ int32_t wave_max(int32_t v) {
  return __builtin_amdgcn_readlane(wave_incl_max(v), kWave - 1);
}

// Orders the wave's own LDS and scratch accesses: one lane's stores before
// the fence are seen by every lane's loads after it (a wave's memory
// operations run in order).  Not a workgroup barrier, so the waves of a
// larger workgroup may run row programs independently.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---- 32-bit key sorts in registers ----
// Value of the lane whose number differs in bit S (S = 1, 2, 4, 8), by DPP
// moves inside a 16-lane row.
constexpr int kDppQuadXor1 = 0xB1, kDppQuadXor2 = 0x4E, kDppQuadXor3 = 0x1B, kDppHalfMirror = 0x141,
              kDppRowRor8 = 0x128;
template <int S>
__device__ __forceinline__ uint32_t lane_xor(uint32_t v) {
  if (S == 1) return __builtin_amdgcn_mov_dpp(v, kDppQuadXor1, 0xf, 0xf, true);
  if (S == 2) return __builtin_amdgcn_mov_dpp(v, kDppQuadXor2, 0xf, 0xf, true);
  if (S == 4)  // i -> 7 - i inside eight lanes, then i -> 3 - i inside four
    return __builtin_amdgcn_mov_dpp(__builtin_amdgcn_mov_dpp(v, kDppHalfMirror, 0xf, 0xf, true), kDppQuadXor3,
                                    0xf, 0xf, true);
  return __builtin_amdgcn_mov_dpp(v, kDppRowRor8, 0xf, 0xf, true);
}
// Compare-exchange with the lane at distance S: the lower lane of the pair
// keeps the smaller key.  At 16 and 32 the lane swaps of gfx950 give every
// lane both keys of its pair.
template <int S>
__device__ __forceinline__ uint32_t cmp_exchange(uint32_t k, bool lower) {
  uint32_t a = k, b;
  if (S == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(k, k, false, false);
    a = r[0];
    b = r[1];
  } else if (S == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(k, k, false, false);
    a = r[0];
    b = r[1];
  } else {
    b = lane_xor<S>(k);
  }
  const uint32_t mn = a < b ? a : b, mx = a < b ? b : a;
  return lower ? mn : mx;
}

// Ascending bitonic sort inside every SEG-lane segment of the wave.
template <int SEG>
__device__ __forceinline__ uint32_t seg_sort32(uint32_t k) {
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t held = 0;
#pragma unroll
  for (int size = 2; size <= SEG; size <<= 1) {
    const uint32_t want = size < SEG ? (uint32_t)-(int32_t)((lane & size) != 0) : 0u;
    k ^= held ^ want;
    held = want;
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const bool lower = (lane & stride) == 0;
      if (stride == 16) k = cmp_exchange<16>(k, lower);
      if (stride == 8) k = cmp_exchange<8>(k, lower);
      if (stride == 4) k = cmp_exchange<4>(k, lower);
      if (stride == 2) k = cmp_exchange<2>(k, lower);
      if (stride == 1) k = cmp_exchange<1>(k, lower);
    }
  }
  return k;
}

// Ascending bitonic sort of the 64 * NS keys k[s] of lane l (key s * 64 + l).
// Blocks a stage sorts downwards are held complemented meanwhile, so every
// exchange keeps the minimum in the lower place: 3 to 5 VALU instructions
// per exchange and no LDS traffic, against two LDS permutes and about ten
// VALU instructions for 64-bit keys.
template <int NS>
__device__ __forceinline__ void wave_sort32(uint32_t (&k)[NS]) {
  const int lane = threadIdx.x & (kWave - 1);
  uint32_t held = 0;  // complement now applied by lane
#pragma unroll
  for (int size = 2; size <= kWave * NS; size <<= 1) {
    const uint32_t want = size < kWave ? (uint32_t)-(int32_t)((lane & size) != 0) : 0u;
#pragma unroll
    for (int s = 0; s < NS; s++) {
      const uint32_t slotWas = size > kWave && (((s * kWave) & (size >> 1)) != 0) ? ~0u : 0u;
      const uint32_t slotNow = size >= kWave && size < kWave * NS && (((s * kWave) & size) != 0) ? ~0u : 0u;
      k[s] ^= held ^ want ^ slotWas ^ slotNow;
    }
    held = want;
#pragma unroll
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      if (stride >= kWave) {
        const int d = stride / kWave;
#pragma unroll
        for (int s = 0; s < NS; s++) {
          if (s & d) continue;
          const uint32_t a = k[s], b = k[s | d];
          k[s] = a < b ? a : b;
          k[s | d] = a < b ? b : a;
        }
        continue;
      }
      const bool lower = (lane & stride) == 0;
#pragma unroll
      for (int s = 0; s < NS; s++) {
        if (stride == 32) k[s] = cmp_exchange<32>(k[s], lower);
        if (stride == 16) k[s] = cmp_exchange<16>(k[s], lower);
        if (stride == 8) k[s] = cmp_exchange<8>(k[s], lower);
        if (stride == 4) k[s] = cmp_exchange<4>(k[s], lower);
        if (stride == 2) k[s] = cmp_exchange<2>(k[s], lower);
        if (stride == 1) k[s] = cmp_exchange<1>(k[s], lower);
      }
    }
  }
}

// Ascending sort of n keys in memory by one wave, any n: a bitonic network
// whose every exchange points upwards (each merge starts with a mirrored
// pass), so keys past n act as the largest and are left out.
__device__ __forceinline__ void wave_sort32_mem(uint32_t* keys, int n) {
  const int lane = threadIdx.x & (kWave - 1);
  int np = 2;
  while (np < n) np <<= 1;
  for (int size = 2; size <= np; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      const bool mirror = stride == (size >> 1);
      for (int t = lane; t < np / 2; t += kWave) {
        const int r = t & (stride - 1);
        const int i = 2 * t - r;
        const int j = mirror ? i + 2 * (stride - r) - 1 : i + stride;
        if (j < n) {
          const uint32_t a = keys[i], b = keys[j];
          if (a > b) {
            keys[i] = b;
            keys[j] = a;
          }
        }
      }
      wave_sync();
    }
  }
}

// Bitonic sort of n keys in L.keys (n <= cap, cap a power of two).  Keys
// beyond n are padded with UINT64_MAX.  The whole wave participates.
__device__ void wave_sort_keys(uint64_t* keys, int n, int cap) {
  int lane = lane_id();
  int np = 64;
  while (np < n) np <<= 1;
  if (np > cap) np = cap;  // n <= cap guaranteed by the caller
  if (n <= 32) {
    // rank sort: keys are distinct (their low word is the position), so each
    // lane's rank is the number of smaller keys, found by broadcasting every
    // key in turn
    uint64_t k = lane < n ? keys[lane] : ~0ull;
    uint32_t klo = (uint32_t)k, khi = (uint32_t)(k >> 32);
    int rank = 0;
    for (int j = 0; j < n; j++) {
      uint32_t jlo = __builtin_amdgcn_readlane(klo, j), jhi = __builtin_amdgcn_readlane(khi, j);
      rank += (jhi < khi || (jhi == khi && jlo < klo)) ? 1 : 0;
    }
    wave_sync();
    if (lane < n) keys[rank] = k;
    wave_sync();
    return;
  }
  for (int i = n + lane; i < np; i += kWave) keys[i] = ~0ull;
  wave_sync();
  if (np == 64) {
    uint64_t k = keys[lane];
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1) {
#pragma unroll
      for (int stride = size >> 1; stride > 0; stride >>= 1) {
        uint64_t o = __shfl_xor(k, stride, kWave);
        bool up = ((lane & size) == 0);
        bool lower = (lane & stride) == 0;
        uint64_t mn = k < o ? k : o, mx = k < o ? o : k;
        k = (lower == up) ? mn : mx;
      }
    }
    keys[lane] = k;
    wave_sync();
    return;
  }
  for (int size = 2; size <= np; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int t = lane; t < np / 2; t += kWave) {
        int i = 2 * t - (t & (stride - 1));
        int j = i + stride;
        bool up = ((i & size) == 0);
        uint64_t a = keys[i], b = keys[j];
        if ((a > b) == up) {
          keys[i] = b;
          keys[j] = a;
        }
      }
      wave_sync();
    }
  }
}

// Order-preserving map of a float to an unsigned key (finite values).
__device__ __forceinline__ uint32_t float_key(float f) {
  uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

struct RowCtx {
  const FillInfo* F;
  const PartInfo* parts;  // this fill's partitions
  const Entry* E;         // this fill's entries
  const int8_t* EW;       // windings
  int32_t y;
  int32_t wx0, wx1;       // window [wx0, wx1)
  int32_t cx0, cx1;       // clip of this row's writes
};

// Adds value v to pixels [a, b) of the window (clipped), via D.
__device__ __forceinline__ void add_run(const RowCtx& C, RowLds& L, int64_t a, int64_t b, int32_t v) {
  int64_t lo = a > C.cx0 ? a : C.cx0;
  int64_t hi = b < C.cx1 ? b : C.cx1;
  if (lo < C.wx0) lo = C.wx0;
  if (hi > C.wx1) hi = C.wx1;
  if (lo >= hi) return;
  atomicAdd(&L.D[lo - C.wx0], v);
  atomicAdd(&L.D[hi - C.wx0], -v);
}

// The walk iterator (paths.nim:1298-1330) over the n sorted hits in L.keys
// (at in the high word, hit position in the low word; windings in L.B by
// position), executed in parallel.  Calls span(prevAt, at) per yielded span.
__device__ __forceinline__ int32_t key_at(uint64_t k) {
  return (int32_t)((uint32_t)(k >> 32) ^ 0x80000000u);
}

// kPacked: the winding is the key's low byte (keys (x, index << 8 | winding))
// instead of L.B[low word].
__device__ __forceinline__ int32_t key_winding(uint64_t k) { return (int32_t)(int8_t)(uint8_t)k; }

// Walk state carried from one 64-hit chunk to the next.
struct WalkCarry {
  int32_t count = 0;      // winding count before the chunk
  int32_t prev = 0;       // prevAt so far (0 before any event)
  bool consumed = false;  // the chunk's first hit was consumed by a skip
};

// One chunk of the walk: lane i holds a sorted hit (at, w) when valid and,
// when hasNext, the hit after it (nextAt, nextW), which for the last lane is
// the next chunk's first hit.  Yields pixie's spans in parallel: winding
// counts by prefix sum, the zero-width skip of a cancelling pair by ballots
// (a skip consumes the next hit, so skips are taken left to right), the
// NonZero shortcut per lane, and prevAt as an exclusive prefix max of the
// event positions.
template <class SpanFn>
__device__ __forceinline__ void walk_chunk(int32_t at, int32_t w, bool valid, bool hasNext, int32_t nextAt,
                                           int32_t nextW, int32_t rule, WalkCarry& c, SpanFn& span) {
  const int lane = lane_id();
  int32_t tot;
  const int32_t countBefore = c.count + wave_excl_scan(w, &tot);
  const bool filling = should_fill(rule, countBefore);
  const bool canSkip = valid && at > 0 && filling && hasNext && nextAt == at && w + nextW == 0;
  uint64_t cm = ballot(canSkip);
  uint64_t skipMask = 0, consMask = c.consumed ? 1ull : 0ull;
  bool carryOut = false;
  while (cm) {
    const int b = __builtin_ctzll(cm);
    cm &= cm - 1;
    if (!((consMask >> b) & 1ull)) {
      skipMask |= 1ull << b;
      if (b + 1 < kWave) consMask |= 1ull << (b + 1);
      else carryOut = true;
    }
  }
  const bool consumed = (consMask >> lane) & 1ull;
  const bool skipStart = (skipMask >> lane) & 1ull;
  // 0 = none, 1 = start (prevAt = at), 2 = end (yield, prevAt = at)
  int ev = 0;
  if (valid && !consumed && !skipStart && at > 0) {
    if (filling) {
      const bool cont = (rule == kNonZero) && hasNext && (countBefore + w != 0);
      ev = cont ? 0 : 2;
    } else {
      ev = 1;
    }
  }
  const int32_t prevHere = wave_excl_max(ev ? at : INT32_MIN);
  const int32_t prevAt = prevHere > c.prev ? prevHere : c.prev;
  if (ev == 2) span(prevAt, at);
  const int32_t lastEv = wave_max(ev ? at : INT32_MIN);
  if (lastEv > c.prev) c.prev = lastEv;
  c.count += tot;
  c.consumed = carryOut;
}

template <bool kPacked = false, class SpanFn>
__device__ void wave_walk(RowLds& L, int n, int32_t rule, SpanFn& span) {
  const int lane = lane_id();
  WalkCarry c;
  for (int base = 0; base < n; base += kWave) {
    const int i = base + lane;
    const bool valid = i < n;
    const uint64_t k = valid ? L.keys[i] : 0ull;
    const int32_t at = valid ? key_at(k) : 0;
    const int32_t w = valid ? (kPacked ? key_winding(k) : L.B[(uint32_t)k]) : 0;
    const bool hasNext = valid && i < n - 1;
    const uint64_t kn = hasNext ? L.keys[i + 1] : 0ull;
    const int32_t nextAt = hasNext ? key_at(kn) : 0;
    const int32_t nextW = hasNext ? (kPacked ? key_winding(kn) : L.B[(uint32_t)kn]) : 0;
    walk_chunk(at, w, valid, hasNext, nextAt, nextW, rule, c, span);
  }
}

// Coverage contributions of one span (computeCoverage 1390-1431).
struct CovSpan {
  const RowCtx* C;
  RowLds* L;
  int32_t sc;        // sampleCoverage
  int32_t covLo, covHi;  // coverage buffer span [startX, startX + pathWidth)
  __device__ void add_px(int64_t x, int32_t v) {
    if (x < covLo || x >= covHi) return;
    if (x < C->wx0 || x >= C->wx1) return;
    atomicAdd(&L->D[x - C->wx0], v);
    atomicAdd(&L->D[x - C->wx0 + 1], -v);
  }
  __device__ void operator()(int32_t prevAt, int32_t at) {
    int64_t fillStart = fx_int(prevAt);
    bool pixelCrossed = fx_int(at) != fx_int(prevAt);
    int32_t leftCover = pixelCrossed ? fx_trunc(prevAt) + 256 - prevAt : at - prevAt;
    if (leftCover != 0) {
      fillStart++;
      add_px(fx_int(prevAt), (int32_t)(uint8_t)fx_int(leftCover * sc));
    }
    if (pixelCrossed) {
      int32_t rightCover = at - fx_trunc(at);
      if (rightCover > 0) add_px(fx_int(at), (int32_t)(uint8_t)fx_int(rightCover * sc));
    }
    int64_t fillEnd = fx_int(at);
    if (fillEnd > fillStart) {
      int64_t lo = fillStart > covLo ? fillStart : covLo;
      int64_t hi = fillEnd < covHi ? fillEnd : covHi;
      if (lo < C->wx0) lo = C->wx0;
      if (hi > C->wx1) hi = C->wx1;
      if (lo < hi) {
        atomicAdd(&L->D[lo - C->wx0], sc);
        atomicAdd(&L->D[hi - C->wx0], -sc);
      }
    }
  }
};

// Fill runs of a walkInteger span (fillHits 1540-1591).
struct FillSpan {
  const RowCtx* C;
  RowLds* L;
  int32_t code;   // value added over the span
  int64_t minX;   // spans are cut below minX (mask mode: left of startX is cleared)
  __device__ void operator()(int32_t prevAt, int32_t at) {
    int64_t s = fx_int(prevAt), e = fx_int(at);
    if (e - s <= 0) return;
    if (s < minX) s = minX;
    add_run(*C, *L, s, e, code);
  }
};

// The row's selected entries.  When the selection fits in one wave (the
// common case), lane i keeps selection i in registers for all sample lines;
// otherwise entries are re-read through L.A.
struct SelCache {
  bool inReg;
  Entry e;
  int32_t w;
};

// Collects the hits of one sample line (paths.nim:1373-1388) from the
// selection L.A[0..ne) into L.keys sorted stably by x; windings go to L.B by
// hit position.  Returns the number of hits.
__device__ __forceinline__ int row_hits(const RowCtx& C, RowLds& L, int ne, float yLine, SelCache S) {
  int lane = lane_id();
  const float Wf = (float)C.F->canvasW;
  int nh = 0;
  for (int base = 0; base < ne; base += kWave) {
    int i = base + lane;
    bool hit = false;
    int32_t at = 0, w = 0;
    if (i < ne) {
      Entry e;
      int32_t ew;
      if (S.inReg) {
        e = S.e;
        ew = S.w;
      } else {
        int k = L.A[i];
        e = C.E[k];
        ew = C.EW[k];
      }
      if (e.aty <= yLine && e.toy >= yLine) {
        float x = e.m == 0.0f ? e.b : (yLine - e.b) / e.m;
        at = fixed32(nim_minf(x, Wf));
        w = ew;
        hit = true;
      }
    }
    uint64_t m = ballot(hit);
    int pos = nh + __popcll(m & ((1ull << lane) - 1ull));
    if (hit) {
      L.keys[pos] = ((uint64_t)((uint32_t)at ^ 0x80000000u) << 32) | (uint32_t)pos;
      L.B[pos] = w;
    }
    nh += __popcll(m);
  }
  wave_sync();
  if (nh > 1) wave_sort_keys(L.keys, nh, L.cap);
  return nh;
}

// ---- sample lines by 32-bit keys ----
// A window's walk needs only the hits inside it: the windings of the hits
// left of it give the count it starts with, and a span open at its end is
// known to end later when the windings of the whole line sum to 0 (the count
// then returns to 0 at a hit that no skip consumes).  So a hit's key is 32
// bits: its 24.8 position from the window's start, its place in the selection
// (pixie's stable order of equal x) and the sign of its winding; the keys
// sort in registers, with no LDS traffic.  A line whose windings do not sum
// to 0 is walked whole (row_hits and wave_walk).
//
// Every span (p, a) of the walk is added as two independent parts, one at
// its start and one at its end: with L = floor((256 - frac p) * sc / 256) and
// R = floor(frac a * sc / 256), D gets L and sc - L at p's pixel and the
// next, R - sc and -R at a's pixel and the next, which sum to what
// computeCoverage (1390-1431) adds.  Only when p and a share a pixel do the
// two roundings differ from the one of (a - p) * sc; the end then adds the
// difference.  Positions are clamped to the columns the coverage may write,
// which clips spans as computeCoverage clips them.
//
// The row program is bound by instruction issue; per 64 hits the 64-bit form
// of this path took about 250 instructions to sort (LDS permutes) and 250 to
// walk (scans, up to six LDS atomics a span), this one 110 and 90 (lane masks,
// two atomics an event): rows of the 4096 x 4096 scene 957 -> 636 us, of the
// 10,000-glyph atlas 617 -> 515 us.
constexpr int kSampleCov = 255 / 5;

// Lanes below this one in its SEG-lane segment, as a 64-bit lane mask.
template <int SEG>
__device__ __forceinline__ uint64_t seg_below() {
  const int lane = lane_id();
  return ((1ull << lane) - 1ull) & ~((1ull << (lane & ~(SEG - 1))) - 1ull);
}
// Set bits of m below this lane in its segment, plus acc.
template <int SEG>
__device__ __forceinline__ int32_t seg_rank(uint64_t m) {
  if (SEG == kWave) return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
  return __popcll(m & seg_below<SEG>());
}

struct Walk32 {
  int32_t count = 0;      // winding count before the chunk (per segment)
  int32_t prev = -1;      // position of the last event before the chunk
  bool consumed = false;  // the chunk's first hit was consumed by a skip
};

// One chunk of the walk over sorted keys (position << IB | order << 1 |
// winding is 1): lane i of a segment holds hit i when valid, kn the key
// after it when hasNext.  Positions are relative to the pixel D points at,
// [lo, hi) are the pixels that may be written.
template <int IB, int SEG>
__device__ __forceinline__ void walk32(uint32_t k, uint32_t kn, bool valid, bool hasNext, int32_t rule, int32_t* D,
                                       int32_t lo, int32_t hi, Walk32& c) {
  const int lane = lane_id();
  const bool up = (k & 1u) != 0;
  const uint64_t pos = ballot(valid && up), neg = ballot(valid && !up);
  const int32_t cb = c.count + seg_rank<SEG>(pos) - seg_rank<SEG>(neg);
  const bool filling = should_fill(rule, cb);
  // a hit and the next at the same x whose windings cancel are skipped
  uint64_t cm = ballot(valid && filling && hasNext && ((k ^ kn) >> IB) == 0 && ((k ^ kn) & 1u));
  bool off = false;
  if (cm != 0 || c.consumed) {
    uint64_t skip = 0, cons = c.consumed ? 1ull : 0ull;
    bool carry = false;
    while (cm) {
      const int b = __builtin_ctzll(cm);
      cm &= cm - 1;
      if (!((cons >> b) & 1ull)) {
        skip |= 1ull << b;
        if (b + 1 < kWave) cons |= 1ull << (b + 1);
        else carry = true;
      }
    }
    off = ((skip | cons) >> lane) & 1ull;
    c.consumed = carry;
  }
  const bool act = valid && !off;
  const bool start = act && !filling;
  const bool end = act && filling && !(rule == kNonZero && cb + (up ? 1 : -1) != 0);
  const int32_t rel = (int32_t)(k >> IB);
  int32_t r = rel > (lo << 8) ? rel : (lo << 8);
  r = r < (hi << 8) ? r : (hi << 8);
  const int32_t f = r & 255, px = r >> 8;
  int32_t v0 = ((start ? 256 - f : f) * kSampleCov) >> 8;
  if (!start) v0 -= kSampleCov;
  int32_t v1 = (start ? kSampleCov : -kSampleCov) - v0;
  // ends whose start may share their pixel: the hit before them does
  const uint64_t em = ballot(start || end);
  const uint32_t kp = __builtin_amdgcn_update_dpp(~0u, k, kDppWaveShr1, 0xf, 0xf, false);
  const bool first = (lane & (SEG - 1)) == 0;
  const bool near = end && (first ? c.prev >> 8 == rel >> 8 : ((kp ^ k) >> (IB + 8)) == 0);
  if (ballot(near)) {
    const uint64_t before = em & seg_below<SEG>();
    const int src = before ? 63 - __builtin_clzll(before) : lane;
    const int32_t ps = __shfl(rel, src, kWave);
    const int32_t p = before ? ps : c.prev;
    if (near && (p >> 8) == (rel >> 8) && p >= 0 && r == rel && px < hi) {
      const int32_t left = ((256 - (p & 255)) * kSampleCov) >> 8;  // what p's start added
      const int32_t whole = ((rel - p) * kSampleCov) >> 8;
      const int32_t fix = whole - (left + v0);
      v0 += fix;
      v1 -= fix;
    }
  }
  if (start || end) {
    atomicAdd(&D[px], v0);
    atomicAdd(&D[px + 1], v1);
  }
  if (SEG == kWave) {
    c.count += __popcll(pos) - __popcll(neg);
    if (em) c.prev = __builtin_amdgcn_readlane(rel, 63 - __builtin_clzll(em));
  }
}

// What a line filled at the window's start or end adds there.
__device__ __forceinline__ void walk32_borders(bool fillStart, bool fillEnd, int32_t* D, int32_t lo, int32_t hi) {
  if (fillStart) atomicAdd(&D[lo], kSampleCov);
  if (fillEnd) atomicAdd(&D[hi], -kSampleCov);
}

// A row window's place for the 32-bit walks, which take windows that end below
// kWin32End: its 24.8 bounds must not leave 32 bits.  (Positions of 2^23 px
// and more saturate to the lowest number, as pixie's conversion does; in a
// window below them they count as hits left of it, which is where pixie's sort
// puts them.)  The lines of a window beyond are walked whole.
constexpr int32_t kWin32End = 1 << 23;
struct Win32 {
  int32_t A, A1, B;  // 24.8 bounds of its hits (a hit at or left of x = 0 only counts)
  int32_t lo, hi;    // columns the coverage may write, from the window's start
};
__device__ __forceinline__ Win32 window32(const RowCtx& C) {
  const int32_t covLo = C.F->startX, covHi = covLo + C.F->pathWidth;
  Win32 w;
  w.A = C.wx0 * 256;
  w.A1 = w.A > 1 ? w.A : 1;
  w.B = C.wx1 * 256;
  w.lo = (covLo > C.wx0 ? covLo : C.wx0) - C.wx0;
  w.hi = (covHi < C.wx1 ? covHi : C.wx1) - C.wx0;
  return w;
}
constexpr int kKeyBits = 15;  // order (14 bits) and winding below the position (17 bits: windows of 512 px)
constexpr int kSegBits = 7;   // of at most 64 entries: order (6 bits) and winding (25 bits: any window)

// 24.8 x of an entry's hit on a sample line (1373-1388).
__device__ __forceinline__ int32_t hit_at(const Entry& e, float yLine, float Wf) {
  const float x = e.m == 0.0f ? e.b : (yLine - e.b) / e.m;
  return fixed32(nim_minf(x, Wf));
}

// The 5-sample coverage of a row that selects at most SEG entries (held by
// lanes 0..ne-1 of S): 64 / SEG sample lines at a time, one per segment of
// the wave -- all five for SEG = 8, two passes for 16, three for 32, five for
// 64.  A segment holds one whole line, so the walk needs no carries.  yLine
// is one step before the first line.  Returns the lines whose windings do
// not sum to 0 (bit m: line m), which are left to be
// walked whole.
template <int SEG>
__device__ __forceinline__ uint32_t row_coverage_seg(const RowCtx& C, RowLds& L, int ne, SelCache S, float yLine,
                                                     float offset, int32_t rule) {
  constexpr int kPer = kWave / SEG;
  constexpr int kPasses = (5 + kPer - 1) / kPer;
  const int lane = lane_id();
  const int grp = lane / SEG, i = lane & (SEG - 1);
  const float Wf = (float)C.F->canvasW;
  const Win32 w = window32(C);
  Entry e = S.e;
  int32_t ew = S.w;
  if (SEG < kWave) {
    e.aty = __shfl(S.e.aty, i, kWave);
    e.toy = __shfl(S.e.toy, i, kWave);
    e.m = __shfl(S.e.m, i, kWave);
    e.b = __shfl(S.e.b, i, kWave);
    ew = __shfl(S.w, i, kWave);
  }
  uint32_t whole = 0;
  const uint64_t segMask = SEG == kWave ? ~0ull : ((1ull << (SEG & 63)) - 1ull) << (grp * SEG);
#pragma unroll 1
  for (int pass = 0; pass < kPasses; pass++) {
    const int sample = pass * kPer + grp;
    float y = yLine;
#pragma unroll
    for (int g = 0; g < kPer && g < 5; g++) {
      yLine += offset;
      y = grp == g ? yLine : y;
    }
    const bool hit = sample < 5 && i < ne && e.aty <= y && e.toy >= y;
    const int32_t at = hit_at(e, y, Wf);
    const uint64_t up = ballot(hit && ew > 0), down = ballot(hit && ew <= 0);
    const bool isLeft = hit && at < w.A1, in = hit && !isLeft && at < w.B;
    const uint64_t inM = ballot(in), leftM = ballot(isLeft);
    const bool open = __popcll(up & segMask) != __popcll(down & segMask);  // the windings do not sum to 0
    const uint64_t openM = ballot(open);
    if (w.lo < w.hi) {
      const int32_t left = __popcll(leftM & up & segMask) - __popcll(leftM & down & segMask);
      const int32_t after = left + __popcll(inM & up & segMask) - __popcll(inM & down & segMask);
      const int n = __popcll(inM & segMask);
      uint32_t k = in ? ((uint32_t)(at - w.A) << kSegBits) | ((uint32_t)i << 1) | (ew > 0 ? 1u : 0u) : ~0u;
      uint32_t ks[1] = {k};
      if (SEG == kWave) wave_sort32<1>(ks);
      k = SEG == kWave ? ks[0] : seg_sort32<SEG>(k);
      const uint32_t kn = __builtin_amdgcn_update_dpp(~0u, k, kDppWaveShl1, 0xf, 0xf, false);
      Walk32 c;
      c.count = left;
      walk32<kSegBits, SEG>(k, kn, i < n && !open, i < n - 1, rule, L.D, w.lo, w.hi, c);
      if (i == 0 && !open) walk32_borders(should_fill(rule, left), should_fill(rule, after), L.D, w.lo, w.hi);
    }
    if (openM)
#pragma unroll
      for (int g = 0; g < kPer && g < 5; g++)
        if ((openM >> (g * SEG)) & 1ull) whole |= 1u << (pass * kPer + g);
  }
  return whole;
}

// Finishes sorting n distinct keys that are nearly in order: odd-even
// transposition passes until one swaps nothing, and a full sort once
// kFixPassesMem passes have not been enough.
constexpr int kFixPassesMem = 16;
__device__ void wave_fix_keys(uint64_t* keys, int n, int cap) {
  const int lane = lane_id();
  for (int pass = 0;; pass++) {
    bool swapped = false;
    for (int par = 0; par < 2; par++) {
      for (int i = 2 * lane + par; i + 1 < n; i += 2 * kWave) {
        const uint64_t a = keys[i], b = keys[i + 1];
        if (a > b) {
          keys[i] = b;
          keys[i + 1] = a;
          swapped = true;
        }
      }
      wave_sync();
    }
    if (ballot(swapped) == 0) return;
    if (pass + 1 >= kFixPassesMem) {
      wave_sort_keys(keys, n, cap);
      return;
    }
  }
}

// The 5-sample coverage of a row of more entries than the wide path takes
// (computeCoverage 1350-1431).  pixie sorts each sample line's hits from
// scratch (sort 1373-1388).  Here the selection is sorted once, by x where
// each entry is nearest the row's middle; every sample line then collects
// its hits in that order, which leaves them sorted except where entries cross
// inside the row, and wave_fix_keys finishes the sort.  The hit keys carry
// the selection index as tie-break, which orders equal x like pixie's
// insertion sort over hits collected in selection order, and the winding in
// their low byte, so the walk reads it from the key.
__device__ __forceinline__ void row_coverage_presorted(const RowCtx& C, RowLds& L, int ne, float yLine,
                                                       float offset, int32_t rule, CovSpan& span) {
  const int lane = lane_id();
  const float Wf = (float)C.F->canvasW;
  const float yMid = (float)C.y + 0.5f;
  // By presorted position: the selection index with the winding in the low
  // byte (the hit key's low word), and the entry index.
  int32_t* order = (int32_t*)L.tx0;
  int32_t* entry = (int32_t*)L.tx1;
  for (int i = lane; i < ne; i += kWave) {
    const int k = L.A[i];
    const Entry e = C.E[k];
    const float yc = yMid < e.aty ? e.aty : (yMid > e.toy ? e.toy : yMid);
    L.keys[i] = ((uint64_t)float_key(solve_x(e.m, e.b, yc)) << 32) | (uint32_t)i;
    L.B[i] = C.EW[k];
  }
  wave_sync();
  wave_sort_keys(L.keys, ne, L.cap);
  for (int j = lane; j < ne; j += kWave) {
    const int s = (int)(uint32_t)L.keys[j];
    order[j] = (s << 8) | (int32_t)(uint8_t)L.B[s];
    entry[j] = L.A[s];
  }
  wave_sync();
#pragma unroll 1
  for (int m = 0; m < 5; m++) {
    yLine += offset;
    int nh = 0;
    for (int base = 0; base < ne; base += kWave) {
      const int j = base + lane;
      bool hit = false;
      int32_t at = 0, s = 0;
      if (j < ne) {
        const Entry e = C.E[entry[j]];
        s = order[j];
        if (e.aty <= yLine && e.toy >= yLine) {
          at = hit_at(e, yLine, Wf);
          hit = true;
        }
      }
      const uint64_t mk = ballot(hit);
      const int pos = nh + __popcll(mk & ((1ull << lane) - 1ull));
      if (hit) L.keys[pos] = ((uint64_t)((uint32_t)at ^ 0x80000000u) << 32) | (uint32_t)s;
      nh += __popcll(mk);
    }
    wave_sync();
    wave_fix_keys(L.keys, nh, L.cap);
    wave_walk<true>(L, nh, rule, span);
    wave_sync();
  }
}

// Sorts n <= 64 * NS staged keys in NS register slots.
template <int NS>
__device__ __forceinline__ void sort32_staged(uint32_t* stage, int n) {
  const int lane = lane_id();
  uint32_t k[NS];
#pragma unroll
  for (int s = 0; s < NS; s++) k[s] = s * kWave + lane < n ? stage[s * kWave + lane] : ~0u;  // padding sorts last
  wave_sort32<NS>(k);
#pragma unroll
  for (int s = 0; s < NS; s++)
    if (s * kWave + lane < n) stage[s * kWave + lane] = k[s];
}

// Sorts and walks n staged keys, any n.  One copy of the walk serves every
// size: the sorted keys go back to the stage.
template <int IB>
__device__ __forceinline__ void walk32_staged(uint32_t* stage, int n, int32_t rule, int32_t* D, int32_t lo,
                                              int32_t hi, Walk32& c) {
  if (n > 4 * kWave)
    wave_sort32_mem(stage, n);
  else if (n > 2 * kWave)
    sort32_staged<4>(stage, n);
  else if (n > kWave)
    sort32_staged<2>(stage, n);
  else
    sort32_staged<1>(stage, n);
  wave_sync();
#pragma unroll 1
  for (int base = 0; base < n; base += kWave) {
    const int i = base + lane_id();
    const uint32_t k = i < n ? stage[i] : ~0u, kn = i < n - 1 ? stage[i + 1] : ~0u;
    walk32<IB, kWave>(k, kn, i < n, i < n - 1, rule, D, lo, hi, c);
  }
}

// The 5-sample coverage of an anti-aliased row that selects 65 to kWideMax
// entries (computeCoverage 1350-1431 with walk 1298-1334).  A selection of at
// most 256 is held in registers (selection j in slot j / 64 of lane j % 64);
// a larger one is read from the band for every sample line (C.E / C.EW start
// at the band, count entries; a hit implies the selection test, which is
// repeated so that the two agree at any y).  Each line's hits inside the
// window are compacted in selection order into L.stage (LDS) as 32-bit keys,
// sorted in register slots and walked.  Returns the lines to be walked
// whole, as row_coverage_seg does.
constexpr int kWideSlots = 4;
constexpr int kWideMax = 8 * kWave;
__device__ __forceinline__ bool wide_fits(const RowLds& L, int ne, int count) {
  return L.ww <= 512 && ne <= L.stageCap && (ne <= kWideSlots * kWave || (ne <= kWideMax && count <= 1 << (kKeyBits - 1)));
}
__device__ __forceinline__ uint32_t row_coverage_wide(const RowCtx& C, RowLds& L, int count, int ne, float scanTop,
                                                      float scanBottom, float yLine, float offset, int32_t rule) {
  const int lane = lane_id();
  const float Wf = (float)C.F->canvasW;
  const Win32 win = window32(C);
  uint32_t* stage = L.stage;
  uint32_t whole = 0;
  const bool inReg = ne <= kWideSlots * kWave;
  Entry e[kWideSlots];
  int32_t w[kWideSlots];
#pragma unroll
  for (int s = 0; s < kWideSlots; s++) {
    e[s] = Entry{0.0f, 0.0f, 0.0f, 0.0f};
    w[s] = 0;
    const int j = s * kWave + lane;
    if (inReg && j < ne) {
      const int k = L.A[j];
      e[s] = C.E[k];
      w[s] = C.EW[k];
    }
  }
#pragma unroll 1
  for (int m = 0; m < 5; m++) {
    yLine += offset;
    int n = 0, left = 0, total = 0, in = 0;  // keys, and winding sums
    auto put = [&](const Entry& ei, int32_t wi, bool sel, int order) {
      const bool hit = sel && ei.aty <= yLine && ei.toy >= yLine;
      const int32_t at = hit_at(ei, yLine, Wf);
      const bool isLeft = hit && at < win.A1, inW = hit && !isLeft && at < win.B;
      const uint64_t up = ballot(hit && wi > 0), down = ballot(hit && wi <= 0), lm = ballot(isLeft), im = ballot(inW);
      total += __popcll(up) - __popcll(down);
      left += __popcll(lm & up) - __popcll(lm & down);
      in += __popcll(im & up) - __popcll(im & down);
      if (inW)
        stage[n + seg_rank<kWave>(im)] =
            ((uint32_t)(at - win.A) << kKeyBits) | ((uint32_t)order << 1) | (wi > 0 ? 1u : 0u);
      n += __popcll(im);
    };
    if (inReg) {
#pragma unroll
      for (int s = 0; s < kWideSlots; s++)
        if (s * kWave < ne) put(e[s], w[s], s * kWave + lane < ne, s * kWave + lane);
    } else {
#pragma unroll 2
      for (int base = 0; base < count; base += kWave) {
        const int i = base + lane;
        Entry ei = {0.0f, 0.0f, 0.0f, 0.0f};
        int32_t wi = 0;
        if (i < count) {
          ei = C.E[i];
          wi = C.EW[i];
        }
        put(ei, wi, i < count && !(ei.toy <= scanTop || ei.aty >= scanBottom), i);
      }
    }
    wave_sync();
    if (total != 0) {
      whole |= 1u << m;
    } else if (win.lo < win.hi) {
      Walk32 c;
      c.count = left;
      walk32_staged<kKeyBits>(stage, n, rule, L.D, win.lo, win.hi, c);
      if (lane == 0)
        walk32_borders(should_fill(rule, left), should_fill(rule, left + in), L.D, win.lo, win.hi);
    }
    wave_sync();
  }
  return whole;
}

// Entries row C.y selects (row_program's selection), so that a caller can
// place the row's arrays before running it: the arrays hold the selection,
// which is often much smaller than the band.
__device__ __forceinline__ int row_selection_count(const RowCtx& C) {
  const FillInfo& F = *C.F;
  const int32_t y = C.y;
  if (y < F.startY || y >= F.pathHeight) return 0;
  int32_t pi = (y - F.startY) / F.bandH;
  if (pi > F.nParts - 1) pi = F.nParts - 1;
  const int count = __builtin_amdgcn_readfirstlane(C.parts[pi].count);
  if (__builtin_amdgcn_readfirstlane(C.parts[pi].flags) & 2) return 2;
  const Entry* E = C.E + __builtin_amdgcn_readfirstlane(C.parts[pi].entryBase);
  const float scanTop = (float)y, scanBottom = (float)(y + 1);
  int ne = 0;
#pragma unroll 2
  for (int base = 0; base < count; base += kWave) {
    const int i = base + lane_id();
    bool s = false;
    if (i < count) {
      const Entry e = E[i];
      s = !(e.toy <= scanTop || e.aty >= scanBottom);
    }
    ne += __popcll(ballot(s));
  }
  return ne;
}

// Runs the row program for (fill, row y, window) and leaves the row's codes
// in L.D (and L.AX).  Returns the row kind; kRowNone means nothing to do and
// -1 means the selection holds more entries than L.cap (nothing was written).
__device__ int32_t row_program(const RowCtx& C, RowLds& L) {
  const FillInfo& F = *C.F;
  const int lane = lane_id();
  const int32_t W = F.canvasW;
  const int32_t y = C.y;
  const bool mask = F.mode == kMask;

  if (y < F.startY || y >= F.pathHeight) {
    if (mask) {  // rows outside the path are cleared (paths.nim:1910-1912)
      if (lane == 0) add_run(C, L, 0, W, kClear);
      wave_sync();
      return kRowOps;
    }
    return kRowNone;
  }
  int32_t pi = (y - F.startY) / F.bandH;
  if (pi > F.nParts - 1) pi = F.nParts - 1;
  PartInfo P = C.parts[pi];  // the same in every lane: scalar registers
  P.entryBase = __builtin_amdgcn_readfirstlane(P.entryBase);
  P.count = __builtin_amdgcn_readfirstlane(P.count);
  P.flags = __builtin_amdgcn_readfirstlane(P.flags);
  const bool aa = P.flags & 1, two = P.flags & 2;
  RowCtx Cp = C;
  Cp.E = C.E + P.entryBase;
  Cp.EW = C.EW + P.entryBase;
  const Entry* E = Cp.E;
  const int8_t* EW = Cp.EW;

  if (two && !aa) {  // paths.nim:1644-1668
    if (mask && lane == 0) add_run(C, L, 0, W, kClear);  // default for mask rows
    if (lane == 0) {
      int64_t left = nim_f2i(E[0].b), right = nim_f2i(E[1].b);
      int64_t minX = left < 0 ? 0 : (left > W ? W : left);
      int64_t maxX = right < 0 ? 0 : (right > W ? W : right);
      if (maxX > minX) add_run(C, L, minX, maxX, mask ? kFill - kClear : kFill);
    }
    wave_sync();
    return kRowOps;
  }

  const float scanTop = (float)y, scanBottom = (float)(y + 1);
  int ne = 0;
  bool allSpan = true;
  if (two) {
    if (lane == 0) {
      L.A[0] = 0;
      L.A[1] = 1;
    }
    ne = 2;
  } else {
#pragma unroll 2
    for (int base = 0; base < P.count; base += kWave) {
      int i = base + lane;
      bool s = false, notSpan = false;
      if (i < P.count) {
        Entry e = E[i];
        s = !(e.toy <= scanTop || e.aty >= scanBottom);
        notSpan = s && (e.aty > scanTop || e.toy < scanBottom);
      }
      uint64_t m = ballot(s);
      int pos = ne + __popcll(m & ((1ull << lane) - 1ull));
      if (s && pos < L.cap) L.A[pos] = i;
      ne += __popcll(m);
      if (ballot(notSpan)) allSpan = false;
    }
  }
  wave_sync();
  // the row's arrays hold the selection (not the whole band); D is untouched
  // so far, so a selection too large for them leaves nothing behind
  if (ne > L.cap) return -1;
  if (mask && lane == 0) add_run(C, L, 0, W, kClear);  // default for mask rows
  const bool inReg = ne <= kWave;
  float sAty = 0.0f, sToy = 0.0f, sM = 0.0f, sB = 0.0f;
  int32_t sW = 0;
  if (inReg && lane < ne) {
    const int k = L.A[lane];
    sAty = E[k].aty;
    sToy = E[k].toy;
    sM = E[k].m;
    sB = E[k].b;
    sW = EW[k];
  }
  const SelCache S{inReg, Entry{sAty, sToy, sM, sB}, sW};

  if (allSpan && (ne % 2) == 0) {  // trapezoid fast path, 1691-1872
    for (int i = lane; i < ne; i += kWave) {
      Entry e = S.e;  // (a conditional copy, not a ?: on the two lvalues: that would keep S in memory)
      if (!S.inReg) e = E[L.A[i]];
      float a = solve_x(e.m, e.b, scanTop), b = solve_x(e.m, e.b, scanBottom);
      L.tx0[i] = a;
      L.tx1[i] = b;
      L.keys[i] = ((uint64_t)float_key(midpoint_x(v2(a, scanTop), v2(b, scanBottom))) << 32) |
                  (uint32_t)i;
    }
    wave_sync();
    if (ne > 1) wave_sort_keys(L.keys, ne, L.cap);
    // the partial coverage areas must not overlap (1720-1728) and the pairs
    // must be simple fills (1731-1745)
    bool bad = false;
    int32_t carry = 0;
    for (int base = 0; base < ne; base += kWave) {
      int i = base + lane;
      bool fail = false;
      int32_t w = 0;
      if (i < ne) {
        int pi0 = (int)(uint32_t)L.keys[i];
        w = EW[L.A[pi0]];
        if (i < ne - 1) {
          int pi1 = (int)(uint32_t)L.keys[i + 1];
          float lmax = nim_maxf(L.tx0[pi0], L.tx1[pi0]);
          float rmin = nim_minf(L.tx0[pi1], L.tx1[pi1]);
          if (nim_f2i(ceilf(lmax)) > nim_f2i(rmin)) fail = true;
        }
      }
      int32_t tot;
      int32_t incl = carry + wave_excl_scan(w, &tot) + w;
      if (i < ne) {
        bool f = should_fill(F.rule, incl);
        if ((i % 2 == 0) != f) fail = true;
      }
      carry += tot;
      if (ballot(fail)) bad = true;
    }
    if (!bad) {
      const int32_t areaCode = mask ? kArea - kClear : kArea;
      for (int p = lane; p < ne / 2; p += kWave) {  // one lane per pair
        int pl = (int)(uint32_t)L.keys[2 * p], pr = (int)(uint32_t)L.keys[2 * p + 1];
        Entry le = E[L.A[pl]], re = E[L.A[pr]];
        float la = L.tx0[pl], lt = L.tx1[pl];
        float ra = L.tx0[pr], rt = L.tx1[pr];
        float leftMaxX = nim_maxf(la, lt);
        float rightMinX = nim_minf(ra, rt);
        int64_t leftCoverEnd = nim_f2i(ceilf(leftMaxX));
        int64_t rightCoverBegin = nim_f2i(truncf(rightMinX));
        {  // left sliver 1772-1809
          bool inverted = la < lt;
          float sliverStart = nim_minf(la, lt);
          float rectStart = leftMaxX;
          float pen = sliverStart, prevPen = pen;
          float penY = inverted ? (float)y : (float)(y + 1);
          float prevPenY = penY;
          int64_t x0 = nim_f2i(sliverStart), x1 = nim_f2i(ceilf(rectStart));
          for (int64_t x = x0; x < x1; x++) {
            prevPen = pen;
            pen = (float)(x + 1);
            float rightRectArea = 0.0f;
            if (pen > rectStart) {
              rightRectArea = pen - rectStart;
              pen = rectStart;
            }
            prevPenY = penY;
            penY = solve_y(le.m, le.b, pen);
            if (x < 0 || x >= W) continue;
            float run = pen - prevPen;
            float triangleArea = 0.5f * run * fabsf(penY - prevPenY);
            float rectArea = inverted ? (prevPenY - (float)y) * run : ((float)(y + 1) - prevPenY) * run;
            float area = triangleArea + rectArea + rightRectArea;
            if (x >= C.cx0 && x < C.cx1 && x >= C.wx0 && x < C.wx1) {
              L.AX[x - C.wx0] = area_factor(area);
              atomicAdd(&L.D[x - C.wx0], areaCode);
              atomicAdd(&L.D[x - C.wx0 + 1], -areaCode);
            }
          }
        }
        {  // right sliver 1811-1847
          bool inverted = ra > rt;
          float rectEnd = rightMinX;
          float sliverEnd = nim_maxf(ra, rt);
          float pen = rectEnd, prevPen = pen;
          float penY = inverted ? (float)(y + 1) : (float)y;
          float prevPenY = penY;
          int64_t x0 = nim_f2i(rectEnd), x1 = nim_f2i(ceilf(sliverEnd));
          for (int64_t x = x0; x < x1; x++) {
            prevPen = pen;
            pen = (float)(x + 1);
            float ap = fabsf(prevPen);
            float leftRectArea = ap - floorf(ap);
            if (pen > sliverEnd) pen = sliverEnd;
            prevPenY = penY;
            penY = solve_y(re.m, re.b, pen);
            if (x < 0 || x >= W) continue;
            float run = pen - prevPen;
            float triangleArea = 0.5f * run * fabsf(penY - prevPenY);
            float rectArea = inverted ? (penY - (float)y) * run : ((float)(y + 1) - penY) * run;
            float area = leftRectArea + triangleArea + rectArea;
            if (x >= C.cx0 && x < C.cx1 && x >= C.wx0 && x < C.wx1) {
              L.AX[x - C.wx0] = area_factor(area);
              atomicAdd(&L.D[x - C.wx0], areaCode);
              atomicAdd(&L.D[x - C.wx0 + 1], -areaCode);
            }
          }
        }
        int64_t fb = leftCoverEnd < 0 ? 0 : (leftCoverEnd > W ? W : leftCoverEnd);
        int64_t fe = rightCoverBegin < 0 ? 0 : (rightCoverBegin > W ? W : rightCoverBegin);
        // interior: fillHits on (fixed32(fb), +1), (fixed32(fe), -1)
        if (fe > fb) add_run(C, L, fb, fe, mask ? kFill - kClear : kFill);
      }
      wave_sync();
      return kRowOps;
    }
    // Not a simple trapezoid row: pixie keeps the midpoint order of the
    // selection for the coverage pass below.
    for (int i = lane; i < ne; i += kWave) L.B[i] = L.A[(int)(uint32_t)L.keys[i]];
    wave_sync();
    for (int i = lane; i < ne; i += kWave) L.A[i] = L.B[i];
    wave_sync();
  }

  // computeCoverage 1350-1431 / fillHits 1898
  const int quality = aa ? 5 : 1;
  const float offset = 1.0f / (float)quality;
  const float initialOffset = offset / 2.0f + 0.00031415926535897936f;
  float yLine = (float)y + initialOffset - offset;
  const int64_t covLo = F.startX, covHi = (int64_t)F.startX + F.pathWidth;
  if (aa) {
    if (mask && lane == 0) add_run(C, L, covLo, covHi, -kClear);  // coverage range
    CovSpan cs{&C, &L, kSampleCov, (int32_t)covLo, (int32_t)covHi};
    uint32_t whole;
    if (Cp.wx1 >= kWin32End) {
      whole = 0x1fu;
    } else if (ne <= 8) {
      whole = row_coverage_seg<8>(Cp, L, ne, S, yLine, offset, F.rule);
    } else if (ne <= 16) {
      whole = row_coverage_seg<16>(Cp, L, ne, S, yLine, offset, F.rule);
    } else if (ne <= 32) {
      whole = row_coverage_seg<32>(Cp, L, ne, S, yLine, offset, F.rule);
    } else if (ne <= kWave) {
      whole = row_coverage_seg<64>(Cp, L, ne, S, yLine, offset, F.rule);
    } else if (wide_fits(L, ne, P.count)) {
      whole = row_coverage_wide(Cp, L, P.count, ne, scanTop, scanBottom, yLine, offset, F.rule);
    } else {
      whole = 0;
      row_coverage_presorted(Cp, L, ne, yLine, offset, F.rule, cs);
    }
    for (; whole != 0; whole >>= 1) {
      yLine += offset;
      if (whole & 1u) {  // pixie's walk of the whole line
        wave_walk(L, row_hits(Cp, L, ne, yLine, S), F.rule, cs);
        wave_sync();
      }
    }
    return kRowCoverage;
  }
  yLine += offset;
  int nh = row_hits(Cp, L, ne, yLine, S);
  FillSpan fs{&C, &L, mask ? kFill - kClear : kFill, mask ? (int64_t)F.startX : (int64_t)INT64_MIN};
  wave_walk(L, nh, F.rule, fs);
  wave_sync();
  return kRowOps;
}

// Applies one pixel's code.  Returns the new pixel value.
__device__ __forceinline__ uint32_t apply_code(int32_t kind, int32_t code, uint32_t ax,
                                               uint32_t dst, uint32_t rgbx, int32_t mode,
                                               bool* touched) {
  if (kind == kRowCoverage) {
    if (code >= kClear) {
      *touched = true;
      return 0;
    }
    uint32_t c = (uint32_t)code & 255u;
    bool doit = (mode == kMask) ? (c != 255u) : (c != 0u);
    if (!doit) return dst;
    *touched = true;
    uint32_t src = mul_cov(rgbx, c);
    return mode == kOverwrite ? src : blend(mode, dst, src);
  }
  if (code == 0) return dst;
  *touched = true;
  if (code >= kClear) return 0;
  uint32_t src = code >= kArea ? mul_cov(rgbx, ax) : rgbx;
  return blend(mode, dst, src);
}

// apply_code for NormalBlend (paths.nim:1700-1770 with blends.nim:60-70), the
// mode of nearly every call, without a branch: the general form's branches
// and its mode switch took a third of the composition's instructions.
__device__ __forceinline__ uint32_t apply_normal(bool coverage, int32_t code, uint32_t ax, uint32_t dst,
                                                 uint32_t rgbx, bool* touched) {
  const bool clear = code >= kClear;
  const uint32_t c = coverage ? (uint32_t)code & 255u : (code >= kArea ? ax : 255u);
  uint32_t s = mul_div255(rgbx, c, 127u);
  if (ballot(c > 255u) != 0) s = mul_cov(rgbx, c);  // an area outside [0, 1]
  const uint32_t sa = ch_a(s);
  uint32_t out = add_channels(s, mul_div255(dst, 255u - sa, 0u));
  out = sa == 0u ? dst : out;
  out = (ch_a(dst) == 0u || sa == 255u) ? s : out;
  *touched = coverage ? clear || c != 0u : code != 0;
  return clear ? 0u : (*touched ? out : dst);
}

// Four neighbouring pixels' codes are whole pixels of an opaque Normal paint:
// the pixels become the paint, whatever they were.
__device__ __forceinline__ bool all_opaque(int32_t kind, const int32_t* code, uint32_t rgbx, int32_t mode) {
  if (mode != kNormal || ch_a(rgbx) != 255u) return false;
  bool full = true;
#pragma unroll
  for (int k = 0; k < 4; k++)
    full = full && (kind == kRowCoverage ? code[k] == 255 : code[k] != 0 && code[k] < kArea);
  return full;
}

// Scans L.D over the window and applies the codes to canvas row `row`.
// Normal without branches and whole opaque pixels without reading them halve
// the instructions of a 3,686 x 3,686 rounded rectangle on an A8 canvas (30 to
// 15 million, 141 a pixel before).
// Leaves L.D zeroed for the next row.  Canvas rows are W pixels wide.
__device__ uint32_t row_epilogue(const RowCtx& C, RowLds& L, int32_t kind, uint32_t* canvas,
                                 int32_t W, uint32_t rgbx, int32_t mode) {
  const int lane = lane_id();
  const int32_t wlen = C.wx1 - C.wx0;
  uint32_t* rowp = canvas + (size_t)C.y * (size_t)W;
  const bool vec_ok = ((W & 3) == 0) && ((C.wx0 & 3) == 0);
  int32_t carry = 0;
  uint32_t ntouch = 0;
  for (int base = 0; base < wlen; base += 4 * kWave) {
    int i0 = base + 4 * lane;
    int32_t d0 = 0, d1 = 0, d2 = 0, d3 = 0;
    if (i0 < wlen + 1) {  // D has ww + 4 entries; indices up to ww + 3 valid
      d0 = L.D[i0];
      d1 = L.D[i0 + 1];
      d2 = L.D[i0 + 2];
      d3 = L.D[i0 + 3];
      L.D[i0] = 0;
      L.D[i0 + 1] = 0;
      L.D[i0 + 2] = 0;
      L.D[i0 + 3] = 0;
    }
    int32_t c0 = d0, c1 = c0 + d1, c2 = c1 + d2, c3 = c2 + d3;
    int32_t tot;
    int32_t off = carry + wave_excl_scan(c3, &tot);
    carry += tot;
    int32_t code[4] = {off + c0, off + c1, off + c2, off + c3};
    bool any = false;
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (i0 + k < wlen && code[k] != 0) any = true;
    if (kind == kRowCoverage && mode == kMask) any = true;  // mask coverage rows write every pixel
    if (!any) continue;
    int32_t x0 = C.wx0 + i0;
    uint32_t px[4];
    bool full = vec_ok && (i0 + 3 < wlen);
    if (full && all_opaque(kind, code, rgbx, mode)) {
      *(uint4*)(rowp + x0) = make_uint4(rgbx, rgbx, rgbx, rgbx);
      ntouch += 4;
      continue;
    }
    if (full) {
      uint4 v = *(const uint4*)(rowp + x0);
      px[0] = v.x; px[1] = v.y; px[2] = v.z; px[3] = v.w;
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) px[k] = (i0 + k < wlen) ? rowp[x0 + k] : 0u;
    }
    bool touched = false;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (i0 + k < wlen) {
        uint32_t ax = (code[k] >= kArea && code[k] < kClear && kind == kRowOps) ? L.AX[i0 + k] : 0u;
        bool t = false;
        px[k] = mode == kNormal ? apply_normal(kind == kRowCoverage, code[k], ax, px[k], rgbx, &t)
                                : apply_code(kind, code[k], ax, px[k], rgbx, mode, &t);
        ntouch += t ? 1u : 0u;
        touched |= t;
      }
    }
    if (!touched) continue;
    if (full) {
      *(uint4*)(rowp + x0) = make_uint4(px[0], px[1], px[2], px[3]);
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (i0 + k < wlen) rowp[x0 + k] = px[k];
    }
  }
  // clear the tail entries the loop did not visit
  for (int i = lane; i < 4; i += kWave) {
    int idx = ((wlen + 4 * kWave - 1) / (4 * kWave)) * 4 * kWave + i;
    if (idx < L.ww + 4) L.D[idx] = 0;
  }
  wave_sync();
  return ntouch;
}

// Epilogue for an A8 target (masks, glyph atlas): pixel v reads as
// rgbx(v,v,v,v) and the alpha of the result is stored.
__device__ uint32_t row_epilogue_a8(const RowCtx& C, RowLds& L, int32_t kind, uint8_t* canvas,
                                    int32_t W, uint32_t rgbx, int32_t mode) {
  const int lane = lane_id();
  const int32_t wlen = C.wx1 - C.wx0;
  uint8_t* rowp = canvas + (size_t)C.y * (size_t)W;
  const bool vec_ok = ((W & 3) == 0) && ((C.wx0 & 3) == 0);
  int32_t carry = 0;
  uint32_t ntouch = 0;
  for (int base = 0; base < wlen; base += 4 * kWave) {
    int i0 = base + 4 * lane;
    int32_t d0 = 0, d1 = 0, d2 = 0, d3 = 0;
    if (i0 < wlen + 1) {
      d0 = L.D[i0];
      d1 = L.D[i0 + 1];
      d2 = L.D[i0 + 2];
      d3 = L.D[i0 + 3];
      L.D[i0] = 0;
      L.D[i0 + 1] = 0;
      L.D[i0 + 2] = 0;
      L.D[i0 + 3] = 0;
    }
    int32_t c0 = d0, c1 = c0 + d1, c2 = c1 + d2, c3 = c2 + d3;
    int32_t tot;
    int32_t off = carry + wave_excl_scan(c3, &tot);
    carry += tot;
    int32_t code[4] = {off + c0, off + c1, off + c2, off + c3};
    bool any = kind == kRowCoverage && mode == kMask;
#pragma unroll
    for (int k = 0; k < 4; k++)
      if (i0 + k < wlen && code[k] != 0) any = true;
    if (!any) continue;
    int32_t x0 = C.wx0 + i0;
    uint32_t px[4];
    bool full = vec_ok && (i0 + 3 < wlen);
    if (full && all_opaque(kind, code, rgbx, mode)) {
      *(uint32_t*)(rowp + x0) = ~0u;
      ntouch += 4;
      continue;
    }
    if (full) {
      uint32_t v = *(const uint32_t*)(rowp + x0);
#pragma unroll
      for (int k = 0; k < 4; k++) px[k] = ((v >> (8 * k)) & 255u) * 0x01010101u;
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) px[k] = (i0 + k < wlen) ? rowp[x0 + k] * 0x01010101u : 0u;
    }
    bool touched = false;
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (i0 + k < wlen) {
        uint32_t ax = (code[k] >= kArea && code[k] < kClear && kind == kRowOps) ? L.AX[i0 + k] : 0u;
        bool t = false;
        px[k] = mode == kNormal ? apply_normal(kind == kRowCoverage, code[k], ax, px[k], rgbx, &t)
                                : apply_code(kind, code[k], ax, px[k], rgbx, mode, &t);
        ntouch += t ? 1u : 0u;
        touched |= t;
      }
    }
    if (!touched) continue;
    if (full) {
      *(uint32_t*)(rowp + x0) = ch_a(px[0]) | (ch_a(px[1]) << 8) | (ch_a(px[2]) << 16) | (ch_a(px[3]) << 24);
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++)
        if (i0 + k < wlen) rowp[x0 + k] = (uint8_t)ch_a(px[k]);
    }
  }
  for (int i = lane; i < 4; i += kWave) {
    int idx = ((wlen + 4 * kWave - 1) / (4 * kWave)) * 4 * kWave + i;
    if (idx < L.ww + 4) L.D[idx] = 0;
  }
  wave_sync();
  return ntouch;
}

}  // namespace pxh
