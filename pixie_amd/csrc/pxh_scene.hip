// pxh_scene.hip -- the batched form: device geometry, band building and the
// two raster phases of a recorded scene (see pxh_scene.h).
//
// Every stage is exact with respect to the per-call form: flattening,
// stroking, segments, bounds and bands use the same pxh_geom.h functions in
// the same float32 order, and the row program is the same device code.
#include <hip/hip_runtime.h>

#include "pxh_raster.h"
#include "pxh_scene.h"

namespace pxh {

constexpr int kBlock = 256;
constexpr int kStagePts = 4096;  // LDS points of the geometry stage (32 KB)
constexpr int kBigSegGrid = 1024;  // workgroups of the big-fill segment kernels (grid-stride)
constexpr int kStrokeGrid = 2048;  // workgroups of the stroke segment kernels (grid-stride)
constexpr int kSegBandBlocks = 2048;  // workgroups of the band ranges (a wave per 64 segments)
constexpr int kTaskBlocks = 1024;     // workgroups of the work-item kernels (a wave per 64 units)

constexpr int kWinA = 512;    // phase-A column window
constexpr int kWinB = 512;    // phase-B column window (2 chunks of 256 px)
constexpr int kChunksB = kWinB / 256;

// ---------------------------------------------------------------------------
// block helpers (256 threads = 4 waves)
// ---------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ int block_excl_scan_n(int v, int* total, int* sh) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int wt;
  int x = wave_excl_scan(v, &wt);
  __syncthreads();
  if (lane == 0) sh[w] = wt;
  __syncthreads();
  int off = 0, tot = 0;
#pragma unroll
  for (int i = 0; i < NB / 64; i++) {
    int t = sh[i];
    if (i < w) off += t;
    tot += t;
  }
  *total = tot;
  return off + x;
}

// Single-workgroup scans over the big calls use the largest workgroup so that
// they take few serial steps.
constexpr int kScanBlock = 1024;

// ---------------------------------------------------------------------------
// commands (SceneCmd) -> points, commandsToShapes (paths.nim:654-1057)
// ---------------------------------------------------------------------------
__device__ __forceinline__ V2 cmd_end(const SceneCmd& c) {
  switch ((int)c.kind) {
    case 1: case 2: return v2(c.p[0], c.p[1]);  // Move, Line
    case 5: return v2(c.p[4], c.p[5]);          // Cubic
    case 7: return v2(c.p[2], c.p[3]);          // Quad
    default: return v2(c.sx, c.sy);             // Close
  }
}

struct CountEmit {
  int n = 0;
  __device__ void operator()(V2 a, V2 b) {
    V2 d = a - b;
    if (d.x != 0.0f || d.y != 0.0f) n++;  // addSegment skips zero-length pieces
  }
};

// Counts like CountEmit and keeps the first `cap` points in an LDS slice,
// transformed like StoreEmit, so that the emit stage can copy them instead of
// flattening the command again.
struct StageEmit {
  float2* buf;
  int cap;
  const float* mat;
  bool xf;
  bool writer = true;  // lanes of a flattening group count alike; one writes
  int n = 0;
  __device__ void operator()(V2 a, V2 b) {
    V2 d = a - b;
    if (d.x == 0.0f && d.y == 0.0f) return;  // addSegment skips zero-length pieces
    if (writer && n < cap) {
      V2 p = xf ? mat_apply(mat, b) : b;
      buf[n] = make_float2(p.x, p.y);
    }
    n++;
  }
};

// flatten_cubic (paths.nim:677-721) run by a group of G lanes of one wave
// (lanes gbase .. gbase + G - 1, u = lane - gbase).  Each
// round lane u tries the step halved u times; the first candidate in
// halving order that is accepted, or that reaches epsilon, decides the round,
// which is the decision the sequential loop reaches after u halvings (each
// halving and its reuse of the halfway point are exact, so the candidates
// evaluate the same points).  Every lane of the group calls emit alike.
template <int G>
struct Lanes {
  static constexpr int value = G;
};
template <int G, class Emit>
__device__ __forceinline__ int32_t flatten_cubic_group(V2 at, V2 c1, V2 c2, V2 to, float errSq, Emit& emit, int u,
                                       int gbase) {
  float t = 0.0f, step = 1.0f;
  V2 prev = at;
  for (;;) {
    float s = step;
    for (int q = 0; q < u; q++) s /= 2.0f;
    const bool eps = s <= kFltEpsilon;
    bool ok = false;
    V2 next = v2(0.0f, 0.0f);
    if (!eps) {
      next = cubic_at(at, c1, c2, to, t + s);
      const V2 halfway = cubic_at(at, c1, c2, to, t + s / 2.0f);
      const V2 midpoint = (prev + next) / 2.0f;
      const V2 lineTangent = midpoint - prev;
      const V2 curveTangent = cubic_deriv(at, c1, c2, to, t + s / 2.0f);
      const V2 curveTangentScaled = normalize(curveTangent) * len(lineTangent);
      const float error = lensq(midpoint - halfway);
      const float errorTangent = lensq(lineTangent - curveTangentScaled);
      ok = !(error + errorTangent > errSq);
    }
    const uint64_t bm = (__ballot(eps || ok) >> gbase) & ((1ull << G) - 1ull);
    if (bm == 0) {  // every candidate was refined: go on from step / 2^G
      for (int q = 0; q < G; q++) step /= 2.0f;
      continue;
    }
    const int src = gbase + __builtin_ctzll(bm);
    if (__shfl(eps ? 1 : 0, src, 64)) return kErrDiscretize;
    const float sw = __shfl(s, src, 64);
    const V2 nw = v2(__shfl(next.x, src, 64), __shfl(next.y, src, 64));
    emit(prev, nw);
    t += sw;
    if (t == 1.0f) break;
    prev = nw;
    step = nim_minf(sw * 2.0f, 1.0f - t);
  }
  return kOk;
}

struct StoreEmit {
  float2* out;
  int32_t* outPoly;
  int32_t poly;
  const float* mat;
  bool xf;
  int n = 0;
  __device__ void put(V2 p) {
    if (xf) p = mat_apply(mat, p);
    out[n] = make_float2(p.x, p.y);
    outPoly[n] = poly;
    n++;
  }
  __device__ void operator()(V2 a, V2 b) {
    V2 d = a - b;
    if (d.x != 0.0f || d.y != 0.0f) put(b);
  }
};

// Points command i emits (its non-degenerate pieces' end points).
template <class Emit>
__device__ __forceinline__ int32_t cmd_emit(const SceneCmd* cmds, int i, float errSq, Emit& e) {
  const SceneCmd& c = cmds[i];
  int k = (int)c.kind;
  if (k == 1) return kOk;  // Move
  V2 at = cmd_end(cmds[i - 1]);  // a subpath always starts with a Move
  switch (k) {
    case 2: e(at, v2(c.p[0], c.p[1])); return kOk;
    case 5: return flatten_cubic(at, v2(c.p[0], c.p[1]), v2(c.p[2], c.p[3]), v2(c.p[4], c.p[5]), errSq, e);
    case 7: return flatten_quad(at, v2(c.p[0], c.p[1]), v2(c.p[2], c.p[3]), errSq, e);
    case 0: {  // Close: addSegment(at, start) when at != start
      V2 st = v2(c.sx, c.sy);
      if (!veq(at, st)) e(at, st);
      return kOk;
    }
    default: return kErrArg;
  }
}

// ---------------------------------------------------------------------------
// stroke polygons (strokeShapes, paths.nim:1922-2082) -> segments
// ---------------------------------------------------------------------------
struct SegSink {
  // counting when out == nullptr
  float4* out = nullptr;
  int8_t* outW = nullptr;
  int n = 0;
  int err = 0;  // a dash pattern ran past kMaxDashPasses
  Bounds bd;
  __device__ void seg(V2 v1, V2 v2_) {
    Seg s;
    if (!make_segment(v1, v2_, &s)) return;
    if (out) {
      out[n] = make_float4(s.at.x, s.at.y, s.to.x, s.to.y);
      outW[n] = (int8_t)s.w;
      bounds_add(&bd, s);
    }
    n++;
  }
  // shapesToSegments (paths.nim:1069-1090) of one polygon q[0..m)
  __device__ void poly(const V2* q, int m, const SceneItem& I) {
    if (m <= 0) return;
    V2 last = I.identity ? q[m - 1] : mat_apply(I.mat, q[m - 1]);
    V2 vec1 = v2(last.x, quantize_y(last.y));
    for (int i = 0; i < m; i++) {
      V2 p = I.identity ? q[i] : mat_apply(I.mat, q[i]);
      V2 vec2 = v2(p.x, quantize_y(p.y));
      if (i == 0 && veq(vec1, vec2)) continue;
      seg(vec1, vec2);
      vec1 = vec2;
    }
  }
};

// Streams the polygon of makeCircle (paths.nim:1938-1941): the ellipse
// path's first shape.  Its last point equals its first bit for bit (the last
// cubic ends on the Move point), so the closing candidate is always skipped.
struct CircleEmit {
  SegSink* sink;
  const SceneItem* I;
  V2 prevq;
  __device__ void add(V2 p) {
    V2 t = I->identity ? p : mat_apply(I->mat, p);
    V2 q = v2(t.x, quantize_y(t.y));
    sink->seg(prevq, q);
    prevq = q;
  }
  __device__ void operator()(V2 a, V2 b) {
    V2 d = a - b;
    if (d.x != 0.0f || d.y != 0.0f) add(b);
  }
};

// The quarters [q0, q1) of the circle: quarter q's cubic starts where quarter
// q - 1's ends (its last flattened point is its end point exactly: the cubic
// at t = 1 adds zeros to it), so the quarters are independent.
__device__ __forceinline__ void circle_segments(V2 at, int q0, int q1, const SceneItem& I, SegSink& sink) {
  const double K = 4.0 * (-1.0 + 1.4142135623730951) / 3.0;  // splineCircleK (float64)
  const float cx = at.x, cy = at.y, rx = I.halfStroke, ry = I.halfStroke;
  const double mx = K * (double)rx, my = K * (double)ry;
  const float right = cx + rx, left = cx - rx, low = cy + ry, high = cy - ry;
  const float yp = (float)((double)cy + my), yn = (float)((double)cy - my);
  const float xp = (float)((double)cx + mx), xn = (float)((double)cx - mx);
#pragma unroll 1
  for (int q = q0; q < q1; q++) {
    const V2 a = q == 0 ? v2(right, cy) : q == 1 ? v2(cx, low) : q == 2 ? v2(left, cy) : v2(cx, high);
    const V2 c1 = q == 0 ? v2(right, yp) : q == 1 ? v2(xn, low) : q == 2 ? v2(left, yn) : v2(xp, high);
    const V2 c2 = q == 0 ? v2(xp, low) : q == 1 ? v2(left, yp) : q == 2 ? v2(xn, high) : v2(right, yn);
    const V2 to = q == 0 ? v2(cx, low) : q == 1 ? v2(left, cy) : q == 2 ? v2(cx, high) : v2(right, cy);
    const V2 st = I.identity ? a : mat_apply(I.mat, a);
    CircleEmit ce{&sink, &I, v2(st.x, quantize_y(st.y))};
    flatten_cubic(a, c1, c2, to, I.errSq, ce);
  }
}

__device__ __forceinline__ void rect_segments(V2 at, V2 to, const SceneItem& I, SegSink& sink) {  // makeRect
  float hs = I.halfStroke;
  V2 tangent = normalize(to - at);
  V2 normal = v2(tangent.y, tangent.x);
  V2 q[5];
  q[0] = v2(at.x + normal.x * hs, at.y - normal.y * hs);
  q[1] = v2(to.x + normal.x * hs, to.y - normal.y * hs);
  q[2] = v2(to.x - normal.x * hs, to.y + normal.y * hs);
  q[3] = v2(at.x - normal.x * hs, at.y + normal.y * hs);
  q[4] = q[0];
  sink.poly(q, 5, I);
}

__device__ __forceinline__ float fix_angle_d(float a) {  // vmath fixAngle
  const float PI = 3.14159265358979323846f;
  while (a > PI) a -= PI * 2.0f;
  while (a < -PI) a += PI * 2.0f;
  return a;
}

// A round join's circle is left to the caller (*circle = true): it is always
// the last polygon a stroke point emits, so stroke_point draws every circle
// from one place.
__device__ __forceinline__ void join_segments(V2 prevPos, V2 pos, V2 nextPos, const SceneItem& I,
                                              SegSink& sink, bool* circle) {
  const float PI = 3.14159265358979323846f;
  float minArea = I.minArea, hs = I.halfStroke;
  if (I.join == 1) {  // RoundJoin
    float area = PI * hs * hs;
    if (area > minArea) *circle = true;
    return;
  }
  V2 dn = nextPos - pos, dp = prevPos - pos;
  float angle = fix_angle_d(atan2f(dn.y, dn.x) - atan2f(dp.y, dp.x));
  if (fabsf(fabsf(angle) - PI) > 0.00031415926535897936f) {
    V2 a = normalize(pos - prevPos) * hs;
    V2 b = normalize(pos - nextPos) * hs;
    if (angle >= 0.0f) {
      a = v2(-a.y, a.x);
      b = v2(b.y, -b.x);
    } else {
      a = v2(a.y, -a.x);
      b = v2(-b.y, b.x);
    }
    int j = I.join;
    if (j == 0 && fabsf(angle) < I.miterAngleLimit) j = 2;
    if (j == 0) {
      V2 la0 = prevPos + a, la1 = pos + a, lb0 = nextPos + b, lb1 = pos + b;
      V2 s1 = la1 - la0, s2 = lb1 - lb0;
      float den = (-s2.x * s1.y + s1.x * s2.y);
      if (den != 0.0f) {
        float t = (s2.x * (la0.y - lb0.y) - s2.y * (la0.x - lb0.x)) / den;
        V2 at = la0 + s1 * t;
        float bl = lensq(at - pos);
        float areaSq = 0.25f * (lensq(a) * bl + lensq(b) * bl);
        if (areaSq > minArea * minArea) {
          V2 q[5] = {pos + a, at, pos + b, pos, pos + a};
          sink.poly(q, 5, I);
        }
      }
    } else if (j == 2) {
      float areaSq = 0.25f * lensq(a) * lensq(b);
      if (areaSq > minArea * minArea) {
        V2 q[4] = {a + pos, b + pos, pos, a + pos};
        sink.poly(q, 4, I);
      }
    }
  }
}

// The stroke of a call whose joins or caps are circles spreads every point
// over four lanes, one per quarter of its circle.
__device__ __forceinline__ int stroke_lanes(const SceneItem& I) { return (I.join == 1 || I.cap == 1) ? 4 : 1; }

// Segments of point k of a stroked polyline P[0..n), in strokeShapes order:
// its cap or its segment rectangle and join.  A round cap or round join comes
// last, so the one circle a point may need is drawn at the end, from a single
// call site (which keeps I and sink in registers once inlined).  Lane `sub` of
// the point's `lanes` emits its share: lane 0 what precedes the circle, and
// each lane its quarters of the circle.
__device__ __forceinline__ void stroke_point(const float2* P, int k, int n, const SceneItem& I,
                                             const float* dash, SegSink& sink, int sub, int lanes) {
  auto pt = [&](int i) { return v2(P[i].x, P[i].y); };
  bool closed = veq(pt(0), pt(n - 1));
  bool circle = false;
  V2 center = v2(0.0f, 0.0f);
  if (sub > 0) {
    const bool cap = !closed && (k == 0 || k == n - 1) && I.cap == 1;
    const bool join = k > 0 && (k < n - 1 || (closed && n >= 2)) && I.join == 1;
    if (join) join_segments(pt(k), pt(k), pt(k), I, sink, &circle);  // a round join only decides on its circle
    circle = circle || cap;
    center = pt(k);
  } else if (k == 0) {
    if (!closed) {
      if (I.cap == 1) {
        circle = true;
        center = pt(0);
      } else if (I.cap == 2) {
        V2 tangent = normalize(pt(1) - pt(0));
        rect_segments(pt(0) - tangent * I.halfStroke, pt(0), I, sink);
      }
    }
  } else {
    if (I.dashCount > 0) {
      // the dash pattern restarts on every segment (paths.nim:2046-2059)
      const V2 prevPos = pt(k - 1), pos = pt(k);
      float distance = len(prevPos - pos);
      const V2 dir = normalize(pos - prevPos);
      V2 currPos = prevPos;
      bool done = false;
      for (int pass = 0; !done; pass++) {
        if (pass == kMaxDashPasses) {
          sink.err = 1;
          break;
        }
        for (int j = 0; j < I.dashCount; j++) {
          const float d = dash[j];
          if ((j & 1) == 0) rect_segments(currPos, currPos + dir * nim_minf(distance, d), I, sink);
          currPos = currPos + dir * d;
          distance -= d;
          if (distance <= 0.0f) {
            done = true;
            break;
          }
        }
      }
    } else {
      rect_segments(pt(k - 1), pt(k), I, sink);
    }
    if (k < n - 1) {
      join_segments(pt(k - 1), pt(k), pt(k + 1), I, sink, &circle);
      center = pt(k);
    }
    if (k == n - 1) {
      if (closed) {
        if (n >= 2) {
          join_segments(pt(n - 2), pt(n - 1), pt(1), I, sink, &circle);
          center = pt(n - 1);
        }
      } else {
        if (I.cap == 1) {
          circle = true;
          center = pt(n - 1);
        } else if (I.cap == 2) {
          V2 tangent = normalize(pt(n - 1) - pt(n - 2));
          rect_segments(pt(n - 1) + tangent * I.halfStroke, pt(n - 1), I, sink);
        }
      }
    }
  }
  if (circle) {
    const int per = 4 / lanes;
    circle_segments(center, sub * per, (sub + 1) * per, I, sink);
  }
}

// ---------------------------------------------------------------------------
// geometry: one workgroup per call
// ---------------------------------------------------------------------------
// Stage 6 of a fill: the call's bounds (merged from every thread's `bd`)
// give its fill locals and band layout (fill_locals, band_layout).
template <int NB>
__device__ __forceinline__ void geom_finish(const ScenePools& P, const SceneItem& I, int it, Bounds bd, int nseg,
                                            Bounds* sBd) {
  const int tid = threadIdx.x;
  for (int o = 32; o > 0; o >>= 1) {
    Bounds ob;
    ob.xMin = __shfl_xor(bd.xMin, o, 64);
    ob.xMax = __shfl_xor(bd.xMax, o, 64);
    ob.yMin = __shfl_xor(bd.yMin, o, 64);
    ob.yMax = __shfl_xor(bd.yMax, o, 64);
    bd = bounds_merge(bd, ob);
  }
  if ((tid & 63) == 0) sBd[tid >> 6] = bd;
  __syncthreads();
  if (tid != 0) return;
  Bounds b = sBd[0];
  for (int w = 1; w < NB / 64; w++) b = bounds_merge(b, sBd[w]);
  FillInfo f = {};
  f.rgbx = I.rgbx;
  f.mode = I.mode;
  f.rule = I.rule;
  const int32_t r = fill_locals(b, false, P.W, P.H, &f);
  f.status = r;
  if (r == kOk && f.pathWidth > 0) band_layout(&f, nseg);
  P.fills[it] = f;
}

// Marks the 64-segment groups a call has allocated, for the band-range stage.
__device__ __forceinline__ void mark_groups(const ScenePools& P, int it, int segBase, int segs) {
  for (int g = (int)threadIdx.x; g < (segs + 63) / 64; g += (int)blockDim.x) P.groupItem[(segBase >> 6) + g] = it;
}

// Registers the chunks of a stroke's points (the whole workgroup; none when
// the call failed).
__device__ __forceinline__ void stroke_register(const ScenePools& P, const SceneItem& I, int it, int points) {
  __shared__ int sChunk;
  const int per = 256 / stroke_lanes(I);
  const int n = I.strokeNone ? 0 : (points + per - 1) / per;
  if (threadIdx.x == 0) {
    sChunk = n ? atomicAdd(&P.counters[kCntStrokeChunks], n) : 0;
    StrokeCall st = {};
    st.chunkBase = sChunk;
    st.nChunks = n;
    st.err = kOk;
    P.strokes[it] = st;
  }
  __syncthreads();
  for (int c = (int)threadIdx.x; c < n; c += (int)blockDim.x) P.strokeChunk[sChunk + c] = make_int2(it, 0);
}

// Thread per command of the calls of more than kBlock commands (the first
// nBig calls of itemOrder; bigCmdStart holds their command prefix): counts
// its points (emit = 0; a negative count is an error code), or writes them
// at the offsets the front half computed (emit = 1).
__global__ void __launch_bounds__(256) scene_big_cmd_kernel(ScenePools P, int emit) {
  const int gid = blockIdx.x * 256 + threadIdx.x;
  if (gid >= P.bigCmdStart[P.nBig]) return;
  int lo = 0, hi = P.nBig;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (P.bigCmdStart[mid] <= gid) lo = mid;
    else hi = mid;
  }
  const int it = P.itemOrder[lo];
  const SceneItem& I = P.items[it];
  const int i = I.cmdBase + (gid - P.bigCmdStart[lo]);
  const bool xf = !I.stroke && !I.identity;
  if (!emit) {
    CountEmit ce;
    const int32_t r = cmd_emit(P.cmds, i, I.errSq, ce);
    P.cmdCount[i] = r != kOk ? -r : ce.n;
    return;
  }
  if (P.geo[it].status != kOk || P.cmdCount[i] <= 0) return;
  const int o = P.geo[it].ptBase + P.cmdOff[i];
  StoreEmit se{P.pts + o, P.ptPoly + o, P.cmds[i].pad[0], I.mat, xf};
  cmd_emit(P.cmds, i, I.errSq, se);
}

// ---- the segment stage of big fills, spread over the device ----
// Stage 5 of a fill makes a segment from each point and its predecessor
// (the first point of a subpath pairs with its last), skipping horizontal
// ones; segments keep point order.  For a big fill the points are cut into
// chunks of kBigChunk (256 threads x 16 consecutive points): the chunks
// count their segments and bounds, one workgroup per call scans the counts,
// merges the bounds and lays out the call's bands (stage 6), the chunks
// write their segments at the scanned offsets, and one wave per 64-segment
// group finds the band ranges (stage 7).  The result is the one-workgroup
// back half's, segment for segment.

__device__ __forceinline__ bool fill_point_seg(const ScenePools& P, const SceneItem& I, const float2* pts,
                                               const int32_t* ptPoly, int j, Seg* s) {
  const int q = I.polyBase + ptPoly[j];
  const int pb = P.polyPt[q], np = P.polyN[q];
  const float2 pa = j == pb ? pts[pb + np - 1] : pts[j - 1];
  const float2 pc = pts[j];
  const V2 v1 = v2(pa.x, quantize_y(pa.y)), v2_ = v2(pc.x, quantize_y(pc.y));
  return !(j == pb && veq(v1, v2_)) && make_segment(v1, v2_, s);
}

// The big call whose range of `start` (an exclusive prefix, nBig + 1
// entries) holds index c.
__device__ __forceinline__ int big_call_of(const int32_t* start, int nBig, int c) {
  int lo = 0, hi = nBig;
  while (hi - lo > 1) {
    const int mid = (lo + hi) / 2;
    if (start[mid] <= c) lo = mid;
    else hi = mid;
  }
  return lo;
}

// Block-wide bounds of 256 threads (valid in every thread after the call).
__device__ __forceinline__ Bounds block_bounds256(Bounds bd, Bounds* sBd) {
  for (int o = 32; o > 0; o >>= 1) {
    Bounds ob;
    ob.xMin = __shfl_xor(bd.xMin, o, 64);
    ob.xMax = __shfl_xor(bd.xMax, o, 64);
    ob.yMin = __shfl_xor(bd.yMin, o, 64);
    ob.yMax = __shfl_xor(bd.yMax, o, 64);
    bd = bounds_merge(bd, ob);
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sBd[threadIdx.x >> 6] = bd;
  __syncthreads();
  Bounds b = sBd[0];
  for (int w = 1; w < 4; w++) b = bounds_merge(b, sBd[w]);
  return b;
}

// Prefixes over the big calls: subpath chunks of every call (what = 2),
// and point chunks of the fills whose points were laid out (what = 0).
__global__ void __launch_bounds__(kScanBlock) scene_big_plan_kernel(ScenePools P, int what) {
  __shared__ int sh[kScanBlock / 64];
  int32_t* out = what == 2 ? P.bigPolyStart : P.bigChunkStart;
  int carry = 0;
  for (int i0 = 0; i0 < P.nBig; i0 += kScanBlock) {
    const int i = i0 + threadIdx.x;
    int n = 0;
    if (i < P.nBig) {
      const int it = P.itemOrder[i];
      if (what == 2) {
        n = (P.items[it].polyCount + kBigPolyChunk - 1) / kBigPolyChunk;
      } else {
        const ItemGeom g = P.geo[it];
        if (!P.items[it].stroke && g.status == kOk) n = (g.ptCount + kBigChunk - 1) / kBigChunk;
      }
    }
    int t;
    const int off = block_excl_scan_n<kScanBlock>(n, &t, sh);
    if (i < P.nBig) out[i] = carry + off;
    carry += t;
    __syncthreads();
  }
  if (threadIdx.x == 0) out[P.nBig] = carry;
}

// ---- the point layout of big calls (geometry stages 2-3), spread over
// the device: each chunk of kBigPolyChunk subpaths (256 threads x 4)
// counts its subpaths' points and finds count errors, one workgroup per call
// scans the chunk totals and allocates the call's points, and the chunks
// place their subpaths (offsets, per-command offsets, start and closing
// points).  The layout is the one-workgroup front half's, point for point.

// Points of subpath q (stage 2): start + pieces, plus the implicit closing
// point of a fill; *err gets a command's error code.
__device__ __forceinline__ int big_poly_points(const ScenePools& P, const SceneItem& I, int q, int* err) {
  const ScenePoly sp = P.polys[q];
  int n = 0;
  for (int c = 0; c < sp.numCmds; c++) {
    const int k = P.cmdCount[sp.firstCmd + c];
    if (k < 0) *err = max(*err, -k);
    else n += k;
  }
  if (n <= 0) return 0;
  int np = n + 1;
  const SceneCmd& last = P.cmds[sp.firstCmd + sp.numCmds - 1];
  if (!I.stroke && (int)last.kind != 0 && !sp.noClose) {
    V2 d = cmd_end(last) - v2(last.sx, last.sy);
    if (d.x != 0.0f || d.y != 0.0f) np++;
  }
  return np;
}

// emit = 0: points and errors per chunk; emit = 1: subpath placement.
__global__ void __launch_bounds__(256) scene_big_front_kernel(ScenePools P, int emit) {
  __shared__ int sh[4];
  const int nChunks = P.bigPolyStart[P.nBig];
  for (int c = blockIdx.x; c < nChunks; c += gridDim.x) {
    const int bi = big_call_of(P.bigPolyStart, P.nBig, c);
    const int it = P.itemOrder[bi];
    const SceneItem& I = P.items[it];
    const int ql0 = (c - P.bigPolyStart[bi]) * kBigPolyChunk + threadIdx.x * 4;
    if (!emit) {
      int sum = 0, err = kOk;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int ql = ql0 + u;
        if (ql < I.polyCount) {
          const int np = big_poly_points(P, I, I.polyBase + ql, &err);
          P.polyN[I.polyBase + ql] = np;
          sum += np;
        }
      }
      int t;
      block_excl_scan_n<256>(sum, &t, sh);
      for (int o = 32; o > 0; o >>= 1) err = max(err, __shfl_xor(err, o, 64));
      __syncthreads();
      if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = err;
      __syncthreads();
      if (threadIdx.x == 0) P.bigPolyChunk[c] = make_int4(t, max(max(sh[0], sh[1]), max(sh[2], sh[3])), 0, 0);
      __syncthreads();
      continue;
    }
    const ItemGeom g = P.geo[it];
    if (g.status != kOk) continue;  // the same for the whole block
    int np[4], sum = 0;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int ql = ql0 + u;
      np[u] = ql < I.polyCount ? P.polyN[I.polyBase + ql] : 0;
      sum += np[u];
    }
    int t;
    int pb = P.bigPolyChunk[c].z + block_excl_scan_n<256>(sum, &t, sh);
    const bool xf = !I.stroke && !I.identity;
    float2* pts = P.pts + g.ptBase;
    int32_t* ptPoly = P.ptPoly + g.ptBase;
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int ql = ql0 + u;
      if (ql < I.polyCount) {  // stage 3
        const int q = I.polyBase + ql;
        P.polyPt[q] = pb;
        const ScenePoly sp = P.polys[q];
        int off = pb + 1;
        for (int k = 0; k < sp.numCmds; k++) {
          P.cmdOff[sp.firstCmd + k] = off;
          off += P.cmdCount[sp.firstCmd + k];
        }
        if (np[u] > 0) {
          const SceneCmd& mv = P.cmds[sp.firstCmd];
          V2 s = v2(mv.sx, mv.sy);
          V2 w = xf ? mat_apply(I.mat, s) : s;
          pts[pb] = make_float2(w.x, w.y);
          ptPoly[pb] = ql;
          if (off < pb + np[u]) {  // implicit closing point of a fill
            pts[off] = make_float2(w.x, w.y);
            ptPoly[off] = ql;
          }
        }
        pb += np[u];
      }
    }
    __syncthreads();
  }
}

// One workgroup per big call: its point total and errors from the chunks,
// the chunks' point offsets, and the call's point allocation.
__global__ void __launch_bounds__(256) scene_big_front_alloc_kernel(ScenePools P) {
  __shared__ int sh[4];
  const int bi = blockIdx.x;
  const int it = P.itemOrder[bi];
  const SceneItem& I = P.items[it];
  const int c0 = P.bigPolyStart[bi], nc = P.bigPolyStart[bi + 1] - c0;
  int carry = 0, err = kOk;
  for (int k0 = 0; k0 < nc; k0 += 256) {
    const int k = k0 + threadIdx.x;
    int n = 0;
    if (k < nc) {
      const int4 ch = P.bigPolyChunk[c0 + k];
      n = ch.x;
      err = max(err, ch.y);
    }
    int t;
    const int off = block_excl_scan_n<256>(n, &t, sh);
    if (k < nc) P.bigPolyChunk[c0 + k].z = carry + off;
    carry += t;
    __syncthreads();
  }
  for (int o = 32; o > 0; o >>= 1) err = max(err, __shfl_xor(err, o, 64));
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = err;
  __syncthreads();
  err = max(max(sh[0], sh[1]), max(sh[2], sh[3]));
  const int total = carry;
  __syncthreads();
  if (threadIdx.x == 0) {
    int base = 0;
    if (err == kOk) {
      base = atomicAdd(&P.counters[kCntPoints], total);
      if (base + total > P.ptCap) {
        atomicOr(&P.counters[kCntError], 1);
        err = kErrCapacity;
      }
      // strokeShapes checks the dash values once it meets a shape with
      // points (paths.nim:2029-2031)
      if (I.stroke && !I.strokeNone && I.dashBad && total > 0 && err == kOk) err = kErrDash;
    }
    ItemGeom g = {};
    if (err != kOk) {
      g.status = err;
      P.fills[it].status = err;
      P.fills[it].pathWidth = 0;
    } else {
      g.ptBase = base;
      g.ptCount = total;
      g.status = kOk;
    }
    P.geo[it] = g;
    sh[0] = err;
  }
  __syncthreads();
  if (I.stroke) stroke_register(P, I, it, sh[0] == kOk ? total : 0);
}

// Segments and bounds of each chunk (emit = 0), or its segments written at
// the call's segment base plus the chunk's scanned offset (emit = 1).
__global__ void __launch_bounds__(256) scene_big_seg_kernel(ScenePools P, int emit) {
  __shared__ int sh[4];
  __shared__ Bounds sBd[4];
  const int nChunks = P.bigChunkStart[P.nBig];
  for (int c = blockIdx.x; c < nChunks; c += gridDim.x) {
    const int bi = big_call_of(P.bigChunkStart, P.nBig, c);
    const int it = P.itemOrder[bi];
    const SceneItem& I = P.items[it];
    const ItemGeom g = P.geo[it];
    if (emit && g.status != kOk) continue;  // the same for the whole block
    const float2* pts = P.pts + g.ptBase;
    const int32_t* ptPoly = P.ptPoly + g.ptBase;
    const int j0 = (c - P.bigChunkStart[bi]) * kBigChunk + threadIdx.x * 16;
    float4 sg[16];
    int8_t sw[16];
    uint32_t valid = 0;
    Bounds bd = bounds_init();
#pragma unroll
    for (int u = 0; u < 16; u++) {
      const int j = j0 + u;
      Seg s;
      if (j < g.ptCount && fill_point_seg(P, I, pts, ptPoly, j, &s)) {
        sg[u] = make_float4(s.at.x, s.at.y, s.to.x, s.to.y);
        sw[u] = (int8_t)s.w;
        bounds_add(&bd, s);
        valid |= 1u << u;
      }
    }
    const int n = __popc(valid);
    int t;
    const int off = block_excl_scan_n<256>(n, &t, sh);
    if (!emit) {
      const Bounds b = block_bounds256(bd, sBd);
      if (threadIdx.x == 0) {
        P.bigChunkCnt[c] = make_int2(t, 0);
        P.bigChunkBd[c] = make_float4(b.xMin, b.xMax, b.yMin, b.yMax);
      }
    } else {
      const int w = g.segBase + P.bigChunkCnt[c].y + off;
      int k = 0;
#pragma unroll
      for (int u = 0; u < 16; u++)
        if ((valid >> u) & 1u) {
          P.segs[w + k] = sg[u];
          P.segW[w + k] = sw[u];
          k++;
        }
    }
    __syncthreads();
  }
}

// One workgroup per big call: scans its chunk counts, merges their bounds,
// allocates the segments and lays out the fill (stage 6).
__global__ void __launch_bounds__(256) scene_big_seg_alloc_kernel(ScenePools P) {
  __shared__ int sh[4];
  __shared__ Bounds sBd[4];
  const int bi = blockIdx.x;
  const int it = P.itemOrder[bi];
  const SceneItem& I = P.items[it];
  if (I.stroke) return;
  ItemGeom g = P.geo[it];
  if (g.status != kOk) return;  // the front half wrote the error
  const int c0 = P.bigChunkStart[bi], nc = P.bigChunkStart[bi + 1] - c0;
  int carry = 0;
  Bounds bd = bounds_init();
  for (int k0 = 0; k0 < nc; k0 += 256) {
    const int k = k0 + threadIdx.x;
    int n = 0;
    if (k < nc) {
      n = P.bigChunkCnt[c0 + k].x;
      const float4 b = P.bigChunkBd[c0 + k];
      Bounds cb;
      cb.xMin = b.x;
      cb.xMax = b.y;
      cb.yMin = b.z;
      cb.yMax = b.w;
      bd = bounds_merge(bd, cb);
    }
    int t;
    const int off = block_excl_scan_n<256>(n, &t, sh);
    if (k < nc) P.bigChunkCnt[c0 + k].y = carry + off;
    carry += t;
    __syncthreads();
  }
  const Bounds b = block_bounds256(bd, sBd);
  const int nseg = carry;
  if (threadIdx.x == 0) {
    // segments start on a 64-segment group of their own
    const int base = atomicAdd(&P.counters[kCntSegs], (nseg + 63) & ~63);
    FillInfo f = {};
    f.rgbx = I.rgbx;
    f.mode = I.mode;
    f.rule = I.rule;
    if (base + nseg > P.segCap) {
      atomicOr(&P.counters[kCntError], 1);
      f.status = kErrCapacity;
      f.pathWidth = 0;
      g.segBase = 0;
      g.segCount = 0;
      g.status = kErrCapacity;
    } else {
      const int32_t r = fill_locals(b, false, P.W, P.H, &f);
      f.status = r;
      if (r == kOk && f.pathWidth > 0) band_layout(&f, nseg);
      g.segBase = base;
      g.segCount = nseg;
      g.status = r;
    }
    P.fills[it] = f;
    P.geo[it] = g;
    sh[0] = g.status == kErrCapacity ? -1 : base;
  }
  __syncthreads();
  if (sh[0] >= 0) mark_groups(P, it, sh[0], nseg);
}

// ---- strokes, spread over the device (stages 5-6) ----
// A stroke makes tens of segments per point (a round join flattens a circle),
// and segments keep point order.  Its points are cut into chunks of 256 lanes
// (64 points of four lanes, or 256 of one): the chunks count their segments,
// one workgroup per stroke scans the counts and allocates, and the chunks
// write theirs and merge their bounds.  In one workgroup per stroke these
// stages were the tail of the whole geometry: 630 of the 800 thousand cycles
// of the longest call (1,303 points, 26,038 segments) of 100 paths on
// 1,023 x 767, whose geometry took 340 us and now takes 73 + 9 + 7 + 13.

// Order-preserving map of a non-NaN float to an unsigned, for atomic bounds.
__device__ __forceinline__ uint32_t bound_key(float f) {
  const uint32_t u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float bound_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// Without kEmit: the segments of every chunk; with it: the segments written,
// and the bounds.
template <bool kEmit>
__global__ void __launch_bounds__(256) scene_stroke_kernel(ScenePools P) {
  __shared__ int sh[4];
  __shared__ Bounds sBd[4];
  if (P.counters[kCntError]) return;
  const int nChunks = P.counters[kCntStrokeChunks];
  for (int c = blockIdx.x; c < nChunks; c += gridDim.x) {
    const int2 ch = P.strokeChunk[c];
    const int it = ch.x;
    const SceneItem& I = P.items[it];
    const ItemGeom g = P.geo[it];
    if (kEmit && g.status != kOk) continue;  // the same for the whole block
    const int lanes = stroke_lanes(I), sub = (int)threadIdx.x % lanes;
    const int j = (c - P.strokes[it].chunkBase) * (256 / lanes) + (int)threadIdx.x / lanes;
    const float2* pts = P.pts + g.ptBase;
    int n = 0, pb = 0, np = 0;
    int32_t err = 0;
    if (j < g.ptCount) {
      const int q = I.polyBase + P.ptPoly[g.ptBase + j];
      pb = P.polyPt[q];
      np = P.polyN[q];
      // a lane of four keeps up to 254 of its segments in its byte of ptSeg
      // (255: counted again); a point of one lane has the whole word
      if (kEmit) {
        const uint32_t w = (uint32_t)P.ptSeg[g.ptBase + j];
        n = lanes == 1 ? (int)w : (int)((w >> (8 * sub)) & 255u);
      }
      if (!kEmit || (lanes > 1 && n == 255)) {
        SegSink sink;
        stroke_point(pts + pb, j - pb, np, I, P.dashes + I.dashBase, sink, sub, lanes);
        n = sink.n;
        err = sink.err;
      }
    }
    if (!kEmit) {
      if (err) atomicMax(&P.strokes[it].err, (int32_t)kErrCapacity);
      uint32_t w = (uint32_t)n;
      if (lanes > 1) {  // the same for the whole block
        w = (uint32_t)(n < 255 ? n : 255) << (8 * sub);
        w |= (uint32_t)__shfl_xor((int)w, 1, 64);
        w |= (uint32_t)__shfl_xor((int)w, 2, 64);
      }
      if (sub == 0 && j < g.ptCount) P.ptSeg[g.ptBase + j] = (int32_t)w;
    }
    int t;
    const int off = block_excl_scan_n<256>(n, &t, sh);
    if (!kEmit) {
      if (threadIdx.x == 0) P.strokeChunk[c].y = t;
    } else {
      SegSink out;
      out.bd = bounds_init();
      if (n > 0) {
        const int w = g.segBase + ch.y + off;
        out.out = P.segs + w;
        out.outW = P.segW + w;
        stroke_point(pts + pb, j - pb, np, I, P.dashes + I.dashBase, out, sub, lanes);
      }
      const Bounds b = block_bounds256(out.bd, sBd);
      if (threadIdx.x == 0 && t > 0) {
        uint32_t* const bd = P.strokes[it].bd;
        atomicMin(&bd[0], bound_key(b.xMin));
        atomicMax(&bd[1], bound_key(b.xMax));
        atomicMin(&bd[2], bound_key(b.yMin));
        atomicMax(&bd[3], bound_key(b.yMax));
      }
    }
    __syncthreads();
  }
}

// One workgroup per stroke: scans its chunk counts and allocates its segments.
__global__ void __launch_bounds__(256) scene_stroke_alloc_kernel(ScenePools P) {
  __shared__ int sh[4];
  __shared__ int sBase;
  const int it = P.strokeItems[blockIdx.x];
  const SceneItem& I = P.items[it];
  ItemGeom g = P.geo[it];
  if (g.status != kOk) return;  // the point layout wrote the error
  const int chunkBase = P.strokes[it].chunkBase, nChunks = P.strokes[it].nChunks;
  int carry = 0;
  for (int k0 = 0; k0 < nChunks; k0 += 256) {
    const int k = k0 + threadIdx.x;
    const int n = k < nChunks ? P.strokeChunk[chunkBase + k].y : 0;
    int t;
    const int off = block_excl_scan_n<256>(n, &t, sh);
    if (k < nChunks) P.strokeChunk[chunkBase + k].y = carry + off;
    carry += t;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    int32_t status = P.strokes[it].err;
    int base = 0;
    if (status == kOk) {
      // segments start on a 64-segment group of their own
      base = atomicAdd(&P.counters[kCntSegs], (carry + 63) & ~63);
      if (base + carry > P.segCap) {
        atomicOr(&P.counters[kCntError], 1);
        status = kErrCapacity;
      }
    }
    const Bounds b = bounds_init();
    uint32_t* const bd = P.strokes[it].bd;
    bd[0] = bound_key(b.xMin);
    bd[1] = bound_key(b.xMax);
    bd[2] = bound_key(b.yMin);
    bd[3] = bound_key(b.yMax);
    g.segBase = status == kOk ? base : 0;
    g.segCount = status == kOk ? carry : 0;
    g.status = status;
    P.geo[it] = g;
    // the band-range stage writes the fill of a stroke that has segments
    FillInfo f = {};
    f.rgbx = I.rgbx;
    f.mode = I.mode;
    f.rule = kNonZero;
    f.status = status != kOk ? status : fill_locals(b, false, P.W, P.H, &f);
    P.fills[it] = f;
    sBase = status == kOk ? base : -1;
  }
  __syncthreads();
  if (sBase >= 0) mark_groups(P, it, sBase, carry);
}

// A stroke's fill from its merged bounds (stage 6).
__device__ __forceinline__ void stroke_fill(const ScenePools& P, int it, int segCount, FillInfo* f) {
  const uint32_t* bd = P.strokes[it].bd;
  Bounds b;
  b.xMin = bound_value(bd[0]);
  b.xMax = bound_value(bd[1]);
  b.yMin = bound_value(bd[2]);
  b.yMax = bound_value(bd[3]);
  f->status = fill_locals(b, false, P.W, P.H, f);
  if (f->status == kOk && f->pathWidth > 0) band_layout(f, segCount);
}

// Geometry of a call of at most kBlock commands, one workgroup per call: a
// fill's stages 1-6; a stroke ends here with its points (scene_stroke_*).
// The other calls spread their stages over the CUs: scene_big_cmd_kernel
// counts every command's points, scene_big_front_* lay the points out (stages
// 2-3), scene_big_cmd_kernel emits them, and scene_big_seg_* make the
// segments of fills.
__global__ void __launch_bounds__(kBlock) scene_geom_kernel(ScenePools P, int orderBase) {
  constexpr int NB = kBlock;
  __shared__ int sh[NB / 64];
  __shared__ int sBase;
  __shared__ Bounds sBd[NB / 64];
  __shared__ int sErr;
  __shared__ float2 sPts[kStagePts];
  __shared__ int sPre[NB + 1];
  const int it = P.itemOrder[orderBase + blockIdx.x];
  const int tid = threadIdx.x;
  const SceneItem& I = P.items[it];
  const bool xf = !I.stroke && !I.identity;  // fills transform points here
  if (tid == 0) sErr = kOk;
  __syncthreads();

  int total = 0;
  // 1. points per command, kept in an LDS slice per command (thread tid <->
  // command tid in stages 1 and 4), so that stage 4 copies them unless a
  // slice overflowed.  Few commands take 8, 4 or 2 lanes each, so that a
  // cubic's adaptive steps are tried that many halvings at a time.
  const int slice = I.cmdCount > 0 ? kStagePts / I.cmdCount : 0;
  bool staged = false;
  int myN = 0;
  auto group = [&](auto lanesPer) {
    constexpr int G = decltype(lanesPer)::value;
    const int c = tid / G, u = tid % G;
    if (c < I.cmdCount) {
      const int i = I.cmdBase + c;
      StageEmit se{sPts + c * slice, slice, I.mat, xf};
      se.writer = u == 0;
      int32_t r;
      const SceneCmd& cm = P.cmds[i];
      if ((int)cm.kind == 5)
        r = flatten_cubic_group<G>(cmd_end(P.cmds[i - 1]), v2(cm.p[0], cm.p[1]), v2(cm.p[2], cm.p[3]),
                                   v2(cm.p[4], cm.p[5]), I.errSq, se, u, tid & 63 & ~(G - 1));
      else
        r = cmd_emit(P.cmds, i, I.errSq, se);
      if (u == 0) {
        if (r != kOk) atomicMax(&sErr, r);
        P.cmdCount[i] = se.n;
        sPre[c] = se.n;
      }
    }
    __syncthreads();
    if (tid < I.cmdCount) {
      myN = sPre[tid];
      staged = myN <= slice;
    }
  };
  if (I.cmdCount <= NB / 8) {
    group(Lanes<8>{});
  } else if (I.cmdCount <= NB / 4) {
    group(Lanes<4>{});
  } else if (I.cmdCount <= NB / 2) {
    group(Lanes<2>{});
  } else if (tid < I.cmdCount) {
    const int i = I.cmdBase + tid;
    StageEmit se{sPts + tid * slice, slice, I.mat, xf};
    const int32_t r = cmd_emit(P.cmds, i, I.errSq, se);
    if (r != kOk) atomicMax(&sErr, r);
    P.cmdCount[i] = se.n;
    myN = se.n;
    staged = se.n <= slice;
  }
  __syncthreads();
  // Points before each command of the call (sPre[c], and the total in
  // sPre[cmdCount]), so that subpath sums and command offsets take two LDS
  // reads instead of a loop over commands.
  {
    int tot;
    const int pre = block_excl_scan_n<NB>(tid < I.cmdCount ? myN : 0, &tot, sh);
    if (tid < I.cmdCount) sPre[tid] = pre;
    if (tid == 0) sPre[I.cmdCount] = tot;
    __syncthreads();
  }
  // 2. points per subpath: start + pieces (+ the implicit closing point of a fill)
  for (int q0 = 0; q0 < I.polyCount; q0 += NB) {
    int q = I.polyBase + q0 + tid;
    int np = 0;
    if (q0 + tid < I.polyCount) {
      ScenePoly sp = P.polys[q];
      const int cl = sp.firstCmd - I.cmdBase;
      const int n = sPre[cl + sp.numCmds] - sPre[cl];
      if (n > 0) {
        np = n + 1;
        const SceneCmd& last = P.cmds[sp.firstCmd + sp.numCmds - 1];
        if (!I.stroke && (int)last.kind != 0 && !sp.noClose) {
          V2 d = cmd_end(last) - v2(last.sx, last.sy);
          if (d.x != 0.0f || d.y != 0.0f) np++;
        }
      }
    }
    int t;
    int off = block_excl_scan_n<NB>(np, &t, sh);
    if (q0 + tid < I.polyCount) {
      P.polyPt[q] = total + off;
      P.polyN[q] = np;
    }
    total += t;
  }
  if (tid == 0) {
    int base = atomicAdd(&P.counters[kCntPoints], total);
    if (base + total > P.ptCap) {
      atomicOr(&P.counters[kCntError], 1);
      sErr = kErrCapacity;
    }
    // strokeShapes checks the dash values once it meets a shape with points
    // (paths.nim:2029-2031)
    if (I.stroke && !I.strokeNone && I.dashBad && total > 0 && sErr == kOk) sErr = kErrDash;
    sBase = base;
  }
  __syncthreads();
  const int ptBase = sBase;
  if (I.stroke) stroke_register(P, I, it, sErr == kOk ? total : 0);
  if (sErr != kOk) {
    if (tid == 0) {
      P.geo[it].status = sErr;
      P.geo[it].segCount = 0;
      P.fills[it].status = sErr;
      P.fills[it].pathWidth = 0;
    }
    return;
  }
  float2* pts = P.pts + ptBase;
  int32_t* ptPoly = P.ptPoly + ptBase;

  // 3. start and closing points (thread per subpath)
  for (int q0 = 0; q0 < I.polyCount; q0 += NB) {
    int ql = q0 + tid;
    if (ql < I.polyCount) {
      int q = I.polyBase + ql;
      ScenePoly sp = P.polys[q];
      int np = P.polyN[q], pb = P.polyPt[q];
      int off = pb + 1;
      const int cl = sp.firstCmd - I.cmdBase;  // stage 4 derives each command's offset from sPre
      off += sPre[cl + sp.numCmds] - sPre[cl];
      if (np > 0) {
        const SceneCmd& mv = P.cmds[sp.firstCmd];
        V2 s = v2(mv.sx, mv.sy);
        V2 w = xf ? mat_apply(I.mat, s) : s;
        pts[pb] = make_float2(w.x, w.y);
        ptPoly[pb] = ql;
        if (off < pb + np) {  // implicit closing point of a fill
          pts[off] = make_float2(w.x, w.y);
          ptPoly[off] = ql;
        }
      }
    }
  }
  __syncthreads();
  // 4. emit points (thread per command)
  if (tid < I.cmdCount && myN > 0) {
    const int i = I.cmdBase + tid;
    // subpath of command i (the host stores it in pad[0] of every command)
    const int ql = P.cmds[i].pad[0], q = I.polyBase + ql;
    const int o = P.polyPt[q] + 1 + sPre[tid] - sPre[P.polys[q].firstCmd - I.cmdBase];
    if (staged) {
      const float2* src = sPts + tid * slice;
      for (int k = 0; k < myN; k++) {
        pts[o + k] = src[k];
        ptPoly[o + k] = ql;
      }
    } else {
      StoreEmit se{pts + o, ptPoly + o, ql, I.mat, xf};
      cmd_emit(P.cmds, i, I.errSq, se);
    }
  }
  __syncthreads();

  // 5. segments of a fill, thread per point: it makes at most one per point,
  // so it allocates that bound and emits in one pass
  int nseg = 0;
  if (!I.stroke) {
    if (tid == 0) {
      // segments start on a 64-segment group of their own
      int base = atomicAdd(&P.counters[kCntSegs], (total + 63) & ~63);
      if (base + total > P.segCap) {
        atomicOr(&P.counters[kCntError], 1);
        sErr = kErrCapacity;
      }
      sBase = base;
    }
    __syncthreads();
    if (sErr == kOk) {
      // four consecutive points per thread per round, their loads first
      int segOff = 0;
      Bounds bd = bounds_init();
      for (int j0 = 0; j0 < total; j0 += 4 * NB) {
        const int jb = j0 + 4 * tid;
        Seg fs[4];
        int c[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int j = jb + u;
          c[u] = 0;
          if (j < total) {
            const int q = I.polyBase + ptPoly[j];
            const int pb = P.polyPt[q], np = P.polyN[q];
            // shapesToSegments: candidate (prev point -> this point); the
            // first point pairs with the polygon's last point
            const float2 pa = j == pb ? pts[pb + np - 1] : pts[j - 1];
            const float2 pc = pts[j];
            const V2 v1 = v2(pa.x, quantize_y(pa.y)), v2_ = v2(pc.x, quantize_y(pc.y));
            if (!(j == pb && veq(v1, v2_)) && make_segment(v1, v2_, &fs[u])) c[u] = 1;
          }
        }
        int t;
        int w = segOff + block_excl_scan_n<NB>(c[0] + c[1] + c[2] + c[3], &t, sh);
#pragma unroll
        for (int u = 0; u < 4; u++) {
          if (c[u]) {
            P.segs[sBase + w] = make_float4(fs[u].at.x, fs[u].at.y, fs[u].to.x, fs[u].to.y);
            P.segW[sBase + w] = (int8_t)fs[u].w;
            bounds_add(&bd, fs[u]);
            w++;
          }
        }
        segOff += t;
      }
      nseg = segOff;
      geom_finish<NB>(P, I, it, bd, nseg, sBd);
      mark_groups(P, it, sBase, total);
    }
  }
  if (tid == 0) {
    const bool segs = !I.stroke && sErr == kOk;
    ItemGeom g = {};
    g.ptBase = ptBase;
    g.ptCount = total;
    g.segBase = segs ? sBase : 0;
    g.segCount = segs ? nseg : 0;
    g.status = sErr != kOk ? sErr : (I.stroke ? (int32_t)kOk : P.fills[it].status);
    if (sErr != kOk) {
      P.fills[it].status = sErr;
      P.fills[it].pathWidth = 0;
    }
    P.geo[it] = g;
  }
}

// ---------------------------------------------------------------------------
// planning: each call's bands, phase-A tasks and work-item chunks
// ---------------------------------------------------------------------------
// 64 calls per workgroup: wave 0 lays them out (one atomic per workgroup and
// pool: where a call's bands and tasks lie does not matter, only that they
// are consecutive), then all four waves write the band -> call and
// chunk -> call maps.
constexpr int kPlanCalls = 64;
__device__ void plan_calls(const ScenePools& P, int block) {
  __shared__ int sBand[kPlanCalls], sBands[kPlanCalls], sChunk[kPlanCalls], sChunks[kPlanCalls];
  const int lane = threadIdx.x & 63, wave = uni((int)threadIdx.x >> 6);
  const int it0 = block * kPlanCalls;
  if (wave == 0) {
    const int it = it0 + lane;
    int nb = 0, nt = 0, nc = 0;
    ItemGeom g = {};
    FillInfo f = {};
    int4 rows = make_int4(0, 0, 0, 0);
    if (it < P.nItems) {
      g = P.geo[it];
      f = P.fills[it];
      if (P.items[it].stroke && g.status == kOk && g.segCount > 0) {
        stroke_fill(P, it, g.segCount, &f);
        g.status = f.status;
        P.fills[it] = f;
      }
      g.rowStart = 0;
      g.rowCount = 0;
      g.nWin = 0;
      if (g.status == kOk && f.pathWidth > 0) {
        nb = f.nParts;
        int rs = f.startY, re = f.pathHeight;
        if (re > P.H) re = P.H;
        g.rowStart = rs;
        g.rowCount = re > rs ? re - rs : 0;
        int lo = f.mode == kMask ? 0 : (f.xlo & ~3), hi = f.mode == kMask ? P.W : f.xhi;
        g.winBase = lo;
        g.nWin = hi > lo ? (hi - lo + kWinA - 1) / kWinA : 0;
        nt = g.rowCount * g.nWin;
        nc = ((g.rowCount + kRowGroup - 1) / kRowGroup * g.nWin + 63) / 64;
        // a mask call touches every row (it clears the rows outside it)
        rows = f.mode == kMask ? make_int4(0, P.H, 0, P.W)
                               : make_int4(g.rowStart, g.rowStart + g.rowCount, f.xlo, f.xhi);
      }
      P.itemRows[it] = rows;
    }
    int tb, tt, tc;
    const int bOff = wave_excl_scan(nb, &tb), tOff = wave_excl_scan(nt, &tt), cOff = wave_excl_scan(nc, &tc);
    int bBase = 0, tBase = 0, cBase = 0;
    if (lane == 0) {
      bBase = atomicAdd(&P.counters[kCntBands], tb);
      tBase = atomicAdd(&P.counters[kCntTasks], tt);
      cBase = atomicAdd(&P.counters[kCntChunks], tc);
    }
    bBase = uni(bBase);
    tBase = uni(tBase);
    cBase = uni(cBase);
    const bool fits = bBase + tb <= P.bandCap && tBase + tt <= P.taskCap &&
                      cBase + tc <= P.taskCap / 64 + P.nItems + 1;
    if (!fits && lane == 0) atomicOr(&P.counters[kCntError], 2);
    if (it < P.nItems) {
      g.bandBase = bBase + bOff;
      g.taskBase = tBase + tOff;
      ItemGeom* const o = &P.geo[it];  // not its segments, which the band ranges read meanwhile
      o->bandBase = g.bandBase;
      o->rowStart = g.rowStart;
      o->rowCount = g.rowCount;
      o->winBase = g.winBase;
      o->nWin = g.nWin;
      o->taskBase = g.taskBase;
      o->status = g.status;
      // compact per-call record for phase B
      P.itemPaint[it] = make_int4((int)f.rgbx, f.mode, g.taskBase, g.nWin);
      P.itemSpan[it] = make_int4(g.rowStart, g.rowCount, f.xlo, f.xhi);
    }
    sBand[lane] = bBase + bOff;
    sBands[lane] = fits ? nb : 0;
    sChunk[lane] = cBase + cOff;
    sChunks[lane] = fits ? nc : 0;
  }
  __syncthreads();
  for (int c = wave; c < kPlanCalls; c += 4) {
    const int b0 = uni(sBand[c]), nb = uni(sBands[c]), c0 = uni(sChunk[c]), nc = uni(sChunks[c]);
    for (int b = lane; b < nb; b += 64) P.bandItem[b0 + b] = it0 + c;
    for (int k = lane; k < nc; k += 64) P.taskChunk[c0 + k] = make_int2(it0 + c, k);
  }
}

// Stage 7 of every call: one wave per 64-segment group finds the band range
// of each segment (partitionSegments 1201-1213), its requiresAntiAliasing bit
// and the band range of the group.
__device__ void seg_bands(const ScenePools& P, int block, int blocks) {
  const int nGroups = P.counters[kCntSegs] >> 6;
  const int wave = uni((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  for (int gi = block * 4 + wave; gi < nGroups; gi += blocks * 4) {
    const int it = uni(P.groupItem[gi]);
    const int segBase = uni(P.geo[it].segBase), segCount = uni(P.geo[it].segCount);
    FillInfo f = {};
    if (P.items[it].stroke) {
      stroke_fill(P, it, segCount, &f);
    } else {
      const FillInfo& F = P.fills[it];
      f.status = F.status;
      f.pathWidth = F.pathWidth;
      f.startY = F.startY;
      f.nParts = F.nParts;
      f.bandH = F.bandH;
    }
    const int j = gi * 64 + lane - segBase;
    int lo = 0x7fffffff, hi = -1;
    if (j < segCount && f.status == kOk && f.pathWidth > 0) {
      const float4 sg = P.segs[segBase + j];
      uint32_t l = 0, h = 0;
      if (f.nParts > 1)
        partition_range(sg.y, sg.w, (uint32_t)f.startY, (uint32_t)f.bandH, (uint32_t)f.nParts, &l, &h);
      const bool aa = seg_requires_aa(v2(sg.x, sg.y), v2(sg.z, sg.w));
      P.segBand[segBase + j] = make_int2((int)l, (int)h | (aa ? kSegAA : 0));
      lo = (int)l;
      hi = (int)h;
    }
    for (int o = 32; o > 0; o >>= 1) {
      lo = min(lo, __shfl_xor(lo, o, 64));
      hi = max(hi, __shfl_xor(hi, o, 64));
    }
    if (lane == 0) P.segChunk[gi] = make_int2(lo, hi);
  }
}

// The plan and the band ranges need the same inputs and not each other.
__global__ void __launch_bounds__(256) scene_plan_kernel(ScenePools P, int planBlocks) {
  if ((int)blockIdx.x < planBlocks)
    plan_calls(P, blockIdx.x);
  else if (!(P.counters[kCntError] & 1))  // (set by earlier kernels only)
    seg_bands(P, (int)blockIdx.x - planBlocks, (int)gridDim.x - planBlocks);
}

// Band b of its call: top / bottom rows (partitionSegments 1183-1192).
__device__ __forceinline__ void band_rows(const FillInfo& f, int k, float* top, float* bot) {
  *top = (float)(f.startY + k * f.bandH);
  *bot = (k == f.nParts - 1) ? (float)f.pathHeight : (float)(f.startY + (k + 1) * f.bandH);
}


// A grid-stride loop over items [0, n) laid out by XCD: workgroups go to
// the kXcds XCDs round robin, and XCD x takes the x-th contiguous share of
// the items, so that neighbouring items (the bands of one call, which read
// the same segments) share its L2.
constexpr int kXcds = 8;
struct XcdSpan {
  int begin, end, step;
};
__device__ __forceinline__ XcdSpan xcd_span(int n, int block, int blocks) {
  const int per = blocks / kXcds;
  if (per == 0) return XcdSpan{block, n, blocks};
  const int xcd = block % kXcds, li = block / kXcds;
  if (li >= per) return XcdSpan{0, 0, 1};  // beyond the last full round of XCDs
  return XcdSpan{(int)((int64_t)n * xcd / kXcds) + li, (int)((int64_t)n * (xcd + 1) / kXcds), per};
}

// Entry of segment s in band [top, bot]: slope-intercept form of the whole
// segment, y range clipped to the band when the segment spans it
// (partitionSegments 1236-1248).  *clipped receives the clipped segment.
__device__ __forceinline__ Entry band_entry(float4 s, float top, float bot, float4* clipped) {
  V2 at = v2(s.x, s.y), to = v2(s.z, s.w);
  Entry e = init_entry(at, to);
  if (at.y <= top && to.y >= bot) {
    V2 c = v2(0, 0);
    clip_to_line(at, to, top, &c);
    at = c;
    clip_to_line(at, to, bot, &c);
    to = c;
    e.aty = at.y;
    e.toy = to.y;
  }
  *clipped = make_float4(at.x, at.y, to.x, to.y);
  return e;
}

// The segment groups [c0, c1) of a call that may reach band k, four at a
// time so that their loads overlap: calls fn(segBand of this lane's segment
// in each of the four, its index) until fn returns false.
template <class Fn>
__device__ __forceinline__ void band_groups(const ScenePools& P, int k, int c0, int c1, int s1, Fn fn) {
  const int lane = threadIdx.x & 63;
  for (int cb = c0; cb < c1; cb += 64) {
    bool may = false;
    if (cb + lane < c1) {
      const int2 cr = P.segChunk[cb + lane];
      may = k >= cr.x && k <= cr.y;
    }
    uint64_t cm = ballot(may);
    while (cm) {
      int2 sb[4];
      int js[4];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        sb[u] = make_int2(1, 0);  // empty band range
        js[u] = 0;
        if (cm) {
          js[u] = ((cb + __builtin_ctzll(cm)) << 6) + lane;
          cm &= cm - 1;
          if (js[u] < s1) sb[u] = P.segBand[js[u]];
        }
      }
      if (!fn(sb, js)) return;
    }
  }
}

// The bands, in a tile per workgroup (tile t holds bands t,
// t + nTiles, ...: neighbours, which are of one call and about as long, go to
// different workgroups of one XCD).  One launch counts the entries of every
// band, with requiresAntiAliasing, and each tile's; the next finds its tile's
// place by summing the tiles before it (4,096 at most; an atomic per tile on
// one counter took 40 us) and writes the entries.  A wave takes a band by
// itself; when there are few bands (a page of text has a couple of hundred
// with thousands of segment groups), the four waves of a workgroup share one,
// each a quarter of its call's groups.
constexpr int kBandBlocks = kBandTilesMax;  // at most one tile per workgroup
struct BandTiles {
  bool share;  // four waves per band
  int tile, n;
};
__device__ __forceinline__ BandTiles band_tiling(int nb) {
  BandTiles t;
  t.share = nb <= kBandBlocks;
  t.tile = t.share ? 1 : (nb + kBandBlocks - 1) / kBandBlocks;
  t.n = (nb + t.tile - 1) / t.tile;
  return t;
}
// The share of groups [c0, c1) of wave w of four.
__device__ __forceinline__ void quarter(int w, int* c0, int* c1) {
  const int per = (*c1 - *c0 + 3) / 4;
  *c0 += w * per;
  *c1 = *c0 + per < *c1 ? *c0 + per : *c1;
}

__device__ void band_count(const ScenePools& P, int block, int blocks) {
  __shared__ int sSum, sCnt[4];
  const int lane = threadIdx.x & 63, wave = uni((int)threadIdx.x >> 6);
  const int nb = P.counters[kCntBands];
  const BandTiles bt = band_tiling(nb);
  const XcdSpan sp = xcd_span(bt.n, block, blocks);
  for (int t = sp.begin; t < sp.end; t += sp.step) {
    const int bn = (nb - t + bt.n - 1) / bt.n;
    if (threadIdx.x < 4) sCnt[threadIdx.x] = 0;
    if (threadIdx.x == 0) sSum = 0;
    __syncthreads();
    int sum = 0;
    for (int i = bt.share ? 0 : wave; i < bn; i += bt.share ? 1 : 4) {
      const int b = t + i * bt.n, it = uni(P.bandItem[b]);
      const ItemGeom g = P.geo[it];
      const int k = b - uni(g.bandBase), s0 = uni(g.segBase), s1 = s0 + uni(g.segCount);  // s0 is 64-aligned
      int c0 = s0 >> 6, c1 = (s1 + 63) >> 6;
      if (bt.share) quarter(wave, &c0, &c1);
      int cnt = 0;
      bool aa = false;
      band_groups(P, k, c0, c1, s1, [&](const int2* sb, const int*) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const bool in = k >= sb[u].x && k <= (sb[u].y & ~kSegAA);
          cnt += __popcll(ballot(in));
          if (ballot(in && (sb[u].y & kSegAA))) aa = true;
        }
        return true;
      });
      sum += cnt;
      if (bt.share) {
        if (lane == 0) sCnt[wave] = cnt | (aa ? 1 << 30 : 0);
      } else {
        P.parts[b] = PartInfo{0, cnt, aa ? 1 : 0, 0};  // every lane stores the same value
        if (cnt > P.gcap && lane == 0) atomicMax(&P.counters[kCntMaxBand], cnt);
      }
    }
    if (lane == 0 && sum) atomicAdd(&sSum, sum);
    __syncthreads();
    if (threadIdx.x == 0) {
      P.tileSum[t] = sSum;
      if (bt.share) {
        const int m = (1 << 30) - 1;
        P.parts[t] = PartInfo{0, sSum, ((sCnt[0] | sCnt[1] | sCnt[2] | sCnt[3]) >> 30) & 1, 0};
        P.bandQuarter[t] = make_int4(sCnt[0] & m, sCnt[1] & m, sCnt[2] & m, sCnt[3] & m);
        if (sSum > P.gcap) atomicMax(&P.counters[kCntMaxBand], sSum);
      }
    }
    __syncthreads();
  }
}

__global__ void __launch_bounds__(256) scene_band_write_kernel(ScenePools P) {
  __shared__ int sh[4];
  const int lane = threadIdx.x & 63, wave = uni((int)threadIdx.x >> 6);
  if (P.counters[kCntError] & 3) return;  // (not set by this kernel)
  const int nb = P.counters[kCntBands];
  const BandTiles bt = band_tiling(nb);
  const XcdSpan sp = xcd_span(bt.n, blockIdx.x, gridDim.x);
  for (int t = sp.begin; t < sp.end; t += sp.step) {
    const int bn = (nb - t + bt.n - 1) / bt.n;
    // entries of the tiles before this one, and of all
    int before = 0, all = 0;
    for (int i = (int)threadIdx.x; i < bt.n; i += 256) {
      const int v = P.tileSum[i];
      all += v;
      before += i < t ? v : 0;
    }
    int tot;
    block_excl_scan_n<256>(all, &tot, sh);
    int base;
    block_excl_scan_n<256>(before, &base, sh);
    if (t == 0 && threadIdx.x == 0) {
      P.counters[kCntEntries] = tot;
      if (tot > P.entryCap) atomicOr(&P.counters[kCntError], 4);
    }
    if (tot > P.entryCap) return;  // the same in every workgroup
    for (int r0 = 0; r0 < bn; r0 += 64) {  // 64 bands' counts and places at a time
      const int n64 = bn - r0 < 64 ? bn - r0 : 64;
      const PartInfo mine = lane < n64 ? P.parts[t + (r0 + lane) * bt.n] : PartInfo{0, 0, 0, 0};
      int sum64;
      const int place = base + wave_excl_scan(mine.count, &sum64);
      base += sum64;
      for (int i = bt.share ? 0 : wave; i < n64; i += bt.share ? 1 : 4) {
        const int b = t + (r0 + i) * bt.n, it = uni(P.bandItem[b]);
        const int eb = __builtin_amdgcn_readlane(place, i);
        const ItemGeom g = P.geo[it];
        FillInfo f = P.fills[it];
        const int k = b - uni(g.bandBase), s0 = uni(g.segBase), s1 = s0 + uni(g.segCount);
        f.startY = uni(f.startY);
        f.bandH = uni(f.bandH);
        f.nParts = uni(f.nParts);
        f.pathHeight = uni(f.pathHeight);
        float top, bot;
        band_rows(f, k, &top, &bot);
        int c0 = s0 >> 6, c1 = (s1 + 63) >> 6;
        const int count = __builtin_amdgcn_readlane(mine.count, i), flags = __builtin_amdgcn_readlane(mine.flags, i);
        if (!bt.share || wave == 0) P.parts[b].entryBase = eb;  // every lane stores the same value
        int pos = 0, end = count;
        if (bt.share && count != 2) {
          const int4 q = P.bandQuarter[b];
          const int q0 = uni(q.x), q1 = uni(q.y), q2 = uni(q.z);
          quarter(wave, &c0, &c1);
          pos = wave == 0 ? 0 : wave == 1 ? q0 : wave == 2 ? q0 + q1 : q0 + q1 + q2;
          end = wave == 0 ? q0 : wave == 1 ? q0 + q1 : wave == 2 ? q0 + q1 + q2 : count;
        }
        if (count != 2) {
          const uint64_t below = (1ull << lane) - 1ull;
          if (pos < end)
            band_groups(P, k, c0, c1, s1, [&](const int2* sb, const int* js) {
              bool in[4];
              float4 sg[4];
              int8_t sw[4];
#pragma unroll
              for (int u = 0; u < 4; u++) {
                in[u] = k >= sb[u].x && k <= (sb[u].y & ~kSegAA);
                sg[u] = make_float4(0, 0, 0, 0);
                sw[u] = 0;
                if (in[u]) {
                  sg[u] = P.segs[js[u]];
                  sw[u] = P.segW[js[u]];
                }
              }
#pragma unroll
              for (int u = 0; u < 4; u++) {
                const uint64_t m = ballot(in[u]);
                if (in[u]) {
                  const int p = eb + pos + __popcll(m & below);
                  float4 cl;
                  P.entries[p] = band_entry(sg[u], top, bot, &cl);
                  P.entW[p] = sw[u];
                }
                pos += __popcll(m);
              }
              return pos < end;
            });
          continue;
        }
        if (bt.share && wave != 0) continue;
        // two entries: gather both segments into every lane, decide the
        // two-spanning flag and order (1250-1262), then write
        float4 g0 = make_float4(0, 0, 0, 0), g1 = g0;
        int w0 = 0, w1 = 0, found = 0;
        band_groups(P, k, c0, c1, s1, [&](const int2* sb, const int* js) {
#pragma unroll
          for (int u = 0; u < 4; u++) {
            const bool in = k >= sb[u].x && k <= (sb[u].y & ~kSegAA);
            uint64_t m = ballot(in);
            if (!m) continue;
            float4 sg = make_float4(0, 0, 0, 0);
            int wv = 0;
            if (in) {
              sg = P.segs[js[u]];
              wv = P.segW[js[u]];
            }
            while (m != 0 && found < 2) {
              const int src = __builtin_ctzll(m);
              m &= m - 1;
              const float4 t4 = make_float4(__shfl(sg.x, src, 64), __shfl(sg.y, src, 64), __shfl(sg.z, src, 64),
                                            __shfl(sg.w, src, 64));
              const int tw = __shfl(wv, src, 64);
              if (found == 0) {
                g0 = t4;
                w0 = tw;
              } else {
                g1 = t4;
                w1 = tw;
              }
              found++;
            }
          }
          return found < 2;
        });
        float4 a, c;
        Entry first = band_entry(g0, top, bot, &a);
        Entry second = band_entry(g1, top, bot, &c);
        const V2 a0 = v2(a.x, a.y), a1 = v2(a.z, a.w), d0 = v2(c.x, c.y), d1 = v2(c.z, c.w);
        bool swap = false, two = false;
        if (!intersects_inside(a0, a1, d0, d1)) {
          if (a0.y <= top && a1.y >= bot && d0.y <= top && d1.y >= bot) {
            two = true;
            swap = midpoint_x(a0, a1) > midpoint_x(d0, d1);
          }
        }
        // every lane stores the same values (conditional copies, not ?: on the
        // two lvalues, which would keep both entries in memory)
        if (swap) {
          const Entry e = first;
          first = second;
          second = e;
        }
        P.entries[eb] = first;
        P.entries[eb + 1] = second;
        P.entW[eb] = (int8_t)(swap ? w1 : w0);
        P.entW[eb + 1] = (int8_t)(swap ? w0 : w1);
        if (two) P.parts[b].flags = flags | 2;
      }
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// row bins for phase B: a workgroup per bin lists the calls that meet its
// rows, in call order; wave w takes the w-th quarter of the calls
// ---------------------------------------------------------------------------
__device__ void fill_bin(const ScenePools& P, int bin) {
  __shared__ int sCnt[4], sBase;
  const int lane = threadIdx.x & 63, wave = uni((int)threadIdx.x >> 6);
  const int r0 = bin * kBinRows, r1 = r0 + kBinRows;
  const int per = ((P.nItems + 3) / 4 + 63) & ~63;
  const int i0 = wave * per, i1 = i0 + per < P.nItems ? i0 + per : P.nItems;
  int cnt = 0;
#pragma unroll 4
  for (int i = i0; i < i1; i += 64) {
    const int it = i + lane;
    bool in = false;
    if (it < i1) {
      const int4 r = P.itemRows[it];
      in = r.x < r1 && r.y > r0;
    }
    cnt += __popcll(ballot(in));
  }
  if (lane == 0) sCnt[wave] = cnt;
  __syncthreads();
  const int c0 = uni(sCnt[0]), c1 = uni(sCnt[1]), c2 = uni(sCnt[2]), tot = c0 + c1 + c2 + uni(sCnt[3]);
  if (threadIdx.x == 0) {
    const int base = atomicAdd(&P.counters[kCntBinEntries], tot);
    if (base + tot > P.binCap) atomicOr(&P.counters[kCntError], 32);
    P.binOff[bin] = base;
    P.binCount[bin] = tot;
    sBase = base;
  }
  __syncthreads();
  const int base = uni(sBase);
  if (base + tot > P.binCap) return;
  int pos = base + (wave == 0 ? 0 : wave == 1 ? c0 : wave == 2 ? c0 + c1 : c0 + c1 + c2);
#pragma unroll 4
  for (int i = i0; i < i1; i += 64) {
    const int it = i + lane;
    bool in = false;
    if (it < i1) {
      const int4 r = P.itemRows[it];
      in = r.x < r1 && r.y > r0;
    }
    const uint64_t m = ballot(in);
    if (in) P.binList[pos + __popcll(m & ((1ull << lane) - 1ull))] = it;
    pos += __popcll(m);
  }
}

// Both need the plan and not each other.  binBlocks is a multiple of kXcds.
__global__ void __launch_bounds__(256) scene_band_kernel(ScenePools P, int binBlocks) {
  __shared__ int sErr;
  // read once: another workgroup may set the error meanwhile
  if (threadIdx.x == 0) sErr = P.counters[kCntError] & 3;
  __syncthreads();
  if (uni(sErr)) return;
  if ((int)blockIdx.x < binBlocks) {
    if ((int)blockIdx.x < (P.H + kBinRows - 1) / kBinRows) fill_bin(P, blockIdx.x);
  } else {
    band_count(P, (int)blockIdx.x - binBlocks, (int)gridDim.x - binBlocks);
  }
}

// ---------------------------------------------------------------------------
// phase A: row programs of every (call, row, window) -> sparse runs
// ---------------------------------------------------------------------------

// Where this workgroup counts the runs it wrote: one of kUsedSlots, 64 bytes
// apart, which the composition adds up.  Thousands of waves that end together
// and add to one address wait 10 to 20 ns each.
__device__ __forceinline__ int32_t* used_slot(const ScenePools& P) {
  return P.queues + (blockIdx.x % kUsedSlots) * 16;
}

// Takes n entries of a pool counter for the whole wave (also with every lane
// in the atomic; once per chunk of runs).
__device__ __forceinline__ int queue_take(int32_t* counter, int n) {
  const int lane = threadIdx.x & 63;
  int base = atomicAdd(counter, lane == 0 ? n : 0);
  return __builtin_amdgcn_readfirstlane(__shfl(base, 0, 64));
}

// Band of row y of a banded call (partitionSegments' layout).
__device__ __forceinline__ int band_of_row(const FillInfo& F, int y) {
  const int pi = (y - F.startY) / F.bandH;
  return pi > F.nParts - 1 ? F.nParts - 1 : pi;
}
// First cost class of the heavy kernel: one later for a scene of many tasks,
// whose other rows keep the chip busy beside a row that takes one wave long
// (the heavy kernel runs more instructions per row: its benefit is latency).
// Fills, three in ten stroked, by their tasks, from class 10 and 11: 45 k 606
// and 866 us, 69 k 618 and 792, 92 k 738 and 871, 147 k 937 and 1,031, 200 k
// 1,142 and 1,135, 266 k 1,451 and 1,310; all stroked, 102 k 909 and 1,009,
// 147 k 1,145 and 1,142, 228 k 1,598 and 1,472.
constexpr int kManyTasks = 3 << 16;
__device__ __forceinline__ int heavy_class(const ScenePools& P) {
  return P.heavyClass + (P.counters[kCntTasks] > kManyTasks ? 1 : 0);
}
// Cost class of band pi of a call: the bit length of its entry count (below
// the heavy classes when the band needs no anti-aliasing).
__device__ __forceinline__ int band_class(const ScenePools& P, const ItemGeom& g, int pi, int heavyClass) {
  const PartInfo p = P.parts[g.bandBase + pi];
  const int c = p.count <= 0 ? 0 : 32 - __clz(p.count);
  return (p.flags & 1) || c < heavyClass ? c : heavyClass - 1;
}

// The work items of one (call, row group, window) unit, a lane per unit: fn(r,
// class, grouped) is called by every lane alike, with a negative class for
// lanes without an item at row r of their group.
template <class Fn>
__device__ __forceinline__ void unit_items(const ScenePools& P, int unit, const ItemGeom& g, const FillInfo& F,
                                           int heavyClass, Fn fn) {
  const bool on = unit < (g.rowCount + kRowGroup - 1) / kRowGroup * g.nWin;
  const int rg = unit / g.nWin * kRowGroup, win = unit % g.nWin;
  const int rows = !on ? 0 : (rg + kRowGroup < g.rowCount ? kRowGroup : g.rowCount - rg);
  const bool banded = F.nParts > 0 && F.bandH > 0;
  // classes of its rows' bands (every row of a call lies in [startY, pathHeight))
  int cls[kRowGroup], chunk = 0;
#pragma unroll
  for (int q = 0; q < kRowGroup; q++) {
    cls[q] = 0;
    if (banded && q < rows) {
      cls[q] = band_class(P, g, band_of_row(F, g.rowStart + rg + q), heavyClass);
      chunk = cls[q] > chunk ? cls[q] : chunk;
    }
  }
  const bool grouped = chunk <= kGroupMaxClass;
  if (ballot(on && grouped)) fn(rg, on && grouped ? chunk : -1, true);
  if (ballot(on && !grouped)) {
#pragma unroll
    for (int q = 0; q < kRowGroup; q++) {
      // a heavy row's item takes kHeavyWins windows at a time
      const bool own = on && !grouped && q < rows && (cls[q] < heavyClass || win % kHeavyWins == 0);
      fn(rg + q, own ? cls[q] : -1, false);
    }
  }
}

// Counts the work items per cost class (kPlace = false), or places them in
// the order, largest class first (kPlace = true): a wave per 64 units, each
// workgroup a contiguous share of them.  Placing counts the share again and
// reserves its range of every class with one atomic before it deals the
// places out in LDS.
template <bool kPlace>
__global__ void __launch_bounds__(256) scene_task_kernel(ScenePools P) {
  __shared__ int32_t hist[kCostClasses], start[kCostClasses];
  const int lane = threadIdx.x & 63, wave = uni((int)threadIdx.x >> 6);
  if (P.counters[kCntError]) return;
  const int heavyClass = heavy_class(P);
  if (threadIdx.x < kCostClasses) hist[threadIdx.x] = 0;
  __syncthreads();
  const int nChunks = P.counters[kCntChunks];
  const int per = (nChunks + (int)gridDim.x - 1) / (int)gridDim.x;
  const int k0 = (int)blockIdx.x * per, k1 = k0 + per < nChunks ? k0 + per : nChunks;
  for (int k = k0 + wave; k < k1; k += 4) {
    const int2 ch = P.taskChunk[k];
    const int it = uni(ch.x);
    unit_items(P, uni(ch.y) * 64 + lane, P.geo[it], P.fills[it], heavyClass, [&](int, int c, bool) {
      if (c >= 0) atomicAdd(&hist[c], 1);
    });
  }
  __syncthreads();
  if (!kPlace) {
    if (threadIdx.x < kCostClasses && hist[threadIdx.x])
      atomicAdd(&P.counters[kCntClassHist + threadIdx.x], hist[threadIdx.x]);
    return;
  }
  if (wave == 0) {  // lane l: class kCostClasses - 1 - l
    const int c = kCostClasses - 1 - lane;
    const int n = lane < kCostClasses ? P.counters[kCntClassHist + c] : 0;
    int tot;
    const int off = wave_excl_scan(n, &tot);
    if (lane < kCostClasses) {
      start[c] = off + (hist[c] ? atomicAdd(&P.counters[kCntClassCursor + c], hist[c]) : 0);
      if (blockIdx.x == 0 && c == heavyClass - 1) P.counters[kCntHeavy] = off;
      if (blockIdx.x == 0 && c == 0) P.counters[kCntGroups] = tot;
    }
  }
  __syncthreads();
  for (int k = k0 + wave; k < k1; k += 4) {
    const int2 ch = P.taskChunk[k];
    const int it = uni(ch.x);
    const ItemGeom g = P.geo[it];
    const int unit = uni(ch.y) * 64 + lane, first = g.taskBase + unit % g.nWin;
    unit_items(P, unit, g, P.fills[it], heavyClass, [&](int r, int c, bool grouped) {
      if (c >= 0)
        P.taskOrder[atomicAdd(&start[c], 1)] =
            make_int2(first + r * g.nWin, grouped ? (int32_t)((uint32_t)it | 0x80000000u) : it);
    });
  }
}

// A wave's place in the run pool: it appends its runs to chunks it takes one
// at a time (one atomic per chunk, not per task).
struct RunCursor {
  int at = 0, end = 0, used = 0;
};

// Writes a window's codes D[0..wlen] as runs -- the nonzero deltas and, for
// ops rows, the area factors of the pixels whose code is an area code -- in
// one pass, and clears D.  The wave's run chunk is first made to hold the
// most the row can write (wlen + 1 deltas, and wlen area factors on ops
// rows).  D has kWinA + 4 entries and is zero beyond wlen, so a lane with
// i0 <= wlen moves its 4 entries as one 16-byte access.  Returns the number
// of runs and their place in *off.
__device__ __forceinline__ int emit_runs(const ScenePools& P, int32_t* D, const uint32_t* AX, int wx0, int wlen,
                                         bool ops, RunCursor* rc, int* off) {
  const int lane = threadIdx.x & 63;
  wave_sync();
  const int most = ops ? 2 * wlen + 1 : wlen + 1;
  if (rc->at + most > rc->end) {
    rc->at = queue_take(&P.counters[kCntRuns], kRunChunk);
    rc->end = rc->at + kRunChunk;
  }
  *off = rc->at;
  if (rc->end > P.runCap) {
    atomicOr(&P.counters[kCntError], 16);
    for (int i = lane; i <= wlen; i += 64) D[i] = 0;
    wave_sync();
    return 0;
  }
  int carry = 0, written = 0;
  for (int base = 0; base <= wlen; base += 4 * kWave) {
    const int i0 = base + 4 * lane;
    int4 dv = make_int4(0, 0, 0, 0);
    if (i0 <= wlen) dv = *(const int4*)(D + i0);
    const int32_t d[4] = {dv.x, dv.y, dv.z, dv.w};
    bool area[4] = {false, false, false, false};
    if (ops) {
      const int32_t c0 = d[0], c1 = c0 + d[1], c2 = c1 + d[2], c3 = c2 + d[3];
      int32_t tot;
      const int32_t ofs = carry + wave_excl_scan(c3, &tot);
      carry += tot;
      const int32_t code[4] = {ofs + c0, ofs + c1, ofs + c2, ofs + c3};
#pragma unroll
      for (int q = 0; q < 4; q++) area[q] = i0 + q < wlen && code[q] >= kArea && code[q] < kClear;
    }
    int n = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) n += (d[q] != 0 ? 1 : 0) + (area[q] ? 1 : 0);
    int ntot;
    const int p = wave_excl_scan(n, &ntot);
    if (i0 <= wlen) {
      int2* out = P.runs + *off + written + p;
      int w = 0;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int x = wx0 + i0 + q;
        if (d[q] != 0) out[w++] = make_int2(x, d[q]);
        if (area[q]) out[w++] = make_int2(x | kRunArea, (int32_t)AX[i0 + q]);
      }
      *(int4*)(D + i0) = make_int4(0, 0, 0, 0);
    }
    written += ntot;
  }
  rc->at += written;
  rc->used += written;
  wave_sync();
  return written;
}

// ---------------------------------------------------------------------------
// heavy rows: one workgroup per (call, row, kHeavyWins windows)
// ---------------------------------------------------------------------------
// A row of a band of hundreds of entries (a line of text, a stroke with round
// joins) is a long serial chain for one wave, and each of its windows would
// scan the band and sort every hit of the row again.  Here the waves of a
// workgroup share the row: they scan its band once for kHeavyWins windows,
// keep the places of the entries that can meet those windows in LDS, deal the hits of all
// five sample lines into buckets of 4 to 64 pixels, and each wave sorts and
// walks whole buckets.
//
// Walking a bucket [A, B) by itself gives the pixels of pixie's walk over the
// whole line (paths.nim:1298-1330): skipped pairs and equal-x groups share
// one x, so they lie in one bucket; a span that crosses a bucket border
// covers the pixels on both sides as the two spans cut at the border do (the
// border is a whole pixel); before the bucket's first hit only the winding
// count matters, which is the sum over the hits left of A; and a span open at
// B ends at some later hit whenever the windings of the whole line sum to 0
// (the count then returns to 0 at a hit that is not skipped).  A row with a
// line whose windings do not sum to 0 (a sample line through a vertex, where
// float32 leaves no room between them) or with more hits than the key space
// is left to the rows kernel, as is a trapezoid candidate.
//
// An entry's hit position is monotone in y (every float operation of it is),
// so the positions on the first and the last sample line tell whether it can
// meet the windows at all; entries left of them only add to the counts.
//
// Keys are 32 bits: x inside the bucket in 24.8 (14 bits), the entry's place
// in the band (17 bits: pixie's stable order), the winding's sign.
//
// Measured (kernel trace): a 4096-px page of 33,000 glyphs, rows kernel alone
// 2,888 us, heavy rows 139 us + rows kernel 48 us; 100 paths on 1,023 x 767,
// 647 us and 45 us + 140 us.  An item takes 70 thousand cycles when the chip
// is not full (scan 16, deal 14, buckets 24, runs 9), bound by the latency of
// the loads and of the short dependent chains between its barriers.
constexpr int kHeavyThreads = kHeavyWavesPerGroup * 64;
constexpr int kHeavyPx = kHeavyWins * kWinA;
constexpr int kBucketKeyBits = 18;  // order and winding below a bucket's positions
constexpr int kHeavyBuckets = 64;  // most buckets of a line (a wave scans them)
constexpr int kHeavyKeys = 4096;   // hits of the lines dealt together
constexpr int kHeavySel = 1280;    // entries kept
constexpr int kHeavyMaxBand = 65535;  // a bucket's hit count is 16 bits
constexpr int kHeavyMaxWidth = 1 << 22;  // 24.8 positions of a row item stay below 2^31

// What the workgroup needs to know of a work item.
struct HeavyItem {
  int32_t first, it;   // task of its first window (-1 ends the kernel), call
  int32_t y, gx0, nw;  // row, first pixel, windows
  PartInfo part;       // the row's band
  int32_t mode, rule, xhi, covLo, covHi;
};

// Wave 0 reads the records of the next item while the workgroup is busy with
// this one: each step's loads (order -> call -> band) are issued a
// phase before the next step needs them.  The items go round the workgroups
// in their order, longest first; a shared queue would cost each item the
// round trip of an atomic (8 to 14 thousand cycles of 70).
struct HeavyFetch {
  int q;  // place of the next item
  int first, it;
  ItemGeom g;
  FillInfo F;
  PartInfo part;
  __device__ __forceinline__ void step_order(const ScenePools& P, int n) {
    const int2 o = q < n ? P.taskOrder[q] : make_int2(-1, 0);
    first = o.x;
    it = o.y;  // never marked as grouped
  }
  __device__ __forceinline__ void step_call(const ScenePools& P) {
    g = P.geo[it];
    F = P.fills[it];
  }
  __device__ __forceinline__ void step_band(const ScenePools& P, HeavyItem* h) {
    h->first = first;  // every lane stores the same values
    h->it = it;
    if (first < 0) return;
    const int local = first - g.taskBase, win0 = local % g.nWin, y = g.rowStart + local / g.nWin;
    part = P.parts[g.bandBase + band_of_row(F, y)];
    h->y = y;
    h->gx0 = g.winBase + win0 * kWinA;
    h->nw = g.nWin - win0 < kHeavyWins ? g.nWin - win0 : kHeavyWins;
    h->mode = F.mode;
    h->rule = F.rule;
    h->xhi = F.mode == kMask ? P.W : F.xhi;
    h->covLo = F.startX;
    h->covHi = F.startX + F.pathWidth;
  }
};

__global__ void __launch_bounds__(kHeavyThreads, 5) scene_heavy_kernel(ScenePools P) {
  __shared__ __align__(16) int32_t D[kHeavyWins][kWinA + 4];
  __shared__ uint32_t sel[kHeavySel];  // kept entries: place in the band << 1 | winding is 1
  __shared__ uint32_t keys[kHeavyKeys];
  // per line and bucket: hits | windings << 16, then the place of the
  // bucket's next key in its line; and the winding count left of the bucket
  __shared__ uint32_t bkt[5][kHeavyBuckets];
  __shared__ int32_t left0[5][kHeavyBuckets];
  // per line: the winding sums of the hits left of the windows and of all
  // hits, and its hits in the buckets
  __shared__ int32_t sLeft[5], sTotal[5], sHits[5];
  __shared__ int32_t sNe, sNotSpan, sSel;
  __shared__ HeavyItem sItems[2];  // this item's record and the next one's
  const int tid = threadIdx.x, lane = tid & 63, wave = uni(tid >> 6);
  for (int i = tid; i < kHeavyWins * (kWinA + 4); i += kHeavyThreads) ((int32_t*)D)[i] = 0;
  // read once, so that every wave takes the same way when another workgroup
  // sets the error meanwhile
  if (tid == 0) sNe = P.counters[kCntError];
  __syncthreads();
  if (uni(sNe)) return;
  const int nHeavy = P.counters[kCntHeavy];
  RunCursor rc;
  HeavyFetch nx;
  if (wave == 0) {
    nx.q = blockIdx.x;
    nx.step_order(P, nHeavy);
    nx.step_call(P);
    nx.step_band(P, &sItems[0]);
  }
  for (int cur = 0;; cur ^= 1) {
    HeavyItem& sItem = sItems[cur];
    HeavyItem* const next = &sItems[cur ^ 1];
    __syncthreads();  // the item before is done with the shared words
    if (wave == 0) {
      sItem.part = nx.part;
      if (lane == 0) sNe = sNotSpan = sSel = 0;
      if (lane < 5) sLeft[lane] = sTotal[lane] = 0;
      nx.q += gridDim.x;
      nx.step_order(P, nHeavy);
    }
    for (int i = tid; i < 5 * kHeavyBuckets; i += kHeavyThreads) (&bkt[0][0])[i] = 0;
    __syncthreads();
    const int first = uni(sItem.first);
    if (first < 0) break;
    const int y = uni(sItem.y), nw = uni(sItem.nw), count = uni(sItem.part.count);
    const int32_t mode = uni(sItem.mode), rule = uni(sItem.rule);
    const bool mask = mode == kMask;
    const Entry* E = P.entries + uni(sItem.part.entryBase);
    const int8_t* EW = P.entW + uni(sItem.part.entryBase);
    const float scanTop = (float)y, scanBottom = (float)(y + 1);
    const int32_t gx0 = uni(sItem.gx0), cx1 = uni(sItem.xhi);
    const int32_t covLo = uni(sItem.covLo), covHi = uni(sItem.covHi);
    const int32_t A = gx0 * 256, A1 = A > 1 ? A : 1, B = (gx0 + nw * kWinA) * 256;
    const float Wf = (float)P.W;
    float yl[5];
    {
      const float offset = 1.0f / 5.0f;
      float v = (float)y + (offset / 2.0f + 0.00031415926535897936f) - offset;
#pragma unroll
      for (int m = 0; m < 5; m++) yl[m] = v += offset;
    }
    // Buckets of a width that puts 24 to 48 hits into each, at most
    // kHeavyBuckets of them: a row selects about half of its band's entries,
    // half of those meet a sample line, and the windows hold their share of
    // the path's width.
    const int extent = covHi < gx0 + nw * kWinA ? covHi - gx0 : nw * kWinA;
    const int est = covHi - covLo > extent ? (int)((int64_t)count * extent / (covHi - covLo)) : count;
    int sh = 6;
    while (sh > 2 && (extent >> (sh - 1)) < kHeavyBuckets && (est << sh) > 192 * extent) sh--;
    const int px = 1 << sh;
    int nb = (extent + px - 1) >> sh;
    nb = nb < 1 ? 1 : (nb < kHeavyBuckets ? nb : kHeavyBuckets);
    // hits at Bk or beyond lie right of the coverage range: they cover no
    // pixel, and what they end covers the range to its border either way
    const int32_t Bk = A + nb * (px << 8) < B ? A + nb * (px << 8) : B;
    bool leave = !(uni(sItem.part.flags) & 1) || count > P.gcap || count > kHeavyMaxBand || P.W > kHeavyMaxWidth;
    // Scan of the band: the row's selection (paths.nim:1673-1689) with its
    // size and whether every entry spans the row, each line's winding sums and
    // bucket counts, and the list of the entries that can meet the windows.
    // kLoads entries per thread are in flight at a time.
    constexpr int kLoads = 4;
    int ne = 0;
    if (!leave) {
      bool notSpan = false;
      int32_t left[5] = {0, 0, 0, 0, 0}, total[5] = {0, 0, 0, 0, 0};
      auto scan = [&](const Entry& e, int32_t w, bool in) -> bool {
        if (!in || e.toy <= scanTop || e.aty >= scanBottom) return false;
        ne++;
        notSpan |= e.aty > scanTop || e.toy < scanBottom;
        const int32_t a0 = hit_at(e, yl[0], Wf), a4 = hit_at(e, yl[4], Wf);
        const bool isLeft = a0 < A && a4 < A, isRight = a0 >= B && a4 >= B;
#pragma unroll
        for (int m = 0; m < 5; m++) {
          if (!(e.aty <= yl[m] && e.toy >= yl[m])) continue;
          total[m] += w;
          if (isLeft) left[m] += w;
          if (isLeft || isRight) continue;
          const int32_t at = m == 0 ? a0 : m == 4 ? a4 : hit_at(e, yl[m], Wf);
          if (at < A1) left[m] += w;  // (a hit at x = 0 only counts)
          else if (at < Bk) atomicAdd(&bkt[m][(at - A) >> (sh + 8)], 1u + ((uint32_t)w << 16));
        }
        return !isLeft && !isRight;
      };
      for (int i0 = 0; i0 < count; i0 += kLoads * kHeavyThreads) {
        Entry e[kLoads];
        int32_t w[kLoads];
#pragma unroll
        for (int u = 0; u < kLoads; u++) {
          const int i = i0 + u * kHeavyThreads + tid;
          e[u] = Entry{0.0f, 0.0f, 0.0f, 0.0f};
          w[u] = 0;
          if (i < count) {
            e[u] = E[i];
            w[u] = EW[i];
          }
        }
#pragma unroll
        for (int u = 0; u < kLoads; u++) {
          const int i = i0 + u * kHeavyThreads + tid;
          if (scan(e[u], w[u], i < count)) {
            const int at = atomicAdd(&sSel, 1);
            if (at < kHeavySel) sel[at] = ((uint32_t)i << 1) | (w[u] > 0 ? 1u : 0u);
          }
        }
      }
      ne = wave_incl_sum(ne);
      if (lane == 63 && ne) atomicAdd(&sNe, ne);
      if (ballot(notSpan) && lane == 0) sNotSpan = 1;
#pragma unroll
      for (int m = 0; m < 5; m++) {
        left[m] = wave_incl_sum(left[m]);
        total[m] = wave_incl_sum(total[m]);
        if (lane == 63 && left[m]) atomicAdd(&sLeft[m], left[m]);
        if (lane == 63 && total[m]) atomicAdd(&sTotal[m], total[m]);
      }
    }
    if (wave == 0) nx.step_call(P);
    __syncthreads();
    ne = uni(sNe);
    leave = leave || (ne > 0 && !uni(sNotSpan) && (ne % 2) == 0) ||
            (uni(sTotal[0]) | uni(sTotal[1]) | uni(sTotal[2]) | uni(sTotal[3]) | uni(sTotal[4])) != 0;
    if (!leave) {
      if (mask && wave < nw && lane == 0) {
        // a mask row is cleared but for its coverage range
        const int32_t wx0 = gx0 + wave * kWinA, wx1 = wx0 + kWinA < cx1 ? wx0 + kWinA : cx1;
        const int32_t lo = covLo > wx0 ? covLo : wx0, hi = covHi < wx1 ? covHi : wx1;
        atomicAdd(&D[wave][0], kClear);
        atomicAdd(&D[wave][wx1 - wx0], -kClear);
        if (ne > 0 && lo < hi) {
          atomicAdd(&D[wave][lo - wx0], -kClear);
          atomicAdd(&D[wave][hi - wx0], kClear);
        }
      }
      // places of the buckets in their line, and the counts left of them
      for (int m = wave; m < 5; m += kHeavyWavesPerGroup) {
        const uint32_t v = bkt[m][lane];
        int nHit, wAll;
        const int at = wave_excl_scan((int)(v & 0xffffu), &nHit);
        const int cw = uni(sLeft[m]) + wave_excl_scan((int32_t)v >> 16, &wAll);
        bkt[m][lane] = (uint32_t)at;
        left0[m][lane] = cw;
        if (lane == 0) sHits[m] = nHit;
      }
      // the listed entries, or the band's when they do not fit the list
      const int nSel = uni(sSel);
      const bool kept = nSel <= kHeavySel;
      const int nList = kept ? nSel : count;
      for (int l0 = 0; ne > 0 && l0 < 5;) {
        __syncthreads();
        // as many lines at a time as the key space holds
        int base[5], nKeys = 0, l1 = l0;
#pragma unroll
        for (int m = 0; m < 5; m++) {
          base[m] = nKeys;
          const int h = uni(sHits[m]);
          if (m == l1 && nKeys + h <= kHeavyKeys) {
            nKeys += h;
            l1++;
          }
        }
        if (l1 == l0) {  // a line alone exceeds it (the same in every wave)
          leave = true;
          break;
        }
        auto deal = [&](const Entry& e, uint32_t k) {
          if (e.toy <= scanTop || e.aty >= scanBottom) return;
#pragma unroll
          for (int m = 0; m < 5; m++) {
            if (m < l0 || m >= l1 || !(e.aty <= yl[m] && e.toy >= yl[m])) continue;
            const int32_t at = hit_at(e, yl[m], Wf);
            if (at < A1 || at >= Bk) continue;
            const uint32_t rel = (uint32_t)(at - A);
            keys[base[m] + atomicAdd(&bkt[m][rel >> (sh + 8)], 1u)] = ((rel & ((1u << (sh + 8)) - 1u)) << 18) | k;
          }
        };
#pragma unroll 2
        for (int i = tid; i < nList; i += kHeavyThreads) {
          const uint32_t k = kept ? sel[i] : ((uint32_t)i << 1) | (EW[i] > 0 ? 1u : 0u);
          deal(E[k >> 1], k);
        }
        if (wave == 0 && l0 == 0) nx.step_band(P, next);
        __syncthreads();
        // a bucket's place now points past its keys, at the next one's.  The
        // buckets go round the waves: a shared counter read by one lane would
        // put that lane on a path of its own from here to the next round.
        for (int j = wave; j < (l1 - l0) * nb; j += kHeavyWavesPerGroup) {
          const int m = l0 + j / nb, b = j % nb;
          const int o1 = uni((int)bkt[m][b]), o0 = b > 0 ? uni((int)bkt[m][b - 1]) : 0;
          const int32_t cb = uni(left0[m][b]);
          if (o1 == o0 && !should_fill(rule, cb)) continue;
          const int32_t bx0 = gx0 + b * px;
          const int win = (b * px) / kWinA;
          const int32_t wx0 = gx0 + win * kWinA, wx1 = wx0 + kWinA < cx1 ? wx0 + kWinA : cx1;
          const int32_t lo = (bx0 > covLo ? bx0 : covLo) - bx0;
          int32_t hi = bx0 + px < covHi ? bx0 + px : covHi;
          hi = (hi < wx1 ? hi : wx1) - bx0;
          if (lo >= hi) continue;
          const int kb = m == 0 ? base[0] : m == 1 ? base[1] : m == 2 ? base[2] : m == 3 ? base[3] : base[4];
          int32_t* const Db = D[win] + (bx0 - wx0);
          Walk32 c;
          c.count = cb;
          walk32_staged<kBucketKeyBits>(keys + kb + o0, o1 - o0, rule, Db, lo, hi, c);
          if (lane == 0) walk32_borders(should_fill(rule, cb), should_fill(rule, c.count), Db, lo, hi);
        }
        l0 = l1;
        __syncthreads();
      }
      __syncthreads();
    }
    if (leave) {  // to the rows kernel, window by window
      if (wave == 0) nx.step_band(P, next);
      for (int i = tid; i < kHeavyWins * (kWinA + 4); i += kHeavyThreads) ((int32_t*)D)[i] = 0;
      if (tid < nw)
        P.taskOrder[P.taskCap + atomicAdd(&P.counters[kCntLeft], 1)] = make_int2(first + tid, uni(sItem.it));
      continue;
    }
    if (ne == 0 && wave == 0) nx.step_band(P, next);
    if (wave < nw) {
      const int32_t wx0 = gx0 + wave * kWinA, wx1 = wx0 + kWinA < cx1 ? wx0 + kWinA : cx1;
      RowRuns rr;
      rr.kind = ne > 0 ? kRowCoverage : kRowOps;
      rr.pad = 0;
      rr.off = 0;
      rr.n = emit_runs(P, D[wave], nullptr, wx0, wx1 - wx0, false, &rc, &rr.off);
      P.tasks[first + wave] = rr;  // every lane stores the same value
    }
  }
  if (lane == 0 && rc.used) atomicAdd(used_slot(P), rc.used);
}

__global__ void __launch_bounds__(64, 4) scene_rows_kernel(ScenePools P) {
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x;
  const size_t fixedBytes = row_lds_fixed_bytes(kWinA);
  RowLds Ll = row_lds_carve(smem, smem + fixedBytes, P.ldsCap, kWinA);
  RowLds Lg = row_lds_carve(smem, P.gscratch + (size_t)blockIdx.x * row_cap_bytes(P.gcap), P.gcap, kWinA);
  for (int i = lane; i < kWinA + 4; i += 64) Ll.D[i] = 0;
  __syncthreads();
  if (P.counters[kCntError]) return;
  // the rows the heavy kernel left, then the work items after its own
  const int nHeavy = P.counters[kCntHeavy], nLeft = P.counters[kCntLeft];
  const int nItems = nLeft + P.counters[kCntGroups] - nHeavy;
  RunCursor rc;
  for (;;) {
    const int q = queue_next<kRowGranule>(P.queues + kQueues * kQueueStride, nItems);
    if (q >= nItems) break;
    // Work item, call and the call's records are the same in every lane:
    // read them into scalar registers.
    const int2 item = P.taskOrder[q < nLeft ? P.taskCap + q : nHeavy + q - nLeft];
    const int first = uni(item.x), itw = uni(item.y);
    const int it = itw & 0x7fffffff;
    ItemGeom g = P.geo[it];
    g.rowStart = uni(g.rowStart);
    g.nWin = uni(g.nWin);
    g.winBase = uni(g.winBase);
    g.taskBase = uni(g.taskBase);
    g.bandBase = uni(g.bandBase);
    g.rowCount = uni(g.rowCount);
    FillInfo Fu = P.fills[it];
    Fu.startX = uni(Fu.startX);
    Fu.startY = uni(Fu.startY);
    Fu.pathWidth = uni(Fu.pathWidth);
    Fu.pathHeight = uni(Fu.pathHeight);
    Fu.nParts = uni(Fu.nParts);
    Fu.bandH = uni(Fu.bandH);
    Fu.mode = uni(Fu.mode);
    Fu.rule = uni(Fu.rule);
    Fu.xlo = uni(Fu.xlo);
    Fu.xhi = uni(Fu.xhi);
    Fu.canvasW = uni(Fu.canvasW);
    const FillInfo& F = Fu;
    const int local = first - g.taskBase;
    const int win = local % g.nWin;
    const int r0 = local / g.nWin;
    const int r1 = itw >= 0 ? r0 + 1 : (r0 + kRowGroup < g.rowCount ? r0 + kRowGroup : g.rowCount);
    const bool mask = F.mode == kMask;
    for (int r = r0; r < r1; r++) {
      const int y = g.rowStart + r;
      const int task = g.taskBase + r * g.nWin + win;
      RowCtx C;
      C.F = &Fu;
      C.parts = P.parts + g.bandBase;
      C.E = P.entries;
      C.EW = P.entW;
      C.y = y;
      C.cx0 = mask ? 0 : F.xlo;
      C.cx1 = mask ? P.W : F.xhi;
      C.wx0 = g.winBase + win * kWinA;
      C.wx1 = C.wx0 + kWinA < C.cx1 ? C.wx0 + kWinA : C.cx1;
      // band of this row decides where the row scratch lives
      int pi = (y - F.startY) / F.bandH;
      if (pi > F.nParts - 1) pi = F.nParts - 1;
      const int cnt = uni(C.parts[pi].count);
      // a large band's row whose selection fits LDS still runs there
      bool inLds = cnt <= P.ldsCap;
      if (!inLds && cnt <= P.gcap) inLds = row_selection_count(C) <= P.ldsCap;
      RowLds& L = inLds ? Ll : Lg;
      int32_t kind = (inLds || cnt <= P.gcap) ? row_program(C, L) : -1;
      RowRuns rr;
      rr.off = 0;
      rr.n = 0;
      rr.kind = kind;
      rr.pad = 0;
      if (kind < 0) {
        atomicOr(&P.counters[kCntError], 8);
      } else if (kind != kRowNone) {
        const int wlen = C.wx1 - C.wx0;
        rr.n = emit_runs(P, Ll.D, L.AX, C.wx0, wlen, kind == kRowOps, &rc, &rr.off);
      }
      P.tasks[task] = rr;  // every lane stores the same value
    }
  }
  if (threadIdx.x == 0 && rc.used) atomicAdd(used_slot(P), rc.used);
}

// ---------------------------------------------------------------------------
// phase B: canvas row windows in registers, calls applied in order
// ---------------------------------------------------------------------------
// The canvas window lives in LDS (512 px) while the calls are applied, so
// that one copy of the per-pixel blend code serves every pixel: the kernel
// stays small enough for the instruction cache.  Bound by the instructions of
// a call's turn: with its plan made lane by lane beforehand, Normal without
// branches and narrow calls without the queue of changed pixels, 8,192 glyphs
// on 8,192 x 8,192 go from 450 to 395 us (279 with one addition per item
// taken), 4,096 x 4,096 with 2,000 paths from 388 to 356 (334), a document of
// 900 elements from 85 to 62 (60).
constexpr uint32_t kPlanCarry = 1u << 29, kPlanPlain = 1u << 30;
template <bool kA8>
__global__ void __launch_bounds__(64) scene_compose_kernel(ScenePools P, void* canvas,
                                                          unsigned long long* touchedOut,
                                                          int32_t* errOut) {
  __shared__ __align__(16) int32_t D[kWinB + 4];
  __shared__ uint32_t AX[kWinB];
  __shared__ uint32_t WIN[kWinB];
  __shared__ int32_t Q[2 * kWave];  // pixels queued for the blend
  const int lane = threadIdx.x;
  for (int i = lane; i < kWinB + 4; i += 64) D[i] = 0;
  const int W = P.W, H = P.H;
  const int winsPerRow = (W + kWinB - 1) / kWinB;
  const int nUnits = H * winsPerRow;
  const bool vec = ((W & 3) == 0);
  uint32_t ntouch = 0;
  if (blockIdx.x == 0) {  // the runs written, for the host
    const int32_t used = wave_incl_sum(P.queues[lane * 16]);
    if (lane == kWave - 1) P.counters[kCntRunsUsed] = used;
  }
  if (const int32_t err = P.counters[kCntError]) {
    // an earlier stage ran out of a pool: the canvas stays untouched and the
    // error reaches the host through the lane's error word
    if (blockIdx.x == 0 && lane == 0) atomicOr(errOut, err);
    return;
  }
  for (;;) {
    const int unit = queue_next<kComposeGranule>(P.queues + 2 * kQueues * kQueueStride, nUnits);
    if (unit >= nUnits) break;
    const int y = unit / winsPerRow;
    const int b0 = (unit % winsPerRow) * kWinB;
    const int b1 = b0 + kWinB < W ? b0 + kWinB : W;
    bool loaded = false, dirty = false;
    const int bin = y / kBinRows;
    const int l0 = P.binOff[bin], l1 = l0 + P.binCount[bin];
    for (int i0 = l0; i0 < l1; i0 += 64) {
      const int li = i0 + lane;
      bool cov = false;
      int4 paint = make_int4(0, 0, 0, 0), span = paint;
      if (li < l1) {
        const int it = P.binList[li];
        const int4 r = P.itemRows[it];
        cov = y >= r.x && y < r.y && r.w > b0 && r.z < b1;
        if (cov) {  // each lane fetches its call's record: the loads overlap
          paint = P.itemPaint[it];
          span = P.itemSpan[it];
        }
      }
      // Each covering lane also fetches its call's first phase-A window
      // record for this row and window (pre.w = that window, -1 if none) and
      // works out how the call is applied, so that a call's turn begins with
      // two lane reads.  A plain call has all its runs for this row and
      // window in one record of at most 64; one without any is left out.
      int4 pre = make_int4(0, 0, 0, -1);
      uint32_t plan = 0;
      if (cov) {
        const bool mask = paint.y == kMask;
        if (!mask || (y >= span.x && y < span.x + span.y)) {
          const int winBase = mask ? 0 : (span.z & ~3);
          const int d = b0 - kWinA - winBase;  // windows ending before b0 are skipped
          const int w = d > 0 ? (d + kWinA - 1) / kWinA : 0;
          if (w < paint.w && winBase + w * kWinA < b1) {
            const RowRuns rr = P.tasks[paint.z + (y - span.x) * paint.w + w];
            pre = make_int4(rr.off, rr.n, rr.kind, w);
            if ((w + 1 >= paint.w || winBase + (w + 1) * kWinA >= b1) && rr.n <= 64) {
              const int lo = mask ? 0 : (span.z > b0 ? span.z - b0 : 0);
              const int hi = mask ? b1 - b0 : (span.w < b1 ? span.w : b1) - b0;
              plan = (uint32_t)lo | (uint32_t)hi << 11 | (uint32_t)paint.y << 22 | (uint32_t)rr.kind << 27 |
                     (winBase + w * kWinA < b0 ? kPlanCarry : 0u) | kPlanPlain;
              cov = rr.kind != kRowNone;
            }
          } else {
            cov = false;
          }
        }
      }
      uint64_t m = __ballot(cov);
      // a call's first 64 runs are fetched while the call before it is applied
      auto first_runs = [&](uint64_t left) {
        int2 r = make_int2(kRunXMask, 0);  // beyond every window
        if (left) {
          const int s = __builtin_ctzll(left);
          const int off = __builtin_amdgcn_readlane(pre.x, s), n = __builtin_amdgcn_readlane(pre.y, s);
          if (lane < n) r = P.runs[off + lane];
        }
        return r;
      };
      int carry = 0;  // this lane's share of the deltas before b0
      auto scatter = [&](int2 r) {
        const int x = r.x & kRunXMask;
        if (r.x & kRunArea) {
          if (x >= b0 && x < b1) AX[x - b0] = (uint32_t)r.y;
        } else if (x < b0) {
          carry += r.y;
        } else if (x < b1) {
          atomicAdd(&D[x - b0], r.y);
        }
      };
      int2 ahead = first_runs(m);
      while (m) {
        const int src = __builtin_ctzll(m);
        m &= m - 1;
        const int2 runs0 = ahead;
        ahead = first_runs(m);
        const uint32_t rgbx = (uint32_t)__builtin_amdgcn_readlane(paint.x, src);
        const uint32_t how = (uint32_t)__builtin_amdgcn_readlane((int)plan, src);
        if (!loaded) {  // canvas window -> LDS
#pragma unroll
          for (int c = 0; c < kChunksB; c++) {
            const int x0 = b0 + c * 256 + 4 * lane;
            uint4 v = make_uint4(0, 0, 0, 0);
            if (kA8) {
              const uint8_t* row = (const uint8_t*)canvas + (size_t)y * W;
              uint32_t u[4] = {0, 0, 0, 0};
              if (vec && x0 + 3 < b1) {
                uint32_t w4 = *(const uint32_t*)(row + x0);
#pragma unroll
                for (int q = 0; q < 4; q++) u[q] = ((w4 >> (8 * q)) & 255u) * 0x01010101u;
              } else {
#pragma unroll
                for (int q = 0; q < 4; q++) u[q] = (x0 + q < b1) ? row[x0 + q] * 0x01010101u : 0u;
              }
              v = make_uint4(u[0], u[1], u[2], u[3]);
            } else {
              const uint32_t* row = (const uint32_t*)canvas + (size_t)y * W;
              if (vec && x0 + 3 < b1) {
                v = *(const uint4*)(row + x0);
              } else {
                v.x = (x0 < b1) ? row[x0] : 0u;
                v.y = (x0 + 1 < b1) ? row[x0 + 1] : 0u;
                v.z = (x0 + 2 < b1) ? row[x0 + 2] : 0u;
                v.w = (x0 + 3 < b1) ? row[x0 + 3] : 0u;
              }
            }
            const int i4 = c * 256 + 4 * lane;
            WIN[i4] = v.x;
            WIN[i4 + 1] = v.y;
            WIN[i4 + 2] = v.z;
            WIN[i4 + 3] = v.w;
          }
          loaded = true;
        }
        int mode, kind, lo, hi;
        carry = 0;
        if (how & kPlanPlain) {
          lo = (int)(how & 2047u);
          hi = (int)(how >> 11 & 2047u);
          mode = (int)(how >> 22 & 31u);
          kind = (int)(how >> 27 & 3u);
          scatter(runs0);
          if (how & kPlanCarry) carry = __builtin_amdgcn_readlane(wave_incl_sum(carry), kWave - 1);
          __syncthreads();
        } else {
          mode = __builtin_amdgcn_readlane(paint.y, src);
          const int taskBase = __builtin_amdgcn_readlane(paint.z, src);
          const int nWin = __builtin_amdgcn_readlane(paint.w, src);
          const int rowStart = __builtin_amdgcn_readlane(span.x, src);
          const int rowCount = __builtin_amdgcn_readlane(span.y, src);
          const int xlo = __builtin_amdgcn_readlane(span.z, src);
          const int xhi = __builtin_amdgcn_readlane(span.w, src);
          if (mode == kMask && !(y >= rowStart && y < rowStart + rowCount)) {
            // rows outside a mask fill's path are cleared (paths.nim:1910-1912)
            for (int c = 0; c < kChunksB; c++) {
              const int i4 = c * 256 + 4 * lane;
              WIN[i4] = WIN[i4 + 1] = WIN[i4 + 2] = WIN[i4 + 3] = 0u;
              const int x0 = b0 + c * 256 + 4 * lane;
              const int n = b1 - x0;
              ntouch += n <= 0 ? 0 : (n >= 4 ? 4 : n);
            }
            dirty = true;
            continue;
          }
          // gather this call's runs for row y into D / AX.  Every phase-A
          // window's deltas sum to zero, so windows that end before b0 or
          // start at b1 or later change nothing here.
          const int tb = taskBase + (y - rowStart) * nWin;
          const int winBase = mode == kMask ? 0 : (xlo & ~3);
          kind = kRowNone;
          for (int w = 0; w < nWin; w++) {
            const int wx0 = winBase + w * kWinA;
            if (wx0 >= b1) break;
            if (wx0 + kWinA < b0) continue;
            RowRuns rr = P.tasks[tb + w];
            rr.off = uni(rr.off);
            rr.n = uni(rr.n);
            rr.kind = uni(rr.kind);
            if (rr.kind > kind) kind = rr.kind;
            for (int e = lane; e < rr.n; e += 64) scatter(P.runs[rr.off + e]);
          }
          carry = __builtin_amdgcn_readlane(wave_incl_sum(carry), kWave - 1);
          __syncthreads();
          if (kind == kRowNone) continue;
          lo = mode == kMask ? 0 : (xlo > b0 ? xlo - b0 : 0);
          hi = mode == kMask ? b1 - b0 : (xhi < b1 ? xhi : b1) - b0;
        }
        const bool maskCov = kind == kRowCoverage && mode == kMask;  // every pixel is written
        if (mode == kNormal && hi - (lo & ~3) < kWave) {
          // a narrow call: its deltas and pixels are one slice from lo & ~3
          const int idx = (lo & ~3) + lane;
          int32_t d = 0;
          if (idx <= hi) {
            d = D[idx];
            D[idx] = 0;
          }
          const int32_t code = carry + wave_incl_sum(d);
          if (idx >= lo && idx < hi && code != 0) {
            const uint32_t ax = (kind == kRowOps && code >= kArea && code < kClear) ? AX[idx] : 0u;
            bool t = false;
            WIN[idx] = apply_normal(kind == kRowCoverage, code, ax, WIN[idx], rgbx, &t);
            if (t) {
              ntouch++;
              dirty = true;
            }
          }
          __syncthreads();
          continue;
        }
        // The call's deltas lie in [xlo & ~3, xhi] (phase-A windows start on
        // a multiple of 4, and a run may end at xhi): the 64-px slices from
        // lo's to hi's hold them all, since xlo & ~3 shares xlo's slice.
        // Pixel codes in 64-px slices (lane l takes pixel l of the slice).
        // The pixels this call changes are queued, packed as code << 11 |
        // index, and the blend runs on full batches of 64 queued pixels, so
        // partly covered slices do not leave lanes idle in the blend.  A
        // call changes each pixel at most once, so a batch never holds the
        // same pixel twice.
        int s = lo >> 6;
        const int sEnd = (hi >> 6) + 1 < kWinB / 64 ? (hi >> 6) + 1 : kWinB / 64;
        int nq = 0;
        for (;;) {
          while (s < sEnd && nq < kWave) {
            const int idx = s * 64 + lane;
            const int32_t d = D[idx];
            D[idx] = 0;
            const int32_t incl = wave_incl_sum(d);
            const int32_t code = carry + incl;
            carry += __builtin_amdgcn_readlane(incl, kWave - 1);
            const bool work = idx >= lo && idx < hi && (code != 0 || maskCov);
            const uint64_t wm = __ballot(work);
            const int pos = nq + __builtin_amdgcn_mbcnt_hi((uint32_t)(wm >> 32),
                                                           __builtin_amdgcn_mbcnt_lo((uint32_t)wm, 0u));
            if (work) Q[pos] = code * 2048 + idx;
            nq += __popcll(wm);
            s++;
          }
          if (nq == 0) break;
          if (lane < nq) {
            const int32_t v = Q[lane];
            const int idx = v & 2047;
            const int32_t code = v >> 11;
            uint32_t ax = (kind == kRowOps && code >= kArea && code < kClear) ? AX[idx] : 0u;
            bool t = false;
            if (mode == kNormal)
              WIN[idx] = apply_normal(kind == kRowCoverage, code, ax, WIN[idx], rgbx, &t);
            else
              WIN[idx] = apply_code(kind, code, ax, WIN[idx], rgbx, mode, &t);
            if (t) {
              ntouch++;
              dirty = true;
            }
          }
          // keep the overflow (queue positions 64 .. nq-1) for the next batch
          nq = nq > kWave ? nq - kWave : 0;
          if (lane < nq) Q[lane] = Q[kWave + lane];
        }
        __syncthreads();
      }
    }
    if (__ballot(dirty) != 0) {  // LDS window -> canvas
#pragma unroll
      for (int c = 0; c < kChunksB; c++) {
        const int x0 = b0 + c * 256 + 4 * lane;
        const int i4 = c * 256 + 4 * lane;
        const uint4 v = make_uint4(WIN[i4], WIN[i4 + 1], WIN[i4 + 2], WIN[i4 + 3]);
        if (kA8) {
          uint8_t* row = (uint8_t*)canvas + (size_t)y * W;
          if (vec && x0 + 3 < b1) {
            *(uint32_t*)(row + x0) = ch_a(v.x) | (ch_a(v.y) << 8) | (ch_a(v.z) << 16) | (ch_a(v.w) << 24);
          } else {
            if (x0 < b1) row[x0] = (uint8_t)ch_a(v.x);
            if (x0 + 1 < b1) row[x0 + 1] = (uint8_t)ch_a(v.y);
            if (x0 + 2 < b1) row[x0 + 2] = (uint8_t)ch_a(v.z);
            if (x0 + 3 < b1) row[x0 + 3] = (uint8_t)ch_a(v.w);
          }
        } else {
          uint32_t* row = (uint32_t*)canvas + (size_t)y * W;
          if (vec && x0 + 3 < b1) {
            *(uint4*)(row + x0) = v;
          } else {
            if (x0 < b1) row[x0] = v.x;
            if (x0 + 1 < b1) row[x0 + 1] = v.y;
            if (x0 + 2 < b1) row[x0 + 2] = v.z;
            if (x0 + 3 < b1) row[x0 + 3] = v.w;
          }
        }
      }
    }
  }
  if (touchedOut) {
    ntouch = (uint32_t)wave_incl_sum((int32_t)ntouch);
    ntouch = __builtin_amdgcn_readlane(ntouch, kWave - 1);
    if (lane == 0 && ntouch) atomicAdd(touched_slot(touchedOut), (unsigned long long)ntouch);
  }
}

// ---------------------------------------------------------------------------
// launcher
// ---------------------------------------------------------------------------
int scene_set_lds_limits(size_t bytes) {
  if (hipFuncSetAttribute((const void*)scene_rows_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                          (int)(bytes - 1024)) != hipSuccess)
    return kErrDevice;
  return 0;
}

size_t scene_gscratch_bytes(int rowGrid, int gcap) { return (size_t)rowGrid * row_cap_bytes(gcap); }

// Clears the counters and queue heads of a render.  A kernel rather than a
// memset, so that a render captured in a graph holds kernel nodes only.
__global__ void __launch_bounds__(256) scene_clear_kernel(int32_t* counters, int nc, int32_t* queues,
                                                          int nq) {
  for (int i = threadIdx.x; i < nc; i += blockDim.x) counters[i] = 0;
  for (int i = threadIdx.x; i < nq; i += blockDim.x) queues[i] = 0;
}

// Text calls: one wave per glyph instance writes its commands and subpaths
// into the scene's recording (GlyphInst).  Points are transformed as
// Path.transform transforms them (paths.nim:264-333): m * (x, y) in float32.
__global__ void __launch_bounds__(256) scene_expand_kernel(const GlyphInst* inst, int n,
                                                           const SceneCmd* aCmds, const ScenePoly* aPolys,
                                                           SceneCmd* cmds, ScenePoly* polys) {
  const int lane = threadIdx.x & 63;
  for (int w = blockIdx.x * 4 + (threadIdx.x >> 6); w < n; w += gridDim.x * 4) {
    const GlyphInst g = inst[w];
    const float* m = g.m;
    if (g.srcCmd < 0) {  // path.rect(x, y, w, h), clockwise unless m[4] (paths.nim:506-521)
      const float x = m[0], y = m[1], rw = m[2], rh = m[3];
      const bool ccw = m[4] != 0.0f;
      if (lane < 5) {
        SceneCmd c = {};
        c.kind = lane == 0 ? 1.0f : lane == 4 ? 0.0f : 2.0f;
        if (lane == 0) { c.p[0] = x; c.p[1] = y; }
        if (lane == 1) { c.p[0] = ccw ? x : x + rw; c.p[1] = ccw ? y + rh : y; }
        if (lane == 2) { c.p[0] = x + rw; c.p[1] = y + rh; }
        if (lane == 3) { c.p[0] = ccw ? x + rw : x; c.p[1] = ccw ? y : y + rh; }
        c.sx = x;
        c.sy = y;
        c.pad[0] = g.polyIdx;
        cmds[g.dstCmd + lane] = c;
      }
      if (lane == 0) {
        ScenePoly sp = {};
        sp.firstCmd = g.dstCmd;
        sp.numCmds = 5;
        polys[g.dstPoly] = sp;
      }
      continue;
    }
    for (int k = lane; k < g.nCmds; k += 64) {
      SceneCmd c = aCmds[g.srcCmd + k];
      if (!g.identity) {
        const int kind = (int)c.kind;
        const int pts = kind == 5 ? 3 : kind == 7 ? 2 : (kind == 1 || kind == 2) ? 1 : 0;
        for (int q = 0; q < pts; q++) {
          const float x = c.p[2 * q], y = c.p[2 * q + 1];
          c.p[2 * q] = m[0] * x + m[2] * y + m[4];
          c.p[2 * q + 1] = m[1] * x + m[3] * y + m[5];
        }
        const float sx = c.sx, sy = c.sy;
        c.sx = m[0] * sx + m[2] * sy + m[4];
        c.sy = m[1] * sx + m[3] * sy + m[5];
      }
      c.pad[0] += g.polyIdx;
      cmds[g.dstCmd + k] = c;
    }
    for (int k = lane; k < g.nPolys; k += 64) {
      ScenePoly sp = aPolys[g.srcPoly + k];
      sp.firstCmd = sp.firstCmd - g.srcCmd + g.dstCmd;
      polys[g.dstPoly + k] = sp;
    }
  }
}

int scene_launch_expand(const GlyphInst* inst, int32_t n, const SceneCmd* arenaCmds, const ScenePoly* arenaPolys,
                        SceneCmd* cmds, ScenePoly* polys, hipStream_t s) {
  if (n <= 0) return 0;
  int grid = (n + 3) / 4;
  if (grid > 2048) grid = 2048;
  hipLaunchKernelGGL(scene_expand_kernel, dim3(grid), dim3(256), 0, s, inst, n, arenaCmds, arenaPolys, cmds,
                     polys);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_clear(const ScenePools& p, hipStream_t s) {
  hipLaunchKernelGGL(scene_clear_kernel, dim3(1), dim3(256), 0, s, p.counters, (int)kCounterInts,
                     p.queues, kQueueSets * kQueues * kQueueStride);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_geometry(const ScenePools& p, hipStream_t s) {
  if (p.nItems <= 0) return 0;
  // calls of more than kBlock commands (they come first in itemOrder)
  if (p.nBig > 0) {
    const int grid = (p.bigCmds + 255) / 256;
    hipLaunchKernelGGL(scene_big_cmd_kernel, dim3(grid), dim3(256), 0, s, p, 0);
    // point layout: subpath chunks over the device
    hipLaunchKernelGGL(scene_big_plan_kernel, dim3(1), dim3(kScanBlock), 0, s, p, 2);
    hipLaunchKernelGGL(scene_big_front_kernel, dim3(kBigSegGrid), dim3(256), 0, s, p, 0);
    hipLaunchKernelGGL(scene_big_front_alloc_kernel, dim3(p.nBig), dim3(256), 0, s, p);
    hipLaunchKernelGGL(scene_big_front_kernel, dim3(kBigSegGrid), dim3(256), 0, s, p, 1);
    hipLaunchKernelGGL(scene_big_cmd_kernel, dim3(grid), dim3(256), 0, s, p, 1);
    // fills: segments in chunks over the device
    hipLaunchKernelGGL(scene_big_plan_kernel, dim3(1), dim3(kScanBlock), 0, s, p, 0);
    hipLaunchKernelGGL(scene_big_seg_kernel, dim3(kBigSegGrid), dim3(256), 0, s, p, 0);
    hipLaunchKernelGGL(scene_big_seg_alloc_kernel, dim3(p.nBig), dim3(256), 0, s, p);
    hipLaunchKernelGGL(scene_big_seg_kernel, dim3(kBigSegGrid), dim3(256), 0, s, p, 1);
  }
  if (p.nItems > p.nBig)
    hipLaunchKernelGGL(scene_geom_kernel, dim3(p.nItems - p.nBig), dim3(kBlock), 0, s, p, p.nBig);
  if (p.nStrokes > 0) {
    hipLaunchKernelGGL(scene_stroke_kernel<false>, dim3(kStrokeGrid), dim3(256), 0, s, p);
    hipLaunchKernelGGL(scene_stroke_alloc_kernel, dim3(p.nStrokes), dim3(256), 0, s, p);
    hipLaunchKernelGGL(scene_stroke_kernel<true>, dim3(kStrokeGrid), dim3(256), 0, s, p);
  }
  const int planBlocks = (p.nItems + kPlanCalls - 1) / kPlanCalls;
  hipLaunchKernelGGL(scene_plan_kernel, dim3(planBlocks + kSegBandBlocks), dim3(256), 0, s, p, planBlocks);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_bands(const ScenePools& p, hipStream_t s) {
  const int bins = (p.H + kBinRows - 1) / kBinRows, binBlocks = (bins + kXcds - 1) / kXcds * kXcds;
  hipLaunchKernelGGL(scene_band_kernel, dim3(binBlocks + kBandBlocks), dim3(256), 0, s, p, binBlocks);
  hipLaunchKernelGGL(scene_band_write_kernel, dim3(kBandBlocks), dim3(256), 0, s, p);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_tasks(const ScenePools& p, hipStream_t s) {
  hipLaunchKernelGGL(scene_task_kernel<false>, dim3(kTaskBlocks), dim3(256), 0, s, p);
  hipLaunchKernelGGL(scene_task_kernel<true>, dim3(kTaskBlocks), dim3(256), 0, s, p);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_heavy(const ScenePools& p, int numCUs, hipStream_t s) {
  hipLaunchKernelGGL(scene_heavy_kernel, dim3(scene_queue_grid(numCUs * kHeavyGroupsPerCU)), dim3(kHeavyThreads), 0,
                     s, p);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_rows(const ScenePools& p, const RowShape& shape, int numCUs, hipStream_t s) {
  const size_t lds = row_lds_fixed_bytes(kWinA) + row_cap_bytes(shape.ldsCap);
  hipLaunchKernelGGL(scene_rows_kernel, dim3(scene_queue_grid(numCUs * shape.wavesPerCU)), dim3(64), lds, s, p);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

int scene_launch_compose(const ScenePools& p, void* canvas, bool a8, unsigned long long* touched,
                         int32_t* errOut, int grid, hipStream_t s) {
  if (a8)
    hipLaunchKernelGGL(scene_compose_kernel<true>, dim3(grid), dim3(64), 0, s, p, canvas, touched,
                       errOut);
  else
    hipLaunchKernelGGL(scene_compose_kernel<false>, dim3(grid), dim3(64), 0, s, p, canvas, touched,
                       errOut);
  return hipGetLastError() == hipSuccess ? 0 : kErrDevice;
}

}  // namespace pxh
