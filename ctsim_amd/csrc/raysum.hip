// Ray-sum kernels for gfx950 (Scanner::collectProjections,
// libctsim/scanner.cpp:280-656).
//
// One lane owns one (view, detector): it walks the detector's sample rays and
// sums every phantom element's clipped chord times its attenuation in FP64,
// then stores sum / nSample as float (scanner.cpp:522).  All lanes of a wave
// visit the same elements in the same order, so element data is read with
// wave-uniform loads.  The detector and source positions are repeated sums
// along the detector array (scanner.cpp:490-532); a first pass with one lane
// per sum performs that walk so every lane starts from the reference's
// values.
//
//   F64 path    short closed forms with error bounds for ellipses and
//               rectangles, stored where the bounds round to one float32; the
//               rest in the reference's clipping step order: bounding-box
//               reject by Cohen-Sutherland on the polygon outline's box, map
//               to the element frame, circle clip by translate / rotate
//               (atan2, cos, sin) / clamp / rotate back, map back, length.
//   mixed path  the same box reject, then closed-form FP64 chords for
//               ellipses (quadratic in the element frame) and rectangles
//               (slab clip); triangles, segments and sectors keep the
//               reference's clip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include "crmath.h"
#include "scan_plan.h"

#pragma clang fp contract(off)

namespace ctsim {
namespace {

// Per-view constants of projectSingleView, scanner.cpp:449-473.
struct ViewSetup {
  double sdx, sdy, ddx, ddy, ddx2, ddy2, aInc, aSampInc;
};

__device__ __forceinline__ ViewSetup view_setup(const ViewEnds& e, int nDet, unsigned nSample,
                                                int geom, double angDetInc) {
  ViewSetup s;
  s.sdx = (e.xs2 - e.xs1) / nDet;
  s.sdy = (e.ys2 - e.ys1) / nDet;
  s.ddx = s.ddy = s.ddx2 = s.ddy2 = s.aInc = s.aSampInc = 0;
  if (geom == GEOM_EQUIANGULAR) {
    s.aInc = angDetInc;
    s.aSampInc = s.aInc / nSample;
  } else {
    s.ddx = (e.xd2 - e.xd1) / nDet;
    s.ddy = (e.yd2 - e.yd1) / nDet;
    s.ddx2 = s.ddx / nSample;
    s.ddy2 = s.ddy / nSample;
  }
  return s;
}

struct WalkArgs {
  const ViewEnds* ends;
  double4* walk;  // [nView][walk_row]
  int* counter;   // the ray-sum kernels' three counters, zeroed here
  int nView, nDet, geom;
  unsigned nSample;
  double angDetInc, angDetLen;
};

// A view's row of the walk: the four increments, then xs, ys, xd (or the
// detector angle) and yd of every kWalkStep-th detector.  A reader takes the
// last steps itself.
constexpr int kWalkStep = 4;
__host__ __device__ inline int walk_row(int nDet) { return 1 + (nDet + kWalkStep - 1) / kWalkStep; }

// The detector walk of projectSingleView (scanner.cpp:449-531): per view
// four chains of rounded sums (xs, ys, and xd, yd or the detector angle), one
// lane per chain, 16 views per block.
//
// What bounds it: the latency of the chains, nDet adds one after the other.
// The stores go straight to memory, and only every kWalkStep-th state is kept:
// with all of them (47 MB at 1440 views of 1024 detectors), gathered in LDS and
// stored as rows between two barriers, each of which waits for the row's
// stores, the kernel took 48 us there, now 11.
constexpr int kWalkViews = 16;
__global__ __launch_bounds__(64) void raysum_walk_kernel(WalkArgs a) {
  if (blockIdx.x == 0 && threadIdx.x < 3) a.counter[threadIdx.x] = 0;
  const int lane = threadIdx.x, comp = lane & 3, v = blockIdx.x * kWalkViews + (lane >> 2);
  if (v >= a.nView) return;
  const ViewEnds e = a.ends[v];
  const ViewSetup s = view_setup(e, a.nDet, a.nSample, a.geom, a.angDetInc);
  const bool equi = a.geom == GEOM_EQUIANGULAR;
  double x = 0.0, inc = 0.0;
  if (comp == 0) { x = e.xs1 + (s.sdx / 2); inc = s.sdx; }
  else if (comp == 1) { x = e.ys1 + (s.sdy / 2); inc = s.sdy; }
  else if (comp == 2) {
    if (equi) { x = e.detAngle - (a.angDetLen / 2) + s.aSampInc / 2; inc = s.aInc; }
    else { x = e.xd1 + s.ddx2 / 2; inc = s.ddx; }
  } else if (!equi) {  // yd (the equiangular walk keeps 0 here)
    x = e.yd1 + s.ddy2 / 2;
    inc = s.ddy;
  }
  const int n = walk_row(a.nDet);
  double* out = reinterpret_cast<double*>(a.walk + static_cast<size_t>(v) * n) + comp;
  *out = inc;
#pragma unroll 8
  for (int c = 1; c < n; c++) {
    out[4 * c] = x;
#pragma unroll
    for (int j = 0; j < kWalkStep; j++) x += inc;
  }
}

// Detector d's state of view v's walk.
__device__ __forceinline__ double4 walk_at(const double4* walk, int nDet, int v, int d) {
  const double4* row = walk + static_cast<size_t>(v) * walk_row(nDet);
  const double4 inc = row[0];
  double4 w = row[1 + d / kWalkStep];
#pragma unroll
  for (int j = 1; j < kWalkStep; j++)
    if (d % kWalkStep >= j) {
      w.x += inc.x;
      w.y += inc.y;
      w.z += inc.z;
      w.w += inc.w;
    }
  return w;
}

// --------------------------------------------------- reference clipping

__device__ __forceinline__ void xf(const double* m, double& x, double& y) {
  const double xt = x * m[0] + y * m[2] + m[4];
  const double yt = x * m[1] + y * m[3] + m[5];
  x = xt;
  y = yt;
}

// normalizeAngle, libctsupport/mathfuncs.cpp:72-81
__device__ __forceinline__ double normalize_angle(double t) {
  while (t < 0.) t += kTwoPi;
  while (t >= kTwoPi) t -= kTwoPi;
  return t;
}

// rectcode + clip_rect, libctsupport/clip.cpp:332-395
__device__ __forceinline__ int rectcode(double x, double y, const double* r) {
  int c = 0;
  if (x < r[0]) c = 1;
  else if (x > r[2]) c = 2;
  if (y < r[1]) c += 4;
  else if (y > r[3]) c += 8;
  return c;
}
__device__ bool clip_rect(double& x1, double& y1, double& x2, double& y2, const double* r) {
  double x = 0, y = 0;
  int c1 = rectcode(x1, y1, r), c2 = rectcode(x2, y2, r);
  while (c1 || c2) {
    if (c1 & c2) return false;
    const int c = c1 ? c1 : c2;
    if (c & 1) { y = y1 + (y2 - y1) * (r[0] - x1) / (x2 - x1); x = r[0]; }
    else if (c & 2) { y = y1 + (y2 - y1) * (r[2] - x1) / (x2 - x1); x = r[2]; }
    else if (c & 4) { x = x1 + (x2 - x1) * (r[1] - y1) / (y2 - y1); y = r[1]; }
    else if (c & 8) { x = x1 + (x2 - x1) * (r[3] - y1) / (y2 - y1); y = r[3]; }
    if (c == c1) { x1 = x; y1 = y; c1 = rectcode(x1, y1, r); }
    else { x2 = x; y2 = y; c2 = rectcode(x2, y2, r); }
  }
  return true;
}

// clip_circle, libctsupport/clip.cpp:126-198 (rot_mtx2 / xform_mtx2 inlined)
__device__ bool clip_circle(double& x1, double& y1, double& x2, double& y2, double cx, double cy,
                            double radius, double t1, double t2) {
  double xc1 = x1, yc1 = y1, xc2 = x2, yc2 = y2, ccx = cx, ccy = cy;
  const double xtrans = -xc1, ytrans = -yc1;
  xc1 += xtrans; yc1 += ytrans; xc2 += xtrans; yc2 += ytrans; ccx += xtrans; ccy += ytrans;
  const double theta = -crm_atan2(yc2, xc2);
  // correctly rounded cos and sin are exactly even and odd, so rotating back
  // by -theta below reuses them as the reference's cos(-theta), sin(-theta)
  double c, s;
  crm_sincos(theta, &s, &c);
  const double cb = c, sb = -s;
  {  // xform by rot(theta): x' = x c + y (-s) + 0, y' = x s + y c + 0
    double xt = xc2 * c + yc2 * -s + 0.0, yt = xc2 * s + yc2 * c + 0.0;
    xc2 = xt; yc2 = yt;
    xt = ccx * c + ccy * -s + 0.0; yt = ccx * s + ccy * c + 0.0;
    ccx = xt; ccy = yt;
  }
  t1 += theta;
  t2 += theta;
  t1 = normalize_angle(t1);
  t2 = normalize_angle(t2);
  if (xc2 < -kDEps || fabs(yc2) > kFEps) return false;  // reference: ERR_SEVERE, reject
  if (fabs(ccy) > radius) return false;
  const double temp = sqrt(radius * radius - ccy * ccy);
  const double xcmin = ccx - temp, xcmax = ccx + temp;
  if (fabs(t2 - t1) < kDEps) {
    if (xc1 < xcmin) xc1 = xcmin;
    if (xc2 > xcmax) xc2 = xcmax;
  } else if (t1 < t2) {
    if (t1 < kPi && t2 > kPi)
      if (xc1 < xcmin) xc1 = xcmin;
  } else if (t1 > t2) {
    if (t1 < kPi)
      if (xc1 < xcmin) xc1 = xcmin;
    if (xc2 > xcmax) xc2 = xcmax;
  }
  c = cb;
  s = sb;
  {
    double xt = xc1 * c + yc1 * -s + 0.0, yt = xc1 * s + yc1 * c + 0.0;
    xc1 = xt; yc1 = yt;
    xt = xc2 * c + yc2 * -s + 0.0; yt = xc2 * s + yc2 * c + 0.0;
    xc2 = xt; yc2 = yt;
  }
  xc1 += -xtrans; yc1 += -ytrans; xc2 += -xtrans; yc2 += -ytrans;
  x1 = xc1; y1 = yc1; x2 = xc2; y2 = yc2;
  return true;
}

// tcode + clip_triangle, libctsupport/clip.cpp:243-316
__device__ __forceinline__ int tcode(double x, double y, double m, double b, bool clipX) {
  int c = 0;
  if (clipX && y < 0.) c = 1;
  if (y > -m * x + b + kDEps) c += 2;
  if (y > m * x + b + kDEps) c += 4;
  return c;
}
__device__ bool clip_triangle(double& x1, double& y1, double& x2, double& y2, double u, double v,
                              bool clipX) {
  const double m = v / u, b = v;
  int c1 = tcode(x1, y1, m, b, clipX), c2 = tcode(x2, y2, m, b, clipX);
  while (c1 || c2) {
    if (c1 & c2) return false;
    const int c = c1 ? c1 : c2;
    double x = 0, y = 0;
    if (c & 1) {
      x = x1 + (x2 - x1) * (0.0 - y1) / (y2 - y1);
      y = 0.0;
    } else if (c & 2) {
      const double dx = x2 - x1, dy = y2 - y1;
      if (fabs(dx) > kDEps) x = (-y1 + b + x1 * dy / dx) / (m + dy / dx);
      else x = x1;
      y = -m * x + b;
    } else if (c & 4) {
      const double dx = x2 - x1, dy = y2 - y1;
      if (fabs(dx) > kDEps) {
        x = (y1 - b - x1 * dy / dx);
        x /= (m - dy / dx);
      } else {
        x = x1;
      }
      y = m * x + b;
    }
    if (c == c1) { x1 = x; y1 = y; c1 = tcode(x1, y1, m, b, clipX); }
    else { x2 = x; y2 = y; c2 = tcode(x2, y2, m, b, clipX); }
  }
  return true;
}

// clip_segment (libctsupport/clip.cpp:44-77) and clip_sector (clip.cpp:
// 90-111) share the ellipse's clip_circle call below, so the kernel holds
// one copy of the circle clip (and its atan2, sin and cos): each case does
// the same operations in the same order as the reference.

// False only when the segment certainly misses the box: separating axes
// (the box's two axes and the segment's normal) on the box widened by a
// margin far above the rounding of the reference's Cohen-Sutherland clip,
// so every segment that clip keeps passes.  No division.
__device__ __forceinline__ bool seg_may_hit_box(double x1, double y1, double x2, double y2, const double* r) {
  const double scale = fmax(fmax(fabs(r[0]), fabs(r[2])), fmax(fmax(fabs(r[1]), fabs(r[3])), 1.0));
  const double m = 1e-9 * scale;
  const double bx0 = r[0] - m, by0 = r[1] - m, bx1 = r[2] + m, by1 = r[3] + m;
  if (fmax(x1, x2) < bx0 || fmin(x1, x2) > bx1 || fmax(y1, y2) < by0 || fmin(y1, y2) > by1) return false;
  const double nx = y1 - y2, ny = x2 - x1;  // the segment's normal
  const double s0 = nx * (bx0 - x1) + ny * (by0 - y1), s1 = nx * (bx1 - x1) + ny * (by0 - y1);
  const double s2 = nx * (bx0 - x1) + ny * (by1 - y1), s3 = nx * (bx1 - x1) + ny * (by1 - y1);
  const double tol = m * (fabs(nx) + fabs(ny));
  const double lo = fmin(fmin(s0, s1), fmin(s2, s3)), hi = fmax(fmax(s0, s1), fmax(s2, s3));
  return lo <= tol && hi >= -tol;
}

// True only when the segment certainly crosses the box: the same test on the
// box narrowed by that margin, with strict inequalities.  Such a segment is
// kept by the reference's Cohen-Sutherland clip, whose clipped points the
// chord discards, so the clip can be skipped.
__device__ __forceinline__ bool seg_surely_hits_box(double x1, double y1, double x2, double y2, const double* r) {
  const double scale = fmax(fmax(fabs(r[0]), fabs(r[2])), fmax(fmax(fabs(r[1]), fabs(r[3])), 1.0));
  const double m = 1e-9 * scale;
  const double bx0 = r[0] + m, by0 = r[1] + m, bx1 = r[2] - m, by1 = r[3] - m;
  if (!(bx0 < bx1 && by0 < by1)) return false;
  if (!(fmax(x1, x2) > bx0 && fmin(x1, x2) < bx1 && fmax(y1, y2) > by0 && fmin(y1, y2) < by1)) return false;
  const double nx = y1 - y2, ny = x2 - x1;
  const double s0 = nx * (bx0 - x1) + ny * (by0 - y1), s1 = nx * (bx1 - x1) + ny * (by0 - y1);
  const double s2 = nx * (bx0 - x1) + ny * (by1 - y1), s3 = nx * (bx1 - x1) + ny * (by1 - y1);
  const double tol = m * (fabs(nx) + fabs(ny));
  const double lo = fmin(fmin(s0, s1), fmin(s2, s3)), hi = fmax(fmax(s0, s1), fmax(s2, s3));
  return lo < -tol && hi > tol;
}

// False only when the line through the segment certainly misses the unit
// circle of the element frame m (an ellipse): its distance from the centre,
// |p1 x p2| / |p2 - p1| in that frame, exceeds 1 by a margin far above the
// rounding of the reference's circle clip, which then rejects the segment
// (clip.cpp:152, |ccy| > radius).
__device__ __forceinline__ bool line_may_hit_unit_circle(const double* m, double x1, double y1, double x2,
                                                         double y2) {
  const double X1 = x1 * m[0] + y1 * m[2] + m[4], Y1 = x1 * m[1] + y1 * m[3] + m[5];
  const double X2 = x2 * m[0] + y2 * m[2] + m[4], Y2 = x2 * m[1] + y2 * m[3] + m[5];
  const double dx = X2 - X1, dy = Y2 - Y1, cr = X1 * Y2 - X2 * Y1;
  const double sc = fmax(fmax(fabs(X1), fabs(Y1)), fmax(fmax(fabs(X2), fabs(Y2)), 1.0));
  const double r = 1.0 + 1e-9 * sc;
  return cr * cr <= r * r * (dx * dx + dy * dy);
}

// PhantomElement::clipLineWorldCoords / clipLineNormalizedCoords and
// Scanner::projectLineAgainstPElem, phantom.cpp:830-898, scanner.cpp:633-656
__device__ __forceinline__ double chord_ref(const ElemGPU& e, double x1, double y1, double x2, double y2) {
  if (!seg_surely_hits_box(x1, y1, x2, y2, e.lim)) {  // else the box clip keeps the segment
    double cx1 = x1, cy1 = y1, cx2 = x2, cy2 = y2;
    if (!clip_rect(cx1, cy1, cx2, cy2, e.lim)) return 0.0;
  }
  xf(e.p2o, x1, y1);
  xf(e.p2o, x2, y2);
  bool ok = false;
  const int type = e.type;
  if (type == PE_RECT) {
    const double unit[4] = {-1.0, -1.0, 1.0, 1.0};
    ok = clip_rect(x1, y1, x2, y2, unit);
  } else if (type == PE_TRI) {
    ok = clip_triangle(x1, y1, x2, y2, 1.0, 1.0, true);
  } else if (type == PE_ELLIPSE || type == PE_SEGMENT || type == PE_SECTOR) {
    const bool scaled = type != PE_ELLIPSE;  // segment, sector: x * u, y * v
    const double u = e.u, v = e.v;
    double xc1 = x1, yc1 = y1, xc2 = x2, yc2 = y2;
    double ccy = 0.0, radius = 1.0;
    ok = true;
    if (scaled) {
      xc1 = x1 * u; yc1 = y1 * v; xc2 = x2 * u; yc2 = y2 * v;
      if (type == PE_SEGMENT && yc1 > 0. && yc2 > 0.) ok = false;
      radius = sqrt(u * u + v * v);
      ccy = v;
    }
    if (ok) ok = clip_circle(xc1, yc1, xc2, yc2, 0.0, ccy, radius, 0.0, 0.0);
    if (ok && type == PE_SEGMENT) {
      if (yc1 > 0. && yc2 > 0.) {
        ok = false;
      } else if (yc1 > 0.) {
        xc1 = xc1 + (xc2 - xc1) * (0.0 - yc1) / (yc2 - yc1);
        yc1 = 0.0;
      } else if (yc2 > 0.) {
        xc2 = xc1 + (xc2 - xc1) * (0.0 - yc1) / (yc2 - yc1);
        yc2 = 0.0;
      }
    }
    if (ok && type == PE_SECTOR) ok = clip_triangle(xc1, yc1, xc2, yc2, u, v, false);
    if (ok) {
      if (scaled) {
        x1 = xc1 / u; y1 = yc1 / v; x2 = xc2 / u; y2 = yc2 / v;
      } else {
        x1 = xc1; y1 = yc1; x2 = xc2; y2 = yc2;
      }
    }
  }
  if (!ok) return 0.0;
  xf(e.o2p, x1, y1);
  xf(e.o2p, x2, y2);
  const double len = sqrt((x2 - x1) * (x2 - x1) + (y2 - y1) * (y2 - y1));
  return len * e.atten;
}

// ------------------------------------------------- closed-form chords
#pragma clang fp contract(fast)

// Segment-box test by slabs (the reference rejects with Cohen-Sutherland on
// the same box; the two agree except for rays grazing a box corner).
__device__ __forceinline__ bool seg_hits_box(double x1, double y1, double dx, double dy,
                                             const double* r) {
  double t0 = 0.0, t1 = 1.0;
  if (dx != 0.0) {
    const double inv = 1.0 / dx;
    double ta = (r[0] - x1) * inv, tb = (r[2] - x1) * inv;
    if (ta > tb) { const double t = ta; ta = tb; tb = t; }
    t0 = fmax(t0, ta);
    t1 = fmin(t1, tb);
  } else if (x1 < r[0] || x1 > r[2]) {
    return false;
  }
  if (dy != 0.0) {
    const double inv = 1.0 / dy;
    double ta = (r[1] - y1) * inv, tb = (r[3] - y1) * inv;
    if (ta > tb) { const double t = ta; ta = tb; tb = t; }
    t0 = fmax(t0, ta);
    t1 = fmin(t1, tb);
  } else if (y1 < r[1] || y1 > r[3]) {
    return false;
  }
  return t0 <= t1;
}

// The reference's clip chain as a call: the closed form takes it only for
// triangles, segments and sectors, whose registers then stay out of the
// ellipse and rectangle path.
__device__ __attribute__((noinline)) double chord_ref_call(const ElemGPU& e, double x1, double y1, double x2,
                                                           double y2) {
  return chord_ref(e, x1, y1, x2, y2);
}

// Parameter interval of the segment inside the element, in the element frame.
__device__ double chord_closed(const ElemGPU& e, double x1, double y1, double x2, double y2,
                               double segLen) {
  const double dx = x2 - x1, dy = y2 - y1;
  if (!seg_hits_box(x1, y1, dx, dy, e.lim)) return 0.0;
  if (e.type == PE_ELLIPSE || e.type == PE_RECT) {
    const double px = x1 * e.p2o[0] + y1 * e.p2o[2] + e.p2o[4];
    const double py = x1 * e.p2o[1] + y1 * e.p2o[3] + e.p2o[5];
    const double qx = dx * e.p2o[0] + dy * e.p2o[2];
    const double qy = dx * e.p2o[1] + dy * e.p2o[3];
    double t0, t1;
    if (e.type == PE_ELLIPSE) {
      // |p + t q|^2 = 1
      const double a = qx * qx + qy * qy, b = px * qx + py * qy, c = px * px + py * py - 1.0;
      const double disc = b * b - a * c;
      if (!(disc > 0.0)) return 0.0;
      const double sq = sqrt(disc);
      t0 = (-b - sq) / a;
      t1 = (-b + sq) / a;
    } else {
      t0 = -1e300;
      t1 = 1e300;
      if (qx != 0.0) {
        double ta = (-1.0 - px) / qx, tb = (1.0 - px) / qx;
        if (ta > tb) { const double t = ta; ta = tb; tb = t; }
        t0 = fmax(t0, ta);
        t1 = fmin(t1, tb);
      } else if (px < -1.0 || px > 1.0) {
        return 0.0;
      }
      if (qy != 0.0) {
        double ta = (-1.0 - py) / qy, tb = (1.0 - py) / qy;
        if (ta > tb) { const double t = ta; ta = tb; tb = t; }
        t0 = fmax(t0, ta);
        t1 = fmin(t1, tb);
      } else if (py < -1.0 || py > 1.0) {
        return 0.0;
      }
    }
    t0 = fmax(t0, 0.0);
    t1 = fmin(t1, 1.0);
    return t1 > t0 ? (t1 - t0) * segLen * e.atten : 0.0;
  }
  return chord_ref_call(e, x1, y1, x2, y2);
}

#pragma clang fp contract(off)

struct RaysumArgs {
  const ViewEnds* ends;
  const double4* walk;
  const ElemGPU* __restrict__ elems;
  float* sino;
  int* counter;  // items taken so far, items and rays deferred (zeroed by the walk kernel)
  int nView, nDet, nElem, geom, storageOffset;
  unsigned nSample;
  double angDetInc, centerDetLength;
  int unitPulse;
  // the short chord (fast = 0: every ray by the reference's chain) and what it
  // defers: items (view, first detector) and single rays (view, detector)
  const FastElem* __restrict__ fastElems;
  int2* items;
  int2* rays;
  int fast, deferItems;  // deferItems: raysum_f64_kernel follows, for waves the short chord does not suit
  double fastX, fastY, fastR, fastMin, fastFar;
};

// Detector end (a) and source end (b) of sample i of detector d's ray, as
// raysum_ray walks them (to rounding: the hull test below has a margin).
__device__ __forceinline__ void ray_ends(const RaysumArgs& a, const ViewSetup& s, int v, int d, unsigned i,
                                         double& ax, double& ay, double& bx, double& by) {
  const double4 w = walk_at(a.walk, a.nDet, v, d);
  bx = w.x;
  by = w.y;
  if (a.geom == GEOM_EQUIANGULAR) {
    const double ang = w.z + i * s.aSampInc;
    ax = a.centerDetLength * cos(ang);
    ay = a.centerDetLength * sin(ang);
  } else {
    ax = w.z + i * s.ddx2;
    ay = w.w + i * s.ddy2;
  }
}

// Candidate elements of one wave's rays (detectors d0..d1 of view v, every
// sample): lane k tests element 64 c + k's box against the hull of the
// rays, the quadrilateral of the first and the last ray (widened by the
// sagitta of the detector arc in the equiangular geometry and a margin), by
// separating axes; bit k of mask c is set unless the box is certainly
// outside.  Every ray of the wave lies in the hull, so a clear bit marks an
// element whose chords are all exactly zero.
constexpr int kCandChunks = 16;  // up to 1024 elements; more take no culling
__device__ __forceinline__ void wave_candidates(const RaysumArgs& a, const ViewSetup& s, int v, int d0, int d1,
                                                unsigned long long* masks, int nChunks) {
  double px[4], py[4];
  ray_ends(a, s, v, d0, 0, px[0], py[0], px[1], py[1]);
  ray_ends(a, s, v, d1, a.nSample - 1, px[3], py[3], px[2], py[2]);
  double mg = 1e-9 * fmax(fmax(fmax(fabs(px[0]), fabs(px[1])), fmax(fabs(px[2]), fabs(px[3]))),
                          fmax(fmax(fmax(fabs(py[0]), fabs(py[1])), fmax(fabs(py[2]), fabs(py[3]))), 1.0));
  if (a.geom == GEOM_EQUIANGULAR) {  // the detector ends lie on an arc bulging past the chord
    const double cx = px[3] - px[0], cy = py[3] - py[0];
    mg += (cx * cx + cy * cy) / (2.0 * a.centerDetLength) + 1e-12;
  }
  const double qx0 = fmin(fmin(px[0], px[1]), fmin(px[2], px[3])), qx1 = fmax(fmax(px[0], px[1]), fmax(px[2], px[3]));
  const double qy0 = fmin(fmin(py[0], py[1]), fmin(py[2], py[3])), qy1 = fmax(fmax(py[0], py[1]), fmax(py[2], py[3]));
  const int lane = threadIdx.x;
  for (int c = 0; c < nChunks; c++) {
    const int k = 64 * c + lane;
    bool cand = false;
    if (k < a.nElem) {
      const double* r = a.elems[k].lim;
      cand = !(qx1 < r[0] - mg || qx0 > r[2] + mg || qy1 < r[1] - mg || qy0 > r[3] + mg);
#pragma unroll
      for (int ed = 0; ed < 4 && cand; ed++) {
        const int e2 = (ed + 1) & 3;
        const double nx = py[ed] - py[e2], ny = px[e2] - px[ed];
        double h0 = 1e300, h1 = -1e300;
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const double p = nx * px[j] + ny * py[j];
          h0 = fmin(h0, p);
          h1 = fmax(h1, p);
        }
        const double c00 = nx * r[0] + ny * r[1], c10 = nx * r[2] + ny * r[1];
        const double c01 = nx * r[0] + ny * r[3], c11 = nx * r[2] + ny * r[3];
        const double b0 = fmin(fmin(c00, c10), fmin(c01, c11)), b1 = fmax(fmax(c00, c10), fmax(c01, c11));
        const double tol = mg * (fabs(nx) + fabs(ny)) + 1e-300;
        if (b1 < h0 - tol || b0 > h1 + tol) cand = false;
      }
    }
    const unsigned long long bits = __ballot(cand);
    if (lane == 0) masks[c] = bits;
  }
}

// A wave's deferred chords.  The (lane, element) pairs whose chord is
// needed are queued in the reference's element order and computed 64 at a
// time, one pair per lane, so lanes whose rays miss an element do not idle
// through its clip; each lane then adds its own chords in queue order, the
// order of the element list.  Rings of kQueue entries: at most 63 pairs
// wait before an element's (up to 64) are added, and a flush of 64 follows.
constexpr int kQueue = 128;
struct WaveQueue {
  double4 ray[64];                  // each lane's ray: detector end, source end
  double val[kQueue];               // computed chords, by pair slot
  unsigned long long vmask[kQueue];  // per queued element: the lanes that need it
  int vbase[kQueue];                // ... and the slot of its first pair
  int pair[kQueue];                 // lane | element << 6, by pair slot
};

__device__ __forceinline__ int lanes_below(unsigned long long m) {
  return __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(m >> 32),
                                   __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0));
}

__device__ __forceinline__ unsigned long long uniform_u64(unsigned long long x) {
  return (static_cast<unsigned long long>(static_cast<unsigned>(
              __builtin_amdgcn_readfirstlane(static_cast<unsigned>(x >> 32)))) << 32) |
         static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<unsigned>(x)));
}

// One lane's ray sum: detector d of view v (a lane past the last detector,
// active false, only helps its wave's chords).  masks: the nChunks
// candidate masks (wave_candidates), or nullptr for every element.
__device__ __forceinline__ void raysum_ray(const RaysumArgs& a, const ViewSetup& s, int v, int d, bool active,
                                           const unsigned long long* masks, int nChunks, WaveQueue* qp) {
  const int lane = threadIdx.x;
  const double4 w = walk_at(a.walk, a.nDet, v, active ? d : a.nDet - 1);
  const double xs = w.x, ys = w.y;
  double xd = w.z, yd = w.w, ang = w.z;
  double sum = 0.0;
  for (unsigned i = 0; i < a.nSample; i++) {
    if (a.geom == GEOM_EQUIANGULAR) {
      double sa, ca;
      crm_sincos(ang, &sa, &ca);
      xd = a.centerDetLength * ca;
      yd = a.centerDetLength * sa;
    }
    qp->ray[lane] = make_double4(xd, yd, xs, ys);
    // projectSingleLine: the element list is newest-first (phantom.cpp:247).
    // A segment that misses an element's box, or an ellipse's line that
    // misses it, adds the reference's exact zero, which changes no sum: such
    // pairs are never queued (elements outside the wave's hull by the masks,
    // then lane by lane).
    double rsum = 0.0;
    int enq = 0, done = 0, nv = 0, vc = 0;
    auto flush = [&](int n) {
      __syncthreads();  // rays, pairs and visits written above are visible
      if (lane < n) {
        const int slot = (done + lane) & (kQueue - 1);
        const int pr = qp->pair[slot];
        const double4 r = qp->ray[pr & 63];
        qp->val[slot] = chord_ref(a.elems[pr >> 6], r.x, r.y, r.z, r.w);
      }
      __syncthreads();
      const int prev = done;
      done += n;
      // each lane adds its chords among slots [prev, done), element by element
      while (vc < nv) {
        const int vs = vc & (kQueue - 1);
        const unsigned long long vm = uniform_u64(qp->vmask[vs]);
        const int vb = __builtin_amdgcn_readfirstlane(qp->vbase[vs]);
        if ((vm >> lane) & 1) {
          const int slot = vb + lanes_below(vm);
          if (slot >= prev && slot < done) rsum += qp->val[slot & (kQueue - 1)];
        }
        if (vb + __popcll(vm) > done) break;  // the rest of this element comes later
        vc++;
      }
    };
    for (int c = nChunks - 1; c >= 0; c--) {
      unsigned long long m;
      if (masks) {
        m = uniform_u64(masks[c]);
      } else {  // every element of the chunk
        const int rem = a.nElem - 64 * c;
        m = rem >= 64 ? ~0ull : (1ull << rem) - 1;
      }
      while (m) {
        const int b = 63 - __builtin_clzll(m);
        m &= ~(1ull << b);
        const int k = 64 * c + b;
        // an ellipse by its line alone (a line that misses it clips to zero;
        // the rays span the phantom, so the line test queues next to no pair
        // whose segment the clip then rejects)
        const bool may = active && (a.elems[k].type == PE_ELLIPSE
                                        ? line_may_hit_unit_circle(a.elems[k].p2o, xd, yd, xs, ys)
                                        : seg_may_hit_box(xd, yd, xs, ys, a.elems[k].lim));
        const unsigned long long hit = __ballot(may);
        if (!hit) continue;
        if (may) qp->pair[(enq + lanes_below(hit)) & (kQueue - 1)] = lane | (k << 6);
        if (lane == 0) {
          qp->vmask[nv & (kQueue - 1)] = hit;
          qp->vbase[nv & (kQueue - 1)] = enq;
        }
        nv++;
        enq += __popcll(hit);
        if (enq - done >= 64) flush(64);
      }
    }
    if (enq > done) flush(enq - done);
    sum += rsum;
    if (a.geom == GEOM_EQUIANGULAR) ang += s.aSampInc;
    else { xd += s.ddx2; yd += s.ddy2; }
  }
  if (active) {
    float* out = a.sino + static_cast<size_t>(v + a.storageOffset) * a.nDet;
    out[d] = static_cast<float>(sum / a.nSample);
  }
}

// ----------------------------------------------------- the short ray sum
//
// Only float(sum / nSample) of a ray is kept, so its chords are needed exactly
// only when the sum lies within its error of a float32 rounding boundary.
// This kernel sums short closed forms with bounds on their distance from the
// reference's chain and stores a ray whose two bounds round to one float32
// number; the others are deferred to raysum_rays_kernel, which runs the chain.
// The result is the reference's bit for bit either way.
//
// Ellipse: the chord is 2 sqrt(A - (det c)^2) / A per unit of attenuation, A =
// |M d|^2 for the ray's unit direction d and the linear map M onto the unit
// circle, c the signed distance of its centre from the ray: about 40
// instructions where the reference's clip takes an arc tangent, a sine, a
// cosine and four rotations.  With z = t^2 = 1 - (det c)^2 / A, t the half
// chord in the unit frame, against the reference's chain:
//   z < -1e-6: the line passes the ellipse by far more than any rounding; the
//     chain clips to zero;
//   z > edge: the line cuts the polygon that the bounding box is taken from,
//     so the box clip keeps it, and both chords are within
//     80 u (max / min semi-axis) (ray end + centre + semi-axis) (1 + 1 / t) of
//     the exact one (u = 2^-53).  The chain: 17 u T across (T the ends' size in
//     the unit frame, at most (ray end + centre) / min; the transform's own
//     rounding, the arc tangent's, sine's and cosine's and the rotation), hence
//     17 u T / t in the half chord, twice, 14 u T for rotating, moving and
//     mapping both ends back, all times the larger semi-axis; here 8 u of the
//     centre's distance and 6 u aspect in A, 34 u / t in all;
//   between: the ray is deferred.
// Rectangle: the line's parameters at the four sides, each off by a
// coordinate's error (64 u of the ends' size in the unit frame, both
// evaluations) over the direction's component, give an interval that holds
// the chord however the corners are decided; 80 u as above for mapping back.
// Both ends of the ray must lie outside the disc that holds these elements, on
// either side of it (the clip then replaces both), and T below 1e6 keeps the shares above far inside
// the margins on z and in the chain's own tolerances.  The sums add in the same
// order; their roundings are bounded by u times the elements times the sum of
// the sizes, twice.  A wave that meets another type of element is deferred to
// raysum_f64_kernel.
//
// What bounds it: FP64 VALU issue, two thirds of its cycles.  1440 views of 1024
// detectors over 64 ellipses and 4 rectangles: the chain for every ray took
// 452 us, this kernel takes 93 and raysum_rays_kernel 14 for the few rays that
// are deferred (calling the chain from this kernel instead: 388 us, for the
// registers and the lanes that wait).
__device__ __forceinline__ double rcp_f64(double x) {
  const double r = __builtin_amdgcn_rcp(x), e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// Element k's record, the same for the whole wave, through scalar loads.
__device__ __forceinline__ FastElem load_fast(const FastElem* table, int k) {
  typedef const __attribute__((address_space(4))) FastElem* Ptr;
  const Ptr p = (Ptr)(reinterpret_cast<unsigned long long>(table)) + __builtin_amdgcn_readfirstlane(k);
  FastElem f;
  f.m[0] = p->m[0]; f.m[1] = p->m[1]; f.m[2] = p->m[2]; f.m[3] = p->m[3];
  f.cx = p->cx; f.cy = p->cy; f.det2 = p->det2; f.att = p->att;
  f.kappa = p->kappa; f.edge = p->edge; f.kind = p->kind;
  return f;
}

__device__ __forceinline__ bool raysum_short(const RaysumArgs& a, const ViewSetup& s, int v, int d,
                                             const unsigned long long* masks, int nChunks, float* out) {
  const double4 w = walk_at(a.walk, a.nDet, v, d);
  const double xs = w.x, ys = w.y;
  double xd = w.z, yd = w.w, ang = w.z;
  double sum = 0.0, size = 0.0;
  float bound = 0.f;
  bool sure = true;
  for (unsigned i = 0; i < a.nSample; i++) {
    if (a.geom == GEOM_EQUIANGULAR) {
      double sa, ca;
      crm_sincos(ang, &sa, &ca);
      xd = a.centerDetLength * ca;
      yd = a.centerDetLength * sa;
    }
    const double ddx = xs - xd, ddy = ys - yd, L = sqrt(ddx * ddx + ddy * ddy);
    const double dx = ddx / L, dy = ddy / L;
    // the ends lie outside the disc, on either side of it
    const double fx = a.fastX - xd, fy = a.fastY - yd, sx = xs - a.fastX, sy = ys - a.fastY, R2 = a.fastR * a.fastR;
    const double foot = fx * dx + fy * dy;
    const double far = fmax(fabs(xd) + fabs(yd), fabs(xs) + fabs(ys)) + a.fastFar;
    sure = sure && foot > 0.0 && L > foot && fx * fx + fy * fy > R2 && sx * sx + sy * sy > R2 && far < 1e6 * a.fastMin;
    const float farf = static_cast<float>(far);
    const double k0 = xd * dy - yd * dx;
    float e = 0.f;
    double rsum = 0.0;
    // candidates newest first, the next one's record read ahead
    int c = nChunks;
    unsigned long long m = 0;
    auto next = [&]() -> int {
      while (!m) {
        if (c == 0) return -1;
        m = uniform_u64(masks[--c]);
      }
      const int b = 63 - __builtin_clzll(m);
      m &= ~(1ull << b);
      return 64 * c + b;
    };
    int kn = __builtin_amdgcn_readfirstlane(next());
    if (kn >= 0) {
      FastElem fn = load_fast(a.fastElems, kn);
      while (kn >= 0) {
        const FastElem f = fn;
        kn = __builtin_amdgcn_readfirstlane(next());
        if (kn >= 0) fn = load_fast(a.fastElems, kn);
        const double qx = fma(dx, f.m[0], dy * f.m[2]), qy = fma(dx, f.m[1], dy * f.m[3]);
        double chord = 0.0;
        if (f.kind == 1) {
          const double A = fma(qx, qx, qy * qy);
          const double cr = fma(f.cy, dx, fma(-f.cx, dy, k0));
          const double num = fma(-f.det2 * cr, cr, A);
          if (!__any(num > -1e-6 * A)) continue;  // no lane's line comes near
          const double inv = rcp_f64(A);
          const float z = static_cast<float>(num * inv);
          if (z > f.edge) {
            // sqrt(num) by the hardware's reciprocal root and two steps
            const double y = __builtin_amdgcn_rsq(num);
            double g = num * y, h = 0.5 * y;
            const double r1 = fma(-g, h, 0.5);
            g = fma(g, r1, g);
            h = fma(h, r1, h);
            g = fma(fma(-g, g, num), h, g);
            chord = g * inv * f.att;
            e = fmaf(f.kappa, __builtin_amdgcn_rsqf(z), e);
          } else if (!(z < -1e-6f)) {
            sure = false;
          }
        } else {
          const double px = fma(xd, f.m[0], fma(yd, f.m[2], f.cx)), py = fma(xd, f.m[1], fma(yd, f.m[3], f.cy));
          const double ix = rcp_f64(qx), iy = rcp_f64(qy);
          const double cx = -px * ix, cy = -py * iy, hx = fabs(ix), hy = fabs(iy);  // middles and half lengths
          const double err = static_cast<double>(f.edge * farf), gx = err * hx, gy = err * hy;
          const double in = fmin(cx + hx - gx, cy + hy - gy) - fmax(cx - hx + gx, cy - hy + gy);
          const double ou = fmin(cx + hx + gx, cy + hy + gy) - fmax(cx - hx - gx, cy - hy - gy);
          // a line along a side (or no number) is left to the chain
          sure = sure && ou < 1e300 && hx < 1e12 * hy && hy < 1e12 * hx;
          const double lo = fmax(in, 0.0), hi = fmax(ou, 0.0);
          chord = 0.5 * (lo + hi) * f.att;
          if (hi > 0.0) e += f.kappa + static_cast<float>(0.51 * (hi - lo) * fabs(f.att)) * __builtin_amdgcn_rcpf(farf);
        }
        rsum += chord;
        size += fabs(chord);
      }
    }
    sum += rsum;
    bound = fmaf(e, farf, bound);
    if (a.geom == GEOM_EQUIANGULAR) ang += s.aSampInc;
    else { xd += s.ddx2; yd += s.ddy2; }
  }
  const double E = 1.01 * static_cast<double>(bound) + 2.5 * 0x1p-53 * (a.nElem + 2.0 + a.nSample) * size;
  const float f0 = static_cast<float>((sum - E) / a.nSample), f1 = static_cast<float>((sum + E) / a.nSample);
  *out = f0;
  return sure & (__float_as_uint(f0) == __float_as_uint(f1)) & (f0 == f0);
}

// More unsure rays of a wave than this are cheaper 64 at a time, their pairs of
// ray and element packed (raysum_f64_kernel), than a wave each.
constexpr int kDeferRays = 8;

// One wave per block and item (a view, 64 detectors).  The middle of the
// detector comes first, over all views, its ends, whose rays meet few
// elements, last: the short items fill the end of the launch.
__global__ __launch_bounds__(64) void raysum_short_kernel(RaysumArgs a) {
  __shared__ unsigned long long masks[kCandChunks];
  const int blocks = (a.nDet + 63) / 64, nChunks = (a.nElem + 63) / 64;
  const int ring = blockIdx.x / a.nView, v = static_cast<int>(blockIdx.x) - ring * a.nView;
  const int d0 = 64 * (blocks / 2 + ((ring & 1) ? -((ring + 1) / 2) : ring / 2));
  const int d = d0 + static_cast<int>(threadIdx.x), d1 = min(d0 + 63, a.nDet - 1);
  const ViewSetup s = view_setup(a.ends[v], a.nDet, a.nSample, a.geom, a.angDetInc);
  wave_candidates(a, s, v, d0, d1, masks, nChunks);
  __syncthreads();
  // an element of another type among the candidates
  bool other = false;
  for (int c = 0; c < nChunks; c++) {
    const int k = 64 * c + static_cast<int>(threadIdx.x);
    other = other || (((uniform_u64(masks[c]) >> threadIdx.x) & 1) && a.fastElems[k].kind == 0);
  }
  if (__any(other)) {
    if (threadIdx.x == 0) a.items[atomicAdd(a.counter + 1, 1)] = make_int2(v, d0);
    return;
  }
  float f;
  const bool sure = raysum_short(a, s, v, min(d, a.nDet - 1), masks, nChunks, &f);
  if (sure && d < a.nDet) a.sino[static_cast<size_t>(v + a.storageOffset) * a.nDet + d] = f;
  const unsigned long long rest = __ballot(!sure && d < a.nDet);
  if (__popcll(rest) > kDeferRays && a.deferItems) {
    if (threadIdx.x == 0) a.items[atomicAdd(a.counter + 1, 1)] = make_int2(v, d0);
  } else if (rest) {
    int at = 0;
    if (threadIdx.x == 0) at = atomicAdd(a.counter + 2, __popcll(rest));
    at = __builtin_amdgcn_readfirstlane(at) + lanes_below(rest);
    if ((rest >> threadIdx.x) & 1) a.rays[at] = make_int2(v, d);
  }
}

// The deferred rays by the reference's chain, a wave per ray: lane k clips
// element 64 c + k, and the chords are added in the element order.  One chain's
// latency bounds it: a lane per ray would take an element's chain after the
// other.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void raysum_rays_kernel(RaysumArgs a) {
  const int nRays = a.counter[2], nChunks = (a.nElem + 63) / 64, lane = threadIdx.x;
  for (int r = blockIdx.x; r < nRays; r += gridDim.x) {
    const int2 at = a.rays[r];
    const int v = __builtin_amdgcn_readfirstlane(at.x), d = __builtin_amdgcn_readfirstlane(at.y);
    const ViewSetup s = view_setup(a.ends[v], a.nDet, a.nSample, a.geom, a.angDetInc);
    const double4 w = walk_at(a.walk, a.nDet, v, d);
    double xd = w.z, yd = w.w, ang = w.z, sum = 0.0;
    for (unsigned i = 0; i < a.nSample; i++) {
      if (a.geom == GEOM_EQUIANGULAR) {
        double sa, ca;
        crm_sincos(ang, &sa, &ca);
        xd = a.centerDetLength * ca;
        yd = a.centerDetLength * sa;
      }
      double rsum = 0.0;
      for (int c = nChunks - 1; c >= 0; c--) {
        const int k = 64 * c + lane;
        const bool may = k < a.nElem && (a.elems[k].type == PE_ELLIPSE
                                             ? line_may_hit_unit_circle(a.elems[k].p2o, xd, yd, w.x, w.y)
                                             : seg_may_hit_box(xd, yd, w.x, w.y, a.elems[k].lim));
        double chord = 0.0;
        if (may) chord = chord_ref(a.elems[k], xd, yd, w.x, w.y);
        unsigned long long m = __ballot(may);
        const unsigned long long bits = __builtin_bit_cast(unsigned long long, chord);
        while (m) {  // newest first
          const int b = 63 - __builtin_clzll(m);
          m &= ~(1ull << b);
          const unsigned hi = __builtin_amdgcn_readlane(static_cast<int>(bits >> 32), b);
          const unsigned lo = __builtin_amdgcn_readlane(static_cast<int>(bits), b);
          rsum += __builtin_bit_cast(double, (static_cast<unsigned long long>(hi) << 32) | lo);
        }
      }
      sum += rsum;
      if (a.geom == GEOM_EQUIANGULAR) ang += s.aSampInc;
      else { xd += s.ddx2; yd += s.ddy2; }
    }
    if (lane == 0) a.sino[static_cast<size_t>(v + a.storageOffset) * a.nDet + d] = static_cast<float>(sum / a.nSample);
  }
}

// A persistent wave per block takes items (view, 64 detectors; of those that
// raysum_short_kernel deferred, where it ran) from a counter until none is
// left: the rays' work differs widely (a ray through the phantom's middle meets
// many elements), and taking items as waves free up keeps every CU busy to the
// end.
__device__ __forceinline__ void raysum_items(const RaysumArgs& a, WaveQueue* q) {
  const int blocks = (a.nDet + 63) / 64, nItems = a.fast ? a.counter[1] : blocks * a.nView;
  const int nChunks = (a.nElem + 63) / 64;
  const bool cull = nChunks <= kCandChunks;
  __shared__ unsigned long long masks[kCandChunks];  // the wave's candidate masks
  while (true) {
    int item = 0;
    if (threadIdx.x == 0) item = atomicAdd(a.counter, 1);
    item = __builtin_amdgcn_readfirstlane(item);
    if (item >= nItems) break;
    int v = item / blocks, d0 = (item - v * blocks) * 64;
    if (a.fast) {
      const int2 r = a.items[item];
      v = __builtin_amdgcn_readfirstlane(r.x);
      d0 = __builtin_amdgcn_readfirstlane(r.y);
    }
    const int d = d0 + static_cast<int>(threadIdx.x), d1 = min(d0 + 63, a.nDet - 1);
    if (a.unitPulse) {  // scanner.cpp:475-478
      if (d < a.nDet) a.sino[static_cast<size_t>(v + a.storageOffset) * a.nDet + d] = d == a.nDet / 2 ? 1.f : 0.f;
      continue;
    }
    const ViewEnds e = a.ends[v];
    const ViewSetup s = view_setup(e, a.nDet, a.nSample, a.geom, a.angDetInc);
    if (cull) wave_candidates(a, s, v, d0, d1, masks, nChunks);
    raysum_ray(a, s, v, d, d < a.nDet, cull ? masks : nullptr, nChunks, q);
  }
}

// The FP64 path at 4 waves per SIMD: the clip chain's registers are capped
// at 128, the few it then keeps in scratch cost less than the latency a
// fourth wave hides.
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4, 8))) void raysum_f64_kernel(RaysumArgs a) {
  __shared__ WaveQueue q;
  raysum_items(a, &q);
}

// The closed-form chords, a few dozen operations each, one lane per ray over
// every element: culling costs them more than it saves.
__global__ __launch_bounds__(256) void raysum_closed_kernel(RaysumArgs a) {
  const int d = blockIdx.x * blockDim.x + threadIdx.x;
  const int v = blockIdx.y;
  if (d >= a.nDet) return;
  float* out = a.sino + static_cast<size_t>(v + a.storageOffset) * a.nDet;
  if (a.unitPulse) {  // scanner.cpp:475-478
    out[d] = d == a.nDet / 2 ? 1.f : 0.f;
    return;
  }
  const ViewSetup s = view_setup(a.ends[v], a.nDet, a.nSample, a.geom, a.angDetInc);
  const double4 w = walk_at(a.walk, a.nDet, v, d);
  const double xs = w.x, ys = w.y;
  double xd = w.z, yd = w.w, ang = w.z;
  double sum = 0.0;
  for (unsigned i = 0; i < a.nSample; i++) {
    if (a.geom == GEOM_EQUIANGULAR) {
      double sa, ca;
      crm_sincos(ang, &sa, &ca);
      xd = a.centerDetLength * ca;
      yd = a.centerDetLength * sa;
    }
    const double segLen = sqrt((xs - xd) * (xs - xd) + (ys - yd) * (ys - yd));
    double rsum = 0.0;
    for (int k = a.nElem - 1; k >= 0; k--) rsum += chord_closed(a.elems[k], xd, yd, xs, ys, segLen);
    sum += rsum;
    if (a.geom == GEOM_EQUIANGULAR) ang += s.aSampInc;
    else { xd += s.ddx2; yd += s.ddy2; }
  }
  out[d] = static_cast<float>(sum / a.nSample);
}

}  // namespace

int phantom_upload(PhantomPlan& p) {
  if (!p.dirty && p.d_elems.ptr) return CTSIM_OK;
  const size_t n = p.elems.size();
  CTSIM_CHECK(p.d_elems.reserve((n ? n : 1) * (sizeof(ElemGPU) + sizeof(FastElem))));
  if (n) {
    std::vector<unsigned char> all(n * (sizeof(ElemGPU) + sizeof(FastElem)));
    const std::vector<FastElem> fast = phantom_fast_elems(p);
    memcpy(all.data(), p.elems.data(), n * sizeof(ElemGPU));
    memcpy(all.data() + n * sizeof(ElemGPU), fast.data(), n * sizeof(FastElem));
    CTSIM_HIP(hipMemcpy(p.d_elems.ptr, all.data(), all.size(), hipMemcpyHostToDevice));
  }
  p.dirty = false;
  return CTSIM_OK;
}

int raysum_launch(ctsim_ctx* ctx, const ScannerPlan& s, PhantomPlan& p, int precision,
                  int iStartView, int iNumViews, int iOffsetView, int iStorageOffset,
                  float* d_sino, double* h_angles) {
  if (iNumViews <= 0) return CTSIM_OK;
  const hipStream_t st = ctx->stream;
  CTSIM_CHECK(phantom_upload(p));
  const size_t eb = static_cast<size_t>(iNumViews) * sizeof(ViewEnds);
  CTSIM_CHECK(ctx->stage.reserve(eb, st));
  ViewEnds* ends = static_cast<ViewEnds*>(ctx->stage.ptr);
  scanner_view_ends(s, iStartView, iNumViews, iOffsetView, ends);
  if (h_angles)
    for (int v = 0; v < iNumViews; v++) h_angles[v + iStorageOffset] = ends[v].viewAngle;
  CTSIM_CHECK(ctx->stage.upload(ctx->viewConsts, eb, st));
  // the walk, the ray-sum kernels' counters, what the short chord defers
  const size_t walkBytes = static_cast<size_t>(iNumViews) * walk_row(s.nDet) * sizeof(double4);
  const int items = ((s.nDet + 63) / 64) * iNumViews;
  const size_t rays = static_cast<size_t>(iNumViews) * s.nDet;
  // The short chord is for phantoms with an element that it knows and whose
  // size against the scan leaves its bound room (else every ray is deferred).
  const double rim = std::max({hypot(s.xs1, s.ys1), hypot(s.xs2, s.ys2), hypot(s.xd1, s.yd1), hypot(s.xd2, s.yd2),
                               s.centerDetLength});
  const bool fast = precision == CTSIM_PREC_F64 && !p.unitPulse && p.elems.size() <= 64 * kCandChunks &&
                    p.fastR > 0 && 1.5 * rim + p.fastFar < 1e6 * p.fastMin &&
                    raysum_short_pays(s, p, iNumViews, ctx->numCUs);
  // Whole items are deferred where other types are met or a ray may end in the
  // elements' disc.
  const bool deferItems = !p.fastOthers.empty() || !(std::min(s.focalLength, s.centerDetLength) >
                                                     1.001 * (hypot(p.fastX - s.xc, p.fastY - s.yc) + p.fastR));
  CTSIM_CHECK(ctx->scratch.reserve(walkBytes + 256 + (fast ? (items + rays) * sizeof(int2) : 0)));
  int* counter = reinterpret_cast<int*>(static_cast<unsigned char*>(ctx->scratch.ptr) + walkBytes);
  WalkArgs wa{ctx->viewConsts.as<ViewEnds>(), ctx->scratch.as<double4>(), counter, iNumViews, s.nDet,
              s.geom, s.nSample, s.angDetInc, s.angDetLen};
  hipLaunchKernelGGL(raysum_walk_kernel, dim3((iNumViews + kWalkViews - 1) / kWalkViews), dim3(64), 0, st, wa);
  CTSIM_HIP(hipGetLastError());
  int2* deferred = reinterpret_cast<int2*>(reinterpret_cast<unsigned char*>(counter) + 256);
  RaysumArgs ra{ctx->viewConsts.as<ViewEnds>(), ctx->scratch.as<double4>(), p.d_elems.as<ElemGPU>(),
                d_sino, counter, iNumViews, s.nDet, static_cast<int>(p.elems.size()), s.geom, iStorageOffset,
                s.nSample, s.angDetInc, s.centerDetLength, p.unitPulse ? 1 : 0,
                reinterpret_cast<const FastElem*>(p.d_elems.as<ElemGPU>() + p.elems.size()), deferred, deferred + items,
                fast ? 1 : 0, deferItems ? 1 : 0, p.fastX, p.fastY, p.fastR, p.fastMin, p.fastFar};
  if (precision == CTSIM_PREC_F64) {
    // persistent single-wave blocks, as many as are resident at once, no
    // more than the items
    auto resident = [&](auto kern, int n) {
      int perCU = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&perCU, reinterpret_cast<const void*>(kern), 64, 0) != hipSuccess ||
          perCU < 1)
        perCU = 8;
      return dim3(static_cast<unsigned>(std::min(n, ctx->numCUs * perCU)));
    };
    if (fast) {
      hipLaunchKernelGGL(raysum_short_kernel, dim3(items), dim3(64), 0, st, ra);
      CTSIM_HIP(hipGetLastError());
      hipLaunchKernelGGL(raysum_rays_kernel, resident(raysum_rays_kernel, items), dim3(64), 0, st, ra);
      CTSIM_HIP(hipGetLastError());
    }
    if (!fast || deferItems)
      hipLaunchKernelGGL(raysum_f64_kernel, resident(raysum_f64_kernel, items), dim3(64), 0, st, ra);
  } else {
    hipLaunchKernelGGL(raysum_closed_kernel, dim3((s.nDet + 255) / 256, iNumViews), dim3(256), 0, st, ra);
  }
  CTSIM_HIP(hipGetLastError());
  return CTSIM_OK;
}

}  // namespace ctsim

using namespace ctsim;

extern "C" {

int ctsim_phantom_create(ctsim_phantom** out, const char* builtinName) {
  if (!out) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_create: NULL argument");
  *out = nullptr;
  auto* p = new ctsim_phantom();
  if (builtinName && builtinName[0]) {
    const int rc = phantom_builtin(p->plan, builtinName);
    if (rc) { delete p; return rc; }
  }
  *out = p;
  return CTSIM_OK;
}

void ctsim_phantom_destroy(ctsim_phantom* p) { delete p; }

int ctsim_phantom_add_element(ctsim_phantom* p, const char* type, double cx, double cy, double u,
                              double v, double rotDeg, double atten) {
  if (!p) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_add_element: NULL phantom");
  return phantom_add(p->plan, type, cx, cy, u, v, rotDeg, atten);
}

int ctsim_phantom_extent(const ctsim_phantom* p, double* ext4) {
  if (!p || !ext4) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_extent: NULL argument");
  ext4[0] = p->plan.xmin; ext4[1] = p->plan.xmax; ext4[2] = p->plan.ymin; ext4[3] = p->plan.ymax;
  return static_cast<int>(p->plan.elems.size());
}

int ctsim_phantom_element(const ctsim_phantom* p, int index, double* out13) {
  if (!p || !out13) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_element: NULL argument");
  const int n = static_cast<int>(p->plan.elems.size());
  if (index < 0 || index >= n) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_element: index out of range");
  const int k = n - 1 - index;  // the reference's list is newest-first
  const ElemInfo& in = p->plan.infos[k];
  const ElemGPU& e = p->plan.elems[k];
  const double v[13] = {static_cast<double>(in.type), in.cx, in.cy, in.u, in.v, in.rotRad, in.atten,
                        e.lim[0], e.lim[1], e.lim[2], e.lim[3], static_cast<double>(in.nOutline),
                        in.rotDeg};
  for (int i = 0; i < 13; i++) out13[i] = v[i];
  return CTSIM_OK;
}

int ctsim_scanner_create(ctsim_scanner** out, const ctsim_phantom* phm, const char* geometry,
                         int nDet, int nView, int offsetView, int nSample, double rotLen,
                         double focalLengthRatio, double centerDetectorRatio, double viewRatio,
                         double scanRatio) {
  if (!out || !phm) return fail(CTSIM_ERR_INVALID, "ctsim_scanner_create: NULL argument");
  *out = nullptr;
  auto* s = new ctsim_scanner();
  const int rc = scanner_init(s->plan, phm->plan, geometry, nDet, nView, offsetView, nSample, rotLen,
                              focalLengthRatio, centerDetectorRatio, viewRatio, scanRatio);
  if (rc) { delete s; return rc; }
  *out = s;
  return CTSIM_OK;
}

void ctsim_scanner_destroy(ctsim_scanner* s) { delete s; }

int ctsim_scanner_info(const ctsim_scanner* sc, double* o) {
  if (!sc || !o) return fail(CTSIM_ERR_INVALID, "ctsim_scanner_info: NULL argument");
  const ScannerPlan& s = sc->plan;
  o[0] = s.detInc; o[1] = s.detStart; o[2] = s.rotInc; o[3] = s.viewDiameter;
  o[4] = s.focalLength; o[5] = s.sdl; o[6] = s.fanBeamAngle; o[7] = s.viewDiameter / kSqrt2;
  o[8] = s.detLen; o[9] = s.centerDetLength; o[10] = s.scanDiameter; o[11] = s.geom;
  return CTSIM_OK;
}

int ctsim_collect_projections(ctsim_ctx* ctx, const ctsim_scanner* sc, ctsim_phantom* phm,
                              int precision, int iStartView, int iNumViews, int iOffsetView,
                              int iStorageOffset, float* d_sino, double* h_angles) {
  if (!ctx || !sc || !phm || (iNumViews > 0 && !d_sino))
    return fail(CTSIM_ERR_INVALID, "ctsim_collect_projections: NULL argument");
  if (precision != CTSIM_PREC_F64 && precision != CTSIM_PREC_MIXED)
    return fail(CTSIM_ERR_INVALID, "ctsim_collect_projections: unknown precision");
  if (iNumViews < 0 || iStartView < 0 || iStorageOffset < 0)
    return fail(CTSIM_ERR_INVALID, "ctsim_collect_projections: negative view range");
  CTSIM_CHECK(ctx->activate());
  return raysum_launch(ctx, sc->plan, phm->plan, precision, iStartView, iNumViews, iOffsetView,
                       iStorageOffset, d_sino, h_angles);
}

}  // extern "C"
