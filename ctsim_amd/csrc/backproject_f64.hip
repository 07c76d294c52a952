// FP64 fan-beam and IntDiff backprojection for gfx950, linear and cubic
// interpolation.
//
// Fan beam.
// The reference adds every view's contribution to a float32 pixel,
// v = float(double(v) + c) (backprojectors.cpp:656-743), with c built from a
// cosine, a sine, an arc tangent and divisions, each rounded in its own
// order.  Only float(double(v) + c) is ever kept, so c is needed exactly only
// when it lies within its own error of a float32 rounding boundary.  This
// kernel evaluates c by a short FP64 formula with a bound e on its distance
// from the reference's c, forms float(double(v) + (c - e)) and
// float(double(v) + (c + e)), and keeps the result when the two have the
// same bits: rounding is monotone, so the reference's value lies between
// them.  A lane whose two values differ, or whose position lies outside the
// staged window, redoes its update with the reference's own operations
// (fan_exact).  The image is therefore the
// reference's bit for bit; the error bound decides only how often the slow
// path runs.
//
// What bounds it: FP64 VALU issue.  512^2 pixels, 1440 views of 1024 detectors,
// equiangular cubic: 395 lane instructions per update and 4.97 ms with the
// reference's operations for every update, about 57 and 0.90 ms here (of which
// 44 in the update itself, the rest staging and the views' constants; 0.57 of
// the VALU's issue slots, 0.34 of the LDS's); equilinear linear, 501 x 413
// pixels, 731 views: 1.88 and 0.38 ms.  Leaving out the slow path changes
// neither time.  Two or four pixels per lane measured 0.92 and more on the
// first against 0.90 (fewer waves per SIMD), one or two views at a time 1.03
// and 0.95.
#include <hip/hip_runtime.h>

#include <cmath>

#include "bp_plan.h"
#include "crmath.h"
#include "mixed_device.h"

#pragma clang fp contract(off)

namespace ctsim {
namespace {

constexpr int kBlock = 256;
constexpr int kTile = 16;            // a tile is 16 x 16 pixels, one per lane
constexpr int kMaxDeg = 14;          // largest arc-tangent degree (in t^2)
constexpr int kMeta = 128;           // views whose constants are found at a time
constexpr int kViews = 8;            // views staged at a time, two per wave
constexpr int kSeg = 59;             // intervals that 64 consecutive cells give
constexpr size_t kFanLds = 64 * 1024;  // largest staging buffer
using dev::xcd_tile;

// Bounds on the distance between the short formula and the reference's
// contribution (fan_bounds): per view and tile, the position within
//   kPos * ((rA * dA + dPerp) / L + extra) + posC      (cells, equiangular)
//   kPos * (rA * dA + dPerp) * L / fl^2 + posR |pos| + posC   (equilinear)
// where dA is half an ulp of theta - phi and L, fl the tile's nearest
// distances (its farthest L in the numerator); the value within dVal of the
// largest cell and of itself.
struct FanBounds {
  double kPos, rA, dPerp, extra, posR, posC, dVal, kappa, radius;
};

struct FanF64Args {
  int nx, ny, nDet, center, nView;
  int tilesY, W;
  double detInc, F, sdl;
  const double* r;
  const double* phi;
  const double* xs;
  const double* ys;
  const double* f;
  const ViewConstF64* vc;
  float* image;
  double endScale;            // fresh: factor applied to the finished sums
  int fresh;                  // sums start at zero instead of the image
  double posScale;            // equilinear: sdl / detInc
  double atan[kMaxDeg + 1];   // equiangular: series of atan(t)/t in t^2, over detInc
  FanBounds b;
};

// ------------------------------------------------------- the reference's own operations

__device__ __forceinline__ double cubic_row(const double* Y, int n, double x) {
  // CubicPolyInterpolator::interpolate, libctsupport/interpolator.cpp:36-75
  const int l = static_cast<int>(floor(x)) - 1;
  const int hi = l + 3;
  if (l < -1) return 0;
  if (l == -1) return Y[0] + x * (Y[1] - Y[0]);
  if (hi > n) return 0;
  if (hi == n) {
    const double frac = x - (l + 1);
    return Y[n - 2] + frac * (Y[n - 1] - Y[n - 2]);
  }
  const double xd0 = x - l, xd1 = x - (l + 1), xd2 = x - (l + 2), xd3 = x - (l + 3);
  const double oneSixth = (1. / 6.);
  double y = xd1 * xd2 * xd3 * -oneSixth * Y[l];
  y += xd0 * xd2 * xd3 * 0.5 * Y[l + 1];
  y += xd0 * xd1 * xd3 * -0.5 * Y[l + 2];
  y += xd0 * xd1 * xd2 * oneSixth * Y[l + 3];
  return y;
}

// One update of pixel value v by filtered row Y, BackprojectEquiangular /
// BackprojectEquilinear::BackprojectView, backprojectors.cpp:656-743.
template <int KIND, int INTERP>
__device__ __noinline__ float fan_exact(double r, double phi, double theta, double F, double sdl,
                                        double detInc, int center, int nDet, const double* Y, float v) {
  double s, co;
  crm_sincos(theta - phi, &s, &co);
  const double rc = r * co, rs = r * s;
  double pos, wgt;
  if constexpr (KIND == KIND_EQUIANGULAR) {
    const double fl = F + rs;
    pos = crm_atan(rc / fl) / detInc;
    wgt = fl * fl + (rc * rc);
  } else {
    const double U = (F + rs) / F;
    double dp = rc / U;
    dp *= sdl / F;
    pos = dp / detInc;
    wgt = U * U;
  }
  if constexpr (INTERP == INTERP_LINEAR) {
    const double pf = floor(pos);
    const int i = center + static_cast<int>(pf);
    const double frac = pos - pf;
    if (i < 0 || i >= nDet - 1) return v;
    return static_cast<float>(static_cast<double>(v) + (Y[i] + frac * (Y[i + 1] - Y[i])) / wgt);
  } else {
    const double d = center + pos;
    if (!(d >= 0 && d < nDet)) return v;
    return static_cast<float>(static_cast<double>(v) + cubic_row(Y, nDet, d) / wgt);
  }
}

// ------------------------------------------------------------------ the kernel

// The largest of non-negative numbers, less 2^-20 of it at most (which the
// bounds' quarter covers); infinite or no number if one of them is (fmax would
// drop the latter).  Their order is that of their high words.
__device__ __forceinline__ unsigned high_word(double x) {
  return static_cast<unsigned>(__builtin_bit_cast(unsigned long long, x) >> 32);
}
__device__ __forceinline__ double largest(double a, double b, double c, double d = 0.0) {
  const unsigned h = max(max(high_word(a), high_word(b)), max(high_word(c), high_word(d)));
  return __builtin_bit_cast(double, static_cast<unsigned long long>(h) << 32);
}

// Coefficients of detector interval i of row Y: on [i, i + 1) the
// interpolant is a0 + u (a1 + u (a2 + u a3)).  Outside the detector every
// coefficient is -0.0: adding -0.0 leaves any v as it is, and the bounds on a
// v of -0.0 then differ, so that fan_exact decides that one case.
// slope: a bound on |d/du| of this interval and its neighbours (the
// interpolant is continuous, so a position in doubt by less than a cell moves
// the value by no more than that times the doubt), plus kappa times the
// largest cell, which covers the coefficients' rounding; infinite beside the
// detector's ends, where the interpolant jumps to zero, and infinite or no
// number beside a cell that is, which a neighbouring interval may add.
template <int INTERP>
struct FanCell {  // the cubic's coefficients, or the line's two, and the slope bound
  static constexpr int kSlope = INTERP == INTERP_CUBIC ? 4 : 2;
  double v[INTERP == INTERP_CUBIC ? 6 : 4];
};

template <int INTERP>
__device__ __forceinline__ void fan_coef(double ym, double y0, double y1, double y2, double y3, double yp, int i,
                                         int n, double kappa, FanCell<INTERP>* cell) {
  const bool in = i >= 0 && i + 2 <= n;  // the intervals [0, n - 1)
  const double d0 = fabs(y1 - y0), d1 = fabs(y2 - y1), d2 = fabs(y3 - y2);
  const double big = largest(fabs(y0), fabs(y1), fabs(y2), fabs(y3));
  double slope;
  double2* out = reinterpret_cast<double2*>(cell->v);
  if constexpr (INTERP == INTERP_LINEAR) {
    out[0] = make_double2(in ? y1 : -0.0, in ? y2 - y1 : -0.0);
    slope = fma(kappa, big, largest(d0, d1, d2));
  } else {
    const double third = 1. / 3, sixth = 1. / 6;
    const bool interior = i > 0 && i + 2 < n;  // else (in) the first or last interval: a line
    const double b1 = fma(-third, y0, fma(-0.5, y1, fma(-sixth, y3, y2)));
    const double b2 = fma(0.5, y0 + y2, -y1);
    const double b3 = fma(sixth, y3 - y0, 0.5 * (y1 - y2));
    out[0] = make_double2(in ? y1 : -0.0, interior ? b1 : (in ? y2 - y1 : -0.0));
    out[1] = make_double2(interior ? b2 : (in ? 0.0 : -0.0), interior ? b3 : (in ? 0.0 : -0.0));
    // the cubic's slope between its middle cells is at most 1/3, 13/12 and 1/3
    // of its three steps' sizes (the end intervals' lines: 1 of theirs)
    const double dm = fabs(y0 - ym), dp = fabs(yp - y3), m = 1.0834;
    const double s0 = fma(m, d0, third * (dm + d1)), s1 = fma(m, d1, third * (d0 + d2)), s2 = fma(m, d2, third * (d1 + dp));
    slope = fma(kappa, big, largest(s0, s1, s2));
  }
  if ((i >= -1 && i <= 0) || (i >= n - 2 && i <= n - 1)) slope = __builtin_inf();
  if (i < -1 || i > n - 1) slope = 0.0;
  cell->v[FanCell<INTERP>::kSlope] = slope;
}

// The value of the next (dir > 0) or previous lane of the wave.
template <int DIR>
__device__ __forceinline__ double lane_step(double x) {
  constexpr int kCtrl = DIR > 0 ? 0x130 : 0x138;  // wave_shl:1, wave_shr:1
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(u), kCtrl, 0xf, 0xf, true);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(u >> 32), kCtrl, 0xf, 0xf, true);
  return __builtin_bit_cast(double, (static_cast<unsigned long long>(hi) << 32) | lo);
}

// 1 / m: the hardware's estimate (better than 2^-20) and one step of third
// order.
__device__ __forceinline__ double fan_rcp(double m) {
  const double r = __builtin_amdgcn_rcp(m);
  const double e = fma(-m, r, 1.0);
  return fma(r, fma(e, e, e), r);
}

// Window-relative position and weight of a pixel from rc = its offset across
// and fl = its distance along the view's direction through the tile.
template <int KIND, int DEG>
__device__ __forceinline__ void fan_pos(const FanF64Args& a, double rc, double fl, double p0, double& pos,
                                        double& wgt) {
  if constexpr (KIND == KIND_EQUIANGULAR) {
    // one reciprocal serves rc / fl and 1 / L^2
    const double L2 = fma(rc, rc, fl * fl);
    const double rr = fan_rcp(fl * L2);
    const double t = rc * (L2 * rr), z = t * t;
    double p = a.atan[DEG];
#pragma unroll
    for (int k = DEG - 1; k >= 0; k--) p = fma(p, z, a.atan[k]);
    pos = fma(t, p, p0);
    wgt = fl * rr;
  } else {
    const double q = fan_rcp(fl);
    pos = fma(rc * q, a.posScale, p0);
    const double u = a.F * q;
    wgt = u * u;
  }
}

// The kernel's arguments where they are used once in a long while: read again
// each time, instead of being held (and spilled) in scalar registers that the
// inner loop needs.
typedef const __attribute__((address_space(4))) FanF64Args* FanArgsPtr;
__device__ __forceinline__ FanArgsPtr cold_args() {
  FanArgsPtr p = (FanArgsPtr)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}

// One workgroup of 256 lanes owns a tile of 16 x 16 pixels, one per lane
// (lanes along iy), over all views (the float32 sums are in view order).
// Constants and windows are found for 128 views at a time, one view per
// lane, from the tile's corners.  Views are
// staged eight at a time: wave w loads the windows of views w and w + 4 into
// registers while the lanes interpolate the eight before (64 consecutive
// cells give 59 intervals, whose outer cells come from the neighbouring
// lanes), and writes their interval coefficients to LDS between two
// barriers.  Every lane then takes the views four at a time: four independent
// contributions, then the ordered adds.
//
// Equiangular: the view's axis is turned to the tile's centre (angle a0, of
// which cosine, sine and position are exact to an ulp), so that the pixels'
// angles from it are small and a short series of atan(t)/t serves; turning
// costs nothing per pixel, since the turned rc and fl are again affine in x
// and y.
template <int KIND, int INTERP, int DEG>
__global__ __launch_bounds__(kBlock) void bp_fan_f64_kernel(FanF64Args a) {
  using Cell = FanCell<INTERP>;
  extern __shared__ double2 s_dyn[];
  Cell* const s_c = reinterpret_cast<Cell*>(s_dyn);  // [kViews][W]
  __shared__ double s_v[kMeta][6];
  __shared__ int2 s_win[kMeta];  // first interval, intervals
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int ix0 = (tile / a.tilesY) * kTile, iy0 = (tile % a.tilesY) * kTile;
  const int ix = ix0 + t / kTile, iy = iy0 + t % kTile;
  const int cx1 = min(ix0 + kTile - 1, a.nx - 1), cy1 = min(iy0 + kTile - 1, a.ny - 1);
  const bool active = ix < a.nx && iy < a.ny;
  const int W = a.W;
  const double x = a.xs[min(ix, a.nx - 1)], y = a.ys[min(iy, a.ny - 1)];
  const size_t pix = static_cast<size_t>(ix) * a.ny + iy;
  float v = active && !a.fresh ? a.image[pix] : 0.f;

  // the cells of this wave's two views of the eight at view g (zero outside
  // the detector, and for views beyond nb)
  double raw[2][2];
  int vb = 0, nb = 0;
  auto load = [&](int view, int first, int j0) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double*>(a.f + static_cast<size_t>(view) * a.nDet), 0, a.nDet * 8, 0x00020000);
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (first + j0 - 2 + lane) * 8, 0, 0));
  };
  auto window = [&](int v) {
    const int2 w = s_win[v];
    return make_int2(__builtin_amdgcn_readfirstlane(w.x), __builtin_amdgcn_readfirstlane(w.y));
  };
  auto fetch = [&](int g) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int v = g + wave + 4 * q;
      if (v >= nb) break;
      const int2 w = window(v);
      raw[q][0] = load(vb + v, w.x, 0);
      if (w.y > kSeg) raw[q][1] = load(vb + v, w.x, kSeg);
    }
  };
  auto place = [&](int g) {
#pragma unroll
    for (int q = 0; q < 2; q++) {
      const int v = g + wave + 4 * q;
      if (v >= nb) break;
      const int2 w = window(v);
      for (int j0 = 0; j0 < w.y; j0 += kSeg) {
        const double y1 = j0 == 0 ? raw[q][0] : (j0 == kSeg ? raw[q][1] : load(vb + v, w.x, j0));
        const double y2 = lane_step<1>(y1), y3 = lane_step<1>(y2), yp = lane_step<1>(y3);
        const double y0 = lane_step<-1>(y1), ym = lane_step<-1>(y0);
        const int j = j0 + lane - 2;
        if (lane >= 2 && lane < kSeg + 2 && j < w.y)
          fan_coef<INTERP>(ym, y0, y1, y2, y3, yp, w.x + j, a.nDet, a.b.kappa, s_c + (v - g) * W + j);
      }
    }
  };

  for (vb = 0; vb < a.nView; vb += kMeta) {
    nb = min(kMeta, a.nView - vb);
    if (t < nb) {
      const FanArgsPtr ca = cold_args();
      const ViewConstF64 c = ca->vc[vb + t];
      const double xa = ca->xs[ix0], xb = ca->xs[cx1], ya = ca->ys[iy0], yb = ca->ys[cy1];
      double ct = c.a, st = c.b, Fs = 0.0, Fc = ca->F, base = ca->center;
      const double xm = 0.5 * (xa + xb), ym = 0.5 * (ya + yb);
      if constexpr (KIND == KIND_EQUIANGULAR) {
        const double a0 = crm_atan(fma(xm, ct, ym * st) / (ca->F + fma(xm, st, -(ym * ct))));
        double sa, co;
        crm_sincos(a0, &sa, &co);
        const double ct0 = ct, st0 = st;
        ct = fma(ct0, co, -(st0 * sa));
        st = fma(st0, co, ct0 * sa);
        Fs = -ca->F * sa;
        Fc = ca->F * co;
        base += a0 / ca->detInc;
      }
      double pmin = 1e300, pmax = -1e300;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const double cx = (q & 1) ? xb : xa, cy = (q & 2) ? yb : ya;
        double p, w;
        fan_pos<KIND, DEG>(a, fma(cy, st, fma(cx, ct, Fs)), fma(-cy, ct, fma(cx, st, Fc)), base, p, w);
        pmin = fmin(pmin, p);
        pmax = fmax(pmax, p);
      }
      // this view's bound: dA is half an ulp of the largest |theta - phi|
      const double dA = ldexp(0x1p-53, __builtin_amdgcn_frexp_exp(fabs(c.theta) + 3.15) - 1);
      const double flm = fma(-ym, ct, fma(xm, st, Fc)), rcm = fma(ym, st, fma(xm, ct, Fs));
      const double L = sqrt(fma(flm, flm, rcm * rcm));
      const double perp = fma(ca->b.rA, dA, ca->b.dPerp);
      if constexpr (KIND == KIND_EQUIANGULAR) {
        s_v[t][5] = fma(ca->b.kPos, perp / (L - ca->b.radius) + ca->b.extra, ca->b.posC);
      } else {
        const double fl = flm - ca->b.radius;
        s_v[t][5] = fma(ca->b.kPos, perp * (L + ca->b.radius) / (fl * fl),
                        fma(ca->b.posR, fmax(fabs(pmin - base), fabs(pmax - base)), ca->b.posC));
      }
      // positions that are no numbers stage anything: every pixel then fails its tests
      if (!(pmin > -1e9 && pmin < 1e9)) pmin = 0;
      const int lo = static_cast<int>(floor(pmin)) - 2;
      s_win[t] = make_int2(lo, pmax < 1e9 ? min(static_cast<int>(floor(pmax)) + 3 - lo, W) : W);
      s_v[t][0] = ct;
      s_v[t][1] = st;
      s_v[t][2] = Fs;
      s_v[t][3] = Fc;
      s_v[t][4] = base - lo;
    }
    // N views from view vv of the eight at v0 on
    auto step = [&](int v0, int vv, auto count) {
      constexpr int N = decltype(count)::value;
      double lo[N], hi[N], w[N];
      bool in[N], ok = true;
#pragma unroll
      for (int n = 0; n < N; n++) {
        const double* c = s_v[v0 + vv + n];
        double pos;
        fan_pos<KIND, DEG>(a, fma(y, c[1], fma(x, c[0], c[2])), fma(-y, c[0], fma(x, c[1], c[3])), c[4], pos, w[n]);
        const double fr = __builtin_amdgcn_fract(pos);
        const int cell = static_cast<int>(pos);
        const int cl = min(max(cell, 1), W - 1);  // (a position within the window: unchanged)
        const Cell& q = s_c[(vv + n) * W + cl];
        const double2* k = reinterpret_cast<const double2*>(q.v);
        double val;
        if constexpr (INTERP == INTERP_CUBIC) val = fma(fr, fma(fr, fma(fr, k[1].y, k[1].x), k[0].y), k[0].x);
        else val = fma(fr, k[0].y, k[0].x);
        const double e = fma(c[5], q.v[Cell::kSlope], a.b.dVal * fabs(val));
        in[n] = cell == cl;
        lo[n] = val - e;
        hi[n] = val + e;
      }
      // the float32 results of the two bounds: the same bits, and a number
      auto sure = [&](int n, float f0) {
        const float f1 = static_cast<float>(fma(w[n], hi[n], static_cast<double>(v)));
        return in[n] & (__float_as_uint(f0) == __float_as_uint(f1)) & (f0 == f0);
      };
      const float vs = v;
#pragma unroll
      for (int n = 0; n < N; n++) {
        const float f0 = static_cast<float>(fma(w[n], lo[n], static_cast<double>(v)));
        ok = ok & sure(n, f0);
        v = f0;
      }
      if (__builtin_expect(!ok & active, 0)) {  // redo the updates in order, those in doubt by the reference
        v = vs;
#pragma unroll
        for (int n = 0; n < N; n++) {
          const int view = vb + v0 + vv + n;
          const float f0 = static_cast<float>(fma(w[n], lo[n], static_cast<double>(v)));
          if (sure(n, f0)) {
            v = f0;
          } else {
            const FanArgsPtr ca = cold_args();
            v = fan_exact<KIND, INTERP>(ca->r[pix], ca->phi[pix], ca->vc[view].theta, ca->F, ca->sdl, ca->detInc,
                                        ca->center, ca->nDet, ca->f + static_cast<size_t>(view) * ca->nDet, v);
          }
        }
      }
    };
    __syncthreads();  // the constants are there
    fetch(0);
    for (int v0 = 0; v0 < nb; v0 += kViews) {
      const int nv = min(kViews, nb - v0);
      place(v0);
      __syncthreads();
      if (v0 + kViews < nb) fetch(v0 + kViews);  // in flight during the interpolation below
      int vv = 0;
      for (; vv + 4 <= nv; vv += 4) step(v0, vv, std::integral_constant<int, 4>{});
      for (; vv < nv; vv++) step(v0, vv, std::integral_constant<int, 1>{});
      __syncthreads();  // every lane is done reading
    }
  }
  if (active) {
    const FanArgsPtr ca = cold_args();
    ca->image[pix] = ca->fresh ? static_cast<float>(static_cast<double>(v) * ca->endScale) : v;
  }
}

template <int KIND, int INTERP, int DEG>
void launch_fan(const FanF64Args& a, int grid, size_t lds, hipStream_t s) {
  hipLaunchKernelGGL((bp_fan_f64_kernel<KIND, INTERP, DEG>), dim3(grid), dim3(kBlock), lds, s, a);
}

template <int INTERP>
void launch_fan_kind(const BpPlan& p, int deg, const FanF64Args& a, int grid, size_t lds, hipStream_t s) {
  if (p.kind == KIND_EQUILINEAR) launch_fan<KIND_EQUILINEAR, INTERP, 0>(a, grid, lds, s);
  else if (deg == 5) launch_fan<KIND_EQUIANGULAR, INTERP, 5>(a, grid, lds, s);
  else if (deg == 8) launch_fan<KIND_EQUIANGULAR, INTERP, 8>(a, grid, lds, s);
  else launch_fan<KIND_EQUIANGULAR, INTERP, kMaxDeg>(a, grid, lds, s);
}

// ------------------------------------------------------------------ IntDiff

// BackprojectIntDiff (backprojectors.cpp:579-653) walks the image in 32.32
// fixed point.  Every such position is a whole multiple of 2^-32 and, below
// 2^20 cells, an FP64 number: the positions are formed exactly in FP64, the
// interval and the fraction are the fixed-point ones, and scaling the slope by
// 2^-32 and the remainder by 2^32, as the reference does, changes no rounding.
// Linear interpolation then does the reference's own two operations; cubic
// interpolation evaluates the interval's polynomial, within kCubicRound of the
// largest cell of the reference's Lagrange sum, and decides the float32 sum as
// the fan-beam kernel does.  Outside the detector the linear coefficients are
// -0.0, which leaves any v as it is (the reference skips the sample), the
// cubic ones 0.0, which the reference adds.
//
// What bounds it: FP64 VALU issue.  2048^2 pixels, 2880 views, linear: 37.4
// lane instructions per update and 15.1 ms with the fixed-point walk of one
// pixel per lane, about 12 and 4.5 ms here (56 cycles per wave and update, 12
// instructions at the 4.7 cycles that an FP64 instruction takes on this chip);
// 256^2, 320 views: 184 us and 27.
struct IdiffArgs {
  int nx, ny, nDet, nView;
  int tilesY, W, views, half;  // views: staged at a time; half: 32 lanes stage a window
  int fresh;                   // as in FanF64Args
  double endScale;
  const double* f;
  const ViewConstF64* vc;
  float* image;
};

// the reference's Lagrange sum and the staged polynomial (40 u, as in
// fan_bounds), and a quarter more
constexpr double kCubicRound = 1.25 * 40 * 0x1p-53;

template <int INTERP>
struct IdiffCell {  // the line's value and slope, or the cubic's coefficients and rounding bound
  double v[INTERP == INTERP_CUBIC ? 6 : 2];
};

template <int INTERP>
__device__ __forceinline__ void idiff_coef(double y0, double y1, double y2, double y3, int i, int n,
                                           IdiffCell<INTERP>* cell) {
  double2* out = reinterpret_cast<double2*>(cell->v);
  if constexpr (INTERP == INTERP_LINEAR) {
    const bool in = i >= 0 && i < n;  // the last cell's value is held
    out[0] = make_double2(in ? y1 : -0.0, in ? (i < n - 1 ? y2 - y1 : 0.0) : -0.0);
  } else {
    const double third = 1. / 3, sixth = 1. / 6;
    const bool in = i >= 0 && i + 2 <= n, interior = i > 0 && i + 2 < n;  // else (in) the end intervals: a line
    const double b1 = fma(-third, y0, fma(-0.5, y1, fma(-sixth, y3, y2)));
    const double b2 = fma(0.5, y0 + y2, -y1);
    const double b3 = fma(sixth, y3 - y0, 0.5 * (y1 - y2));
    const double big = fmax(fmax(fabs(y0), fabs(y1)), fmax(fabs(y2), fabs(y3)));
    out[0] = make_double2(in ? y1 : 0.0, interior ? b1 : (in ? y2 - y1 : 0.0));
    out[1] = make_double2(interior ? b2 : 0.0, interior ? b3 : 0.0);
    cell->v[4] = in ? kCubicRound * big : 0.0;
  }
}

__device__ __noinline__ float idiff_cubic_exact(const double* Y, int n, double x, float v) {
  return static_cast<float>(static_cast<double>(v) + cubic_row(Y, n, x));
}

// One workgroup of 256 lanes owns a tile of (256 / LY) columns x LY P rows,
// lane (cx, ly) the rows P ly ... P ly + P - 1 of its column, over all views
// in order.  Windows are found for 128 views at a time and staged a.views at
// a time, loaded into registers while the views before are interpolated (64
// lanes a window, or 32 where it is short).  Every lane takes the views U at
// a time.
template <int INTERP, int LY, int P, int U>
__global__ __launch_bounds__(kBlock) void bp_idiff_f64_kernel(IdiffArgs a) {
  using Cell = IdiffCell<INTERP>;
  extern __shared__ double2 s_dyn[];
  Cell* const s_c = reinterpret_cast<Cell*>(s_dyn);  // [views][W]
  __shared__ double s_v[kMeta][4];  // position of the tile's first pixel in the window, steps along x and y
  __shared__ int2 s_win[kMeta];     // first interval, intervals
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  constexpr int kTx = kBlock / LY, kTy = LY * P;
  const int ix0 = (tile / a.tilesY) * kTx, iy0 = (tile % a.tilesY) * kTy;
  const int ix = ix0 + t / LY, iyb = iy0 + (t % LY) * P;
  const int cx1 = min(ix0 + kTx - 1, a.nx - 1), cy1 = min(iy0 + kTy - 1, a.ny - 1);
  const int W = a.W;
  const double cx = t / LY, cy = (t % LY) * P;
  const size_t pix = static_cast<size_t>(ix) * a.ny + iyb;
  float v[P];
#pragma unroll
  for (int k = 0; k < P; k++) v[k] = !a.fresh && ix < a.nx && iyb + k < a.ny ? a.image[pix + k] : 0.f;

  // staging: `group` lanes take one window, 4 or 8 windows a pass; cells gl - 1
  // + j0 of the window, of which the inner ones give intervals
  const int group = a.half ? 32 : 64, gl = lane & (group - 1), inner = group - 3;
  const int perPass = a.half ? 8 : 4, mine = a.half ? 2 * wave + (lane >> 5) : wave;
  double raw[4];
  int vb = 0, nb = 0;
  auto load = [&](int view, int cell) {
    return a.f[static_cast<size_t>(view) * a.nDet + min(max(cell, 0), a.nDet - 1)];
  };
  auto fetch = [&](int g) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int u = q * perPass + mine;
      if (u < a.views && g + u < nb) raw[q] = load(vb + g + u, s_win[g + u].x + gl - 1);
    }
  };
  auto place = [&](int g) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int u = q * perPass + mine;
      if (q * perPass >= a.views) break;
      const bool have = u < a.views && g + u < nb;
      const int2 w = s_win[have ? g + u : g];
      // (the loop's bound is the wave's: with 32 lanes a window, one round)
      for (int j0 = 0; j0 < W; j0 += inner) {
        const int j = j0 + gl - 1;
        const double y1 = j0 == 0 ? raw[q] : load(vb + (have ? g + u : g), w.x + j);
        const double y2 = lane_step<1>(y1), y3 = lane_step<1>(y2), y0 = lane_step<-1>(y1);
        if (have && gl >= 1 && gl <= inner && j < w.y) idiff_coef<INTERP>(y0, y1, y2, y3, w.x + j, a.nDet, s_c + u * W + j);
      }
    }
  };
  // N views from view vv of those staged at v0 on
  auto step = [&](int v0, int vv, auto count) {
    constexpr int N = decltype(count)::value;
    double pos[N][P], val[N][P], e[N][P];
#pragma unroll
    for (int n = 0; n < N; n++) {
      const double* c = s_v[v0 + vv + n];
      pos[n][0] = fma(cx, c[1], fma(cy, c[2], c[0]));  // exact, and so are the steps
#pragma unroll
      for (int k = 1; k < P; k++) pos[n][k] = pos[n][k - 1] + c[2];
#pragma unroll
      for (int k = 0; k < P; k++) {
        const double fr = __builtin_amdgcn_fract(pos[n][k]);
        const int cell = min(max(static_cast<int>(pos[n][k]), 0), W - 1);  // (a pixel's: unchanged)
        const Cell& q = s_c[(vv + n) * W + cell];
        const double2* h = reinterpret_cast<const double2*>(q.v);
        if constexpr (INTERP == INTERP_LINEAR) {
          val[n][k] = h[0].x + fr * h[0].y;
        } else {
          val[n][k] = fma(fr, fma(fr, fma(fr, h[1].y, h[1].x), h[0].y), h[0].x);
          e[n][k] = q.v[4];
        }
      }
    }
    if constexpr (INTERP == INTERP_LINEAR) {
#pragma unroll
      for (int n = 0; n < N; n++)
#pragma unroll
        for (int k = 0; k < P; k++) v[k] = static_cast<float>(static_cast<double>(v[k]) + val[n][k]);
    } else {
#pragma unroll
      for (int n = 0; n < N; n++) {
#pragma unroll
        for (int k = 0; k < P; k++) {
          const double vd = static_cast<double>(v[k]);
          const float f0 = static_cast<float>(vd + (val[n][k] - e[n][k])), f1 = static_cast<float>(vd + (val[n][k] + e[n][k]));
          const bool sure = (__float_as_uint(f0) == __float_as_uint(f1)) & (f0 == f0);
          if (__builtin_expect(!sure, 0)) {
            const int view = vb + v0 + vv + n;
            v[k] = idiff_cubic_exact(a.f + static_cast<size_t>(view) * a.nDet, a.nDet, pos[n][k] + s_win[v0 + vv + n].x, v[k]);
          } else {
            v[k] = f0;
          }
        }
      }
    }
  };

  for (vb = 0; vb < a.nView; vb += kMeta) {
    nb = min(kMeta, a.nView - vb);
    if (t < nb) {
      const ViewConstF64 c = a.vc[vb + t];
      long long dx, dy, cs;
      __builtin_memcpy(&dx, &c.a, 8);
      __builtin_memcpy(&dy, &c.b, 8);
      __builtin_memcpy(&cs, &c.c, 8);
      const long long p0 = cs + ix0 * dx + iy0 * dy, p1 = cs + cx1 * dx + iy0 * dy;
      const long long p2 = cs + ix0 * dx + cy1 * dy, p3 = cs + cx1 * dx + cy1 * dy;
      const int lo = static_cast<int>(min(min(p0, p1), min(p2, p3)) >> 32);
      const int hi = static_cast<int>(max(max(p0, p1), max(p2, p3)) >> 32);
      s_win[t] = make_int2(lo, min(hi + 1 - lo, W));
      s_v[t][0] = static_cast<double>(p0 - (static_cast<long long>(lo) << 32)) * 0x1p-32;
      s_v[t][1] = static_cast<double>(dx) * 0x1p-32;
      s_v[t][2] = static_cast<double>(dy) * 0x1p-32;
    }
    __syncthreads();  // the windows are there
    fetch(0);
    for (int v0 = 0; v0 < nb; v0 += a.views) {
      const int nv = min(a.views, nb - v0);
      place(v0);
      __syncthreads();
      if (v0 + a.views < nb) fetch(v0 + a.views);  // in flight during the interpolation below
      int vv = 0;
      for (; vv + U <= nv; vv += U) step(v0, vv, std::integral_constant<int, U>{});
      for (; vv < nv; vv++) step(v0, vv, std::integral_constant<int, 1>{});
      __syncthreads();  // every lane is done reading
    }
  }
#pragma unroll
  for (int k = 0; k < P; k++)
    if (ix < a.nx && iyb + k < a.ny)
      a.image[pix + k] = a.fresh ? static_cast<float>(static_cast<double>(v[k]) * a.endScale) : v[k];
}

// Cells of a window of tileX x tileY pixels, exactly: the positions of a
// tile span at most the steps times its sides, and one cell for the ends.
int idiff_window(const BpPlan& p, int tileX, int tileY) {
  const double sx = (tileX - 1) * fabs(p.xInc) / p.detInc, sy = (tileY - 1) * fabs(p.yInc) / p.detInc;
  const double w = ceil(sqrt(sx * sx + sy * sy) * (1 + 1e-9) + 1e-3) + 2;
  return w < 4096 ? static_cast<int>(w) : 0;
}

size_t idiff_cell(const BpPlan& p) {
  return p.interp == INTERP_CUBIC ? sizeof(IdiffCell<INTERP_CUBIC>) : sizeof(IdiffCell<INTERP_LINEAR>);
}

// Largest distance of a pixel from the origin.
double pixel_radius(const BpPlan& p) {
  const double rx = fmax(fabs(p.xMin), fabs(p.xMax)), ry = fmax(fabs(p.yMin), fabs(p.yMax));
  return sqrt(rx * rx + ry * ry);
}

// Sine of the largest angle between the axis to a tile's centre and one of
// its pixels: a point at distance h from the axis' target subtends at most
// asin(h / L).
double tile_sine(const BpPlan& p, double* radius) {
  const double hx = 0.5 * (kTile - 1) * fabs(p.xInc), hy = 0.5 * (kTile - 1) * fabs(p.yInc);
  const double h = sqrt(hx * hx + hy * hy);
  if (radius) *radius = h;
  return h / (p.F - pixel_radius(p));
}

// Degree of the arc-tangent series: the first term left out is below 2^-56
// (0: none is).
int atan_degree(const BpPlan& p) {
  const double sn = tile_sine(p, nullptr);
  if (!(sn < 0.5)) return 0;
  const double z = sn * sn / (1 - sn * sn);
  for (int d : {5, 8, kMaxDeg})
    if (sqrt(z) * pow(z, d + 1) / (2 * d + 3) < 0x1p-56) return d;
  return 0;
}

// Staging bytes of windows of W intervals.
size_t fan_lds(int W, bool cubic) {
  return static_cast<size_t>(kViews) * W * (cubic ? sizeof(FanCell<INTERP_CUBIC>) : sizeof(FanCell<INTERP_LINEAR>));
}

// Whether a tile's windows can be staged and its views turned.
bool fan_tile_ok(const BpPlan& p) {
  const int W = bp_window_bound(p, kTile, kTile);
  return W > 0 && fan_lds(W, p.interp == INTERP_CUBIC) <= kFanLds &&
         (p.kind == KIND_EQUILINEAR || atan_degree(p) > 0);
}

// Half an ulp of the numbers up to x in size.
double half_ulp(double x) { return 0x1p-53 * exp2(floor(log2(x))); }

// The bounds of FanBounds, from the roundings of both evaluations in units of
// u = 2^-53 (half an ulp of 1, the relative rounding of one operation).  R is
// the largest pixel radius; (rc, fl) the pixel's offset across the view's axis
// and its distance along it.
//   dPerp, what moves the pixel across its own ray (r per unit of radius):
//     reference   cos, sin rounded to u / 2 each (0.71 r), the two products
//                 (1 r), F + rs, which lies along the axis: (F + R) R / F;
//     both        x, y stand for r cos phi, r sin phi: phi's error is at most
//                 0.55 ulp of pi (2.2 r), r's three roundings 2 r: 3 r;
//     here        the view's cosine and sine 0.55 u each (0.78 r).
//       equiangular: turning them doubles the inputs' error and adds two
//                 roundings each (2.9 r in all); F's turned part across the
//                 axis 2 R; the first fused step 1.5 R, the second is small;
//                 errors of fl (F's turned part and two steps, 4 (F + R) +
//                 3 R) count by the tile's sine.
//       equilinear: two fused steps each, across 2.5 R, along 2 (F + R) R / F.
//   rA dA, the reference's rounding of theta - phi at radius R.
//   extra, the angle (equiangular): the reference's quotient 0.5 and arc
//     tangent 0.5, here the quotient, the series and its left-out term 0.3
//     and 10 of the tile's sine.
//   posC, posR, the position: half an ulp for each rounding of a whole
//     position (nDet) or one counted from the centre (half of it); the
//     products and quotients of the equilinear position 9 u of it.
//   dVal: the weight moves by 2 D / L, D the whole displacement of (rc, fl)
//     (the reference's 2 R and dA R, F + rs; here 6 R, 6 R, 3 F, 3 (F + R)),
//     the reciprocal, the quotients and the products by 24; a cubic's
//     coefficients, Horner steps and the reference's Lagrange sum by 40 of
//     the largest of the four cells (kappa, as a share of the least
//     position bound, since it is multiplied by the position bound).
// A quarter is added for the higher orders left out.
void fan_bounds(const BpPlan& p, int W, FanBounds& b) {
  const double u = 0x1p-53, R = pixel_radius(p), F = p.F, L = F - R, sinMax = R / F;
  const double sn = tile_sine(p, &b.radius);
  const bool cubic = p.interp == INTERP_CUBIC;
  const double whole = half_ulp(p.nDet), side = half_ulp(0.5 * p.nDet + 2);
  b.rA = R;
  if (p.kind == KIND_EQUIANGULAR) {
    b.dPerp = u * (R * (1.71 + 3 + 2.9 + 3.5) + sinMax * (F + R) + sn * (4 * (F + R) + 3 * R));
    b.extra = u * (1.3 + 10 * sn);
    b.kPos = 1.25 / p.detInc;
    b.posR = 0;
    b.posC = 1.25 * (2 * side + 2 * whole + 4 * W * u);
  } else {
    b.dPerp = u * (R * (1.71 + 3 + 0.78 + 2.5) + 3 * sinMax * (F + R));
    b.extra = 0;
    b.kPos = 1.25 * p.sdl / p.detInc;
    b.posR = 1.25 * 9 * u;
    b.posC = 1.25 * (whole + 2 * W * u);
  }
  const double D = R * (16 + 15) + 4 * (F + R) + 3 * F;
  b.dVal = 1.25 * u * (2 * D / L + 24 + 4);
  b.kappa = 1.25 * (cubic ? 40 : 4) * u / b.posC;
}

}  // namespace

// The rule of the dispatch: everything the bounds and the staging cover goes
// here, since the short formula is faster at every size measured (a 24^2 image
// as well as 2048^2); the general kernel keeps what is left: a source near or
// inside the image, windows of more cells than LDS holds, angles beyond 28.
bool bp_fan_f64_ok(const BpPlan& p, double maxAngle) {
  if (p.kind != KIND_EQUIANGULAR && p.kind != KIND_EQUILINEAR) return false;
  if (p.interp == INTERP_NEAREST) return false;
  // a source well outside the image, and angles of a few turns (16 u in the
  // bounds is half an ulp of theta - phi below 32)
  return p.F > 1.05 * pixel_radius(p) && p.detInc > 0 && p.sdl > 0 && maxAngle < 28.0 && fan_tile_ok(p);
}

int bp_fan_f64_launch(ctsim_ctx* ctx, const BpPlan& p, const double* d_filtered, const ViewConstF64* d_vc,
                      int nView, float* d_image, bool fresh) {
  const bool cubic = p.interp == INTERP_CUBIC, equi = p.kind == KIND_EQUIANGULAR;
  FanF64Args a{};
  a.nx = p.nx; a.ny = p.ny; a.nDet = p.nDet; a.center = p.iDetCenter; a.nView = nView;
  a.tilesY = (p.ny + kTile - 1) / kTile;
  const int grid = (p.nx + kTile - 1) / kTile * a.tilesY;
  a.W = bp_window_bound(p, kTile, kTile);
  const size_t lds = fan_lds(a.W, cubic);
  a.detInc = p.detInc; a.F = p.F; a.sdl = p.sdl;
  const size_t n = p.r.size();
  a.r = p.d_rphi.as<double>();
  a.phi = a.r + n;
  a.xs = a.r + 2 * n;
  a.ys = a.xs + p.nx;
  a.f = d_filtered; a.vc = d_vc; a.image = d_image;
  a.fresh = fresh; a.endScale = p.rotScale;
  const int deg = equi ? atan_degree(p) : 0;
  for (int k = 0; k <= deg; k++) a.atan[k] = (k & 1 ? -1.0 : 1.0) / ((2 * k + 1) * p.detInc);
  a.posScale = p.sdl / p.detInc;
  fan_bounds(p, a.W, a.b);
  ctx->prof_begin();
  if (cubic) launch_fan_kind<INTERP_CUBIC>(p, deg, a, grid, lds, ctx->stream);
  else launch_fan_kind<INTERP_LINEAR>(p, deg, a, grid, lds, ctx->stream);
  ctx->prof_end();
  CTSIM_HIP(hipGetLastError());
  return CTSIM_OK;
}

// The IntDiff kernel: positions below 2^20 cells (exact in FP64) and windows
// that fit LDS four views at a time.
bool bp_idiff_f64_ok(const BpPlan& p) {
  if (p.kind != KIND_IDIFF || p.interp == INTERP_NEAREST || !(p.detInc > 0)) return false;
  const double far = (fabs(p.xMin) + fabs(p.xMax) + fabs(p.yMin) + fabs(p.yMax)) / p.detInc + p.nDet;
  const int W = idiff_window(p, 32, 32);
  return far < 0x1p20 && W > 0 && 4 * W * idiff_cell(p) <= kFanLds;
}

int bp_idiff_f64_launch(ctsim_ctx* ctx, const BpPlan& p, const double* d_filtered, const ViewConstF64* d_vc,
                        int nView, float* d_image, bool fresh) {
  const bool cubic = p.interp == INTERP_CUBIC;
  IdiffArgs a{};
  a.nx = p.nx; a.ny = p.ny; a.nDet = p.nDet; a.nView = nView;
  a.f = d_filtered; a.vc = d_vc; a.image = d_image;
  a.fresh = fresh; a.endScale = p.rotScale;
  // four rows per lane where that leaves four workgroups per CU, else one.
  // Per slice with the FFT filter, one / four rows, linear: 256^2 47 / 96 us,
  // 512^2 145 / 206, 1024^2 791 / 722; 2048^2 (convolution) 7.30 / 6.24 ms.
  // Views at a time: 4 with one row, 2 (linear) or 1 (cubic, whose bounds take
  // the registers) with four, each the fastest of 1, 2, 4 and 8.
  const int P = static_cast<size_t>(p.nx) * p.ny >= static_cast<size_t>(4) * 4 * kBlock * ctx->numCUs ? 4 : 1;
  const int side = P == 4 ? 32 : 16;
  a.W = idiff_window(p, side, side);
  a.tilesY = (p.ny + side - 1) / side;
  const int grid = (p.nx + side - 1) / side * a.tilesY;
  a.half = a.W <= 29;
  for (a.views = 16; a.views > 4 && a.views * a.W * idiff_cell(p) > kFanLds; a.views /= 2) {
  }
  const size_t lds = a.views * a.W * idiff_cell(p);
  const dim3 g(grid), b(kBlock);
  const hipStream_t s = ctx->stream;
  ctx->prof_begin();
  if (cubic) {
    if (P == 4) hipLaunchKernelGGL((bp_idiff_f64_kernel<INTERP_CUBIC, 8, 4, 1>), g, b, lds, s, a);
    else hipLaunchKernelGGL((bp_idiff_f64_kernel<INTERP_CUBIC, 16, 1, 4>), g, b, lds, s, a);
  } else {
    if (P == 4) hipLaunchKernelGGL((bp_idiff_f64_kernel<INTERP_LINEAR, 8, 4, 2>), g, b, lds, s, a);
    else hipLaunchKernelGGL((bp_idiff_f64_kernel<INTERP_LINEAR, 16, 1, 4>), g, b, lds, s, a);
  }
  ctx->prof_end();
  CTSIM_HIP(hipGetLastError());
  return CTSIM_OK;
}

}  // namespace ctsim
