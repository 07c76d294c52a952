// Fan-beam to parallel rebinning (Projections::interpolateToParallel,
// libctsim/projections.cpp:1250-1328, with ParallelRaysums, 1339-1469).
//
// Every fan sample is a parallel ray (theta, t).  The reference sorts all
// samples by (t, theta); detector g of the new sinogram is the g-th run of
// nView samples (one fan detector, all views, increasing theta).  It then
// interpolates each run linearly to evenly spaced view angles, and each new
// view linearly to evenly spaced detector positions, storing floats after
// each pass.  The sort depends only on the geometry and the view angles, so
// the plan does it once on the host (the reference's expressions, glibc
// trig, no contraction); the two interpolation passes run on the device, one
// block per new view, in FP64 with the reference's expression order.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <functional>
#include <cmath>
#include <numeric>
#include <vector>

#include "ctsim_internal.h"

#pragma clang fp contract(off)

namespace ctsim {
namespace {

constexpr int kRebinLds = 5120;  // detectors whose positions and row fit 60 KB of LDS

struct RebinPlan {
  int geom = 0, nDet = 0, nView = 0;
  double newRotInc = 0, newDetStart = 0, newDetInc = 0;
  std::vector<double> newAngles;
  DevBuf d_theta;   // [nView][nDet] sorted theta of each run
  DevBuf d_src;     // [nView][nDet] source sample (v * nDet + d) of each run entry
  DevBuf d_t;       // [nDet] t of each run
  DevBuf d_angles;  // [nView] new view angles
  DevBuf d_pos;     // [nDet] new detector positions
  DevBuf d_mid;     // [nView][nDet] float after the theta pass (two launches)
};

// The largest i with dX >= X(i), or -1.  guess: tried first with its
// neighbours, three loads at once, before the binary search.
template <class XF>
__device__ __forceinline__ int lower_index(const XF& X, int n, double dX, int guess) {
  const int g = min(max(guess, 1), n - 2);
  if (n >= 3) {
    const double a = X(g - 1), b = X(g), c = X(g + 1);
    if (dX >= a && dX < c) return dX >= b ? g : g - 1;
  }
  int iLower = -1, iUpper = n;
  while (iUpper - iLower > 1) {
    const int iMiddle = (iUpper + iLower) >> 1;
    if (dX >= X(iMiddle)) iLower = iMiddle;
    else iUpper = iMiddle;
  }
  return iLower;
}

// LinearInterpolator<double>::interpolate with abscissae and values clamped
// outside (include/interpolator.h:203-262), the search done; the search hint
// the reference passes does not change the result for increasing abscissae.
template <class XF, class YF>
__device__ __forceinline__ double lin_interp(const XF& X, const YF& Y, int n, double dX, int iLower) {
  if (iLower < 0 || dX == X(0)) return Y(0);
  if (dX >= X(n - 1)) return Y(n - 1);
  const double y0 = Y(iLower), y1 = Y(iLower + 1);
  return y0 + (y1 - y0) * ((dX - X(iLower)) / (X(iLower + 1) - X(iLower)));
}

struct RebinArgs {
  const float* in;
  const double* theta;
  const int* src;
  const double* t;
  const double* angles;
  const double* pos;
  float* mid;
  float* out;
  int nDet, nView;
};

// Run g at new view v (projections.cpp:1285-1298).  A run's angles are nearly
// evenly spaced, so its interval is guessed from its ends.  The runs' tables lie
// [entry][run], so that a wave's lanes, whose entries are nearly the same, read
// adjacent runs.
__device__ __forceinline__ float run_value(const RebinArgs& a, int g, double dX) {
  const int nDet = a.nDet, nView = a.nView;
  auto X = [&a, g, nDet](int i) { return a.theta[static_cast<size_t>(i) * nDet + g]; };
  auto Y = [&a, g, nDet](int i) { return static_cast<double>(a.in[a.src[static_cast<size_t>(i) * nDet + g]]); };
  const double x0 = X(0), x1 = X(nView - 1);
  const float guess = static_cast<float>(dX - x0) / static_cast<float>(x1 - x0) * (nView - 1);
  const int g0 = static_cast<int>(fminf(fmaxf(guess, 0.f), static_cast<float>(nView)));  // (no number: 0)
  return static_cast<float>(lin_interp(X, Y, nView, dX, lower_index(X, nView, dX, g0)));
}

// A view's row of runs (positions t) at new detector position d
// (projections.cpp:1300-1325), searched from d on.
__device__ __forceinline__ float row_value(const RebinArgs& a, const double* t, const float* row, int d) {
  auto X = [t](int i) { return t[i]; };
  auto Y = [row](int i) { return static_cast<double>(row[i]); };
  const double p = a.pos[d];
  return static_cast<float>(lin_interp(X, Y, a.nDet, p, lower_index(X, a.nDet, p, d)));
}

// One block per new view, the row of floats between the two passes in LDS.
//
// What bounds it: the latency of the searches.  720 views of 512 detectors:
// 16.1 us a call in two launches with binary searches in memory and the row
// between them, 9.0 now (8.2 in the kernel).
__global__ __launch_bounds__(512) void rebin_kernel(RebinArgs a) {
  extern __shared__ double s_t[];
  const int v = blockIdx.x, nDet = a.nDet;
  float* row = reinterpret_cast<float*>(s_t + nDet);
  const double dX = a.angles[v];
  for (int g = threadIdx.x; g < nDet; g += blockDim.x) {
    s_t[g] = a.t[g];
    row[g] = run_value(a, g, dX);
  }
  __syncthreads();
  for (int d = threadIdx.x; d < nDet; d += blockDim.x)
    a.out[static_cast<size_t>(v) * nDet + d] = row_value(a, s_t, row, d);
}

// The two passes as launches of their own, a lane per value, the rows between
// them in a.mid: for rows that do not fit LDS, for an output that overlaps the
// input (the first pass has read it all), and where one block per view would go
// through long rows alone (ctsim_rebin_run).
__global__ __launch_bounds__(256) void rebin_runs_kernel(RebinArgs a) {
  const int v = blockIdx.x, g = blockIdx.y * 256 + threadIdx.x;
  if (g < a.nDet) a.mid[static_cast<size_t>(v) * a.nDet + g] = run_value(a, g, a.angles[v]);
}
__global__ __launch_bounds__(256) void rebin_rows_kernel(RebinArgs a) {
  const int v = blockIdx.x, d = blockIdx.y * 256 + threadIdx.x;
  const size_t row = static_cast<size_t>(v) * a.nDet;
  if (d < a.nDet) a.out[row + d] = row_value(a, a.t, a.mid + row, d);
}

}  // namespace
}  // namespace ctsim

using namespace ctsim;

struct ctsim_rebin {
  RebinPlan p;
};

extern "C" {

int ctsim_rebin_create(ctsim_ctx* ctx, ctsim_rebin** out, int geometry, int nDet, int nView,
                       double detStart, double detInc, double focalLength,
                       double sourceDetectorLength, double viewDiameter, double rotStart,
                       const double* h_angles) {
  if (!ctx || !out || !h_angles) return fail(CTSIM_ERR_INVALID, "ctsim_rebin_create: NULL argument");
  if (geometry != GEOM_EQUIANGULAR && geometry != GEOM_EQUILINEAR)
    return fail(CTSIM_ERR_INVALID, "ctsim_rebin_create: fan-beam geometry expected "
                                   "(parallel projections are returned unchanged by the reference)");
  if (nDet < 2 || nView < 2) return fail(CTSIM_ERR_INVALID, "ctsim_rebin_create: too few samples");
  *out = nullptr;
  CTSIM_CHECK(ctx->activate());
  auto* r = new ctsim_rebin();
  RebinPlan& p = r->p;
  p.geom = geometry;
  p.nDet = nDet;
  p.nView = nView;
  p.newRotInc = kTwoPi / nView;
  p.newDetStart = -viewDiameter / 2;
  p.newDetInc = viewDiameter / nDet;
  if (nDet % 2 == 0) p.newDetInc = viewDiameter / (nDet - 1);
  // ParallelRaysums coordinates, view-major (projections.cpp:1352-1379)
  const size_t nc = static_cast<size_t>(nView) * nDet;
  std::vector<double> th(nc), tt(nc);
  for (int iV = 0; iV < nView; iV++) {
    const double dViewAngle = h_angles[iV];
    double dDetPos = detStart;
    for (int iD = 0; iD < nDet; iD++) {
      const size_t k = static_cast<size_t>(iV) * nDet + iD;
      double theta, t;
      if (geometry == GEOM_EQUILINEAR) {
        const double dFanAngle = atan(dDetPos / sourceDetectorLength);
        theta = dViewAngle + dFanAngle;
        t = focalLength * sin(dFanAngle);
      } else {
        theta = dViewAngle + dDetPos;
        t = focalLength * sin(dDetPos);
      }
      while (theta < 0.) theta += kTwoPi;  // normalizeAngle, mathfuncs.cpp:72-81
      while (theta >= kTwoPi) theta -= kTwoPi;
      th[k] = theta;
      tt[k] = t;
      dDetPos += detInc;
    }
  }
  // compareByT (include/projections.h:50-52); exact ties keep view-major order
  std::vector<int> idx(nc);
  std::iota(idx.begin(), idx.end(), 0);
  std::sort(idx.begin(), idx.end(), [&](int a, int b) {
    if (tt[a] != tt[b]) return tt[a] < tt[b];
    if (th[a] != th[b]) return th[a] < th[b];
    return a < b;
  });
  std::vector<double> theta(nc), tRun(nDet), pos(nDet);
  std::vector<int> src(nc);
  for (int g = 0; g < nDet; g++)
    for (int k = 0; k < nView; k++) {
      const size_t to = static_cast<size_t>(k) * nDet + g;
      src[to] = idx[static_cast<size_t>(g) * nView + k];
      theta[to] = th[src[to]];
    }
  for (int g = 0; g < nDet; g++) tRun[g] = tt[idx[static_cast<size_t>(g) * nView]];
  p.newAngles.resize(nView);
  double a = rotStart;
  for (int v = 0; v < nView; v++, a += p.newRotInc) p.newAngles[v] = a;
  double x = p.newDetStart;
  for (int d = 0; d < nDet; d++, x += p.newDetInc) pos[d] = x;
  int rc = CTSIM_OK;
  auto up = [&](DevBuf& d, const void* src, size_t n) {
    if (rc != CTSIM_OK) return;
    if ((rc = d.reserve(n)) != CTSIM_OK) return;
    if (hipMemcpy(d.ptr, src, n, hipMemcpyHostToDevice) != hipSuccess)
      rc = fail(CTSIM_ERR_HIP, "ctsim_rebin_create: upload failed");
  };
  up(p.d_theta, theta.data(), nc * sizeof(double));
  up(p.d_src, src.data(), nc * sizeof(int));
  up(p.d_t, tRun.data(), nDet * sizeof(double));
  up(p.d_angles, p.newAngles.data(), nView * sizeof(double));
  up(p.d_pos, pos.data(), nDet * sizeof(double));
  if (rc == CTSIM_OK) rc = p.d_mid.reserve(nc * sizeof(float));
  if (rc != CTSIM_OK) {
    delete r;
    return rc;
  }
  *out = r;
  return CTSIM_OK;
}

void ctsim_rebin_destroy(ctsim_rebin* r) { delete r; }

int ctsim_rebin_info(const ctsim_rebin* r, double* out4, double* h_newAngles) {
  if (!r || !out4) return fail(CTSIM_ERR_INVALID, "ctsim_rebin_info: NULL argument");
  out4[0] = 0;  // rotStart of the new projections (projections.cpp:1272)
  out4[1] = r->p.newRotInc;
  out4[2] = r->p.newDetStart;
  out4[3] = r->p.newDetInc;
  if (h_newAngles) std::copy(r->p.newAngles.begin(), r->p.newAngles.end(), h_newAngles);
  return CTSIM_OK;
}

int ctsim_rebin_run(ctsim_ctx* ctx, ctsim_rebin* r, const float* d_in, float* d_out) {
  if (!ctx || !r || !d_in || !d_out) return fail(CTSIM_ERR_INVALID, "ctsim_rebin_run: NULL argument");
  CTSIM_CHECK(ctx->activate());
  RebinPlan& p = r->p;
  const RebinArgs a{d_in,
                    p.d_theta.as<double>(),
                    p.d_src.as<int>(),
                    p.d_t.as<double>(),
                    p.d_angles.as<double>(),
                    p.d_pos.as<double>(),
                    p.d_mid.as<float>(),
                    d_out,
                    p.nDet,
                    p.nView};
  const size_t n = static_cast<size_t>(p.nView) * p.nDet;
  const std::less<const float*> before;
  const bool overlap = before(d_in, d_out + n) && before(d_out, d_in + n);
  // One launch while a block goes over its row in one or two rounds, and for
  // longer rows where the views give every CU a block (three rounds) or two.  One
  // / two launches: 1024 x 4 5.7 / 6.9 us, 1024 x 720 14 / 21, 1536 x 64 9.6 / 7.8,
  // 1536 x 360 14 / 16, 2048 x 360 20 / 19, 4096 x 64 23 / 8.8, 4096 x 720 50 / 55.
  const int rounds = (p.nDet + 511) / 512;
  if (p.nDet <= kRebinLds && !overlap && p.nView >= std::min(2, std::max(0, rounds - 2)) * ctx->numCUs) {
    hipLaunchKernelGGL(rebin_kernel, dim3(p.nView), dim3(std::min(512, (p.nDet + 63) / 64 * 64)),
                       p.nDet * (sizeof(double) + sizeof(float)), ctx->stream, a);
  } else {
    const dim3 grid(p.nView, (p.nDet + 255) / 256);
    hipLaunchKernelGGL(rebin_runs_kernel, grid, dim3(256), 0, ctx->stream, a);
    hipLaunchKernelGGL(rebin_rows_kernel, grid, dim3(256), 0, ctx->stream, a);
  }
  CTSIM_HIP(hipGetLastError());
  return CTSIM_OK;
}

}  // extern "C"
