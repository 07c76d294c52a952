// Phantom rasterisation on the device (Phantom::convertToImagefile,
// libctsim/phantom.cpp:463-538; the phm2if tool).
//
// Each pixel is the average over nsample x nsample sample points of the
// summed attenuation of the elements containing them.  One lane owns one
// pixel and walks the elements in the reference's list order (newest first),
// adding each element's double sum of sample attenuations into the float
// pixel, as the reference does; sample coordinates follow the reference's
// repeated additions (column and row starts from host tables built the same
// way), so the image is bit-identical.
//
// A wave owns 8 x 8 pixels and first tests 64 elements at a time, one per
// lane, against its square: an element certainly outside it adds nothing (a
// sum of zero changes a pixel only if that is -0.0, which attenuations of
// ordinary size do not leave: `cull`), one that certainly contains it adds its
// nsample^2 attenuations, summed on the host in the reference's order, and
// only the others' samples are tested point by point.
//
// What bounds it: FP64 VALU issue of the point tests.  512^2 pixels, 2 x 2
// samples, 69 elements: 70 us with every lane walking every element, 10 us
// here.
#include <hip/hip_runtime.h>

#include <vector>

#include "scan_plan.h"

#pragma clang fp contract(off)

namespace ctsim {
namespace {

struct RasterArgs {
  const ElemGPU* elems;
  int nElem, nx, ny, nsample;
  int tilesY, cull;
  double kxinc, kyinc, kxofs, kyofs, factor;
  const double* xs;   // column starts x, by repeated addition
  const double* ys;   // row starts y
  const double* sum;  // per element its attenuation added nsample^2 times
  float* img;         // [nx][ny] column-major
};

// PhantomElement::isPointInside with PHM_COORD, phantom.cpp:913-975.
__device__ __forceinline__ bool point_inside(const ElemGPU& e, double x, double y) {
  const double xt = x * e.p2o[0] + y * e.p2o[2] + e.p2o[4];
  const double yt = x * e.p2o[1] + y * e.p2o[3] + e.p2o[5];
  x = xt;
  y = yt;
  switch (e.type) {
    case PE_RECT:
      return !(x > 1. || x < -1. || y > 1. || y < -1.);
    case PE_TRI:
      return !(y < 0. || y > 1. - x || y > 1. + x);
    case PE_ELLIPSE:
      if (x > 1. || x < -1. || y > 1. || y < -1.) return false;
      return !(x * x + y * y > 1.);
    case PE_SEGMENT:
      if (x > 1. || x < -1. || y > 0.) return false;
      x *= e.u;
      y *= e.v;
      return !(x * x + (y - e.v) * (y - e.v) > e.u * e.u + e.v * e.v);
    case PE_SECTOR:
      if (x > 1. || x < -1. || y > 1.) return false;
      if (y > 1. - x || y > 1. + x) return false;
      x *= e.u;
      y *= e.v;
      return !(x * x + (y - e.v) * (y - e.v) > e.u * e.u + e.v * e.v);
  }
  return false;
}

// Where the square of centre (x, y) and half sides (hx, hy) lies to an element:
// -1 certainly outside, 1 certainly inside, 0 to be tested.  The square's
// image in the element's frame is bounded by its centre and half extents; the
// margins cover the rounding of the point test, and values that are no
// numbers fail every comparison.
__device__ __forceinline__ int square_place(const ElemGPU& e, double x, double y, double hx, double hy) {
  const double cx = x * e.p2o[0] + y * e.p2o[2] + e.p2o[4], cy = x * e.p2o[1] + y * e.p2o[3] + e.p2o[5];
  const double mag = 1 + fabs(e.p2o[4]) + fabs(e.p2o[5]) + (fabs(x) + hx) * (fabs(e.p2o[0]) + fabs(e.p2o[1])) +
                     (fabs(y) + hy) * (fabs(e.p2o[2]) + fabs(e.p2o[3]));
  const double m = 1e-12 * mag;
  const double ex = fabs(e.p2o[0]) * hx + fabs(e.p2o[2]) * hy + m, ey = fabs(e.p2o[1]) * hx + fabs(e.p2o[3]) * hy + m;
  if (fabs(cx) - ex > 1 || cy - ey > (e.type == PE_SEGMENT ? 0 : 1)) return -1;
  if (e.type == PE_RECT || e.type == PE_ELLIPSE) {
    if (cy + ey < -1) return -1;
    const double far = fabs(cx) + ex, low = fabs(cy) + ey;
    if (e.type == PE_RECT) return far < 1 && low < 1 ? 1 : 0;
    const double nx = fmax(fabs(cx) - ex, 0.0), ny = fmax(fabs(cy) - ey, 0.0);
    if (nx * nx + ny * ny > 1 + 1e-12) return -1;
    return far * far + low * low < 1 - 1e-12 ? 1 : 0;
  }
  if (e.type == PE_TRI && cy + ey < 0) return -1;
  return 0;
}

__global__ __launch_bounds__(256) void raster_kernel(RasterArgs a) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // waves 0 ... 3 own the quarters of a 16 x 16 tile
  const int bx = static_cast<int>(blockIdx.x) / a.tilesY * 16 + (wave >> 1) * 8;
  const int by = static_cast<int>(blockIdx.x) % a.tilesY * 16 + (wave & 1) * 8;
  if (bx >= a.nx || by >= a.ny) return;
  const int ix = bx + (lane >> 3), iy = by + (lane & 7);
  const double x = a.xs[min(ix, a.nx - 1)], y = a.ys[min(iy, a.ny - 1)];
  // the samples' range
  const double xa = a.xs[bx] + a.kxofs, xb = a.xs[min(bx + 7, a.nx - 1)] + a.kxofs + (a.nsample - 1) * a.kxinc;
  const double ya = a.ys[by] + a.kyofs, yb = a.ys[min(by + 7, a.ny - 1)] + a.kyofs + (a.nsample - 1) * a.kyinc;
  float v = 0.f;
  for (int e0 = (a.nElem - 1) & ~63; e0 >= 0; e0 -= 64) {
    const int ek = e0 + lane;
    int place = -1;
    if (ek < a.nElem)
      place = a.cull ? square_place(a.elems[ek], 0.5 * (xa + xb), 0.5 * (ya + yb), 0.5 * fabs(xb - xa), 0.5 * fabs(yb - ya))
                     : 0;
    unsigned long long todo = __ballot(place >= 0);
    const unsigned long long whole = __ballot(place > 0);
    while (todo) {  // newest first
      const int b = 63 - __builtin_clzll(todo);
      todo &= ~(1ull << b);
      const int el = e0 + b;
      double dAtten = 0;
      if ((whole >> b) & 1) {
        dAtten = a.sum[el];
      } else {
        const ElemGPU& e = a.elems[el];
        double xi = x + a.kxofs;
        for (int kx = 0; kx < a.nsample; kx++, xi += a.kxinc) {
          double yi = y + a.kyofs;
          for (int ky = 0; ky < a.nsample; ky++, yi += a.kyinc)
            if (point_inside(e, xi, yi)) dAtten += e.atten;
        }
      }
      v += dAtten;
    }
  }
  if (a.nsample > 1) v *= a.factor;
  if (ix < a.nx && iy < a.ny) a.img[static_cast<size_t>(ix) * a.ny + iy] = v;
}

}  // namespace
}  // namespace ctsim

using namespace ctsim;

extern "C" int ctsim_phantom_rasterize(ctsim_ctx* ctx, ctsim_phantom* phm, int nx, int ny,
                                       double viewRatio, int nsample, float* d_image,
                                       double* ext4) {
  if (!ctx || !phm || !d_image) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_rasterize: NULL argument");
  if (nx < 2 || ny < 2) return fail(CTSIM_ERR_INVALID, "ctsim_phantom_rasterize: image smaller than 2x2");
  CTSIM_CHECK(ctx->activate());
  PhantomPlan& p = phm->plan;
  CTSIM_CHECK(phantom_upload(p));
  if (nsample < 1) nsample = 1;
  // phantom.cpp:474-500
  const double dx = p.xmax - p.xmin, dy = p.ymax - p.ymin;
  const double xcent = p.xmin + dx / 2, ycent = p.ymin + dy / 2;
  const double maxAxis = dx > dy ? dx : dy;
  const double dHalflen = viewRatio * ((kSqrt2 * maxAxis) / kSqrt2 / 2);
  const double xmin = xcent - dHalflen, xmax = xcent + dHalflen;
  const double ymin = ycent - dHalflen, ymax = ycent + dHalflen;
  const double xinc = (xmax - xmin) / nx, yinc = (ymax - ymin) / ny;
  const size_t nElem = p.elems.size();
  const size_t bytes = (static_cast<size_t>(nx) + ny + nElem) * sizeof(double);
  CTSIM_CHECK(ctx->stage.reserve(bytes, ctx->stream));
  double* tab = static_cast<double*>(ctx->stage.ptr);
  double x = xmin;
  for (int ix = 0; ix < nx; ix++, x += xinc) tab[ix] = x;
  double y = ymin;
  for (int iy = 0; iy < ny; iy++, y += yinc) tab[nx + iy] = y;
  bool cull = true;
  for (size_t k = 0; k < nElem; k++) {
    const double atten = p.elems[k].atten;
    double sum = 0;
    for (int q = 0; q < nsample * nsample; q++) sum += atten;
    tab[static_cast<size_t>(nx) + ny + k] = sum;
    if (!(atten == 0 || fabs(atten) > 1e-20)) cull = false;
  }
  CTSIM_CHECK(ctx->rasterTab.reserve(bytes));
  CTSIM_CHECK(ctx->stage.upload(ctx->rasterTab, bytes, ctx->stream));
  RasterArgs a{};
  a.elems = p.d_elems.as<ElemGPU>();
  a.nElem = static_cast<int>(nElem);
  a.nx = nx;
  a.ny = ny;
  a.nsample = nsample;
  a.kxinc = xinc / nsample;
  a.kyinc = yinc / nsample;
  a.kxofs = a.kxinc / 2;
  a.kyofs = a.kyinc / 2;
  a.factor = 1.0 / static_cast<double>(nsample * nsample);
  a.xs = ctx->rasterTab.as<double>();
  a.ys = a.xs + nx;
  a.sum = a.ys + ny;
  a.cull = cull ? 1 : 0;
  a.img = d_image;
  a.tilesY = (ny + 15) / 16;
  const size_t tiles = static_cast<size_t>((nx + 15) / 16) * a.tilesY;
  hipLaunchKernelGGL(raster_kernel, dim3(static_cast<unsigned>(tiles)), dim3(256), 0, ctx->stream, a);
  CTSIM_HIP(hipGetLastError());
  CTSIM_HIP(hipStreamSynchronize(ctx->stream));
  if (ext4) {
    ext4[0] = xmin; ext4[1] = xmax; ext4[2] = ymin; ext4[3] = ymax;
  }
  return CTSIM_OK;
}
