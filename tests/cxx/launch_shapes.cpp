// Host decisions of the launches, printed for test_launch_shapes.py.
//
//   slice GEOMETRY NDET NVIEW NX NY METHOD INTERP: the mixed launch shape by rule
//     and the one that a whole slice runs (kernel, rows per lane, lanes along y,
//     view groups), its scratch, and the default shape's scratch, then the
//     detector windows of the rule's tile and of 8 and 16 lanes with 4 rows
//   fan64 ANGLE...: the largest angle in size, and whether the FP64 fan-beam
//     kernel's bounds cover it
//   scan GEOMETRY NDET NVIEW FOCAL CENTER ELLIPSES RECTANGLES TRIANGLES SIZE (or a
//     phantom's name): whether the short ray sums run
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "bp_plan.h"
#include "filter_plan.h"
#include "scan_plan.h"

using namespace ctsim;

static int slice(char** v) {
  const int geom = atoi(v[0]), nDet = atoi(v[1]), nView = atoi(v[2]), nx = atoi(v[3]), ny = atoi(v[4]);
  const double d = 2 * std::sqrt(2.0), F = d, sdl = 2 * d, pi = 3.14159265358979323846;
  const double fan = 2 * std::asin(0.5);
  const double inc = geom == GEOM_PARALLEL ? d / nDet : (geom == GEOM_EQUILINEAR ? 2 * sdl * std::tan(fan / 2) : fan) / nDet;
  BpPlan p;
  if (bp_plan_init(p, geom, nDet, inc, nView, d, F, sdl, "idiff", v[6], 1, nx, ny, nullptr) != CTSIM_OK) return 1;
  FilterPlan f;
  if (filter_plan_init(f, "abs_hanning", v[5], 1 / inc, inc, nDet, 1.0, "frequency", "direct", 1, 1, geom, F, sdl) != CTSIM_OK)
    return 1;
  std::vector<double> angles(nView);
  for (int k = 0; k < nView; k++) angles[k] = k * ((geom == GEOM_PARALLEL ? pi : 2 * pi) / nView);
  std::vector<ViewConstF32> vc(nView);
  const MirrorViews mv = bp_view_consts_f32(p, angles.data(), nView, vc.data());
  SymViews sv = bp_sym_views(angles.data(), nView);
  sv.NM = mv.NM;
  sv.mapO = mv.mapO;
  const MixedShape a = bp_auto_shape(p, sv, nView), b = fbp_slice_shape(f, p, sv, nView);
  std::printf("rule %d %d %d %d slice %d %d %d %d scratch %zu default %zu windows %d %d %d\n", a.sym, a.P, a.lanesY, a.split, b.sym, b.P,
              b.lanesY, b.split, fbp_slice_scratch(f, p, b, nView).total(), fbp_slice_scratch(f, p, p.mixed, nView).total(), a.W,
              bp_window_bound(p, 32, 32), bp_window_bound(p, 16, 64));
  return 0;
}

static int fan64(int n, char** v) {
  std::vector<double> angles(n);
  for (int k = 0; k < n; k++) angles[k] = std::atof(v[k]);
  BpPlan p;
  const double d = 2 * std::sqrt(2.0);
  if (bp_plan_init(p, GEOM_EQUIANGULAR, 257, 0.004, n, d, d, 2 * d, "idiff", "linear", 1, 128, 128, nullptr) != CTSIM_OK) return 1;
  const double m = bp_max_angle(angles.data(), n);
  std::printf("%g %d\n", m, bp_fan_f64_ok(p, m) ? 1 : 0);
  return 0;
}

static int scan(int n, char** v) {
  PhantomPlan p;
  if (n == 6) {
    if (phantom_builtin(p, v[5]) != CTSIM_OK) return 1;
  } else {
    phantom_add(p, "rectangle", 0, 0, 1, 1, 0, 0.1);
    unsigned seed = 1;
    auto at = [&]() { return ((seed = seed * 1664525u + 1013904223u) >> 8) / 16777216.0 - 0.5; };
    const char* const types[] = {"ellipse", "rectangle", "triangle"};
    for (int t = 0; t < 3; t++)
      for (int k = 0; k < std::atoi(v[5 + t]); k++) {
        const double x = at(), y = at(), size = t == 2 ? std::atof(v[8]) : 0.1;
        phantom_add(p, types[t], x, y, size, size, 360 * at(), 0.3);
      }
  }
  ScannerPlan s;
  if (scanner_init(s, p, v[0], std::atoi(v[1]), std::atoi(v[2]), 0, 1, v[0][0] == 'p' ? 3.14159265358979323846 : 6.28318530717958647692,
                   std::atof(v[3]), std::atof(v[4]), 1, 1) != CTSIM_OK)
    return 1;
  phantom_fast_elems(p);
  std::printf("%d\n", raysum_short_pays(s, p, s.nView, 256) ? 1 : 0);
  return 0;
}

int main(int argc, char** argv) {
  if (argc >= 8 && !std::strcmp(argv[1], "scan")) return scan(argc - 2, argv + 2);
  if (argc > 2 && !std::strcmp(argv[1], "fan64")) return fan64(argc - 2, argv + 2);
  if (argc == 9 && !std::strcmp(argv[1], "slice")) return slice(argv + 2);
  return 2;
}
