// Host check of the range walk's float32 filter with the kernel's own error bound
// (rel_err) and thresholds (range_filter): pairs of a query within ext of a centre
// and a leaf anywhere, radii at, just below and just above their distance and far
// from it; a pair surely inside r_max or nearer than r_min is so exactly, and one
// surely outside or not nearer is so too.  The packet walk's bounds (rel_upper,
// rel_lower) with that error bound hold as well.
#include "../../fasttree_amd/csrc/ft_traverse.hpp"
#include <cmath>
#include <cstdio>
#include <random>
using namespace ft;

static long tests = 0, unsure = 0;

template <typename T, int MK> static long check(std::mt19937_64 &g, Metric m, double side, double origin) {
  using D = typename CoordTraits<T>::D;
  std::uniform_real_distribution<double> U(0.0, 1.0);
  const bool fp = CoordTraits<T>::fp, wrap = MK == MK_WRAP;
  long bad = 0;
  auto put = [&](double v) -> T {
    if (wrap) v = std::fmod(std::fmod(v, side) + side, side);
    if (!fp && v < 0) v = 0;
    return (T)(fp ? v + origin : std::min(std::floor(v), side - 1));
  };
  for (int it = 0; it < 200000; ++it) {
    const double ext0 = side * std::pow(10.0, -6.0 * U(g)) * 0.2;
    T c[3], q[3], x[3];
    float fq[3], fx[3], ext = 0.f;
    for (int a = 0; a < 3; ++a) {
      const double cc = U(g) * side, qq = cc + (2 * U(g) - 1) * ext0;
      const int mode = (int)(g() % 3);
      const double gap = mode == 0 ? U(g) * side * 0.4 : mode == 1 ? ext0 * U(g) : ext0 * 1e-4 * U(g);
      c[a] = put(cc); q[a] = put(qq); x[a] = put(qq + ((g() & 1) ? gap : -gap));
      fq[a] = rel_coord<T, MK>(m, q[a], c[a]);
      fx[a] = rel_coord<T, MK>(m, x[a], c[a]);
      ext = std::fmax(ext, std::fabs(fq[a]));
    }
    const double E = rel_err<T, MK>(m, ext, c[0], c[1], c[2]);
    const D d2 = leaf_d2<T>(m, q[0], q[1], q[2], x[0], x[1], x[2]);
    const float fd = fpf_sq(fq[0] - fx[0], fq[1] - fx[1], fq[2] - fx[2]);
    const double v = (double)d2;
    for (double r2 : {v, std::nextafter(v, 1e300), std::nextafter(v, 0.0), v * (1 + 1e-7), v * (1 - 1e-7),
                      v * U(g), v * (1 + U(g)), 0.0}) {
      const D R = (D)r2;
      const double rad = std::sqrt((double)R);
      if (wrap && !(ext + rad < 0.249 * side)) continue;  // the kernel's own limit
      const RangeFilter f = range_filter<D>(R, R, E);
      ++tests;
      bad += (fd < f.f_in && !(d2 <= R)) || (fd > f.f_out && d2 <= R);
      if (!(R <= D(0))) bad += (fd < f.g_out && d2 >= R) || (fd > f.g_in && !(d2 >= R));
      bad += d2 <= R && !(fd <= rel_upper((float)R, (float)E));
      bad += !wrap && d2 >= R && !(fd >= rel_lower((float)R, (float)E));
      unsure += !(fd < f.f_in) && fd <= f.f_out;
    }
  }
  return bad;
}

int main() {
  std::mt19937_64 g(31);
  long bad = 0;
  for (double L : {1.0, 100.0, 1e6}) {
    bad += check<double, MK_WRAP>(g, Metric{21, 1, 0, 0, L}, L, 0.0);
    bad += check<double, MK_OPEN>(g, Metric{21, 0, 0, 0, 0.0}, L, 0.0);
    bad += check<double, MK_OPEN>(g, Metric{21, 0, 0, 0, 0.0}, L, -1e9);  // far from the origin
  }
  for (int b : {10, 21}) {
    bad += check<uint64_t, MK_WRAP>(g, Metric{b, 1, 0, 0, 0.0}, (double)(1u << b), 0.0);
    bad += check<uint32_t, MK_WRAP>(g, Metric{b, 1, 0, 0, 0.0}, (double)(1u << b), 0.0);
    bad += check<uint64_t, MK_OPEN>(g, Metric{b, 0, 0, 0, 0.0}, (double)(1u << b), 0.0);
    bad += check<uint32_t, MK_OPEN>(g, Metric{b, 0, 0, 0, 0.0}, (double)(1u << b), 0.0);
  }
  // radii that are not numbers have no hits, zero and tiny ones go to the exact test
  const RangeFilter n = range_filter<double>(0.0, std::nan(""), 1e-9);
  bad += n.f_in != -1.f || n.f_out != -1.f;
  for (double r2 : {0.0, 1e-300, 1e-45, 1e-31}) bad += range_filter<double>(0.0, r2, 0.0).f_in != 0.f;
  printf("range filter tests %ld (%ld left to the exact test), failures: %ld\n", tests, unsure, bad);
  return bad != 0;
}
