// Host check of the packet walk's relative float32 filter (rel_coord,
// rel_upper, rel_lower): pairs of a query within ext of a centre and a leaf
// anywhere, doubles and integers, periodic (no wrap in the filter, bounds
// within a quarter period less ext) and open; the filter passes every leaf
// within the bound and none above a floor falls below it.
#include "../../fasttree_amd/csrc/ft_traverse.hpp"
#include <cmath>
#include <cstdio>
#include <random>
using namespace ft;

template <typename T, int MK> static long check(std::mt19937_64 &g, Metric m, double side, long &tests) {
  std::uniform_real_distribution<double> U(0.0, 1.0);
  const bool fp = CoordTraits<T>::fp, wrap = MK == MK_WRAP;
  long bad = 0;
  auto put = [&](double v) -> T {
    if (wrap) v = std::fmod(std::fmod(v, side) + side, side);
    if (v < 0) v = 0;
    return (T)(fp ? v : std::min(std::floor(v), side - 1));
  };
  for (int it = 0; it < 300000; ++it) {
    const double ext0 = side * std::pow(10.0, -6.0 * U(g)) * 0.2;
    T c[3], q[3], x[3];
    float fq[3], fx[3], ext = 0.f;
    for (int a = 0; a < 3; ++a) {
      const double cc = U(g) * side, qq = cc + (2 * U(g) - 1) * ext0;
      const int mode = (int)(g() % 3);
      const double gap = mode == 0 ? U(g) * side : mode == 1 ? ext0 * U(g) : ext0 * 1e-4 * U(g);
      c[a] = put(cc); q[a] = put(qq); x[a] = put(qq + ((g() & 1) ? gap : -gap));
      fq[a] = rel_coord<T, MK>(m, q[a], c[a]);
      fx[a] = rel_coord<T, MK>(m, x[a], c[a]);
      ext = std::fmax(ext, std::fabs(fq[a]));
    }
    float E = 2.02f * 0x1p-24f * ext;
    if (fp) E += (float)(0x1p-50 * (side + ext + (wrap ? m.box : 0.0)));
    const auto d2 = leaf_d2<T>(m, q[0], q[1], q[2], x[0], x[1], x[2]);
    const float fd = fpf_sq(fq[0] - fx[0], fq[1] - fx[1], fq[2] - fx[2]);
    const double room = 0.249 * side - ext;
    if (!wrap || (room > 0 && (double)d2 <= room * room)) {
      ++tests;
      bad += !(fd <= rel_upper((float)d2, E));
      if (!fp && wrap) bad += !(fd <= wrap_filter_bound((uint64_t)d2));
    }
    // (periodic: a leaf farther than half a period may look farther than it is)
    if (!wrap || (room > 0 && (double)d2 <= room * room)) bad += !(fd >= rel_lower((float)d2, E));
    // a leaf beyond the room is never taken for one inside it
    if (wrap && room > 0 && (double)d2 > room * room * 1.01)
      bad += !(fd > rel_upper((float)(0.9 * room * room), E));
  }
  return bad;
}

int main() {
  std::mt19937_64 g(29);
  long tests = 0, bad = 0;
  for (double L : {1.0, 100.0, 1e6}) {
    bad += check<double, MK_WRAP>(g, Metric{21, 1, 0, 0, L}, L, tests);
    bad += check<double, MK_OPEN>(g, Metric{21, 0, 0, 0, 0.0}, L, tests);
  }
  for (int b : {10, 21, 22}) {
    bad += check<uint64_t, MK_WRAP>(g, Metric{b, 1, 0, 0, 0.0}, (double)(1u << b), tests);
    bad += check<uint32_t, MK_WRAP>(g, Metric{b, 1, 0, 0, 0.0}, (double)(1u << b), tests);
  }
  for (int b : {10, 21, 31}) {
    bad += check<uint64_t, MK_OPEN>(g, Metric{b, 0, 0, 0, 0.0}, (double)(1u << b), tests);
    bad += check<uint32_t, MK_OPEN>(g, Metric{b, 0, 0, 0, 0.0}, (double)(1u << b), tests);
  }
  // tiny and huge magnitudes of the bound itself
  for (double d : {0.0, 1e-300, 1e-45, 1e-39, 1e-31, 1e-29, 1.0, 1e30, 1e38, 1e300}) {
    const float fd = (float)d;
    bad += !(fd <= rel_upper(fd, 0.f)) || !(fd >= rel_lower(fd, 0.f) || std::isinf(fd));
    tests += 1;
  }
  printf("relative filter tests %ld, failures: %ld\n", tests, bad);
  return bad != 0;
}
