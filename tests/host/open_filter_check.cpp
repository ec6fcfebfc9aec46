// Host check of the float32 pre-filter for integer coordinates in an open box
// (fpf_* with the coordinates converted to float and scaled by 2^-dshift): it
// passes every leaf whose exact squared distance is at most the bound, and
// with a floor never puts one below it; and of leaf_f32, whose widened value
// is leaf_d2 of float coordinates.
#include "../../fasttree_amd/csrc/ft_traverse.hpp"
#include <cmath>
#include <cstdio>
#include <random>
using namespace ft;

template <typename T> static long check(std::mt19937_64 &g, int bits, long &tests) {
  Metric m{bits, 0, bits > 31 ? bits - 31 : 0, 0, 0.0};
  const T top = (T)(~(T)0) >> (sizeof(T) * 8 - bits);
  const float fs = 1.0f / (float)(1ull << m.dshift);
  const double E = fpf_err((double)top * fs, 0.0, false) + (m.dshift ? 1.0 : 0.0);
  long bad = 0;
  for (int it = 0; it < 200000; ++it) {
    T p[3], q[3];
    float fp[3], fq[3];
    for (int a = 0; a < 3; ++a) {
      p[a] = (T)g() & top;
      const int mode = (int)(g() % 4);  // anywhere, close, closer, the same
      const T gap = mode == 0 ? (T)g() & top : mode == 1 ? (T)(g() & 0xFFFF) : mode == 2 ? (T)(g() & 7) : 0;
      q[a] = (g() & 1) ? (p[a] > gap ? (T)(p[a] - gap) : 0) : (top - p[a] > gap ? (T)(p[a] + gap) : top);
      fp[a] = (float)p[a] * fs;
      fq[a] = (float)q[a] * fs;
    }
    const uint64_t d = leaf_d2<T>(m, p[0], p[1], p[2], q[0], q[1], q[2]);
    const float fd = fpf_sq(fpf_gap(fp[0], fq[0], 0.f, false), fpf_gap(fp[1], fq[1], 0.f, false),
                            fpf_gap(fp[2], fq[2], 0.f, false));
    for (uint64_t w : {d, d + 1}) bad += !(fd <= fpf_upper((double)w, E));
    for (uint64_t lo : {d, d ? d - 1 : 0}) bad += !(fd >= fpf_lower((double)lo, E));
    tests += 4;
  }
  return bad;
}

int main() {
  std::mt19937_64 g(23);
  long tests = 0, bad = 0;
  for (int b : {1, 10, 21, 24, 31, 32}) bad += check<uint32_t>(g, b, tests);
  for (int b : {10, 21, 31, 32, 42}) bad += check<uint64_t>(g, b, tests);
  std::uniform_real_distribution<float> U(0.f, 100.f);
  for (int wrap = 0; wrap < 2; ++wrap) {
    Metric m{21, wrap, 0, 0, 100.0};
    for (int it = 0; it < 200000; ++it, ++tests) {
      const float v[6] = {U(g), U(g), U(g), U(g), U(g), U(g)};
      const double d = leaf_d2<float>(m, v[0], v[1], v[2], v[3], v[4], v[5]);
      const float f = wrap ? leaf_f32<MK_WRAP>(m, v[0], v[1], v[2], v[3], v[4], v[5])
                           : leaf_f32<MK_OPEN>(m, v[0], v[1], v[2], v[3], v[4], v[5]);
      bad += (double)f != d;
    }
  }
  printf("open filter tests %ld, failures: %ld\n", tests, bad);
  return bad != 0;
}
