// Host check of the point-location bins (salvus_amd/csrc/element_bins.h): for
// boxes of ordinary, graded, needle-shaped and random elements and for boxes
// that are not finite, every element whose box holds a point (as a scan over
// all boxes decides) is listed in the point's bin, ascending and once, and the
// bins hold at most kMaxBinEntries elements for each element of the mesh.
// Exits non-zero if any check fails.
#include <cstdio>
#include <limits>
#include <random>

#include "element_bins.h"

using namespace sem;

static int failures = 0;

static void check(const char *name, int dim, const std::vector<double> &bbox, const std::vector<double> &pts) {
  const int64_t E = (int64_t)bbox.size() / (2 * dim);
  ElementBins B;
  bin_elements(B, dim, E, bbox.data());
  const int64_t nb = (int64_t)B.n[0] * B.n[1] * B.n[2];
  long missing = 0, disorder = 0;
  for (size_t i = 0; i + dim <= pts.size(); i += dim) {
    const double *pt = &pts[i];
    const int64_t bin = bin_of(B, dim, pt);
    if (bin < 0 || bin >= nb) { ++disorder; continue; }
    const auto begin = B.elem.begin() + B.start[bin], end = B.elem.begin() + B.start[bin + 1];
    for (auto it = begin; it != end; ++it)
      if (*it < 0 || *it >= E || (it != begin && *it <= *(it - 1))) ++disorder;
    for (int64_t e = 0; e < E; ++e) {
      bool out = false;
      for (int a = 0; a < dim; ++a) out = out || pt[a] < bbox[e * 2 * dim + a] || pt[a] > bbox[e * 2 * dim + dim + a];
      if (!out && !std::binary_search(begin, end, (int32_t)e)) ++missing;
    }
  }
  const bool many = nb > 1 && (int64_t)B.elem.size() > kMaxBinEntries * E;
  const bool ok = !missing && !disorder && !many && B.start[nb] == (int64_t)B.elem.size();
  std::printf("%s dim %d: %lld elements, %lld bins, %lld entries: %s\n", name, dim, (long long)E, (long long)nb,
              (long long)B.elem.size(), ok ? "ok" : "FAILED");
  failures += !ok;
}

int main() {
  std::mt19937_64 rng(7);
  const auto uni = [&](double lo, double hi) { return lo + (hi - lo) * std::uniform_real_distribution<double>()(rng); };
  const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
  for (int dim = 2; dim <= 3; ++dim) {
    const int n = dim == 2 ? 40 : 12;
    const auto grid = [&](double power) {  // a lattice of n^dim boxes, coordinates raised to `power`
      std::vector<double> b;
      for (int k = 0; k < (dim == 3 ? n : 1); ++k)
        for (int j = 0; j < n; ++j)
          for (int i = 0; i < n; ++i) {
            const int at[3] = {i, j, k};
            for (int h = 0; h < 2; ++h)
              for (int a = 0; a < dim; ++a) b.push_back(std::pow((at[a] + h) / (double)n, a == 0 ? power : 1.0));
          }
      return b;
    };
    const auto points = [&](const std::vector<double> &b, double lo, double hi) {
      std::vector<double> p;
      for (int i = 0; i < 200 * dim; ++i) p.push_back(uni(lo, hi));
      for (size_t e = 0; e < b.size() / (2 * dim); e += 7)  // corners of boxes too
        for (int h = 0; h < 2; ++h)
          for (int a = 0; a < dim; ++a)
            if (std::isfinite(b[e * 2 * dim + h * dim + a])) p.push_back(b[e * 2 * dim + h * dim + a]);
            else p.push_back(0.5);
      const double far[] = {-1e300, 1e300, inf, -inf, 0.0, -0.0, 1e-310};
      for (double x : far)
        for (int a = 0; a < dim; ++a) p.push_back(x);
      return p;
    };
    std::vector<double> b = grid(1.0);
    check("lattice", dim, b, points(b, -0.1, 1.1));
    b = grid(6.0);
    check("graded", dim, b, points(b, -0.1, 1.1));
    // needles along the diagonal, side by side: each box is nearly the whole domain
    const int ne = dim == 2 ? 4000 : 8000;
    b.clear();
    for (int e = 0; e < ne; ++e) {
      double lo[3];
      for (int a = 0; a < dim; ++a) b.push_back(lo[a] = a == 0 ? e / (double)ne * 0.01 : 0.0);
      for (int a = 0; a < dim; ++a) b.push_back(lo[a] + 1.0);
    }
    check("needles", dim, b, points(b, -0.1, 1.1));
    b.clear();
    for (int e = 0; e < 500; ++e) {
      double lo[3];
      for (int a = 0; a < dim; ++a) b.push_back(lo[a] = uni(-5, 5));
      for (int a = 0; a < dim; ++a) b.push_back(lo[a] + std::pow(10.0, uni(-6, 1)));
    }
    check("random", dim, b, points(b, -6, 6));
    // one element, a point-like one, extents past a double's range
    b.assign(2 * dim, 0.25);
    check("point", dim, b, points(b, 0, 1));
    for (int which = 0; which < 5; ++which) {
      b = grid(1.0);
      const size_t at = (b.size() / (2 * dim) / 2) * 2 * dim;
      const double values[5] = {inf, -inf, nan, 1e308, -1e308};
      b[at + (which & 1)] = which == 1 || which == 4 ? values[which] : b[at + (which & 1)];
      if (which != 1 && which != 4) b[at + dim + (which & 1)] = values[which];
      if (which == 2) b[at] = nan;
      check("one box not finite or far", dim, b, points(b, -0.1, 1.1));
    }
    b.clear();
    for (int e = 0; e < 20; ++e)
      for (int h = 0; h < 2; ++h)
        for (int a = 0; a < dim; ++a) b.push_back(e == 0 ? (h ? 1e308 : -1e308) : h ? inf : -inf);
    check("whole range", dim, b, points(b, -1, 1));
    b.assign(20 * 2 * dim, nan);
    check("no number", dim, b, points(b, -1, 1));
  }
  if (!failures) std::printf("all bins ok\n");
  return failures ? 1 : 0;
}
