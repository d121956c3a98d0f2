// Point location (host): bins over the elements' bounding boxes.  Standard
// library only, so that host checks compile it alone.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <vector>

namespace sem {

// The elements whose box meets bin b are elem[start[b] .. start[b + 1]),
// ascending.
struct ElementBins {
  int n[3] = {1, 1, 1};
  double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0}, inv[3] = {0, 0, 0};  // inv: bins per unit length
  std::vector<int64_t> start;
  std::vector<int32_t> elem;
  // bin coordinate of x along axis a; monotone in x
  int at(int a, double x) const {
    const double f = (x - lo[a]) * inv[a];
    return !(f > 0) ? 0 : f >= n[a] ? n[a] - 1 : (int)f;
  }
};

// Bins of about one element each over the box of E > 0 elements (bbox: per
// element dim lower, then dim upper bounds), filled by a counting sort in
// element order.  Where the boxes overlap so much that the bins would hold more
// than kMaxBinEntries elements for each element of the mesh (long thin elements
// across the axes: half of them of a 1:1000 needle's box each), the bins are
// made larger.  A box that is not finite counts as the whole axis: its element
// is a candidate everywhere, as in a scan over all of them.
constexpr int64_t kMaxBinEntries = 64;
inline void bin_elements(ElementBins &B, int dim, int64_t E, const double *bbox) {
  double cells = 1, w[3] = {0, 0, 0};
  for (int a = 0; a < dim; ++a) {
    B.lo[a] = 1e300;
    B.hi[a] = -1e300;
    for (int64_t e = 0; e < E; ++e) {
      const double l = bbox[e * 2 * dim + a], h = bbox[e * 2 * dim + dim + a];
      if (std::isfinite(l) && l < B.lo[a]) B.lo[a] = l;
      if (std::isfinite(h) && h > B.hi[a]) B.hi[a] = h;
    }
    w[a] = B.hi[a] - B.lo[a];
    cells *= std::max(w[a], 1e-300);
  }
  double h = std::pow(cells / (double)E, 1.0 / dim);  // about an element
  const double most = 4.0 * std::pow((double)E, 1.0 / dim) + 1.0;
  int64_t nb = 1;
  const auto each = [&](auto &&f) {
    for (int64_t e = 0; e < E; ++e) {
      const double *bb = &bbox[e * 2 * dim];
      int lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
      for (int a = 0; a < dim; ++a) {
        lo[a] = std::isfinite(bb[a]) ? B.at(a, bb[a]) : 0;
        hi[a] = std::isfinite(bb[dim + a]) ? B.at(a, bb[dim + a]) : B.n[a] - 1;
      }
      f((int32_t)e, lo, hi);
    }
  };
  for (;; h *= 2) {
    nb = 1;
    for (int a = 0; a < dim; ++a) {
      // (extents past the range of a double make h infinite: one bin)
      const double k = std::isfinite(h) && std::isfinite(w[a]) && h > 0 ? w[a] / h : 1.0;
      B.n[a] = (int)std::min(std::max(k, 1.0), most);
      B.inv[a] = w[a] > 0 && std::isfinite(w[a]) ? B.n[a] / w[a] : 0.0;
      nb *= B.n[a];
    }
    int64_t entries = 0;
    each([&](int32_t, const int *lo, const int *hi) {
      entries += (int64_t)(hi[0] - lo[0] + 1) * (hi[1] - lo[1] + 1) * (hi[2] - lo[2] + 1);
    });
    if (nb == 1 || entries <= kMaxBinEntries * E) break;
  }
  const auto bins_of = [&](auto &&f) {
    each([&](int32_t e, const int *lo, const int *hi) {
      for (int z = lo[2]; z <= hi[2]; ++z)
        for (int y = lo[1]; y <= hi[1]; ++y)
          for (int x = lo[0]; x <= hi[0]; ++x) f(x + (int64_t)B.n[0] * (y + (int64_t)B.n[1] * z), e);
    });
  };
  B.start.assign(nb + 1, 0);
  bins_of([&](int64_t b, int32_t) { ++B.start[b + 1]; });
  for (int64_t b = 0; b < nb; ++b) B.start[b + 1] += B.start[b];
  B.elem.resize(B.start[nb]);
  std::vector<int64_t> cur(B.start.begin(), B.start.end() - 1);
  bins_of([&](int64_t b, int32_t e) { B.elem[cur[b]++] = e; });
}

// The bin of a point that is no NaN.
inline int64_t bin_of(const ElementBins &B, int dim, const double *pt) {
  int64_t bin = 0;
  for (int a = dim - 1; a >= 0; --a) bin = bin * B.n[a] + B.at(a, pt[a]);
  return bin;
}

}  // namespace sem
