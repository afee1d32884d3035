// lowrank.hpp -- the PSF of all planes as combinations of a few planes' PSFs
// (host code).
//
// For plans whose caller chose it (spect_plan_create_images).  The taps of plane
// i are a Gaussian (or any profile) whose width varies smoothly with the distance
// to the detector, so the planes' 2-D kernels k_i = y taps (x) z taps span,
// numerically, far fewer dimensions than there are planes: over a range of planes
// whose widths differ by at most a factor of two, about ten of them reproduce
// every other one to 2^-22 of its norm
// (128^3 at 4.8 mm, sigma = 0.03 d + 0.1 cm: 29 kernels for 182 planes).  With
//   k_i = sum_r c[i][r] k_(node r)
// the ray sum of blurred planes is the sum of a few blurred images,
//   sum_i k_i * V_i = sum_r k_(node r) * (sum_i c[i][r] V_i),
// and the blurred projection of every plane is a combination of a few.
//
// Planes are taken in units of 16 (one MFMA tile of planes).  Consecutive
// units form a group while their widths (plus kLrWidthOffset: narrow kernels
// reach few pixels whatever their ratio) stay within kLrRatio of each other: a
// node is then never much wider than the planes it stands for (one basis for all
// planes would need 20 images instead of 29, but puts 2^-24 of the widest
// kernel under the narrowest).  The planes' tails are not kept: where a plane's
// own tap is smaller, up to 6e-8 of its peak remains of the combination, and tap
// products above 1e-4 of the peak are off by up to 1.6e-3 of themselves.  Keeping
// every tap within 1e-6 of itself takes a width ratio of 1.2 and 90 images at
// 128^3, whose blurs cost as much as the planes'.  Consecutive groups whose nodes fill at most
// kLrRows rows share a segment (one MFMA tile of images).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <exception>
#include <system_error>
#include <thread>
#include <vector>

#include "tiers.hpp"

namespace spect {

constexpr int kLrUnit = 16;        // planes per unit
constexpr int kLrRows = 16;        // image rows per segment
constexpr int kLrMaxSegments = 8;  // segments per radius
constexpr double kLrTol = 1.0 / (1 << 22);
constexpr double kLrRatio = 2.0;
constexpr double kLrWidthOffset = 0.75;  // pixels

// Taps of an image are stored with zeros to either side, so that the entries of
// the Toeplitz tiles within reach (at most 16 ND + 15 from the centre) are all
// there: rows of this many, the centre in the middle.
inline int lr_tap_stride(int H) { return 2 * (16 * (H > 16 ? 2 : 1) + 15) + 1; }

// One radius: segments of whole units, and the images (nodes) of each.
struct LrRadius {
  std::vector<int> seg_unit;  // nseg + 1 unit bounds
  std::vector<int> seg_rows;  // nseg: rows in use
  struct Image {
    int seg, row, node, he;  // node: plane whose taps the image is blurred with
  };
  std::vector<Image> images;
  std::vector<double> coef;  // [P][kLrRows]: row weights of each plane in its segment
};

namespace lr_detail {

// Standard deviation of a plane's y taps in pixels.
template <typename T> double tap_width(const T *w, int H) {
  double s = 0.0, m = 0.0;
  for (int d = -H; d <= H; ++d) {
    s += std::fabs((double)w[H + d]);
    m += std::fabs((double)w[H + d]) * d * d;
  }
  return s > 0.0 ? std::sqrt(m / s) : 0.0;
}

// Nodes and coefficients of planes [lo, hi): pivoted Cholesky factorisation of
// the Gram matrix <k_i, k_j> = <y_i, y_j> <z_i, z_j> of the normalised
// kernels, stopped when every plane's remainder is below kLrTol (the squared
// remainders are held in extended precision: 2^-44 of the diagonal).  False
// when more than max_nodes are needed.
template <typename T>
bool fit_group(const T *ty, const T *tz, int H, int lo, int hi, int max_nodes, std::vector<int> &nodes,
               std::vector<double> &coef) {
  using X = long double;
  const int K = 2 * H + 1, n = hi - lo;
  auto dot = [&](const T *a, const T *b) {
    X s = 0;
    for (int t = 0; t < K; ++t) s += (X)a[t] * (X)b[t];
    return s;
  };
  std::vector<X> norm(n), rest(n, 1);
  for (int i = 0; i < n; ++i) {
    const T *y = ty + (size_t)(lo + i) * K, *z = tz + (size_t)(lo + i) * K;
    norm[i] = std::sqrt(dot(y, y) * dot(z, z));
    if (!(norm[i] > 0)) return false;
  }
  std::vector<std::vector<X>> L;  // L[r][i]: row r of the factor, over all planes
  nodes.clear();
  for (;;) {
    int k = 0;
    for (int i = 1; i < n; ++i)
      if (rest[i] > rest[k]) k = i;
    if (rest[k] <= (X)kLrTol * (X)kLrTol) break;
    if ((int)nodes.size() == max_nodes) return false;
    const X piv = std::sqrt(rest[k]);
    std::vector<X> row(n);
    const T *yk = ty + (size_t)(lo + k) * K, *zk = tz + (size_t)(lo + k) * K;
    for (int i = 0; i < n; ++i) {
      const T *y = ty + (size_t)(lo + i) * K, *z = tz + (size_t)(lo + i) * K;
      X v = dot(y, yk) * dot(z, zk) / (norm[i] * norm[k]);
      for (size_t r = 0; r < L.size(); ++r) v -= L[r][i] * L[r][k];
      row[i] = v / piv;
    }
    for (int i = 0; i < n; ++i) rest[i] = std::max((X)0, rest[i] - row[i] * row[i]);
    rest[k] = 0;
    nodes.push_back(k);
    L.push_back(std::move(row));
  }
  const int R = (int)nodes.size();
  // c = L_nodes^-T L_i per plane, rescaled from normalised kernels
  coef.assign((size_t)n * R, 0.0);
  std::vector<X> c(R);
  for (int i = 0; i < n; ++i) {
    const auto self = std::find(nodes.begin(), nodes.end(), i);
    if (self != nodes.end()) {
      coef[(size_t)i * R + (self - nodes.begin())] = 1.0;
      continue;
    }
    for (int r = R - 1; r >= 0; --r) {
      X v = L[r][i];
      for (int q = r + 1; q < R; ++q) v -= L[r][nodes[q]] * c[q];
      c[r] = v / L[r][nodes[r]];
    }
    for (int r = 0; r < R; ++r) coef[(size_t)i * R + r] = (double)(c[r] * norm[i] / norm[nodes[r]]);
  }
  for (int &k : nodes) k += lo;
  return true;
}

}  // namespace lr_detail

// The segments and images of one radius from its taps ([P][2H+1] each), or
// false when they do not pay: more than kLrMaxSegments segments, or more
// images than half the planes (a PSF that does not vary smoothly).
template <typename T>
bool lowrank_fit(const T *ty, const T *tz, int P, int H, LrRadius &out) {
  const int K = 2 * H + 1, units = (P + kLrUnit - 1) / kLrUnit;
  std::vector<double> width(P);
  for (int i = 0; i < P; ++i)
    width[i] = std::max(lr_detail::tap_width(ty + (size_t)i * K, H), lr_detail::tap_width(tz + (size_t)i * K, H));
  struct Group {
    int u0, u1;
    std::vector<int> nodes;
    std::vector<double> coef;
  };
  std::vector<Group> groups;
  for (int u = 0; u < units;) {
    // the longest run of units whose widths stay within the ratio, shortened
    // until it fits the rows
    int e = u;
    double lo = 1e300, hi = 0.0;
    while (e < units) {
      double l = lo, h = hi;
      for (int i = e * kLrUnit; i < std::min(P, (e + 1) * kLrUnit); ++i) {
        l = std::min(l, width[i] + kLrWidthOffset);
        h = std::max(h, width[i] + kLrWidthOffset);
      }
      if (e > u && h > kLrRatio * l) break;
      lo = l;
      hi = h;
      ++e;
    }
    Group g;
    for (; e > u; --e)
      if (lr_detail::fit_group(ty, tz, H, u * kLrUnit, std::min(P, e * kLrUnit), kLrRows, g.nodes, g.coef)) break;
    if (e == u) return false;
    g.u0 = u;
    g.u1 = e;
    groups.push_back(std::move(g));
    u = e;
  }
  out = LrRadius{};
  out.coef.assign((size_t)P * kLrRows, 0.0);
  for (const Group &g : groups) {
    const int R = (int)g.nodes.size();
    if (out.seg_rows.empty() || out.seg_rows.back() + R > kLrRows) {
      out.seg_unit.push_back(g.u0);
      out.seg_rows.push_back(0);
    }
    const int seg = (int)out.seg_rows.size() - 1, row0 = out.seg_rows.back();
    for (int r = 0; r < R; ++r) {
      const size_t t = (size_t)g.nodes[r] * K;
      out.images.push_back({seg, row0 + r, g.nodes[r], plane_half_width(ty + t, tz + t, H, kTierEps32)});
    }
    const int lo = g.u0 * kLrUnit, hi = std::min(P, g.u1 * kLrUnit);
    for (int i = lo; i < hi; ++i)
      for (int r = 0; r < R; ++r) out.coef[(size_t)i * kLrRows + row0 + r] = g.coef[(size_t)(i - lo) * R + r];
    out.seg_rows.back() += R;
  }
  out.seg_unit.push_back(units);
  return (int)out.seg_rows.size() <= kLrMaxSegments && 2 * (int)out.images.size() <= P;
}

// The tables of LrTables (lowrank_launch.hpp) for all radii.
struct LrHostTables {
  int nseg = 0, nimg = 0, quads = 0;
  struct Img {
    int32_t seg, row, he, unused;
  };
  std::vector<int32_t> seg_unit, seg_rows, count;
  std::vector<Img> img;
  std::vector<float> taps, cf, cb;
};

// Fits every radius (taps [n_radii][P][2H+1]) and packs the tables; false when
// a radius has no such representation or a tap is negative or not a number
// (the kernels clamp sums of non-negative samples at zero).
template <typename T>
bool lowrank_tables(const T *taps_y, const T *taps_z, int n_radii, int P, int H, LrHostTables &t) {
  const int K = 2 * H + 1, units = (P + kLrUnit - 1) / kLrUnit;
  for (size_t k = 0; k < (size_t)n_radii * P * K; ++k)
    if (!(taps_y[k] >= T(0)) || !(taps_z[k] >= T(0))) return false;
  // a body-contour orbit has a radius per angle, 0.1 to 0.6 ms each: a thread
  // per 16 radii, this one for those that the system does not give.  Nothing may
  // leave a thread, nor this function with threads running: the entry is C.
  std::vector<LrRadius> fits(n_radii);
  std::vector<char> ok(n_radii, 0);
  const int nt = std::max(1, std::min(8, n_radii / 16));
  auto work = [&](int first) noexcept {
    for (int r = first; r < n_radii; r += nt) {
      try {
        ok[r] = lowrank_fit<T>(taps_y + (size_t)r * P * K, taps_z + (size_t)r * P * K, P, H, fits[r]) ? 1 : 0;
      } catch (const std::exception &) {  // out of memory: blur planes
      }
    }
  };
  std::vector<std::thread> threads(nt);
  for (int k = 1; k < nt; ++k) {
    try {
      threads[k] = std::thread(work, k);
    } catch (const std::system_error &) {
      work(k);
    }
  }
  work(0);
  for (auto &th : threads)
    if (th.joinable()) th.join();
  t = LrHostTables{};
  for (int r = 0; r < n_radii; ++r) {
    if (!ok[r]) return false;
    t.nseg = std::max(t.nseg, (int)fits[r].seg_rows.size());
    t.nimg = std::max(t.nimg, (int)fits[r].images.size());
  }
  t.quads = 4 * units;
  t.seg_unit.assign((size_t)n_radii * (t.nseg + 1), units);
  t.seg_rows.assign((size_t)n_radii * t.nseg, 0);
  t.count.assign(n_radii, 0);
  t.img.assign((size_t)n_radii * t.nimg, {0, 0, 0, 0});
  const int KP = lr_tap_stride(H);
  t.taps.assign((size_t)n_radii * t.nimg * 2 * KP, 0.0f);
  t.cf.assign((size_t)n_radii * t.quads * 64, 0.0f);
  t.cb.assign((size_t)n_radii * units * 256, 0.0f);
  for (int r = 0; r < n_radii; ++r) {
    const LrRadius &f = fits[r];
    std::copy(f.seg_unit.begin(), f.seg_unit.end(), t.seg_unit.begin() + (size_t)r * (t.nseg + 1));
    std::copy(f.seg_rows.begin(), f.seg_rows.end(), t.seg_rows.begin() + (size_t)r * t.nseg);
    t.count[r] = (int)f.images.size();
    for (int k = 0; k < t.count[r]; ++k) {
      const auto &m = f.images[k];
      t.img[(size_t)r * t.nimg + k] = {m.seg, m.row, m.he, 0};
      for (int x = 0; x < K; ++x) {
        const size_t src = ((size_t)r * P + m.node) * K + x;
        const size_t dst = ((size_t)r * t.nimg + k) * 2 * KP + KP / 2 - H + x;
        t.taps[dst] = (float)taps_z[src];
        t.taps[dst + KP] = (float)taps_y[src];
      }
    }
    for (int i = 0; i < P; ++i)
      for (int q = 0; q < kLrRows; ++q) {
        const float c = (float)f.coef[(size_t)i * kLrRows + q];
        t.cf[((size_t)r * t.quads + i / 4) * 64 + (i % 4) * 16 + q] = c;
        t.cb[((size_t)r * units + i / 16) * 256 + (q / 4) * 64 + (q % 4) * 16 + i % 16] = c;
      }
  }
  return true;
}

}  // namespace spect
