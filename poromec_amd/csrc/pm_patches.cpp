// pm_patches.cpp -- which elements the element products serve (pm_affine.hip),
// and in which patches.  Plain host code without device calls.
#include "pm_patches.h"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <exception>
#include <functional>
#include <thread>
#include <utility>

// The bilinear and trilinear parts of the element's map, taken back to the
// reference cube by the linear part J: the map is J (I + E) with
// |E| <= 3 y for the largest component y, and the element's matrix differs from
// that of the parallelepiped by a few y of its norm, whatever the ratio of the
// edges (taken against the longest edge it would be that ratio times as much).
// 1e-12 is what coordinates i * h leave in a mesh of a few thousand cells a
// side.
bool pm_is_parallelepiped(const int *v, const double *x) {
  static const int sr[8] = {1, -1, -1, 1, 1, -1, -1, 1}, ss[8] = {1, 1, -1, -1, 1, 1, -1, -1},
                   st[8] = {1, 1, 1, 1, -1, -1, -1, -1};
  double c[7][3] = {};  // r, s, t, rs, st, rt, rst
  for (int k = 0; k < 8; k++) {
    const int s[7] = {sr[k], ss[k], st[k], sr[k] * ss[k], ss[k] * st[k], sr[k] * st[k],
                      sr[k] * ss[k] * st[k]};
    for (int d = 0; d < 3; d++) {
      const double xk = x[(size_t)(v[k] - 1) * 3 + d];
      for (int i = 0; i < 7; i++) c[i][d] += s[i] * xk;
    }
  }
  double adj[3][3];  // rows of det J J^-1
  for (int i = 0; i < 3; i++) {
    const double *a = c[(i + 1) % 3], *b = c[(i + 2) % 3];
    for (int d = 0; d < 3; d++)
      adj[i][d] = a[(d + 1) % 3] * b[(d + 2) % 3] - a[(d + 2) % 3] * b[(d + 1) % 3];
  }
  const double det = c[0][0] * adj[0][0] + c[0][1] * adj[0][1] + c[0][2] * adj[0][2];
  if (!std::isfinite(det) || det == 0.0) return false;
  for (int i = 0; i < 3; i++)
    for (int m = 3; m < 7; m++) {
      const double y = adj[i][0] * c[m][0] + adj[i][1] * c[m][1] + adj[i][2] * c[m][2];
      if (!(std::fabs(y) <= 1.0e-12 * std::fabs(det))) return false;
    }
  return true;
}

// Slots and patches: the elements of each connected part of the mesh split in
// two along its longest side (in mean element sizes), again and again, at
// multiples of L elements, so that only a part's last patch is not full.
//
// Centroids are kept in FP32 from the first element's corner: at map
// coordinates of 7e6 the neighbours of a 0.25 mesh would share theirs.
void pm_element_patches(int numel, int nen, int nnodev, const int *ix, const int *id,
                        const double *x, int L, std::vector<int> &ord, std::vector<int> &ps) {
  std::vector<float> cen((size_t)numel * 3);
  double size[3] = {0, 0, 0}, corner[3];
  for (int d = 0; d < 3; d++) {
    corner[d] = x[(size_t)(ix[0] - 1) * 3 + d];
    for (int k = 1; k < 8; k++) corner[d] = std::min(corner[d], x[(size_t)(ix[k] - 1) * 3 + d]);
  }
  std::vector<int> part((size_t)nnodev);
  for (int n = 0; n < nnodev; n++) part[n] = n;
  auto root = [&](int n) {
    while (part[n] != n) n = part[n] = part[part[n]];
    return n;
  };
  for (int e = 0; e < numel; e++) {
    const int *v = ix + (size_t)e * 21;
    const int r = root(v[0] - 1);
    for (int k = 1; k < 8; k++) {
      const int q = root(v[k] - 1);
      if (q != r) part[q] = r;
    }
    for (int d = 0; d < 3; d++) {
      double lo = x[(size_t)(v[0] - 1) * 3 + d], hi = lo, sum = 0.0;
      for (int k = 0; k < 8; k++) {
        const double xk = x[(size_t)(v[k] - 1) * 3 + d];
        lo = std::min(lo, xk);
        hi = std::max(hi, xk);
        sum += xk;
      }
      cen[(size_t)e * 3 + d] = (float)(0.125 * sum - corner[d]);
      size[d] += hi - lo;
    }
  }
  for (int d = 0; d < 3; d++)
    if (!(size[d] > 0.0)) size[d] = 1.0;
  for (int e = 0; e < numel; e++)
    for (int d = 0; d < 3; d++) cen[(size_t)e * 3 + d] *= (float)(numel / size[d]);
  // parts in the order of their lowest equation, as the matrix has them
  std::vector<int> key((size_t)nnodev, INT32_MAX);
  for (int e = 0; e < numel; e++) {
    int lo = INT32_MAX;
    for (int k = 0; k < nen; k++)
      for (int d = 0; d < 4; d++) {
        const int q = id[(size_t)(ix[(size_t)e * 21 + k] - 1) * 4 + d];
        if (q > 0) lo = std::min(lo, q);
      }
    int &kr = key[root(ix[(size_t)e * 21] - 1)];
    kr = std::min(kr, lo);
  }
  ord.resize((size_t)numel);
  std::vector<std::pair<int, int>> pk((size_t)numel);
  for (int e = 0; e < numel; e++) {
    const int r = root(ix[(size_t)e * 21] - 1);
    pk[e] = {key[r] == INT32_MAX ? INT32_MAX : key[r], r};
    ord[e] = e;
  }
  std::stable_sort(ord.begin(), ord.end(), [&](int a, int b) { return pk[a] < pk[b]; });
  std::function<void(int, int, int)> split = [&](int lo, int hi, int fork) {
    const int n = hi - lo;
    if (n <= L) return;
    float mn[3] = {1e30f, 1e30f, 1e30f}, mx[3] = {-1e30f, -1e30f, -1e30f};
    for (int i = lo; i < hi; i++)
      for (int d = 0; d < 3; d++) {
        const float v = cen[(size_t)ord[i] * 3 + d];
        mn[d] = std::min(mn[d], v);
        mx[d] = std::max(mx[d], v);
      }
    int ax = 0;
    for (int d = 1; d < 3; d++)
      if (mx[d] - mn[d] > (mx[ax] - mn[ax]) * 1.001f + 0.01f) ax = d;
    const int mid = lo + ((n + L - 1) / L) / 2 * L;
    std::nth_element(ord.begin() + lo, ord.begin() + mid, ord.begin() + hi, [&](int a, int b) {
      const float va = cen[(size_t)a * 3 + ax], vb = cen[(size_t)b * 3 + ax];
      return va != vb ? va < vb : a < b;
    });
    std::thread t;
    if (fork > 0 && n > 20000) {
      try {
        t = std::thread([&] { split(lo, mid, fork - 1); });
      } catch (const std::exception &) {  // no thread, or no memory for one
      }
    }
    // nothing below allocates but threads, so nothing throws past a running one
    if (!t.joinable()) split(lo, mid, fork - 1);
    split(mid, hi, fork - 1);
    if (t.joinable()) t.join();
  };
  ps.assign(1, 0);
  for (int a = 0; a < numel;) {
    int b = a + 1;
    while (b < numel && pk[ord[b]] == pk[ord[a]]) b++;
    split(a, b, 3);
    for (int q = a; q < b; q += L) ps.push_back(std::min(q + L, b));
    a = b;
  }
}
