// pm_patches.cpp -- which elements the element products serve (pm_affine.hip).
// Plain host code without device calls.
#include "pm_patches.h"

#include <cmath>
#include <cstddef>

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
