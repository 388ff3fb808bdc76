// pm_affine.hip -- element loops and matrix products over parallelepiped
// elements, without forming element matrices.
//
// On an element with a constant Jacobian the integrals of elmt17_pm
// (Elmlib03.f:2022-2526) and of the Q1/Q1 element separate in the products
// of Legendre polynomials P_a(r) P_b(s) P_c(t): the 20 serendipity functions
// span the products with at most one degree 2 and the others <= 1, the 8
// trilinear ones those with degrees <= 1.  In that basis
//   * nodal values become coefficients by sums and differences of the
//     vertices and of the mid-edges (pm_modal_fwd; the transpose
//     pm_modal_back takes coefficient forces to nodal forces),
//   * a derivative moves a coefficient one degree down (P1' = P0, P2' = 3 P1),
//   * the 4^3 (2^3) Gauss rule is exact for every product that occurs, so the
//     17 derivative modes are orthogonal and D acts on each mode alone.
// An element's K_e u_e is then 1,624 FP64 instructions (Q1/Q1 637) instead of
// the 64-point loops' ~2 million operations, and needs its 15 coefficients
// (128 B) instead of the matrix's 37 KB of stored values.
//
// In large meshes a lane takes an element (2,800 vector instructions a
// wavefront of 64, patch and scalars included).  In small ones four lanes do:
// lanes 0-2 one displacement component each, lane 3 the pressure; the stress of
// a mode exchanges gradients inside the quad by DPP (four wavefronts of 1,600
// for the same 64).  A wavefront sums the vectors of its 64 or 16 neighbouring
// elements in LDS and writes the patch's nodes to ye; a second kernel sums
// every node's patches in a fixed order: no colours, the same result every
// time.
#include <algorithm>
#include <cstring>
#include <new>

#include "pm_affine.h"
#include "pm_elemlib.h"
#include "pm_fused.h"
#include "pm_patches.h"

#define PM_EC 16  // doubles of element coefficients
// 0-8 g[i][x] = d r_i / d x, then det J times: 9 a (1 - b), 10 a b, 11 a c,
// 12 alpha, 13 1/M, 14 dt perm (+ the Q1/Q1 stabilization), 15 one

template <int CTRL>
__device__ __forceinline__ double pm_quad(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffll), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xf, 0xf, true);
  return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned int)lo);
}
#define PM_QP(a, b, c, d) ((a) | ((b) << 2) | ((c) << 4) | ((d) << 6))

__host__ __device__ constexpr int pm_md(int a, int b, int c) { return a * 9 + b * 3 + c; }
// modes of the element's displacement basis
template <int NEN>
__host__ __device__ constexpr bool pm_is_mode(int a, int b, int c) {
  const int twos = (a == 2) + (b == 2) + (c == 2);
  return a <= 2 && b <= 2 && c <= 2 && twos <= (NEN == 20 ? 1 : 0);
}

// sums and differences of the 8 vertex values (not scaled): h[a*4+b*2+c]
__host__ __device__ __forceinline__ void pm_hadamard8(const double *v, double *h) {
#pragma unroll
  for (int c = 0; c < 2; c++) {
    double q[4];
#pragma unroll
    for (int k = 0; k < 4; k++) q[k] = c == 0 ? v[k] + v[k + 4] : v[k] - v[k + 4];
    // vertices of a face: 0 (+,+), 1 (-,+), 2 (-,-), 3 (+,-)
    const double p1 = q[0] + q[1], m1 = q[0] - q[1], p2 = q[3] + q[2], m2 = q[3] - q[2];
    h[0 + c] = p1 + p2;
    h[2 + c] = p1 - p2;
    h[4 + c] = m1 + m2;
    h[6 + c] = m1 - m2;
  }
}
// the transpose: h[a*4+b*2+c] to the 8 vertices
__device__ __forceinline__ void pm_hadamard8t(const double *h, double *v) {
  double q[2][4];
#pragma unroll
  for (int c = 0; c < 2; c++) {
    const double p1 = h[0 + c] + h[2 + c], p2 = h[0 + c] - h[2 + c];
    const double m1 = h[4 + c] + h[6 + c], m2 = h[4 + c] - h[6 + c];
    q[c][0] = p1 + m1;
    q[c][1] = p1 - m1;
    q[c][3] = p2 + m2;
    q[c][2] = p2 - m2;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) {
    v[k] = q[0][k] + q[1][k];
    v[k + 4] = q[0][k] - q[1][k];
  }
}
// the 4 mid-edges of one direction, given in the order (+,+), (-,+), (-,-),
// (+,-) of the two other directions' signs: e[b*2+c]
__host__ __device__ __forceinline__ void pm_hadamard4(double a, double b, double c, double d, double *e) {
  const double p1 = a + b, m1 = a - b, p2 = d + c, m2 = d - c;
  e[0] = p1 + p2;  // 1
  e[1] = p1 - p2;  // second sign
  e[2] = m1 + m2;  // first sign
  e[3] = m1 - m2;
}

// nodal values -> Legendre coefficients.  kap = 2/3 for a displacement
// component; 0 for the pressure, whose degree-2 coefficients vanish (its
// mid-edge values are passed as zero).
template <int NEN>
__host__ __device__ __forceinline__ void pm_modal_fwd(const double *v, double kap, double *co) {
  double h[8];
  pm_hadamard8(v, h);
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] *= 0.125;
  if constexpr (NEN == 8) {
#pragma unroll
    for (int i = 0; i < 8; i++) co[pm_md(i >> 2, (i >> 1) & 1, i & 1)] = h[i];
    return;
  } else {
    double er[4], es[4], et[4];
    // first/second sign: (t, s) for r-edges, (t, r) for s-edges, (s, r) for t-edges
    pm_hadamard4(v[8], v[12], v[14], v[10], er);
    pm_hadamard4(v[11], v[15], v[13], v[9], es);
    pm_hadamard4(v[16], v[19], v[18], v[17], et);
    double b[8];
#pragma unroll
    for (int i = 0; i < 8; i++) b[i] = h[i];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        // (2, b = p, c = q): e index = first sign t (c), second sign s (b)
        const double c2 = kap * (h[0 * 4 + p * 2 + q] - 0.25 * er[q * 2 + p]);
        co[pm_md(2, p, q)] = c2;
        b[0 * 4 + p * 2 + q] -= c2;
        // (a = p, 2, c = q)
        const double d2 = kap * (h[p * 4 + 0 * 2 + q] - 0.25 * es[q * 2 + p]);
        co[pm_md(p, 2, q)] = d2;
        b[p * 4 + 0 * 2 + q] -= d2;
        // (a = p, b = q, 2)
        const double f2 = kap * (h[p * 4 + q * 2 + 0] - 0.25 * et[q * 2 + p]);
        co[pm_md(p, q, 2)] = f2;
        b[p * 4 + q * 2 + 0] -= f2;
      }
#pragma unroll
    for (int i = 0; i < 8; i++) co[pm_md(i >> 2, (i >> 1) & 1, i & 1)] = b[i];
  }
}

// coefficient forces -> nodal forces (the transpose of pm_modal_fwd)
template <int NEN>
__device__ __forceinline__ void pm_modal_back(const double *f, double kap, double *v) {
  double h[8];
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] = f[pm_md(i >> 2, (i >> 1) & 1, i & 1)];
  if constexpr (NEN == 20) {
    double base[8], er[4], es[4], et[4];
#pragma unroll
    for (int i = 0; i < 8; i++) base[i] = h[i];
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const double w1 = kap * (f[pm_md(2, p, q)] - base[0 * 4 + p * 2 + q]);
        h[0 * 4 + p * 2 + q] += w1;
        er[q * 2 + p] = -0.25 * w1;
        const double w2 = kap * (f[pm_md(p, 2, q)] - base[p * 4 + 0 * 2 + q]);
        h[p * 4 + 0 * 2 + q] += w2;
        es[q * 2 + p] = -0.25 * w2;
        const double w3 = kap * (f[pm_md(p, q, 2)] - base[p * 4 + q * 2 + 0]);
        h[p * 4 + q * 2 + 0] += w3;
        et[q * 2 + p] = -0.25 * w3;
      }
    auto edge = [](const double *e, double &pp, double &mp, double &mm, double &pm) {
      const double a = e[0] + e[1], b = e[0] - e[1], c = e[2] + e[3], d = e[2] - e[3];
      pp = a + c;  // first +, second +
      mp = a - c;  // first -, second +
      pm = b + d;  // first +, second -
      mm = b - d;
    };
    edge(er, v[8], v[12], v[14], v[10]);
    edge(es, v[11], v[15], v[13], v[9]);
    edge(et, v[16], v[19], v[18], v[17]);
  }
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] *= 0.125;
  pm_hadamard8t(h, v);
}

struct AffineArgs {
  int npatch, max_nodes;
  const int *ps;             // (npatch + 1) first slot of each patch
  const unsigned int *pn;    // (npatch + 1) first entry of each patch in pw
  const unsigned int *pw;    // free-dof words of the patches' nodes
  const unsigned short *loc; // (numel, nen) patch node of each element node
  const int *ord;
  const double *ec;
  double *ye;
  const double *x;  // equation vector (OP)
  const int *ix;    // (numel, nen) nodes (RHS2, RHS4)
  const double *u;  // (nnode, 4)
  const double *dp; // (nnode)
  const int *mat;
  const double *e;  // (numat, 15)
  double grav[3];
  const PmScalars *S;
};

enum { AF_OP = 0, AF_RHS2 = 1, AF_RHS4 = 2 };

// One lane's share of an element vector: the nodal values v of component c (3:
// pressure) become the nodal forces of K_e, or (AF_RHS4) of isw 4.
template <int NEN, int MODE>
__device__ __forceinline__ void pm_element_vector(const AffineArgs &A, int slot, int c, double *v,
                                                  const double *dpv) {
  const double *ec = A.ec + (size_t)slot * PM_EC;
  // the lane's physical axes in cyclic order: its own first (lane 3: x, y, z)
  double g[3][3];
#pragma unroll
  for (int k = 0; k < 3; k++) {
    int ax = (c == 3 ? 0 : c) + k;
    ax = ax >= 3 ? ax - 3 : ax;
#pragma unroll
    for (int i = 0; i < 3; i++) g[k][i] = ec[3 * i + ax];
  }
  const bool pr = c == 3;
  const double dtk = ec[14];
  const double cA = pr ? -dtk : ec[9], cB = pr ? 0.0 : ec[10], cC = pr ? -dtk : ec[11];
  const double cR = pr ? 0.0 : 1.0, cP = pr ? 0.0 : -ec[12];
  const double cM = pr ? -ec[13] : 0.0, cT = pr ? -ec[12] : 0.0;
  const double kap = pr ? 0.0 : 2.0 / 3.0;
  double co[27], f[27], dpm[8];
  pm_modal_fwd<NEN>(v, kap, co);
  if constexpr (MODE == AF_RHS4) pm_hadamard8(dpv, dpm);  // every lane holds dp
#pragma unroll
  for (int i = 0; i < 27; i++) f[i] = 0.0;
  constexpr double nrm[3] = {2.0, 2.0 / 3.0, 2.0 / 5.0};
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
      for (int d = 0; d < 3; d++) {
        if (!pm_is_mode<NEN>(a, b, d)) continue;
        const bool hr = a < 2 && pm_is_mode<NEN>(a + 1, b, d);
        const bool hs = b < 2 && pm_is_mode<NEN>(a, b + 1, d);
        const bool ht = d < 2 && pm_is_mode<NEN>(a, b, d + 1);
        const bool base = a < 2 && b < 2 && d < 2;  // a pressure mode
        if (!hr && !hs && !ht && !base) continue;
        const double nd = nrm[a] * nrm[b] * nrm[d];
        const double sr = a == 1 ? 3.0 : 1.0, ss = b == 1 ? 3.0 : 1.0, st = d == 1 ? 3.0 : 1.0;
        double F[3] = {0.0, 0.0, 0.0};
        if (hr || hs || ht) {
          const double dr = hr ? sr * co[pm_md(a + 1, b, d)] : 0.0;
          const double ds = hs ? ss * co[pm_md(a, b + 1, d)] : 0.0;
          const double dt = ht ? st * co[pm_md(a, b, d + 1)] : 0.0;
#pragma unroll
          for (int k = 0; k < 3; k++) {
            double s = 0.0;
            if (hr) s = g[k][0] * dr;
            if (hs) s = hr ? fma(g[k][1], ds, s) : g[k][1] * ds;
            if (ht) s = (hr || hs) ? fma(g[k][2], dt, s) : g[k][2] * dt;
            F[k] = s;
          }
          const double tr = pm_quad<PM_QP(0, 0, 0, 0)>(F[0]) + pm_quad<PM_QP(1, 1, 1, 1)>(F[0]) +
                            pm_quad<PM_QP(2, 2, 2, 2)>(F[0]);
          // shear partners: lane c + 1's gradient along c is its third in
          // cyclic order, lane c + 2's its second
          const double r1 = pm_quad<PM_QP(1, 2, 0, 3)>(F[2]);
          const double r2 = pm_quad<PM_QP(2, 0, 1, 3)>(F[1]);
          double s0 = fma(cB, tr, cA * F[0]);
          if (base) {
            const double p = MODE == AF_RHS4 ? 0.125 * dpm[a * 4 + b * 2 + d]
                                             : pm_quad<PM_QP(3, 3, 3, 3)>(co[pm_md(a, b, d)]);
            s0 = fma(cP, p, s0);
          }
          double s1 = cC * fma(cR, r1, F[1]);
          double s2 = cC * fma(cR, r2, F[2]);
          if (MODE == AF_RHS4 && a + b + d == 0) {  // gravity's flux dt perm rho_f g
            const double *em = A.e + (size_t)A.mat[A.ord[slot]] * PM_PROP;
            const double fd = pr ? em[6] * 1.0e-06 * dtk : 0.0;
            s0 = fma(fd, A.grav[0], s0);
            s1 = fma(fd, A.grav[1], s1);
            s2 = fma(fd, A.grav[2], s2);
          }
          s0 *= nd;
          s1 *= nd;
          s2 *= nd;
          if (hr) {
            const double q = fma(g[2][0], s2, fma(g[1][0], s1, g[0][0] * s0));
            f[pm_md(a + 1, b, d)] = fma(sr, q, f[pm_md(a + 1, b, d)]);
          }
          if (hs) {
            const double q = fma(g[2][1], s2, fma(g[1][1], s1, g[0][1] * s0));
            f[pm_md(a, b + 1, d)] = fma(ss, q, f[pm_md(a, b + 1, d)]);
          }
          if (ht) {
            const double q = fma(g[2][2], s2, fma(g[1][2], s1, g[0][2] * s0));
            f[pm_md(a, b, d + 1)] = fma(st, q, f[pm_md(a, b, d + 1)]);
          }
          if (base && MODE != AF_RHS4) f[pm_md(a, b, d)] = fma(nd * cT, tr, f[pm_md(a, b, d)]);
        }
        if (base && MODE != AF_RHS4)
          f[pm_md(a, b, d)] = fma(nd * cM, co[pm_md(a, b, d)], f[pm_md(a, b, d)]);
        if (MODE == AF_RHS4 && a + b + d == 0) {  // - rho g on the displacement rows
          const double *em = A.e + (size_t)A.mat[A.ord[slot]] * PM_PROP;
          const double gc = c == 0 ? A.grav[0] : c == 1 ? A.grav[1] : c == 2 ? A.grav[2] : 0.0;
          f[0] -= nd * ec[15] * (em[5] * 1.0e-06) * gc;
        }
      }
  pm_modal_back<NEN>(f, kap, v);
}

// The same with one lane per element, all four components in its registers:
// no exchanges, a quarter of the instructions per element; for meshes large
// enough to fill the chip with 64 elements a wavefront.  x: 4 components of
// every node on entry, the nodal forces on exit.  The transforms' 1/8 each way
// and the modes' norms are folded into the material coefficients.
template <int NEN>
__device__ __forceinline__ void pm_modal_fwd8(const double *v, double *co) {  // 8 x coefficients
  double h[8];
  pm_hadamard8(v, h);
  if constexpr (NEN == 20) {
    double er[4], es[4], et[4];
    pm_hadamard4(v[8], v[12], v[14], v[10], er);
    pm_hadamard4(v[11], v[15], v[13], v[9], es);
    pm_hadamard4(v[16], v[19], v[18], v[17], et);
    double b[8];
#pragma unroll
    for (int i = 0; i < 8; i++) b[i] = h[i];
    constexpr double k1 = 2.0 / 3.0, k2 = -4.0 / 3.0;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const double c2 = fma(k2, er[q * 2 + p], k1 * h[0 * 4 + p * 2 + q]);
        const double d2 = fma(k2, es[q * 2 + p], k1 * h[p * 4 + 0 * 2 + q]);
        const double f2 = fma(k2, et[q * 2 + p], k1 * h[p * 4 + q * 2 + 0]);
        co[pm_md(2, p, q)] = c2;
        co[pm_md(p, 2, q)] = d2;
        co[pm_md(p, q, 2)] = f2;
        b[0 * 4 + p * 2 + q] -= c2;
        b[p * 4 + 0 * 2 + q] -= d2;
        b[p * 4 + q * 2 + 0] -= f2;
      }
#pragma unroll
    for (int i = 0; i < 8; i++) h[i] = b[i];
  }
#pragma unroll
  for (int i = 0; i < 8; i++) co[pm_md(i >> 2, (i >> 1) & 1, i & 1)] = h[i];
}

// 8 x the transpose
template <int NEN>
__device__ __forceinline__ void pm_modal_back8(const double *f, double *v) {
  double h[8];
#pragma unroll
  for (int i = 0; i < 8; i++) h[i] = f[pm_md(i >> 2, (i >> 1) & 1, i & 1)];
  if constexpr (NEN == 20) {
    double base[8], er[4], es[4], et[4];
#pragma unroll
    for (int i = 0; i < 8; i++) base[i] = h[i];
    constexpr double k1 = 2.0 / 3.0, k2 = -4.0 / 3.0;
#pragma unroll
    for (int p = 0; p < 2; p++)
#pragma unroll
      for (int q = 0; q < 2; q++) {
        const double w1 = f[pm_md(2, p, q)] - base[0 * 4 + p * 2 + q];
        const double w2 = f[pm_md(p, 2, q)] - base[p * 4 + 0 * 2 + q];
        const double w3 = f[pm_md(p, q, 2)] - base[p * 4 + q * 2 + 0];
        h[0 * 4 + p * 2 + q] = fma(k1, w1, h[0 * 4 + p * 2 + q]);
        h[p * 4 + 0 * 2 + q] = fma(k1, w2, h[p * 4 + 0 * 2 + q]);
        h[p * 4 + q * 2 + 0] = fma(k1, w3, h[p * 4 + q * 2 + 0]);
        er[q * 2 + p] = k2 * w1;
        es[q * 2 + p] = k2 * w2;
        et[q * 2 + p] = k2 * w3;
      }
    auto edge = [](const double *e, double &pp, double &mp, double &mm, double &pm) {
      const double a = e[0] + e[1], b = e[0] - e[1], c = e[2] + e[3], d = e[2] - e[3];
      pp = a + c;
      mp = a - c;
      pm = b + d;
      mm = b - d;
    };
    edge(er, v[8], v[12], v[14], v[10]);
    edge(es, v[11], v[15], v[13], v[9]);
    edge(et, v[16], v[19], v[18], v[17]);
  }
  pm_hadamard8t(h, v);
}

// adds v to f, or starts it
__device__ __forceinline__ void pm_acc(bool &on, double &f, double k, double v) {
  f = on ? fma(k, v, f) : k * v;
  on = true;
}

template <int NEN, int MODE>
__device__ __forceinline__ void pm_element_lane(const AffineArgs &A, int slot,
                                                double (&x)[4][NEN], const double *dpv) {
  const double *ec = A.ec + (size_t)slot * PM_EC;
  double g[3][3];  // g[i][y] = d r_i / d y
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int y = 0; y < 3; y++) g[i][y] = ec[3 * i + y];
  constexpr double s64 = 1.0 / 64.0;
  const double cA = s64 * ec[9], cB = s64 * ec[10], cC = s64 * ec[11], cP = -s64 * ec[12];
  const double cM = -s64 * ec[13], cK = -s64 * ec[14];
  double co[4][27], f[4][27];
#pragma unroll
  for (int c = 0; c < 3; c++) pm_modal_fwd8<NEN>(x[c], co[c]);
  pm_modal_fwd8<8>(x[3], co[3]);
  double dpm[8];
  if constexpr (MODE == AF_RHS4) pm_hadamard8(dpv, dpm);
  bool fon[4][27];
#pragma unroll
  for (int c = 0; c < 4; c++)
#pragma unroll
    for (int i = 0; i < 27; i++) {
      fon[c][i] = false;
      f[c][i] = 0.0;
    }
  constexpr double nrm[3] = {2.0, 2.0 / 3.0, 2.0 / 5.0};
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
      for (int d = 0; d < 3; d++) {
        if (!pm_is_mode<NEN>(a, b, d)) continue;
        const int e[3] = {a, b, d};
        const double nd = nrm[a] * nrm[b] * nrm[d];
        const bool base = a < 2 && b < 2 && d < 2;
        const int m = pm_md(a, b, d);
        bool has[3], hasp[3];
        int src[3];
        double sc[3];
#pragma unroll
        for (int i = 0; i < 3; i++) {
          const int q[3] = {a + (i == 0), b + (i == 1), d + (i == 2)};
          has[i] = e[i] < 2 && pm_is_mode<NEN>(q[0], q[1], q[2]);
          hasp[i] = e[i] < 1 && pm_is_mode<8>(q[0], q[1], q[2]);
          src[i] = q[0] * 9 + q[1] * 3 + q[2];
          sc[i] = e[i] == 1 ? 3.0 : 1.0;
        }
        const bool any = has[0] || has[1] || has[2];
        double tr = 0.0;
        if (any) {
          double F[3][3];  // F[u][y] = d u / d y
#pragma unroll
          for (int u = 0; u < 3; u++) {
            bool on[3] = {false, false, false};
#pragma unroll
            for (int i = 0; i < 3; i++) {
              if (!has[i]) continue;
              const double di = sc[i] == 1.0 ? co[u][src[i]] : sc[i] * co[u][src[i]];
#pragma unroll
              for (int y = 0; y < 3; y++) {
                F[u][y] = on[y] ? fma(g[i][y], di, F[u][y]) : g[i][y] * di;
                on[y] = true;
              }
            }
          }
          tr = F[0][0] + F[1][1] + F[2][2];
          double T = (nd * cB) * tr;
          if (base) T = fma(nd * cP, MODE == AF_RHS4 ? dpm[a * 4 + b * 2 + d] : co[3][m], T);
          double S[3][3];
#pragma unroll
          for (int u = 0; u < 3; u++) S[u][u] = fma(nd * cA, F[u][u], T);
          S[0][1] = S[1][0] = (nd * cC) * (F[0][1] + F[1][0]);
          S[1][2] = S[2][1] = (nd * cC) * (F[1][2] + F[2][1]);
          S[0][2] = S[2][0] = (nd * cC) * (F[0][2] + F[2][0]);
#pragma unroll
          for (int u = 0; u < 3; u++)
#pragma unroll
            for (int i = 0; i < 3; i++) {
              if (!has[i]) continue;
              const double q = fma(g[i][2], S[u][2], fma(g[i][1], S[u][1], g[i][0] * S[u][0]));
              if (sc[i] == 1.0) {
                f[u][src[i]] = fon[u][src[i]] ? f[u][src[i]] + q : q;
                fon[u][src[i]] = true;
              } else {
                pm_acc(fon[u][src[i]], f[u][src[i]], sc[i], q);
              }
            }
        }
        if (hasp[0] || hasp[1] || hasp[2]) {
          double P[3];
          bool on = false;
#pragma unroll
          for (int i = 0; i < 3; i++) {
            if (!hasp[i]) continue;
#pragma unroll
            for (int y = 0; y < 3; y++)
              P[y] = on ? fma(g[i][y], co[3][src[i]], P[y]) : g[i][y] * co[3][src[i]];
            on = true;
          }
#pragma unroll
          for (int y = 0; y < 3; y++) P[y] *= nd * cK;
          if (MODE == AF_RHS4 && a + b + d == 0) {  // gravity's flux dt perm rho_f g
            const double *em = A.e + (size_t)A.mat[A.ord[slot]] * PM_PROP;
            const double fd = nd * 0.125 * ec[14] * (em[6] * 1.0e-06);
#pragma unroll
            for (int y = 0; y < 3; y++) P[y] = fma(fd, A.grav[y], P[y]);
          }
#pragma unroll
          for (int i = 0; i < 3; i++) {
            if (!hasp[i]) continue;
            const double q = fma(g[i][2], P[2], fma(g[i][1], P[1], g[i][0] * P[0]));
            f[3][src[i]] = fon[3][src[i]] ? f[3][src[i]] + q : q;
            fon[3][src[i]] = true;
          }
        }
        if (base && MODE != AF_RHS4) {
          pm_acc(fon[3][m], f[3][m], nd * cM, co[3][m]);
          if (any) pm_acc(fon[3][m], f[3][m], nd * cP, tr);
        }
        if (MODE == AF_RHS4 && a + b + d == 0) {  // - rho g on the displacement rows
          const double *em = A.e + (size_t)A.mat[A.ord[slot]] * PM_PROP;
          const double w = -nd * 0.125 * ec[15] * (em[5] * 1.0e-06);
#pragma unroll
          for (int u = 0; u < 3; u++) pm_acc(fon[u][m], f[u][m], w, A.grav[u]);
        }
      }
#pragma unroll
  for (int c = 0; c < 3; c++) pm_modal_back8<NEN>(f[c], x[c]);
  pm_modal_back8<8>(f[3], x[3]);
}

// ---------------------------------------------------------------------------
// patches
// ---------------------------------------------------------------------------
// A wavefront takes a patch of up to 64 (16) elements, a brick of 4 x 4 x 4
// (4 x 2 x 2) in a box.  It reads every node of the patch once into LDS, forms
// the element vectors, adds them up in LDS and writes one vector per patch
// node: 425 (141) nodes for 1280 (320) element nodes with hexa20/8, 125 (45)
// for 512 (128) with Q1/Q1.  The additions are LDS atomics
// in a fixed order: a wavefront's instructions execute in turn, and within
// one no two elements share the node (checked when the patches are built).
//
// Large meshes wait for memory (hexa20/8 87^3: 1.6 GFLOP, 46 us of issue and
// 0.4 GB in 199 us; 425 nodes of LDS allow eleven wavefronts a CU), small ones
// for the chain load, transform, stress, transform, store (24^3: 10.8 us).
// With the node part the product of an SQMR iteration takes 0.37 ms at 87^3
// against 2.9 ms from the stored matrix in FP64 and 1.9 in FP32, Q1/Q1 64^3
// 38 us against 192 and 118; without patches it was 71 us there, with patches
// of four lanes an element 54.
__device__ __forceinline__ void pm_wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// wavefronts of a workgroup: two where a patch's nodes take 14 KB of LDS
__host__ __device__ constexpr int pm_patch_waves(int nen, int lpe) {
  return nen == 20 && lpe == 1 ? 2 : PM_WAVES;
}

// doubles of LDS a wavefront needs: the patch's nodes and a dummy for
// restrained ones, four values each
__host__ __device__ inline int pm_patch_lds(int max_nodes) { return (max_nodes + 1) * 4; }

// four lanes an element: buf holds the patch nodes' values (AF_OP) on entry and
// their sums on exit, n4 = 4 * nodes values; written to ye
template <int NEN, int MODE>
__device__ __forceinline__ void pm_patch(const AffineArgs &A, int p, int lane, int n4, double *buf) {
  const int c = lane & 3;
  const int slot = A.ps[p] + (lane >> 2);
  const bool on = slot < A.ps[p + 1];
  double v[NEN], dpv[8];
  int l[NEN];
  if (on) {
    const uint2 *lp = reinterpret_cast<const uint2 *>(A.loc + (size_t)slot * NEN);
#pragma unroll
    for (int k = 0; k < NEN / 4; k++) {
      const uint2 q = lp[k];
      l[4 * k] = (int)(q.x & 0xffffu) * 4 + c;
      l[4 * k + 1] = (int)(q.x >> 16) * 4 + c;
      l[4 * k + 2] = (int)(q.y & 0xffffu) * 4 + c;
      l[4 * k + 3] = (int)(q.y >> 16) * 4 + c;
    }
    if constexpr (MODE == AF_OP) {
#pragma unroll
      for (int k = 0; k < NEN; k++) v[k] = buf[l[k]];
    } else {
      const int4 *np = reinterpret_cast<const int4 *>(A.ix + (size_t)A.ord[slot] * NEN);
      int no[NEN];
#pragma unroll
      for (int k = 0; k < NEN / 4; k++) {
        const int4 q = np[k];
        no[4 * k] = q.x;
        no[4 * k + 1] = q.y;
        no[4 * k + 2] = q.z;
        no[4 * k + 3] = q.w;
      }
#pragma unroll
      for (int k = 0; k < NEN; k++) v[k] = (k < 8 || c < 3) ? A.u[(size_t)no[k] * 4 + c] : 0.0;
      if constexpr (MODE == AF_RHS4)
#pragma unroll
        for (int k = 0; k < 8; k++) dpv[k] = A.dp[no[k]];
    }
    pm_element_vector<NEN, MODE>(A, slot, c, v, dpv);
  }
  pm_wave_lds_fence();  // every element has its values: the buffer turns into the sums
  for (int i = lane; i < n4 + 4; i += 64) buf[i] = 0.0;
  pm_wave_lds_fence();
  if (on) {
#pragma unroll
    for (int k = 0; k < NEN; k++)
      if (k < 8 || c < 3)
        __hip_atomic_fetch_add(&buf[l[k]], v[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
  pm_wave_lds_fence();
  double *y = A.ye + (size_t)A.pn[p] * 4;
  for (int i = lane; i < n4; i += 64) y[i] = buf[i];
  pm_wave_lds_fence();
}

// One lane an element, 64 elements a patch.  buf is component-major here (ld
// values a component), so that the lanes' nodes fall on different banks.
template <int NEN, int MODE>
__device__ __forceinline__ void pm_patch_lane(const AffineArgs &A, int p, int lane, int n4, int ld,
                                              double *buf) {
  const int slot = A.ps[p] + lane;
  const bool on = slot < A.ps[p + 1];
  double x[4][NEN], dpv[8];
  int l[NEN];
  if (on) {
    const uint2 *lp = reinterpret_cast<const uint2 *>(A.loc + (size_t)slot * NEN);
#pragma unroll
    for (int k = 0; k < NEN / 4; k++) {
      const uint2 q = lp[k];
      l[4 * k] = (int)(q.x & 0xffffu);
      l[4 * k + 1] = (int)(q.x >> 16);
      l[4 * k + 2] = (int)(q.y & 0xffffu);
      l[4 * k + 3] = (int)(q.y >> 16);
    }
    if constexpr (MODE == AF_OP) {
#pragma unroll
      for (int c = 0; c < 4; c++)
#pragma unroll
        for (int k = 0; k < (c < 3 ? NEN : 8); k++) x[c][k] = buf[c * ld + l[k]];
    } else {
      const int *no = A.ix + (size_t)A.ord[slot] * NEN;
#pragma unroll
      for (int k = 0; k < NEN; k++) {
        const double2 *up = reinterpret_cast<const double2 *>(A.u + (size_t)no[k] * 4);
        const double2 q0 = up[0], q1 = up[1];
        x[0][k] = q0.x;
        x[1][k] = q0.y;
        x[2][k] = q1.x;
        x[3][k] = q1.y;
        if (MODE == AF_RHS4 && k < 8) dpv[k] = A.dp[no[k]];
      }
    }
    pm_element_lane<NEN, MODE>(A, slot, x, dpv);
  }
  pm_wave_lds_fence();
  for (int i = lane; i < 4 * ld; i += 64) buf[i] = 0.0;
  pm_wave_lds_fence();
  if (on) {
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
      for (int k = 0; k < (c < 3 ? NEN : 8); k++)
        __hip_atomic_fetch_add(&buf[c * ld + l[k]], x[c][k], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_WAVEFRONT);
  }
  pm_wave_lds_fence();
  double *y = A.ye + (size_t)A.pn[p] * 4;
  for (int i = lane; i < n4; i += 64) y[i] = buf[(i & 3) * ld + (i >> 2)];
  pm_wave_lds_fence();
}

// row of dof c in a free-dof word
__device__ __forceinline__ unsigned int pm_word_row(unsigned int w, int c) {
  return (w >> 4) + __popc(w & ((1u << c) - 1u));
}

// place of value i = 4 * node + component in a patch's buffer
template <int LPE>
__device__ __forceinline__ int pm_at(int i, int ld) {
  return LPE == 4 ? i : (i & 3) * ld + (i >> 2);
}

// Patch vectors of K_e x_e (AF_OP: x an equation vector, restrained dofs
// zero; AF_RHS2: the nodal state) or of isw 4 (AF_RHS4); LPE lanes an element.
// The right-hand sides of hexa20/8 40^3 take 20 us and 12 us to subtract; eight
// colours of one workgroup an element took 4.3 ms (isw 4).
template <int NEN, int MODE, int LPE>
__global__ __launch_bounds__(64 * pm_patch_waves(NEN, LPE)) void k_affine_elements(AffineArgs A) {
  if (MODE == AF_OP && A.S != nullptr && A.S->done) return;
  extern __shared__ double s_dyn[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 3;
  const int ld = A.max_nodes + 1;
  double *buf = s_dyn + (size_t)wave * pm_patch_lds(A.max_nodes);
  const int p = pm_xcd_block(blockIdx.x, gridDim.x) * pm_patch_waves(NEN, LPE) + wave;
  if (p >= A.npatch) return;
  const unsigned int n0 = A.pn[p];
  const int n4 = (int)(A.pn[p + 1] - n0) * 4;
  if (MODE == AF_OP) {
    for (int i = lane; i < n4 + 4; i += 64) {
      const unsigned int w = i < n4 ? A.pw[n0 + (i >> 2)] : 0u;
      buf[pm_at<LPE>(i, ld)] = ((w >> c) & 1u) ? A.x[pm_word_row(w, c)] : 0.0;
    }
    pm_wave_lds_fence();
  }
  if constexpr (LPE == 4) pm_patch<NEN, MODE>(A, p, lane, n4, buf);
  else pm_patch_lane<NEN, MODE>(A, p, lane, n4, ld, buf);
}

// Pass A of the fused iteration (pm_fused.h), element part: the patch vectors
// of q_new = t + beta q, a patch per wavefront.  The patch's nodes are loaded
// while the scalars are formed.
template <int NEN, PmMethod MT, int LPE, bool BATCH>
__global__ __launch_bounds__(64 * pm_patch_waves(NEN, LPE)) void k_affine_pass_elements(
    AffineArgs A, PmVecs V, PmIterState *st, int cur, int first, double tol, int nblk,
    const double *pb, PmMap M) {
  extern __shared__ double s_dyn[];
  // nodes in registers, 16 a step: 160 or 48 (four lanes an element), 432 or 128
  constexpr int NB = LPE == 4 ? (NEN == 20 ? 10 : 3) : (NEN == 20 ? 27 : 8);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = lane & 3;
  const int ld = A.max_nodes + 1;
  double *buf = s_dyn + (size_t)wave * pm_patch_lds(A.max_nodes);
  const PmPart P = pm_part<BATCH, PM_PASS_ELEMS>(M, A.npatch, st, pb, nblk, nullptr);
  const int p = (int)P.lo + P.wg * pm_patch_waves(NEN, LPE) + wave;
  const bool on = p < P.hi;
  const unsigned int n0 = on ? A.pn[p] : 0u;
  const int n4 = on ? (int)(A.pn[p + 1] - n0) * 4 : 0;
  double tv[NB], qv[NB];
  unsigned int wv[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    // no branches around the loads: past the nodes lane 0's word, restrained
    // dofs row 0, dropped below
    const int i = b * 64 + lane;
    wv[b] = A.pw[i < n4 ? n0 + (unsigned int)(i >> 2) : 0u];
  }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const unsigned int row = (wv[b] >> c) & 1u ? pm_word_row(wv[b], c) : 0u;
    tv[b] = V.t[row];
    qv[b] = V.q[row];
  }
  double beta;
  {
    const PmIter s =
        pm_iter_begin<MT, pm_patch_waves(NEN, LPE), BATCH>(P.st, cur, first, tol, P.nin, P.in);
    if (P.wg == 0 && threadIdx.x == 0) P.st->it[cur ^ 1] = s;
    if (s.done || s.pending || !on) return;
    beta = s.beta;
  }
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int i = b * 64 + lane;
    if (i < n4 + 4)
      buf[pm_at<LPE>(i, ld)] = i < n4 && ((wv[b] >> c) & 1u) ? tv[b] + beta * qv[b] : 0.0;
  }
  for (int i = NB * 64 + lane; i < n4 + 4; i += 64) {  // a wider patch
    const unsigned int w = i < n4 ? A.pw[n0 + (i >> 2)] : 0u;
    const unsigned int row = pm_word_row(w, c);
    buf[pm_at<LPE>(i, ld)] = ((w >> c) & 1u) ? V.t[row] + beta * V.q[row] : 0.0;
  }
  pm_wave_lds_fence();
  if constexpr (LPE == 4) pm_patch<NEN, AF_OP>(A, p, lane, n4, buf);
  else pm_patch_lane<NEN, AF_OP>(A, p, lane, n4, ld, buf);
}

// element coefficients: geometry and material, dt folded in.  One lane an
// element, bound by its scattered vertex loads: 10 us at 64,000 elements, 300
// at 2.1 M, once a pass over the elements.
__global__ __launch_bounds__(PM_WG) void k_affine_coefs(int numel, int nen, const int *ord,
                                                        const int *ix, const double *xv,
                                                        const int *mat, const double *e,
                                                        double dt, double gmod, int stab,
                                                        double *ec, int *err) {
  const int slot = blockIdx.x * PM_WG + threadIdx.x;
  if (slot >= numel) return;
  const int el = ord[slot];
  const int *nodes = ix + (size_t)el * nen;
  double J[3][3] = {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}};
  for (int k = 0; k < 8; k++)
    for (int j = 0; j < 3; j++) {
      const double x = 0.125 * xv[(size_t)nodes[k] * 3 + j];
      J[0][j] += c_rn[k] * x;
      J[1][j] += c_sn[k] * x;
      J[2][j] += c_tn[k] * x;
    }
  const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) -
                     J[0][1] * (J[1][0] * J[2][2] - J[1][2] * J[2][0]) +
                     J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
  if (det <= 1.0e-14) atomicExch(err, PM_ERR_JACOBIAN);
  double *o = ec + (size_t)slot * PM_EC;
  // o[3 i + x] = d r_i / d x
  o[0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]) / det;
  o[1] = -(J[1][0] * J[2][2] - J[1][2] * J[2][0]) / det;
  o[2] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) / det;
  o[3] = -(J[0][1] * J[2][2] - J[0][2] * J[2][1]) / det;
  o[4] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) / det;
  o[5] = -(J[0][0] * J[2][1] - J[0][1] * J[2][0]) / det;
  o[6] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) / det;
  o[7] = -(J[0][0] * J[1][2] - J[0][2] * J[1][0]) / det;
  o[8] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) / det;
  const double *em = e + (size_t)mat[el] * PM_PROP;
  const ElemMat M = elem_material(em, dt, gmod);
  double dtk = M.dt_perm;
  if (stab && em[8] != 0.0) {  // the Q1/Q1 element's pressure stabilization (k_q1_isw2)
    const double h = cbrt(8.0 * det);
    dtk += em[8] * h * h / M.a;
  }
  o[9] = det * M.a * (1.0 - M.b);
  o[10] = det * M.a * M.b;
  o[11] = det * M.a * M.c;
  o[12] = det * M.coef_biot;
  o[13] = det * M.imod_biot;
  o[14] = det * dtk;
  o[15] = det;
}

// ---------------------------------------------------------------------------
// sums of the patch vectors per node
// ---------------------------------------------------------------------------
// Four lanes take a row block (a node) and sum its patches' entries, eight at
// a time in a fixed tree; lane c holds dof c.  Every node has `stride` offsets
// (8 in a box, two or three of them used on average; the others point to a
// zero), so their loads need no pointer first.  Bound by memory: with SQMR's
// updates 0.79 GB in 172 us at hexa20/8 87^3 (4.6 TB/s), 157 us at Q1/Q1 128^3
// (194 and 174 with the patches' nodes in the elements' order);
// 5-6 us, a chain of three loads, where the vectors stay in cache.
struct GatherArgs {
  int nrn, stride;
  const unsigned int *gnode;  // (nrn) first row << 4 | free dofs
  const unsigned int *gsrc;   // (nrn, stride) offsets in ye; past the last, of a zero
  const double *ye;
  unsigned int zero;
};

__device__ __forceinline__ double pm_gather_sum(const GatherArgs &G, int64_t k, int c) {
  const uint4 *src = reinterpret_cast<const uint4 *>(G.gsrc + (size_t)k * G.stride);
  double s = 0.0;
  for (int p = 0; p < G.stride; p += 8) {
    const uint4 a = src[p / 4];
    const uint4 b = p + 4 < G.stride ? src[p / 4 + 1] : uint4{G.zero, G.zero, G.zero, G.zero};
    double t[8];
    t[0] = G.ye[a.x + (unsigned int)c];
    t[1] = G.ye[a.y + (unsigned int)c];
    t[2] = G.ye[a.z + (unsigned int)c];
    t[3] = G.ye[a.w + (unsigned int)c];
    if (b.x != G.zero) {  // only the nodes of five patches and more
      t[4] = G.ye[b.x + (unsigned int)c];
      t[5] = G.ye[b.y + (unsigned int)c];
      t[6] = G.ye[b.z + (unsigned int)c];
      t[7] = G.ye[b.w + (unsigned int)c];
    } else {
      t[4] = t[5] = t[6] = t[7] = 0.0;
    }
    s += ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
  }
  return s;
}

template <int NV, bool SCALE_M>
__global__ __launch_bounds__(PM_WG) void k_affine_gather(GatherArgs G, double *__restrict__ y,
                                                         const double *__restrict__ w,
                                                         const double *__restrict__ m,
                                                         double *partials, const PmScalars *S) {
  if (S != nullptr && S->done) return;
  const int lb = pm_xcd_block(blockIdx.x, gridDim.x);
  int64_t k0, k1;
  pm_chunk(G.nrn, lb, gridDim.x, k0, k1);
  const int c = threadIdx.x & 3;
  double v[2] = {0.0, 0.0};
  for (int64_t k = k0 + (threadIdx.x >> 2); k < k1; k += PM_WG / 4) {
    const unsigned int w4 = G.gnode[k];
    if (!((w4 >> c) & 1u)) continue;
    const unsigned int row = (w4 >> 4) + __popc(w4 & ((1u << c) - 1u));
    double s = pm_gather_sum(G, k, c);
    if (SCALE_M) s *= m[row];
    y[row] = s;
    if (NV >= 1) v[0] += s * w[row];
    if (NV >= 2) v[1] += s * s;
  }
  pm_block_partials<NV>(v, partials);
}

// Pass A, node part: y = A q_new with the row's update and the dot q_new . y
template <PmMethod MT, bool BATCH>
__global__ __launch_bounds__(PM_WG) void k_affine_pass_gather(GatherArgs G, PmVecs V,
                                                              PmIterState *st, int nxt, double *pa,
                                                              PmMap M) {
  const PmPart P = pm_part<BATCH, PM_PASS_NODES>(M, G.nrn, st, nullptr, 0, pa);
  int64_t k0, k1;
  pm_share(P, k0, k1);
  const int c = threadIdx.x & 3;
  double v[1] = {0.0};
  int64_t k = k0 + (threadIdx.x >> 2);
  // the first node's sum does not wait for the scalars
  unsigned int w4 = 0;
  double y = 0.0;
  if (k < k1) {
    w4 = G.gnode[k];
    y = pm_gather_sum(G, k, c);
  }
  const PmIter s = P.st->it[nxt];  // written by the element part
  if (s.done) return;
  while (k < k1) {
    if ((w4 >> c) & 1u) {
      const unsigned int row = (w4 >> 4) + __popc(w4 & ((1u << c) - 1u));
      const double qn = pm_row_update<MT>(V, s, row);
      if (!s.pending) {
        V.y[row] = y;
        v[0] += y * qn;
      }
    }
    k += PM_WG / 4;
    if (k < k1) {
      w4 = G.gnode[k];
      y = pm_gather_sum(G, k, c);
    }
  }
  pm_dots_partials<1>(v, P.out, P.slot);
}

__global__ __launch_bounds__(PM_WG) void k_affine_subtract(GatherArgs G, double *b) {
  const int64_t k = (int64_t)pm_xcd_block(blockIdx.x, gridDim.x) * (PM_WG / 4) + (threadIdx.x >> 2);
  const int c = threadIdx.x & 3;
  if (k >= G.nrn) return;
  const unsigned int w4 = G.gnode[k];
  if (!((w4 >> c) & 1u)) return;
  const unsigned int row = (w4 >> 4) + __popc(w4 & ((1u << c) - 1u));
  b[row] -= pm_gather_sum(G, k, c);
}

// b -= the face loads of each loaded node's elements, in list order
__global__ __launch_bounds__(256) void k_face_subtract(int n4, const int *node, const int *ptr,
                                                       const int *src, const double *fv,
                                                       const int *eq, double *b) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const int j = i >> 2, c = i & 3;
  const int row = eq[(size_t)node[j] * 4 + c];
  if (row < 0) return;
  double s = 0.0;
  for (int q = ptr[j]; q < ptr[j + 1]; q++) s += fv[(size_t)src[q] * 4 + c];
  b[row] -= s;
}

// ---------------------------------------------------------------------------
// the matrix, one row block per group of lanes
// ---------------------------------------------------------------------------
// Integrals over the reference element, m, n nodes and q, s pressure vertices:
//   R[m][ij][n] = int d_i N_m d_j N_n    M[m][j][q] = int d_j N_m Np_q
//   T[q][j][n] = M[n][j][q]              Z[q][s] = int Np_q Np_s
//   L[q][ij][s] = int d_i Np_q d_j Np_s
template <int NEN>
struct RefTab {
  static constexpr int R = 0, M = R + NEN * 9 * NEN, T = M + NEN * 3 * 8, Z = T + 8 * 3 * NEN,
                       L = Z + 64, SIZE = L + 8 * 9 * 8;
};

// g g^T of every element, the symmetric products of its coefficients
__global__ __launch_bounds__(PM_WG) void k_affine_metric(int numel, const double *ec, double *gg) {
  const int slot = blockIdx.x * PM_WG + threadIdx.x;
  if (slot >= numel) return;
  const double *g = ec + (size_t)slot * PM_EC;
  double *o = gg + (size_t)slot * PM_EC;
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++)
      o[3 * i + j] = g[3 * i] * g[3 * j] + g[3 * i + 1] * g[3 * j + 1] + g[3 * i + 2] * g[3 * j + 2];
}

// Each matrix value is written once: the lanes of a group walk the row node's
// incident elements, lane (b, x) forming the column of node b's component x
// (then lanes 0..7 the pressure columns), and add into the block's rows in
// LDS.  A pair's 3 x 3 block is J^-T R J^-1 contracted with D: ~45
// multiply-adds a lane instead of 64 Gauss points'.  Bound by instruction
// issue, so the places of all the elements' nodes in the block's column list
// are found first, a node a lane (bisection in LDS): three searches a row
// block instead of sixteen (hexa20/8 vertices); with 64 lanes a block its
// elements' data are scalar loads.  hexa20/8 40^3: 1.87 ms (2.53 with the
// places searched one by one) against 8.3 in eight colours of one workgroup an
// element; 87^3 19.0 against 67; Q1/Q1 64^3 1.60 against 3.6, 128^3 12.4
// against 20.  The sums keep a multiply and an add apart, in the row's order.
template <int NEN>
__global__ __launch_bounds__(PM_WG) void k_affine_matrix(
    int nrn, int max_cols, int mstride, const unsigned int *__restrict__ minc,
    const unsigned int *__restrict__ gnode, const unsigned int *__restrict__ en,
    const double *__restrict__ ec, const double *__restrict__ gg_all,
    const double *__restrict__ tab, const int *__restrict__ nr,
    const int64_t *__restrict__ colptr, const int64_t *__restrict__ valptr,
    const int *__restrict__ ncol, double *__restrict__ val, int *err) {
  constexpr int LPB = NEN == 20 ? 64 : 32;  // 60 (24) displacement columns an element
  constexpr int GR = PM_WG / LPB;
  using RT = RefTab<NEN>;
  extern __shared__ double s_dyn[];
  int grp = threadIdx.x / LPB;
  const int l = threadIdx.x % LPB;
  if (LPB == 64) grp = __builtin_amdgcn_readfirstlane(grp);
  double *row = s_dyn + (size_t)grp * max_cols * 4;
  int *cols = reinterpret_cast<int *>(s_dyn + (size_t)GR * max_cols * 4) + (size_t)grp * max_cols;
  // place << 4 | free dofs of every node of the incident elements
  int *place = reinterpret_cast<int *>(s_dyn + (size_t)GR * max_cols * 4) + (size_t)GR * max_cols +
               (size_t)grp * mstride * NEN;
  const int64_t k = (int64_t)pm_xcd_block(blockIdx.x, gridDim.x) * GR + grp;
  const bool live = k < nrn;
  const int n = live ? nr[k] : 0;
  const int64_t cp = live ? colptr[k] : 0;
  const int cnt = live ? (int)(colptr[k + 1] - cp) : 0;
  for (int j = l; j < cnt; j += LPB) cols[j] = ncol[cp + j];
  for (int j = l; j < n * cnt; j += LPB) row[j] = 0.0;
  __syncthreads();
  if (!live) return;  // no workgroup barrier follows
  const unsigned int *inc = minc + (size_t)k * mstride;
  for (int i = l; i < mstride * NEN; i += LPB) {
    const int p = i / NEN, b = i - p * NEN;
    const unsigned int code = inc[p];
    if (code == 0xffffffffu) break;
    const unsigned int w = en[(size_t)(code >> 5) * NEN + b];
    int lo = 0, hi = cnt;
    const int col = (int)(w >> 4);
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (cols[mid] < col) lo = mid + 1;
      else hi = mid;
    }
    unsigned int m = w & 15u;
    if (m && (lo >= cnt || cols[lo] != col)) {  // pattern does not hold the pair
      atomicExch(err, PM_ERR_STATE);
      m = 0;
    }
    place[i] = (lo << 4) | (int)m;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const unsigned int mk = gnode[k] & 15u;
  const int q1 = (int)(mk & 1u), q2 = (int)__popc(mk & 3u), q3 = (int)__popc(mk & 7u);
  double *r0 = row, *r1 = row + q1 * cnt, *r2 = row + q2 * cnt, *r3 = row + q3 * cnt;
  const int b = l / 3, x = l - 3 * b;
  for (int p = 0; p < mstride; p++) {
    unsigned int code = inc[p];
    if (LPB == 64) code = __builtin_amdgcn_readfirstlane(code);
    if (code == 0xffffffffu) break;
    const unsigned int slot = code >> 5;
    const int a = (int)(code & 31u);  // the row's local node
    const double *eq = ec + (size_t)slot * PM_EC, *gg = gg_all + (size_t)slot * PM_EC;
    double g[9];
#pragma unroll
    for (int i = 0; i < 9; i++) g[i] = eq[i];
    const double cb = eq[10], cd = eq[9] + cb, cc = eq[11], al = eq[12];
    if (l < 3 * NEN) {
      const int w = place[p * NEN + b];
      if ((w >> x) & 1) {
        const int pos = (w >> 4) + __popc(w & ((1 << x) - 1));
        const double gx[3] = {x == 0 ? g[0] : x == 1 ? g[1] : g[2],
                              x == 0 ? g[3] : x == 1 ? g[4] : g[5],
                              x == 0 ? g[6] : x == 1 ? g[7] : g[8]};
        const double *tr = tab + RT::R + a * 9 * NEN + b;
        double H[3] = {0, 0, 0}, Ht[3] = {0, 0, 0}, lap = 0.0;
#pragma unroll
        for (int i = 0; i < 3; i++)
#pragma unroll
          for (int j = 0; j < 3; j++) {
            const double r = tr[(3 * i + j) * NEN];
            H[i] = fma(r, gx[j], H[i]);    // int d_i N_a dN_b/dx
            Ht[j] = fma(r, gx[i], Ht[j]);  // int dN_a/dx d_j N_b
            lap = fma(r, gg[3 * i + j], lap);
          }
        // row y, column x: D's normal and shear parts
        double v[3];
#pragma unroll
        for (int y = 0; y < 3; y++) {
          const double Gyx = g[y] * H[0] + g[3 + y] * H[1] + g[6 + y] * H[2];
          const double Gxy = g[y] * Ht[0] + g[3 + y] * Ht[1] + g[6 + y] * Ht[2];
          v[y] = y == x ? cd * Gyx + cc * (lap - Gyx) : cb * Gyx + cc * Gxy;
        }
        if (mk & 1u) r0[pos] += v[0];
        if (mk & 2u) r1[pos] += v[1];
        if (mk & 4u) r2[pos] += v[2];
        if (a < 8 && (mk & 8u)) {  // pressure row
          const double *tt = tab + RT::T + a * 3 * NEN + b;
          r3[pos] -= al * fma(gx[2], tt[2 * NEN], fma(gx[1], tt[NEN], gx[0] * tt[0]));
        }
      }
    }
    if (l < 8) {  // pressure columns
      const int w = place[p * NEN + l];
      if (w & 8) {
        const int pos = (w >> 4) + __popc(w & 7);
        const double *tm = tab + RT::M + a * 3 * 8 + l;
        const double m0 = tm[0], m1 = tm[8], m2 = tm[16];
        if (mk & 1u) r0[pos] -= al * fma(g[6], m2, fma(g[3], m1, g[0] * m0));
        if (mk & 2u) r1[pos] -= al * fma(g[7], m2, fma(g[4], m1, g[1] * m0));
        if (mk & 4u) r2[pos] -= al * fma(g[8], m2, fma(g[5], m1, g[2] * m0));
        if (a < 8 && (mk & 8u)) {
          const double *tl = tab + RT::L + a * 9 * 8 + l;
          double lap = 0.0;
#pragma unroll
          for (int i = 0; i < 9; i++) lap = fma(tl[i * 8], gg[i], lap);
          r3[pos] -= eq[13] * tab[RT::Z + a * 8 + l] + eq[14] * lap;
        }
      }
    }
    // the next element's lanes add into what these lanes wrote
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  double *out = val + valptr[k];
  for (int j = l; j < n * cnt; j += LPB) out[j] = row[j];
}

// the reference integrals from the shape functions' Legendre coefficients
template <int NEN>
static std::vector<double> reference_integrals() {
  using RT = RefTab<NEN>;
  std::vector<double> t((size_t)RT::SIZE, 0.0);
  const double nrm[3] = {2.0, 2.0 / 3.0, 2.0 / 5.0};
  auto coefs = [](int nodes, int k, double *co) {
    double v[20] = {0};
    for (int i = 0; i < 27; i++) co[i] = 0.0;
    v[k] = 1.0;
    if (nodes == 20) pm_modal_fwd<20>(v, 2.0 / 3.0, co);
    else pm_modal_fwd<8>(v, 2.0 / 3.0, co);
  };
  auto derive = [](const double *co, int dir, double *d) {
    for (int i = 0; i < 27; i++) d[i] = 0.0;
    for (int m = 0; m < 27; m++) {
      int e[3] = {m / 9, (m / 3) % 3, m % 3};
      const double s = e[dir] == 2 ? 3.0 : 1.0;
      if (e[dir] == 0) continue;
      e[dir]--;
      d[e[0] * 9 + e[1] * 3 + e[2]] += s * co[m];
    }
  };
  auto dot = [&](const double *p, const double *q) {
    double s = 0.0;
    for (int m = 0; m < 27; m++) s += p[m] * q[m] * (nrm[m / 9] * nrm[(m / 3) % 3] * nrm[m % 3]);
    return s;
  };
  double N[20][27], dN[20][3][27], P[8][27], dP[8][3][27];
  for (int k = 0; k < NEN; k++) {
    coefs(NEN, k, N[k]);
    for (int i = 0; i < 3; i++) derive(N[k], i, dN[k][i]);
  }
  for (int k = 0; k < 8; k++) {
    coefs(8, k, P[k]);
    for (int i = 0; i < 3; i++) derive(P[k], i, dP[k][i]);
  }
  for (int m = 0; m < NEN; m++)
    for (int i = 0; i < 3; i++)
      for (int j = 0; j < 3; j++)
        for (int n = 0; n < NEN; n++) t[RT::R + (m * 9 + 3 * i + j) * NEN + n] = dot(dN[m][i], dN[n][j]);
  for (int q = 0; q < 8; q++) {
    for (int m = 0; m < NEN; m++)
      for (int j = 0; j < 3; j++) {
        const double v = dot(dN[m][j], P[q]);
        t[RT::M + (m * 3 + j) * 8 + q] = v;
        t[RT::T + (q * 3 + j) * NEN + m] = v;
      }
    for (int s = 0; s < 8; s++) {
      t[RT::Z + q * 8 + s] = dot(P[q], P[s]);
      for (int i = 0; i < 3; i++)
        for (int j = 0; j < 3; j++) t[RT::L + (q * 9 + 3 * i + j) * 8 + s] = dot(dP[q][i], dP[s][j]);
    }
  }
  return t;
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
void pm_affine_free(PmAffine *a) {
  if (!a) return;
  for (void *p : {(void *)a->ord, (void *)a->ps, (void *)a->pn, (void *)a->pw, (void *)a->loc,
                  (void *)a->en, (void *)a->gsrc, (void *)a->gnode, (void *)a->minc,
                  (void *)a->ec_op, (void *)a->ec, (void *)a->ye, (void *)a->tab})
    if (p) (void)hipFree(p);
  delete a;
}

static int affine_setup(pm_ctx *c, const double *x, const PmHostPattern &pat) {
  const std::vector<int> &eq_block = pat.eq_block;
  const PmHostMesh &m = c->mesh;
  const int nen = m.nen, numel = m.numel, nrn = c->A.nrn;
  if (m.neq >= (1 << 28) || (int64_t)numel * nen * 4 + 4 >= ((int64_t)1 << 32) || numel >= (1 << 27))
    return PM_OK;
  for (int e = 0; e < numel; e++)
    if (!pm_is_parallelepiped(m.ix20.data() + (size_t)e * 21, x)) return PM_OK;
  // each node's free dofs: first equation << 4 | mask, and its row block
  std::vector<unsigned int> word((size_t)m.nnode, 0);
  std::vector<int> block((size_t)m.nnode, -1);
  std::vector<unsigned int> gnode((size_t)nrn, 0);
  for (int n = 0; n < m.nnode; n++) {
    const int nd = m.fnno[n] == 1 ? 4 : 3;
    unsigned int mk = 0;
    int first = -1;
    for (int d = 0; d < nd; d++) {
      const int q = m.id[(size_t)n * 4 + d];
      if (q <= 0) continue;
      if (first < 0) first = q - 1;
      mk |= 1u << d;
    }
    if (first < 0) continue;
    word[n] = ((unsigned int)first << 4) | mk;
    block[n] = eq_block[first];
    gnode[block[n]] = word[n];
  }
  int max_cols = 0;
  for (int k = 0; k < nrn; k++)
    max_cols = std::max(max_cols, (int)(pat.colptr[k + 1] - pat.colptr[k]));
  std::vector<int> ord, ps;
  // one lane an element from 50,000 elements (800 wavefronts): below, four
  // times the wavefronts hide more latency.  SQMR iteration, four lanes / one:
  // Q1/Q1 32^3 17.5 / 18.3 us, 36^3 20.5 / 19.7, 40^3 22.8 / 21.6, 48^3 32.9 /
  // 28.7, 64^3 62.6 / 48.9; hexa20/8 24^3 20.0 / 25.1, 32^3 28.8 / 31.1, 36^3
  // 38.3 / 37.2, 40^3 47.8 / 43.3, 48^3 74.1 / 69.8.  Between the crossing,
  // near 40,000, and the line the two are within 4 %.
  const int lpe = numel >= 50000 ? 1 : 4;
  pm_element_patches(numel, nen, m.nnodev, m.ix20.data(), m.id.data(), x, 64 / lpe, ord, ps);
  const int npatch = (int)ps.size() - 1;
  // patch nodes; restrained nodes share the dummy after the last
  std::vector<unsigned int> en((size_t)numel * nen), pn((size_t)npatch + 1, 0), pw;
  std::vector<int> pblock;  // row block of each entry of pw
  std::vector<unsigned short> loc((size_t)numel * nen);
  std::vector<int> at((size_t)m.nnode, -1), seen((size_t)m.nnode, -1);
  std::vector<int> pcnt((size_t)nrn, 0), mcnt((size_t)nrn, 0);
  std::vector<int> patch_first((size_t)npatch, -1), patch_last((size_t)npatch, -1);
  std::vector<int> nodes;  // of a patch
  int max_nodes = 0, step = 0;
  pw.reserve((size_t)numel * nen / 2);
  pblock.reserve((size_t)numel * nen / 2);
  for (int p = 0; p < npatch; p++) {
    const int n0 = (int)pw.size();
    for (int s = ps[p]; s < ps[p + 1]; s++)
      for (int k = 0; k < nen; k++) {
        const int n = m.ix20[(size_t)ord[s] * 21 + k] - 1;
        en[(size_t)s * nen + k] = word[n];
        if (block[n] < 0) continue;
        mcnt[block[n]]++;
        if (at[n] < n0) {
          at[n] = n0;
          nodes.push_back(n);
        }
      }
    // in the order of their equations: neighbouring lanes read and write
    // neighbouring entries of the vectors
    std::sort(nodes.begin(), nodes.end(), [&](int i, int j) { return word[i] < word[j]; });
    for (int n : nodes) {
      at[n] = (int)pw.size();
      pw.push_back(word[n]);
      pblock.push_back(block[n]);
      pcnt[block[n]]++;
    }
    nodes.clear();
    const int nn = (int)pw.size() - n0;
    max_nodes = std::max(max_nodes, nn);
    for (int k = 0; k < nen; k++, step++)
      for (int s = ps[p]; s < ps[p + 1]; s++) {
        const int n = m.ix20[(size_t)ord[s] * 21 + k] - 1;
        loc[(size_t)s * nen + k] = (unsigned short)(block[n] < 0 ? nn : at[n] - n0);
        if (seen[n] == step) return PM_OK;  // two elements add to a node at once
        seen[n] = step;
      }
    pn[p + 1] = (unsigned int)pw.size();
    if (nn > 0) {
      patch_first[p] = pblock[n0];
      patch_last[p] = pblock.back();
    }
  }
  auto widest = [](const std::vector<int> &v) {
    return ((v.empty() ? 0 : *std::max_element(v.begin(), v.end())) + 3) & ~3;
  };
  const int stride = widest(pcnt), mstride = widest(mcnt);
  if (stride > 32 || mstride > 32) return PM_OK;  // a fan of elements: keep the stored matrix
  // a workgroup of patches may ask for 64 KB of LDS (bricks take 27 KB at most)
  if ((size_t)pm_patch_lds(max_nodes) * pm_patch_waves(nen, lpe) * sizeof(double) > 65536)
    return PM_OK;
  const unsigned int zero = pn[npatch] * 4u;
  std::vector<unsigned int> gsrc((size_t)nrn * stride, zero),
      minc((size_t)nrn * mstride, 0xffffffffu);
  std::fill(pcnt.begin(), pcnt.end(), 0);
  std::fill(mcnt.begin(), mcnt.end(), 0);
  for (size_t i = 0; i < pw.size(); i++)
    gsrc[(size_t)pblock[i] * stride + pcnt[pblock[i]]++] = (unsigned int)i * 4u;
  for (int s = 0; s < numel; s++)
    for (int k = 0; k < nen; k++) {
      const int b = block[m.ix20[(size_t)ord[s] * 21 + k] - 1];
      if (b >= 0) minc[(size_t)b * mstride + mcnt[b]++] = ((unsigned int)s << 5) | (unsigned int)k;
    }
  const std::vector<double> tab = nen == 20 ? reference_integrals<20>() : reference_integrals<8>();
  PmAffine *a = new PmAffine();
  a->max_cols = max_cols;
  a->stride = stride;
  a->zero = zero;
  a->numel = numel;
  a->npatch = npatch;
  a->lpe = lpe;
  a->patch_first = std::move(patch_first);
  a->patch_last = std::move(patch_last);
  a->max_nodes = max_nodes;
  a->mstride = mstride;
  a->nen = nen;
  a->nrn = nrn;
  bool ok = true;
  auto up = [&](void **d, const void *h, size_t bytes) {
    ok = ok && hipMalloc(d, bytes) == hipSuccess &&
         (!h || hipMemcpy(*d, h, bytes, hipMemcpyHostToDevice) == hipSuccess);
  };
  up((void **)&a->ord, ord.data(), sizeof(int) * ord.size());
  up((void **)&a->ps, ps.data(), sizeof(int) * ps.size());
  up((void **)&a->pn, pn.data(), sizeof(unsigned int) * pn.size());
  up((void **)&a->pw, pw.data(), sizeof(unsigned int) * std::max<size_t>(pw.size(), 1));
  up((void **)&a->loc, loc.data(), sizeof(unsigned short) * loc.size());
  up((void **)&a->minc, minc.data(), sizeof(unsigned int) * std::max<size_t>(minc.size(), 1));
  up((void **)&a->en, en.data(), sizeof(unsigned int) * en.size());
  up((void **)&a->gsrc, gsrc.data(), sizeof(unsigned int) * gsrc.size());
  up((void **)&a->gnode, gnode.data(), sizeof(unsigned int) * gnode.size());
  up((void **)&a->ec_op, nullptr, sizeof(double) * PM_EC * (size_t)numel);
  up((void **)&a->ec, nullptr, sizeof(double) * PM_EC * (size_t)numel);
  up((void **)&a->tab, tab.data(), sizeof(double) * tab.size());
  // the patch vectors, then four zeros for the gathers' missing entries
  up((void **)&a->ye, nullptr, sizeof(double) * ((size_t)zero + 4));
  // on the stream of its readers, which the null stream does not wait for
  ok = ok && hipMemsetAsync(a->ye + zero, 0, 4 * sizeof(double), c->stream) == hipSuccess;
  if (!ok) {  // the stored-matrix path needs none of this
    (void)hipGetLastError();
    pm_affine_free(a);
    return PM_OK;
  }
  c->affine = a;
  return PM_OK;
}

int pm_affine_setup(pm_ctx *c, const double *x, const PmHostPattern &pat) {
  try {
    return affine_setup(c, x, pat);
  } catch (const std::bad_alloc &) {  // the stored-matrix path needs none of this
    return PM_OK;
  }
}

// c->affine's element loops stand for elmt17_pm and the Q1/Q1 element with
// constant properties, summed in any order
static bool affine_elements(const pm_ctx *c) {
  return c->affine && !c->ordered && !c->vprop[0];
}

// From 3.6 million stored values on with FP64 values, 4.5 with FP32: below,
// the stored product is the shorter chain (one pass against two).  An SQMR
// iteration on boxes, stored / elements, FP64 and FP32: hexa20/8 11^3 (3.2 M
// values) 13.9 / 16.4 us and 13.5 / 16.1, 12^3 (4.2 M) 17.6 / 16.1 and 15.2 /
// 16.1, 14^3 (6.7 M) 22.7 / 16.1 and 20.2 / 16.3; Q1/Q1 18^3 (2.4 M) 12.1 /
// 14.6 and 12.3 / 15.2, 20^3 (3.3 M) 14.7 / 15.4 and 13.7 / 14.8, 22^3 (4.4 M)
// 17.7 / 14.8 and 14.9 / 14.7, 24^3 (5.8 M) 20.7 / 15.0 and 17.8 / 15.3.
bool pm_affine_product(const pm_ctx *c, int use32) {
  return affine_elements(c) && c->affine->op_valid && c->A.values_valid &&
         c->A.nnz >= (use32 ? 4500000 : 3600000);
}

static GatherArgs gather_args(const pm_ctx *c) {
  const PmAffine *a = c->affine;
  return GatherArgs{a->nrn, a->stride, a->gnode, a->gsrc, a->ye, a->zero};
}

static size_t patch_lds(const PmAffine *a) {
  return (size_t)pm_patch_lds(a->max_nodes) * pm_patch_waves(a->nen, a->lpe) * sizeof(double);
}

template <int MODE>
static void launch_elements(pm_ctx *c, AffineArgs A) {
  const int pw = pm_patch_waves(c->affine->nen, c->affine->lpe);
  const dim3 g(((A.npatch + pw - 1) / pw + 7) & ~7), bl(64 * pw);
  const size_t lds = patch_lds(c->affine);
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, bl, lds, c->stream, A); };
  if (c->affine->nen == 20) {
    if (c->affine->lpe == 4) go(k_affine_elements<20, MODE, 4>);
    else go(k_affine_elements<20, MODE, 1>);
  } else {
    if (c->affine->lpe == 4) go(k_affine_elements<8, MODE, 4>);
    else go(k_affine_elements<8, MODE, 1>);
  }
}

static AffineArgs affine_args(const pm_ctx *c) {
  AffineArgs A{};
  const PmAffine *a = c->affine;
  A.npatch = a->npatch;
  A.max_nodes = a->max_nodes;
  A.ps = a->ps;
  A.pn = a->pn;
  A.pw = a->pw;
  A.loc = a->loc;
  A.ord = a->ord;
  A.ye = a->ye;
  return A;
}

void pm_affine_elements(pm_ctx *c, const double *x, const PmScalars *S) {
  AffineArgs A = affine_args(c);
  A.ec = c->affine->ec_op;
  A.x = x;
  A.S = S;
  launch_elements<AF_OP>(c, A);
}

int pm_affine_gather(pm_ctx *c, double *y, const double *w, const double *m, int nv, bool scale_m,
                     const PmScalars *S) {
  const GatherArgs G = gather_args(c);
  int g = (G.nrn + PM_WG / 4 - 1) / (PM_WG / 4);
  g = (std::min(g, PM_MAX_GRID) + 7) & ~7;
  const dim3 gr(g), bl(PM_WG);
  if (scale_m) {
    if (nv == 1)
      hipLaunchKernelGGL((k_affine_gather<1, true>), gr, bl, 0, c->stream, G, y, w, m,
                         c->d_partials, S);
    else
      hipLaunchKernelGGL((k_affine_gather<0, true>), gr, bl, 0, c->stream, G, y, w, m,
                         c->d_partials, S);
  } else if (nv == 2) {
    hipLaunchKernelGGL((k_affine_gather<2, false>), gr, bl, 0, c->stream, G, y, w, m,
                       c->d_partials, S);
  } else if (nv == 1) {
    hipLaunchKernelGGL((k_affine_gather<1, false>), gr, bl, 0, c->stream, G, y, w, m,
                       c->d_partials, S);
  } else {
    hipLaunchKernelGGL((k_affine_gather<0, false>), gr, bl, 0, c->stream, G, y, w, m,
                       c->d_partials, S);
  }
  return g;
}

// the element part's kernel for the mesh, called with it
template <PmMethod MT, bool BATCH, class Go>
static void pass_elements(const PmAffine *a, Go go) {
  if (a->nen == 20) {
    if (a->lpe == 4) go(k_affine_pass_elements<20, MT, 4, BATCH>);
    else go(k_affine_pass_elements<20, MT, 1, BATCH>);
  } else {
    if (a->lpe == 4) go(k_affine_pass_elements<8, MT, 4, BATCH>);
    else go(k_affine_pass_elements<8, MT, 1, BATCH>);
  }
}

template <PmMethod MT>
static int affine_pass(pm_ctx *c, const PmVecs &V, PmIterState *st, int cur, int first, double tol,
                       int nblk, const double *pb, double *pa) {
  AffineArgs A = affine_args(c);
  A.ec = c->affine->ec_op;
  const int pw = pm_affine_patch_waves(c);
  const dim3 ge(((A.npatch + pw - 1) / pw + 7) & ~7), bl(64 * pw);
  const size_t lds = patch_lds(c->affine);
  pass_elements<MT, false>(c->affine, [&](auto kernel) {
    hipLaunchKernelGGL(kernel, ge, bl, lds, c->stream, A, V, st, cur, first, tol, nblk, pb, PmMap{});
  });
  const GatherArgs G = gather_args(c);
  const int g = (std::min((G.nrn + PM_WG / 4 - 1) / (PM_WG / 4), PM_MAX_GRID) + 7) & ~7;
  hipLaunchKernelGGL((k_affine_pass_gather<MT, false>), dim3(g), dim3(PM_WG), 0, c->stream, G, V,
                     st, cur ^ 1, pa, PmMap{});
  return g;
}

int pm_affine_pass(pm_ctx *c, PmMethod mt, const PmVecs &V, PmIterState *st, int cur, int first,
                   double tol, int nblk, const double *pb, double *pa) {
  return mt == PM_IT_SQMR ? affine_pass<PM_IT_SQMR>(c, V, st, cur, first, tol, nblk, pb, pa)
                          : affine_pass<PM_IT_PCG>(c, V, st, cur, first, tol, nblk, pb, pa);
}

template <PmMethod MT>
static void affine_pass_boxes(pm_ctx *c, const PmVecs &V, PmIterState *st, int cur, int first,
                              double tol, const double *pb, double *pa, const PmMap &elems,
                              int n_elems, const PmMap &nodes, int n_nodes) {
  AffineArgs A = affine_args(c);
  A.ec = c->affine->ec_op;
  const size_t lds = patch_lds(c->affine);
  pass_elements<MT, true>(c->affine, [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(n_elems), dim3(64 * pm_affine_patch_waves(c)), lds, c->stream,
                       A, V, st, cur, first, tol, 0, pb, elems);
  });
  hipLaunchKernelGGL((k_affine_pass_gather<MT, true>), dim3(n_nodes), dim3(PM_WG), 0, c->stream,
                     gather_args(c), V, st, cur ^ 1, pa, nodes);
}

void pm_affine_pass_boxes(pm_ctx *c, PmMethod mt, const PmVecs &V, PmIterState *st, int cur,
                          int first, double tol, const double *pb, double *pa, const PmMap &elems,
                          int n_elems, const PmMap &nodes, int n_nodes) {
  if (mt == PM_IT_SQMR)
    affine_pass_boxes<PM_IT_SQMR>(c, V, st, cur, first, tol, pb, pa, elems, n_elems, nodes, n_nodes);
  else
    affine_pass_boxes<PM_IT_PCG>(c, V, st, cur, first, tol, pb, pa, elems, n_elems, nodes, n_nodes);
}

int pm_affine_patch_waves(const pm_ctx *c) { return pm_patch_waves(c->affine->nen, c->affine->lpe); }

bool pm_affine_box_patches(const pm_ctx *c, const std::vector<int> &blk0, std::vector<int> &p0) {
  const std::vector<int> &first = c->affine->patch_first, &last = c->affine->patch_last;
  const int nbox = (int)blk0.size() - 1;
  p0.assign(nbox + 1, 0);
  int box = 0;
  for (size_t p = 0; p < first.size(); p++) {
    if (first[p] < 0) continue;  // no free node: with the patch before
    if (first[p] < blk0[box]) return false;  // patches out of the boxes' order
    while (first[p] >= blk0[box + 1]) p0[++box] = (int)p;
    // elements of two boxes that share restrained nodes: every box has scalars
    // of its own, a patch can have one box's only
    if (last[p] >= blk0[box + 1]) return false;
  }
  while (box < nbox) p0[++box] = (int)first.size();
  return true;
}

// LDS of a workgroup of k_affine_matrix: every group's rows, columns and places
static size_t matrix_lds(const PmAffine *a) {
  return (size_t)(PM_WG / (a->nen == 20 ? 64 : 32)) *
         (a->max_cols * (4 * sizeof(double) + sizeof(int)) + a->mstride * a->nen * sizeof(int));
}

bool pm_affine_loops(const pm_ctx *c, int isw, int lhs) {
  // row blocks too wide for the 64 KB of LDS a workgroup may ask for keep the
  // scattered assembly (437 columns; a box's vertex has 270, 108 with Q1/Q1)
  return affine_elements(c) && (isw != 2 || !lhs || matrix_lds(c->affine) <= 65536);
}

int pm_affine_pform(pm_ctx *c, const ElemArgs &E, int isw, int lhs, int rhs) {
  PmAffine *a = c->affine;
  const PmDevMatrix &M = c->A;
  double *ec = isw == 2 && lhs ? a->ec_op : a->ec;
  if (isw == 2 && lhs) a->op_valid = false;
  hipLaunchKernelGGL(k_affine_coefs, dim3((a->numel + PM_WG - 1) / PM_WG), dim3(PM_WG), 0,
                     c->stream, a->numel, a->nen, a->ord, E.ix, E.xv, E.mat, E.e, E.dt, E.gmod,
                     a->nen == 8 && isw == 2, ec, E.err);
  if (rhs) {
    AffineArgs A = affine_args(c);
    A.ec = ec;
    A.ix = E.ix;
    A.u = E.u;
    A.dp = E.dp;
    A.mat = E.mat;
    A.e = E.e;
    for (int d = 0; d < 3; d++) A.grav[d] = E.grav[d];
    if (isw == 2) launch_elements<AF_RHS2>(c, A);
    else launch_elements<AF_RHS4>(c, A);
    const GatherArgs G = gather_args(c);
    const int g = ((G.nrn + PM_WG / 4 - 1) / (PM_WG / 4) + 7) & ~7;
    hipLaunchKernelGGL(k_affine_subtract, dim3(g), dim3(PM_WG), 0, c->stream, G, E.b);
    if (isw == 4 && c->n_face_elems > 0) {
      if (a->nen == 20) PM_TRY(pm_hexa20_faces(E, c->n_face_elems, c->d_face_elems, c->d_face_vec, c->stream));
      else PM_TRY(pm_q1_faces(E, c->n_face_elems, c->d_face_elems, c->d_face_vec, c->stream));
      const int n4 = c->n_face_nodes * 4;
      hipLaunchKernelGGL(k_face_subtract, dim3((n4 + 255) / 256), dim3(256), 0, c->stream, n4,
                         c->d_face_node, c->d_face_ptr, c->d_face_src, c->d_face_vec, E.eq, E.b);
    }
  }
  if (isw == 2 && lhs) {
    const int gr = PM_WG / (a->nen == 20 ? 64 : 32);
    const dim3 g((unsigned)(((a->nrn + gr - 1) / gr + 7) & ~7));
    const size_t lds = matrix_lds(a);
    hipLaunchKernelGGL(k_affine_metric, dim3((a->numel + PM_WG - 1) / PM_WG), dim3(PM_WG), 0,
                       c->stream, a->numel, ec, a->ec);
    if (a->nen == 20)
      hipLaunchKernelGGL(k_affine_matrix<20>, g, dim3(PM_WG), lds, c->stream, a->nrn, a->max_cols,
                         a->mstride, a->minc, a->gnode, a->en, ec, a->ec, a->tab, M.nr, M.colptr, M.valptr,
                         M.ncol, M.val, E.err);
    else
      hipLaunchKernelGGL(k_affine_matrix<8>, g, dim3(PM_WG), lds, c->stream, a->nrn, a->max_cols,
                         a->mstride, a->minc, a->gnode, a->en, ec, a->ec, a->tab, M.nr, M.colptr, M.valptr,
                         M.ncol, M.val, E.err);
  }
  PM_CHECK_HIP(hipGetLastError());
  return PM_OK;
}
