// pm_fused.hip -- SQMR (Iters.f:6100-6436) and PCG (Iters.f:299-595) in two
// passes an iteration, without finisher kernels between them (pm_fused.h):
//
//   A  beta (and SQMR's tau, c) from pass B's dots; q_new = t + beta q formed
//      at every gathered column and stored by its row's owner together with
//      the update of d and x; y = A q_new; the dot q_new . y
//   B  alpha from that dot; r -= alpha y, t = M r; the dots r . r and r . t
//      (PCG: x += alpha q too)
//
// The values are those of the separate loops, expression by expression.  What
// bounds a small system is the chain of dependent kernels: six of 1.4-8 us an
// iteration before, two (three through the elements) now.
#include <algorithm>
#include <cstring>

#include "pm_affine.h"
#include "pm_fused.h"
#include "pm_spmv.h"

// ---------------------------------------------------------------------------
// pass A on the stored matrix: a wavefront per node block, UNR columns a lane
// ---------------------------------------------------------------------------
template <typename VT, int UNR, PmMethod MT>
__global__ __launch_bounds__(PM_WG) void k_stored_pass(
    int nrn, const int *__restrict__ fr, const int *__restrict__ nr,
    const int64_t *__restrict__ colptr, const int64_t *__restrict__ valptr,
    const int *__restrict__ ncol, const VT *__restrict__ val, PmVecs V, PmIterState *st, int cur,
    int first, double tol, int nblk, const double *pb, double *pa) {
  const PmIter s = pm_iter_begin<MT>(st, cur, first, tol, nblk, pb);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->it[cur ^ 1] = s;
  if (s.done) return;
  constexpr int GROUPS = PM_WG / 64;
  const int lane = threadIdx.x & 63;
  const int grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
  const int lb = pm_xcd_block(blockIdx.x, gridDim.x);
  int64_t k0, k1;
  pm_chunk(nrn, lb, gridDim.x, k0, k1);
  const int qr = pm_row_of(lane);
  double dot[1] = {0.0};
  for (int64_t k = k0 + grp; k < k1; k += GROUPS) {
    const PmBlockMeta m = pm_uniform<64>(pm_block_meta(k, k1, colptr, valptr, nr));
    const int f = fr[k];
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    if (!s.pending) {
      for (int j0 = 0; j0 < m.c; j0 += UNR * 64) {
        // past the block's columns a lane takes the last one and drops it
        // after the load; past its rows, row 0 (summed, never stored)
        int col[UNR];
        VT w[UNR][4];
#pragma unroll
        for (int u = 0; u < UNR; u++) {
          const int j = j0 + u * 64 + lane, jc = j < m.c ? j : m.c - 1;
          col[u] = ncol[m.cp + jc];
#pragma unroll
          for (int q = 0; q < 4; q++) w[u][q] = val[m.vp + (int64_t)(q < m.n ? q : 0) * m.c + jc];
        }
        double xq[UNR];
#pragma unroll
        for (int u = 0; u < UNR; u++) xq[u] = V.t[col[u]] + s.beta * V.q[col[u]];
#pragma unroll
        for (int u = 0; u < UNR; u++) {
          const double x = j0 + u * 64 + lane < m.c ? xq[u] : 0.0;
#pragma unroll
          for (int q = 0; q < 4; q++) a[q] += (double)w[u][q] * x;
        }
      }
    }
    const double y = pm_rows4_sum<64>(lane, a);
    if (lane < 4 && qr < m.n) {
      const int row = f + qr;
      const double qn = pm_row_update<MT>(V, s, row);
      if (!s.pending) {
        V.y[row] = y;
        dot[0] += y * qn;
      }
    }
  }
  pm_dots_partials<1>(dot, pa);
}

// ---------------------------------------------------------------------------
// initial vectors and pass B
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(PM_WG) void k_fused_init(int64_t n, const double *b, const double *m,
                                                      double *x, double *r, double *t, double *q,
                                                      double *d, double *pb) {
  double v[2] = {0.0, 0.0};
  for (int64_t i = (int64_t)blockIdx.x * PM_WG + threadIdx.x; i < n; i += (int64_t)gridDim.x * PM_WG) {
    const double bi = b[i], ti = bi * m[i];
    x[i] = 0.0;
    r[i] = bi;
    t[i] = ti;
    q[i] = 0.0;
    d[i] = 0.0;
    v[0] += bi * bi;
    v[1] += bi * ti;
  }
  pm_dots_partials<2>(v, pb);
}

template <PmMethod MT>
__global__ __launch_bounds__(PM_WG) void k_fused_b(int64_t n, PmIterState *st, int nxt, int nblk,
                                                   const double *pa, const double *y,
                                                   const double *m, const double *q, double *x,
                                                   double *r, double *t, double *pb) {
  const PmIter s = st->it[nxt];
  if (s.done || s.pending) return;
  // XCD-contiguous chunks; the first row's loads do not wait for the sums
  int64_t i0, i1;
  pm_chunk(n, pm_xcd_block(blockIdx.x, gridDim.x), gridDim.x, i0, i1);
  int64_t i = i0 + threadIdx.x;
  const bool on = i < i1;
  double yi = on ? y[i] : 0.0, ri = on ? r[i] : 0.0, mi = on ? m[i] : 0.0;
  double sum[1];
  pm_sum_dots<1>(nblk, pa, sum);
  if (MT == PM_IT_SQMR && sum[0] == 0.0) {
    if (blockIdx.x == 0 && threadIdx.x == 0) st->step.broken = 1;
    return;
  }
  const double alpha = s.ro / sum[0];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->step.alpha = alpha;
    st->step.broken = 0;
  }
  double v[2] = {0.0, 0.0};
  while (i < i1) {
    if (MT == PM_IT_PCG) x[i] = x[i] + alpha * q[i];
    const double rn = ri - alpha * yi;
    r[i] = rn;
    const double tn = rn * mi;
    t[i] = tn;
    if (MT == PM_IT_SQMR) v[0] += rn * rn;
    v[1] += rn * tn;
    i += PM_WG;
    if (i < i1) {
      yi = y[i];
      ri = r[i];
      mi = m[i];
    }
  }
  pm_dots_partials<2>(v, pb);
}

// the update and the stop test of the last iteration launched
template <PmMethod MT>
__global__ __launch_bounds__(PM_WG) void k_fused_tail(int64_t n, PmVecs V, PmIterState *st, int cur,
                                                      int nblk, const double *pb) {
  PmIter s = pm_iter_begin<MT>(st, cur, 0, 0.0, nblk, pb);
  const bool update = !s.done;
  if (s.pending) s.done = s.pending;
  if (blockIdx.x == 0 && threadIdx.x == 0) st->it[cur ^ 1] = s;
  if (!update) return;
  for (int64_t i = (int64_t)blockIdx.x * PM_WG + threadIdx.x; i < n; i += (int64_t)gridDim.x * PM_WG)
    (void)pm_row_update<MT>(V, s, i);
}

// ---------------------------------------------------------------------------
// driver
// ---------------------------------------------------------------------------
// Always through the elements; on the stored matrix up to 12 million values
// (FP32: 24).  Beyond, the product's two gathers a column cost more than the
// finishers: an SQMR iteration, three passes with the tuned SpMV shape / fused,
// takes 44.5 / 33.6 us at 12.2 M values (hexa20/8 17^3), 57.9 / 47.3 at 20 M,
// 88.8 / 102 at 35 M; Q1/Q1 41.5 / 41.7 at 13.8 M (32^3), 61.0 / 76.1 at 27 M;
// FP32 59.2 / 57.1 at 35 M, Q1/Q1 53.5 / 53.8 at 27 M.
bool pm_fused_usable(const pm_ctx *c, int use32) {
  if (c->ordered) return false;
  return pm_affine_product(c, use32) || c->A.nnz <= (use32 ? 24000000 : 12000000);
}

template <typename VT, PmMethod MT>
static int stored_pass(pm_ctx *c, const VT *val, const PmVecs &V, PmIterState *st, int cur,
                       int first, double tol, int nblk, const double *pb, double *pa) {
  const PmDevMatrix &A = c->A;
  int g = (A.nrn + PM_WG / 64 - 1) / (PM_WG / 64);
  g = (std::min(g, PM_MAX_GRID) + 7) & ~7;
  hipLaunchKernelGGL((k_stored_pass<VT, 3, MT>), dim3(g), dim3(PM_WG), 0, c->stream, A.nrn, A.fr,
                     A.nr, A.colptr, A.valptr, A.ncol, val, V, st, cur, first, tol, nblk, pb, pa);
  return g;
}

// grid of the vector passes: a row per thread up to 512 workgroups (their
// partials are summed by every workgroup of the next pass A; two rows a thread
// measured the same, four 0.5-1 us an iteration more), 1024 beyond
static int vec_grid(int64_t n) {
  const int64_t g = (n + PM_WG - 1) / PM_WG;
  return (int)((std::min<int64_t>(g, n > 2000000 ? 1024 : 512) + 7) & ~7);
}

template <PmMethod MT>
static int solve(pm_ctx *c, int n, const double *b, double *x, const double *m, double tol,
                 int maxit, int use32, pm_solve_info *info, int *converged) {
  double *y = c->d_wk[0], *r = c->d_wk[1], *t = c->d_wk[2], *d = c->d_wk[3];
  double *q[2] = {c->d_wk[4], c->d_wk[5]};
  double *pa = c->d_partials, *pb = c->d_partials + 8192;
  PmIterState *st = c->d_iter;
  *converged = 0;
  const bool elems = pm_affine_product(c, use32);
  const int gv = vec_grid(n);
  hipLaunchKernelGGL(k_fused_init, dim3(gv), dim3(PM_WG), 0, c->stream, (int64_t)n, b, m, x, r, t,
                     q[0], d, pb);
  int launched = 0;
  PmIter h{};
  while (launched < maxit) {
    const int chunk = std::min(launched < 32 ? 8 : launched < 256 ? 32 : 64, maxit - launched);
    for (int k = 0; k < chunk; k++) {
      const int it = launched + k, cur = it & 1;
      const PmVecs V{t, q[cur], q[cur ^ 1], d, x, y};
      c->cur_iter = it + 1;
      pm_spmv_time_begin(c);
      const int ga =
          elems ? pm_affine_pass(c, MT, V, st, cur, it == 0, tol, gv, pb, pa)
          : use32 ? stored_pass<float, MT>(c, c->A.val32, V, st, cur, it == 0, tol, gv, pb, pa)
                  : stored_pass<double, MT>(c, c->A.val, V, st, cur, it == 0, tol, gv, pb, pa);
      pm_spmv_time_end(c, use32);
      hipLaunchKernelGGL(k_fused_b<MT>, dim3(gv), dim3(PM_WG), 0, c->stream, (int64_t)n, st,
                         cur ^ 1, ga, pa, y, m, V.qn, x, r, t, pb);
      (use32 ? info->spmv32 : info->spmv64)++;
    }
    launched += chunk;
    int last = launched & 1;  // slot written by the last pass A
    if (launched >= maxit) {
      const PmVecs V{t, q[last], q[last ^ 1], d, x, y};
      hipLaunchKernelGGL(k_fused_tail<MT>, dim3(gv), dim3(PM_WG), 0, c->stream, (int64_t)n, V, st,
                         last, gv, pb);
      last ^= 1;
    }
    PM_CHECK_HIP(hipGetLastError());
    PM_CHECK_HIP(hipMemcpyAsync(c->h_iter, &st->it[last], sizeof(PmIter), hipMemcpyDeviceToHost,
                                c->stream));
    PM_CHECK_HIP(hipStreamSynchronize(c->stream));
    h = *c->h_iter;
    pm_progress(launched, h.resid);
    if (c->tev_used) pm_spmv_harvest(c, h.done | h.pending, h.it);
    if (h.done || h.pending) break;  // pending: the last pass A made the update
  }
  const int end = h.done ? h.done : h.pending;
  if (end < 0) return end;
  *converged = end == 1;
  if (*converged) {
    info->iters += h.it;
    info->resid = h.resid;
  }
  return PM_OK;
}

int pm_fused_solve(pm_ctx *c, PmMethod mt, int n, const double *b, double *x, const double *m,
                   double tol, int maxit, int use32, pm_solve_info *info, int *converged) {
  return mt == PM_IT_SQMR ? solve<PM_IT_SQMR>(c, n, b, x, m, tol, maxit, use32, info, converged)
                          : solve<PM_IT_PCG>(c, n, b, x, m, tol, maxit, use32, info, converged);
}
