// pm_fused.h -- scalars of the fused SQMR and PCG iterations (pm_fused.hip).
//
// An iteration is a product pass A and a vector pass B.  Each pass leaves
// workgroup partials of its dots; the workgroups of the next pass sum them
// again, all in the same fixed order, and so all hold the same scalars
// without a finisher kernel between the passes.  Workgroup 0 writes the
// scalars for the passes after that one.  A pass never reads what its own
// launch writes: A takes slot it & 1 to slot (it + 1) & 1, B writes PmStep.
#pragma once
#include "pm_device.h"
#include "pm_spmv.h"

enum PmMethod { PM_IT_SQMR, PM_IT_PCG };

struct PmIter {
  double conv;         // stop threshold of the recurrence residual
  double ro, tau, v0;  // SQMR: rho, tau, theta; PCG: ro = r . M^-1 r
  double t1, t2, beta; // coefficients of the pending update of d and q
  double resid;        // recurrence residual of the last finished iteration
  int done;            // 0 running, 1 converged, < 0 PM_ERR_* code
  int pending;         // converged (1) or broken down (< 0): this pass A still
                       // makes the finished iteration's update, then done
  int it;              // iterations started
  int pad;
};
struct PmStep {
  double alpha;
  int broken;  // the product's dot vanished (SQMR)
  int pad;
};
struct PmIterState {  // device
  PmIter it[2];
  PmStep step;
};

// Sums of the partials of nblk workgroups, the same in every workgroup: as
// pm_sum_partials, the wavefront sums by DPP instead of six LDS permutes each
// (they sit on every pass's critical path).
template <int NV, int WAVES = PM_WAVES>
__device__ __forceinline__ void pm_sum_dots(int nblk, const double *partials, double *out) {
  __shared__ double sh[NV][WAVES];
  double acc[NV];
#pragma unroll
  for (int i = 0; i < NV; i++) acc[i] = 0.0;
  for (int b = threadIdx.x; b < nblk; b += WAVES * 64)
#pragma unroll
    for (int i = 0; i < NV; i++) acc[i] += partials[(size_t)b * NV + i];
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const double w = pm_group_sum<64>(acc[i]);
    if ((threadIdx.x & 63) == 63) sh[i][threadIdx.x >> 6] = w;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NV; i++) {
    out[i] = sh[i][0];
    for (int w = 1; w < WAVES; w++) out[i] += sh[i][w];
  }
}

// workgroup partials of NV dots, DPP sums
template <int NV>
__device__ __forceinline__ void pm_dots_partials(const double *v, double *partials, int wg) {
  __shared__ double sh[NV][PM_WAVES];
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const double w = pm_group_sum<64>(v[i]);
    if ((threadIdx.x & 63) == 63) sh[i][threadIdx.x >> 6] = w;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double acc = sh[threadIdx.x][0];
    for (int w = 1; w < PM_WAVES; w++) acc += sh[threadIdx.x][w];
    partials[(size_t)wg * NV + threadIdx.x] = acc;
  }
}

// Scalars of the iteration that pass A starts: from the partials of pass B
// of the last one (first: of the initial vectors), RPSQMR (Iters.f:6100-6436)
// and PCG (Iters.f:299-595).  Called by whole workgroups; every thread
// receives the same values.
template <PmMethod MT, int WAVES = PM_WAVES, bool BATCH = false>
__device__ __forceinline__ PmIter pm_iter_begin(const PmIterState *st, int cur, int first, double tol,
                                                int nblk, const double *partials) {
  PmIter s = st->it[cur];
  if (first) {
    double r[2];
    pm_sum_dots<2, WAVES>(nblk, partials, r);
    s.v0 = s.t1 = s.t2 = s.beta = 0.0;
    s.resid = 0.0;
    s.done = s.pending = 0;
    s.it = 1;
    if (MT == PM_IT_SQMR) {
      s.conv = tol * sqrt(fabs(r[0]));
      s.tau = sqrt(r[0]);
      s.ro = r[1];
    } else {
      s.conv = tol * sqrt(fabs(r[1]));
      s.tau = 0.0;
      s.ro = r[1];
    }
    if (BATCH && r[0] == 0.0) {  // a box without load: x = 0
      s.done = 1;
      s.it = 0;
    }
    return s;
  }
  if (s.done) return s;
  if (s.pending) {  // the update was made by the last pass A
    s.done = s.pending;
    return s;
  }
  if (MT == PM_IT_SQMR && st->step.broken) {
    s.done = PM_ERR_BREAKDOWN;
    return s;
  }
  double r[2];
  pm_sum_dots<2, WAVES>(nblk, partials, r);
  if (MT == PM_IT_SQMR) {
    const double normr = sqrt(r[0]);
    const double vn = normr / s.tau;
    const double cn = 1.0 / sqrt(1.0 + vn * vn);
    s.tau = s.tau * vn * cn;
    s.t1 = cn * cn * s.v0 * s.v0;
    s.t2 = cn * cn * st->step.alpha;
    s.v0 = vn;
    if (s.ro == 0.0) {
      s.pending = PM_ERR_BREAKDOWN;
      return s;
    }
    s.beta = r[1] / s.ro;
    s.ro = r[1];
    s.resid = normr;
    if (normr < s.conv) s.pending = 1;
  } else {
    s.beta = r[1] / s.ro;
    s.ro = r[1];
    s.resid = sqrt(fabs(r[1]));
    if (s.resid < s.conv) s.pending = 1;
  }
  if (!s.pending) s.it += 1;
  return s;
}

// vectors of an iteration: q_new = t + beta q; SQMR also d = t1 d + t2 q,
// x += d (PCG moves x in pass B)
struct PmVecs {
  const double *t, *q;
  double *qn, *d, *x, *y;
};

// one row of pass A's update; returns q_new
template <PmMethod MT>
__device__ __forceinline__ double pm_row_update(const PmVecs &V, const PmIter &s, int64_t i) {
  const double qi = V.q[i];
  if (MT == PM_IT_SQMR) {
    const double di = s.t1 * V.d[i] + s.t2 * qi;
    V.d[i] = di;
    V.x[i] = V.x[i] + di;
  }
  const double qn = V.t[i] + s.beta * qi;
  V.qn[i] = qn;
  return qn;
}

// The batching form: every box its own scalars, partials and workgroups.  A
// pass's workgroups are listed in a map (x box, y the workgroup's number among
// the box's, z their number) that holds the open boxes only; a box's own
// numbers never change, so neither do its sums.
struct PmBoxInfo {
  int p0, p1, k0, k1, e0, e1;  // patches, row blocks, equations
  int na, abase, nb, bbase;    // workgroups of passes A (node part) and B, first partials
};
struct PmMap {
  const int4 *wg;
  const PmBoxInfo *box;
};

// a workgroup's part of a pass: number `wg` of `nwg`, on items [lo, hi)
struct PmPart {
  int wg, nwg, slot;  // slot: of its partials
  int64_t lo, hi;
  PmIterState *st;
  const double *in;
  int nin;
  double *out;
};
enum PmPass { PM_PASS_ELEMS, PM_PASS_NODES, PM_PASS_B };

template <bool BATCH, PmPass PASS>
__device__ __forceinline__ PmPart pm_part(const PmMap &M, int64_t n, PmIterState *st,
                                          const double *in, int nin, double *out) {
  if constexpr (BATCH) {
    const int4 w = M.wg[blockIdx.x];
    const PmBoxInfo B = M.box[w.x];
    PmPart P{w.y, w.z, w.y, 0, 0, st + w.x, nullptr, 0, nullptr};
    if (PASS == PM_PASS_ELEMS) {
      P.lo = B.p0;
      P.hi = B.p1;
    } else if (PASS == PM_PASS_NODES) {
      P.lo = B.k0;
      P.hi = B.k1;
    } else {
      P.lo = B.e0;
      P.hi = B.e1;
    }
    P.in = PASS == PM_PASS_B ? in + B.abase : in + 2 * B.bbase;
    P.nin = PASS == PM_PASS_B ? B.na : B.nb;
    P.out = PASS == PM_PASS_B ? out + 2 * B.bbase : out + B.abase;
    return P;
  } else {
    return PmPart{pm_xcd_block(blockIdx.x, gridDim.x), (int)gridDim.x, (int)blockIdx.x, 0, n, st,
                  in, nin, out};
  }
}
// the part's contiguous share of its items
__device__ __forceinline__ void pm_share(const PmPart &P, int64_t &a, int64_t &b) {
  pm_chunk(P.hi - P.lo, P.wg, P.nwg, a, b);
  a += P.lo;
  b += P.lo;
}

// pass A of every open box through the elements: maps of the element and the
// node part
void pm_affine_pass_boxes(pm_ctx *c, PmMethod mt, const PmVecs &V, PmIterState *st, int cur,
                          int first, double tol, const double *pb, double *pa, const PmMap &elems,
                          int n_elems, const PmMap &nodes, int n_nodes);
// patches of the row blocks [blk0[b], blk0[b + 1]); false if they do not split so
bool pm_affine_box_patches(const pm_ctx *c, const std::vector<int> &blk0, std::vector<int> &p0);
int pm_affine_patch_waves(const pm_ctx *c);

struct PmFusedBoxes;  // buffers of the batched solve
void pm_fused_boxes_free(PmFusedBoxes *f);
// SQMR or PCG on every box (eq0, blk0: nbox + 1 first equations and blocks);
// iters and done per box (1 converged, < 0 error, 0 open).  cap != 0: once
// half the boxes have converged at iteration L, stop at 4 L.  *usable = 0 and
// nothing done where the elements do not serve.
int pm_fused_batch_solve(pm_ctx *c, PmFusedBoxes **fb, const std::vector<int> &eq0,
                         const std::vector<int> &blk0, PmMethod mt, const double *b, double *x,
                         const double *m, double tol, int maxit, int use32, int cap,
                         std::vector<int> &iters, std::vector<int> &done,
                         std::vector<double> &resid, int *launched, int *usable);

// pass A through the elements (pm_affine.hip); returns the grid of its partials
int pm_affine_pass(pm_ctx *c, PmMethod mt, const PmVecs &V, PmIterState *st, int cur, int first,
                   double tol, int nblk, const double *pb, double *pa);

// true if the solve can run fused
bool pm_fused_usable(const pm_ctx *c, int use32);
int pm_fused_solve(pm_ctx *c, PmMethod mt, int n, const double *b, double *x, const double *m,
                   double tol, int maxit, int use32, pm_solve_info *info, int *converged);
