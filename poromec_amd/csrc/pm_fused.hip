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
// iteration before, two (three through the elements) now (an iteration of the
// 4x4x40 column of hexa20/8 25 -> 12.8 us, of batched boxes of 8^3-12^3 59.8 ->
// 18.8).  Pass B of a large one is bound by memory: 0.35 GB in 71 us at 8.7 M
// equations (4.9 TB/s; a copy reaches 5.5).
#include <algorithm>
#include <cstring>

#include "pm_affine.h"
#include "pm_fused.h"
#include "pm_spmv.h"

// ---------------------------------------------------------------------------
// pass A on the stored matrix: a wavefront per node block, UNR columns a lane
// ---------------------------------------------------------------------------
template <typename VT>
struct PmStoredPart {  // UNR columns a lane of a node block: values, t and q
  static constexpr int UNR = 3;
  VT w[UNR][4];
  double t[UNR], q[UNR];
  __device__ __forceinline__ void load(const PmBlockMeta &m, int j0, int lane, const int *ncol,
                                       const VT *val, const PmVecs &V) {
    // past the block's columns a lane takes the last one and drops it after
    // the load; past its rows, row 0 (summed, never stored)
    int col[UNR];
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const int j = j0 + u * 64 + lane, jc = j < m.c ? j : m.c - 1;
      col[u] = ncol[m.cp + jc];
#pragma unroll
      for (int k = 0; k < 4; k++) w[u][k] = val[m.vp + (int64_t)(k < m.n ? k : 0) * m.c + jc];
    }
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      t[u] = V.t[col[u]];
      q[u] = V.q[col[u]];
    }
  }
  __device__ __forceinline__ void add(const PmBlockMeta &m, int j0, int lane, double beta,
                                      double *a) const {
#pragma unroll
    for (int u = 0; u < UNR; u++) {
      const double xq = t[u] + beta * q[u];
      const double x = j0 + u * 64 + lane < m.c ? xq : 0.0;
#pragma unroll
      for (int k = 0; k < 4; k++) a[k] += (double)w[u][k] * x;
    }
  }
};

// The first block's loads are in flight while the scalars form.
template <typename VT, PmMethod MT>
__global__ __launch_bounds__(PM_WG) void k_stored_pass(
    int nrn, const int *__restrict__ fr, const int *__restrict__ nr,
    const int64_t *__restrict__ colptr, const int64_t *__restrict__ valptr,
    const int *__restrict__ ncol, const VT *__restrict__ val, PmVecs V, PmIterState *st, int cur,
    int first, double tol, int nblk, const double *pb, double *pa) {
  constexpr int GROUPS = PM_WG / 64;
  const int lane = threadIdx.x & 63;
  const int grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
  const int lb = pm_xcd_block(blockIdx.x, gridDim.x);
  int64_t k0, k1;
  pm_chunk(nrn, lb, gridDim.x, k0, k1);
  int64_t k = k0 + grp;
  PmBlockMeta m = pm_uniform<64>(pm_block_meta(k, k1, colptr, valptr, nr));
  constexpr int UNR = PmStoredPart<VT>::UNR;
  PmStoredPart<VT> D;
  int f = 0;
  if (k < k1) {
    D.load(m, 0, lane, ncol, val, V);
    f = fr[k];
  }
  const PmIter s = pm_iter_begin<MT>(st, cur, first, tol, nblk, pb);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->it[cur ^ 1] = s;
  if (s.done) return;
  const int qr = pm_row_of(lane);
  double dot[1] = {0.0};
  while (k < k1) {
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    if (!s.pending) {
      D.add(m, 0, lane, s.beta, a);
      for (int j0 = UNR * 64; j0 < m.c; j0 += UNR * 64) {
        D.load(m, j0, lane, ncol, val, V);
        D.add(m, j0, lane, s.beta, a);
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
    k += GROUPS;
    if (k < k1) {
      m = pm_uniform<64>(pm_block_meta(k, k1, colptr, valptr, nr));
      D.load(m, 0, lane, ncol, val, V);
      f = fr[k];
    }
  }
  pm_dots_partials<1>(dot, pa, blockIdx.x);
}

// The same with one run of <= 4 columns per lane and 32 lanes per block
// (k_spmv_chg's layout; two blocks a wavefront): a third of the index words
// and of the loads a column, two runs' descriptors and the first runs' values
// and gathers in flight while the scalars form.
template <typename VT>
struct PmRunPart {  // a lane's run: values of the block's rows, t and q
  int len;
  VT v[4][4];
  double t[4], q[4];
  // base: the block's columns before this pass, returned after it
  __device__ __forceinline__ unsigned int load(unsigned int d, bool valid, unsigned long long gmask,
                                               unsigned int base, unsigned int voff,
                                               unsigned int rowb, __amdgpu_buffer_rsrc_t vr,
                                               __amdgpu_buffer_rsrc_t tr,
                                               __amdgpu_buffer_rsrc_t qr) {
    const unsigned int l1 = d & 3u;
    const unsigned long long bv = __ballot(valid) & gmask;
    const unsigned long long b0 = __ballot(valid && (l1 & 1u)) & gmask;
    const unsigned long long b1 = __ballot(valid && (l1 & 2u)) & gmask;
    const unsigned int off =
        base + pm_lanes_below(bv) + pm_lanes_below(b0) + 2u * pm_lanes_below(b1);
    len = valid ? (int)l1 + 1 : 0;
    // a lane without a run reads past the resources' ends: zeros
    const unsigned int o = valid ? (voff + off) * (unsigned int)sizeof(VT) : PM_PAST_END;
    const unsigned int xo = valid ? (d >> 2) * 8u : 0xffffff00u;
    typedef unsigned int u4 __attribute__((ext_vector_type(4)));
    constexpr int VPR = sizeof(VT) == 4 ? 1 : 2;  // 16-byte loads a row
#pragma unroll
    for (int k = 0; k < 4; k++) {
      u4 w[VPR];
#pragma unroll
      for (int h = 0; h < VPR; h++)
        w[h] = __builtin_bit_cast(u4, __builtin_amdgcn_raw_buffer_load_b128(
                                          vr, o + (unsigned int)k * rowb + 16u * h, 0, 0));
      __builtin_memcpy(v[k], w, sizeof(v[k]));
    }
#pragma unroll
    for (int j = 0; j < 4; j++) {
      t[j] = pm_bload<double, 0>(tr, xo + (unsigned int)j * 8u);
      q[j] = pm_bload<double, 0>(qr, xo + (unsigned int)j * 8u);
    }
    return base + (unsigned int)(__popcll(bv) + __popcll(b0) + 2 * __popcll(b1));
  }
  __device__ __forceinline__ void add(double beta, double *a) const {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const bool in = j == 0 || j < len;  // past the run: other columns, other rows
      const double xq = t[j] + beta * q[j];
      const double x = in ? xq : 0.0;
#pragma unroll
      for (int k = 0; k < 4; k++) a[k] += (double)(in ? v[k][j] : VT(0)) * x;
    }
  }
};

template <typename VT, PmMethod MT>
__global__ __launch_bounds__(PM_WG) void k_stored_runs(
    int nrn, int neq, const int *__restrict__ fr, const int *__restrict__ nr,
    const int64_t *__restrict__ colptr, const int64_t *__restrict__ valptr,
    const int64_t *__restrict__ chptr, const unsigned int *__restrict__ chunk,
    const VT *__restrict__ val, PmVecs V, PmIterState *st, int cur, int first, double tol,
    int nblk, const double *pb, double *pa) {
  constexpr int GROUPS = PM_WG / 64;
  const int lane = threadIdx.x & 63, gi = lane >> 5, gl = lane & 31;
  const unsigned long long gmask = 0xffffffffull << (gi * 32);
  const int grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / 64));
  const int lb = pm_xcd_block(blockIdx.x, gridDim.x);
  int64_t p0, p1;
  pm_chunk(((int64_t)nrn + 1) / 2, lb, gridDim.x, p0, p1);
  int64_t p = p0 + grp;
  const __amdgpu_buffer_rsrc_t tr = pm_rsrc(V.t, (unsigned int)neq * 8u);
  const __amdgpu_buffer_rsrc_t qr = pm_rsrc(V.q, (unsigned int)neq * 8u);
  PmBlocksMeta<2> m;
  PmRunMeta me;
  PmRunPart<VT> D;
  unsigned int d1 = 0, base = 0;
  int f = 0;
  auto descriptor = [&](int h0) {  // of run h0 + gl of the group's block
    const __amdgpu_buffer_rsrc_t hr =
        pm_rsrc(chunk + m.b[0].hp, (unsigned int)(m.b[0].nh + m.b[1].nh) * 4u);
    const unsigned int at = (unsigned int)(me.hp - m.b[0].hp) + (unsigned int)(h0 + gl);
    return (unsigned int)__builtin_amdgcn_raw_buffer_load_b32(hr, at * 4u, 0, 0);
  };
  auto load = [&](int h0, unsigned int d) {
    const __amdgpu_buffer_rsrc_t vr =
        pm_rsrc(val + m.b[0].vp,
                (unsigned int)(m.b[0].n * m.b[0].c + m.b[1].n * m.b[1].c + 3) *
                    (unsigned int)sizeof(VT));
    base = D.load(d, h0 + gl < me.nh, gmask, base, (unsigned int)(me.vp - m.b[0].vp),
                  (unsigned int)me.c * (unsigned int)sizeof(VT), vr, tr, qr);
  };
  auto start = [&] {
    m = pm_blocks_meta<2>(p, p1, nrn, colptr, valptr, nr, chptr);
    me = pm_pick<2>(m, gi);
    const unsigned int d0 = descriptor(0);
    d1 = descriptor(32);
    f = me.n > 0 ? fr[2 * p + gi] : 0;
    base = 0;
    load(0, d0);
  };
  if (p < p1) start();
  const PmIter s = pm_iter_begin<MT>(st, cur, first, tol, nblk, pb);
  if (blockIdx.x == 0 && threadIdx.x == 0) st->it[cur ^ 1] = s;
  if (s.done) return;
  const int row = pm_row_of(gl);
  double dot[1] = {0.0};
  while (p < p1) {
    double a[4] = {0.0, 0.0, 0.0, 0.0};
    if (!s.pending) {
      D.add(s.beta, a);
      const int passes = max(m.b[0].nh, m.b[1].nh);  // the wavefront's
      for (int h0 = 32; h0 < passes; h0 += 32) {
        load(h0, h0 == 32 ? d1 : descriptor(h0));
        D.add(s.beta, a);
      }
    }
    const double y = pm_rows4_sum<32>(gl, a);
    if (gl < 4 && row < me.n) {
      const double qn = pm_row_update<MT>(V, s, f + row);
      if (!s.pending) {
        V.y[f + row] = y;
        dot[0] += y * qn;
      }
    }
    p += GROUPS;
    if (p < p1) start();
  }
  pm_dots_partials<1>(dot, pa, blockIdx.x);
}

// ---------------------------------------------------------------------------
// initial vectors and pass B
// ---------------------------------------------------------------------------
template <bool BATCH>
__global__ __launch_bounds__(PM_WG) void k_fused_init(int64_t n, const double *b, const double *m,
                                                      double *x, double *r, double *t, double *q,
                                                      double *d, double *pb, PmMap M) {
  const PmPart P = pm_part<BATCH, PM_PASS_B>(M, n, nullptr, nullptr, 0, pb);
  double v[2] = {0.0, 0.0};
  const int64_t i0 = P.lo + (int64_t)P.slot * PM_WG + threadIdx.x;
  for (int64_t i = i0; i < P.hi; i += (int64_t)P.nwg * PM_WG) {
    const double bi = b[i], ti = bi * m[i];
    x[i] = 0.0;
    r[i] = bi;
    t[i] = ti;
    q[i] = 0.0;
    d[i] = 0.0;
    v[0] += bi * bi;
    v[1] += bi * ti;
  }
  pm_dots_partials<2>(v, P.out, P.slot);
}

template <PmMethod MT, bool BATCH>
__global__ __launch_bounds__(PM_WG) void k_fused_b(int64_t n, PmIterState *st, int nxt, int nblk,
                                                   const double *pa, const double *y,
                                                   const double *m, const double *q, double *x,
                                                   double *r, double *t, double *pb, PmMap M) {
  const PmPart P = pm_part<BATCH, PM_PASS_B>(M, n, st, pa, nblk, pb);
  // contiguous shares; the first row's loads wait for neither scalars nor sums
  int64_t i0, i1;
  pm_share(P, i0, i1);
  int64_t i = i0 + threadIdx.x;
  const int64_t il = i < i1 ? i : P.lo;
  double yi = y[il], ri = r[il], mi = m[il];
  const PmIter s = P.st->it[nxt];
  if (s.done || s.pending) return;
  double sum[1];
  pm_sum_dots<1>(P.nin, P.in, sum);
  const bool lead = P.wg == 0 && threadIdx.x == 0;
  if (MT == PM_IT_SQMR && sum[0] == 0.0) {
    if (lead) P.st->step.broken = 1;
    return;
  }
  const double alpha = s.ro / sum[0];
  if (lead) {
    P.st->step.alpha = alpha;
    P.st->step.broken = 0;
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
  pm_dots_partials<2>(v, P.out, P.slot);
}

// the update and the stop test of the last iteration launched
template <PmMethod MT, bool BATCH>
__global__ __launch_bounds__(PM_WG) void k_fused_tail(int64_t n, PmVecs V, PmIterState *st, int cur,
                                                      int nblk, const double *pb, PmMap M) {
  PmPart P = pm_part<BATCH, PM_PASS_B>(M, n, st, pb, nblk, nullptr);
  if (BATCH) {  // pass B's partials come in here
    const PmBoxInfo B = M.box[M.wg[blockIdx.x].x];
    P.in = pb + 2 * B.bbase;
    P.nin = B.nb;
  }
  PmIter s = pm_iter_begin<MT>(P.st, cur, 0, 0.0, P.nin, P.in);
  const bool update = !s.done;
  if (s.pending) s.done = s.pending;
  if (P.wg == 0 && threadIdx.x == 0) P.st->it[cur ^ 1] = s;
  if (!update) return;
  int64_t i0, i1;
  pm_share(P, i0, i1);
  for (int64_t i = i0 + threadIdx.x; i < i1; i += PM_WG) (void)pm_row_update<MT>(V, s, i);
}

// ---------------------------------------------------------------------------
// driver
// ---------------------------------------------------------------------------
// The stored product by runs of columns from 2 million values on where the
// runs are long enough to fill a lane's four values.  us an SQMR iteration,
// by columns / by runs: hexa20/8 1.2 M 11.8 / 12.2, 2.4 M 13.3 / 13.3, 3.2 M
// 17.2 / 14.2, 6.7 M 25.6 / 22.3, 12.2 M 33.8 / 34.5, 20 M 48.4 / 44.8; Q1/Q1
// 2.4 M 15.2 / 12.6, 5.8 M 23.1 / 20.4, 13.8 M 40.0 / 34.2; FP32 values 14.7 /
// 13.6 at 3.2 M, Q1/Q1 34.1 / 30.7 at 13.8 M.
static bool stored_runs(const PmDevMatrix &A) {
  return A.nnz >= 2000000 && A.ncols >= 2 * A.nchunks;
}

// Always through the elements; on the stored matrix by runs up to 30 million
// values (FP32: 40), by columns up to 12 (24).  Beyond, the product's two
// gathers a column cost more than the finishers: an SQMR iteration in three
// passes / by runs takes 52.4 / 44.8 us at 20 M values (hexa20/8 20^3), 84.8 /
// 85.3 at 35 M, 136 / 145 at 56 M; Q1/Q1 61.3 / 52.8 at 27 M (40^3), 110 / 115
// at 47 M; FP32 60.3 / 52.7 at 35 M, 81.3 / 87.5 at 56 M, Q1/Q1 73.7 / 64.2 at
// 47 M.  By columns 41.5 / 41.7 at 13.8 M.
bool pm_fused_usable(const pm_ctx *c, int use32) {
  if (c->ordered) return false;
  const int64_t most = stored_runs(c->A) ? (use32 ? 40000000 : 30000000)
                                         : (use32 ? 24000000 : 12000000);
  return pm_affine_product(c, use32) || c->A.nnz <= most;
}

template <typename VT, PmMethod MT>
static int stored_pass(pm_ctx *c, const VT *val, const PmVecs &V, PmIterState *st, int cur,
                       int first, double tol, int nblk, const double *pb, double *pa) {
  const PmDevMatrix &A = c->A;
  if (stored_runs(A)) {
    int g = (A.nrn + PM_WG / 32 - 1) / (PM_WG / 32);
    g = (std::min(g, PM_MAX_GRID) + 7) & ~7;
    hipLaunchKernelGGL((k_stored_runs<VT, MT>), dim3(g), dim3(PM_WG), 0, c->stream, A.nrn, A.neq,
                       A.fr, A.nr, A.colptr, A.valptr, A.chptr, A.chunk, val, V, st, cur, first,
                       tol, nblk, pb, pa);
    return g;
  }
  int g = (A.nrn + PM_WG / 64 - 1) / (PM_WG / 64);
  g = (std::min(g, PM_MAX_GRID) + 7) & ~7;
  hipLaunchKernelGGL((k_stored_pass<VT, MT>), dim3(g), dim3(PM_WG), 0, c->stream, A.nrn, A.fr,
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
  hipLaunchKernelGGL(k_fused_init<false>, dim3(gv), dim3(PM_WG), 0, c->stream, (int64_t)n, b, m, x,
                     r, t, q[0], d, pb, PmMap{});
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
      hipLaunchKernelGGL((k_fused_b<MT, false>), dim3(gv), dim3(PM_WG), 0, c->stream, (int64_t)n,
                         st, cur ^ 1, ga, pa, y, m, V.qn, x, r, t, pb, PmMap{});
      (use32 ? info->spmv32 : info->spmv64)++;
    }
    launched += chunk;
    int last = launched & 1;  // slot written by the last pass A
    if (launched >= maxit) {
      const PmVecs V{t, q[last], q[last ^ 1], d, x, y};
      hipLaunchKernelGGL((k_fused_tail<MT, false>), dim3(gv), dim3(PM_WG), 0, c->stream, (int64_t)n,
                         V, st, last, gv, pb, PmMap{});
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

// ---------------------------------------------------------------------------
// every box of a batch its own solve
// ---------------------------------------------------------------------------
struct PmFusedBoxes {
  int nbox = 0;
  std::vector<PmBoxInfo> box;
  PmBoxInfo *d_box = nullptr;
  int4 *d_wg = nullptr;  // the three maps, one after the other
  size_t wg_cap = 0;
  PmIterState *d_st = nullptr, *h_st = nullptr;
  double *d_part = nullptr;
  size_t pa_len = 0;
  ~PmFusedBoxes() {
    (void)hipFree(d_box);
    (void)hipFree(d_wg);
    (void)hipFree(d_st);
    (void)hipFree(d_part);
    if (h_st) (void)hipHostFree(h_st);
  }
};

void pm_fused_boxes_free(PmFusedBoxes *f) { delete f; }

static int boxes_setup(pm_ctx *c, PmFusedBoxes **fb, const std::vector<int> &eq0,
                       const std::vector<int> &blk0) {
  std::vector<int> p0;
  if (!pm_affine_box_patches(c, blk0, p0)) return PM_OK;
  const int nbox = (int)eq0.size() - 1, pw = pm_affine_patch_waves(c);
  PmFusedBoxes *f = new PmFusedBoxes();
  f->nbox = nbox;
  f->box.resize(nbox);
  size_t na = 0, nb = 0, ne = 0;
  for (int b = 0; b < nbox; b++) {
    PmBoxInfo &B = f->box[b];
    B.p0 = p0[b];
    B.p1 = p0[b + 1];
    B.k0 = blk0[b];
    B.k1 = blk0[b + 1];
    B.e0 = eq0[b];
    B.e1 = eq0[b + 1];
    // as in the single solve: 64 nodes and a row per thread a workgroup, up
    // to 256 and 128 workgroups a box
    B.na = std::min(256, std::max(1, (B.k1 - B.k0 + PM_WG / 4 - 1) / (PM_WG / 4)));
    B.nb = std::min(128, std::max(1, (B.e1 - B.e0 + PM_WG - 1) / PM_WG));
    B.abase = (int)na;
    B.bbase = (int)nb;
    na += B.na;
    nb += B.nb;
    ne += std::max(1, (B.p1 - B.p0 + pw - 1) / pw);
  }
  f->pa_len = na;
  f->wg_cap = ne + na + nb;
  bool ok = hipMalloc((void **)&f->d_box, sizeof(PmBoxInfo) * nbox) == hipSuccess &&
            hipMalloc((void **)&f->d_wg, sizeof(int4) * f->wg_cap) == hipSuccess &&
            hipMalloc((void **)&f->d_st, sizeof(PmIterState) * nbox) == hipSuccess &&
            hipMalloc((void **)&f->d_part, sizeof(double) * (na + 2 * nb)) == hipSuccess &&
            hipHostMalloc((void **)&f->h_st, sizeof(PmIterState) * nbox, hipHostMallocDefault) ==
                hipSuccess &&
            hipMemcpy(f->d_box, f->box.data(), sizeof(PmBoxInfo) * nbox, hipMemcpyHostToDevice) ==
                hipSuccess;
  if (!ok) {  // the stored-matrix batch needs none of this
    (void)hipGetLastError();
    delete f;
    return PM_OK;
  }
  *fb = f;
  return PM_OK;
}

template <PmMethod MT>
static int batch_solve(pm_ctx *c, PmFusedBoxes *f, const double *b, double *x, const double *m,
                       double tol, int maxit, int use32, int cap, std::vector<int> &iters,
                       std::vector<int> &done, std::vector<double> &resid, int *out_launched) {
  double *y = c->d_wk[0], *r = c->d_wk[1], *t = c->d_wk[2], *d = c->d_wk[3];
  double *q[2] = {c->d_wk[4], c->d_wk[5]};
  double *pa = f->d_part, *pb = f->d_part + f->pa_len;
  const int nbox = f->nbox, pw = pm_affine_patch_waves(c);
  PmIterState *st = f->d_st;
  done.assign(nbox, 0);
  iters.assign(nbox, 0);
  resid.assign(nbox, 0.0);
  // maps of the open boxes' workgroups; a box keeps its own numbers
  PmMap me{nullptr, f->d_box}, mn = me, mb = me;
  int ne = 0, nn = 0, nv = 0;
  auto build = [&]() -> int {
    std::vector<int4> w;
    for (int pass = 0; pass < 3; pass++) {
      const size_t at = w.size();
      for (int k = 0; k < nbox; k++) {
        if (done[k]) continue;
        const PmBoxInfo &B = f->box[k];
        const int g = pass == 0 ? std::max(1, (B.p1 - B.p0 + pw - 1) / pw) : pass == 1 ? B.na : B.nb;
        for (int i = 0; i < g; i++) w.push_back(int4{k, i, g, 0});
      }
      (pass == 0 ? me : pass == 1 ? mn : mb).wg = f->d_wg + at;
      (pass == 0 ? ne : pass == 1 ? nn : nv) = (int)(w.size() - at);
    }
    if (!w.empty())
      PM_CHECK_HIP(hipMemcpy(f->d_wg, w.data(), sizeof(int4) * w.size(), hipMemcpyHostToDevice));
    return PM_OK;
  };
  PM_TRY(build());
  hipLaunchKernelGGL(k_fused_init<true>, dim3(nv), dim3(PM_WG), 0, c->stream, (int64_t)0, b, m, x, r,
                     t, q[0], d, pb, mb);
  int launched = 0, open = nbox, open_last = nbox, half_at = -1;
  while (open > 0 && launched < maxit) {
    if (cap && half_at >= 0 && launched >= 4 * std::max(half_at, 64)) break;
    const int chunk = std::min(launched < 32 ? 8 : 32, maxit - launched);
    for (int k = 0; k < chunk; k++) {
      const int it = launched + k, cur = it & 1;
      const PmVecs V{t, q[cur], q[cur ^ 1], d, x, y};
      pm_affine_pass_boxes(c, MT, V, st, cur, it == 0, tol, pb, pa, me, ne, mn, nn);
      hipLaunchKernelGGL((k_fused_b<MT, true>), dim3(nv), dim3(PM_WG), 0, c->stream, (int64_t)0, st,
                         cur ^ 1, 0, pa, y, m, V.qn, x, r, t, pb, mb);
    }
    launched += chunk;
    int last = launched & 1;
    const bool end = launched >= maxit ||
                     (cap && half_at >= 0 && launched >= 4 * std::max(half_at, 64));
    if (end) {
      const PmVecs V{t, q[last], q[last ^ 1], d, x, y};
      hipLaunchKernelGGL((k_fused_tail<MT, true>), dim3(nv), dim3(PM_WG), 0, c->stream, (int64_t)0,
                         V, st, last, 0, pb, mb);
      last ^= 1;
    }
    PM_CHECK_HIP(hipGetLastError());
    PM_CHECK_HIP(hipMemcpyAsync(f->h_st, st, sizeof(PmIterState) * nbox, hipMemcpyDeviceToHost,
                                c->stream));
    PM_CHECK_HIP(hipStreamSynchronize(c->stream));
    double worst = 0.0;
    for (int k = 0; k < nbox; k++) {
      if (done[k]) continue;
      const PmIter &s = f->h_st[k].it[last];
      iters[k] = s.it;
      resid[k] = s.resid;
      worst = std::max(worst, s.resid);
      done[k] = s.done ? s.done : s.pending;  // pending: the last pass A made the update
      open -= done[k] != 0;
    }
    pm_progress(launched, worst);
    if (half_at < 0 && 2 * (nbox - open) >= nbox) half_at = launched;
    if (end) break;
    // the finished boxes' workgroups leave when a quarter of them is idle
    if (open > 0 && 4 * open <= 3 * open_last) {
      PM_TRY(build());
      open_last = open;
    }
  }
  *out_launched = launched;
  return PM_OK;
}

int pm_fused_batch_solve(pm_ctx *c, PmFusedBoxes **fb, const std::vector<int> &eq0,
                         const std::vector<int> &blk0, PmMethod mt, const double *b, double *x,
                         const double *m, double tol, int maxit, int use32, int cap,
                         std::vector<int> &iters, std::vector<int> &done,
                         std::vector<double> &resid, int *launched, int *usable) {
  *usable = 0;
  if (!pm_affine_product(c, use32)) return PM_OK;
  if (!*fb) PM_TRY(boxes_setup(c, fb, eq0, blk0));
  if (!*fb) return PM_OK;
  *usable = 1;
  return mt == PM_IT_SQMR ? batch_solve<PM_IT_SQMR>(c, *fb, b, x, m, tol, maxit, use32, cap, iters,
                                                    done, resid, launched)
                          : batch_solve<PM_IT_PCG>(c, *fb, b, x, m, tol, maxit, use32, cap, iters,
                                                   done, resid, launched);
}
