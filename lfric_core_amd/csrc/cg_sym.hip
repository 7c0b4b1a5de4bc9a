// Conjugate gradient iteration over the symmetric-packed copy of a lowest-order W0 operator, in three
// kernels: units, gather with the residual's update, and the step of x and p.
//   Bound: HBM.  Against the apply in two kernels, the update and aypx in one each, A p is not written and read
// back, p is read once less and there is a launch less: FP32 C96x70 112 + 20 + 22 + 11.5 us an iteration ->
// 110 (5.8 TB/s) + 28 (4.6) + 14.6 (5.4), and the mixed solve 53.3 -> 49.4 ms.
#include <hip/hip_runtime.h>

#include "block_reduce.h"
#include "device_common.h"
#include "internal.h"
#include "kernels.h"
#include "sym_apply.h"

namespace lfric {
namespace {

// Kernels of iteration it carry phases 3 it, 3 it + 1, 3 it + 2.  The one that ends the solve stores its phase + 1
// in SolverState::stop (block 0, one store), so that its own later blocks still finish it and every later
// kernel returns.
__device__ inline bool stopped(const SolverState *st, int phase) {
  const int s = st->stop;
  return s != 0 && s - 1 < phase;
}

constexpr int kUnitThreads = 512, kGatherThreads = 1024, kGatherBlocks = 512, kStepBlocks = 2048;

// phase 1 of the apply on p, and the block's partial of p . A p: the sum over units of p at the unit's 4 dofs
// times the unit's outputs is the sum over dofs of p times A p, so alpha is known before the outputs are
// gathered.  Products and sums in FP64.  A block leaves one partial (stored by the logical block, so the order of
// the sum does not depend on the XCD window); blocks of 512 keep them few enough for the next kernel's blocks
// to add all of them.
template <typename T>
__global__ __launch_bounds__(kUnitThreads) void k_cg_sym_units(const T *__restrict__ sym, size_t gss,
                                                               const T *__restrict__ p,
                                                               const int4 *__restrict__ cellcol, T *__restrict__ z,
                                                               int ncells, int nl, SolverState *st, int phase,
                                                               int xwin, double *__restrict__ partials) {
  if (stopped(st, phase)) return;
  // a solve that the initial residual ended: nothing after this kernel runs
  if (phase == 0 && blockIdx.x == 0 && threadIdx.x == 0 && st->done) st->stop = 1;
  const int lb = xcd_block(blockIdx.x, gridDim.x, xwin);
  int k, m;
  T x0[4], out[4];
  double d[1] = {0.0};
  if (sym_unit<T>(sym, gss, p, cellcol, ncells, nl, static_cast<long long>(lb) * kUnitThreads + threadIdx.x, k, m, x0,
                  out)) {
    T *zp = z + static_cast<size_t>(k) * 4 * (nl + 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      zp[static_cast<size_t>(i) * (nl + 1) + m] = out[i];
      d[0] += to_d(x0[i]) * to_d(out[i]);
    }
  }
  double tot[1];
  block_sum_nt<kUnitThreads, 1>(d, tot);
  if (threadIdx.x == 0) partials[lb] = tot[0];
}

// phase 2 with the residual's update: (A p) at each point (the units' outputs in colour order, as
// k_sym_gather), r -= alpha A p, z = r / diag and the block's partials of r . r and r . z.  A p is neither
// written nor read back, and p is read by the next kernel alone.
template <typename T>
__global__ __launch_bounds__(kGatherThreads) void k_cg_sym_gather(const T *__restrict__ u, T *__restrict__ r,
                                                                  T *__restrict__ z, const T *__restrict__ diag,
                                                                  const int2 *__restrict__ cols,
                                                                  const int4 *__restrict__ zu, int ncols, int nl,
                                                                  SolverState *st, int phase, int par,
                                                                  const double *__restrict__ pzp, int npz,
                                                                  double *__restrict__ partials) {
  if (stopped(st, phase)) return;
  double tp[1];
  sum_partials<kGatherThreads, 1>(pzp, npz, tp);
  const double pz = tp[0], alpha = st->rzb[par] / pz;  // alpha = <r,z> / <p,A.p>
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (lead) st->pz = pz;
  if (pz != pz || pz == 0.0) {
    if (lead) {
      st->status = pz != pz ? LFRIC_NAN : LFRIC_BREAKDOWN;
      st->done = 1;
      st->stop = phase + 1;
    }
    return;
  }
  if (lead) st->alpha = alpha;
  const T ma = static_cast<T>(-alpha);
  const unsigned H = nl + 1, total = static_cast<unsigned>(ncols) * H, stride = gridDim.x * kGatherThreads;
  constexpr int kU = 4;
  double v[2] = {0.0, 0.0};
  for (unsigned t0 = blockIdx.x * kGatherThreads + threadIdx.x; t0 < total; t0 += kU * stride) {
    T q[kU][4], rv[kU], dv[kU];
    size_t dof[kU];
    int4 us[kU];
    bool ok[kU];
    unsigned m[kU];
#pragma unroll
    for (int e = 0; e < kU; ++e) {
      const unsigned t = t0 + e * stride;
      ok[e] = t < total && t >= t0;
      const unsigned col = ok[e] ? t / H : 0;
      m[e] = ok[e] ? t - col * H : 0;
      us[e] = zu[col];
      dof[e] = static_cast<size_t>(cols[col].x) + m[e];
    }
#pragma unroll
    for (int e = 0; e < kU; ++e) {
      const int w[4] = {us[e].x, us[e].y, us[e].z, us[e].w};
#pragma unroll
      for (int s = 0; s < 4; ++s) q[e][s] = ok[e] && w[s] >= 0 ? u[static_cast<size_t>(w[s]) * H + m[e]] : T(0);
      rv[e] = ok[e] ? r[dof[e]] : T(0);
      dv[e] = ok[e] && diag ? diag[dof[e]] : T(1);
    }
#pragma unroll
    for (int e = 0; e < kU; ++e) {
      if (!ok[e]) continue;
      const int w[4] = {us[e].x, us[e].y, us[e].z, us[e].w};
      T acc = q[e][0];
#pragma unroll
      for (int s = 1; s < 4; ++s)
        if (w[s] >= 0) acc = acc + q[e][s];
      const T ri = rv[e] + ma * acc;             // r%axpy(-alpha, A.p)
      const T zi = diag ? ri / dv[e] : ri;       // prec%apply(r,z)
      r[dof[e]] = ri;
      z[dof[e]] = zi;
      v[0] += to_d(ri) * to_d(ri);
      v[1] += to_d(ri) * to_d(zi);
    }
  }
  double tot[2];
  block_sum_nt<kGatherThreads, 2>(v, tot);
  if (threadIdx.x < 2) partials[2 * blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? tot[0] : tot[1];
}

// x += alpha p (here, where p is read anyway), the convergence test, and p = z + beta p unless the solve ends here (x is updated all the same)
template <typename T>
__global__ __launch_bounds__(kBlock) void k_cg_sym_step(T *__restrict__ x, T *__restrict__ p, const T *__restrict__ z,
                                                        long long n, SolverState *st, int phase, int par,
                                                        const double *__restrict__ partials, int np) {
  if (stopped(st, phase)) return;
  double tot[2];
  sum_partials<kBlock, 2>(partials, np, tot);
  const double rn = sqrt(tot[0]), beta = tot[1] / st->rzb[par];
  const bool nan = rn != rn;
  const bool conv = !nan && st->monitor && (rn / st->r_nrm0 <= st->r_tol || rn <= st->a_tol);
  const T a = static_cast<T>(st->alpha), b = static_cast<T>(beta);
  const long long stride = static_cast<long long>(gridDim.x) * kBlock;
  constexpr int kU = 4;
  for (long long i0 = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i0 < n; i0 += kU * stride) {
    T xv[kU], pv[kU], zv[kU];
#pragma unroll
    for (int e = 0; e < kU; ++e) {
      const long long i = i0 + e * stride;
      xv[e] = i < n ? x[i] : T(0);
      pv[e] = i < n ? p[i] : T(0);
      zv[e] = i < n ? z[i] : T(0);
    }
#pragma unroll
    for (int e = 0; e < kU; ++e) {
      const long long i = i0 + e * stride;
      if (i >= n) continue;
      x[i] = xv[e] + a * pv[e];                        // x%axpy(alpha,p)
      if (!nan && !conv) p[i] = b * pv[e] + zv[e];     // p%aypx(beta,z)
    }
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    const int iter = st->iter + 1;
    st->iter = iter;
    st->r_nrm = rn;
    bool end = nan || conv;
    if (nan) {
      st->status = LFRIC_NAN;
    } else {
      st->red0 = tot[0];
      st->red1 = tot[1];
      if (conv) {
        st->converged = 1;
      } else {
        st->beta = beta;
        st->rz = tot[1];
        st->rzb[par ^ 1] = tot[1];
        end = iter >= st->max_iter;
      }
    }
    if (end) {
      st->done = 1;
      st->stop = phase + 1;
    }
  }
}

template <typename T>
int iteration_t(const lfric_op *op, T *x, T *r, T *z, T *p, const T *diag, SolverState *st, long long it,
                double *unit_partials, double *partials) {
  const FunctionSpace &f = *op->to;
  const int phase = static_cast<int>(3 * it), par = static_cast<int>(it & 1);
  const int nu = cg_sym_partials(op), H = f.nlayers + 1;
  const int ng = grid_for(static_cast<long long>(f.gather_ncols) * H, kGatherThreads, kGatherBlocks);
  hipLaunchKernelGGL(k_cg_sym_units<T>, dim3(nu), dim3(kUnitThreads), 0, cur_stream(), static_cast<const T *>(op->sym),
                     op->gss, p, op->d_symcol, static_cast<T *>(op->symz), f.ncells, f.nlayers, st, phase, op->xwin,
                     unit_partials);
  hipLaunchKernelGGL(k_cg_sym_gather<T>, dim3(ng), dim3(kGatherThreads), 0, cur_stream(),
                     static_cast<const T *>(op->symz), r, z, diag, f.d_gcol, op->d_symzu, f.gather_ncols, f.nlayers, st,
                     phase + 1, par, unit_partials, nu, partials);
  hipLaunchKernelGGL(k_cg_sym_step<T>, dim3(grid_for(f.undf, 4 * kBlock, kStepBlocks)), dim3(kBlock), 0, cur_stream(), x,
                     p, z, static_cast<long long>(f.undf), st, phase + 2, par, partials, ng);
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

}  // namespace

int cg_sym_partials(const lfric_op *op) {
  return grid_for(s1_threads(static_cast<long long>(op->to->ncells) * (op->to->nlayers + 1)), kUnitThreads);
}

bool cg_sym_usable(const lfric_op *op) {
  return op->sym && op->to == op->from && op->to->ndf == 8 && op->sym_seg == 0 && op->d_symzu && op->d_symcol &&
         static_cast<long long>(op->to->gather_ncols) * (op->to->nlayers + 1) < (1LL << 31) &&
         cg_sym_partials(op) <= kSymUnitPartials;
}

int launch_cg_sym_iteration(const lfric_op *op, void *x, void *r, void *z, void *p, const void *diag, SolverState *st,
                            long long it) {
  double *up = ctx().d_partials + 4 * kRedBlocks, *gp = ctx().d_partials;
  return op->precision == LFRIC_R64
             ? iteration_t<double>(op, static_cast<double *>(x), static_cast<double *>(r), static_cast<double *>(z),
                                   static_cast<double *>(p), static_cast<const double *>(diag), st, it, up, gp)
             : iteration_t<float>(op, static_cast<float *>(x), static_cast<float *>(r), static_cast<float *>(z),
                                  static_cast<float *>(p), static_cast<const float *>(diag), st, it, up, gp);
}

}  // namespace lfric
