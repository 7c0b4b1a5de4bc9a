// Conjugate gradient iteration over the element layout of a small lowest-order W0 operator, in two kernels.
#include <hip/hip_runtime.h>

#include "device_common.h"
#include "internal.h"
#include "kernels.h"
#include "w0_table.h"

namespace lfric {
namespace {

// the sum of nb partials of NV values, in one fixed order in every block (for at most 8 kBlock of them the order of the
// separate kernels' reduce_partials); 8 of a thread's are requested before any is added
template <int NV>
__device__ inline void sum_partials(const double *__restrict__ p, int nb, double (&tot)[NV]) {
  constexpr int kU = 8;
  double s[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) s[q] = 0.0;
  for (int b = threadIdx.x; b < nb; b += kU * kBlock) {
    double t[kU][NV];
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int q = 0; q < NV; ++q) t[u][q] = b + u * kBlock < nb ? p[static_cast<size_t>(b + u * kBlock) * NV + q] : 0.0;
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int q = 0; q < NV; ++q) s[q] += t[u][q];
  }
  block_sum<NV>(s, tot);
}

// ||r|| and r.z after the iterations so far (np partials of the update), and whether the solve ends with them
struct Test {
  double rn, rz;
  bool nan, conv;
};
__device__ inline Test test_of(const SolverState *st, const double *__restrict__ partials, int np) {
  double tot[2];
  sum_partials<2>(partials, np, tot);
  Test t;
  t.rn = sqrt(tot[0]);
  t.rz = tot[1];
  t.nan = t.rn != t.rn;
  t.conv = !t.nan && st->monitor && (t.rn / st->r_nrm0 <= st->r_tol || t.rn <= st->a_tol);
  return t;
}
// Whether the solve has ended before this kernel.  The update does not set `done` on a NaN or zero p.q but
// leaves that to the kernel after it, here: set there, `done` would be read by the later waves of blocks whose
// earlier waves started without it, and such a block would add an incomplete p.q and step x with it.
// (record sets `done` while blocks of the apply start; a block it divides writes p and q alone, which a solve that
// has ended does not read.)
__device__ inline bool ended(SolverState *st, bool lead) {
  if ((st->done | st->status) == 0) return false;  // one load of both
  if (lead) st->done = 1;
  return true;
}
// one thread: the state after `it` iterations
__device__ inline void record(SolverState *st, const Test &t, int it) {
  st->iter = it;
  st->r_nrm = t.rn;
  if (t.nan)
    st->status = LFRIC_NAN;
  else if (t.conv)
    st->converged = 1;
  if (t.nan || t.conv || it >= st->max_iter) st->done = 1;
}

// Iteration it: the previous iteration's convergence test and beta from its partials (each block adds them
// itself, in one order), p = z + beta p formed where the apply reads it, q = A p (k_lma_gather's chain) and the
// block's partial of p.q.  The thread of a point also stores its p, in the other of two buffers, since its
// neighbours still read the old one.  With it = 0 p is z.
//   Bound: latency.  Forming p here doubles the loads of x but leaves two launches of the three (gather, update,
// aypx: 6.6 + 5.7 + 6.5 us at C12x20, FP64); a point's element rows are requested before the partials are added.
// AHEAD: so are z and the old p, which takes 364 registers in FP64 (one wave on a SIMD).
template <typename T, bool AHEAD>
__global__ __launch_bounds__(kBlock) void k_cg_w0_apply(const T *__restrict__ A, size_t gs,
                                                        const W0Col *__restrict__ tab, const T *__restrict__ z,
                                                        const T *__restrict__ pold, T *__restrict__ pnew,
                                                        T *__restrict__ q, int ncols, int nl, SolverState *st, int it,
                                                        const double *__restrict__ partials, int np,
                                                        double *__restrict__ pq) {
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (ended(st, lead)) return;
  constexpr int V = chunk_entries<T>(), NC = 8 / V;
  typedef T VecT __attribute__((ext_vector_type(V)));
  const unsigned H = nl + 1, g = blockIdx.x * kBlock + threadIdx.x;
  const bool valid = g < static_cast<unsigned>(ncols) * H;
  const unsigned col = valid ? g / H : 0;
  const int m = valid ? static_cast<int>(g - col * H) : 0;
  const W0Col *tc = tab + col;
  const int4 eb4 = tc->ebase, head = tc->head;
  const int eb[4] = {eb4.x, eb4.y, eb4.z, eb4.w}, cnt = valid ? head.y : 0;
  const bool has_m = m < nl, has_p = m > 0;
  int4 xc[4];
  VecT top[4][NC], bot[4][NC];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    xc[k] = tc->xcol[k];
    const int i = (head.z >> (8 * k)) & 255;
    const long long e = static_cast<long long>(eb[k]) + m;
    const T *Ae = A + static_cast<size_t>(e >> 6) * gs + static_cast<size_t>(e & 63) * V;
    const T *rt = Ae + static_cast<size_t>(i + 4) * NC * 64 * V, *rb = Ae + static_cast<size_t>(i) * NC * 64 * V;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      top[k][c] = k < cnt && has_p ? *reinterpret_cast<const VecT *>(rt + static_cast<size_t>(c) * 64 * V) : VecT{};
      bot[k][c] = k < cnt && has_m ? *reinterpret_cast<const VecT *>(rb + static_cast<size_t>(c) * 64 * V) : VecT{};
    }
  }
  T zl[AHEAD ? 4 : 1][3][4], pl[AHEAD ? 4 : 1][3][4];
  if constexpr (AHEAD) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int c4[4] = {xc[k].x, xc[k].y, xc[k].z, xc[k].w};
#pragma unroll
      for (int l = 0; l < 3; ++l)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          // dof 0 where there is no such point
          const int d = k < cnt && (l > 0 || has_p) && (l < 2 || has_m) ? c4[j] + m + l - 1 : 0;
          zl[k][l][j] = z[d];
          pl[k][l][j] = pold[d];
        }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  T b = T(0);
  if (it > 0) {
    const Test t = test_of(st, partials, np);
    if (lead) record(st, t, it);
    if (t.nan || t.conv || it >= st->max_iter) return;
    const double beta = t.rz / st->rzb[(it - 1) & 1];
    if (lead) {
      st->beta = beta;
      st->rz = t.rz;
      st->rzb[it & 1] = t.rz;
    }
    b = static_cast<T>(beta);
  }
  auto pf = [&](int d) { return fma(b, pold[d], z[d]); };  // p%aypx(beta,z)
  T acc = T(0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k >= cnt) break;
    const int c4[4] = {xc[k].x, xc[k].y, xc[k].z, xc[k].w};
    T xl[3][4];  // p of the cell's 4 columns at levels m-1, m, m+1
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (AHEAD) {
#pragma unroll
        for (int l = 0; l < 3; ++l) xl[l][j] = fma(b, pl[k][l][j], zl[k][l][j]);
      } else {
        xl[0][j] = has_p ? pf(c4[j] + m - 1) : T(0);
        xl[1][j] = pf(c4[j] + m);
        xl[2][j] = has_m ? pf(c4[j] + m + 1) : T(0);
      }
    }
    if (has_p) {
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fma(top[k][j / V][j % V], j < 4 ? xl[0][j] : xl[1][j - 4], acc);
    }
    if (has_m) {
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fma(bot[k][j / V][j % V], j < 4 ? xl[1][j] : xl[2][j - 4], acc);
    }
  }
  double v[1] = {0.0};
  if (valid) {
    const T p = pf(head.x + m);
    pnew[head.x + m] = p;
    q[head.x + m] = acc;
    v[0] = to_d(acc) * to_d(p);
  }
  double tot[1];
  block_sum<1>(v, tot);
  if (threadIdx.x == 0) pq[blockIdx.x] = tot[0];
}

// alpha = rz / p.q, x += alpha p, r -= alpha q, z = r / diag and the block's partials of r.r and r.z
template <typename T>
__global__ __launch_bounds__(kBlock) void k_cg_w0_update(T *__restrict__ x, T *__restrict__ r, T *__restrict__ z,
                                                         const T *__restrict__ p, const T *__restrict__ q,
                                                         const T *__restrict__ diag, int n, SolverState *st, int it,
                                                         const double *__restrict__ pq, int npq,
                                                         double *__restrict__ partials) {
  if (st->done) return;
  const int i = blockIdx.x * kBlock + threadIdx.x;
  const bool ok = i < n;
  const T xv = ok ? x[i] : T(0), rv = ok ? r[i] : T(0), pv = ok ? p[i] : T(0), qv = ok ? q[i] : T(0);
  const T dv = ok && diag ? diag[i] : T(1);
  double tp[1];
  sum_partials<1>(pq, npq, tp);
  const double pz = tp[0], alpha = st->rzb[it & 1] / pz;  // alpha = <r,z> / <p,A.p>
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (lead) st->pz = pz;
  if (pz != pz || pz == 0.0) {
    if (lead) st->status = pz != pz ? LFRIC_NAN : LFRIC_BREAKDOWN;
    return;
  }
  if (lead) st->alpha = alpha;
  double v[2] = {0.0, 0.0};
  if (ok) {
    x[i] = xv + static_cast<T>(alpha) * pv;         // x%axpy(alpha,p)
    const T ri = rv + static_cast<T>(-alpha) * qv;  // r%axpy(-alpha,z)
    const T zi = diag ? ri / dv : ri;               // prec%apply(r,z)
    r[i] = ri;
    z[i] = zi;
    v[0] = to_d(ri) * to_d(ri);
    v[1] = to_d(ri) * to_d(zi);
  }
  double tot[2];
  block_sum<2>(v, tot);
  if (threadIdx.x < 2) partials[2 * blockIdx.x + threadIdx.x] = threadIdx.x == 0 ? tot[0] : tot[1];
}

// the test after `it` iterations, for the host's read (the next iteration's first kernel forms it again)
__global__ __launch_bounds__(kBlock) void k_cg_w0_test(SolverState *st, int it, const double *__restrict__ partials,
                                                       int np) {
  if (ended(st, threadIdx.x == 0)) return;
  const Test t = test_of(st, partials, np);
  if (threadIdx.x == 0) record(st, t, it);
}

constexpr int kUnits = 256;  // compute units

template <typename T>
int iteration_t(const lfric_op *op, void *const (&v)[6], const T *diag, SolverState *st, int it) {
  const FunctionSpace &f = *op->to;
  const int n = f.undf, nb = grid_for(n);
  T *x = static_cast<T *>(v[0]), *r = static_cast<T *>(v[1]), *z = static_cast<T *>(v[2]), *q = static_cast<T *>(v[3]);
  T *pold = static_cast<T *>(v[4 + (it & 1)]), *pnew = static_cast<T *>(v[4 + ((it + 1) & 1)]);
  double *part = ctx().d_partials, *pq = part + 2 * kCgW0Blocks;
  // loads ahead while all blocks are resident at once (a wave on a SIMD in FP64, two in FP32).  Solves without -> with,
  // FP64: C12x20 (72 blocks) 283 -> 257 us, C20x25 (244) 321 -> 288, C24x30 (419) 423 -> 438; FP32: C12x20 167 -> 149,
  // C24x36 (500) 216 -> 191
  auto apply = nb <= (sizeof(T) == 4 ? 2 : 1) * kUnits ? k_cg_w0_apply<T, true> : k_cg_w0_apply<T, false>;
  hipLaunchKernelGGL(apply, dim3(nb), dim3(kBlock), 0, cur_stream(), static_cast<const T *>(op->d), op->gs,
                     static_cast<const W0Col *>(f.d_w0tab), z, it > 0 ? pold : z, pnew, q, f.w0tab_cols, f.nlayers, st,
                     it, part, nb, pq);
  hipLaunchKernelGGL(k_cg_w0_update<T>, dim3(nb), dim3(kBlock), 0, cur_stream(), x, r, z, pnew, q, diag, n, st, it, pq,
                     nb, part);
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

}  // namespace

// Up to the blocks that are resident at once without loads ahead (two on a compute unit in FP64, three in FP32).  There
// the launches that it saves outweigh reading two vectors where the apply of three kernels reads one; the first
// block beyond takes a second round of the whole kernel.  16 iterations, three kernels -> two, FP64: 18186 dofs 367 ->
// 262 us, 107198 504 -> 475, 127946 (500 blocks) 530 -> 502, 138320 (541) 557 -> 610, 176358 617 -> 717; FP32: 18186
// 357 -> 253, 176358 468 -> 440, 192946 (754 blocks) 485 -> 452, 211770 (828) 512 -> 588, 374906 631 -> 704.
bool cg_w0_usable(const lfric_op *op) {
  const FunctionSpace &f = *op->to;
  return f.d_w0tab && op->to == op->from && !op->sym && f.undf == f.w0tab_cols * (f.nlayers + 1) &&
         grid_for(f.undf) <= (op->precision == LFRIC_R64 ? 2 : 3) * kUnits;
}

int launch_cg_w0_iteration(const lfric_op *op, void *const (&v)[6], const void *diag, SolverState *st, int it) {
  return op->precision == LFRIC_R64 ? iteration_t<double>(op, v, static_cast<const double *>(diag), st, it)
                                    : iteration_t<float>(op, v, static_cast<const float *>(diag), st, it);
}

int launch_cg_w0_test(const lfric_op *op, SolverState *st, int it) {
  hipLaunchKernelGGL(k_cg_w0_test, dim3(1), dim3(kBlock), 0, cur_stream(), st, it, ctx().d_partials,
                     grid_for(op->to->undf));
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

}  // namespace lfric
