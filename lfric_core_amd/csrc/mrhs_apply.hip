// The LMA apply of several right-hand sides: gather, colour-ordered and matrix-core forms and their
// dispatch.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "colour_apply.h"
#include "device_common.h"
#include "internal.h"
#include "kernels.h"
#include "mfma_apply.h"
#include "role_kind.h"

namespace lfric {
namespace {

// Several right-hand sides over the row-gathered copy: each RHS accumulates exactly as
// k_lma_gather_rows_w0 (and so as k_lma_gather_mrhs), x and y hold NR values per dof, RHS
// fastest.  The matrix streams once for all right-hand sides.
template <typename T, int NR>
__global__ __launch_bounds__(kBlock) void k_lma_gather_rows_w0_mrhs(const T *__restrict__ rows, size_t gsr,
                                                                    const T *__restrict__ x, T *__restrict__ y,
                                                                    const int *__restrict__ map2,
                                                                    const int2 *__restrict__ cols,
                                                                    const int *__restrict__ off,
                                                                    const int *__restrict__ ent, int ncols, int nl,
                                                                    int xwin) {
  rows_point_w0_mrhs<T, NR>(rows, gsr, x, y, map2, cols, off, ent, ncols, nl,
                            static_cast<long long>(xcd_block(blockIdx.x, gridDim.x, xwin)) * kBlock + threadIdx.x);
}

// ---- several right-hand sides ------------------------------------------------------------
// Multi-RHS vectors hold NR values per dof, RHS fastest: (dof, r) at dof*NR + r.  Every RHS
// is accumulated exactly as the one-RHS kernels do (same fma order), so column r of a
// multi-RHS apply equals the one-RHS apply of column r bit for bit.

// gather form, NR right-hand sides per thread (see k_lma_gather)
template <typename T, int N2, int NR, class R>
__global__ __launch_bounds__(kBlock) void k_lma_gather_mrhs(const T *__restrict__ A, size_t gs,
                                                            const int *__restrict__ ebase, const T *__restrict__ x,
                                                            T *__restrict__ y, const int *__restrict__ map2,
                                                            const int2 *__restrict__ cols, const int *__restrict__ off,
                                                            const int *__restrict__ ent, int ncols, int nl, R roles,
                                                            int xwin) {
  typedef typename RVec<T, NR>::type VR;
  const int H = nl + 1;
  const long long t = static_cast<long long>(xcd_block(blockIdx.x, gridDim.x, xwin)) * kBlock + threadIdx.x;
  if (t >= static_cast<long long>(ncols) * H) return;
  const int col = static_cast<int>(t / H);
  const int m = static_cast<int>(t - static_cast<long long>(col) * H);
  const int2 ci = cols[col];
  if (m == nl && !ci.y) return;
  const bool has_m = m < nl, has_p = m > 0;
  VR acc = {};
  const int q1 = off[col + 1];
  for (int q = off[col]; q < q1; ++q) {
    const int en = ent[q];
    const int pos = en >> 5, i = en & 31;
    const int pt = roles.partner(i);
    const long long e = static_cast<long long>(ebase[pos]) + m;
    int b[N2];
#pragma unroll
    for (int j = 0; j < N2; ++j) b[j] = map2[static_cast<size_t>(pos) * N2 + j];
    if (pt >= 0 && has_p) row_dot_mrhs<T, N2, NR>(A, gs, e, pt, x, b, m - 1, acc);
    if (has_m) row_dot_mrhs<T, N2, NR>(A, gs, e, i, x, b, m, acc);
  }
  *reinterpret_cast<VR *>(y + (static_cast<size_t>(ci.x) + m) * NR) = acc;
}

// colour-ordered scatter form, NR right-hand sides per thread, one (cell, level) unit per thread
// (see colour_apply.h)
template <typename T, int N1, int N2, int NR, class R>
__global__ __launch_bounds__(kBlock) void k_lma_colour_mrhs(const T *__restrict__ A, size_t gs,
                                                            const int *__restrict__ ebase, const T *__restrict__ x,
                                                            T *__restrict__ y, const int *__restrict__ map1,
                                                            const int *__restrict__ map2,
                                                            const uint32_t *__restrict__ first, int pos0, int npos,
                                                            int nl, R roles, int xwin) {
  const int H = nl + 1;
  const int t = xcd_block(blockIdx.x, gridDim.x, xwin) * kBlock + threadIdx.x;
  if (t >= npos * H) return;
  const int lp = t / H;
  const int m = t - lp * H;
  const int pos = pos0 + lp;
  colour_unit_mrhs<T, N1, N2, NR>(A, gs, static_cast<long long>(ebase[pos]) + m, map1 + static_cast<size_t>(pos) * N1,
                                  map2 + static_cast<size_t>(pos) * N2, first[pos], x, y, m, nl, roles);
}

// Colour-ordered multi-RHS apply of a lowest-order W0 FP32 operator on the matrix cores (see
// mfma_apply.h): 64 (cell, level) units per 256-thread block, 4 lanes per unit.
template <int NR>
__global__ __launch_bounds__(kBlock) void k_lma_colour_mrhs_mfma(const float *__restrict__ A, size_t gs,
                                                                 const int *__restrict__ ebase,
                                                                 const float *__restrict__ x, float *__restrict__ y,
                                                                 const int *__restrict__ map1,
                                                                 const int *__restrict__ map2,
                                                                 const uint32_t *__restrict__ first, int pos0,
                                                                 int npos, int nl, int xwin) {
  const int H = nl + 1;
  const long long u = static_cast<long long>(xcd_block(blockIdx.x, gridDim.x, xwin)) * (kBlock / 4) + (threadIdx.x >> 2);
  const bool valid = u < static_cast<long long>(npos) * H;
  const int lp = valid ? static_cast<int>(u / H) : 0;
  const int m = valid ? static_cast<int>(u - static_cast<long long>(lp) * H) : 0;
  const int pos = pos0 + lp;
  mfma_unit_w0<NR>(A, gs, static_cast<long long>(ebase[pos]) + m, map1 + static_cast<size_t>(pos) * 8,
                   map2 + static_cast<size_t>(pos) * 8, first[pos], x, y, m, nl, valid);
}

}  // namespace

#define LAUNCH(kernel, grid, ...) hipLaunchKernelGGL((kernel), dim3(grid), dim3(kBlock), 0, cur_stream(), __VA_ARGS__)
#define CHECK_LAUNCH() LF_HIP(hipGetLastError())

// ---- multi-RHS dispatch ---------------------------------------------------------------------
template <typename T, int N2, int NR, class R>
static int launch_gather_mrhs_r(const lfric_op *op, const T *x, T *y, R roles) {
  const FunctionSpace &to = *op->to, &from = *op->from;
  const int grid = grid_for(static_cast<long long>(to.gather_ncols) * (to.nlayers + 1));
  if constexpr (N2 == 27 && std::is_same<R, RolesW0K1>::value) {
    if (sym27_ready(op)) return launch_sym27_mrhs(op, x, y, NR);
  }
  if constexpr (N2 == 8 && std::is_same<R, RolesW0K0>::value) {
    if (op->rows) {  // the row-gathered copy (lowest-order W0, launch_build_rows)
      LAUNCH((k_lma_gather_rows_w0_mrhs<T, NR>), grid, static_cast<const T *>(op->rows), op->gsr, x, y, from.d_map,
             to.d_gcol, to.d_goff, to.d_gent, to.gather_ncols, to.nlayers, op->xwin);
      return LFRIC_OK;
    }
  }
  LAUNCH((k_lma_gather_mrhs<T, N2, NR, R>), grid, static_cast<const T *>(op->d), op->gs, to.d_ebase, x, y,
         from.d_map, to.d_gcol, to.d_goff, to.d_gent, to.gather_ncols, to.nlayers, roles, op->xwin);
  return LFRIC_OK;
}

template <typename T, int N1, int N2, int NR, class R>
static void launch_colour_mrhs_r(const lfric_op *op, const T *x, T *y, R roles) {
  const FunctionSpace &to = *op->to, &from = *op->from;
  for (int c = 0; c < to.ncolours; ++c) {
    const int pos0 = to.colour_start[c], npos = to.colour_start[c + 1] - pos0;
    if (npos == 0) continue;
    LAUNCH((k_lma_colour_mrhs<T, N1, N2, NR, R>), grid_for(static_cast<long long>(npos) * (to.nlayers + 1)),
           static_cast<const T *>(op->d), op->gs, to.d_ebase, x, y, to.d_map, from.d_map, to.d_first, pos0, npos,
           to.nlayers, roles, op->xwin);
  }
}

template <typename T, int N1, int N2, int NR>
static int launch_mrhs_n(int variant, RoleKind rk, const lfric_op *op, const T *x, T *y) {
  const Roles rr = roles_of(*op->to);
  const bool colour = variant == LFRIC_MRHS_COLOUR;
  // each role table belongs to one element size
  if constexpr (N1 == 8 && N2 == 8) {
    if (rk == RoleKind::W0K0) {
      if (!colour) return launch_gather_mrhs_r<T, N2, NR>(op, x, y, RolesW0K0{});
      launch_colour_mrhs_r<T, N1, N2, NR>(op, x, y, RolesW0K0{});
      return LFRIC_OK;
    }
  }
  if constexpr (N1 == 27 && N2 == 27) {
    if (rk == RoleKind::W0K1) {
      if (!colour) return launch_gather_mrhs_r<T, N2, NR>(op, x, y, RolesW0K1{});
      if (colour_rows27_faster(op, NR)) return launch_colour_rows27(op, x, y, NR, nullptr);
      launch_colour_mrhs_r<T, N1, N2, NR>(op, x, y, RolesW0K1{});
      return LFRIC_OK;
    }
  }
  if constexpr (N1 == 6 && N2 == 6) {
    if (rk == RoleKind::W2K0) {
      if (!colour) return launch_gather_mrhs_r<T, N2, NR>(op, x, y, RolesW2K0{});
      launch_colour_mrhs_r<T, N1, N2, NR>(op, x, y, RolesW2K0{});
      return LFRIC_OK;
    }
  }
  if (rk == RoleKind::None) {
    if (!colour) return launch_gather_mrhs_r<T, N2, NR>(op, x, y, RolesNone{});
    launch_colour_mrhs_r<T, N1, N2, NR>(op, x, y, RolesNone{});
    return LFRIC_OK;
  }
  if (!colour) return launch_gather_mrhs_r<T, N2, NR>(op, x, y, RolesRuntime{rr});
  launch_colour_mrhs_r<T, N1, N2, NR>(op, x, y, RolesRuntime{rr});
  return LFRIC_OK;
}

template <typename T, int NR>
static int mrhs_nr(int variant, const lfric_op *op, const T *x, T *y) {
  const RoleKind rk = role_kind(*op->to);
  const int n1 = op->to->ndf, n2 = op->from->ndf;
#define MRHS_CASE(A, B)                                      \
  if (n1 == A && n2 == B) {                                  \
    if (int rc = launch_mrhs_n<T, A, B, NR>(variant, rk, op, x, y)) return rc; \
    CHECK_LAUNCH();                                          \
    return LFRIC_OK;                                         \
  }
  MRHS_CASE(8, 8)
  MRHS_CASE(27, 27)
  MRHS_CASE(6, 6)
  MRHS_CASE(1, 1)
#undef MRHS_CASE
  return fail(LFRIC_E_UNSUPPORTED, "lma_apply_mrhs: unsupported (ndf_to, ndf_from)");
}

template <typename T>
static int mrhs_t(int variant, int nrhs, const lfric_op *op, const T *x, T *y) {
  if (variant == LFRIC_MRHS_GATHER)
    if (int rc = prepare_gather(*op->to)) return rc;
  switch (nrhs) {
    case 2: return mrhs_nr<T, 2>(variant, op, x, y);
    case 4: return mrhs_nr<T, 4>(variant, op, x, y);
    case 8: return mrhs_nr<T, 8>(variant, op, x, y);
  }
  return fail(LFRIC_E_UNSUPPORTED, "lma_apply_mrhs: nrhs must be 1, 2, 4 or 8");
}

template <int NR>
static void launch_mrhs_mfma_nr(const lfric_op *op, const float *x, float *y) {
  const FunctionSpace &to = *op->to, &from = *op->from;
  for (int c = 0; c < to.ncolours; ++c) {
    const int pos0 = to.colour_start[c], npos = to.colour_start[c + 1] - pos0;
    if (npos == 0) continue;
    LAUNCH((k_lma_colour_mrhs_mfma<NR>), grid_for(static_cast<long long>(npos) * (to.nlayers + 1), kBlock / 4),
           static_cast<const float *>(op->d), op->gs, to.d_ebase, x, y, to.d_map, from.d_map, to.d_first, pos0, npos,
           to.nlayers, op->xwin);
  }
}

bool mfma_apply_supported(const lfric_op *op) {
  return op->precision == LFRIC_R32 && op->to == op->from && op->to->ndf == 8 && role_kind(*op->to) == RoleKind::W0K0;
}

int batch_colour_form(const lfric_op *op) {
  if (mfma_apply_supported(op)) return 1;
  if (op->precision == LFRIC_R32 && op->to == op->from && op->to->ndf == 27 && role_kind(*op->to) == RoleKind::W0K1)
    return 2;
  return 0;
}

static int mrhs_mfma(const lfric_op *op, const void *xv, void *yv, int nrhs) {
  LF_CHECK(mfma_apply_supported(op), LFRIC_E_UNSUPPORTED,
           "lma_apply_mrhs: the MFMA variant is for square lowest-order W0 FP32 operators");
  const float *x = static_cast<const float *>(xv);
  float *y = static_cast<float *>(yv);
  switch (nrhs) {
    case 1: launch_mrhs_mfma_nr<1>(op, x, y); break;
    case 2: launch_mrhs_mfma_nr<2>(op, x, y); break;
    case 4: launch_mrhs_mfma_nr<4>(op, x, y); break;
    case 8: launch_mrhs_mfma_nr<8>(op, x, y); break;
    default: return fail(LFRIC_E_UNSUPPORTED, "lma_apply_mrhs: nrhs must be 1, 2, 4 or 8");
  }
  CHECK_LAUNCH();
  return LFRIC_OK;
}

int launch_lma_apply_mrhs(const lfric_op *op, const void *x, void *y, int nrhs, int variant) {
  if (variant == LFRIC_MRHS_AUTO) {
    // measured: an operator with a row-gathered copy is fastest in the gather form over the
    // copy; otherwise the colour-ordered form with register-staged x is the fastest from a few
    // hundred thousand cells up (C96x70 W0, 4 FP32 RHS: 0.310 ms vs gather 0.354); on small
    // meshes its one launch per colour leaves the GPU idle and the gather form wins
    // (order 1: from 8000 cells, with its rows split over threads; C12x10, 4 FP32 RHS 30 us against 55,
    // C6x20, 2 FP32 RHS 24 against 20; not 8 FP64 RHS, C24x30 702 us against 631)
    const long long nc3 = static_cast<long long>(op->to->ncells) * op->to->nlayers;
    const bool rows27 = role_kind(*op->to) == RoleKind::W0K1 && op->from->ndf == 27 &&
                        !(op->precision == LFRIC_R64 && nrhs == 8);
    variant = (nrhs > 1 && nc3 >= (rows27 ? 8000 : 200000) && !op->rows && !sym27_ready(op)) ? LFRIC_MRHS_COLOUR : LFRIC_MRHS_GATHER;
  }
  LF_CHECK(variant == LFRIC_MRHS_GATHER || variant == LFRIC_MRHS_COLOUR || variant == LFRIC_MRHS_MFMA, LFRIC_E_ARG,
           "unknown multi-RHS variant");
  if (variant == LFRIC_MRHS_MFMA) return mrhs_mfma(op, x, y, nrhs);
  if (nrhs == 1)
    return variant == LFRIC_MRHS_GATHER ? launch_lma_apply_gather(op, x, y) : launch_lma_apply(op, x, y, nullptr);
  if (op->precision == LFRIC_R64)
    return mrhs_t<double>(variant, nrhs, op, static_cast<const double *>(x), static_cast<double *>(y));
  return mrhs_t<float>(variant, nrhs, op, static_cast<const float *>(x), static_cast<float *>(y));
}

}  // namespace lfric
