// Gather apply of lowest-order W0 operators over their element layout, from one table entry per dof
// column.
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "device_common.h"
#include "internal.h"
#include "kernels.h"
#include "role_kind.h"
#include "w0_table.h"

namespace lfric {
namespace {

// Thread (column, level m): w0_point.
//   Bound: HBM on large meshes, the chain of dependent loads on small ones.  The column's cells, rows
// and vertex columns come with one round of loads where the lists take three (offsets, entries, map),
// and there is one launch where the colours take four that each re-read x and y.  FP64 / FP32,
// colour-ordered sums: C12x20 20.4 -> 4.9 / 18.4 -> 4.5 us, C48x70 126 -> 95 / 60 -> 43 us, C96x70
// 451 -> 360 / 231 -> 181 us (5.7 TB/s); gather sums: C12x20 6.9 -> 5.8 / 6.6 -> 5.0 us, C96x70
// 400 -> 359 / 191 -> 180 us.
template <typename T, bool COLOUR, bool DOT>
__global__ __launch_bounds__(kBlock) void k_w0_gather(const T *__restrict__ A, size_t gs,
                                                      const W0Col *__restrict__ tab, const T *__restrict__ x,
                                                      T *__restrict__ y, int ncols, int nl, double *partials,
                                                      const int *skip, int xwin) {
  if (skip && *skip) return;
  const int H = nl + 1;
  const int lb = xcd_block(blockIdx.x, gridDim.x, xwin);
  const unsigned t = static_cast<unsigned>(lb) * kBlock + threadIdx.x;
  const bool valid = t < static_cast<unsigned>(ncols) * static_cast<unsigned>(H);
  const unsigned col = valid ? t / H : 0;
  const int m = valid ? static_cast<int>(t - col * H) : 0;
  const W0Col *tc = tab + col;
  const int4 head = tc->head;
  const T acc = w0_point<T, COLOUR>(A, gs, tc, head, valid ? head.y : 0, m, nl, [&](int d) { return x[d]; });
  if (valid) y[static_cast<size_t>(head.x) + m] = acc;
  if constexpr (DOT) {
    double v[1] = {valid ? to_d(acc) * to_d(x[static_cast<size_t>(head.x) + m]) : 0.0};
    block_partials<1>(v, partials, lb);
  }
}

template <typename T>
int launch_t(const lfric_op *op, const T *x, T *y, bool colour, double *partials, const int *skip) {
  const FunctionSpace &f = *op->to;
  const int grid = grid_for(static_cast<long long>(f.w0tab_cols) * (f.nlayers + 1));
  const T *A = static_cast<const T *>(op->d);
  const W0Col *tab = static_cast<const W0Col *>(f.d_w0tab);
#define W0_LAUNCH(C, D)                                                                                          \
  hipLaunchKernelGGL((k_w0_gather<T, C, D>), dim3(grid), dim3(kBlock), 0, cur_stream(), A, op->gs, tab, x, y,    \
                     f.w0tab_cols, f.nlayers, partials, skip, op->xwin)
  if (colour)
    W0_LAUNCH(true, false);
  else if (partials)
    W0_LAUNCH(false, true);
  else
    W0_LAUNCH(false, false);
#undef W0_LAUNCH
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

}  // namespace

int build_w0_table(FunctionSpace &f) {
  static std::mutex mu;  // spaces are shared between the operators of several threads
  std::lock_guard<std::mutex> lock(mu);
  if (f.d_w0tab || f.ndf != 8 || role_kind(f) != RoleKind::W0K0) return LFRIC_OK;
  // columns in the order of their base dofs, each one's cells in colour order
  std::vector<int> col(static_cast<size_t>(f.undf), 0);  // cells of the column based there, then its number
  for (int c = 0; c < f.ncells; ++c)
    for (int i = 0; i < 4; ++i)
      if (++col[f.dofmap[static_cast<size_t>(c) * 8 + i] - 1] > 4) return LFRIC_OK;
  std::vector<W0Col> tab;
  for (int d = 0; d < f.undf; ++d) {
    if (!col[d]) continue;
    col[d] = static_cast<int>(tab.size());
    tab.push_back(W0Col{});
    tab.back().head.x = d;
  }
  if (static_cast<long long>(tab.size()) * (f.nlayers + 1) >= (1LL << 31)) return LFRIC_OK;
  for (int p = 0; p < f.ncells; ++p) {
    const int *row = &f.dofmap[static_cast<size_t>(f.cell_of_pos[p]) * 8];
    for (int i = 0; i < 4; ++i) {
      W0Col &t = tab[col[row[i] - 1]];
      const int k = t.head.y++;
      (&t.ebase.x)[k] = f.ebase[p];
      t.head.z |= i << (8 * k);
      t.xcol[k] = make_int4(row[0] - 1, row[1] - 1, row[2] - 1, row[3] - 1);
    }
  }
  const size_t bytes = sizeof(W0Col) * tab.size();
  void *d = nullptr;
  if (int rc = dmalloc(&d, bytes)) return rc;
  hipError_t e = hipMemcpy(d, tab.data(), bytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    dfree(d, bytes);
    return fail(LFRIC_E_HIP, hipGetErrorString(e));
  }
  f.w0tab_cols = static_cast<int>(tab.size());
  f.w0tab_bytes = bytes;
  f.d_w0tab = d;
  return LFRIC_OK;
}

int launch_w0_gather(const lfric_op *op, const void *x, void *y, bool colour, double *partials, const int *skip) {
  return op->precision == LFRIC_R64
             ? launch_t<double>(op, static_cast<const double *>(x), static_cast<double *>(y), colour, partials, skip)
             : launch_t<float>(op, static_cast<const float *>(x), static_cast<float *>(y), colour, partials, skip);
}

}  // namespace lfric
