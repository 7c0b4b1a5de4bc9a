// One unit of the symmetric-packed lowest-order W0 apply, shared by the plain apply and the conjugate
// gradient's.
//
// Cells take slots in cell-id order, so that the threads of a window of blocks work on neighbouring cells and
// share their x entries in one L2: unit t = k*(nl+1) + m is (k-th cell, level m).  Slot t of the copy holds
// the upper triangle of that cell's layer-m element (m < nl; the slot of m = nl is empty), entry q at
// (t/64)*gss + ((q/V)*64 + t%64)*V + q%V.  A unit's thread forms the bottom rows' chains c_i of its element (x at
// levels m, m+1) and the top rows' chains of the same element, which belong to unit m+1: the next lane takes
// them with one shuffle.  Every chain is the colour kernel's (same entries, same x, same order).
#pragma once
#include <hip/hip_runtime.h>

#include "device_common.h"

namespace lfric {
namespace {

__host__ __device__ constexpr int tri_index(int i, int j) { return i * 8 - i * (i - 1) / 2 + (j - i); }

// A wavefront takes 63 new units and repeats, in lane 0, the previous wavefront's last unit (whose outputs it
// does not write), so that every unit's lower neighbour is the previous lane; s1_threads gives the launch's
// thread count.
inline long long s1_threads(long long units) { return (units + 62) / 63 * 64; }

// Thread g's unit: its 4 outputs, its cell's slot k and level m, and x at level m; false where nothing is
// written.  cellcol[k]: the 0-based base dofs of the k-th cell's 4 bottom vertex columns.
template <typename T>
__device__ inline bool sym_unit(const T *__restrict__ sym, size_t gss, const T *__restrict__ x,
                                const int4 *__restrict__ cellcol, int ncells, int nl, long long g, int &k, int &m,
                                T (&x0)[4], T (&out)[4]) {
  constexpr int V = chunk_entries<T>(), NCH = 36 / V;
  typedef T VecT __attribute__((ext_vector_type(V)));
  const unsigned H = nl + 1, units = static_cast<unsigned>(ncells) * H;
  const int lane = threadIdx.x & 63;
  const long long ts = (g >> 6) * 63 + lane - 1;
  const bool valid = ts >= 0 && ts < static_cast<long long>(units);
  const unsigned t = valid ? static_cast<unsigned>(ts) : 0;
  k = static_cast<int>(t / H);
  m = static_cast<int>(t - k * H);
  const bool has_m = valid && m < nl, has_p = valid && m > 0;
  const T *St = sym + static_cast<size_t>(t >> 6) * gss + static_cast<size_t>(t & 63) * V;
  VecT tri[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c)
    tri[c] = has_m ? __builtin_nontemporal_load(reinterpret_cast<const VecT *>(St + static_cast<size_t>(c) * 64 * V))
                   : VecT{};
  int b[4] = {0, 0, 0, 0};
  if (valid) {
    const int4 bb = cellcol[k];
    b[0] = bb.x;
    b[1] = bb.y;
    b[2] = bb.z;
    b[3] = bb.w;
  }
  T x1[4];  // x at level m+1
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    x0[j] = valid ? x[b[j] + m] : T(0);
    x1[j] = has_m ? x[b[j] + m + 1] : T(0);
  }
  auto at = [&](int q) { return tri[q / V][q % V]; };
  T c[4], cn[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    T s = T(0), sn = T(0);
    if (has_m) {
#pragma unroll
      for (int j = 0; j < 8; ++j) s = fma(at(j >= i ? tri_index(i, j) : tri_index(j, i)), j < 4 ? x0[j] : x1[j - 4], s);
#pragma unroll
      for (int j = 0; j < 8; ++j)
        sn = fma(at(j >= i + 4 ? tri_index(i + 4, j) : tri_index(j, i + 4)), j < 4 ? x0[j] : x1[j - 4], sn);
    }
    c[i] = s;
    cn[i] = sn;
  }
  // the top rows of the layer-(m-1) element: the previous lane's unit (m-1 of the same cell)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const T cp = __shfl_up(cn[i], 1, 64);
    out[i] = c[i] + (has_p ? cp : T(0));
  }
  return valid && lane != 0;
}

}  // namespace
}  // namespace lfric
