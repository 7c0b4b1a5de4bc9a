// The table entry of a lowest-order W0 dof column, and one point of the apply from it.  The small conjugate
// gradient's apply (cg_w0.hip) reads the same entries and states the same gather chain with its loads of z and
// the old p placed for it; tests hold the two to the same bits.
#pragma once
#include <hip/hip_runtime.h>

#include "device_common.h"

namespace lfric {
namespace {

// Table entry of a dof column (W0Col in int4 units): the element slot bases of its cells in colour
// order, its base dof with the cell count and each cell's bottom row, and each cell's 4 bottom
// vertex columns (the top vertices lie one level up in the same columns).
struct W0Col {
  int4 ebase;   // of cell 0..3
  int4 head;    // base dof, cells, row of cell 0..3 (one byte each), 0
  int4 xcol[4];
};
static_assert(sizeof(W0Col) == 96, "W0Col is read as 6 int4");

// (A x)(column, level m), x given by xf(dof).  The roles of a W0 space put a cell's top vertex j+4 one level
// above its bottom vertex j, so its two rows' x are 4 columns at 3 levels, each loaded once.  COLOUR: each cell's
// bottom row of layer m and top row of layer m-1 are two chains from zero and their sum is added, as
// k_lma_colour does; else one chain runs through the cells, as in k_lma_gather.  cnt: the column's cells.
template <typename T, bool COLOUR, class F>
__device__ inline T w0_point(const T *__restrict__ A, size_t gs, const W0Col *__restrict__ tc, int4 head, int cnt, int m,
                             int nl, F &&xf) {
  constexpr int V = chunk_entries<T>(), NC = 8 / V;
  typedef T VecT __attribute__((ext_vector_type(V)));
  const int4 eb4 = tc->ebase;
  int4 xc[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) xc[k] = tc->xcol[k];
  const int eb[4] = {eb4.x, eb4.y, eb4.z, eb4.w};
  const bool has_m = m < nl, has_p = m > 0;
  T acc = T(0);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (k >= cnt) break;
    const int i = (head.z >> (8 * k)) & 255;
    const long long e = static_cast<long long>(eb[k]) + m;
    const T *Ae = A + static_cast<size_t>(e >> 6) * gs + static_cast<size_t>(e & 63) * V;
    const T *rt = Ae + static_cast<size_t>(i + 4) * NC * 64 * V, *rb = Ae + static_cast<size_t>(i) * NC * 64 * V;
    VecT top[NC], bot[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      top[c] = has_p ? *reinterpret_cast<const VecT *>(rt + static_cast<size_t>(c) * 64 * V) : VecT{};
      bot[c] = has_m ? *reinterpret_cast<const VecT *>(rb + static_cast<size_t>(c) * 64 * V) : VecT{};
    }
    const int b[4] = {xc[k].x, xc[k].y, xc[k].z, xc[k].w};
    T xl[3][4];  // x of the cell's 4 columns at levels m-1, m, m+1
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      xl[0][j] = has_p ? xf(b[j] + m - 1) : T(0);
      xl[1][j] = xf(b[j] + m);
      xl[2][j] = has_m ? xf(b[j] + m + 1) : T(0);
    }
    if constexpr (COLOUR) {
      T c = T(0), cp = T(0);
      if (has_m) {
#pragma unroll
        for (int j = 0; j < 8; ++j) c = fma(bot[j / V][j % V], j < 4 ? xl[1][j] : xl[2][j - 4], c);
      }
      if (has_p) {
#pragma unroll
        for (int j = 0; j < 8; ++j) cp = fma(top[j / V][j % V], j < 4 ? xl[0][j] : xl[1][j - 4], cp);
      }
      const T out = c + cp;
      acc = k == 0 ? out : acc + out;
    } else {
      if (has_p) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = fma(top[j / V][j % V], j < 4 ? xl[0][j] : xl[1][j - 4], acc);
      }
      if (has_m) {
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = fma(bot[j / V][j % V], j < 4 ? xl[1][j] : xl[2][j - 4], acc);
      }
    }
  }
  return acc;
}

}  // namespace
}  // namespace lfric
