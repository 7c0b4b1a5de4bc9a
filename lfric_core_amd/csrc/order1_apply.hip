// Colour-ordered apply of order-1 W0 operators over their element layout, split by rows.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "colour_apply.h"
#include "device_common.h"
#include "internal.h"
#include "kernels.h"

namespace lfric {
namespace {

// The 27 rows of an order-1 W0 element feed 18 outputs of a unit (cell position, level m): 9
// dofs with a top partner (the bottom face, the 4 bottom edges, the 4 bottom vertices), whose
// output is a row of layer m plus the partner's row of layer m-1, and 9 without (the volume, the 4
// side faces, the 4 vertical edges).
constexpr int kPairs27 = 9;
__device__ inline int pair27(int q) { return q == 0 ? 5 : q < 5 ? 6 + q : 14 + q; }
__device__ inline int partner27(int q) { return q == 0 ? 6 : q < 5 ? 14 + q : 18 + q; }
__device__ inline int single27(int q) { return q < 5 ? q : 6 + q; }

// Row r of a 27 x 27 element held in registers as the 16-byte chunks that cover it (14 in FP64; 7 or
// 8 in FP32, the row starting s entries into its first chunk).  All of them are requested before
// the first is used: left to itself the compiler waits for each chunk of an FP64 row in turn.
template <typename T>
struct Row27 {
  static constexpr int V = chunk_entries<T>(), NCH = (27 + 2 * (V - 1)) / V;
  typedef T VecT __attribute__((ext_vector_type(V)));
  VecT v[NCH];
  int s;
  __device__ inline void load(const T *__restrict__ Ae, int r) {
    const int p0 = r * 27;
    s = p0 % V;
    const T *Ar = Ae + static_cast<size_t>(p0 / V) * 64 * V;
#pragma unroll
    for (int c = 0; c < NCH; ++c)
      if (c * V < 27 || c * V < 27 + s) v[c] = *reinterpret_cast<const VecT *>(Ar + static_cast<size_t>(c) * 64 * V);
  }
  template <int S, class F>
  __device__ inline void entries_s(F &&f) const {
#pragma unroll
    for (int j = 0; j < 27; ++j) f(j, v[(j + S) / V][(j + S) % V]);
  }
  template <class F>
  __device__ inline void entries(F &&f) const {  // f(j, a_rj), j in order; s is the same in every lane
    if constexpr (V == 2) {
      if (s)
        entries_s<1>(f);
      else
        entries_s<0>(f);
    } else {
      switch (s) {
        case 0: entries_s<0>(f); break;
        case 1: entries_s<1>(f); break;
        case 2: entries_s<2>(f); break;
        default: entries_s<3>(f); break;
      }
    }
  }
};

// One colour's pass with a unit's 27 rows over G threads: thread g takes 9/G of the outputs with a
// partner and 9/G of those without, so every thread has as many rows.  Each row is one fma chain
// in df2 order from zero and an output is c + cp, as in the one-thread-per-unit kernels
// (k_lma_colour, colour_unit_mrhs): the results are theirs bit for bit.
//   Bound: the element matrices from HBM.  With one thread per unit a colour of a C24x30 mesh is 420
// wavefronts on 1024 SIMDs, each with 5.8 KB to read in turn.  FP64, C24x30, one right-hand side:
// 712 us -> 146 us (4.2 TB/s of matrix, y and x); C32x70 892 -> 554 us (4.6 TB/s).  FP32: 180 -> 86 us;
// C48x70 639 -> 631 us; 8 right-hand sides there 2763 -> 1568 us.
//   Blocks: 8 consecutive unit blocks for g = 0, then the same 8 for g = 1, ...; workgroups go to the 8
// XCDs in turn, so the threads of one unit share an L2 and its x and row-boundary chunks.
template <typename T, int NR, int G>
__global__ __launch_bounds__(kBlock) void k_lma_colour_rows27(const T *__restrict__ A, size_t gs,
                                                              const int *__restrict__ ebase, const T *__restrict__ x,
                                                              T *__restrict__ y, const int *__restrict__ map1,
                                                              const int *__restrict__ map2,
                                                              const uint32_t *__restrict__ first, int pos0, int npos,
                                                              int nl, const int *__restrict__ skip, int nub) {
  typedef typename RVec<T, NR>::type VR;
  constexpr int V = chunk_entries<T>();
  constexpr int Q = kPairs27 / G;                     // pairs, and singles, of this thread
  constexpr bool kHold = sizeof(T) * 27 * NR <= 512;  // a level's x in registers
  if (skip && *skip) return;
  const int w = blockIdx.x / (8 * G), rr = blockIdx.x - w * (8 * G);
  const int ub = w * 8 + (rr & 7), g = rr >> 3;
  const int H = nl + 1;
  const int t = ub * kBlock + threadIdx.x;
  if (ub >= nub || t >= npos * H) return;
  const int lp = t / H, m = t - lp * H, pos = pos0 + lp;
  const int *m1 = map1 + static_cast<size_t>(pos) * 27, *m2 = map2 + static_cast<size_t>(pos) * 27;
  const uint32_t ft = first[pos];
  const bool has_m = m < nl, has_p = m > 0;
  const long long e = static_cast<long long>(ebase[pos]) + m;
  const T *Ae = A + static_cast<size_t>(e >> 6) * gs + static_cast<size_t>(e & 63) * V;
  int b[27];
#pragma unroll
  for (int j = 0; j < 27; ++j) b[j] = m2[j];
  VR X[kHold ? 27 : 1];
  auto xat = [&](int j, int lev) { return *reinterpret_cast<const VR *>(x + (static_cast<size_t>(b[j]) + lev) * NR); };
  auto hold = [&](int lev) {
    if constexpr (kHold) {
#pragma unroll
      for (int j = 0; j < 27; ++j) X[j] = xat(j, lev);
    }
  };
  auto chain = [&](int r, int lev) {
    Row27<T> row;
    row.load(Ae, r);
    __builtin_amdgcn_sched_barrier(0);
    VR c = {};
    row.entries([&](int j, T a) {
      const VR xv = kHold ? X[kHold ? j : 0] : xat(j, lev);
#pragma unroll
      for (int k = 0; k < NR; ++k) c[k] = fma(a, xv[k], c[k]);
    });
    return c;
  };
  auto put = [&](int i, const VR &v) {
    VR *yd = reinterpret_cast<VR *>(y + (static_cast<size_t>(m1[i]) + m) * NR);
    if ((ft >> i) & 1u)
      *yd = v;
    else
      *yd = *yd + v;
  };
  VR c[Q], cp[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) c[q] = cp[q] = VR{};
  if (has_m) {
    hold(m);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int is = single27(g * Q + q);
      c[q] = chain(pair27(g * Q + q), m);
      put(is, chain(is, m));
    }
  }
  if (has_p) {
    hold(m - 1);
#pragma unroll
    for (int q = 0; q < Q; ++q) cp[q] = chain(partner27(g * Q + q), m - 1);
  }
#pragma unroll
  for (int q = 0; q < Q; ++q) put(pair27(g * Q + q), c[q] + cp[q]);
}

template <typename T, int NR, int G>
void launch_g(const lfric_op *op, const T *x, T *y, const int *skip) {
  const FunctionSpace &to = *op->to, &from = *op->from;
  for (int c = 0; c < to.ncolours; ++c) {
    const int pos0 = to.colour_start[c], npos = to.colour_start[c + 1] - pos0;
    if (npos == 0) continue;
    const int nub = grid_for(static_cast<long long>(npos) * (to.nlayers + 1));
    hipLaunchKernelGGL((k_lma_colour_rows27<T, NR, G>), dim3((nub + 7) / 8 * 8 * G), dim3(kBlock), 0, cur_stream(),
                       static_cast<const T *>(op->d), op->gs, to.d_ebase, x, y, to.d_map, from.d_map, to.d_first, pos0,
                       npos, to.nlayers, skip, nub);
  }
}

// units of the operator's largest colour
long long colour_units(const lfric_op *op) {
  const FunctionSpace &to = *op->to;
  return static_cast<long long>(*std::max_element(to.npc.begin(), to.npc.end())) * (to.nlayers + 1);
}

// 9 threads a unit, except where the measured time of 3 was lower: 4 FP32 right-hand sides from 16384
// units a colour (C24x30 110 us against 130, C12x10 48 against 30), and 8 FP64 ones, whose 9-way
// kernel spills (C24x30 702 us against 952)
template <typename T>
int launch_t(const lfric_op *op, const T *x, T *y, int nrhs, const int *skip) {
  switch (nrhs) {
    case 1: launch_g<T, 1, 9>(op, x, y, skip); break;
    case 2: launch_g<T, 2, 9>(op, x, y, skip); break;
    case 4:
      if (sizeof(T) == 4 && colour_units(op) > 16384)
        launch_g<T, 4, 3>(op, x, y, skip);
      else
        launch_g<T, 4, 9>(op, x, y, skip);
      break;
    case 8: launch_g<T, 8, sizeof(T) == 8 ? 3 : 9>(op, x, y, skip); break;
    default: return fail(LFRIC_E_UNSUPPORTED, "lma_apply_mrhs: nrhs must be 1, 2, 4 or 8");
  }
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

}  // namespace

bool colour_rows27_faster(const lfric_op *op, int nrhs) {
  const int es = op->precision == LFRIC_R64 ? 8 : 4;
  return nrhs == 1 || es * 27 * nrhs > 512 || colour_units(op) <= 32768;
}

int launch_colour_rows27(const lfric_op *op, const void *x, void *y, int nrhs, const int *skip) {
  return op->precision == LFRIC_R64
             ? launch_t<double>(op, static_cast<const double *>(x), static_cast<double *>(y), nrhs, skip)
             : launch_t<float>(op, static_cast<const float *>(x), static_cast<float *>(y), nrhs, skip);
}

}  // namespace lfric
