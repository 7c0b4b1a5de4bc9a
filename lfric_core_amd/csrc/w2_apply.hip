// Lowest-order W2 operators over small tables of the mesh: the gather apply of 6 x 6 mass matrices from
// one table entry per dof column, and for W2 <-> W3 operators (1 x 6 elements), over each cell's side neighbours,
// the transpose apply in one launch and the Helmholtz composite in one kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "device_common.h"
#include "internal.h"
#include "kernels.h"
#include "role_kind.h"

namespace lfric {
namespace {

// Each cell position's neighbour across its side faces W, S, E, N as neighbour position * 8 + the face's
// number there, -1 where there is none.  False where the kernels below do not hold, as a caller's dofmap may
// have it: a side face of more than two cells, or a bottom-face column (dof 4) that other faces share.
bool w2_neighbours(const FunctionSpace &f, std::vector<int4> &tab) {
  struct Item {
    int base, pos, df;
  };
  std::vector<Item> items;
  items.reserve(static_cast<size_t>(f.ncells) * 5);
  for (int p = 0; p < f.ncells; ++p)
    for (int d = 0; d < 5; ++d) items.push_back({f.dofmap[static_cast<size_t>(f.cell_of_pos[p]) * 6 + d], p, d});
  std::sort(items.begin(), items.end(), [](const Item &a, const Item &b) { return a.base < b.base; });
  tab.assign(f.ncells, make_int4(-1, -1, -1, -1));
  for (size_t q = 1; q < items.size(); ++q) {
    const Item &a = items[q - 1], &b = items[q];
    if (a.base != b.base) continue;
    if (a.df == 4 || b.df == 4 || (q + 1 < items.size() && items[q + 1].base == b.base)) return false;
    (&tab[a.pos].x)[a.df] = b.pos * 8 + b.df;
    (&tab[b.pos].x)[b.df] = a.pos * 8 + a.df;
  }
  return true;
}

// Table entry of a W2 dof column, read as int4s: base dof; cells, row of cell 0 and 1 and whether the column is
// the bottom/top-face one (a byte each); the cells' element slot bases in colour order; and the cells' six
// dof columns.
struct W2Col {
  int base, info, ebase[2];
  int xcol[2][6];
};
static_assert(sizeof(W2Col) == 64, "W2Col is read as 4 int4");

// y = A x for a 6 x 6 operator: thread (column, level m).  COLOUR: the colour-ordered apply's sums (a chain per
// row from zero, then added), else one chain through the column's cells as in k_lma_gather; bit for bit in
// both.  bc: the ends of the bottom/top-face columns are written as 0 (enforce_bc).
//   Bound: HBM.  The table gives a thread its cells, rows and x columns in one round of loads where the lists
// take three, and both of a point's rows are in flight together.  C48x50 FP64, mass apply with boundary conditions:
// 65.1 us in two launches -> 50.9 us (59.9 with the second row requested after the first was summed).
template <typename T, bool COLOUR, bool DOT>
__global__ __launch_bounds__(kBlock) void k_w2_gather(const T *__restrict__ A, size_t gs,
                                                      const W2Col *__restrict__ tab, const T *__restrict__ x,
                                                      T *__restrict__ y, int ncols, int nl, double *partials,
                                                      const int *skip, int xwin, int bc) {
  if (skip && *skip) return;
  constexpr int V = chunk_entries<T>();
  typedef T VecT __attribute__((ext_vector_type(V)));
  const unsigned H = nl + 1;
  const int lb = xcd_block(blockIdx.x, gridDim.x, xwin);
  const unsigned t = static_cast<unsigned>(lb) * kBlock + threadIdx.x;
  bool valid = t < static_cast<unsigned>(ncols) * H;
  const unsigned col = valid ? t / H : 0;
  const int m = valid ? static_cast<int>(t - col * H) : 0;
  const int4 *tc = reinterpret_cast<const int4 *>(tab + col);
  const int4 h = tc[0], q1 = tc[1], q2 = tc[2], q3 = tc[3];
  const int b[2][6] = {{q1.x, q1.y, q1.z, q1.w, q2.x, q2.y}, {q2.z, q2.w, q3.x, q3.y, q3.z, q3.w}};
  const int eb[2] = {h.z, h.w}, cnt = h.y & 255;
  const bool tall = (h.y >> 24) != 0, has_m = m < nl, has_p = tall && m > 0;
  valid = valid && (has_m || tall);
  const bool zero = bc && tall && (m == 0 || !has_m);
  // the point's two rows: of a side face's two cells, or a bottom/top-face column's top face of layer m-1 and
  // bottom face of layer m.  Both are requested before either is used.
  const int row[2] = {tall ? 5 : (h.y >> 8) & 255, tall ? 4 : (h.y >> 16) & 255};
  const bool use[2] = {valid && !zero && (!tall || has_p), valid && !zero && (tall ? has_m : cnt > 1)};
  T a[2][6], xv[2][6];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const long long e = static_cast<long long>(tall ? eb[0] : eb[k]) + m;
    const int r = row[k], lev = k == 0 && tall ? m - 1 : m;
    const T *Ae = A + static_cast<size_t>(e >> 6) * gs + static_cast<size_t>(e & 63) * V;
    if constexpr (V == 2) {  // 3 whole chunks
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const VecT v = use[k] ? *reinterpret_cast<const VecT *>(Ae + static_cast<size_t>(3 * r + c) * 64 * V) : VecT{};
        a[k][2 * c] = v[0];
        a[k][2 * c + 1] = v[1];
      }
    } else {  // entries 6r .. 6r+5 in two chunks of 4, starting 0 (r even) or 2 (r odd) entries in
      const T *Ar = Ae + static_cast<size_t>((6 * r) >> 2) * 64 * V;
      const VecT u = use[k] ? *reinterpret_cast<const VecT *>(Ar) : VecT{};
      const VecT w = use[k] ? *reinterpret_cast<const VecT *>(Ar + 64 * V) : VecT{};
      const bool odd = r & 1;
      a[k][0] = odd ? u[2] : u[0];
      a[k][1] = odd ? u[3] : u[1];
      a[k][2] = odd ? w[0] : u[2];
      a[k][3] = odd ? w[1] : u[3];
      a[k][4] = odd ? w[2] : w[0];
      a[k][5] = odd ? w[3] : w[1];
    }
#pragma unroll
    for (int j = 0; j < 6; ++j) xv[k][j] = use[k] ? x[static_cast<size_t>(tall ? b[0][j] : b[k][j]) + lev] : T(0);
  }
  T acc = T(0);
  if constexpr (COLOUR) {
    T c[2] = {T(0), T(0)};
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (use[k]) {
#pragma unroll
        for (int j = 0; j < 6; ++j) c[k] = fma(a[k][j], xv[k][j], c[k]);
      }
    acc = use[1] || tall ? c[0] + c[1] : c[0];
  } else {
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (use[k]) {
#pragma unroll
        for (int j = 0; j < 6; ++j) acc = fma(a[k][j], xv[k][j], acc);
      }
  }
  if (valid) y[static_cast<size_t>(h.x) + m] = acc;
  if constexpr (DOT) {
    double v[1] = {valid ? to_d(acc) * to_d(x[static_cast<size_t>(h.x) + m]) : 0.0};
    block_partials<1>(v, partials, lb);
  }
}

// The six entries of a 1 x 6 element
template <typename T>
__device__ inline void element6(const T *__restrict__ A, size_t gs, long long e, T (&v)[6]) {
  constexpr int V = chunk_entries<T>(), NC = (6 + V - 1) / V;
  typedef T VecT __attribute__((ext_vector_type(V)));
  const T *Ae = A + static_cast<size_t>(e >> 6) * gs + static_cast<size_t>(e & 63) * V;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const VecT x = *reinterpret_cast<const VecT *>(Ae + static_cast<size_t>(c) * 64 * V);
#pragma unroll
    for (int q = 0; q < V; ++q)
      if (c * V + q < 6) v[c * V + q] = x[q];
  }
}

// y = A^T x.  Thread (cell position, level m) writes the W2 dofs its cell touches first: the
// bottom-face column's level m, and for each such side face its own term plus the neighbour's.  Each
// term is k_transpose_colour's chain and a face has at most two, so the sums are its bit for bit
// (first written, second added).
//   Bound: HBM (the elements once, about half of them again for the neighbours' entries).  The colours took
// four launches, each reading its elements again for one face of a chunk.  C48x50 FP64: 4 x 8.1 us -> 14.5 us.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_transpose_w2(const T *__restrict__ A, size_t gs,
                                                         const int *__restrict__ ebase, const int4 *__restrict__ nbr,
                                                         const T *__restrict__ x, T *__restrict__ y,
                                                         const int *__restrict__ map3, const int *__restrict__ map2,
                                                         const uint32_t *__restrict__ first, int npos, int nl) {
  const unsigned H = nl + 1, t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= static_cast<unsigned>(npos) * H) return;
  const int pos = static_cast<int>(t / H), m = static_cast<int>(t - pos * H);
  const int4 n4 = nbr[pos];
  const int nb[4] = {n4.x, n4.y, n4.z, n4.w};
  const int *mf = map2 + static_cast<size_t>(pos) * 6;
  const uint32_t ft = first[pos];
  const int b3 = map3[pos];
  const long long e = static_cast<long long>(ebase[pos]) + m;
  const bool has_m = m < nl;
  T a[6], xn[4], an[4];
  if (has_m) element6<T>(A, gs, e, a);
  const T x0 = has_m ? x[b3 + m] : T(0);
  const T x1 = m > 0 ? x[b3 + m - 1] : T(0), a5 = m > 0 ? A[aidx<T>(gs, e - 1, 5)] : T(0);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bool use = has_m && ((ft >> j) & 1u) && nb[j] >= 0;
    const int p = use ? nb[j] >> 3 : pos;
    an[j] = use ? A[aidx<T>(gs, static_cast<long long>(ebase[p]) + m, nb[j] & 7)] : T(0);
    xn[j] = use ? x[map3[p] + m] : T(0);
  }
  T acc = has_m ? fma(a[4], x0, T(0)) : T(0);
  if (m > 0) acc = fma(a5, x1, acc);
  y[static_cast<size_t>(mf[4]) + m] = acc;
  if (!has_m) return;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (!((ft >> j) & 1u)) continue;
    T s = fma(a[j], x0, T(0));
    if (nb[j] >= 0) s = s + fma(an[j], xn[j], T(0));
    y[static_cast<size_t>(mf[j]) + m] = s;
  }
}

// The composite's copy of D and M3, one array per entry in the thread order u = pos * nl + m: row j of D
// at [j * nu + u], M3 at [6 * nu + u], and the neighbour's entry of side face j at [(7 + j) * nu + u] (0 where
// there is none).  The element layout pads a 1 x 6 element to two or three 16-byte chunks and a 1 x 1 element
// to one; the copy is read coalesced and holds the values alone.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_build_helm(const T *__restrict__ D, size_t gsd, const T *__restrict__ M3,
                                                       size_t gs3, const int *__restrict__ ebase,
                                                       const int4 *__restrict__ nbr, int ncells, int nl,
                                                       T *__restrict__ out) {
  const int nu = ncells * nl;
  const int u = blockIdx.x * kBlock + threadIdx.x;
  if (u >= nu) return;
  const int pos = u / nl, m = u - pos * nl;
  const long long e = static_cast<long long>(ebase[pos]) + m;
  const int4 n4 = nbr[pos];
  const int nb[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
  for (int j = 0; j < 6; ++j) out[static_cast<size_t>(j) * nu + u] = D[aidx<T>(gsd, e, j)];
  out[static_cast<size_t>(6) * nu + u] = M3[aidx<T>(gs3, e, 0)];
#pragma unroll
  for (int j = 0; j < 4; ++j)
    out[static_cast<size_t>(7 + j) * nu + u] =
        nb[j] >= 0 ? D[aidx<T>(gsd, static_cast<long long>(ebase[nb[j] >> 3]) + m, nb[j] & 7)] : T(0);
}

// y = M3 x + tau D diag(M2)^-1 D^T x.  Thread (cell, layer) forms the gradient of its six faces itself: each
// face has this cell's term and at most one neighbour's, so what a cell's two neighbours share is formed
// twice and the W2 field between the two products is neither written nor read.  Every operation is that of
// the transpose, the division, the divergence, the M3 apply and the axpy, in their order (a face's two terms
// commute), so the result is the chain's bit for bit.
//   Bound: HBM, 13 values per cell and layer beside m2 (a face read by both its cells).  Against the transpose
// and the divergence as two kernels: C48x50 FP32 16.1 + 8.4 us -> 12.5 us, FP64 19.2 + 13.5 -> 20.1 us.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_helm(const T *__restrict__ dc, const int4 *__restrict__ nb3,
                                                 const T *__restrict__ m2, const int *__restrict__ map2,
                                                 const T *__restrict__ x, const int *__restrict__ map3,
                                                 T *__restrict__ y, int ncells, int nl, T tau) {
  const unsigned nu = static_cast<unsigned>(ncells) * nl, u = blockIdx.x * kBlock + threadIdx.x;
  if (u >= nu) return;
  const int pos = static_cast<int>(u / static_cast<unsigned>(nl)), m = static_cast<int>(u - pos * nl);
  const int4 n4 = nb3[pos];
  const int nb[4] = {n4.x, n4.y, n4.z, n4.w}, b3 = map3[pos];
  const int *b2 = map2 + static_cast<size_t>(pos) * 6;
  const bool up = m + 1 < nl, dn = m > 0;
  T D[6], Dn[4], mm[6], xn[4];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    D[j] = dc[static_cast<size_t>(j) * nu + u];
    mm[j] = m2[static_cast<size_t>(b2[j]) + m];
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    Dn[j] = dc[static_cast<size_t>(7 + j) * nu + u];
    xn[j] = nb[j] >= 0 ? x[nb[j] + m] : T(0);
  }
  const T M3 = dc[static_cast<size_t>(6) * nu + u];
  const T Dup = up ? dc[static_cast<size_t>(4) * nu + u + 1] : T(0), Ddn = dn ? dc[static_cast<size_t>(5) * nu + u - 1] : T(0);
  const T x0 = x[b3 + m], xup = up ? x[b3 + m + 1] : T(0), xdn = dn ? x[b3 + m - 1] : T(0);
  T acc = T(0);
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    T s;
    if (j == 4) {  // the bottom face: its bottom-face term of this layer, then the layer below's top face
      s = fma(D[4], x0, T(0));
      if (dn) s = fma(Ddn, xdn, s);
    } else if (j == 5) {  // the top face is the bottom face of the layer above
      s = up ? fma(Dup, xup, T(0)) : T(0);
      s = fma(D[5], x0, s);
    } else {
      s = fma(D[j], x0, T(0));
      if (nb[j] >= 0) s = s + fma(Dn[j], xn[j], T(0));
    }
    acc = fma(D[j], s / mm[j], acc);
  }
  const T y3 = fma(M3, x0, T(0));
  y[static_cast<size_t>(b3) + m] = y3 + tau * acc;
}

template <typename T>
int transpose_t(const lfric_op *op, const T *x, T *y) {
  const FunctionSpace &to = *op->to, &from = *op->from;
  hipLaunchKernelGGL(k_transpose_w2<T>, dim3(grid_for(static_cast<long long>(from.ncells) * (from.nlayers + 1))),
                     dim3(kBlock), 0, cur_stream(), static_cast<const T *>(op->d), op->gs, from.d_ebase,
                     static_cast<const int4 *>(from.d_w2tab), x, y, to.d_map, from.d_map, from.d_first, from.ncells,
                     from.nlayers);
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

template <typename T>
int gather_t(const lfric_op *op, const T *x, T *y, bool colour, double *partials, const int *skip, int bc) {
  const FunctionSpace &f = *op->to;
  const int grid = grid_for(static_cast<long long>(f.w2_ncols) * (f.nlayers + 1));
#define W2_LAUNCH(C, D)                                                                                         \
  hipLaunchKernelGGL((k_w2_gather<T, C, D>), dim3(grid), dim3(kBlock), 0, cur_stream(),                        \
                     static_cast<const T *>(op->d), op->gs, static_cast<const W2Col *>(f.d_w2col), x, y, f.w2_ncols, \
                     f.nlayers, partials, skip, op->xwin, bc)
  if (colour)
    W2_LAUNCH(true, false);
  else if (partials)
    W2_LAUNCH(false, true);
  else
    W2_LAUNCH(false, false);
#undef W2_LAUNCH
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

template <typename T>
int helm_t(const lfric_linop *L, const T *x, T *y) {
  const FunctionSpace &w2 = *L->D->from, &w3 = *L->D->to;
  const int grid = grid_for(static_cast<long long>(w3.ncells) * w3.nlayers);
  if (L->helm_dver != L->D->version || L->helm_mver != L->M3->version) {  // (re)build the copy
    if (!L->d_helm) {
      L->helm_bytes = 11 * sizeof(T) * static_cast<size_t>(w3.ncells) * w3.nlayers;
      if (int rc = dmalloc(&L->d_helm, L->helm_bytes)) return rc;
    }
    hipLaunchKernelGGL(k_build_helm<T>, dim3(grid), dim3(kBlock), 0, cur_stream(), static_cast<const T *>(L->D->d),
                       L->D->gs, static_cast<const T *>(L->M3->d), L->M3->gs, w3.d_ebase,
                       static_cast<const int4 *>(w2.d_w2tab), w3.ncells, w3.nlayers, static_cast<T *>(L->d_helm));
    LF_HIP(hipGetLastError());
    L->helm_dver = L->D->version;
    L->helm_mver = L->M3->version;
  }
  hipLaunchKernelGGL(k_helm<T>, dim3(grid), dim3(kBlock), 0, cur_stream(), static_cast<const T *>(L->d_helm),
                     static_cast<const int4 *>(L->d_hcol), static_cast<const T *>(L->m2->d), w2.d_map, x, w3.d_map, y,
                     w3.ncells, w3.nlayers, static_cast<T>(L->tau));
  LF_HIP(hipGetLastError());
  return LFRIC_OK;
}

}  // namespace

// columns in the order of their base dofs, each one's cells in colour order; nbr as w2_neighbours gives it
static std::vector<W2Col> w2_columns(const FunctionSpace &f, const std::vector<int4> &nbr) {
  std::vector<W2Col> tab;
  for (int p = 0; p < f.ncells; ++p) {
    const int *row = &f.dofmap[static_cast<size_t>(f.cell_of_pos[p]) * 6];
    for (int j = 0; j < 5; ++j) {
      const int nb = j < 4 ? (&nbr[p].x)[j] : -1;
      if (nb >= 0 && (nb >> 3) < p) continue;  // entered with its first cell
      W2Col c{};
      c.base = row[j] - 1;
      c.info = (nb >= 0 ? 2 : 1) | j << 8 | (nb >= 0 ? (nb & 7) << 16 : 0) | (j == 4 ? 1 << 24 : 0);
      const int cells[2] = {p, nb >= 0 ? nb >> 3 : p};
      for (int k = 0; k < 2; ++k) {
        c.ebase[k] = f.ebase[cells[k]];
        for (int q = 0; q < 6; ++q) c.xcol[k][q] = f.dofmap[static_cast<size_t>(f.cell_of_pos[cells[k]]) * 6 + q] - 1;
      }
      tab.push_back(c);
    }
  }
  std::sort(tab.begin(), tab.end(), [](const W2Col &a, const W2Col &b) { return a.base < b.base; });
  return tab;
}

static int to_device(const void *src, size_t bytes, void **out) {
  void *d = nullptr;
  if (int rc = dmalloc(&d, bytes)) return rc;
  hipError_t e = hipMemcpy(d, src, bytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    dfree(d, bytes);
    return fail(LFRIC_E_HIP, hipGetErrorString(e));
  }
  *out = d;
  return LFRIC_OK;
}

int build_w2_table(FunctionSpace &f, bool columns) {
  static std::mutex mu;  // spaces are shared between the operators of several threads
  std::lock_guard<std::mutex> lock(mu);
  if (f.ndf != 6 || role_kind(f) != RoleKind::W2K0 || f.ncells >= (1 << 28) ||
      static_cast<long long>(f.ncells) * 5 * (f.nlayers + 1) + kBlock >= (1LL << 31))
    return LFRIC_OK;
  if (!f.d_w2tab) {
    if (f.w2_nbr.empty() && !w2_neighbours(f, f.w2_nbr)) {
      f.w2_nbr.clear();
      return LFRIC_OK;
    }
    f.w2tab_bytes = sizeof(int4) * f.w2_nbr.size();
    if (int rc = to_device(f.w2_nbr.data(), f.w2tab_bytes, &f.d_w2tab)) return rc;
  }
  if (columns && !f.d_w2col) {
    const std::vector<W2Col> tab = w2_columns(f, f.w2_nbr);
    f.w2_ncols = static_cast<int>(tab.size());
    f.w2col_bytes = sizeof(W2Col) * tab.size();
    if (int rc = to_device(tab.data(), f.w2col_bytes, &f.d_w2col)) return rc;
  }
  return LFRIC_OK;
}

int launch_w2_gather(const lfric_op *op, const void *x, void *y, bool colour, double *partials, const int *skip,
                     int bc) {
  return op->precision == LFRIC_R64
             ? gather_t<double>(op, static_cast<const double *>(x), static_cast<double *>(y), colour, partials, skip, bc)
             : gather_t<float>(op, static_cast<const float *>(x), static_cast<float *>(y), colour, partials, skip, bc);
}

int launch_transpose_w2(const lfric_op *op, const void *x, void *y) {
  return op->precision == LFRIC_R64 ? transpose_t<double>(op, static_cast<const double *>(x), static_cast<double *>(y))
                                    : transpose_t<float>(op, static_cast<const float *>(x), static_cast<float *>(y));
}

int build_helm_table(const lfric_linop *L) {
  if (L->hcol_state) return LFRIC_OK;
  FunctionSpace &w2 = *L->D->from;
  const FunctionSpace &w3 = *L->D->to;
  if (int rc = build_w2_table(w2, false)) return rc;
  if (!w2.d_w2tab) {
    L->hcol_state = -1;
    return LFRIC_OK;
  }
  std::vector<int4> tab = w2.w2_nbr;
  for (int4 &t : tab)
    for (int j = 0; j < 4; ++j) {
      int &v = (&t.x)[j];
      if (v >= 0) v = w3.dofmap[w3.cell_of_pos[v >> 3]] - 1;
    }
  L->hcol_bytes = sizeof(int4) * tab.size();
  if (int rc = to_device(tab.data(), L->hcol_bytes, &L->d_hcol)) return rc;
  L->hcol_state = 1;
  return LFRIC_OK;
}

int launch_helm(const lfric_linop *L, const void *x, void *y) {
  return L->precision == LFRIC_R64 ? helm_t<double>(L, static_cast<const double *>(x), static_cast<double *>(y))
                                   : helm_t<float>(L, static_cast<const float *>(x), static_cast<float *>(y));
}

}  // namespace lfric
