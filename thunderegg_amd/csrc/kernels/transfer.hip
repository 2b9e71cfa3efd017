// Inter-level transfer.  Restriction is computed per coarse cell (a gather, so
// every coarse cell is written exactly once and no atomics are needed);
// interpolation is computed per fine cell.
//  - LinearRestrictor (GMG/LinearRestrictor.h:101-155): coarse[(i+s)/2] += fine[i]/2^D
//    for children with an orthant on the parent, coarse[i] += fine[i] for copies;
//    MPIRestrictor::restrict zeroes the coarse vector with ghosts first (:73).  With
//    extrapolate_boundary_ghosts (:49-92, 138-155) the coarse ghost cells over a child's
//    exterior sides get (3 ghost - interior) / 2^D of the child's side cells, the corner of
//    the child's orthant, when it has no neighbour there, 3 ghost - interior of the child's
//    corner cell, and copies take the ghost cells too.
//  - DirectInterpolator (GMG/DirectInterpolator.h:60-91): fine[i] += coarse[(i+s)/2].
// Children of a coarse patch are visited in increasing fine local index and fine
// cells in x-fastest order, the order in which the reference accumulates them.
#include <algorithm>

#include "../te_internal.h"
#include "ghost2d.h"

namespace te {
namespace {

// the coarse ghost cell at (X, Y, Z) of patch p with extrapolate_boundary_ghosts: the sum
// over p's children in increasing local order, each term as the reference forms it
template <typename TI, int D>
__device__ TI extrapolated_ghost(const DevPatch* __restrict__ fdp, const int32_t* __restrict__ child,
                                 const int32_t* __restrict__ nchild, const int32_t* __restrict__ orth,
                                 const TI* __restrict__ fine, const Layout& L, int p, int c, int X, int Y, int Z,
                                 int rem)
{
  // 3 g - i rounded after the product, as the reference's expression (no fused multiply-add)
#pragma clang fp contract(off)
  const int cx[3] = { X, Y, Z };
  int outn = 0, bits = 0, axis = 0;
#pragma unroll
  for (int a = 0; a < D; a++) {
    if (cx[a] < 0 || cx[a] >= L.n[a]) {
      outn++;
      axis = a;
      if (cx[a] >= L.n[a]) bits |= 1 << a;
    }
  }
  TI acc = TI(0);
  const int nc = nchild[p];
  for (int k = 0; k < nc; k++) {
    const int f = child[p * 8 + k];
    const int o = orth[f];
    if (o < 0) {  // copyToParent: every cell, ghosts included
      acc += fine[f * L.ps + rem];
      continue;
    }
    if (outn == 1) {  // a side ghost: the child whose exterior side and half it lies over
      const int up = (bits >> axis) & 1;
      if (((o >> axis) & 1) != up) continue;
      int lo[2] = { 0, 0 }, hi[2] = { 0, 0 }, fa[2] = { 0, 0 }, nf = 0;
      bool mine = true;
#pragma unroll
      for (int b = 0; b < D; b++) {
        if (b == axis) continue;
        const int st = ((o >> b) & 1) ? L.n[b] : 0;
        int t0 = 2 * cx[b] - st, t1 = t0 + 1;  // the fine cells with (t + st) / 2 == cx[b]
        if (t0 < 0) t0 = 0;
        if (t1 > L.n[b] - 1) t1 = L.n[b] - 1;
        if (t0 > t1) mine = false;
        fa[nf] = b;
        lo[nf] = t0;
        hi[nf] = t1;
        nf++;
      }
      if (!mine) continue;
      const int ga = up ? L.n[axis] : -1, ia = up ? L.n[axis] - 1 : 0;
      // the side's slice, first free axis fastest
      for (int j = (D == 3 ? lo[1] : 0); j <= (D == 3 ? hi[1] : 0); j++)
        for (int i = lo[0]; i <= hi[0]; i++) {
          int xg[3] = { 0, 0, 0 }, xi[3] = { 0, 0, 0 };
          xg[axis] = ga;
          xi[axis] = ia;
          xg[fa[0]] = xi[fa[0]] = i;
          if (D == 3) xg[fa[1]] = xi[fa[1]] = j;
          const TI g = fine[lin(L, f, c, xg[0], xg[1], xg[2])], in = fine[lin(L, f, c, xi[0], xi[1], xi[2])];
          acc += (TI(3) * g - in) / TI(1 << D);
        }
    } else if (outn == D) {  // the corner of the child's orthant, when nothing lies across it
      if (o != bits || fdp[f].type[bits] >= 0) continue;
      int xg[3] = { 0, 0, 0 }, xi[3] = { 0, 0, 0 };
#pragma unroll
      for (int a = 0; a < D; a++) {
        xg[a] = ((bits >> a) & 1) ? L.n[a] : -1;
        xi[a] = ((bits >> a) & 1) ? L.n[a] - 1 : 0;
      }
      acc += TI(3) * fine[lin(L, f, c, xg[0], xg[1], xg[2])] - fine[lin(L, f, c, xi[0], xi[1], xi[2])];
    }
  }
  return acc;
}

template <typename TI, typename TO, int D, bool EX>
__global__ void __launch_bounds__(256) restrict_kernel(const int32_t* __restrict__ child,
                                                       const int32_t* __restrict__ nchild,
                                                       const int32_t* __restrict__ orth, const TI* __restrict__ fine,
                                                       TO* __restrict__ coarse, Layout L, int np_coarse,
                                                       const DevPatch* __restrict__ fdp)
{
  long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  long total = (long)np_coarse * L.ps;
  if (gid >= total) return;
  int idx = (int)gid;
  int p = idx / L.ps;
  int rem = idx - p * L.ps;
  int c = rem / L.cs;
  int q = rem - c * L.cs;
  int X, Y, Z = 0;
  if (D == 2) {
    Y = q / L.sx;
    X = q - Y * L.sx;
  } else {
    Z = q / L.sy;
    int r2 = q - Z * L.sy;
    Y = r2 / L.sx;
    X = r2 - Y * L.sx;
    Z -= 1;
  }
  X -= 1;
  Y -= 1;
  bool inter = X >= 0 && X < L.n[0] && Y >= 0 && Y < L.n[1] && (D == 2 || (Z >= 0 && Z < L.n[2]));
  if (!inter) {
    coarse[idx] = EX ? TO(extrapolated_ghost<TI, D>(fdp, child, nchild, orth, fine, L, p, c, X, Y, Z, rem)) : TO(0);
    return;
  }
  int nc = nchild[p];
  TI acc = TI(0);
  const TI w = TI(1.0 / (1 << D));
  for (int k = 0; k < nc; k++) {
    int f = child[p * 8 + k];
    int o = orth[f];
    if (o < 0) {  // copyToParent
      acc += fine[lin(L, f, c, X, Y, Z)];
      continue;
    }
    int s0 = (o & 1) ? L.n[0] : 0, s1 = (o & 2) ? L.n[1] : 0, s2 = (o & 4) ? L.n[2] : 0;
    int z0 = D == 3 ? 2 * Z - s2 : 0, z1 = D == 3 ? z0 + 1 : 0;
    for (int zz = z0; zz <= z1; zz++) {
      if (D == 3 && (zz < 0 || zz >= L.n[2])) continue;
      for (int yy = 2 * Y - s1; yy <= 2 * Y - s1 + 1; yy++) {
        if (yy < 0 || yy >= L.n[1]) continue;
        for (int xx = 2 * X - s0; xx <= 2 * X - s0 + 1; xx++) {
          if (xx < 0 || xx >= L.n[0]) continue;
          acc += fine[lin(L, f, c, xx, yy, zz)] * w;
        }
      }
    }
  }
  coarse[idx] = TO(acc);
}

// V values of type T from addresses that are multiples of T only: one access
template <typename T, int V, class Out>
__device__ __forceinline__ void load_at(const T* q, Out put)
{
  if (V == 2) {
    typedef T T2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    const T2 v = *reinterpret_cast<const T2*>(q);
    put(0, v[0]);
    put(1, v[1]);
  } else {
    put(0, *q);
  }
}
template <typename T, int V, class Get>
__device__ __forceinline__ void store_at(T* q, Get get)
{
  if (V == 2) {
    typedef T T2 __attribute__((ext_vector_type(2), aligned(sizeof(T))));
    T2 v;
    v[0] = get(0);
    v[1] = get(1);
    *reinterpret_cast<T2*>(q) = v;
  } else {
    *q = get(0);
  }
}

// One patch, or a run of its values, per workgroup (3D) or wavefront (2D) in both kernels below, so
// that the link's records are wave-uniform, and pairs of values along rows (even cells per side).
// Bound by memory on large levels.  One thread per cell with its place found by divisions -> these,
// us, FP64, restriction / interpolation: 4,096 fine patches of 16^3 81 / 90 -> 29 / 56; 65,536 of
// 16^2 79 / 76 -> 30 / 59; 64 of 64^2 4.7 / 4.2 -> 4.1 / 4.1 (16 / 9.5 with one wave a patch).

// Restriction where every coarse cell has one child over it (te_level_link::regular): a thread
// forms the two coarse cells of an aligned pair, each from 2^(D - 1) accesses of two fine cells,
// in the order of the general kernel above.
template <typename TI, typename TO, int D>
__global__ void __launch_bounds__(256) restrict_regular_kernel(const int32_t* __restrict__ child,
                                                               const int32_t* __restrict__ orth,
                                                               const TI* __restrict__ fine, TO* __restrict__ coarse,
                                                               Layout L, int np_coarse, FastDiv per_row, FastDiv rows,
                                                               int split)
{
  constexpr bool WAVE = D == 2;
  __shared__ int tabs[4][8], copies[4];  // the child of each octant (-1: none), or a copied child in entry 0
  const int b = xcd_item(blockIdx.x, gridDim.x);
  const int w = WAVE ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int unit = WAVE ? b * 4 + w : b, p = unit >> split;
  const bool live = p < np_coarse;
  const int t = WAVE ? threadIdx.x & 63 : threadIdx.x, nt = WAVE ? 64 : blockDim.x;
  // the link's records of the patch by one lane each (entries past the last child are -1)
  if (t < 8) {
    const int f = live ? child[p * 8 + t] : -1, o = f >= 0 ? orth[f] : -1;
    if (f >= 0 && o < 0) copies[w] = 1;  // the only child then (t = 0)
    else if (t == 0) copies[w] = 0;
    tabs[w][t] = -1;
    wave_sync();
    if (f >= 0) tabs[w][o < 0 ? 0 : o] = f;
  }
  __syncthreads();
  const bool copy = copies[w] != 0;
  if (!live) return;
  const int n0 = L.n[0], n1 = L.n[1], n2 = D == 3 ? L.n[2] : 1, h0 = n0 / 2, h1 = n1 / 2, h2 = n2 / 2;
  const int per = (n0 + 2) / 2;
  int first;
  const int last = split_range(per * (n1 + 2) * (D == 3 ? n2 + 2 : 1), split, unit & ((1 << split) - 1), &first);
  const TI wt = TI(1.0 / (1 << D));
  for (int c = 0; c < L.ncomp; c++) {
    for (int i = first + t; i < last; i += nt) {
      const int row = per_row(i);
      const int Z = D == 3 ? rows(row) - 1 : 0, Y = D == 3 ? row - (Z + 1) * (n1 + 2) - 1 : row - 1;
      const int X0 = 2 * (i - row * per) - 1;
      const bool in = Y >= 0 && Y < n1 && (D == 2 || (Z >= 0 && Z < n2));
      TI v[2][D == 3 ? 8 : 4];
      bool has[2];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int X = X0 + j;
        const int o = (X >= h0 ? 1 : 0) | (Y >= h1 ? 2 : 0) | (D == 3 && Z >= h2 ? 4 : 0);
        const int f = tabs[w][copy ? 0 : o];
        has[j] = in && X >= 0 && X < n0 && f >= 0;
        if (!has[j]) continue;
        if (copy) {
          v[j][0] = fine[lin(L, f, c, X, Y, Z)];
          continue;
        }
        const TI* q = fine + lin(L, f, c, 2 * X - (X >= h0 ? n0 : 0), 2 * Y - (Y >= h1 ? n1 : 0),
                                 D == 3 ? 2 * Z - (Z >= h2 ? n2 : 0) : 0);
#pragma unroll
        for (int r = 0; r < (D == 3 ? 4 : 2); r++)
          load_at<TI, 2>(q + (r & 1) * L.sx + (r >> 1) * L.sy, [&](int e, TI x) { v[j][2 * r + e] = x; });
      }
      TO res[2];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        TI acc = TI(0);
        if (has[j]) {
          if (copy) {
            acc += v[j][0];
          } else {
#pragma unroll
            for (int r = 0; r < (D == 3 ? 8 : 4); r++) acc += v[j][r] * wt;
          }
        }
        res[j] = TO(acc);
      }
      store_at<TO, 2>(coarse + p * L.ps + c * L.cs + 2 * i, [&](int j) { return res[j]; });
    }
  }
}

constexpr int kInterpItems = 2;  // pairs in flight a thread

// DirectInterpolator: fine += the coarse cell over it, over the interior rows of each fine patch
template <typename TC, typename TF, int D, int V>
__global__ void __launch_bounds__(256) interp_kernel(const int32_t* __restrict__ parent,
                                                     const int32_t* __restrict__ orth, const TC* __restrict__ coarse,
                                                     TF* __restrict__ fine, Layout L, FastDiv per_row, FastDiv rows,
                                                     int split)
{
  constexpr bool WAVE = D == 2;
  constexpr int U = kInterpItems;
  const int b = xcd_item(blockIdx.x, gridDim.x);
  const int unit = WAVE ? __builtin_amdgcn_readfirstlane(b * 4 + (threadIdx.x >> 6)) : b, p = unit >> split;
  if (p >= L.np) return;
  const int t = WAVE ? threadIdx.x & 63 : threadIdx.x, nt = WAVE ? 64 : blockDim.x;
  const int n0 = L.n[0], n1 = L.n[1], n2 = D == 3 ? L.n[2] : 1;
  const int per = V == 2 ? n0 / 2 + 1 : n0;
  int first;
  const int last = split_range(per * n1 * n2, split, unit & ((1 << split) - 1), &first);
  const int cp = parent[p], o = orth[p], sh = o < 0 ? 0 : 1;
  const int s0 = sh && (o & 1) ? n0 : 0, s1 = sh && (o & 2) ? n1 : 0, s2 = sh && (o & 4) ? n2 : 0;
  for (int c = 0; c < L.ncomp; c++) {
    const TC* cb = coarse + cp * L.ps + c * L.cs;
    TF* fb = fine + p * L.ps + c * L.cs;
    for (int i0 = first + t; i0 < last; i0 += U * nt) {
      TF fv[U][V];
      TC cv[U][V];
      int off[U], x0[U];
#pragma unroll
      for (int k = 0; k < U; k++) {
        const int i = i0 + k * nt;
        if (i >= last) continue;
        const int row = per_row(i), z = D == 3 ? rows(row) : 0, y = row - z * n1;
        x0[k] = V == 2 ? 2 * (i - row * per) - 1 : i - row * per;
        const int up = D == 3 ? L.sy : 0;
        off[k] = (z + 1) * up + (y + 1) * L.sx + x0[k] + 1;
        load_at<TF, V>(fb + off[k], [&](int j, TF v) { fv[k][j] = v; });
        const int crow = (((z + s2) >> sh) + 1) * up + (((y + s1) >> sh) + 1) * L.sx + 1;
#pragma unroll
        for (int j = 0; j < V; j++) {
          const int x = min(max(x0[k] + j, 0), n0 - 1);  // an end pair's ghost value is not written
          cv[k][j] = cb[crow + ((x + s0) >> sh)];
        }
      }
#pragma unroll
      for (int k = 0; k < U; k++) {
        const int i = i0 + k * nt;
        if (i >= last) continue;
#pragma unroll
        for (int j = 0; j < V; j++) fv[k][j] = TF(fv[k][j] + TF(cv[k][j]));
        if (V == 1 || (x0[k] >= 0 && x0[k] + 1 < n0)) store_at<TF, V>(fb + off[k], [&](int j) { return fv[k][j]; });
        else if (x0[k] < 0) fb[off[k] + 1] = fv[k][V - 1];
        else fb[off[k]] = fv[k][0];
      }
    }
  }
}

template <typename TI, typename TO>
void restrict_t(const te_level_link* l, const TI* fine, TO* coarse, int ncomp, bool ex, hipStream_t s)
{
  const te_domain* c = l->coarse;
  Layout L = make_layout(c->dim, c->ns, ncomp, l->fine->np);
  long total = (long)c->np * L.ps;
  if (total == 0) return;
  if (!ex && l->regular) {
    const int per = (L.n[0] + 2) / 2, rows = L.n[1] + 2;
    const int items = per * rows * (c->dim == 3 ? L.n[2] + 2 : 1);
    const int block = c->dim == 2 ? 256 : std::min(256, (items + 63) / 64 * 64), unit = c->dim == 2 ? 64 : block;
    const int split = patch_split(c->np, items, unit, unit / 64, items), units = c->np << split;
    if (c->dim == 2)
      hipLaunchKernelGGL((restrict_regular_kernel<TI, TO, 2>), dim3(xcd_grid((units + 3) / 4)), dim3(block), 0, s,
                         l->d_child, l->d_orth, fine, coarse, L, c->np, FastDiv(per), FastDiv(rows), split);
    else
      hipLaunchKernelGGL((restrict_regular_kernel<TI, TO, 3>), dim3(xcd_grid(units)), dim3(block), 0, s, l->d_child,
                         l->d_orth, fine, coarse, L, c->np, FastDiv(per), FastDiv(rows), split);
    return;
  }
  const int B = 256;
  int grid = (int)((total + B - 1) / B);
#define TE_RK(D_, EX_)                                                                                             \
  hipLaunchKernelGGL((restrict_kernel<TI, TO, D_, EX_>), dim3(grid), dim3(B), 0, s, l->d_child, l->d_nchild,        \
                     l->d_orth, fine, coarse, L, c->np, l->fine->d_patches)
  if (c->dim == 2) {
    if (ex) TE_RK(2, true);
    else TE_RK(2, false);
  } else {
    if (ex) TE_RK(3, true);
    else TE_RK(3, false);
  }
#undef TE_RK
}

template <typename TC, typename TF>
void interp_t(const te_level_link* l, const TC* coarse, TF* fine, int ncomp, hipStream_t s)
{
  const te_domain* f = l->fine;
  if (f->np == 0) return;
  Layout L = make_layout(f->dim, f->ns, ncomp, f->np);
  const int V = L.n[0] % 2 == 0 ? 2 : 1, per = V == 2 ? L.n[0] / 2 + 1 : L.n[0];
  const int items = per * L.n[1] * (f->dim == 3 ? L.n[2] : 1);
  const int block = f->dim == 2 ? 256 : std::min(256, (items / kInterpItems + 63) / 64 * 64);
  const int unit = f->dim == 2 ? 64 : block;
  const int split = patch_split(f->np, items, unit * kInterpItems, unit / 64, items), units = f->np << split;
  const int grid = xcd_grid(f->dim == 2 ? (units + 3) / 4 : units);
#define TE_IP(D_, V_)                                                                                              \
  hipLaunchKernelGGL((interp_kernel<TC, TF, D_, V_>), dim3(grid), dim3(block), 0, s, l->d_parent, l->d_orth, coarse, \
                     fine, L, FastDiv(per), FastDiv(L.n[1]), split)
  if (f->dim == 2) {
    if (V == 2) TE_IP(2, 2);
    else TE_IP(2, 1);
  } else {
    if (V == 2) TE_IP(3, 2);
    else TE_IP(3, 1);
  }
#undef TE_IP
}

}  // namespace

int launch_restrict(const te_level_link* l, int dti, const void* fine, int dto, void* coarse, int ncomp,
                    hipStream_t s, bool extrapolate)
{
  const bool ex = extrapolate;
  if (dti == TE_F64 && dto == TE_F64) restrict_t<double, double>(l, (const double*)fine, (double*)coarse, ncomp, ex, s);
  else if (dti == TE_F32 && dto == TE_F32) restrict_t<float, float>(l, (const float*)fine, (float*)coarse, ncomp, ex, s);
  else if (dti == TE_F32 && dto == TE_F64) restrict_t<float, double>(l, (const float*)fine, (double*)coarse, ncomp, ex, s);
  else restrict_t<double, float>(l, (const double*)fine, (float*)coarse, ncomp, ex, s);
  TE_HIP(hipGetLastError());
  return TE_OK;
}

int launch_interpolate(const te_level_link* l, int dtc, const void* coarse, int dtf, void* fine, int ncomp,
                       hipStream_t s)
{
  if (dtc == TE_F64 && dtf == TE_F64) interp_t<double, double>(l, (const double*)coarse, (double*)fine, ncomp, s);
  else if (dtc == TE_F32 && dtf == TE_F32) interp_t<float, float>(l, (const float*)coarse, (float*)fine, ncomp, s);
  else if (dtc == TE_F64 && dtf == TE_F32) interp_t<double, float>(l, (const double*)coarse, (float*)fine, ncomp, s);
  else interp_t<float, double>(l, (const float*)coarse, (double*)fine, ncomp, s);
  TE_HIP(hipGetLastError());
  return TE_OK;
}

}  // namespace te
