// Star stencils: Poisson (Poisson/StarPatchOperator.h:75-101) and VarPoisson
// (VarPoisson/StarPatchOperator.h:61-109), 5-point in 2D and 7-point in 3D,
// optionally fused with the residual r = f - A u of Cycle::restrict
// (GMG/Cycle.h:57-65) and with the ghost fill before it (PatchOperator.h:126-143).  Ghost cells
// of the output are written 0 (f.setWithGhost(0), PatchOperator.h:136), interior cells get
// the stencil.  Physical-boundary ghosts of u are applied inline
// (enforceBoundaryConditions, :115-144): -u (Dirichlet) or +u (Neumann).
#include <algorithm>

#include "../te_internal.h"
#include "dft.h"
#include "ghost2d.h"
#include "ghost3d.h"

namespace te {
namespace {

constexpr int kNoFill = -1;

// One patch, or a run of its slices (3D) or rows (2D), per workgroup (3D) or wavefront (2D), so that
// its neighbour records and spacings are wave-uniform and a cell's place takes one or two
// multiply-shift divisions.  FILL (a te_filler_kind): the side ghosts next to the unit's cells
// first, written to u for the caller; they depend on interior cells only, so no unit waits for
// another's, and the stencil then reads them back from this workgroup's cache.  The stencil runs over the padded patch in groups of V = 2
// values (rows of even length start on them): one 16-byte (FP64) or 8-byte access per row
// neighbour and for the output, kStarItems groups in flight a thread.  Patches go to the XCDs in
// contiguous eighths (xcd_item), which takes 9 to 10 us off both cases below: the ghost phase
// reads most of the neighbours' lines.
// A u with ghosts, two launches of one thread per cell before / this one, vectors rotated so that
// the caches do not keep them: 4,096 patches of 16^3 in FP64 240 / 157 us (a copy of the padded
// vector 110), VarPoisson in FP32 209 / 133; 65,536 patches of 16^2 in FP64 (one set of vectors)
// 203 / 104, VarPoisson 248 / 143; few patches: 64 of 32^2 8.0 / 4.4, 4 of 1024^2 59 / 27.
// Marching each thread along z (three rows' loads together) was 3 to 4 us slower in 3D.
constexpr int kStarItems = 2;
// 3D faces (z) of more cells are filled by a launch of their own where a patch is split: one unit
// would fill such a face alone (64^3: 16 passes of its threads; 32^3: 4)
constexpr int kFusedFace = 1024;

template <typename T, typename TF, typename TO, int D, int OP, int FILL, int V>
__global__ void __launch_bounds__(256) star_kernel(const DevPatch* __restrict__ dp, const int4* __restrict__ ring, T* u,
                                                   const T* __restrict__ cf, const TF* __restrict__ fin,
                                                   TO* __restrict__ out, Layout L, int neumann, FastDiv per_row,
                                                   FastDiv rows, int split)
{
  constexpr bool WAVE = D == 2;
  const int b = xcd_item(blockIdx.x, gridDim.x);
  const int unit = WAVE ? __builtin_amdgcn_readfirstlane(b * 4 + (threadIdx.x >> 6)) : b;
  const int p = unit >> split, part = unit & ((1 << split) - 1);
  if (p >= L.np) return;
  const int t = WAVE ? threadIdx.x & 63 : threadIdx.x, nt = WAVE ? 64 : blockDim.x;
  const int n0 = L.n[0], n1 = L.n[1], n2 = D == 3 ? L.n[2] : 1;
  const int per = (n0 + 2) / V;
  const DevPatch& P = dp[p];
  int first, last;  // the unit's groups
  if (FILL == kNoFill) {
    last = split_range(per * (n1 + 2) * (D == 3 ? n2 + 2 : 1), split, part, &first);
  } else {
    // whole rows (2D) or slices (3D), lo <= r < hi of the interior ones
    const int nr = D == 3 ? n2 : n1, group = D == 3 ? per * (n1 + 2) : per;
    last = split_range(nr + 2, split, part, &first);
    const int lo = max(first, 1) - 1, hi = min(last, nr + 1) - 1;
    const bool low = lo == 0 && hi > lo, high = hi == nr && hi > lo;
    first *= group;
    last *= group;
    if (D == 2) {
      // ring cells: west and east of the rows, then south and north where they are the unit's
      const int m = max(hi - lo, 0), sides = 2 * m + (low ? n0 : 0) + (high ? n0 : 0);
      for (int i = t; i < sides; i += 64) {
        int g = i - 2 * m + 2 * n1 + (low ? 0 : n0);
        if (i < m) g = lo + i;
        else if (i < 2 * m) g = n1 + lo + i - m;
        int s, tt;
        const int4 r = ring[ring_index(p, g, n0, n1, &s, &tt)];
        if (r.x >= 0) fill_ring_cell<T, FILL == TE_BILINEAR ? TE_BILINEAR : TE_BIQUADRATIC>(r, s, tt, u, L, p);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");  // one wave wrote what it reads below
    } else {
      const int f0[6] = { lo * n1, lo * n1, lo * n0, lo * n0, 0, 0 };
      const int f1[6] = { hi * n1, hi * n1, hi * n0, hi * n0, low ? n0 * n1 : 0, high ? n0 * n1 : 0 };
      const int face = largest_face(L);
      if (face <= kSmallFace && split == 0) fill_faces3_small<T>(L, P, u, p, t, nt, face);
      else fill_faces3<T>(L, P, u, p, t, nt, f0, f1);
      __syncthreads();
    }
  }
  constexpr int SB = D == 2 ? 4 : 20;
  bool phys[2 * D];
  T ih2[D];
#pragma unroll
  for (int a = 0; a < D; a++) {
    ih2[a] = T(P.inv_h2[a]);
    phys[2 * a] = P.type[SB + 2 * a] < 0;
    phys[2 * a + 1] = P.type[SB + 2 * a + 1] < 0;
  }
  const T bs = (OP == 0 && neumann) ? T(1) : T(-1);
  for (int c = 0; c < L.ncomp; c++) {
    const int base = p * L.ps + c * L.cs, cbase = p * L.cs;
    for (int i0 = first + t; i0 < last; i0 += kStarItems * nt) {
      // a group and its row neighbours: below / above along y and z; single values left and right of it
      struct Cells {
        T m[V], yl[V], yu[V], zl[V], zu[V], lf, rt;
      };
      Cells U[kStarItems], C[OP == 1 ? kStarItems : 1];  // u, and the coefficients
      TF fv[kStarItems][V];
      int xx[kStarItems], yy[kStarItems], zz[kStarItems];
      bool in[kStarItems];
      auto load = [](auto& dst, const auto* src) {
        typedef typename std::remove_const<typename std::remove_reference<decltype(*src)>::type>::type E;
        if (V == 2) {
          typedef E E2 __attribute__((ext_vector_type(2), aligned(sizeof(E))));
          const E2 v = *reinterpret_cast<const E2*>(src);
          dst[0] = v[0];
          dst[V - 1] = v[1];
        } else {
          dst[0] = *src;
        }
      };
      auto cells = [&](Cells& d, const T* q) {
        load(d.m, q);
        load(d.yl, q - L.sx);
        load(d.yu, q + L.sx);
        if (D == 3) {
          load(d.zl, q - L.sy);
          load(d.zu, q + L.sy);
        }
        d.lf = q[-1];
        d.rt = q[V];
      };
#pragma unroll
      for (int k = 0; k < kStarItems; k++) {
        const int i = i0 + k * nt;
        const int row = per_row(i);
        zz[k] = D == 3 ? rows(row) : 1;
        yy[k] = D == 3 ? row - zz[k] * (n1 + 2) : row;
        xx[k] = V * (i - row * per) - 1;
        in[k] = i < last && yy[k] >= 1 && yy[k] <= n1 && zz[k] >= 1 && zz[k] <= n2;
        if (V == 1) in[k] = in[k] && xx[k] >= 0 && xx[k] < n0;
        if (!in[k]) continue;
        cells(U[k], u + base + V * i);
        if (OP == 1) cells(C[OP == 1 ? k : 0], cf + cbase + V * i);
        if (fin) load(fv[k], fin + base + V * i);
      }
#pragma unroll
      for (int k = 0; k < kStarItems; k++) {
        const int i = i0 + k * nt;
        if (i >= last) continue;
        TO res[V];
#pragma unroll
        for (int j = 0; j < V; j++) {
          res[j] = TO(0);
          const int x = xx[k] + j;
          if (!in[k] || x < 0 || x >= n0) continue;
          const Cells& u_ = U[k];
          const Cells& c_ = C[OP == 1 ? k : 0];
          const T mid = u_.m[j];
          const T bc = bs * mid;
          T acc = T(0);
          auto axis = [&](int a, T lower, T upper, T cl, T cu, int cells, int at0) {
            if (at0 == 0 && phys[2 * a]) lower = bc;
            if (at0 == cells - 1 && phys[2 * a + 1]) upper = bc;
            if (OP == 0) {
              acc += (upper - T(2) * mid + lower) * ih2[a];
            } else {
              const T cm = c_.m[j];
              acc += ((cu + cm) * (upper - mid) - (cl + cm) * (mid - lower)) * (ih2[a] * T(0.5));
            }
          };
          auto left = [&](const Cells& q) { return j == 0 ? q.lf : q.m[0]; };
          auto right = [&](const Cells& q) { return j == V - 1 ? q.rt : q.m[V - 1]; };
          axis(0, left(u_), right(u_), left(c_), right(c_), n0, x);
          axis(1, u_.yl[j], u_.yu[j], c_.yl[j], c_.yu[j], n1, yy[k] - 1);
          if (D == 3) axis(D - 1, u_.zl[j], u_.zu[j], c_.zl[j], c_.zu[j], n2, zz[k] - 1);
          res[j] = fin ? TO(T(fv[k][j]) - acc) : TO(acc);
        }
        TO* o = out + base + V * i;
        if (V == 2) {
          typedef TO O2 __attribute__((ext_vector_type(2)));
          O2 w;
          w[0] = res[0];
          w[1] = res[V - 1];
          *reinterpret_cast<O2*>(o) = w;
        } else {
          *o = res[0];
        }
      }
    }
  }
}

// The ghost fill and the stencil of 3D patches of N^3 cells through LDS, on levels of more patches
// than CUs: a workgroup stages its patch as it lies in memory (padded, 16-byte loads), puts the
// face ghosts into it (and into u for the caller) and each thread forms 16 bytes of the padded
// result at a time, its z and y neighbours by wide LDS reads.  star_kernel above reads each cell
// seven times through the vector L1 and its stencil waits for the ghosts' stores; here it waits
// for LDS only.  Bound by memory.  Operator / residual with the ghost fill, star_kernel -> this
// one, us, vectors rotated so that the caches do not keep them: 2,500 patches of 16^3 (refined
// octree, FP32) 60 / 75 -> 51 / 62 (a copy of the padded vector 25); 4,096 of 16^3 in FP32 91 / 111
// -> 79 / 91, VarPoisson in FP64 226 / 236 -> 213 / 224; 4,096 of 8^3 in FP32 23.7 / 23.8 -> 13.0 /
// 14.7, in FP64 33 / 41 -> 20 / 29; 512 of 8^3 6.9 -> 5.2.  Not for 16^3 Poisson in FP64 (157 / 178
// against 163 / 189: three workgroups of 46 KB a CU) and VarPoisson in FP32 (133 / 142 against 152 /
// 157: its coefficients are read cell by cell here).
template <typename T, typename TF, typename TO, int OP, int N>
__global__ void __launch_bounds__(N == 16 ? 256 : 64) star3_tile_kernel(const DevPatch* __restrict__ dp, T* u,
                                                                        const T* __restrict__ cf,
                                                                        const TF* __restrict__ fin,
                                                                        TO* __restrict__ out, Layout L, int neumann)
{
  constexpr int SX = N + 2, SY = SX * SX, PS = SX * SY, NT = N == 16 ? 256 : 64;
  constexpr int W = 16 / sizeof(T);  // values a group
  static_assert(PS % W == 0 && SY % W == 0 && N * N == NT, "whole groups; a cell of each face per thread");
  __shared__ __align__(16) T tile[PS];
  const int p = xcd_item(blockIdx.x, gridDim.x);
  if (p >= L.np) return;
  const DevPatch& P = dp[p];
  const int t = threadIdx.x, fi = t % N, fj = t / N;
  const T ih2[3] = { T(P.inv_h2[0]), T(P.inv_h2[1]), T(P.inv_h2[2]) };
  typedef T VecT __attribute__((ext_vector_type(W), aligned(sizeof(T))));
  typedef TF VecF __attribute__((ext_vector_type(W), aligned(sizeof(TF))));
  typedef TO VecO __attribute__((ext_vector_type(W), aligned(sizeof(TO))));
  // the component: a grid axis, since a loop over components keeps every face's and group's offsets
  // in registers (100 instead of 39 of them, FP32 16^3)
  const int c = blockIdx.y;
  T* uc = component(L, u, p, c);
  TO* oc = component(L, out, p, c);
  const TF* fc = fin ? component(L, fin, p, c) : nullptr;
  const int cbase = p * L.cs;
  T G[6];
#pragma unroll
  for (int s = 0; s < 6; s++) {
    if (P.type[20 + s] >= 0) {
      G[s] = face_ghost3<T>(L, P.type[20 + s], P.orth[20 + s], P.nbr[20 + s], u, p, c, s, fi, fj);
    } else {
      const T b = at(uc, side_cell3(L, 0, 0, s, 0, fi, fj));
      G[s] = (OP == 0 && neumann) ? b : -b;
    }
  }
  for (int k = t; k < PS / W; k += NT)
    *reinterpret_cast<VecT*>(tile + W * k) = *reinterpret_cast<const VecT*>(&at(uc, W * k));
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 6; s++) {
    tile[side_cell3(L, 0, 0, s, -1, fi, fj)] = G[s];
    if (P.type[20 + s] >= 0) at(uc, side_cell3(L, 0, 0, s, -1, fi, fj)) = G[s];
  }
  __syncthreads();
  for (int k = t; k < PS / W; k += NT) {
    VecO res;
    const int q0 = W * k;
#pragma unroll
    for (int j = 0; j < W; j++) res[j] = TO(0);
    if (q0 >= SY && q0 < PS - SY) {  // whole groups lie in or out of the ghost planes
      VecF fv;
      if (fin) fv = *reinterpret_cast<const VecF*>(&at(fc, q0));
#pragma unroll
      for (int j = 0; j < W; j++) {  // rows' ghosts too (every neighbour lies in the tile), set to zero below
        const int q = q0 + j, y = q / SX % SX, x = q % SX;
        const T mid = tile[q];
        T acc = T(0);
        const int st[3] = { 1, SX, SY };
#pragma unroll
        for (int a = 0; a < 3; a++) {
          const T lower = tile[q - st[a]], upper = tile[q + st[a]];
          if (OP == 0) {
            acc += (upper - T(2) * mid + lower) * ih2[a];
          } else {
            const int ci = cbase + q;
            const T cm = at(cf, ci), cl = at(cf, ci - st[a]), cu = at(cf, ci + st[a]);
            acc += ((cu + cm) * (upper - mid) - (cl + cm) * (mid - lower)) * (ih2[a] * T(0.5));
          }
        }
        const bool in = x >= 1 && x <= N && y >= 1 && y <= N;
        res[j] = in ? (fin ? TO(T(fv[j]) - acc) : TO(acc)) : TO(0);
      }
    }
    *reinterpret_cast<VecO*>(&at(oc, q0)) = res;
  }
}

template <typename T, typename TF, typename TO, int D, int OP>
int launch_one(const te_ghost_filler* g, T* u, const T* cf, const TF* fin, TO* out, int ncomp, int neumann, bool fill,
                hipStream_t s)
{
  const te_domain* d = g->d;
  Layout L = make_layout(d->dim, d->ns, ncomp, d->np);
  // star3_tile_kernel's levels: those that fill the CUs, of the patch sizes it is written for; 16^3
  // patches only where it is the faster one (its comment)
  if constexpr (D == 3) {
    const bool cube = L.n[1] == L.n[0] && L.n[2] == L.n[0];
    const bool tile = fill && cube && d->np > cu_count();
    if (tile && L.n[0] == 8) {
      hipLaunchKernelGGL((star3_tile_kernel<T, TF, TO, OP, 8>), dim3(xcd_grid(d->np), ncomp), dim3(64), 0, s,
                         d->d_patches, u, cf, fin, out, L, neumann);
      return TE_OK;
    }
    if constexpr ((OP == 0) == (sizeof(T) == 4)) {
      if (tile && L.n[0] == 16) {
        hipLaunchKernelGGL((star3_tile_kernel<T, TF, TO, OP, 16>), dim3(xcd_grid(d->np), ncomp), dim3(256), 0, s,
                           d->d_patches, u, cf, fin, out, L, neumann);
        return TE_OK;
      }
    }
  }
  const bool pairs = L.n[0] % 2 == 0 && (uintptr_t)u % (2 * sizeof(T)) == 0 && (uintptr_t)fin % (2 * sizeof(TF)) == 0 &&
                     (uintptr_t)out % (2 * sizeof(TO)) == 0;
  const int V = pairs ? 2 : 1, per = (L.n[0] + 2) / V;
  const int items = per * (L.n[1] + 2) * (D == 3 ? L.n[2] + 2 : 1);
  const int block = D == 2 ? 256 : std::min(256, (items / kStarItems + 63) / 64 * 64);
  // the unit: a wave in 2D, the workgroup in 3D
  const int threads = D == 2 ? 64 : block, pass = threads * kStarItems;
  // rows of two passes and more: a unit of a 16-waves-a-CU split is a few rows, walked for so long that
  // its neighbours' rows have left the L2 when it reads them again.  With 64 waves a CU 16 patches of
  // 1024^2 take 46 us instead of 80 (FP64, filled ghosts), 16 of 512^2 13.4 instead of 17.6; shorter
  // rows lose in FP32 (256 patches of 256^2 22.5 to 25.1)
  const int per_cu = D == 2 && per >= 2 * pass ? 64 : 16;
  int split = patch_split(d->np, items, pass, threads / 64, fill ? (D == 3 ? L.n[2] : L.n[1]) + 2 : items, per_cu);
  if (fill && D == 3 && split > 0 && L.n[0] * L.n[1] > kFusedFace) {
    int rc = launch_ghost_fill_faces(g, sizeof(T) == 8 ? TE_F64 : TE_F32, u, ncomp, s);
    if (rc) return rc;
    fill = false;
    split = patch_split(d->np, items, pass, threads / 64, items);
  }
  const int units = d->np << split, grid = xcd_grid(D == 2 ? (units + 3) / 4 : units);
#define TE_ST(F_, V_)                                                                                               \
  hipLaunchKernelGGL((star_kernel<T, TF, TO, D, OP, F_, V_>), dim3(grid), dim3(block), 0, s, d->d_patches,          \
                     (const int4*)d->d_ring, u, cf, fin, out, L, neumann, FastDiv(per), FastDiv(L.n[1] + 2), split)
#define TE_SF(F_)          \
  do {                     \
    if (V == 2) TE_ST(F_, 2); \
    else TE_ST(F_, 1);     \
  } while (0)
  if (!fill) TE_SF(kNoFill);
  else if (D == 3) TE_SF((D == 3 ? TE_TRILINEAR : kNoFill));
  else if (g->kind == TE_BILINEAR) TE_SF((D == 2 ? TE_BILINEAR : kNoFill));
  else TE_SF((D == 2 ? TE_BIQUADRATIC : kNoFill));
#undef TE_SF
#undef TE_ST
  return TE_OK;
}

template <typename T, typename TF, typename TO>
int launch_dim(const te_ghost_filler* g, int op_kind, T* u, const T* cf, const TF* fin, TO* out, int ncomp,
                int neumann, bool fill, hipStream_t s)
{
  if (g->d->dim == 2) {
    if (op_kind == 0) return launch_one<T, TF, TO, 2, 0>(g, u, cf, fin, out, ncomp, neumann, fill, s);
    return launch_one<T, TF, TO, 2, 1>(g, u, cf, fin, out, ncomp, neumann, fill, s);
  }
  if (op_kind == 0) return launch_one<T, TF, TO, 3, 0>(g, u, cf, fin, out, ncomp, neumann, fill, s);
  return launch_one<T, TF, TO, 3, 1>(g, u, cf, fin, out, ncomp, neumann, fill, s);
}

// Cycle::restrict (GMG/Cycle.h:57-65) of 3D patches of N^3 cells in one launch: a workgroup stages
// its patch in LDS as it lies in memory (padded, 16-byte loads), writes the face ghosts into it
// (face_ghost3; physical sides by the boundary condition), and each thread forms the coarse cells
// of a child cell block: eight residuals, averaged in restrict_kernel's order (a copied child: the
// residuals themselves).  The residual vector is never stored.  T: arithmetic, u; TF: f; TC: the
// coarse f.  2,535 patches of 16^3 (FP32): 44 us against 60 + 29 for the residual (with its
// ghosts) and its restriction apart.
template <typename T, typename TF, typename TC, int OP, int N>
__global__ void __launch_bounds__(N == 16 ? 256 : 64) resid_restrict3_kernel(
  const DevPatch* __restrict__ dp, const T* __restrict__ u, const T* __restrict__ cf, const TF* __restrict__ f,
  TC* __restrict__ fc, const int32_t* __restrict__ parent, const int32_t* __restrict__ orth, Layout L, int neumann)
{
  constexpr int SX = N + 2, SY = SX * SX, PS = SX * SY, H = N / 2, NT = N == 16 ? 256 : 64;
  __shared__ __align__(16) T tile[PS];
  const int p = xcd_item(blockIdx.x, gridDim.x);
  if (p >= L.np) return;
  const DevPatch& P = dp[p];
  const int t = threadIdx.x;
  // the face ghosts (no thread's depends on another's ghost) while the patch is on its way
  constexpr int FC = N * N / NT;  // 1
  static_assert(FC == 1, "a cell of each face per thread");
  const int fi = t % N, fj = t / N;
  T G[6];
#pragma unroll
  for (int s = 0; s < 6; s++) {
    G[s] = T(0);
    if (P.type[20 + s] >= 0) {
      G[s] = face_ghost3<T>(L, P.type[20 + s], P.orth[20 + s], P.nbr[20 + s], u, p, 0, s, fi, fj);
    } else {
      const T b = at(u, side_cell3(L, p, 0, s, 0, fi, fj));
      G[s] = (OP == 0 && neumann) ? b : -b;
    }
  }
  typedef T Vec __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
  constexpr int W = 16 / sizeof(T);
  static_assert(PS % W == 0, "whole accesses");
  for (int k = t; k < PS / W; k += NT)
    *reinterpret_cast<Vec*>(tile + W * k) = *reinterpret_cast<const Vec*>(&at(u, p * PS + W * k));
  __syncthreads();
#pragma unroll
  for (int s = 0; s < 6; s++) tile[side_cell3(L, 0, 0, s, -1, fi, fj)] = G[s];
  __syncthreads();
  const T ih2[3] = { T(P.inv_h2[0]), T(P.inv_h2[1]), T(P.inv_h2[2]) };
  auto resid = [&](int k, T fv) {  // k: padded index in the patch
    const T mid = tile[k];
    T acc = T(0);
    const int st[3] = { 1, SX, SY };
#pragma unroll
    for (int a = 0; a < 3; a++) {
      const T lower = tile[k - st[a]], upper = tile[k + st[a]];
      if (OP == 0) {
        acc += (upper - T(2) * mid + lower) * ih2[a];
      } else {
        const int ci = p * PS + k;
        const T cm = at(cf, ci), cl = at(cf, ci - st[a]), cu = at(cf, ci + st[a]);
        acc += ((cu + cm) * (upper - mid) - (cl + cm) * (mid - lower)) * (ih2[a] * T(0.5));
      }
    }
    return T(fv - acc);
  };
  const int cp = parent[p], o = orth[p];
  if (o < 0) {  // copyToParent
    for (int k = t; k < N * N * N; k += NT) {
      const int q = (k % N) + 1 + SX * (k / N % N + 1) + SY * (k / (N * N) + 1);
      at(fc, cp * PS + q) = TC(resid(q, T(at(f, p * PS + q))));
    }
    return;
  }
  const int c0 = cp * PS + ((o & 1) ? H : 0) + 1 + SX * (((o & 2) ? H : 0) + 1) + SY * (((o & 4) ? H : 0) + 1);
#pragma unroll
  for (int k = t; k < H * H * H; k += NT) {
    const int X = k % H, Y = k / H % H, Z = k / (H * H);
    const int q = 2 * X + 1 + SX * (2 * Y + 1) + SY * (2 * Z + 1);
    TF fv[8];
#pragma unroll
    for (int r = 0; r < 4; r++) {
      typedef TF F2 __attribute__((ext_vector_type(2), aligned(sizeof(TF))));
      const F2 v = *reinterpret_cast<const F2*>(&at(f, p * PS + q + (r & 1) * SX + (r >> 1) * SY));
      fv[2 * r] = v[0];
      fv[2 * r + 1] = v[1];
    }
    T acc = T(0);
#pragma unroll
    for (int r = 0; r < 8; r++) acc += resid(q + (r & 1) + ((r >> 1) & 1) * SX + (r >> 2) * SY, T(fv[r])) * T(0.125);
    at(fc, c0 + X + SX * Y + SY * Z) = TC(acc);
  }
}

template <typename T, typename TF, typename TC>
void launch_rr3(const te_ghost_filler* g, const te_level_link* l, int op_kind, int neumann, const void* coeffs,
                const void* f, const void* u, void* fc, hipStream_t s)
{
  const te_domain* d = g->d;
  const Layout L = make_layout(3, d->ns, 1, d->np);
#define TE_RR3(OP_, N_)                                                                                             \
  hipLaunchKernelGGL((resid_restrict3_kernel<T, TF, TC, OP_, N_>), dim3(xcd_grid(d->np)), dim3(N_ == 16 ? 256 : 64), \
                     0, s, d->d_patches, (const T*)u, (const T*)coeffs, (const TF*)f, (TC*)fc, l->d_parent,         \
                     l->d_orth, L, neumann)
  if (d->ns[0] == 16) {
    if (op_kind == 0) TE_RR3(0, 16);
    else TE_RR3(1, 16);
  } else {
    if (op_kind == 0) TE_RR3(0, 8);
    else TE_RR3(1, 8);
  }
#undef TE_RR3
}

}  // namespace

bool resid_restrict3_supported(const te_ghost_filler* g, const te_level_link* link)
{
  const te_domain* d = g->d;
  return d->dim == 3 && (d->ns[0] == 8 || d->ns[0] == 16) && d->ns[1] == d->ns[0] && d->ns[2] == d->ns[0] &&
         link->regular && link->covered && link->fine == d;
}

int launch_resid_restrict3(const te_ghost_filler* g, const te_level_link* link, int op_kind, int neumann,
                           const void* coeffs, int dt, int dtf, const void* f, const void* u, int dtc, void* fc,
                           hipStream_t s)
{
  if (g->d->np == 0) return TE_OK;
  if (!resid_restrict3_supported(g, link)) {
    set_error("internal: 3D residual / restriction needs 8^3 or 16^3 patches and a regular, covered link");
    return TE_ERR_UNSUPPORTED;
  }
  if (dt == TE_F64 && dtf == TE_F64 && dtc == TE_F64)
    launch_rr3<double, double, double>(g, link, op_kind, neumann, coeffs, f, u, fc, s);
  else if (dt == TE_F32 && dtf == TE_F32 && dtc == TE_F32)
    launch_rr3<float, float, float>(g, link, op_kind, neumann, coeffs, f, u, fc, s);
  else if (dt == TE_F32 && dtf == TE_F64 && dtc == TE_F32)
    launch_rr3<float, double, float>(g, link, op_kind, neumann, coeffs, f, u, fc, s);
  else if (dt == TE_F32 && dtf == TE_F32 && dtc == TE_F64)
    launch_rr3<float, float, double>(g, link, op_kind, neumann, coeffs, f, u, fc, s);
  else if (dt == TE_F32 && dtf == TE_F64 && dtc == TE_F64)
    launch_rr3<float, double, double>(g, link, op_kind, neumann, coeffs, f, u, fc, s);
  else {
    set_error("unsupported dtype combination for the 3D residual / restriction");
    return TE_ERR_UNSUPPORTED;
  }
  TE_HIP(hipGetLastError());
  return TE_OK;
}

// fin != nullptr: out = fin - A u (residual); else out = A u.  dt: type of u and coeffs,
// dtf: type of fin, dto: type of out.  Supported: (f64,f64,f64), (f32,f32,f32), (f32,f64,f32).
int launch_star(const te_ghost_filler* g, int dt, int dtf, int dto, int op_kind, int neumann, const void* coeffs,
                const void* fin, void* u, void* out, int ncomp, bool fill, hipStream_t s)
{
  if (g->d->np == 0) return TE_OK;
  int rc = TE_OK;
  if (fill) {
    rc = launch_ghost_fill_lowdim(g, dt, u, ncomp, s);
    if (rc) return rc;
  }
  if (dt == TE_F64 && dtf == TE_F64 && dto == TE_F64)
    rc = launch_dim<double, double, double>(g, op_kind, (double*)u, (const double*)coeffs, (const double*)fin, (double*)out,
                                       ncomp, neumann, fill, s);
  else if (dt == TE_F32 && dtf == TE_F32 && dto == TE_F32)
    rc = launch_dim<float, float, float>(g, op_kind, (float*)u, (const float*)coeffs, (const float*)fin, (float*)out, ncomp,
                                    neumann, fill, s);
  else if (dt == TE_F32 && dtf == TE_F64 && dto == TE_F32)
    rc = launch_dim<float, double, float>(g, op_kind, (float*)u, (const float*)coeffs, (const double*)fin, (float*)out,
                                     ncomp, neumann, fill, s);
  else {
    set_error("unsupported dtype combination for the star stencil");
    return TE_ERR_UNSUPPORTED;
  }
  if (rc) return rc;
  TE_HIP(hipGetLastError());
  return TE_OK;
}

}  // namespace te
