// Ghost filling as a race-free gather ("pull"): every ghost cell facing a
// neighbour is computed by exactly one thread from the closed-form weights of
// the reference's push-style fillers (MPIGhostFiller.h:1055-1092 with
// BiLinearGhostFiller.cpp, BiQuadraticGhostFiller.cpp, TriLinearGhostFiller.cpp).
// Terms are summed in the order the reference accumulates them: self terms
// first (fillGhostCellsForLocalPatch runs before processLocalFills), then the
// neighbour contributions in the order their calls are enumerated.
#include <algorithm>

#include "../te_internal.h"
#include "ghost2d.h"
#include "ghost3d.h"

namespace te {
namespace {

constexpr int NB_NORMAL = 0, NB_COARSE = 1;

// 2D side ghosts: one wavefront per patch walks the patch's ring of side ghost cells
// (ring_cell order: the two x faces, then the two y faces, so the y faces' ghost rows are
// written by consecutive lanes).  One 16-byte ring-table record per cell names the
// neighbour its formula reads; the closed forms are ghost2d.h's (self terms, then the
// neighbour terms, in the reference's order).  Patches are split over the XCDs
// (xcd_range), so a patch and most of its neighbours are read through one L2.
template <typename T, int KIND>
__global__ void __launch_bounds__(256) ghost_ring_2d(const int4* __restrict__ ring, T* __restrict__ u, Layout L)
{
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int n0 = L.n[0], n1 = L.n[1], nr = 2 * (n0 + n1);
  const XcdRange xr = xcd_range(blockIdx.x, gridDim.x, L.np, 4);
  for (int p = xr.first + wave; p < xr.end; p += xr.step) {
    for (int g = lane; g < nr; g += 64) {
      int s, t;
      const int4 r = ring[ring_index(p, g, n0, n1, &s, &t)];
      if (r.x < 0) continue;  // a physical side: the operators apply its condition themselves
      fill_ring_cell<T, KIND>(r, s, t, u, L, p);
    }
  }
}

// 2D corners (fill type Corners).  BiLinearGhostFiller.cpp:167-264,
// BiQuadraticGhostFiller.cpp:239-334.
template <typename T, int KIND>
__global__ void ghost_corners_2d(const DevPatch* __restrict__ dp, T* __restrict__ u, Layout L)
{
  int gid = blockIdx.x * blockDim.x + threadIdx.x;
  int p = gid >> 2;
  if (p >= L.np) return;
  int cr = gid & 3;
  int type = dp[p].type[cr];
  if (type < 0) return;
  int q = dp[p].nbr[cr][0];
  int ux = cr & 1, uy = (cr >> 1) & 1;
  int nx = L.n[0], ny = L.n[1];
  for (int c = 0; c < L.ncomp; c++) {
    // interior corner cell of patch p at corner cr, and its (1,1) inner cell
    T P0 = u[lin(L, p, c, ux ? nx - 1 : 0, uy ? ny - 1 : 0, 0)];
    T P1 = u[lin(L, p, c, ux ? nx - 2 : 1, uy ? ny - 2 : 1, 0)];
    // neighbour's interior cell at the opposite corner
    T Q0 = u[lin(L, q, c, ux ? 0 : nx - 1, uy ? 0 : ny - 1, 0)];
    T Q1 = u[lin(L, q, c, ux ? 1 : nx - 2, uy ? 1 : ny - 2, 0)];
    T G;
    if (type == NB_NORMAL) {
      G = Q0;
    } else if (type == NB_COARSE) {
      if (KIND == TE_BILINEAR) G = P0 / T(3) + T(2) * Q0 / T(3);
      else G = (T(2) * P0 / T(3) - P1 / T(5)) + T(8) * Q0 / T(15);
    } else {
      if (KIND == TE_BILINEAR) G = -P0 / T(3) + T(4) * Q0 / T(3);
      else G = -P0 / T(15) + (T(2) * Q0 / T(3) + T(2) * Q1 / T(5));
    }
    u[lin(L, p, c, ux ? nx : -1, uy ? ny : -1, 0)] = G;
  }
}

// 3D faces, so that a wave's patch (and side) and with it the neighbour records are uniform and a
// cell's place on the face takes one division (FP64, one thread per ghost cell of all patches -> the form):
//  FACES_SMALL, faces of at most 16 cells: a wave per patch, the six faces' cells in a row
//    (fill_faces3_small; 32,768 patches of 4^3: 36 -> 26 us, 48 as FACES_SIDES);
//  FACES_SIDES, up to 64 cells: a workgroup per patch, a wave per side (4,096 of 8^3: 23 -> 12);
//  FACES_PARTS, more: as FACES_SIDES, the patch's faces shared by several workgroups, on large
//    levels in parts of under three passes of a wave (4,096 of 12^3: 42 -> 27, of 16^3 77 -> 49, of
//    32^3 327 -> 318; in one workgroup a patch, a thread the same cell of all six sides: 32, 60 and
//    356), on small ones in as many as fill the card (512 of 16^3: 11.8 -> 7.1; 64 of 64^3: 13.1 ->
//    12.4; 8 of 128^3: 6.8 -> 5.1).  Up to one patch a CU they are dealt to the XCDs in turn:
//    contiguous eighths take 15.3 us for 64 of 64^3, but 6.8 against 9.9 for 512 of 16^3
enum FaceForm { FACES_SMALL, FACES_SIDES, FACES_PARTS };

template <typename T, int FORM>
__global__ void __launch_bounds__(FORM == FACES_SMALL ? 256 : 384)
  ghost_faces_3d(const DevPatch* __restrict__ dp, T* u, Layout L, int split, bool in_turn)
{
  const int b = FORM == FACES_PARTS && in_turn ? blockIdx.x : xcd_item(blockIdx.x, gridDim.x);
  if (FORM == FACES_SMALL) {
    const int q = __builtin_amdgcn_readfirstlane(b * 4 + (threadIdx.x >> 6));
    if (q < L.np) fill_faces3_small<T>(L, dp[q], u, q, threadIdx.x & 63, 64, largest_face(L));
    return;
  }
  const int p = FORM == FACES_PARTS ? b >> split : b;
  if (p >= L.np) return;
  const DevPatch& P = dp[p];
  const int s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int type = P.type[20 + s], ni = L.n[s < 2 ? 1 : 0], nj = L.n[s < 4 ? 2 : 1];
  if (type < 0) return;
  auto fill = [&](int k) {
    const int j = k / ni;
    for (int c = 0; c < L.ncomp; c++) {
      const T G = face_ghost3<T>(L, type, P.orth[20 + s], P.nbr[20 + s], u, p, c, s, k - j * ni, j);
      at(component(L, u, p, c), side_cell3(L, 0, 0, s, -1, k - j * ni, j)) = G;
    }
  };
  if (FORM == FACES_SIDES) {
    if (lane < ni * nj) fill(lane);
  } else {
    int first;
    const int last = split_range(ni * nj, split, b & ((1 << split) - 1), &first);
    for (int k = first + lane; k < last; k += 64) fill(k);
  }
}

// 3D edge e (Face<3,1>): free axis = e >> 2; fixed sides in axis order with
// bit k of e = upper on the k-th fixed axis (Face.h:504-515).
__device__ __forceinline__ int edge_cell3(const Layout& L, int p, int c, int e, int k, int i)
{
  int fa = e >> 2;
  int x[3];
  int kk = 0;
  for (int a = 0; a < 3; a++) {
    if (a == fa) {
      x[a] = i;
    } else {
      int up = (e >> kk) & 1;
      x[a] = up ? L.n[a] - 1 - k : k;
      kk++;
    }
  }
  return lin(L, p, c, x[0], x[1], x[2]);
}

// 3D edges and corners (fill types Edges / Corners), TriLinearGhostFiller.cpp:188-405.
template <typename T>
__global__ void ghost_lowdim_3d(const DevPatch* __restrict__ dp, T* __restrict__ u, Layout L, int nmax,
                                int with_corners)
{
  int gid = blockIdx.x * blockDim.x + threadIdx.x;
  int per = 12 * nmax + 8;
  int p = gid / per;
  if (p >= L.np) return;
  int r = gid - p * per;
  if (r < 12 * nmax) {
    int e = r / nmax;
    int i = r - e * nmax;
    int n = L.n[e >> 2];
    if (i >= n) return;
    int slot = 8 + e;
    int type = dp[p].type[slot];
    if (type < 0) return;
    int eo = e ^ 3;  // opposite edge
    for (int c = 0; c < L.ncomp; c++) {
      T G;
      if (type == NB_NORMAL) {
        G = u[edge_cell3(L, dp[p].nbr[slot][0], c, eo, 0, i)];
      } else if (type == NB_COARSE) {
        int q = dp[p].nbr[slot][0];
        int off = dp[p].orth[slot] == 1 ? n : 0;
        G = T(0);
        for (int tp = i - 1; tp <= i + 1; tp++) {
          if (tp < 0 || tp >= n) continue;
          T sv = u[edge_cell3(L, p, c, e, 0, tp)];
          if (tp == i) {
            G += T(2.0 / 3.0) * sv;
          } else {
            int partner = ((tp + off) % 2 == 0) ? tp + 1 : tp - 1;
            if (partner == i) G += T(-1.0 / 3.0) * sv;
          }
        }
        G += T(2.0 / 3.0) * u[edge_cell3(L, q, c, eo, 0, (i + off) / 2)];
      } else {
        G = T(-1.0 / 3.0) * u[edge_cell3(L, p, c, e, 0, i)];
        for (int k = 0; k < 2; k++) {
          int q = dp[p].nbr[slot][k];
          int off = k * n;
          for (int fi = 2 * i - off; fi <= 2 * i - off + 1; fi++) {
            if (fi < 0 || fi >= n) continue;
            G += T(2.0 / 3.0) * u[edge_cell3(L, q, c, eo, 0, fi)];
          }
        }
      }
      u[edge_cell3(L, p, c, e, -1, i)] = G;
    }
  } else {
    if (!with_corners) return;
    int cr = r - 12 * nmax;
    int type = dp[p].type[cr];
    if (type < 0) return;
    int q = dp[p].nbr[cr][0];
    int ux = cr & 1, uy = (cr >> 1) & 1, uz = (cr >> 2) & 1;
    int nx = L.n[0], ny = L.n[1], nz = L.n[2];
    for (int c = 0; c < L.ncomp; c++) {
      T P0 = u[lin(L, p, c, ux ? nx - 1 : 0, uy ? ny - 1 : 0, uz ? nz - 1 : 0)];
      T Q0 = u[lin(L, q, c, ux ? 0 : nx - 1, uy ? 0 : ny - 1, uz ? 0 : nz - 1)];
      T G;
      if (type == NB_NORMAL) G = Q0;
      else if (type == NB_COARSE) G = P0 / T(3) + T(2) * Q0 / T(3);
      else G = -P0 / T(3) + T(4) * Q0 / T(3);
      u[lin(L, p, c, ux ? nx : -1, uy ? ny : -1, uz ? nz : -1)] = G;
    }
  }
}

template <typename T>
int ghost_fill_t(const te_ghost_filler* g, T* u, int ncomp, bool faces, bool lowdim, hipStream_t s)
{
  const te_domain* d = g->d;
  if (d->np == 0) return TE_OK;
  Layout L = make_layout(d->dim, d->ns, ncomp, d->np);
  const int B = 256;
  if (d->dim == 2) {
    // a wave per patch (4 per workgroup), at most 8192 workgroups walking the rest
    const int ngroups = (d->np + 3) / 4;
    const int grid = ngroups < 8192 ? ngroups : 8192;
    if (!faces) {
    } else if (g->kind == TE_BILINEAR)
      hipLaunchKernelGGL((ghost_ring_2d<T, TE_BILINEAR>), dim3(grid), dim3(B), 0, s, (const int4*)d->d_ring, u, L);
    else
      hipLaunchKernelGGL((ghost_ring_2d<T, TE_BIQUADRATIC>), dim3(grid), dim3(B), 0, s, (const int4*)d->d_ring, u,
                         L);
    if (lowdim && g->fill_type == TE_CORNERS) {
      int cg = (d->np * 4 + B - 1) / B;
      if (g->kind == TE_BILINEAR)
        hipLaunchKernelGGL((ghost_corners_2d<T, TE_BILINEAR>), dim3(cg), dim3(B), 0, s, d->d_patches, u, L);
      else
        hipLaunchKernelGGL((ghost_corners_2d<T, TE_BIQUADRATIC>), dim3(cg), dim3(B), 0, s, d->d_patches, u, L);
    }
  } else {
    const int face = largest_face(L);
    int split = patch_split(d->np, face, 64, 2, face);  // of FACES_PARTS: short waves, so 48 of them a CU
    while ((face >> split) >= 3 * 64) split++;
#define TE_GF(FORM_, UNITS_, BLOCK_)                                                                                \
  hipLaunchKernelGGL((ghost_faces_3d<T, FORM_>), dim3(xcd_grid(UNITS_)), dim3(BLOCK_), 0, s, d->d_patches, u, L, split, \
                     d->np <= cu_count())
    if (!faces) {
    } else if (face <= kSmallFace) {
      TE_GF(FACES_SMALL, (d->np + 3) / 4, B);
    } else if (face <= 64) {
      TE_GF(FACES_SIDES, d->np, 384);
    } else {
      TE_GF(FACES_PARTS, d->np << split, 384);
    }
#undef TE_GF
    if (lowdim && g->fill_type != TE_FACES) {
      int tmax = d->ns[0];
      for (int a = 1; a < 3; a++) tmax = d->ns[a] > tmax ? d->ns[a] : tmax;
      long tl = (long)d->np * (12 * tmax + 8);
      int lg = (int)((tl + B - 1) / B);
      hipLaunchKernelGGL((ghost_lowdim_3d<T>), dim3(lg), dim3(B), 0, s, d->d_patches, u, L, tmax,
                         g->fill_type == TE_CORNERS ? 1 : 0);
    }
  }
  TE_HIP(hipGetLastError());
  return TE_OK;
}

}  // namespace

int launch_ghost_fill(const te_ghost_filler* g, int dtype, void* u, int ncomp, hipStream_t s)
{
  if (dtype == TE_F64) return ghost_fill_t<double>(g, (double*)u, ncomp, true, true, s);
  return ghost_fill_t<float>(g, (float*)u, ncomp, true, true, s);
}

// the face ghosts alone
int launch_ghost_fill_faces(const te_ghost_filler* g, int dtype, void* u, int ncomp, hipStream_t s)
{
  if (dtype == TE_F64) return ghost_fill_t<double>(g, (double*)u, ncomp, true, false, s);
  return ghost_fill_t<float>(g, (float*)u, ncomp, true, false, s);
}

// the edge and corner ghosts alone (nothing for fill type Faces)
int launch_ghost_fill_lowdim(const te_ghost_filler* g, int dtype, void* u, int ncomp, hipStream_t s)
{
  if (g->fill_type == TE_FACES) return TE_OK;
  if (dtype == TE_F64) return ghost_fill_t<double>(g, (double*)u, ncomp, false, true, s);
  return ghost_fill_t<float>(g, (float*)u, ncomp, false, true, s);
}

}  // namespace te
