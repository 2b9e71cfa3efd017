// 3D face ghosts (TriLinearGhostFiller.cpp:33-175) as a gather: the value of ghost cell (i, j) on
// side s of a patch from its own and its neighbours' interior cells, the terms in the order the
// reference accumulates them (self terms, then the neighbours').
#pragma once

#include "../te_internal.h"

namespace te {

// cells along axis a (selects: a lane's own a would index the kernel's arguments in memory)
__device__ __forceinline__ int axis_cells(const Layout& L, int a)
{
  return a == 0 ? L.n[0] : a == 1 ? L.n[1] : L.n[2];
}

// cell (i, j) of the slice on side s at depth k (k = -1: the ghost layer); the free axes are the
// two other axes in increasing order.  LANE: s differs from lane to lane.
template <bool LANE = false>
__device__ __forceinline__ int side_cell3(const Layout& L, int p, int c, int s, int k, int i, int j)
{
  int a = s >> 1, up = s & 1;
  int ca = up ? (LANE ? axis_cells(L, a) : L.n[a]) - 1 - k : k;
  if (LANE) return lin(L, p, c, a == 0 ? ca : i, a == 0 ? i : a == 1 ? ca : j, a == 2 ? ca : j);
  if (a == 0) return lin(L, p, c, ca, i, j);
  if (a == 1) return lin(L, p, c, i, ca, j);
  return lin(L, p, c, i, j, ca);
}

// type 0 same level (neighbour q[0]), 1 coarser (q[0], orth: where on its side), 2 finer (q[0..3])
template <typename T, bool LANE = false>
__device__ __forceinline__ T face_ghost3(const Layout& L, int type, int orth, const int* q, const T* u, int p, int c,
                                         int s, int i, int j)
{
  const int a = s >> 1, ni = a == 0 ? L.n[1] : L.n[0], nj = a == 2 ? L.n[1] : L.n[2];
  auto U = [&](int qq, int side, int ii, int jj) {
    return at(component(L, u, qq, c), side_cell3<LANE>(L, 0, 0, side, 0, ii, jj));
  };
  if (type == 0) return U(q[0], s ^ 1, i, j);
  T G = T(0);
  if (type == 1) {
    const int oi = (orth & 1) ? ni : 0, oj = (orth & 2) ? nj : 0;
    const int pi = ((i + oi) % 2 == 0) ? i + 1 : i - 1;
    const int pj = ((j + oj) % 2 == 0) ? j + 1 : j - 1;
    G += T(5.0 / 6.0) * U(p, s, i, j);
    G -= T(1.0 / 6.0) * U(p, s, pi, j);
    G -= T(1.0 / 6.0) * U(p, s, i, pj);
    G -= T(1.0 / 6.0) * U(p, s, pi, pj);
    G += T(4.0 / 6.0) * U(q[0], s ^ 1, (i + oi) / 2, (j + oj) / 2);
    return G;
  }
  // the 2 x 2 fine cells against it: even cells per side (TriLinearGhostFiller.cpp:576-584), so
  // all four lie in the finer neighbour that covers this quarter of the side
  const int hi = 2 * i >= ni, hj = 2 * j >= nj;
  const int fq = q[hi + 2 * hj], fi = 2 * i - (hi ? ni : 0), fj = 2 * j - (hj ? nj : 0);
  G -= T(1.0 / 3.0) * U(p, s, i, j);
#pragma unroll
  for (int dj = 0; dj < 2; dj++)
#pragma unroll
    for (int di = 0; di < 2; di++) G += T(1.0 / 3.0) * U(fq, s ^ 1, fi + di, fj + dj);
  return G;
}

// The face ghosts first[s] <= k < last[s] of each side s of patch p (k: the face's cells, first
// free axis fastest), by the nt threads t = 0 .. nt - 1: each thread takes a cell of all six sides
// at a time, so that their loads are in flight together.
template <typename T>
__device__ __forceinline__ void fill_faces3(const Layout& L, const DevPatch& P, T* u, int p, int t, int nt,
                                            const int (&first)[6], const int (&last)[6])
{
  int cells[6], most = 0;
#pragma unroll
  for (int s = 0; s < 6; s++) {
    cells[s] = P.type[20 + s] < 0 ? 0 : last[s] - first[s];
    most = cells[s] > most ? cells[s] : most;
  }
  for (int c = 0; c < L.ncomp; c++)
    for (int i = t; i < most; i += nt) {
      T G[6];
#pragma unroll
      for (int s = 0; s < 6; s++) {
        if (i >= cells[s]) continue;
        const int ni = L.n[s < 2 ? 1 : 0], k = first[s] + i, j = k / ni;
        G[s] = face_ghost3<T>(L, P.type[20 + s], P.orth[20 + s], P.nbr[20 + s], u, p, c, s, k - j * ni, j);
      }
#pragma unroll
      for (int s = 0; s < 6; s++) {
        if (i >= cells[s]) continue;
        const int ni = L.n[s < 2 ? 1 : 0], k = first[s] + i, j = k / ni;
        at(component(L, u, p, c), side_cell3(L, 0, 0, s, -1, k - j * ni, j)) = G[s];
      }
    }
}

// The same for all face ghosts of patches whose largest face has `face` <= 16 cells: the threads
// take the six faces' cells in a row, since a face's cells alone would leave most lanes idle.
template <typename T>
__device__ __forceinline__ void fill_faces3_small(const Layout& L, const DevPatch& P, T* u, int p, int t, int nt, int face)
{
  for (int g = t; g < 6 * face; g += nt) {
    const int s = g / face, k = g - s * face, a = s >> 1;
    const int ni = a == 0 ? L.n[1] : L.n[0], nj = a == 2 ? L.n[1] : L.n[2], j = k / ni, i = k - j * ni;
    const int type = P.type[20 + s];
    if (type < 0 || j >= nj) continue;
    const int orth = P.orth[20 + s];
    for (int c = 0; c < L.ncomp; c++)
      at(component(L, u, p, c), side_cell3<true>(L, 0, 0, s, -1, i, j)) =
        face_ghost3<T, true>(L, type, orth, P.nbr[20 + s], u, p, c, s, i, j);
  }
}
// faces of at most this many cells: fill_faces3_small (4^3; 6^3's 36 cells fill a wave's lanes by themselves)
constexpr int kSmallFace = 16;
__host__ __device__ inline int largest_face(const Layout& L)
{
  const int a = L.n[0] * L.n[1], b = L.n[1] * L.n[2], c = L.n[0] * L.n[2], m = a > b ? a : b;
  return m > c ? m : c;
}

}  // namespace te
