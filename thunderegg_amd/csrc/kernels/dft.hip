// Poisson::DFTPatchSolver::solveSinglePatch (Poisson/DFTPatchSolver.h:420-450) for
// every patch of a level in one launch, generic (VALU) form for any n: a workgroup holds
// PPW patches, TPP threads each (by a rule, or a variant of the autotuner's table, tune.h).
// Each patch is staged in LDS; each axis transform y = M x (executePlan, :205-265) is a
// dense n x n product over all lines of that axis; eigenvalues (:320-361) come from a
// per-axis sin^2 table.
//
// Template parameters: T = arithmetic / u type, TF = type of f, TO = type of
// the output.  UZERO: u is known to be identically zero (the first smoothing
// sweep of a freshly zeroed level), so the interface terms of
// modifyRHSForInternalBoundaryConditions vanish and u is not read.
#include <algorithm>

#include "../te_internal.h"
#include "dft.h"
#include "blas.h"
#include "dft_wave.h"
#include "ghost2d.h"
#include "ghost3d.h"
#include "../tune.h"

namespace te {
namespace {

// The launch's geometry: LDS pitches and the divisions by run-time sizes.
struct DftGeom {
  int px;      // row pitch of the staged patch (odd where it fits, so that a wave's lines spread over the banks)
  int mp;      // pitch of a transposed matrix; a multiple of 4 (vec) where it fits
  int nmat;    // matrices per direction and copy: one per axis, or one for all of equal sizes and types
  bool vec, share;  // share: one copy for the whole workgroup (every patch has the same types)
  bool one;         // a thread per cell: one output a task, the cell's interface terms formed by its thread
  FastDiv d0, d1, lines[3], na[3];
};

// GM (2D): 0 = the ghost values of u are read from u (filled beforehand); 1 = they are
// computed here from the neighbours' cells (ghost2d.h, the filler's closed forms); 2 = the same
// on u + P uc (DirectInterpolator applied on the fly: uc is the coarser level's solution).
// With GM != 0, out must not alias u.
//
// A task of an axis transform is one line and four of its outputs: per step of the product one
// staged value and four matrix values (one wide LDS read, the same for a wave's lanes, which
// take consecutive lines) feed four multiply-adds.  The last forward transform divides by the
// eigenvalues as it writes, the last inverse one writes the result.  The interface terms are
// formed first, a thread per side cell (in 2D from one ring-table record each).  Where the patch
// has a thread per cell (G.one, small levels) a task is one output, and a thread forms the terms
// of its own cell from the filled ghosts: the launch then lasts as long as one thread's chain,
// and four outputs, a barrier per axis and terms apart make that longer (16 patches of 8^2 in FP64
// 7.8 us, 5.3 so; 8 of 4^3 9.7, 6.4).
// Bound by LDS reads on large levels, by the chain of loads and barriers on small ones.
// Measured against one output a thread and task everywhere, the terms formed cell by cell (apply
// from zero with its zeroed ghosts / sweep on filled ghosts, us): 1,024 patches of 24^2 in FP64
// 44 -> 14.7 / 41.6 -> 14.9; 512 of 12^3 in FP32 36.6 -> 15.5 / 34.0 -> 17.9; 512 of 6^3 in
// FP32 10.3 -> 6.7 / 8.6 -> 7.5; 1,024 of 7^2 7.9 -> 5.3 / 7.1 -> 6.0; 48 problems
// together, a third of them on 8^2 patches, 12.2 -> 10.7 ms.
template <typename T, typename TF, typename TO, int D, int OP, bool UZERO, int GM = 0, int KIND = 0, typename TC = T>
__global__ void __launch_bounds__(256) dft_kernel(const DevPatch* __restrict__ dp, const int* __restrict__ ptype,
                                                  const T* __restrict__ mats, const T* __restrict__ s2tab,
                                                  const TF* __restrict__ f, const T* u, const T* __restrict__ coeffs,
                                                  TO* out, Layout L, int ppw, FusedArgs<T, TC> fa,
                                                  const int4* __restrict__ ring, DftGeom G, bool zero_ghosts)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  const int n0 = L.n[0], n1 = L.n[1], n2 = D == 3 ? L.n[2] : 1;
  const int nn[3] = { n0, n1, n2 }, N = n0 * n1 * n2, NP = G.px * n1 * n2;
  const int nmax = n0 > n1 ? (n0 > n2 ? n0 : n2) : (n1 > n2 ? n1 : n2);
  const int msz = nmax * G.mp, nr = UZERO ? 0 : D == 2 ? 2 * (n0 + n1) : 2 * (n1 * n2 + n0 * n2 + n0 * n1);
  // this thread's patch (sub-block of tpp threads) and its index t within it; the threads
  // of a patch past the last one take part in the barriers only
  const int tpp = blockDim.x / ppw, sub = threadIdx.x / tpp, t = threadIdx.x - sub * tpp;
  const bool live = blockIdx.x * ppw + sub < L.np;
  const int p = live ? blockIdx.x * ppw + sub : L.np - 1;
  // LDS: the matrices (forward, then inverse; one copy or one per patch), then per patch two
  // buffers, the second of which first holds the interface terms
  T* M = reinterpret_cast<T*>(smem_raw) + (G.share ? 0 : sub * 2 * G.nmat * msz);
  T* A = reinterpret_cast<T*>(smem_raw) + (G.share ? 1 : ppw) * 2 * G.nmat * msz + sub * (NP + (NP > nr ? NP : nr));
  T* B = A + NP;
  T* term = B;  // consumed before the first transform writes B
  // transform and eigenvalue types per axis, zero mode; without Neumann sides (share) DST-II, Dirichlet
  int tf[D], te[D], zero_mode = 0;
#pragma unroll
  for (int a = 0; a < D; a++) {
    tf[a] = 3;
    te[a] = 2;
  }
  if (!G.share) {
    const int* pt = ptype + p * 8;
#pragma unroll
    for (int a = 0; a < D; a++) {
      tf[a] = pt[a];
      te[a] = pt[3 + a];
    }
    zero_mode = pt[6];
  }
  const DevPatch& P = dp[p];
  if (UZERO && zero_ghosts && live)  // the patch's results follow after the barriers
    for (int k = t; k < L.cs; k += tpp) out[p * L.ps + k] = TO(0);
  {
    const int m0 = G.share ? threadIdx.x : t, step = G.share ? blockDim.x : tpp;
#pragma unroll
    for (int a = 0; a < D; a++) {
      if (a >= G.nmat) break;
      const int ti = tf[a] == 0 ? 1 : (tf[a] == 3 ? 4 : tf[a]);  // DCT_II->DCT_III, DST_II->DST_III, IV types self-inverse
      for (int i = m0; i < nn[a] * nn[a]; i += step) {
        const int k = G.na[a](i), j = i - k * nn[a];
        M[a * msz + j * G.mp + k] = mats[(tf[a] * 3 + a) * kDftMatStride + i];
        M[(G.nmat + a) * msz + j * G.mp + k] = mats[(ti * 3 + a) * kDftMatStride + i];
      }
    }
  }
  // f_copy = f, then modifyRHSForInternalBoundaryConditions (Poisson :165-180, VarPoisson
  // :168-186), sides in the reference's order: here (a thread per cell), or term by term below
  const bool here = !UZERO && GM == 0 && G.one;
  for (int o = t; o < N; o += tpp) {
    const int row = G.d0(o), x = o - row * n0, z = D == 3 ? G.d1(row) : 0, y = row - z * n1;
    const int c = lin(L, p, 0, x, y, z), c3[3] = { x, y, z };
    T v = T(f[c]);
    if (here) {
#pragma clang fp contract(off)  // a term is rounded before it is subtracted, as below: the same bits for every launch shape
      const T ub = u[c], cb = OP == 1 ? coeffs[c] : T(0);
#pragma unroll
      for (int s = 0; s < 2 * D; s++) {
        const int a = s >> 1, st = a == 0 ? 1 : (a == 1 ? L.sx : L.sy), g = s & 1 ? c + st : c - st;
        if (c3[a] != (s & 1 ? nn[a] - 1 : 0) || P.type[(D == 2 ? 4 : 20) + s] < 0) continue;
        const T ih2 = T(P.inv_h2[a]), w = u[g] + ub;
        if (OP == 0) v -= w * ih2;
        else v -= w * (cb + coeffs[g]) * (ih2 * T(0.5));
      }
    }
    A[row * G.px + x] = v;
  }
  if (!UZERO && !here && D == 2) {
    for (int g = t; g < nr; g += tpp) {
      int s, tt;
      const int ri = ring_index(p, g, n0, n1, &s, &tt);
      const int a = s >> 1, up = s & 1, nt = a == 0 ? n1 : n0;
      T v = T(0);
      if (P.type[4 + s] >= 0) {
        int bx, by;
        side_xy(s, 0, tt, nn[a], &bx, &by);
        const int bi = lin(L, p, 0, bx, by, 0), gi = bi + (up ? 1 : -1) * (a == 0 ? 1 : L.sx);
        if (GM == 0) {
          v = u[gi] + u[bi];
        } else {
          const int4 r = ring[ri];
          const int par = GM == 2 ? fa.parent[p] : 0, o = GM == 2 ? fa.porth[p] : -1;
          // u, or u + P uc with q's parent and orthant, at a cell of patch q
          auto val = [&](int q, int qpar, int qo, int x, int y) {
            T w = at(u, lin(L, q, 0, x, y, 0));
            if (GM == 2) {
              const int cx = qo >= 0 ? (x + ((qo & 1) ? n0 : 0)) / 2 : x, cy = qo >= 0 ? (y + ((qo & 2) ? n1 : 0)) / 2 : y;
              w = T(w + T(at(fa.uc, lin(L, qpar, 0, cx, cy, 0))));
            }
            return w;
          };
          T gv[4] = { T(0), T(0), T(0), T(0) };
          ghost2d_gather<KIND>(r.x, r.y, r.z, s, tt, nn[a], nt,
                               [&](int k, int q, int x, int y) { gv[k] = val(q, r.w >> 3, (r.w & 7) - 1, x, y); });
          const T ug = ghost2d_combine<T, KIND>(r.x, r.y, tt, nt,
                                                [&](int k, int e) {
                                                  int x, y;
                                                  side_xy(s, k, e, nn[a], &x, &y);
                                                  return val(p, par, o, x, y);
                                                },
                                                gv);
          v = ug + val(p, par, o, bx, by);
        }
        const T ih2 = T(P.inv_h2[a]);
        if (OP == 0) v = v * ih2;
        else v = v * (coeffs[bi] + coeffs[gi]) * (ih2 * T(0.5));
      }
      term[g] = v;
    }
  }
  // 3D face cell g of axis a: its side and cell (first free axis fastest)
  auto face_cell = [&](int a, int g, int* up, int (&c3)[3]) {
    const int f0 = a == 0 ? 1 : 0, f1 = a == 2 ? 1 : 2, cells = nn[f0] * nn[f1];
    *up = g >= cells ? 1 : 0;
    const int q = g - *up * cells, j = a == 0 ? G.d1(q) : G.d0(q);
    c3[a] = *up ? nn[a] - 1 : 0;
    c3[f0] = q - j * nn[f0];
    c3[f1] = j;
  };
  auto faces = [&](int a) { return 2 * N / nn[a]; };
  if (!UZERO && !here && D == 3) {
#pragma unroll
    for (int a = 0; a < D; a++) {
      const int g0 = a == 0 ? 0 : a == 1 ? faces(0) : faces(0) + faces(1);
      const T ih2 = T(P.inv_h2[a]);
      for (int g = t; g < faces(a); g += tpp) {
        int up, c3[3];
        face_cell(a, g, &up, c3);
        T v = T(0);
        if (P.type[20 + 2 * a + up] >= 0) {
          const int bi = lin(L, p, 0, c3[0], c3[1], c3[2]), st = a == 0 ? 1 : (a == 1 ? L.sx : L.sy);
          const int gi = up ? bi + st : bi - st;
          v = u[gi] + u[bi];
          if (OP == 0) v = v * ih2;
          else v = v * (coeffs[bi] + coeffs[gi]) * (ih2 * T(0.5));
        }
        term[g0 + g] = v;
      }
    }
  }
  __syncthreads();
  if (!UZERO && !here) {
#pragma unroll
    for (int a = 0; a < D; a++) {
      if (D == 2) {
        const int nt = a == 0 ? n1 : n0, g0 = a == 0 ? 0 : 2 * n1;
        for (int g = t; g < 2 * nt; g += tpp) {
          int s, tt, bx, by;
          ring_cell(g0 + g, n0, n1, &s, &tt);
          side_xy(s, 0, tt, nn[a], &bx, &by);
          A[by * G.px + bx] -= term[g0 + g];
        }
      } else {
        const int g0 = a == 0 ? 0 : a == 1 ? faces(0) : faces(0) + faces(1);
        for (int g = t; g < faces(a); g += tpp) {
          int up, c3[3];
          face_cell(a, g, &up, c3);
          A[c3[0] + G.px * (c3[1] + n1 * c3[2])] -= term[g0 + g];
        }
      }
      __syncthreads();
    }
  }
  T lam[D];
#pragma unroll
  for (int a = 0; a < D; a++) lam[a] = T(4.0 / (P.h[a] * P.h[a]));
  T scale = T(1);
#pragma unroll
  for (int a = 0; a < D; a++) scale *= T(2.0) / T(nn[a]);
  // one transform (DST-II / DCT-II / DCT-IV / DST-IV and their inverses) along axis a
  // (pre(l, k0): task (l, k0)'s values for its outputs, loaded before its product)
  auto transform = [&](int a, const T* Mt, const T* src, auto pre, auto put) {
    const int na = nn[a], sta = a == 0 ? 1 : (a == 1 ? G.px : G.px * n1), nl = (int)G.lines[a].d;
    const int tasks = G.one ? nl * na : nl * ((na + 3) / 4);
    for (int i = t; i < tasks; i += tpp) {
      const int kb = G.lines[a](i), l = i - kb * nl, k0 = G.one ? kb : 4 * kb;
      int base;
      if (a == 0) {
        base = l * G.px;
      } else {
        const int q = G.d0(l);
        base = l - q * n0 + (a == 1 ? q * G.px * n1 : q * G.px);
      }
      const auto e = pre(l, k0);
      T acc[4] = { T(0), T(0), T(0), T(0) };
      if (G.one) {
#pragma unroll 4
        for (int j = 0; j < na; j++) acc[0] += Mt[j * G.mp + k0] * src[base + j * sta];
        put(l, k0, base + k0 * sta, acc[0], e, 0);
        continue;
      }
      if (G.vec) {
        typedef T V4 __attribute__((ext_vector_type(4)));
#pragma unroll 4
        for (int j = 0; j < na; j++) {
          const T v = src[base + j * sta];
          const V4 m = *reinterpret_cast<const V4*>(Mt + j * G.mp + k0);
#pragma unroll
          for (int r = 0; r < 4; r++) acc[r] += m[r] * v;
        }
      } else {
        int k[4];
#pragma unroll
        for (int r = 0; r < 4; r++) k[r] = k0 + r < na ? k0 + r : na - 1;
        for (int j = 0; j < na; j++) {
          const T v = src[base + j * sta];
#pragma unroll
          for (int r = 0; r < 4; r++) acc[r] += Mt[j * G.mp + k[r]] * v;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; r++)
        if (k0 + r < na) put(l, k0 + r, base + (k0 + r) * sta, acc[r], e, r);
    }
  };
  // the eigenvalues (:320-361) of a task's outputs of the last forward transform
  struct Eig {
    T v[4];
  };
  auto eigen = [&](int l, int k0) {
    const int y = D == 3 ? G.d0(l) : 0, x = l - y * n0;
    const T sx = s2tab[te[0] * 3 * kDftMatDim + x], sy = D == 3 ? s2tab[(te[1] * 3 + 1) * kDftMatDim + y] : T(0);
    T sl[4];
#pragma unroll
    for (int r = 0; r < 4; r++)  // loaded together (a load under each output's bound would wait for the one before)
      sl[r] = s2tab[(te[D - 1] * 3 + D - 1) * kDftMatDim + (k0 + r < nn[D - 1] ? k0 + r : nn[D - 1] - 1)];
    Eig e;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      T eig = T(0);
      eig -= lam[0] * sx;
      if (D == 3) eig -= lam[1] * sy;
      eig -= lam[D - 1] * sl[r];
      e.v[r] = eig;
    }
    return e;
  };
  T* src = A;
  T* dst = B;
#pragma unroll
  for (int a = 0; a < D; a++) {
    transform(a, M + (G.nmat == 1 ? 0 : a) * msz, src, [&](int l, int k0) { return a < D - 1 ? Eig{} : eigen(l, k0); },
              [&](int l, int k, int at_, T v, const Eig& e, int r) {
                if (a == D - 1) {
                  v = v / e.v[r];
                  if (zero_mode && l == 0 && k == 0) v = T(0);  // all-Neumann patch without neighbours (:438-440)
                }
                dst[at_] = v;
              });
    __syncthreads();
    T* sw = src;
    src = dst;
    dst = sw;
  }
#pragma unroll
  for (int a = 0; a < D; a++) {
    transform(a, M + (G.nmat + (G.nmat == 1 ? 0 : a)) * msz, src, [](int, int) { return 0; },
              [&](int l, int k, int at_, T v, int, int) {
                if (a < D - 1) {
                  dst[at_] = v;
                } else if (live) {
                  const int y = D == 3 ? G.d0(l) : k, x = D == 3 ? l - y * n0 : l;
                  out[lin(L, p, 0, x, y, D == 3 ? k : 0)] = TO(v * scale);
                }
              });
    if (a < D - 1) __syncthreads();
    T* sw = src;
    src = dst;
    dst = sw;
  }
}

// pitches, sharing and the launch's LDS bytes for ppw patches a workgroup
size_t dft_geom(const te_dft_plan* pl, size_t esz, int ppw, bool terms, DftGeom* G)
{
  const te_domain* d = pl->g->d;
  const int D = d->dim, n0 = d->ns[0], n1 = d->ns[1], n2 = D == 3 ? d->ns[2] : 1;
  const int nmax = std::max(n0, std::max(n1, n2)), N = n0 * n1 * n2;
  const bool cubic = n0 == n1 && (D == 2 || n2 == n0);
  G->share = pl->mask == 0;
  G->nmat = G->share && cubic ? 1 : D;
  auto bytes = [&]() {
    const size_t np = (size_t)G->px * n1 * n2;
    return esz * ((size_t)(G->share ? 1 : ppw) * 2 * G->nmat * nmax * G->mp +
                  (size_t)ppw * (np + std::max<size_t>(np, !terms ? 0 : D == 2 ? 2 * (n0 + n1) : 2 * (n1 * n2 + n0 * n2 + n0 * n1))));
  };
  G->px = n0 | 1;
  G->mp = (nmax + 3) / 4 * 4;
  G->vec = true;
  if (bytes() > 65536) {  // large patches: unpadded
    G->px = n0;
    G->mp = nmax;
    G->vec = nmax % 4 == 0;
  }
  G->d0 = FastDiv(n0);
  G->d1 = FastDiv(n1);
  const int nn[3] = { n0, n1, n2 };
  for (int a = 0; a < 3; a++) {
    G->na[a] = FastDiv(nn[a]);
    G->lines[a] = FastDiv(N / nn[a]);
  }
  return bytes();
}

inline int patch_cells(const te_domain* d) { return d->ns[0] * d->ns[1] * (d->dim == 3 ? d->ns[2] : 1); }

// patches per workgroup and threads per patch: the autotuner's choice for this shape, or (variant
// 0) a thread per four outputs of a transform, in powers of two from 32 to 256 threads (up to one
// per cell while the level does not fill the CUs with 512 threads each), and as many patches as
// make 256 threads and at most 48 KB of LDS.  The sweep at 256 / 512 / 1,024 threads a CU: 512
// patches of 6^3 in FP32 9.9 / 7.5 / 7.5 us, 4,096 of 10^2 in FP64 9.9 / 9.9 / 11.7
DftGenericVariant dft_shape(const te_dft_plan* pl, size_t esz, bool terms)
{
  const te_domain* d = pl->g->d;
  const int v = tune_variant(TUNE_DFT_GENERIC, d->dim, d->ns[0], esz == 8 ? TE_F64 : TE_F32);
  if (v != 0) return dft_generic_variant(v);
  const int N = patch_cells(d);
  DftGenericVariant w{ 1, 32 };
  while (w.tpp < 256 && (w.tpp * 4 < N || (w.tpp < N && (long)d->np * w.tpp < 512 * cu_count()))) w.tpp *= 2;
  DftGeom G;
  for (w.ppw = 256 / w.tpp; w.ppw > 1 && dft_geom(pl, esz, w.ppw, terms, &G) > 49152; w.ppw /= 2) {
  }
  return w;
}

// The same solve for 3D patches of 16^3 cells on the matrix cores.  Every axis transform is a
// chain of 16x16x4 MFMAs with the transform matrices in registers: per z-slice the x product's
// accumulator is the y product's operand (with a matching K order), the patch crosses LDS once
// to the z products (per y-row: forward, eigenvalues, inverse, chained through registers) and
// once back to the inverse y-x chain.  Wave w owns the slices (then rows) w, w + 4, w + 8,
// w + 12; in a slice lane l = c + 16 g holds the cells x = 4g .. 4g + 3 of row y = c.  The loads
// of a batch of slices (f, and at the faces the ghost and boundary values of u) are issued
// before its first product: 2 slices in FP32, 1 in FP64 (registers).
// Latency-bound on small levels (one patch a CU): 8 patches in FP32 take 6.4 us where one LDS
// round trip per axis (six, with barriers between) took 20.6; on large ones bound by memory:
// 2,535 patches 43 us (the vectors' padded lines in 36 at a copy's rate) against 95.
// FILL: the ghosts of u's faces are formed here (face_ghost3, one of the 256 cells of each face
// a thread, into LDS) instead of read from u; out may not be u then, since other patches' ghosts
// are formed from it.  A cycle's sweep with its ghosts on 2,535 patches: 53 us against 28 + 43 apart.
constexpr int k3N = 16, k3Row = 20, k3Slice = 16 * k3Row + 4, k3Slab = 16 * k3Slice;

template <typename T, typename TF, typename TO, int OP, bool UZERO, bool FILL>
__global__ void __launch_bounds__(256) dft3_mfma_kernel(const DevPatch* __restrict__ dp, const int* __restrict__ ptype,
                                                        const T* __restrict__ mats, const T* __restrict__ s2tab,
                                                        const TF* __restrict__ f, const T* u,
                                                        const T* __restrict__ coeffs, TO* out, Layout L,
                                                        bool zero_ghosts)
{
  __shared__ __align__(16) T slab[k3Slab];
  __shared__ T ghost[FILL ? 6 : 1][FILL ? k3N * k3N : 1];
  typedef typename Mf<T>::V V;
  constexpr int SB = sizeof(T) == 4 ? 2 : 1;
  const int p = FILL ? xcd_item(blockIdx.x, gridDim.x) : blockIdx.x;
  if (p >= L.np) return;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int* pt = ptype + p * 8;  // fwd type per axis [0..2], eig type per axis [3..5], zero mode [6]
  const DevPatch& P = dp[p];
  const int row0 = p * L.ps + (c + 1) * L.sx + 4 * g + 1;  // the lane's cells in slice z: row0 + (z + 1) * sy
  T F[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++) load_row4(f, row0 + (w + 4 * i + 1) * L.sy, F[i]);
  if (FILL) {
    const int i = threadIdx.x & 15, j = threadIdx.x >> 4;
    T G[6];
#pragma unroll
    for (int s = 0; s < 6; s++)
      G[s] = P.type[20 + s] < 0 ? T(0) : face_ghost3<T>(L, P.type[20 + s], P.orth[20 + s], P.nbr[20 + s], u, p, 0, s, i, j);
#pragma unroll
    for (int s = 0; s < 6; s++) ghost[FILL ? s : 0][FILL ? threadIdx.x : 0] = G[s];
  }
  // the transform matrices M[i][j] (y_i = sum_j M[i][j] x_j) as MFMA operands: lane (c, g), step
  // s holds M[c][K], K the product's K order (4g + s from memory, Mf<T>::row from an accumulator)
  auto mat = [&](int t, int a, int i, int j) { return mats[(t * 3 + a) * kDftMatStride + i * k3N + j]; };
  T SxB[4], SyA[4], SzA[4], SziA[4], SxiB[4], SyiA[4];
  int tf[3], ti[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    tf[a] = pt[a];
    ti[a] = tf[a] == 0 ? 1 : (tf[a] == 3 ? 4 : tf[a]);  // DCT_II->DCT_III, DST_II->DST_III, IV types self-inverse
  }
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int k1 = 4 * g + s, k2 = Mf<T>::row(s, g);
    SxB[s] = mat(tf[0], 0, c, k1);
    SyA[s] = mat(tf[1], 1, c, k2);
    SzA[s] = mat(tf[2], 2, c, k1);
    SziA[s] = mat(ti[2], 2, c, k2);
    SxiB[s] = mat(ti[0], 0, c, k1);
    SyiA[s] = mat(ti[1], 1, c, k2);
  }
  if (UZERO && zero_ghosts)  // 16-byte stores; the patch's results follow after the barriers
    for (int k = threadIdx.x; k < 18 * 18 * 18 * (int)sizeof(TO) / 16; k += 256)
      reinterpret_cast<float4*>(out + p * L.ps)[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  // f_copy = f, then modifyRHSForInternalBoundaryConditions (Poisson :165-180, VarPoisson
  // :168-186), sides in the reference's order
  bool has[6];
#pragma unroll
  for (int s = 0; s < 6; s++) has[s] = P.type[20 + s] >= 0;
  const bool onx = (g == 0 && has[0]) || (g == 3 && has[1]);
  const bool ony = (c == 0 && has[2]) || (c == k3N - 1 && has[3]);
  const T ih[3] = { T(P.inv_h2[0]), T(P.inv_h2[1]), T(P.inv_h2[2]) };
  // the values of v on a face of the lane's cells: x its one boundary cell and the ghost, y and z
  // the row of four and the ghosts over it
  struct Face {
    T xb, xg, b[4], y[4], z[4];
  };
  // (own: u's, whose ghosts are in LDS with FILL)
  auto faces = [&](const T* v, int z, bool own, Face& q) {
    const int r = row0 + (z + 1) * L.sy;
    const bool onz = (z == 0 && has[4]) || (z == k3N - 1 && has[5]), lds = FILL && own;
    if (onx) {
      q.xb = at(v, g == 0 ? r : r + 3);
      q.xg = lds ? ghost[g == 0 ? 0 : (FILL ? 1 : 0)][FILL ? c + 16 * z : 0] : at(v, g == 0 ? r - 1 : r + 4);
    }
    if (ony || onz) load_row4(v, r, q.b);
    if (lds) {
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if (ony) q.y[k] = ghost[FILL ? (c == 0 ? 2 : 3) : 0][FILL ? 4 * g + k + 16 * z : 0];
        if (onz) q.z[k] = ghost[FILL ? (z == 0 ? 4 : 5) : 0][FILL ? 4 * g + k + 16 * c : 0];
      }
    } else {
      if (ony) load_row4(v, c == 0 ? r - L.sx : r + L.sx, q.y);
      if (onz) load_row4(v, z == 0 ? r - L.sy : r + L.sy, q.z);
    }
  };
  if (FILL) __syncthreads();
#pragma unroll
  for (int i0 = 0; i0 < 4; i0 += SB) {
    Face q[SB], cq[OP == 1 ? SB : 1];
    if (!UZERO) {
#pragma unroll
      for (int j = 0; j < SB; j++) {
        faces(u, w + 4 * (i0 + j), true, q[j]);
        if (OP == 1) faces(coeffs, w + 4 * (i0 + j), false, cq[OP == 1 ? j : 0]);
      }
    }
#pragma unroll
    for (int j = 0; j < SB; j++) {
      const int z = w + 4 * (i0 + j);
      T(&Fz)[4] = F[i0 + j];
      if (!UZERO) {
        const Face& Q = q[j];
        const Face& C = cq[OP == 1 ? j : 0];
        auto sub = [&](T& v, T ug, T ub, T cg, T cb, T h) {
          if (OP == 0) v -= (ug + ub) * h;
          else v -= (ug + ub) * (cb + cg) * (h * T(0.5));
        };
        if (g == 0 && has[0]) sub(Fz[0], Q.xg, Q.xb, C.xg, C.xb, ih[0]);
        if (g == 3 && has[1]) sub(Fz[3], Q.xg, Q.xb, C.xg, C.xb, ih[0]);
        if (ony) {
#pragma unroll
          for (int k = 0; k < 4; k++) sub(Fz[k], Q.y[k], Q.b[k], C.y[k], C.b[k], ih[1]);
        }
        if ((z == 0 && has[4]) || (z == k3N - 1 && has[5])) {
#pragma unroll
          for (int k = 0; k < 4; k++) sub(Fz[k], Q.z[k], Q.b[k], C.z[k], C.b[k], ih[2]);
        }
      }
      V d1 = { 0, 0, 0, 0 };  // D1[y][kx] = sum_x F[y][x] Sx[kx][x]
#pragma unroll
      for (int s = 0; s < 4; s++) d1 = Mf<T>::mma(Fz[s], SxB[s], d1);
      V d2 = { 0, 0, 0, 0 };  // D2[ky][kx] = sum_y Sy[ky][y] D1[y][kx]
#pragma unroll
      for (int s = 0; s < 4; s++) d2 = Mf<T>::mma(SyA[s], d1[s], d2);
#pragma unroll
      for (int r = 0; r < 4; r++) slab[z * k3Slice + Mf<T>::row(r, g) * k3Row + c] = d2[r];
    }
  }
  __syncthreads();
  const T lx = T(4.0 / (P.h[0] * P.h[0])), ly = T(4.0 / (P.h[1] * P.h[1])), lz = T(4.0 / (P.h[2] * P.h[2]));
  const T s2x = s2tab[(pt[3] * 3 + 0) * kDftMatDim + c];
  T s2z[4];
#pragma unroll
  for (int r = 0; r < 4; r++) s2z[r] = s2tab[(pt[5] * 3 + 2) * kDftMatDim + Mf<T>::row(r, g)];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int ky = w + 4 * i;
    V b = { 0, 0, 0, 0 };  // W[kz][kx] = sum_z Sz[kz][z] D2[z][ky][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) b = Mf<T>::mma(SzA[s], slab[(4 * g + s) * k3Slice + ky * k3Row + c], b);
    const T s2y = s2tab[(pt[4] * 3 + 1) * kDftMatDim + ky];
#pragma unroll
    for (int r = 0; r < 4; r++) {  // divide by the eigenvalues (:320-361)
      T eig = T(0);
      eig -= lx * s2x;
      eig -= ly * s2y;
      eig -= lz * s2z[r];
      b[r] = b[r] / eig;
      // all-Neumann patch without neighbours (:438-440)
      if (pt[6] && ky == 0 && c == 0 && Mf<T>::row(r, g) == 0) b[r] = T(0);
    }
    V b2 = { 0, 0, 0, 0 };  // W'[z][kx] = sum_kz Szi[z][kz] W[kz][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) b2 = Mf<T>::mma(SziA[s], b[s], b2);
#pragma unroll
    for (int r = 0; r < 4; r++) slab[Mf<T>::row(r, g) * k3Slice + ky * k3Row + c] = b2[r];
  }
  __syncthreads();
  const T scale = T(2.0) / T(16) * (T(2.0) / T(16)) * (T(2.0) / T(16));
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int z = w + 4 * i;
    V r1 = { 0, 0, 0, 0 };  // R[ky][x] = sum_kx Q[ky][kx] Sxi[x][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) r1 = Mf<T>::mma(slab[z * k3Slice + c * k3Row + 4 * g + s], SxiB[s], r1);
    V u2 = { 0, 0, 0, 0 };  // U[y][x] = sum_ky Syi[y][ky] R[ky][x]
#pragma unroll
    for (int s = 0; s < 4; s++) u2 = Mf<T>::mma(SyiA[s], r1[s], u2);
#pragma unroll
    for (int r = 0; r < 4; r++)
      at(out, p * L.ps + (z + 1) * L.sy + (Mf<T>::row(r, g) + 1) * L.sx + c + 1) = TO(u2[r] * scale);
  }
}

// The same solve for 3D patches of 8^3 cells, one wavefront per patch (four to a workgroup) and
// no workgroup barrier.  A 16 x 16 product takes four 8 x 8 planes at once, arranged 2 x 2, with
// the axis matrix twice on the diagonal (half the matrix work is on zeros; it stays far below the
// loads): the x and y products on four z-slices, the z products on the (z, x) planes of four
// y-rows.  Chained through registers like dft3_mfma_kernel, with one crossing of the wave's own
// LDS to the z products and one back, on pitches that spread each access over all banks.
// Plane q = (column half) + 2 (row half) of tile t is slice (or row) 4t + q.
// Latency of loads and LDS; 4,096 patches in FP32: 11.1 us from zero and 12.6 with interface
// terms, where one 128-thread group per patch with dense products in VALU took 40 and 47.
// FILL: as in dft3_mfma_kernel, one of the 64 cells of each face a lane.
constexpr int k3Pitch8 = 72, k3Slab8 = 8 * k3Pitch8;  // words of a slice, of the patch

template <typename T, typename TF, typename TO, int OP, bool UZERO, bool FILL>
__global__ void __launch_bounds__(256) dft3_tile8_kernel(const DevPatch* __restrict__ dp, const int* __restrict__ ptype,
                                                         const T* __restrict__ mats, const T* __restrict__ s2tab,
                                                         const TF* __restrict__ f, const T* u,
                                                         const T* __restrict__ coeffs, TO* out, Layout L,
                                                         bool zero_ghosts)
{
  constexpr int SX = 10, SY = 100, PS = 1000;
  __shared__ T slabs[4 * k3Slab8];
  __shared__ T ghosts[FILL ? 4 * 6 * 64 : 1];
  typedef typename Mf<T>::V V;
  const int p = __builtin_amdgcn_readfirstlane((FILL ? xcd_item(blockIdx.x, gridDim.x) : blockIdx.x) * 4 +
                                               (threadIdx.x >> 6));
  if (p >= L.np) return;
  T* ghost = ghosts + (FILL ? (threadIdx.x >> 6) * 6 * 64 : 0);
  T* slab = slabs + (threadIdx.x >> 6) * k3Slab8;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int* pt = ptype + p * 8;  // fwd type per axis [0..2], eig type per axis [3..5], zero mode [6]
  const DevPatch& P = dp[p];
  // as an operand lane (c, g) holds four cells x = 4 (g & 1) ... of row y = c & 7 in plane qa; in an
  // accumulator register r is row Mf::row(r, g) and column c of the tile
  const int y = c & 7, xlow = 4 * (g & 1), qa = (g >> 1) + 2 * (c >> 3);
  const int row0 = p * PS + (y + 1) * SX + xlow + 1;
  T F[2][4];
#pragma unroll
  for (int t = 0; t < 2; t++) load_row4(f, row0 + (4 * t + qa + 1) * SY, F[t]);
  int tf[3], ti[3];
#pragma unroll
  for (int a = 0; a < 3; a++) {
    tf[a] = pt[a];
    ti[a] = tf[a] == 0 ? 1 : (tf[a] == 3 ? 4 : tf[a]);  // DCT_II->DCT_III, DST_II->DST_III, IV types self-inverse
  }
  if (FILL) {
    T G[6];
#pragma unroll
    for (int s = 0; s < 6; s++)
      G[s] = P.type[20 + s] < 0
               ? T(0)
               : face_ghost3<T>(L, P.type[20 + s], P.orth[20 + s], P.nbr[20 + s], u, p, 0, s, lane & 7, lane >> 3);
#pragma unroll
    for (int s = 0; s < 6; s++) ghost[FILL ? s * 64 + lane : 0] = G[s];
    wave_sync();
  }
  // element (i, j) of the doubled matrix of axis a
  auto mat = [&](int t, int a, int i, int j) {
    const T m = mats[(t * 3 + a) * kDftMatStride + (i & 7) * 8 + (j & 7)];
    return (i ^ j) & 8 ? T(0) : m;
  };
  T SxB[4], SyA[4], SzA[4], SziA[4], SxiB[4], SyiA[4];
#pragma unroll
  for (int s = 0; s < 4; s++) {
    const int k1 = 4 * g + s, k2 = Mf<T>::row(s, g);
    SxB[s] = mat(tf[0], 0, c, k1);
    SyA[s] = mat(tf[1], 1, c, k2);
    SzA[s] = mat(tf[2], 2, c, k1);
    SziA[s] = mat(ti[2], 2, c, k2);
    SxiB[s] = mat(ti[0], 0, c, k1);
    SyiA[s] = mat(ti[1], 1, c, k2);
  }
  if (UZERO && zero_ghosts)  // 16-byte stores; the patch's results follow below
    for (int k = lane; k < PS * (int)sizeof(TO) / 16; k += 64)
      reinterpret_cast<float4*>(out + p * PS)[k] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (!UZERO) {
    // modifyRHSForInternalBoundaryConditions (Poisson :165-180, VarPoisson :168-186), sides in the
    // reference's order; every lane has one cell on an x face
    bool has[6];
    T ih[3];
#pragma unroll
    for (int s = 0; s < 6; s++) has[s] = P.type[20 + s] >= 0;
#pragma unroll
    for (int a = 0; a < 3; a++) ih[a] = T(P.inv_h2[a]);
    const int xc = xlow ? 3 : 0;  // the lane's cell on its x face
    const bool onx = xlow ? has[1] : has[0], ony = (y == 0 && has[2]) || (y == 7 && has[3]);
    struct Face {
      T xb, xg, b[4], y[4], z[4];
    };
    auto faces = [&](const T* v, int z, bool own, Face& q) {
      const int r = row0 + (z + 1) * SY;
      const bool onz = (z == 0 && has[4]) || (z == 7 && has[5]), lds = FILL && own;
      if (onx) {
        q.xb = at(v, r + xc);
        q.xg = lds ? ghost[FILL ? (xlow ? 64 : 0) + y + 8 * z : 0] : at(v, xlow ? r + 4 : r - 1);
      }
      if (ony || onz) load_row4(v, r, q.b);
      if (lds) {
#pragma unroll
        for (int k = 0; k < 4; k++) {
          if (ony) q.y[k] = ghost[FILL ? (y == 0 ? 2 : 3) * 64 + xlow + k + 8 * z : 0];
          if (onz) q.z[k] = ghost[FILL ? (z == 0 ? 4 : 5) * 64 + xlow + k + 8 * y : 0];
        }
      } else {
        if (ony) load_row4(v, y == 0 ? r - SX : r + SX, q.y);
        if (onz) load_row4(v, z == 0 ? r - SY : r + SY, q.z);
      }
    };
    Face q[2], cq[OP == 1 ? 2 : 1];
#pragma unroll
    for (int t = 0; t < 2; t++) {
      faces(u, 4 * t + qa, true, q[t]);
      if (OP == 1) faces(coeffs, 4 * t + qa, false, cq[OP == 1 ? t : 0]);
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
      const int z = 4 * t + qa;
      const Face& Q = q[t];
      const Face& C = cq[OP == 1 ? t : 0];
      auto sub = [&](T& v, T ug, T ub, T cg, T cb, T h) {
        if (OP == 0) v -= (ug + ub) * h;
        else v -= (ug + ub) * (cb + cg) * (h * T(0.5));
      };
      if (onx && !xlow) sub(F[t][0], Q.xg, Q.xb, C.xg, C.xb, ih[0]);
      if (onx && xlow) sub(F[t][3], Q.xg, Q.xb, C.xg, C.xb, ih[0]);
      if (ony) {
#pragma unroll
        for (int k = 0; k < 4; k++) sub(F[t][k], Q.y[k], Q.b[k], C.y[k], C.b[k], ih[1]);
      }
      if ((z == 0 && has[4]) || (z == 7 && has[5])) {
#pragma unroll
        for (int k = 0; k < 4; k++) sub(F[t][k], Q.z[k], Q.b[k], C.z[k], C.b[k], ih[2]);
      }
    }
  }
  // the place of accumulator register r of tile t: its plane's row and column, and the plane
  auto arow = [&](int r) { return Mf<T>::row(r, g) & 7; };
  auto aplane = [&](int t, int r) { return 4 * t + (c >> 3) + 2 * (Mf<T>::row(r, g) >> 3); };
#pragma unroll
  for (int t = 0; t < 2; t++) {
    V d1 = { 0, 0, 0, 0 };  // D1[y][kx] = sum_x F[y][x] Sx[kx][x]
#pragma unroll
    for (int s = 0; s < 4; s++) d1 = Mf<T>::mma(F[t][s], SxB[s], d1);
    V d2 = { 0, 0, 0, 0 };  // D2[ky][kx] = sum_y Sy[ky][y] D1[y][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) d2 = Mf<T>::mma(SyA[s], d1[s], d2);
#pragma unroll
    for (int r = 0; r < 4; r++) slab[aplane(t, r) * k3Pitch8 + arow(r) * 8 + (c & 7)] = d2[r];
  }
  wave_sync();
  const T lx = T(4.0 / (P.h[0] * P.h[0])), ly = T(4.0 / (P.h[1] * P.h[1])), lz = T(4.0 / (P.h[2] * P.h[2]));
  const T s2x = s2tab[(pt[3] * 3 + 0) * kDftMatDim + (c & 7)];
  V wz[2];
#pragma unroll
  for (int t = 0; t < 2; t++) {
    V b = { 0, 0, 0, 0 };  // W[kz][kx] = sum_z Sz[kz][z] D2[z][ky][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const int z = (4 * g + s) & 7, ky = 4 * t + (c >> 3) + 2 * (g >> 1);
      b = Mf<T>::mma(SzA[s], slab[z * k3Pitch8 + ky * 8 + (c & 7)], b);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {  // divide by the eigenvalues (:320-361)
      const int kz = arow(r), ky = aplane(t, r);
      T eig = T(0);
      eig -= lx * s2x;
      eig -= ly * s2tab[(pt[4] * 3 + 1) * kDftMatDim + ky];
      eig -= lz * s2tab[(pt[5] * 3 + 2) * kDftMatDim + kz];
      b[r] = b[r] / eig;
      // all-Neumann patch without neighbours (:438-440)
      if (pt[6] && ky == 0 && kz == 0 && (c & 7) == 0) b[r] = T(0);
    }
    V b2 = { 0, 0, 0, 0 };  // W'[z][kx] = sum_kz Szi[z][kz] W[kz][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) b2 = Mf<T>::mma(SziA[s], b[s], b2);
    wz[t] = b2;
  }
  wave_sync();
#pragma unroll
  for (int t = 0; t < 2; t++)
#pragma unroll
    for (int r = 0; r < 4; r++) slab[arow(r) * k3Pitch8 + aplane(t, r) * 8 + (c & 7)] = wz[t][r];
  wave_sync();
  if (UZERO && zero_ghosts) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
  const T scale = T(2.0) / T(8) * (T(2.0) / T(8)) * (T(2.0) / T(8));
#pragma unroll
  for (int t = 0; t < 2; t++) {
    V r1 = { 0, 0, 0, 0 };  // R[ky][x] = sum_kx Q[ky][kx] Sxi[x][kx]
#pragma unroll
    for (int s = 0; s < 4; s++) r1 = Mf<T>::mma(slab[(4 * t + qa) * k3Pitch8 + y * 8 + xlow + s], SxiB[s], r1);
    V u2 = { 0, 0, 0, 0 };  // U[y][x] = sum_ky Syi[y][ky] R[ky][x]
#pragma unroll
    for (int s = 0; s < 4; s++) u2 = Mf<T>::mma(SyiA[s], r1[s], u2);
#pragma unroll
    for (int r = 0; r < 4; r++)
      at(out, p * PS + (aplane(t, r) + 1) * SY + (arow(r) + 1) * SX + (c & 7) + 1) = TO(u2[r] * scale);
  }
}

template <typename T, typename TF, typename TO, int D>
void launch_d(const te_dft_plan* pl, const TF* f, const T* u, TO* out, bool uzero, bool zg, bool fill,
              hipStream_t s)
{
  const te_domain* d = pl->g->d;
  Layout L = make_layout(d->dim, d->ns, 1, d->np);
  const T* mats = (const T*)(sizeof(T) == 8 ? (const void*)pl->d_mats64 : (const void*)pl->d_mats32);
  const T* s2 = (const T*)(sizeof(T) == 8 ? (const void*)pl->d_s2_64 : (const void*)pl->d_s2_32);
  const T* cf = (const T*)(sizeof(T) == 8 ? (const void*)pl->d_coeffs64 : (const void*)pl->d_coeffs32);
  if (D == 3 && dft3_mfma_supported(pl)) {
    const bool big = d->ns[0] == 16;
    const int groups = big ? d->np : (d->np + 3) / 4, grid = fill && !uzero ? xcd_grid(groups) : groups;
#define TE_D3(OP_, UZ_, F_)                                                                                         \
  do {                                                                                                              \
    if (big)                                                                                                        \
      hipLaunchKernelGGL((dft3_mfma_kernel<T, TF, TO, OP_, UZ_, F_>), dim3(grid), dim3(256), 0, s, d->d_patches,    \
                         pl->d_ptype, mats, s2, f, u, cf, out, L, zg);                                              \
    else                                                                                                            \
      hipLaunchKernelGGL((dft3_tile8_kernel<T, TF, TO, OP_, UZ_, F_>), dim3(grid), dim3(256), 0, s, d->d_patches,   \
                         pl->d_ptype, mats, s2, f, u, cf, out, L, zg);                                              \
  } while (0)
#define TE_D3O(OP_)                        \
  do {                                     \
    if (uzero) TE_D3(OP_, true, false);    \
    else if (fill) TE_D3(OP_, false, true); \
    else TE_D3(OP_, false, false);         \
  } while (0)
    if (pl->op_kind == 0) TE_D3O(0);
    else TE_D3O(1);
#undef TE_D3O
#undef TE_D3
    return;
  }
  const DftGenericVariant v = dft_shape(pl, sizeof(T), !uzero);
  DftGeom G;
  const size_t shmem = dft_geom(pl, sizeof(T), v.ppw, !uzero, &G);
  G.one = patch_cells(d) <= v.tpp;
  const int grid = (d->np + v.ppw - 1) / v.ppw;
  const FusedArgs<T, T> fa{ nullptr, nullptr, nullptr };
#define TE_DL(OP_, UZ_)                                                                                          \
  hipLaunchKernelGGL((dft_kernel<T, TF, TO, D, OP_, UZ_>), dim3(grid), dim3(v.ppw * v.tpp), shmem, s,          \
                     d->d_patches, pl->d_ptype, mats, s2, f, u, cf, out, L, v.ppw, fa, nullptr, G, zg)
  if (pl->op_kind == 0) {
    if (uzero) TE_DL(0, true); else TE_DL(0, false);
  } else {
    if (uzero) TE_DL(1, true); else TE_DL(1, false);
  }
#undef TE_DL
}

template <typename T, typename TF, typename TO>
void launch_t(const te_dft_plan* pl, const void* f, const void* u, void* out, bool uzero, bool zg,
              bool fill, hipStream_t s)
{
  if (pl->g->d->dim == 2) launch_d<T, TF, TO, 2>(pl, (const TF*)f, (const T*)u, (TO*)out, uzero, zg, fill, s);
  else launch_d<T, TF, TO, 3>(pl, (const TF*)f, (const T*)u, (TO*)out, uzero, zg, fill, s);
}

// the fused sweeps of the generic kernel, 2D: gm 0 (ghosts read from u), 1 (computed here),
// 2 (computed here on u + P uc)
template <typename T, typename TF, typename TO, typename TC>
void launch_fused_t(const te_dft_plan* pl, const void* fv, const void* uv, void* outv, bool uzero, int gm,
                    const void* ucv, const te_level_link* link, hipStream_t s)
{
  const te_domain* d = pl->g->d;
  Layout L = make_layout(2, d->ns, 1, d->np);
  const T* mats = (const T*)(sizeof(T) == 8 ? (const void*)pl->d_mats64 : (const void*)pl->d_mats32);
  const T* s2 = (const T*)(sizeof(T) == 8 ? (const void*)pl->d_s2_64 : (const void*)pl->d_s2_32);
  const T* cf = (const T*)(sizeof(T) == 8 ? (const void*)pl->d_coeffs64 : (const void*)pl->d_coeffs32);
  const DftGenericVariant v = dft_shape(pl, sizeof(T), !uzero);
  DftGeom G;
  const size_t shmem = dft_geom(pl, sizeof(T), v.ppw, !uzero, &G);
  G.one = patch_cells(d) <= v.tpp;
  const int grid = (d->np + v.ppw - 1) / v.ppw;
  const int4* ring = (const int4*)(gm == 2 ? link->d_ring : d->d_ring);
  const FusedArgs<T, TC> fa{ (const TC*)ucv, link ? link->d_parent : nullptr, link ? link->d_orth : nullptr };
  const TF* f = (const TF*)fv;
  const T* u = (const T*)uv;
  TO* out = (TO*)outv;
  const int kind = pl->g->kind;
#define TE_DF(OP_, UZ_, GM_, K_)                                                                                 \
  hipLaunchKernelGGL((dft_kernel<T, TF, TO, 2, OP_, UZ_, GM_, K_, TC>), dim3(grid), dim3(v.ppw * v.tpp), shmem, \
                     s, d->d_patches, pl->d_ptype, mats, s2, f, u, cf, out, L, v.ppw, fa, ring, G, false)
#define TE_DFO(OP_)                                                        \
  do {                                                                     \
    if (uzero) TE_DF(OP_, true, 0, 0);                                     \
    else if (gm == 0) TE_DF(OP_, false, 0, 0);                             \
    else if (gm == 1 && kind == TE_BILINEAR) TE_DF(OP_, false, 1, TE_BILINEAR); \
    else if (gm == 1) TE_DF(OP_, false, 1, TE_BIQUADRATIC);                \
    else if (kind == TE_BILINEAR) TE_DF(OP_, false, 2, TE_BILINEAR);       \
    else TE_DF(OP_, false, 2, TE_BIQUADRATIC);                             \
  } while (0)
  if (pl->op_kind == 0) TE_DFO(0);
  else TE_DFO(1);
#undef TE_DFO
#undef TE_DF
}

}  // namespace

bool dft_generic_fused_supported(const te_dft_plan* pl)
{
  const te_domain* d = pl->g->d;
  return d->dim == 2 && d->ns[0] % 2 == 0 && d->ns[1] % 2 == 0 &&
         (pl->g->kind == TE_BILINEAR || pl->g->kind == TE_BIQUADRATIC);
}

int launch_dft_fused(const te_dft_plan* pl, int dt, int dtf, int dto, const void* f, const void* u, void* out,
                     bool uzero, int gm, int dtc, const void* uc, const te_level_link* link, hipStream_t s)
{
  if (pl->use_mfma && dft_mfma_supported(pl))
    return launch_dft_mfma_fused(pl, dt, dtf, dto, f, u, out, uzero, gm, dtc, uc, link, s);
  if (pl->g->d->np == 0) return TE_OK;
  if (!dft_generic_fused_supported(pl)) {
    set_error("fused DFT sweep: needs 2D, even cells per side, BiLinear or BiQuadratic ghosts");
    return TE_ERR_UNSUPPORTED;
  }
  if (gm == 2 && (!uc || !link)) {
    set_error("fused interpolation needs the coarser level's u and the level link");
    return TE_ERR_ARG;
  }
  if (gm != 0 && !uzero && out == u) {
    set_error("internal: a fused sweep that computes ghosts must not write its input");
    return TE_ERR_ARG;
  }
  const bool c64 = gm != 2 || dtc == TE_F64;
#define TE_LF(T_, TF_, TO_)                                                                      \
  do {                                                                                           \
    if (c64) launch_fused_t<T_, TF_, TO_, double>(pl, f, u, out, uzero, gm, uc, link, s);        \
    else launch_fused_t<T_, TF_, TO_, float>(pl, f, u, out, uzero, gm, uc, link, s);             \
  } while (0)
  if (dt == TE_F64 && dtf == TE_F64 && dto == TE_F64) {
    if (!c64) {
      set_error("FP64 level with an FP32 coarser level is not supported");
      return TE_ERR_UNSUPPORTED;
    }
    launch_fused_t<double, double, double, double>(pl, f, u, out, uzero, gm, uc, link, s);
  } else if (dt == TE_F32 && dtf == TE_F32 && dto == TE_F32) {
    TE_LF(float, float, float);
  } else if (dt == TE_F32 && dtf == TE_F64 && dto == TE_F32) {
    TE_LF(float, double, float);
  } else if (dt == TE_F32 && dtf == TE_F64 && dto == TE_F64) {
    TE_LF(float, double, double);
  } else if (dt == TE_F32 && dtf == TE_F32 && dto == TE_F64) {
    TE_LF(float, float, double);
  } else {
    set_error("unsupported dtype combination for the DFT patch solver");
    return TE_ERR_UNSUPPORTED;
  }
#undef TE_LF
  TE_HIP(hipGetLastError());
  return TE_OK;
}

bool dft3_mfma_supported(const te_dft_plan* pl)
{
  const te_domain* d = pl->g->d;
  return pl->use_mfma && d->dim == 3 && (d->ns[0] == 8 || d->ns[0] == 16) && d->ns[1] == d->ns[0] &&
         d->ns[2] == d->ns[0];
}

int launch_dft(const te_dft_plan* pl, int dt, int dtf, int dto, const void* f, const void* u, void* out, bool uzero,
               hipStream_t s, bool zero_ghosts, bool fill)
{
  const te_domain* d = pl->g->d;
  if (d->np == 0) return TE_OK;
  // the kernels of this file zero the ghosts themselves (the 3D matrix-core ones by 16-byte stores)
  const bool own = uzero && f != out &&
                   (dft3_mfma_supported(pl) ? (uintptr_t)out % 16 == 0 : !(pl->use_mfma && dft_mfma_supported(pl)));
  if (fill && !uzero && (!dft3_mfma_supported(pl) || out == u)) {
    set_error("internal: a 3D sweep that forms ghosts needs 8^3 or 16^3 patches and another buffer for its result");
    return TE_ERR_ARG;
  }
  const bool zg = zero_ghosts && own;
  if (zero_ghosts && !own) {
    int rc = launch_vec_op(d, dto, VOP_SET_WITH_GHOST, out, nullptr, nullptr, 0.0, 0, 0, 1, s);
    if (rc) return rc;
  }
  if (pl->use_mfma && dft_mfma_supported(pl)) return launch_dft_mfma(pl, dt, dtf, dto, f, u, out, uzero, s);
  if (dt == TE_F64 && dtf == TE_F64 && dto == TE_F64) launch_t<double, double, double>(pl, f, u, out, uzero, zg, fill, s);
  else if (dt == TE_F32 && dtf == TE_F32 && dto == TE_F32) launch_t<float, float, float>(pl, f, u, out, uzero, zg, fill, s);
  else if (dt == TE_F32 && dtf == TE_F64 && dto == TE_F32) launch_t<float, double, float>(pl, f, u, out, uzero, zg, fill, s);
  else if (dt == TE_F32 && dtf == TE_F64 && dto == TE_F64) launch_t<float, double, double>(pl, f, u, out, uzero, zg, fill, s);
  else {
    set_error("unsupported dtype combination for the DFT patch solver");
    return TE_ERR_UNSUPPORTED;
  }
  TE_HIP(hipGetLastError());
  return TE_OK;
}

}  // namespace te
