// Iterative::PatchSolver<D>(BiCGStab, op) smoothing sweep
// (Iterative/PatchSolver.h:134-175 inside PatchSolver::smooth, PatchSolver.h:142-170):
// every patch runs its own inner BiCGStab (Iterative/BiCGStab.h:111-203) on the
// single-patch operator with internal boundary conditions, started from the
// current u.  One workgroup per patch keeps the whole Krylov state on chip: each thread owns
// CPT cells of every Krylov vector in registers.  Patches iterate independently (per-patch
// termination), so a level is one launch.
//
// What bounds it: an iteration is a serial chain (operator, inner product, scalar, update,
// operator, ...) and moves no memory, so its length is latency.  Hence
//  - inner products sum across a wave with DPP moves (6 dependent adds, no LDS round trips),
//    then over the waves through double-buffered LDS slots with one barrier;
//  - three of them per iteration: s.s joins As.s and As.As (the s-norm test of
//    BiCGStab.h:162-167 is then made after As is known, with the same outcome), r.rhat joins r.r;
//  - the stopping tests compare squares and take the square root and the quotient only within
//    1e-7 of the limit (same decisions);
//  - square 2D patches of 8, 16 and 32 cells a side run patch_bicgstab_tile, whose threads own
//    strips of a column: x neighbours come from the adjacent lanes, y neighbours from registers,
//    only the strip ends cross LDS, and VarPoisson's face weights stay in registers; 8 and 16
//    are one wave without any barrier (wave_sync orders their LDS exchanges).  Every other shape runs patch_bicgstab_kernel, whose
//    operand passes through a padded LDS patch.
// Measured against one 256-thread workgroup per patch for every shape, with cross-lane shuffles,
// the operand in LDS and the cells' places worked out in every apply: 64 patches of 32^2 in FP64
// to 1e-12, two sweeps, 720 -> 319 us; a VarPoisson solve on 754 patches of 32^2 (7 levels, 280
// sweeps of at most 50 iterations, FP32) 51.2 -> 23.7 ms.  32^2 on 128 or 512 threads instead of
// 256: 1.1 to 1.3 times slower (more cells per thread; more waves to sum).
#include "../te_internal.h"
#include "blas.h"
#include "ghost2d.h"

namespace te {
namespace {

constexpr int kThreads = 256;

// v moved across lanes by a DPP control (0 in lanes without a source)
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ int dpp(int v)
{
  return __builtin_amdgcn_update_dpp(0, v, CTRL, ROWS, 0xf, ROWS == 0xf);
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp(float v)
{
  return __int_as_float(dpp<CTRL, ROWS>(__float_as_int(v)));
}
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp(double v)
{
  return __hiloint2double(dpp<CTRL, ROWS>(__double2hiint(v)), dpp<CTRL, ROWS>(__double2loint(v)));
}
constexpr int kRowShr = 0x110, kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShl1 = 0x130, kWaveShr1 = 0x138;

// the sum over the wave, valid in lane 63 (lanes without a source add 0)
__device__ __forceinline__ double wave_sum63(double v)
{
  v += dpp<kRowShr + 1>(v);
  v += dpp<kRowShr + 2>(v);
  v += dpp<kRowShr + 4>(v);
  v += dpp<kRowShr + 8>(v);
  v += dpp<kRowBcast15, 0xa>(v);
  v += dpp<kRowBcast31, 0xc>(v);
  return v;
}

// sums over the workgroup of NV values per thread, returned to every thread; `buf` alternates
// between the two halves of `red` from call to call, so that a call's writes cannot meet the
// previous call's reads and one barrier suffices (the one before it orders the call before).
// Every call orders the LDS accesses before it before those after it, in one wave too.
template <int NV, int NT>
__device__ __forceinline__ void wg_sums(double (&v)[NV], double (*red)[3 * (NT / 64)], int& buf)
{
  constexpr int W = NT / 64;
#pragma unroll
  for (int j = 0; j < NV; j++) v[j] = wave_sum63(v[j]);
  if (W == 1) {
#pragma unroll
    for (int j = 0; j < NV; j++)
      v[j] = __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v[j]), 63),
                              __builtin_amdgcn_readlane(__double2loint(v[j]), 63));
    wave_sync();
    return;
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  double* rb = red[buf];
  if (lane == 63)
#pragma unroll
    for (int j = 0; j < NV; j++) rb[j * W + w] = v[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NV; j++) {
    double r = rb[j * W];
#pragma unroll
    for (int k = 1; k < W; k++) r += rb[j * W + k];
    v[j] = r;
  }
  buf ^= 1;
}

// sqrt(n2) / r0 against tol: by squares where they are far enough apart that rounding cannot
// change the outcome, else as written (a NaN fails both tests)
struct Limit {
  double r0, tol, lo, hi;
  __device__ Limit(double r0_, double tol_) : r0(r0_), tol(tol_), lo(0.0), hi(0.0)
  {
    const double t2 = tol * r0 * (tol * r0);
    if (tol > 0.0 && t2 > 1e-280) {
      lo = t2 * (1.0 - 1e-7);
      hi = t2 * (1.0 + 1e-7);
    }
  }
  __device__ bool above(double n2) const
  {
    if (hi > 0.0 && n2 > hi) return true;
    if (hi > 0.0 && n2 < lo) return false;
    return sqrt(n2) / r0 > tol;
  }
  __device__ bool within(double n2) const
  {
    if (hi > 0.0 && n2 > hi) return false;
    if (hi > 0.0 && n2 < lo) return true;
    return sqrt(n2) / r0 <= tol;
  }
};

// BiCGStab::solve (Iterative/BiCGStab.h:111-203) on a thread's CPT cells of one patch: x from
// the initial guess to the solution for b.  `op` is the patch's operator, called by every
// thread of the workgroup: op.init(v, out) applies it, and op.ready<SET>(c, a) before a
// reduction with op.apply<SET>(v, m, out) after it applies it to v = c m + a, which lets the
// neighbours' values cross with the reduction's barrier (m, the reduction's result, is what
// they lack).  Cells that the thread does not own hold zeros, which the operator keeps.
template <typename T, int CPT, int NT, class Op>
__device__ __forceinline__ int patch_solve(T (&x)[CPT], const T (&b)[CPT], int max_it, double tol,
                                           double (*red)[3 * (NT / 64)], bool* broke, Op& op)
{
  T r[CPT], rhat[CPT], pv[CPT], ap[CPT], s[CPT], as[CPT];
  int rbuf = 0;
  op.init(x, r);
  double v3[3] = { 0.0, 0.0, 0.0 };
#pragma unroll
  for (int k = 0; k < CPT; k++) {
    r[k] = r[k] * T(-1) + b[k];
    rhat[k] = r[k];
    pv[k] = r[k];
    ap[k] = T(0);
    v3[0] += double(b[k]) * double(b[k]);
    v3[1] += double(r[k]) * double(r[k]);
  }
  op.template ready<1>(ap, r);  // p = r
  T pm = T(0);
  wg_sums<3, NT>(v3, red, rbuf);
  const double r0_norm = sqrt(v3[0]);
  double rho = v3[1], rr = v3[1];
  int its = 0;
  *broke = false;
  if (r0_norm == 0.0) return its;
  const Limit lim(r0_norm, tol);
  while (its < max_it && lim.above(rr)) {
    if (rho == 0.0) {
      *broke = true;
      break;
    }
    op.template apply<1>(pv, pm, ap);
    double v1[1] = { 0.0 };
#pragma unroll
    for (int k = 0; k < CPT; k++) v1[0] += double(rhat[k]) * double(ap[k]);
    op.template ready<0>(ap, r);
    wg_sums<1, NT>(v1, red, rbuf);
    const double alpha = rho / v1[0];
#pragma unroll
    for (int k = 0; k < CPT; k++) s[k] = r[k] + ap[k] * T(-alpha);
    op.template apply<0>(s, T(-alpha), as);
    v3[0] = v3[1] = v3[2] = 0.0;
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      v3[0] += double(as[k]) * double(s[k]);
      v3[1] += double(as[k]) * double(as[k]);
      v3[2] += double(s[k]) * double(s[k]);
    }
    wg_sums<3, NT>(v3, red, rbuf);
    if (lim.within(v3[2])) {
#pragma unroll
      for (int k = 0; k < CPT; k++) x[k] += pv[k] * T(alpha);
      break;
    }
    const double omega = v3[0] / v3[1];
    double v2[2] = { 0.0, 0.0 };
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      x[k] += pv[k] * T(alpha) + s[k] * T(omega);
      r[k] += ap[k] * T(-alpha) + as[k] * T(-omega);
      pv[k] += ap[k] * T(-omega);
      v2[0] += double(r[k]) * double(rhat[k]);
      v2[1] += double(r[k]) * double(r[k]);
    }
    op.template ready<1>(pv, r);
    wg_sums<2, NT>(v2, red, rbuf);
    const double beta = v2[0] * alpha / (rho * omega);
    pm = T(beta);
#pragma unroll
    for (int k = 0; k < CPT; k++) pv[k] = pv[k] * pm + r[k];
    its++;
    rho = v2[0];
    rr = v2[1];
  }
  return its;
}

// Square 2D patches of N1 cells a side: thread (x, strip) owns the CPT cells y = strip * CPT ...
// of column x.  x neighbours are the adjacent lanes (a row of cells is 8, 16 or 32 consecutive
// lanes), y neighbours the thread's own registers, and the cells at a strip's ends go through
// LDS.  The single-patch operator's side ghosts (Poisson/StarPatchOperator.h:75-101 with
// internal = true) are -interior, on physical Neumann sides +interior.
template <typename T, int OP, int N1, int NT>
struct TileOp {
  static constexpr int CPT = N1 * N1 / NT, S = N1 / CPT;
  // each strip's first and last row of the two vectors of a set (ready / apply)
  struct Edges {
    T first[2][S][N1], last[2][S][N1];
  };
  Edges* e;
  int x0, st;
  bool xl, xr, yl, yr;
  T sg[4];      // the sign of each side's ghost
  T ihx, ihy;
  T wl[OP == 1 ? CPT : 1], wr[OP == 1 ? CPT : 1], wy[OP == 1 ? CPT + 1 : 1];  // VarPoisson: face weights

  template <int SET>
  __device__ __forceinline__ void ready(const T (&c)[CPT], const T (&a)[CPT])
  {
    e[SET].first[0][st][x0] = c[0];
    e[SET].first[1][st][x0] = a[0];
    e[SET].last[0][st][x0] = c[CPT - 1];
    e[SET].last[1][st][x0] = a[CPT - 1];
  }
  __device__ __forceinline__ void init(const T (&v)[CPT], T (&out)[CPT])
  {
    T zero[CPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) zero[k] = T(0);
    ready<0>(zero, v);
    __syncthreads();
    apply<0>(v, T(0), out);
  }
  template <int SET>
  __device__ __forceinline__ void apply(const T (&v)[CPT], T m, T (&out)[CPT])
  {
    // the reads are issued unconditionally and waited for only where they are used
    const int sb = yl ? 0 : st - 1, sa = yr ? S - 1 : st + 1;
    const T bc = e[SET].last[0][sb][x0], ba = e[SET].last[1][sb][x0];
    const T ac = e[SET].first[0][sa][x0], aa = e[SET].first[1][sa][x0];
    T west[CPT], east[CPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      const T l = dpp<kWaveShr1>(v[k]), r = dpp<kWaveShl1>(v[k]);  // from lane - 1, lane + 1
      west[k] = xl ? sg[0] * v[k] : l;
      east[k] = xr ? sg[1] * v[k] : r;
    }
    T lower = yl ? sg[2] * v[0] : bc * m + ba;
    const T above = yr ? sg[3] * v[CPT - 1] : ac * m + aa;
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      const T mid = v[k];
      const T upper = k == CPT - 1 ? above : v[k + 1 < CPT ? k + 1 : k];
      if (OP == 0) {
        T acc = (east[k] - T(2) * mid + west[k]) * ihx;
        acc += (upper - T(2) * mid + lower) * ihy;
        out[k] = acc;
      } else {
        T acc = wr[k] * (east[k] - mid) - wl[k] * (mid - west[k]);
        acc += wy[k + 1] * (upper - mid) - wy[k] * (mid - lower);
        out[k] = acc;
      }
      lower = mid;
    }
  }
};

template <typename T, int OP, int N1, int NT>
__global__ void __launch_bounds__(NT) patch_bicgstab_tile(const DevPatch* __restrict__ dp, const T* __restrict__ coeffs,
                                                          const T* __restrict__ f, T* __restrict__ u, int neumann,
                                                          int max_it, double tol, int32_t* __restrict__ iters,
                                                          int32_t* __restrict__ breakdown)
{
  typedef TileOp<T, OP, N1, NT> Tile;
  constexpr int CPT = Tile::CPT, S = Tile::S, SX = N1 + 2, PS = SX * SX;
  __shared__ typename Tile::Edges edges[2];
  __shared__ double red[2][3 * (NT / 64)];
  const int p = blockIdx.x;
  const DevPatch& P = dp[p];
  const int x0 = threadIdx.x & (N1 - 1), st = threadIdx.x / N1;
  const bool xl = x0 == 0, xr = x0 == N1 - 1, yl = st == 0, yr = st == S - 1;
  const T ihx = T(P.inv_h2[0]), ihy = T(P.inv_h2[1]);
  Tile op{ edges, x0, st, xl, xr, yl, yr, {}, ihx, ihy, {}, {}, {} };
  bool nb[4];  // a patch lies across the side
#pragma unroll
  for (int s = 0; s < 4; s++) {
    nb[s] = P.type[4 + s] >= 0;
    op.sg[s] = (OP == 0 && neumann && !nb[s]) ? T(1) : T(-1);
  }
  const int base = p * PS + (st * CPT + 1) * SX + x0 + 1;

  // VarPoisson (VarPoisson/StarPatchOperator.h:61-109): the weight of each face, (c + c') / (2 h^2)
  if (OP == 1) {
    T below = at(coeffs, base - SX);
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      const int g = base + k * SX;
      const T c = at(coeffs, g);
      op.wl[k] = (at(coeffs, g - 1) + c) * (ihx * T(0.5));
      op.wr[k] = (at(coeffs, g + 1) + c) * (ihx * T(0.5));
      op.wy[k] = (below + c) * (ihy * T(0.5));
      below = c;
    }
    op.wy[CPT] = (below + at(coeffs, base + CPT * SX)) * (ihy * T(0.5));
  }

  // f_copy = f; modifyRHSForInternalBoundaryConditions (Poisson :165-180, VarPoisson :168-186)
  T x[CPT], b[CPT];
#pragma unroll
  for (int k = 0; k < CPT; k++) {
    const int g = base + k * SX;
    x[k] = u[g];
    b[k] = at(f, g);
  }
  auto side = [&](int k, int off, T w) { b[k] -= (u[base + k * SX + off] + x[k]) * w; };
#pragma unroll
  for (int k = 0; k < CPT; k++) {
    if (xl && nb[0]) side(k, -1, OP == 0 ? ihx : op.wl[OP == 1 ? k : 0]);
    if (xr && nb[1]) side(k, 1, OP == 0 ? ihx : op.wr[OP == 1 ? k : 0]);
  }
  if (yl && nb[2]) side(0, -SX, OP == 0 ? ihy : op.wy[0]);
  if (yr && nb[3]) side(CPT - 1, SX, OP == 0 ? ihy : op.wy[OP == 1 ? CPT : 0]);

  bool broke;
  const int its = patch_solve<T, CPT, NT>(x, b, max_it, tol, red, &broke, op);
#pragma unroll
  for (int k = 0; k < CPT; k++) u[base + k * SX] = x[k];
  if (threadIdx.x == 0) {
    if (iters) iters[p] = its;
    if (broke) breakdown[0] = 1;
  }
}

// an operator that stages its whole operand (patch_solve)
template <typename T, int CPT, class F>
struct StagedOp {
  F& f;
  __device__ __forceinline__ void init(const T (&v)[CPT], T (&out)[CPT]) { f(v, out); }
  template <int SET>
  __device__ __forceinline__ void ready(const T (&)[CPT], const T (&)[CPT])
  {
  }
  template <int SET>
  __device__ __forceinline__ void apply(const T (&v)[CPT], T, T (&out)[CPT])
  {
    f(v, out);
  }
};

// Any patch shape of at most 16 * 256 cells: thread t owns the cells t + k * NT (x fastest),
// the operand of an apply is staged in a padded LDS patch (VarPoisson: the coefficients too,
// once).  A cell's place in the patch and the sides it touches are worked out once (bit s:
// the cell lies on side s, bit 8 + s: its ghost there is +interior).
template <typename T, int D, int OP, int CPT, int NT>
__global__ void __launch_bounds__(NT) patch_bicgstab_kernel(
  const DevPatch* __restrict__ dp, const T* __restrict__ coeffs, const T* __restrict__ f, T* __restrict__ u,
  Layout L, int neumann, int max_it, double tol, int32_t* __restrict__ iters, int32_t* __restrict__ breakdown)
{
  extern __shared__ __align__(16) unsigned char smem_raw[];
  T* pad = reinterpret_cast<T*>(smem_raw);  // padded patch of the operand being applied
  T* cfl = pad + L.cs;                      // VarPoisson: the patch's coefficients (with ghosts)
  __shared__ double red[2][3 * (NT / 64)];
  const int p = blockIdx.x;
  const DevPatch& P = dp[p];
  const int n0 = L.n[0], n1 = L.n[1];
  const int N = n0 * n1 * (D == 3 ? L.n[2] : 1);
  const int st[3] = { 1, L.sx, L.sy };
  const int sb = D == 2 ? 4 : 20;
  T ih2[3];
#pragma unroll
  for (int a = 0; a < 3; a++) ih2[a] = T(P.inv_h2[a]);

  int gidx[CPT];  // index within the padded patch, -1: no cell
  int edge[CPT];
#pragma unroll
  for (int k = 0; k < CPT; k++) {
    const int o = threadIdx.x + k * NT;
    gidx[k] = -1;
    edge[k] = 0;
    if (o >= N) continue;
    const int yz = o / n0, z = D == 3 ? yz / n1 : 0;
    const int c3[3] = { o - yz * n0, yz - z * n1, z };
    gidx[k] = lin(L, 0, 0, c3[0], c3[1], c3[2]);
#pragma unroll
    for (int a = 0; a < D; a++) {
#pragma unroll
      for (int up = 0; up < 2; up++) {
        if (c3[a] != (up ? L.n[a] - 1 : 0)) continue;
        const int s = 2 * a + up;
        edge[k] |= 1 << s;
        if (OP == 0 && neumann && P.type[sb + s] < 0) edge[k] |= 256 << s;
      }
    }
  }
  const int base = p * L.ps;
  if (OP == 1)
    for (int k = threadIdx.x; k < L.cs; k += NT) cfl[k] = at(coeffs, base + k);

  // applySinglePatchWithInternalBoundaryConditions (Poisson/StarPatchOperator.h:75-101 with
  // internal = true): every side ghost is -interior, except physical Neumann sides (+interior)
  auto apply = [&](const T (&v)[CPT], T (&out)[CPT]) {
#pragma unroll
    for (int k = 0; k < CPT; k++)
      if (gidx[k] >= 0) pad[gidx[k]] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < CPT; k++) {
      out[k] = T(0);
      if (gidx[k] < 0) continue;
      const int g = gidx[k], e = edge[k];
      const T mid = v[k];
      T acc = T(0);
#pragma unroll
      for (int a = 0; a < D; a++) {
        const T lo = pad[g - st[a]], hi = pad[g + st[a]];
        const T lower = (e >> (2 * a)) & 1 ? ((e >> (8 + 2 * a)) & 1 ? mid : -mid) : lo;
        const T upper = (e >> (2 * a + 1)) & 1 ? ((e >> (9 + 2 * a)) & 1 ? mid : -mid) : hi;
        if (OP == 0) {
          acc += (upper - T(2) * mid + lower) * ih2[a];
        } else {
          const T cm = cfl[g], cl = cfl[g - st[a]], cu = cfl[g + st[a]];
          acc += ((cu + cm) * (upper - mid) - (cl + cm) * (mid - lower)) * (ih2[a] * T(0.5));
        }
      }
      out[k] = acc;
    }
  };

  // f_copy = f; modifyRHSForInternalBoundaryConditions (Poisson :165-180, VarPoisson :168-186)
  T x[CPT], b[CPT];
#pragma unroll
  for (int k = 0; k < CPT; k++) {
    x[k] = T(0);
    b[k] = T(0);
    if (gidx[k] < 0) continue;
    const int g = base + gidx[k];
    x[k] = u[g];
    T v = at(f, g);
#pragma unroll
    for (int s = 0; s < 2 * D; s++) {
      if (!((edge[k] >> s) & 1) || P.type[sb + s] < 0) continue;
      const int a = s >> 1, gg = s & 1 ? g + st[a] : g - st[a];
      if (OP == 0) v -= (u[gg] + x[k]) * ih2[a];
      else v -= (u[gg] + x[k]) * (at(coeffs, g) + at(coeffs, gg)) * (ih2[a] * T(0.5));
    }
    b[k] = v;
  }
  StagedOp<T, CPT, decltype(apply)> op{ apply };
  bool broke;
  const int its = patch_solve<T, CPT, NT>(x, b, max_it, tol, red, &broke, op);
#pragma unroll
  for (int k = 0; k < CPT; k++)
    if (gidx[k] >= 0) u[base + gidx[k]] = x[k];
  if (threadIdx.x == 0) {
    if (iters) iters[p] = its;
    if (broke) breakdown[0] = 1;
  }
}

template <typename T, int D, int OP>
int launch_cpt(const te_domain* d, int N, const T* coeffs, const T* f, T* u, int neumann, int max_it, double tol,
               int32_t* iters, int32_t* bd, hipStream_t s)
{
  if (D == 2 && d->ns[0] == d->ns[1]) {
#define TE_PT(N_, NT_)                                                                                            \
  hipLaunchKernelGGL((patch_bicgstab_tile<T, OP, N_, NT_>), dim3(d->np), dim3(NT_), 0, s, d->d_patches, coeffs, f, \
                     u, neumann, max_it, tol, iters, bd)
    switch (d->ns[0]) {
      case 8: TE_PT(8, 64); return TE_OK;
      case 16: TE_PT(16, 64); return TE_OK;
      case 32: TE_PT(32, 256); return TE_OK;
      default: break;
    }
#undef TE_PT
  }
  Layout L = make_layout(d->dim, d->ns, 1, d->np);
  size_t shmem = sizeof(T) * (size_t)L.cs * (OP == 1 ? 2 : 1);
#define TE_PB(C_, NT_)                                                                                         \
  hipLaunchKernelGGL((patch_bicgstab_kernel<T, D, OP, C_, NT_>), dim3(d->np), dim3(NT_), shmem, s, d->d_patches, \
                     coeffs, f, u, L, neumann, max_it, tol, iters, bd)
  // up to 256 cells in one wave (no barriers), else four
  if (N <= 64) TE_PB(1, 64);
  else if (N <= 128) TE_PB(2, 64);
  else if (N <= 256) TE_PB(4, 64);
  else if (N <= 512) TE_PB(2, kThreads);
  else if (N <= 1024) TE_PB(4, kThreads);
  else if (N <= 2048) TE_PB(8, kThreads);
  else TE_PB(16, kThreads);
#undef TE_PB
  return TE_OK;
}

}  // namespace

int launch_patch_bicgstab(const te_domain* d, int dtype, int op_kind, int neumann, const void* coeffs, const void* f,
                          void* u, int max_it, double tol, int32_t* iters, int32_t* bd, hipStream_t s)
{
  if (d->np == 0) return TE_OK;
  int N = d->ns[0] * d->ns[1] * (d->dim == 3 ? d->ns[2] : 1);
  if (N > 16 * kThreads) {
    set_error("patch BiCGStab smoother supports at most 4096 cells per patch");
    return TE_ERR_UNSUPPORTED;
  }
#define TE_PD(T)                                                                                                   \
  if (d->dim == 2) {                                                                                               \
    if (op_kind == 0) launch_cpt<T, 2, 0>(d, N, (const T*)coeffs, (const T*)f, (T*)u, neumann, max_it, tol, iters, bd, s); \
    else launch_cpt<T, 2, 1>(d, N, (const T*)coeffs, (const T*)f, (T*)u, neumann, max_it, tol, iters, bd, s);      \
  } else {                                                                                                         \
    if (op_kind == 0) launch_cpt<T, 3, 0>(d, N, (const T*)coeffs, (const T*)f, (T*)u, neumann, max_it, tol, iters, bd, s); \
    else launch_cpt<T, 3, 1>(d, N, (const T*)coeffs, (const T*)f, (T*)u, neumann, max_it, tol, iters, bd, s);      \
  }
  if (dtype == TE_F64) {
    TE_PD(double)
  } else {
    TE_PD(float)
  }
#undef TE_PD
  TE_HIP(hipGetLastError());
  return TE_OK;
}

}  // namespace te
