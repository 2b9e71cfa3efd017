// Vector<D> BLAS-1 over interior cells (Vector.h:391-611) and deterministic
// two-pass reductions: a fixed grid writes one partial per block (wavefront
// shuffles, then LDS), a single-block pass folds the partials in a fixed order.
#include "../te_internal.h"
#include "blas.h"

namespace te {
namespace {

// V values at consecutive addresses: one access
template <typename T, int V>
struct Pack {
  typedef T Vec __attribute__((ext_vector_type(V)));
};
template <typename T>
struct Pack<T, 1> {
  typedef T Vec;
};
template <typename T, int V>
__device__ __forceinline__ T& lane(typename Pack<T, V>::Vec& v, int k)
{
  return reinterpret_cast<T*>(&v)[k];
}

template <typename T, int OP>
__device__ __forceinline__ T vec_value(T x, T a, T b, T alpha, T beta, T gamma)
{
  switch (OP) {
    case VOP_SET: return alpha;
    case VOP_SCALE: return x * alpha;
    case VOP_SHIFT: return x + alpha;
    case VOP_COPY: return a;
    case VOP_ADD: return x + a;
    case VOP_ADD_SCALED: return x + a * alpha;
    case VOP_ADD_SCALED2: return x + (a * alpha + b * beta);
    case VOP_SCALE_THEN_ADD: return x * alpha + a;
    case VOP_SCALE_THEN_ADD_SCALED: return x * alpha + a * beta;
    default: return x * alpha + a * beta + b * gamma;
  }
}

// Every padded value in groups of V consecutive ones, ghost rows too: V * i, or -1 for a group
// without an interior cell; *g: its place in the row.  V divides the row
struct FlatGroups {
  FastDiv per_row, ry, rz;
  int items, n1, n2, last;
  FlatGroups(const Layout& L, int V)
      : per_row(L.sx / V), ry(L.n[1] + 2), rz(L.dim == 3 ? L.n[2] + 2 : 1), items((int)((long)L.np * L.ps / V)),
        n1(L.n[1]), n2(L.dim == 3 ? L.n[2] : 0), last(L.sx / V - 1)
  {
  }
  template <int V>
  __device__ __forceinline__ int at(int i, int* g) const
  {
    const int row = per_row(i), zz = ry(row), y = row - zz * (int)ry.d;
    *g = i - row * (int)per_row.d;
    bool in = y >= 1 && y <= n1 && (V > 1 || (*g > 0 && *g < last));
    if (n2) {
      const int z = zz - rz(zz) * (int)rz.d;
      in = in && z >= 1 && z <= n2;
    }
    return in ? V * i : -1;
  }
};

// One interior update.  HBM bound: a thread takes one group, neighbours in memory are neighbours in
// the launch, and the ghost rows' threads leave.  Lines are then read in the order in which they
// lie: four groups of interior rows a thread (Rows, below) made the streams of large vectors
// slower, at 32768 patches of 16^3 in FP64 (1.5 GB a vector) x = a 888 us, x += a y 830, with
// two such terms 1075, against 763, 723 and 975 here; one FP64 value a thread with its place found
// by five divisions took 786, 743 and 941, and in FP32 590, 619 and 642 against 376, 381 and 512.
// At 4096 patches x = a 95 us, x += a y 92 (4.9 TB/s with the ghost values of the lines it touches).
// A row's end groups hold a ghost value, which is read and not written.
template <typename T, int OP, int V>
__global__ void __launch_bounds__(256) vec_op_kernel(FlatGroups R, T* __restrict__ x, const T* __restrict__ a,
                                                     const T* __restrict__ b, T alpha, T beta, T gamma)
{
  typedef typename Pack<T, V>::Vec P;
  constexpr bool RX = OP != VOP_SET && OP != VOP_COPY, RA = OP >= VOP_COPY,
                 RB = OP == VOP_ADD_SCALED2 || OP == VOP_SCALE_THEN_ADD_SCALED2;
  const int i = blockIdx.x * 256 + threadIdx.x;
  int g = 0;
  const int k = i < R.items ? R.at<V>(i, &g) : -1;
  if (k < 0) return;
  P vx, va, vb, r;
  if (RX) vx = *reinterpret_cast<const P*>(x + k);
  if (RA) va = *reinterpret_cast<const P*>(a + k);
  if (RB) vb = *reinterpret_cast<const P*>(b + k);
#pragma unroll
  for (int j = 0; j < V; j++)
    lane<T, V>(r, j) = vec_value<T, OP>(RX ? lane<T, V>(vx, j) : T(0), RA ? lane<T, V>(va, j) : T(0),
                                        RB ? lane<T, V>(vb, j) : T(0), alpha, beta, gamma);
  if (V == 1 || (g > 0 && g < R.last)) *reinterpret_cast<P*>(x + k) = r;
  else if (g == 0) x[k + 1] = lane<T, V>(r, V - 1);
  else x[k] = lane<T, V>(r, 0);
}

// every padded value of a vector: V at a time (16 bytes, or 1 where x starts off that grid),
// the few values past the last whole group singly
template <typename T, int V>
__global__ void __launch_bounds__(256) vec_fill_kernel(long n, T* __restrict__ x, T alpha)
{
  typedef typename Pack<T, V>::Vec P;
  P r;
#pragma unroll
  for (int j = 0; j < V; j++) lane<T, V>(r, j) = alpha;
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * V;
  if (i + V <= n) *reinterpret_cast<P*>(x + i) = r;
  else
    for (long k = i; k < n; k++) x[k] = alpha;
}

template <typename TD, typename TS>
__global__ void __launch_bounds__(256) convert_kernel(long n, TD* __restrict__ d, const TS* __restrict__ s)
{
  long gid = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (gid < n) d[gid] = TD(s[gid]);
}

}  // namespace

namespace {

// One partial per workgroup over the interior cells (groups of interior rows: te::Rows), kRedItems
// groups a thread and step so that their loads are in flight together: dot product 88 -> 55 us,
// norm of a vector just written 77 -> 31 us (the same vectors; one load in flight before)
constexpr int kRedItems = 4;

template <typename T, int OP, int V>
__global__ void __launch_bounds__(256) reduce_partial_kernel(Rows R, const T* __restrict__ a, const T* __restrict__ b,
                                                             const DevPatch* __restrict__ dp, FastDiv ps,
                                                             double* __restrict__ partial)
{
  typedef typename Pack<T, V>::Vec P;
  double acc[kRedItems];  // max starts at 0: Vector::infNorm is max(0, max v)
#pragma unroll
  for (int k = 0; k < kRedItems; k++) acc[k] = 0.0;
  for (int i0 = blockIdx.x * (256 * kRedItems) + threadIdx.x; i0 < R.items; i0 += gridDim.x * (256 * kRedItems)) {
    int idx[kRedItems], g[kRedItems];
    P va[kRedItems], vb[kRedItems];
#pragma unroll
    for (int k = 0; k < kRedItems; k++) {
      const int i = i0 + k * 256;
      idx[k] = i < R.items ? R.at<V>(i, &g[k]) : -1;
      if (idx[k] < 0) continue;
      va[k] = *reinterpret_cast<const P*>(a + idx[k]);
      if (OP == RED_DOT) vb[k] = *reinterpret_cast<const P*>(b + idx[k]);
    }
#pragma unroll
    for (int k = 0; k < kRedItems; k++) {
      if (idx[k] < 0) continue;
#pragma unroll
      for (int j = 0; j < V; j++) {
        if (V == 2 && ((j == 0 && g[k] == 0) || (j == 1 && g[k] == R.last))) continue;  // the row's ghosts
        const double v = double(lane<T, V>(va[k], j));
        if (OP == RED_DOT) {
          acc[k] += v * double(lane<T, V>(vb[k], j));
        } else if (OP == RED_SUMSQ) {
          acc[k] += v * v;
        } else if (OP == RED_INTEGRAL) {
          const double* h = dp[ps(idx[k])].h;  // h[2] = 1 in 2D
          acc[k] += v * (h[0] * h[1] * h[2]);
        } else {
          acc[k] = fmax(acc[k], v);
        }
      }
    }
  }
  double t = acc[0];
#pragma unroll
  for (int k = 1; k < kRedItems; k++) t = red_combine<OP>(t, acc[k]);
  const double r = block_reduce<OP>(t);
  if (threadIdx.x == 0) partial[blockIdx.x] = r;
}

template <int OP>
__global__ void __launch_bounds__(256) reduce_final_kernel(const double* __restrict__ partial, int n,
                                                           double* __restrict__ out, int sqrt_out)
{
  double acc = 0.0;
  // a fixed order: thread t folds the partials t, t + 256, ..., whose loads do not wait for each other
  double v[kMaxPartials / 256];
#pragma unroll
  for (int k = 0; k < kMaxPartials / 256; k++) {
    const int i = threadIdx.x + k * 256;
    v[k] = i < n ? partial[i] : 0.0;
  }
#pragma unroll
  for (int k = 0; k < kMaxPartials / 256; k++) acc = red_combine<OP>(acc, v[k]);
  double r = block_reduce<OP>(acc);
  if (threadIdx.x == 0) out[0] = sqrt_out ? sqrt(r) : r;
}

}  // namespace

namespace {

// values a group: 2 where rows start on its multiples (even cells per row) in every operand
template <typename T>
int group_of(const Layout& L, const void* x, const void* a, const void* b)
{
  const uintptr_t all = (uintptr_t)x | (uintptr_t)a | (uintptr_t)b;
  return L.n[0] % 2 == 0 && all % (2 * sizeof(T)) == 0 ? 2 : 1;
}

template <typename T>
void vec_op_t(const Layout& L, int op, T* x, const T* a, const T* b, double alpha, double beta, double gamma,
                     hipStream_t s)
{
  if (op == VOP_SET_WITH_GHOST) {
    const long n = (long)L.np * L.ps;
    constexpr int W = 16 / sizeof(T);
    if ((uintptr_t)x % 16 == 0)
      hipLaunchKernelGGL((vec_fill_kernel<T, W>), dim3((unsigned)((n + 256 * W - 1) / (256 * W))), dim3(256), 0, s, n,
                         x, T(alpha));
    else
      hipLaunchKernelGGL((vec_fill_kernel<T, 1>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, x, T(alpha));
    return;
  }
  // FP64 with three streams or more by single values: x += a y at 32768 patches of 16^3 723 us
  // against 772 in pairs, with two terms 975 against 1018 (8^3: 117 against 126, 154 against 164).
  // Pairs for fewer streams (x = a at 512 patches of 64^3 454 us against 529) and in FP32 (x = a
  // at 32768 patches of 16^3 376 against 590)
  const int V = sizeof(T) == 8 && op >= VOP_ADD ? 1 : group_of<T>(L, x, a, b);
  const FlatGroups R(L, V);
  const int grid = (int)(((long)R.items + 255) / 256);
#define TE_VO(OP_)                                                                                                  \
  case OP_:                                                                                                         \
    if (V == 2)                                                                                                     \
      hipLaunchKernelGGL((vec_op_kernel<T, OP_, 2>), dim3(grid), dim3(256), 0, s, R, x, a, b, T(alpha), T(beta),    \
                         T(gamma));                                                                                 \
    else                                                                                                            \
      hipLaunchKernelGGL((vec_op_kernel<T, OP_, 1>), dim3(grid), dim3(256), 0, s, R, x, a, b, T(alpha), T(beta),    \
                         T(gamma));                                                                                 \
    break
  switch (op) {
    TE_VO(VOP_SET);
    TE_VO(VOP_SCALE);
    TE_VO(VOP_SHIFT);
    TE_VO(VOP_COPY);
    TE_VO(VOP_ADD);
    TE_VO(VOP_ADD_SCALED);
    TE_VO(VOP_ADD_SCALED2);
    TE_VO(VOP_SCALE_THEN_ADD);
    TE_VO(VOP_SCALE_THEN_ADD_SCALED);
    TE_VO(VOP_SCALE_THEN_ADD_SCALED2);
    default: break;
  }
#undef TE_VO
}

}  // namespace

int launch_vec_op(const te_domain* d, int dtype, int op, void* x, const void* a, const void* b, double alpha,
                  double beta, double gamma, int ncomp, hipStream_t s)
{
  if (d->np == 0) return TE_OK;
  Layout L = make_layout(d->dim, d->ns, ncomp, d->np);
  if (dtype == TE_F64) vec_op_t<double>(L, op, (double*)x, (const double*)a, (const double*)b, alpha, beta, gamma, s);
  else vec_op_t<float>(L, op, (float*)x, (const float*)a, (const float*)b, alpha, beta, gamma, s);
  TE_HIP(hipGetLastError());
  return TE_OK;
}

namespace {

template <typename T>
int reduce_t(const te_domain* d, const Layout& L, int op, const T* a, const T* b, hipStream_t s)
{
  const int V = group_of<T>(L, a, op == RED_DOT ? b : nullptr, nullptr);
  const Rows R(L, V);
  const int want = (R.items + 256 * kRedItems - 1) / (256 * kRedItems);
  const int g = want < kMaxPartials ? want : kMaxPartials;
  const FastDiv ps(L.ps);
#define TE_RP(OP_)                                                                                                  \
  do {                                                                                                              \
    if (V == 2)                                                                                                     \
      hipLaunchKernelGGL((reduce_partial_kernel<T, OP_, 2>), dim3(g), dim3(256), 0, s, R, a, b, d->d_patches, ps,   \
                         d->d_scratch);                                                                             \
    else                                                                                                            \
      hipLaunchKernelGGL((reduce_partial_kernel<T, OP_, 1>), dim3(g), dim3(256), 0, s, R, a, b, d->d_patches, ps,   \
                         d->d_scratch);                                                                             \
  } while (0)
  if (op == RED_DOT) TE_RP(RED_DOT);
  else if (op == RED_SUMSQ) TE_RP(RED_SUMSQ);
  else if (op == RED_INTEGRAL) TE_RP(RED_INTEGRAL);
  else TE_RP(RED_MAX);
#undef TE_RP
  return g;
}

}  // namespace

int launch_reduce(const te_domain* d, int dtype, int op, const void* a, const void* b, int ncomp, double* d_out,
                  hipStream_t s)
{
  Layout L = make_layout(d->dim, d->ns, ncomp, d->np);
  const int g = dtype == TE_F64 ? reduce_t<double>(d, L, op, (const double*)a, (const double*)b, s)
                                : reduce_t<float>(d, L, op, (const float*)a, (const float*)b, s);
  if (op == RED_MAX)
    hipLaunchKernelGGL((reduce_final_kernel<RED_MAX>), dim3(1), dim3(256), 0, s, d->d_scratch, g, d_out, 0);
  else
    hipLaunchKernelGGL((reduce_final_kernel<RED_SUM>), dim3(1), dim3(256), 0, s, d->d_scratch, g, d_out,
                       op == RED_SUMSQ ? 1 : 0);
  TE_HIP(hipGetLastError());
  return TE_OK;
}

int launch_convert(long n, int dtd, void* dst, int dts, const void* src, hipStream_t s)
{
  if (n == 0) return TE_OK;
  int grid = (int)((n + 255) / 256);
  if (dtd == TE_F64 && dts == TE_F32)
    hipLaunchKernelGGL((convert_kernel<double, float>), dim3(grid), dim3(256), 0, s, n, (double*)dst,
                       (const float*)src);
  else if (dtd == TE_F32 && dts == TE_F64)
    hipLaunchKernelGGL((convert_kernel<float, double>), dim3(grid), dim3(256), 0, s, n, (float*)dst,
                       (const double*)src);
  else if (dtd == TE_F64)
    hipLaunchKernelGGL((convert_kernel<double, double>), dim3(grid), dim3(256), 0, s, n, (double*)dst,
                       (const double*)src);
  else
    hipLaunchKernelGGL((convert_kernel<float, float>), dim3(grid), dim3(256), 0, s, n, (float*)dst,
                       (const float*)src);
  TE_HIP(hipGetLastError());
  return TE_OK;
}

}  // namespace te
