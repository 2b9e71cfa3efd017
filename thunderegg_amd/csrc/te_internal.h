// Internal declarations shared by the host code and the HIP kernels of
// libthunderegg_amd.  Not part of the public C ABI.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/thunderegg_amd.h"

namespace te {

void set_error(const std::string& msg);

// 64 bytes of page-locked host memory that every device writes, for results that the host reads
// after a stream synchronisation (no copy); nullptr when there is none to be had
double* take_result();
void give_result(double* r);

#define TE_HIP(call)                                                                                 \
  do {                                                                                               \
    hipError_t e_ = (call);                                                                          \
    if (e_ != hipSuccess) {                                                                          \
      ::te::set_error(std::string(#call) + ": " + hipGetErrorString(e_));                            \
      return TE_ERR_HIP;                                                                             \
    }                                                                                                \
  } while (0)

// Per-patch neighbour table on the device.  Slots as in te_patch_info.
struct DevPatch {
  int type[26];
  int orth[26];
  int nbr[26][4];
  double h[3];
  double inv_h2[3];
  int any_nbr;
  int pad;
};

// Vector layout: [patch][comp][z][y][x], each axis padded by one ghost cell.
struct Layout {
  int dim;
  int n[3];   // cells per axis (n[2] = 1 in 2D)
  int ncomp;
  int sx;     // stride of y  (= n0 + 2)
  int sy;     // stride of z  (= (n0 + 2)(n1 + 2))
  int cs;     // component stride (padded cells of one component)
  int ps;     // patch stride (= cs * ncomp)
  int np;     // number of patches
};

inline Layout make_layout(int dim, const int* n, int ncomp, int np)
{
  Layout L{};
  L.dim = dim;
  L.n[0] = n[0];
  L.n[1] = n[1];
  L.n[2] = dim == 3 ? n[2] : 1;
  L.ncomp = ncomp;
  L.sx = L.n[0] + 2;
  L.sy = (L.n[0] + 2) * (L.n[1] + 2);
  L.cs = dim == 3 ? L.sy * (L.n[2] + 2) : L.sy;
  L.ps = L.cs * ncomp;
  L.np = np;
  return L;
}

// base[idx] for idx >= 0 with the byte offset formed in 32 bits (tables and vectors of one
// component stay below 2 GiB, checked when domains are created), so a load or store can address
// from a scalar base plus a 32-bit vector offset instead of a 64-bit vector address.  Vectors of
// several components reach 16 GiB: there the base is one component of one patch (component).
template <typename T>
__device__ __forceinline__ const T& at(const T* base, int idx)
{
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + (unsigned)idx * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T& at(T* base, int idx)
{
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + (unsigned)idx * (unsigned)sizeof(T));
}

// component c of patch p: all its padded values lie within 32-bit offsets of it
template <typename T>
__device__ __forceinline__ T* component(const Layout& L, T* u, int p, int c)
{
  return u + (p * L.ps + c * L.cs);
}

// x / d for 0 <= x < 2^31 and a fixed d >= 1 as one high product and a shift
struct FastDiv {
  unsigned d = 1, mul = 1u << 31, sh = 0;
  FastDiv() = default;
  explicit FastDiv(unsigned dd) : d(dd)
  {
    while ((1ull << sh) < dd) sh++;
    // mul = floor(2^(31 + sh) / d) + 1 exceeds 2^(31 + sh) / d by at most 1 <= 2^sh / d, so the
    // quotient is exact below 2^31
    mul = (unsigned)((1ull << (31 + sh)) / dd + 1);
  }
  __host__ __device__ __forceinline__ int operator()(int x) const
  {
    return (int)((((unsigned long long)((unsigned)x << 1) * mul) >> 32) >> sh);
  }
};

// The item of workgroup b when the grid is 8 * ceil(n / 8) workgroups and XCD x (workgroups are
// dealt round-robin over the 8) takes the x-th contiguous eighth of n items: patches are in
// Morton order, so most neighbours are then read through the same L2.  n or more: no item.
__host__ __device__ inline int xcd_grid(int n) { return (n + 7) / 8 * 8; }
__device__ __forceinline__ int xcd_item(int b, int grid) { return (b & 7) * (grid >> 3) + (b >> 3); }

// part k of n items in 2^split equal parts: [*first, the return value)
__device__ __forceinline__ int split_range(int n, int split, int k, int* first)
{
  *first = (int)(((long)n * k) >> split);
  return (int)(((long)n * (k + 1)) >> split);
}

// The interior cells of a padded vector as items of V consecutive padded values: row after row
// (ghost rows left out), each row the V-wide groups that cover its cells.  V = 2 (even n[0],
// so that every row starts a group) puts the row's first and last cell into groups with a ghost.
struct Rows {
  FastDiv per_row, ny, nyz;  // groups per row, rows per slice, rows per patch and component
  int items;                 // groups in all
  int sx, sy, cs, last;      // last: index of a row's last group
  Rows() = default;
  Rows(const Layout& L, int V)
  {
    const int nz = L.dim == 3 ? L.n[2] : 1, groups = V == 2 ? L.n[0] / 2 + 1 : L.n[0];
    per_row = FastDiv(groups);
    ny = FastDiv(L.n[1]);
    nyz = FastDiv(L.n[1] * nz);
    items = groups * L.n[1] * nz * L.np * L.ncomp;
    sx = L.sx;
    sy = L.dim == 3 ? L.sy : 0;
    cs = L.cs;
    last = groups - 1;
  }
  // the padded index of item i's first value; *g: its place in the row
  template <int V>
  __device__ __forceinline__ int at(int i, int* g) const
  {
    const int row = per_row(i), pc = nyz(row), rem = row - pc * (int)nyz.d, z = ny(rem), y = rem - z * (int)ny.d;
    *g = i - row * (int)per_row.d;
    return pc * cs + (sy ? (z + 1) * sy : 0) + (y + 1) * sx + V * *g + (V == 1 ? 1 : 0);
  }
};

__host__ __device__ inline int lin(const Layout& L, int p, int c, int x, int y, int z)
{
  return p * L.ps + c * L.cs + (x + 1) + (y + 1) * L.sx + (L.dim == 3 ? (z + 1) * L.sy : 0);
}

}  // namespace te

struct te_domain {
  int dim;
  int ns[3];
  int np;
  std::vector<te_patch_info> patches;
  std::vector<int32_t> nbr_local;  // np * 26 * 4
  te::DevPatch* d_patches = nullptr;
  int any_coarse_fine = 0;         // some face/edge/corner is a coarse/fine interface
  double* d_scratch = nullptr;     // reduction partials
  double* result = nullptr;        // a reduction's result: host memory that the kernels write (take_result)
  int32_t* d_flags = nullptr;      // breakdown flags
  int32_t* d_ring = nullptr;       // 2D: ring table (te::ring_table), pq fields 0
};

struct te_ghost_filler {
  const te_domain* d;
  int kind;
  int fill_type;
};

struct te_level_link {
  const te_domain* fine;
  const te_domain* coarse;
  std::vector<int32_t> parent;      // per fine patch
  int32_t* d_parent = nullptr;      // per fine patch
  int32_t* d_orth = nullptr;        // per fine patch orth_on_parent (-1 copy)
  // per coarse patch: children (fine local indexes) in increasing local-index order
  int32_t* d_child = nullptr;       // [np_coarse][8]
  int32_t* d_nchild = nullptr;      // [np_coarse]
  int32_t* d_ring = nullptr;        // 2D: ring table of the fine level with the pq fields set
  // even cells per side, and every coarse patch has either one copied child or children of
  // distinct orthants: each coarse cell then lies under one child
  bool regular = true;
  // every coarse patch has a copied child or one per orthant: no coarse cell is without a child
  bool covered = true;
};

namespace te {

// 2D ring table: for patch p, side s and half h of that side (h = 1 for ghost cells
// t >= n / 2), the int4 record at [(p * 4 + s) * 2 + h] = {type, orth, q, pq} of what a
// ghost cell there reads: the side's neighbour type and orth_on_coarse, the neighbour
// patch q (for finer neighbours the one facing that half; -1 on a physical side) and,
// when the table belongs to a level link, q's parent * 8 + orth_on_parent(q) + 1 in the
// coarser level (0 otherwise).  One 16-byte load gives a lane everything it needs to
// issue the neighbour reads of its ghost cell.
std::vector<int32_t> ring_table(const te_domain* d, const int32_t* parent, const int32_t* orth_on_parent);

// compute units of the current device (queried once per device)
int cu_count();
// Each of np patches is shared by 2^s units (workgroups or wavefronts) of `waves` waves, `pass` of
// its `items` work items a pass: s grows while a unit would take more than two passes and the
// launch has fewer than per_cu waves a CU, and not past `most` units.  A patch that one wave walks
// alone takes as long as its cells: the operator on 4 patches of 1024^2 (FP64) 3,460 us as one wave
// a patch, 26 shared; 8 of 64^3 148 and 17; 64 of 32^2 7.0 and 4.4.  Neither more nor fewer than 16
// (1,024 patches of 128^2 in FP32 at 8 / 16 / 32 waves a CU: 41 / 30 / 34 us; 512 of 16^3 in FP64:
// 17 / 16 / 20), but for the long rows that launch_one (stencil.hip) names.
int patch_split(int np, long items, int pass, int waves, long most, int per_cu = 16);
// workgroups of `block` threads and `shmem` dynamic LDS bytes of `kernel` resident at once
// on the whole current device (occupancy query, cached)
int resident_blocks(const void* kernel, int block, size_t shmem);

// Timings on a stream for the solvers (timer.cpp): a domain timing (domain_id, or INT_MAX
// for none) started / stopped by events on s.  A null timer makes both no-ops.
int timer_start_stream(te_timer* t, const char* name, int domain_id, hipStream_t s);
int timer_stop_stream(te_timer* t, const char* name, int domain_id, hipStream_t s);
bool timer_has_domain(const te_timer* t, int domain_id);

// ---- launchers (defined in kernels/*.hip) ----
int launch_ghost_fill(const te_ghost_filler* g, int dtype, void* u, int ncomp, hipStream_t s);
int launch_ghost_fill_faces(const te_ghost_filler* g, int dtype, void* u, int ncomp, hipStream_t s);
int launch_ghost_fill_lowdim(const te_ghost_filler* g, int dtype, void* u, int ncomp, hipStream_t s);
// out = A u, or fin - A u where fin is given.  fill: u's ghosts are filled first (as
// launch_ghost_fill) in the same launch; otherwise they are read as they are.
int launch_star(const te_ghost_filler* g, int dt, int dtf, int dto, int op_kind, int neumann, const void* coeffs,
                const void* fin, void* u, void* out, int ncomp, bool fill, hipStream_t s);
// extrapolate: LinearRestrictor's extrapolate_boundary_ghosts
int launch_restrict(const te_level_link* l, int dtype_in, const void* fine, int dtype_out, void* coarse, int ncomp,
                    hipStream_t s, bool extrapolate = false);
int launch_interpolate(const te_level_link* l, int dtype_c, const void* coarse, int dtype_f, void* fine, int ncomp,
                       hipStream_t s);
// boundary data (kernels/bc.hip): values per patch, sum over sides of the face cell counts
long boundary_stride(const te_domain* d);
int launch_bc_rhs(const te_domain* d, int dtype, void* f, const double* g, const double* c, bool neumann,
                  hipStream_t s);

}  // namespace te
