// libbmg: cells of a level, boundaries and coefficients, shared by the
// kernels of the grids and those of trees' uniform levels (which do not
// include the grids' kernels).  The storage is described in bmg_kernels.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace bmg {

constexpr int kBlock = 256;

// homogeneous boundary description of one level
struct BCH {
  int periodic[3];
  int sigma[6];  // right, left, top, bottom, front, back
  int tree;      // edge/corner ghosts by the tree rule (see bilinear_at)
};

// inhomogeneous boundary of `a` on the finest level: ghost = c + sigma * s,
// with the cell size (x / Delta is computed as x * invD when Delta is a
// power of two, which rounds identically)
struct BCA {
  int periodic[3];
  int sigma[6];
  const double* c[6];  // n^(DIM-1) values per side, or null for 0
  double invD;
  int pow2;
};

// cell indices fit in 32 bits (at most 2^30 cells per level)
using idx_t = uint32_t;

// two adjacent values as one vector load/store
template <typename T>
struct Vec2;
template <>
struct Vec2<float> {
  using type = float2;
};
template <>
struct Vec2<double> {
  using type = double2;
};

template <int DIM>
struct Geo {
  int n, log2n;
  __device__ __forceinline__ void decode(idx_t idx, int c[3]) const {
    const idx_t m = (idx_t)(n - 1);
    if (DIM == 3) {
      c[2] = (int)(idx & m);
      c[1] = (int)((idx >> log2n) & m);
      c[0] = (int)(idx >> (2 * log2n));
    } else if (DIM == 2) {
      c[2] = 0;
      c[1] = (int)(idx & m);
      c[0] = (int)(idx >> log2n);
    } else {
      c[0] = (int)idx;
      c[1] = c[2] = 0;
    }
  }
  __device__ __forceinline__ idx_t stride(int d) const {
    if (DIM == 3) return d == 0 ? (idx_t)1 << (2 * log2n) : d == 1 ? (idx_t)1 << log2n : 1u;
    if (DIM == 2) return d == 0 ? (idx_t)1 << log2n : 1u;
    return 1u;
  }
  __device__ __forceinline__ idx_t index(const int c[3]) const {
    if (DIM == 3) return ((((idx_t)c[0] << log2n) + (idx_t)c[1]) << log2n) + (idx_t)c[2];
    if (DIM == 2) return ((idx_t)c[0] << log2n) + (idx_t)c[1];
    return (idx_t)c[0];
  }
  // index on the wall normal to d (tangential coordinates in order)
  __device__ __forceinline__ idx_t wall(int d, const int c[3]) const {
    if (DIM == 3)
      return d == 0 ? ((idx_t)c[1] << log2n) + c[2] : d == 1 ? ((idx_t)c[0] << log2n) + c[2]
                                                           : ((idx_t)c[0] << log2n) + c[1];
    if (DIM == 2) return d == 0 ? (idx_t)c[1] : (idx_t)c[0];
    return 0u;
  }
  __device__ __forceinline__ idx_t ncell() const { return (idx_t)1 << (DIM * log2n); }
};

// Blocks are dispatched round-robin over the 8 XCDs; give each XCD a
// contiguous run of logical blocks so that neighbouring rows and planes of
// a stencil share one L2.
__device__ __forceinline__ idx_t logical_block() {
  idx_t b = blockIdx.x, nb = gridDim.x;
  if ((nb & 7) == 0) b = (b & 7) * (nb >> 3) + (b >> 3);
  return b;
}

// index of the neighbour of cell c along d (dir +1 or -1): the cell itself
// when the neighbour is a non-periodic ghost.  `ghost` tells which.
template <int DIM>
__device__ __forceinline__ idx_t nbr_index(const Geo<DIM>& g, const int* periodic, idx_t idx, const int c[3],
                                           int d, int dir, bool& ghost) {
  const idx_t s = g.stride(d);
  const bool inside = dir > 0 ? c[d] < g.n - 1 : c[d] > 0;
  const idx_t wrapoff = (idx_t)(g.n - 1) * s;
  const idx_t step = dir > 0 ? idx + s : idx - s;
  const idx_t wrapped = dir > 0 ? idx - wrapoff : idx + wrapoff;
  ghost = !inside && !periodic[d];
  return inside ? step : (periodic[d] ? wrapped : idx);
}

// value of field f at the neighbour of cell c along d (dir +1 or -1), with
// the homogeneous ghost mapping (branch-free: a ghost reads the cell itself
// and scales it by sigma)
template <int DIM, typename T>
__device__ __forceinline__ T nbr_h(const T* __restrict__ f, const Geo<DIM>& g, const BCH& bc, idx_t idx,
                                   const int c[3], int d, int dir, T self) {
  bool ghost;
  idx_t iq = nbr_index<DIM>(g, bc.periodic, idx, c, d, dir, ghost);
  T v = ghost ? self : f[iq];
  return ghost ? T(bc.sigma[2 * d + (dir < 0)]) * v : v;
}

// alpha on the high face of cell c along d (one load from a selected address)
template <int DIM, typename T>
__device__ __forceinline__ T alpha_hi(const T* __restrict__ lo, const T* __restrict__ wall, const Geo<DIM>& g,
                                      idx_t idx, const int c[3], int d) {
  const T* p = c[d] < g.n - 1 ? lo + idx + g.stride(d) : wall + g.wall(d, c);
  return *p;
}

template <typename T>
struct Coef {
  const T* lo[3];
  const T* wall[3];
  T alpha;        // used when lo[0] is null (constant alpha, unityf)
  const T* lam;   // null: constant lam_c
  T lam_c;
};

// a ghost cell outside along two or three dimensions, from the value v of
// the interior cell diagonal to it.  Multigrid (grid/multigrid.h:543-594,
// one reflection per direction): the product of the sigmas times v.  Tree
// (grid/tree.h:1168-1258): b1 + b2 - v, or b1 + b2 + b3 - 2 v, with
// b = sigma v per crossed side (sums of +-v, so exact in any order).
template <typename T>
__device__ __forceinline__ T corner2(T v, T sa, T sb, bool tree) {
  return tree ? (sb * v + sa * v) - v : (sa * sb) * v;
}
template <typename T>
__device__ __forceinline__ T corner3(T v, T sx, T sy, T sz, bool gx, bool gy, bool gz, bool tree) {
  int k = (int)gx + (int)gy + (int)gz;
  if (!tree || k < 2) return ((sx * sy) * sz) * v;
  if (k == 2) return ((gz ? sz * v : T(0)) + (gy ? sy * v : T(0)) + (gx ? sx * v : T(0))) - v;
  return ((sz * v + sy * v) + sx * v) - T(2) * v;
}

// --- arguments of the kernels that run all coarse levels in one workgroup --

// levels 0..12 at most (4096 cells in 1D)
constexpr int kCoarseLevels = 13;

template <typename T, int DIM>
struct CoarseLevel {
  T* da;
  T* da2;  // Jacobi output
  T* res;
  Coef<T> k;
  Geo<DIM> g;
  BCH bc;
  T D2;
};

template <typename T, int DIM>
struct CoarseArgs {
  CoarseLevel<T, DIM> L[kCoarseLevels];
  int minlevel, top, nrelax, jacobi, gs;  // gs: the in-place Gauss-Seidel order, through da2
  double* a;  // k_coarse_rb: where the finest level ends the cycle, the solution it corrects (or null)
};

}  // namespace bmg
