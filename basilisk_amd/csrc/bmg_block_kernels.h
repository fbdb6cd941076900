// libbmg: red-black sweeps of whole levels or tiles held on chip, 2D and 3D.
//
// Below the sizes that stream from HBM a sweep is bound by its two dependent
// launches (3.5-5 us each whatever the size up to 64^3 or 512^2 cells).  The
// kernels here run several half-sweeps per launch with a workgroup barrier
// between them:
//   k_coarse_rb  the coarsest levels of a cycle (up to 4096 cells), one
//                workgroup
//   k_rb_tile    the sweeps of one larger level, tiles with a halo of two
//                cells per sweep that every workgroup recomputes
// Same arithmetic, in the same order, as relax_value and bilinear_at.
//
// A thread owns a block of 2^DIM cells (even corner, so every block has its
// red cells at the same places): their values, -D2 res, the denominators,
// which do not change over the sweeps, and the faces, those inside the block
// once, are in registers.  Of a cell's 2 DIM neighbours DIM are in its own
// block; the others are read from LDS, where the field is stored by place in
// the block and then by block, so that the lanes of a wave read consecutive
// words (row-major pairs of cells cost two-way bank conflicts and twice the
// LDS reads: 1.4 us instead of 0.6 us for a half-sweep of 4096 cells).
#pragma once

#include "bmg_cells.h"

namespace bmg {

// place p of a block: its coordinate along d (the last dimension fastest)
template <int DIM>
__device__ __forceinline__ constexpr int place_bit(int d) {
  return 1 << (DIM - 1 - d);
}
__device__ __forceinline__ constexpr int place_colour(int p) { return (p ^ (p >> 1) ^ (p >> 2)) & 1; }

template <int DIM, typename T, bool ALPHAF>
struct RBBlock {
  static constexpr int NC = 1 << DIM, NF = NC / 2;
  T v[NC];           // values
  T m[NC], d[NC];    // -D2 res, denominators
  T face[ALPHAF ? DIM : 1][3][ALPHAF ? NF : 1];  // faces normal to each dimension: low, middle, high
  int lo[DIM], hi[DIM];  // LDS offsets of the blocks below and above
  int wall;              // bits 2 d, 2 d + 1: a wall (not periodic) below, above

  // index of place p among the places with the same coordinate along d
  static __device__ __forceinline__ constexpr int across(int p, int d) {
    const int b = place_bit<DIM>(d);
    return (p & (b - 1)) | ((p >> 1) & ~(b - 1));
  }
  // the coefficients of the block whose first cell is c (index idx)
  __device__ __forceinline__ void load(const T* __restrict__ res, const Coef<T>& k, const Geo<DIM>& g, idx_t idx,
                                       const int c[3], T D2) {
    using V2 = typename Vec2<T>::type;
#pragma unroll
    for (int p = 0; p < NC; p += 2) {
      idx_t at = idx;
#pragma unroll
      for (int e = 0; e < DIM - 1; e++)
        if (p & place_bit<DIM>(e)) at += g.stride(e);
      m[p] = -D2 * res[at];
      m[p + 1] = -D2 * res[at + 1];
      V2 lam;
      lam.x = lam.y = k.lam_c;
      if (k.lam) lam = *reinterpret_cast<const V2*>(k.lam + at);
      d[p] = -lam.x * D2;
      d[p + 1] = -lam.y * D2;
      if (ALPHAF) {
#pragma unroll
        for (int e = 0; e < DIM; e++) {
          const V2 f = *reinterpret_cast<const V2*>(k.lo[e] + at);
          const int x0 = p & place_bit<DIM>(e) ? 1 : 0;
          face[ALPHAF ? e : 0][x0][ALPHAF ? across(p, e) : 0] = f.x;
          face[ALPHAF ? e : 0][e == DIM - 1 ? 1 : x0][ALPHAF ? across(p + 1, e) : 0] = f.y;
        }
      }
    }
    if (ALPHAF) {
#pragma unroll
      for (int e = 0; e < DIM; e++)
#pragma unroll
        for (int p = 0; p < NC; p++)
          if (p & place_bit<DIM>(e)) {
                  idx_t at = idx;
            int cp[3] = {c[0], c[1], c[2]};
#pragma unroll
            for (int q = 0; q < DIM; q++)
              if (p & place_bit<DIM>(q)) {
                at += g.stride(q);
                cp[q]++;
              }
            face[ALPHAF ? e : 0][2][ALPHAF ? across(p, e) : 0] =
                alpha_hi<DIM, T>(k.lo[e], k.wall[e], g, at, cp, e);
          }
    }
#pragma unroll
    for (int p = 0; p < NC; p++)
#pragma unroll
      for (int e = 0; e < DIM; e++) {
        if (ALPHAF) d[p] += high(p, e) + low(p, e);
        else d[p] += k.alpha + k.alpha;
      }
  }
  __device__ __forceinline__ T low(int p, int e) const {
    return face[ALPHAF ? e : 0][p & place_bit<DIM>(e) ? 1 : 0][ALPHAF ? across(p, e) : 0];
  }
  __device__ __forceinline__ T high(int p, int e) const {
    return face[ALPHAF ? e : 0][p & place_bit<DIM>(e) ? 2 : 1][ALPHAF ? across(p, e) : 0];
  }
  // relax the cells of one colour; f: this block in LDS, plane: the distance
  // between places there
  __device__ __forceinline__ void relax(int colour, T* f, int plane, T alpha, const BCH& bc) {
#pragma unroll
    for (int p = 0; p < NC; p++) {
      if (place_colour(p) != colour) continue;
      T n = m[p];
#pragma unroll
      for (int e = 0; e < DIM; e++) {
        const int b = place_bit<DIM>(e), q = p ^ b;
        const bool up = p & b;  // the upper cell of the block along e
        T x = f[q * plane + (up ? hi[e] : lo[e])];
        if (wall & (1 << (2 * e + (up ? 1 : 0)))) x = T(bc.sigma[2 * e + (up ? 0 : 1)]) * v[p];
        const T ah = ALPHAF ? high(p, e) : alpha, al = ALPHAF ? low(p, e) : alpha;
        n += ah * (up ? x : v[q]) + al * (up ? v[q] : x);
      }
      v[p] = n / d[p];
    }
#pragma unroll
    for (int p = 0; p < NC; p++)
      if (place_colour(p) == colour) f[p * plane] = v[p];
  }
};

// bilinear values of the 2^DIM children of coarse cell c (of an n^DIM level)
// as bilinear_at; at(q) reads the coarse cell at q
template <int DIM, typename T, typename At>
__device__ __forceinline__ void bilinear_block(const int c[3], int n, const BCH& bc, const At& at, T* v) {
  const bool tree = bc.tree != 0;
  int q[3][3];   // per dimension: below, the cell, above
  T sg[3][3];
  bool gh[3][3];
#pragma unroll
  for (int d = 0; d < 3; d++)
#pragma unroll
    for (int o = -1; o <= 1; o++) {
      const int x = d < DIM ? c[d] + o : 0;
      const bool out = d < DIM && (x < 0 || x >= n);
      gh[d][o + 1] = out && !bc.periodic[d];
      q[d][o + 1] = !out ? x : bc.periodic[d] ? (x < 0 ? x + n : x - n) : c[d];
      sg[d][o + 1] = gh[d][o + 1] ? T(bc.sigma[2 * d + (o < 0)]) : T(1);
    }
  constexpr int NR = DIM == 3 ? 27 : 9;
  T r[NR];
#pragma unroll
  for (int m = 0; m < NR; m++) {
    const int i = DIM == 3 ? m / 9 : m / 3, j = DIM == 3 ? (m / 3) % 3 : m % 3, l = DIM == 3 ? m % 3 : 0;
    const int x[3] = {q[0][i], q[1][j], DIM == 3 ? q[2][l] : 0};
    r[m] = at(x);
  }
#pragma unroll
  for (int p = 0; p < (1 << DIM); p++) {
    if (DIM == 2) {
      const int i = p & 2 ? 2 : 0, j = p & 1 ? 2 : 0;
      const T sx = sg[0][i], sy = sg[1][j];
      T c00 = r[4], c10 = sx * r[i * 3 + 1], c01 = sy * r[3 + j];
      T c11 = gh[0][i] && gh[1][j] ? corner2(r[i * 3 + j], sx, sy, tree) : (sx * sy) * r[i * 3 + j];
      v[p] = (T(9) * c00 + T(3) * (c10 + c01) + c11) / T(16);
    } else {
      const int i = p & 4 ? 2 : 0, j = p & 2 ? 2 : 0, l = p & 1 ? 2 : 0;
      const T sx = sg[0][i], sy = sg[1][j], sz = sg[2][l];
      const bool gx = gh[0][i], gy = gh[1][j], gz = gh[2][l];
#define BR(x, y, z) r[((x)*3 + (y)) * 3 + (z)]
      T c000 = BR(1, 1, 1), c100 = sx * BR(i, 1, 1), c010 = sy * BR(1, j, 1), c001 = sz * BR(1, 1, l);
      T c110 = gx && gy ? corner2(BR(i, j, 1), sx, sy, tree) : (sx * sy) * BR(i, j, 1);
      T c101 = gx && gz ? corner2(BR(i, 1, l), sx, sz, tree) : (sx * sz) * BR(i, 1, l);
      T c011 = gy && gz ? corner2(BR(1, j, l), sy, sz, tree) : (sy * sz) * BR(1, j, l);
      T c111 = corner3(BR(i, j, l), sx, sy, sz, gx, gy, gz, tree);
#undef BR
      v[p] = (T(27) * c000 + T(9) * (c100 + c010 + c001) + T(3) * (c110 + c101 + c011) + c111) / T(64);
    }
  }
}

// k_prolong with one thread per coarse cell: its 2^DIM children from the
// 3^DIM cells around it, each read once (the children one by one read them
// 64 times: 34 us at 256^3 FP32), the two children along the last dimension
// written as one vector
template <int DIM, typename T>
__global__ __launch_bounds__(kBlock) void k_prolong_children(const T* __restrict__ coarse, T* __restrict__ fine,
                                                             Geo<DIM> gf, BCH bcc) {
  using V2 = typename Vec2<T>::type;
  const Geo<DIM> gc{gf.n >> 1, gf.log2n - 1};
  const idx_t idx = logical_block() * kBlock + threadIdx.x;
  if (idx >= gc.ncell()) return;
  int c[3];
  gc.decode(idx, c);
  T v[1 << DIM];
  bilinear_block<DIM, T>(c, gc.n, bcc, [&](const int* q) { return coarse[gc.index(q)]; }, v);
  const int f[3] = {2 * c[0], 2 * c[1], 2 * c[2]};
  const idx_t b = gf.index(f);
#pragma unroll
  for (int p = 0; p < (1 << DIM); p += 2) {
    idx_t at = b;
#pragma unroll
    for (int d = 0; d < DIM - 1; d++)
      if (p & place_bit<DIM>(d)) at += gf.stride(d);
    V2 w;
    w.x = v[p];
    w.y = v[p + 1];
    *reinterpret_cast<V2*>(fine + at) = w;
  }
}

// --- all coarse levels in one workgroup, red-black ------------------------
//
// Levels minlevel..top of the cycle (top of at most 16^3 or 32^2 cells):
// restriction of res down to minlevel, then from minlevel up the zero
// or bilinear initial guess and nrelax sweeps, a thread per block of the
// level.  res and da of every level end in memory too.  On a grid that ends
// there the correction is added as well (a launch of 4 us otherwise).
//
// NT: the blocks of the largest level it takes.  2D: 256 (32^2).  3D: 512
// (16^3), but with a face field in FP64 a block's 60 values leave no
// registers at two waves per SIMD (99 us with spills), so 64 (8^3, one wave).
template <int DIM, typename T, bool ALPHAF>
constexpr int kCoarseThreads = DIM == 2 ? 256 : sizeof(T) == 8 && ALPHAF ? 64 : 512;

template <int DIM, typename T, bool ALPHAF>
__global__ __launch_bounds__((kCoarseThreads<DIM, T, ALPHAF>)) void k_coarse_rb(CoarseArgs<T, DIM> A) {
  constexpr int NC = 1 << DIM, kBlocks = kCoarseThreads<DIM, T, ALPHAF>;
  constexpr int kRes = 2 * kBlocks;  // the cells of all levels below the largest
  // the fields of the level and of the one below it (by turns: the larger
  // part for the levels of top's parity)
  __shared__ T big[NC * kBlocks], small[kBlocks], rs[kRes];
  const int t = threadIdx.x;
  auto roff = [](int l) { return ((1 << (DIM * l)) - 1) / ((1 << DIM) - 1); };
  for (int l = A.top - 1; l >= A.minlevel; l--) {
    const CoarseLevel<T, DIM>& C = A.L[l];
    const Geo<DIM> gc = C.g, gf = A.L[l + 1].g;
    const T* F = l + 1 == A.top ? A.L[l + 1].res : rs + roff(l + 1);
    for (idx_t idx = t; idx < gc.ncell(); idx += blockDim.x) {
      int c[3];
      gc.decode(idx, c);
      int f[3] = {2 * c[0], 2 * c[1], 2 * c[2]};
      const idx_t b = gf.index(f);
      T sum = T(0);
#pragma unroll
      for (int m = 0; m < NC / 2; m++) {
        const idx_t q = b + (DIM == 3 ? (idx_t)(m >> 1) * gf.stride(0) + (idx_t)(m & 1) * gf.stride(1)
                                      : (idx_t)m * gf.stride(0));
        sum += F[q];
        sum += F[q + 1];
      }
      sum = sum / T(NC);
      rs[roff(l) + idx] = sum;
      C.res[idx] = sum;
    }
    __syncthreads();
  }
  for (int l = A.minlevel; l <= A.top; l++) {
    const CoarseLevel<T, DIM>& L = A.L[l];
    const Geo<DIM> g = L.g;
    const int n = g.n;
    T* cur = ((A.top - l) & 1) == 0 ? big : small;
    const T* prev = ((A.top - l) & 1) == 0 ? small : big;
    if (n == 1) {
      // one cell, red, its ghosts sigma times itself
      if (t == 0) {
        T v = T(0);
        for (int it = 0; it < A.nrelax; it++) {
          T nn = -L.D2 * (A.top == 0 ? L.res[0] : rs[0]), dd = -(L.k.lam ? L.k.lam[0] : L.k.lam_c) * L.D2;
          for (int d = 0; d < DIM; d++) {
            const T ah = L.k.lo[0] ? L.k.wall[d][0] : L.k.alpha, al = L.k.lo[0] ? L.k.lo[d][0] : L.k.alpha;
            const T ap = L.bc.periodic[d] ? v : T(L.bc.sigma[2 * d]) * v;
            const T am = L.bc.periodic[d] ? v : T(L.bc.sigma[2 * d + 1]) * v;
            nn += ah * ap + al * am;
            dd += ah + al;
          }
          v = nn / dd;
        }
        cur[0] = v;
        L.da[0] = v;
        if (A.a && A.top == 0) A.a[0] += (double)v;
      }
      __syncthreads();
      continue;
    }
    // blocks of this level and of the previous one, per dimension
    const int lb = g.log2n - 1, nb = n >> 1, lp = g.log2n - 2;
    const int plane = 1 << (DIM * lb), pplane = lp < 0 ? 1 : 1 << (DIM * lp);
    const bool on = t < plane;
    RBBlock<DIM, T, ALPHAF> B;
    T* f = cur + t;
    idx_t idx = 0;
    if (on) {
      int cb[3] = {0, 0, 0};
      Geo<DIM>{nb, lb}.decode((idx_t)t, cb);
      const int c[3] = {2 * cb[0], 2 * cb[1], DIM == 3 ? 2 * cb[2] : 0};
      idx = g.index(c);
      B.wall = 0;
#pragma unroll
      for (int d = 0; d < DIM; d++) {
        const int s = 1 << ((DIM - 1 - d) * lb);
        const bool per = L.bc.periodic[d] != 0, first = cb[d] == 0, last = cb[d] == nb - 1;
        B.lo[d] = first ? (per ? (nb - 1) * s : 0) : -s;
        B.hi[d] = last ? (per ? -(nb - 1) * s : 0) : s;
        if (!per) B.wall |= (first ? 1 << (2 * d) : 0) | (last ? 2 << (2 * d) : 0);
      }
      if (l == A.minlevel) {
#pragma unroll
        for (int p = 0; p < NC; p++) B.v[p] = T(0);
      } else {
        // cell q of the previous level: place, then block (one cell: both 0)
        auto at = [&](const int* q) {
          if (lp < 0) return prev[0];
          int p = 0, b = 0;
#pragma unroll
          for (int d = 0; d < DIM; d++) {
            p = p * 2 + (q[d] & 1);
            b = (b << lp) + (q[d] >> 1);
          }
          return prev[p * pplane + b];
        };
        bilinear_block<DIM, T>(cb, nb, A.L[l - 1].bc, at, B.v);
      }
      B.load(l == A.top ? L.res : rs + roff(l), L.k, g, idx, c, L.D2);
#pragma unroll
      for (int p = 0; p < NC; p++) f[p * plane] = B.v[p];
    }
    __syncthreads();
    for (int it = 0; it < A.nrelax; it++)
#pragma unroll
      for (int col = 0; col < 2; col++) {
        if (on) B.relax(col, f, plane, L.k.alpha, L.bc);
        __syncthreads();
      }
    if (on) {
#pragma unroll
      for (int p = 0; p < NC; p += 2) {
        idx_t at = idx;
#pragma unroll
        for (int e = 0; e < DIM - 1; e++)
          if (p & place_bit<DIM>(e)) at += g.stride(e);
        typename Vec2<T>::type w;
        w.x = B.v[p];
        w.y = B.v[p + 1];
        *reinterpret_cast<typename Vec2<T>::type*>(L.da + at) = w;
        if (A.a && l == A.top) {
          double2 x = *reinterpret_cast<const double2*>(A.a + at);
          x.x += (double)w.x;
          x.y += (double)w.y;
          *reinterpret_cast<double2*>(A.a + at) = x;
        }
      }
    }
  }
}

// --- the sweeps of one level, by tiles ------------------------------------
//
// ns sweeps of a level in one launch.  A workgroup loads a region of
// 2 B0 x 2 B1 (x 2 B2) cells, a thread per block, and relaxes all of it that
// lies in the level, 2 ns times.  Values next to the region's edge are wrong
// from the first half-sweep on and spread one cell per half-sweep, so a halo
// of 2 ns cells on every side that is not a wall or a whole dimension keeps
// the tile itself right; the tile (region minus halo) is written, to `out`.
// Along a periodic dimension the region's coordinates wrap.  The field comes
// from `dold`, or with `coarse` is the bilinear initial guess interpolated
// here; with `a` the launch ends the cycle and adds the correction to the
// solution too.
struct TileArgs {
  int ns;
  int tile[3];   // cells of a tile per dimension (even)
  int halo[3];   // 2 ns, or 0 where the region spans the dimension
  int ntile[3];
};

template <int DIM, typename T, bool ALPHAF, int B0, int B1, int B2>
__global__ __launch_bounds__(B0* B1* B2) void k_rb_tile(const T* __restrict__ dold, const T* __restrict__ coarse,
                                                        T* __restrict__ out, double* __restrict__ a,
                                                        const T* __restrict__ res, Coef<T> k, Geo<DIM> g, BCH bc,
                                                        BCH bcc, T D2, TileArgs A) {
  using V2 = typename Vec2<T>::type;
  constexpr int NC = 1 << DIM, NT = B0 * B1 * B2;
  constexpr int S0 = DIM == 3 ? B1 * B2 : B1, S1 = DIM == 3 ? B2 : 1;  // LDS strides of a block step
  // every place's plane has S0 words on either side, which the region's edge
  // blocks read for neighbours outside it
  constexpr int plane = NT + 2 * S0;
  __shared__ T buf[NC * plane];
  const int n = g.n, t = threadIdx.x;
  T* const f = buf + S0 + t;
  idx_t blk = logical_block();
  int tl[3] = {0, 0, 0};
#pragma unroll
  for (int d = DIM - 1; d >= 0; d--) {
    tl[d] = (int)(blk % (idx_t)A.ntile[d]);
    blk /= (idx_t)A.ntile[d];
  }
  const int r[3] = {t / S0, DIM == 3 ? t / S1 % B1 : t % S0, DIM == 3 ? t % S1 : 0};
  RBBlock<DIM, T, ALPHAF> B;
  B.wall = 0;
  int c[3] = {0, 0, 0};
  bool in = true, own = true;
#pragma unroll
  for (int d = 0; d < DIM; d++) {
    const int u = tl[d] * A.tile[d] - A.halo[d] + 2 * r[d];
    own = own && u >= tl[d] * A.tile[d] && u < (tl[d] + 1) * A.tile[d] && u < n;
    c[d] = bc.periodic[d] ? u & (n - 1) : u;
    in = in && c[d] >= 0 && c[d] < n;
    if (!bc.periodic[d]) B.wall |= (c[d] == 0 ? 1 << (2 * d) : 0) | (c[d] + 2 == n ? 2 << (2 * d) : 0);
    const int s = d == 0 ? S0 : d == 1 ? S1 : 1;
    B.lo[d] = -s;
    B.hi[d] = s;
  }
  const idx_t idx = in ? g.index(c) : 0u;
  if (in) {
    B.load(res, k, g, idx, c, D2);
    if (coarse) {
      const Geo<DIM> gc{n >> 1, g.log2n - 1};
      const int cc[3] = {c[0] >> 1, c[1] >> 1, c[2] >> 1};
      bilinear_block<DIM, T>(cc, gc.n, bcc, [&](const int* q) { return coarse[gc.index(q)]; }, B.v);
    } else {
#pragma unroll
      for (int p = 0; p < NC; p += 2) {
        idx_t at = idx;
#pragma unroll
        for (int e = 0; e < DIM - 1; e++)
          if (p & place_bit<DIM>(e)) at += g.stride(e);
        const V2 w = *reinterpret_cast<const V2*>(dold + at);
        B.v[p] = w.x;
        B.v[p + 1] = w.y;
      }
    }
#pragma unroll
    for (int p = 0; p < NC; p++) f[p * plane] = B.v[p];
  }
  __syncthreads();
  for (int it = 0; it < A.ns; it++)
#pragma unroll
    for (int col = 0; col < 2; col++) {
      if (in) B.relax(col, f, plane, k.alpha, bc);
      __syncthreads();
    }
  if (own) {
#pragma unroll
    for (int p = 0; p < NC; p += 2) {
      idx_t at = idx;
#pragma unroll
      for (int e = 0; e < DIM - 1; e++)
        if (p & place_bit<DIM>(e)) at += g.stride(e);
      V2 w;
      w.x = B.v[p];
      w.y = B.v[p + 1];
      *reinterpret_cast<V2*>(out + at) = w;
      if (a) {
        double2 x = *reinterpret_cast<const double2*>(a + at);
        x.x += (double)w.x;
        x.y += (double)w.y;
        *reinterpret_cast<double2*>(a + at) = x;
      }
    }
  }
}

}  // namespace bmg
