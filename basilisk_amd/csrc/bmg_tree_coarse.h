// libbmg: the uniform coarse levels of a tree's cycle on chip.
//
// The levels of a tree without leaves above them are full grids, stored in
// cache order: the 2^dim children of a cell are consecutive slots, which is
// the block of cells a thread owns in k_coarse_rb.  This is that kernel on
// slots: levels minlevel..top (at most 32^2 or 16^3 cells) in one workgroup,
// restriction of res, initial guesses and red-black sweeps.  As batched small
// operations each half-sweep was a chain of dependent loads through the
// tables, 2.6 us; here it takes 0.2 us (levels 1-5 of a quadtree 170 -> 24
// us a cycle, FP64; 1-4 of an octree 133 -> 38 us, FP32).
#pragma once

#include "bmg_block_kernels.h"
#include "bmg_tree_kernels.h"

namespace bmgt {

constexpr int kCoarseTop = 5;

template <typename T>
struct TreeCoarse {
  T *da, *res;
  RelaxCoef<T> k;
  const int* nbr;
  bmg::BCH bc;
  int minlevel, top, nrelax;
  int off[kCoarseTop + 1], abase[kCoarseTop + 1];  // first slot, first entry of the neighbour table
  T D2[kCoarseTop + 1];
};

// cache order of the cells of a full level: the bits of the coordinates
// interleaved, the last dimension's lowest
template <int DIM>
__host__ __device__ __forceinline__ int cache_index(const int c[3], int bits) {
  int r = 0;
  for (int b = 0; b < bits; b++)
    for (int d = 0; d < DIM; d++) r |= ((c[d] >> b) & 1) << (DIM * b + DIM - 1 - d);
  return r;
}
template <int DIM>
__host__ __device__ __forceinline__ void cache_cell(int r, int bits, int c[3]) {
  for (int d = 0; d < 3; d++) c[d] = 0;
  for (int b = 0; b < bits; b++)
    for (int d = 0; d < DIM; d++) c[d] |= ((r >> (DIM * b + DIM - 1 - d)) & 1) << b;
}

template <int DIM, typename T, bool ALPHAF>
__global__ __launch_bounds__((bmg::kCoarseThreads<DIM, T, ALPHAF>)) void k_t_coarse(TreeCoarse<T> A) {
  constexpr int NC = 1 << DIM, kBlocks = bmg::kCoarseThreads<DIM, T, ALPHAF>;
  __shared__ T big[NC * kBlocks], small[kBlocks], rs[2 * kBlocks];
  const int t = threadIdx.x;
  auto roff = [](int l) { return ((1 << (DIM * l)) - 1) / (NC - 1); };
  // (the levels below minlevel too: relax() may read their res)
  for (int l = A.top - 1; l >= 0; l--) {
    for (int q = t; q < 1 << (DIM * l); q += (int)blockDim.x) {
      const T* c = l + 1 == A.top ? A.res + A.off[l + 1] + q * NC : rs + roff(l + 1) + q * NC;
      T sum = T(0);
#pragma unroll
      for (int m = 0; m < NC; m++) sum += c[m];
      sum = sum / T(NC);
      rs[roff(l) + q] = sum;
      A.res[A.off[l] + q] = sum;
    }
    __syncthreads();
  }
  for (int l = A.minlevel; l <= A.top; l++) {
    const int lb = l - 1, nb = 1 << lb, plane = 1 << (DIM * lb);
    T* cur = ((A.top - l) & 1) == 0 ? big : small;
    const T* prev = ((A.top - l) & 1) == 0 ? small : big;
    const bool on = t < plane;
    const int s0 = A.off[l] + t * NC;
    bmg::RBBlock<DIM, T, ALPHAF> B;
    T* f = cur + t;
    if (on) {
      int cb[3];
      cache_cell<DIM>(t, lb, cb);
      B.wall = 0;
#pragma unroll
      for (int d = 0; d < DIM; d++) {
        const bool first = cb[d] == 0, last = cb[d] == nb - 1;
        int q[3] = {cb[0], cb[1], cb[2]};
        q[d] = first ? cb[d] : cb[d] - 1;
        B.lo[d] = cache_index<DIM>(q, lb) - t;
        q[d] = last ? cb[d] : cb[d] + 1;
        B.hi[d] = cache_index<DIM>(q, lb) - t;
        B.wall |= (first ? 1 << (2 * d) : 0) | (last ? 2 << (2 * d) : 0);
      }
      if (l == A.minlevel) {
#pragma unroll
        for (int p = 0; p < NC; p++) B.v[p] = T(0);
      } else {
        auto at = [&](const int* q) {
          int p = 0, h[3];
#pragma unroll
          for (int d = 0; d < 3; d++) {
            if (d < DIM) p = p * 2 + (q[d] & 1);
            h[d] = q[d] >> 1;
          }
          return prev[p * (plane >> DIM) + cache_index<DIM>(h, lb - 1)];
        };
        bmg::bilinear_block<DIM, T>(cb, nb, A.bc, at, B.v);
      }
      const T* res = l == A.top ? A.res + s0 : rs + roff(l) + t * NC;
      const int* nb0 = A.nbr + (size_t)(A.abase[l] + t * NC) * 2 * DIM;
#pragma unroll
      for (int p = 0; p < NC; p++) {
        B.m[p] = -A.D2[l] * res[p];
        B.d[p] = -(A.k.lam ? A.k.lam[s0 + p] : A.k.lam_c) * A.D2[l];
        if (ALPHAF) {
#pragma unroll
          for (int e = 0; e < DIM; e++) {
            const bool up = p & bmg::place_bit<DIM>(e);
            const int a = ALPHAF ? B.across(p, e) : 0;
            B.face[ALPHAF ? e : 0][up ? 1 : 0][a] = A.k.alpha[e][s0 + p];
            if (up) B.face[ALPHAF ? e : 0][2][a] = A.k.alpha[e][nb0[p * 2 * DIM + 2 * e + 1]];
          }
        }
      }
#pragma unroll
      for (int p = 0; p < NC; p++)
#pragma unroll
        for (int e = 0; e < DIM; e++) {
          if (ALPHAF) B.d[p] += B.high(p, e) + B.low(p, e);
          else B.d[p] += A.k.alpha_c + A.k.alpha_c;
        }
#pragma unroll
      for (int p = 0; p < NC; p++) f[p * plane] = B.v[p];
    }
    __syncthreads();
    for (int it = 0; it < A.nrelax; it++)
#pragma unroll
      for (int col = 0; col < 2; col++) {
        if (on) B.relax(col, f, plane, A.k.alpha_c, A.bc);
        __syncthreads();
      }
    if (on) {
#pragma unroll
      for (int p = 0; p < NC; p++) A.da[s0 + p] = B.v[p];
    }
  }
}

}  // namespace bmgt
