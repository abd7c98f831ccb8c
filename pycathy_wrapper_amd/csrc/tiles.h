// tiles.h -- the column preconditioner and the PCG iteration of small and
// medium meshes in two launches (tile_kernels.hip).
//
// In the column ordering z = (L L^T)^-1 t takes five dependent launches (three
// colours forward, two back).  A mesh of up to a few hundred thousand nodes does not fill
// them: a launch of 4 - 8 us moves what takes 1 us.  Here the surface is cut
// into tiles of neighbouring columns, one work-group each, and a work-group
// computes all five phases for its tile in LDS.  A phase needs the results of the
// one before on neighbouring columns too, so each phase runs on the tile
// plus the columns the later phases reach (about twice the tile's own rows in all),
// recomputed by every tile that needs them: no work-group waits for another.
// Every row is computed by the same operations wherever it is computed, so
// the copies agree bit for bit.
//
// The recomputed rows and the factor read again are free only while the GPU has room.
// Where solves share it, the same mesh runs by the colour launches (Flow::crowded), with
// its columns' recurrences level by level and its sums by tile, as here: the same bits.
#pragma once

#include "flow_kernels.h"

namespace cg {

// What a k_tile launch computes: kTilePcg the alpha half of an iteration and z, kTileSolve
// out = (L L^T)^-1 in, kTileFwd out = L^-1 in, kTileBwd out = L^-T in.
enum TileMode { kTilePcg = 0, kTileSolve, kTileFwd, kTileBwd };
constexpr int kTileThreads = 1024;  // at most; a launch takes as many as a phase has rows
// LDS: x / y of the tile's columns, the recurrence coefficients of a phase
inline size_t tile_lds(int nloc, int coef, int len) { return sizeof(double) * (size_t)(nloc + coef) * len; }

// Sums of two partial arrays in a fixed order by the first 256 threads of a
// work-group of any size, in every thread (sh: 16 doubles).
// U: partials per thread and array that are loaded without a wait between them.
template <int U>
struct Partials {
  double a[U], b[U];
};
template <int U>
__device__ __forceinline__ Partials<U> partials_load(const double *pa, const double *pb, int cnt) {
  Partials<U> q{};
  if (threadIdx.x < 256) {
    int i = threadIdx.x;
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (i + 256 * u < cnt) {
        q.a[u] = pa[i + 256 * u];
        q.b[u] = pb[i + 256 * u];
      }
    for (i += 256 * U; i < cnt; i += 256) {
      q.a[0] += pa[i];
      q.b[0] += pb[i];
    }
  }
  return q;
}
template <int U>
__device__ __forceinline__ double2 partials_sum(const Partials<U> &q, double *sh) {
  if (threadIdx.x < 256) {
    double va = q.a[0], vb = q.b[0];
#pragma unroll
    for (int u = 1; u < U; ++u) {
      va += q.a[u];
      vb += q.b[u];
    }
    va = wave_sum(va);
    vb = wave_sum(vb);
    if ((threadIdx.x & 63) == 0) {
      sh[2 * (threadIdx.x >> 6)] = va;
      sh[2 * (threadIdx.x >> 6) + 1] = vb;
    }
  }
  __syncthreads();
  const double2 t = make_double2((sh[0] + sh[2]) + (sh[4] + sh[6]), (sh[1] + sh[3]) + (sh[5] + sh[7]));
  __syncthreads();
  return t;
}
// Block sums of two values, in thread 0 (sh: 2 * waves doubles).
__device__ __forceinline__ double2 tile_sum2(double a, double b, double *sh) {
  a = wave_sum(a);
  b = wave_sum(b);
  const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    sh[2 * w] = a;
    sh[2 * w + 1] = b;
  }
  __syncthreads();
  double2 t = make_double2(0.0, 0.0);
  if (threadIdx.x == 0)
    for (int k = 0; k < nw; ++k) {
      t.x += sh[2 * k];
      t.y += sh[2 * k + 1];
    }
  return t;
}

// The recurrence v_k = b_k - a_k v_(k -+ 1) of one column in place (v: b in, v out,
// planes nloc apart; a: planes cnt apart), k ascending or, UP, descending; SCALE
// stores v_k d_k instead.  Eight levels' coefficients are in registers ahead of
// the serial part: the LDS stores would otherwise hold back the loads.
template <bool UP, bool SCALE>
__device__ __forceinline__ void tile_chain(double *v, int nloc, const double *a, const double *d, int cnt, int len) {
  const int sv = UP ? -nloc : nloc, sa = UP ? -cnt : cnt;
  if (UP) {
    v += (len - 1) * nloc;
    a += (len - 1) * cnt;
  }
  double y = 0.0;
  int k = 0;
  for (; k + 8 <= len; k += 8) {
    double b[8], c[8], e[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      b[u] = v[u * sv];
      c[u] = a[u * sa];
      if (SCALE) e[u] = d[u * sa];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      y = fma(-c[u], y, b[u]);
      v[u * sv] = SCALE ? y * e[u] : y;
    }
    v += 8 * sv;
    a += 8 * sa;
    if (SCALE) d += 8 * sa;
  }
  if (k < len) {  // the last levels: reads past the end stay on the last one
    const int m = len - 1 - k;
    double b[8], c[8], e[8];
#pragma unroll
    for (int u = 0; u < 7; ++u) {
      const int q = min(u, m);
      b[u] = v[q * sv];
      c[u] = a[q * sa];
      if (SCALE) e[u] = d[q * sa];
    }
#pragma unroll
    for (int u = 0; u < 7; ++u) {
      if (u > m) break;
      y = fma(-c[u], y, b[u]);
      v[u * sv] = SCALE ? y * e[u] : y;
    }
  }
}

template <typename FT, int MODE, int RPT>
__global__ void k_tile(TileSet T, TileCols C, const FT *F, TilePcg P, const double *in, double *out,
                       const int *done);
__global__ void k_spmv_beta(Sell sl, FacTab ft, TilePcg P, int ntile);
__global__ void k_pcg_check(TilePcg P, int ntile);
template <int RPT>
__global__ void k_tile_dots(TileSet T, TileCols C, TilePcg P);
template <typename FT, int MODE, int RPT>
__global__ void kb_tile(const int *start, int nmem, const MemberDev *md, int vin, int vout);
__global__ void kb_spmv_beta(const int *start, int nmem, const MemberDev *md);
__global__ void kb_pcg_check(const int *start, int nmem, const MemberDev *md);
template <int RPT>
__global__ void kb_tile_dots(const int *start, int nmem, const MemberDev *md);

}  // namespace cg
