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
#pragma once

#include "flow_kernels.h"

namespace cg {

// What a k_tile launch computes: kTilePcg the alpha half of an iteration and z, kTileSolve
// out = (L L^T)^-1 in, kTileFwd out = L^-1 in, kTileBwd out = L^-T in.
enum TileMode { kTilePcg = 0, kTileSolve, kTileFwd, kTileBwd };
constexpr int kTileThreads = 1024;  // at most; a launch takes as many as a phase has rows
// LDS: x / y of the tile's columns, the recurrence coefficients of a phase
inline size_t tile_lds(int nloc, int coef, int len) { return sizeof(double) * (size_t)(nloc + coef) * len; }

template <typename FT, int MODE, int RPT>
__global__ void k_tile(TileSet T, TileCols C, const FT *F, TilePcg P, const double *in, double *out,
                       const int *done);
__global__ void k_spmv_beta(Sell sl, FacTab ft, TilePcg P, int ntile);
__global__ void k_pcg_check(TilePcg P, int ntile);
template <typename FT, int MODE, int RPT>
__global__ void kb_tile(const int *start, int nmem, const MemberDev *md, int vin, int vout);
__global__ void kb_spmv_beta(const int *start, int nmem, const MemberDev *md);
__global__ void kb_pcg_check(const int *start, int nmem, const MemberDev *md);

}  // namespace cg
