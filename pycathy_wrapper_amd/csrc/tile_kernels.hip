// tile_kernels.hip -- the column preconditioner over surface tiles and the PCG
// iteration in two launches (tiles.h).
#include "tiles.h"

#include <type_traits>

namespace cg {

// Element i of an array of fewer than 2^32 bytes: one 32-bit offset on a uniform base.
template <typename T>
__device__ __forceinline__ T at(const T *p, int i) {
  return *(const T *)((const char *)p + (size_t)((uint32_t)i * (uint32_t)sizeof(T)));
}
template <typename T>
__device__ __forceinline__ void put(T *p, int i, T v) {
  *(T *)((char *)p + (size_t)((uint32_t)i * (uint32_t)sizeof(T))) = v;
}

// The stopping test after iteration `it` (graddp.f:1348-1377) from its
// partials; every work-group takes it alike.
struct PcgTest {
  double err, beta;
  bool stop;
};
__device__ __forceinline__ PcgTest pcg_test(const TilePcg &P, const Partials<1> &q, int it, double *sh) {
  const double2 s = partials_sum(q, sh);
  PcgTest t;
  t.beta = -s.x / P.sc->pb;
  const double xl = P.sc->xlung;
  t.err = xl > 0.0 ? sqrt(s.y / xl) : sqrt(s.y / P.n);
  t.stop = !(t.err > P.sc->tol && it < P.sc->imax);
  return t;
}

// ----------------------------------------------- first launch: p, B = A p --
// Iteration b = it + 1: the stopping test of iteration it (b > 1), then p = z + beta p
// formed for the row and for each neighbour it gathers (the same fma
// everywhere), B = A p and partial (p, r), (p, B).  Joins k_pcg_beta to k_spmv_dot2
// for one more gather per entry.  The scalars a launch reads (it) are written by the
// other launch of the iteration, those it writes (niter, err, stop) it does
// not read.  Bound: the dependent loads (slice offset, column code, neighbour)
// on small meshes, in flight together with the partials; the gathers on large ones.
// 7.9 us at 4,851 nodes, 16.9 at 214,221, 12.9 at 8 x 26,896 (k_spmv_dot2 and
// k_pcg_beta before: 13, 24 and 16 us).  Held to four waves per SIMD it spills: 9.0 and
// 19.8 us.
__device__ __forceinline__ void spmv_beta_body(Blk bk, const Sell &sl, const FacTab &ft, const TilePcg &P, int ntile) {
  __shared__ double sh[16];
  const int stopped = *P.done, it = P.sc->it;
  const Partials<1> q = partials_load<1>(P.part_bz, P.part_rr, ntile);
  const int i = bk.b * blockDim.x + threadIdx.x;
  const bool on = i < P.n;
  double a[kUnroll], zv[kUnroll], v[kUnroll], zi = 0.0, pi = 0.0, ri = 0.0;
  int w = 0, c[kUnroll];
  // every load of the row goes out before the partials are summed
  if (on) {
    const int s = __builtin_amdgcn_readfirstlane(i >> 6);
    const int o0 = sl.so[s], q0 = o0 + (i & 63);
    w = (sl.so[s + 1] - o0) >> 6;
    const RowPos rp = row_pos(sl, i);
    uint32_t cw[kUnroll];
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) cw[j] = code_word(sl, rp, min(j, w - 1));
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) c[j] = j < w ? code_col(sl, rp.k, cw[j]) : 0;
    if (ft.w) {  // lower entries through the transpose (see sell_row_dot_sym)
      const int jd = sell_diag(sl, rp, i);
      const uint32_t *tw = ft.w + (size_t)fac_class(rp.k, sl.nplane) * kFacWords * ft.nchain + rp.g;
      uint32_t wt[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) wt[u] = tw[(size_t)(34 + u) * ft.nchain];
#pragma unroll
      for (int j = 0; j < kUnroll; ++j) {
        const int b = (int)((wt[j >> 2] >> (8 * (j & 3))) & 0xFFu);
        a[j] = P.A[j < jd ? sl.so[c[j] >> 6] + (c[j] & 63) + 64 * b : (j < w ? q0 + 64 * j : 0)];
      }
    } else {
#pragma unroll
      for (int j = 0; j < kUnroll; ++j) a[j] = P.A[j < w ? q0 + 64 * j : 0];
    }
  }
  if (stopped) return;
  const double *po = P.p[(it + 1) & 1], *r = P.r[it & 1];
  double *pn = P.p[it & 1];
  // iteration 1 takes p as it is: the same loads, from p in place of z
  const double *po1 = it > 0 ? po : pn, *z = it > 0 ? P.z : pn;
  if (on) {
    zi = at(z, i);
    pi = at(po1, i);
    ri = at(r, i);
#pragma unroll
    for (int j = 0; j < kUnroll; ++j) {
      zv[j] = at(z, c[j]);
      v[j] = at(po1, c[j]);
    }
  }
  double beta = 0.0;
  if (it > 0) {
    const PcgTest t = pcg_test(P, q, it, sh);
    if (bk.b == 0 && threadIdx.x == 0) {
      P.sc->err = t.err;
      if (t.stop) P.sc->stop = 1;
    }
    if (t.stop) return;
    beta = t.beta;
  }
  if (bk.b == 0 && threadIdx.x == 0) P.sc->niter = it + 1;
  double apr = 0.0, apb = 0.0;
  if (on) {
    double acc = 0.0;
    if (it > 0) {
#pragma unroll
      for (int j = 0; j < kUnroll; ++j) acc = fma(j < w ? a[j] : 0.0, fma(beta, v[j], zv[j]), acc);
      pi = fma(beta, pi, zi);
      pn[i] = pi;
    } else {
#pragma unroll
      for (int j = 0; j < kUnroll; ++j) acc = fma(j < w ? a[j] : 0.0, v[j], acc);
    }
    P.B[i] = acc;
    apr = pi * ri;
    apb = pi * acc;
  }
  const double2 t = tile_sum2(apr, apb, sh);
  if (threadIdx.x == 0) {
    P.part_pr[bk.b] = t.x;
    P.part_pb[bk.b] = t.y;
  }
}
__global__ __launch_bounds__(kBlock) void k_spmv_beta(Sell sl, FacTab ft, TilePcg P, int ntile) {
  spmv_beta_body(self_xcd_blk(), sl, ft, P, ntile);
}

// The stopping test of the last iteration of a launch batch, before the host reads
// the flag (the next batch's first launch would take it again, alike).
__device__ __forceinline__ void pcg_check_body(const TilePcg &P, int ntile) {
  if (P.sc->stop) return;
  __shared__ double sh[16];
  const PcgTest t = pcg_test(P, partials_load<1>(P.part_bz, P.part_rr, ntile), P.sc->it, sh);
  if (threadIdx.x == 0) {
    P.sc->err = t.err;
    if (t.stop) P.sc->stop = 1;
    else P.sc->niter = P.sc->it + 1;
  }
}
__global__ __launch_bounds__(256) void k_pcg_check(TilePcg P, int ntile) { pcg_check_body(P, ntile); }

// --------------------------------------- second launch: alpha, r, x, z, (B, z) --
// Bound: five phases one after the other, each of them first-touch load latency,
// the serial recurrences along the columns (8 - 25 cycles a level) and four LDS
// barriers; on the largest meshes also the factor, read two to three times through L2.
// Loads run ahead across the barriers (lds_barrier leaves them under way).
// 13.3 us at 4,851 nodes, 25 at 214,221, 25 at 8 x 26,896; the five sweep launches,
// alpha and (B, z) took 29, 34 and 32 us.  16 columns a tile instead of 25: 30 us at
// 8 x 26,896 (more copies of the columns between tiles), 13.9 at 4,851.
// A row of a phase.  Its ids and table words are loaded two phases ahead, its
// factor entries, 1 / L_rr and right-hand side one phase ahead: a first touch of a
// line in a launch costs 0.8 us, as much as a phase computes.
struct TileIds {
  int v, i, k;       // LDS index of its value, item within the phase (-1: none), plane
  int2 rb;           // row id, SELL position of its slot 0
  uint32_t meta, w[kTileSlots / 2];
};
template <typename FT>
struct TileRow {
  FT f[kTileSlots], fc, fu;  // window, the chain's entry, the successor's where the last colour turns round
  double di, t, b;           // 1 / L_rr, right-hand side, B of the row (alpha update)
};

// Entry e of a row's packed words: LDS index of the neighbour, from that of the
// tile's first column one plane up.
__device__ __forceinline__ int tile_nbr(const uint32_t (&w)[kTileSlots / 2], int e, int above) {
  return above + (int)((w[e >> 1] >> (16 * (e & 1))) & 0xFFFFu);
}

// RPT: rows of a phase per thread (the host checks that every phase fits).  flag: the
// launch returns where it is set (null: never).
template <typename FT, int MODE, int RPT>
__device__ __forceinline__ void tile_body(Blk bk, double *smem, const TileSet &T, const TileCols &C,
                                          const FT *__restrict__ F, const TilePcg &P, const double *__restrict__ in,
                                          double *out, const int *flag) {
  __shared__ double sh[2 * kTileThreads / 64];
  const int stopped = flag ? *flag : 0;
  const TileDesc d = T.desc[bk.b];
  const int body = MODE == kTilePcg ? P.sc->niter : 0;  // written by this iteration's first launch
  if (stopped) {
    if (MODE == kTilePcg && bk.b == 0 && threadIdx.x == 0) *P.done = 1;  // the flag read is sc->stop (see PcgScal)
    return;
  }
  const int len = C.c[0].len, kl = len - 1, tid = threadIdx.x, nt = T.threads;
  const int off1 = d.n[0], off2 = d.n[0] + d.n[1], nloc = off2 + d.n[2];
  double *V = smem, *W = smem + nloc * len;  // y / x by [plane][column]; coefficients of a phase
  const int2 *rows = T.rows + d.row;
  const double *ro = nullptr, *pc = nullptr;
  double *rn = nullptr;
  if (MODE == kTilePcg) {
    ro = P.r[(body - 1) & 1];
    rn = P.r[body & 1];
    pc = P.p[(body - 1) & 1];
  }
  TileIds S[RPT], X[RPT];
  TileRow<FT> R[RPT];
  double alfa = 0.0, rr = 0.0, bz = 0.0;
  // ids of a phase over cnt columns from l0; BACK: backward sweep; NW: its entry
  // window (0: none)
  auto ids = [&](auto back, auto win, int l0, int cnt) {
    constexpr bool BACK = decltype(back)::value;
    constexpr int NW = decltype(win)::value;
    int k = cnt > 0 && tid < nt ? tid / cnt : len, l = cnt > 0 ? tid - k * cnt : 0;
    const int dk = cnt > 0 ? nt / cnt : 0, dl = cnt > 0 ? nt - dk * cnt : 0;
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      TileIds &Y = S[u];
      Y.i = -1;
      if (k < len) {
        Y.k = k;
        Y.i = __mul24(k, cnt) + l;
        Y.v = __mul24(k, nloc) + l0 + l;
        Y.rb = at(rows, Y.v);
        const int tw = (k == 0 ? 0 : (k == kl ? 2 : 1)) * kTileWords * T.ntot + d.off + l0 + l;
        Y.meta = at(T.tab + (size_t)(kTileWords - 1) * T.ntot, tw);
#pragma unroll
        for (int q = 0; q < NW / 2; ++q) Y.w[q] = at(T.tab + (size_t)((BACK ? kTileSlots / 2 : 0) + q) * T.ntot, tw);
      }
      k += dk;
      l += dl;
      if (cnt > 0 && l >= cnt) {
        l -= cnt;
        k += 1;
      }
    }
  };
  // values of the phase whose ids are in S (kept in X)
  auto load = [&](auto back, auto turn, auto win) {
    constexpr bool BACK = decltype(back)::value, TURN = decltype(turn)::value;
    constexpr int NW = decltype(win)::value;
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      X[u] = S[u];
      if (S[u].i < 0) continue;
      TileRow<FT> &Y = R[u];
      const int k = S[u].k, r = S[u].rb.x, base = S[u].rb.y, jd = (int)(S[u].meta & 0xFFu);
      // one offset per row; a window of slots from it, 64 apart (the factor's
      // allocation holds a window past its last slot)
      const int f0 = base + 64 * (BACK ? jd + (k < kl ? 2 : 1) : 0), q = base + 64 * jd;
      const FT *f = (const FT *)((const char *)F + (size_t)((uint32_t)f0 * (uint32_t)sizeof(FT)));
#pragma unroll
      for (int j = 0; j < NW; ++j) Y.f[j] = f[64 * j];
      Y.fc = BACK ? (k < kl ? at(F, q + 64) : FT(0)) : (k > 0 ? at(F, q - 64) : FT(0));
      if (TURN) Y.fu = k < kl ? at(F, q + 64) : FT(0);
      Y.di = at(P.dinv, r);
      if (!BACK || MODE == kTileBwd) Y.t = MODE == kTilePcg ? at(ro, r) : at(in, r);
      if (MODE == kTilePcg && !BACK) Y.b = at((const double *)P.B, r);
    }
  };
  // a phase's rows: b_k = (t - sum f v) / L_rr into V, the chain's coefficients into W
  auto solve = [&](auto back, auto turn, auto win, int cnt, int own) {
    constexpr bool BACK = decltype(back)::value, TURN = decltype(turn)::value;
    constexpr int NW = decltype(win)::value;
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      if (X[u].i < 0) continue;
      TileRow<FT> &Y = R[u];
      const int k = X[u].k, r = X[u].rb.x, nj = (int)((X[u].meta >> (BACK ? 16 : 8)) & 0xFFu);
      double s = BACK && MODE != kTileBwd ? V[X[u].v] : Y.t;
      if (MODE == kTilePcg && !BACK) {
        s = fma(-alfa, Y.b, s);
        if (X[u].i - __mul24(k, cnt) < own) {  // the tile's own rows take the alpha update
          put(rn, r, s);
          put(P.x, r, fma(alfa, at(pc, r), at((const double *)P.x, r)));
          if (!at(P.isdir, r)) rr = fma(s, s, rr);
        }
      }
      if (NW > 0) {
        const int above = __mul24(k - 1, nloc);
        double yv[NW > 0 ? NW : 1];
#pragma unroll
        for (int j = 0; j < NW; ++j) yv[j] = V[tile_nbr(X[u].w, j, above)];
#pragma unroll
        for (int j = 0; j < NW; ++j) s = j < nj ? fma(-(double)Y.f[j], yv[j], s) : s;
      }
      V[X[u].v] = s * Y.di;
      W[X[u].i] = (double)Y.fc * Y.di;
      if (TURN) {
        W[__mul24(cnt, len) + X[u].i] = (double)Y.fu * Y.di;
        W[2 * __mul24(cnt, len) + X[u].i] = Y.di;
      }
    }
  };
  const std::integral_constant<bool, true> yes{};
  const std::integral_constant<bool, false> no{};
  const std::integral_constant<bool, MODE != kTileFwd> turn{};
  const std::integral_constant<int, 0> w0{};
  const std::integral_constant<int, kTileSlots1> w1{};
  const std::integral_constant<int, kTileSlots> w2{};
  // own rows (columns o of the three colours in turn): LDS index and row id
  const int nown = d.own[0] + d.own[1] + d.own[2];
  auto own_ids = [&] {
    int k = nown > 0 && tid < nt ? tid / nown : len, o = nown > 0 ? tid - k * nown : 0;
    const int dk = nown > 0 ? nt / nown : 0, dl = nown > 0 ? nt - dk * nown : 0;
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      S[u].i = -1;
      if (k < len) {
        const int l = o < d.own[0] ? o : (o < d.own[0] + d.own[1] ? off1 + o - d.own[0] : off2 + o - d.own[0] - d.own[1]);
        S[u].i = 0;
        S[u].v = __mul24(k, nloc) + l;
        S[u].rb = at(rows, S[u].v);
      }
      k += dk;
      o += dl;
      if (nown > 0 && o >= nown) {
        o -= nown;
        k += 1;
      }
    }
  };
  if (MODE != kTileBwd) {
    Partials<4> q{};
    if (MODE == kTilePcg) q = partials_load<4>(P.part_pr, P.part_pb, (P.n + kBlock - 1) / kBlock);
    ids(no, w0, 0, d.n[0]);
    load(no, no, w0);
    ids(no, w1, off1, d.n[1]);
    if (MODE == kTilePcg) {
      const double2 s = partials_sum(q, sh);
      alfa = s.x / s.y;
      if (bk.b == 0 && tid == 0) {
        P.sc->pb = s.y;
        P.sc->alpha = alfa;
        P.sc->it = body;
      }
    }
    solve(no, no, w0, d.n[0], d.own[0]);
    load(no, no, w1);
    ids(no, w2, off2, d.n[2]);
    lds_barrier();
    if (tid < d.n[0]) tile_chain<false, false>(V + tid, nloc, W + tid, nullptr, d.n[0], len);
    lds_barrier();
    solve(no, no, w1, d.n[1], d.own[1]);
    load(no, turn, w2);
    if (MODE != kTileFwd) ids(yes, w1, off1, d.x1);
    lds_barrier();
    if (tid < d.n[1]) tile_chain<false, false>(V + off1 + tid, nloc, W + tid, nullptr, d.n[1], len);
    lds_barrier();
    solve(no, turn, w2, d.n[2], d.own[2]);
  } else {
    ids(yes, w0, off2, d.n[2]);
    load(yes, no, w0);
    ids(yes, w1, off1, d.x1);
    solve(yes, no, w0, d.n[2], 0);
  }
  if (MODE != kTileFwd) {
    load(yes, no, w1);
    ids(yes, w2, 0, d.own[0]);
  } else {
    own_ids();
  }
  lds_barrier();
  if (tid < d.n[2]) {
    double *v = V + off2 + tid, *w = W + tid;
    const int cnt = d.n[2];
    if (MODE == kTileBwd) {
      tile_chain<true, false>(v, nloc, w, nullptr, cnt, len);
    } else if (MODE == kTileFwd) {
      tile_chain<false, false>(v, nloc, w, nullptr, cnt, len);
    } else {  // down, then x_k = y_k d_k - u_k x_(k+1) up
      tile_chain<false, true>(v, nloc, w, w + 2 * cnt * len, cnt, len);
      tile_chain<true, false>(v, nloc, w + cnt * len, nullptr, cnt, len);
    }
  }
  lds_barrier();
  if (MODE != kTileFwd) {
    solve(yes, no, w1, d.x1, 0);
    load(yes, no, w2);
    own_ids();
    lds_barrier();
    if (tid < d.x1) tile_chain<true, false>(V + off1 + tid, nloc, W + tid, nullptr, d.x1, len);
    lds_barrier();
    solve(yes, no, w2, d.own[0], 0);
    double B[RPT];
    if (MODE == kTilePcg)
#pragma unroll
      for (int u = 0; u < RPT; ++u) B[u] = S[u].i >= 0 ? at((const double *)P.B, S[u].rb.x) : 0.0;
    lds_barrier();
    if (tid < d.own[0]) tile_chain<true, false>(V + tid, nloc, W + tid, nullptr, d.own[0], len);
    lds_barrier();
    if (MODE == kTilePcg)
#pragma unroll
      for (int u = 0; u < RPT; ++u)
        if (S[u].i >= 0) bz = fma(B[u], V[S[u].v], bz);
  }
#pragma unroll
  for (int u = 0; u < RPT; ++u)
    if (S[u].i >= 0) put(out, S[u].rb.x, V[S[u].v]);
  if (MODE == kTilePcg) {
    const double2 t = tile_sum2(bz, rr, sh);
    if (tid == 0) {
      P.part_bz[bk.b] = t.x;
      P.part_rr[bk.b] = t.y;
    }
  }
}
template <typename FT, int MODE, int RPT>
__global__ __launch_bounds__(kTileThreads) void k_tile(TileSet T, TileCols C, const FT *F, TilePcg P,
                                                       const double *in, double *out, const int *done) {
  extern __shared__ double smem[];
  tile_body<FT, MODE, RPT>(self_xcd_blk(), smem, T, C, F, P, in, out, MODE == kTilePcg ? &P.sc->stop : done);
}
#define CG_INST_TILE(FT, MODE)                                                                                       \
  template __global__ void k_tile<FT, MODE, 1>(TileSet, TileCols, const FT *, TilePcg, const double *, double *, const int *); \
  template __global__ void k_tile<FT, MODE, 2>(TileSet, TileCols, const FT *, TilePcg, const double *, double *, const int *);
#define CG_INST_TILES(FT)                                                                        \
  CG_INST_TILE(FT, kTilePcg) CG_INST_TILE(FT, kTileSolve) CG_INST_TILE(FT, kTileFwd) CG_INST_TILE(FT, kTileBwd)
CG_INST_TILES(float)
CG_INST_TILES(double)
#undef CG_INST_TILES
#undef CG_INST_TILE

// ---------------------- the dots of a tile's own rows, for the colour launches --
// (B, z) and ||r||^2 by tile, by the thread and in the order k_tile takes them: a mesh on tiles
// whose solve runs by the colour launches (Flow::crowded) sums the same partials, so the
// two ways give the same bits.  Takes the place of k_dot.  A tile's own columns of a colour
// are neighbouring chains, so their rows follow from the first.  Bound by latency: the values of all
// items go out together (threads without a row read the tile's first).  16 x 26,896 nodes 9.8 us (k_dot 3.8);
// phase after phase, with the rows read from the table, 11.7.
template <int RPT>
__device__ __forceinline__ void tile_dots_body(Blk bk, const TileSet &T, const TileCols &C, const TilePcg &P) {
  __shared__ double sh[2 * kTileThreads / 64];
  const int stopped = *P.done;
  const TileDesc d = T.desc[bk.b];
  if (stopped) return;
  const int tid = threadIdx.x, nt = T.threads, len = C.c[0].len;
  const int off1 = d.n[0], off2 = d.n[0] + d.n[1], nown = d.own[0] + d.own[1] + d.own[2];
  // first own row of each colour (surface plane)
  const int2 *rows = T.rows + d.row;
  const int row0[3] = {d.own[0] > 0 ? rows[0].x : 0, d.own[1] > 0 ? rows[off1].x : 0,
                       d.own[2] > 0 ? rows[off2].x : 0};
  const int any = d.own[0] > 0 ? row0[0] : (d.own[1] > 0 ? row0[1] : row0[2]);
  // phase c's items as k_tile's solve takes them (c = 3: its own rows)
  int r[4][RPT];
  bool on[4][RPT];
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const int cnt = c < 3 ? d.n[c] : nown, own = c < 3 ? d.own[c] : nown;
    int k = cnt > 0 && tid < nt ? tid / cnt : len, l = cnt > 0 ? tid - k * cnt : 0;
    const int dk = cnt > 0 ? nt / cnt : 0, dl = cnt > 0 ? nt - dk * cnt : 0;
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      on[c][u] = k < len && l < own;
      int row;
      if (c < 3) row = row0[c] + k * C.c[c].nc + l;
      else if (l < d.own[0]) row = row0[0] + k * C.c[0].nc + l;
      else if (l < d.own[0] + d.own[1]) row = row0[1] + k * C.c[1].nc + l - d.own[0];
      else row = row0[2] + k * C.c[2].nc + l - d.own[0] - d.own[1];
      r[c][u] = on[c][u] ? row : any;
      k += dk;
      l += dl;
      if (cnt > 0 && l >= cnt) {
        l -= cnt;
        k += 1;
      }
    }
  }
  double s[3][RPT], b[RPT], z[RPT], rr = 0.0, bz = 0.0;
  uint8_t dir[3][RPT];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int u = 0; u < RPT; ++u) {
      s[c][u] = at((const double *)P.r[0], r[c][u]);
      dir[c][u] = at(P.isdir, r[c][u]);
    }
#pragma unroll
  for (int u = 0; u < RPT; ++u) {
    b[u] = at((const double *)P.B, r[3][u]);
    z[u] = at((const double *)P.z, r[3][u]);
  }
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int u = 0; u < RPT; ++u) rr = on[c][u] && !dir[c][u] ? fma(s[c][u], s[c][u], rr) : rr;
#pragma unroll
  for (int u = 0; u < RPT; ++u) bz = on[3][u] ? fma(b[u], z[u], bz) : bz;
  const double2 t = tile_sum2(bz, rr, sh);
  if (tid == 0) {
    P.part_bz[bk.b] = t.x;
    P.part_rr[bk.b] = t.y;
  }
}
template <int RPT>
__global__ __launch_bounds__(kTileThreads) void k_tile_dots(TileSet T, TileCols C, TilePcg P) {
  tile_dots_body<RPT>(self_xcd_blk(), T, C, P);
}
template __global__ void k_tile_dots<1>(TileSet, TileCols, TilePcg);
template __global__ void k_tile_dots<2>(TileSet, TileCols, TilePcg);

// ------------------------------------------ batched ensemble launches --
#define CG_TILE_HEAD                                       \
  const int g_ = xcd_group();                              \
  const int m_ = batch_member(start, nmem, g_);            \
  const MemberDev &d = md[m_];                             \
  const Blk bk{g_ - start[m_], start[m_ + 1] - start[m_]};
__device__ __forceinline__ double *member_vec(const MemberDev &d, int v) {
  return v == kVecTnoti ? d.tnoti : (v == kVecPdiff ? d.pdiff : (v == kVecR ? d.tpcg.r[0] : (v == kVecP ? d.tpcg.p[0] : d.z)));
}
template <typename FT, int MODE, int RPT>
__global__ __launch_bounds__(kTileThreads) void kb_tile(const int *start, int nmem, const MemberDev *md, int vin,
                                                        int vout) {
  extern __shared__ double smem[];
  CG_TILE_HEAD
  const FT *F = sizeof(FT) == 4 ? (const FT *)d.F32 : (const FT *)d.F64;
  const TileCols C{{d.col[0], d.col[1], d.col[2]}};
  if (MODE == kTilePcg) tile_body<FT, MODE, RPT>(bk, smem, d.tiles, C, F, d.tpcg, nullptr, d.z, &d.tpcg.sc->stop);
  else tile_body<FT, MODE, RPT>(bk, smem, d.tiles, C, F, d.tpcg, member_vec(d, vin), member_vec(d, vout), nullptr);
}
#define CG_INST_BTILE(FT, MODE)                                                          \
  template __global__ void kb_tile<FT, MODE, 1>(const int *, int, const MemberDev *, int, int); \
  template __global__ void kb_tile<FT, MODE, 2>(const int *, int, const MemberDev *, int, int);
CG_INST_BTILE(float, kTilePcg)
CG_INST_BTILE(float, kTileSolve)
CG_INST_BTILE(double, kTilePcg)
CG_INST_BTILE(double, kTileSolve)
#undef CG_INST_BTILE
__global__ __launch_bounds__(kBlock) void kb_spmv_beta(const int *start, int nmem, const MemberDev *md) {
  CG_TILE_HEAD
  spmv_beta_body(bk, d.sl, d.fts, d.tpcg, d.tiles.ntile);
}
__global__ __launch_bounds__(256) void kb_pcg_check(const int *start, int nmem, const MemberDev *md) {
  CG_TILE_HEAD
  (void)bk;
  pcg_check_body(d.tpcg, d.tiles.ntile);
}
template <int RPT>
__global__ __launch_bounds__(kTileThreads) void kb_tile_dots(const int *start, int nmem, const MemberDev *md) {
  CG_TILE_HEAD
  tile_dots_body<RPT>(bk, d.tiles, TileCols{{d.col[0], d.col[1], d.col[2]}}, d.tpcg);
}
template __global__ void kb_tile_dots<1>(const int *, int, const MemberDev *);
template __global__ void kb_tile_dots<2>(const int *, int, const MemberDev *);
#undef CG_TILE_HEAD

}  // namespace cg
