// guess.hip -- the learned initial iterate's network on gfx950: bf16 MFMA
// convolution (inference, training forward, backward-data), weight
// gradients, Adam, and the cathy_gpu_guess_* C entries.
//
// MFMA operand layout (v_mfma_f32_16x16x16bf16_1k, D = A B + C, 16x16x16):
//   lane l holds A[l%16][4(l/16)+t], B[4(l/16)+t][l%16], D[4(l/16)+t][l%16],
//   t = 0..3.
// Convolution as a GEMM per 16-level block of one column: rows = levels,
// K = (tap k, input channel ci) with kk = k*CIN + ci, A(l, kk) =
// in[l + k - 1][ci] (zero outside the column), N = output channels.
#include <hip/hip_runtime.h>

#include <cmath>
#include <map>
#include <mutex>

#include "cathy_gpu.h"
#include "guess.h"

static_assert(CATHY_GPU_EINVAL == -1 && CATHY_GPU_ENOMEM == -3, "status codes of guarded()");

namespace cg {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// fp32 -> bf16, round to nearest even (finite inputs).
__device__ __forceinline__ unsigned short f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ int wave_id() { return (int)((blockIdx.x * (size_t)blockDim.x + threadIdx.x) >> 6); }

// ------------------------------------------------------------- packs --
// Forward B operand of one layer: entry (j, b, lane) holds W[kk][co],
// kk = 16j + 4(lane/16) + t, co = 16b + lane%16 (W[k][ci][co] flattened
// as kk*cout + co).
__global__ void k_gpack_fwd(const float *__restrict__ w, int off_w, int cin, int cout, int nchunk, int nb,
                            bf16x4 *__restrict__ out) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nchunk * nb * 64) return;
  const int lane = e & 63, jn = e >> 6, j = jn / nb, b = jn - j * nb;
  const int co = 16 * b + (lane & 15);
  bf16x4 r;
  for (int t = 0; t < 4; ++t) {
    const int kk = 16 * j + 4 * (lane >> 4) + t;
    const float val = (kk < 3 * cin && co < cout) ? w[off_w + kk * cout + co] : 0.f;
    r[t] = (short)f2bf(val);
  }
  out[e] = r;
}

// Backward-data operand: the input gradient is the convolution of the
// output gradient (cin_b channels, cout real) with W'[k'][c][ci] =
// W[2-k'][ci][c]; output channels = cin (4 blocks of 16).
__global__ void k_gpack_bwd(const float *__restrict__ w, int off_w, int cin, int cout, int cin_b, int nchunk_b,
                            bf16x4 *__restrict__ out) {
  const int nb = cin / 16;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nchunk_b * nb * 64) return;
  const int lane = e & 63, jn = e >> 6, j = jn / nb, b = jn - j * nb;
  const int ci = 16 * b + (lane & 15);
  bf16x4 r;
  for (int t = 0; t < 4; ++t) {
    const int kk = 16 * j + 4 * (lane >> 4) + t;
    const int kp = kk / cin_b, c = kk - kp * cin_b;
    const float val = (kp < 3 && c < cout) ? w[off_w + ((2 - kp) * cin + ci) * cout + c] : 0.f;
    r[t] = (short)f2bf(val);
  }
  out[e] = r;
}

// -------------------------------------------------------- convolution --
// One wavefront: levels [16 rb, 16 rb + 16) of one column, all 16*NB
// output channels.  out = act(conv + bias), zero at levels >= L; with a
// mask tensor (same layout as out) entries whose mask is not > 0 are zero
// (the ReLU derivative in the backward pass).  out32 takes channel 0 in
// fp32 (the network output).
template <int CIN, int NB>
__global__ __launch_bounds__(256) void k_gconv(int ncol, int Lp, int L, const int *__restrict__ idx,
                                               const unsigned short *__restrict__ in,
                                               const bf16x4 *__restrict__ wp, const float *__restrict__ bias,
                                               int cout, int relu, const unsigned short *__restrict__ mask,
                                               unsigned short *__restrict__ out, float *__restrict__ out32) {
  constexpr int K = 3 * CIN, NCH = (K + 15) / 16, OS = 16 * NB;
  const int lane = threadIdx.x & 63;
  const int wv = wave_id();
  const int rbs = Lp >> 4;
  if (wv >= ncol * rbs) return;
  const int col = wv / rbs, rb = wv - col * rbs;
  const size_t src = idx ? (size_t)idx[col] : (size_t)col;
  const unsigned short *xin = in + src * Lp * CIN;
  const int grp = lane >> 4, r16 = lane & 15;
  const int l = rb * 16 + r16;
  f32x4 acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int kk = 16 * j + 4 * grp;
    bf16x4 a = {0, 0, 0, 0};
    if (kk < K) {
      const int k = kk / CIN, ci = kk - k * CIN;
      const int lv = l + k - 1;
      if (lv >= 0 && lv < L) a = *(const bf16x4 *)(xin + (size_t)lv * CIN + ci);
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
      acc[b] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, wp[(j * NB + b) * 64 + lane], acc[b], 0, 0, 0);
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int co = 16 * b + r16;
    const float bv = (bias && co < cout) ? bias[co] : 0.f;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int lo = rb * 16 + 4 * grp + t;
      const size_t o = ((size_t)col * Lp + lo) * OS + co;
      float v = acc[b][t] + bv;
      if (relu) v = fmaxf(v, 0.f);
      if (lo >= L) v = 0.f;
      if (mask && !(bf2f(mask[o]) > 0.f)) v = 0.f;
      if (out) out[o] = f2bf(v);
      if (out32 && co == 0) out32[(size_t)col * Lp + lo] = v;
    }
  }
}

// ---------------------------------------------------- weight gradient --
// dW[kk][co] = sum over positions of A(pos, kk) g(pos, co); row kk = 3*CIN
// is the bias (A = 1 at live levels).  MFMA with M = kk, K = 16 positions
// (one level block), N = co.  A wavefront owns one 16x16 tile over a
// contiguous range of level blocks (split); partials [split][rows][GS].
template <int CIN, int GS>
__global__ __launch_bounds__(256) void k_gdw(int ncol, int Lp, int L, const int *__restrict__ idx,
                                             const unsigned short *__restrict__ in,
                                             const unsigned short *__restrict__ g, int nsplit,
                                             float *__restrict__ part) {
  constexpr int K = 3 * CIN, NCW = (K + 1 + 15) / 16, NB = GS / 16, T = NCW * NB;
  const int lane = threadIdx.x & 63;
  const int wv = wave_id();
  if (wv >= T * nsplit) return;
  const int tile = wv % T, split = wv / T;
  const int j = tile / NB, b = tile - j * NB;
  const int rbs = Lp >> 4;
  const long R = (long)ncol * rbs;
  const long r0 = R * split / nsplit, r1 = R * (split + 1) / nsplit;
  const int grp = lane >> 4, r16 = lane & 15;
  const int kk = 16 * j + r16;
  const bool isw = kk < K, isb = kk == K;
  const int kdx = isw ? kk / CIN : 0, ci = isw ? kk - kdx * CIN : 0;
  const int co = 16 * b + r16;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (long r = r0; r < r1; ++r) {
    const int col = (int)(r / rbs), rb = (int)(r - (long)col * rbs);
    const size_t src = idx ? (size_t)idx[col] : (size_t)col;
    const unsigned short *xin = in + src * Lp * CIN;
    const unsigned short *gc = g + (size_t)col * Lp * GS;
    bf16x4 a, bb;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int lv = rb * 16 + 4 * grp + t;
      unsigned short av = 0;
      if (isw) {
        const int ls = lv + kdx - 1;
        if (ls >= 0 && ls < L) av = xin[(size_t)ls * CIN + ci];
      } else if (isb && lv < L) {
        av = 0x3F80;  // 1.0
      }
      a[t] = (short)av;
      bb[t] = (short)gc[(size_t)lv * GS + co];
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bb, acc, 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
    part[((size_t)split * NCW * 16 + 16 * j + 4 * grp + t) * GS + co] = acc[t];
}

// ------------------------------------------------------- loss, Adam --
// Mean squared error over live levels: gradient 2 d / (ncol L) into the
// head's 16-channel gradient tensor (channel 0), per-block sums of d^2.
__global__ __launch_bounds__(256) void k_gloss(int ncol, int Lp, int L, const float *__restrict__ y,
                                               const int *__restrict__ idx, const float *__restrict__ t,
                                               float inv, unsigned short *__restrict__ gh,
                                               float *__restrict__ lossp) {
  __shared__ float red[256];
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  float d2 = 0.f;
  if (e < ncol * Lp) {
    const int col = e / Lp, l = e - col * Lp;
    float gv = 0.f;
    if (l < L) {
      const size_t src = idx ? (size_t)idx[col] : (size_t)col;
      const float d = y[e] - t[src * Lp + l];
      d2 = d * d;
      gv = 2.f * d * inv;
    }
    unsigned short *o = gh + (size_t)e * 16;
    o[0] = f2bf(gv);
    for (int c = 1; c < 16; ++c) o[c] = 0;
  }
  red[threadIdx.x] = d2;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) lossp[blockIdx.x] = red[0];
}

// Where the partials of a gradient lie: entry (kk, co) of layer l of split p
// at part[off[l] + p * stride[l] + kk * gs[l] + co] (row kk = K: the bias).
struct GradParts {
  const float *part;
  size_t off[kGuessLayers], stride[kGuessLayers];
  int gs[kGuessLayers], nsplit;
};
// The layers' parameter and pack layout (GuessLayer) for k_gstep.
struct GradLayers {
  int off_w[kGuessLayers], cin[kGuessLayers], cout[kGuessLayers], nb[kGuessLayers];
  unsigned fpack[kGuessLayers], bpack[kGuessLayers];  // bf16x4 units
};

// Sums the split partials into the gradient vector (STEP: and takes the Adam
// step and rewrites the parameter's entries of the MFMA packs, whose padding
// entries stay zero); work-group 0 also sums the loss partials.  A
// work-group owns kStepCols consecutive parameters: its 16 groups of 64 lanes
// read every 16th split of the 64 parameters side by side, and their sums
// meet in LDS in a fixed order.  One thread per parameter adding 256 splits
// one after the other took 63 us a layer, and the packs nine launches of
// 4.4 us; here all layers, Adam and the packs are one launch of 18 us at 256
// splits (48 MB of partials, 2.7 TB/s).
constexpr int kStepCols = 64, kStepRows = 16;
template <bool STEP>
__global__ __launch_bounds__(kStepCols *kStepRows) void k_gstep(GradParts gp, GradLayers ly, const float *__restrict__ lossp,
                                                                 int nloss, float inv, float *__restrict__ slot,
                                                                 float *__restrict__ grad, float *__restrict__ w,
                                                                 float *__restrict__ m, float *__restrict__ v, float lr_t,
                                                                 float b1, float b2, float eps, short *__restrict__ pack) {
  __shared__ float sh[kStepRows][kStepCols];
  const int c = threadIdx.x % kStepCols, q = threadIdx.x / kStepCols;
  if (blockIdx.x == 0) {
    float s = 0.f;
    for (int i = threadIdx.x; i < nloss; i += kStepCols * kStepRows) s += lossp[i];
    sh[q][c] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
      float t = 0.f;
      for (int i = 0; i < kStepRows; ++i) {
        float u = 0.f;
        for (int k = 0; k < kStepCols; ++k) u += sh[i][k];
        t += u;
      }
      slot[0] = t * inv;
    }
    __syncthreads();
  }
  const int e = blockIdx.x * kStepCols + c;
  int l = 0, kk = 0, co = 0;
  float s = 0.f;
  if (e < kGuessParams) {
#pragma unroll
    for (int i = 1; i < kGuessLayers; ++i)
      if (e >= ly.off_w[i]) l = i;
    kk = (e - ly.off_w[l]) / ly.cout[l];  // the bias follows the weights: row K
    co = (e - ly.off_w[l]) - kk * ly.cout[l];
    const float *p = gp.part + gp.off[l] + (size_t)kk * gp.gs[l] + co;
    const size_t st = gp.stride[l];
    float a[4] = {0.f, 0.f, 0.f, 0.f};  // four loads in flight
    int i = q;
    for (; i + 3 * kStepRows < gp.nsplit; i += 4 * kStepRows)
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] += p[(size_t)(i + u * kStepRows) * st];
    for (; i < gp.nsplit; i += kStepRows) a[0] += p[(size_t)i * st];
    s = (a[0] + a[1]) + (a[2] + a[3]);
  }
  sh[q][c] = s;
  __syncthreads();
  if (q != 0 || e >= kGuessParams) return;
  float gi = 0.f;
#pragma unroll
  for (int i = 0; i < kStepRows; i += 4)
    gi += (sh[i][c] + sh[i + 1][c]) + (sh[i + 2][c] + sh[i + 3][c]);
  grad[e] = gi;
  if (!STEP) return;
  const float mi = b1 * m[e] + (1.f - b1) * gi;
  const float vi = b2 * v[e] + (1.f - b2) * gi * gi;
  const float wi = w[e] - lr_t * mi / (sqrtf(vi) + eps);
  m[e] = mi;
  v[e] = vi;
  w[e] = wi;
  if (kk >= 3 * ly.cin[l]) return;  // a bias: not packed
  const short h = (short)f2bf(wi);
  const int r = kk & 15;
  pack[4 * ((size_t)ly.fpack[l] + ((kk >> 4) * ly.nb[l] + (co >> 4)) * 64 + (r >> 2) * 16 + (co & 15)) + (r & 3)] = h;
  if (l > 0) {  // k_gpack_bwd: row kp * cin_b + co with kp = 2 - k, column ci
    const int cin = ly.cin[l], k = kk / cin, ci = kk - k * cin;
    const int kb = (2 - k) * 16 * ly.nb[l] + co, rb = kb & 15;
    pack[4 * ((size_t)ly.bpack[l] + ((kb >> 4) * (cin >> 4) + (ci >> 4)) * 64 + (rb >> 2) * 16 + (ci & 15)) + (rb & 3)] = h;
  }
}

// ------------------------------------------------ the network in one launch --
// Columns of at most kTileRows levels (Lp <= 64): a work-group takes tiles of
// whole columns (64 / Lp of them) through all layers in LDS, and in training
// on through the loss and every layer's gradients, so activations and
// gradients never reach HBM.  Wave w computes output channels 16w .. 16w+15
// of every layer (waves w and w + 4 share them and take every other row block),
// with the layer's B operand (the k_gpack_* packs, 24 VGPRs) loaded once per
// tile; the weight gradients of the 16 output channels accumulate in MFMA
// tiles (25 a wave, 100 VGPRs: w the input channels 0 .. 31 and the
// biases, w + 4 the others and the head) over all tiles of the work-group and are
// written once, as one split of the partials k_gstep sums.  Rounding points are those of the layer-by-layer
// kernels (bf16 inputs, weights, activations, gradients; fp32 sums).
// Bound by LDS latency and barriers (about 18 us per tile, two tiles a group at 1024
// columns of 31 levels) and by writing the partials (48 MB, 10 us); the products alone
// would take 7 us at the card's rate.  A training step on 1024 columns of 31 levels took 550 us
// in 31 launches, 65 us of them convolutions and 87 us weight gradients; it
// takes 51 us here and 18 us in k_gstep.  With four waves instead of
// eight (448 registers each) this kernel took 63 us.
// A row of an LDS tile is padded to 136 bytes (40 for 16 channels) so that the
// 16 rows of an operand read start in different banks; row kTileRows is zero and
// stands for the levels outside a column.
constexpr int kTileRows = 64, kTileBlocks = kTileRows / 16;
constexpr int kTrainGroups = 256;  // one work-group per CU, one split of the partials each
constexpr int kFwdGroups = 1024;   // four per CU
constexpr int kWS = kGuessWidth + 4, kXS = kGuessIn + 4;  // row strides (shorts)
constexpr int kPartSize = 4 * 16 * 64 + 3 * 13 * 16 * 64 + 13 * 16 * 16;  // floats of one split
constexpr int kPartOff[kGuessLayers] = {0, 4096, 4096 + 13312, 4096 + 2 * 13312, 4096 + 3 * 13312};
static_assert(kPartSize == 4096 + 3 * 13312 + 3328, "partial layout");

struct FusedNet {
  const bf16x4 *pack;
  const float *w;
  size_t fpack[kGuessLayers], bpack[kGuessLayers];
  int off_b[kGuessLayers];
};

// LDS row of a level's neighbour: row `row` of the tile holds level `lv` of
// its column (zero row outside [0, L)).
__device__ __forceinline__ int tile_row(int row, int lv, int L) { return lv >= 0 && lv < L ? row : kTileRows; }

// acc = conv of row block rb of the LDS tile `in` with the wave's B operand.
template <int CIN, int SS>
__device__ __forceinline__ f32x4 tile_conv(const short *in, const bf16x4 (&wr)[3 * CIN / 16], int rb, int lv0, int L,
                                           int grp, int r16) {
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const short *src = in + tile_row(rb * 16 + r16 + k - 1, lv0 + r16 + k - 1, L) * SS + 4 * grp;
#pragma unroll
    for (int cb = 0; cb < CIN / 16; ++cb)
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*(const bf16x4 *)(src + 16 * cb), wr[k * (CIN / 16) + cb], acc, 0,
                                                      0, 0);
  }
  return acc;
}
// the wave's B operand of a layer: chunk j of output block b
template <int N>
__device__ __forceinline__ void load_pack(bf16x4 (&wr)[N], const bf16x4 *p, int nb, int b, int lane) {
#pragma unroll
  for (int j = 0; j < N; ++j) wr[j] = p[(j * nb + b) * 64 + lane];
}
// Weight-gradient tiles of one row block: dw[3 cb-blocks k][c] += x_k^T g for the channel
// blocks [C0, C0 + NC) of `in`, g = the block's gradient operand.
template <int NC, int SS>
__device__ __forceinline__ void tile_dw(f32x4 *dw, const short *in, int c0, bf16x4 g, int rb, int lv0, int L, int grp,
                                        int r16) {
#pragma unroll
  for (int cb = 0; cb < NC; ++cb) {
    short u[6];
#pragma unroll
    for (int q = 0; q < 6; ++q)
      u[q] = in[tile_row(rb * 16 + 4 * grp + q - 1, lv0 + 4 * grp + q - 1, L) * SS + 16 * (c0 + cb) + r16];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      const bf16x4 a = {u[k], u[k + 1], u[k + 2], u[k + 3]};
      dw[k * NC + cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, g, dw[k * NC + cb], 0, 0, 0);
    }
  }
}

template <bool TRAIN>
__global__ __launch_bounds__(512, 2) void k_gfused(FusedNet net, int ncol, int Lp, int L, const int *__restrict__ idx,
                                                   const unsigned short *__restrict__ x, const float *__restrict__ t,
                                                   float inv, float *__restrict__ y, float *__restrict__ lossp,
                                                   float *__restrict__ part) {
  __shared__ __align__(16) short xs[(kTileRows + 1) * kXS];
  __shared__ __align__(16) short act[TRAIN ? 4 : 2][(kTileRows + 1) * kWS];
  __shared__ __align__(16) short gr[TRAIN ? 2 : 1][TRAIN ? (kTileRows + 1) * kWS : 4];
  __shared__ __align__(16) short gh[TRAIN ? (kTileRows + 1) * kXS : 4];
  __shared__ float red[4];
  const int lane = threadIdx.x & 63, w = (threadIdx.x >> 6) & 3, h = threadIdx.x >> 8;
  const int grp = lane >> 4, r16 = lane & 15;
  const int rbs = Lp >> 4, cpt = kTileBlocks / rbs, nrb = cpt * rbs;  // columns and row blocks per tile
  const int ntile = (ncol + cpt - 1) / cpt;
  for (int i = threadIdx.x; i < (kTileRows + 1) * kXS; i += 512) {
    xs[i] = 0;
    if (TRAIN) gh[i] = 0;
  }
  for (int i = threadIdx.x; i < kWS; i += 512) {
#pragma unroll
    for (int a = 0; a < (TRAIN ? 4 : 2); ++a) act[a][kTileRows * kWS + i] = 0;
    if (TRAIN) gr[0][kTileRows * kWS + i] = gr[1][kTileRows * kWS + i] = 0;
  }
  f32x4 dwe[4], dw[3][7];  // input layer (h = 0) or head (h = 1), hidden layers (last tile: the bias)
  float d2 = 0.f;
  if (TRAIN) {
#pragma unroll
    for (int i = 0; i < 4; ++i) dwe[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int l = 0; l < 3; ++l)
#pragma unroll
      for (int i = 0; i < 7; ++i) dw[l][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    __syncthreads();  // the previous tile's readers (and the zero rows) are done
    // an offset the compiler cannot see through: it would keep every layer's B
    // operand (180 VGPRs) in registers across the tiles, and spill
    int opaque = 0;
    asm volatile("" : "+s"(opaque));
    const bf16x4 *pack = net.pack + opaque;
    if (threadIdx.x < 4 * kTileRows) {
      const int row = threadIdx.x >> 2, c4 = 4 * (threadIdx.x & 3);
      const int col = tile * cpt + row / Lp, lv = row % Lp;
      bf16x4 v = {0, 0, 0, 0};
      if (row < nrb * 16 && col < ncol)
        v = *(const bf16x4 *)(x + ((size_t)(idx ? idx[col] : col) * Lp + lv) * kGuessIn + c4);
      *(bf16x4 *)(xs + row * kXS + c4) = v;
    }
    // ---- forward: hidden layers
    bf16x4 w3[3], w12[12];
    load_pack(w3, pack + net.fpack[0], 4, w, lane);
#pragma unroll
    for (int l = 0; l < 4; ++l) {
      const float bias = net.w[net.off_b[l] + 16 * w + r16];
      if (l > 0) load_pack(w12, pack + net.fpack[l], 4, w, lane);
      __syncthreads();
      short *out = act[TRAIN ? l : l & 1];
      const short *in = l == 0 ? xs : act[TRAIN ? l - 1 : (l - 1) & 1];
#pragma unroll
      for (int i = 0; i < kTileBlocks / 2; ++i) {
        const int rb = 2 * i + h;
        if (rb >= nrb) break;
        const int lv0 = (rb % rbs) * 16;
        const f32x4 acc = l == 0 ? tile_conv<kGuessIn, kXS>(in, w3, rb, lv0, L, grp, r16)
                                 : tile_conv<kGuessWidth, kWS>(in, w12, rb, lv0, L, grp, r16);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          float v = fmaxf(acc[u] + bias, 0.f);
          if (lv0 + 4 * grp + u >= L) v = 0.f;
          out[(rb * 16 + 4 * grp + u) * kWS + 16 * w + r16] = (short)f2bf(v);
        }
      }
    }
    // ---- head: wave w takes row block w; channel 0 is the output
    const short *last = act[TRAIN ? 3 : 1];
    load_pack(w12, pack + net.fpack[4], 1, 0, lane);
    __syncthreads();
    if (h == 0 && w < nrb) {
      const int lv0 = (w % rbs) * 16, col = tile * cpt + w / rbs;
      const f32x4 acc = tile_conv<kGuessWidth, kWS>(last, w12, w, lv0, L, grp, r16);
      if (r16 == 0) {
        const float bias = net.w[net.off_b[4]];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int lv = lv0 + 4 * grp + u;
          const float v = lv < L ? acc[u] + bias : 0.f;
          if (TRAIN) {
            float gv = 0.f;
            if (lv < L && col < ncol) {
              const float d = v - t[(size_t)(idx ? idx[col] : col) * Lp + lv];
              d2 += d * d;
              gv = 2.f * d * inv;
            }
            gh[(w * 16 + 4 * grp + u) * kXS] = (short)f2bf(gv);
          } else if (col < ncol) {
            y[(size_t)col * Lp + lv] = v;
          }
        }
      }
    }
    if constexpr (TRAIN) {
      // ---- backward: head, then hidden layers 3, 2, 1
      load_pack(w3, pack + net.bpack[4], 4, w, lane);
      __syncthreads();
#pragma unroll
      for (int l = 4; l >= 0; --l) {
        // gradient at layer l's output: gh (head), else gr[l & 1]; its inputs
        // are act[l - 1] (xs for layer 0); the next gradient goes to gr[(l - 1) & 1]
        const short *g = l == 4 ? gh : gr[l & 1];
        const int gs = l == 4 ? kXS : kWS, gc = l == 4 ? r16 : 16 * w + r16;
#pragma unroll 1
        for (int rb = 0; rb < nrb; ++rb) {
          const int lv0 = (rb % rbs) * 16;
          bf16x4 gv, one;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            gv[u] = g[(rb * 16 + 4 * grp + u) * gs + gc];
            one[u] = r16 == 0 && lv0 + 4 * grp + u < L ? (short)0x3F80 : (short)0;
          }
          if (l == 4) {  // input channels 16w .. 16w+15, w = 0 also the bias
            if (h == 1) {
              tile_dw<1, kWS>(dwe, act[3], w, gv, rb, lv0, L, grp, r16);
              if (w == 0) dwe[3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(one, gv, dwe[3], 0, 0, 0);
            }
          } else if (l == 0) {
            if (h == 0) {
              tile_dw<1, kXS>(dwe, xs, 0, gv, rb, lv0, L, grp, r16);
              dwe[3] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(one, gv, dwe[3], 0, 0, 0);
            }
          } else {
            tile_dw<2, kWS>(dw[l - 1], act[l - 1], 2 * h, gv, rb, lv0, L, grp, r16);
            if (h == 0) dw[l - 1][6] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(one, gv, dw[l - 1][6], 0, 0, 0);
          }
        }
        if (l > 0) {
#pragma unroll
          for (int i = 0; i < kTileBlocks / 2; ++i) {
            const int rb = 2 * i + h;
            if (rb >= nrb) break;
            const int lv0 = (rb % rbs) * 16;
            const f32x4 acc = l == 4 ? tile_conv<kGuessIn, kXS>(g, w3, rb, lv0, L, grp, r16)
                                     : tile_conv<kGuessWidth, kWS>(g, w12, rb, lv0, L, grp, r16);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int o = (rb * 16 + 4 * grp + u) * kWS + 16 * w + r16;
              float v = acc[u];
              if (lv0 + 4 * grp + u >= L) v = 0.f;
              if (!(bf2f((unsigned short)act[l - 1][o]) > 0.f)) v = 0.f;
              gr[(l - 1) & 1][o] = (short)f2bf(v);
            }
          }
        }
        if (l > 1) load_pack(w12, pack + net.bpack[l - 1], 4, w, lane);
        if (l > 0) __syncthreads();
      }
    }
  }
  if constexpr (TRAIN) {
    // hidden tile 2k + cb of wave half h is chunk 4k + 2h + cb, head tile k chunk
    // 4k + w; the last tile is the bias chunk
    float *P = part + (size_t)blockIdx.x * kPartSize;
#pragma unroll
    for (int l = 0; l < 3; ++l)
#pragma unroll
      for (int i = 0; i < 7; ++i) {
        if (i == 6 && h == 1) break;
        const int j = i == 6 ? 12 : 4 * (i >> 1) + 2 * h + (i & 1);
#pragma unroll
        for (int u = 0; u < 4; ++u) P[kPartOff[l + 1] + (16 * j + 4 * grp + u) * 64 + 16 * w + r16] = dw[l][i][u];
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (h == 0) P[kPartOff[0] + (16 * i + 4 * grp + u) * 64 + 16 * w + r16] = dwe[i][u];
        else if (i < 3 || w == 0) P[kPartOff[4] + (16 * (i < 3 ? 4 * i + w : 12) + 4 * grp + u) * 16 + r16] = dwe[i][u];
      }
    for (int o = 32; o > 0; o >>= 1) d2 += __shfl_down(d2, o, 64);
    if (lane == 0 && h == 0) red[w] = d2;
    __syncthreads();
    if (threadIdx.x == 0) lossp[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}

// ------------------------------------------------------ flow-side ops --
// Features of (surface node s, level l): raw fp32 values and the
// standardised bf16 network input; levels >= L are zero.
__global__ void k_guess_features(int nnod, int L, int Lp, const int *__restrict__ colrow,
                                 const double *__restrict__ ptimep, const double *__restrict__ pprev,
                                 double ratio, const double *__restrict__ swtimep,
                                 const float *__restrict__ stat, const double *__restrict__ atmpot,
                                 const double *__restrict__ arenod, float ldt, GuessScale sc,
                                 float *__restrict__ raw, unsigned short *__restrict__ x) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nnod * Lp) return;
  const int s = e / Lp, l = e - s * Lp;
  float f[kGuessIn];
  for (int c = 0; c < kGuessIn; ++c) f[c] = 0.f;
  const bool live = l < L;
  if (live) {
    const int row = colrow[s * L + l];
    const float *sn = stat + ((size_t)s * L + l) * 5;
    f[0] = (float)ptimep[row];
    f[1] = (float)(swtimep[row] * (double)sn[4]);
    f[2] = sn[0];
    f[3] = sn[1];
    f[4] = sn[2];
    f[5] = (float)(atmpot[s] / arenod[s]);
    f[6] = ldt;
    f[7] = sn[3];
    f[8] = (float)(ratio * (ptimep[row] - pprev[row]));
  }
  for (int c = 0; c < kGuessIn; ++c) {
    if (raw) raw[(size_t)e * kGuessIn + c] = f[c];
    if (x) x[(size_t)e * kGuessIn + c] = live ? f2bf((f[c] - sc.mu[c]) / sc.sd[c]) : (unsigned short)0;
  }
}

// One thread per column: E_l = ratio (PTIMEP - PPREV), s = rms_l E_l +
// floor, PNEW = PTIMEP + beta E + s out clamp(y, -10, 10) on every node
// except the surface nodes that are Dirichlet at the start of the attempt
// (IFATM != 0) and, with band >= 0, the nodes where PTIMEP or the guess is
// above -band (at or near saturation, where the Picard linearisation of
// the storage term changes branch).
__global__ void k_guess_apply(int nnod, int L, int Lp, const int *__restrict__ colrow,
                              const int *__restrict__ ifatm, const double *__restrict__ ptimep,
                              const double *__restrict__ pprev, double ratio, const float *__restrict__ y,
                              double beta, double out, double floor_abs, double band,
                              double *__restrict__ pnew) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= nnod) return;
  const int *cr = colrow + (size_t)s * L;
  double e2 = 0.0;
  for (int l = 0; l < L; ++l) {
    const double d = ratio * (ptimep[cr[l]] - pprev[cr[l]]);
    e2 += d * d;
  }
  const double scol = sqrt(e2 / L) + floor_abs;
  for (int l = (ifatm[s] != 0) ? 1 : 0; l < L; ++l) {
    const int row = cr[l];
    const double pt = ptimep[row];
    const double yl = fmin(fmax((double)y[(size_t)s * Lp + l], -10.0), 10.0);
    const double gv = pt + beta * (ratio * (pt - pprev[row])) + scol * out * yl;
    if (band >= 0.0 && (pt > -band || gv > -band)) continue;
    pnew[row] = gv;
  }
}

__global__ void k_guess_target(int nnod, int L, int Lp, const int *__restrict__ colrow,
                               const double *__restrict__ ptimep, const double *__restrict__ pnew,
                               float *__restrict__ target) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nnod * Lp) return;
  const int s = e / Lp, l = e - s * Lp;
  float v = 0.f;
  if (l < L) {
    const int row = colrow[s * L + l];
    v = (float)(pnew[row] - ptimep[row]);
  }
  target[e] = v;
}

void guess_features(hipStream_t st, int nnod, int L, int Lp, const int *colrow, const double *ptimep,
                    const double *pprev, double ratio, const double *swtimep, const float *stat,
                    const double *atmpot, const double *arenod, double dt, const GuessScale &sc, float *raw,
                    unsigned short *x) {
  hipLaunchKernelGGL(k_guess_features, dim3(grid_for((size_t)nnod * Lp)), dim3(kBlock), 0, st, nnod, L, Lp,
                     colrow, ptimep, pprev, ratio, swtimep, stat, atmpot, arenod, (float)std::log10(dt), sc, raw,
                     x);
}

void guess_apply(hipStream_t st, int nnod, int L, int Lp, const int *colrow, const int *ifatm,
                 const double *ptimep, const double *pprev, double ratio, const float *y, const GuessScale &sc,
                 double *pnew) {
  hipLaunchKernelGGL(k_guess_apply, dim3(grid_for((size_t)nnod)), dim3(kBlock), 0, st, nnod, L, Lp, colrow, ifatm,
                     ptimep, pprev, ratio, y, (double)sc.beta, (double)sc.out, (double)sc.floor, (double)sc.band,
                     pnew);
}

void guess_target(hipStream_t st, int nnod, int L, int Lp, const int *colrow, const double *ptimep,
                  const double *pnew, float *target) {
  hipLaunchKernelGGL(k_guess_target, dim3(grid_for((size_t)nnod * Lp)), dim3(kBlock), 0, st, nnod, L, Lp,
                     colrow, ptimep, pnew, target);
}

// ------------------------------------------------------------ GuessNet --
static int waves_blocks(long waves) { return (int)((waves * 64 + kBlock - 1) / kBlock); }

static int split_count(int ncol, int Lp) {
  const long r = (long)ncol * (Lp / 16);
  long s = r / 8;
  if (s < 1) s = 1;
  if (s > 256) s = 256;
  return (int)s;
}

GuessNet::GuessNet(int levels) : L(levels) {
  CG_REQUIRE(levels >= 2 && levels <= 4096, "guess net: levels out of range");
  Lp = (L + 15) / 16 * 16;
  CG_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
  const int cin[kGuessLayers] = {kGuessIn, 64, 64, 64, 64}, cout[kGuessLayers] = {64, 64, 64, 64, 1};
  int off = 0;
  size_t fp = 0;
  for (int l = 0; l < kGuessLayers; ++l) {
    GuessLayer &g = ly[l];
    g.cin = cin[l];
    g.cout = cout[l];
    g.nb = (g.cout + 15) / 16;
    g.K = 3 * g.cin;
    g.nchunk = (g.K + 15) / 16;
    g.nchunk_w = (g.K + 1 + 15) / 16;
    g.off_w = off;
    off += g.K * g.cout;
    g.off_b = off;
    off += g.cout;
    g.cin_b = g.nb * 16;
    g.nchunk_b = l == 0 ? 0 : (3 * g.cin_b + 15) / 16;
    g.fpack = fp;
    fp += (size_t)g.nchunk * g.nb * 64;
  }
  for (int l = 1; l < kGuessLayers; ++l) {
    ly[l].bpack = fp;
    fp += (size_t)ly[l].nchunk_b * (ly[l].cin / 16) * 64;
  }
  CG_REQUIRE(off == kGuessParams, "guess net: parameter layout");
  pack.alloc(fp);
  for (DBuf<float> *b : {&w, &m, &v, &grad}) b->alloc(kGuessParams);
  CG_HIP(hipMemsetAsync(w.p, 0, sizeof(float) * kGuessParams, st));
  CG_HIP(hipMemsetAsync(m.p, 0, sizeof(float) * kGuessParams, st));
  CG_HIP(hipMemsetAsync(v.p, 0, sizeof(float) * kGuessParams, st));
  for (int c = 0; c < kGuessIn; ++c) { scale.mu[c] = 0.f; scale.sd[c] = 1.f; }
  scale.out = 1.f;
  scale.floor = 1e-5f;
  scale.beta = 1.f;
  scale.band = 0.1f;
  repack();
  CG_HIP(hipStreamSynchronize(st));
}

GuessNet::~GuessNet() {
  if (st) {
    (void)hipStreamSynchronize(st);
    (void)hipStreamDestroy(st);
  }
}

void GuessNet::repack() {
  for (int l = 0; l < kGuessLayers; ++l) {
    const GuessLayer &g = ly[l];
    const int nf = g.nchunk * g.nb * 64;
    hipLaunchKernelGGL(k_gpack_fwd, dim3(grid_for(nf)), dim3(kBlock), 0, st, w.p, g.off_w, g.cin, g.cout,
                       g.nchunk, g.nb, pack.p + g.fpack);
    if (l > 0) {
      const int nbk = g.nchunk_b * (g.cin / 16) * 64;
      hipLaunchKernelGGL(k_gpack_bwd, dim3(grid_for(nbk)), dim3(kBlock), 0, st, w.p, g.off_w, g.cin, g.cout,
                         g.cin_b, g.nchunk_b, pack.p + g.bpack);
    }
  }
}

void GuessNet::set_params(const float *p, const GuessScale *s) {
  if (p) {
    w.upload(p, kGuessParams, st);
    CG_HIP(hipMemsetAsync(m.p, 0, sizeof(float) * kGuessParams, st));
    CG_HIP(hipMemsetAsync(v.p, 0, sizeof(float) * kGuessParams, st));
    adam_t = 0;
    repack();
  }
  if (s) {
    for (int c = 0; c < kGuessIn; ++c) CG_REQUIRE(s->sd[c] > 0.f, "guess net: feature scales must be > 0");
    CG_REQUIRE(s->floor >= 0.f, "guess net: floor must be >= 0");
    scale = *s;
  }
  CG_HIP(hipStreamSynchronize(st));
}

void GuessNet::get_params(float *p, GuessScale *s) {
  if (p) {
    w.download(p, kGuessParams, st);
    CG_HIP(hipStreamSynchronize(st));
  }
  if (s) *s = scale;
}

void GuessNet::ensure(int ncol) {
  CG_REQUIRE(ncol > 0, "guess net: no columns");
  if (ncol <= cap) return;
  const size_t pos = (size_t)ncol * Lp;
  cap = 0;  // should an allocation fail
  xs.alloc(pos * kGuessIn);
  y32.alloc(pos);
  ts.alloc(pos);
  if (!hist.p) hist.alloc(1);
  if (!fused()) {
    for (auto &a : act) a.alloc(pos * kGuessWidth);
    for (auto &a : gb) a.alloc(pos * kGuessWidth);
    ghead.alloc(pos * 16);
    lossp.alloc(grid_for(pos));
    const int nsplit = split_count(ncol, Lp);
    size_t po = 0;
    for (int l = 0; l < kGuessLayers; ++l) {
      ly[l].part = po;
      po += (size_t)nsplit * ly[l].nchunk_w * 16 * ly[l].nb * 16;
    }
    part.alloc(po);
  }
  cap = ncol;
}

// Columns of at most kTileRows levels run through k_gfused (a tile of 64 rows
// keeps the activations and gradients of a training pass in 58 KB of LDS);
// deeper ones do not fit a tile and run layer by layer.
bool GuessNet::fused() const { return Lp <= kTileRows; }
int GuessNet::tiles(int ncol) const {
  const int cpt = kTileBlocks / (Lp >> 4);
  return (ncol + cpt - 1) / cpt;
}

static FusedNet fused_net(const GuessNet &g) {
  FusedNet f{};
  f.pack = g.pack.p;
  f.w = g.w.p;
  for (int l = 0; l < kGuessLayers; ++l) {
    f.fpack[l] = g.ly[l].fpack;
    f.bpack[l] = g.ly[l].bpack;
    f.off_b[l] = g.ly[l].off_b;
  }
  return f;
}

void GuessNet::forward(const unsigned short *x, const int *idx, int ncol, float *y) {
  ensure(ncol);
  if (fused()) {
    hipLaunchKernelGGL(k_gfused<false>, dim3(std::min(tiles(ncol), kFwdGroups)), dim3(512), 0, st, fused_net(*this), ncol,
                       Lp, L, idx, x, (const float *)nullptr, 0.f, y, (float *)nullptr, (float *)nullptr);
    return;
  }
  const int gw = waves_blocks((long)ncol * (Lp / 16));
  const float *W = w.p;
  hipLaunchKernelGGL((k_gconv<kGuessIn, 4>), dim3(gw), dim3(kBlock), 0, st, ncol, Lp, L, idx, x, pack.p + ly[0].fpack,
                     W + ly[0].off_b, 64, 1, (const unsigned short *)nullptr, act[0].p, (float *)nullptr);
  for (int l = 1; l < 4; ++l)
    hipLaunchKernelGGL((k_gconv<64, 4>), dim3(gw), dim3(kBlock), 0, st, ncol, Lp, L, (const int *)nullptr,
                       act[l - 1].p, pack.p + ly[l].fpack, W + ly[l].off_b, 64, 1, (const unsigned short *)nullptr,
                       act[l].p, (float *)nullptr);
  hipLaunchKernelGGL((k_gconv<64, 1>), dim3(gw), dim3(kBlock), 0, st, ncol, Lp, L, (const int *)nullptr, act[3].p,
                     pack.p + ly[4].fpack, W + ly[4].off_b, 1, 0, (const unsigned short *)nullptr,
                     (unsigned short *)nullptr, y);
}

// One gradient of the mean squared error into grad and its loss into
// loss_slot; with lr the Adam step on it (the packs follow the weights).
void GuessNet::gradient(const unsigned short *x, const int *idx, const float *t, int ncol, float *loss_slot,
                        const float *lr) {
  ensure(ncol);
  const float inv = 1.0f / ((float)ncol * (float)L);
  GradParts gp{};
  int nloss;
  if (fused()) {
    const int G = std::min(tiles(ncol), kTrainGroups);
    if (part.n < (size_t)G * kPartSize) part.alloc((size_t)G * kPartSize);
    if (lossp.n < (size_t)G) lossp.alloc(G);
    hipLaunchKernelGGL(k_gfused<true>, dim3(G), dim3(512), 0, st, fused_net(*this), ncol, Lp, L, idx, x, t, inv,
                       (float *)nullptr, lossp.p, part.p);
    nloss = gp.nsplit = G;
    for (int l = 0; l < kGuessLayers; ++l) {
      gp.off[l] = kPartOff[l];
      gp.stride[l] = kPartSize;
    }
  } else {
    nloss = layered_gradient(x, idx, t, ncol, inv);
    gp.nsplit = split_count(ncol, Lp);
    for (int l = 0; l < kGuessLayers; ++l) {
      gp.off[l] = ly[l].part;
      gp.stride[l] = (size_t)ly[l].nchunk_w * 16 * ly[l].nb * 16;
    }
  }
  gp.part = part.p;
  GradLayers gl{};
  for (int l = 0; l < kGuessLayers; ++l) {
    gp.gs[l] = ly[l].nb * 16;
    gl.off_w[l] = ly[l].off_w;
    gl.cin[l] = ly[l].cin;
    gl.cout[l] = ly[l].cout;
    gl.nb[l] = ly[l].nb;
    gl.fpack[l] = (unsigned)ly[l].fpack;
    gl.bpack[l] = (unsigned)ly[l].bpack;
  }
  const dim3 g(grid_for(kGuessParams, kStepCols)), b(kStepCols * kStepRows);
  short *pk = reinterpret_cast<short *>(pack.p);
  if (!lr) {
    hipLaunchKernelGGL(k_gstep<false>, g, b, 0, st, gp, gl, lossp.p, nloss, inv, loss_slot, grad.p, w.p, m.p, v.p, 0.f,
                       0.f, 0.f, 0.f, pk);
    return;
  }
  ++adam_t;
  const double b1 = 0.9, b2 = 0.999;
  const double lr_t = *lr * std::sqrt(1.0 - std::pow(b2, (double)adam_t)) / (1.0 - std::pow(b1, (double)adam_t));
  hipLaunchKernelGGL(k_gstep<true>, g, b, 0, st, gp, gl, lossp.p, nloss, inv, loss_slot, grad.p, w.p, m.p, v.p,
                     (float)lr_t, (float)b1, (float)b2, 1e-8f, pk);
}

// The gradient's partials layer by layer; returns the count of loss partials.
int GuessNet::layered_gradient(const unsigned short *x, const int *idx, const float *t, int ncol, float inv) {
  forward(x, idx, ncol, y32.p);
  const int gl = grid_for((size_t)ncol * Lp);
  hipLaunchKernelGGL(k_gloss, dim3(gl), dim3(kBlock), 0, st, ncol, Lp, L, y32.p, idx, t, inv, ghead.p, lossp.p);
  const int ns = split_count(ncol, Lp);
  const int gw = waves_blocks((long)ncol * (Lp / 16));
  auto dw_blocks = [&](const GuessLayer &g) { return waves_blocks((long)g.nchunk_w * g.nb * ns); };
  // head
  hipLaunchKernelGGL((k_gdw<64, 16>), dim3(dw_blocks(ly[4])), dim3(kBlock), 0, st, ncol, Lp, L,
                     (const int *)nullptr, act[3].p, ghead.p, ns, part.p + ly[4].part);
  hipLaunchKernelGGL((k_gconv<16, 4>), dim3(gw), dim3(kBlock), 0, st, ncol, Lp, L, (const int *)nullptr, ghead.p,
                     pack.p + ly[4].bpack, (const float *)nullptr, 64, 0, act[3].p, gb[0].p, (float *)nullptr);
  // hidden layers 3, 2, 1: gradient in gb[cur], input activation act[l-1]
  int cur = 0;
  for (int l = 3; l >= 1; --l) {
    hipLaunchKernelGGL((k_gdw<64, 64>), dim3(dw_blocks(ly[l])), dim3(kBlock), 0, st, ncol, Lp, L,
                       (const int *)nullptr, act[l - 1].p, gb[cur].p, ns, part.p + ly[l].part);
    hipLaunchKernelGGL((k_gconv<64, 4>), dim3(gw), dim3(kBlock), 0, st, ncol, Lp, L, (const int *)nullptr,
                       gb[cur].p, pack.p + ly[l].bpack, (const float *)nullptr, 64, 0, act[l - 1].p,
                       gb[1 - cur].p, (float *)nullptr);
    cur = 1 - cur;
  }
  hipLaunchKernelGGL((k_gdw<kGuessIn, 64>), dim3(dw_blocks(ly[0])), dim3(kBlock), 0, st, ncol, Lp, L, idx, x, gb[cur].p,
                     ns, part.p + ly[0].part);
  return gl;
}

// ------------------------------------------------------------ handles --
static std::mutex g_gmu;
static std::map<int64_t, std::shared_ptr<GuessNet>> g_nets;
static int64_t g_gnext = 1;

std::shared_ptr<GuessNet> guess_lookup(int64_t h) {
  std::lock_guard<std::mutex> lk(g_gmu);
  auto it = g_nets.find(h);
  if (it == g_nets.end()) throw Error(CATHY_GPU_EHANDLE, "unknown guess-net handle");
  return it->second;
}

}  // namespace cg

using namespace cg;

static GuessScale scale_from(const float *s) {
  GuessScale g;
  for (int c = 0; c < kGuessIn; ++c) {
    g.mu[c] = s[c];
    g.sd[c] = s[kGuessIn + c];
  }
  g.out = s[2 * kGuessIn];
  g.floor = s[2 * kGuessIn + 1];
  g.beta = s[2 * kGuessIn + 2];
  g.band = s[2 * kGuessIn + 3];
  return g;
}

extern "C" {

int cathy_gpu_guess_create(int64_t *net, const int *levels, int *nparam) {
  return guarded([&] {
    CG_REQUIRE(net && levels, "null argument");
    auto g = std::make_shared<GuessNet>(*levels);
    std::lock_guard<std::mutex> lk(g_gmu);
    *net = g_gnext++;
    g_nets[*net] = std::move(g);
    if (nparam) *nparam = kGuessParams;
    return 0;
  });
}

int cathy_gpu_guess_destroy(int64_t *net) {
  return guarded([&] {
    std::lock_guard<std::mutex> lk(g_gmu);
    if (!net || !g_nets.count(*net)) throw Error(CATHY_GPU_EHANDLE, "unknown guess-net handle");
    g_nets.erase(*net);
    *net = 0;
    return 0;
  });
}

int cathy_gpu_guess_set(int64_t *net, const float *params, const float *scale) {
  return guarded([&] {
    CG_REQUIRE(net, "null argument");
    auto g = guess_lookup(*net);
    std::lock_guard<std::mutex> lk(g->mu);
    GuessScale s;
    if (scale) s = scale_from(scale);
    g->set_params(params, scale ? &s : nullptr);
    return 0;
  });
}

int cathy_gpu_guess_get(int64_t *net, float *params, float *scale) {
  return guarded([&] {
    CG_REQUIRE(net, "null argument");
    auto g = guess_lookup(*net);
    std::lock_guard<std::mutex> lk(g->mu);
    GuessScale s;
    g->get_params(params, &s);
    if (scale) {
      for (int c = 0; c < kGuessIn; ++c) {
        scale[c] = s.mu[c];
        scale[kGuessIn + c] = s.sd[c];
      }
      scale[2 * kGuessIn] = s.out;
      scale[2 * kGuessIn + 1] = s.floor;
      scale[2 * kGuessIn + 2] = s.beta;
      scale[2 * kGuessIn + 3] = s.band;
    }
    return 0;
  });
}

int cathy_gpu_guess_forward(int64_t *net, const int *ncol, const uint16_t *x, float *y) {
  return guarded([&] {
    CG_REQUIRE(net && ncol && x && y && *ncol > 0, "bad argument");
    auto g = guess_lookup(*net);
    std::lock_guard<std::mutex> lk(g->mu);
    g->ensure(*ncol);
    const size_t pos = (size_t)*ncol * g->Lp;
    g->xs.upload(x, pos * kGuessIn, g->st);
    g->forward(g->xs.p, nullptr, *ncol, g->y32.p);
    g->y32.download(y, pos, g->st);
    CG_HIP(hipStreamSynchronize(g->st));
    return 0;
  });
}

int cathy_gpu_guess_gradient(int64_t *net, const int *ncol, const uint16_t *x, const float *t, float *loss,
                             float *grad) {
  return guarded([&] {
    CG_REQUIRE(net && ncol && x && t && *ncol > 0, "bad argument");
    auto g = guess_lookup(*net);
    std::lock_guard<std::mutex> lk(g->mu);
    g->ensure(*ncol);
    const size_t pos = (size_t)*ncol * g->Lp;
    g->xs.upload(x, pos * kGuessIn, g->st);
    g->ts.upload(t, pos, g->st);
    g->gradient(g->xs.p, nullptr, g->ts.p, *ncol, g->hist.p, nullptr);
    if (loss) g->hist.download(loss, 1, g->st);
    if (grad) g->grad.download(grad, kGuessParams, g->st);
    CG_HIP(hipStreamSynchronize(g->st));
    return 0;
  });
}

int cathy_gpu_guess_load(int64_t *net, const int64_t *nsamp, const uint16_t *x, const float *t) {
  return guarded([&] {
    CG_REQUIRE(net && nsamp && x && t && *nsamp > 0, "bad argument");
    auto g = guess_lookup(*net);
    std::lock_guard<std::mutex> lk(g->mu);
    const size_t pos = (size_t)*nsamp * g->Lp;
    g->nsamp = 0;  // no training set should an allocation fail
    g->X.alloc(pos * kGuessIn);
    g->T.alloc(pos);
    g->X.upload(x, pos * kGuessIn, g->st);
    g->T.upload(t, pos, g->st);
    g->nsamp = *nsamp;
    CG_HIP(hipStreamSynchronize(g->st));
    return 0;
  });
}

int cathy_gpu_guess_train(int64_t *net, const int *nsteps, const int *batch, const int *idx, const float *lr,
                          float *loss) {
  return guarded([&] {
    CG_REQUIRE(net && nsteps && batch && idx && lr && *nsteps > 0 && *batch > 0, "bad argument");
    auto g = guess_lookup(*net);
    std::lock_guard<std::mutex> lk(g->mu);
    CG_REQUIRE(g->nsamp > 0, "no training set loaded");
    const size_t nidx = (size_t)*nsteps * *batch;
    for (size_t i = 0; i < nidx; ++i)
      CG_REQUIRE(idx[i] >= 0 && idx[i] < g->nsamp, "sample index out of range");
    g->ensure(*batch);
    g->bidx.alloc(nidx);
    g->bidx.upload(idx, nidx, g->st);
    DBuf<float> h(*nsteps);
    for (int s = 0; s < *nsteps; ++s)
      g->gradient(g->X.p, g->bidx.p + (size_t)s * *batch, g->T.p, *batch, h.p + s, lr);
    if (loss) h.download(loss, *nsteps, g->st);
    CG_HIP(hipStreamSynchronize(g->st));
    CG_HIP(hipGetLastError());
    return 0;
  });
}

}  // extern "C"
