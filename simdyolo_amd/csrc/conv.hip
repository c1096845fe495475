// Convolution: weight preparation, algorithm routing and the gfx950 kernels,
// but for the two that multiply float32 as f16 pairs, which most layers run:
// split_gemm.hip (implicit GEMM) and split_conv3.hip (3x3 from an LDS patch).
//
//  * implicit GEMM on FP32 MFMA (v_mfma_f32_32x32x2f32): M = output pixels
//    (NHWC rows), N = output channels, K = (ky, kx, ic).  A rows are gathered
//    from the NHWC input on load (im2col never materialised), B is the packed
//    weight matrix [ocp][kp]; both are staged through LDS, double buffered.
//    Epilogue fuses bias, SiLU, the Bottleneck residual add and the write into
//    a channel slice of a concat buffer.
//  * Winograd F(4x4,3x3) for 3x3 s1 p1: input transform V = B^T d B per 6x6
//    patch, 36 batched MFMA GEMMs M[p] = V[p] U[p]^T (the implicit-GEMM kernel
//    with K = ic), inverse transform Y = A^T M A with the same epilogue.
//  * direct low-channel conv for the stem (ic = 3), reading the network's
//    NCHW input directly so the boundary layout change costs no extra pass.
//
// Routing mirrors DeviceConv (src/SimdYolo/VulkanExecution.cs:337-350).
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <utility>

#include "igemm.h"
#include "sy_internal.h"

namespace sy {

// KIND only separates the instantiations by caller (0 convolution, 1 Winograd
// plane GEMM, 2 plain GEMM) so that profilers report them apart.  MODE picks
// the A-row addressing:
//   0  general im2col: (ky, kx, ic) recovered from k per K tile;
//   1  IC % 16 == 0: every K tile lies inside one tap, so (ky, kx, ic0) are
//      uniform counters advanced per tile and a row costs one add and a
//      bounds test;
//   2  plain GEMM rows (1x1 s1 p0 conv, Winograd planes, gemm_nt): A row m
//      starts at x + m * ldx.
//
// PF is the number of K tiles in flight ahead of the one being multiplied:
// PF = 1 loads tile k+1 into registers while tile k is multiplied from LDS;
// PF = 2 keeps two register sets, so a tile's loads are issued two
// iterations before its LDS store and have two tiles' MFMA time to land
// (short-K and HBM-bound shapes, where one tile of MFMAs does not cover the
// memory latency).
template <int KIND, int MODE, int BM, int BN, int WM, int WN, int BK, int PF = 1>
// Occupancy targets where VGPRs, not LDS, would limit it: four-wave tiles of
// at most 64 x 64 (20 KiB of LDS at K tiles of 16: eight workgroups per CU)
// are compiled for eight waves per SIMD (64 VGPRs), 128 x 64 tiles with K
// tiles of 16 (31 KiB) for four (at most 128 VGPRs); neither spills.
// Measured on YOLOv8n: batch 1 0.7% faster, batch 32 unchanged.
__global__ __launch_bounds__(WM* WN * 64, (BM * BN <= 64 * 64 && WM * WN == 4)                   ? 8
                                          : (BM == 128 && BN == 64 && BK == 16 && WM * WN == 4) ? 4
                                                                                                  : 1) void igemm_kernel(
    const IgemmArgs a) {
  constexpr int NT = WM * WN * 64;
  constexpr int LDK = BK + 4;
  constexpr int QK = BK / 4;  // float4 chunks per K-tile row
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int A_IT = (BM * QK + NT - 1) / NT;
  constexpr int B_IT = (BN * QK + NT - 1) / NT;
  static_assert(BK == 16 || BK == 32, "K tile is 16 or 32");
  static_assert(TM >= 1 && TN >= 1, "wave tile must hold a 32x32 MFMA block");
  __shared__ __attribute__((aligned(16))) float As[2][BM][LDK];
  __shared__ __attribute__((aligned(16))) float Bs[2][BN][LDK];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wid = tid >> 6;
  const int wm = wid / WN, wn = wid % WN;
  const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
  const float* __restrict__ x = a.x + (long long)blockIdx.z * a.xb;
  const float* __restrict__ wt = a.w + (long long)blockIdx.z * a.wb;
  float* __restrict__ y = a.y + (long long)blockIdx.z * a.yb;
  const int quad = tid % QK;

  // Rows of A this thread gathers.  MODE 2: the row start.  Otherwise the
  // image base, the offset of the top-left tap (may point outside the image;
  // only dereferenced after the bounds test) and its coordinates.
  const float* a_img[A_IT];
  const float* a_up[A_IT];  // MODE 3: the row's half-resolution pixel
  int a_iy[A_IT], a_ix[A_IT], a_pix[A_IT];
  bool a_ok[A_IT];
#pragma unroll
  for (int i = 0; i < A_IT; ++i) {
    int r = (tid + i * NT) / QK;
    int m = m0 + r;
    a_ok[i] = (tid + i * NT) < BM * QK && m < a.M;
    int mm = a_ok[i] ? m : 0;
    if (MODE == 2 || MODE == 3) {
      a_img[i] = x + (long long)mm * a.ldx;
      a_iy[i] = a_ix[i] = a_pix[i] = 0;
      if (MODE == 3) {
        const int ox = mm % a.W, t = mm / a.W, oy = t % a.H, n = t / a.H;
        a_up[i] = a.xu + ((long long)(n * (a.H >> 1) + (oy >> 1)) * (a.W >> 1) + (ox >> 1)) * a.ldxu;
      }
    } else {
      int ox = mm % a.OW;
      int t = mm / a.OW;
      int oy = t % a.OH;
      int n = t / a.OH;
      a_iy[i] = oy * a.SH - a.PH;
      a_ix[i] = ox * a.SW - a.PW;
      a_pix[i] = (a_iy[i] * a.W + a_ix[i]) * a.ldx;
      a_img[i] = x + (long long)n * a.H * a.W * a.ldx;
    }
  }
  // Split K: this workgroup's K range (a whole number of K tiles).
  const int kbeg = a.part ? (int)blockIdx.z * a.kchunk : 0;
  const int kend = a.part ? min(a.K, kbeg + a.kchunk) : a.K;
  // MODE 1: tap and channel offset of the next K tile to load (uniform).
  int t_ic = kbeg % a.IC, t_ky = (kbeg / a.IC) / a.KW, t_kx = (kbeg / a.IC) % a.KW;

  // Operand loads are branch-free: a lane whose element lies outside the
  // operand (padding, ragged M or K) loads from a valid base address instead
  // and its value is replaced by zero when it is stored to LDS.  A load under
  // a branch makes the compiler wait for it right away to merge the branch's
  // registers, so the prefetch would not overlap the MFMAs.
  struct Stage {
    f32x4 a[A_IT], b[B_IT];
    bool aok[A_IT], bok[B_IT];
  };
  Stage st0, st1;
  auto gload = [&](int k0, Stage& g) {
    const int k = k0 + quad * 4;
    const bool kok = MODE == 1 || k < kend;
    if (MODE == 2) {
#pragma unroll
      for (int i = 0; i < A_IT; ++i) {
        g.aok[i] = a_ok[i] && kok;
        g.a[i] = *(const f32x4*)(g.aok[i] ? a_img[i] + k : x);
      }
    } else if (MODE == 3) {
      const bool up = k0 < a.ku;  // uniform: ku is a whole number of K tiles
#pragma unroll
      for (int i = 0; i < A_IT; ++i) {
        g.aok[i] = a_ok[i] && kok;
        g.a[i] = *(const f32x4*)(g.aok[i] ? (up ? a_up[i] + k : a_img[i] + (k - a.ku)) : x);
      }
    } else if (MODE == 1) {
      const int dy = t_ky * a.DH, dx = t_kx * a.DW;
      const int off = (dy * a.W + dx) * a.ldx + t_ic + quad * 4;
#pragma unroll
      for (int i = 0; i < A_IT; ++i) {
        const int iy = a_iy[i] + dy, ix = a_ix[i] + dx;
        g.aok[i] = a_ok[i] && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
        g.a[i] = *(const f32x4*)(a_img[i] + (g.aok[i] ? a_pix[i] + off : 0));
      }
      t_ic += BK;
      if (t_ic == a.IC) {
        t_ic = 0;
        if (++t_kx == a.KW) {
          t_kx = 0;
          ++t_ky;
        }
      }
    } else {
      int tap = k / a.IC;
      int ic = k - tap * a.IC;
      int ky = tap / a.KW, kx = tap - (tap / a.KW) * a.KW;
#pragma unroll
      for (int i = 0; i < A_IT; ++i) {
        int iy = a_iy[i] + ky * a.DH, ix = a_ix[i] + kx * a.DW;
        g.aok[i] = a_ok[i] && kok && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
        g.a[i] = *(const f32x4*)(a_img[i] + (g.aok[i] ? ((long long)iy * a.W + ix) * a.ldx + ic : 0));
      }
    }
#pragma unroll
    for (int i = 0; i < B_IT; ++i) {
      const int idx = tid + i * NT;
      const int row = n0 + idx / QK;
      // Packed conv weights are zero-padded to [ocp][kp]; other B operands
      // (e.g. mask prototypes) are bounds-checked instead.
      g.bok[i] = idx < BN * QK && (!a.bguard || (row < a.Nb && kok));
      g.b[i] = *(const f32x4*)(wt + (g.bok[i] ? (long long)row * a.Kp + k0 + quad * 4 : 0));
    }
  };
  auto sstore = [&](int buf, const Stage& g) {
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < A_IT; ++i) {
      int idx = tid + i * NT;
      if (idx < BM * QK) *(f32x4*)&As[buf][idx / QK][quad * 4] = g.aok[i] ? g.a[i] : z;
    }
#pragma unroll
    for (int i = 0; i < B_IT; ++i) {
      int idx = tid + i * NT;
      if (idx < BN * QK) *(f32x4*)&Bs[buf][idx / QK][quad * 4] = g.bok[i] ? g.b[i] : z;
    }
  };

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int half = lane >> 5, r32 = lane & 31;
  const int nk = (kend - kbeg + BK - 1) / BK;
  // Multiplies the K tile held in LDS buffer cur.
  auto mma = [&](int cur) {
    // Lane half h consumes k = (BK/2) h + s at MFMA step s; A and B agree.
    constexpr int HK = BK / 8;  // float4 reads per row and lane half
    f32x4 av[TM][HK], bv[TN][HK];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const float* p = &As[cur][wm * (BM / WM) + i * 32 + r32][half * (BK / 2)];
#pragma unroll
      for (int q = 0; q < HK; ++q) av[i][q] = *(const f32x4*)(p + 4 * q);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const float* p = &Bs[cur][wn * (BN / WN) + j * 32 + r32][half * (BK / 2)];
#pragma unroll
      for (int q = 0; q < HK; ++q) bv[j][q] = *(const f32x4*)(p + 4 * q);
    }
#pragma unroll
    for (int s = 0; s < BK / 2; ++s)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i][s >> 2][s & 3], bv[j][s >> 2][s & 3], acc[i][j], 0,
                                                           0, 0);
  };
  if (PF == 1) {
    gload(kbeg, st0);
    sstore(0, st0);
    __syncthreads();
    for (int kc = 0; kc < nk; ++kc) {
      const int cur = kc & 1;
      if (kc + 1 < nk) gload(kbeg + (kc + 1) * BK, st0);
      mma(cur);
      if (kc + 1 < nk) sstore(cur ^ 1, st0);
      __syncthreads();
    }
  } else {
    // Stage st0 carries even K tiles, st1 odd ones; the loop is unrolled by
    // two so both stay in registers.  While tile kc is multiplied, tile
    // kc + 2 is loaded and tile kc + 1 (loaded one tile earlier) is stored
    // into the other LDS buffer.
    gload(kbeg, st0);
    if (nk > 1) gload(kbeg + BK, st1);
    sstore(0, st0);
    __syncthreads();
    int kc = 0;
    for (; kc + 1 < nk; kc += 2) {
      if (kc + 2 < nk) gload(kbeg + (kc + 2) * BK, st0);
      mma(0);
      sstore(1, st1);
      __syncthreads();
      if (kc + 3 < nk) gload(kbeg + (kc + 3) * BK, st1);
      mma(1);
      if (kc + 2 < nk) sstore(0, st0);
      __syncthreads();
    }
    if (kc < nk) mma(0);  // odd tile count: the last tile sits in buffer 0
  }

  // D layout of the 32x32 MFMA: lane holds column (lane & 31) and rows
  // 8*(r/4) + 4*(lane/32) + (r%4) for r = 0..15.
  const int rbase = m0 + wm * (BM / WM) + 4 * half;
  if (a.part) {
    float* __restrict__ P = a.part + (long long)blockIdx.z * a.M * a.ldp;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int col = n0 + wn * (BN / WN) + j * 32 + r32;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = rbase + i * 32 + 8 * (r >> 2) + (r & 3);
          if (row < a.M) P[(long long)row * a.ldp + col] = acc[i][j][r];
        }
    }
    return;
  }
  if (MODE == 2 && a.shuf > 0) {
    store_shuf<TM, TN>(a, y, acc, rbase, n0 + wn * (BN / WN) + r32);
    return;
  }
  store_acc<TM, TN>(a, y, acc, rbase, n0 + wn * (BN / WN) + r32);
}

struct TileCfg {
  int bm, bn, wm, wn, bk, pf;
};

// Macro tile, wave grid, K depth and prefetch depth of each igemm instantiation.
#define SY_TILE_LIST(X)             \
  X(0, 128, 128, 2, 2, 16, 1)       \
  X(1, 128, 64, 2, 2, 16, 1)        \
  X(2, 64, 64, 2, 2, 16, 1)         \
  X(3, 128, 32, 4, 1, 16, 1)        \
  X(4, 64, 32, 2, 1, 16, 1)         \
  X(5, 256, 64, 4, 1, 16, 1)        \
  X(6, 128, 64, 2, 1, 16, 1)        \
  X(7, 128, 64, 2, 2, 32, 1)        \
  X(8, 128, 128, 2, 2, 32, 1)       \
  X(9, 256, 32, 4, 1, 16, 1)        \
  X(10, 256, 128, 4, 2, 16, 1)      \
  X(11, 64, 64, 2, 2, 32, 1)        \
  X(12, 128, 32, 4, 1, 32, 1)       \
  X(13, 64, 32, 2, 1, 32, 1)        \
  X(14, 64, 64, 2, 2, 32, 2)        \
  X(15, 128, 64, 2, 2, 32, 2)       \
  X(16, 64, 64, 2, 2, 16, 2)        \
  X(17, 128, 32, 4, 1, 16, 2)       \
  X(18, 256, 64, 4, 1, 16, 2)       \
  X(19, 128, 128, 2, 2, 16, 2)      \
  X(20, 64, 32, 2, 1, 32, 2)        \
  X(21, 128, 32, 4, 1, 32, 2)       \
  X(22, 64, 96, 2, 3, 16, 2)        \
  X(23, 64, 96, 2, 3, 32, 1)

#define SY_TILE_CFG(i, bm, bn, wm, wn, bk, pf) {bm, bn, wm, wn, bk, pf},
static const TileCfg kTiles[] = {SY_TILE_LIST(SY_TILE_CFG)};
#undef SY_TILE_CFG
static constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);
// Output-channel rows the packed weights are zero-padded to: the last column
// block of every tile (32, 64, 96 or 128 wide) reads inside them.
static int oc_pad(int oc) { return std::max((oc + 127) / 128 * 128, (oc + 95) / 96 * 96); }

// ------------------------------------------------------------ weight-stationary row GEMM
//
// y[m][n] = sum_k x[m][k] w[n][k] for skinny plain-row GEMMs (1x1 s1
// convolutions, Winograd planes): many rows, K and N small.  A workgroup copies
// its 32*NW x K slab of the weights into LDS once and keeps it there while each
// wave streams 32-row blocks of A from HBM straight into registers and
// multiplies them against the slab on 32x32x2 MFMAs.  Lane half h holds
// k in [h*KC/2, (h+1)*KC/2) of a KC-wide K chunk, so every lane loads
// contiguous float4s of its own row and the B fragments are float4 LDS reads
// of the same k.  The next chunk (of this row block or of the wave's next
// one) is loaded while the current one is multiplied.  Waves walk their row
// blocks with a grid-wide stride, so the weights are read once per workgroup
// instead of once per output tile.
constexpr int kPwWaves = 4;
constexpr int kPwBase = 32;               // tile ids kPwBase + NW - 1 select this kernel (NW = 1..4)
constexpr int kPwLdsMax = 64 * 1024;      // weight slab bytes per workgroup

static bool is_pw_tile(int t) { return t >= kPwBase && t < kPwBase + 4; }
static int pw_kc(int K) { return K % 64 == 0 ? 64 : K % 32 == 0 ? 32 : 16; }
static bool pw_fits(int K, int nw) { return K > 0 && K % 16 == 0 && (size_t)32 * nw * (K + 4) * 4 <= kPwLdsMax; }

template <int NW, int KC>
__global__ __launch_bounds__(kPwWaves * 64) void pw_kernel(const IgemmArgs a, int tiles32, int per_wave) {
  extern __shared__ __attribute__((aligned(16))) float ws[];  // [32*NW][K + 4]
  constexpr int NB = 32 * NW, HK = KC / 8;
  const int K = a.K, LDW = K + 4, K4 = K >> 2;
  const int n0 = blockIdx.y * NB;
  const float* __restrict__ wt = a.w + (long long)blockIdx.z * a.wb;
  const float* __restrict__ x = a.x + (long long)blockIdx.z * a.xb;
  float* __restrict__ y = a.y + (long long)blockIdx.z * a.yb;
  // The slab loads go out in batches of eight per thread before their LDS
  // stores (clamped in-range rows, zero past Nb), so their latencies overlap.
  for (int i0 = 0; i0 < NB * K4; i0 += 8 * kPwWaves * 64) {
    f32x4 sv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = min(i0 + u * kPwWaves * 64 + (int)threadIdx.x, NB * K4 - 1);
      const int r = i / K4, q = i - r * K4;
      const int row = n0 + r;
      const f32x4 t = *(const f32x4*)(wt + (long long)min(row, a.Nb - 1) * a.Kp + 4 * q);
      sv[u] = row < a.Nb ? t : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * kPwWaves * 64 + (int)threadIdx.x;
      if (i < NB * K4) {
        const int r = i / K4, q = i - r * K4;
        *(f32x4*)(ws + r * LDW + 4 * q) = sv[u];
      }
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int h = lane >> 5, r32 = lane & 31;
  const int stride = gridDim.x * kPwWaves;
  const int t0 = blockIdx.x * kPwWaves + wave;
  if (t0 >= tiles32) return;
  const int mine = min(per_wave, (tiles32 - 1 - t0) / stride + 1);
  const int nch = K / KC;
  float bias[NW];
#pragma unroll
  for (int j = 0; j < NW; ++j) {
    const int col = n0 + j * 32 + r32;
    bias[j] = (a.bias && col < a.OC) ? a.bias[col] : 0.f;
  }
  // Branch-free: rows past M read row M-1 and are zeroed by a select, so the
  // loads carry no control flow and their waits stay exact.
  auto load = [&](int tile, int c, f32x4* dst) {
    const int row = tile * 32 + r32;
    const bool ok = row < a.M;
    const float* src = x + (long long)min(row, a.M - 1) * a.ldx + c * KC + h * (KC / 2);
#pragma unroll
    for (int q = 0; q < HK; ++q) {
      const f32x4 v = *(const f32x4*)(src + 4 * q);
      dst[q] = ok ? v : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  f32x16 acc[NW];
#pragma unroll
  for (int j = 0; j < NW; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
  f32x4 cur[HK], nxt[HK];
  int tile = t0, c = 0;
  load(tile, 0, cur);
  const int iters = mine * nch;
  for (int it = 0; it < iters; ++it) {
    int nc = c + 1, ntile = tile;
    if (nc == nch) {
      nc = 0;
      ntile = tile + stride;
    }
    // Unconditional (the last iteration reloads its own chunk), so the wait
    // for this iteration's operands does not also wait for the prefetch.
    if (it + 1 < iters) load(ntile, nc, nxt);
    else load(tile, c, nxt);
    const float* wb = ws + r32 * LDW + c * KC + h * (KC / 2);
#pragma unroll
    for (int q = 0; q < HK; ++q) {
      f32x4 bv[NW];
#pragma unroll
      for (int j = 0; j < NW; ++j) bv[j] = *(const f32x4*)(wb + j * 32 * LDW + 4 * q);
#pragma unroll
      for (int st = 0; st < 4; ++st)
#pragma unroll
        for (int j = 0; j < NW; ++j) acc[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(cur[q][st], bv[j][st], acc[j], 0, 0, 0);
    }
    if (c == nch - 1) {
      // D layout: lane holds column (lane & 31), rows 8*(r/4) + 4*h + (r%4).
      // A block wholly inside the rows stores without per-row tests; each
      // column block's residual values are loaded before its stores.
      const int row0 = tile * 32 + 4 * h;
      const bool inner = tile * 32 + 32 <= a.M;
#pragma unroll
      for (int j = 0; j < NW; ++j) {
        const int col = n0 + j * 32 + r32;
        if (col < a.OC) {
          float* yr = y + (long long)row0 * a.ldy + col;
          float v[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            v[r] = acc[j][r] + bias[j];
            if (a.silu) v[r] = silu_fast(v[r]);
          }
          if (a.res) {
            const float* rr = a.res + (long long)row0 * a.ldr + col;
            float rv[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int dr = 8 * (r >> 2) + (r & 3);
              rv[r] = (inner || row0 + dr < a.M) ? rr[dr * a.ldr] : 0.f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) v[r] = rv[r] + v[r];
          }
          if (inner) {
#pragma unroll
            for (int r = 0; r < 16; ++r) yr[(8 * (r >> 2) + (r & 3)) * a.ldy] = v[r];
          } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int dr = 8 * (r >> 2) + (r & 3);
              if (row0 + dr < a.M) yr[dr * a.ldy] = v[r];
            }
          }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
      }
    }
#pragma unroll
    for (int q = 0; q < HK; ++q) cur[q] = nxt[q];
    tile = ntile;
    c = nc;
  }
}

template <int NW, int KC>
static int launch_pw_kc(sy_ctx* ctx, const IgemmArgs& a, int batch) {
  const int tiles32 = (a.M + 31) / 32;
  const int gy = (a.OC + 32 * NW - 1) / (32 * NW);
  const size_t lds = (size_t)32 * NW * (a.K + 4) * sizeof(float);
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pw_kernel<NW, KC>, kPwWaves * 64, lds) != hipSuccess ||
      per_cu < 1)
    per_cu = 1;
  const long long cap_waves = (long long)(ctx->cu_count > 0 ? ctx->cu_count : 256) * per_cu * kPwWaves;
  const long long groups = (long long)gy * batch;
  long long per_wave = ((long long)tiles32 * groups + cap_waves - 1) / cap_waves;
  if (per_wave < 1) per_wave = 1;
  long long gx = (tiles32 + kPwWaves * per_wave - 1) / (kPwWaves * per_wave);
  if (gy > 1) gx = (gx + 7) / 8 * 8;  // siblings along y share an XCD (and its L2 copy of the rows)
  SY_CHECK(gx <= 0x7fffffff && batch <= 65535 && gy <= 65535, SY_EUNSUPPORTED, "row GEMM grid too large");
  hipLaunchKernelGGL((pw_kernel<NW, KC>), dim3((unsigned)gx, gy, batch), dim3(kPwWaves * 64), lds, ctx->stream, a,
                     tiles32, (int)per_wave);
  return SY_OK;
}

// ------------------------------------------------------------ 3x3 conv, 16 input channels
//
// The C2f bottlenecks at 160x160 (16 -> 16) and the 16 -> 32 stride-2 conv
// are too narrow for 32-column MFMA tiles.  Here a workgroup stages the input
// patch of an 8x32 (stride 1) or 4x32 (stride 2) output tile in LDS (20
// floats per pixel: 16 channels + 4 of padding, which spreads a float4 read
// by 8 consecutive pixels over distinct banks) and each wave multiplies
// 16-pixel rows against the weights, held in registers, on 16x16x4 FP32
// MFMAs: lane l supplies pixel l % 16 and channels 4*(l/16)..+3 of a tap, one
// float4 feeding four MFMA steps; B lanes hold the same channels of weight
// row l % 16.  K = 9 taps x 16 channels; OC is one or two 16-column blocks.
constexpr int kC16Tile = 40;  // tile id that selects this kernel for a conv

template <int OC, int S, int TH>
__global__ __launch_bounds__(256) void conv_c16_kernel(const IgemmArgs a) {
  constexpr int TW = 32;
  constexpr int PH = (TH - 1) * S + 3, PW = (TW - 1) * S + 3, PS = 20;
  constexpr int NB = OC / 16;
  __shared__ __attribute__((aligned(16))) float patch[PH * PW * PS];
  const int tiles_x = (a.OW + TW - 1) / TW, tiles_y = (a.OH + TH - 1) / TH;
  int b = blockIdx.x;
  const int tx = b % tiles_x;
  b /= tiles_x;
  const int ty = b % tiles_y;
  const int n = b / tiles_y;
  if (n >= a.N) return;
  const int oy0 = ty * TH, ox0 = tx * TW;
  const int iy0 = oy0 * S - a.PH, ix0 = ox0 * S - a.PW;
  const float* __restrict__ img = a.x + (long long)n * a.H * a.W * a.ldx;
  // All of a thread's patch loads are issued before the first LDS store
  // (clamped, always in-bounds addresses; zero outside the image), so their
  // latencies overlap instead of adding up.
  constexpr int NP = PH * PW * 4, NI = (NP + 255) / 256;
  f32x4 pv[NI];
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int i = min(it * 256 + (int)threadIdx.x, NP - 1);
    const int q = i & 3, pix = i >> 2;
    const int py = pix / PW, px = pix - py * PW;
    const int iy = iy0 + py, ix = ix0 + px;
    const bool ok = (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
    const int cy = min(max(iy, 0), a.H - 1), cx = min(max(ix, 0), a.W - 1);
    const f32x4 t = *(const f32x4*)(img + ((long long)cy * a.W + cx) * a.ldx + 4 * q);
    pv[it] = ok ? t : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int i = it * 256 + (int)threadIdx.x;
    if (i < NP) *(f32x4*)&patch[(i >> 2) * PS + 4 * (i & 3)] = pv[it];
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l16 = lane & 15, kq = lane >> 4;
  // Packed weights [oc][tap * 16 + ic], Kp apart.
  f32x4 wr[NB][9];
  float bias[NB];
#pragma unroll
  for (int ob = 0; ob < NB; ++ob) {
    const float* wrow = a.w + (long long)(ob * 16 + l16) * a.Kp + 4 * kq;
#pragma unroll
    for (int t = 0; t < 9; ++t) wr[ob][t] = *(const f32x4*)(wrow + 16 * t);
    bias[ob] = a.bias ? a.bias[ob * 16 + l16] : 0.f;
  }
  __syncthreads();
  constexpr int RB = TW / 16;  // 16-pixel blocks per output row
  for (int pb = wave; pb < TH * RB; pb += 4) {
    const int r = pb / RB, xo = (pb % RB) * 16;
    // This block's residual values, loaded before its MFMAs so that the wait
    // for them does not fall between the block's stores.
    float rv[4][NB];
    if (a.res) {
      const int oy = min(oy0 + r, a.OH - 1);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int ox = min(ox0 + xo + 4 * kq + i, a.OW - 1);
        const long long pix = ((long long)n * a.OH + oy) * a.OW + ox;
#pragma unroll
        for (int ob = 0; ob < NB; ++ob) rv[i][ob] = a.res[pix * a.ldr + ob * 16 + l16];
      }
    }
    f32x4 acc[NB];
#pragma unroll
    for (int ob = 0; ob < NB; ++ob) acc[ob] = f32x4{0.f, 0.f, 0.f, 0.f};
    const float* prow = patch + ((r * S) * PW + (xo + l16) * S) * PS + 4 * kq;
#pragma unroll
    for (int ky = 0; ky < 3; ++ky)
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) {
        const f32x4 av = *(const f32x4*)(prow + (ky * PW + kx) * PS);
#pragma unroll
        for (int st = 0; st < 4; ++st)
#pragma unroll
          for (int ob = 0; ob < NB; ++ob)
            acc[ob] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[st], wr[ob][ky * 3 + kx][st], acc[ob], 0, 0, 0);
      }
    // D layout: lane holds column l16 of pixels 4*kq + i.
    const int oy = oy0 + r;
    if (oy >= a.OH) continue;
    float o[4][NB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ob = 0; ob < NB; ++ob) {
        float v = acc[ob][i] + bias[ob];
        if (a.silu) v = silu_fast(v);
        if (a.res) v = rv[i][ob] + v;
        o[i][ob] = v;
      }
    const long long pix0 = ((long long)n * a.OH + oy) * a.OW + ox0 + xo + 4 * kq;
    float* yp = a.y + pix0 * a.ldy + l16;
    if (ox0 + xo + 16 <= a.OW) {
      // All 16 pixels of the block lie inside the row: no per-pixel tests.
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int ob = 0; ob < NB; ++ob) yp[(long long)i * a.ldy + ob * 16] = o[i][ob];
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (ox0 + xo + 4 * kq + i >= a.OW) continue;
#pragma unroll
        for (int ob = 0; ob < NB; ++ob) yp[(long long)i * a.ldy + ob * 16] = o[i][ob];
      }
    }
  }
}

static bool c16_ok(const IgemmArgs& a) {
  return a.IC == 16 && (a.OC == 16 || a.OC == 32) && a.KH == 3 && a.KW == 3 && a.SH == a.SW &&
         (a.SH == 1 || a.SH == 2) && a.DH == 1 && a.DW == 1 && a.shuf == 0 && a.xb == 0 &&
         ((uintptr_t)a.x & 15) == 0 && a.ldx % 4 == 0 && a.Kp % 4 == 0 && a.Nb >= a.OC && a.K == 144;
}

static int launch_c16(sy_ctx* ctx, const IgemmArgs& a) {
  const int TH = a.SH == 1 ? 8 : 4, TW = 32;
  const long long blocks = (long long)a.N * ((a.OH + TH - 1) / TH) * ((a.OW + TW - 1) / TW);
  SY_CHECK(blocks <= 0x7fffffff, SY_EUNSUPPORTED, "conv grid too large");
  const dim3 grid((unsigned)blocks);
  void (*k)(const IgemmArgs) = nullptr;
#define SY_C16(oc, s, th) if (a.OC == oc && a.SH == s && TH == th) k = conv_c16_kernel<oc, s, th>;
  SY_C16(16, 1, 8) SY_C16(32, 1, 8) SY_C16(16, 2, 4) SY_C16(32, 2, 4)
#undef SY_C16
  SY_CHECK(k != nullptr, SY_EUNSUPPORTED, "no 16-channel conv kernel for oc %d stride %d rows %d", a.OC, a.SH, TH);
  hipLaunchKernelGGL(k, grid, dim3(256), 0, ctx->stream, a);
  return SY_OK;
}

template <int NW>
static int launch_pw(sy_ctx* ctx, const IgemmArgs& a, int batch) {
  switch (pw_kc(a.K)) {
    case 64: return launch_pw_kc<NW, 64>(ctx, a, batch);
    case 32: return launch_pw_kc<NW, 32>(ctx, a, batch);
    default: return launch_pw_kc<NW, 16>(ctx, a, batch);
  }
}

// SIMDYOLO_HIP_TILE pins the GEMM tile of convolutions whose tile is not
// chosen by the tuner (an explicit algorithm): 0..kNumTiles-1 igemm tiles,
// kPwBase..kPwBase+3 the weight-stationary row kernel.
static int env_tile() {
  const char* env = getenv("SIMDYOLO_HIP_TILE");
  return (env && *env) ? atoi(env) : -1;
}

static int pick_tile(sy_ctx* ctx, int M, int OC, int batch) {
  const int et = env_tile();
  if (et >= 0 && et < kNumTiles) return et;
  const long long want = 2LL * (ctx->cu_count > 0 ? ctx->cu_count : 256);
  int order[5];
  int no = 0;
  if (OC > 64) {
    order[no++] = 0; order[no++] = 1; order[no++] = 2; order[no++] = 4;
  } else if (OC > 32) {
    order[no++] = 1; order[no++] = 2; order[no++] = 4;
  } else {
    order[no++] = 3; order[no++] = 4;
  }
  int best = order[no - 1];
  for (int i = 0; i < no; ++i) {
    const TileCfg& c = kTiles[order[i]];
    long long wgs = (long long)((M + c.bm - 1) / c.bm) * ((OC + c.bn - 1) / c.bn) * batch;
    if (wgs >= want) return order[i];
  }
  return best;
}

// Profile name of an instantiation: igemm_m<MODE>_<BM>x<BN>_<WM><WN>_k<BK>
// for convolutions, wino_gemm_<...> for the Winograd plane GEMMs.
static const char* tile_name(int t, bool wino, int mode) {
  if (is_pw_tile(t)) {
    static const char* pw[2][4] = {{"pw_gemm_n32", "pw_gemm_n64", "pw_gemm_n96", "pw_gemm_n128"},
                                   {"wino_pw_n32", "wino_pw_n64", "wino_pw_n96", "wino_pw_n128"}};
    return pw[wino ? 1 : 0][t - kPwBase];
  }
  // Filled once, on first use (a function-local static: safe when contexts
  // on several threads launch for the first time together).
  struct Names {
    std::string n[2][4][kNumTiles];
    Names() {
      for (int w = 0; w < 2; ++w)
        for (int m = 0; m < 4; ++m)
          for (int i = 0; i < kNumTiles; ++i) {
            const TileCfg& c = kTiles[i];
            char buf[64];
            char pf[8] = "";
            if (c.pf > 1) snprintf(pf, sizeof pf, "_p%d", c.pf);
            if (w)
              snprintf(buf, sizeof buf, "wino_gemm_%dx%d_%d%d_k%d%s", c.bm, c.bn, c.wm, c.wn, c.bk, pf);
            else
              snprintf(buf, sizeof buf, "igemm_m%d_%dx%d_%d%d_k%d%s", m, c.bm, c.bn, c.wm, c.wn, c.bk, pf);
            n[w][m][i] = buf;
          }
    }
  };
  static const Names names;
  return names.n[wino ? 1 : 0][mode][t].c_str();
}

template <int KIND, int MODE>
static void launch_tile(int t, dim3 grid, hipStream_t st, const IgemmArgs& a) {
  switch (t) {
#define SY_TILE_CASE(i, bm, bn, wm, wn, bk, pf)                                                                \
  case i:                                                                                                      \
    hipLaunchKernelGGL((igemm_kernel<KIND, MODE, bm, bn, wm, wn, bk, pf>), grid, dim3(wm * wn * 64), 0, st, a); \
    break;
    SY_TILE_LIST(SY_TILE_CASE)
#undef SY_TILE_CASE
    default: break;
  }
}

// Whether tile t exists for these operands: every igemm tile runs plain-row
// and im2col operands; the weight-stationary kernel needs plain 16-byte rows,
// K % 16 == 0 and a weight slab that fits its LDS budget.
static bool gemm_tile_ok(int t, bool) { return t >= 0 && t < kNumTiles; }
static bool pw_ok(int t, const IgemmArgs& a, bool rows) {
  return is_pw_tile(t) && rows && a.shuf == 0 && ((uintptr_t)a.x & 15) == 0 && a.ldx % 4 == 0 && a.Kp % 4 == 0 &&
         a.xb % 4 == 0 && a.wb % 4 == 0 && pw_fits(a.K, t - kPwBase + 1);
}

// Split-K epilogue: y = [res +] act(sum_z part[z] + bias), summed in z order
// (deterministic), one thread per output element.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S, int M, int ldp,
                                                            int OC, const float* __restrict__ bias, int silu,
                                                            const float* __restrict__ res, int ldr,
                                                            float* __restrict__ y, int ldy) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)M * OC) return;
  const int m = (int)(i / OC), n = (int)(i - (long long)m * OC);
  const long long plane = (long long)M * ldp;
  const float* p = part + (long long)m * ldp + n;
  float v = p[0];
  for (int z = 1; z < S; ++z) v += p[z * plane];
  v += bias ? bias[n] : 0.f;
  if (silu) v = silu_fast(v);
  if (res) v = res[(long long)m * ldr + n] + v;
  y[(long long)m * ldy + n] = v;
}

// Largest split-K partial buffer (floats) a conv may use, and the largest
// unsplit grid (workgroups) for which splitting is tried.
constexpr long long kSplitMaxFloats = 8LL << 20;
constexpr long long kSplitGridMax = 256;

// K chunk (a whole number of K tiles) and effective split count for S.
static void split_chunks(int K, int bk, int S, int* kchunk, int* splits) {
  const int nt = (K + bk - 1) / bk;
  const int per = (nt + S - 1) / S;
  *kchunk = per * bk;
  *splits = (K + *kchunk - 1) / *kchunk;
}

static int env_split() {
  const char* env = getenv("SIMDYOLO_HIP_SPLIT");
  return (env && *env) ? atoi(env) : 1;
}

// ------------------------------------------------------------ in-workgroup split-K GEMM
//
// For small grids (batch 1), instead of splitting K over workgroups and
// reducing the partials in a second launch: one workgroup per 32x32 output
// tile, KW waves each taking a contiguous share of the K chunks.  A wave
// streams its own A and B fragments from global memory straight into MFMA
// operands (there is nothing to share between the waves of a tile): lane
// (row r = lane % 32, half h = lane / 32) loads the BK/2 consecutive k of its
// row that half h consumes, as float4s, one chunk ahead of the multiply.  The
// KW partial 32x32 tiles meet in LDS and are summed in wave order (the result
// does not depend on timing), then each wave finishes 16 / KW of the MFMA
// result registers with the epilogue.  MODE 1: IC % BK == 0, every K chunk
// lies inside one tap; MODE 2: plain rows (1x1 s1).
constexpr int kKsBase = 48;  // tile ids kKsBase + i select this kernel with 4 << i waves
static bool is_ks_tile(int t) { return t >= kKsBase && t < kKsBase + 3; }

template <int MODE, int KW, int BK>
__global__ __launch_bounds__(KW * 64) void igemm_ks_kernel(const IgemmArgs a) {
  constexpr int HK = BK / 8;  // float4 loads per lane and chunk, for A and for B
  static_assert(16 % KW == 0 || KW == 16, "waves divide the 16 result registers");
  __shared__ float red[KW][16][64];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int half = lane >> 5, r32 = lane & 31;
  const int m0 = blockIdx.x * 32, n0 = blockIdx.y * 32;
  const int m = m0 + r32;
  const bool mok = m < a.M;
  const int nch = (a.K + BK - 1) / BK;
  const int per = (nch + KW - 1) / KW;
  const int c0 = wid * per, c1 = min(nch, c0 + per);
  // This lane's A row: MODE 2 the row start; MODE 1 the image, the top-left
  // tap's coordinates (only dereferenced after the bounds test).
  const float* __restrict__ arow = a.x;
  int oy0 = 0, ox0 = 0;
  if (MODE == 2) {
    arow = a.x + (long long)(mok ? m : 0) * a.ldx;
  } else {
    const int mm = mok ? m : 0;
    const int ox = mm % a.OW, t = mm / a.OW, oy = t % a.OH, n = t / a.OH;
    oy0 = oy * a.SH - a.PH;
    ox0 = ox * a.SW - a.PW;
    arow = a.x + (long long)n * a.H * a.W * a.ldx;
  }
  const float* __restrict__ brow = a.w + (long long)(n0 + r32) * a.Kp + half * (BK / 2);
  auto load = [&](int c, f32x4* av, f32x4* bv) {
    const int k = c * BK + half * (BK / 2);
    if (MODE == 2) {
#pragma unroll
      for (int q = 0; q < HK; ++q)
        av[q] = (mok && k + 4 * q < a.K) ? *(const f32x4*)(arow + k + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
      const int tap = (c * BK) / a.IC, ic = k - tap * a.IC;
      const int ky = tap / a.KW, kx = tap - ky * a.KW;
      const int iy = oy0 + ky * a.DH, ix = ox0 + kx * a.DW;
      const bool ok = mok && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
      const float* src = arow + ((long long)iy * a.W + ix) * a.ldx + ic;
#pragma unroll
      for (int q = 0; q < HK; ++q) av[q] = ok ? *(const f32x4*)(src + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // Packed weights are zero-padded to [ocp][kp]: every read is in bounds.
#pragma unroll
    for (int q = 0; q < HK; ++q) bv[q] = *(const f32x4*)(brow + c * BK + 4 * q);
  };
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
  f32x4 av[2][HK], bv[2][HK];
  if (c0 < c1) load(c0, av[0], bv[0]);
  for (int c = c0; c < c1; ++c) {
    const int cur = (c - c0) & 1;
    if (c + 1 < c1) load(c + 1, av[cur ^ 1], bv[cur ^ 1]);
#pragma unroll
    for (int s = 0; s < BK / 2; ++s)
      acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av[cur][s >> 2][s & 3], bv[cur][s >> 2][s & 3], acc, 0, 0, 0);
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) red[wid][r][lane] = acc[r];
  __syncthreads();
  // D layout: lane holds column (lane & 31) and rows 8*(r/4) + 4*(lane/32) + (r%4).
  constexpr int RW = 16 / KW;
  const int col = n0 + r32;
  if (col < a.OC) {
    const float bvl = a.bias ? a.bias[col] : 0.f;
    // Residual values first: a wait for a load also waits for earlier stores.
    float rv[RW];
    if (a.res) {
#pragma unroll
      for (int i = 0; i < RW; ++i) {
        const int r = wid * RW + i;
        const int row = min(m0 + 8 * (r >> 2) + 4 * half + (r & 3), a.M - 1);
        rv[i] = a.res[(long long)row * a.ldr + col];
      }
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const int r = wid * RW + i;
      const int row = m0 + 8 * (r >> 2) + 4 * half + (r & 3);
      if (row >= a.M) continue;
      float v = red[0][r][lane];
#pragma unroll
      for (int w = 1; w < KW; ++w) v += red[w][r][lane];
      v += bvl;
      if (a.silu) v = silu_fast(v);
      if (a.res) v = rv[i] + v;
      a.y[(long long)row * a.ldy + col] = v;
    }
  }
}

// Operands the in-workgroup split-K kernel takes: a convolution (no batched
// GEMM, no sub-pixel scatter), plain rows or whole K chunks per tap, 16-byte
// aligned rows, 32-bit A offsets.
static int ks_mode(const IgemmArgs& a, bool rows, int* bk) {
  if (a.shuf || a.xb || ((uintptr_t)a.x & 15) || a.ldx % 4 || a.Kp % 4) return -1;
  if ((long long)a.H * a.W * a.ldx >= (1LL << 31) || (long long)a.M * a.ldx >= (1LL << 31)) return -1;
  if (rows) {
    *bk = 32;
    return 2;
  }
  if (a.IC % 16) return -1;
  *bk = a.IC % 32 == 0 ? 32 : 16;
  return 1;
}

// Names of the split-K forms [waves][mode][bk 16 / 32], filled once.
struct KsNames {
  std::string n[3][3][2];
  explicit KsNames(const char* fmt) {
    for (int i = 0; i < 3; ++i)
      for (int m = 0; m < 3; ++m)
        for (int b = 0; b < 2; ++b) {
          char buf[48];
          snprintf(buf, sizeof buf, fmt, 4 << i, m, b ? 32 : 16);
          n[i][m][b] = buf;
        }
  }
};

static const char* ks_name(int t, int mode, int bk) {
  static const KsNames names("igemm_ks%d_m%d_k%d");
  return names.n[t - kKsBase][mode][bk == 32 ? 1 : 0].c_str();
}

static int launch_ks(sy_ctx* ctx, int t, int mode, int bk, const IgemmArgs& a) {
  const dim3 grid((a.M + 31) / 32, (a.OC + 31) / 32);
  void (*k)(const IgemmArgs) = nullptr;
#define SY_KS(md, kw, b) \
  if (mode == md && (4 << (t - kKsBase)) == kw && bk == b) k = igemm_ks_kernel<md, kw, b>;
  SY_KS(1, 4, 16) SY_KS(1, 8, 16) SY_KS(1, 16, 16) SY_KS(1, 4, 32) SY_KS(1, 8, 32) SY_KS(1, 16, 32)
  SY_KS(2, 4, 32) SY_KS(2, 8, 32) SY_KS(2, 16, 32)
#undef SY_KS
  SY_CHECK(k != nullptr, SY_EINVAL, "no in-workgroup split-K kernel for mode %d tile %d", mode, t);
  hipLaunchKernelGGL(k, grid, dim3((4 << (t - kKsBase)) * 64), 0, ctx->stream, a);
  return SY_OK;
}

// ------------------------------------------------------------ in-workgroup split-K GEMM, 16x16 tiles
//
// The same scheme on 16x16 output tiles (v_mfma_f32_16x16x4f32): four times
// the workgroups of igemm_ks_kernel for a batch-1 grid, at the same matrix
// rate per SIMD.  A 3x3 128->128 conv at 20x20 gives 52 workgroups of 32x32
// on 256 CUs; here 200.  Lane (row l16 = lane % 16, group q = lane / 16)
// loads the BK/4 consecutive k of its row that group q consumes (MFMA step
// (h, s) of a chunk takes k = BK/4 * q + 4h + s from group q, for A and B
// alike), and a wave issues the loads of up to kKs16Ahead of its K chunks
// before their first MFMA (clamped to its last chunk, so every address is
// valid), one memory round trip per kKs16Ahead chunks.  The KW partial tiles
// are summed in LDS in wave order; waves 0..3 each finish one result
// register (rows 4q + r of column l16).
constexpr int kKs16Base = 52;   // tile ids kKs16Base + i select this kernel with 4 << i waves
constexpr int kKs16Ahead = 4;   // K chunks per round trip
static bool is_ks16_tile(int t) { return t >= kKs16Base && t < kKs16Base + 3; }

template <int MODE, int KW, int BK, bool BG>
__global__ __launch_bounds__(KW * 64) void igemm_ks16_kernel(const IgemmArgs a) {
  constexpr int HQ = BK / 16;  // float4 loads per lane and chunk, for A and for B
  static_assert(KW >= 4, "waves 0..3 finish the four result registers");
  __shared__ float red[KW][4][64];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int q = lane >> 4, l16 = lane & 15;
  const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16;
  const int m = m0 + l16;
  const bool mok = m < a.M;
  const int nch = (a.K + BK - 1) / BK;
  const int per = (nch + KW - 1) / KW;
  const int c0 = wid * per, c1 = min(nch, c0 + per);
  const float* __restrict__ arow = a.x;
  int oy0 = 0, ox0 = 0;
  if (MODE == 2) {
    arow = a.x + (long long)(mok ? m : 0) * a.ldx;
  } else {
    const int mm = mok ? m : 0;
    const int ox = mm % a.OW, t = mm / a.OW, oy = t % a.OH, n = t / a.OH;
    oy0 = oy * a.SH - a.PH;
    ox0 = ox * a.SW - a.PW;
    arow = a.x + (long long)n * a.H * a.W * a.ldx;
  }
  // B: packed conv weights are zero-padded to [ocp][kp], so every read is in
  // bounds; a plain row operand (BG, from a.bguard) has exactly Nb rows of K
  // values, so its reads use a clamped row and k and read zero past them.
  const bool brow_ok = !BG || n0 + l16 < a.Nb;
  const float* __restrict__ brow = a.w + (long long)(BG ? min(n0 + l16, a.Nb - 1) : n0 + l16) * a.Kp + q * (BK / 4);
  auto load = [&](int c, f32x4* av, f32x4* bv) {
    const int k = c * BK + q * (BK / 4);
    if (MODE == 2) {
#pragma unroll
      for (int h = 0; h < HQ; ++h)
        av[h] = (mok && k + 4 * h < a.K) ? *(const f32x4*)(arow + k + 4 * h) : f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
      const int tap = (c * BK) / a.IC, ic = k - tap * a.IC;
      const int ky = tap / a.KW, kx = tap - ky * a.KW;
      const int iy = oy0 + ky * a.DH, ix = ox0 + kx * a.DW;
      const bool ok = mok && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
      const float* src = arow + ((long long)iy * a.W + ix) * a.ldx + ic;
#pragma unroll
      for (int h = 0; h < HQ; ++h) av[h] = ok ? *(const f32x4*)(src + 4 * h) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int h = 0; h < HQ; ++h) {
      const int kk = c * BK + 4 * h;  // this float4's offset past brow's group start
      const f32x4 v = *(const f32x4*)(brow + (BG ? min(kk, a.K - 4 - q * (BK / 4)) : kk));
      bv[h] = (!BG || (brow_ok && k + 4 * h < a.K)) ? v : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  };
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int cb = c0; cb < c1; cb += kKs16Ahead) {
    f32x4 av[kKs16Ahead][HQ], bv[kKs16Ahead][HQ];
#pragma unroll
    for (int d = 0; d < kKs16Ahead; ++d) load(min(cb + d, c1 - 1), av[d], bv[d]);
#pragma unroll
    for (int d = 0; d < kKs16Ahead; ++d) {
      if (cb + d < c1) {
#pragma unroll
        for (int h = 0; h < HQ; ++h)
#pragma unroll
          for (int st = 0; st < 4; ++st)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[d][h][st], bv[d][h][st], acc, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) red[wid][r][lane] = acc[r];
  __syncthreads();
  if (wid >= 4) return;
  // D layout of the 16x16 MFMA: lane holds column l16 of rows 4q + r.
  const int r = wid, row = m0 + 4 * q + r, col = n0 + l16;
  if (row >= a.M || col >= a.OC) return;
  const float rv = a.res ? a.res[(long long)row * a.ldr + col] : 0.f;
  float v = red[0][r][lane];
#pragma unroll
  for (int w = 1; w < KW; ++w) v += red[w][r][lane];
  v += a.bias ? a.bias[col] : 0.f;
  if (a.silu) v = silu_fast(v);
  if (a.res) v = rv + v;
  a.y[(long long)row * a.ldy + col] = v;
}

static const char* ks16_name(int t, int mode, int bk) {
  static const KsNames names("igemm_ks%d_t16_m%d_k%d");
  return names.n[t - kKs16Base][mode][bk == 32 ? 1 : 0].c_str();
}

static int launch_ks16(sy_ctx* ctx, int t, int mode, int bk, const IgemmArgs& a) {
  const dim3 grid((a.M + 15) / 16, (a.OC + 15) / 16);
  void (*k)(const IgemmArgs) = nullptr;
  const bool bg = a.bguard != 0;
#define SY_KS16(md, kw, b, g) \
  if (mode == md && (4 << (t - kKs16Base)) == kw && bk == b && bg == g) k = igemm_ks16_kernel<md, kw, b, g>;
  SY_KS16(1, 4, 16, false) SY_KS16(1, 8, 16, false) SY_KS16(1, 16, 16, false) SY_KS16(1, 4, 32, false)
  SY_KS16(1, 8, 32, false) SY_KS16(1, 16, 32, false) SY_KS16(2, 4, 32, false) SY_KS16(2, 8, 32, false)
  SY_KS16(2, 16, 32, false) SY_KS16(2, 4, 32, true) SY_KS16(2, 8, 32, true) SY_KS16(2, 16, 32, true)
#undef SY_KS16
  SY_CHECK(k != nullptr, SY_EINVAL, "no 16x16 in-workgroup split-K kernel for mode %d tile %d", mode, t);
  hipLaunchKernelGGL(k, grid, dim3((4 << (t - kKs16Base)) * 64), 0, ctx->stream, a);
  return SY_OK;
}

static int launch_igemm(sy_ctx* ctx, const IgemmArgs& a, int batch, bool wino, double flops, double bytes,
                        const char* name = nullptr) {
  const bool rows = a.KH == 1 && a.KW == 1 && a.SH == 1 && a.SW == 1 && a.PH == 0 && a.PW == 0 && a.OH == a.H &&
                    a.OW == a.W;
  const int ft = ctx->force_tile >= 0 ? ctx->force_tile : env_tile();
  if (ft == kC16Tile && batch == 1 && !name && !wino && c16_ok(a)) {
    const char* pn = a.SH == 1 ? (a.OC == 16 ? "conv3x3_c16_oc16_s1" : "conv3x3_c16_oc32_s1")
                               : (a.OC == 16 ? "conv3x3_c16_oc16_s2" : "conv3x3_c16_oc32_s2");
    ProfScope prof(ctx, pn, flops, bytes);
    SY_TRY(launch_c16(ctx, a));
    return check_launch(pn);
  }
  if (is_x3_tile(ft) && batch == 1 && !name && !wino) {
    const int mode = rows ? (a.ku > 0 ? 3 : 2) : (a.IC % 32 == 0 && (long long)a.H * a.W * a.ldx < (1LL << 31) ? 1 : 0);
    SY_CHECK(a.ku == 0 || (rows && a.ku % 32 == 0), SY_EINVAL,
             "an upsampled input part needs a plain 1x1 GEMM whose K tile divides it");
    const char* pn = x3_name(ft, mode);
    ProfScope prof(ctx, pn, flops, bytes);
    SY_TRY(launch_x3(ctx, ft, mode, a));
    return check_launch(pn);
  }
  if (is_ks_tile(ft) && batch == 1 && !name && !wino && a.ku == 0) {
    int bk = 0;
    const int mode = ks_mode(a, rows, &bk);
    if (mode > 0) {
      const char* pn = ks_name(ft, mode, bk);
      ProfScope prof(ctx, pn, flops, bytes);
      SY_TRY(launch_ks(ctx, ft, mode, bk, a));
      return check_launch(pn);
    }
  }
  if (is_ks16_tile(ft) && batch == 1 && !name && !wino && a.ku == 0) {
    int bk = 0;
    const int mode = ks_mode(a, rows, &bk);
    if (mode > 0) {
      const char* pn = ks16_name(ft, mode, bk);
      ProfScope prof(ctx, pn, flops, bytes);
      SY_TRY(launch_ks16(ctx, ft, mode, bk, a));
      return check_launch(pn);
    }
  }
  if (name && batch == 1 && !wino && a.ku == 0 && a.shuf == 0 && ft < 0 && rows && a.K >= 128) {
    // Named row GEMMs (the attention products) are not tuned: at batch 1 a
    // deep-K product whose tiled grid would leave most CUs idle runs on the
    // 16x16 in-workgroup split-K kernel, its waves sized to the K chunks.
    const TileCfg& c = kTiles[pick_tile(ctx, a.M, a.OC, 1)];
    const long long grid = (long long)((a.M + c.bm - 1) / c.bm) * ((a.OC + c.bn - 1) / c.bn);
    IgemmArgs b = a;
    b.xb = b.wb = b.yb = 0;
    int bk = 0;
    if (4 * grid < (ctx->cu_count > 0 ? ctx->cu_count : 256) && ks_mode(b, rows, &bk) == 2) {
      const int nch = (a.K + 31) / 32;
      const int t = kKs16Base + (nch >= 64 ? 2 : nch >= 24 ? 1 : 0);  // 16, 8 or 4 waves
      ProfScope prof(ctx, name, flops, bytes);
      SY_TRY(launch_ks16(ctx, t, 2, bk, b));
      return check_launch(name);
    }
  }
  if (a.ku == 0 && pw_ok(ft, a, rows)) {
    const char* pn = name ? name : tile_name(ft, wino, 2);
    ProfScope prof(ctx, pn, flops, bytes);
    switch (ft - kPwBase) {
      case 0: SY_TRY(launch_pw<1>(ctx, a, batch)); break;
      case 1: SY_TRY(launch_pw<2>(ctx, a, batch)); break;
      case 2: SY_TRY(launch_pw<3>(ctx, a, batch)); break;
      default: SY_TRY(launch_pw<4>(ctx, a, batch)); break;
    }
    return check_launch(pn);
  }
  int t = gemm_tile_ok(ctx->force_tile, rows) ? ctx->force_tile : pick_tile(ctx, a.M, a.OC, batch);
  if (!gemm_tile_ok(t, rows)) t = 2;
  const int kind = name ? 2 : (wino ? 1 : 0);
  const int want = ctx->force_split > 1 ? ctx->force_split : env_split();
  const bool split = want > 1 && kind == 0 && batch == 1 && a.shuf == 0;
  const TileCfg& c = kTiles[t];
  dim3 grid((a.M + c.bm - 1) / c.bm, (a.OC + c.bn - 1) / c.bn, batch);
  const bool fits32 = (long long)a.H * a.W * a.ldx < (1LL << 31);
  const int mode = rows ? (a.ku > 0 ? 3 : 2) : (a.IC % c.bk == 0 && fits32 ? 1 : 0);
  SY_CHECK(a.ku == 0 || (rows && kind == 0 && a.ku % c.bk == 0), SY_EINVAL,
           "an upsampled input part needs a plain 1x1 GEMM whose K tile divides it");
  if (split) {
    int kchunk = 0, S = 1;
    split_chunks(a.K, c.bk, want, &kchunk, &S);
    const int ldp = grid.y * c.bn;
    SY_CHECK((long long)S * a.M * ldp <= kSplitMaxFloats, SY_EUNSUPPORTED,
             "split-K partials of %lld floats exceed the %lld limit", (long long)S * a.M * ldp, kSplitMaxFloats);
    SY_TRY(ensure_scratch(ctx, (size_t)S * a.M * ldp * sizeof(float)));
    IgemmArgs b = a;
    b.part = (float*)ctx->scratch;
    b.kchunk = kchunk;
    b.ldp = ldp;
    b.xb = b.wb = b.yb = 0;
    grid.z = S;
    char pn[80];
    snprintf(pn, sizeof pn, "%s_sk%d", tile_name(t, false, mode), want);
    {
      ProfScope prof(ctx, pn, flops, bytes);
      if (mode == 3) launch_tile<0, 3>(t, grid, ctx->stream, b);
      else if (mode == 2) launch_tile<0, 2>(t, grid, ctx->stream, b);
      else if (mode == 1) launch_tile<0, 1>(t, grid, ctx->stream, b);
      else launch_tile<0, 0>(t, grid, ctx->stream, b);
      SY_TRY(check_launch(pn));
    }
    const long long outs = (long long)a.M * a.OC;
    ProfScope prof(ctx, "splitk_reduce", 0,
                   4.0 * ((double)S * a.M * a.OC + (double)outs * (a.res ? 2 : 1)));
    hipLaunchKernelGGL(splitk_reduce_kernel, dim3((unsigned)((outs + 255) / 256)), dim3(256), 0, ctx->stream,
                       b.part, S, a.M, ldp, a.OC, a.bias, a.silu, a.res, a.ldr, a.y, a.ldy);
    return check_launch("splitk_reduce");
  }
  ProfScope prof(ctx, name ? name : tile_name(t, wino, mode), flops, bytes);
  if (kind == 1) {
    SY_CHECK(mode == 2, SY_EINVAL, "Winograd plane GEMM needs row addressing");
    launch_tile<1, 2>(t, grid, ctx->stream, a);
  } else if (kind == 2) {
    SY_CHECK(mode == 2, SY_EINVAL, "GEMM needs row addressing");
    launch_tile<2, 2>(t, grid, ctx->stream, a);
  } else if (mode == 3) {
    launch_tile<0, 3>(t, grid, ctx->stream, a);
  } else if (mode == 2) {
    launch_tile<0, 2>(t, grid, ctx->stream, a);
  } else if (mode == 1) {
    launch_tile<0, 1>(t, grid, ctx->stream, a);
  } else {
    launch_tile<0, 0>(t, grid, ctx->stream, a);
  }
  return check_launch(name ? name : tile_name(t, wino, mode));
}

// C[m][n] = sum_k A[m][k] * B[n][k] (+ C's batch strides) on the same MFMA
// kernel: A rows are 1x1 "pixels", B rows are bounds-checked against N and K.
int gemm_nt(sy_ctx* ctx, const float* A, int M, int K, int lda, const float* B, int N, int ldb, float* C, int ldc,
            const char* name, int batch, long long a_stride, long long b_stride, long long c_stride) {
  SY_CHECK(((uintptr_t)A & 15) == 0 && ((uintptr_t)B & 15) == 0 && lda % 4 == 0 && ldb % 4 == 0 && K % 4 == 0 &&
               a_stride % 4 == 0 && b_stride % 4 == 0,
           SY_EINVAL, "GEMM operands must be 16-byte aligned with K, lda, ldb multiples of 4");
  IgemmArgs a;
  a.x = A; a.N = 1; a.H = 1; a.W = M; a.IC = K; a.ldx = lda;
  a.w = B; a.Kp = ldb; a.bias = nullptr; a.res = nullptr; a.ldr = 0;
  a.y = C; a.OH = 1; a.OW = M; a.OC = N; a.ldy = ldc;
  a.KH = a.KW = a.SH = a.SW = 1; a.PH = a.PW = 0; a.DH = a.DW = 1;
  a.K = K; a.M = M; a.silu = 0;
  a.xb = a_stride; a.wb = b_stride; a.yb = c_stride;
  a.Nb = N; a.bguard = 1;
  return launch_igemm(ctx, a, batch, false, 2.0 * batch * M * N * K,
                      4.0 * batch * ((double)M * K + (double)N * K + (double)M * N), name);
}

// ------------------------------------------------------------ Winograd F(4,3)

// Input transform V = B^T d B on the 6x6 patch at (4ty-1, 4tx-1), zero
// outside the image.  One thread per (tile, VEC channels): consecutive threads
// take consecutive channel groups, so the loads and stores of a wave are
// contiguous runs.  VEC trades load-instruction count against the registers
// the 36-value patch needs (and so occupancy); 4 measures fastest on the
// YOLO shapes although it leaves 2 waves per SIMD.  V layout [36][tiles][ic].
typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int VEC> struct VecT;
template <> struct VecT<1> { typedef float T; };
template <> struct VecT<2> { typedef f32x2 T; };
template <> struct VecT<4> { typedef f32x4 T; };

// One column (or row) of the input transform B^T d, the rows of
// F(4x4, 3x3)'s B^T as in CpuWinograd4.cs:36, with the shared sums formed
// once: 14 operations per six values instead of the 24 the rows spell out.
template <class T>
__device__ __forceinline__ void winograd_bt6(const T (&d)[6], T (&o)[6]) {
  const T s12 = d[1] + d[2], s34 = d[3] + d[4];
  const T m12 = d[1] - d[2], m43 = d[4] - d[3];
  const T a = d[4] - d[2], b = d[3] - d[1];
  o[0] = 4.f * d[0] + (d[4] - 5.f * d[2]);
  o[1] = s34 - 4.f * s12;
  o[2] = m43 + 4.f * m12;
  o[3] = a + 2.f * b;
  o[4] = a - 2.f * b;
  o[5] = 4.f * d[1] + (d[5] - 5.f * d[3]);
}

template <int VEC>
__global__ __launch_bounds__(256) void wino_in_kernel(const float* __restrict__ x, int N, int H, int W, int IC,
                                                      int ldx, int TH, int TW, float* __restrict__ V,
                                                      long long plane) {
  typedef typename VecT<VEC>::T vec;
  const int CG = IC / VEC;
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long total = (long long)N * TH * TW * CG;
  if (gid >= total) return;
  // Index decode in 32 bits when the grid allows (every YOLO shape): 64-bit
  // division and remainder are long instruction sequences per thread.
  int c, tx, ty, n;
  long long t;
  if (total < (1LL << 31)) {
    const unsigned g = (unsigned)gid, cg = (unsigned)CG, tw = (unsigned)TW, th = (unsigned)TH;
    const unsigned tt = g / cg, q = tt / tw;
    c = VEC * (int)(g - tt * cg);
    tx = (int)(tt - q * tw);
    ty = (int)(q % th);
    n = (int)(q / th);
    t = tt;
  } else {
    c = VEC * (int)(gid % CG);
    t = gid / CG;
    tx = (int)(t % TW);
    const long long r = t / TW;
    ty = (int)(r % TH);
    n = (int)(r / TH);
  }
  const float* base = x + (long long)n * H * W * ldx + c;
  const int y0 = ty * 4 - 1, x0 = tx * 4 - 1;
  // All 36 loads are issued before the first use (one HBM round trip, not six).
  vec ld[6][6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const int cx = min(max(x0 + j, 0), W - 1);
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int cy = min(max(y0 + i, 0), H - 1);
      ld[i][j] = *(const vec*)(base + ((long long)cy * W + cx) * ldx);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  vec t1[6][6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    vec d[6];
    const int ix = x0 + j;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int iy = y0 + i;
      d[i] = ((unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W) ? ld[i][j] : vec(0.f);
    }
    vec col[6];
    winograd_bt6(d, col);
#pragma unroll
    for (int i = 0; i < 6; ++i) t1[i][j] = col[i];
  }
  float* out = V + t * IC + c;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    vec v[6];
    winograd_bt6(t1[i], v);
#pragma unroll
    for (int j = 0; j < 6; ++j) *(vec*)(out + (long long)(i * 6 + j) * plane) = v[j];
  }
}

// Input transform into the MFMA-blocked V of wino_go_kernel,
// V[p][tile / 32][k / 8][lane][4] with lane = 32 * ((k / 4) % 2) + tile % 32
// (one float4 per lane is a whole 32-tile x 8-channel A fragment).  A
// workgroup covers one 32-tile block and 32 channels (four fragments).  The
// loads run along the channels: lane l of wave w takes tile 8w + l / 8 and
// channels 4 * (l % 8) .. + 3, so eight lanes read 128 contiguous bytes of a
// pixel (a lane order equal to the fragment's would make every 16-byte load
// its own L1 access).  Each lane transforms its own 6x6 x 4-channel patch in
// registers; the results are regrouped into fragments through LDS, six
// planes at a time, and each wave stores one fragment per plane as a
// contiguous 1 KiB write.
constexpr int kInTilePad = 9;  // float4s per tile row in the exchange (8 + 1: conflict-free reads)

__global__ __launch_bounds__(256) void wino_in_blk_kernel(const float* __restrict__ x, int H, int W, int IC,
                                                          int ldx, int TH, int TW, long long tiles,
                                                          float* __restrict__ V, long long plane) {
  __shared__ f32x4 S[2][6][32 * kInTilePad];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nkc = IC >> 3, nkg = (nkc + 3) >> 2;
  const long long tb = blockIdx.x / nkg;
  const int g = (int)(blockIdx.x - tb * nkg);
  // Phase 1: this lane's tile and channel group (clamped into range; lanes
  // past the end compute values nobody stores).
  const int ti = 8 * wave + (lane >> 3), c4 = lane & 7;
  const long long t = min(tb * 32 + ti, tiles - 1);
  const int c = min(g * 32 + 4 * c4, IC - 4);
  const int tx = (int)(t % TW);
  const long long r = t / TW;
  const int ty = (int)(r % TH);
  const int n = (int)(r / TH);
  const float* base = x + (long long)n * H * W * ldx + c;
  const int y0 = ty * 4 - 1, x0 = tx * 4 - 1;
  // All 36 patch loads are issued before the first use, each at a row
  // offset plus a column offset (clamped into the image).
  long long ro[6], co[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    ro[i] = (long long)min(max(y0 + i, 0), H - 1) * W * ldx;
    co[i] = (long long)min(max(x0 + i, 0), W - 1) * ldx;
  }
  f32x4 ld[6][6];
#pragma unroll
  for (int j = 0; j < 6; ++j)
#pragma unroll
    for (int i = 0; i < 6; ++i) ld[i][j] = *(const f32x4*)(base + (ro[i] + co[j]));
  __builtin_amdgcn_sched_barrier(0);
  f32x4 t1[6][6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    f32x4 d[6];
    const int ix = x0 + j;
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int iy = y0 + i;
      d[i] = ((unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W) ? ld[i][j] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    f32x4 col[6];
    winograd_bt6(d, col);
#pragma unroll
    for (int i = 0; i < 6; ++i) t1[i][j] = col[i];
  }
  // Phase 2: regroup.  Wave w stores fragment kc = 4g + w; its lane L holds
  // tile L % 32 and channels 4 * (L / 32) .. + 3 of that fragment, i.e.
  // channel group c4 = 2w + L / 32 of the workgroup.
  const int kc = g * 4 + wave;
  const int rt = lane & 31, rc = 2 * wave + (lane >> 5);
  float* out = V + (tb * nkc + kc) * 256 + lane * 4;
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    f32x4 v[6];
    winograd_bt6(t1[i], v);
    f32x4(*B)[32 * kInTilePad] = S[i & 1];
#pragma unroll
    for (int j = 0; j < 6; ++j) B[j][ti * kInTilePad + c4] = v[j];
    // One barrier per plane row: the double buffer keeps the next row's
    // writes off the buffer this row is still being read from.
    __syncthreads();
    if (kc < nkc) {
#pragma unroll
      for (int j = 0; j < 6; ++j) *(f32x4*)(out + (long long)(i * 6 + j) * plane) = B[j][rt * kInTilePad + rc];
    }
  }
}

// One column (or row) of the output transform A^T m, the rows of
// F(4x4, 3x3)'s A^T as in CpuWinograd4.cs:36, with the shared sums formed
// once (10 operations per four outputs).
__device__ __forceinline__ void winograd_at6(const float (&m)[6], float (&u)[4]) {
  const float a = m[1] + m[2], b = m[1] - m[2], c = m[3] + m[4], d = m[3] - m[4];
  u[0] = m[0] + a + c;
  u[1] = b + 2.f * d;
  u[2] = a + 4.f * c;
  u[3] = b + 8.f * d + m[5];
}

// Inverse transform Y = A^T M A + bias, SiLU, residual; 4x4 outputs per tile,
// clipped at the right/bottom edge.  One thread per (tile, channel), channels
// fastest, for the same coalescing and occupancy reasons as the input pass.
__global__ __launch_bounds__(256) void wino_out_kernel(const float* __restrict__ Mt, long long plane, int ldm,
                                                       int N, int TH, int TW, int OH, int OW, int OC,
                                                       const float* __restrict__ bias, int silu,
                                                       const float* __restrict__ res, int ldr,
                                                       float* __restrict__ y, int ldy) {
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long total = (long long)N * TH * TW * OC;
  if (gid >= total) return;
  // Index decode in 32 bits when the grid allows (as in wino_in_kernel).
  int c, tx, ty, n;
  long long t;
  if (total < (1LL << 31)) {
    const unsigned g = (unsigned)gid, oc = (unsigned)OC, tw = (unsigned)TW, th = (unsigned)TH;
    const unsigned tt = g / oc, q = tt / tw;
    c = (int)(g - tt * oc);
    tx = (int)(tt - q * tw);
    ty = (int)(q % th);
    n = (int)(q / th);
    t = tt;
  } else {
    c = (int)(gid % OC);
    t = gid / OC;
    tx = (int)(t % TW);
    const long long r = t / TW;
    ty = (int)(r % TH);
    n = (int)(r / TH);
  }
  const float* src = Mt + t * ldm + c;
  // All 36 loads are issued before the first use (one HBM round trip, not six).
  float ld[36];
#pragma unroll
  for (int p = 0; p < 36; ++p) ld[p] = src[(long long)p * plane];
  __builtin_amdgcn_sched_barrier(0);
  float u[4][6];
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    float m[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) m[i] = ld[i * 6 + j];
    float col[4];
    winograd_at6(m, col);
#pragma unroll
    for (int i = 0; i < 4; ++i) u[i][j] = col[i];
  }
  const float b = bias ? bias[c] : 0.f;
  float o[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    winograd_at6(u[i], o[i]);
#pragma unroll
    for (int j = 0; j < 4; ++j) o[i][j] += b;
    if (silu) {
#pragma unroll
      for (int j = 0; j < 4; ++j) o[i][j] = silu_fast(o[i][j]);
    }
  }
  // One 64-bit base per tile; interior tiles store without per-pixel tests.
  const int oy0 = ty * 4, ox0 = tx * 4;
  const long long pix0 = ((long long)n * OH + oy0) * OW + ox0;
  float* yp = y + pix0 * ldy + c;
  const float* rp = res ? res + pix0 * ldr + c : nullptr;
  const int ystep = OW * ldy, rstep = OW * ldr;
  if (oy0 + 4 <= OH && ox0 + 4 <= OW) {
    if (rp) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) o[i][j] = rp[i * rstep + j * ldr] + o[i][j];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) yp[i * ystep + j * ldy] = o[i][j];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (oy0 + i < OH && ox0 + j < OW) {
          float v = o[i][j];
          if (rp) v = rp[i * rstep + j * ldr] + v;
          yp[i * ystep + j * ldy] = v;
        }
      }
  }
}

// ------------------------------------------------------------ Winograd, GEMM + inverse

// The 36 plane GEMMs M[p] = V[p] U[p]^T fused with the inverse transform, so
// the transformed output M never goes to HBM.  A workgroup owns 32 tiles x 32
// output channels; each of four waves accumulates nine planes (nine 32x32
// MFMA accumulators).  V and U are stored in MFMA-operand blocks (one float4 per
// lane is a whole 32 x 8 fragment, contiguous), so the K loop has no LDS, no
// barrier and fully coalesced 1 KiB loads; fragments are loaded eight planes
// (32 MFMAs, about 2000 cycles) ahead of their use, which covers a read of V
// from HBM with one wave per SIMD.  The epilogue exchanges the accumulators through LDS,
// half the tiles at a time to keep the LDS small, and applies Y = A^T M A, bias, SiLU and the
// residual.  Workgroups are ordered so that the channel blocks of one tile
// block run on the same XCD (workgroup i runs on XCD i % 8) and read V from
// its L2.
struct WinoGoArgs {
  const float* V;  // [36][ntb][nkc][64][4]
  const float* U;  // [36][nob][nkc][64][4]
  const float* bias;
  const float* res;
  int ldr;
  float* y;
  int ldy, OC;
  int TH, TW, OH, OW;
  long long tiles;
  int ntb, nob, nkc, silu;
  // wino_fx_kernel only: the NHWC input it transforms.
  const float* x;
  int H, W, IC, ldx;
};

// Accumulator exchange: a pass moves 16 of the 32 tiles as 8 pairs.  LDS row
// (plane p, pair k) holds 64 floats, the 32 channels of tile 8*(k/4) + (k%4)
// and then those of tile 8*(k/4) + 4 + (k%4) (the two lane halves of one
// accumulator register), so every exchange access of a wave is 256
// contiguous bytes.
constexpr int kGoPairs = 8;

constexpr int kGoWaves = 4, kGoPlanes = 36 / kGoWaves;
constexpr int kGoRing = 9;  // fragment ring slots (divides kGoPlanes)
// Wave layouts: NW = 4, the four MFMA waves alone (two workgroups per CU:
// one's epilogue overlaps the other's K loop); NW = 8, four more waves that
// skip the K loop and share the inverse transform (for grids that leave one
// workgroup per CU, where nothing else would overlap the epilogue).  Both
// sum in the same order and give the same bits.
constexpr int kGoVariants = 2;

template <int NW>
__device__ __forceinline__ void wino_go_epilogue(const WinoGoArgs& a, float* E, const f32x16 (&acc)[kGoPlanes],
                                                 int tb, int ob, int wave, int lane, bool mfma_wave, int p0,
                                                 float bias);

template <int NW>
__global__ __launch_bounds__(64 * NW, NW == kGoWaves ? 2 : 1) void wino_go_kernel(const WinoGoArgs a) {
  __shared__ float E[36 * kGoPairs * 64];  // [plane][pair][2 tiles x 32 channels]
  // The wave index is made explicitly uniform so that every fragment address
  // is a scalar base plus one per-lane offset: 64-bit per-lane pointers for
  // the 18 streams would take the registers the load ring needs.
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = gridDim.x, L = blockIdx.x;
  const int xcd = L & 7, kk = L >> 3;
  const int q8 = G >> 3, rem = G & 7;
  const int P = xcd * q8 + (xcd < rem ? xcd : rem) + kk;
  const int tb = P / a.nob, ob = P - (P / a.nob) * a.nob;
  const long long vps = (long long)a.ntb * a.nkc * 256, ups = (long long)a.nob * a.nkc * 256;
  const bool mfma_wave = wave < kGoWaves;
  const int p0 = kGoPlanes * (mfma_wave ? wave : 0);
  const float* vp = a.V + ((long long)p0 * a.ntb + tb) * a.nkc * 256;
  const float* up = a.U + ((long long)p0 * a.nob + ob) * a.nkc * 256;
  const int lo = lane * 4;
  // The epilogue's bias, loaded before any store is issued.
  const float bias = (ob * 32 + (lane & 31) < a.OC) ? a.bias[ob * 32 + (lane & 31)] : 0.f;

  f32x16 acc[kGoPlanes];
#pragma unroll
  for (int q = 0; q < kGoPlanes; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
  if (mfma_wave) {
    // Fragments stream through a ring of kGoRing slots: while plane q of chunk
    // kc is multiplied, plane q + kGoRing - 1 (of this chunk, or of the next)
    // is loaded.
    static_assert(kGoPlanes % kGoRing == 0, "ring slots must divide the planes per wave");
    constexpr int kGoAhead = kGoRing - 1;
    f32x4 av[kGoRing], bv[kGoRing];
    // Issued in plane order (pinned by the scheduling barriers): the loop's
    // wait before plane q counts the loads issued after plane q's, and one
    // wait count serves every iteration, the first included.
#pragma unroll
    for (int q = 0; q < kGoAhead; ++q) {
      av[q] = *(const f32x4*)(vp + q * vps + lo);
      bv[q] = *(const f32x4*)(up + q * ups + lo);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int kc = 0; kc < a.nkc; ++kc) {
      const long long cur = (long long)kc * 256;
#pragma unroll
      for (int q = 0; q < kGoPlanes; ++q) {
        const int ld = q + kGoAhead;  // plane index of the load issued now
        if (ld < kGoPlanes) {
          av[ld % kGoRing] = *(const f32x4*)(vp + (ld * vps + cur) + lo);
          bv[ld % kGoRing] = *(const f32x4*)(up + (ld * ups + cur) + lo);
        } else {
          // The last chunk reloads its own fragments (never used): with no
          // branch around the loads, each plane waits for its own loads only,
          // not for every load in flight.
          const long long nxt = kc + 1 < a.nkc ? cur + 256 : cur;
          av[ld % kGoRing] = *(const f32x4*)(vp + ((ld - kGoPlanes) * vps + nxt) + lo);
          bv[ld % kGoRing] = *(const f32x4*)(up + ((ld - kGoPlanes) * ups + nxt) + lo);
        }
        // Keep the loads just issued ahead of this plane's MFMAs: left alone,
        // the scheduler sinks each load next to its use and every plane then
        // waits for all outstanding loads.
        __builtin_amdgcn_sched_barrier(0);
        const f32x4 x0 = av[q % kGoRing], w0 = bv[q % kGoRing];
        // Lane half h holds k = 4h + s at step s, for A and B alike.
#pragma unroll
        for (int st = 0; st < 4; ++st) acc[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(x0[st], w0[st], acc[q], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }

  wino_go_epilogue<NW>(a, E, acc, tb, ob, wave, lane, mfma_wave, p0, bias);
}

// Epilogue of the plane GEMM: the accumulators of waves 0-3 (nine planes
// each, 32 tiles x 32 channels) go through the LDS exchange E, and waves
// 0..NW-1 apply Y = A^T M A, bias, SiLU and the residual.  D layout: lane
// holds channel (lane & 31) of tiles 8*(r/4) + 4*(lane/32) + (r%4), so
// registers 8*hp .. 8*hp + 7 hold tiles 16*hp .. 16*hp + 15 and register
// 8*hp + k is pair k of pass hp.  The caller has passed a barrier after its
// last read of E's memory.
// On this GPU a wait for a load also waits for every store issued before
// it, so the epilogue issues no load after a store of the same pass: the
// bias was loaded before the K loop, and each pass loads all of its
// residual values before its first store.
template <int NW>
__device__ __forceinline__ void wino_go_epilogue(const WinoGoArgs& a, float* E, const f32x16 (&acc)[kGoPlanes],
                                                 int tb, int ob, int wave, int lane, bool mfma_wave, int p0,
                                                 float bias) {
  const int r32 = lane & 31, h = lane >> 5;
  const int tiles_per_img = a.TH * a.TW;
  const int oc = ob * 32 + r32;
  const bool oc_ok = oc < a.OC;
  constexpr int kPairsPerWave = (kGoPairs + NW - 1) / NW;
#pragma unroll
  for (int hp = 0; hp < 2; ++hp) {
    if (hp) __syncthreads();  // the first pass's reads are done
    if (mfma_wave) {
#pragma unroll
      for (int q = 0; q < kGoPlanes; ++q)
#pragma unroll
        for (int k = 0; k < kGoPairs; ++k) E[((p0 + q) * kGoPairs + k) * 64 + lane] = acc[q][8 * hp + k];
    }
    __syncthreads();
    // Wave w applies the inverse to pairs w, w + NW, ...: lane half h takes
    // the pair's second tile, lane r32 channel r32.  Tile indices fit 32
    // bits (the host caps the tile count at 2^30).
    bool ok[kPairsPerWave], inner[kPairsPerWave];
    long long pix[kPairsPerWave];
    int oy0[kPairsPerWave], ox0[kPairsPerWave];
    float rv[kPairsPerWave][16];
#pragma unroll
    for (int kk = 0; kk < kPairsPerWave; ++kk) {
      const int k = wave + NW * kk;
      const int tile = tb * 32 + 16 * hp + 8 * (k >> 2) + 4 * h + (k & 3);
      ok[kk] = k < kGoPairs && tile < a.tiles && oc_ok;
      const int n = tile / tiles_per_img;
      const int trem = tile - n * tiles_per_img;
      const int ty = trem / a.TW, tx = trem - (trem / a.TW) * a.TW;
      oy0[kk] = ty * 4;
      ox0[kk] = tx * 4;
      inner[kk] = oy0[kk] + 4 <= a.OH && ox0[kk] + 4 <= a.OW;
      pix[kk] = ((long long)n * a.OH + oy0[kk]) * a.OW + ox0[kk];
      if (a.res && ok[kk]) {
        const float* rp = a.res + pix[kk] * a.ldr + oc;
        const int rstep = a.OW * a.ldr;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
            rv[kk][i * 4 + jj] = (inner[kk] || (oy0[kk] + i < a.OH && ox0[kk] + jj < a.OW))
                                     ? rp[i * rstep + jj * a.ldr] : 0.f;
      }
    }
#pragma unroll
    for (int kk = 0; kk < kPairsPerWave; ++kk) {
      if (!ok[kk]) continue;
      const int k = wave + NW * kk;
      const float* e = E + k * 64 + lane;
      float u[4][6];
#pragma unroll
      for (int jj = 0; jj < 6; ++jj) {
        float m[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) m[i] = e[(i * 6 + jj) * kGoPairs * 64];
        float col[4];
        winograd_at6(m, col);
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i][jj] = col[i];
      }
      const float b = bias;
      float o[4][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        winograd_at6(u[i], o[i]);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) o[i][jj] += b;
        if (a.silu) {
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) o[i][jj] = silu_fast(o[i][jj]);
        }
      }
      if (a.res) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) o[i][jj] = rv[kk][i * 4 + jj] + o[i][jj];
      }
      // One 64-bit base per tile, 32-bit offsets within it; interior tiles
      // (all 16 pixels inside the image) store without per-pixel tests.
      float* yp = a.y + pix[kk] * a.ldy + oc;
      const int ystep = a.OW * a.ldy;
      if (inner[kk]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) yp[i * ystep + jj * a.ldy] = o[i][jj];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj)
            if (oy0[kk] + i < a.OH && ox0[kk] + jj < a.OW) yp[i * ystep + jj * a.ldy] = o[i][jj];
      }
    }
  }
}

// ------------------------------------------------------------ fused Winograd

// The plane GEMM and inverse of wino_go_kernel with the input transform
// inside, so V never goes to HBM.  A workgroup owns 32 tiles x 32 output
// channels; wave w accumulates planes 9w .. 9w + 8 over 8-channel K chunks,
// reading its A fragments from an LDS double buffer that the same 256
// threads fill one chunk ahead: thread t transforms tile t / 8, channel
// t % 8 of the next chunk (36 patch loads, eight lanes reading a pixel's 32
// contiguous bytes, issued before the current chunk's MFMAs and used after
// them), V = B^T d B in registers, then 36 LDS stores in fragment order.  B
// fragments stream from L2 through the same ring as in wino_go_kernel.  Two
// workgroups per CU, so one's transform runs beside the other's MFMAs.  The
// transform, the fragment order, the summation order and the epilogue are
// those of wino_in_blk_kernel + wino_go_kernel: both forms give the same
// bits.  Input channels past IC (IC % 8 != 0) read as zero.
constexpr int kFxBuf = 36 * 256;  // floats of one chunk's A fragments [plane][64 lanes][4]
constexpr int kFxOob = 0x40000000;  // buffer offset past every record: the load returns zero
constexpr int kBufferWord3 = 0x00020000;  // raw buffer resource, word 3 (gfx9 family)

// Float offset of fragment lane L within a plane: lanes 32..63 are kept
// with tile bits 2 and 3 flipped, so that the transform's stores (eight
// lanes per tile, channels 0..7) fall in distinct banks whether a store is
// served 64 lanes over 64 banks or 32 lanes over 32 banks at a time; the
// MFMA reads stay one 16-byte slot per lane over a contiguous 1 KiB.
__device__ __forceinline__ int fx_slot(int L) { return L < 32 ? 4 * L : 128 + 4 * ((L - 32) ^ 12); }

template <int RING, int GR>
__global__ __launch_bounds__(256 * GR, GR == 1 ? 2 : 1) void wino_fx_kernel(const WinoGoArgs a) {
  constexpr int kE = 36 * kGoPairs * 64;  // floats of one exchange
  // GR = 1: two chunks of fragments, then the exchange.  GR = 2: two phases
  // of two chunks, then one exchange per group.
  __shared__ __attribute__((aligned(16))) float S[GR * kE];
  static_assert(2 * kFxBuf <= kE, "the fragment double buffer fits the exchange");
  static_assert(GR == 1 || GR == 2, "one or two groups of four waves");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2, wq = wave & 3;  // group, wave within the group
  const int G = gridDim.x, L = blockIdx.x;
  const int xcd = L & 7, kx = L >> 3;
  const int q8 = G >> 3, rem = G & 7;
  const int P = xcd * q8 + (xcd < rem ? xcd : rem) + kx;
  const int nobk = (a.nob + GR - 1) / GR;  // workgroups per tile block
  const int tb = P / nobk;
  // Group g multiplies output block GR * (P % nobk) + g; a block past the
  // last one (odd block count) reads the last block's fragments and stores
  // nothing (its channels fail the epilogue's channel test).
  const int ob = (P - tb * nobk) * GR + grp, obc = min(ob, a.nob - 1);
  const long long ups = (long long)a.nob * a.nkc * 256;
  const int p0 = kGoPlanes * wq;
  const float* up = a.U + ((long long)p0 * a.nob + obc) * a.nkc * 256 + lane * 4;
  const float bias = (ob * 32 + (lane & 31) < a.OC) ? a.bias[ob * 32 + (lane & 31)] : 0.f;

  // This thread's transform unit: tile tt of the block, channel cu of each
  // chunk.  The patch is read through a buffer resource based at the image
  // of the block's first tile, so per-lane byte offsets stay within 32 bits
  // (the host caps the span of a block's images): a row or column outside
  // the image, or a tile past the end, takes offset kFxOob and reads as zero
  // (two such offsets sum to 2^31, no wrap), and the chunk's channel offset
  // is the scalar soffset.  No select, clamp or 64-bit address per load.
  const int tt = (tid & 255) >> 3, cu = tid & 7;
  const bool tok = (long long)tb * 32 + tt < a.tiles;
  const int tile = tok ? tb * 32 + tt : (int)(a.tiles - 1);
  const int tiles_per_img = a.TH * a.TW;
  const int n0 = (tb * 32) / tiles_per_img;
  const int n = tile / tiles_per_img, trem = tile - n * tiles_per_img;
  const int ty = trem / a.TW, tx = trem - (trem / a.TW) * a.TW;
  const long long img = (long long)a.H * a.W * a.ldx;
  const long long span = 4 * ((a.tiles / tiles_per_img - n0) * img - a.ldx + a.IC);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + n0 * img), (short)0, (int)min(span, (long long)kFxOob), kBufferWord3);
  int ro[6], co[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const int iy = 4 * ty - 1 + i, ix = 4 * tx - 1 + i;
    ro[i] = tok && (unsigned)iy < (unsigned)a.H ? 4 * ((n - n0) * (int)img + iy * a.W * a.ldx) : kFxOob;
    co[i] = (unsigned)ix < (unsigned)a.W ? 4 * (ix * a.ldx + cu) : kFxOob;
  }
  const int wslot = (cu < 4 ? 4 * tt : 128 + 4 * (tt ^ 12)) + (cu & 3);
  const int rslot = fx_slot(lane);

  float d[36];
  // Each row offset passes through an empty asm per chunk: hoisted out of the
  // loop, the 36 sums would hold 36 registers through the MFMAs.
  auto load_x = [&](int kc) {
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      int r = ro[i];
      asm volatile("" : "+v"(r));
#pragma unroll
      for (int j = 0; j < 6; ++j)
        d[i * 6 + j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, r + co[j], 32 * kc, 0));
    }
  };
  auto transform_store = [&](int kc, float* buf) {
    // Channels past IC (a last chunk that IC % 8 leaves partial) read other
    // data of the pixel: zero them.
    if (kc * 8 + 8 > a.IC) {
      if (kc * 8 + cu >= a.IC) {
#pragma unroll
        for (int p = 0; p < 36; ++p) d[p] = 0.f;
      }
    }
    float t1[6][6];
#pragma unroll
    for (int j = 0; j < 6; ++j) {
      float dc[6], col[6];
#pragma unroll
      for (int i = 0; i < 6; ++i) dc[i] = d[i * 6 + j];
      winograd_bt6(dc, col);
#pragma unroll
      for (int i = 0; i < 6; ++i) t1[i][j] = col[i];
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      float v[6];
      winograd_bt6(t1[i], v);
#pragma unroll
      for (int j = 0; j < 6; ++j) buf[(i * 6 + j) * 256 + wslot] = v[j];
    }
  };

  f32x16 acc[kGoPlanes];
#pragma unroll
  for (int q = 0; q < kGoPlanes; ++q)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
  static_assert(kGoPlanes % RING == 0, "ring slots must divide the planes per wave");
  constexpr int kAhead = RING - 1;
  f32x4 bv[RING];
  // One chunk of MFMAs: the A fragment of plane q + 1 is read from LDS while
  // plane q multiplies; the ring's loads run RING - 1 planes ahead across
  // chunk boundaries, as in wino_go_kernel (the last chunk reloads its own).
  // mid() issues the next chunk's patch loads right after plane 0's ring
  // load: a wait counts loads in issue order, so with a full ring (RING = 9)
  // every B fragment of this chunk is issued before them and no plane waits
  // for the patch.
  auto gemm_chunk = [&](int kc, const float* vbuf, auto&& mid) {
    const float* vb = vbuf + rslot + p0 * 256;
    const long long cur = (long long)kc * 256;
    const long long nxt = kc + 1 < a.nkc ? cur + 256 : cur;
    f32x4 av[2];
    av[0] = *(const f32x4*)vb;
#pragma unroll
    for (int q = 0; q < kGoPlanes; ++q) {
      const int ld = q + kAhead;
      if (ld < kGoPlanes)
        bv[ld % RING] = *(const f32x4*)(up + (ld * ups + cur));
      else
        bv[ld % RING] = *(const f32x4*)(up + ((ld - kGoPlanes) * ups + nxt));
      __builtin_amdgcn_sched_barrier(0);
      if (q == 0) {
        mid();
        __builtin_amdgcn_sched_barrier(0);
      }
      if (q + 1 < kGoPlanes) av[(q + 1) & 1] = *(const f32x4*)(vb + (q + 1) * 256);
      __builtin_amdgcn_sched_barrier(0);
      const f32x4 x0 = av[q & 1], w0 = bv[q % RING];
#pragma unroll
      for (int st = 0; st < 4; ++st) acc[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(x0[st], w0[st], acc[q], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Phase ph covers chunks GR ph .. GR ph + GR - 1 in buffer ph % 2; group g
  // transforms chunk GR ph + g of the next phase while both groups multiply
  // the current one (a chunk past the last reads as zero and is not
  // multiplied).
  const int nph = (a.nkc + GR - 1) / GR;
  auto vbuf = [&](int ph, int c) { return S + ((ph & 1) * GR + c) * kFxBuf; };
  load_x(grp);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int q = 0; q < kAhead; ++q) {
    bv[q] = *(const f32x4*)(up + q * ups);
    __builtin_amdgcn_sched_barrier(0);
  }
  transform_store(grp, vbuf(0, grp));
  __syncthreads();
  // A phase's MFMAs run between the loads and the transform of the next
  // phase; one barrier per phase orders both buffers (a buffer is rewritten
  // only after every wave has passed the barrier that follows its last read).
  for (int ph = 0; ph + 1 < nph; ++ph) {
    gemm_chunk(GR * ph, vbuf(ph, 0), [&] { load_x(GR * (ph + 1) + grp); });
    if (GR == 2) gemm_chunk(GR * ph + 1, vbuf(ph, 1), [] {});
    transform_store(GR * (ph + 1) + grp, vbuf(ph + 1, grp));
    __syncthreads();
  }
  gemm_chunk(GR * (nph - 1), vbuf(nph - 1, 0), [] {});
  if (GR == 2 && GR * (nph - 1) + 1 < a.nkc) gemm_chunk(GR * (nph - 1) + 1, vbuf(nph - 1, 1), [] {});
  __syncthreads();
  wino_go_epilogue<kGoWaves>(a, S + grp * kE, acc, tb, ob, wq, lane, true, p0, bias);
}

// Warp-specialized form of the fused Winograd kernel, one 512-thread
// workgroup per CU: waves 0-3 only multiply (nine planes each, as above) and
// waves 4-7 only transform, 16 input channels (two K chunks) at a time, into
// an LDS double buffer of 144 KiB.  A producer thread takes tile t / 8 and
// channels 2 (t % 8), + 1 of the 16: eight lanes read a pixel's 64
// contiguous bytes as float2, and the loads for the next 16 channels are in
// flight while the current ones are transformed.  The producers' VALU work
// runs beside the MFMA waves on the same SIMDs; one barrier per 16
// channels.  The two roles take separate code paths (with the same barrier
// sequence) so that only the MFMA waves hold accumulators; all eight waves
// share the inverse transform.  Same bits as the other Winograd forms.
constexpr int kFusedForms = 3;  // four-wave, warp-specialized, two four-wave groups over 64 output channels
constexpr int kFwSub = kFxBuf + 32;      // floats per K chunk (pad: the two chunks' stores use other banks)
constexpr int kFwBuf = 2 * kFwSub + 64;  // floats per 16-channel buffer

__global__ __launch_bounds__(512, 1) void wino_fw_kernel(const WinoGoArgs a) {
  __shared__ __attribute__((aligned(16))) float S[2 * kFwBuf];  // two 16-channel buffers, then E
  static_assert(2 * kFwBuf * 4 <= 160 * 1024 && 36 * kGoPairs * 64 <= 2 * kFwBuf, "LDS layout");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = gridDim.x, L = blockIdx.x;
  const int xcd = L & 7, kx = L >> 3;
  const int q8 = G >> 3, rem = G & 7;
  const int P = xcd * q8 + (xcd < rem ? xcd : rem) + kx;
  const int tb = P / a.nob, ob = P - (P / a.nob) * a.nob;
  const int nsc = (a.nkc + 1) >> 1;  // 16-channel steps
  const float bias = (ob * 32 + (lane & 31) < a.OC) ? a.bias[ob * 32 + (lane & 31)] : 0.f;

  if (wave < kGoWaves) {
    // ------------------------------------------------ MFMA waves
    const long long ups = (long long)a.nob * a.nkc * 256;
    const int p0 = kGoPlanes * wave;
    const float* up = a.U + ((long long)p0 * a.nob + ob) * a.nkc * 256 + lane * 4;
    const int rslot = fx_slot(lane) + p0 * 256;
    f32x16 acc[kGoPlanes];
#pragma unroll
    for (int q = 0; q < kGoPlanes; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[q][r] = 0.f;
    constexpr int kAhead = kGoRing - 1;
    f32x4 bv[kGoRing];
    auto gemm_chunk = [&](int kc, const float* vb) {
      const long long cur = (long long)kc * 256;
      const long long nxt = kc + 1 < a.nkc ? cur + 256 : cur;
      f32x4 av[2];
      av[0] = *(const f32x4*)vb;
#pragma unroll
      for (int q = 0; q < kGoPlanes; ++q) {
        const int ld = q + kAhead;
        if (ld < kGoPlanes)
          bv[ld % kGoRing] = *(const f32x4*)(up + (ld * ups + cur));
        else
          bv[ld % kGoRing] = *(const f32x4*)(up + ((ld - kGoPlanes) * ups + nxt));
        if (q + 1 < kGoPlanes) av[(q + 1) & 1] = *(const f32x4*)(vb + (q + 1) * 256);
        __builtin_amdgcn_sched_barrier(0);
        const f32x4 x0 = av[q & 1], w0 = bv[q % kGoRing];
#pragma unroll
        for (int st = 0; st < 4; ++st)
          acc[q] = __builtin_amdgcn_mfma_f32_32x32x2f32(x0[st], w0[st], acc[q], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
#pragma unroll
    for (int q = 0; q < kAhead; ++q) {
      bv[q] = *(const f32x4*)(up + q * ups);
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();  // 16 channels transformed
    for (int sc = 0; sc < nsc; ++sc) {
      const float* vb = S + (sc & 1) * kFwBuf + rslot;
      gemm_chunk(2 * sc, vb);
      if (2 * sc + 1 < a.nkc) gemm_chunk(2 * sc + 1, vb + kFwSub);
      __syncthreads();  // this buffer read; the next one written
    }
    wino_go_epilogue<2 * kGoWaves>(a, S, acc, tb, ob, wave, lane, true, p0, bias);
  } else {
    // ------------------------------------------------ transform waves
    const int pt = tid - 64 * kGoWaves;
    const int tt = pt >> 3, c2 = pt & 7;
    // Patch addressing as in wino_fx_kernel: a buffer resource at the image
    // of the block's first tile, zero-reading offsets outside the image,
    // the 16-channel step's offset in soffset.
    const bool tok = (long long)tb * 32 + tt < a.tiles;
    const int tile = tok ? tb * 32 + tt : (int)(a.tiles - 1);
    const int tiles_per_img = a.TH * a.TW;
    const int n0 = (tb * 32) / tiles_per_img;
    const int n = tile / tiles_per_img, trem = tile - n * tiles_per_img;
    const int ty = trem / a.TW, tx = trem - (trem / a.TW) * a.TW;
    const long long img = (long long)a.H * a.W * a.ldx;
    const long long span = 4 * ((a.tiles / tiles_per_img - n0) * img - a.ldx + a.IC);
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(a.x + n0 * img), (short)0, (int)min(span, (long long)kFxOob), kBufferWord3);
    int ro[6], co[6];
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      const int iy = 4 * ty - 1 + i, ix = 4 * tx - 1 + i;
      ro[i] = tok && (unsigned)iy < (unsigned)a.H ? 4 * ((n - n0) * (int)img + iy * a.W * a.ldx) : kFxOob;
      co[i] = (unsigned)ix < (unsigned)a.W ? 4 * (ix * a.ldx + 2 * c2) : kFxOob;
    }
    // Channels 2 c2, 2 c2 + 1 of the 16: K chunk c2 / 4, fragment lane half
    // (c2 / 2) % 2, elements 2 (c2 % 2) and 2 (c2 % 2) + 1.
    const int wofs = (c2 >> 2) * kFwSub + fx_slot(32 * ((c2 >> 1) & 1) + tt) + 2 * (c2 & 1);
    f32x2 d[36];
    auto load_x = [&](int sc) {
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        int r = ro[i];
        asm volatile("" : "+v"(r));
#pragma unroll
        for (int j = 0; j < 6; ++j)
          d[i * 6 + j] = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(xr, r + co[j], 64 * sc, 0));
      }
    };
    auto transform_store = [&](int sc, float* buf) {
      // Channel pairs past IC (IC % 4 == 0: both channels or neither) read
      // other data of the pixel: zero them.
      if (16 * sc + 16 > a.IC) {
        if (16 * sc + 2 * c2 >= a.IC) {
#pragma unroll
          for (int p = 0; p < 36; ++p) d[p] = f32x2{0.f, 0.f};
        }
      }
      f32x2 t1[6][6];
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        f32x2 dc[6], col[6];
#pragma unroll
        for (int i = 0; i < 6; ++i) dc[i] = d[i * 6 + j];
        winograd_bt6(dc, col);
#pragma unroll
        for (int i = 0; i < 6; ++i) t1[i][j] = col[i];
      }
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        f32x2 v[6];
        winograd_bt6(t1[i], v);
#pragma unroll
        for (int j = 0; j < 6; ++j) *(f32x2*)(buf + (i * 6 + j) * 256 + wofs) = v[j];
      }
    };
    load_x(0);
    transform_store(0, S);
    if (nsc > 1) load_x(1);
    __syncthreads();  // 16 channels transformed
    for (int sc = 0; sc < nsc; ++sc) {
      if (sc + 1 < nsc) {
        transform_store(sc + 1, S + ((sc + 1) & 1) * kFwBuf);
        if (sc + 2 < nsc) load_x(sc + 2);
      }
      __syncthreads();  // the MFMA waves are done with buffer sc & 1
    }
    f32x16 none[kGoPlanes];
#pragma unroll
    for (int q = 0; q < kGoPlanes; ++q)
#pragma unroll
      for (int r = 0; r < 16; ++r) none[q][r] = 0.f;
    wino_go_epilogue<2 * kGoWaves>(a, S, none, tb, ob, wave, lane, false, 0, bias);
  }
}

// ------------------------------------------------------------ depthwise

// Depthwise conv (groups == channels): one thread per output pixel and 4
// channels (float4 along the NHWC channel axis, so a wave reads 64 x 16
// contiguous bytes per tap), + bias, SiLU and the residual.  HBM-bound.
// vec4 = 0 falls back to one channel per thread for unaligned views.
__global__ __launch_bounds__(256) void depthwise_kernel(const float* __restrict__ x, int ldx, int N, int H, int W,
                                                        int C, const float* __restrict__ w, int ldw,
                                                        const float* __restrict__ bias, int silu,
                                                        const float* __restrict__ res, int ldr,
                                                        float* __restrict__ y, int ldy, int OH, int OW, int KH, int KW,
                                                        int SH, int SW, int PH, int PW, int DH, int DW, int vec4) {
  const int cg = vec4 ? (C >> 2) : C;
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long total = (long long)N * OH * OW * cg;
  if (gid >= total) return;
  const int g = (int)(gid % cg);
  const long long p = gid / cg;
  const int ox = (int)(p % OW);
  const long long t = p / OW;
  const int oy = (int)(t % OH);
  const long long n = t / OH;
  const float* img = x + n * H * W * ldx;
  if (vec4) {
    const int c = g * 4;
    f32x4 acc = *(const f32x4*)(bias + c);
    for (int ky = 0; ky < KH; ++ky) {
      const int iy = oy * SH - PH + ky * DH;
      if ((unsigned)iy >= (unsigned)H) continue;
      for (int kx = 0; kx < KW; ++kx) {
        const int ix = ox * SW - PW + kx * DW;
        if ((unsigned)ix >= (unsigned)W) continue;
        const f32x4 v = *(const f32x4*)(img + ((long long)iy * W + ix) * ldx + c);
        const f32x4 k = *(const f32x4*)(w + (ky * KW + kx) * ldw + c);
        acc += v * k;
      }
    }
    if (silu) {
      acc[0] = silu_fast(acc[0]);
      acc[1] = silu_fast(acc[1]);
      acc[2] = silu_fast(acc[2]);
      acc[3] = silu_fast(acc[3]);
    }
    if (res) acc = *(const f32x4*)(res + p * ldr + c) + acc;
    *(f32x4*)(y + p * ldy + c) = acc;
  } else {
    const int c = g;
    float acc = bias[c];
    for (int ky = 0; ky < KH; ++ky) {
      const int iy = oy * SH - PH + ky * DH;
      if ((unsigned)iy >= (unsigned)H) continue;
      for (int kx = 0; kx < KW; ++kx) {
        const int ix = ox * SW - PW + kx * DW;
        if ((unsigned)ix >= (unsigned)W) continue;
        acc += img[((long long)iy * W + ix) * ldx + c] * w[(ky * KW + kx) * ldw + c];
      }
    }
    if (silu) acc = silu_f(acc);
    if (res) acc = res[p * ldr + c] + acc;
    y[p * ldy + c] = acc;
  }
}

// Depthwise 3x3 (pad 1, dilation 1), four channels and four consecutive
// output columns per thread: the nine weight float4s stay in registers and
// each input row is read once for the four outputs (3S + 3 float4 loads per
// row instead of 12), which keeps the L1 under the HBM rate.  Lanes take
// consecutive channel groups first, so every load is a contiguous run of an
// NHWC row.
template <int S>
__global__ __launch_bounds__(256) void dw3_kernel(const float* __restrict__ x, int ldx, int N, int H, int W, int C,
                                                  const float* __restrict__ w, int ldw,
                                                  const float* __restrict__ bias, int silu,
                                                  const float* __restrict__ res, int ldr, float* __restrict__ y,
                                                  int ldy, int OH, int OW) {
  constexpr int R = 4;              // output columns per thread
  constexpr int IWN = R * S + 3 - S;  // input columns they touch
  const int cg = C >> 2;
  const int strips = (OW + R - 1) / R;
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long total = (long long)N * OH * strips * cg;
  if (gid >= total) return;
  // Index decode in 32 bits when the grid allows (64-bit division is a long
  // instruction sequence per thread).
  int g, sx, oy;
  long long n;
  if (total < (1LL << 31)) {
    const unsigned gg = (unsigned)gid, ucg = (unsigned)cg, ust = (unsigned)strips, uoh = (unsigned)OH;
    const unsigned q = gg / ucg, t = q / ust;
    g = (int)(gg - q * ucg);
    sx = (int)(q - t * ust);
    oy = (int)(t % uoh);
    n = t / uoh;
  } else {
    g = (int)(gid % cg);
    const long long q = gid / cg;
    sx = (int)(q % strips);
    const long long t = q / strips;
    oy = (int)(t % OH);
    n = t / OH;
  }
  const int c = 4 * g;
  const int ox0 = sx * R;
  const int ix0 = ox0 * S - 1;
  const float* img = x + n * H * W * ldx + c;
  // Every input load is issued before the arithmetic, without branches:
  // clamped (in-bounds) addresses, zero outside the image.
  f32x4 v[3][IWN];
#pragma unroll
  for (int ky = 0; ky < 3; ++ky) {
    const int iy = oy * S - 1 + ky;
    const bool rok = (unsigned)iy < (unsigned)H;
    const float* row = img + (long long)min(max(iy, 0), H - 1) * W * ldx;
#pragma unroll
    for (int i = 0; i < IWN; ++i) {
      const int ix = ix0 + i;
      const f32x4 u = *(const f32x4*)(row + (long long)min(max(ix, 0), W - 1) * ldx);
      v[ky][i] = rok && (unsigned)ix < (unsigned)W ? u : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  f32x4 k[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) k[i] = *(const f32x4*)(w + i * ldw + c);
  const f32x4 b = *(const f32x4*)(bias + c);
  f32x4 acc[R];
#pragma unroll
  for (int j = 0; j < R; ++j) acc[j] = b;
#pragma unroll
  for (int ky = 0; ky < 3; ++ky)
#pragma unroll
    for (int j = 0; j < R; ++j)
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) acc[j] += v[ky][j * S + kx] * k[ky * 3 + kx];
  const long long pix0 = (n * OH + oy) * OW + ox0;
#pragma unroll
  for (int j = 0; j < R; ++j) {
    if (ox0 + j >= OW) break;
    f32x4 o = acc[j];
    if (silu) {
      o[0] = silu_fast(o[0]);
      o[1] = silu_fast(o[1]);
      o[2] = silu_fast(o[2]);
      o[3] = silu_fast(o[3]);
    }
    if (res) o = *(const f32x4*)(res + (pix0 + j) * ldr + c) + o;
    *(f32x4*)(y + (pix0 + j) * ldy + c) = o;
  }
}

// Depthwise 3x3, stride 1, pad 1, with no LDS and no barrier: a thread owns
// one output column, four channels and SEG consecutive output rows.  It
// loads the (SEG + 2) x 3 input pixels its window slides over (clamped
// in-bounds addresses, zero outside the image, all issued before the
// arithmetic), so every input row leaves HBM once per segment; the left and
// right columns are the neighbouring threads' centre columns and come from
// L1.  Lanes take consecutive channel groups first, so every load and store
// is a contiguous run of an NHWC row.
template <int SEG>
__global__ __launch_bounds__(256) void dw3_col_kernel(const float* __restrict__ x, int ldx, int N, int H, int W, int C,
                                                      const float* __restrict__ w, int ldw,
                                                      const float* __restrict__ bias, int silu,
                                                      const float* __restrict__ res, int ldr, float* __restrict__ y,
                                                      int ldy) {
  const int cg = C >> 2;
  const int segs = (H + SEG - 1) / SEG;
  const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long total = (long long)N * segs * W * cg;
  if (gid >= total) return;
  int g, ox, sg;
  long long n;
  if (total < (1LL << 31)) {
    const unsigned gg = (unsigned)gid, ucg = (unsigned)cg, uw = (unsigned)W, us = (unsigned)segs;
    const unsigned q = gg / ucg, t = q / uw;
    g = (int)(gg - q * ucg);
    ox = (int)(q - t * uw);
    sg = (int)(t % us);
    n = t / us;
  } else {
    g = (int)(gid % cg);
    const long long q = gid / cg;
    ox = (int)(q % W);
    const long long t = q / W;
    sg = (int)(t % segs);
    n = t / segs;
  }
  const int c = 4 * g, oy0 = sg * SEG;
  const float* img = x + n * H * W * ldx + c;
  f32x4 v[SEG + 2][3];
#pragma unroll
  for (int r = 0; r < SEG + 2; ++r) {
    const int iy = oy0 - 1 + r;
    const bool rok = (unsigned)iy < (unsigned)H;
    const float* row = img + (long long)min(max(iy, 0), H - 1) * W * ldx;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      const int ix = ox - 1 + j;
      const f32x4 u = *(const f32x4*)(row + (long long)min(max(ix, 0), W - 1) * ldx);
      v[r][j] = rok && (unsigned)ix < (unsigned)W ? u : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  f32x4 k[9];
#pragma unroll
  for (int i = 0; i < 9; ++i) k[i] = *(const f32x4*)(w + i * ldw + c);
  const f32x4 b = *(const f32x4*)(bias + c);
  const long long pix0 = (n * H + oy0) * W + ox;
  // Residual values before the first store (a wait for a load also waits for
  // the stores issued before it).
  f32x4 rv[SEG];
  if (res) {
#pragma unroll
    for (int r = 0; r < SEG; ++r) rv[r] = *(const f32x4*)(res + (pix0 + (long long)min(r, H - 1 - oy0) * W) * ldr + c);
  }
#pragma unroll
  for (int r = 0; r < SEG; ++r) {
    if (oy0 + r >= H) break;
    f32x4 o = b;
#pragma unroll
    for (int ky = 0; ky < 3; ++ky)
#pragma unroll
      for (int kx = 0; kx < 3; ++kx) o += v[r + ky][kx] * k[ky * 3 + kx];
    if (silu) {
      o[0] = silu_fast(o[0]);
      o[1] = silu_fast(o[1]);
      o[2] = silu_fast(o[2]);
      o[3] = silu_fast(o[3]);
    }
    if (res) o = rv[r] + o;
    *(f32x4*)(y + (pix0 + (long long)r * W) * ldy + c) = o;
  }
}

// Depthwise 3x3, stride 1, pad 1, from an LDS tile with a one-pixel halo:
// a workgroup covers kDwRows output rows x TX columns x 32 channels of one
// image.  The (kDwRows + 2) x (TX + 2) input pixels are loaded once with
// eight lanes per pixel (one 128-byte line of its 32 channels), so each
// input line leaves HBM once per tile instead of once per tap.  Each
// (column, channel group) item then slides the 3x3 window down the tile's
// rows in registers: three LDS reads per output row.  TX = 20 for widths that
// are multiples of 20 (every YOLO level of a 640 input), else 32.
constexpr int kDwRows = 8, kDwGroups = 8;  // output rows, float4 channel groups per workgroup

template <int TX>
__global__ __launch_bounds__(256) void dw3_tile_kernel(const float* __restrict__ x, int ldx, int H, int W, int C,
                                                       const float* __restrict__ w, int ldw,
                                                       const float* __restrict__ bias, int silu,
                                                       const float* __restrict__ res, int ldr, float* __restrict__ y,
                                                       int ldy, int tiles_x, int tiles_y, int cblocks) {
  constexpr int IX = TX + 2, IY = kDwRows + 2;
  __shared__ f32x4 t[IY][IX][kDwGroups];
  int b = blockIdx.x;
  const int cb = b % cblocks;
  b /= cblocks;
  const int bx = b % tiles_x;
  b /= tiles_x;
  const int by = b % tiles_y;
  const int n = b / tiles_y;
  const int cg = C >> 2, g0 = cb * kDwGroups;
  const int oy0 = by * kDwRows, ox0 = bx * TX;
  const float* img = x + (long long)n * H * W * ldx;
  // Stage the input tile; pixels outside the image and channel groups past
  // C read as zero (clamped in-bounds addresses, no branches around loads).
  constexpr int NE = IY * IX * kDwGroups;
  constexpr int U = (NE + 255) / 256;
  f32x4 v[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = min(u * 256 + (int)threadIdx.x, NE - 1);
    const int g = e % kDwGroups, px = e / kDwGroups;
    const int iy = oy0 - 1 + px / IX, ix = ox0 - 1 + px % IX;
    const bool ok = (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W && g0 + g < cg;
    const f32x4 a = *(const f32x4*)(img + ((long long)min(max(iy, 0), H - 1) * W + min(max(ix, 0), W - 1)) * ldx +
                                    4 * min(g0 + g, cg - 1));
    v[u] = ok ? a : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int e = u * 256 + (int)threadIdx.x;
    if (e < NE) (&t[0][0][0])[e] = v[u];
  }
  __syncthreads();
  for (int it = threadIdx.x; it < TX * kDwGroups; it += 256) {
    const int g = it % kDwGroups, col = it / kDwGroups;
    const int ox = ox0 + col, c = 4 * (g0 + g);
    if (ox >= W || g0 + g >= cg) continue;
    f32x4 k[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) k[i] = *(const f32x4*)(w + i * ldw + c);
    const f32x4 bv = *(const f32x4*)(bias + c);
    f32x4 r0[3], r1[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      r0[j] = t[0][col + j][g];
      r1[j] = t[1][col + j][g];
    }
#pragma unroll
    for (int r = 0; r < kDwRows; ++r) {
      f32x4 r2[3];
#pragma unroll
      for (int j = 0; j < 3; ++j) r2[j] = t[r + 2][col + j][g];
      f32x4 o = bv;
#pragma unroll
      for (int j = 0; j < 3; ++j) o += r0[j] * k[j] + r1[j] * k[3 + j] + r2[j] * k[6 + j];
      const int oy = oy0 + r;
      if (oy < H) {
        if (silu) {
          o[0] = silu_fast(o[0]);
          o[1] = silu_fast(o[1]);
          o[2] = silu_fast(o[2]);
          o[3] = silu_fast(o[3]);
        }
        const long long pix = ((long long)n * H + oy) * W + ox;
        if (res) o = *(const f32x4*)(res + pix * ldr + c) + o;
        *(f32x4*)(y + pix * ldy + c) = o;
      }
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        r0[j] = r1[j];
        r1[j] = r2[j];
      }
    }
  }
}

// ------------------------------------------------------------ direct (stem)

// The network stem: 3x3 stride-2 pad-1 conv of the 3-channel NCHW input
// (VulkanLowChannels.cs:28-46).  A workgroup owns 4 output rows x 64 output
// columns of one image.  It reads the 3 x 9 x 129 input patch once, with
// row-contiguous loads all issued before the first use, into LDS split into
// even and odd columns (the stride-2 taps of adjacent pixels are then
// adjacent words).  Each wave forms one output row: the 27-tap dot products
// run on v_mfma_f32_16x16x4f32 with M = 16 pixels, K = 4 taps (27 padded to
// 28 with a zero weight row) and N = 16 output channels, so the VALU only
// applies SiLU and the stores.
constexpr int kStemRows = 4, kStemCols = 64;

template <int OC>
__global__ __launch_bounds__(256) void stem_kernel(const float* __restrict__ x, int H, int W,
                                                   const float* __restrict__ w, int ocd,
                                                   const float* __restrict__ bias, int silu, float* __restrict__ y,
                                                   int OH, int OW, int ldy) {
  constexpr int PR = 2 * kStemRows + 1;              // patch rows
  constexpr int PE = kStemCols + 1, PO = kStemCols;  // even / odd patch columns
  constexpr int PC = PE + PO;                        // 2 * kStemCols + 1 input columns
  constexpr int TOTAL = 3 * PR * PC;
  constexpr int IT = (TOTAL + 255) / 256;
  constexpr int NB = OC / 16;                        // 16-channel output blocks
  __shared__ float patch[3 * PR * PE + 3 * PR * PO];  // even columns, then odd
  float* pe = patch;
  float* po = patch + 3 * PR * PE;
  const int tid = threadIdx.x;
  const int n = blockIdx.z;
  const int oy0 = blockIdx.y * kStemRows, ox0 = blockIdx.x * kStemCols;
  const int iy0 = 2 * oy0 - 1, ix0 = 2 * ox0 - 1;
  const float* img = x + (long long)n * 3 * H * W;
  // Issue every patch load before the first use: clamped (always in-bounds)
  // addresses, zeroed where the tap falls outside the image.  With W % 4 == 0
  // a patch row is read as 33 aligned float4s starting 3 columns left of the
  // patch (a float4 then lies wholly inside or wholly outside the image row);
  // otherwise one float per thread and column.
  constexpr int Q4 = (PC + 3 + 3) / 4;  // float4s per patch row
  constexpr int TOTAL4 = 3 * PR * Q4;
  constexpr int IT4 = (TOTAL4 + 255) / 256;
  const bool vec = (W & 3) == 0 && ((uintptr_t)x & 15) == 0;
  float v[IT];
  f32x4 v4[IT4];
  if (vec) {
#pragma unroll
    for (int it = 0; it < IT4; ++it) {
      const int i = tid + it * 256;
      const int c = i / (PR * Q4);
      const int rem = i - c * (PR * Q4);
      const int r = rem / Q4, j = rem - r * Q4;
      const int iy = iy0 + r, ix = ix0 - 3 + 4 * j;
      const bool ok = i < TOTAL4 && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
      const int cc = min(c, 2), cy = min(max(iy, 0), H - 1), cx = min(max(ix, 0), W - 4);
      const f32x4 t = *(const f32x4*)(img + ((long long)cc * H + cy) * W + cx);
      v4[it] = ok ? t : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  } else {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int i = tid + it * 256;
      const int c = i / (PR * PC);
      const int rem = i - c * (PR * PC);
      const int r = rem / PC, col = rem - r * PC;
      const int iy = iy0 + r, ix = ix0 + col;
      const bool ok = i < TOTAL && (unsigned)iy < (unsigned)H && (unsigned)ix < (unsigned)W;
      const int cc = min(c, 2), cy = min(max(iy, 0), H - 1), cx = min(max(ix, 0), W - 1);
      const float t = img[((long long)cc * H + cy) * W + cx];
      v[it] = ok ? t : 0.f;
    }
  }
  // B operand of k-step s for this lane: weight row kk = 4 s + lane / 16 (rows
  // ordered (ky, kx, c)), output channel 16 nb + lane % 16; row 27 is zero.
  const int lane = tid & 63, g = lane >> 4, q = lane & 15;
  float bw[7][NB];
#pragma unroll
  for (int st = 0; st < 7; ++st) {
    const int kk = 4 * st + g;
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) bw[st][nb] = kk < 27 ? w[kk * ocd + 16 * nb + q] : 0.f;
  }
  if (vec) {
#pragma unroll
    for (int it = 0; it < IT4; ++it) {
      const int i = tid + it * 256;
      if (i < TOTAL4) {
        const int c = i / (PR * Q4);
        const int rem = i - c * (PR * Q4);
        const int r = rem / Q4, j = rem - r * Q4;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int col = 4 * j + e - 3;  // patch column
          if (col >= 0 && col < PC) {
            if (col & 1) po[(c * PR + r) * PO + (col >> 1)] = v4[it][e];
            else pe[(c * PR + r) * PE + (col >> 1)] = v4[it][e];
          }
        }
      }
    }
  } else {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int i = tid + it * 256;
      if (i < TOTAL) {
        const int c = i / (PR * PC);
        const int rem = i - c * (PR * PC);
        const int r = rem / PC, col = rem - r * PC;
        if (col & 1) po[(c * PR + r) * PO + (col >> 1)] = v[it];
        else pe[(c * PR + r) * PE + (col >> 1)] = v[it];
      }
    }
  }
  __syncthreads();
  // Wave w forms output rows w, w + 4, ... of the tile.
  typedef float f32x4v __attribute__((ext_vector_type(4)));
#pragma unroll 1
  for (int rr = 0; rr < kStemRows / 4; ++rr) {
    const int ty = (tid >> 6) + 4 * rr;
    const int oy = oy0 + ty;
    if (oy >= OH) return;
    // A operand of k-step s: MFMA row q = lane % 16 holds pixel 16 mb + pm with
    // pm = 4 (q % 4) + q / 4, tap kk = 4 s + lane / 16, so that D register i of
    // lane group g is pixel 16 mb + 4 i + g and one store covers four adjacent
    // pixels (256 contiguous bytes at 16 channels).  Tap 27 (padding) re-reads
    // tap 26 of the same pixel; its weight row is 0.
    const int pm = 4 * (q & 3) + (q >> 2);
    int off[7];
#pragma unroll
    for (int st = 0; st < 7; ++st) {
      const int kk = min(4 * st + g, 26);
      const int t = kk / 3, c = kk - 3 * t;
      const int ky = t / 3, kx = t - 3 * ky;
      const int row = 2 * ty + ky;
      off[st] = kx == 1 ? 3 * PR * PE + (c * PR + row) * PO + pm : (c * PR + row) * PE + pm + (kx >> 1);
    }
    f32x4v acc[4][NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const float b0 = bias[16 * nb + q];
#pragma unroll
      for (int mb = 0; mb < 4; ++mb) acc[mb][nb] = f32x4v{b0, b0, b0, b0};
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
      for (int st = 0; st < 7; ++st) {
        const float a = patch[off[st] + 16 * mb];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bw[st][nb], acc[mb][nb], 0, 0, 0);
      }
    // D layout: lane holds channel 16 nb + lane % 16 of MFMA rows 4 (lane / 16) + i,
    // i.e. pixels 16 mb + 4 i + lane / 16.
    float* out = y + ((long long)n * OH + oy) * OW * ldy;
    if (silu) {
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[mb][nb][i] = silu_fast(acc[mb][nb][i]);
    }
    if (ox0 + kStemCols <= OW) {
      // The row's 64 pixels all lie inside the output: no per-pixel tests.
      float* o = out + (long long)(ox0 + g) * ldy + q;
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) o[(16 * mb + 4 * i) * ldy + 16 * nb] = acc[mb][nb][i];
    } else {
#pragma unroll
      for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int ox = ox0 + 16 * mb + 4 * i + g;
          if (ox < OW) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) out[(long long)ox * ldy + 16 * nb + q] = acc[mb][nb][i];
          }
        }
    }
  }
}

// One thread per output pixel and 16 output channels; weights [K][ocd] of
// this 16-channel block staged in LDS.  Input NCHW (dense) or an NHWC view.
__global__ __launch_bounds__(256) void direct_kernel(const float* __restrict__ x, int nchw, int N, int H, int W,
                                                     int IC, int ldx, const float* __restrict__ w, int ocd,
                                                     const float* __restrict__ bias, int silu, float* __restrict__ y,
                                                     int OH, int OW, int OC, int ldy, int KH, int KW, int SH, int SW,
                                                     int PH, int PW, int DH, int DW) {
  extern __shared__ float wl[];  // [K][16]
  const int K = KH * KW * IC;
  const int oc0 = blockIdx.y * 16;
  for (int i = threadIdx.x; i < K * 16; i += blockDim.x) wl[i] = w[(long long)(i >> 4) * ocd + oc0 + (i & 15)];
  __syncthreads();
  const long long m = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const long long M = (long long)N * OH * OW;
  if (m >= M) return;
  const int ox = (int)(m % OW);
  const long long t = m / OW;
  const int oy = (int)(t % OH);
  const int n = (int)(t / OH);
  float acc[16];
#pragma unroll
  for (int o = 0; o < 16; ++o) acc[o] = bias[oc0 + o];
  for (int ky = 0; ky < KH; ++ky) {
    const int iy = oy * SH - PH + ky * DH;
    if ((unsigned)iy >= (unsigned)H) continue;
    for (int kx = 0; kx < KW; ++kx) {
      const int ix = ox * SW - PW + kx * DW;
      if ((unsigned)ix >= (unsigned)W) continue;
      const float* wk = wl + (ky * KW + kx) * IC * 16;
      for (int ic = 0; ic < IC; ++ic) {
        const float v = nchw ? x[(((long long)n * IC + ic) * H + iy) * W + ix]
                             : x[(((long long)n * H + iy) * W + ix) * ldx + ic];
#pragma unroll
        for (int o = 0; o < 16; ++o) acc[o] += v * wk[ic * 16 + o];
      }
    }
  }
  float* dst = y + m * ldy + oc0;
  const int lim = OC - oc0 < 16 ? OC - oc0 : 16;
  if (lim == 16 && (ldy & 3) == 0 && (((uintptr_t)dst) & 15) == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = silu ? silu_f(acc[q * 4 + e]) : acc[q * 4 + e];
      *(f32x4*)(dst + q * 4) = v;
    }
  } else {
    for (int o = 0; o < lim; ++o) dst[o] = silu ? silu_f(acc[o]) : acc[o];
  }
}

// ------------------------------------------------------------ preparation

static int upload(sy_ctx* ctx, const std::vector<float>& h, float** d) {
  SY_CHECK(!ctx->capturing, SY_ESTATE, "weight upload during graph capture");
  // The copy runs on the legacy null stream: wait until no other context has
  // a capture open (bounded, so that a thread holding a capture of its own
  // on another context gets an error instead of waiting on itself).
  std::unique_lock<std::shared_timed_mutex> lock(capture_lock(), std::defer_lock);
  SY_CHECK(lock.try_lock_for(std::chrono::seconds(60)), SY_ESTATE,
           "weight upload waited 60 s for graph captures on other contexts to end");
  void* p = nullptr;
  SY_HIP(hipMalloc(&p, h.size() * sizeof(float)));
  ctx->owned.push_back(p);
  SY_HIP(hipMemcpy(p, h.data(), h.size() * sizeof(float), hipMemcpyHostToDevice));
  *d = (float*)p;
  return SY_OK;
}

static inline int round_up(int v, int m) { return (v + m - 1) / m * m; }

// The fused Winograd kernels address a 32-tile block's input in 32 bits from
// the image of its first tile: the images such a block spans (at most
// 31 / tiles-per-image + 2) must stay below the zero-read buffer offset.
static bool fused_wino_fits(const sy_tensor* x) {
  const long long tpi = (long long)((x->h + 3) / 4) * ((x->w + 3) / 4);
  const long long img = (long long)x->h * x->w * x->ldc;
  return 4 * img * (31 / tpi + 2) < kFxOob;
}

// 3x3 pad-1 undilated ungrouped convolution of that stride on whole float4s.
static bool conv3x3(const ConvPlan* p, int stride) {
  return p->groups == 1 && p->kh == 3 && p->kw == 3 && p->sh == stride && p->sw == stride && p->dh == 1 &&
         p->dw == 1 && p->pt == 1 && p->pl == 1 && p->pb == 1 && p->pr == 1 && p->ic % 4 == 0 && !p->up2;
}
static bool conv3x3_patch(const ConvPlan* p) { return conv3x3(p, 1) || conv3x3(p, 2); }

bool conv_supports(const ConvPlan* p, int algo) {
  const bool g1 = p->groups == 1;
  switch (algo) {
    case kIgemm: return g1 && p->ic % 4 == 0;
    case kWinograd: return conv3x3(p, 1) && p->oc % 4 == 0;
    case kDirect: return g1 && p->kh * p->kw * p->ic <= 1024;
    case kWinograd3: return conv_supports(p, kWinograd);
    case kDepthwise: return p->groups == p->ic && p->ic == p->oc;
    case kWinograd2: return conv_supports(p, kWinograd) && p->ic % 8 == 0;
    default: return false;
  }
}

static int auto_algo(const ConvPlan* p) {
  const char* wenv = getenv("SIMDYOLO_HIP_WINOGRAD");
  const bool wino_on = !(wenv && strcmp(wenv, "0") == 0);
  if (conv_supports(p, kDepthwise)) return kDepthwise;
  if (p->groups == 1 && p->ic % 4 != 0 && conv_supports(p, kDirect)) return kDirect;
  if (wino_on && conv_supports(p, kWinograd) && p->ic >= 16) {
    // Without the tuner the rule keeps the three-kernel form: the routing
    // rule does not see the input size, and the fused kernels, fastest on
    // large grids, leave most CUs idle on small ones (batch 1, 20x20
    // layers).  The fused kernel is selectable (SIMDYOLO_HIP_WINO_FUSED=1
    // or SY_CONV_WINOGRAD).
    const char* f = getenv("SIMDYOLO_HIP_WINO_FUSED");
    return (f && strcmp(f, "1") == 0) ? kWinograd : kWinograd3;
  }
  if (conv_supports(p, kIgemm)) return kIgemm;
  if (conv_supports(p, kDirect)) return kDirect;
  return -1;
}

// Whether the device weights the given algorithm reads are there.
static bool weights_packed(const ConvPlan* p, int algo, int tile) {
  if (algo == kIgemm) return (is_x3_tile(tile) ? p->w_x3 : is_c3_tile(tile) ? p->w_c3 : p->w_gemm) != nullptr;
  if (algo == kDirect) return p->w_direct != nullptr;
  if (algo == kDepthwise) return p->w_dw != nullptr;
  return (algo == kWinograd2 || algo == kWinograd ? p->w_wino_b : p->w_wino) != nullptr;
}

// Packs them (once).
static int pack_weights(sy_ctx* ctx, ConvPlan* p, int algo, int tile) {
  const bool x3 = algo == kIgemm && is_x3_tile(tile), c3 = algo == kIgemm && is_c3_tile(tile);
  SY_CHECK(!ctx->capturing || weights_packed(p, algo, tile), SY_ESTATE, "weight packing during graph capture");
  const int oc = p->oc, ic = p->ic, kh = p->kh, kw = p->kw;
  const float* W = p->host_w.data();
  if ((x3 && !p->w_x3) || (c3 && !p->w_c3)) {
    SY_CHECK(p->finite, SY_EUNSUPPORTED, "the f16-split kernels take finite weights only");
    // Split weights in the GEMM's or the 3x3 patch kernel's operand order
    // (igemm.h), then the channels' inverse scales.
    const int taps = kh * kw, K = taps * ic, nkt = (K + 31) / 32, ng = (ic + 15) / 16, ocp = oc_pad(oc);
    const size_t units = x3 ? (size_t)(ocp / 32) * nkt * kX3Units : (size_t)(ocp / 32) * ng * taps * 128;
    std::vector<float> h(units * 4 + ocp, 0.f);
    uint16_t* q = (uint16_t*)h.data();
    std::vector<uint16_t> hi(K), lo(K);
    for (int o = 0; o < oc; ++o) {
      const float* g = W + (size_t)o * K;
      float big = 0.f;
      for (int i = 0; i < K; ++i) big = std::max(big, std::fabs(g[i]));
      const float scale = x3_weight_scale(big);
      h[units * 4 + o] = 1.f / scale;
      x3_split(g, K, scale, hi.data(), lo.data());
      for (int c = 0; c < ic; ++c)
        for (int t = 0; t < taps; ++t) {
          const int k = x3 ? t * ic + c : c;
          const size_t unit = x3 ? ((size_t)(o >> 5) * nkt + (k >> 5)) * kX3Units + ((k >> 4) & 1) * 128
                                 : (((size_t)(o >> 5) * ng + (c >> 4)) * taps + t) * 128;
          const size_t at = (unit + ((k >> 3) & 1) * 32 + (o & 31)) * 8 + (k & 7);
          q[at] = hi[c * taps + t];
          q[at + 512] = lo[c * taps + t];
        }
    }
    float* d = nullptr;
    SY_TRY(upload(ctx, h, &d));
    (x3 ? p->w_x3 : p->w_c3) = d;
    (x3 ? p->w_x3s : p->w_c3s) = d + units * 4;
  }
  if (algo == kIgemm && !x3 && !c3 && !p->w_gemm) {
    const int K = kh * kw * ic;
    p->kp = round_up(K, 32);  // the deepest K tile
    p->ocp = oc_pad(oc);
    std::vector<float> h((size_t)p->ocp * p->kp, 0.f);
    for (int o = 0; o < oc; ++o)
      for (int c = 0; c < ic; ++c)
        for (int ky = 0; ky < kh; ++ky)
          for (int kx = 0; kx < kw; ++kx)
            h[(size_t)o * p->kp + (ky * kw + kx) * ic + c] = W[(((size_t)o * ic + c) * kh + ky) * kw + kx];
    SY_TRY(upload(ctx, h, &p->w_gemm));
  }
  if ((algo == kWinograd2 || algo == kWinograd) && !p->w_wino_b) {
    // U = G g G^T in double, stored as MFMA B-operand blocks
    // [36][oc / 32][ic / 8][lane = 32 * ((k / 4) % 2) + oc % 32][k % 4]
    // (output channels and a last partial K chunk padded with zeros).
    static const double G[6][3] = {{0.25, 0, 0},
                                   {-1.0 / 6, -1.0 / 6, -1.0 / 6},
                                   {-1.0 / 6, 1.0 / 6, -1.0 / 6},
                                   {1.0 / 24, 1.0 / 12, 1.0 / 6},
                                   {1.0 / 24, -1.0 / 12, 1.0 / 6},
                                   {0, 0, 1}};
    const int nob = (oc + 31) / 32, nkc = (ic + 7) / 8;
    std::vector<float> h((size_t)36 * nob * nkc * 256, 0.f);
    for (int o = 0; o < oc; ++o)
      for (int c = 0; c < ic; ++c) {
        const float* g = W + ((size_t)o * ic + c) * 9;
        double tmp[6][3];
        for (int i = 0; i < 6; ++i)
          for (int j = 0; j < 3; ++j) tmp[i][j] = G[i][0] * g[0 * 3 + j] + G[i][1] * g[1 * 3 + j] + G[i][2] * g[2 * 3 + j];
        const int lanev = 32 * ((c >> 2) & 1) + (o & 31);
        for (int i = 0; i < 6; ++i)
          for (int j = 0; j < 6; ++j) {
            double u = tmp[i][0] * G[j][0] + tmp[i][1] * G[j][1] + tmp[i][2] * G[j][2];
            const size_t blk = ((size_t)(i * 6 + j) * nob + (o >> 5)) * nkc + (c >> 3);
            h[blk * 256 + lanev * 4 + (c & 3)] = (float)u;
          }
      }
    SY_TRY(upload(ctx, h, &p->w_wino_b));
  }
  if (algo == kWinograd3 && !p->w_wino) {
    // U = G g G^T (6x6) per (oc, ic), computed in double.
    static const double G[6][3] = {{0.25, 0, 0},
                                   {-1.0 / 6, -1.0 / 6, -1.0 / 6},
                                   {-1.0 / 6, 1.0 / 6, -1.0 / 6},
                                   {1.0 / 24, 1.0 / 12, 1.0 / 6},
                                   {1.0 / 24, -1.0 / 12, 1.0 / 6},
                                   {0, 0, 1}};
    p->kpw = round_up(ic, 32);
    p->ocw = oc_pad(oc);
    std::vector<float> h((size_t)36 * p->ocw * p->kpw, 0.f);
    for (int o = 0; o < oc; ++o)
      for (int c = 0; c < ic; ++c) {
        const float* g = W + ((size_t)o * ic + c) * 9;
        double tmp[6][3];
        for (int i = 0; i < 6; ++i)
          for (int j = 0; j < 3; ++j) tmp[i][j] = G[i][0] * g[0 * 3 + j] + G[i][1] * g[1 * 3 + j] + G[i][2] * g[2 * 3 + j];
        for (int i = 0; i < 6; ++i)
          for (int j = 0; j < 6; ++j) {
            double u = tmp[i][0] * G[j][0] + tmp[i][1] * G[j][1] + tmp[i][2] * G[j][2];
            h[((size_t)(i * 6 + j) * p->ocw + o) * p->kpw + c] = (float)u;
          }
      }
    SY_TRY(upload(ctx, h, &p->w_wino));
  }
  if (algo == kDirect && !p->w_direct) {
    const int K = kh * kw * ic;
    p->ocd = round_up(oc, 16);
    std::vector<float> h((size_t)K * p->ocd, 0.f);
    for (int o = 0; o < oc; ++o)
      for (int c = 0; c < ic; ++c)
        for (int ky = 0; ky < kh; ++ky)
          for (int kx = 0; kx < kw; ++kx)
            h[(size_t)((ky * kw + kx) * ic + c) * p->ocd + o] = W[(((size_t)o * ic + c) * kh + ky) * kw + kx];
    SY_TRY(upload(ctx, h, &p->w_direct));
  }
  if (algo == kDepthwise && !p->w_dw) {
    // [tap][channel], channels contiguous for float4 loads.
    const int C4 = round_up(oc, 4);
    std::vector<float> h((size_t)kh * kw * C4, 0.f);
    for (int o = 0; o < oc; ++o)
      for (int t = 0; t < kh * kw; ++t) h[(size_t)t * C4 + o] = W[(size_t)o * kh * kw + t];
    SY_TRY(upload(ctx, h, &p->w_dw));
  }
  if (!p->bias) {
    std::vector<float> h((size_t)oc_pad(oc), 0.f);
    for (int o = 0; o < oc; ++o) h[o] = p->host_b[o];
    SY_TRY(upload(ctx, h, &p->bias));
  }
  return SY_OK;
}

int conv_prepare(sy_ctx* ctx, ConvPlan* p) {
  int algo = p->algo == kAuto ? auto_algo(p) : p->algo;
  SY_CHECK(algo > 0, SY_EUNSUPPORTED,
           "convolution oc=%d ic=%d k=%dx%d groups=%d is not supported by the HIP backend", p->oc, p->ic, p->kh,
           p->kw, p->groups);
  p->algo = algo;
  for (float w : p->host_w) p->finite = p->finite && std::isfinite(w);
  return pack_weights(ctx, p, algo, -1);
}

void conv_out_size(const ConvPlan* p, int h, int w, int* oh, int* ow) {
  if (p->up2) {
    *oh = 2 * h;
    *ow = 2 * w;
    return;
  }
  long long hn = (long long)h + p->pt + p->pb - (long long)p->dh * (p->kh - 1) - 1;
  long long wn = (long long)w + p->pl + p->pr - (long long)p->dw * (p->kw - 1) - 1;
  *oh = hn < 0 ? 0 : (int)(hn / p->sh + 1);
  *ow = wn < 0 ? 0 : (int)(wn / p->sw + 1);
}

size_t conv_scratch_bytes(const ConvPlan* p, int n, int h, int w) {
  // The largest need of any Winograd form the tuner may route this conv to:
  // three kernels keep V and M, two kernels keep V in 32-tile blocks.
  const long long tiles = (long long)n * ((h + 3) / 4) * ((w + 3) / 4);
  size_t need = 0;
  // Split-K partials of the implicit GEMM (small grids only).
  if (p->user_algo ? p->algo == kIgemm : conv_supports(p, kIgemm)) {
    int oh = 0, ow = 0;
    conv_out_size(p, h, w, &oh, &ow);
    const long long M = (long long)n * oh * ow;
    const long long ldp = (p->oc + 127) / 128 * 128;
    const long long fl = std::min(16 * M * ldp, kSplitMaxFloats);
    // Some tile's grid is small enough to be split when the largest tile's is.
    if (!p->up2 && (M + 255) / 256 * ((p->oc + 127) / 128) * 2 <= kSplitGridMax) need = (size_t)fl * sizeof(float);
  }
  if (p->user_algo ? p->algo == kWinograd3 : conv_supports(p, kWinograd3))
    need = std::max<size_t>(need, (size_t)36 * tiles * ((size_t)p->ic + p->oc) * sizeof(float) + (size_t)256);
  if (p->user_algo ? p->algo == kWinograd2 : conv_supports(p, kWinograd2)) {
    const size_t b = (size_t)36 * ((tiles + 31) / 32 * 32) * p->ic * sizeof(float) + 256;
    if (b > need) need = b;
  }
  return need;
}

namespace {
struct ForceTile {
  sy_ctx* ctx;
  int saved, saved_split;
  ForceTile(sy_ctx* c, int t, int split) : ctx(c), saved(c->force_tile), saved_split(c->force_split) {
    ctx->force_tile = t;
    ctx->force_split = split;
  }
  ~ForceTile() {
    ctx->force_tile = saved;
    ctx->force_split = saved_split;
  }
};
// Shape tag appended to profile names of the kernels one conv launches;
// cleared on exit so later non-conv kernels carry no stale tag.
struct ProfTag {
  sy_ctx* ctx;
  explicit ProfTag(sy_ctx* c) : ctx(c) {}
  ~ProfTag() { ctx->prof_tag.clear(); }
};
}  // namespace

static int conv_exec(sy_ctx* ctx, ConvPlan* p, const sy_tensor* x, const sy_tensor* y, const sy_tensor* res,
                     ConvChoice ch) {
  SY_TRY(check_view(x, "conv input", true));
  SY_TRY(check_view(y, "conv output"));
  if (res) SY_TRY(check_view(res, "conv residual"));
  SY_CHECK(x->c == p->ic, SY_EINVAL, "conv input has %d channels, weights expect %d", x->c, p->ic);
  int oh, ow;
  conv_out_size(p, x->h, x->w, &oh, &ow);
  SY_CHECK(oh > 0 && ow > 0, SY_EINVAL, "convolution kernel exceeds the padded input dimensions");
  const int yc = p->up2 ? p->up2 : p->oc;
  SY_CHECK(y->n == x->n && y->c == yc && y->h == oh && y->w == ow, SY_EINVAL,
           "conv output view %dx%dx%dx%d does not match expected %dx%dx%dx%d", y->n, y->c, y->h, y->w, x->n, yc, oh,
           ow);
  SY_CHECK(!p->up2 || (!res && ch.algo == kIgemm && x->layout == SY_LAYOUT_NHWC), SY_EUNSUPPORTED,
           "the transposed conv runs as an implicit GEMM without residual");
  if (res)
    SY_CHECK(res->n == y->n && res->c == y->c && res->h == y->h && res->w == y->w, SY_EINVAL,
             "residual shape does not match the conv output");
  const bool nchw = x->layout == SY_LAYOUT_NCHW;
  const int algo = ch.algo;
  SY_TRY(pack_weights(ctx, p, algo, ch.tile >= 0 ? ch.tile : env_tile()));
  ForceTile force(ctx, ch.tile, ch.split);
  ProfTag tag_scope(ctx);
  if (ctx->profile_shapes) {
    char tag[96];
    snprintf(tag, sizeof tag, "%dx%d s%d ic%d oc%d %dx%d n%d%s", p->kh, p->kw, p->sh, p->ic, p->oc, x->h, x->w, x->n,
             res ? " +res" : "");
    ctx->prof_tag = tag;
  }
  if (nchw) {
    SY_CHECK(algo == kDirect, SY_EUNSUPPORTED, "NCHW input is only supported by the direct low-channel conv");
    SY_CHECK(!res, SY_EUNSUPPORTED, "residual is not supported by the direct conv");
  }
  if (algo == kDepthwise) {
    const long long px = (long long)x->n * oh * ow;
    const bool v4 = (p->oc & 3) == 0 && (((uintptr_t)x->data | (uintptr_t)y->data) & 15) == 0 &&
                    ((x->ldc | y->ldc) & 3) == 0 &&
                    (!res || ((((uintptr_t)res->data) & 15) == 0 && (res->ldc & 3) == 0));
    const int cg = v4 ? p->oc / 4 : p->oc;
    const long long threads = px * cg;
    const double dw_flops = 2.0 * px * p->oc * p->kh * p->kw;
    const double dw_bytes = 4.0 * ((double)x->n * x->h * x->w * x->c + (double)px * p->oc * (res ? 2 : 1));
    if (v4 && p->kh == 3 && p->kw == 3 && p->sh == p->sw && (p->sh == 1 || p->sh == 2) && p->pt == 1 &&
        p->pl == 1 && p->dh == 1 && p->dw == 1) {
      // 3x3 stride 1 or 2 on 16-byte channel groups.  Kernel: the tuned
      // choice, else SIMDYOLO_HIP_TILE (0 register, 1 LDS tile, 2 / 3 column
      // with 4- / 8-row segments), else the LDS tile for whole 32-channel
      // blocks (measured 7-29% faster than the register kernel on the
      // YOLO11n batch-32 shapes) and the register kernel otherwise.  The
      // tile and column kernels are stride 1 only.
      const int et = ctx->force_tile >= 0 ? ctx->force_tile : env_tile();
      if (p->sh == 1 && (et == 2 || et == 3)) {
        const int seg = et == 2 ? 4 : 8;
        const long long t = (long long)x->n * ((oh + seg - 1) / seg) * ow * cg;
        SY_CHECK(t < (1LL << 40), SY_EUNSUPPORTED, "depthwise grid too large");
        ProfScope prof(ctx, seg == 4 ? "depthwise_col4" : "depthwise_col8", dw_flops, dw_bytes);
        if (seg == 4)
          hipLaunchKernelGGL(dw3_col_kernel<4>, dim3((unsigned)((t + 255) / 256)), dim3(256), 0, ctx->stream, x->data,
                             x->ldc, x->n, x->h, x->w, p->oc, p->w_dw, round_up(p->oc, 4), p->bias, p->silu,
                             res ? res->data : nullptr, res ? res->ldc : 0, y->data, y->ldc);
        else
          hipLaunchKernelGGL(dw3_col_kernel<8>, dim3((unsigned)((t + 255) / 256)), dim3(256), 0, ctx->stream, x->data,
                             x->ldc, x->n, x->h, x->w, p->oc, p->w_dw, round_up(p->oc, 4), p->bias, p->silu,
                             res ? res->data : nullptr, res ? res->ldc : 0, y->data, y->ldc);
        return check_launch("depthwise_conv");
      }
      if (p->sh == 1 && (et == 1 || (et != 0 && p->oc % 32 == 0))) {
        const int tx = ow % 20 == 0 ? 20 : 32;
        const int tiles_x = (ow + tx - 1) / tx, tiles_y = (oh + kDwRows - 1) / kDwRows;
        const int cblocks = (cg + kDwGroups - 1) / kDwGroups;
        const long long wgs = (long long)x->n * tiles_y * tiles_x * cblocks;
        SY_CHECK(wgs < (1LL << 31), SY_EUNSUPPORTED, "depthwise grid too large");
        ProfScope prof(ctx, tx == 20 ? "depthwise_tile20" : "depthwise_tile32", dw_flops, dw_bytes);
        if (tx == 20)
          hipLaunchKernelGGL(dw3_tile_kernel<20>, dim3((unsigned)wgs), dim3(256), 0, ctx->stream, x->data, x->ldc,
                             x->h, x->w, p->oc, p->w_dw, round_up(p->oc, 4), p->bias, p->silu,
                             res ? res->data : nullptr, res ? res->ldc : 0, y->data, y->ldc, tiles_x, tiles_y, cblocks);
        else
          hipLaunchKernelGGL(dw3_tile_kernel<32>, dim3((unsigned)wgs), dim3(256), 0, ctx->stream, x->data, x->ldc,
                             x->h, x->w, p->oc, p->w_dw, round_up(p->oc, 4), p->bias, p->silu,
                             res ? res->data : nullptr, res ? res->ldc : 0, y->data, y->ldc, tiles_x, tiles_y, cblocks);
        return check_launch("depthwise_conv");
      }
      const long long t4 = (long long)x->n * oh * ((ow + 3) / 4) * cg;
      const dim3 grid((unsigned)((t4 + 255) / 256));
      ProfScope prof(ctx, p->sh == 1 ? "depthwise_reg_s1" : "depthwise_reg_s2", dw_flops, dw_bytes);
      if (p->sh == 1)
        hipLaunchKernelGGL(dw3_kernel<1>, grid, dim3(256), 0, ctx->stream, x->data, x->ldc, x->n, x->h, x->w, p->oc,
                           p->w_dw, round_up(p->oc, 4), p->bias, p->silu, res ? res->data : nullptr,
                           res ? res->ldc : 0, y->data, y->ldc, oh, ow);
      else
        hipLaunchKernelGGL(dw3_kernel<2>, grid, dim3(256), 0, ctx->stream, x->data, x->ldc, x->n, x->h, x->w, p->oc,
                           p->w_dw, round_up(p->oc, 4), p->bias, p->silu, res ? res->data : nullptr,
                           res ? res->ldc : 0, y->data, y->ldc, oh, ow);
      return check_launch("depthwise_conv");
    }
    ProfScope prof(ctx, "depthwise_conv", dw_flops, dw_bytes);
    hipLaunchKernelGGL(depthwise_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, x->data,
                       x->ldc, x->n, x->h, x->w, p->oc, p->w_dw, round_up(p->oc, 4), p->bias, p->silu,
                       res ? res->data : nullptr, res ? res->ldc : 0, y->data, y->ldc, oh, ow, p->kh, p->kw, p->sh,
                       p->sw, p->pt, p->pl, p->dh, p->dw, v4 ? 1 : 0);
    return check_launch("depthwise_conv");
  }
  if (algo == kDirect) {
    SY_CHECK(!res, SY_EUNSUPPORTED, "residual is not supported by the direct conv");
    const int K = p->kh * p->kw * p->ic;
    const long long M = (long long)x->n * oh * ow;
    const bool stem = nchw && p->ic == 3 && p->kh == 3 && p->kw == 3 && p->sh == 2 && p->sw == 2 && p->pt == 1 &&
                      p->pl == 1 && p->dh == 1 && p->dw == 1 && (p->oc == 16 || p->oc == 32 || p->oc == 48 ||
                                                                  p->oc == 64) &&
                      ((uintptr_t)y->data & 15) == 0 && (y->ldc & 3) == 0;
    if (stem) {
      dim3 grid((unsigned)((ow + kStemCols - 1) / kStemCols), (unsigned)((oh + kStemRows - 1) / kStemRows),
                (unsigned)x->n);
      ProfScope prof(ctx, "stem_conv", 2.0 * M * p->oc * K,
                     4.0 * ((double)x->n * x->c * x->h * x->w + (double)M * p->oc + (double)K * p->oc));
      switch (p->oc) {
        case 16: hipLaunchKernelGGL(stem_kernel<16>, grid, dim3(256), 0, ctx->stream, x->data, x->h, x->w, p->w_direct, p->ocd, p->bias, p->silu, y->data, oh, ow, y->ldc); break;
        case 32: hipLaunchKernelGGL(stem_kernel<32>, grid, dim3(256), 0, ctx->stream, x->data, x->h, x->w, p->w_direct, p->ocd, p->bias, p->silu, y->data, oh, ow, y->ldc); break;
        case 48: hipLaunchKernelGGL(stem_kernel<48>, grid, dim3(256), 0, ctx->stream, x->data, x->h, x->w, p->w_direct, p->ocd, p->bias, p->silu, y->data, oh, ow, y->ldc); break;
        default: hipLaunchKernelGGL(stem_kernel<64>, grid, dim3(256), 0, ctx->stream, x->data, x->h, x->w, p->w_direct, p->ocd, p->bias, p->silu, y->data, oh, ow, y->ldc); break;
      }
      return check_launch("stem_conv");
    }
    dim3 grid((unsigned)((M + 255) / 256), (unsigned)((p->oc + 15) / 16));
    ProfScope prof(ctx, "direct_conv", 2.0 * M * p->oc * K,
                   4.0 * ((double)x->n * x->c * x->h * x->w + (double)M * p->oc + (double)K * p->oc));
    hipLaunchKernelGGL(direct_kernel, grid, dim3(256), (size_t)K * 16 * sizeof(float), ctx->stream, x->data,
                       nchw ? 1 : 0, x->n, x->h, x->w, x->c, x->ldc, p->w_direct, p->ocd, p->bias, p->silu, y->data,
                       oh, ow, p->oc, y->ldc, p->kh, p->kw, p->sh, p->sw, p->pt, p->pl, p->dh, p->dw);
    return check_launch("direct_conv");
  }
  // float4 gathers need 16-byte aligned channel groups.
  SY_CHECK(((uintptr_t)x->data & 15) == 0 && (x->ldc & 3) == 0, SY_EINVAL,
           "conv input view must be 16-byte aligned with ldc %% 4 == 0");
  const int et = ch.tile >= 0 ? ch.tile : env_tile();
  if (algo == kIgemm && is_c3_tile(et)) {
    C3Args a{};
    a.x = x->data; a.N = x->n; a.H = x->h; a.W = x->w; a.IC = x->c; a.ldx = x->ldc;
    a.S = p->sh; a.OH = oh; a.OW = ow;
    a.w = p->w_c3; a.ws = p->w_c3s; a.bias = p->bias;
    a.res = res ? res->data : nullptr; a.ldr = res ? res->ldc : 0;
    a.y = y->data; a.ldy = y->ldc; a.OC = p->oc; a.silu = p->silu; a.ng = (p->ic + 15) / 16;
    if (!conv3x3_patch(p) || ctx->up_src || !c3_fits(a)) {
      // Views past the kernel's 32-bit offsets (the tuned choice is kept by
      // shape, not by pitch) take the routing rule.
      SY_CHECK(ch.tile >= 0, SY_EUNSUPPORTED,
               "the 3x3 patch kernel needs a 3x3 stride-1 or -2 pad-1 convolution of 32-bit extent");
      return conv_exec(ctx, p, x, y, res, ConvChoice{p->algo, -1});
    }
    const double px = (double)x->n * oh * ow;
    const char* pn = c3_name(et - kC3Base);
    ProfScope prof(ctx, pn, 2.0 * 9 * px * p->ic * p->oc,
                   4.0 * ((double)x->n * x->h * x->w * p->ic + px * p->oc * (res ? 2 : 1) + 9.0 * p->ic * p->oc));
    SY_TRY(launch_c3(ctx, et - kC3Base, a));
    return check_launch(pn);
  }
  if (algo == kIgemm) {
    IgemmArgs a;
    a.x = x->data; a.N = x->n; a.H = x->h; a.W = x->w; a.IC = x->c; a.ldx = x->ldc;
    a.w = p->w_gemm; a.Kp = p->kp; a.bias = p->bias;
    a.w3 = p->w_x3; a.w3s = p->w_x3s; a.nkt = (p->kh * p->kw * p->ic + 31) / 32;
    a.res = res ? res->data : nullptr; a.ldr = res ? res->ldc : 0;
    a.y = y->data; a.OH = oh; a.OW = ow; a.OC = p->oc; a.ldy = y->ldc;
    a.KH = p->kh; a.KW = p->kw; a.SH = p->sh; a.SW = p->sw; a.PH = p->pt; a.PW = p->pl; a.DH = p->dh; a.DW = p->dw;
    a.K = p->kh * p->kw * p->ic; a.M = x->n * oh * ow; a.silu = p->silu;
    a.xb = a.wb = a.yb = 0;
    a.Nb = p->ocp; a.bguard = 0;
    if (p->up2) {  // GEMM over input pixels; the epilogue scatters to 2x2 sub-pixels
      a.OH = x->h; a.OW = x->w; a.M = x->n * x->h * x->w; a.shuf = p->up2;
    }
    if (ctx->up_src) {  // channels [0, ku) read from the half-resolution view
      a.xu = ctx->up_src->data; a.ldxu = ctx->up_src->ldc; a.ku = ctx->up_src->c;
      a.x = x->data + a.ku;
    }
    const double in_b = (double)x->n * x->h * x->w * x->c, out_b = (double)a.M * p->oc;
    return launch_igemm(ctx, a, 1, false, 2.0 * a.M * p->oc * a.K,
                        4.0 * (in_b + out_b * (res ? 2 : 1) + (double)a.K * p->oc));
  }
  // Winograd
  SY_CHECK(((uintptr_t)y->data & 15) == 0 && (y->ldc & 3) == 0, SY_EINVAL,
           "Winograd output view must be 16-byte aligned with ldc %% 4 == 0");
  if (res)
    SY_CHECK(((uintptr_t)res->data & 15) == 0 && (res->ldc & 3) == 0, SY_EINVAL,
             "Winograd residual view must be 16-byte aligned with ldc %% 4 == 0");
  const int TH = (oh + 3) / 4, TW = (ow + 3) / 4;
  const long long tiles = (long long)x->n * TH * TW;
  SY_CHECK(tiles * p->ic <= (1LL << 31) && tiles <= (1LL << 30), SY_EUNSUPPORTED, "Winograd tensor too large");
  if (algo == kWinograd) {
    SY_CHECK(fused_wino_fits(x), SY_EUNSUPPORTED, "fused Winograd image too large");
    const int ntb = (int)((tiles + 31) / 32), nob = (p->oc + 31) / 32, nkc = (p->ic + 7) / 8;
    WinoGoArgs a{};
    a.V = nullptr; a.U = p->w_wino_b; a.bias = p->bias;
    a.res = res ? res->data : nullptr; a.ldr = res ? res->ldc : 0;
    a.y = y->data; a.ldy = y->ldc; a.OC = p->oc;
    a.TH = TH; a.TW = TW; a.OH = oh; a.OW = ow; a.tiles = tiles;
    a.ntb = ntb; a.nob = nob; a.nkc = nkc; a.silu = p->silu;
    a.x = x->data; a.H = x->h; a.W = x->w; a.IC = x->c; a.ldx = x->ldc;
    const long long wgs = (long long)ntb * nob;
    SY_CHECK(wgs < (1LL << 31), SY_EUNSUPPORTED, "Winograd grid too large");
    const double px = (double)x->n * oh * ow;
    // Form: the tuned choice, else SIMDYOLO_HIP_TILE for an explicit
    // algorithm, else the four-wave kernel (1: warp-specialized; 2: two
    // groups of four waves over 64 output channels sharing each transform,
    // one workgroup per CU).
    int variant = ctx->force_tile >= 0 ? ctx->force_tile : env_tile();
    if (variant < 0 || variant >= kFusedForms) variant = 0;
    static const char* const kNames[kFusedForms] = {"wino_fused", "wino_fused_ws", "wino_fused_g2"};
    ProfScope prof(ctx, kNames[variant], 2.0 * 36 * tiles * p->ic * p->oc,
                   4.0 * ((double)x->n * x->h * x->w * x->c + px * p->oc * (res ? 2 : 1) + 36.0 * p->ic * p->oc));
    if (variant == 1) {
      SY_CHECK(((uintptr_t)x->data & 7) == 0 && (x->ldc & 1) == 0, SY_EINVAL,
               "warp-specialized Winograd input view must be 8-byte aligned with an even ldc");
      hipLaunchKernelGGL(wino_fw_kernel, dim3((unsigned)wgs), dim3(512), 0, ctx->stream, a);
    } else if (variant == 2) {
      const long long wgs2 = (long long)ntb * ((nob + 1) / 2);
      hipLaunchKernelGGL((wino_fx_kernel<9, 2>), dim3((unsigned)wgs2), dim3(512), 0, ctx->stream, a);
    } else {
      hipLaunchKernelGGL((wino_fx_kernel<9, 1>), dim3((unsigned)wgs), dim3(256), 0, ctx->stream, a);
    }
    return check_launch("wino_fused");
  }
  SY_TRY(ensure_scratch(ctx, conv_scratch_bytes(p, x->n, x->h, x->w)));
  if (algo == kWinograd2) {
    SY_CHECK(p->ic % 8 == 0, SY_EUNSUPPORTED, "two-kernel Winograd needs ic %% 8 == 0");
    const int ntb = (int)((tiles + 31) / 32), nob = (p->oc + 31) / 32, nkc = p->ic / 8;
    float* Vb = (float*)ctx->scratch;
    {
      const long long blocks = (long long)ntb * ((nkc + 3) / 4);
      SY_CHECK(blocks < (1LL << 31), SY_EUNSUPPORTED, "Winograd grid too large");
      ProfScope prof(ctx, "wino_input_blk", 0, 4.0 * ((double)x->n * x->h * x->w * x->c + 36.0 * tiles * p->ic));
      hipLaunchKernelGGL(wino_in_blk_kernel, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, x->data, x->h, x->w,
                         x->c, x->ldc, TH, TW, tiles, Vb, (long long)ntb * 32 * p->ic);
      SY_TRY(check_launch("wino_input_blk"));
    }
    WinoGoArgs a{};
    a.V = Vb; a.U = p->w_wino_b; a.bias = p->bias;
    a.res = res ? res->data : nullptr; a.ldr = res ? res->ldc : 0;
    a.y = y->data; a.ldy = y->ldc; a.OC = p->oc;
    a.TH = TH; a.TW = TW; a.OH = oh; a.OW = ow; a.tiles = tiles;
    a.ntb = ntb; a.nob = nob; a.nkc = nkc; a.silu = p->silu;
    const long long wgs = (long long)ntb * nob;
    SY_CHECK(wgs < (1LL << 31), SY_EUNSUPPORTED, "Winograd grid too large");
    const double px = (double)x->n * oh * ow;
    // Wave layout: the tuned choice, else SIMDYOLO_HIP_TILE for an explicit
    // algorithm, else four waves.
    int variant = ctx->force_tile >= 0 ? ctx->force_tile : env_tile();
    if (variant < 0 || variant >= kGoVariants) variant = 0;
    ProfScope prof(ctx, variant ? "wino_gemm_out_w8" : "wino_gemm_out", 2.0 * 36 * tiles * p->ic * p->oc,
                   4.0 * (36.0 * tiles * p->ic + px * p->oc * (res ? 2 : 1) + 36.0 * p->ic * p->oc));
    if (variant)
      hipLaunchKernelGGL(wino_go_kernel<2 * kGoWaves>, dim3((unsigned)wgs), dim3(128 * kGoWaves), 0, ctx->stream, a);
    else
      hipLaunchKernelGGL(wino_go_kernel<kGoWaves>, dim3((unsigned)wgs), dim3(64 * kGoWaves), 0, ctx->stream, a);
    return check_launch("wino_gemm_out");
  }
  float* V = (float*)ctx->scratch;
  float* Mt = V + 36 * tiles * p->ic;
  {
    const long long threads = tiles * (p->ic / 4);
    ProfScope prof(ctx, "wino_input", 0, 4.0 * ((double)x->n * x->h * x->w * x->c + 36.0 * tiles * p->ic));
    hipLaunchKernelGGL((wino_in_kernel<4>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, x->data,
                       x->n, x->h, x->w, x->c, x->ldc,
                         TH, TW, V, tiles * p->ic);
    SY_TRY(check_launch("wino_input"));
  }
  {
    IgemmArgs a;
    a.x = V; a.N = 1; a.H = 1; a.W = (int)tiles; a.IC = p->ic; a.ldx = p->ic;
    a.w = p->w_wino; a.Kp = p->kpw; a.bias = nullptr; a.res = nullptr; a.ldr = 0;
    a.y = Mt; a.OH = 1; a.OW = (int)tiles; a.OC = p->oc; a.ldy = p->oc;
    a.KH = a.KW = a.SH = a.SW = 1; a.PH = a.PW = 0; a.DH = a.DW = 1;
    a.K = p->ic; a.M = (int)tiles; a.silu = 0;
    a.xb = tiles * p->ic; a.wb = (long long)p->ocw * p->kpw; a.yb = tiles * p->oc;
    a.Nb = p->ocw; a.bguard = 0;
    SY_TRY(launch_igemm(ctx, a, 36, true, 2.0 * 36 * tiles * p->ic * p->oc,
                        4.0 * 36 * ((double)tiles * (p->ic + p->oc) + (double)p->ic * p->oc)));
  }
  {
    const long long threads = tiles * p->oc;
    ProfScope prof(ctx, "wino_output", 0,
                   4.0 * (36.0 * tiles * p->oc + (double)x->n * oh * ow * p->oc * (res ? 2 : 1)));
    hipLaunchKernelGGL(wino_out_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, ctx->stream, Mt,
                       tiles * p->oc, p->oc, x->n, TH, TW, oh, ow, p->oc, p->bias, p->silu,
                       res ? res->data : nullptr, res ? res->ldc : 0, y->data, y->ldc);
    SY_TRY(check_launch("wino_output"));
  }
  return SY_OK;
}


// ------------------------------------------------------------ autotuning

static bool autotune_enabled() {
  const char* e = getenv("SIMDYOLO_HIP_AUTOTUNE");
  return !(e && strcmp(e, "0") == 0);
}

// Times every (algorithm, tile) candidate of this conv on the given views and
// keeps the fastest for the input shape: the counterpart of the reference's
// timestamp autotuning of Winograd/conv tiles (VulkanWinograd.cs:83-117).
// Runs outside graph capture only; the candidates all write y.
// Key of a tuning decision: conv geometry, input shape, residual.
// The last field: 1 with a residual, plus 2 with an upsampled input part.
static std::string tune_key(const ConvPlan* p, const sy_tensor* x, const sy_tensor* res, int ku) {
  char k[160];
  snprintf(k, sizeof k, "%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d,%d:%d,%d,%d,%d", p->oc, p->ic, p->kh, p->kw, p->sh,
           p->sw, p->pt, p->pl, p->pb, p->pr, p->dh, p->dw, p->groups, p->silu, p->up2, x->n, x->h, x->w,
           (res ? 1 : 0) + (ku > 0 ? 2 : 0));
  return k;
}

// What the tile numbers of a saved table mean: the form lists' sizes and bases.
static std::string tune_header() {
  char h[80];
  snprintf(h, sizeof h, "simdyolo_hip tune3 %d %d %d %d %d %d", kNumTiles, kPwBase, kX3Base, x3_num_tiles(), kC3Base,
           c3_num_forms());
  return h;
}

int tune_save(const sy_ctx* ctx, const char* path) {
  FILE* f = fopen(path, "w");
  SY_CHECK(f != nullptr, SY_EINVAL, "cannot open %s for writing", path);
  fprintf(f, "%s\n", tune_header().c_str());
  for (const auto& kv : ctx->tune_table)
    fprintf(f, "%s %d %d %d\n", kv.first.c_str(), kv.second.algo, kv.second.tile, kv.second.split);
  const bool ok = fclose(f) == 0;
  SY_CHECK(ok, SY_EINVAL, "writing %s failed", path);
  return SY_OK;
}

int tune_load(sy_ctx* ctx, const char* path) {
  FILE* f = fopen(path, "r");
  SY_CHECK(f != nullptr, SY_EINVAL, "cannot open %s", path);
  char line[128] = "";
  const bool head = fgets(line, sizeof line, f) != nullptr;
  line[strcspn(line, "\r\n")] = 0;
  if (!head || line != tune_header()) {
    fclose(f);
    SY_CHECK(false, SY_EINVAL, "%s is not a tuning table of this library build", path);
  }
  char key[160];
  int algo, tile, split;
  std::map<std::string, ConvChoice> table;
  while (fscanf(f, "%159s %d %d %d", key, &algo, &tile, &split) == 4) table[key] = ConvChoice{algo, tile, split};
  fclose(f);
  for (const auto& kv : table) ctx->tune_table[kv.first] = kv.second;
  return SY_OK;
}

// The (algorithm, tile) candidates the tuner times for this conv and input
// view; empty when the conv keeps its routing rule.
static std::vector<ConvChoice> conv_candidates_all(const ConvPlan* p, const sy_tensor* x) {
  std::vector<ConvChoice> cand;
  const bool nchw = x->layout == SY_LAYOUT_NCHW;
  const bool aligned = ((uintptr_t)x->data & 15) == 0 && (x->ldc & 3) == 0;
  if (p->algo == kDepthwise) {
    // 3x3 stride-1 depthwise on 16-byte views: the register kernel (0), the
    // LDS-tile kernel (1) and the column kernel with 4- or 8-row segments.
    const bool v4 = (p->oc & 3) == 0 && aligned;
    if (v4 && p->kh == 3 && p->kw == 3 && p->sh == 1 && p->sw == 1 && p->pt == 1 && p->pl == 1 && p->dh == 1 &&
        p->dw == 1)
      for (int t = 0; t < 4; ++t) cand.push_back(ConvChoice{kDepthwise, t});
    return cand;
  }
  if (p->algo == kDirect || nchw || !aligned) return cand;
  const bool rows1x1 = p->kh == 1 && p->kw == 1 && p->sh == 1 && p->sw == 1 && p->pt == 0 && p->pl == 0 &&
                       p->pb == 0 && p->pr == 0;
  int oh = 0, ow = 0;
  conv_out_size(p, x->h, x->w, &oh, &ow);
  const long long M = (long long)x->n * oh * ow;
  const int K = p->kh * p->kw * p->ic;
  // The f16-split kernels.  Where 64 x 64 output tiles fill the CUs twice over,
  // no other candidate is timed: of 98 such layers of YOLOv8n, s and m at 640
  // (batch 1 to 32) they are the fastest at 97, by 1.02 to 2.5 times (1x1 384 ->
  // 128 at 40 x 40, batch 32: 30 us against 58; 3x3 64 -> 64 at 80 x 80: 52 against
  // 73; 3x3 stride 2 64 -> 128: 38 against 82), and 1% behind at one (1x1 48 -> 32
  // at 160 x 160, bound by memory).  Smaller grids and shallow products, where the
  // in-workgroup split-K and row kernels can win, time all.
  if (conv_supports(p, kIgemm) && p->finite && M * p->oc < (1LL << 40)) {
    for (int i = 0; i < x3_num_tiles(); ++i) cand.push_back(ConvChoice{kIgemm, kX3Base + i});
    const long long wide = (M + 63) / 64 * ((p->oc + 63) / 64);
    if (conv3x3_patch(p)) {
      // Forms whose waves share out the channel groups: only while the plain
      // ones leave most CUs idle, and with a group for most of the waves.
      for (int i = 0; i < c3_num_forms(); ++i) {
        const int kw = c3_form_groups(i);
        if (kw == 1 || (wide < 256 && (p->ic + 15) / 16 * 4 >= 3 * kw)) cand.push_back(ConvChoice{kIgemm, kC3Base + i});
      }
    }
    if (wide >= 512 && K >= 64 && p->ic >= 32) return cand;
  }
  for (int algo : {(int)kIgemm, (int)kWinograd3}) {
    if (!conv_supports(p, algo)) continue;
    for (int t = 0; t < kNumTiles; ++t) {
      if (!gemm_tile_ok(t, algo == kWinograd3 || rows1x1)) continue;
      // The 96-wide tiles serve convs with 80-odd output channels (a detect
      // head's class branch); as Winograd plane GEMMs they win the timed
      // launch at batch 1 but cost the three-kernel path's extra launches
      // in the captured forward.
      if (algo == kWinograd3 && kTiles[t].bn == 96) continue;
      // 32-column tiles re-read a plane's V once per 32 output channels (a
      // 128x32 plane GEMM moved 3.8x its algorithmic bytes in YOLOv8n's
      // batch-32 forward): for wider outputs they are not offered.
      if (algo == kWinograd3 && kTiles[t].bn == 32 && p->oc > 32) continue;
      cand.push_back(ConvChoice{algo, t});
      // Split K when the tile grid leaves most of the GPU idle (small
      // batches): two to sixteen workgroups per output tile, each at least
      // two K tiles deep.
      const TileCfg& c = kTiles[t];
      const long long grid = (M + c.bm - 1) / c.bm * ((p->oc + c.bn - 1) / c.bn);
      // The partials must fit what conv_scratch_bytes reserves for this
      // shape: a branch stream's scratch is sized from it before capture.
      if (algo == kIgemm && !p->up2 && grid * 2 <= kSplitGridMax && t == 2)
        for (int i = 0; i < 3; ++i)
          if ((long long)K >= 2LL * (4 << i) * 16 && (rows1x1 || p->ic % 16 == 0) &&
              ((long long)M * x->ldc < (1LL << 31))) {
            cand.push_back(ConvChoice{algo, kKsBase + i});
            cand.push_back(ConvChoice{algo, kKs16Base + i});
          }
      if (algo == kIgemm && !p->up2 && grid * 2 <= kSplitGridMax)
        for (int sp = 2; sp <= 16; sp *= 2) {
          int kchunk = 0, S = 1;
          split_chunks(K, c.bk, sp, &kchunk, &S);
          const long long ldp = (p->oc + c.bn - 1) / c.bn * c.bn;
          const size_t part = (size_t)S * M * ldp * sizeof(float);
          if (S == sp && kchunk >= 2 * c.bk && (long long)S * M * ldp <= kSplitMaxFloats &&
              part <= conv_scratch_bytes(p, x->n, x->h, x->w))
            cand.push_back(ConvChoice{algo, t, sp});
        }
    }
    // Weight-stationary row GEMM: A rows are the input pixels (1x1) or the
    // transformed tiles (Winograd, K = ic, 16-byte aligned scratch).
    if (algo == kWinograd3 || (rows1x1 && aligned))
      for (int nw = 1; nw <= 4; ++nw)
        if (pw_fits(p->ic, nw) && (nw == 1 || 32 * (nw - 1) < p->oc)) cand.push_back(ConvChoice{algo, kPwBase + nw - 1});
  }
  if (conv_supports(p, kIgemm) && p->ic == 16 && (p->oc == 16 || p->oc == 32) && p->kh == 3 && p->kw == 3 &&
      p->sh == p->sw && (p->sh == 1 || p->sh == 2) && p->dh == 1 && p->dw == 1 && !p->up2 && aligned)
    cand.push_back(ConvChoice{kIgemm, kC16Tile});
  if (conv_supports(p, kWinograd) && p->ic >= 8 && fused_wino_fits(x))
    for (int v = 0; v < kFusedForms; ++v)
      if (v != 2 || p->oc > 32) cand.push_back(ConvChoice{kWinograd, v});
  if (conv_supports(p, kWinograd2))
    for (int v = 0; v < kGoVariants; ++v) cand.push_back(ConvChoice{kWinograd2, v});
  return cand;
}

// With an upsampled input part of ku channels (conv_run_upsampled) only the
// plain implicit-GEMM tiles whose K tile divides ku, split or not, apply.
static std::vector<ConvChoice> conv_candidates(const ConvPlan* p, const sy_tensor* x, int ku) {
  std::vector<ConvChoice> cand = conv_candidates_all(p, x);
  if (ku == 0) return cand;
  std::vector<ConvChoice> keep;
  for (const ConvChoice& c : cand)
    if (c.algo == kIgemm && (is_x3_tile(c.tile) ? ku % 32 == 0
                                                : c.tile >= 0 && c.tile < kNumTiles && ku % kTiles[c.tile].bk == 0))
      keep.push_back(c);
  return keep;
}

static int up_channels(const sy_ctx* ctx) { return ctx->up_src ? ctx->up_src->c : 0; }

static int conv_tune(sy_ctx* ctx, ConvPlan* p, const sy_tensor* x, const sy_tensor* y, const sy_tensor* res,
                     ConvChoice* out) {
  const std::vector<ConvChoice> cand = conv_candidates(p, x, up_channels(ctx));
  if (cand.size() <= 1) {
    *out = cand.empty() ? ConvChoice{p->algo, -1} : cand[0];
    return SY_OK;
  }
  const bool prof = ctx->profiling;
  ctx->profiling = false;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = SY_OK;
  float best = 1e30f;
  ConvChoice pick{p->algo, -1};
  if (hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
    rc = SY_EDEVICE;
    set_error("hipEventCreate failed");
  }
  // Rounds over all candidates, each timed over three launches and kept by its
  // best: the clock moves with the load, so candidates next to each other in
  // time are compared, not the first with the last.  After the first round only
  // those within 30% of the best go on.
  constexpr int kReps = 3, kRounds = 4;
  std::vector<float> ms(cand.size(), 1e30f);
  for (int round = 0; rc == SY_OK && round < kRounds; ++round) {
    const float limit = 1.3f * best;
    for (size_t i = 0; rc == SY_OK && i < cand.size(); ++i) {
      if (round > 0 && ms[i] > limit) continue;
      if (round == 0) rc = conv_exec(ctx, p, x, y, res, cand[i]);  // warm: packs weights, touches caches
      if (rc == SY_OK && hipEventRecord(e0, ctx->stream) != hipSuccess) rc = SY_EDEVICE;
      for (int r = 0; rc == SY_OK && r < kReps; ++r) rc = conv_exec(ctx, p, x, y, res, cand[i]);
      if (rc != SY_OK) break;
      float w = 0.f;
      if (hipEventRecord(e1, ctx->stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
          hipEventElapsedTime(&w, e0, e1) != hipSuccess) {
        rc = SY_EDEVICE;
        set_error("event timing failed while tuning a convolution");
        break;
      }
      ms[i] = std::min(ms[i], w);
      if (ms[i] < best) {
        best = ms[i];
        pick = cand[i];
      }
    }
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  ctx->profiling = prof;
  SY_TRY(rc);
  *out = pick;
  return SY_OK;
}

bool views_overlap(const sy_tensor* a, const sy_tensor* b) {
  auto span = [](const sy_tensor* t) {
    const size_t px = (size_t)t->n * t->h * t->w;
    const size_t floats = t->layout == SY_LAYOUT_NCHW ? px * t->c : (px - 1) * t->ldc + t->c;
    const uintptr_t lo = (uintptr_t)t->data;
    return std::make_pair(lo, lo + floats * sizeof(float));
  };
  const auto ra = span(a), rb = span(b);
  if (!(ra.first < rb.second && rb.first < ra.second)) return false;
  if (a->layout != SY_LAYOUT_NHWC || b->layout != SY_LAYOUT_NHWC || a->ldc != b->ldc) return true;
  // Channel slices of one NHWC buffer (same pixel stride L): every element of
  // a view sits at a float address whose residue mod L falls in its channel
  // arc; disjoint arcs on that circle mean disjoint views.
  const long long L = a->ldc;
  if (a->c >= L || b->c >= L) return true;
  const long long ra0 = (long long)((uintptr_t)a->data / sizeof(float) % (uintptr_t)L);
  const long long rb0 = (long long)((uintptr_t)b->data / sizeof(float) % (uintptr_t)L);
  auto within = [L](long long x, long long start, long long len) { return ((x - start) % L + L) % L < len; };
  return within(ra0, rb0, b->c) || within(rb0, ra0, a->c);
}

int conv_run(sy_ctx* ctx, ConvPlan* p, const sy_tensor* x, const sy_tensor* y, const sy_tensor* res) {
  ConvChoice ch{p->algo, -1};
  // Timing candidates re-runs the conv; an output that overlaps one of its
  // inputs (an in-place residual y += f(x)) would then read its own result.
  const bool rerunnable = x && y && !views_overlap(x, y) && !(res && views_overlap(res, y));
  const int ku = up_channels(ctx);
  if (!p->user_algo && rerunnable && autotune_enabled()) {
    const auto key = std::make_tuple(x->n, x->h, x->w, (res ? 1 : 0) + (ku > 0 ? 2 : 0));
    auto it = p->tuned.find(key);
    if (it != p->tuned.end()) {
      ch = it->second;
    } else {
      // A choice recorded for the same geometry and input shape (this
      // context's earlier tuning or a loaded table) is reused when it is one
      // of this conv's candidates; otherwise the candidates are timed.
      const std::string tkey = tune_key(p, x, res, ku);
      auto rec = ctx->tune_table.find(tkey);
      bool reused = false;
      if (rec != ctx->tune_table.end()) {
        for (const ConvChoice& c : conv_candidates(p, x, ku))
          if (c.algo == rec->second.algo && c.tile == rec->second.tile && c.split == rec->second.split)
            reused = true;
      }
      if (reused && ctx->capturing && !weights_packed(p, rec->second.algo, rec->second.tile)) {
        // A first run inside a capture, which cannot upload: the routing rule,
        // whose weights are there from the start, for this call alone.
      } else if (reused) {
        ch = rec->second;
        p->tuned[key] = ch;
      } else if (!ctx->capturing) {
        // Validate the views before timing candidates on them.
        SY_TRY(conv_exec(ctx, p, x, y, res, ch));
        SY_TRY(conv_tune(ctx, p, x, y, res, &ch));
        p->tuned[key] = ch;
        ctx->tune_table[tkey] = ch;
      }
    }
  }
  return conv_exec(ctx, p, x, y, res, ch);
}

// Resolves ctx->up_src for the duration of one conv and restores it.
struct UpSource {
  sy_ctx* ctx;
  const sy_tensor* saved;
  UpSource(sy_ctx* c, const sy_tensor* xu) : ctx(c), saved(c->up_src) { ctx->up_src = xu; }
  ~UpSource() { ctx->up_src = saved; }
};

int conv_run_upsampled(sy_ctx* ctx, ConvPlan* p, const sy_tensor* xu, const sy_tensor* x, const sy_tensor* y,
                       const sy_tensor* res) {
  SY_CHECK(xu && x, SY_EINVAL, "null conv input");
  SY_TRY(check_view(xu, "upsampled conv source"));
  SY_TRY(check_view(x, "conv input"));
  SY_CHECK(xu->layout == SY_LAYOUT_NHWC && x->layout == SY_LAYOUT_NHWC && xu->n == x->n && 2 * xu->h == x->h &&
               2 * xu->w == x->w && xu->c > 0 && xu->c < x->c,
           SY_EINVAL, "the upsampled source must be a half-size NHWC view of the input's leading channels");
  // The kernel's form: a plain 1x1 implicit GEMM whose K tiles (16 or 32
  // channels) never straddle the two parts, 16-byte views, and an upsampled
  // part that the tuner may route to no other kernel.
  const bool fits = p->algo == kIgemm && p->kh == 1 && p->kw == 1 && p->sh == 1 && p->sw == 1 && p->pt == 0 &&
                    p->pl == 0 && p->pb == 0 && p->pr == 0 && p->groups == 1 && !p->up2 && !p->user_algo &&
                    xu->c % 32 == 0 && ((uintptr_t)xu->data & 15) == 0 && (xu->ldc & 3) == 0 &&
                    ((uintptr_t)x->data & 15) == 0 && (x->ldc & 3) == 0 &&
                    (long long)xu->n * xu->h * xu->w * xu->ldc < (1LL << 40);
  if (!fits) {
    sy_tensor head = *x;
    head.c = xu->c;
    SY_TRY(op_resize_nearest(ctx, xu, &head));
    return conv_run(ctx, p, x, y, res);
  }
  UpSource up(ctx, xu);
  return conv_run(ctx, p, x, y, res);
}

}  // namespace sy
