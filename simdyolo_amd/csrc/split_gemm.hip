// Float32 implicit GEMM on the f16 matrix cores, with error-corrected products
// (Ootomo and Yokota, 2022).
//
// Every float32 operand, scaled by a power of two (exact), is written as
// hi + lo / 2048 with hi = f16(v) and lo = f16(2048 (v - hi)): v - hi is exact
// and lo keeps 11 more significand bits, so the pair is within 2^-23 of v.  A
// product is three f16 products, each exact in the float32 accumulators:
// hi hi in one, hi lo + lo hi (2048 times too large) in the other.  The lo lo
// left out is below 2^-22 of it, with either sign.  Where every operand has its
// pair in full the result is closer to float64 than the float32 MFMA's, whose
// accumulator rounds once per two terms: the main one here rounds once per
// sixteen.
//
// Scales.  Weights: one power of two per output channel, chosen when they are
// packed.  Activations: one per workgroup, from the largest magnitude of the
// K tiles seen so far: 2^2 <= largest < 2^15 after scaling, so f16 does not
// overflow.  The first guess, 16, suits largest values from 0.25 to 2047; a K
// tile that leaves the range is split again with another scale (into
// [2^11, 2^12)) and the accumulators take the exact ratio.
//
// Range.  f16 ends at 2^-24: the pair of a scaled value is within 2^-23 of it down
// to 2^-13, and within 2^-36 absolute below.  So that one row (pixel) does not pay
// for another's magnitude, a workgroup in which a row has nonzero elements but
// none of 2^-13 or more, or that reads a value of 2^16 or more, computes its tile
// again in plain float32 from the same operands, at about the speed of the
// float32 tiles.  What is left is, per element, 2^-23 of its row's largest.
//
// Why: v_mfma_f32_32x32x16_f16 multiplies 16 K steps in 32 cycles per SIMD,
// three of them replace eight 64-cycle v_mfma_f32_32x32x2f32 (measured raw
// issue: 2,090 against 149 TFLOP/s, so 697 TFLOP/s of float32 work).  The
// split costs four VALU operations per A element and K tile, beside the
// MFMAs of other waves; B is split once, when the weights are packed.  At batch
// 32, against the float32 tiles: 1x1 384 -> 128 at 40 x 40 58 -> 30 us (105 MB
// at 3.6 TB/s), 3x3 stride 2 64 -> 128 at 80 x 80 82 -> 38 us.
//
// Non-finite operands: infinities take the plain path too, and convolutions with
// non-finite weights are not routed here: infinities and NaN propagate as they do
// in the float32 kernels.
#include <cmath>
#include <cstring>
#include <string>

#include "igemm.h"
#include "split.h"

namespace sy {

// Four zeros: the source of elements outside the operand.
__device__ const float kX3Zeros[4] = {0.f, 0.f, 0.f, 0.f};

// A wave's blocks in plain float32, on the float32 matrix cores, operands straight
// from memory.  Lane half h takes k = 8 q + 4 h .. + 3 of its row and column.
template <int MODE, int TM, int TN>
__device__ __forceinline__ void x3_plain(const IgemmArgs& a, int row0, int col0, int lane, f32x16 (&acc)[TM][TN]) {
  const int half = lane >> 5, r32 = lane & 31;
  int m[TM], n[TM], oy[TM], ox[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    m[i] = row0 + i * 32 + r32;
    const int t = m[i] / a.OW;
    ox[i] = m[i] - t * a.OW;
    n[i] = t / a.OH;
    oy[i] = t - n[i] * a.OH;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  }
  const _Float16* w[TN];
  float ws[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = col0 + j * 32 + r32;
    w[j] = (const _Float16*)a.w3 + ((long long)(col >> 5) * a.nkt * kX3Units + (col & 31)) * 8;
    ws[j] = a.w3s[col];
  }
  for (int k8 = 0; k8 < a.K; k8 += 8) {
    const int k = k8 + 4 * half;
    const int tap = k / a.IC, ic = k - tap * a.IC, ky = tap / a.KW, kx = tap - ky * a.KW;
    f32x4 xv[TM], wv[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      bool ok = m[i] < a.M && k < a.K;
      const float* x;
      if (MODE == 2) {
        x = a.x + (long long)m[i] * a.ldx + k;
      } else if (MODE == 3) {
        x = k < a.ku ? a.xu + ((long long)(n[i] * (a.H >> 1) + (oy[i] >> 1)) * (a.W >> 1) + (ox[i] >> 1)) * a.ldxu + k
                     : a.x + (long long)m[i] * a.ldx + (k - a.ku);
      } else {
        const int iy = oy[i] * a.SH - a.PH + ky * a.DH, ix = ox[i] * a.SW - a.PW + kx * a.DW;
        ok = ok && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
        x = a.x + (((long long)n[i] * a.H + iy) * a.W + ix) * a.ldx + ic;
      }
      xv[i] = *(const f32x4*)(ok ? x : kX3Zeros);
    }
#pragma unroll
    for (int j = 0; j < TN; ++j)
      wv[j] = join4(w[j] + ((long long)(k >> 5) * kX3Units + ((k >> 4) & 1) * 128 + ((k >> 3) & 1) * 32) * 8 + (k & 7),
                    ws[j]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[i][e], wv[j][e], acc[i][j], 0, 0, 0);
  }
}

// One BM x BN tile per workgroup, K tiles of 32.  A is gathered from the
// NHWC input (MODE as in igemm_kernel), split in registers and stored to LDS
// as two f16 planes; B arrives split, in MFMA operand order.  The next K
// tile's loads are in flight while the current one multiplies; LDS holds one
// K tile (two barriers per tile), and the other workgroups on the CU
// multiply while one stages.
template <int MODE, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(WM* WN * 64, (BM / WM) * (BN / WN) >= 3072   ? 2
                                          : (BM / WM) * (BN / WN) >= 2048 ? 3
                                                                          : 4) void x3_kernel(const IgemmArgs a,
                                                                                              int nblk) {
  constexpr int NT = WM * WN * 64, NW = WM * WN;
  constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
  constexpr int LDA = 40;  // halves per A row: 16-byte reads of 32 rows fall in distinct banks
  constexpr int A_IT = BM * 8 / NT;
  constexpr int BU = BN / 32 * kX3Units;  // 16-byte units of a B tile
  constexpr int B_IT = (BU + NT - 1) / NT;
  static_assert(BM * 8 % NT == 0, "every thread stages whole rows");
  __shared__ __attribute__((aligned(16))) unsigned short As[2][BM][LDA];
  __shared__ __attribute__((aligned(16))) u32x4 Bs[BU];
  __shared__ float red[NW];
  __shared__ int low;  // a row lies below the range of the workgroup's scale

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  if (tid == 0) low = 0;
  const int wm = wid / WN, wn = wid % WN;
  // Each XCD (workgroups L, L + 8, ...) takes a contiguous run of tiles, a
  // row block's column blocks next to each other: they share its A rows in
  // that XCD's L2.
  const int G = gridDim.x, L = blockIdx.x;
  const int xcd = L & 7, q8 = G >> 3, rem = G & 7;
  const int P = xcd * q8 + (xcd < rem ? xcd : rem) + (L >> 3);
  const int m0 = P / nblk * BM, n0 = (P % nblk) * BN;
  const int quad = tid & 7, nkt = a.nkt;

  const float* a_img[A_IT];
  const float* a_up[A_IT];
  int a_iy[A_IT], a_ix[A_IT], a_pix[A_IT];
  bool a_ok[A_IT];
#pragma unroll
  for (int i = 0; i < A_IT; ++i) {
    const int m = m0 + (tid + i * NT) / 8;
    a_ok[i] = m < a.M;
    const int mm = a_ok[i] ? m : 0;
    if (MODE == 2 || MODE == 3) {
      a_img[i] = a.x + (long long)mm * a.ldx + quad * 4;
      if (MODE == 3) {
        const int ox = mm % a.W, t = mm / a.W, oy = t % a.H, n = t / a.H;
        a_up[i] = a.xu + ((long long)(n * (a.H >> 1) + (oy >> 1)) * (a.W >> 1) + (ox >> 1)) * a.ldxu + quad * 4;
      }
    } else {
      const int ox = mm % a.OW, t = mm / a.OW, oy = t % a.OH, n = t / a.OH;
      a_iy[i] = oy * a.SH - a.PH;
      a_ix[i] = ox * a.SW - a.PW;
      a_pix[i] = (a_iy[i] * a.W + a_ix[i]) * a.ldx;
      a_img[i] = a.x + (long long)n * a.H * a.W * a.ldx;
    }
  }
  int t_ic = 0, t_ky = 0, t_kx = 0;  // MODE 1: tap and channel of the next K tile (uniform)
  const u32x4* bp[B_IT];
#pragma unroll
  for (int i = 0; i < B_IT; ++i) {
    const int u = tid + i * NT;
    bp[i] = (const u32x4*)a.w3 + ((long long)(n0 / 32 + u / kX3Units) * nkt) * kX3Units + u % kX3Units;
  }

  f32x4 ar[A_IT];
  u32x4 br[B_IT];
  unsigned seen[A_IT] = {};  // hi parts of the thread's share of its rows, or'ed
  // Branch-free loads: an element outside the operand is read from the zeros.
  auto gload = [&](int kt) {
    const int k0 = kt * 32;
    if (MODE == 2) {
      const bool kok = k0 + quad * 4 < a.K;
#pragma unroll
      for (int i = 0; i < A_IT; ++i) ar[i] = *(const f32x4*)(a_ok[i] && kok ? a_img[i] + k0 : kX3Zeros);
    } else if (MODE == 3) {
      const bool up = k0 < a.ku, kok = k0 + quad * 4 < a.K;
#pragma unroll
      for (int i = 0; i < A_IT; ++i)
        ar[i] = *(const f32x4*)(a_ok[i] && kok ? (up ? a_up[i] + k0 : a_img[i] + (k0 - a.ku)) : kX3Zeros);
    } else if (MODE == 1) {
      const int dy = t_ky * a.DH, dx = t_kx * a.DW;
      const int off = (dy * a.W + dx) * a.ldx + t_ic + quad * 4;
#pragma unroll
      for (int i = 0; i < A_IT; ++i) {
        const bool ok = a_ok[i] && (unsigned)(a_iy[i] + dy) < (unsigned)a.H && (unsigned)(a_ix[i] + dx) < (unsigned)a.W;
        ar[i] = *(const f32x4*)(ok ? a_img[i] + (a_pix[i] + off) : kX3Zeros);
      }
      t_ic += 32;
      if (t_ic == a.IC) {
        t_ic = 0;
        if (++t_kx == a.KW) {
          t_kx = 0;
          ++t_ky;
        }
      }
    } else {
      const int k = k0 + quad * 4;
      const int tap = k / a.IC, ic = k - tap * a.IC, ky = tap / a.KW, kx = tap - (tap / a.KW) * a.KW;
#pragma unroll
      for (int i = 0; i < A_IT; ++i) {
        const int iy = a_iy[i] + ky * a.DH, ix = a_ix[i] + kx * a.DW;
        const bool ok = a_ok[i] && k < a.K && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
        ar[i] = *(const f32x4*)(ok ? a_img[i] + (((long long)iy * a.W + ix) * a.ldx + ic) : kX3Zeros);
      }
    }
#pragma unroll
    for (int i = 0; i < B_IT; ++i)
      if (BU % NT == 0 || tid + i * NT < BU) br[i] = bp[i][(long long)kt * kX3Units];
  };
  auto stage = [&](float s) {
#pragma unroll
    for (int i = 0; i < A_IT; ++i) {
      u32x2 hi, lo;
      split4(ar[i], s, hi, lo);
      seen[i] |= hi[0] | hi[1];
      const int row = (tid + i * NT) / 8;
      *(u32x2*)&As[0][row][quad * 4] = hi;
      *(u32x2*)&As[1][row][quad * 4] = lo;
    }
  };

  f32x16 acc[TM][TN], crs[TM][TN];  // sums of hi hi, and of hi lo + lo hi
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = crs[i][j][r] = 0.f;
  const int half = lane >> 5, r32 = lane & 31;
  int se = kSplitExpGuess;
  float big = 0.f;  // largest magnitude so far

  gload(0);
  for (int kt = 0; kt < nkt; ++kt) {
    if (kt > 0) __syncthreads();  // the last tile's reads are done
    float m = 0.f;
#pragma unroll
    for (int i = 0; i < A_IT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) m = fmaxf(m, __builtin_fabsf(ar[i][e]));
    m = wave_max63(m);
    if (lane == 63) red[wid] = m;
    stage(exp_float(se));
#pragma unroll
    for (int i = 0; i < B_IT; ++i)
      if (BU % NT == 0 || tid + i * NT < BU) Bs[tid + i * NT] = br[i];
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) big = fmaxf(big, red[w]);
    int ne;
    if (!scale_fits(big, se, &ne)) {
      if (kt > 0) rescale<TM, TN>(se, ne, acc, crs);
      se = ne;
#pragma unroll
      for (int i = 0; i < A_IT; ++i) seen[i] = 0;  // what counts is the rows under this scale
      stage(exp_float(se));
      __syncthreads();
    }
    if (kt + 1 < nkt) gload(kt + 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      f16x8 av[TM][2], bv[TN][2];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          av[i][p] = *(const f16x8*)&As[p][wm * (BM / WM) + i * 32 + r32][ks * 16 + half * 8];
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          bv[j][p] = __builtin_bit_cast(f16x8, Bs[(wn * TN + j) * kX3Units + (ks * 2 + p) * 64 + lane]);
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          crs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i][1], bv[j][0], crs[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i][0], bv[j][0], acc[i][j], 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          crs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[i][0], bv[j][1], crs[i][j], 0, 0, 0);
    }
  }

  // Rows with no element in the pairs' full range, unless they are all zero.
  unsigned below = 0;
#pragma unroll
  for (int i = 0; i < A_IT; ++i) below |= (a_ok[i] && !(or_lanes<8>(seen[i]) & kSplitFull)) << i;
  if (__any(below != 0)) {
    unsigned nz[A_IT] = {};
    t_ic = t_ky = t_kx = 0;
    for (int kt = 0; kt < nkt; ++kt) {
      gload(kt);
#pragma unroll
      for (int i = 0; i < A_IT; ++i) nz[i] |= magnitude_bits(ar[i]);
    }
#pragma unroll
    for (int i = 0; i < A_IT; ++i)
      if ((below >> i & 1) && nz[i]) low = 1;
  }
  __syncthreads();

  const int row0 = m0 + wm * (BM / WM), col0 = n0 + wn * (BN / WN);
  if (big >= kSplitHuge || low) {
    x3_plain<MODE, TM, TN>(a, row0, col0, lane, acc);
  } else {
    float ws[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) ws[j] = a.w3s[col0 + j * 32 + r32];
    unscale<TM, TN>(ws, se, acc, crs);
  }
  if (MODE == 2 && a.shuf > 0)
    store_shuf<TM, TN>(a, a.y, acc, row0 + 4 * half, col0 + r32);
  else
    store_acc<TM, TN>(a, a.y, acc, row0 + 4 * half, col0 + r32);
}

#define SY_X3_LIST(X) \
  X(0, 128, 128, 2, 2) X(1, 64, 64, 2, 2) X(2, 64, 128, 2, 2) X(3, 128, 32, 4, 1) X(4, 64, 32, 2, 1)

#define SY_X3_CFG(i, bm, bn, wm, wn) {bm, bn, wm, wn},
const X3Tile kX3Tiles[] = {SY_X3_LIST(SY_X3_CFG)};
#undef SY_X3_CFG
static constexpr int kNumX3 = sizeof(kX3Tiles) / sizeof(kX3Tiles[0]);
int x3_num_tiles() { return kNumX3; }

const char* x3_name(int t, int mode) {
  struct Names {
    std::string n[4][kNumX3];
    Names() {
      for (int m = 0; m < 4; ++m)
        for (int i = 0; i < kNumX3; ++i) {
          const X3Tile& c = kX3Tiles[i];
          char buf[64];
          snprintf(buf, sizeof buf, "igemm_m%d_x3_%dx%d_%d%d", m, c.bm, c.bn, c.wm, c.wn);
          n[m][i] = buf;
        }
    }
  };
  static const Names names;
  return names.n[mode][t - kX3Base].c_str();
}

// Nearest f16 (ties to even) of a float below 65520 in magnitude, and back.
// Both branches are computed and one taken, so that loops vectorise.
static inline uint32_t f16_bits(float v) {
  uint32_t u, m;
  std::memcpy(&u, &v, 4);
  const uint32_t sign = (u >> 16) & 0x8000u;
  u &= 0x7fffffffu;
  // Below 2^-14: a multiple of 2^-24, rounded in the float addition.
  const float s = std::fabs(v) * 0x1p24f + 0x1p23f;
  std::memcpy(&m, &s, 4);
  const uint32_t n = (u + 0xfffu + ((u >> 13) & 1) - 0x38000000u) >> 13;
  return sign | (u < 0x38800000u ? m & 0x7fffffu : n);
}
static inline float f16_value(uint32_t h) {
  const uint32_t u = h & 0x7fffu, n = (u << 13) + 0x38000000u;
  float v;
  std::memcpy(&v, &n, 4);
  v = u < 0x400u ? (float)(int)u * 0x1p-24f : v;
  return h & 0x8000u ? -v : v;
}

void x3_split(const float* v, int n, float scale, uint16_t* hi, uint16_t* lo) {
  for (int i = 0; i < n; ++i) {
    const float s = v[i] * scale;
    const uint32_t h = f16_bits(s);
    hi[i] = (uint16_t)h;
    lo[i] = (uint16_t)f16_bits((s - f16_value(h)) * 2048.f);
  }
}

float x3_weight_scale(float largest) {
  if (!(largest > 0.f)) return 1.f;
  int e = 0;
  (void)std::frexp(largest, &e);  // largest in [2^(e-1), 2^e)
  return std::ldexp(1.f, std::min(12 - e, 120));
}

int launch_x3(sy_ctx* ctx, int t, int mode, const IgemmArgs& a) {
  const X3Tile& c = kX3Tiles[t - kX3Base];
  const int nblk = (a.OC + c.bn - 1) / c.bn;
  const long long grid = (long long)((a.M + c.bm - 1) / c.bm) * nblk;
  SY_CHECK(grid < (1LL << 31), SY_EUNSUPPORTED, "convolution grid too large");
  void (*k)(const IgemmArgs, int) = nullptr;
#define SY_X3_CASE(i, bm, bn, wm, wn)                                                        \
  if (t - kX3Base == i)                                                                       \
    k = mode == 0   ? x3_kernel<0, bm, bn, wm, wn>                                            \
        : mode == 1 ? x3_kernel<1, bm, bn, wm, wn>                                            \
        : mode == 2 ? x3_kernel<2, bm, bn, wm, wn>                                            \
                    : x3_kernel<3, bm, bn, wm, wn>;
  SY_X3_LIST(SY_X3_CASE)
#undef SY_X3_CASE
  SY_CHECK(k != nullptr, SY_EINVAL, "no split GEMM tile %d", t);
  hipLaunchKernelGGL(k, dim3((unsigned)grid), dim3(c.wm * c.wn * 64), 0, ctx->stream, a, nblk);
  return SY_OK;
}

}  // namespace sy
