// Shared by the implicit-GEMM kernels: operand description and epilogues.
#pragma once

#include "sy_internal.h"

namespace sy {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ __forceinline__ float silu_f(float v) { return v / (1.0f + __expf(-v)); }
// SiLU with the hardware reciprocal (within 1 ulp of the division) for GEMM
// epilogues, where the IEEE division sequence is a large share of the VALU.
__device__ __forceinline__ float silu_fast(float v) { return v * __builtin_amdgcn_rcpf(1.0f + __expf(-v)); }

// ------------------------------------------------------------ implicit GEMM

struct IgemmArgs {
  const float* x;
  int N, H, W, IC, ldx;
  const float* w;
  int Kp;
  const float* bias;
  const float* res;
  int ldr;
  float* y;
  int OH, OW, OC, ldy;
  int KH, KW, SH, SW, PH, PW, DH, DW;
  int K, M, silu;
  long long xb, wb, yb;  // per-blockIdx.z strides (floats) for batched GEMMs
  int Nb, bguard;        // B rows present; check B reads against Nb and K
  int shuf = 0;          // > 0: column q * shuf + o goes to pixel (2y + q/2, 2x + q%2), channel o
  // Split K: workgroup z sums k in [z * kchunk, (z + 1) * kchunk) and stores
  // the raw partial tile to part[z][m][ldp]; splitk_reduce_kernel finishes.
  float* part = nullptr;
  int kchunk = 0, ldp = 0;
  // MODE 3 (1x1 over concat(upsample2x(xu), x)): K columns [0, ku) of row
  // (n, oy, ox) come from xu's pixel (n, oy / 2, ox / 2) of an (H/2) x (W/2)
  // image, columns [ku, K) from x's row (x points at that part's first
  // channel).  ku is a whole number of K tiles.
  const float* xu = nullptr;
  int ldxu = 0, ku = 0;
  const void* w3 = nullptr;  // split weights (split_gemm.hip) when the tile reads them
  const float* w3s = nullptr;  // per column: 1 / their scale
  int nkt = 0;               // their K tiles of 32
};

// Epilogue of a GEMM tile: y = [res +] act(acc + bias) for the 32x32 MFMA
// blocks of one wave.  rbase is the wave's first output row (plus the lane
// half's 4-row offset), col0 its first column plus the lane's column.  D
// layout of the 32x32 MFMA: lane holds column (lane & 31) and rows
// 8*(r/4) + 4*(lane/32) + (r%4) for r = 0..15.  Every bias and residual
// value is loaded before the first store: a wait for a load also waits for
// the stores issued before it, so interleaving them would serialise the
// stores' round trips.
template <int TM, int TN>
__device__ __forceinline__ void store_acc(const IgemmArgs& a, float* __restrict__ y, const f32x16 (&acc)[TM][TN],
                                          int rbase, int col0) {
  float bv[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) bv[j] = (a.bias && col0 + j * 32 < a.OC) ? a.bias[col0 + j * 32] : 0.f;
  // A wave tile wholly inside the output (every row below M, every column
  // below OC) stores without per-element tests: one branch for the tile
  // instead of one per store.
  const bool inner = rbase - 4 * ((threadIdx.x & 63) >> 5) + TM * 32 <= a.M &&
                     col0 - (threadIdx.x & 31) + TN * 32 <= a.OC;
  if (__builtin_amdgcn_readfirstlane((int)inner)) {
    float v[TM][TN][16];
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float t = acc[i][j][r] + bv[j];
          v[i][j][r] = a.silu ? silu_fast(t) : t;
        }
    if (a.res) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const float* rr = a.res + (long long)(rbase + i * 32) * a.ldr + col0 + j * 32;
          float rv[16];
#pragma unroll
          for (int r = 0; r < 16; ++r) rv[r] = rr[(8 * (r >> 2) + (r & 3)) * a.ldr];
#pragma unroll
          for (int r = 0; r < 16; ++r) v[i][j][r] = rv[r] + v[i][j][r];
        }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        float* yr = y + (long long)(rbase + i * 32) * a.ldy + col0 + j * 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) yr[(8 * (r >> 2) + (r & 3)) * a.ldy] = v[i][j][r];
      }
    return;
  }
  float rv[TM][TN][16];
  if (a.res) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int col = col0 + j * 32, row0 = rbase + i * 32;
        const float* rr = a.res + (long long)row0 * a.ldr + col;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int dr = 8 * (r >> 2) + (r & 3);
          rv[i][j][r] = (col < a.OC && row0 + dr < a.M) ? rr[dr * a.ldr] : 0.f;
        }
      }
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = col0 + j * 32;
    if (col >= a.OC) continue;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int row0 = rbase + i * 32;
      float* yr = y + (long long)row0 * a.ldy + col;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int dr = 8 * (r >> 2) + (r & 3);
        if (row0 + dr >= a.M) continue;
        float v = acc[i][j][r] + bv[j];
        if (a.silu) v = silu_fast(v);
        if (a.res) v = rv[i][j][r] + v;
        yr[dr * a.ldy] = v;
      }
    }
  }
}

// Epilogue of a transposed 2x2 stride-2 conv's GEMM: scatter each column to
// its sub-pixel (rbase, col0 as in store_acc).
template <int TM, int TN>
__device__ __forceinline__ void store_shuf(const IgemmArgs& a, float* __restrict__ y, const f32x16 (&acc)[TM][TN],
                                           int rbase, int col0) {
  const int hw = a.H * a.W;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int col = col0 + j * 32;
    if (col >= a.OC) continue;
    const float bv = a.bias ? a.bias[col] : 0.f;
    const int q = col / a.shuf, o = col - q * a.shuf;
    const int dy = q >> 1, dx = q & 1;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = rbase + i * 32 + 8 * (r >> 2) + (r & 3);
        if (row >= a.M) continue;
        const int n = row / hw, rem = row - n * hw;
        const int yy = rem / a.W, xx = rem - yy * a.W;
        const long long pix = ((long long)n * 2 * a.H + 2 * yy + dy) * (2 * a.W) + 2 * xx + dx;
        float v = acc[i][j][r] + bv;
        if (a.silu) v = silu_fast(v);
        y[pix * a.ldy + o] = v;
      }
  }
}

// ------------------------------------------------------------ f16 split GEMM

// Packed operand of the split GEMM (split_gemm.hip): weight column o at
// k = 32 kt + 16 ks + 8 h + e, split s (0 hi, 1 lo), sits in f16 element e of
// 16-byte unit ((o / 32 * nkt + kt) * 4 + 2 ks + s) * 64 + 32 h + o % 32.
constexpr int kX3Units = 256;  // 16-byte units of one (32-column block, 32-deep K tile)
constexpr int kX3Base = 64;    // tile ids kX3Base + i select the i-th split-GEMM tile
struct X3Tile {
  int bm, bn, wm, wn;
};
extern const X3Tile kX3Tiles[];
int x3_num_tiles();
inline bool is_x3_tile(int t) { return t >= kX3Base && t < kX3Base + x3_num_tiles(); }
const char* x3_name(int t, int mode);
// hi and lo of n (finite) weights times their channel's scale, within 2^-23 of
// them, and that power of two for the channel's largest magnitude.
void x3_split(const float* v, int n, float scale, uint16_t* hi, uint16_t* lo);
float x3_weight_scale(float largest);
int launch_x3(sy_ctx* ctx, int t, int mode, const IgemmArgs& a);

// ------------------------------------------------------------ 3x3 from an LDS patch, f16 split

// split_conv3.hip: 3x3 pad-1 convolution of stride S = 1 or 2.  Packed weights: channel o,
// input channel c, tap, split s in f16 element c % 8 of 16-byte unit
// (((o / 32) ng + c / 16) 9 + tap) 128 + 64 s + 32 ((c / 8) % 2) + o % 32.
struct C3Args {
  const float* x;
  int N, H, W, IC, ldx, S, OH, OW;
  const void* w;
  const float* ws;    // per output channel: 1 / the weights' scale
  const float* bias;  // padded to whole column blocks
  const float* res;
  int ldr;
  float* y;
  int ldy, OC, silu;
  int ng;  // groups of 16 input channels
  // Filled by launch_c3: pixels; TH x TW outputs per tile, rows per image, tiles
  // per row, column blocks, reciprocals of TW (2^16) and of the patch width
  // (2^16, at stride 2 2^20), rounded up.
  int M, TH, TW, rpi, ntx, nblk, inv_tw, inv_pw;
};
constexpr int kC3Base = 96;  // tile ids kC3Base + i select the i-th form
int c3_num_forms();
inline bool is_c3_tile(int t) { return t >= kC3Base && t < kC3Base + c3_num_forms(); }
int c3_form_groups(int f);  // waves that share out a block's channel groups (1: none)
const char* c3_name(int f);
bool c3_fits(const C3Args& a);
int launch_c3(sy_ctx* ctx, int f, C3Args a);

}  // namespace sy
