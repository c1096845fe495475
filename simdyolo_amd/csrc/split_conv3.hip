// 3x3 convolution, stride 1 or 2, on the f16 matrix cores, from an LDS patch.
//
// The arithmetic is split_gemm.hip's (float32 as scaled f16 pairs, three
// products).  Its implicit GEMM stages and splits every input value once per
// tap; here a workgroup stages the input patch of its output tile (TH x TW
// outputs, (TH + 2) x (TW + 2) inputs at stride 1, (2 TH + 1) x (2 TW + 1) at
// stride 2) once, up to 64 channels at a time, and the nine taps read it at
// shifted pixels.  All of a chunk's loads are issued together: 16 channels at a
// time left too few bytes in flight, and every wait for weights behind them
// (loads return in order) cost a memory latency.  Weights stream from L2
// straight into MFMA operands: their packed order makes each read of a wave
// 1 KiB contiguous, and the workgroup's waves read the same ones.
//
// Scales are split_gemm.hip's, by chunk instead of K tile.  A workgroup that reads
// a value of 2^16 or more, or a pixel whose channels of a chunk are not all zero
// but all below the pairs' full range, computes its tile again in plain float32, at
// about the speed of the float32 tiles: an element's error is at most 2^-23 of its
// pixel's largest of the chunk, whatever the other pixels hold.  The test costs two
// operations per four values: 80 -> 80 at 80 x 80, batch 32, 98.7 -> 100.5 us, at
// 45 x 75, batch 4, 10.5 -> 10.7, 64 -> 64 at 40 x 40, batch 1, 5.0 -> 5.1, at 80 x 80,
// batch 32, 53.8 -> 53.6.  Bits kept per pixel for all chunks took up to 10% (spills).
//
// A wave owns TM 32-pixel blocks x TN 32-channel blocks.  Per (tap, 16
// channels) it reads 2 TM KiB from LDS and 2 TN KiB from L1 / L2 for 3 TM TN
// MFMAs of 32 cycles.
//
// Measured at 64 -> 64 channels, 80 x 80, batch 32 (15.1 GFLOP direct): 52 - 54 us on
// random inputs (41 - 44 on zeros: the clock follows the power), against 73 us for the fastest float32 Winograd form.  The matrix cores are busy for 38% of its
// cycles (SQ_VALU_MFMA_BUSY_CYCLES over GRBM_GUI_ACTIVE); the patch loads
// (8,000 of a 128-pixel workgroup's 29,000 cycles), the epilogue (6,000)
// and a thin last round of 1,600 workgroups on 256 CUs take the rest.
// Workgroups that run through several tiles with the next patch loaded behind
// the last taps measured the same, 16-channel double buffering 57 - 60 us.
// At batch 1 the chain of taps is the time: sharing a block's groups out over
// four or eight waves (KW) takes 64 -> 64 at 40 x 40 from 6.3 to 5.0 us, 128 -> 128
// at 20 x 20 from 9.3 to 6.0, 256 -> 64 at 20 x 20 from 15.5 to 8.1.
// Stride 2, batch 32, against the implicit GEMM of split_gemm.hip, which stages
// every input per tap: 64 -> 128 at 80 x 80 42 -> 38 us, 32 -> 64 at 160 x 160
// 49 -> 41, 16 -> 32 at 320 x 320 88 -> 70 (315 MB), 128 -> 128 at 40 x 40 33 -> 22.
//
// LDS holds the patch as planes of 8 channels, [split][8-channel block][pixel]
// [8].  ds_read_b128 serves 16 lanes a cycle over 64 banks, lanes 0-3, 12-15,
// 20-23, 24-27 together and the other 16 of each half wave together (measured:
// 232 B/clk per CU without conflicts, 126 with 32 consecutive pixels on 32
// consecutive lanes); c3_row gives the lanes of one such group 16 consecutive
// pixels.  The planes' pitch spreads a staged pixel's 8-byte writes over the
// banks.
#include <cmath>
#include <cstring>
#include <string>

#include "igemm.h"
#include "split.h"

namespace sy {

constexpr int kC3Oob = 0x40000000;       // buffer offset past every record: the load returns zero
constexpr int kC3BufWord3 = 0x00020000;  // raw buffer resource, word 3 (gfx9 family)

// LDS pixels a patch may take for a tile of BM outputs.
constexpr int c3_patch(int bm, int s) {
  return s == 1 ? (bm == 32 ? 72 : bm == 64 ? 112 : 192) : (bm == 32 ? 168 : bm == 64 ? 304 : 568);
}
constexpr int c3_extent(int n, int s) { return s * (n - 1) + 3; }  // inputs under n outputs

// Low 32 bits of the product of two values below 2^24 (a full-rate instruction,
// a 32-bit multiply is a quarter-rate one).
__device__ __forceinline__ int mul24(int x, int y) { return (int)__umul24((unsigned)x, (unsigned)y); }

// Pixel of a 32-pixel block that MFMA row r (lane r of a half wave) holds.
__device__ __forceinline__ int c3_row(int r) { return ((0x73261540 >> (r & 28)) & 7) * 4 + (r & 3); }

// Four zeros: the source of input outside the image.
__device__ const float kC3Zeros[4] = {0.f, 0.f, 0.f, 0.f};

// A wave's blocks in plain float32, on the float32 matrix cores, operands straight
// from memory: channel groups g0, g0 + gs, ...  Lane half h takes channels
// 8 q + 4 h .. + 3 of its pixel and column.
template <int TM, int TN>
__device__ __forceinline__ void c3_plain(const C3Args& a, const int* opix, int ob0, int g0, int gs, int lane,
                                         f32x16 (&acc)[TM][TN]) {
  const int half = lane >> 5, r32 = lane & 31;
  const float* img[TM];
  int iy0[TM], ix0[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int pix = opix[i * 32 + r32], t = pix / a.OW, n = t / a.OH;
    img[i] = a.x + (long long)n * a.H * a.W * a.ldx;
    iy0[i] = pix < a.M ? (t - n * a.OH) * a.S - 1 : -4;  // -4: every tap is outside
    ix0[i] = (pix - t * a.OW) * a.S - 1;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  }
  float ws[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) ws[j] = a.ws[(ob0 + j) * 32 + r32];
  for (int g = g0; g < a.ng; g += gs) {
    for (int k = 0; k < 18; ++k) {
      const int tap = k >> 1, h8 = k & 1, c = 16 * g + 8 * h8 + 4 * half;
      f32x4 xv[TM], wv[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int iy = iy0[i] + tap / 3, ix = ix0[i] + tap % 3;
        const bool ok = c < a.IC && (unsigned)iy < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
        xv[i] = *(const f32x4*)(ok ? img[i] + ((long long)iy * a.W + ix) * a.ldx + c : kC3Zeros);
      }
#pragma unroll
      for (int j = 0; j < TN; ++j)
        wv[j] = join4((const _Float16*)a.w +
                          ((((long long)(ob0 + j) * a.ng + g) * 9 + tap) * 128 + 32 * h8 + r32) * 8 + 4 * half,
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
}

// Waves per SIMD the registers are allocated for (each measured without spills
// that matter).
constexpr int c3_waves(int s, int g, int nw, int blocks, int kw, bool one) {
  if (kw > 1) return s == 1 ? 4 : 2;
  if (one) return blocks == 2 ? (s == 2 ? 2 : 3) : (s == 2 ? 3 : 4);
  if (blocks == 2) return g == 4 || s == 2 ? 2 : 3;
  return (g == 4 || s == 2) && nw == 2 ? 2 : 3;
}

// S: stride.  G: 16-channel groups per chunk.  At stride 2 a patch row holds its
// even columns, then the odd ones, so that the operand reads of neighbouring
// outputs are neighbours at every tap.  KW > 1: the tile's channel groups shared
// out over KW waves (small grids: a fourth or an eighth of the chain of taps),
// their sums joined through LDS, each wave finishing 16 / KW of the rows.
// ONE: all channels fit one chunk, whose staging registers are free again before
// the sums exist.
template <int S, int G, int WM, int WN, int TM, int TN, int KW, bool ONE>
__global__ __launch_bounds__(WM* WN * KW * 64, c3_waves(S, G, WM * WN, TM * TN, KW, ONE)) void conv3_kernel(
    const C3Args a) {
  constexpr int NW = WM * WN * KW, NT = NW * 64, BM = WM * TM * 32, NPX = c3_patch(BM, S);
  constexpr int PL = (NPX * 8 + 127) / 128 * 128 + 64 / G;  // halves per plane
  constexpr int L_IT = (NPX * 4 * G + NT - 1) / NT;         // float4 loads per thread and chunk
  __shared__ __attribute__((aligned(16))) _Float16 P[G * 4 * PL];
  static_assert(KW == 1 || G * 4 * PL * 2 >= KW * 4096, "the partial sums fit the patch's memory");
  __shared__ __attribute__((aligned(16))) int opix[BM];
  __shared__ float red[NW];  // the waves' largest magnitudes, negative: a pixel is below the scale's range

  const int tid = threadIdx.x, lane = tid & 63, wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  static_assert(KW == 1 || (WM * WN * TM * TN == 1 && 16 % KW == 0), "split sums: one block per workgroup");
  const int wk = wid % KW, wm = wid / KW / WN, wn = wid / KW % WN;
  const int half = lane >> 5, r32 = lane & 31;
  // Each XCD (workgroups L, L + 8, ...) takes a contiguous run of tiles, a
  // tile's channel blocks next to each other (they read the same patch) and
  // neighbouring tiles after it.
  const int grid = gridDim.x, L = blockIdx.x;
  const int xcd = L & 7, q8 = grid >> 3, rem = grid & 7;
  const int T = xcd * q8 + (xcd < rem ? xcd : rem) + (L >> 3);
  const int tile = T / a.nblk, ob0 = (T - tile * a.nblk) * (WN * TN) + wn * TN;
  const int trow = tile / a.ntx, ox0 = (tile - trow * a.ntx) * a.TW;
  // Tile rows run over virtual output rows, rpi per image: OH + 1 with tiles
  // that may span images (the inputs of the row past OH are the zero rows
  // between two images), or a multiple of TH with tiles inside one image.
  const int v0 = trow * a.TH, nb = v0 / a.rpi, y0 = v0 - nb * a.rpi;
  const int PW = c3_extent(a.TW, S), npx = c3_extent(a.TH, S) * PW, odd = (PW + 1) >> 1;

  // Patch values this thread stages: its i-th float4 is channels 4 q4 .. + 3 of
  // the chunk, of patch pixel px0 + i NT / 4G.  Byte offsets from the tile's
  // first image; pixels outside their image read as zero.
  const long long img = (long long)a.H * a.W * a.ldx;
  const long long span = 4 * ((a.N - nb) * img - a.ldx + a.IC);
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.x + nb * img), (short)0, (int)min(span, (long long)kC3Oob), kC3BufWord3);
  const int q4 = tid % (4 * G), px0 = tid / (4 * G);
  // Row of patch pixel px: at most 568 pixels, the quotient by a 2^16 or 2^20
  // reciprocal is exact.
  auto patch_row = [&](int px) { return mul24(px, a.inv_pw) >> (S == 1 ? 16 : 20); };
  f32x4 d[L_IT];
  auto xload = [&](int ch) __attribute__((always_inline)) {
    const bool cok = ch * (16 * G) + 4 * q4 < a.IC;
#pragma unroll
    for (int i = 0; i < L_IT; ++i) {
      const int px = px0 + i * (NT / (4 * G)), pr = patch_row(px), ix = S * ox0 - 1 + px - mul24(pr, PW);
      const int row = S * y0 - 1 + pr;
      const bool wrap = a.rpi > a.OH && row >= S * a.rpi;  // into the next image
      const int y = wrap ? row - S * a.rpi : row;
      const bool ok =
          cok && px < npx && nb + wrap < a.N && (unsigned)y < (unsigned)a.H && (unsigned)ix < (unsigned)a.W;
      const int off = ok ? 4 * ((wrap ? (int)img : 0) + mul24(mul24(y, a.W) + ix, a.ldx) + 4 * q4) : kC3Oob;
      d[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, off, ch * (64 * G), 0));
    }
  };
  // Weights run kRing taps ahead of their use, across groups and chunks (the
  // last group loads its own first taps again): uniform base of the wave's
  // channel blocks, 32-bit lane offset.
  constexpr int kRing = 3;
  f16x8 bv[kRing][TN][2];
  const int wob = a.ng * (9 * 128 * 16);  // bytes per 32-channel block
  const char* wbase = (const char*)a.w + (long long)ob0 * wob;
  const unsigned wlane = lane * 16;
  auto wload = [&](int g, int tap) __attribute__((always_inline)) {
    const char* wg = wbase + min(g, a.ng - 1) * (9 * 128 * 16);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int p = 0; p < 2; ++p)
        bv[tap % kRing][j][p] = *(const f16x8*)(wg + (j * wob + (tap * 2 + p) * 1024) + wlane);
  };

  // A chunk into LDS.  A pixel is below the scale's range if its channels of the
  // chunk are not all zero and none is in the pairs' full range (2^-13 or more,
  // scaled).  Few are: the first test is on any four channels of a thread.
  static_assert(L_IT <= 32, "a bit per staged pixel");
  auto stage = [&](int ch, int se, bool first) __attribute__((always_inline)) {
    const float s = exp_float(se);
    const unsigned range = (unsigned)(241 - se) << 23;  // bits of 2^-13 / s
    float m = 0.f;
    unsigned least = ~0u;  // bits of the smallest nonzero maximum, less one
#pragma unroll
    for (int i = 0; i < L_IT; ++i) {
      const float mi = max4(d[i]);
      m = fmaxf(m, mi);
      least = min(least, __builtin_bit_cast(unsigned, mi) - 1);
      const int px = px0 + i * (NT / (4 * G));
      u32x2 hi, lo;
      split4(d[i], s, hi, lo);
      if (S == 2 ? px < npx : (L_IT * NT == NPX * 4 * G || px < NPX)) {
        int at = px;
        if (S == 2) {
          const int row = mul24(patch_row(px), PW), c = px - row;
          at = row + (c >> 1) + (c & 1 ? odd : 0);
        }
        _Float16* dst = P + (q4 >> 1) * PL + at * 8 + (q4 & 1) * 4;
        *(u32x2*)dst = hi;
        *(u32x2*)(dst + 2 * G * PL) = lo;
      }
    }
    if (first) {
#pragma unroll
      for (int t = 0; t < kRing; ++t) wload(wk, t);
    }
    m = wave_max63(m);
    if (__builtin_expect(__any(least < range - 1), 0)) {
      unsigned full = 0, some = 0;  // a bit per pixel
      if (S == 2 && !ONE) xload(ch);  // their many registers are not kept until here
#pragma unroll
      for (int i = 0; i < L_IT; ++i) {
        const float mi = max4(d[i]);
        if (mi > 0.f) some |= 1u << i;
        if (__builtin_bit_cast(unsigned, mi) >= range) full |= 1u << i;
      }
      if (__any(or_lanes<4 * G>(some) & ~or_lanes<4 * G>(full))) m = -m;
    }
    if (lane == 63) red[wid] = m;
  };
  xload(0);
  // The epilogue's operands, loaded before they are waited for.
  const int col0 = ob0 * 32 + r32;
  float bias[TN], ws[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    bias[j] = col0 + j * 32 < a.OC ? a.bias[col0 + j * 32] : 0.f;
    ws[j] = a.ws[col0 + j * 32];
  }
  // This tile's output pixels by MFMA row; M, past the output, for none.
  for (int p = tid; p < BM; p += NT) {
    const int q = (p & ~31) + c3_row(p & 31), py = mul24(q, a.inv_tw) >> 16, ox = ox0 + q - mul24(py, a.TW);
    const bool wrap = y0 + py >= a.rpi;
    const int n = wrap ? nb + 1 : nb, oy = wrap ? y0 + py - a.rpi : y0 + py;
    opix[p] = py < a.TH && n < a.N && oy < a.OH && ox < a.OW ? mul24(mul24(n, a.OH) + oy, a.OW) + ox : a.M;
  }
  // LDS offset (halves) of this lane's operand rows at tap (0, 0).
  int arow[TM];
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int p = (wm * TM + i) * 32 + c3_row(r32), py = mul24(p, a.inv_tw) >> 16;
    arow[i] = (S * mul24(min(py, a.TH - 1), PW) + p - mul24(py, a.TW)) * 8 + half * PL;
  }
  int se = kSplitExpGuess;
  float big = 0.f;  // largest magnitude so far
  f32x16 acc[TM][TN], crs[TM][TN];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = crs[i][j][r] = 0.f;
  };
  int low = 0;  // negative: a chunk had a pixel below the range of its scale
  auto maxima = [&]() __attribute__((always_inline)) {
    int l = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      big = fmaxf(big, __builtin_fabsf(red[w]));
      l |= __builtin_bit_cast(int, red[w]);
    }
    return __builtin_amdgcn_readfirstlane(l);
  };
  // Chunk ch (loaded already) into LDS.
  auto enter = [&](int ch) __attribute__((always_inline)) {
    stage(ch, se, ch == 0);
    __syncthreads();
    int l = maxima(), ne;
    if (!scale_fits(big, se, &ne)) {  // rare: the chunk again with another scale
      if (!ONE && ch > 0) rescale<TM, TN>(se, ne, acc, crs);
      se = ne;
      xload(ch);
      __syncthreads();  // every wave has read the maxima
      stage(ch, se, false);
      __syncthreads();
      l = maxima();
    }
    low |= l;
  };
  if (ONE) enter(0);
  clear();

  // KW waves take a group each per step (KW == G), so a chunk is one step.
  static_assert(KW == 1 || KW == G, "a group per wave and chunk");
  for (int gs = 0; gs < a.ng; gs += KW) {
    if (!ONE && gs % G == 0) {
      if (gs > 0) {
        xload(gs / G);
        __syncthreads();  // the last chunk's operand reads are done
      }
      enter(gs / G);
    }
    const int g = gs + wk;
    if (KW > 1 && g >= a.ng) continue;
    const _Float16* pg = P + (g % G) * (2 * PL);
    f16x8 av[2][TM][2];
    auto aload = [&](int tap) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p)
          av[tap & 1][i][p] =
              *(const f16x8*)(pg + p * (2 * G * PL) + arow[i] +
                              ((tap / 3) * PW + (S == 1 ? tap % 3 : tap % 3 == 1 ? odd : tap % 3 / 2)) * 8);
    };
    aload(0);
    // The barriers pin the order: operands of the next tap, this tap's MFMAs,
    // the weights three taps on.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      if (tap + 1 < 9) aload(tap + 1);
      __builtin_amdgcn_sched_barrier(0);
      const auto& w = bv[tap % kRing];
      const auto& x = av[tap & 1];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          crs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i][1], w[j][0], crs[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i][0], w[j][0], acc[i][j], 0, 0, 0);
        }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          crs[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[i][0], w[j][1], crs[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      wload(tap + kRing < 9 ? g : g + KW, (tap + kRing) % 9);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  const int* po = opix + wm * TM * 32;
  if (__builtin_expect(__builtin_amdgcn_readfirstlane((int)(big >= kSplitHuge)) || low < 0, 0)) {
    // Lane and arguments read anew: the rare path keeps no register of the main one.
    int l = lane;
    auto p = (const __attribute__((address_space(4))) C3Args*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+v"(l), "+s"(p));
    c3_plain<TM, TN>(*(const C3Args*)p, po, ob0, wk, KW, l, acc);
  } else {
    unscale<TM, TN>(ws, se, acc, crs);
  }
  if (KW > 1) {
    // Rows r of the sums belong to wave r KW / 16.
    float* sums = (float*)P;
    __syncthreads();  // the patch's reads are done
#pragma unroll
    for (int r = 0; r < 16; ++r) sums[(wk * 16 + r) * 64 + lane] = acc[0][0][r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      if (r * KW / 16 != wk) continue;
      float v = sums[r * 64 + lane];
#pragma unroll
      for (int w = 1; w < KW; ++w) v += sums[(w * 16 + r) * 64 + lane];
      acc[0][0][r] = v;
    }
  }
  // Buffer accesses: a pixel or channel past the output has an offset past the
  // resource, whose load gives zero and whose store is dropped.
  const __amdgpu_buffer_rsrc_t yr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)a.y, (short)0, 4 * ((a.M - 1) * a.ldy + a.OC), kC3BufWord3);
  const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
      (void*)a.res, (short)0, a.res ? 4 * ((a.M - 1) * a.ldr + a.OC) : 0, kC3BufWord3);
  // D layout: lane holds column r32 of rows 8 (r / 4) + 4 half + r % 4.
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    int px[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      px[r] = po[i * 32 + 8 * (r >> 2) + 4 * half + (r & 3)];
      if (KW > 1 && r * KW / 16 != wk) px[r] = a.M;  // another wave's row
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const unsigned col = col0 + j * 32 < a.OC ? 4u * (col0 + j * 32) : 0x80000000u;
      float v[16], rv[16];
      if (a.res) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          rv[r] = __builtin_bit_cast(float,
                                     __builtin_amdgcn_raw_buffer_load_b32(rr, mul24(px[r], 4 * a.ldr) + col, 0, 0));
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        v[r] = acc[i][j][r] + bias[j];
        if (a.silu) v[r] = silu_fast(v[r]);
        if (a.res) v[r] = rv[r] + v[r];
      }
#pragma unroll
      for (int r = 0; r < 16; ++r)
        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v[r]), yr, mul24(px[r], 4 * a.ldy) + col, 0,
                                              0);
    }
  }
}

// Wave grid (pixels x channels), 32 x 32 blocks per wave, waves per block.
#define SY_C3_LIST(X)                                                                                 \
  X(0, 2, 2, 2, 1, 1) X(1, 4, 1, 1, 1, 1) X(2, 2, 1, 1, 1, 1) X(3, 2, 2, 1, 1, 1) X(4, 2, 3, 1, 1, 1) \
  X(5, 1, 1, 1, 1, 4) X(6, 1, 1, 1, 1, 8)

struct C3Form {
  int wm, wn, tm, tn, kw;
};
#define SY_C3_CFG(i, wm, wn, tm, tn, kw) {wm, wn, tm, tn, kw},
static const C3Form kC3Forms[] = {SY_C3_LIST(SY_C3_CFG)};
#undef SY_C3_CFG
static constexpr int kNumC3 = sizeof(kC3Forms) / sizeof(kC3Forms[0]);
int c3_form_groups(int f) { return kC3Forms[f].kw; }
int c3_num_forms() { return kNumC3; }

const char* c3_name(int f) {
  struct Names {
    std::string n[kNumC3];
    Names() {
      for (int i = 0; i < kNumC3; ++i) {
        char buf[48];
        const C3Form& c = kC3Forms[i];
        int len = snprintf(buf, sizeof buf, "conv3_x3_%dx%d_%d%d", c.wm * c.tm * 32, c.wn * c.tn * 32, c.wm, c.wn);
        if (c.kw > 1) snprintf(buf + len, sizeof buf - len, "_ks%d", c.kw);
        n[i] = buf;
      }
    }
  };
  static const Names names;
  return names.n[f].c_str();
}

// Output tile of at most bm pixels whose patch fits, with the fewest tiles:
// TW from 4 to bm columns (a multiple of 16 among equals: its operand reads are
// free of bank conflicts), tiles inside one image or over virtual rows.
static bool pick_tile_shape(int bm, const C3Args& a, int* th, int* tw, int* rpi, long long* tiles, int* ntx) {
  const int S = a.S, N = a.N, H = a.OH, W = a.OW;
  long long best = -1;
  for (int w = 4; w <= bm && w <= ((W + 3) & ~3); ++w) {
    const int rows = c3_patch(bm, S) / c3_extent(w, S);
    const int h = std::min(bm / w, (rows - 3) / S + 1);
    if (rows < 3 || h < 1) continue;
    const int tx = (W + w - 1) / w;
    for (int span = 0; span < 2; ++span) {
      // A tile spans at most two images.
      const int hh = span ? std::min(h, H - 1) : std::min(h, H);
      if (hh < 1) continue;
      const int r = span ? H + 1 : (H + hh - 1) / hh * hh;
      const long long t = ((long long)N * r + hh - 1) / hh * tx;
      if (best < 0 || t < best || (t == best && w % 16 == 0)) {
        best = t;
        *th = hh;
        *tw = w;
        *rpi = r;
        *ntx = tx;
      }
    }
  }
  *tiles = best;
  return best > 0;
}

bool c3_fits(const C3Args& a) {
  // 32-bit byte offsets: the two images a tile may span below the zero-read
  // offset, outputs and residuals below 2^31; pixel counts for 24-bit multiplies.
  const long long img = 4LL * a.H * a.W * a.ldx, M = (long long)a.N * a.OH * a.OW;
  return 2 * img < kC3Oob && 4 * M * a.ldy < (1LL << 31) && 4 * M * a.ldr < (1LL << 31) && M < (1LL << 24) &&
         4LL * a.ldy < (1LL << 24) && 4LL * a.ldr < (1LL << 24) && a.ldx < (1LL << 24) &&
         (long long)a.H * a.W < (1LL << 24) &&
         (long long)a.N * (a.H + 64) < (1LL << 24) && (long long)a.ng * (9 * 128 * 16 * 4) < (1LL << 31);
}

// Chunks of up to 64 channels for the wide forms at stride 1; 32 for the
// 32-channel forms (twice the workgroups per CU: 80 -> 80 at 80 x 80, batch 32,
// 104 against 119 us) and for stride 2 (four times the patch); a group per wave
// where waves share a block out.
template <int WM, int WN, int TM, int TN, int KW>
static auto c3_pick(int stride, int ng) -> void (*)(const C3Args) {
  if constexpr (KW > 1) {
    return stride == 2 ? conv3_kernel<2, KW, WM, WN, TM, TN, KW, false> : conv3_kernel<1, KW, WM, WN, TM, TN, KW, false>;
  } else {
    if (stride == 2)
      return ng == 1   ? conv3_kernel<2, 1, WM, WN, TM, TN, 1, true>
             : ng == 2 ? conv3_kernel<2, 2, WM, WN, TM, TN, 1, true>
                       : conv3_kernel<2, 2, WM, WN, TM, TN, 1, false>;
    if (ng == 1) return conv3_kernel<1, 1, WM, WN, TM, TN, 1, true>;
    if (ng == 2) return conv3_kernel<1, 2, WM, WN, TM, TN, 1, true>;
    if constexpr (WN * TN == 1)
      return conv3_kernel<1, 2, WM, WN, TM, TN, 1, false>;
    else
      return ng <= 4 ? conv3_kernel<1, 4, WM, WN, TM, TN, 1, true> : conv3_kernel<1, 4, WM, WN, TM, TN, 1, false>;
  }
}

int launch_c3(sy_ctx* ctx, int f, C3Args a) {
  const C3Form& c = kC3Forms[f];
  const int bm = c.wm * c.tm * 32;
  long long tiles = 0;
  SY_CHECK(pick_tile_shape(bm, a, &a.TH, &a.TW, &a.rpi, &tiles, &a.ntx), SY_EUNSUPPORTED, "no tile for a %dx%d image",
           a.H, a.W);
  a.M = a.N * a.OH * a.OW;
  a.nblk = ((a.OC + 31) / 32 + c.wn * c.tn - 1) / (c.wn * c.tn);
  a.inv_tw = 65536 / a.TW + 1;
  a.inv_pw = (a.S == 1 ? 1 << 16 : 1 << 20) / c3_extent(a.TW, a.S) + 1;
  SY_CHECK(tiles * a.nblk < (1LL << 31), SY_EUNSUPPORTED, "convolution grid too large");
  void (*k)(const C3Args) = nullptr;
#define SY_C3_CASE(i, wm, wn, tm, tn, kw)                                                              \
  if (f == i) k = c3_pick<wm, wn, tm, tn, kw>(a.S, a.ng);
  SY_C3_LIST(SY_C3_CASE)
#undef SY_C3_CASE
  SY_CHECK(k != nullptr, SY_EINVAL, "no split 3x3 form %d", f);
  hipLaunchKernelGGL(k, dim3((unsigned)(tiles * a.nblk)), dim3(c.wm * c.wn * c.kw * 64), 0,
                     ctx->stream, a);
  return SY_OK;
}

}  // namespace sy
