// Multi-head attention core of the C2PSA block (PtModel.Attention,
// src/SimdYolo/PtModel.cs:429-437): from the qkv 1x1 conv output, viewed as
// [B, heads, 2*kd + hd, N], compute S = q^T k * scale, softmax over the last
// axis, o = v S^T, written as an NHWC [B, heads*hd, H, W] view; also emits v
// as a dense NHWC tensor for the depthwise `pe` conv.  The reference runs
// this as DeviceMatMul + Scale (op 4) + Softmax (op 25) + DeviceMatMul
// (VulkanExecution.cs:499-541, tensor.comp:62-68).
//
// Key dims up to 32 and head dims up to 64 (every YOLO11 / YOLO26 block: 32 and
// 64) run in one kernel that keeps the scores in registers.  Other geometries,
// and outputs that overlap the input or each other, run both products on the
// FP32-MFMA GEMM (gemm_nt); S rows and V^T rows are padded to N4 = round_up(N, 4)
// with zeros so K stays a multiple of 4.
#include <cfloat>
#include <cmath>

#include "split.h"
#include "sy_internal.h"

namespace sy {

struct AttnArgs {
  const float* qkv;
  int ldq, N, heads, kd, hd, qtiles;
  float scale;
  float* o;
  int ldo;
  float* v;
  int ldv;
};

// One query's output in plain float32 by one wave: lane `lane`'s channel.  Weights
// are normalised before they meet the values, so that no finite average overflows.
__device__ __forceinline__ float attn_row(const AttnArgs& a, const float* base, int q, int lane) {
  const float* qr = base + (long long)q * a.ldq;
  auto score = [&](int j) {
    if (j >= a.N) return -INFINITY;
    const float* kr = base + (long long)j * a.ldq + a.kd;
    float s = 0.f;
    for (int c = 0; c < a.kd; ++c) s = __builtin_fmaf(qr[c], kr[c], s);
    return s * a.scale;
  };
  float mx = -INFINITY, sum = 0.f, acc = 0.f;
  for (int j = lane; j < a.N; j += 64) mx = fmaxf(mx, score(j));
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  for (int j = lane; j < a.N; j += 64) sum += expf(score(j) - mx);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  const float inv = 1.f / sum;
  for (int j0 = 0; j0 < a.N; j0 += 64) {
    const float e = j0 + lane < a.N ? expf(score(j0 + lane) - mx) * inv : 0.f;
    for (int t = 0; t < min(64, a.N - j0); ++t) {
      const float et = __shfl(e, t);
      if (lane < a.hd) acc = __builtin_fmaf(et, base[(long long)(j0 + t) * a.ldq + 2 * a.kd + lane], acc);
    }
  }
  return acc;
}

// e^x for x up to a few units: 2^t of the hardware at t = x log2(e) rounded, times 1 plus the
// first-order term of t's exact rounding error and of log2(e)'s.  Below -150,
// where the result is under every float, 0; NaN stays.
__device__ __forceinline__ float exp_neg(float x) {
  constexpr float kLog2e = 1.4426950408889634f, kLog2eLow = (float)(1.4426950408889634 - (double)kLog2e);
  x = x < -150.f ? -150.f : x;
  const float t = x * kLog2e, r = __builtin_fmaf(x, kLog2eLow, __builtin_fmaf(x, kLog2e, -t));
  const float p = __builtin_amdgcn_exp2f(t);
  return __builtin_fmaf(p, r * 0.69314718f, p);
}

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Eight floats as three bf16 parts each, v = p[0] + p[1] + p[2] exactly.
__device__ __forceinline__ void parts8(const f32x4& x, const f32x4& y, bf16x8 (&p)[3]) {
  u32x4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f32x2v v = i < 2 ? f32x2v{x[2 * i], x[2 * i + 1]} : f32x2v{y[2 * i - 4], y[2 * i - 3]};
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      const unsigned b = __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
      w[s][i] = b;
      if (s < 2) {
        v[0] -= __builtin_bit_cast(float, b << 16);
        v[1] -= __builtin_bit_cast(float, b & 0xffff0000u);
      }
    }
  }
#pragma unroll
  for (int s = 0; s < 3; ++s) p[s] = __builtin_bit_cast(bf16x8, w[s]);
}

// main + rest += a b: the leading parts' product in main, the five next ones in
// rest.
__device__ __forceinline__ void mfma_parts(const bf16x8 (&a)[3], const bf16x8 (&b)[3], f32x16& main, f32x16& rest) {
  rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b[0], rest, 0, 0, 0);
  main = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[0], main, 0, 0, 0);
  rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[1], rest, 0, 0, 0);
  rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[2], rest, 0, 0, 0);
  rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b[0], rest, 0, 0, 0);
  rest = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b[1], rest, 0, 0, 0);
}

// 32 queries of one head and image per workgroup.  Wave w takes the 32-key
// tiles w, w + 4, ... with a running maximum, sum and output of its own; the
// four are joined through LDS at the end.  Nothing else is shared: operands go
// from L2 straight into MFMA registers.
//
// Scores are computed as S^T = K Q^T, so that a lane holds one query's scores
// (keys 8 (r / 4) + 4 half + r % 4): the maximum and sum over keys are in-lane
// but for one exchange between the wave's halves, and the probabilities are
// already the B operand of O^T = V^T P^T under the key order
// 8 (e / 4) + 4 half + e % 4 of a 16-key step, in which V is loaded.
//
// Both products take float32 operands as three bf16 parts (Henry, Tang and
// Heinecke, 2019), which hold a float's 24 significand bits over its whole exponent
// range (parts below 2^-126, of values below 2^-110, may be lost): no operand's
// precision depends on another's size, as it would with f16 pairs under common
// scales.  Six of the nine part products are taken, the rest is below 2^-24 of the
// product.  Where a part is not finite (infinities, NaN, values that round to 2^128
// in bf16) or a sum overflows, the query's output is not finite either and is
// computed again in plain float32.
//
// The running maximum (online softmax: Milakov and Gimelshein, 2018) moves, and the
// sums with it, only where a score passes it by kSlack; until then weights reach
// e^kSlack.  The test is on the difference, which is exact between floats this near:
// the sum of maximum and slack rounds, from 2^23 on to more than the slack.
//
// Bound by VALU work (the parts of K, V and P 350 operations per tile, the
// exponentials and sums about 220, beside 36 MFMAs) and, at 400 tokens, by the
// latency of its few tiles.  Measured, us, against two GEMMs, a softmax and a copy
// with the scores in memory / float32 MFMAs for both products / f16 pairs: 2 heads,
// 400 tokens, batch 16 74 / 28 / 21.6 -> 19.6, batch 1 25 / 18 / 14.5 -> 13.0;
// 4 heads, 1,600 tokens, batch 8 858 / 206 / 141 -> 145.  Error against float64 at
// 400 tokens 1.4e-7 (1.9e-7 with f16 pairs, 2.0e-7 with float32 MFMAs summed tile by
// tile).  Three waves per SIMD spill registers: 178 us at 1,600 tokens.
constexpr float kSlack = 2.5f;
__global__ __launch_bounds__(256, 2) void attention_kernel(const AttnArgs a) {
  constexpr int NQ = 32;  // queries
  __shared__ float O[4][NQ][65];
  __shared__ float M[4][NQ], Lsum[4][NQ];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = lane >> 5, r32 = lane & 31;
  const int qt = blockIdx.x % a.qtiles, bh = blockIdx.x / a.qtiles, head = bh % a.heads, b = bh / a.heads;
  const int per = 2 * a.kd + a.hd, q0 = qt * NQ;
  const float* base = a.qkv + (long long)b * a.N * a.ldq + head * per;
  float* ob = a.o + (long long)b * a.N * a.ldo + head * a.hd;
  float* vb = a.v + (long long)b * a.N * a.ldv + head * a.hd;

  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // Row `row`'s channels 16 ks + 8 half + 4 i .. + 3 from `at`.
  auto row4 = [&](int row, int at, int ks, int i) {
    const int c = 16 * ks + 8 * half + 4 * i;
    return c < a.kd ? *(const f32x4*)(base + min(row, a.N - 1) * a.ldq + at + c) : zero;
  };
  // A tile's keys and values; past the last key both read the last key's row.  Past
  // kd the keys' last channels are read again, which the queries' zeros cancel.  In a
  // whole tile the value rows' addresses are scalar, with one offset per lane.
  f32x4 k[2][2];
  float v[2][16];
  int kcol[2][2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
#pragma unroll
    for (int i = 0; i < 2; ++i) kcol[ks][i] = min(16 * ks + 8 * half + 4 * i, a.kd - 4);
  const int vrow = 4 * half * a.ldq + 2 * a.kd, vcol[2] = {min(r32, a.hd - 1), min(32 + r32, a.hd - 1)};
  auto load_k = [&](int j0) __attribute__((always_inline)) {
    const float* tb = base + j0 * a.ldq + a.kd;
    const int row = min(r32, a.N - 1 - j0) * a.ldq;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) k[ks][i] = *(const f32x4*)(tb + (unsigned)(row + kcol[ks][i]));
  };
  auto load_v = [&](int j0) __attribute__((always_inline)) {
    if (j0 + 32 <= a.N) {
      const float* tb = base + j0 * a.ldq;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float* vr = tb + (16 * (e >> 3) + 8 * ((e >> 2) & 1) + (e & 3)) * a.ldq;
#pragma unroll
        for (int d = 0; d < 2; ++d) v[d][e] = vr[(unsigned)(vrow + vcol[d])];
      }
      return;
    }
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const int j = min(j0 + 16 * (e >> 3) + 8 * ((e >> 2) & 1) + 4 * half + (e & 3), a.N - 1);
      const float* vr = base + j * a.ldq + 2 * a.kd;
#pragma unroll
      for (int d = 0; d < 2; ++d) v[d][e] = vr[vcol[d]];
    }
  };
  const int tiles = (a.N + 31) / 32;

  bf16x8 q[2][3];
  {
    f32x4 t[2][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i) t[ks][i] = row4(q0 + r32, 0, ks, i);
    load_k(min(wave, tiles - 1) * 32);
    load_v(min(wave, tiles - 1) * 32);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) parts8(t[ks][0], t[ks][1], q[ks]);
  }

  f32x16 acc[2], rest[2];
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[d][r] = rest[d][r] = 0.f;
  float mrun = -INFINITY, lrun = 0.f;

  for (int kt = wave; kt < tiles; kt += 4) {
    const int j0 = kt * 32;
    const int jn = min(kt + 4, tiles - 1) * 32;  // the next tile (the last loads its own again)
    f32x16 s, c;
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = c[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8 kp[3];
      parts8(k[ks][0], k[ks][1], kp);
      mfma_parts(kp, q[ks], s, c);
    }
    load_k(jn);
#pragma unroll
    for (int r = 0; r < 16; ++r) s[r] = (s[r] + c[r]) * a.scale;
    if (j0 + 32 > a.N) {
      asm volatile("");  // a branch, not 16 selects in every tile
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (j0 + 8 * (r >> 2) + 4 * half + (r & 3) >= a.N) s[r] = -INFINITY;
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if (__any(mx - mrun > kSlack)) {
      mx = fmaxf(mx, mrun);
      const float f = exp_neg(mrun - (mx == -INFINITY ? 0.f : mx));
      mrun = mx;
      lrun *= f;
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          acc[d][r] *= f;
          rest[d][r] *= f;
        }
    }
    const float from = mrun == -INFINITY ? 0.f : mrun;  // no weight yet: all are 0
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = exp_neg(s[r] - from);
      sum += s[r];
    }
    lrun += sum;
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      bf16x8 p[3];
      parts8(f32x4{s[8 * st], s[8 * st + 1], s[8 * st + 2], s[8 * st + 3]},
             f32x4{s[8 * st + 4], s[8 * st + 5], s[8 * st + 6], s[8 * st + 7]}, p);
#pragma unroll
      for (int d = 0; d < 2; ++d) {
        bf16x8 vp[3];
        parts8(f32x4{v[d][8 * st], v[d][8 * st + 1], v[d][8 * st + 2], v[d][8 * st + 3]},
               f32x4{v[d][8 * st + 4], v[d][8 * st + 5], v[d][8 * st + 6], v[d][8 * st + 7]}, vp);
        mfma_parts(vp, p, acc[d], rest[d]);
      }
    }
    load_v(jn);
  }

  const float l = lrun + __shfl_xor(lrun, 32);
  if (half == 0) {
    M[wave][r32] = mrun;
    Lsum[wave][r32] = l;
  }
#pragma unroll
  for (int d = 0; d < 2; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) O[wave][r32][32 * d + 8 * (r >> 2) + 4 * half + (r & 3)] = acc[d][r] + rest[d][r];
  // v of these rows, dense, for the positional conv: thread (row q, dim lane).
  float vd[NQ / 4];
#pragma unroll
  for (int i = 0; i < NQ / 4; ++i)
    vd[i] = base[min(q0 + wave + 4 * i, a.N - 1) * a.ldq + 2 * a.kd + min(lane, a.hd - 1)];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NQ / 4; ++i)
    if (q0 + wave + 4 * i < a.N && lane < a.hd) vb[(long long)(q0 + wave + 4 * i) * a.ldv + lane] = vd[i];
  // Joins the waves' partial outputs; a wave without keys weighs nothing.
  unsigned again = 0;  // rows to compute in plain float32
#pragma unroll
  for (int i = 0; i < NQ / 4; ++i) {
    const int q = wave + 4 * i;
    float mx = M[0][q];
#pragma unroll
    for (int w = 1; w < 4; ++w) mx = fmaxf(mx, M[w][q]);
    float l = 0.f, s = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float f = M[w][q] == -INFINITY ? 0.f : expf(M[w][q] - mx);
      l = __builtin_fmaf(Lsum[w][q], f, l);
      s = __builtin_fmaf(O[w][q][lane], f, s);
    }
    const float y = s / l;
    const bool here = q0 + q < a.N && lane < a.hd;
    again |= (__any(here && !(__builtin_fabsf(y) <= FLT_MAX)) ? 1u : 0u) << i;
    if (here) ob[(long long)(q0 + q) * a.ldo + lane] = y;
  }
  for (; again; again &= again - 1) {
    const int row = q0 + wave + 4 * __builtin_ctz(again);
    const float y = attn_row(a, base, row, lane);
    if (lane < a.hd) ob[(long long)row * a.ldo + lane] = y;
  }
}

// What the fused kernel takes: operands in its 32-channel steps, row offsets
// within an image in 32 bits, outputs of their own (its workgroups write them
// while others still read qkv; the GEMMs copy v and form all scores first).
static bool attention_fused(const sy_tensor* qkv, int kd, int hd, const sy_tensor* o, const sy_tensor* v) {
  return kd <= 32 && hd <= 64 && (long long)qkv->h * qkv->w * qkv->ldc < (1LL << 31) && !views_overlap(o, qkv) &&
         !views_overlap(v, qkv) && !views_overlap(o, v);
}

// One wavefront per row: y = softmax(x * scale) over n entries (max-subtracted),
// zeroing the padding columns [n, ld).
__global__ __launch_bounds__(256) void softmax_rows_kernel(float* __restrict__ s, long long rows, int n, int ld,
                                                           float scale) {
  const long long row = (long long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63;
  float* r = s + row * ld;
  float mx = -INFINITY;
  for (int j = lane; j < n; j += 64) mx = fmaxf(mx, r[j] * scale);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off));
  float sum = 0.f;
  for (int j = lane; j < n; j += 64) {
    const float e = expf(r[j] * scale - mx);
    r[j] = e;
    sum += e;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
  const float inv = 1.0f / sum;
  for (int j = lane; j < n; j += 64) r[j] *= inv;
  for (int j = n + lane; j < ld; j += 64) r[j] = 0.f;
}

// v of head h -> vt[b][h][d][j] (rows padded to ld with zeros) and the dense
// NHWC copy vd[b][j][h*hd + d].
__global__ __launch_bounds__(256) void split_v_kernel(const float* __restrict__ qkv, int ldq, int N, int heads,
                                                      int kd, int hd, int B, float* __restrict__ vt, int ld,
                                                      float* __restrict__ vd, int ldv) {
  const long long total = (long long)B * heads * hd * ld;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const int j = (int)(i % ld);
  const long long r = i / ld;
  const int d = (int)(r % hd);
  const long long bh = r / hd;
  const int h = (int)(bh % heads);
  const long long b = bh / heads;
  float v = 0.f;
  if (j < N) {
    v = qkv[(b * N + j) * ldq + h * (2 * kd + hd) + 2 * kd + d];
    vd[(b * N + j) * ldv + h * hd + d] = v;
  }
  vt[i] = v;
}

int op_attention(sy_ctx* ctx, const sy_tensor* qkv, int heads, int kd, int hd, float scale, const sy_tensor* o,
                 const sy_tensor* v) {
  SY_TRY(check_view(qkv, "attention qkv"));
  SY_TRY(check_view(o, "attention output"));
  SY_TRY(check_view(v, "attention v"));
  SY_CHECK(heads > 0 && kd > 0 && hd > 0, SY_EINVAL, "invalid attention geometry");
  const int per = 2 * kd + hd;
  SY_CHECK(qkv->c == heads * per, SY_EINVAL, "qkv has %d channels, expected heads*(2*kd+hd) = %d", qkv->c,
           heads * per);
  const int B = qkv->n, N = qkv->h * qkv->w, C = heads * hd;
  SY_CHECK(o->n == B && o->c == C && o->h == qkv->h && o->w == qkv->w, SY_EINVAL, "attention output shape mismatch");
  SY_CHECK(v->n == B && v->c == C && v->h == qkv->h && v->w == qkv->w, SY_EINVAL, "attention v shape mismatch");
  SY_CHECK(qkv->ldc == qkv->c || qkv->ldc % 4 == 0, SY_EINVAL, "qkv view stride");
  SY_CHECK(kd % 4 == 0 && per % 4 == 0 && hd % 4 == 0, SY_EUNSUPPORTED,
           "attention needs key/head dims that are multiples of 4");
  SY_CHECK(((uintptr_t)qkv->data & 15) == 0 && qkv->ldc % 4 == 0, SY_EINVAL,
           "attention qkv view must be 16-byte aligned with ldc %% 4 == 0");
  if (attention_fused(qkv, kd, hd, o, v)) {
    AttnArgs a{qkv->data, qkv->ldc, N, heads, kd, hd, (N + 31) / 32, scale, o->data, o->ldc, v->data, v->ldc};
    const long long grid = (long long)B * heads * a.qtiles;
    SY_CHECK(grid < (1LL << 31), SY_EUNSUPPORTED, "attention grid too large");
    ProfScope prof(ctx, "attention", 2.0 * B * heads * N * (double)N * (kd + hd),
                   4.0 * (double)B * N * (heads * per + 2.0 * C));
    hipLaunchKernelGGL(attention_kernel, dim3((unsigned)grid), dim3(256), 0, ctx->stream, a);
    return check_launch("attention");
  }
  const int N4 = (N + 3) / 4 * 4;
  const size_t s_floats = (size_t)B * heads * N * N4, vt_floats = (size_t)B * heads * hd * N4;
  SY_TRY(ensure_scratch(ctx, (s_floats + vt_floats) * sizeof(float) + 512));
  float* S = (float*)ctx->scratch;
  float* Vt = S + ((s_floats + 63) / 64 * 64);
  {
    const long long total = (long long)B * heads * hd * N4;
    ProfScope prof(ctx, "attn_split_v", 0, 4.0 * (double)B * N * C * 3);
    hipLaunchKernelGGL(split_v_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, ctx->stream, qkv->data,
                       qkv->ldc, N, heads, kd, hd, B, Vt, N4, v->data, v->ldc);
    SY_TRY(check_launch("attn_split_v"));
  }
  for (int h = 0; h < heads; ++h) {
    const float* q = qkv->data + h * per;
    SY_TRY(gemm_nt(ctx, q, N, kd, qkv->ldc, q + kd, N, qkv->ldc, S + (size_t)h * N * N4, N4, "attn_qk", B,
                   (long long)N * qkv->ldc, (long long)N * qkv->ldc, (long long)heads * N * N4));
  }
  {
    const long long rows = (long long)B * heads * N;
    ProfScope prof(ctx, "attn_softmax", 4.0 * rows * N, 8.0 * rows * N4);
    hipLaunchKernelGGL(softmax_rows_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, ctx->stream, S, rows, N,
                       N4, scale);
    SY_TRY(check_launch("attn_softmax"));
  }
  for (int h = 0; h < heads; ++h)
    SY_TRY(gemm_nt(ctx, S + (size_t)h * N * N4, N, N4, N4, Vt + (size_t)h * hd * N4, hd, N4, o->data + h * hd,
                   o->ldc, "attn_av", B, (long long)heads * N * N4, (long long)heads * hd * N4,
                   (long long)N * o->ldc));
  return SY_OK;
}

size_t attention_scratch_bytes(int B, int H, int W, int heads, int kd, int hd) {
  if (kd <= 32 && hd <= 64) return 0;  // the fused kernel
  const size_t N = (size_t)H * W, N4 = (N + 3) / 4 * 4;
  return ((size_t)B * heads * N * N4 + 64 + (size_t)B * heads * hd * N4) * sizeof(float) + 512;
}

}  // namespace sy

extern "C" int sy_attention(sy_ctx* ctx, const sy_tensor* qkv, int heads, int key_dim, int head_dim, float scale,
                            const sy_tensor* o, const sy_tensor* v) {
  SY_CHECK(ctx, SY_EINVAL, "null context");
  return sy::op_attention(ctx, qkv, heads, key_dim, head_dim, scale, o, v);
}
