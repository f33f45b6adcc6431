// dgi/csrc/mix/chunk_split.h — fp32 operands as bf16 parts, decays as powers, the order of sequences: what chunk_parts.hip and chunk_delta.hip share.
#pragma once
#include "chunk_args.h"

namespace {

constexpr int C = 32;              // tokens per chunk
constexpr float MOST = 3.38e38f;   // beyond, a first part would round to infinity
constexpr double LOG2E = 1.4426950408889634;

__device__ __forceinline__ double softplus_d(double x) { return fmax(x, 0.) + log1p(exp(-fabs(x))); }

__device__ __forceinline__ short4v read_tr(const char* p) { return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)p); }

// two values in three bf16 parts each; x becomes what is left for the next
__device__ __forceinline__ uint32_t part_of(float& x0, float& x1) {
  const uint32_t p = pack_bf16x2(x0, x1);
  x0 -= __uint_as_float(p << 16);
  x1 -= __uint_as_float(p & 0xffff0000u);
  return p;
}
template <int PARTS>
__device__ __forceinline__ void split8(const float* x, u32x4* p) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
    if constexpr (PARTS == 1) {
      p[0][i] = pack_bf16x2(a, b);
    } else {
      p[0][i] = part_of(a, b);
      p[1][i] = part_of(a, b);
      p[2][i] = pack_bf16x2(a, b);
    }
  }
}
// 3 / 2 2^(16 + the exponent of the largest): added and taken off again, it rounds to multiples of 2^-7 of it
__device__ __forceinline__ float grid_of(float most) { return __uint_as_float(((__float_as_uint(most) & 0x7f800000u) + 0x08000000u) | 0x00400000u); }
// Parts of products x f (l: what f lacks of more bits), with what they lack in 32 bits.  GRID: the first part is a multiple of what grid says.
template <bool GRID>
__device__ __forceinline__ void split2_of(const float* x, const float* f, const float* l, float grid, int i, u32x4* p) {
  float a = x[2 * i] * f[2 * i], b = x[2 * i + 1] * f[2 * i + 1];
  float ea = fmaf(x[2 * i], f[2 * i], -a), eb = fmaf(x[2 * i + 1], f[2 * i + 1], -b);
  if constexpr (GRID) {
    ea = fmaf(x[2 * i], l[2 * i], ea);
    eb = fmaf(x[2 * i + 1], l[2 * i + 1], eb);
    const float a0 = (a + grid) - grid, b0 = (b + grid) - grid;
    p[0][i] = pack_bf16x2(a0, b0);
    a = (a - a0) + ea;
    b = (b - b0) + eb;
    p[1][i] = part_of(a, b);
    p[2][i] = part_of(a, b);
    p[3][i] = pack_bf16x2(a, b);
  } else {
    p[0][i] = part_of(a, b);
    p[1][i] = part_of(a, b);
    p[2][i] = pack_bf16x2(a + ea, b + eb);
  }
}

__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}
// products of N operands' parts by one's (or its own: BN = N), for sums of their own: all but the first two parts', smallest first, to lo; multiply: those to hi, too.
// Sums take turns, none waits for its own last product.
template <int PA, int PB, int N, int BN>
__device__ __forceinline__ void small(const u32x4 (&a)[N][PA], const u32x4 (&b)[BN][PB], f32x4 (&lo)[N]) {
#pragma unroll
  for (int x = 2; x > 0; --x)                        // parts that together are x smaller than the first
#pragma unroll
    for (int p = x; p >= 0; --p)
      if (p < PA && x - p < PB) {
#pragma unroll
        for (int i = 0; i < N; ++i) lo[i] = mfma(a[i][p], b[i % BN][x - p], lo[i]);
      }
}
template <int PA, int PB, int N, int BN>
__device__ __forceinline__ void multiply(const u32x4 (&a)[N][PA], const u32x4 (&b)[BN][PB], f32x4 (&lo)[N], f32x4 (&hi)[N]) {
  small<PA, PB, N, BN>(a, b, lo);
#pragma unroll
  for (int i = 0; i < N; ++i) hi[i] = mfma(a[i][0], b[i % BN][0], hi[i]);
}

// 2^(whole + part), part within [-2, 2]
__device__ __forceinline__ float power(float whole, float part) {
  return __builtin_amdgcn_ldexpf(__builtin_amdgcn_exp2f(part), (int)whole);
}
__device__ __forceinline__ void whole_and_part(double x, float& whole, float& part) {
  x = fmin(fmax(x, -1e6), 1e6);
  const double i = rint(x);
  whole = (float)i;
  part = (float)(x - i);
}
// 2^x, rounded about once, and what it lacks: 2^part - 1 by its series, part within [-0.5, 0.5] (the first term left out is 5.2e-9)
__device__ __forceinline__ float power_once(double x, float* rest = nullptr) {
  float i, f;
  whole_and_part(x, i, f);
  const float y = f * 0.693147181f;
  float p = 1.f / 5040.f;
  p = fmaf(p, y, 1.f / 720.f);
  p = fmaf(p, y, 1.f / 120.f);
  p = fmaf(p, y, 1.f / 24.f);
  p = fmaf(p, y, 1.f / 6.f);
  p = fmaf(p, y, 0.5f);
  const float t = fmaf(p * y, y, y), r = 1.f + t;
  if (rest) *rest = __builtin_amdgcn_ldexpf((1.f - r) + t, (int)i);
  return __builtin_amdgcn_ldexpf(r, (int)i);
}

// chunks of all sequences one after the other
__device__ __forceinline__ int first_chunk(int row0, int seq) { return row0 / C + seq; }

// longest sequences first among at most 16
constexpr int MOST_SEQ = 16;
__device__ __forceinline__ int ranked(const ChunkArgs& a, int seq) {
  if (a.n_seq > MOST_SEQ || a.n_seq == 1) return seq;
  const int lane = threadIdx.x & 63, i = min(lane, a.n_seq - 1);
  const int len = lane < a.n_seq ? max(a.seq_row0[i + 1] - a.seq_row0[i], 0) : -1;
  if (!__any(len > a.skip_rows)) return seq;         // none is this launch's
  int before = 0;                                    // sequences that are longer, or as long and earlier
  for (int j = 0; j < a.n_seq; ++j) {
    const int other = __builtin_amdgcn_readlane(len, j);
    before += other > len || (other == len && j < lane);
  }
  return __ffsll((unsigned long long)__ballot(lane < a.n_seq && before == seq)) - 1;
}

}  // namespace
