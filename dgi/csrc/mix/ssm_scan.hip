// dgi/csrc/mix/ssm_scan.hip — Mamba-2 selective scan over packed rows with the state in a slot, and
// the gated group RMS norm that follows it.
//
// Per sequence of the step and head h (group g = h / (heads / G)), for its rows in order:
//
//     dt  = softplus(dt_raw[t][h] + dt_bias[h])             a = exp(-exp(a_log[h]) * dt)
//     S  <- a * S + dt * B_t x_t^T                          S: [N, dv] fp32
//     y_t = S^T C_t + d_skip[h] * x_t
//
// S starts as state[slot][h] (stored transposed, [dv][N]; zero when the portion starts at position 0) and goes back there after
// the last row.  This kernel takes decode rows and short portions, long ones go through chunk_scan.hip.  x | B | C come as one fp32 row (the convolution's output).
//
// Work split: a workgroup owns (sequence, head, 16 value columns); thread (column v, n-lane l) keeps
// S[n][v] for n = 4 l + 64 q + j in registers, so the y reduction over n is four DPP rotate-adds inside a
// 16-lane row.  The serial loop over tokens never waits for global memory: B, C, x and the step
// sizes of 16 tokens are staged in LDS (the next tile's loads are in flight, in registers, while the
// current one is consumed; softplus and the decay are computed once per token while staging), and a
// token costs two 16-byte LDS reads per four state values.  The state is stored value-major,
// [slot][head][v][n], so a thread's values are contiguous.  Everything is fp32 (softplus in its
// overflow-free form max(z, 0) + log1p(exp(-|z|))).
//
// gated_group_norm: g = y * silu(z), each of `groups` equal parts of a row divided by its own root
// mean square (eps inside the root), times w.
#include <algorithm>

#include "../common.h"

using namespace dgi;

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ldf<uint16_t>(const uint16_t* p) { return bf16_to_f32(*p); }
template <typename T> __device__ __forceinline__ void stf(T* p, float v);
template <> __device__ __forceinline__ void stf<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void stf<uint16_t>(uint16_t* p, float v) { *p = f32_to_bf16(v); }

// Sum over the 16 lanes of a DPP row (lanes 16 r .. 16 r + 15), result in every lane: four rotate-and-add
// steps in the VALU (row_ror 8, 4, 2, 1) — no trip through the LDS permute unit, which a per-token
// reduction inside a serial loop would otherwise wait for four times.
__device__ __forceinline__ float row16_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x122, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xf, 0xf, false));
  return v;
}

constexpr int COLS = 16;     // value columns per workgroup
constexpr int NL = 16;       // n-lanes per column
constexpr int TT = 16;       // tokens per staged tile

// NQ: float4 groups of state per thread (N <= 64 * NQ); thread (column v, n-lane l) owns
// n = 4 l + 64 q + j, j < 4.  LDS tile: B [TT][NP], C [TT][NP] (NP = 64 NQ, zero beyond N), x [TT][COLS],
// dt [TT], decay [TT].
template <typename TD, int NQ>
__global__ __launch_bounds__(COLS * NL) void ssm_scan_kernel(
    float* __restrict__ y, const float* __restrict__ xbc, int xbc_stride, const TD* __restrict__ dt_raw, int dt_stride,
    const float* __restrict__ dt_bias, const float* __restrict__ a_log, const float* __restrict__ d_skip,
    float* __restrict__ state, const int* __restrict__ positions, const int* __restrict__ seq_row0,
    const int* __restrict__ seq_slots, int heads, int dv, int N, int G, int most) {
  constexpr int NP = 64 * NQ;
  constexpr int PB = (TT * NP) / (COLS * NL);          // B (and C) values a thread stages per tile
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* sB = sm;
  float* sC = sB + TT * NP;
  float* sX = sC + TT * NP;
  float* sDt = sX + TT * COLS;
  float* sDa = sDt + TT;
  const int seq = blockIdx.x, h = blockIdx.y;
  const int tid = threadIdx.x;
  const int l = tid & (NL - 1), col = tid >> 4;
  const int v = blockIdx.z * COLS + col;
  const int r0 = seq_row0[seq], r1 = seq_row0[seq + 1];
  if (r1 <= r0 || (most > 0 && r1 - r0 > most)) return;          // longer portions: chunk_scan.hip, in a launch of its own
  const bool vok = v < dv;
  const int g = h / (heads / G);
  const int inner = heads * dv;
  const float* bp = xbc + inner + (size_t)g * N;
  const float* cp = bp + (size_t)G * N;
  float* sp = state + (((size_t)seq_slots[seq] * heads + h) * dv + v) * N;     // [..][head][v][n]
  const bool fresh = positions[r0] == 0;
  float S[NQ][4];
  const bool vec = (N & 3) == 0 && ((uintptr_t)state & 15) == 0;
#pragma unroll
  for (int q = 0; q < NQ; ++q) {
    const int n = 4 * l + 64 * q;
    if (vec) {
      // read and written once a step, and the other layers' come in between: marked so, the chip's caches give it up first, and whole
      // quads are one access (64 x 128, four layers: 32 rows of 64 heads 189 us -> 122, 4.4 TB/s; of 16 heads 64 -> 40; 4 rows 39 -> 25; sixteen
      // layers, more than the caches hold, 32 rows of 64 heads 47 us a layer -> 30)
      f32x4 s = {0.f, 0.f, 0.f, 0.f};
      if (!fresh && vok && n < N) s = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(sp + n));
#pragma unroll
      for (int j = 0; j < 4; ++j) S[q][j] = s[j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) S[q][j] = (!fresh && vok && n + j < N) ? sp[n + j] : 0.f;
    }
  }
  const float na = -expf(a_log[h]), bias = dt_bias[h], dsk = d_skip[h];

  float rb[PB], rc[PB], rx = 0.f, rdt = 0.f;
  auto prefetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      const int idx = tid + i * (COLS * NL);
      const int tok = idx / NP, n = idx - tok * NP;
      const bool ok = t0 + tok < r1 && n < N;
      rb[i] = ok ? bp[(size_t)(t0 + tok) * xbc_stride + n] : 0.f;
      rc[i] = ok ? cp[(size_t)(t0 + tok) * xbc_stride + n] : 0.f;
    }
    {
      const int tok = tid / COLS, c = tid - tok * COLS;            // TT * COLS == blockDim
      const int vv = blockIdx.z * COLS + c;
      rx = (t0 + tok < r1 && vv < dv) ? xbc[(size_t)(t0 + tok) * xbc_stride + (size_t)h * dv + vv] : 0.f;
    }
    if (tid < TT) rdt = t0 + tid < r1 ? ldf<TD>(dt_raw + (size_t)(t0 + tid) * dt_stride + h) : 0.f;
  };
  prefetch(r0);
  for (int t0 = r0; t0 < r1; t0 += TT) {
    __syncthreads();                                     // the previous tile is fully consumed
#pragma unroll
    for (int i = 0; i < PB; ++i) {
      sB[tid + i * (COLS * NL)] = rb[i];
      sC[tid + i * (COLS * NL)] = rc[i];
    }
    sX[tid] = rx;
    if (tid < TT) {
      const float z = rdt + bias;
      const float dt = fmaxf(z, 0.f) + log1pf(expf(-fabsf(z)));
      sDt[tid] = dt;
      sDa[tid] = expf(na * dt);
    }
    __syncthreads();
    if (t0 + TT < r1) prefetch(t0 + TT);                 // in flight while this tile is consumed
    const int cnt = min(TT, r1 - t0);
    for (int k = 0; k < cnt; ++k) {
      const float a = sDa[k], xv = sX[k * COLS + col];
      const float dx = sDt[k] * xv;
      float acc = 0.f;
#pragma unroll
      for (int q = 0; q < NQ; ++q) {
        const float4 b4 = *reinterpret_cast<const float4*>(sB + k * NP + 4 * l + 64 * q);
        const float4 c4 = *reinterpret_cast<const float4*>(sC + k * NP + 4 * l + 64 * q);
        S[q][0] = a * S[q][0] + b4.x * dx;
        S[q][1] = a * S[q][1] + b4.y * dx;
        S[q][2] = a * S[q][2] + b4.z * dx;
        S[q][3] = a * S[q][3] + b4.w * dx;
        acc += S[q][0] * c4.x + S[q][1] * c4.y + S[q][2] * c4.z + S[q][3] * c4.w;
      }
      acc = row16_sum(acc);
      if (l == 0 && vok) y[(size_t)(t0 + k) * inner + (size_t)h * dv + v] = acc + dsk * xv;
    }
  }
  if (vok) {
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const int n = 4 * l + 64 * q;
      if (vec) {
        if (n < N) __builtin_nontemporal_store(f32x4{S[q][0], S[q][1], S[q][2], S[q][3]}, reinterpret_cast<f32x4*>(sp + n));
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (n + j < N) sp[n + j] = S[q][j];
      }
    }
  }
}

template <typename TZ, typename TO>
__global__ __launch_bounds__(256) void gated_group_norm_kernel(
    TO* __restrict__ out, const float* __restrict__ y, const TZ* __restrict__ z, int z_stride,
    const float* __restrict__ w, int C, int groups, float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x, grp = blockIdx.y;
  const int gs = C / groups;
  const float* yp = y + (size_t)row * C + (size_t)grp * gs;
  const TZ* zp = z + (size_t)row * z_stride + (size_t)grp * gs;
  float ss = 0.f;
  for (int i = threadIdx.x; i < gs; i += 256) {
    const float zz = ldf<TZ>(zp + i);
    const float gv = yp[i] * zz / (1.f + expf(-zz));
    ss += gv * gv;
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float r = 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)gs + eps);
  for (int i = threadIdx.x; i < gs; i += 256) {
    const float zz = ldf<TZ>(zp + i);
    const float gv = yp[i] * zz / (1.f + expf(-zz));
    stf<TO>(out + (size_t)row * C + (size_t)grp * gs + i, gv * r * w[(size_t)grp * gs + i]);
  }
}

template <typename T> __device__ __forceinline__ void ld4(const T* p, float* f);
template <> __device__ __forceinline__ void ld4<float>(const float* p, float* f) {
  const float4 v = *reinterpret_cast<const float4*>(p);
  f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w;
}
template <> __device__ __forceinline__ void ld4<uint16_t>(const uint16_t* p, float* f) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
}
template <typename T> __device__ __forceinline__ void st4(T* p, const float* f);
template <> __device__ __forceinline__ void st4<float>(float* p, const float* f) {
  *reinterpret_cast<float4*>(p) = make_float4(f[0], f[1], f[2], f[3]);
}
template <> __device__ __forceinline__ void st4<uint16_t>(uint16_t* p, const float* f) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]));
}

// One pass: a group of up to 256 * 4 * VPT values stays in registers between the sum of squares and the
// store (y and z are read once); groups in fours of columns, 16-byte accesses.
template <typename TZ, typename TO, int VPT>
__global__ __launch_bounds__(256) void gated_group_norm_reg_kernel(
    TO* __restrict__ out, const float* __restrict__ y, const TZ* __restrict__ z, int z_stride,
    const float* __restrict__ w, int C, int groups, float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x, grp = blockIdx.y;
  const int gs = C / groups;
  const float* yp = y + (size_t)row * C + (size_t)grp * gs;
  const TZ* zp = z + (size_t)row * z_stride + (size_t)grp * gs;
  float gv[VPT][4];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = (threadIdx.x + 256 * i) * 4;
    if (c < gs) {
      float yy[4], zz[4];
      ld4<float>(yp + c, yy);
      ld4<TZ>(zp + c, zz);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        gv[i][k] = yy[k] * zz[k] / (1.f + expf(-zz[k]));
        ss += gv[i][k] * gv[i][k];
      }
    }
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float r = 1.f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)gs + eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = (threadIdx.x + 256 * i) * 4;
    if (c < gs) {
      float ww[4], o[4];
      ld4<float>(w + (size_t)grp * gs + c, ww);
#pragma unroll
      for (int k = 0; k < 4; ++k) o[k] = gv[i][k] * r * ww[k];
      st4<TO>(out + (size_t)row * C + (size_t)grp * gs + c, o);
    }
  }
}

}  // namespace

extern "C" int dgi_chunk_scan(float* y, int mode, const void* q, int q_stride, const void* k, int k_stride, const void* v,
                              int v_stride, int in_f32, const void* aux1, int aux1_stride, const void* aux2, int aux2_stride,
                              int aux_bf16, const float* par1, const float* par2, const float* par3, float cap, float* state,
                              float* norm, float* mx, float* norm_new, float* mx_new, const int* positions, const int* seq_row0,
                              const int* seq_slots, int n_seq, int H, int G, int dk, int dv, int skip_rows,
                              int segs, int seg_rows, float* ws, float* wsd, float* parts, int parts_chunks, int rows, hipStream_t st);

extern "C" int dgi_chunk_scan_ok(int mode, int dk, const void* q, int q_stride, const void* k, int k_stride, int in_f32);
bool dgi_chunk_parts_takes(int mode, int dk, int H, int G, int in_f32);

// chunked: portions go 32 tokens at a time through the matrix cores (chunk_parts.hip; sixteen, chunk_scan.hip, where groups have fewer than four heads or
// channels are more than 128).  Its workgroups have a
// compute unit to themselves and a pipeline to fill, so among more than APART_FROM sequences the short ones stay with this file's kernel: those
// of at most 48 rows while the workgroups find a place each (12 portions of 39 rows, 32 heads: 31 us against 51 there), longer ones when they
// wait for each other (64 columns, this file's time and that one's: 11 portions of 100 rows, 16 heads 35, 41; 128 rows 42, 41; 16 portions of 128
// rows, 64 heads 158, 162; 200 rows 242, 222).  recur.scan_chunks decides for whole steps, by the last two of these lines.
constexpr int APART_FROM = 8;
// In chunks of 32: 88 rows there (12 portions of 96 rows of 128 channels, 64 heads 88, 89; 128 rows 114, 104).
static int apart_rows(int n_seq, int heads, int dv, int N, int G) {
  const long units = (long)n_seq * heads * ((dv + 63) / 64);
  return n_seq <= APART_FROM ? 0 : units <= 128 ? 48 : dgi_chunk_parts_takes(5, N, heads, G, 1) ? 88 : units <= 256 ? 112 : 144;
}

// Segments (of *seg_rows rows) that a chunked step's portions are cut into (1: whole portions).  Together they are as long as the step: a portion
// may have all of its rows, beside sequences without any.
// Two passes over a segment take 2 (seg_rows / 16 + 5) chunks' time and the state pass some 10 us, one over a whole portion
// rows / 16 + 5: worth it from about 512 rows on while the workgroups (32 columns of a head) leave half of the chip idle.  Every segment's
// workgroups have a compute unit to themselves, so the rows are shared out over 256 of them, less one segment for each portion that may end in a
// part of one; a second round of workgroups costs more than shorter segments give (1444 rows, 16 heads of 64: whole 123 us, 11 segments
// 82, 8 segments 50; 2 x 2000 rows whole 166, 6 of 672 117, 7 of 576 101).  At most 24 segments, of 64 rows at least: the state pass goes through them one by one.
extern "C" int dgi_ssm_segments(int n_seq, int heads, int dv, int rows, int* seg_rows) {
  const long one = (long)heads * ((dv + 31) / 32), groups = n_seq * one;
  *seg_rows = 0;
  if (groups <= 0 || groups > 128 || rows - n_seq + 1 < 512) return 1;
  const long places = 256 - (n_seq - 1) * one;
  const long share = std::max({64l, (rows * one + places - 1) / places, (rows + 23l) / 24});
  const int each = (int)((share + 31) / 32 * 32), segs = (rows + each - 1) / each;
  if (segs < 3) return 1;
  *seg_rows = each;
  return segs;
}

// Whether such a step goes whole all the same: in chunks of 32 (chunk_parts.hip) a portion takes half to two thirds of the above, so three segments are too
// few, and with more than 64 workgroups segments are worth it from 1024 rows on (us in segments, whole, 64 channels: 8 heads, 8 x 65 rows 25, 11; 600 rows
// beside 7 45, 31; 16 heads, 4 x 192 29, 16; 600 beside 3 36, 31; 32 heads, 2 x 400 40, 26; 2 x 2000 120, 92).
extern "C" int dgi_ssm_whole(int n_seq, int heads, int dv, int N, int G, int rows, int segs) {
  return dgi_chunk_parts_takes(5, N, heads, G, 1) && (segs <= 3 || ((long)n_seq * heads * ((dv + 31) / 32) > 64 && rows - n_seq + 1 < 1024));
}

extern "C" int dgi_ssm_scan(float* y, const float* xbc, int xbc_stride, const void* dt_raw, int dt_f32, int dt_stride,
                            const float* dt_bias, const float* a_log, const float* d_skip, float* state,
                            const int* positions, const int* seq_row0, const int* seq_slots, int n_seq, int heads,
                            int dv, int N, int G, int chunked, int segs, int seg_rows, float* ws, float* wsd, float* parts,
                            int parts_chunks, hipStream_t s) {
  if (n_seq == 0) return 0;
  if (G <= 0 || heads % G) return -2;
  if (N > 256 || N <= 0 || dv <= 0) return -3;
  if (heads > 65535 || (dv + COLS - 1) / COLS > 65535) return -4;
  int most = 0;
  const float* B = xbc + (size_t)heads * dv;
  if (chunked && dgi_chunk_scan_ok(5, N, B + (size_t)G * N, xbc_stride, B, xbc_stride, 1)) {
    most = apart_rows(n_seq, heads, dv, N, G);
    const int rc = dgi_chunk_scan(y, 5, B + (size_t)G * N, xbc_stride, B, xbc_stride, xbc, xbc_stride, 1, dt_raw, dt_stride, nullptr, 0,
                                  !dt_f32, a_log, dt_bias, d_skip, 0.f, state, nullptr, nullptr, nullptr, nullptr, positions, seq_row0,
                                  seq_slots, n_seq, heads, G, N, dv, most, segs, seg_rows, ws, wsd, parts, parts_chunks, 0, s);
    if (rc || !most) return rc;
  }
  const int nq = (N + 63) / 64;
  const dim3 grid(n_seq, heads, (dv + COLS - 1) / COLS);
#define DGI_SCAN(TD, NQ)                                                                                              \
  ssm_scan_kernel<TD, NQ><<<grid, COLS * NL, (size_t)(2 * TT * 64 * NQ + TT * COLS + 2 * TT) * 4, s>>>(             \
      y, xbc, xbc_stride, (const TD*)dt_raw, dt_stride, dt_bias, a_log, d_skip, state, positions, seq_row0, seq_slots, \
      heads, dv, N, G, most)
  if (dt_f32) {
    if (nq <= 1) DGI_SCAN(float, 1); else if (nq <= 2) DGI_SCAN(float, 2); else DGI_SCAN(float, 4);
  } else {
    if (nq <= 1) DGI_SCAN(uint16_t, 1); else if (nq <= 2) DGI_SCAN(uint16_t, 2); else DGI_SCAN(uint16_t, 4);
  }
#undef DGI_SCAN
  DGI_CHECK_LAUNCH();
  return 0;
}

extern "C" int dgi_gated_group_norm(void* out, int out_f32, const float* y, const void* z, int z_f32, int z_stride,
                                    const float* w, int T, int C, int groups, float eps, hipStream_t s) {
  if (T == 0) return 0;
  if (groups <= 0 || C % groups || groups > 65535) return -2;
  const dim3 grid(T, groups);
  const int gs = C / groups;
  if (gs % 4 == 0 && gs <= 256 * 4 * 8 && z_stride % 4 == 0 &&
      (((uintptr_t)out | (uintptr_t)y | (uintptr_t)z | (uintptr_t)w) & 15) == 0 && z_f32 == out_f32) {
    if (z_f32) {
      if (gs <= 256 * 4 * 2)
        gated_group_norm_reg_kernel<float, float, 2><<<grid, 256, 0, s>>>((float*)out, y, (const float*)z, z_stride, w, C, groups, eps);
      else
        gated_group_norm_reg_kernel<float, float, 8><<<grid, 256, 0, s>>>((float*)out, y, (const float*)z, z_stride, w, C, groups, eps);
    } else {
      if (gs <= 256 * 4 * 2)
        gated_group_norm_reg_kernel<uint16_t, uint16_t, 2><<<grid, 256, 0, s>>>((uint16_t*)out, y, (const uint16_t*)z, z_stride, w, C, groups, eps);
      else
        gated_group_norm_reg_kernel<uint16_t, uint16_t, 8><<<grid, 256, 0, s>>>((uint16_t*)out, y, (const uint16_t*)z, z_stride, w, C, groups, eps);
    }
    DGI_CHECK_LAUNCH();
    return 0;
  }
  if (z_f32 && out_f32)
    gated_group_norm_kernel<float, float><<<grid, 256, 0, s>>>((float*)out, y, (const float*)z, z_stride, w, C, groups, eps);
  else if (!z_f32 && !out_f32)
    gated_group_norm_kernel<uint16_t, uint16_t><<<grid, 256, 0, s>>>((uint16_t*)out, y, (const uint16_t*)z, z_stride, w, C, groups, eps);
  else
    return -3;
  DGI_CHECK_LAUNCH();
  return 0;
}
