// dgi/csrc/mix/masked_attention.hip — row-wise softmax attention over the paged KV pool for any
// head geometry, in bf16 or fp32, with a block ("chunk") mask and an output gate.
//
// decode_attention.hip and prefill_attention.hip are MFMA kernels for bf16 heads of 64 / 128
// dims whose keys and values share one size.  This kernel is the general form the other
// geometries run on (key size != value size, sizes that are no multiple of 16, fp32 caches)
// and the one both step phases share: every query row — a decode row or one row of a prompt
// portion — is one wave that walks its own visible keys
//
//     [first(p), p],   first(p) = floor(p / mask) * mask   (mask > 0: keys of the row's own block
//                                                            of `mask` positions, counted from
//                                                            position 0 of the sequence)
//                      first(p) = 0                          (mask == 0: plain causal)
//                      first(p) = max(0, p + mask + 1)       (mask < 0: the last -mask positions, a sliding window)
//
// straight from the cache (this step's keys are written before it runs), so the result does
// not depend on how the prompt was cut into steps or on what else is in the batch.
// Scores, the online softmax and the output accumulation are fp32; exp is the accurate expf.
// Optional distance bias: dist_bias[min(p - j, n_dist - 1)][head] (fp32, one row per distance, the
// last row for everything farther) is added to the scaled score of key j before the softmax.
// Optional head factors: the scaled score is multiplied by head_scale[head] (fp32, any sign).
// Optional soft cap: the scaled (and biased) score s becomes softcap * tanh(s / softcap).
// Optional sinks: exp(sinks[head]) joins the softmax denominator of that head (a logit that has no
// key and no value; it is neither scaled nor capped).
// Optional epilogue: out *= sigmoid(gate), element by element or one gate per head (`gate_heads`): the mixer's
// output gate, read from the same fused projection row as q.
//
// Wave layout: lane j scores key first + 64 i + j (a contiguous dk-vector per lane, 16-byte
// loads where dk allows); the 64 probabilities go through LDS and every lane accumulates the
// value dims d = lane + 64 c, so the V reads of one key are one coalesced row.
// grid = (rows, H), 64 threads.
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

constexpr int MAXC = 8;       // value dims per lane: dv <= 64 * MAXC
constexpr int MAXDK = 512;    // query vector staged in LDS

__device__ __forceinline__ float dot_row(const float* __restrict__ qs, const float* __restrict__ k, int dk) {
  float acc = 0.f;
  if ((dk & 3) == 0) {
    for (int e = 0; e < dk; e += 4) {
      const float4 v = *reinterpret_cast<const float4*>(k + e);
      acc += qs[e] * v.x + qs[e + 1] * v.y + qs[e + 2] * v.z + qs[e + 3] * v.w;
    }
  } else {
    for (int e = 0; e < dk; ++e) acc += qs[e] * k[e];
  }
  return acc;
}

__device__ __forceinline__ float dot_row(const float* __restrict__ qs, const uint16_t* __restrict__ k, int dk) {
  float acc = 0.f;
  if ((dk & 7) == 0) {
    for (int e = 0; e < dk; e += 8) {
      float f[8];
      unpack8(*reinterpret_cast<const u32x4*>(k + e), f);
#pragma unroll
      for (int j = 0; j < 8; ++j) acc += qs[e + j] * f[j];
    }
  } else {
    for (int e = 0; e < dk; ++e) acc += qs[e] * bf16_to_f32(k[e]);
  }
  return acc;
}

template <typename T>
__global__ __launch_bounds__(64) void masked_attn_rows_kernel(
    const T* __restrict__ q, int q_stride, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ cu_seqlens, int n_seqs,
    const int* __restrict__ positions, int G, int dk, int dv, int bs, float scale, int mask,
    const T* __restrict__ gate, int gate_stride, T* __restrict__ out, int out_stride,
    const float* __restrict__ dist_bias, int n_dist, float softcap, const float* __restrict__ sinks,
    const float* __restrict__ head_scale, int gate_heads) {
  __shared__ float qs[MAXDK];
  __shared__ float ps[64];
  __shared__ long long vo[64];

  const int row = blockIdx.x, head = blockIdx.y, H = gridDim.y;
  const int lane = threadIdx.x;
  const int kvh = head / (H / G);
  // the row's sequence: row index itself (decode rows), or the portion holding it (cu_seqlens)
  int seq = row;
  if (cu_seqlens) {
    int lo = 0, hi = n_seqs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (cu_seqlens[mid] <= row) lo = mid; else hi = mid - 1;
    }
    seq = lo;
  }
  const int* bt = block_tables + (size_t)seq * bt_stride;
  const int pos = positions[row];
  const int first = mask > 0 ? (pos / mask) * mask : (mask < 0 ? max(0, pos + mask + 1) : 0);

  const T* qp = q + (size_t)row * q_stride + (size_t)head * dk;
  for (int e = lane; e < dk; e += 64) qs[e] = ldf<T>(qp + e);
  __syncthreads();

  float m_run = -__builtin_inff(), l_run = 0.f;
  float o[MAXC];
#pragma unroll
  for (int c = 0; c < MAXC; ++c) o[c] = 0.f;
  const int nc = (dv + 63) >> 6;

  for (int k0 = first; k0 <= pos; k0 += 64) {
    const int key = k0 + lane;
    const bool ok = key <= pos;
    float s = -__builtin_inff();
    long long vbase = 0;
    if (ok) {
      const int blk = bt[key / bs];
      const long long slot = ((long long)blk * G + kvh) * bs + (key % bs);
      s = dot_row(qs, k_cache + slot * dk, dk) * scale;
      if (head_scale) s *= head_scale[head];
      if (dist_bias) s += dist_bias[(size_t)min(pos - key, n_dist - 1) * H + head];
      if (softcap > 0.f) s = softcap * tanhf(s / softcap);
      vbase = slot * dv;
    }
    const float m_new = fmaxf(m_run, wave_max(s));     // lane 0's key k0 is always visible: finite
    const float p = ok ? expf(s - m_new) : 0.f;
    const float corr = expf(m_run - m_new);            // first tile: exp(-inf) = 0
    l_run = l_run * corr + wave_sum(p);
    m_run = m_new;
    __syncthreads();                                   // previous tile's ps / vo fully read
    ps[lane] = p;
    vo[lane] = vbase;
    __syncthreads();
    const int n = min(64, pos - k0 + 1);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      if (c < nc) {
        const int d = lane + 64 * c;
        float acc = o[c] * corr;
        if (d < dv)
          for (int j = 0; j < n; ++j) acc += ps[j] * ldf<T>(v_cache + vo[j] + d);
        o[c] = acc;
      }
    }
  }
  float inv = 1.f / l_run;
  if (sinks) {
    // the sink logit joins the denominator only: out = o / (l + exp(sink - m)), with the larger of the two as reference
    const float sk = sinks[head], m2 = fmaxf(m_run, sk);
    const float f = expf(m_run - m2);
    inv = f / (l_run * f + expf(sk - m2));
  }
  T* op = out + (size_t)row * out_stride + (size_t)head * dv;
  const T* gp = gate ? gate + (size_t)row * gate_stride + (gate_heads ? (size_t)head : (size_t)head * dv) : nullptr;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    const int d = lane + 64 * c;
    if (c < nc && d < dv) {
      float v = o[c] * inv;
      if (gp) v *= 1.f / (1.f + expf(-ldf<T>(gate_heads ? gp : gp + d)));
      stf<T>(op + d, v);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Grouped kernel (fp32, and bf16 heads of more than 128 dims): one workgroup per (row, kv head) serves all R = H / G query heads of the group
// from ONE pass over the keys, with 16-byte cache reads.  Eight waves take 64-key tiles round
// robin; in a tile a 16-lane group owns one key at a time (lane c of the group its 16-byte chunk c,
// against the same chunk of the R queries in registers), so one wave instruction reads four whole K
// rows and a row's lines are fetched once; the scores and then the probabilities go through LDS,
// and the values are read the same way.
// Partial outputs are combined over the four lane groups by shuffles and over the waves in LDS.
// Needs dk, dv multiples of 8 (bf16) / 4 (fp32), H / G <= 8 and (H / G) * dv <= 1024.
// A step of few rows over many keys is cut into gridDim.z runs of a row's tiles (one workgroup each; a run may be
// empty): every run leaves its maximum, sum of weights and unnormalised output in part_ml / part_o, and
// masked_attn_reduce_kernel combines them, adds the sink and applies the gate.
constexpr int GNW = 8;        // waves per workgroup

// sum over the 16 lanes of a row (every lane gets it)
__device__ __forceinline__ float row16_total(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x124, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x122, 0xf, 0xf, false));
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x121, 0xf, 0xf, false));
  return v;
}

template <typename T, int R, int VP>
__global__ __launch_bounds__(64 * GNW) void masked_attn_group_kernel(
    const T* __restrict__ q, int q_stride, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    const int* __restrict__ block_tables, int bt_stride, const int* __restrict__ cu_seqlens, int n_seqs,
    const int* __restrict__ positions, int H, int dk, int dv, int bs, float scale, int mask,
    const T* __restrict__ gate, int gate_stride, T* __restrict__ out, int out_stride,
    const float* __restrict__ dist_bias, int n_dist, float softcap, const float* __restrict__ sinks,
    const float* __restrict__ head_scale, int gate_heads, float* __restrict__ part_o, float* __restrict__ part_ml) {
  constexpr int E = 16 / sizeof(T);
  extern __shared__ __attribute__((aligned(16))) float smem[];
  const int row = blockIdx.x, kvh = blockIdx.y, G = gridDim.y;
  const int r = H / G;
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int lg = lane >> 4, lc = lane & 15;
  float* qs = smem;                                  // [R][dk]
  float* ps = qs + R * dk;                           // [GNW][R][64]
  int* vs = reinterpret_cast<int*>(ps + GNW * R * 64);   // [GNW][64] cache slot of each key of the wave's tile
  float* cm = reinterpret_cast<float*>(vs + GNW * 64);   // [GNW][R] running max, then [GNW][R] sums
  float* co = cm + 2 * GNW * R;                      // [GNW][R][dv] partial outputs

  int seq = row;
  if (cu_seqlens) {
    int lo = 0, hi = n_seqs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (cu_seqlens[mid] <= row) lo = mid; else hi = mid - 1;
    }
    seq = lo;
  }
  const int* bt = block_tables + (size_t)seq * bt_stride;
  const int pos = positions[row];
  const int first = mask > 0 ? (pos / mask) * mask : (mask < 0 ? max(0, pos + mask + 1) : 0);

  const T* qp = q + (size_t)row * q_stride + (size_t)kvh * r * dk;
  for (int e = tid; e < r * dk; e += 64 * GNW) qs[e] = ldf<T>(qp + e);
  __syncthreads();

  // this lane's chunks of the queries: in registers where they fit, else read from LDS again for every key
  constexpr bool QREG = R * VP * E <= 64;
  constexpr int U = VP == 1 ? 8 : 4;
  float qr[QREG ? R : 1][QREG ? VP : 1][E];
  if constexpr (QREG) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int p = 0; p < VP; ++p)
#pragma unroll
        for (int j = 0; j < E; ++j) {
          const int c = (lc + 16 * p) * E + j;
          qr[i][p][j] = i < r && c < dk ? qs[i * dk + c] : 0.f;
        }
  }
  float m[R], l[R], o[R][VP][E];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    m[i] = -__builtin_inff();
    l[i] = 0.f;
#pragma unroll
    for (int p = 0; p < VP; ++p)
#pragma unroll
      for (int j = 0; j < E; ++j) o[i][p][j] = 0.f;
  }
  float* psw = ps + w * R * 64;
  int* vsw = vs + w * 64;
  const int ntiles = (pos - first) / 64 + 1;
  const int tpr = (ntiles + (int)gridDim.z - 1) / (int)gridDim.z;      // tiles per run
  const int t_end = min(ntiles, ((int)blockIdx.z + 1) * tpr);
  for (int tile = blockIdx.z * tpr + w; tile < t_end; tile += GNW) {
    const int k0 = first + tile * 64;
    const int key = k0 + lane;
    const bool ok = key <= pos;
    const int kq = min(key, pos);                        // lanes past the last key point at it: every load stays in bounds
    vsw[lane] = (bt[kq / bs] * G + kvh) * bs + (kq % bs);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int n = min(64, pos - k0 + 1);
    // U keys per group at a time, all their rows requested before the first is used; places past n repeat the last key
    u32x4 raw[U][VP];
    auto load_rows = [&](const T* cache, int d, int kk0) {
      int sl[U];
#pragma unroll
      for (int u = 0; u < U; ++u) sl[u] = vsw[kk0 + 4 * u + lg];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int p = 0; p < VP; ++p) {
          const int c = (lc + 16 * p) * E;
          raw[u][p] = c < d ? *reinterpret_cast<const u32x4*>(cache + (size_t)sl[u] * d + c) : u32x4{0u, 0u, 0u, 0u};
        }
    };
    auto as_floats = [&](const u32x4& v, float* f) {
      if constexpr (sizeof(T) == 2) {
        unpack8(v, f);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) f[j] = __uint_as_float(v[j]);
      }
    };
    for (int kk0 = 0; kk0 < n; kk0 += 4 * U) {
      load_rows(k_cache, dk, kk0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float acc[R];
#pragma unroll
        for (int i = 0; i < R; ++i) acc[i] = 0.f;
#pragma unroll
        for (int p = 0; p < VP; ++p) {
          float kf[E];
          as_floats(raw[u][p], kf);
          const int c = (lc + 16 * p) * E;
#pragma unroll
          for (int i = 0; i < R; ++i) {
            if constexpr (QREG) {
#pragma unroll
              for (int j = 0; j < E; ++j) acc[i] += qr[i][p][j] * kf[j];
            } else if (i < r && c < dk) {
#pragma unroll
              for (int j = 0; j < E; ++j) acc[i] += qs[i * dk + c + j] * kf[j];
            }
          }
        }
        float mine = 0.f;                                // lane i of the group keeps head i's score
#pragma unroll
        for (int i = 0; i < R; ++i) {
          const float tot = row16_total(acc[i]);
          mine = lc == i ? tot : mine;
        }
        if (lc < R) psw[lc * 64 + kk0 + 4 * u + lg] = mine;
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (i < r) {
        float s = -__builtin_inff();
        if (ok) {
          s = psw[i * 64 + lane] * scale;
          if (head_scale) s *= head_scale[kvh * r + i];
          if (dist_bias) s += dist_bias[(size_t)min(pos - key, n_dist - 1) * H + kvh * r + i];
          if (softcap > 0.f) s = softcap * tanhf(s / softcap);
        }
        const float m_new = fmaxf(m[i], wave_max(s));       // key k0 (lane 0) is visible: finite
        const float p = ok ? expf(s - m_new) : 0.f;
        const float corr = expf(m[i] - m_new);
        l[i] = l[i] * corr + wave_sum(p);
        m[i] = m_new;
#pragma unroll
        for (int vp = 0; vp < VP; ++vp)
#pragma unroll
          for (int j = 0; j < E; ++j) o[i][vp][j] *= corr;
        psw[i * 64 + lane] = p;                          // over the lane's own score
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int kk0 = 0; kk0 < n; kk0 += 4 * U) {
      load_rows(v_cache, dv, kk0);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float pk[R];                                     // 0 past n
#pragma unroll
        for (int i = 0; i < R; ++i) pk[i] = i < r ? psw[i * 64 + kk0 + 4 * u + lg] : 0.f;
#pragma unroll
        for (int vp = 0; vp < VP; ++vp) {
          float vf[E];
          as_floats(raw[u][vp], vf);
#pragma unroll
          for (int i = 0; i < R; ++i)
#pragma unroll
            for (int j = 0; j < E; ++j) o[i][vp][j] += pk[i] * vf[j];
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  // lane groups -> lane group 0, then waves -> LDS
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int vp = 0; vp < VP; ++vp)
#pragma unroll
      for (int j = 0; j < E; ++j) {
        float v = o[i][vp][j];
        v += __shfl_xor(v, 16, 64);
        v += __shfl_xor(v, 32, 64);
        o[i][vp][j] = v;
      }
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      cm[w * R + i] = m[i];
      cm[GNW * R + w * R + i] = l[i];
    }
  }
  if (lg == 0) {
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (i < r)
#pragma unroll
        for (int vp = 0; vp < VP; ++vp) {
          const int c = (lc + 16 * vp) * E;
          if (c < dv)
#pragma unroll
            for (int j = 0; j < E; ++j) co[((size_t)w * R + i) * dv + c + j] = o[i][vp][j];
        }
  }
  __syncthreads();
  for (int idx = tid; idx < r * dv; idx += 64 * GNW) {
    const int i = idx / dv, d = idx - i * dv;
    const int head = kvh * r + i;
    if (part_o) {
      float M = -__builtin_inff(), L = 0.f, O = 0.f;
#pragma unroll
      for (int ww = 0; ww < GNW; ++ww) M = fmaxf(M, cm[ww * R + i]);
      if (M != -__builtin_inff()) {                    // an empty run leaves zeros
#pragma unroll
        for (int ww = 0; ww < GNW; ++ww) {
          const float f = expf(cm[ww * R + i] - M);
          L += cm[GNW * R + ww * R + i] * f;
          O += co[((size_t)ww * R + i) * dv + d] * f;
        }
      }
      const size_t slot = ((size_t)blockIdx.z * gridDim.x + row) * H + head;
      part_o[slot * dv + d] = O;
      if (d == 0) {
        part_ml[2 * slot] = M;
        part_ml[2 * slot + 1] = L;
      }
      continue;
    }
    float M = sinks ? sinks[head] : -__builtin_inff();
#pragma unroll
    for (int ww = 0; ww < GNW; ++ww) M = fmaxf(M, cm[ww * R + i]);
    float L = sinks ? expf(sinks[head] - M) : 0.f, O = 0.f;      // the sink: one more term of the denominator
#pragma unroll
    for (int ww = 0; ww < GNW; ++ww) {
      const float f = expf(cm[ww * R + i] - M);          // waves without a tile: exp(-inf) = 0
      L += cm[GNW * R + ww * R + i] * f;
      O += co[((size_t)ww * R + i) * dv + d] * f;
    }
    float v = O / L;
    if (gate) v *= 1.f / (1.f + expf(-ldf<T>(gate + (size_t)row * gate_stride + (gate_heads ? (size_t)head : (size_t)head * dv + d))));
    stf<T>(out + (size_t)row * out_stride + (size_t)head * dv + d, v);
  }
}

// ---------------------------------------------------------------------------------------------
// The grouped kernel for bf16 heads of up to 128 dims.  Bounded by the cached rows' bytes, so what counts is how many of them are
// under way: a wave holds one tile of 64 keys in flight all the time.  The keys' registers are loaded again with the tile's values
// as the products consume them, those again with the next tile's keys as the values are summed, and the pages of the next tile are
// looked up a tile ahead.  32 rows of 1500 to 2500 keys, 8 groups of 4 heads of 128 dims, cap, sinks and gate: 54.4 us (the kernel above with
// 16 lanes per key on the vector ALUs, each batch of rows waited for: 68), 4.7 TB/s in all, 5.8 while the longest row is read; 100 rows of
// 600 keys, at most 1024 in a block: 87 -> 57; 1 row of 7000 keys of 64 dims in 13 runs: 31 -> 20.  Scores are matrix products (16 keys by up to 16 heads, products of bf16 numbers exact, sums in fp32);
// they change to one key per lane through LDS for the softmax, whose weights and the values' sums stay in fp32 on the vector ALUs.
// NW waves take tiles in turn; runs over gridDim.z as above.
template <int CTRL>
__device__ __forceinline__ float row_max_step(float v) {
  return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false)));
}
// maximum over the wave (every lane gets it)
__device__ __forceinline__ float wave_max_all(float v) {
  v = row_max_step<0x128>(v);
  v = row_max_step<0x124>(v);
  v = row_max_step<0x122>(v);
  v = row_max_step<0x121>(v);
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

template <bool ONCE>
__device__ __forceinline__ u32x4 cached_row(const uint16_t* p) {
  if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return *reinterpret_cast<const u32x4*>(p);
}

struct RowsArgs {
  const uint16_t *q, *k, *v, *gate;
  uint16_t* out;
  const int *block_tables, *cu_seqlens, *positions;
  const float *dist_bias, *sinks, *head_scale;
  float *part_o, *part_ml;
  int q_stride, bt_stride, n_seqs, H, dk, dv, bs, mask, gate_stride, out_stride, n_dist, gate_heads;
  float scale, softcap;
};

// R: heads of a group, rounded up to 2, 4 or 8; D: dims, rounded up to 64 or 128; ONCE: cached rows are marked as what nothing reads again
// soon, so that the chip's caches give them up first
template <int R, int D, int NW, bool ONCE>
__global__ __launch_bounds__(64 * NW, R == 8 ? 2 : 3) void masked_attn_tiles_kernel(const RowsArgs a) {
  constexpr int KS = D / 32;                         // loads (and products) of a block of 16 keys
  constexpr int LK = D / 8, KL = 64 / LK;            // lanes of a value row, rows of a load
  constexpr int VB = 16 / KL;                        // loads of 16 value rows
  constexpr int QP = D + 8;
  __shared__ __attribute__((aligned(16))) uint16_t qs[R * QP];
  __shared__ __attribute__((aligned(16))) float ps[NW][64 * R];        // scores, then weights: [key][head]
  __shared__ int vs[NW][2][64];                      // cache slot of each key of the wave's tile, and of the next one
  __shared__ float cm[NW][R], cl[NW][R];
  __shared__ float co[NW][R][D];
  const int row = blockIdx.x, kvh = blockIdx.y, G = gridDim.y, r = a.H / G;
  const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int n16 = lane & 15, g = lane >> 4;
  const int lc = lane & (LK - 1), lg = lane / LK;
  const int dk = a.dk, dv = a.dv, bs = a.bs;

  int seq = row;
  if (a.cu_seqlens) {
    int lo = 0, hi = a.n_seqs - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (a.cu_seqlens[mid] <= row) lo = mid; else hi = mid - 1;
    }
    seq = lo;
  }
  const int* bt = a.block_tables + (size_t)seq * a.bt_stride;
  const int pos = a.positions[row];
  const int first = a.mask > 0 ? (pos / a.mask) * a.mask : (a.mask < 0 ? max(0, pos + a.mask + 1) : 0);
  const int ntiles = pos < 0 ? 0 : (pos - first) / 64 + 1;       // a row without a position sees no keys
  const int tpr = (ntiles + (int)gridDim.z - 1) / (int)gridDim.z;      // tiles per run
  const int t_end = min(ntiles, ((int)blockIdx.z + 1) * tpr);
  int tile = blockIdx.z * tpr + w;
  // slot of this lane's key of a tile; lanes past the last key point at it: every load stays in bounds
  auto slot = [&](int t) {
    const int kq = max(min(first + t * 64 + lane, pos), 0);
    return (bt[kq / bs] * G + kvh) * bs + kq % bs;
  };
  const int slot0 = slot(min(tile, ntiles - 1));

  const uint16_t* qp = a.q + (size_t)row * a.q_stride + (size_t)kvh * r * dk;
  for (int e = tid; e < R * D; e += 64 * NW) {
    const int i = e / D, c = e % D;
    qs[i * QP + c] = i < r && c < dk ? qp[i * dk + c] : 0;
  }
  __syncthreads();
  u32x4 qf[KS];                                      // query n16 (0 past R), dims 32 s + 8 g
#pragma unroll
  for (int s = 0; s < KS; ++s)
    qf[s] = n16 < R ? *reinterpret_cast<const u32x4*>(&qs[(n16 < R ? n16 : 0) * QP + 32 * s + 8 * g]) : u32x4{0u, 0u, 0u, 0u};

  float m[R], l[R], o[R][8];                         // l: this lane's keys alone
#pragma unroll
  for (int i = 0; i < R; ++i) {
    m[i] = -__builtin_inff();
    l[i] = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[i][j] = 0.f;
  }
  float* psw = ps[w];
  auto meet = [] {                                   // the wave's LDS writes before, its reads after
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  static_assert(KS == VB, "16 keys and 16 values take the same registers");
  u32x4 raw[4][KS];
  // chunks past a row's end: its last one again (keys: zeros when they are used; values: sums that nobody reads)
  const u32x4 zero = {0u, 0u, 0u, 0u};
  int ck[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) ck[s] = min(32 * s + 8 * g, dk - 8);
  const int cv = min(8 * lc, dv - 8);
  auto load_k = [&](const int* sl, int u) {          // keys 16 u ..
    const uint16_t* p = a.k + (size_t)sl[16 * u + n16] * dk;
#pragma unroll
    for (int s = 0; s < KS; ++s) raw[u][s] = cached_row<ONCE>(p + ck[s]);
  };
  auto load_v = [&](const int* sl, int u) {
#pragma unroll
    for (int x = 0; x < VB; ++x)
      raw[u][x] = cached_row<ONCE>(a.v + (size_t)sl[16 * u + KL * x + lg] * dv + cv);
  };
  auto add_v = [&](int u) {
#pragma unroll
    for (int x = 0; x < VB; ++x) {
      float f[8], p[R];
      unpack8(raw[u][x], f);
#pragma unroll
      for (int i = 0; i < R; ++i) p[i] = psw[(16 * u + KL * x + lg) * R + i];      // 0 past the last key
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) o[i][j] += p[i] * f[j];
    }
  };
  if (tile < t_end) {
    vs[w][0][lane] = slot0;
    meet();
#pragma unroll
    for (int u = 0; u < 4; ++u) load_k(vs[w][0], u);
    for (int cur = 0;; cur ^= 1) {
      const bool more = tile + NW < t_end;
      const int next = slot(min(tile + NW, ntiles - 1));
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (dk < D) {
#pragma unroll
          for (int s = 0; s < KS; ++s) raw[u][s] = 32 * s + 8 * g < dk ? raw[u][s] : zero;
        }
        f32x4 sc = {0.f, 0.f, 0.f, 0.f};             // keys 16 u + 4 g + i, head n16
#pragma unroll
        for (int s = 0; s < KS; ++s) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(raw[u][s]), as_bf16x8(qf[s]), sc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);           // a block's values take the place of its keys
        load_v(vs[w][cur], u);
        if (n16 < R) {
#pragma unroll
          for (int i = 0; i < 4; ++i) psw[(16 * u + 4 * g + i) * R + n16] = sc[i];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      meet();
      const int key = first + tile * 64 + lane;
      const bool ok = key <= pos;
      float p[R];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        p[i] = 0.f;
        if (i < r) {
          float s = -__builtin_inff();
          if (ok) {
            s = psw[lane * R + i] * a.scale;
            if (a.head_scale) s *= a.head_scale[kvh * r + i];
            if (a.dist_bias) s += a.dist_bias[(size_t)min(pos - key, a.n_dist - 1) * a.H + kvh * r + i];
            if (a.softcap > 0.f) s = a.softcap * tanhf(s / a.softcap);
          }
          const float m_new = fmaxf(m[i], wave_max_all(s));      // the tile's first key (lane 0) is visible: finite
          const float corr = expf(m[i] - m_new);
          p[i] = ok ? expf(s - m_new) : 0.f;
          l[i] = l[i] * corr + p[i];
          m[i] = m_new;
#pragma unroll
          for (int j = 0; j < 8; ++j) o[i][j] *= corr;
        }
      }
#pragma unroll
      for (int i = 0; i < R; ++i) psw[lane * R + i] = p[i];      // over the lane's own scores
      vs[w][cur ^ 1][lane] = next;
      meet();
      if (!more) break;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        add_v(u);
        __builtin_amdgcn_sched_barrier(0);
        load_k(vs[w][cur ^ 1], u);
        __builtin_amdgcn_sched_barrier(0);
      }
      meet();
      tile += NW;
    }
    // only a wave's last tile can end early: what is there instead of its missing values may be infinite, and 0 times that is no number
    const int n = pos - (first + tile * 64) + 1;
    if (n < 64) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int x = 0; x < VB; ++x) raw[u][x] = 16 * u + KL * x + lg < n ? raw[u][x] : zero;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      add_v(u);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // lane groups -> lane group 0, then waves -> LDS
#pragma unroll
  for (int i = 0; i < R; ++i) {
    l[i] = wave_sum(l[i]);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
#pragma unroll
      for (int s = LK; s < 64; s *= 2) o[i][j] += __shfl_xor(o[i][j], s, 64);
    }
  }
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      cm[w][i] = m[i];
      cl[w][i] = l[i];
    }
  }
  if (lg == 0) {
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) co[w][i][8 * lc + j] = o[i][j];
  }
  __syncthreads();
  for (int idx = tid; idx < r * dv; idx += 64 * NW) {
    const int i = idx / dv, d = idx - i * dv;
    const int head = kvh * r + i;
    float M = a.sinks && !a.part_o ? a.sinks[head] : -__builtin_inff();
#pragma unroll
    for (int ww = 0; ww < NW; ++ww) M = fmaxf(M, cm[ww][i]);
    float L = a.sinks && !a.part_o ? expf(a.sinks[head] - M) : 0.f, O = 0.f;      // the sink: one more term of the denominator
    if (pos < 0) {                                   // no keys at all: zeros
      M = 0.f;
      L = 1.f;
    } else if (M != -__builtin_inff()) {             // an empty run leaves zeros
#pragma unroll
      for (int ww = 0; ww < NW; ++ww) {
        const float f = expf(cm[ww][i] - M);         // waves without a tile: exp(-inf) = 0
        L += cl[ww][i] * f;
        O += co[ww][i][d] * f;
      }
    }
    if (a.part_o) {
      const size_t at = ((size_t)blockIdx.z * gridDim.x + row) * a.H + head;
      a.part_o[at * dv + d] = O;
      if (d == 0) {
        a.part_ml[2 * at] = M;
        a.part_ml[2 * at + 1] = L;
      }
      continue;
    }
    float v = O / L;
    if (a.gate) v *= 1.f / (1.f + expf(-bf16_to_f32(a.gate[(size_t)row * a.gate_stride + (a.gate_heads ? (size_t)head : (size_t)head * dv + d)])));
    a.out[(size_t)row * a.out_stride + (size_t)head * dv + d] = f32_to_bf16(v);
  }
}

// combines the runs of the two kernels above; grid (rows, H)
template <typename T>
__global__ __launch_bounds__(128) void masked_attn_reduce_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                 int nsplit, int dv, const float* __restrict__ sinks,
                                                                 const T* __restrict__ gate, int gate_stride, int gate_heads,
                                                                 T* __restrict__ out, int out_stride) {
  const int row = blockIdx.x, head = blockIdx.y, rows = gridDim.x, H = gridDim.y;
  float M = sinks ? sinks[head] : -__builtin_inff();
  for (int z = 0; z < nsplit; ++z) M = fmaxf(M, part_ml[2 * (((size_t)z * rows + row) * H + head)]);     // run 0 is never empty
  float L = sinks ? expf(sinks[head] - M) : 0.f;
  for (int z = 0; z < nsplit; ++z) {
    const size_t slot = ((size_t)z * rows + row) * H + head;
    L += part_ml[2 * slot + 1] * expf(part_ml[2 * slot] - M);
  }
  const float inv = 1.f / L;
  for (int d = threadIdx.x; d < dv; d += 128) {
    float O = 0.f;
    for (int z = 0; z < nsplit; ++z) {
      const size_t slot = ((size_t)z * rows + row) * H + head;
      O += part_o[slot * dv + d] * expf(part_ml[2 * slot] - M);
    }
    float v = O * inv;
    if (gate) v *= 1.f / (1.f + expf(-ldf<T>(gate + (size_t)row * gate_stride + (gate_heads ? (size_t)head : (size_t)head * dv + d))));
    stf<T>(out + (size_t)row * out_stride + (size_t)head * dv + d, v);
  }
}

// The same for four runs and more.  It is a launch and a chain of latencies: lane z holds run z's factor, eight runs' sums are under way at a time, the first
// eight while the factors are formed.  Four layers of one row of 16 heads of 128 dims, 8000 keys in 16 runs, 94 us with the one above, so 69; 6 runs 75, 68; 4 runs 135, 132;
// but 3 runs 92.6, 92.2 and 2 59.4, 63.1.
constexpr int MANY_RUNS = 4;
template <typename T>
__global__ __launch_bounds__(128) void masked_attn_reduce_many_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                                 int nsplit, int dv, const float* __restrict__ sinks,
                                                                 const T* __restrict__ gate, int gate_stride, int gate_heads,
                                                                 T* __restrict__ out, int out_stride) {
  constexpr int BATCH = 8;
  const int row = blockIdx.x, head = blockIdx.y, rows = gridDim.x, H = gridDim.y, lane = threadIdx.x & 63;
  auto slot = [&](int z) { return ((size_t)min(z, nsplit - 1) * rows + row) * H + head; };
  auto own = [&](int z0) {                             // maximum and sum of run z0 + lane
    const float2 e = *reinterpret_cast<const float2*>(part_ml + 2 * slot(z0 + lane));
    return z0 + lane < nsplit ? e : make_float2(-__builtin_inff(), 0.f);
  };
  float p[BATCH];
  auto load = [&](int d, int z0) {
#pragma unroll
    for (int i = 0; i < BATCH; ++i) p[i] = part_o[slot(z0 + i) * dv + min(d, dv - 1)];
  };
  const float2 e0 = own(0);
  load(threadIdx.x, 0);
  float M = e0.x;                                      // run 0 is never empty
  for (int z0 = 64; z0 < nsplit; z0 += 64) M = fmaxf(M, own(z0).x);
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
  if (sinks) M = fmaxf(sinks[head], M);
  auto factor = [&](const float2& e) { return expf(e.x - M); };      // no run: exp(-inf) = 0
  float L = e0.y * factor(e0);
  for (int z0 = 64; z0 < nsplit; z0 += 64) {
    const float2 e = own(z0);
    L += e.y * factor(e);
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) L += __shfl_xor(L, o, 64);
  if (sinks) L += expf(sinks[head] - M);
  const float inv = 1.f / L;
  for (int d0 = 0; d0 < dv; d0 += 128) {
    const int d = d0 + threadIdx.x;
    if (d0 > 0) load(d, 0);
    float O = 0.f, f = 0.f;
    for (int z0 = 0; z0 < nsplit; z0 += BATCH) {
      if ((z0 & 63) == 0) f = factor(z0 == 0 ? e0 : own(z0));
#pragma unroll
      for (int i = 0; i < BATCH; ++i)
        if (z0 + i < nsplit) O += p[i] * __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), (z0 + i) & 63));
      if (z0 + BATCH < nsplit) load(d, z0 + BATCH);
    }
    if (d >= dv) continue;
    float v = O * inv;
    if (gate) v *= 1.f / (1.f + expf(-ldf<T>(gate + (size_t)row * gate_stride + (gate_heads ? (size_t)head : (size_t)head * dv + d))));
    stf<T>(out + (size_t)row * out_stride + (size_t)head * dv + d, v);
  }
}

template <typename T>
void launch_reduce(const float* part_o, const float* part_ml, int rows, int H, int nsplit, int dv, const float* sinks, const void* gate, int gate_stride,
                   int gate_heads, void* out, int out_stride, hipStream_t s) {
  auto kernel = nsplit >= MANY_RUNS ? masked_attn_reduce_many_kernel<T> : masked_attn_reduce_kernel<T>;
  kernel<<<dim3(rows, H), 128, 0, s>>>(part_o, part_ml, nsplit, dv, sinks, (const T*)gate, gate_stride, gate_heads, (T*)out, out_stride);
}

template <int R, int D>
void launch_tiles_dims(const RowsArgs& a, int rows, int G, int nsplit, hipStream_t s) {
  // A workgroup per compute unit or fewer: eight waves each (30 rows of 2000 keys, 8 groups of 4 heads of 64 dims: 14.9 us, with four
  // waves 16.8); more of them: four, so that more workgroups share a unit (128 rows of 500 keys, groups of 2: 30.4, with eight 30.9).
  // Where nearly all units have work to the end, cached rows are marked as read once (8 groups of 4 heads of 128 dims, us marked and not: 32
  // rows of 2000 keys 54.9, 56.6, 31 rows 54.2, 55.8, 64 of 1000 52.2, 54.3, 100 of 300 30.6, 32.2).  Where some wait for others, each
  // reads faster without the mark (20 rows of 2000 49.0, 44.2, 28 of 1000 28.0, 27.3; 36 rows of 2000, 64 heads 93.8, 85.4, 40 of 64 dims 47.7,
  // 43.6), and smaller steps' rows the caches may still hold (4 rows of 300 11.9, 11.4).
  const long long units = (long long)rows * G * nsplit;
  const dim3 grid(rows, G, nsplit);
  if (units >= 448) masked_attn_tiles_kernel<R, D, 4, true><<<grid, 256, 0, s>>>(a);
  else if (units > 256) masked_attn_tiles_kernel<R, D, 4, false><<<grid, 256, 0, s>>>(a);
  else if (units >= 240) masked_attn_tiles_kernel<R, D, 8, true><<<grid, 512, 0, s>>>(a);
  else masked_attn_tiles_kernel<R, D, 8, false><<<grid, 512, 0, s>>>(a);
}

template <int R>
void launch_tiles_heads(const RowsArgs& a, int rows, int G, int nsplit, hipStream_t s) {
  if (a.dk <= 64 && a.dv <= 64) launch_tiles_dims<R, 64>(a, rows, G, nsplit, s);
  else launch_tiles_dims<R, 128>(a, rows, G, nsplit, s);
}

void launch_tiles(RowsArgs a, int rows, int G, int nsplit, hipStream_t s) {
  const int r = a.H / G;
  if (nsplit < 2) a.part_o = a.part_ml = nullptr;
  if (r <= 2) launch_tiles_heads<2>(a, rows, G, nsplit, s);
  else if (r <= 4) launch_tiles_heads<4>(a, rows, G, nsplit, s);
  else launch_tiles_heads<8>(a, rows, G, nsplit, s);
  if (nsplit > 1)
    launch_reduce<uint16_t>(a.part_o, a.part_ml, rows, a.H, nsplit, a.dv, a.sinks, a.gate, a.gate_stride, a.gate_heads, a.out, a.out_stride, s);
}

template <typename T, int R, int VP>
int launch_group(const void* q, int q_stride, const void* k_cache, const void* v_cache, const int* block_tables,
                 int bt_stride, const int* cu_seqlens, int n_seqs, const int* positions, int rows, int H, int G, int dk,
                 int dv, int bs, float scale, int mask, const void* gate, int gate_stride, void* out, int out_stride,
                 const float* dist_bias, int n_dist, float softcap, const float* sinks, const float* head_scale, int gate_heads,
                 int nsplit, float* part_o, float* part_ml, hipStream_t s) {
  const size_t lds = (size_t)(R * dk + GNW * R * 64 + GNW * 64 + 2 * GNW * R + GNW * R * dv) * 4;
  if (lds > 64 * 1024) return -1;
  if (nsplit < 2) part_o = part_ml = nullptr;
  masked_attn_group_kernel<T, R, VP><<<dim3(rows, G, nsplit), 64 * GNW, lds, s>>>(
      (const T*)q, q_stride, (const T*)k_cache, (const T*)v_cache, block_tables, bt_stride, cu_seqlens, n_seqs,
      positions, H, dk, dv, bs, scale, mask, (const T*)gate, gate_stride, (T*)out, out_stride, dist_bias, n_dist,
      softcap, sinks, head_scale, gate_heads, part_o, part_ml);
  if (nsplit > 1)
    launch_reduce<T>(part_o, part_ml, rows, H, nsplit, dv, sinks, gate, gate_stride, gate_heads, out, out_stride, s);
  return 0;
}

template <typename T>
int dispatch_group(int r, int vpn, const void* q, int q_stride, const void* k_cache, const void* v_cache,
                   const int* block_tables, int bt_stride, const int* cu_seqlens, int n_seqs, const int* positions,
                   int rows, int H, int G, int dk, int dv, int bs, float scale, int mask, const void* gate,
                   int gate_stride, void* out, int out_stride, const float* dist_bias, int n_dist, float softcap,
                   const float* sinks, const float* head_scale, int gate_heads, int nsplit, float* part_o, float* part_ml, hipStream_t s) {
#define DGI_GRP(RV, VPV)                                                                                       \
  return launch_group<T, RV, VPV>(q, q_stride, k_cache, v_cache, block_tables, bt_stride, cu_seqlens, n_seqs, \
                                  positions, rows, H, G, dk, dv, bs, scale, mask, gate, gate_stride, out, out_stride, dist_bias, \
                                  n_dist, softcap, sinks, head_scale, gate_heads, nsplit, part_o, part_ml, s)
  if constexpr (sizeof(T) == 4) {                    // bf16 heads of up to 128 dims: masked_attn_tiles_kernel
    if (vpn == 1) {
      if (r == 1) DGI_GRP(1, 1);
      if (r == 2) DGI_GRP(2, 1);
      if (r <= 4) DGI_GRP(4, 1);
      DGI_GRP(8, 1);
    }
  }
  if (r == 1) DGI_GRP(1, 2);
  if (r == 2) DGI_GRP(2, 2);
  if (r <= 4) DGI_GRP(4, 2);
  DGI_GRP(8, 2);
#undef DGI_GRP
}

}  // namespace

// q / gate / out: row-major with their own row strides (elements); cu_seqlens (n_seqs + 1 row
// offsets) maps rows to block-table rows, nullptr: row i uses block-table row i.  nsplit > 1: runs of keys per row for
// the grouped kernel (the other one takes a row in one go), with part_o [nsplit, rows, H, dv] and part_ml
// [nsplit, rows, H, 2] fp32 to meet in.
extern "C" int dgi_masked_attn_rows(const void* q, int q_stride, const void* k_cache, const void* v_cache,
                                    const int* block_tables, int bt_stride, const int* cu_seqlens, int n_seqs,
                                    const int* positions, int rows, int H, int G, int dk, int dv, int block_size,
                                    float scale, int mask, const void* gate, int gate_stride, void* out,
                                    int out_stride, int is_f32, const float* dist_bias, int n_dist, float softcap,
                                    const float* sinks, const float* head_scale, int gate_heads, int nsplit, float* part_o,
                                    float* part_ml, hipStream_t s) {
  if (rows == 0) return 0;
  if (G <= 0 || H % G) return -2;
  if (dk > MAXDK || dv > 64 * MAXC || dk <= 0 || dv <= 0) return -3;
  if (H > 65535) return -4;
  if (nsplit < 1 || nsplit > 65535 || (nsplit > 1 && (!part_o || !part_ml))) return -6;
  if (dist_bias && n_dist < 1) return -5;
  {
    // grouped kernels where the geometry allows (see masked_attn_tiles_kernel and masked_attn_group_kernel)
    const int E = is_f32 ? 4 : 8, r = H / G;
    const int vpn = (std::max(dk, dv) + 16 * E - 1) / (16 * E);
    const bool aligned = ((uintptr_t)k_cache | (uintptr_t)v_cache) % 16 == 0;
    if (!is_f32 && dk % 8 == 0 && dv % 8 == 0 && r <= 8 && vpn == 1 && aligned && G <= 65535) {
      RowsArgs a;
      a.q = (const uint16_t*)q; a.k = (const uint16_t*)k_cache; a.v = (const uint16_t*)v_cache; a.gate = (const uint16_t*)gate;
      a.out = (uint16_t*)out;
      a.block_tables = block_tables; a.cu_seqlens = cu_seqlens; a.positions = positions;
      a.dist_bias = dist_bias; a.sinks = sinks; a.head_scale = head_scale;
      a.part_o = part_o; a.part_ml = part_ml;
      a.q_stride = q_stride; a.bt_stride = bt_stride; a.n_seqs = n_seqs; a.H = H; a.dk = dk; a.dv = dv; a.bs = block_size; a.mask = mask;
      a.gate_stride = gate_stride; a.out_stride = out_stride; a.n_dist = n_dist; a.gate_heads = gate_heads;
      a.scale = scale; a.softcap = softcap;
      launch_tiles(a, rows, G, nsplit, s);
      DGI_CHECK_LAUNCH();
      return 0;
    }
    if (dk % E == 0 && dv % E == 0 && r <= 8 && vpn <= 2 && r * dv <= 1024 && aligned && G <= 65535) {
      const int rc = is_f32 ? dispatch_group<float>(r, vpn, q, q_stride, k_cache, v_cache, block_tables, bt_stride, cu_seqlens,
                                                    n_seqs, positions, rows, H, G, dk, dv, block_size, scale, mask, gate,
                                                    gate_stride, out, out_stride, dist_bias, n_dist, softcap, sinks, head_scale,
                                                    gate_heads, nsplit, part_o, part_ml, s)
                            : dispatch_group<uint16_t>(r, vpn, q, q_stride, k_cache, v_cache, block_tables, bt_stride,
                                                       cu_seqlens, n_seqs, positions, rows, H, G, dk, dv, block_size, scale,
                                                       mask, gate, gate_stride, out, out_stride, dist_bias, n_dist, softcap,
                                                       sinks, head_scale, gate_heads, nsplit, part_o, part_ml, s);
      if (rc == 0) {
        DGI_CHECK_LAUNCH();
        return 0;
      }
    }
  }
  const dim3 grid(rows, H);
  if (is_f32)
    masked_attn_rows_kernel<float><<<grid, 64, 0, s>>>(
        (const float*)q, q_stride, (const float*)k_cache, (const float*)v_cache, block_tables, bt_stride, cu_seqlens,
        n_seqs, positions, G, dk, dv, block_size, scale, mask, (const float*)gate, gate_stride, (float*)out, out_stride,
        dist_bias, n_dist, softcap, sinks, head_scale, gate_heads);
  else
    masked_attn_rows_kernel<uint16_t><<<grid, 64, 0, s>>>(
        (const uint16_t*)q, q_stride, (const uint16_t*)k_cache, (const uint16_t*)v_cache, block_tables, bt_stride,
        cu_seqlens, n_seqs, positions, G, dk, dv, block_size, scale, mask, (const uint16_t*)gate, gate_stride,
        (uint16_t*)out, out_stride, dist_bias, n_dist, softcap, sinks, head_scale, gate_heads);
  DGI_CHECK_LAUNCH();
  return 0;
}
