// dgi/csrc/stream_gemm.hip — products of few rows (a decode step's batch) with weights that are read once.
//
//   stream_gemm        y[m][n] = x[m] . w[n] (+ bias), m < M <= 128, as bf16; as SwiGLU over w = [gate; up]; or, with K cut into parts
//                      that run side by side, as fp32 partial sums [part][M][N] for one of the kernels below, which read them where
//                      they would have read y:
//   add_rmsnorm_parts  x = bf16(sum of the parts), residual += x, out = rmsnorm(residual) * gamma
//   rope_cache_parts   q and k rotated, q to rows, k and v to the paged cache (rope_cache.hip)
//   sum_parts          y
//
// stream_gemm is bounded by the weights' bytes.  A unit is 128 weight rows (GLU: 64 outputs, gate and up rows interleaved so that both
// projections of an output meet in one lane) and one part of K; a workgroup per compute unit takes units in turn, its eight waves
// own 16 of the rows each and share the rows of x.  Both come straight to LDS in stages of 64 of K, some six ahead, a load 8 rows x
// 128 bytes: whole lines, which one compute unit reads at 54 GB/s (16 rows x 64 bytes, the products' own order: 37).  Narrow
// projections are cut along K until there are some 256 units, each with one part of x, so that the rows of x are read once per
// 128 rows of weights; the parts cost no pass of their own.  What the memory's rate hangs on (28672 x 4096, reads alone): loads marked
// as read once 46 us, not 50, and units that each start at a stage of their own 36; part by part, not tile by tile, so that an
// XCD's workgroups spread over the parts (8192 x 8192 in 4 parts: 29 -> 23).
//
// Rows, and times in us against the vendor's product (x and weights cold; + the passes that it needs and these do without):
//                       1             16            64            96            128
//   28672 x 4096  GLU   38.5 (63+4.6) 38.6 (65+4.6) 41 (52+4.6)   48 (54+4.6)   53.5 (54.5+4.6)
//   4096 x 14336  parts 21 (27)       21 (27)       23 (39)       27 (63)       29 (75)
//   6144 x 4096   parts 10.5 (14.5)   11 (14.4)     13 (18)       15 (23)       17 (25)
//   4096 x 4096   parts 8.1 (15)      8.8 (16)      10.4 (15)     12 (22)       13 (24)
//   128256 x 4096       158 (187)     155 (190)     179 (208)     205 (224)     227 (233)
//   57344 x 8192  GLU   147 (178+5)   143 (179+5)   154 (184+5)   181 (189+5)   205 (192+5)
#include "common.h"

#include <type_traits>

using namespace dgi;

namespace {

struct StreamArgs {
  const uint16_t* x;
  const uint16_t* w;
  const uint16_t* bias;
  void* out;                                           // bf16 [M, ldo], or fp32 [parts, M, N]
  long long ldx, ldo;
  int M, N, K, parts, per;                             // N: outputs; per: stages of a part
};

enum { ROWS = 0, GLU = 1, PARTS = 2 };

__device__ __forceinline__ void load_lds16(const char* src, char* lds) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// the same for data that nothing reads again soon (nt): the chip's caches give it up first
__device__ __forceinline__ void load_lds16_once(const char* src, char* lds) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds, 16, 0, 2);
}

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// MB: blocks of 16 rows of x; D: stages in LDS
template <int MB, int D, int MODE>
__global__ __launch_bounds__(512) void stream_gemm_kernel(const StreamArgs a) {
  constexpr int STAGE = (16 + 2 * MB) * 1024;          // 128 rows of weights, 16 MB rows of x, 128 bytes each
  constexpr int CA = (2 * MB + 7) / 8, PER = 2 + CA;   // a wave's loads of x, all its loads of a stage
  __shared__ __attribute__((aligned(16))) char lds[D * STAGE];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  constexpr int NO = MODE == GLU ? 64 : 128;
  const int tiles = (a.N + NO - 1) / NO, units = tiles * a.parts;     // (part of K, tile of weight rows)
  // piece c of LDS row r is piece c ^ (r & 7) of the row's 64 elements: reads of 8 rows spread over all banks
  const int row8 = lane >> 3, piece = ((lane & 7) ^ row8) << 4;
  int xi[CA];
#pragma unroll
  for (int i = 0; i < CA; ++i) xi[i] = (w + 8 * i) % (2 * MB);       // where there are fewer than 8 CA, some waves load the same
  auto stages = [&](int u) { return min(a.per, (a.K >> 6) - u / tiles * a.per); };
  // the loader is D - 1 stages ahead, also across the units
  const char *wp[2], *xp[CA];
  int l_unit = blockIdx.x, l_left = 0, l_wrap = 0, l_slot = 0;
  auto load = [&]() {
    if (l_left == 0) {
      if (l_unit >= units) return false;
      // a unit starts at a stage of its own and comes round to the stages before: workgroups in step with each other would read
      // the same offset of rows that are all the same power of two apart, from a few channels of the memory at a time
      l_left = stages(l_unit);
      const int first = (l_unit + (l_unit >> 3)) % l_left;
      l_wrap = l_left - first;
      const size_t koff = (size_t)(l_unit / tiles * a.per + first) * 128 + piece;
      const int n0 = l_unit % tiles * NO;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = 16 * w + 8 * i + row8;
        const int n = min(n0 + (MODE == GLU ? 2 * (r >> 2) + (r & 1) : r), a.N - 1) + (MODE == GLU && (r & 2) ? a.N : 0);
        wp[i] = reinterpret_cast<const char*>(a.w + (size_t)n * a.K) + koff;
      }
#pragma unroll
      for (int i = 0; i < CA; ++i) xp[i] = reinterpret_cast<const char*>(a.x + (size_t)min(8 * xi[i] + row8, a.M - 1) * a.ldx) + koff;
    }
    char* st = lds + l_slot * STAGE;
#pragma unroll
    for (int i = 0; i < 2; ++i) load_lds16_once(wp[i], st + (2 * w + i) * 1024);
#pragma unroll
    for (int i = 0; i < CA; ++i) load_lds16(xp[i], st + 16384 + xi[i] * 1024);
    const long long step = --l_wrap == 0 ? 128 - 128ll * stages(l_unit) : 128;
#pragma unroll
    for (int i = 0; i < 2; ++i) wp[i] += step;
#pragma unroll
    for (int i = 0; i < CA; ++i) xp[i] += step;
    if (--l_left == 0) l_unit += gridDim.x;
    l_slot = l_slot + 1 == D ? 0 : l_slot + 1;
    return true;
  };
  const int at0 = lr * 128 + ((lg ^ (lr & 7)) << 4), at1 = lr * 128 + (((4 + lg) ^ (lr & 7)) << 4);
  bool more = false;                                   // D - 1 stages are under way; uniform over the workgroup
#pragma unroll
  for (int s = 0; s < D - 1; ++s) more = load();
  int slot = 0;
  for (int unit = blockIdx.x; unit < units; unit += gridDim.x) {
    f32x4 acc[MB];
#pragma unroll
    for (int i = 0; i < MB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = stages(unit); s > 0; --s) {
      if (more) wait_loads<(D - 2) * PER>();
      else wait_loads<0>();
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      more = load();                                   // into the stage that every wave has read before the barrier
      const char* st = lds + slot * STAGE;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int at = h ? at1 : at0;
        const bf16x8 fw = *reinterpret_cast<const bf16x8*>(st + w * 2048 + at);
        bf16x8 fx[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i) fx[i] = *reinterpret_cast<const bf16x8*>(st + 16384 + i * 2048 + at);
#pragma unroll
        for (int i = 0; i < MB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw, fx[i], acc[i], 0, 0, 0);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    const int n0 = unit % tiles * NO;
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const int m = 16 * i + lr;
      if (m >= a.M) continue;
      if constexpr (MODE == GLU) {
        const int n = n0 + 8 * w + 2 * lg;             // N is even
        if (n < a.N) {
          float v[2];
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            // as silu_mul on bf16 rows
            const float g = bf16_to_f32(f32_to_bf16(acc[i][j])), u = bf16_to_f32(f32_to_bf16(acc[i][2 + j]));
            v[j] = g * __builtin_amdgcn_rcpf(1.f + __expf(-g)) * u;
          }
          *reinterpret_cast<uint32_t*>(reinterpret_cast<uint16_t*>(a.out) + (size_t)m * a.ldo + n) = pack_bf16x2(v[0], v[1]);
        }
      } else {
        const int n = n0 + 16 * w + 4 * lg;            // N is a multiple of 4
        if (n < a.N) {
          if constexpr (MODE == PARTS) {
            *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.out) + ((size_t)(unit / tiles) * a.M + m) * a.N + n) = acc[i];
          } else {
            float v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = acc[i][j] + (a.bias ? bf16_to_f32(a.bias[n + j]) : 0.f);
            *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.out) + (size_t)m * a.ldo + n) =
                make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
          }
        }
      }
    }
  }
}

template <int MODE>
int launch(const StreamArgs& a, hipStream_t s) {
  const int tiles = (a.N + (MODE == GLU ? 63 : 127)) / (MODE == GLU ? 64 : 128);
  const long long units = (long long)tiles * a.parts;
  if (units > 0x3fffffff) return -4;
  const int grid = (int)(units < 256 ? units : 256);   // one workgroup a compute unit
  if (a.M <= 16) stream_gemm_kernel<1, 8, MODE><<<grid, 512, 0, s>>>(a);
  else if (a.M <= 32) stream_gemm_kernel<2, 7, MODE><<<grid, 512, 0, s>>>(a);
  else if (a.M <= 48) stream_gemm_kernel<3, 6, MODE><<<grid, 512, 0, s>>>(a);
  else if (a.M <= 64) stream_gemm_kernel<4, 6, MODE><<<grid, 512, 0, s>>>(a);
  else if (a.M <= 96) stream_gemm_kernel<6, 5, MODE><<<grid, 512, 0, s>>>(a);
  else stream_gemm_kernel<8, 5, MODE><<<grid, 512, 0, s>>>(a);
  return 0;
}

// eight neighbouring sums over the parts, part 0 first, rounded to bf16 as a product's output is
__device__ __forceinline__ void sum_parts8(const float* p, size_t stride, int parts, float* v) {
  float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
  for (int i = 1; i < parts; ++i) {
    const float4 a = *reinterpret_cast<const float4*>(p + i * stride), b = *reinterpret_cast<const float4*>(p + i * stride + 4);
    lo.x += a.x; lo.y += a.y; lo.z += a.z; lo.w += a.w;
    hi.x += b.x; hi.y += b.y; hi.z += b.z; hi.w += b.w;
  }
  v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
  v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
}

template <int NC>
__global__ __launch_bounds__(256) void add_rmsnorm_parts_kernel(uint16_t* __restrict__ out, const float* __restrict__ parts, int nparts,
                                                                uint16_t* __restrict__ residual, const uint16_t* __restrict__ gamma, int H,
                                                                float eps) {
  const int row = blockIdx.x, tid = threadIdx.x, nchunk = H >> 3;
  const size_t stride = (size_t)gridDim.x * H;
  const float* p = parts + (size_t)row * H;
  u32x4* rr = reinterpret_cast<u32x4*>(residual + (size_t)row * H);
  float v[NC][8];
  u32x4 ra[NC], ga[NC];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = tid + c * 256;
    if (i < nchunk) {
      ra[c] = rr[i];
      ga[c] = reinterpret_cast<const u32x4*>(gamma)[i];
      sum_parts8(p + 8 * i, stride, nparts, v[c]);
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = tid + c * 256;
    if (i < nchunk) {
      float r[8];
      unpack8(ra[c], r);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[c][j] = bf16_to_f32(f32_to_bf16(v[c][j])) + r[j];
      const u32x4 q = pack8(v[c]);                     // the residual stream is bf16
      rr[i] = q;
      unpack8(q, v[c]);
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += v[c][j] * v[c][j];
    }
  }
  __shared__ float red[4];
  ss = wave_sum(ss);
  if ((tid & 63) == 0) red[tid >> 6] = ss;
  __syncthreads();
  const float inv = rsqrtf((red[0] + red[1] + red[2] + red[3]) / (float)H + eps);
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int i = tid + c * 256;
    if (i < nchunk) {
      float g[8], o[8];
      unpack8(ga[c], g);
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = v[c][j] * inv * g[j];
      reinterpret_cast<u32x4*>(out + (size_t)row * H)[i] = pack8(o);
    }
  }
}

__global__ __launch_bounds__(256) void sum_parts_kernel(uint16_t* __restrict__ out, const float* __restrict__ parts, int nparts,
                                                        const uint16_t* __restrict__ bias, int N, size_t stride, int chunks) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= chunks) return;
  float v[8];
  sum_parts8(parts + (size_t)i * 8, stride, nparts, v);
  if (bias) {
    float b[8];
    unpack8(*reinterpret_cast<const u32x4*>(bias + (size_t)i * 8 % N), b);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] += b[j];
  }
  *reinterpret_cast<u32x4*>(out + (size_t)i * 8) = pack8(v);
}

// rope_cache_kernel on the parts of the fused q | k | v rows: NeoX pairing (mode 0) or interleaved pairs (mode 1) over the first rd dims of
// a head; q (rotated) to out [T, nh * hd], k (rotated) and v to the cache.  Items are 8 dims (mode 0: and their partners).
__global__ __launch_bounds__(256) void rope_cache_parts_kernel(uint16_t* __restrict__ out, const float* __restrict__ parts, int nparts,
                                                               const uint16_t* __restrict__ bias, const int* __restrict__ positions,
                                                               const float* __restrict__ cos_sin, int nh, int nkv, int hd, int rd, int mode,
                                                               const int* __restrict__ slot_mapping, uint16_t* __restrict__ k_cache,
                                                               uint16_t* __restrict__ v_cache, int block_size) {
  const int t = blockIdx.x, W = (nh + 2 * nkv) * hd, rhalf = rd >> 1;
  const int rot = mode == 0 ? rhalf >> 3 : rd >> 3, per = rot + ((hd - rd) >> 3), vper = hd >> 3;      // items of a q or k head, of a v head
  const size_t stride = (size_t)gridDim.x * W;
  const float* row = parts + (size_t)t * W;
  const float* cs = cos_sin + (size_t)positions[t] * rd;
  const int slot = slot_mapping[t];
  const int blk = slot >= 0 ? slot / block_size : 0, off = slot >= 0 ? slot - blk * block_size : 0;
  auto take = [&](int col, float* v) {
    sum_parts8(row + col, stride, nparts, v);
    if (bias) {
      float b[8];
      unpack8(*reinterpret_cast<const u32x4*>(bias + col), b);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] += b[j];
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = bf16_to_f32(f32_to_bf16(v[j]));
  };
  for (int it = blockIdx.y * 256 + threadIdx.x; it < (nh + nkv) * per + nkv * vper; it += 256 * gridDim.y) {
    const bool is_v = it >= (nh + nkv) * per;
    const int j = is_v ? it - (nh + nkv) * per : it;
    const int head = is_v ? nh + nkv + j / vper : j / per, c = is_v ? j % vper : j % per;
    if (head >= nh && slot < 0) continue;
    uint16_t* dst = head < nh ? out + (size_t)t * nh * hd + (size_t)head * hd
                              : (is_v ? v_cache : k_cache) + (((size_t)blk * nkv + (head - nh) % nkv) * block_size + off) * hd;
    float a[8], o[8];
    if (is_v || c >= rot) {                            // v, and dims that do not rotate
      const int d = is_v ? 8 * c : rd + 8 * (c - rot);
      take(head * hd + d, a);
      *reinterpret_cast<u32x4*>(dst + d) = pack8(a);
    } else if (mode == 0) {
      float b[8], p[8];
      take(head * hd + 8 * c, a);
      take(head * hd + rhalf + 8 * c, b);
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float co = cs[8 * c + i], si = cs[rhalf + 8 * c + i];
        o[i] = a[i] * co - b[i] * si;
        p[i] = b[i] * co + a[i] * si;
      }
      *reinterpret_cast<u32x4*>(dst + 8 * c) = pack8(o);
      *reinterpret_cast<u32x4*>(dst + rhalf + 8 * c) = pack8(p);
    } else {
      take(head * hd + 8 * c, a);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float co = cs[4 * c + i], si = cs[rhalf + 4 * c + i];
        o[2 * i] = a[2 * i] * co - a[2 * i + 1] * si;
        o[2 * i + 1] = a[2 * i + 1] * co + a[2 * i] * si;
      }
      *reinterpret_cast<u32x4*>(dst + 8 * c) = pack8(o);
    }
  }
}

}  // namespace

// mode 0: out bf16 [M, ldo]; 1: SwiGLU, w [2 N, K]; 2: fp32 parts [parts, M, N].  K a multiple of 64, N of 4, x rows and w at 16-byte
// boundaries.  A part is per stages of 64 of K; no part may be empty.
extern "C" int dgi_stream_gemm(const void* x, long long ldx, const void* w, const void* bias, void* out, long long ldo, int M, int N, int K,
                               int mode, int parts, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (M < 0 || M > 128 || N < 0 || N % 4 || K <= 0 || K % 64 || ldx % 8 || parts < 1 || parts > K / 64 || (mode != PARTS && parts != 1)) return -2;
  if ((((uintptr_t)x | (uintptr_t)w) & 15) || ((uintptr_t)out & (mode == PARTS ? 15 : 7)) || (mode != PARTS && ldo % 4)) return -3;
  StreamArgs a{(const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, out, ldx, ldo, M, N, K, parts, 0};
  a.per = (K / 64 + parts - 1) / parts;
  if ((long long)(parts - 1) * a.per >= K / 64) return -2;
  int rc;
  switch (mode) {
    case ROWS: rc = launch<ROWS>(a, s); break;
    case GLU: rc = launch<GLU>(a, s); break;
    case PARTS: rc = launch<PARTS>(a, s); break;
    default: return -2;
  }
  if (rc) return rc;
  DGI_CHECK_LAUNCH();
  return 0;
}

extern "C" int dgi_add_rmsnorm_parts(void* out, const float* parts, int nparts, void* residual, const void* gamma, int T, int H, float eps,
                                     hipStream_t s) {
  if (H % 8 || H <= 0 || nparts < 1) return -2;
  if (T == 0) return 0;
#define DGI_NORM(NC_)                                                                                                                    \
  add_rmsnorm_parts_kernel<NC_><<<T, 256, 0, s>>>((uint16_t*)out, parts, nparts, (uint16_t*)residual, (const uint16_t*)gamma, H, eps)
  const int nc = (H / 8 + 255) / 256;
  if (nc == 1) DGI_NORM(1);
  else if (nc == 2) DGI_NORM(2);
  else if (nc <= 4) DGI_NORM(4);
  else if (nc <= 8) DGI_NORM(8);
  else return -1;
#undef DGI_NORM
  DGI_CHECK_LAUNCH();
  return 0;
}

extern "C" int dgi_sum_parts(void* out, const float* parts, int nparts, const void* bias, int M, int N, hipStream_t s) {
  if (N % 8 || nparts < 1) return -2;
  const long long chunks = (long long)M * N / 8;
  if (chunks == 0) return 0;
  if (chunks > 0x3fffffff) return -4;
  sum_parts_kernel<<<(int)((chunks + 255) / 256), 256, 0, s>>>((uint16_t*)out, parts, nparts, (const uint16_t*)bias, N, (size_t)M * N, (int)chunks);
  DGI_CHECK_LAUNCH();
  return 0;
}

extern "C" int dgi_rope_cache_parts(void* out, const float* parts, int nparts, const void* bias, int T, const int* positions,
                                    const float* cos_sin, int nh, int nkv, int hd, int rd, int mode, const int* slot_mapping, void* k_cache,
                                    void* v_cache, int block_size, hipStream_t s) {
  if (hd % 8 || rd > hd || rd <= 0 || nparts < 1 || nkv <= 0) return -2;
  if ((mode == 0 && rd % 16) || (mode == 1 && rd % 8) || (mode != 0 && mode != 1)) return -3;
  if (T == 0) return 0;
  rope_cache_parts_kernel<<<dim3(T, 2), 256, 0, s>>>((uint16_t*)out, parts, nparts, (const uint16_t*)bias, positions, cos_sin, nh, nkv, hd, rd,
                                                     mode, slot_mapping, (uint16_t*)k_cache, (uint16_t*)v_cache, block_size);
  DGI_CHECK_LAUNCH();
  return 0;
}
