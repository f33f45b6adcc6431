// dgi/csrc/mix/latent_decode.hip — the two products around attention over cached latents, for steps of few rows (bf16):
//
//   latent_fold    q_lat[h][t] = uk[h]^T q[t][h][:dim]      the unrotated query part through the key up-projection uk [H, dim, kr]
//   latent_values  out[t][h]   = uv[h] o[h][t]              the weighted latent sums through the value up-projection uv [H, vdim, kr],
//                                                           times sigmoid(gate), heads side by side
//
// Both are bounded by launches and latency (2 MB and 4 MB of weights at 32 heads of 64 + 128 dims on 512), not by work: the
// library's batched products took 12 and 5 us for 32 rows, and between them and after them ran a pass that combines the
// runs of keys and one that puts the heads side by side.  latent_values reads the runs' partial sums itself.
#include <cfloat>

#include "../common.h"

using namespace dgi;

namespace {

// A workgroup owns a head and 64 latent dims, wave w 16 of them; its slab of uk lies in LDS and is read transposed (the
// product's A operand: latent dims by query dims).  DS = dim / 32 steps; rows sixteen at a time.
template <int DS>
__global__ __launch_bounds__(256) void latent_fold_kernel(uint16_t* __restrict__ q_lat, const uint16_t* __restrict__ q, int q_stride,
                                                          const uint16_t* __restrict__ uk, int T, int qk, int kr) {
  constexpr int DIM = 32 * DS;
  __shared__ __attribute__((aligned(16))) uint16_t slab[DIM * 64];
  const int head = blockIdx.x, c0 = blockIdx.y * 64;
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  u32x4 v[DS];
  const uint16_t* src = uk + (size_t)head * DIM * kr + c0;
#pragma unroll
  for (int i = 0; i < DS; ++i) {
    const int idx = threadIdx.x + 256 * i;                 // chunk of eight: row idx / 8
    v[i] = *reinterpret_cast<const u32x4*>(src + (size_t)(idx >> 3) * kr + (idx & 7) * 8);
  }
  const uint16_t* qp = q + (size_t)head * qk + 8 * lg;
  auto load_q = [&](int t0, u32x4 (&b)[DS]) {
    const uint16_t* p = qp + (size_t)min(t0 + lr, T - 1) * q_stride;
#pragma unroll
    for (int s = 0; s < DS; ++s) b[s] = *reinterpret_cast<const u32x4*>(p + 32 * s);
  };
  u32x4 b[DS];
  load_q(0, b);
#pragma unroll
  for (int i = 0; i < DS; ++i) *reinterpret_cast<u32x4*>(slab + (threadIdx.x + 256 * i) * 8) = v[i];
  __syncthreads();
  const int tq = lr >> 2, tp = lr & 3;
  u32x4 a[DS];
#pragma unroll
  for (int s = 0; s < DS; ++s) {
    const uint16_t* p = slab + (32 * s + 8 * lg + tq) * 64 + 16 * w + 4 * tp;
    const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)p);
    const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(p + 4 * 64));
    a[s][0] = (uint32_t)(uint16_t)lo[0] | ((uint32_t)(uint16_t)lo[1] << 16);
    a[s][1] = (uint32_t)(uint16_t)lo[2] | ((uint32_t)(uint16_t)lo[3] << 16);
    a[s][2] = (uint32_t)(uint16_t)hi[0] | ((uint32_t)(uint16_t)hi[1] << 16);
    a[s][3] = (uint32_t)(uint16_t)hi[2] | ((uint32_t)(uint16_t)hi[3] << 16);
  }
  for (int t0 = 0; t0 < T; t0 += 16) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DS; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[s]), as_bf16x8(b[s]), acc, 0, 0, 0);
    if (t0 + 16 < T) load_q(t0 + 16, b);
    if (t0 + lr < T)
      *reinterpret_cast<uint2*>(q_lat + ((size_t)head * T + t0 + lr) * kr + c0 + 16 * w + 4 * lg) =
          make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
  }
}

// A workgroup owns a head and rb rows: 16, fewer where the step has few rows, so that 256 workgroups share the partial sums
// (32 rows of 32 heads, 8 runs: 64 workgroups that also read the runs' maxima one by one took 15.7 us, 256 so 10.5), and more than eight
// runs are shared out over the lanes that have no row of their own (8 rows of 32 runs 20.6 us -> 11.0, 1 row of 31 runs 15.4 -> 10.4; 8 runs 10.5,
// so 11.2); its eight waves take 64 of the 512 latent dims each (operands straight from
// memory), and their sums meet in LDS.  runs > 1: o comes as the partial sums of that many runs of keys (at most 64),
// [runs, H, T, 512] relative to each run's maximum (ml: maximum and sum of weights), else as o_lat [H, T, 512].  The loads of
// the weights and of the first four runs are under way while the runs' factors are formed.
constexpr int KR = 512, VMAX = 8, RUNS = 64, SHARE = 8;

template <bool SHARED>
__global__ __launch_bounds__(512) void latent_values_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ o_lat,
                                                            const float* __restrict__ part, const float* __restrict__ ml, int runs,
                                                            const float* __restrict__ sinks, const uint16_t* __restrict__ uv,
                                                            const uint16_t* __restrict__ gate, int gate_stride, int per_head, int T,
                                                            int H, int vdim, int rb) {
  __shared__ __attribute__((aligned(16))) float sums[8][VMAX][64][4];
  const int head = blockIdx.x, t0 = blockIdx.y * rb, t1 = min(t0 + rb, T);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  // SHARED: lanes past the rows take part of the runs, lane lr row lr % rb and every (16 / rb)-th run
  const int r = SHARED ? lr & (rb - 1) : lr, grp = SHARED ? lr / rb : 0, ng = SHARED ? 16 / rb : 1;
  const int t = min(t0 + r, t1 - 1), nv = vdim >> 4, k = w * 64 + 8 * lg;
  u32x4 a[VMAX][2];
  auto load_uv = [&]() {
#pragma unroll
    for (int j = 0; j < VMAX; ++j)
#pragma unroll
      for (int s = 0; s < 2; ++s)
        a[j][s] = *reinterpret_cast<const u32x4*>(uv + ((size_t)head * vdim + min(16 * j, vdim - 16) + lr) * KR + k + 32 * s);
  };
  u32x4 b[2];
  if (runs > 1) {
    const size_t next = (size_t)H * T, first = (size_t)head * T + t;
    // factors e^(m - M) / L of every run and row, through LDS (rows [z][16], then 1 / L)
    float (*fac)[16] = reinterpret_cast<float (*)[16]>(&sums[0][0][0][0]);
    float* len = &sums[1][0][0][0];                        // [RUNS][16]
    constexpr int PER = RUNS * 16 / 512;
    float2 e[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = threadIdx.x + 512 * i, z = min(idx >> 4, runs - 1), tt = min(t0 + (idx & 15), t1 - 1);
      e[i] = *reinterpret_cast<const float2*>(ml + 2 * ((size_t)z * next + (size_t)head * T + tt));
    }
    float4 p[4][2][2];
    auto load_runs = [&](int z0) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float* src = part + (first + (size_t)min(z0 + u * ng + grp, runs - 1) * next) * KR + k;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i) p[u][s][i] = *reinterpret_cast<const float4*>(src + 32 * s + 4 * i);
      }
    };
    load_runs(0);
    load_uv();
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int idx = threadIdx.x + 512 * i;
      (&fac[0][0])[idx] = e[i].x;
      len[idx] = e[i].y;
    }
    __syncthreads();
    float M = -FLT_MAX, L = 0.f;                           // of this lane's row; finite also where no run has keys
    for (int z = grp; z < runs; z += ng) M = fmaxf(M, fac[z][r]);
    if constexpr (SHARED)
      for (int o = rb; o < 16; o <<= 1) M = fmaxf(M, __shfl_xor(M, o, 64));
    for (int z = grp; z < runs; z += ng) L += len[z * 16 + r] * expf(fac[z][r] - M);
    if constexpr (SHARED)
      for (int o = rb; o < 16; o <<= 1) L += __shfl_xor(L, o, 64);
    float inv = L == 0.f ? 0.f : 1.f / L;
    if (sinks) {                                           // one more logit in the denominator, relative to the larger of the two
      const float sink = sinks[head], top = fmaxf(M, sink), f = expf(M - top);
      inv = f / (L * f + expf(sink - top));
    }
    float x[2][8];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) x[s][i] = 0.f;
    for (int z0 = 0; z0 < runs; z0 += 4 * ng) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int z = z0 + u * ng + grp;
        const float f = z < runs ? expf(fac[min(z, runs - 1)][r] - M) : 0.f;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            x[s][4 * i] += p[u][s][i].x * f; x[s][4 * i + 1] += p[u][s][i].y * f;
            x[s][4 * i + 2] += p[u][s][i].z * f; x[s][4 * i + 3] += p[u][s][i].w * f;
          }
      }
      if (z0 + 4 * ng < runs) load_runs(z0 + 4 * ng);
    }
    if constexpr (SHARED)
      for (int o = rb; o < 16; o <<= 1)
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int i = 0; i < 8; ++i) x[s][i] += __shfl_xor(x[s][i], o, 64);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int i = 0; i < 8; ++i) x[s][i] *= inv;
      b[s] = pack8(x[s]);
    }
    __syncthreads();                                       // the factors are read before the sums take their place
  } else {
#pragma unroll
    for (int s = 0; s < 2; ++s) b[s] = *reinterpret_cast<const u32x4*>(o_lat + ((size_t)head * T + t) * KR + k + 32 * s);
    load_uv();
  }
#pragma unroll
  for (int j = 0; j < VMAX; ++j) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[j][s]), as_bf16x8(b[s]), acc, 0, 0, 0);
    *reinterpret_cast<f32x4*>(sums[w][j][lane]) = acc;
  }
  __syncthreads();
  if (w >= nv || t0 + lr >= t1) return;                    // wave w finishes value dims 16 w .. + 15; no barrier follows
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int ww = 0; ww < 8; ++ww) {
    const f32x4 p = *reinterpret_cast<const f32x4*>(sums[ww][w][lane]);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] += p[i];
  }
  const int c = head * vdim + 16 * w + 4 * lg;
  if (gate) {
    const uint16_t* gp = gate + (size_t)t * gate_stride;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= 1.f / (1.f + expf(-bf16_to_f32(gp[per_head ? head : c + i])));
  }
  *reinterpret_cast<uint2*>(out + (size_t)t * H * vdim + c) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}

}  // namespace

// q [T, >= H * qk] (the first dim entries of a head are used), uk [H, dim, kr], q_lat [H, T, kr]; 16-byte rows throughout
extern "C" int dgi_latent_fold(void* q_lat, const void* q, int q_stride, const void* uk, int T, int H, int dim, int qk, int kr,
                               hipStream_t s) {
  if (T == 0) return 0;
  if (H <= 0 || dim % 32 || dim < 32 || dim > 128 || kr % 64 || qk % 8 || q_stride % 8 || (((uintptr_t)q | (uintptr_t)uk) & 15) ||
      ((uintptr_t)q_lat & 7))
    return -2;
  const dim3 grid(H, kr / 64);
#define DGI_LF(N_)                                                                                                             \
  latent_fold_kernel<N_><<<grid, 256, 0, s>>>((uint16_t*)q_lat, (const uint16_t*)q, q_stride, (const uint16_t*)uk, T, qk, kr)
  switch (dim / 32) {
    case 1: DGI_LF(1); break;
    case 2: DGI_LF(2); break;
    case 3: DGI_LF(3); break;
    default: DGI_LF(4);
  }
#undef DGI_LF
  DGI_CHECK_LAUNCH();
  return 0;
}

// o_lat [H, T, 512] or, with runs > 1, part [runs, H, T, 512] and ml [runs, H, T, 2]; uv [H, vdim, 512]; out [T, H * vdim]
extern "C" int dgi_latent_values(void* out, const void* o_lat, const float* part, const float* ml, int runs, const float* sinks,
                                 const void* uv, const void* gate, int gate_stride, int per_head, int T, int H, int vdim,
                                 hipStream_t s) {
  if (T == 0) return 0;
  if (H <= 0 || vdim % 16 || vdim < 16 || vdim > 16 * VMAX || runs < 1 || runs > RUNS || (runs > 1 ? !part || !ml : !o_lat)) return -2;
  if ((((uintptr_t)uv | (uintptr_t)o_lat | (uintptr_t)part) & 15) || ((uintptr_t)out & 7) || ((uintptr_t)ml & 7)) return -3;
  int rb = 16;
  while (rb > 1 && ((long long)H * ((T + rb - 1) / rb) < 256 || rb / 2 >= T)) rb >>= 1;       // fewer rows each while compute units are left over
  if ((T + rb - 1) / rb > 65535) return -4;
  auto kernel = runs > SHARE && rb < 16 ? latent_values_kernel<true> : latent_values_kernel<false>;
  kernel<<<dim3(H, (T + rb - 1) / rb), 512, 0, s>>>((uint16_t*)out, (const uint16_t*)o_lat, part, ml, runs, sinks, (const uint16_t*)uv,
                                                    (const uint16_t*)gate, gate_stride, per_head, T, H, vdim, rb);
  DGI_CHECK_LAUNCH();
  return 0;
}
