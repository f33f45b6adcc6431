// dgi/csrc/mix/latent_decode.hip — the two products around attention over cached latents, for steps of few rows (bf16):
//
//   latent_fold    q_lat[h][t] = uk[h]^T q[t][h][:dim]      the unrotated query part through the key up-projection uk [H, dim, kr]
//   latent_values  out[t][h]   = uv[h] o[h][t]              the weighted latent sums through the value up-projection uv [H, vdim, kr],
//                                                           times sigmoid(gate), heads side by side
//
// Both are bounded by launches and latency (2 MB and 4 MB of weights at 32 heads of 64 + 128 dims on 512), not by work: the
// library's batched products took 12 and 5 us for 32 rows, and between them and after them ran a pass that combines the
// runs of keys and one that puts the heads side by side.  latent_values reads the runs' partial sums itself.
#include <algorithm>
#include <cfloat>

#include "../common.h"

using namespace dgi;

namespace {

// A workgroup owns a head and 64 latent dims, wave w 16 of them; its slab of uk lies in LDS and is read transposed (the
// product's A operand: latent dims by query dims).  DS = dim / 32 steps; FOLD rows, sixteen at a time (128 rows of 16
// heads one behind the other 5.7 us, so 4.5).
constexpr int FOLD = 32;
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
  const int from = blockIdx.z * FOLD, to = min(T, from + FOLD);
  u32x4 b[DS];
  load_q(from, b);
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
  for (int t0 = from; t0 < to; t0 += 16) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DS; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[s]), as_bf16x8(b[s]), acc, 0, 0, 0);
    if (t0 + 16 < to) load_q(t0 + 16, b);
    if (t0 + lr < to)
      *reinterpret_cast<uint2*>(q_lat + ((size_t)head * T + t0 + lr) * kr + c0 + 16 * w + 4 * lg) =
          make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
  }
}

// A workgroup owns a head, rb rows (at most 16) and np sixteens of value dims.  runs > 1: o comes as the partial sums of that many runs of keys (at
// most 64), [runs, H, T, 512] relative to each run's maximum (ml: maximum and sum of weights), else as o_lat [H, T, 512].
//
// What bounds it is its bytes through the caches (32 rows of 32 heads, 8 runs: 17 MB of partial sums and 128 KB of uv a workgroup) and a chain of
// latencies.  The partial sums are read as they lie, four dims a thread, 128 threads a row; rows fewer than four leave their threads to
// others of the row's runs, and those sums meet in LDS.  Lane z holds run z's factor, so that nobody waits for another wave's.  The rows then go
// through LDS to the product, whose waves take sixteen value dims each over 512 / KP latent dims.  The weights, the gate and the first runs are
// under way while the factors are formed.  Before, a wave had 64 latent dims of all value dims, lanes without a row of their own read another's again, and
// few rows a workgroup meant all of uv for each: us then and now, rows x heads x runs: 32 x 32 x 8 10.7, 8.0; 3 x 16 x 6 8.6, 4.7; 8 x 16 x 32 10.7, 6.4;
// 11 x 32 x 23 18.8, 9.3; 44 x 16 x 5 16.6, 7.1; without runs 24 x 32 10.4, 4.1; 2 x 32 5.6, 4.0.
constexpr int KR = 512, RUNS = 64, BATCH = 8;

template <int KP>
__global__ __launch_bounds__(512) void latent_values_kernel(uint16_t* __restrict__ out, const uint16_t* __restrict__ o_lat,
                                                            const float* __restrict__ part, const float* __restrict__ ml, int runs,
                                                            const float* __restrict__ sinks, const uint16_t* __restrict__ uv,
                                                            const uint16_t* __restrict__ gate, int gate_stride, int per_head, int T,
                                                            int H, int vdim, int rb, int np) {
  constexpr int NS = KR / 32 / KP, ROW = KR + 8;           // steps of 32 latent dims; a row in LDS, banks apart
  __shared__ __attribute__((aligned(16))) uint16_t rows[16][ROW];
  __shared__ __attribute__((aligned(16))) float4 others[3][KR / 4];      // rows whose runs are shared: at most three times 512 dims
  __shared__ __attribute__((aligned(16))) f32x4 sums[KP > 1 ? 8 : 1][64];
  const int head = blockIdx.x, t0 = blockIdx.y * rb, nr = min(rb, T - t0);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, lr = lane & 15, lg = lane >> 4;
  const int j = w % np, kp = w / np;                       // of the product: value dims 16 (blockIdx.z np + j), dims 512 / KP kp
  const bool multiplies = kp < KP;
  const int v0 = 16 * (blockIdx.z * np + j), k = min(kp, KP - 1) * (KR / KP) + 8 * lg;
  u32x4 a[NS];
  auto load_uv = [&]() {
#pragma unroll
    for (int s = 0; s < NS; ++s) a[s] = *reinterpret_cast<const u32x4*>(uv + ((size_t)head * vdim + v0 + lr) * KR + k + 32 * s);
  };
  const int c = head * vdim + v0 + 4 * lg;
  uint16_t gates[4] = {0, 0, 0, 0};
  auto load_gate = [&]() {
    if (!gate || kp > 0) return;
    const uint16_t* gp = gate + (size_t)(t0 + min(lr, nr - 1)) * gate_stride;
#pragma unroll
    for (int i = 0; i < 4; ++i) gates[i] = gp[per_head ? head : c + i];
  };
  u32x4 b[NS];
  if (runs > 1) {
    const int apart = min(rb, 4), sharers = 4 / apart;     // rows at a time, groups of threads of a row
    const int group = w >> 1, sub = group / apart, col = threadIdx.x & 127;
    const size_t next = (size_t)H * T;
    float4 p[BATCH];
    auto load_runs = [&](int r, int i0) {                  // the batch of this group's runs, sub + sharers i
      const float* src = part + ((size_t)head * T + t0 + min(r, nr - 1)) * KR + 4 * col;
#pragma unroll
      for (int i = 0; i < BATCH; ++i) p[i] = *reinterpret_cast<const float4*>(src + (size_t)min(sub + (i0 + i) * sharers, runs - 1) * next * KR);
    };
    int r = group % apart;
    auto load_ml = [&](int r) {
      return *reinterpret_cast<const float2*>(ml + 2 * ((size_t)min(lane, runs - 1) * next + (size_t)head * T + t0 + min(r, nr - 1)));
    };
    float2 e = load_ml(r);
    load_runs(r, 0);
    load_uv();
    load_gate();
    for (; r < rb; r += apart) {
      const float m = lane < runs ? e.x : -__builtin_inff();
      float M = fmaxf(m, -FLT_MAX);                        // finite also where no run has keys
      // few runs: the lanes that have them; a loop of more turns costs what it saves
      auto turns = [&](auto f) {
        if (runs > 8) {
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) f(o);
        } else {
          for (int o = 1; o < runs; o <<= 1) f(o);
        }
      };
      turns([&](int o) { M = fmaxf(M, __shfl_xor(M, o, 64)); });
      const float f = expf(m - M);
      float L = lane < runs ? e.y * f : 0.f;
      turns([&](int o) { L += __shfl_xor(L, o, 64); });
      float inv = L == 0.f ? 0.f : 1.f / L;
      if (sinks) {                                         // one more logit in the denominator, relative to the larger of the two
        const float sink = sinks[head], top = fmaxf(M, sink), g = expf(M - top);
        inv = g / (L * g + expf(sink - top));
      }
      inv = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(inv), 0));
      const bool more = r + apart < rb;
      if (more) e = load_ml(r + apart);
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int i0 = 0; sub + i0 * sharers < runs; i0 += BATCH) {
#pragma unroll
        for (int i = 0; i < BATCH; ++i) {
          const int z = sub + (i0 + i) * sharers;
          if (z < runs) {
            const float fz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f), z));
            x.x += p[i].x * fz; x.y += p[i].y * fz; x.z += p[i].z * fz; x.w += p[i].w * fz;
          }
        }
        if (sub + (i0 + BATCH) * sharers < runs) load_runs(r, i0 + BATCH);
        else if (more) load_runs(r + apart, 0);
      }
      if (sharers > 1) {                                   // one row a group: all pass these once
        if (sub > 0) others[(sub - 1) * apart + r][col] = x;
        __syncthreads();
        if (sub > 0) break;
        for (int q = 1; q < sharers; ++q) {
          const float4 y = others[(q - 1) * apart + r][col];
          x.x += y.x; x.y += y.y; x.z += y.z; x.w += y.w;
        }
      }
      *reinterpret_cast<uint2*>(&rows[r][4 * col]) = make_uint2(pack_bf16x2(x.x * inv, x.y * inv), pack_bf16x2(x.z * inv, x.w * inv));
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) b[s] = *reinterpret_cast<const u32x4*>(&rows[min(lr, rb - 1)][k + 32 * s]);
  } else {
#pragma unroll
    for (int s = 0; s < NS; ++s) b[s] = *reinterpret_cast<const u32x4*>(o_lat + ((size_t)head * T + t0 + min(lr, nr - 1)) * KR + k + 32 * s);
    load_uv();
    load_gate();
  }
  f32x4 acc[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a[s]), as_bf16x8(b[s]), acc[s & 3], 0, 0, 0);
  f32x4 v = (acc[0] + acc[1]) + (acc[2] + acc[3]);
  if constexpr (KP > 1) {
    sums[w][lane] = v;
    __syncthreads();
    if (kp == 0)
#pragma unroll
      for (int q = 1; q < KP; ++q) v += sums[q * np + j][lane];
  }
  if (!multiplies || kp > 0 || lr >= nr) return;
  if (gate)
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= 1.f / (1.f + expf(-bf16_to_f32(gates[i])));
  *reinterpret_cast<uint2*>(out + (size_t)(t0 + lr) * H * vdim + c) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}

}  // namespace

// q [T, >= H * qk] (the first dim entries of a head are used), uk [H, dim, kr], q_lat [H, T, kr]; 16-byte rows throughout
extern "C" int dgi_latent_fold(void* q_lat, const void* q, int q_stride, const void* uk, int T, int H, int dim, int qk, int kr,
                               hipStream_t s) {
  if (T == 0) return 0;
  if (H <= 0 || dim % 32 || dim < 32 || dim > 128 || kr % 64 || qk % 8 || q_stride % 8 || (((uintptr_t)q | (uintptr_t)uk) & 15) ||
      ((uintptr_t)q_lat & 7))
    return -2;
  if ((T + FOLD - 1) / FOLD > 65535) return -4;
  const dim3 grid(H, kr / 64, (T + FOLD - 1) / FOLD);
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
  if (H <= 0 || vdim % 16 || vdim < 16 || vdim > 128 || runs < 1 || runs > RUNS || (runs > 1 ? !part || !ml : !o_lat)) return -2;
  if ((((uintptr_t)uv | (uintptr_t)o_lat | (uintptr_t)part) & 15) || ((uintptr_t)out & 7) || ((uintptr_t)ml & 7)) return -3;
  // Rows and value dims of a workgroup: the fewest bytes of one (KB: 2 a row and run, 1 a row without runs, 16 for sixteen value dims), times the
  // rounds of 256 workgroups.  A layer of 32 rows, 32 heads, 8 runs: 8 rows and half of the value dims 40.2 us, 4 rows and all 41.3 (and their
  // partial sums come once); 24 rows of 32 heads without runs: 16 rows, 32 value dims 4.1 us, 2 rows and all 10.4
  const int nv = vdim >> 4;
  int rb = 16, np = nv;
  long long best = -1;
  for (int r = 16; r >= 1; r >>= 1) {
    if (r > 1 && r / 2 >= T) continue;
    for (int z = 1; z <= 8; z <<= 1) {
      if (nv % z) break;
      const long long groups = (long long)H * ((T + r - 1) / r) * z;
      const long long cost = (groups + 255) / 256 * ((long long)std::min(r, T) * (runs > 1 ? 2 * runs : 1) + 16 * nv / z);
      if (best < 0 || cost < best) { best = cost; rb = r; np = nv / z; }
    }
  }
  if ((T + rb - 1) / rb > 65535) return -4;
  const dim3 grid(H, (T + rb - 1) / rb, nv / np);
#define DGI_LV(N_)                                                                                                                      \
  latent_values_kernel<N_><<<grid, 512, 0, s>>>((uint16_t*)out, (const uint16_t*)o_lat, part, ml, runs, sinks, (const uint16_t*)uv,     \
                                                (const uint16_t*)gate, gate_stride, per_head, T, H, vdim, rb, np)
  if (np == 1) DGI_LV(8);
  else if (np == 2) DGI_LV(4);
  else if (np <= 4) DGI_LV(2);
  else DGI_LV(1);
#undef DGI_LV
  DGI_CHECK_LAUNCH();
  return 0;
}
