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
// product's A operand: latent dims by query dims).  DS = dim / 32 steps; `fold` rows, sixteen at a time: 32 (128 rows of
// 16 heads one behind the other 5.7 us, so 4.5), 64 where heads alone fill the chip (256 rows of 32 heads: all 7.7, by 64 8.0, by 32 8.2).
template <int DS>
__global__ __launch_bounds__(256) void latent_fold_kernel(uint16_t* __restrict__ q_lat, const uint16_t* __restrict__ q, int q_stride,
                                                          const uint16_t* __restrict__ uk, int T, int qk, int kr, int fold) {
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
  const int from = blockIdx.z * fold, to = min(T, from + fold);
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
// through LDS to the product, whose waves take sixteen value dims each over 512 / KP latent dims (so do rows without runs where most waves read the same dims).
// Two to four runs: a group asks for four or two rows at once, so that eight loads are under way.  The weights, the gate and the first runs are
// under way while the factors are formed.  Before, a wave had 64 latent dims of all value dims, lanes without a row of their own read another's again, and
// few rows a workgroup meant all of uv for each: us then and now, rows x heads x runs: 32 x 32 x 8 11.3, 8.5; 3 x 16 x 6 8.6, 4.7; 8 x 16 x 16 10.3, 5.9;
// 24 x 32 x 16 20.3, 9.5; 48 x 16 x 4 14.1, 7.0; 64 x 32 x 2 9.2, 7.0; 4 9.7, 9.4; 128 x 32 x 2 10.7, 8.7; without runs 24 x 32 10.9, 4.8; 2 x 32 5.6, 3.7; 128 x 32 7.1, 6.6 (each wave reading all rows
// from memory 9.8); 256 x 32 12.0, 10.5.
constexpr int KR = 512, RUNS = 64, BATCH = 8;

// RP: rows of a group of threads at once, where a row's runs are BATCH / RP at most
template <int KP, int RP>
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
    const int apart = RP > 1 ? 4 : min(rb, 4), sharers = 4 / apart;        // rows at a time, groups of threads of a row
    const int group = w >> 1, sub = group / apart, col = threadIdx.x & 127;
    const size_t next = (size_t)H * T;
    constexpr int S = BATCH / RP;
    float4 p[RP][S];
    float2 e[RP];
    auto load_runs = [&](int r, int i0) {                // the batch of this group's runs, sub + sharers i
#pragma unroll
      for (int u = 0; u < RP; ++u) {
        const float* src = part + ((size_t)head * T + t0 + min(r + u * apart, nr - 1)) * KR + 4 * col;
#pragma unroll
        for (int i = 0; i < S; ++i) p[u][i] = *reinterpret_cast<const float4*>(src + (size_t)min(sub + (i0 + i) * sharers, runs - 1) * next * KR);
      }
    };
    auto load_ml = [&](int r) {
#pragma unroll
      for (int u = 0; u < RP; ++u)
        e[u] = *reinterpret_cast<const float2*>(ml + 2 * ((size_t)min(lane, runs - 1) * next + (size_t)head * T + t0 + min(r + u * apart, nr - 1)));
    };
    int r = group % apart;
    load_ml(r);
    load_runs(r, 0);
    load_uv();
    load_gate();
    for (; RP == 4 || r < rb; r += RP * apart) {           // RP 4: rb is 16
      float f[RP], inv[RP];
      // few runs: the lanes that have them; a loop of more turns costs what it saves
      auto turns = [&](auto g) {
        if (runs > 8) {
#pragma unroll
          for (int o = 1; o < 64; o <<= 1) g(o);
        } else {
          for (int o = 1; o < runs; o <<= 1) g(o);
        }
      };
#pragma unroll
      for (int u = 0; u < RP; ++u) {
        const float m = lane < runs ? e[u].x : -__builtin_inff();
        float M = fmaxf(m, -FLT_MAX);                    // finite also where no run has keys
        turns([&](int o) { M = fmaxf(M, __shfl_xor(M, o, 64)); });
        f[u] = expf(m - M);
        float L = lane < runs ? e[u].y * f[u] : 0.f;
        turns([&](int o) { L += __shfl_xor(L, o, 64); });
        float v = L == 0.f ? 0.f : 1.f / L;
        if (sinks) {                                     // one more logit in the denominator, relative to the larger of the two
          const float sink = sinks[head], top = fmaxf(M, sink), g = expf(M - top);
          v = g / (L * g + expf(sink - top));
        }
        inv[u] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), 0));
      }
      const bool more = RP < 4 && r + RP * apart < rb;
      if (more) load_ml(r + RP * apart);
      float4 x[RP];
#pragma unroll
      for (int u = 0; u < RP; ++u) x[u] = make_float4(0.f, 0.f, 0.f, 0.f);
      for (int i0 = 0; sub + i0 * sharers < runs; i0 += S) {
#pragma unroll
        for (int u = 0; u < RP; ++u)
#pragma unroll
          for (int i = 0; i < S; ++i) {
            const int z = sub + (i0 + i) * sharers;
            if (z < runs) {
              const float fz = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(f[u]), z));
              x[u].x += p[u][i].x * fz; x[u].y += p[u][i].y * fz; x[u].z += p[u][i].z * fz; x[u].w += p[u][i].w * fz;
            }
          }
        if (sub + (i0 + S) * sharers < runs) load_runs(r, i0 + S);
        else if (more) load_runs(r + RP * apart, 0);
      }
      if (RP == 1 && sharers > 1) {                      // one row a group: all pass these once
        if (sub > 0) others[(sub - 1) * apart + r][col] = x[0];
        __syncthreads();
        if (sub > 0) break;
        for (int q = 1; q < sharers; ++q) {
          const float4 y = others[(q - 1) * apart + r][col];
          x[0].x += y.x; x[0].y += y.y; x[0].z += y.z; x[0].w += y.w;
        }
      }
#pragma unroll
      for (int u = 0; u < RP; ++u)
        *reinterpret_cast<uint2*>(&rows[r + u * apart][4 * col]) =
            make_uint2(pack_bf16x2(x[u].x * inv[u], x[u].y * inv[u]), pack_bf16x2(x[u].z * inv[u], x[u].w * inv[u]));
      if (RP == 4) break;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) b[s] = *reinterpret_cast<const u32x4*>(&rows[min(lr, rb - 1)][k + 32 * s]);
  } else if constexpr (KP <= 2) {                            // most waves read the same dims: through LDS, a row a wave
    u32x4 v[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) v[i] = *reinterpret_cast<const u32x4*>(o_lat + ((size_t)head * T + t0 + min(w + 8 * i, nr - 1)) * KR + 8 * lane);
    load_uv();
    load_gate();
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(&rows[w + 8 * i][8 * lane]) = v[i];
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) b[s] = *reinterpret_cast<const u32x4*>(&rows[lr][k + 32 * s]);
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
  const int fold = H * (kr / 64) >= 256 ? 64 : 32;
  if ((T + fold - 1) / fold > 65535) return -4;
  const dim3 grid(H, kr / 64, (T + fold - 1) / fold);
#define DGI_LF(N_)                                                                                                             \
  latent_fold_kernel<N_><<<grid, 256, 0, s>>>((uint16_t*)q_lat, (const uint16_t*)q, q_stride, (const uint16_t*)uk, T, qk, kr, fold)
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
#define DGI_LV(N_, R_)                                                                                                                  \
  latent_values_kernel<N_, R_><<<grid, 512, 0, s>>>((uint16_t*)out, (const uint16_t*)o_lat, part, ml, runs, sinks, (const uint16_t*)uv, \
                                                    (const uint16_t*)gate, gate_stride, per_head, T, H, vdim, rb, np)
#define DGI_LV_ROWS(N_)                                                              \
  if (runs == 2 && rb == 16) DGI_LV(N_, 4);                                          \
  else if (runs > 1 && runs <= 4 && rb >= 8) DGI_LV(N_, 2);                          \
  else DGI_LV(N_, 1)
  if (np == 1) { DGI_LV_ROWS(8); }
  else if (np == 2) { DGI_LV_ROWS(4); }
  else if (np <= 4) { DGI_LV_ROWS(2); }
  else { DGI_LV_ROWS(1); }
#undef DGI_LV_ROWS
#undef DGI_LV
  DGI_CHECK_LAUNCH();
  return 0;
}
