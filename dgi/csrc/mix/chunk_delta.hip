// dgi/csrc/mix/chunk_delta.hip — long prompt portions of the gated delta rule (linear_scan.hip has its definition), 32 tokens at a time on the
// bf16 matrix cores.
//
// For tokens t, s of a chunk that starts from the state S, with D[t, s] the product of the decays of the tokens after s up to t, A_t that of all up to
// t, F_s = D[31, s], and k, q of unit length (q times dk^-1/2):
//
//     x = beta (v - A k S)      u = M x,  M = (I + T)^-1,  T[t, s] = beta_t D[t, s] (k_t . k_s) below the diagonal
//     o = A q S + P u,  P[t, s] = D[t, s] (q_t . k_s)      S <- A_31 S + k^T F u
//
// M does not depend on S, so what u would be is folded into what multiplies it: with G = k^T F M and P M, made for all chunks side by side beforehand, a
// chunk's chain is k S, x, A_31 S + G x, and no substitution.  delta_prepare_kernel: a wave has a chunk of (two) heads; scores on the matrix cores, M forward
// in 64 bits in blocks of sixteen, G and P M as the parts and in the lanes in which the chain takes them.  delta_chain_kernel: a workgroup owns (sequence,
// head, two blocks of 16 value columns), one barrier a chunk: state waves with the state's rows of 16 columns in registers (k S of the next chunk before
// the barrier), output waves a chunk behind them, waves that fetch what was prepared and waves that bring k and q in parts.  fp32 operands are three bf16
// parts each (chunk_parts.hip).
//
// What bounds it: a chunk of the chain takes 1.3 us (chunk_scan.hip: 1.2 for sixteen tokens), 48 products of 16 cycles and 230 vector instructions, which
// one wave does not overlap (alone on its unit the state waves would take 1.03); preparing 4096 rows of 64 heads 50 us, 150 MB of G and P M to memory, which
// nothing reads soon, and then once: stores and loads say so (without, they take the place of q, k and v in the caches, 170 us for 149).  Two
// prompts of 4096 rows in all, 64 heads of 64 x 64: 178 us -> 144; one of 2048 rows 154 -> 103; bf16 rows of
// 128 channels, 4 of 1024 rows, 32 heads, 255 -> 157.  Only long portions are taken, see
// dgi_linear_scan_parts.  Tried: M and P themselves prepared, u by a product more in the chain: 122 us a chain for 105; two state waves a block of columns, half
// the channels each: 138 for 142 without the rest (x is both's, and the unit has no instructions to spare).
//
// Precision (2-norm against 64 bits over that of chunk_scan.hip's substitution, outputs and states, 800 rows, 16 heads): random rows 0.89, 0.90 (fp32, 64
// channels), 0.97, 0.86 (bf16), 0.94, 0.87 (128); after SiLU 0.95 - 1.01, 0.87; rows that share a direction twice their spread 0.87 - 0.99, 0.87 (the loop's states
// are up to 14 % closer there: terms of the folded inverse are large beside their sum); with decays near 1 a fifth, 0.15.
#include <type_traits>
#include "chunk_split.h"

using namespace dgi;

namespace {

typedef double f64x4 __attribute__((ext_vector_type(4)));
// What a chunk of a head has in the workspace (bytes), operands as their lanes hold them: G, three parts of every tile of 16 channels; P M, three parts
// of the rows 0 .. 15 by tokens 0 .. 15 (8 bytes a lane) and of the rows 16 .. 31 by all (16 bytes); factors of its tokens: beta, or NaN where something
// of the chunk is not finite; beta A / |k|; A dk^-1/2 / |q|; the decay; beta; then A of the last token
constexpr int PART = 512 + 1024, MAT = 3 * PART, FACTORS = MAT, ALL = FACTORS + 5 * 128, REST = 6 * 1024;
static_assert(ALL + 16 <= REST, "whole loads of a wave");
__host__ __device__ constexpr int g_bytes(int NT) { return NT * 3 * 1024; }
__host__ __device__ constexpr int each(int NT) { return g_bytes(NT) + REST; }

// 8 channels of a row; channels past dk and rows past the end read zeros
template <typename TI>
__device__ __forceinline__ void row_load8(Rows rows, unsigned off, int ch, int dk, Raw4<TI> (&x)[2]) {
  constexpr unsigned E = sizeof(TI);
  x[0] = row_load<Raw4<TI>>(rows, ch < dk ? off + E * ch : 0x7fffffffu, 0);
  x[1] = row_load<Raw4<TI>>(rows, ch + 4 < dk ? off + E * (ch + 4) : 0x7fffffffu, 0);
}

// ------------------------------------------------------------------------------------------------ what the columns of a head share
// A wave has a chunk of HP heads that share q and k: lane 32 h + t is token t (or column t of M) of the h-th.
template <typename TI, int NK>
struct Prepare {
  static constexpr int PQ = sizeof(TI) == 2 ? 1 : 3, ROWB = 64 * NK, PARTB = C * ROWB;
  static constexpr int TR = 36, TM = 32 * TR + 16;     // padded rows of T; a head's
  static constexpr int MB = 16 * 16 + 16;              // a block of M, in 64 bits; four of them
  static constexpr int DIAG = 4 * MB * 8;              // and the blocks between them, in 32: [2][16][16]
  static constexpr int KB = PARTB > DIAG + 2048 ? PARTB : DIAG + 2048;     // a part of k, then T, then M
  static_assert(2 * TM * 4 <= KB, "T before M");
  static constexpr int EACH_WAVE = KB + 8 * 64 * 4;    // and [8][64] factors of the tokens
};
template <typename TI, int NK, int HP>
__global__ __launch_bounds__(256, 3) void delta_prepare_kernel(const ChunkArgs a) {
  using L = Prepare<TI, NK>;
  constexpr int PQ = L::PQ, NT = 2 * NK, TR = L::TR, TM = L::TM, MB = L::MB;
  constexpr unsigned E = sizeof(TI);
  __shared__ __attribute__((aligned(16))) char all[4][L::EACH_WAVE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
  const int t32 = lane & 31, hl = HP == 2 ? lane >> 5 : 0;
  const int head0 = (blockIdx.x * 4 + wave) * HP;
  int seq = 0, hi = a.n_seq - 1;
  while (seq < hi) {
    const int mid = (seq + hi + 1) >> 1;
    if (first_chunk(a.seq_row0[mid], mid) <= (int)blockIdx.y) seq = mid;
    else hi = mid - 1;
  }
  const int row0 = a.seq_row0[seq], n = a.seq_row0[seq + 1] - row0, first = ((int)blockIdx.y - first_chunk(row0, seq)) * C;
  if (n <= a.skip_rows || first >= n || head0 >= a.H) return;
  const int left = n - first, kvh = head0 / (a.H / a.G), head = head0 + hl;
  char* const K = all[wave];
  float* const T = reinterpret_cast<float*>(K);
  float* const F = reinterpret_cast<float*>(K + L::KB);
  enum { EI, EF, BI, BF, F2, QROW, ROW, COL };
  char* const ws = (char*)a.parts + ((size_t)blockIdx.y * a.H + head0) * each(NT);
  auto place = [&](int row, int ch16) { return row * L::ROWB + ((ch16 ^ (row & 7)) << 4); };

  const size_t tok = (size_t)row0 + first + min(t32, left - 1);
  const float ga = ((const float*)a.aux1)[tok * a.aux1_stride + head], gb = ((const float*)a.aux2)[tok * a.aux2_stride + head];
  Raw4<TI> kr[2][NK][2], qr[2][NK][2];                 // rows 16 h + n16, channels 32 b + 8 g ..
  {
    const unsigned stq = a.q_stride * E, stk = a.k_stride * E, have = min(left, C);
    const Rows pq = rows_at((const TI*)a.q + (size_t)(row0 + first) * a.q_stride + (size_t)kvh * a.dk, (have - 1) * stq + E * a.dk);
    const Rows pk = rows_at((const TI*)a.k + (size_t)(row0 + first) * a.k_stride + (size_t)kvh * a.dk, (have - 1) * stk + E * a.dk);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int b = 0; b < NK; ++b) {
        const unsigned row = 16 * h + n16;
        row_load8<TI>(pk, row < have ? row * stk : 0x70000000u, 32 * b + 8 * g, a.dk, kr[h][b]);
        row_load8<TI>(pq, row < have ? row * stq : 0x70000000u, 32 * b + 8 * g, a.dk, qr[h][b]);
      }
  }
  const double p1 = -exp((double)a.par1[head]) * LOG2E, dt = softplus_d((double)gb + a.par2[head]);
  const bool ok = t32 < left;
  double Z = ok ? p1 * dt : 0.;
  const float beta = ok ? 1.f / (1.f + expf(-ga)) : 0.f;
  bool bad = ok && !(fabs(Z) < 1e30 && beta <= 1.f);
  const float decay = ok ? exp2f((float)Z) : 1.f;
  Z = fmin(fmax(Z, -20000.), 0.);                      // 32 of them stay within the whole numbers' range
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const double y = __shfl_up(Z, o, 32);
    if (t32 >= o) Z += y;
  }
  const double end = __shfl(Z, 31, 32);
  {
    float w, f;
    whole_and_part(Z, w, f);
    F[EI * 64 + lane] = w;
    F[EF * 64 + lane] = f;
    F[BI * 64 + lane] = -w;
    F[BF * 64 + lane] = -f;
  }
  // scores: tiles of tokens s (rows 4 g + r) and t (columns n16): both early, early and late, both late
  f32x4 kk[3], qk[3];
  u32x4 kT[NT][PQ];                                    // k, channels by tokens, as the chain's tiles have them
  {
    u32x4 kp[NK][2][PQ];
    f32x4 kl[3], ql[3], kb[3], qb[3];
    float k2[2] = {0.f, 0.f}, q2[2] = {0.f, 0.f};      // squared norms
#pragma unroll
    for (int i = 0; i < 3; ++i) kk[i] = kl[i] = qk[i] = ql[i] = kb[i] = qb[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NK; ++b) {
      u32x4 kf[3][PQ], kt[3][PQ], qt[3][PQ];           // early, early, late by early, late, late
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        float x[8], y[8];
        widen(kr[h][b][0], x);
        widen(kr[h][b][1], x + 4);
        widen(qr[h][b][0], y);
        widen(qr[h][b][1], y + 4);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          k2[h] = fmaf(x[i], x[i], k2[h]);
          q2[h] = fmaf(y[i], y[i], q2[h]);
        }
        split8<PQ>(x, kp[b][h]);
        split8<PQ>(y, qt[2 * h]);
      }
#pragma unroll
      for (int p = 0; p < PQ; ++p) {
        kf[0][p] = kf[1][p] = kt[0][p] = kp[b][0][p];
        kf[2][p] = kt[1][p] = kt[2][p] = kp[b][1][p];
        qt[1][p] = qt[2][p];
      }
      // the last block's first parts start from the small ones' sum: one rounding less at the sum's size
      small<PQ, PQ, 3, 3>(kf, kt, kl);
      small<PQ, PQ, 3, 3>(kf, qt, ql);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const bool second = NK == 4 && b == 2;
        f32x4 &k = second ? kb[i] : b + 1 < NK ? kk[i] : kl[i], &q = second ? qb[i] : b + 1 < NK ? qk[i] : ql[i];
        k = mfma(kf[i][0], kt[i][0], k);
        q = mfma(kf[i][0], qt[i][0], q);
      }
    }
#pragma unroll
    for (int p = 0; p < PQ; ++p) {
#pragma unroll
      for (int b = 0; b < NK; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) *reinterpret_cast<u32x4*>(K + place(16 * h + n16, 4 * b + g)) = kp[b][h][p];
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const short4v w = read_tr(K + place(16 * h + 4 * g + (n16 >> 2), 4 * (i >> 1) + (n16 & 3)) + 8 * (i & 1));
          kT[i][p][2 * h] = (uint32_t)(uint16_t)w[0] | ((uint32_t)(uint16_t)w[1] << 16);
          kT[i][p][2 * h + 1] = (uint32_t)(uint16_t)w[2] | ((uint32_t)(uint16_t)w[3] << 16);
        }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) { kk[i] += kb[i] + kl[i]; qk[i] += qb[i] + ql[i]; }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      k2[h] += __shfl_xor(k2[h], 16, 64);
      q2[h] += __shfl_xor(q2[h], 16, 64);
      k2[h] += __shfl_xor(k2[h], 32, 64);
      q2[h] += __shfl_xor(q2[h], 32, 64);
      if (g < 2) {
        F[ROW * 64 + 32 * g + 16 * h + n16] = k2[h];
        F[COL * 64 + 32 * g + 16 * h + n16] = q2[h];
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  {
    const float sk = F[ROW * 64 + lane], sq = F[COL * 64 + lane];
    bad |= ok && !(sk < 1e30f && sq < 1e30f);
    const float ik = 1.f / sqrtf(sk + 1e-6f), iq = (1.f / sqrtf((float)a.dk)) / sqrtf(sq + 1e-6f);
    __builtin_amdgcn_wave_barrier();
    F[ROW * 64 + lane] = beta * ik;
    F[COL * 64 + lane] = ik;
    F[QROW * 64 + lane] = iq;
    F[F2 * 64 + lane] = ok ? ik * power_once(end - Z) : 0.f;
    const unsigned long long any = __ballot(bad);
    if (HP == 2 || lane < 32) {
      char* to = ws + hl * each(NT) + g_bytes(NT);
      float* f = (float*)(to + FACTORS) + t32;
      const float A = power_once(Z);
      f[0] = (hl == 0 ? any & 0xffffffffull : any >> 32) != 0 ? __builtin_nanf("") : beta;
      f[32] = beta * ik * A;
      f[64] = iq * A;
      f[96] = decay;
      f[128] = beta;
      if (t32 == 31) *(float*)(to + ALL) = A;
    }
  }
  __builtin_amdgcn_wave_barrier();
  // D[t, s] / |k_s| of tile i, four tokens s
  auto decays = [&](int h, int i, float (&w)[4]) __attribute__((always_inline)) {
    const int s = 32 * h + (i == 2 ? 16 : 0), t = 32 * h + (i > 0 ? 16 : 0);
    const float ei = F[EI * 64 + t + n16], ef = F[EF * 64 + t + n16];
    const float4 bi = ld4(F + BI * 64 + s + 4 * g), bf = ld4(F + BF * 64 + s + 4 * g), co = ld4(F + COL * 64 + s + 4 * g);
    const float bis[4] = {bi.x, bi.y, bi.z, bi.w}, bfs[4] = {bf.x, bf.y, bf.z, bf.w}, cos[4] = {co.x, co.y, co.z, co.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) w[r] = i == 1 || 4 * g + r <= n16 ? power(ei + bis[r], ef + bfs[r]) * cos[r] : 0.f;
  };
  // T[t, s] below the diagonal
#pragma unroll
  for (int h = 0; h < HP; ++h)
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int s = i == 2 ? 16 : 0, t = i > 0 ? 16 : 0;
      const float row = F[ROW * 64 + 32 * h + t + n16];
      float w[4], y[4];
      decays(h, i, w);
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = i == 1 || 4 * g + r < n16 ? kk[i][r] * (w[r] * row) : 0.f;
      *reinterpret_cast<float4*>(T + h * TM + (t + n16) * TR + s + 4 * g) = make_float4(y[0], y[1], y[2], y[3]);
    }
  __builtin_amdgcn_wave_barrier();
  // (I + T) M = I in 64 bits: blocks of sixteen tokens forward, a lane has a column of a head's early or late one, and
  // - M2 T21 M1 between the two (a 64-bit product's register r is row 4 r + g: as the next one's operand has it)
  double* const MD = reinterpret_cast<double*>(K);
  {
    const float* Tc = T + (HP == 2 ? g >> 1 : 0) * TM + (g & 1) * (16 * TR + 16);
    double M[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      double s[2] = {t == n16 ? 1. : 0., 0.};
#pragma unroll
      for (int j = 0; j < t; j += 4) {
        const float4 x = ld4(Tc + t * TR + j);
        const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (j + r < t) s[r & 1] -= (double)xs[r] * M[j + r];
      }
      M[t] = s[0] + s[1];
    }
    float t21[HP][4];
#pragma unroll
    for (int h = 0; h < HP; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) t21[h][j] = T[h * TM + (16 + n16) * TR + 4 * j + g];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < 16; ++t) MD[g * MB + 16 * t + n16] = M[t];
    __builtin_amdgcn_wave_barrier();
    f64x4 w[HP], m21[HP];
#pragma unroll
    for (int h = 0; h < HP; ++h) {
      w[h] = m21[h] = f64x4{0., 0., 0., 0.};
#pragma unroll
      for (int j = 0; j < 4; ++j) w[h] = __builtin_amdgcn_mfma_f64_16x16x4f64((double)t21[h][j], MD[2 * h * MB + 16 * (4 * j + g) + n16], w[h], 0, 0, 0);
    }
#pragma unroll
    for (int h = 0; h < HP; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) m21[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(-MD[(2 * h + 1) * MB + 16 * n16 + 4 * j + g], w[h][j], m21[h], 0, 0, 0);
    // behind the blocks: rows of M21 as floats
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < HP; ++h)
#pragma unroll
      for (int r = 0; r < 4; ++r) reinterpret_cast<float*>(K + L::DIAG)[256 * h + 16 * (4 * r + g) + n16] = (float)m21[h][r];
  }
  __builtin_amdgcn_wave_barrier();
  // G = k^T F M / |k| and P M, transposed as they come: lane = channel (or row of P), four tokens s
#pragma unroll 1
  for (int h = 0; h < HP; ++h) {
    char* const to = ws + h * each(NT);
    const float* M21 = reinterpret_cast<const float*>(K + L::DIAG) + 256 * h;
    u32x4 m[2][3], f[2][3];                            // columns s = 16 hs + n16 of M and F M / |k|
#pragma unroll
    for (int hs = 0; hs < 2; ++hs) {
      float x[8], y[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int t = 16 * (i >> 2) + 4 * g + (i & 3);
        x[i] = hs == 1 && i < 4 ? 0.f : hs == 0 && i >= 4 ? M21[16 * (t - 16) + n16] : (float)MD[(2 * h + hs) * MB + 16 * (t & 15) + n16];
        y[i] = x[i] * F[F2 * 64 + 32 * h + t];
      }
      split8<3>(x, m[hs]);
      split8<3>(y, f[hs]);
    }
    auto four = [&](const f32x4& v, u32x2 (&p)[3]) __attribute__((always_inline)) {
      float x[4] = {v[0], v[1], v[2], v[3]};
#pragma unroll
      for (int j = 0; j < 2; ++j) { p[j][0] = part_of(x[0], x[1]); p[j][1] = part_of(x[2], x[3]); }
      p[2][0] = pack_bf16x2(x[0], x[1]);
      p[2][1] = pack_bf16x2(x[2], x[3]);
    };
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      f32x4 l[2], v[2];
      u32x4 k1[1][PQ];
#pragma unroll
      for (int p = 0; p < PQ; ++p) k1[0][p] = kT[i][p];
#pragma unroll
      for (int hs = 0; hs < 2; ++hs) l[hs] = v[hs] = f32x4{0.f, 0.f, 0.f, 0.f};
      multiply<3, PQ, 2, 1>(f, k1, l, v);
      u32x2 p0[3], p1[3];
      four(v[0] + l[0], p0);
      four(v[1] + l[1], p1);
#pragma unroll
      for (int j = 0; j < 3; ++j) __builtin_nontemporal_store(u32x4{p0[j][0], p0[j][1], p1[j][0], p1[j][1]}, reinterpret_cast<u32x4*>(to + (3 * i + j) * 1024 + 16 * lane));
    }
    u32x4 P[2][3];                                     // rows t = 16 ht + n16
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const float row = F[QROW * 64 + 32 * h + (i > 0 ? 16 : 0) + n16];
      float w[4];
      decays(h, i, w);
      f32x4 x;
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = qk[i][r] * (w[r] * row);
      u32x2 p[3];
      four(x, p);
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        if (i == 0) P[0][j] = u32x4{p[j][0], p[j][1], 0, 0};
        if (i == 1) { P[1][j][0] = p[j][0]; P[1][j][1] = p[j][1]; }
        if (i == 2) { P[1][j][2] = p[j][0]; P[1][j][3] = p[j][1]; }
      }
    }
    f32x4 l[3], v[3];
    u32x4 ma[3][3], pa[3][3];                          // s early and late by t early, early, late
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      ma[0][j] = ma[1][j] = m[0][j];
      ma[2][j] = m[1][j];
      pa[0][j] = P[0][j];
      pa[1][j] = pa[2][j] = P[1][j];
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) l[i] = v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    multiply<3, 3, 3, 3>(ma, pa, l, v);
    u32x2 p[3][3];
#pragma unroll
    for (int i = 0; i < 3; ++i) four(v[i] + l[i], p[i]);
    char* const pm = to + g_bytes(NT);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      __builtin_nontemporal_store(p[0][j], reinterpret_cast<u32x2*>(pm + j * PART + 8 * lane));
      __builtin_nontemporal_store(u32x4{p[1][j][0], p[1][j][1], p[2][j][0], p[2][j][1]}, reinterpret_cast<u32x4*>(pm + j * PART + 512 + 16 * lane));
    }
  }
}

// ------------------------------------------------------------------------------------------------ the chain
template <typename TI, int NK_>
struct Lay {
  static constexpr int NK = NK_, DP = 32 * NK, NB = 2, PQ = sizeof(TI) == 2 ? 1 : 3;
  // k S of the next chunk before the barrier between the two, where LDS has room for a chunk more
  static constexpr bool AHEAD = NK == 2;
  static constexpr int KN = AHEAD ? 3 : 2, RN = AHEAD ? 4 : 3;
  // Waves: state, output, two that fetch what was prepared, k's and q's: waves four apart share a SIMD, and the state's have one almost to themselves
  static constexpr int OUT = NB, FETCH = 2 * NB, PREP = FETCH + 2, WAVES = PREP + 2;
  static constexpr int ROWB = 2 * DP, PARTB = C * ROWB, ARRB = PQ * PARTB, SB = 3 * NK * 1024;       // bytes of a row, a part, q or k, a block's state in parts
  static constexpr int K = 0, Q = K + KN * ARRB;       // [KN], [2][PQ][32][ROWB]
  static constexpr int SP = Q + 2 * ARRB;              // [2][NB] state before the chunk
  static constexpr int X = SP + 2 * NB * SB;           // [2][NB][3][64] parts of x
  static constexpr int G = X + 2 * NB * 3072;          // [2] G
  static constexpr int RING = G + 2 * g_bytes(2 * NK); // [RN] the rest of what was prepared
  static constexpr int END = RING + RN * REST;
};

template <typename TI, int NK>
__global__ __launch_bounds__((64 * Lay<TI, NK>::WAVES), 2) void delta_chain_kernel(const ChunkArgs a) {
  using L = Lay<TI, NK>;
  constexpr int PQ = L::PQ, NT = 2 * NK;
  constexpr unsigned E = sizeof(TI);
  extern __shared__ __attribute__((aligned(16))) char sm[];
  const int head = blockIdx.x % a.H, zb = blockIdx.x / a.H / a.n_seq;
  const int seq = __builtin_amdgcn_readfirstlane(ranked(a, blockIdx.x / a.H % a.n_seq));
  const int row0 = a.seq_row0[seq], n = a.seq_row0[seq + 1] - row0;
  if (n <= a.skip_rows) return;
  const int H = a.H, dk = a.dk, dv = a.dv, kvh = head / (H / a.G);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n16 = lane & 15, g = lane >> 4;
  const int chunks = (n + C - 1) / C;
  constexpr int EACH = each(NT);
  const char* const ws = (const char*)a.parts + ((size_t)first_chunk(row0, seq) * H + head) * EACH;
  // Every wave passes 1 + chunks barriers.
  auto place = [&](int row, int ch16) { return row * L::ROWB + ((ch16 ^ (row & 7)) << 4); };      // eight rows' 16 bytes are eight places
  auto keys_at = [&](int c) { return sm + L::K + (L::KN == 3 ? c % 3 : c & 1) * L::ARRB; };
  auto rest = [&](int c) { return sm + L::RING + (L::RN == 4 ? c & 3 : c % 3) * REST; };
  if (wave >= L::FETCH && wave < L::PREP) {
    // ============================================================================================== what was prepared, to LDS: each every other KB
    const int odd = wave - L::FETCH;
    // G of chunk c and the rest of chunk cr
    auto fetch = [&](int c, bool g, int cr) __attribute__((always_inline)) {
      const char* p = ws + (size_t)min(c, chunks - 1) * H * EACH + 1024 * odd + 16 * lane;
      char* const to = sm + L::G + (c & 1) * g_bytes(NT) + 1024 * odd;
      if (g) {
#pragma unroll
        for (int i = 0; i < g_bytes(NT); i += 2048)
          __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(p + i), (__attribute__((address_space(3))) void*)(to + i), 16, 0, 2);
      }
      const char* r = ws + (size_t)min(cr, chunks - 1) * H * EACH + g_bytes(NT) + 1024 * odd + 16 * lane;
#pragma unroll
      for (int i = 0; i < REST; i += 2048)
        __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(r + i), (__attribute__((address_space(3))) void*)(rest(cr) + 1024 * odd + i), 16, 0, 2);
    };
    fetch(0, true, 0);
    if (L::RN == 4) fetch(0, false, 1);
    __builtin_amdgcn_s_waitcnt(0x0F70);                // vmcnt(0)
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {
      fetch(c + 1, true, c + L::RN - 2);
      __builtin_amdgcn_s_waitcnt(0x0F70);
      __syncthreads();
    }
    return;
  }
  if (wave >= L::PREP) {
    // ============================================================================================== parts of k or q to LDS
    constexpr int PER = L::DP / 8, RPT = 64 / PER, TASKS = C / RPT;      // pieces of eight channels of a row; rows of a task; a lane's tasks
    const bool is_k = wave == L::PREP;
    const int stride = is_k ? a.k_stride : a.q_stride, piece = lane % PER, r0 = lane / PER;
    const TI* const from = (const TI*)(is_k ? a.k : a.q) + (size_t)row0 * stride + (size_t)kvh * dk;
    const unsigned st = stride * E;
    Raw4<TI> raw[2][TASKS][2];
    auto load = [&](int c, auto set) __attribute__((always_inline)) {
      const int first = min(c * C, n - 1), have = min(n - first, C);
      const Rows p = rows_at(from + (size_t)first * stride, (have - 1) * st + dk * E);
#pragma unroll
      for (int j = 0; j < TASKS; ++j) row_load8<TI>(p, (RPT * j + r0) * st, 8 * piece, dk, raw[set.value][j]);      // rows past the end: zeros (or anything: nothing takes them)
    };
    auto put = [&](int c, auto set) __attribute__((always_inline)) {
      char* const to = is_k ? keys_at(c) : sm + L::Q + (c & 1) * L::ARRB;
#pragma unroll
      for (int j = 0; j < TASKS; ++j) {
        float x[8];
        widen(raw[set.value][j][0], x);
        widen(raw[set.value][j][1], x + 4);
        u32x4 p[3];
        split8<PQ>(x, p);
#pragma unroll
        for (int i = 0; i < PQ; ++i) *reinterpret_cast<u32x4*>(to + i * L::PARTB + place(RPT * j + r0, piece)) = p[i];
      }
    };
    constexpr std::integral_constant<int, 0> even;
    constexpr std::integral_constant<int, 1> odd;
    const int lead = is_k ? L::KN - 2 : 0;             // chunks k is ahead of q
    // In step c the rows of chunk c + 1 (+ lead), which have had a step to come, are written, those of the next asked for.
    auto step = [&](int c, auto now, auto next) __attribute__((always_inline)) {
      load(c + 2 + lead, next);
      put(c + 1 + lead, now);
      __syncthreads();
    };
    load(0, even);
    load(lead, odd);
    put(0, even);
    if (lead) put(1, odd);
    load(1 + lead, odd);
    __syncthreads();
    for (int c = 0; c < chunks; c += 2) {
      step(c, odd, even);
      if (c + 1 < chunks) step(c + 1, even, odd);
    }
    return;
  }
  const bool outputs = wave >= L::OUT;
  const int block = wave % L::NB;
  const int col = (zb * L::NB + block) * 16 + n16, colc = min(col, dv - 1);
  const bool cok = col < dv;
  if ((zb * L::NB + block) * 16 >= dv) {
    for (int i = 0; i <= chunks; ++i) __syncthreads();
    return;
  }
  // token 16 h + 4 g + r is value 4 h + r
  auto tok = [&](int i) { return 16 * (i >> 2) + 4 * g + (i & 3); };
  auto chan = [](int g, int i, int r) { return 32 * (i >> 1) + 8 * g + 4 * (i & 1) + r; };
  auto read_factor = [&](const char* p, int i, f32x4 (&f)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) f[h] = *reinterpret_cast<const f32x4*>(p + FACTORS + 128 * i + 64 * h + 16 * g);
  };
  auto read_rows = [&](const char* from, int b, u32x4 (&x)[2][PQ]) __attribute__((always_inline)) {      // of k or q: rows 16 h + n16, channels 32 b + 8 g ..
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < PQ; ++p) x[h][p] = *reinterpret_cast<const u32x4*>(from + p * L::PARTB + place(16 * h + n16, 4 * b + g));
  };
  auto parts_at = [&](int c, int b, int j) { return reinterpret_cast<u32x4*>(sm + L::SP + ((c & 1) * L::NB + block) * L::SB + (3 * b + j) * 1024 + 16 * lane); };
  float* const yb = a.y + (size_t)row0 * H * dv + (size_t)head * dv;

  if (outputs) {
    // ============================================================================================== output waves
    const unsigned sy = H * dv * 4u;
    unsigned vy[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) vy[i] = cok ? tok(i) * sy + colc * 4u : 0x7fffffffu;       // columns past dv: nothing written
    f32x4 qS[2];
    u32x4 P[2][3], up[1][3];
    f32x4 fo[2];
    bool cold = false;
    auto before = [&](int c) __attribute__((always_inline)) {      // x of chunk c, and what it is multiplied by
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        up[0][j] = *reinterpret_cast<const u32x4*>(sm + L::X + ((c & 1) * L::NB + block) * 3072 + 1024 * j + 16 * lane);
        const u32x2 x = *reinterpret_cast<const u32x2*>(rest(c) + j * PART + 8 * lane);
        P[0][j] = u32x4{x[0], x[1], 0, 0};
        P[1][j] = *reinterpret_cast<const u32x4*>(rest(c) + j * PART + 512 + 16 * lane);
      }
      read_factor(rest(c), 2, fo);
      // x that is not a number anywhere: the state wave has written the outputs
      float none = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) none = fmaf(__uint_as_float(up[0][0][i] << 16), 0.f, fmaf(__uint_as_float(up[0][0][i] & 0xffff0000u), 0.f, none));
      cold = __any(none != 0.f);
    };
    auto finish = [&](int c) __attribute__((always_inline)) {
      f32x4 o[2], oh[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) o[h] = f32x4{0.f, 0.f, 0.f, 0.f};
      small<3, 3, 2, 1>(P, up, o);
#pragma unroll
      for (int h = 0; h < 2; ++h) oh[h] = mfma(P[h][0], up[0][0], f32x4{0.f, 0.f, 0.f, 0.f});
      const Rows p = rows_at(yb + (size_t)c * C * H * dv, cold ? 0 : min(n - c * C, C) * sy);
#pragma unroll
      for (int i = 0; i < 8; ++i) row_store(p, oh[i >> 2][i & 3] + fmaf(fo[i >> 2][i & 3], qS[i >> 2][i & 3], o[i >> 2][i & 3]), vy[i], 0);
    };
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {
      if (c > 0) {
        before(c - 1);
        finish(c - 1);
      }
      // the state's part of this one's
      f32x4 lo[2], hi[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) lo[h] = hi[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < NK; ++b) {
        u32x4 sp[1][3], x[2][PQ];
        read_rows(sm + L::Q + (c & 1) * L::ARRB, b, x);
#pragma unroll
        for (int j = 0; j < 3; ++j) sp[0][j] = *parts_at(c, b, j);
        small<PQ, 3, 2, 1>(x, sp, lo);
#pragma unroll
        for (int h = 0; h < 2; ++h) (b + 1 < NK ? hi : lo)[h] = mfma(x[h][0], sp[0][0], (b + 1 < NK ? hi : lo)[h]);
      }
#pragma unroll
      for (int h = 0; h < 2; ++h) qS[h] = hi[h] + lo[h];
      __syncthreads();
    }
    before(chunks - 1);
    finish(chunks - 1);
    return;
  }

  // ================================================================================================ state waves
  f32x4 S[NT];
  const size_t sbase = ((size_t)a.seq_slots[seq] * H + head) * dk * dv;
  auto sat = [&](int ch) { return sbase + (size_t)ch * dv + colc; };
  {
    const bool stored = a.positions[row0] > 0;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ch = chan(g, i, r);
        S[i][r] = (stored && ch < dk && cok) ? a.state[sat(ch)] : 0.f;
      }
  }
  u32x4 sp[NK][1][3];
  auto parts = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NK; ++b) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = S[2 * b + (i >> 2)][i & 3];
      split8<3>(v, sp[b][0]);
#pragma unroll
      for (int j = 0; j < 3; ++j) *parts_at(c, b, j) = sp[b][0][j];
    }
  };
  const TI* vb = (const TI*)a.v + (size_t)row0 * a.v_stride + (size_t)head * dv;
  TI rv[8];
  // the lanes' offsets are kept: rows past the end read zeros (or anything: nothing takes them)
  const unsigned sv = a.v_stride * E;
  unsigned vv[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) vv[i] = tok(i) * sv + colc * E;
  auto load_v = [&](int c) __attribute__((always_inline)) {
    const int first = min(c * C, n - 1), have = min(n - first, C);
    const Rows p = rows_at(vb + (size_t)first * a.v_stride, (have - 1) * sv + dv * E);
#pragma unroll
    for (int i = 0; i < 8; ++i) rv[i] = row_load<TI>(p, vv[i], 0);
  };
  // A chunk with something that is not finite goes token by token, as the recurrence is written: parts of an infinity are no numbers, and a matrix
  // product multiplies a token's values by the zeros of those before it.
  auto by_token = [&](int c) __attribute__((always_inline)) {
    const int have = min(n - c * C, C);
    const float* F = (const float*)(rest(c) + FACTORS);
#pragma unroll 1
    for (int t = 0; t < have; ++t) {
      const size_t row = (size_t)row0 + c * C + t;
      const Rows rk = rows_at((const TI*)a.k + row * a.k_stride + (size_t)kvh * dk, E * dk);
      const Rows rq = rows_at((const TI*)a.q + row * a.q_stride + (size_t)kvh * dk, E * dk);
      const float own = ldf<TI>(vb + (size_t)(c * C + t) * a.v_stride + colc), beta = F[128 + t], decay = F[96 + t];
      float k2 = 0.f, q2 = 0.f, kS = 0.f;
      auto add = [](float x) { x += __shfl_xor(x, 16, 64); return x + __shfl_xor(x, 32, 64); };
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        float k[4], q[4];
        widen(row_load<Raw4<TI>>(rk, chan(g, i, 0) * E, 0), k);
        widen(row_load<Raw4<TI>>(rq, chan(g, i, 0) * E, 0), q);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          S[i][x] *= decay;
          k2 = fmaf(k[x], k[x], k2);
          q2 = fmaf(q[x], q[x], q2);
          kS = fmaf(k[x], S[i][x], kS);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      const float ik = 1.f / sqrtf(add(k2) + 1e-6f), iq = (1.f / sqrtf((float)dk)) / sqrtf(add(q2) + 1e-6f);
      const float u = beta * (own - add(kS) * ik) * ik;
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        float k[4], q[4];
        widen(row_load<Raw4<TI>>(rk, chan(g, i, 0) * E, 0), k);
        widen(row_load<Raw4<TI>>(rq, chan(g, i, 0) * E, 0), q);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          S[i][x] = fmaf(k[x], u, S[i][x]);
          o = fmaf(q[x], S[i][x], o);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      o = add(o) * iq;
      if (g == 0 && cok) yb[(size_t)(c * C + t) * H * dv + colc] = o;
    }
  };
  auto read_g = [&](int c, int j, u32x4 (&x)[2][3]) __attribute__((always_inline)) {      // two tiles
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int p = 0; p < 3; ++p) x[y][p] = *reinterpret_cast<const u32x4*>(sm + L::G + (c & 1) * g_bytes(NT) + (3 * (j + y) + p) * 1024 + 16 * lane);
  };
  // k S of a chunk, and its factors
  u32x4 rows[NK][2][PQ];
  f32x4 f0[2], f1[2], kS[2];
  float tail;
  auto read_keys = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NK; ++b) read_rows(keys_at(c), b, rows[b]);
    read_factor(rest(c), 0, f0);
    read_factor(rest(c), 1, f1);
    tail = *reinterpret_cast<const float*>(rest(c) + ALL);
  };
  auto by_keys = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) kS[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NK; ++b) small<PQ, 3, 2, 1>(rows[b], sp[b], kS);
#pragma unroll
    for (int b = 0; b < NK; ++b)
#pragma unroll
      for (int h = 0; h < 2; ++h) kS[h] = mfma(rows[b][h][0], sp[b][0][0], kS[h]);
  };
  parts(0);
  load_v(0);
  __syncthreads();
  if constexpr (L::AHEAD) {
    read_keys(0);
    by_keys();
  }
  for (int c = 0; c < chunks; ++c) {
    bool warm = true;
    for (; c < chunks; ++c) {
      // the loop
      u32x4 G[2][2][3], xp[1][3];
      read_g(c, 0, G[0]);
      if constexpr (!L::AHEAD) {
        read_keys(c);
        __builtin_amdgcn_sched_barrier(0);
        by_keys();
      }
      // x = beta v - beta A k S / |k|
      float x[8];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int r = 0; r < 4; ++r) x[4 * h + r] = fmaf(-f1[h][r], kS[h][r], f0[h][r] * ldf<TI>(&rv[4 * h + r]));
      }
      // what the parts lack is a number only where x is one (and not too large for them)
      float lack = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        xp[0][0][i] = part_of(x[2 * i], x[2 * i + 1]);
        xp[0][1][i] = part_of(x[2 * i], x[2 * i + 1]);
        xp[0][2][i] = pack_bf16x2(x[2 * i], x[2 * i + 1]);
        lack += x[2 * i] + x[2 * i + 1];
      }
#pragma unroll
      for (int j = 0; j < 3; ++j) *reinterpret_cast<u32x4*>(sm + L::X + ((c & 1) * L::NB + block) * 3072 + 1024 * j + 16 * lane) = xp[0][j];
      load_v(c + 1);                                   // not where the step begins: the other waves' loads all start there
      const float at = tail;
      if constexpr (L::AHEAD) read_keys(c + 1);
      // S <- A S + G x.  Whether x is one is looked at where the products are done: a branch before them would keep them from being mixed with its parts.
      f32x4 s[NT];
#pragma unroll
      for (int j = 0; j < NT; j += 2) {
        if (j + 2 < NT) read_g(c, j + 2, G[(j / 2 + 1) & 1]);
        f32x4 two[2];
#pragma unroll
        for (int y = 0; y < 2; ++y) two[y] = f32x4{0.f, 0.f, 0.f, 0.f};
        small<3, 3, 2, 1>(G[j / 2 & 1], xp, two);
#pragma unroll
        for (int y = 0; y < 2; ++y) s[j + y] = mfma(G[j / 2 & 1][y][0], xp[0][0], two[y]);
      }
      warm = !__any(!finite(lack));
      if (__builtin_expect(!warm, 0)) break;
#pragma unroll
      for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = fmaf(at, S[i][r], s[i][r]);
      parts(c + 1);
      if constexpr (L::AHEAD) by_keys();
      __syncthreads();
    }
    if (warm) break;
    by_token(c);
    parts(c + 1);
    if constexpr (L::AHEAD) by_keys();
    __syncthreads();
  }
  // addresses are made anew: those of the loads would be kept all the way
  int ge = g;
  asm volatile("" : "+v"(ge));
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ch = chan(ge, i, r);
      if (cok && ch < dk) a.state[sat(ch)] = S[i][r];
    }
}

template <typename TI, int NK>
int launch(const ChunkArgs& a, dim3 grid, hipStream_t st) {
  constexpr int lds = Lay<TI, NK>::END;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = delta_chain_kernel<TI, NK>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
  }
  // a wave takes two heads that share q and k where there are such
  if (a.H / a.G % 2 == 0) delta_prepare_kernel<TI, NK, 2><<<dim3((a.H + 7) / 8, a.parts_chunks), 256, 0, st>>>(a);
  else delta_prepare_kernel<TI, NK, 1><<<dim3((a.H + 3) / 4, a.parts_chunks), 256, 0, st>>>(a);
  kernel<<<grid, 64 * Lay<TI, NK>::WAVES, lds, st>>>(a);
  return 0;
}

}  // namespace

// Floats of workspace for T rows of n_seq sequences (0: they are not taken)
long long dgi_chunk_delta_floats(int dk, int H, int T, int n_seq, int in_f32, int* chunks) {
  *chunks = T / C + n_seq;
  const long long floats = (long long)*chunks * H * (each(dk <= 64 ? 4 : 8) / 4);
  return dk > (in_f32 ? 64 : 128) || *chunks > 65535 || floats > 1ll << 28 ? 0 : floats;
}

// grid: n_seq * H * (blocks of 32 value columns)
int dgi_chunk_delta(const ChunkArgs& a, int in_f32, dim3 grid, hipStream_t st) {
  if (a.dk <= 64) return in_f32 ? launch<float, 2>(a, grid, st) : launch<uint16_t, 2>(a, grid, st);
  return in_f32 ? -3 : launch<uint16_t, 4>(a, grid, st);
}
