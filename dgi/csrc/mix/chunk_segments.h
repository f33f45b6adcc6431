// dgi/csrc/mix/chunk_segments.h — prompt portions of recurrences that carry a matrix S [dk, dv] per head (mlstm, light: one decay per token; gla: one per
// token and key channel; linear_scan.hip has their definitions), 32 tokens at a time on the bf16 matrix cores, long portions in segments that run side by side
// (segments.h).
//
// For tokens t, s of a chunk that starts from the state S, with W[t, s] the product of the decays of the tokens after s up to t
// times the write factor of s, A_t the product of all decays up to t and F_s = W[31, s]:
//
//     o_t = A_t S^T q_t + sum_(s <= t) P[t, s] u_s,   P[t, s] = W[t, s] (q_t . k_s)          S <- A_31 S + sum_s k_s (F_s u_s)^T
//
// light: u = v;  mlstm: o divided by the normaliser, itself such a recurrence with u = 1;  gla: with q~ = A_t q_t and k~ = k_s / A_s (A per channel) P[t, s] =
// q~_t . k~_s, S <- A_31 (S + sum_s k~_s v_s^T).
//
// fp32 operands of a product are three bf16 parts each, x = x0 + x1 + x2 (each rounded to nearest, so together all 24 bits of values from 2^-110 on;
// below, what is smaller than the smallest bf16 number is lost): the six products of parts that reach into 24 bits (three where the other
// operand is bf16 as it is) run at sixteen times the rate of an fp32 product.  The five small ones are summed by themselves, so that a sum over
// channels or tokens is rounded at its own size once per 32 of them; scores of 128 channels are summed as a tree.
//
// A workgroup owns (segment, head, up to 64 or 128 value columns).  A column wave has 16 columns: its state, all channels of them, stays in
// registers in the layout the products leave it, which is also that of their operand (a channel's place within its 32 is chosen so).  Four helpers
// make what columns share: parts of q and k (loaded a chunk ahead), P, the gates.  Two halves a chunk, a barrier after each:
//     columns  read-out, update                     |  P u, the store, parts of the next chunk's u and F u
//     helpers  parts of the next chunk's q and k    |  its P; gates of the two chunks after it
// mlstm: one column wave more, whose columns are the normaliser's (u = 1).
//
// What bounds a chunk is the instructions of a SIMD's waves: taking an operand to parts above all, seven instructions for two values.
#pragma once
#include "chunk_split.h"
#include "segments.h"

#include <type_traits>

using namespace dgi;

namespace {

constexpr int GLA = 3;
// gla: a chunk whose decays multiply to less (or to more than its inverse), or whose values are larger, goes by token: k~ v stays far from the largest number
constexpr float GLA_LEAST = 1e-16f, GLA_MOST_K = 1e27f, GLA_MOST_V = 1e10f;
// gates of a chunk, [32] each: W[t, s] = 2^(E_t + B_s), whole numbers and fractions; A; F; a token's own decay and write
// factor; mlstm: exp(-maximum), what F lacks of more bits; then A of the last token, whether something is not finite
constexpr int EI = 0, EF = 32, BI = 64, BF = 96, GA = 128, GF = 160, RA = 192, RC = 224, ALL = 256, BAD = 257, GX = 260, GL = 292;

template <int MODE, typename TI, int NK_, int NB_, bool ONLY_>
struct Lay {
  static constexpr int NK = NK_, DP = 32 * NK, NT = 2 * NK, NB = NB_;      // dk <= DP, 16-channel tiles, column blocks
  static constexpr bool ONLY = ONLY_;                          // states only
  static constexpr int PQ = sizeof(TI) == 2 && MODE == MLSTM ? 1 : 3, PU = sizeof(TI) == 2 && MODE != LIGHT ? 1 : 3;      // parts of q and k, of u
  static constexpr int NORM = NB, HELP = NB + (MODE == MLSTM ? 1 : 0), WAVES = HELP + 4;
  static constexpr int PREPS = MODE == MLSTM ? 3 : 4;          // helpers that take q and k to parts: mlstm's gates are a wave's work of their own
  static constexpr int ROWB = DP * 2, PARTB = C * ROWB, ARRB = PQ * PARTB;       // bytes of q or k
  static constexpr int PB = 3 * C * 64;                        // a chunk's P: parts, 32 rows of 32
  static constexpr int GC = 4, GN = MODE == MLSTM ? 324 : 260; // gates: chunks kept, floats of one
  // bytes
  static constexpr int K = 0, Q = K + 2 * ARRB, P = Q + (ONLY ? 0 : 2 * ARRB);
  static constexpr int NRM = P + (ONLY ? 0 : 2 * PB);          // mlstm: [2][2][32] 1 / normaliser, and what that lacks of it
  static constexpr int NX = NRM + (MODE == MLSTM ? 512 : 0);   // mlstm: [GC][4][32] bf16 parts of F (the normaliser's x)
  static constexpr int GT = NX + (MODE == MLSTM ? GC * 256 : 0);       // gla: [2][DP] decays of a chunk, [2][4][DP] of its eights of tokens
  static constexpr int FLAG = GT + (MODE == GLA ? 10 * DP * 4 : GC * GN * 4);      // [2][4] something not finite among q and k
  static constexpr int POW = FLAG + 32;                        // light: powers 0 .. 32 of the decay
  static constexpr int END = POW + (MODE == LIGHT ? 36 * 4 : 0);
  // two workgroups of eight waves to a compute unit, where LDS has room for them
  static constexpr int PER_SIMD = WAVES <= 8 && END <= 80 * 1024 ? 4 : WAVES <= 8 ? 2 : 3;
};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
// x less the low or the high half of p: exact, in one instruction (p finite; its other half times zero is added)
__device__ __forceinline__ float less_low(uint32_t p, float x) {
  uint32_t c = 0x0000bf80u;
  asm("" : "+s"(c));                                           // not as a literal: that would be taken for both halves
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p), __builtin_bit_cast(bf16x2, c), x, false);
}
__device__ __forceinline__ float less_high(uint32_t p, float x) {
  uint32_t c = 0xbf800000u;
  asm("" : "+s"(c));
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, p), __builtin_bit_cast(bf16x2, c), x, false);
}
// as part_of and split8 of chunk_split.h; what is not finite makes its neighbour's rest none, too
__device__ __forceinline__ uint32_t take_part(float& x0, float& x1) {
  const uint32_t p = pack_bf16x2(x0, x1);
  x0 = less_low(p, x0);
  x1 = less_high(p, x1);
  return p;
}
template <int PARTS>
__device__ __forceinline__ float take_parts8(const float* x, u32x4* p) {      // not 0: one of three parts' was not a finite number
  float none = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i], b = x[2 * i + 1];
    if constexpr (PARTS == 1) {
      p[0][i] = pack_bf16x2(a, b);
    } else {
      p[0][i] = take_part(a, b);
      p[1][i] = take_part(a, b);
      p[2][i] = pack_bf16x2(a, b);
      none = fmaf(a, 0.f, none);
    }
  }
  return none;
}
template <bool GRID>
__device__ __forceinline__ void take_products(const float* x, const float* f, const float* l, float grid, u32x4* p) {      // as split2_of
#pragma clang fp contract(off)
  // (a - a0 as one operation with the product would hold what ea adds once more)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float a = x[2 * i] * f[2 * i], b = x[2 * i + 1] * f[2 * i + 1];
    float ea = fmaf(x[2 * i], f[2 * i], -a), eb = fmaf(x[2 * i + 1], f[2 * i + 1], -b);
    if constexpr (GRID) {
      ea = fmaf(x[2 * i], l[2 * i], ea);
      eb = fmaf(x[2 * i + 1], l[2 * i + 1], eb);
      const float a0 = (a + grid) - grid, b0 = (b + grid) - grid;
      p[0][i] = pack_bf16x2(a0, b0);
      a = (a - a0) + ea;
      b = (b - b0) + eb;
      p[1][i] = take_part(a, b);
      p[2][i] = take_part(a, b);
      p[3][i] = pack_bf16x2(a, b);
    } else {
      p[0][i] = take_part(a, b);
      p[1][i] = take_part(a, b);
      p[2][i] = pack_bf16x2(a + ea, b + eb);
    }
  }
}

// Sums and maxima over lanes up to the own one, within 16 lanes and on to the next 16 of 32, through the lanes' own data paths
template <int CTRL, int ROWS>
__device__ __forceinline__ double from_lane(double x, double none) {
  const long long v = __builtin_bit_cast(long long, x), o = __builtin_bit_cast(long long, none);
  const int lo = __builtin_amdgcn_update_dpp((int)o, (int)v, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(o >> 32), (int)(v >> 32), CTRL, ROWS, 0xf, false);
  return __builtin_bit_cast(double, (long long)hi << 32 | (unsigned)lo);
}
template <typename F>
__device__ __forceinline__ double scan32(double x, double none, F f) {
  x = f(x, from_lane<0x111, 0xf>(x, none));                    // row_shr 1, 2, 4, 8
  x = f(x, from_lane<0x112, 0xf>(x, none));
  x = f(x, from_lane<0x114, 0xf>(x, none));
  x = f(x, from_lane<0x118, 0xf>(x, none));
  return f(x, from_lane<0x142, 0xa>(x, none));                 // row_bcast15: lane 15 (47) to the next row
}

template <int MODE, typename TI, int NK, int NB, bool ONLY>
__global__ __launch_bounds__((64 * Lay<MODE, TI, NK, NB, ONLY>::WAVES), (Lay<MODE, TI, NK, NB, ONLY>::PER_SIMD)) void chunk_segments_kernel(const ChunkArgs a) {
  using L = Lay<MODE, TI, NK, NB, ONLY>;
  constexpr int DP = L::DP, NT = L::NT, PQ = L::PQ, PU = L::PU, GC = L::GC;
  extern __shared__ __attribute__((aligned(16))) char sm[];
  Segment at;
  if (!a.ws) {                                                 // all portions whole
    at = {(int)blockIdx.y, 0, 1, 0, 0};
    at.each = a.seq_row0[at.seq + 1] - a.seq_row0[at.seq];
    if (at.each <= a.skip_rows) return;
  } else if (!find_segment(a.seq_row0, a.n_seq, a.skip_rows, a.seg_rows, a.share, C, blockIdx.y, reinterpret_cast<int*>(sm), at)) {
    return;
  }
  const int index = at.place;
  const int seq = at.seq, seg = at.seg, segs = at.segs;
  if (ONLY && seg + 1 == segs) return;
  const int H = a.H, dk = a.dk, dv = a.dv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n16 = lane & 15, g = lane >> 4;
  const int head = blockIdx.x % H, zb = blockIdx.x / H;        // consecutive workgroups go to different XCDs
  const int all0 = a.seq_row0[seq], slot = a.seq_slots[seq];
  const int len = a.seq_row0[seq + 1] - all0;
  const int row0 = all0 + seg * at.each, n = min(at.each, len - seg * at.each), chunks = (n + C - 1) / C;
  const bool stored = a.positions[all0] > 0;
  const float qscale = 1.f / sqrtf((float)dk);
  auto gates_of = [&](int c) { return reinterpret_cast<float*>(sm + L::GT) + (c & (GC - 1)) * L::GN; };
  auto chunk_decay = [&](int c) { return reinterpret_cast<float*>(sm + L::GT) + (c & 1) * DP; };      // gla
  // 16 bytes (8 channels) of a row of q or k: chunks of 16 bytes change places by row, so that eight rows' are eight places
  auto place = [&](int row, int ch16) { return row * L::ROWB + ((ch16 ^ (row & 7)) << 4); };
  // 16 bytes (8 tokens) of a row of P.  Tokens lie as the waves hold them: token 16 h + 4 g + r at 8 g + 4 h + r
  auto p_place = [&](int row, int g8) { return row * 64 + ((g8 ^ ((row >> 1) & 3)) << 4); };

  // The workspace has, of every segment and head, the blocks' registers (the normaliser's last) and two doubles: the product of its decays (mlstm: their
  // sum) and the maximum;  gla: the product of each channel's.
  auto wsd_at = [&](int index) { return reinterpret_cast<const double*>(a.wsd) + ((size_t)index * H + head) * 2; };
  auto wsd_to = [&](int index) { return reinterpret_cast<double*>(a.wsd) + ((size_t)index * H + head) * 2; };
  auto channels_at = [&](int index) { return a.wsd + ((size_t)index * H + head) * dk; };      // gla
  const double NOTHING = -1e30;                                // mlstm: the maximum of no tokens
  // mlstm: the running maximum that the segment starts from
  auto first_maximum = [&]() {
    if (seg == 0) return !stored ? 0. : !ONLY && segs > 1 ? wsd_at(index + segs - 1)[1] : (double)a.mx[(size_t)slot * H + head];
    double m = NOTHING, after = 0.;
    if constexpr (!ONLY) {
      for (int i = 1; i <= seg; ++i) {
        const double* d = wsd_at(index - i);
        m = fmax(m, d[1] + after);
        after += d[0];
      }
    }
    return m;
  };

  if (wave >= L::HELP) {
    // ============================================================================================== helpers
    const int help = wave - L::HELP;
    const TI* qb = (const TI*)a.q + (size_t)row0 * a.q_stride + (size_t)head * dk;
    const TI* kb = (const TI*)a.k + (size_t)row0 * a.k_stride + (size_t)head * dk;
    const unsigned sk = a.k_stride * (unsigned)sizeof(TI), sq = a.q_stride * (unsigned)sizeof(TI);
    // a lane takes eight channels of a row, a unit of a wave is RPU rows of k, or of q, units go round the waves
    constexpr int PER = DP / 8, RPU = 64 / PER, HALF = C / RPU, UNITS = ONLY ? HALF : 2 * HALF, TASKS = (UNITS + L::PREPS - 1) / L::PREPS;
    const int piece = lane % PER, r0 = lane / PER;
    Raw4<TI> raw[TASKS][2];
    // gla: a lane takes two channels of TPL tokens of the wave's eight; what the eights decay by is there a chunk before
    constexpr int PAIRS = DP / 2, HALVES = 64 / PAIRS, TPL = 8 / HALVES;
    typedef std::conditional_t<sizeof(TI) == 2, uint32_t, u32x2> Pair;
    const int pair = lane % PAIRS, half = lane / PAIRS;
    Pair rq[TPL], rk[TPL];
    u32x2 rd[TPL], rn[TPL];                                    // decays of the next chunk, of the one after it
    auto eights = [&](int c) { return reinterpret_cast<float*>(sm + L::GT) + (2 + 4 * (c & 1)) * DP; };
    float prod[2] = {1.f, 1.f};                                // gla: of the segment's decays
    auto load_qk = [&](int c) __attribute__((always_inline)) {
      const int first = min(c * C, n - 1), rows = min(n - first, C);
      const unsigned width = dk * (unsigned)sizeof(TI);
      if constexpr (MODE == GLA) {
        const Rows pk = rows_at(kb + (size_t)first * a.k_stride, (rows - 1) * sk + width), pq = rows_at(qb + (size_t)first * a.q_stride, (rows - 1) * sq + width);
        const unsigned ch = min(2 * pair, dk - 2);
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
          const unsigned row = 8 * help + TPL * half + i;
          rk[i] = row_load<Pair>(pk, row * sk + ch * (unsigned)sizeof(TI), 0);
          if constexpr (!ONLY) rq[i] = row_load<Pair>(pq, row * sq + ch * (unsigned)sizeof(TI), 0);
        }
      } else {
#pragma unroll
        for (int j = 0; j < TASKS; ++j) {
          const int u = help + L::PREPS * j;
          if (L::PREPS * TASKS > UNITS && u >= UNITS) break;
          const unsigned s = u < HALF ? sk : sq, to = (r0 + u % HALF * RPU) * s;
          const Rows p = rows_at(u < HALF ? kb + (size_t)first * a.k_stride : qb + (size_t)first * a.q_stride, (rows - 1) * s + width);
          raw[j][0] = row_load<Raw4<TI>>(p, to + min(8 * piece, dk - 4) * (unsigned)sizeof(TI), 0);
          raw[j][1] = row_load<Raw4<TI>>(p, to + min(8 * piece + 4, dk - 4) * (unsigned)sizeof(TI), 0);
        }
      }
    };
    auto load_decays = [&](int c) __attribute__((always_inline)) {
      if constexpr (MODE == GLA) {
        const int first = min(c * C, n - 1), rows = min(n - first, C);
        const unsigned sd = a.aux1_stride * 4u, ch = min(2 * pair, dk - 2);
        const Rows pd = rows_at((const float*)a.aux1 + (size_t)(row0 + first) * a.aux1_stride + (size_t)head * dk, (rows - 1) * sd + dk * 4u);
#pragma unroll
        for (int i = 0; i < TPL; ++i) rn[i] = row_load<u32x2>(pd, (8 * help + TPL * half + i) * sd + ch * 4u, 0);
      }
    };
    auto take_decays = [&](int c) __attribute__((always_inline)) {      // of chunk c, then the loads of the next
      if constexpr (MODE == GLA) {
        float own[2] = {1.f, 1.f};
#pragma unroll
        for (int i = 0; i < TPL; ++i)
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const float f = 2 * pair < dk && c * C + 8 * help + TPL * half + i < n ? __uint_as_float(rn[i][x]) : 1.f;
            own[x] *= f;
            rd[i][x] = __float_as_uint(f);
          }
        if constexpr (HALVES == 2) {
          own[0] *= __shfl_xor(own[0], 32, 64);
          own[1] *= __shfl_xor(own[1], 32, 64);
        }
        if (half == 0) *reinterpret_cast<float2*>(eights(c) + help * DP + 2 * pair) = make_float2(own[0], own[1]);
        load_decays(c + 1);
      }
    };
    auto put_qk = [&](int c) __attribute__((always_inline)) {  // then the loads of the next
      const int left = n - c * C, buf = c & 1;
      float most = 0.f, none = 0.f;
      bool bad = false;
      if constexpr (MODE == GLA) {
        const bool in = 2 * pair < dk;
        auto both = [](const Pair& r, float* f) {
          if constexpr (sizeof(TI) == 2) {
            f[0] = __uint_as_float(r << 16); f[1] = __uint_as_float(r & 0xffff0000u);
          } else {
            f[0] = __uint_as_float(r[0]); f[1] = __uint_as_float(r[1]);
          }
        };
        float run[2] = {1.f, 1.f}, least = 1.f, top = 1.f;     // product of the decays up to a token
#pragma unroll
        for (int j = 0; j < 3; ++j)
          if (j < help) {
            const float2 f = *reinterpret_cast<const float2*>(eights(c) + j * DP + 2 * pair);
            run[0] *= f.x;
            run[1] *= f.y;
          }
        if constexpr (HALVES == 2) {
          float own[2] = {1.f, 1.f};
#pragma unroll
          for (int i = 0; i < TPL; ++i)
#pragma unroll
            for (int x = 0; x < 2; ++x) own[x] *= __uint_as_float(rd[i][x]);
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const float other = __shfl_xor(own[x], 32, 64);
            run[x] *= half ? other : 1.f;
          }
        }
#pragma unroll
        for (int i = 0; i < TPL; ++i) {
          const int row = 8 * help + TPL * half + i;
          float k[2], q[2];
          both(rk[i], k);
          if constexpr (!ONLY) both(rq[i], q);
#pragma unroll
          for (int x = 0; x < 2; ++x) {
            const bool ok = in && row < left;
            run[x] *= __uint_as_float(rd[i][x]);
            least = fminf(least, run[x]);
            top = fmaxf(top, run[x]);
            k[x] = ok ? k[x] * __builtin_amdgcn_rcpf(run[x]) : 0.f;
            if constexpr (!ONLY) q[x] = ok ? q[x] * qscale * run[x] : 0.f;
          }
          most = larger3(most, k[0], k[1]);
          const int to = buf * L::ARRB + place(row, pair >> 2) + 4 * (pair & 3);
          auto put = [&](char* at, float* x) __attribute__((always_inline)) {
            *reinterpret_cast<uint32_t*>(at) = take_part(x[0], x[1]);
            *reinterpret_cast<uint32_t*>(at + L::PARTB) = take_part(x[0], x[1]);
            *reinterpret_cast<uint32_t*>(at + 2 * L::PARTB) = pack_bf16x2(x[0], x[1]);
            none = fmaf(x[0], 0.f, none);
          };
          put(sm + L::K + to, k);
          if constexpr (!ONLY) put(sm + L::Q + to, q);
        }
        bad = !(most < GLA_MOST_K && least > GLA_LEAST && top < 1.f / GLA_LEAST);
        if (help == 3 && half == HALVES - 1) {
          *reinterpret_cast<float2*>(chunk_decay(c) + 2 * pair) = make_float2(run[0], run[1]);
          if (ONLY && left > 0) {
            prod[0] *= run[0];
            prod[1] *= run[1];
          }
        }
        take_decays(c + 1);
      } else {
#pragma unroll
        for (int j = 0; j < TASKS; ++j) {
          const int u = help + L::PREPS * j;
          if (L::PREPS * TASKS > UNITS && u >= UNITS) break;
          const int row = r0 + u % HALF * RPU;
          float x[8];
          widen(raw[j][0], x);
          widen(raw[j][1], x + 4);
          if constexpr (MODE == LIGHT) {
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = silu(x[i]);     // zeros stay zeros
          }
          if (left < C || dk < DP) {                           // rows past the portion, channels past dk: zeros
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = row < left && 8 * piece + i < dk ? x[i] : 0.f;
          }
          u32x4 p[3];
#pragma unroll
          for (int i = 0; i < 8; i += 2) most = larger3(most, x[i], x[i + 1]);
          none += take_parts8<PQ>(x, p);                       // one part: what is not a number stays in its channel
          char* to = sm + (u < HALF ? L::K : L::Q) + buf * L::ARRB + place(row, piece);
#pragma unroll
          for (int i = 0; i < PQ; ++i) *reinterpret_cast<u32x4*>(to + i * L::PARTB) = p[i];
        }
        bad = !(most < MOST);
      }
      bad = __any(bad || none != 0.f);
      if (lane == 0) reinterpret_cast<int*>(sm + L::FLAG)[buf * 4 + help] = bad;
      load_qk(c + 1);
    };

    if (help == 3) {
      // -------------------------------------------------------------------------------------------- gates
      // A call takes 64 tokens, one per lane: chunks 2 j and 2 j + 1
      const int t = lane & 31;
      const float base = MODE == LIGHT ? a.par1[head] : 0.f;
      const double qs2 = MODE == MLSTM ? -0.5 * log2((double)dk) : 0.;
      double m_run = 0., sum = 0.;                             // mlstm: running maximum, sum of the decays
      float ga = 0.f, gb = 0.f;                                // raw gates of the next call's tokens
      auto load_gates = [&](int j) __attribute__((always_inline)) {
        if constexpr (MODE == MLSTM) {
          const size_t at = row0 + min(64 * j + lane, n - 1);
          ga = ((const float*)a.aux1)[at * a.aux1_stride + head];
          gb = ((const float*)a.aux2)[at * a.aux2_stride + head];
        }
      };
      // mlstm: in three steps, a half of a chunk each; what they hand on:
      double ld = 0., lc = 0., E = 0., B = 0.;                 // forget and input gate, natural
      bool bad = false;
      float mine = 0.f, before = 0.f;                          // the maximum, and that of the token before
      auto gates1 = [&](int j) __attribute__((always_inline)) {
        if constexpr (MODE == MLSTM) {
          const bool ok = 64 * j + lane < n;
          const float z = ok ? logsigmoid_f(a.cap * tanhf(gb / a.cap)) : 0.f, x = ok ? a.cap * tanhf(ga / a.cap) : -1e30f;
          ld = z;
          lc = x;
          bad = ok && !(fabsf(z) < 1e30f && fabsf(x) < 1e30f);
          load_gates(j + 1);
        }
      };
      auto gates2 = [&](int j) __attribute__((always_inline)) {
        const int c = 2 * j + (lane >> 5);
        const bool ok = 64 * j + lane < n;
        float* G = gates_of(c);
        if constexpr (MODE == LIGHT) {
          // powers of the decay: rows past the portion do not decay
          const float* pw = reinterpret_cast<const float*>(sm + L::POW);
          const int end = min(n - c * C, C);
          G[GA + t] = pw[min(t + 1, max(end, 0))];
          G[GF + t] = t < end ? pw[end - 1 - t] : 0.f;
          G[RA + t] = t < end ? base : 1.f;
          G[RC + t] = t < end ? 1.f : 0.f;
          if (t == 0) {
            G[ALL] = pw[max(end, 0)];
            G[BAD] = finite(pw[32]) ? 0.f : 1.f;
          }
        } else if constexpr (MODE == MLSTM) {
          const bool cold = __any(bad);
          if (t == 0) G[BAD] = cold ? 1.f : 0.f;
          const double Z = scan32(ld, 0., [](double x, double y) { return x + y; });      // sums within each chunk
          if constexpr (ONLY) sum += __shfl(Z, 31, 64) + __shfl(Z, 63, 64);
          // m_t = Z_t + max(m_0, max over s <= t of i_s - Z_s), in 64 bits: its rounding would be the state's, which the loop's is free of (a maximum
          // that only decays has a factor of exactly 1 there)
          double top = scan32(lc - Z, -1e300, [](double x, double y) { return fmax(x, y); });
          const double mid = __shfl(Z, 31, 64) + fmax(m_run, __shfl(top, 31, 64));
          double own = lane < 32 ? m_run : mid;                // the chunk's starting maximum
          top = fmax(own, top);
          E = -top * LOG2E;
          B = ok ? (lc - Z) * LOG2E : -1e5;
          double m = Z + top;
          const double end = __shfl(E, 31, 32);
          if (__builtin_expect(cold, 0)) {                     // one after the other, as the loop does
            float x = (float)m_run;
#pragma unroll 1
            for (int j = 0; j < 64; ++j) {
              x = fmaxf(__shfl((float)ld, j, 64) + x, __shfl((float)lc, j, 64));
              if (lane == j) m = x;
              if (j == 31 && lane >= 32) own = x;
            }
          }
          m_run = __shfl(m, 63, 64);
          mine = (float)m;
          before = __shfl_up(mine, 1, 32);
          if (t == 0) before = (float)own;
          own *= LOG2E;
          G[GA + t] = power_once(E + own + qs2);
          float rest = 0.f, F = power_once(end + B, &rest);
          F = ok ? F : 0.f;
          rest = ok ? rest : 0.f;
          G[GF + t] = F;
          G[GL + t] = rest;
          // the normaliser's operand: as take_products
          float most = F;
#pragma unroll
          for (int o = 16; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o, 32));
          const float grid = grid_of(most), x0 = (F + grid) - grid;
          float x = (F - x0) + rest, none = 0.f;
          uint16_t* X = reinterpret_cast<uint16_t*>(sm + L::NX + (c & (GC - 1)) * 256) + 8 * ((t >> 2) & 3) + 4 * (t >> 4) + (t & 3);
          X[0] = (uint16_t)pack_bf16x2(x0, 0.f);
          X[32] = (uint16_t)part_of(x, none);
          X[64] = (uint16_t)part_of(x, none);
          X[96] = (uint16_t)pack_bf16x2(x, 0.f);
          if (t == 31) G[ALL] = power_once(end + own);
        }
      };
      auto gates3 = [&](int j) __attribute__((always_inline)) {
        if constexpr (MODE == MLSTM) {
          const int c = 2 * j + (lane >> 5);
          const bool ok = 64 * j + lane < n;
          float* G = gates_of(c);
          G[RA + t] = ok ? expf((float)ld + before - mine) : 1.f;
          G[RC + t] = ok ? expf((float)lc - mine) : 0.f;
          G[GX + t] = expf(-mine);
          float i, f;
          whole_and_part(E + qs2, i, f);
          G[EI + t] = i;
          G[EF + t] = f;
          whole_and_part(B, i, f);
          G[BI + t] = i;
          G[BF + t] = f;
        }
      };
      load_gates(0);
      if constexpr (MODE == GLA) {
        load_decays(0);
        take_decays(0);
        __syncthreads();
      }
      if (L::PREPS == 4) load_qk(0);
      else if (lane < 2) reinterpret_cast<int*>(sm + L::FLAG)[4 * lane + 3] = 0;
      if constexpr (MODE == LIGHT) {
        float* pw = reinterpret_cast<float*>(sm + L::POW);
        double p = 1.;
        for (int i = 0; i < 33; ++i) {
          if (lane == 0) pw[i] = (float)p;
          p *= (double)base;
        }
        __builtin_amdgcn_wave_barrier();
      }
      if constexpr (MODE == MLSTM) {
        m_run = first_maximum();
        if (ONLY && seg == 0 && stored && zb == 0 && lane == 0) wsd_to(index + segs - 1)[1] = m_run;
      }
      gates1(0);
      gates2(0);
      gates3(0);
      if (L::PREPS == 4) put_qk(0);
      __syncthreads();
      if constexpr (!ONLY) __syncthreads();
      for (int c = 0; c < chunks; ++c) {
        // those of chunks c + 2 and c + 3 from an even step on
        const int j = c / 2 + 1;
        const bool there = 2 * j < chunks, due = there && !(c & 1), late = there && (c & 1);
        if (L::PREPS == 4) put_qk(c + 1);
        if (due) gates1(j);
        if constexpr (ONLY) {
          if (late) gates2(j);
          if (late) gates3(j);
        } else {
          if (late) gates3(j);
          __syncthreads();
          if (due) gates2(j);
        }
        __syncthreads();
      }
      if constexpr (ONLY) {
        if (zb > 0) return;
        if constexpr (MODE == GLA) {
          if (half == HALVES - 1 && 2 * pair < dk) *reinterpret_cast<float2*>(a.wsd + ((size_t)index * H + head) * dk + 2 * pair) = make_float2(prod[0], prod[1]);
        } else if (lane == 0) {
          if constexpr (MODE == LIGHT) {
            sum = 1.;
            double x = (double)base;
            for (int e = n; e > 0; e >>= 1) {
              if (e & 1) sum *= x;
              x *= x;
            }
          }
          wsd_to(index)[0] = sum;
          if constexpr (MODE == MLSTM) wsd_to(index)[1] = m_run;
        }
      } else if (MODE == MLSTM && seg + 1 == segs && zb == 0 && lane == 0) {
        (a.mx_new ? a.mx_new[(size_t)seq * H + head] : a.mx[(size_t)slot * H + head]) = (float)m_run;
      }
      return;
    }

    // ---------------------------------------------------------------------------------------------- scores
    load_qk(0);
    if constexpr (MODE == GLA) {
      load_decays(0);
      take_decays(0);
      __syncthreads();
    }
    put_qk(0);
    if constexpr (ONLY) {
      __syncthreads();
      for (int c = 0; c < chunks; ++c) {
        put_qk(c + 1);
        __syncthreads();
      }
    } else {
      // P of tokens after the row's own: never written again
      for (int i = help * 64 + lane; i < 2 * L::PB / 16; i += 192) *reinterpret_cast<u32x4*>(sm + L::P + 16 * i) = u32x4{0, 0, 0, 0};
      // tiles of tokens s (rows 4 g + r) and t (columns n16): 0: s and t early, 1: s early, t late, 2: both late
      const int s = help == 2, t = help > 0;
      float wl[4];
      auto scores = [&](int c) __attribute__((always_inline)) {
        f32x4 hi = {0.f, 0.f, 0.f, 0.f}, lo[1] = {{0.f, 0.f, 0.f, 0.f}}, mid = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < NK; ++b) {
          u32x4 kf[1][PQ], qf[1][PQ];
#pragma unroll
          for (int p = 0; p < PQ; ++p) {
            kf[0][p] = *reinterpret_cast<const u32x4*>(sm + L::K + (c & 1) * L::ARRB + p * L::PARTB + place(16 * s + n16, 4 * b + g));
            qf[0][p] = *reinterpret_cast<const u32x4*>(sm + L::Q + (c & 1) * L::ARRB + p * L::PARTB + place(16 * t + n16, 4 * b + g));
          }
          small<PQ, PQ, 1, 1>(kf, qf, lo);                     // as read_out's sums; of four blocks a tree
          f32x4& to = NK == 4 && b == 2 ? mid : b + 1 < NK ? hi : lo[0];
          to = mfma(kf[0][0], qf[0][0], to);
        }
        const f32x4 qk = NK == 4 ? hi + (mid + lo[0]) : hi + lo[0];
        float w[4], x[4], rest[4];
        if constexpr (MODE == LIGHT) {
#pragma unroll
          for (int r = 0; r < 4; ++r) w[r] = wl[r];
        } else if constexpr (MODE == MLSTM) {
          const float* G = gates_of(c);
          const float4 bi = ld4(G + BI + 16 * s + 4 * g), bf = ld4(G + BF + 16 * s + 4 * g);
          const float ei = G[EI + 16 * t + n16], ef = G[EF + 16 * t + n16];
          w[0] = power(ei + bi.x, ef + bf.x); w[1] = power(ei + bi.y, ef + bf.y);
          w[2] = power(ei + bi.z, ef + bf.z); w[3] = power(ei + bi.w, ef + bf.w);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool in = help == 1 || 4 * g + r <= n16;
          x[r] = in ? MODE == GLA ? qk[r] : qk[r] * w[r] : 0.f;
          rest[r] = MODE != GLA && in ? fmaf(qk[r], w[r], -x[r]) : 0.f;
        }
        char* to = sm + L::P + (c & 1) * L::PB + p_place(16 * t + n16, g) + 8 * s;
        uint2 p;
        p.x = take_part(x[0], x[1]); p.y = take_part(x[2], x[3]);
        *reinterpret_cast<uint2*>(to) = p;
        p.x = take_part(x[0], x[1]); p.y = take_part(x[2], x[3]);
        *reinterpret_cast<uint2*>(to + C * 64) = p;
        p.x = pack_bf16x2(x[0] + rest[0], x[1] + rest[1]); p.y = pack_bf16x2(x[2] + rest[2], x[3] + rest[3]);
        *reinterpret_cast<uint2*>(to + 2 * C * 64) = p;
      };
      __syncthreads();
      if constexpr (MODE == LIGHT) {                           // W is every chunk's
        const float* pw = reinterpret_cast<const float*>(sm + L::POW);
#pragma unroll
        for (int r = 0; r < 4; ++r) wl[r] = pw[max((help == 1 ? 16 : 0) + n16 - 4 * g - r, 0)];
      }
      scores(0);
      __syncthreads();
      for (int c = 0; c < chunks; ++c) {
        put_qk(c + 1);
        __syncthreads();
        if (c + 1 < chunks) scores(c + 1);
        __syncthreads();
      }
    }
    return;
  }

  // ================================================================================================ columns
  const bool ones = MODE == MLSTM && wave == L::NORM;          // the normaliser's columns are all the same
  const int block = ones ? 0 : zb * NB + wave, col = block * 16 + n16, colc = ones ? 0 : min(col, dv - 1);
  const bool cok = !ones && col < dv;
  if (!ones && block * 16 >= dv) {
    for (int i = 0; i < (ONLY ? chunks + 1 : 2 * chunks + 2) + (MODE == GLA ? 1 : 0); ++i) __syncthreads();
    return;
  }
  auto tok = [&](int i) { return 16 * (i >> 2) + 4 * g + (i & 3); };      // token 16 h + 4 g + r is value 4 h + r
  const TI* vb = (const TI*)a.v + (size_t)row0 * a.v_stride + (size_t)head * dv;
  TI rv[8];
  const unsigned sv = a.v_stride * (unsigned)sizeof(TI), vv = 4 * g * sv + colc * (unsigned)sizeof(TI);
  auto load_v = [&](int c) __attribute__((always_inline)) {
    const int first = min(c * C, n - 1), rows = min(n - first, C);
    const Rows p = rows_at(vb + (size_t)first * a.v_stride, (rows - 1) * sv + dv * (unsigned)sizeof(TI));
    const bool full = rows == C;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned off = (16 * (i >> 2) + (i & 3)) * sv;
      rv[i] = row_load<TI>(p, vv + (full ? 0 : off), full ? off : 0);
    }
  };
  auto from_gates = [&](const float* G, float* f) {            // this lane's tokens' factors
    const float4 x = ld4(G + 4 * g), y = ld4(G + 16 + 4 * g);
    f[0] = x.x; f[1] = x.y; f[2] = x.z; f[3] = x.w; f[4] = y.x; f[5] = y.y; f[6] = y.z; f[7] = y.w;
  };
  float* yb = a.y + (size_t)row0 * H * dv + (size_t)head * dv;
  // tile i, register r of a state is channel 32 (i / 2) + 8 g + 4 (i % 2) + r, so tiles 2 b and 2 b + 1 are the operand of channels 32 b .. + 31
  auto chan = [](int g, int i, int r) { return 32 * (i >> 1) + 8 * g + 4 * (i & 1) + r; };

  // 1 / x, and what it lacks (0 of one that is not finite): an output is rounded once by its division
  auto put_quotient = [&](int c, int t, float x) {
    float* to = reinterpret_cast<float*>(sm + L::NRM) + (c & 1) * 64 + t;
    const float f = 1.f / x, rest = f * fmaf(-x, f, 1.f);
    to[0] = f;
    to[32] = finite(rest) ? rest : 0.f;
  };
  f32x4 S[NT];
  // A chunk with something that is not finite goes token by token, as the recurrence is written: parts of an infinity are no numbers, and a matrix
  // product multiplies a token's values by the zeros of those before it.  Each wave decides for itself.
  auto by_token = [&](int c) __attribute__((always_inline)) {
    const float* G = gates_of(c);
    const int end = min(n - c * C, C);
    int ge = g, ce = colc;                                     // addresses are made here, not kept all the way
    asm volatile("" : "+v"(ge), "+v"(ce));
    auto row_of = [&](const void* rows, int stride, int t) {   // channels past dk read zeros
      return rows_at((const TI*)rows + (size_t)(row0 + c * C + t) * stride + (size_t)head * dk, dk * (unsigned)sizeof(TI));
    };
    auto values = [&](Rows r, int i, float* f) __attribute__((always_inline)) {
      widen(row_load<Raw4<TI>>(r, chan(ge, i, 0) * (unsigned)sizeof(TI), 0), f);
#pragma unroll
      for (int x = 0; x < 4; ++x) f[x] = MODE == LIGHT ? silu(f[x]) : f[x];
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int t = 0; t < end; ++t) {
      float own = ones ? 1.f : ldf<TI>(vb + (size_t)(c * C + t) * a.v_stride + ce);
      if constexpr (MODE == LIGHT) own = silu(own);
      const float decay = MODE == GLA ? 0.f : G[RA + t], ut = MODE == GLA ? own : own * G[RC + t];
      float o = 0.f;
      const Rows rk = row_of(a.k, a.k_stride, t), rq = row_of(a.q, a.q_stride, t);
      const Rows rd = rows_at((const float*)a.aux1 + (size_t)(row0 + c * C + t) * a.aux1_stride + (size_t)head * dk, MODE == GLA ? dk * 4u : 0u);
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        float k[4], q[4];
        u32x2 d[2];
        values(rk, i, k);
        if constexpr (!ONLY) values(rq, i, q);
        if constexpr (MODE == GLA) {
          d[0] = row_load<u32x2>(rd, chan(ge, i, 0) * 4u, 0);
          d[1] = row_load<u32x2>(rd, chan(ge, i, 2) * 4u, 0);
        }
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          S[i][x] = fmaf(k[x], ut, S[i][x] * (MODE == GLA ? __uint_as_float(d[x >> 1][x & 1]) : decay));
          if constexpr (!ONLY) o = fmaf(q[x], S[i][x], o);
        }
      }
      if constexpr (!ONLY) {
        o += __shfl_xor(o, 16, 64);
        o += __shfl_xor(o, 32, 64);
        if constexpr (MODE != LIGHT) o *= qscale;
        if (ones) put_quotient(c, t, fmaxf(fabsf(o), G[GX + t]) + 1e-6f);
        else if (ge == 0 && cok) yb[(size_t)(c * C + t) * H * dv + ce] = o;      // mlstm: still to be divided
      }
    }
  };

  // ------------------------------------------------------------------------------------------------ the state
  const size_t sbase = ((size_t)slot * H + head) * dk * dv, nbase = ((size_t)slot * H + head) * dk;
  auto sat = [&](int ch) { return ones ? (size_t)ch : (size_t)ch * dv + colc; };
  auto begin = [&]() __attribute__((always_inline)) {
    const float* from = ones ? a.norm + nbase : a.state + sbase;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = (stored && chan(g, i, r) < dk && (cok || ones)) ? from[sat(chan(g, i, r))] : 0.f;
  };
  const int blocks = a.blocks;
  auto ws_at = [&](int index) { return reinterpret_cast<f32x4*>(a.ws) + (((size_t)index * H + head) * blocks + (ones ? blocks - 1 : block)) * (NT * 64) + lane; };
  auto write_ws = [&](int index) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NT; ++i) ws_at(index)[64 * i] = S[i];
  };
  auto read_ws = [&](int index, f32x4 (&X)[NT]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NT; ++i) X[i] = ws_at(index)[64 * i];
  };
  load_v(0);
  if constexpr (MODE == GLA) __syncthreads();
  if (seg == 0) {
    if (!ONLY && segs > 1 && stored) read_ws(index + segs - 1, S);
    else begin();
    if (ONLY && stored) write_ws(index + segs - 1);
  } else {
#pragma unroll
    for (int i = 0; i < NT; ++i) S[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (!ONLY) {
      // the states before, the latest first, each times the decays of those after it; the next one under way
      const double m = MODE == MLSTM ? first_maximum() : 0.;
      double after = MODE == MLSTM ? 0. : 1.;
      f32x4 X[NT], factor[MODE == GLA ? NT : 1];
#pragma unroll
      for (int i = 0; i < (MODE == GLA ? NT : 1); ++i) factor[i] = f32x4{1.f, 1.f, 1.f, 1.f};
      constexpr bool AHEAD = NK == 2;                          // else there are no registers for it
      if (AHEAD) read_ws(index - 1, X);
      for (int i = 1; i <= seg; ++i) {
        f32x4 Y[NT];
        if (AHEAD) read_ws(index - min(i + 1, seg), Y);
        else read_ws(index - i, X);
        float w = 0.f;
        if constexpr (MODE != GLA) {
          const double* d = wsd_at(index - i);
          w = MODE == MLSTM ? power_once((d[1] + after - m) * LOG2E) : (float)after;
          after = MODE == MLSTM ? after + d[0] : after * d[0];
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if constexpr (MODE == GLA) {
              S[j][r] = fmaf(factor[j][r], X[j][r], S[j][r]);
              factor[j][r] *= channels_at(index - i)[min(chan(g, j, r), dk - 1)];
            } else {
              S[j][r] = fmaf(w, X[j][r], S[j][r]);
            }
          }
          if (AHEAD) X[j] = Y[j];
        }
      }
    }
  }
  auto keep_state = [&]() __attribute__((always_inline)) {
    if constexpr (ONLY) {
      write_ws(index);
      return;
    }
    if (seg + 1 < segs) return;
    float* to = ones ? (a.norm_new ? a.norm_new + ((size_t)seq * H + head) * dk : a.norm + nbase) : a.state + sbase;
    const bool keep = ones ? zb == 0 && n16 == 0 : cok;
    // addresses are made anew: those of the loads would be kept all the way
    int ge = g;
    asm volatile("" : "+v"(ge));
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ch = chan(ge, i, r);
        if (keep && ch < dk) to[sat(ch)] = S[i][r];
      }
  };
  // N tiles of k, channels by tokens
  constexpr int N = 2;
  auto read_k = [&](int c, int j, u32x4 (&kf)[N][PQ]) __attribute__((always_inline)) {
    const char* K = sm + L::K + (c & 1) * L::ARRB;
    const int tq = n16 >> 2, tp = n16 & 3;
#pragma unroll
    for (int y = 0; y < N; ++y)
#pragma unroll
      for (int p = 0; p < PQ; ++p)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const short4v v = read_tr(K + p * L::PARTB + place(16 * h + 4 * g + tq, 4 * ((j + y) >> 1) + tp) + 8 * ((j + y) & 1));
          kf[y][p][2 * h] = (uint32_t)(uint16_t)v[0] | ((uint32_t)(uint16_t)v[1] << 16);
          kf[y][p][2 * h + 1] = (uint32_t)(uint16_t)v[2] | ((uint32_t)(uint16_t)v[3] << 16);
        }
  };
  // Parts of x = F u.  A bf16 product cuts off what lies 24 bits below the largest term of eight, which of a state that consists of its
  // last few tokens (mlstm's, whose decays are fast) would be twice a rounding.  So there the first parts of a column are multiples of one
  // 2^-7 of the largest: their products' sum is exact, the others' is 2^-8 smaller (state 5.3e-8 from 64 bits without, the token loop's 4.4e-8).
  constexpr bool GRID = MODE == MLSTM;
  constexpr int XP = GRID ? 4 : MODE == GLA ? PU : 3;
  u32x4 xp[MODE == GLA ? 1 : XP], up[PU];                      // parts of F u, of u (gla: these are both)
  bool odd = false;                                            // one of them is not a finite number, or too large for its parts
  auto take_v = [&](int c) __attribute__((always_inline)) {
    if (ones) {
#pragma unroll
      for (int i = 0; i < XP; ++i) xp[i] = *reinterpret_cast<const u32x4*>(sm + L::NX + (c & (GC - 1)) * 256 + 64 * i + 16 * g);
      return;
    }
    float u[8], f[8], l[8], most = 0.f, grid = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) u[i] = ldf<TI>(&rv[i]);        // rows past the portion: zeros (or, of rows that overlap, anything: nothing takes them)
    if constexpr (MODE == LIGHT) {
#pragma unroll
      for (int i = 0; i < 8; ++i) u[i] = silu(u[i]);
    }
    load_v(c + 1);
    if constexpr (MODE == GLA) {
#pragma unroll
      for (int i = 0; i < 8; i += 2) most = larger3(most, u[i], u[i + 1]);
      float none = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) none = fmaf(u[i], 0.f, none);
      odd = !(most < GLA_MOST_V) || none != 0.f;
      take_parts8<PU>(u, up);
      return;
    }
    from_gates(gates_of(c) + GF, f);
    if constexpr (GRID) from_gates(gates_of(c) + GL, l);
    // a factor is finite (else its chunk goes by token anyway), so only a value that is none makes a product that is none
#pragma unroll
    for (int i = 0; i < 8; i += 2) most = larger3(most, u[i] * f[i], u[i + 1] * f[i + 1]);
    if constexpr (GRID) {
      odd = !(most < 1e30f);
      most = fmaxf(most, __shfl_xor(most, 16, 64));
      most = fmaxf(most, __shfl_xor(most, 32, 64));
      grid = grid_of(most);
    } else {
      odd = !(most < MOST);
    }
    take_products<GRID>(u, f, l, grid, xp);
    if constexpr (!ONLY && PU == 3) {
      float largest = 0.f;
#pragma unroll
      for (int i = 0; i < 8; i += 2) largest = larger3(largest, u[i], u[i + 1]);
      const float none = take_parts8<PU>(u, up);
      odd |= !(largest < MOST) || none != 0.f;
    } else {
      float none = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) none = fmaf(u[i], 0.f, none);
      odd |= none != 0.f;
      if constexpr (!ONLY) take_parts8<PU>(u, up);
    }
  };
  if (ones) {
    up[0] = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};      // P of rows past the portion is 0
#pragma unroll
    for (int i = 1; i < PU; ++i) up[i] = u32x4{0, 0, 0, 0};
  }
  auto state_big = [&]() {
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      most = larger3(most, S[i][0], S[i][1]);
      most = larger3(most, S[i][2], S[i][3]);
    }
    return !(most < MOST);
  };
  auto flagged = [&](int c) __attribute__((always_inline)) {
    const int4 F = *reinterpret_cast<const int4*>(sm + L::FLAG + (c & 1) * 16);
    return __builtin_amdgcn_readfirstlane((MODE != GLA && gates_of(c)[BAD] != 0.f) | F.x | F.y | F.z | F.w) != 0;
  };
  // S <- A S + k^T x
  auto update = [&](int c) __attribute__((always_inline)) {
    const float at = MODE == GLA ? 1.f : gates_of(c)[ALL];
    const u32x4* xs = MODE == GLA ? up : xp;
    constexpr int KEPT = PQ == 1 ? 2 : 1;                      // the next two tiles' under way, where registers are left
    u32x4 kf[KEPT][N][PQ];
    if (KEPT == 2) read_k(c, 0, kf[0]);
#pragma unroll
    for (int j = 0; j < NT; j += N) {
      u32x4(&kj)[N][PQ] = kf[j / N % KEPT];
      if (KEPT == 1) read_k(c, j, kj);
      else if (j + N < NT) read_k(c, j + N, kf[(j / N + 1) % KEPT]);
      f32x4 lo[N], hi[N];
#pragma unroll
      for (int y = 0; y < N; ++y) lo[y] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = GRID ? 3 : 2; t > 0; --t)
#pragma unroll
        for (int p = t; p >= 0; --p)
          if (p < PQ && t - p < XP) {
#pragma unroll
            for (int y = 0; y < N; ++y) lo[y] = mfma(kj[y][p], xs[t - p], lo[y]);
          }
#pragma unroll
      for (int y = 0; y < N; ++y) hi[y] = mfma(kj[y][0], xs[0], GRID ? f32x4{0.f, 0.f, 0.f, 0.f} : lo[y]);
#pragma unroll
      for (int y = 0; y < N; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if constexpr (MODE != GLA) S[j + y][r] = GRID ? hi[y][r] + fmaf(at, S[j + y][r], lo[y][r]) : fmaf(at, S[j + y][r], hi[y][r]);
      if constexpr (MODE == GLA) {                             // rounded once at the state's size
#pragma unroll
        for (int y = 0; y < N; ++y) {
          const f32x4 b = *reinterpret_cast<const f32x4*>(chunk_decay(c) + chan(g, j + y, 0));
#pragma unroll
          for (int r = 0; r < 4; ++r) S[j + y][r] = fmaf(b[r], S[j + y][r], b[r] * hi[y][r]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  if constexpr (ONLY) {
    // a chunk and a barrier; chunks by token outside the inner loop, so that their registers are not that one's
    __syncthreads();
    for (int c = 0; c < chunks; ++c) {
      bool warm = true;
      for (; c < chunks; ++c) {
        take_v(c);
        warm = !(flagged(c) || __any(odd || state_big()));
        if (__builtin_expect(!warm, 0)) break;
        update(c);
        __syncthreads();
      }
      if (warm) break;
      by_token(c);
      __syncthreads();
    }
    keep_state();
    return;
  }

  // ------------------------------------------------------------------------------------------------ read-outs
  f32x4 qS[2];                                                 // S^T q, tokens as tok()
  auto read_out = [&](int c) __attribute__((always_inline)) {
    f32x4 hi[2], lo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) hi[h] = lo[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < NK; ++b) {
      u32x4 qf[2][PQ], sp[1][3];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < PQ; ++p) qf[h][p] = *reinterpret_cast<const u32x4*>(sm + L::Q + (c & 1) * L::ARRB + p * L::PARTB + place(16 * h + n16, 4 * b + g));
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = S[2 * b + (i >> 2)][i & 3];
      take_parts8<3>(v, sp[0]);
      // the last block's first parts start from the small ones' sum: one rounding less at the sum's size
      small<PQ, 3, 2, 1>(qf, sp, lo);
#pragma unroll
      for (int h = 0; h < 2; ++h) (b + 1 < NK ? hi : lo)[h] = mfma(qf[h][0], sp[0][0], (b + 1 < NK ? hi : lo)[h]);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) qS[h] = hi[h] + lo[h];
  };
  float out[8];
  // P u and what the state gave
  auto finish = [&](int c) __attribute__((always_inline)) {
    const char* P = sm + L::P + (c & 1) * L::PB;
    float fA[8];
    u32x4 pf[2][3];
    if constexpr (MODE != GLA) from_gates(gates_of(c) + GA, fA);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int p = 0; p < 3; ++p) pf[h][p] = *reinterpret_cast<const u32x4*>(P + p * C * 64 + p_place(16 * h + n16, g));
    f32x4 lo[2], hi[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) lo[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 2; t > 0; --t)
#pragma unroll
      for (int p = t; p >= 0; --p)
        if (t - p < PU) {
#pragma unroll
          for (int h = 0; h < 2; ++h) lo[h] = mfma(pf[h][p], up[t - p], lo[h]);
        }
#pragma unroll
    for (int h = 0; h < 2; ++h) hi[h] = mfma(pf[h][0], up[0], lo[h]);
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = MODE == GLA ? qS[i >> 2][i & 3] + hi[i >> 2][i & 3] : fmaf(fA[i], qS[i >> 2][i & 3], hi[i >> 2][i & 3]);
  };
  const unsigned sy = H * dv * 4u, vy = cok ? 4 * g * sy + colc * 4u : 0x7fffffffu;      // columns past dv: nothing written
  auto store = [&](int c, const float* o, bool ok) __attribute__((always_inline)) {
    const int rows = min(n - c * C, C);
    const unsigned at = ok ? vy : 0x7fffffffu;
    const Rows p = rows_at(yb + (size_t)c * C * H * dv, rows * sy);
    const bool full = rows == C;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const unsigned off = (16 * (i >> 2) + (i & 3)) * sy;
      row_store(p, o[i], at + (full ? 0 : off), full ? off : 0);
    }
  };
  bool was_cold = false;
  auto divide = [&](int c) __attribute__((always_inline)) {    // mlstm: chunk c, a step later
    float f[8], rest[8], o[8];
    const float* from = reinterpret_cast<const float*>(sm + L::NRM) + (c & 1) * 64;
    from_gates(from, f);
    from_gates(from + 32, rest);
    if (__builtin_expect(was_cold, 0)) {
#pragma unroll
      for (int i = 0; i < 8; ++i) out[i] = yb[(size_t)min(c * C + tok(i), n - 1) * H * dv + colc];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = fmaf(out[i], f[i], __builtin_amdgcn_fmed3f(out[i], -MOST, MOST) * rest[i]);      // an infinite one stays one
    store(c, o, true);
  };

  auto first_half = [&](int c) __attribute__((always_inline)) {      // false: the chunk goes by token
    if constexpr (MODE == MLSTM) {
      if (c > 0 && !ones) divide(c - 1);
    }
    was_cold = flagged(c) || __any(odd || state_big());
    return !was_cold;
  };
  auto second_half = [&](int c) __attribute__((always_inline)) {
    __syncthreads();
    if (!was_cold) {
      finish(c);
      if (ones) {
        float o = out[0];                                      // lane n16's token
#pragma unroll
        for (int i = 1; i < 8; ++i) {
          float x = out[i];
          asm("" : "+v"(x));                                   // values, not a place in memory, are chosen from
          o = (n16 & 7) == i ? x : o;
        }
        const int t = tok(n16 & 7);
        o = fmaxf(fabsf(o), gates_of(c)[GX + t]) + 1e-6f;
        if (n16 < 8) put_quotient(c, t, o);
      }
      if constexpr (MODE != MLSTM) store(c, out, true);
    }
    if (c + 1 < chunks) take_v(c + 1);
    __syncthreads();
  };
  __syncthreads();
  take_v(0);
  __syncthreads();
  for (int c = 0; c < chunks; ++c) {
    bool warm = true;
    for (; c < chunks; ++c) {
      warm = first_half(c);
      if (__builtin_expect(!warm, 0)) break;
      read_out(c);
      update(c);
      second_half(c);
    }
    if (warm) break;
    by_token(c);
    second_half(c);
  }
  if constexpr (MODE == MLSTM) {
    if (!ones) divide(chunks - 1);
  }
  keep_state();
}

template <int MODE, typename TI, int NK, int NB, bool ONLY>
int launch_one(const ChunkArgs& a, dim3 grid, hipStream_t st) {
  using L = Lay<MODE, TI, NK, NB, ONLY>;
  static_assert(L::END <= 160 * 1024, "LDS");
  auto kernel = chunk_segments_kernel<MODE, TI, NK, NB, ONLY>;
  if (L::END > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, L::END);
    if (e != hipSuccess) return (int)e;
  }
  kernel<<<grid, 64 * L::WAVES, L::END, st>>>(a);
  return 0;
}

template <int MODE, typename TI>
int launch_dims(const ChunkArgs& a, bool only, dim3 grid, hipStream_t st) {
#define DGI_SEG(NK_, NB_) (only ? launch_one<MODE, TI, NK_, NB_, true>(a, grid, st) : launch_one<MODE, TI, NK_, NB_, false>(a, grid, st))
  if constexpr (MODE != MLSTM) {
    if (a.dv > 64) return a.dk <= 64 ? DGI_SEG(2, 8) : DGI_SEG(4, 8);
    if (a.dk > 64) return DGI_SEG(4, 4);
  }
  return DGI_SEG(2, 4);
#undef DGI_SEG
}

template <int MODE>
int launch_type(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st) {
  return in_f32 ? launch_dims<MODE, float>(a, only, grid, st) : launch_dims<MODE, uint16_t>(a, only, grid, st);
}

}  // namespace
