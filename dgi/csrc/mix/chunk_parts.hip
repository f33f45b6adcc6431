// dgi/csrc/mix/chunk_parts.hip — prompt portions of the recurrences that carry a matrix S [dk, dv] per head under one decay per
// token (mlstm, light: linear_scan.hip has their definitions; ssm: ssm_scan.hip), 32 tokens at a time on the bf16 matrix cores.
//
// For tokens t, s of a chunk that starts from the state S, with W[t, s] the product of the decays of the tokens after s up to t
// times the write factor of s, A_t the product of all decays up to t and F_s = W[31, s]:
//
//     o_t = A_t S^T q_t + sum_(s <= t) P[t, s] u_s,   P[t, s] = W[t, s] (q_t . k_s)          S <- A_31 S + sum_s k_s (F_s u_s)^T
//
// light: u = v;  ssm: q = C, k = B, u = x, the skip factor on P's diagonal;  mlstm: o divided by the normaliser, itself such a recurrence with u = 1.
//
// fp32 operands of a product are three bf16 parts each, x = x0 + x1 + x2 (each rounded to nearest, so together all 24 bits of values from 2^-110 on;
// below, what is smaller than the smallest bf16 number is lost): the six products of parts that reach into 24 bits (three where the other
// operand is bf16 as it is) run at sixteen times the rate of an fp32 product.  The five small ones are summed by themselves, so that a sum over
// channels or tokens is rounded at its own size once per 32 of them; scores of 128 channels are summed as a tree.
//
// A workgroup owns (sequence, head, two blocks of 16 value columns) and is a pipeline of waves that hand chunks on through LDS, one barrier
// per chunk:
//   preparing waves  load q and k a chunk ahead in registers and write their parts to LDS (ssm of more than 64 channels, long steps: parts and scores come
//                    from a pass before, as the heads of a group and their columns share them);
//   gates wave       sums of log2 decays of 64 tokens at a time (in 64 bits), as whole number and fraction, A and F;
//   scores wave      q . k and P in parts;
//   state waves      one per block of 16 columns: the state's rows of all channels in registers, in the layout the products leave them, which is
//                    also that of their operand (a channel's place within its 32 is chosen so); the state before a chunk goes to LDS;
//   output waves     one per block: parts of that state, read-out, P u (a step later) and the store;
//   normaliser wave  (mlstm) both of a block whose u is 1.
// What bounds a chunk is the longest role's instructions: a wave issues one every four cycles, making three parts of a value is five and a half, and a
// wave's own products (16 cycles) and vector instructions do not overlap, only those of two waves of a SIMD do, in part.  So state and read-out are two
// waves', parts of the next operand are made between the products, what goes token by token is kept out of the loops' registers, and operands
// are asked for a chunk ahead (as buffers: a row is a scalar offset).  Measured against chunk_scan.hip, sixteen tokens at a time in fp32 products, on inputs that change from pass to pass:
//   ssm, 2 prompts of 4096 rows, 64 heads of 128 x 64     210 us -> 168 (of it 15 the pass before)
//   mlstm, 5 prompts of 3001 bf16 rows, 32 heads of 64     83 -> 49;  of 128 197 -> 137;  fp32 rows 105 -> 74
//   light, 2 prompts of 4096 bf16 rows, 64 heads of 64    158 -> 113
// mlstm on fp32 rows of 128 channels stays there (its waves would spill: 213 -> 230 us); delta: chunk_delta.hip; steps of mlstm and light of many short portions
// or few long ones: chunk_segments.h.
//
// Precision: results and states are no further from 64 bits than the token loop's, nor (2-norm) by more than a hundredth than in chunk_scan.hip, whose P u is in
// 64 bits.  512 rows, 16 heads, errors over that kernel's of outputs and states: ssm 0.78, 0.92 (7.0e-8; the loop 1.03e-7); light 0.46, 0.31; mlstm 0.94, 0.76 (64
// channels), 0.95, 0.84 (128); with decays near 1 at most 0.4.  mlstm's outputs by the geometric mean of tokens: bf16 rows 1.03, fp32 0.92.  What gives that:
// decays are summed as logarithms in 64 bits and a running maximum is kept in 64 bits, since its rounding would be the state's.
#include <type_traits>
#include "chunk_split.h"

using namespace dgi;

namespace {

template <int MODE, typename TI, int NK_, bool PRE_ = false>
struct Lay {
  static constexpr int NK = NK_, DP = 32 * NK, NT = 2 * NK, NB = 2;       // dk <= DP, 16-channel tiles, column blocks
  static constexpr bool PRE = PRE_;                            // ssm: parts and scores were made before
  static constexpr int PQ = sizeof(TI) == 2 && MODE != LIGHT ? 1 : 3, PU = sizeof(TI) == 2 && MODE == MLSTM ? 1 : 3;      // parts of q and k, of u
  // Waves: state, output, normaliser, gates, scores, preparing; waves four apart share a SIMD
  static constexpr int NP = PRE ? 0 : PQ == 1 ? (NK == 2 ? 1 : 2) : MODE == MLSTM ? (NK == 2 ? 2 : 4) : 4;
  static constexpr int OUT = NB, NORM = 2 * NB, GATES = NORM + (MODE == MLSTM ? 1 : 0), SCORES = GATES + 1, PREP = SCORES + 1, WAVES = PREP + NP;
  static constexpr int LEAD = MODE == MLSTM ? 3 : 2;           // steps after a chunk is prepared until it is done
  static constexpr int ROWB = DP * 2, PARTB = C * ROWB, ARRB = PQ * PARTB;       // bytes of q or k
  static constexpr int PB = 3 * C * 64;                        // a chunk's P: parts, 32 rows of 32
  static constexpr int SB = NT * 1024;                         // a block's state
  static constexpr int GR = 8, GN = 10 * 32 + 4;               // gates: chunks kept, floats of one
  // bytes
  static constexpr int Q = 0, K = Q + (PRE ? 0 : 2 * ARRB), P = K + (PRE ? 0 : 2 * ARRB);
  static constexpr int ST = P + 2 * PB;                        // [2][NB][NT][64][4] state before the chunk, as the state wave holds it
  static constexpr int NRM = ST + 2 * NB * SB;                 // mlstm: [4][2][32] 1 / normaliser, and what that lacks of it
  static constexpr int NX = NRM + (MODE == MLSTM ? 4 * 64 * 4 : 0);       // mlstm: [GR][4][32] bf16 parts of F (the normaliser's x)
  static constexpr int GT = NX + (MODE == MLSTM ? GR * 256 : 0);
  static constexpr int FLAG = GT + GR * GN * 4;                // [2][NP] something not finite among q and k
  static constexpr int SBAD = FLAG + 32;                       // [2][NB] something not finite in the state
  static constexpr int POW = SBAD + 16;                        // light: powers 0 .. 32 of the decay
  static constexpr int END = POW + 36 * 4;
  // two workgroups of eight waves to a compute unit, where LDS has room for them
  static constexpr int PER_SIMD = !PRE && WAVES <= 8 && END <= 80 * 1024 ? 4 : 2;
};
// gates of a chunk, [32] each: W[t, s] = 2^(E_t + B_s) (ssm: times the write factor), whole numbers and fractions; A; F; a token's own decay and write
// factor; mlstm: exp(-maximum), what F lacks of more bits; then A of the last token, whether something is not finite
constexpr int EI = 0, EF = 32, BI = 64, BF = 96, GA = 128, GF = 160, RA = 192, RC = 224, GX = 256, GL = 288, ALL = 320, BAD = 321;

// ssm, of each chunk and group: the parts, three score tiles and a flag (a multiple of 16 bytes)
__host__ __device__ constexpr int parts_floats(int DP) { return 2 * 3 * C * DP / 2 + 3 * 256 + 4; }

template <int MODE, typename TI, int NK, bool PRE>
__global__ __launch_bounds__((64 * Lay<MODE, TI, NK, PRE>::WAVES), (Lay<MODE, TI, NK, PRE>::PER_SIMD)) void chunk_parts_kernel(const ChunkArgs a) {
  using L = Lay<MODE, TI, NK, PRE>;
  constexpr int DP = L::DP, NT = L::NT, PQ = L::PQ, PU = L::PU, LEAD = L::LEAD;
  extern __shared__ __attribute__((aligned(16))) char sm[];
  // consecutive workgroups go to different XCDs: ssm: so that the heads of a group share one's cache (a multiple of 8 heads)
  int head = blockIdx.x % a.H;
  if (L::PRE && a.H % 8 == 0) head = head % 8 * (a.H / 8) + head / 8;
  const int zb = blockIdx.x / a.H / a.n_seq, seg = MODE == SSM ? blockIdx.y : 0;
  const int seq = __builtin_amdgcn_readfirstlane(ranked(a, blockIdx.x / a.H % a.n_seq));
  int row0 = a.seq_row0[seq], n = a.seq_row0[seq + 1] - row0;
  if (n <= a.skip_rows) return;
  const int slot = a.seq_slots[seq];
  // ssm in segments: 1 the state of a segment from nothing, to the workspace; 2 outputs from the state found there
  bool stored = MODE == SSM ? a.positions[row0] != 0 : a.positions[row0] > 0, last = true;      // as the loops of their files
  if (MODE == SSM && a.pass) {
    row0 += seg * a.seg_rows;
    n -= seg * a.seg_rows;
    last = n <= a.seg_rows;
    if (n <= 0 || (last && a.pass == 1)) return;
    n = min(n, a.seg_rows);
    stored = a.pass == 2;
  }
  const int chunk0 = first_chunk(a.seq_row0[seq], seq) + (MODE == SSM && a.pass ? seg * a.seg_rows / C : 0);      // ssm: its place in the workspace
  const int H = a.H, dk = a.dk, dv = a.dv;
  const int kvh = head / (H / a.G);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n16 = lane & 15, g = lane >> 4;
  const int chunks = (n + C - 1) / C;
  const float qscale = 1.f / sqrtf((float)dk);
  // Every role passes chunks + LEAD barriers.
  auto barriers = [&](int m) {
    for (int i = 0; i < m; ++i) __syncthreads();
  };
  auto gates_of = [&](int c) { return reinterpret_cast<float*>(sm + L::GT) + (c & (L::GR - 1)) * L::GN; };
  // 16 bytes (8 channels) of a row of q or k: chunks of 16 bytes change places by row, so that eight rows' are eight places
  auto place = [&](int row, int ch16) { return row * L::ROWB + ((ch16 ^ (row & 7)) << 4); };
  // 16 bytes (8 tokens) of a row of P or M.  Tokens lie as the column waves hold them: token 16 h + 4 g + r at 8 g + 4 h + r
  auto p_place = [&](int row, int g8) { return row * 64 + ((g8 ^ ((row >> 1) & 3)) << 4); };

  if constexpr (!L::PRE) {
  if (wave >= L::PREP) {
    // ============================================================================================== preparing waves
    const int prep = wave - L::PREP;
    constexpr int PER = DP / 8, TASKS = PER / L::NP;           // 64 times eight channels: q and k of a chunk are PER of them
    static_assert(TASKS * L::NP == PER && TASKS % 2 == 0, "tasks");
    const TI* qb = (const TI*)a.q + (size_t)row0 * a.q_stride + (size_t)kvh * dk;
    const TI* kb = (const TI*)a.k + (size_t)row0 * a.k_stride + (size_t)kvh * dk;
    Raw4<TI> raw[TASKS][2];
    const int piece = lane % PER, r0 = lane / PER;             // task j (of q, then of k): rows (64 / PER) j + r0
    constexpr int RPT = 64 / PER;
    auto first_of = [&](int j) { return RPT * (prep * (TASKS / 2) + j % (TASKS / 2)); };
    auto row_of = [&](int j) { return first_of(j) + r0; };
    const unsigned c0 = min(8 * piece, dk - 4) * (unsigned)sizeof(TI), c1 = min(8 * piece + 4, dk - 4) * (unsigned)sizeof(TI);
    const unsigned sq = a.q_stride * (unsigned)sizeof(TI), sk = a.k_stride * (unsigned)sizeof(TI), oq = r0 * sq, ok = r0 * sk;
    auto load = [&](int c) {
      const int first = min(c * C, n - 1), rows = min(n - first, C);
      const unsigned width = dk * (unsigned)sizeof(TI);
      const Rows pq = rows_at(qb + (size_t)first * a.q_stride, (rows - 1) * sq + width), pk = rows_at(kb + (size_t)first * a.k_stride, (rows - 1) * sk + width);
      const bool full = rows == C;
#pragma unroll
      for (int j = 0; j < TASKS; ++j) {
        const bool is_q = j < TASKS / 2;
        const unsigned off = first_of(j) * (is_q ? sq : sk), in = (is_q ? oq : ok) + (full ? 0 : off), row = full ? off : 0;
        raw[j][0] = row_load<Raw4<TI>>(is_q ? pq : pk, in + c0, row);
        raw[j][1] = row_load<Raw4<TI>>(is_q ? pq : pk, in + c1, row);
      }
    };
    load(0);
    for (int c = 0; c < chunks; ++c) {
      const int buf = c & 1, left = n - c * C;
      float most = 0.f;
#pragma unroll
      for (int j = 0; j < TASKS; ++j) {
        const bool is_q = j < TASKS / 2;
        const int row = row_of(j);
        float x[8];
        widen(raw[j][0], x);
        widen(raw[j][1], x + 4);
        if constexpr (MODE == LIGHT) {
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = silu(x[i]);       // zeros stay zeros
        }
        if (left < C || dk < DP) {                             // rows past the portion, channels past dk: zeros
#pragma unroll
          for (int i = 0; i < 8; ++i) x[i] = row < left && 8 * piece + i < dk ? x[i] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 8; i += 2) most = larger3(most, x[i], x[i + 1]);
        u32x4 p[3];
        split8<PQ>(x, p);
        char* to = sm + (is_q ? L::Q : L::K) + buf * L::ARRB + place(row, piece);
#pragma unroll
        for (int i = 0; i < PQ; ++i) *reinterpret_cast<u32x4*>(to + i * L::PARTB) = p[i];
      }
      load(c + 1);
      const bool bad = __any(!(most < MOST));
      if (lane == 0) reinterpret_cast<int*>(sm + L::FLAG)[buf * L::NP + prep] = bad;
      __syncthreads();
    }
    barriers(LEAD);
    return;
  }
  }

  if (wave == L::SCORES) {
    // ============================================================================================== scores wave
    // P of tokens after the row's own: never written again
    for (int i = lane; i < 2 * L::PB / 16; i += 64) *reinterpret_cast<u32x4*>(sm + L::P + 16 * i) = u32x4{0, 0, 0, 0};
    // tiles of tokens s (rows 4 g + r) and t (columns n16): 0: s and t early, 1: s early, t late, 2: both late
    f32x4 qk[3];
    const char* from = (const char*)a.parts + ((size_t)(chunk0 * a.G + kvh) * parts_floats(DP)) * 4 + 2 * L::ARRB;
    auto load_scores = [&](int c) {
      const Rows p = rows_at(from + (size_t)min(c, chunks - 1) * a.G * parts_floats(DP) * 4, 3 * 1024);
#pragma unroll
      for (int i = 0; i < 3; ++i) qk[i] = row_load<f32x4>(p, 16 * lane, 1024 * i);
    };
    auto products = [&](int c) {
      const char* Q = sm + L::Q + (c & 1) * L::ARRB;
      const char* K = sm + L::K + (c & 1) * L::ARRB;
      f32x4 hi[3], lo[3], mid[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) hi[i] = lo[i] = mid[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int b = 0; b < NK; ++b) {
        u32x4 kf[3][PQ], qf[3][PQ];                  // early, early, late by early, late, late
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int p = 0; p < PQ; ++p) {
            const int at = p * L::PARTB + place(16 * h + n16, 4 * b + g);
            kf[2 * h][p] = *reinterpret_cast<const u32x4*>(K + at);
            qf[2 * h][p] = *reinterpret_cast<const u32x4*>(Q + at);
          }
#pragma unroll
        for (int p = 0; p < PQ; ++p) { kf[1][p] = kf[0][p]; qf[1][p] = qf[2][p]; }
        small<PQ, PQ, 3, 3>(kf, qf, lo);             // as read_out's sums; of four blocks a tree
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          f32x4& sum = NK == 4 && b == 2 ? mid[i] : b + 1 < NK ? hi[i] : lo[i];
          sum = mfma(kf[i][0], qf[i][0], sum);
        }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) qk[i] = NK == 4 ? hi[i] + (mid[i] + lo[i]) : hi[i] + lo[i];
    };
    float wl[3][4];                                  // light: W is every chunk's
    const float skip = MODE == SSM ? a.par3[head] : 0.f;
    // four values (and what they lack) of row t, tokens 4 g + r of half h
    auto put = [&](char* to, int t, int h, const float* hi, const float* lo) {
      float x[4] = {hi[0], hi[1], hi[2], hi[3]};
      char* at = to + p_place(t, g) + 8 * h;
      uint2 p;
      p.x = part_of(x[0], x[1]); p.y = part_of(x[2], x[3]);
      *reinterpret_cast<uint2*>(at) = p;
      p.x = part_of(x[0], x[1]); p.y = part_of(x[2], x[3]);
      *reinterpret_cast<uint2*>(at + C * 64) = p;
      p.x = pack_bf16x2(x[0] + lo[0], x[1] + lo[1]); p.y = pack_bf16x2(x[2] + lo[2], x[3] + lo[3]);
      *reinterpret_cast<uint2*>(at + 2 * C * 64) = p;
    };
    auto finish = [&](int c) __attribute__((always_inline)) {
      const float* G = gates_of(c);
      char* P = sm + L::P + (c & 1) * L::PB;
      float bi[2][4], bf[2][4], wr[2][4], ei[2], ef[2];
      if constexpr (MODE != LIGHT) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const float4 x = ld4(G + BI + 16 * h + 4 * g), y = ld4(G + BF + 16 * h + 4 * g);
          bi[h][0] = x.x; bi[h][1] = x.y; bi[h][2] = x.z; bi[h][3] = x.w;
          bf[h][0] = y.x; bf[h][1] = y.y; bf[h][2] = y.z; bf[h][3] = y.w;
          if constexpr (MODE == SSM) {
            const float4 z = ld4(G + RC + 16 * h + 4 * g);
            wr[h][0] = z.x; wr[h][1] = z.y; wr[h][2] = z.z; wr[h][3] = z.w;
          }
          ei[h] = G[EI + 16 * h + n16];
          ef[h] = G[EF + 16 * h + n16];
        }
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int s = i == 2, t = i > 0;
        float hi[4], lo[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool in = i == 1 || 4 * g + r <= n16;
          float w;
          if constexpr (MODE == LIGHT) w = wl[i][r];
          else w = in ? power(ei[t] + bi[s][r], ef[t] + bf[s][r]) : 0.f;
          if constexpr (MODE == SSM) w *= wr[s][r];
          hi[r] = in ? qk[i][r] * w : 0.f;
          lo[r] = in ? fmaf(qk[i][r], w, -hi[r]) : 0.f;
          if constexpr (MODE == SSM) {
            if (i != 1) {
              const float add = 4 * g + r == n16 ? skip : 0.f, sum = hi[r] + add, b = sum - hi[r];
              lo[r] += (hi[r] - (sum - b)) + (add - b);
              hi[r] = sum;
            }
          }
        }
        put(P, 16 * t + n16, s, hi, lo);
      }
    };
    if constexpr (L::PRE) load_scores(0);
    __syncthreads();                                 // light: the powers are there
    if constexpr (MODE == LIGHT) {
      const float* pw = reinterpret_cast<const float*>(sm + L::POW);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int d = (i == 1 ? 16 : 0) + n16 - 4 * g - r;
          wl[i][r] = d >= 0 ? pw[d] : 0.f;
        }
    }
    for (int c = 0; c < chunks; ++c) {
      if constexpr (!L::PRE) products(c);
      finish(c);
      if constexpr (L::PRE) load_scores(c + 1);
      __syncthreads();
    }
    barriers(LEAD - 1);
    return;
  }

  if (wave == L::GATES) {
    // ============================================================================================== gates, 64 tokens (one per lane) in two steps
    double p1 = 0.;
    float p2 = 0.f, ga = 0.f, gb = 0.f;              // raw gates of the next 64 tokens
    int flag = 0;                                    // ssm: whether what was prepared of their chunk is not finite
    if constexpr (MODE == SSM) { p1 = -exp((double)a.par1[head]) * LOG2E; p2 = a.par2[head]; }
    const bool odd = MODE == SSM && !finite(a.par3[head]);
    const float base = MODE == LIGHT ? a.par1[head] : 0.f;
    const double qs2 = MODE == MLSTM ? -0.5 * log2((double)dk) : 0.;
    double m_run = 0.;
    if constexpr (MODE == MLSTM) {
      if (stored) m_run = a.mx[(size_t)slot * H + head];
    }
    auto load_gates = [&](int b) {
      const size_t t = row0 + min(b * 64 + lane, n - 1);
      if constexpr (MODE == MLSTM) {
        ga = ((const float*)a.aux1)[t * a.aux1_stride + head];
        gb = ((const float*)a.aux2)[t * a.aux2_stride + head];
      } else if constexpr (MODE == SSM) {
        const size_t at = t * a.aux1_stride + head;
        ga = a.aux_bf16 ? bf16_to_f32(((const uint16_t*)a.aux1)[at]) : ((const float*)a.aux1)[at];
        if constexpr (L::PRE) flag = *(const int*)((const char*)a.parts + ((size_t)(chunk0 + min(2 * b + (lane >> 5), chunks - 1)) * a.G + kvh) * parts_floats(DP) * 4 + 2 * L::ARRB + 3 * 1024);
      }
    };
    double ld = 0., lc = 0.;                         // log2 of the decay;  mlstm: forget and input gate, natural
    float decay = 0.f, write = 0.f;                  // the decay itself, where the chunk goes by token;  ssm: the write factor
    bool bad = false;
    auto first = [&](int b) {
      const bool ok = b * 64 + lane < n;
      bad = odd || flag != 0;
      if constexpr (MODE == SSM) {
        const double dt = softplus_d((double)ga + p2);
        ld = ok ? p1 * dt : 0.;
        write = ok ? (float)dt : 0.f;
        bad |= ok && !(fabs(ld) < 1e30 && dt < 1e30);
        decay = exp2f((float)ld);
        ld = fmin(fmax(ld, -20000.), 0.);            // 32 of them stay within the whole numbers' range
      } else if constexpr (MODE == MLSTM) {
        const float z = ok ? logsigmoid_f(a.cap * tanhf(gb / a.cap)) : 0.f, x = ok ? a.cap * tanhf(ga / a.cap) : -1e30f;
        ld = z;
        lc = x;
        bad |= ok && !(fabsf(z) < 1e30f && fabsf(x) < 1e30f);
      }
      load_gates(b + 1);
    };
    auto second = [&](int b) {
      const bool ok = b * 64 + lane < n;
      const int t = lane & 31, c = 2 * b + (lane >> 5);
      float* G = gates_of(c);
      const unsigned long long any = __ballot(bad);
      if (t == 0) G[BAD] = (MODE == MLSTM ? any : (lane ? any >> 32 : any & 0xffffffffull)) != 0 ? 1.f : 0.f;
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
      } else {
        double Z = ld;                               // sums within each chunk
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) {
          const double y = __shfl_up(Z, o, 32);
          if (t >= o) Z += y;
        }
        double E = Z, B = -Z, end = __shfl(Z, 31, 32), own = 0.;      // own: the chunk's starting maximum
        float mine = 0.f, before = 0.f;
        if constexpr (MODE == MLSTM) {
          // m_t = Z_t + max(m_0, max over s <= t of i_s - Z_s), in 64 bits: its rounding would be the state's, which the loop's is free of (a maximum
          // that only decays has a factor of exactly 1 there)
          double top = lc - Z;
#pragma unroll
          for (int o = 1; o < 32; o <<= 1) {
            const double y = __shfl_up(top, o, 32);
            if (t >= o) top = fmax(top, y);
          }
          const double mid = __shfl(Z, 31, 64) + fmax(m_run, __shfl(top, 31, 64));
          own = lane < 32 ? m_run : mid;
          top = fmax(own, top);
          E = -top * LOG2E;
          B = ok ? (lc - Z) * LOG2E : -1e5;
          double m = Z + top;
          end = __shfl(E, 31, 32);
          if (__builtin_expect(any != 0, 0)) {       // one after the other, as the loop does
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
        }
        float i, f;
        G[GA + t] = power_once(E + own + qs2);
        float rest = 0.f, F = power_once(end + B, MODE == MLSTM ? &rest : nullptr) * (MODE == SSM ? write : 1.f);
        F = ok ? F : 0.f;
        G[GF + t] = F;
        if constexpr (MODE == MLSTM) {
          rest = ok ? rest : 0.f;
          G[GL + t] = rest;
          // the normaliser's operand: as split2_of
          float most = F;
#pragma unroll
          for (int o = 16; o > 0; o >>= 1) most = fmaxf(most, __shfl_xor(most, o, 32));
          const float grid = grid_of(most), x0 = (F + grid) - grid;
          float x = (F - x0) + rest, none = 0.f;
          uint16_t* X = reinterpret_cast<uint16_t*>(sm + L::NX + (c & (L::GR - 1)) * 256) + 8 * ((t >> 2) & 3) + 4 * (t >> 4) + (t & 3);
          X[0] = (uint16_t)pack_bf16x2(x0, 0.f);
          X[32] = (uint16_t)part_of(x, none);
          X[64] = (uint16_t)part_of(x, none);
          X[96] = (uint16_t)pack_bf16x2(x, 0.f);
        }
        if (t == 31) G[ALL] = power_once(end + own);
        if constexpr (MODE == MLSTM) {
          G[RA + t] = ok ? expf((float)ld + before - mine) : 1.f;
          G[RC + t] = ok ? expf((float)lc - mine) : 0.f;
          G[GX + t] = expf(-mine);
        } else {
          G[RA + t] = decay;
          G[RC + t] = write;
        }
        whole_and_part(E + qs2, i, f);
        G[EI + t] = i;
        G[EF + t] = f;
        whole_and_part(B, i, f);
        G[BI + t] = i;
        G[BF + t] = f;
      }
    };
    if constexpr (MODE == LIGHT) {
      float* pw = reinterpret_cast<float*>(sm + L::POW);
      double p = 1.;
      for (int i = 0; i < 33; ++i) {
        if (lane == 0) pw[i] = (float)p;
        p *= (double)base;
      }
      __builtin_amdgcn_wave_barrier();
    }
    load_gates(0);
    first(0);
    second(0);
    for (int i = 0; i < chunks + LEAD; ++i) {        // chunks 2 b and 2 b + 1 are there before step 2 b
      const int b = (i >> 1) + 1;
      if (b * 64 < n) {
        if (i & 1) second(b);
        else first(b);
      }
      __syncthreads();
    }
    if constexpr (MODE == MLSTM) {
      if (zb == 0 && lane == 0) (a.mx_new ? a.mx_new[(size_t)seq * H + head] : a.mx[(size_t)slot * H + head]) = (float)m_run;
    }
    return;
  }

  // ================================================================================================== state, output and normaliser waves
  const bool outputs = wave >= L::OUT && wave < L::NORM, ones = MODE == MLSTM && wave == L::NORM;      // the normaliser's columns are all the same
  const int block = ones ? 0 : wave % L::NB;
  const int col = (zb * L::NB + block) * 16 + n16, colc = ones ? 0 : min(col, dv - 1);
  const bool cok = !ones && col < dv;
  if (!ones && (zb * L::NB + block) * 16 >= dv) {
    barriers(chunks + LEAD);
    return;
  }
  // token 16 h + 4 g + r is value 4 h + r
  auto tok = [&](int i) { return 16 * (i >> 2) + 4 * g + (i & 3); };
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
  auto take_v = [&](int c, float* u) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) u[i] = ldf<TI>(&rv[i]);        // rows past the portion: zeros (or, of rows that overlap, anything: nothing takes them)
    if constexpr (MODE == LIGHT) {
#pragma unroll
      for (int i = 0; i < 8; ++i) u[i] = silu(u[i]);
    }
    load_v(c + 1);
  };
  // one of eight values not a finite number (or too large for three parts)
  auto big = [](const float* x) {
    bool b = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) b |= !(fabsf(x[i]) < MOST);
    return b;
  };
  auto from_gates = [&](const float* G, float* f) {  // this lane's tokens' factors
    const float4 x = ld4(G + 4 * g), y = ld4(G + 16 + 4 * g);
    f[0] = x.x; f[1] = x.y; f[2] = x.z; f[3] = x.w; f[4] = y.x; f[5] = y.y; f[6] = y.z; f[7] = y.w;
  };
  float* yb = a.y + (size_t)row0 * H * dv + (size_t)head * dv;
  // tile i, register r of a state is channel 32 (i / 2) + 8 g + 4 (i % 2) + r, so tiles 2 b and 2 b + 1 are the operand of channels 32 b .. + 31
  auto chan = [](int g, int i, int r) { return 32 * (i >> 1) + 8 * g + 4 * (i & 1) + r; };
  char* const ST = sm + L::ST + block * L::SB + 16 * lane;

  // ssm: what was prepared, as operands: [block of channels][half][part], then [tile][part], 64 lanes each
  constexpr unsigned each = (unsigned)parts_floats(DP) * 4;
  const char* from_parts = (const char*)a.parts + (size_t)(chunk0 * a.G + kvh) * each;
  const size_t step = (size_t)a.G * each;
  auto parts_of = [&](int c) { return rows_at(from_parts + min(c, chunks - 1) * step, each); };
  float bad_next = 0.f, all_next = 1.f;              // of the gates (the state's: read before the barrier, after which LDS is busy)
  auto next_gates = [&](int c) {
    bad_next = gates_of(c)[BAD];
    all_next = gates_of(c)[ALL];
  };
  auto flagged = [&](int c) __attribute__((always_inline)) {
    int f = (outputs ? gates_of(c)[BAD] : bad_next) != 0.f;
    if (outputs) f |= reinterpret_cast<const int*>(sm + L::SBAD)[(c & 1) * L::NB + block];
    if constexpr (!L::PRE) {
      const int* F = reinterpret_cast<const int*>(sm + L::FLAG) + (c & 1) * L::NP;
#pragma unroll
      for (int i = 0; i < L::NP; ++i) f |= F[i];
    }
    return __builtin_amdgcn_readfirstlane(f) != 0;
  };

  // 1 / x, and what it lacks (0 of one that is not finite): an output is rounded once by its division
  auto put_quotient = [&](int c, int t, float x) {
    float* to = reinterpret_cast<float*>(sm + L::NRM) + (c & 3) * 64 + t;
    const float f = 1.f / x, rest = f * fmaf(-x, f, 1.f);
    to[0] = f;
    to[32] = finite(rest) ? rest : 0.f;
  };
  // A chunk with something that is not finite goes token by token, as the recurrence is written: parts of an infinity are no numbers, and a matrix
  // product multiplies a token's values by the zeros of those before it.  Each wave decides for itself: the state's for S, the outputs' (on
  // a copy of the state before the chunk) for their rows.
  auto by_token = [&](int c, f32x4 (&S)[NT], bool writes) __attribute__((always_inline)) {
    const float* G = gates_of(c);
    const int end = min(n - c * C, C);
    auto row_of = [&](const void* rows, int stride, int t) {        // channels past dk read zeros
      return rows_at((const TI*)rows + (size_t)(row0 + c * C + t) * stride + (size_t)kvh * dk, dk * (unsigned)sizeof(TI));
    };
    auto values = [&](Rows r, int i, float* f) __attribute__((always_inline)) {
      widen(row_load<Raw4<TI>>(r, chan(g, i, 0) * (unsigned)sizeof(TI), 0), f);
#pragma unroll
      for (int x = 0; x < 4; ++x) f[x] = MODE == LIGHT ? silu(f[x]) : f[x];
      __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll 1
    for (int t = 0; t < end; ++t) {
      float own = ones ? 1.f : ldf<TI>(vb + (size_t)(c * C + t) * a.v_stride + colc);
      if constexpr (MODE == LIGHT) own = silu(own);
      const float decay = G[RA + t], ut = own * G[RC + t];
      float o = 0.f;
      const Rows rk = row_of(a.k, a.k_stride, t), rq = row_of(a.q, a.q_stride, t);
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        float k[4], q[4];
        values(rk, i, k);
        values(rq, i, q);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          S[i][x] = fmaf(k[x], ut, S[i][x] * decay);
          o = fmaf(q[x], S[i][x], o);
        }
      }
      o += __shfl_xor(o, 16, 64);
      o += __shfl_xor(o, 32, 64);
      if constexpr (MODE == SSM) o += a.par3[head] * own;
      if constexpr (MODE == MLSTM) o *= qscale;
      if (ones) put_quotient(c, t, fmaxf(fabsf(o), G[GX + t]) + 1e-6f);
      else if (writes && g == 0 && cok) yb[(size_t)(c * C + t) * H * dv + colc] = o;      // mlstm: still to be divided
    }
  };

  // ---------------------------------------------------------------------------------------------- the state
  f32x4 S[NT];
  const size_t sbase = ((size_t)slot * H + head) * dk * dv, wbase = (((size_t)seq * gridDim.y + seg) * H + head) * dk * dv;
  const size_t nbase = ((size_t)slot * H + head) * dk;
  auto sat = [&](int ch) { return ones ? (size_t)ch : MODE == SSM ? (size_t)colc * dk + ch : (size_t)ch * dv + colc; };
  auto begin = [&]() __attribute__((always_inline)) {
    const float* from = ones ? a.norm + nbase : MODE == SSM && a.pass ? a.ws + wbase : a.state + sbase;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = (stored && chan(g, i, r) < dk && (cok || ones)) ? from[sat(chan(g, i, r))] : 0.f;
  };
  auto keep_state = [&]() __attribute__((always_inline)) {
    // addresses are made anew: those of the loads would be kept all the way
    int ge = g;
    asm volatile("" : "+v"(ge));
    float* to = ones ? (a.norm_new ? a.norm_new + ((size_t)seq * H + head) * dk : a.norm + nbase) : MODE == SSM && a.pass == 1 ? a.ws + wbase : a.state + sbase;
    const bool keep = ones ? zb == 0 && n16 == 0 : cok && (a.pass != 2 || last);
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ch = chan(ge, i, r);
        if (keep && ch < dk) to[sat(ch)] = S[i][r];
      }
  };
  auto to_lds = [&](int c) {                         // the state before chunk c
#pragma unroll
    for (int i = 0; i < NT; ++i) *reinterpret_cast<f32x4*>(ST + (c & 1) * L::NB * L::SB + 1024 * i) = S[i];
  };
  // N tiles of k, channels by tokens.  ssm: all tiles are kept, the next chunk's under way as soon as this one's are used
  constexpr int N = 2, KEPT = L::PRE ? NT / N : 2;
  u32x4 kf[KEPT][N][PQ];
  auto read_k = [&](int c, int j, u32x4 (&kf)[N][PQ]) __attribute__((always_inline)) {
    if constexpr (L::PRE) {
      const Rows p = parts_of(c);
#pragma unroll
      for (int y = 0; y < N; ++y)
#pragma unroll
        for (int x = 0; x < PQ; ++x) kf[y][x] = row_load<u32x4>(p, 16 * lane, L::ARRB + ((j + y) * PQ + x) * 1024);
    } else {
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
    }
  };
  // Parts of x = F u of the next chunk.  A bf16 product cuts off what lies 24 bits below the largest term of eight, which of a state that consists of its
  // last few tokens (mlstm's, whose decays are fast) would be twice a rounding.  So there the first parts of a column are multiples of one
  // 2^-7 of the largest: their products' sum is exact, the others' is 2^-8 smaller (state 5.3e-8 from 64 bits without, the token loop's 4.4e-8).
  constexpr bool GRID = MODE == MLSTM;
  constexpr int XP = GRID ? 4 : 3;
  u32x4 xp[XP];
  float xu[8], xf[8], xl[8], grid = 0.f;
  // true: one is not a finite number, or too large for its parts (a factor may be 0: it shows in the product all the same)
  auto begin_x = [&](int c) __attribute__((always_inline)) {
    take_v(c, xu);
    from_gates(gates_of(c) + GF, xf);
    if constexpr (GRID) from_gates(gates_of(c) + GL, xl);
    float x[8], most = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = xu[i] * xf[i];
    if constexpr (GRID) {
#pragma unroll
      for (int i = 0; i < 8; i += 2) most = larger3(most, x[i], x[i + 1]);
      most = fmaxf(most, __shfl_xor(most, 16, 64));
      most = fmaxf(most, __shfl_xor(most, 32, 64));
      grid = grid_of(most);
    }
    bool odd = false;
#pragma unroll
    for (int i = 0; i < 8; ++i) odd |= !(fabsf(x[i]) < (GRID ? 1e30f : MOST));
    return odd;
  };
  auto make_x = [&](int c) __attribute__((always_inline)) {
    const bool odd = begin_x(c);
#pragma unroll
    for (int i = 0; i < 4; ++i) split2_of<GRID>(xu, xf, xl, grid, i, xp);
    return odd;
  };
  auto state_big = [&]() {
    float most = 0.f;
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      most = larger3(most, S[i][0], S[i][1]);
      most = larger3(most, S[i][2], S[i][3]);
    }
    return !(most < MOST);
  };
  // S <- A S + k^T x, and x of the next chunk beside the products
  auto read_x = [&](int c) __attribute__((always_inline)) {      // the normaliser's
#pragma unroll
    for (int i = 0; i < XP; ++i) xp[i] = *reinterpret_cast<const u32x4*>(sm + L::NX + (c & (L::GR - 1)) * 256 + 64 * i + 16 * g);
  };
  auto update = [&](int c, auto one) __attribute__((always_inline)) {
    const float at = all_next;
    u32x4 xs[XP];
#pragma unroll
    for (int i = 0; i < XP; ++i) xs[i] = xp[i];
    bool odd = false;
    if constexpr (one.value) read_x(c + 1);
    else odd = begin_x(c + 1);
#pragma unroll
    for (int j = 0; j < NT; j += N) {
      __builtin_amdgcn_sched_barrier(0);
      u32x4(&kj)[N][PQ] = kf[j / N % KEPT];
      if (!L::PRE && j + N < NT) read_k(c, j + N, kf[(j / N + 1) % KEPT]);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!one.value && i * (NT / N) / 4 == j / N) split2_of<GRID>(xu, xf, xl, grid, i, xp);
      f32x4 lo[N], hi[N];
#pragma unroll
      for (int y = 0; y < N; ++y) lo[y] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = XP - 1; t > 0; --t)
#pragma unroll
        for (int p = t; p >= 0; --p)
          if (p < PQ) {
#pragma unroll
            for (int y = 0; y < N; ++y) lo[y] = mfma(kj[y][p], xs[t - p], lo[y]);
          }
#pragma unroll
      for (int y = 0; y < N; ++y) hi[y] = mfma(kj[y][0], xs[0], GRID ? f32x4{0.f, 0.f, 0.f, 0.f} : lo[y]);
      if constexpr (L::PRE) read_k(c + 1, j, kj);
#pragma unroll
      for (int y = 0; y < N; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[j + y][r] = GRID ? hi[y][r] + fmaf(at, S[j + y][r], lo[y][r]) : fmaf(at, S[j + y][r], hi[y][r]);
      if (!L::PRE && j + N < NT) __builtin_amdgcn_sched_group_barrier(0x100, N * PQ * 2, 0);
      constexpr int M = N * (GRID ? (PQ == 1 ? 4 : 9) : PQ == 1 ? 3 : 6);
#pragma unroll
      for (int i = 0; i < M; ++i) {                  // a product and some of the next parts in turn
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 4, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    return odd;
  };

  // ---------------------------------------------------------------------------------------------- read-outs
  f32x4 qS[2];                                      // S^T q of the chunk to be finished, tokens as tok()
  u32x4 up[PU];                                      // parts of its u
  bool was_cold = false;                             // or its outputs are there already
  f32x4 T[NT];                                       // the state, from LDS
  constexpr int QK = L::PRE ? NK : 2;
  u32x4 qf[QK][2][PQ];                              // rows of q: as those of k
  auto read_q = [&](int c, int b, u32x4 (&x)[2][PQ]) __attribute__((always_inline)) {
    if constexpr (L::PRE) {
      const Rows p = parts_of(c);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int y = 0; y < PQ; ++y) x[h][y] = row_load<u32x4>(p, 16 * lane, ((2 * b + h) * PQ + y) * 1024);
    } else {
      const char* Q = sm + L::Q + (c & 1) * L::ARRB;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int p = 0; p < PQ; ++p) x[h][p] = *reinterpret_cast<const u32x4*>(Q + p * L::PARTB + place(16 * h + n16, 4 * b + g));
    }
  };
  auto read_ahead = [&](int c) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NT; ++i) {
      T[i] = *reinterpret_cast<const f32x4*>(ST + (c & 1) * L::NB * L::SB + 1024 * i);
    }
    if constexpr (!L::PRE) read_q(c, 0, qf[0]);
  };
  auto read_out = [&](int c, const f32x4 (&X)[NT], auto one) __attribute__((always_inline)) {      // true: one of u is not a finite number
    f32x4 hi[2], lo[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) hi[h] = lo[h] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 sp[2][1][3];
    auto split = [&](int b) __attribute__((always_inline)) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = X[2 * b + (i >> 2)][i & 3];
      split8<3>(v, sp[b & 1][0]);
    };
    split(0);
    bool odd = false;
#pragma unroll
    for (int b = 0; b < NK; ++b) {
      __builtin_amdgcn_sched_barrier(0);
      if (b + 1 < NK) {
        if constexpr (!L::PRE) read_q(c, b + 1, qf[(b + 1) % QK]);
        split(b + 1);
      } else if constexpr (one.value) {
        up[0] = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};      // P of rows past the portion is 0
#pragma unroll
        for (int i = 1; i < PU; ++i) up[i] = u32x4{0, 0, 0, 0};
      } else {
        float u[8];
        take_v(c, u);
        odd = big(u);
        split8<PU>(u, up);
      }
      // the last block's first parts start from the small ones' sum: one rounding less at the sum's size
      small<PQ, 3, 2, 1>(qf[b % QK], sp[b & 1], lo);
#pragma unroll
      for (int h = 0; h < 2; ++h) (b + 1 < NK ? hi : lo)[h] = mfma(qf[b % QK][h][0], sp[b & 1][0][0], (b + 1 < NK ? hi : lo)[h]);
      if constexpr (L::PRE) read_q(c + 1, b, qf[b % QK]);
      if (!L::PRE) __builtin_amdgcn_sched_group_barrier(0x100, 2 * PQ, 0);      // reads, then a product and some of the next parts in turn
      constexpr int M = 2 * (PQ == 1 ? 3 : 6);
#pragma unroll
      for (int i = 0; i < M; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, (48 + M - 1) / M, 0);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) qS[h] = hi[h] + lo[h];
    return odd;
  };
  float out[8];
  u32x4 pf[2][3];
  float fA[8];
  auto read_p = [&](int c) __attribute__((always_inline)) {
    const char* P = sm + L::P + (c & 1) * L::PB;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float4 x = ld4(gates_of(c) + GA + 16 * h + 4 * g);
      fA[4 * h] = x.x; fA[4 * h + 1] = x.y; fA[4 * h + 2] = x.z; fA[4 * h + 3] = x.w;
#pragma unroll
      for (int p = 0; p < 3; ++p) pf[h][p] = *reinterpret_cast<const u32x4*>(P + p * C * 64 + p_place(16 * h + n16, g));
    }
  };
  // P u and what the state gave
  auto finish = [&]() __attribute__((always_inline)) {
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
    for (int i = 0; i < 8; ++i) out[i] = fmaf(fA[i], qS[i >> 2][i & 3], hi[i >> 2][i & 3]);
  };

  // In all loops: what goes by token is outside the inner loop, so that its registers are not that one's.
  if constexpr (MODE == MLSTM) {
    if (ones) {
      begin();
      __syncthreads();
      auto done = [&](int c) __attribute__((always_inline)) {
        finish();
        float o = out[0];                            // lane n16's token
#pragma unroll
        for (int i = 1; i < 8; ++i) {
          float x = out[i];
          asm("" : "+v"(x));                         // values, not a place in memory, are chosen from
          o = (n16 & 7) == i ? x : o;
        }
        const int t = tok(n16 & 7);
        o = fmaxf(fabsf(o), gates_of(c)[GX + t]) + 1e-6f;
        if (n16 < 8 && !was_cold && c >= 0) put_quotient(c, t, o);
      };
      read_x(0);
      next_gates(0);
      bool odd = state_big();
      for (int c = 0; c < chunks; ++c) {
        bool warm = true;
        for (; c < chunks; ++c) {
          read_p(c - 1);
          read_q(c, 0, qf[0]);
          done(c - 1);
          was_cold = flagged(c) || __any(odd);
          warm = !was_cold;
          if (__builtin_expect(!warm, 0)) break;
          read_out(c, S, std::true_type{});
          read_k(c, 0, kf[0]);
          update(c, std::true_type{});
          odd = state_big();
          next_gates(c + 1);
          __syncthreads();
        }
        if (warm) break;
        by_token(c, S, true);
        read_x(c + 1);
        odd = state_big();
        next_gates(c + 1);
        __syncthreads();
      }
      read_p(chunks - 1);
      done(chunks - 1);
      barriers(LEAD - 1);
      keep_state();
      return;
    }
  }

  // The loads before the loops come in the loops' order, in which what is waited for is counted.
  if (!outputs) {
    load_v(0);
    begin();
    to_lds(0);
    auto state_flag = [&](int c) {
      const bool b = __any(state_big());
      if (lane == 0) reinterpret_cast<int*>(sm + L::SBAD)[(c & 1) * L::NB + block] = b;
      return b;
    };
    bool odd = state_flag(0);
    __syncthreads();
    odd |= make_x(0);
    if constexpr (L::PRE) {
#pragma unroll
      for (int j = 0; j < NT; j += N) read_k(0, j, kf[j / N]);
    }
    next_gates(0);
    float all = 1.f;                                 // ssm, pass 1: decay of the segment
    for (int c = 0; c < chunks; ++c) {
      bool warm = true;
      for (; c < chunks; ++c) {
        if constexpr (!L::PRE) read_k(c, 0, kf[0]);
        if constexpr (MODE == SSM) all *= all_next;
        warm = !(flagged(c) || __any(odd));
        if (__builtin_expect(!warm, 0)) break;
        odd = update(c, std::false_type{});
        to_lds(c + 1);
        odd |= state_flag(c + 1);
        next_gates(c + 1);
        __syncthreads();
      }
      if (warm) break;
      by_token(c, S, false);
      to_lds(c + 1);
      odd = state_flag(c + 1);
      odd |= make_x(c + 1);
      next_gates(c + 1);
      if constexpr (L::PRE) {
#pragma unroll
        for (int j = 0; j < NT; j += N) read_k(c + 1, j, kf[j / N]);
      }
      __syncthreads();
    }
    barriers(LEAD - 1);
    keep_state();
    if (MODE == SSM && a.pass == 1 && zb == 0 && wave == 0 && lane == 0) a.wsd[((size_t)seq * gridDim.y + seg) * H + head] = all;
    return;
  }

  if (MODE == SSM && a.pass == 1) {
    barriers(chunks + LEAD);
    return;
  }
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
  bool cold_out = false;
  auto done = [&](int c) __attribute__((always_inline)) {      // chunk c is finished in step c + 2
    cold_out = was_cold;
    finish();
    if constexpr (MODE != MLSTM) store(c, out, c >= 0 && !was_cold);
  };
  auto divide = [&](int c) __attribute__((always_inline)) {    // and divided by the normaliser in step c + 3
    if constexpr (MODE == MLSTM) {
      float f[8], rest[8], o[8];
      from_gates(reinterpret_cast<const float*>(sm + L::NRM) + (c & 3) * 64, f);
      from_gates(reinterpret_cast<const float*>(sm + L::NRM) + (c & 3) * 64 + 32, rest);
      if (__builtin_expect(cold_out && c >= 0, 0)) {
#pragma unroll
        for (int i = 0; i < 8; ++i) out[i] = yb[(size_t)min(c * C + tok(i), n - 1) * H * dv + colc];
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) o[i] = fmaf(out[i], f[i], __builtin_amdgcn_fmed3f(out[i], -MOST, MOST) * rest[i]);      // an infinite one stays one
      store(c, o, c >= 0);
    }
  };
  if constexpr (L::PRE) {
#pragma unroll
    for (int b = 0; b + 1 < NK; ++b) read_q(0, b, qf[b]);
    load_v(0);
    read_q(0, NK - 1, qf[NK - 1]);
  } else {
    load_v(0);
  }
  __syncthreads();
  for (int c = 0; c < chunks; ++c) {
    bool warm = true;
    for (; c < chunks; ++c) {
      read_p(c - 1);
      read_ahead(c);
      const bool bad = flagged(c);
      divide(c - 2);
      done(c - 1);
      const bool odd = read_out(c, T, std::false_type{});      // in any case: it loads for the next
      was_cold = bad || __any(odd);
      warm = !was_cold;
      if (__builtin_expect(!warm, 0)) break;
      __syncthreads();
    }
    if (warm) break;
    by_token(c, T, true);
    __syncthreads();
  }
  divide(chunks - 2);
  read_p(chunks - 1);
  done(chunks - 1);
  __syncthreads();
  if constexpr (MODE == MLSTM) {
    divide(chunks - 1);
    __syncthreads();
  }
}

// What the heads of a state-space group and their columns share, for every chunk: the parts of C and B as the waves' operands, the scores as the scores
// wave holds them, whether something is not finite.  A workgroup owns (chunk, group).
__global__ __launch_bounds__(256) void ssm_parts_kernel(const ChunkArgs a) {
  constexpr int NK = 4;
  using L = Lay<SSM, float, NK, true>;
  constexpr int DP = L::DP, PER = DP / 8, TASKS = 2 * C * PER / 256;
  extern __shared__ __attribute__((aligned(16))) char sm[];
  __shared__ int any_bad;
  const int grp = blockIdx.x;
  // the sequence whose chunk this is: its chunks start at first_chunk
  int lo = 0, hi = a.n_seq - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (first_chunk(a.seq_row0[mid], mid) <= (int)blockIdx.y) lo = mid;
    else hi = mid - 1;
  }
  const int row0 = a.seq_row0[lo], n = a.seq_row0[lo + 1] - row0, first = ((int)blockIdx.y - first_chunk(row0, lo)) * C;
  if (n <= a.skip_rows || first >= n) return;
  const int left = n - first;
  const float* qb = (const float*)a.q + (size_t)(row0 + first) * a.q_stride + (size_t)grp * a.dk;
  const float* kb = (const float*)a.k + (size_t)(row0 + first) * a.k_stride + (size_t)grp * a.dk;
  char* to = (char*)a.parts + ((size_t)blockIdx.y * a.G + grp) * parts_floats(DP) * 4;
  if (threadIdx.x == 0) any_bad = 0;
  f32x4 raw[TASKS][2];
  const int piece = threadIdx.x % PER;
  const int c0 = min(8 * piece, a.dk - 4), c1 = min(8 * piece + 4, a.dk - 4);
#pragma unroll
  for (int j = 0; j < TASKS; ++j) {
    const bool is_q = j < TASKS / 2;
    const int row = min((j % (TASKS / 2)) * (256 / PER) + (int)threadIdx.x / PER, left - 1);
    const float* p = is_q ? qb + (size_t)row * a.q_stride : kb + (size_t)row * a.k_stride;
    raw[j][0] = *reinterpret_cast<const f32x4*>(p + c0);
    raw[j][1] = *reinterpret_cast<const f32x4*>(p + c1);
  }
  __syncthreads();
  float most = 0.f;
  auto place = [&](int row, int ch16) { return row * L::ROWB + ((ch16 ^ (row & 7)) << 4); };
#pragma unroll
  for (int j = 0; j < TASKS; ++j) {
    const int row = (j % (TASKS / 2)) * (256 / PER) + threadIdx.x / PER;
    float x[8];
    widen(raw[j][0], x);
    widen(raw[j][1], x + 4);
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = row < left && 8 * piece + i < a.dk ? x[i] : 0.f;
#pragma unroll
    for (int i = 0; i < 8; i += 2) most = larger3(most, x[i], x[i + 1]);
    u32x4 p[3];
    split8<3>(x, p);
    char* at = sm + (j < TASKS / 2 ? 0 : L::ARRB) + place(row, piece);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(at + i * L::PARTB) = p[i];
  }
  if (__any(!(most < MOST)) && (threadIdx.x & 63) == 0) any_bad = 1;
  __syncthreads();
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
  if (threadIdx.x == 0) *reinterpret_cast<int*>(to + 2 * L::ARRB + 3 * 1024) = any_bad;
  // operands: q's rows, k's channels by tokens
  constexpr int FRAGS = 2 * NK * 3 / 4;
#pragma unroll
  for (int j = 0; j < FRAGS; ++j) {
    const int f = wave * FRAGS + j, p = f % 3, i = f / 3;      // q: block i / 2, half i % 2;  k: tile i
    *reinterpret_cast<u32x4*>(to + f * 1024 + 16 * lane) = *reinterpret_cast<const u32x4*>(sm + p * L::PARTB + place(16 * (i & 1) + n16, 4 * (i >> 1) + g));
    u32x4 kf;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const short4v v = read_tr(sm + L::ARRB + p * L::PARTB + place(16 * h + 4 * g + (n16 >> 2), 4 * (i >> 1) + (n16 & 3)) + 8 * (i & 1));
      kf[2 * h] = (uint32_t)(uint16_t)v[0] | ((uint32_t)(uint16_t)v[1] << 16);
      kf[2 * h + 1] = (uint32_t)(uint16_t)v[2] | ((uint32_t)(uint16_t)v[3] << 16);
    }
    *reinterpret_cast<u32x4*>(to + L::ARRB + f * 1024 + 16 * lane) = kf;
  }
  if (wave == 3) return;
  const int s = wave == 2, t = wave > 0;
  f32x4 h1[1] = {{0.f, 0.f, 0.f, 0.f}}, m1 = h1[0], l1[1] = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int b = 0; b < NK; ++b) {
    u32x4 kf[1][3], qf[1][3];
#pragma unroll
    for (int p = 0; p < 3; ++p) {
      kf[0][p] = *reinterpret_cast<const u32x4*>(sm + L::ARRB + p * L::PARTB + place(16 * s + n16, 4 * b + g));
      qf[0][p] = *reinterpret_cast<const u32x4*>(sm + p * L::PARTB + place(16 * t + n16, 4 * b + g));
    }
    small<3, 3, 1, 1>(kf, qf, l1);                     // as the scores wave's sums
    f32x4& sum = b == 2 ? m1 : b + 1 < NK ? h1[0] : l1[0];
    sum = mfma(kf[0][0], qf[0][0], sum);
  }
  *reinterpret_cast<f32x4*>(to + 2 * L::ARRB + 1024 * wave + 16 * lane) = h1[0] + (m1 + l1[0]);
}

}  // namespace

template <int MODE, typename TI, int NK, bool PRE = false>
static int launch(const ChunkArgs& a, dim3 grid, hipStream_t st) {
  constexpr int lds = Lay<MODE, TI, NK, PRE>::END;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = chunk_parts_kernel<MODE, TI, NK, PRE>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return (int)e;
  }
  kernel<<<grid, 64 * Lay<MODE, TI, NK, PRE>::WAVES, lds, st>>>(a);
  return 0;
}

static int launch_ssm(const ChunkArgs& a, dim3 grid, hipStream_t st) {
  if (a.dk <= 64) return launch<SSM, float, 2>(a, grid, st);
  if (!a.parts) return launch<SSM, float, 4>(a, grid, st);
  if (a.pass != 2) {
    constexpr int lds = 2 * Lay<SSM, float, 4, true>::ARRB;
    ssm_parts_kernel<<<dim3(a.G, a.parts_chunks), 256, lds, st>>>(a);
  }
  return launch<SSM, float, 4, true>(a, grid, st);
}

template <int MODE>
static int launch_mode(const ChunkArgs& a, int in_f32, dim3 grid, hipStream_t st) {
  if (in_f32) {
    if (a.dk <= 64) return launch<MODE, float, 2>(a, grid, st);
    if constexpr (MODE == MLSTM) return -3;
    else return launch<MODE, float, 4>(a, grid, st);
  }
  return a.dk <= 64 ? launch<MODE, uint16_t, 2>(a, grid, st) : launch<MODE, uint16_t, 4>(a, grid, st);
}

// Floats of workspace of a state-space step whose parts and scores are made in a pass before (0: there is none), for T rows of n_seq sequences: steps of
// 65 to 128 channels that are long, or may have a portion of 1500 rows (512 beside many decode rows).  The pass costs 3 us and its operands come from the L2s; without it every
// workgroup makes them, on waves of their own.  us without and with, 128 channels (16, 64 heads): 4 x 256 rows 49, 54 and 48, 52; 4 x 400 61, 69 and 57, 69;
// 8 x 192 24, 45 and 28, 47 (16, 32 heads); 600 beside 16 53, 67 and 50, 62; 2000 142, 144 and 120, 122 (16 heads beside 7 rows; 64 heads alone); 8 x 1000 of 64 heads 317 and 303.  Of 64 channels:
// 8 x 80 rows, 16 heads 12 and 16; 4 x 1000, 32 heads 49 and 57; 2000, 64 heads 87 and 93; 4 x 2000, 16 heads 142 and 134.
extern "C" long long dgi_ssm_parts_floats(int dk, int H, int G, int T, int n_seq, int* chunks) {
  *chunks = T / C + n_seq;
  if (dk <= 64 || !dgi_chunk_parts_takes(SSM, dk, H, G, 1) || !(T >= 320l * n_seq || T - n_seq >= 1536 || (T - n_seq >= 512 && T <= 48l * n_seq))) return 0;
  const long long floats = (long long)*chunks * G * parts_floats(128);
  return *chunks > 65535 || floats > 1ll << 28 ? 0 : floats;
}

bool dgi_chunk_parts_takes(int mode, int dk, int H, int G, int in_f32) {
  return mode == SSM ? dk <= 128 && H >= 4 * G : mode == LIGHT ? dk <= 128 : mode == MLSTM && dk <= (in_f32 ? 64 : 128);
}

// one launch of chunk_scan.hip's dgi_chunk_scan; grid: n_seq * H * (blocks of 32 value columns), segments
int dgi_chunk_parts(const ChunkArgs& a, int mode, int in_f32, dim3 grid, hipStream_t st) {
  switch (mode) {
    case MLSTM: return launch_mode<MLSTM>(a, in_f32, grid, st);
    case LIGHT: return launch_mode<LIGHT>(a, in_f32, grid, st);
    case SSM: return launch_ssm(a, grid, st);
  }
  return -2;
}
