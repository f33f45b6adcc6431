// dgi/csrc/mix/chunk_scan.hip — prompt portions of the recurrences that carry a matrix S [dk, dv] per head (linear_scan.hip has
// their definitions, ssm_scan.hip that of ssm), sixteen tokens at a time in fp32 matrix products (v_mfma_f32_16x16x4_f32).  Those that chunk_parts.hip
// takes (light; mlstm, but for fp32 rows of more than 64 channels; ssm of groups of four heads) go there, long portions of delta to chunk_delta.hip, steps of gla,
// light and mlstm that dgi_chunk_segments_plan says to chunk_segments.h.
//
// For tokens t, s of a chunk that starts from the state S, with D[t, s] the product of the decays of the tokens after s up to t
// and A_t that of all tokens up to t:
//
//     o_t = A_t S^T q_t + sum_(s <= t) P[t, s] u_s,   P[t, s] = D[t, s] (q_t . k_s) c_s          S <- A_15 S + sum_s D[15, s] c_s k_s u_s^T
//
// ssm: q = C, k = B, u = x, c = dt;  mlstm: c = the input gate, o divided by the normaliser;
// wkv: the decays are per key channel, so they sit inside the products: q_t and k_s are scaled by the decays between them and
// the middle of the chunk (so chunk halves, not chunks, have to stay in the fp32 range), the state products use prefix and suffix
// products and no division;  it reads before it writes: s < t, and the bonus on the diagonal;
// delta: u solves (I + T) u = beta (v - A S^T k), T[t, s] = beta_t D[t, s] (k_t . k_s) below the diagonal: block forward
// substitution with blocks of four tokens, each block one matrix product with M_b = [inverse of its diagonal block - I;
// - T below it times that inverse].  (gla: chunk_segments.h, chunk_scan_decay.hip.)
//
// A workgroup owns (sequence, head, NC blocks of 16 value columns: two, or four, see four_blocks) and is a pipeline of waves that hand chunks on through LDS, one
// barrier per chunk:
//   preparing waves  load q / k (and the channel decays) two chunks ahead in registers and write them (scaled) to LDS;
//   gates wave       gates of 64 tokens at a time (in four steps, so that none is long), D and A of each chunk;
//   scores waves     two that take turns: q . k, P and (delta) M;
//   state waves      one per column block: the state rows of all key channels of its 16 columns stay in registers, in the layout the
//                    products leave them (the key index inside a product is permuted so that the registers are its operand as
//                    they are; delta permutes the tokens the same way, so u is an operand as it is), so no wave waits for
//                    another's partial sums; the state before the chunk goes to LDS;  a normaliser wave beside them (mlstm);
//   output waves     one per column block: read-out of that state, P u, the store.
// So a chunk's products (per column block 2 dk / 4 + 4 of 32 cycles each, delta 3 dk / 4 + 8, beside dk / 4 or dk / 2 for the scores)
// spread over the compute unit's four matrix cores; what bounds a chunk is the longest role's chain: the state wave's (delta: read-out
// by k, substitution, update) or a preparing wave's arithmetic (wkv): a wave issues an instruction every four to five cycles at best, so
// addresses are lane offsets kept in registers, and rows past the end a branch of their own.  Measured, a step of 2 prompts of 4096 rows in
// all, 64 heads, states 64 x 64 (ssm 128 x 64), against the same token by token on the vector ALUs (linear_scan.hip, ssm_scan.hip):
// delta 178 us (726), ssm 199 (637; 210 with flat loads), wkv 232 (some 630).
//
// Precision: results and states are no further from 64 bits than the token loop's (2-norm over 1300 to 4096 rows: ssm 7.8e-8, the loop 8.0e-8;
// delta 1.17e-7, 1.18e-7; wkv 9.8e-8, 1.01e-7; but states of wkv on bf16 rows 7.34e-8, 7.28e-8: the loop's products of bf16 keys and values
// are exact, here a decayed key is rounded).  Regrouping alone does not do that: with the sums over channels in two running sums, P and the decays
// rounded product by product and P u in 32 bits the same were 1.25e-7, 1.57e-7 and 1.30e-7.  So sums over channels are added as trees, a sum over
// tokens starts with the oldest, the per-token decays and wkv's suffix products carry their rounding errors along, and P and P u are 64-bit
// (four v_mfma_f64_16x16x4_f64 per chunk and output wave).  It costs 3 % of delta's time; wkv's was not the longest role.
//
// Half-chunk products of channel decays below 1e-28, or q and k so large or small that their scaled values leave the fp32 range: the wave that
// prepares such channels sums their scores token by token instead.  An infinity or NaN among a chunk's u takes a path that keeps it from the tokens
// before it (a matrix product multiplies it by their zeros).  A portion at position 0 reads no state.
#include <type_traits>
#include "chunk_args.h"

using namespace dgi;

namespace {

constexpr int C = 16;              // tokens per chunk
constexpr int TR = 20, PR = 18;    // padded rows of sixteen tokens; in 64 bits
constexpr float SAFE = 1e-28f;
typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float softplus_f(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

// e^x to about an ulp: 2^(x log2 e) with the product in two parts.  x within [-200, 6], where e^-e^x covers every fp32 value below 1.
__device__ __forceinline__ float exp_2part(float x) {
  const float h = x * 1.44269502f, l = fmaf(x, 1.44269502f, -h) + x * 1.92596299e-8f;
  const float e = __builtin_amdgcn_exp2f(h);
  return fmaf(e, l * 0.693147181f, e);
}
__device__ __forceinline__ float exp_neg_exp(float x) {
  const float r = exp_2part(-exp_2part(fminf(fmaxf(x, -200.f), 5.f)));
  return x == x ? r : x;
}

// Sums of sixteen values over the 64 lanes: lane l gets the total of v[l & 15].  Each step halves the values a lane keeps.
__device__ __forceinline__ float sum16(const float* v, int lane) {
  const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4, b3 = lane & 8;
  float w[8], x[4], z[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) w[i] = (b0 ? v[2 * i + 1] : v[2 * i]) + dpp_move<0xB1>(b0 ? v[2 * i] : v[2 * i + 1]);
#pragma unroll
  for (int i = 0; i < 4; ++i) x[i] = (b1 ? w[2 * i + 1] : w[2 * i]) + dpp_move<0x4E>(b1 ? w[2 * i] : w[2 * i + 1]);
#pragma unroll
  for (int i = 0; i < 2; ++i) z[i] = (b2 ? x[2 * i + 1] : x[2 * i]) + __shfl_xor(b2 ? x[2 * i] : x[2 * i + 1], 4, 64);
  float r = (b3 ? z[1] : z[0]) + dpp_move<0x128>(b3 ? z[0] : z[1]);
  r += __shfl_xor(r, 16, 64);
  return r + __shfl_xor(r, 32, 64);
}

// LDS (floats) and roles of a workgroup.  NT: 16-channel tiles (dk <= 16 NT).  A chunk's steps, in order: q / k written, scores (two
// steps; one for NT 16, whose buffers must be fewer), state, output: an array read d steps after it is written has d + 1 buffers.
template <int MODE, int NT, int COLS>
struct Lay {
  static constexpr bool CH = MODE == WKV;                      // decays per key channel
  static constexpr bool TURNS = CH;                            // two sets of preparing waves take turns, two steps a chunk
  static constexpr int NC = COLS / 16, W2 = NT <= 8 ? 2 : 1;         // column blocks, scores waves
  static constexpr int NS = NT / 4;                            // preparing waves of 64 channels
  static constexpr int NA = NT == 4 ? 4 : 8;                   // sums side by side of a sum over the channels: state waves
  static constexpr int NO = MODE == WKV || (MODE == DELTA && NT == 8) ? 8 : 4;      // output waves (delta, 128 channels: with 4 results were 2 % further off than the loop's)
  // Waves: state, output, then gates and normaliser (or preparing waves), scores, (more) preparing waves: waves four apart share a SIMD,
  // and the scores' products are best beside the output waves', the fewest.
  static constexpr int SETS = CH && NT == 4 ? 2 : 1;           // channel decays: one set of preparing waves for the scores, one for the state
  static constexpr int PREPS = (TURNS ? 2 : 1) * NS * SETS;    // preparing waves, EARLY of them before the scores waves
  static constexpr int EARLY = NC == 1 ? 0 : (CH ? 2 : (MODE == MLSTM ? 0 : 1));
  static constexpr int OUT = NC, GATES = 2 * NC, NORM = GATES + 1, SCORES = NC == 1 ? 3 : 2 * NC + 2, PREP = SCORES + W2;
  static constexpr int WAVES = PREP + PREPS - EARLY;
  // every wave has one role: a wave left over would run as an output wave of columns that are another workgroup's
  static_assert(SCORES - EARLY == (CH ? GATES : MODE == MLSTM ? NORM + 1 : GATES + 1), "state, output, gates, normaliser, preparing, scores");
  static constexpr int LEAD = 2 + W2 + (TURNS ? 1 : 0);        // steps before the first output
  static constexpr int DP = 16 * NT, QR = DP + 4, ROWS = C * QR;
  static constexpr int QB = 3 + W2, KB = 2 + W2;               // buffers of q and k
  static constexpr int Q = 0;                                  // [QB][16][QR] q (channel decays: times the prefix products)
  static constexpr int K = Q + QB * ROWS;                      // [KB][16][QR] k, rows by place (read by its tokens: no bank twice); channel decays: [2][16][QR] scaled for the scores
  static constexpr int QT = K + (CH ? 2 : KB) * ROWS;          // CH: [2][16][QR] q scaled for the scores
  static constexpr int KT = QT + (CH ? 2 * ROWS : 0);          // CH: [KB][DP][TR] k times the suffix products, by channel
  static constexpr int DEC = KT + (CH ? KB * DP * TR : 0);     // CH: [KB][DP] decay of the whole chunk
  static constexpr int ST = DEC + (CH ? KB * DP : 0);          // [2][NC][NT][64][4] state before the chunk, as the state wave holds it
  static constexpr int U = ST + 2 * NC * DP * 16;              // DELTA: [2][NC][64][4] u
  static constexpr int P = U + (MODE == DELTA ? 2 * NC * 256 : 0);     // [3][16][PR] in 64 bits
  static constexpr int M = P + 6 * C * PR;                     // DELTA: [2][16][TR]
  static constexpr int T = M + (MODE == DELTA ? 2 * C * TR : 0);       // DELTA: [2][16][TR]
  static constexpr int SC = T + (MODE == DELTA ? 2 * C * TR : 0);      // [4][96] per-token factors, see below
  static constexpr int GT = SC + (CH ? 0 : 4 * 96);            // [2][3][64] gates of 64 tokens
  static constexpr int DM = GT + (CH ? 0 : 384);               // [4][64][4] D as the scores wave holds P^T, [4][16] A
  static constexpr int NRM = DM + (CH ? 0 : 4 * 272);              // DELTA: [4][NS][32] squared norms;  MLSTM: [DP] normaliser
  static constexpr int RAW = NRM + (MODE == DELTA ? 4 * NS * 32 : (MODE == MLSTM ? DP : 0));      // CH: [2][NS][RAWN]
  static constexpr int RAWN = 276;
  static constexpr int END = RAW + (CH ? 2 * NS * RAWN : 0);
};
// per-token factors [16] each: 0 of the state read-out, 16 of the state update, 32 delta: beta, mlstm: row sums of P, then 1 / normaliser,
// 48 delta: -beta A / |k|, mlstm: exp(-maximum), 64 mlstm: A, 80 (one number) decay of the chunk.  Where they meet the registers of u or of
// an output they lie as those do, token t at place(t), so do the columns of P: register r of lane group g holds token 4 r + g, and a sum
// over the tokens starts with the oldest, which under a decay are the small ones.
__device__ __forceinline__ constexpr int place(int t) { return 4 * (t & 3) + (t >> 2); }      // its own inverse

// Steps whose workgroups of two column blocks do not find a compute unit each: four blocks share what does not depend on the columns
// (q, k, gates, scores), at SLOW hundredths of two blocks' time per chunk.  Only the lengths say which is the faster (decode rows and short portions
// take no place for long), so the workgroups decide: all chunks over 256 units and a part of the longest sequence's for the last round, or the longest
// sequence's if that is more.  seq, the seq-th longest before, becomes the sequence itself.
//   us before (two blocks, sequences in their order) and now, 64-wide heads       delta
//   5 prompts of 3001 bf16 rows in all, 32 heads                                  97, 91
//   12 prompts of 4000, 64 heads                                                  173, 158
//   9 prompts of 1500, 32 heads                                                   51, 54
//   1 prompt of 2048 and 3 decode rows, 64 heads (stays at two blocks)            242, 157
constexpr int MOST_SEQ = 16;       // more would be decode rows mostly, whose workgroups should be gone soon
__device__ __forceinline__ bool four_blocks(const ChunkArgs& a, int& seq, int& row0, int& n) {
  constexpr int SLOW = 150;
  const int lane = threadIdx.x & 63, i = min(lane, a.n_seq - 1);
  const int from = a.seq_row0[i], len = lane < a.n_seq ? max(a.seq_row0[i + 1] - from, 0) : -1;
  int before = 0;                                    // sequences that are longer, or as long and earlier
  for (int j = 0; j < a.n_seq; ++j) {
    const int other = __builtin_amdgcn_readlane(len, j);
    before += other > len || (other == len && j < lane);
  }
  seq = __ffsll((unsigned long long)__ballot(lane < a.n_seq && before == seq)) - 1;
  row0 = __builtin_amdgcn_readlane(from, seq);
  n = __builtin_amdgcn_readlane(len, seq);
  const float own = len > a.skip_rows ? (float)((len + C - 1) / C + 5) : 0.f;      // the pipeline fills in some five
  float sum = own, most = own;
#pragma unroll
  for (int o = MOST_SEQ / 2; o > 0; o >>= 1) {
    sum += __shfl_xor(sum, o, 64);
    most = fmaxf(most, __shfl_xor(most, o, 64));
  }
  const float units = (float)__popcll(__ballot(own > 0.f)) * a.H, part = sum * a.H / 256.f;
  auto time = [&](int blocks) { return fmaxf(most, part * blocks + (units * blocks > 256.f ? most * 0.5f : 0.f)); };
  return __builtin_amdgcn_readfirstlane(time((a.dv + 31) / 32) * 100.f > time((a.dv + 63) / 64) * SLOW);
}

// two waves per SIMD at least: within 256 registers the products take ordinary registers, without moves to accumulation ones
template <int MODE, typename TI, int NT, int COLS>
__global__ __launch_bounds__((64 * Lay<MODE, NT, COLS>::WAVES), 2) void chunk_scan_kernel(const ChunkArgs a) {
  using L = Lay<MODE, NT, COLS>;
  constexpr int QR = L::QR, DP = L::DP, NS = L::NS, LEAD = L::LEAD;
  extern __shared__ __attribute__((aligned(16))) float sm[];
  // consecutive workgroups (which go to different XCDs) own consecutive heads; a head's workgroups come n_seq * H later
  const int head = blockIdx.x % a.H, zb = blockIdx.x / a.H / a.n_seq, seg = MODE == SSM ? blockIdx.y : 0;
  int seq = blockIdx.x / a.H % a.n_seq, blocks = L::NC;      // blocks: of columns, this workgroup's
  int row0, n;
  if constexpr (COLS == 64) {
    blocks = four_blocks(a, seq, row0, n) ? 4 : 2;       // the same in every workgroup
    if (zb * blocks * 16 >= a.dv) return;            // the grid is that of two blocks each
  } else {
    row0 = a.seq_row0[seq];
    n = a.seq_row0[seq + 1] - row0;
  }
  if (n <= a.skip_rows) return;
  const int slot = a.seq_slots[seq];
  // ssm in segments (see below): 1 the state of a segment from nothing, to the workspace; 2 outputs from the state found there
  bool stored = MODE == SSM ? a.positions[row0] != 0 : a.positions[row0] > 0, last = true;      // as the loops of their files
  if (MODE == SSM && a.pass) {
    row0 += seg * a.seg_rows;
    n -= seg * a.seg_rows;
    last = n <= a.seg_rows;
    if (n <= 0 || (last && a.pass == 1)) return;
    n = min(n, a.seg_rows);
    stored = a.pass == 2;
  }
  const int H = a.H, dk = a.dk, dv = a.dv;
  const int kvh = head / (H / a.G);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n16 = lane & 15, g = lane >> 4;
  const int chunks = ((n + C - 1) / C + 1) & ~1;      // an even number: a chunk past the end changes nothing
  const float qscale = 1.f / sqrtf((float)dk);
  const TI* qb = (const TI*)a.q + (size_t)row0 * a.q_stride + (size_t)kvh * dk;
  const TI* kb = (const TI*)a.k + (size_t)row0 * a.k_stride + (size_t)kvh * dk;

  // Every role passes chunks + LEAD barriers.  Loads run unconditionally (rows and channels clamped into the portion) in loops of two
  // chunks: a load behind a branch, or one whose registers are renamed at the end of a loop, would be waited for on the spot.
  auto barriers = [&](int m) {
    for (int i = 0; i < m; ++i) __syncthreads();
  };
  // Products over the channels 16 i .. + 15.  A sum over all channels runs in several sums side by side that are added as a tree at the
  // end, so that its error is a tree's.
  auto channels = [](auto& acc, int i, const float4& x, const f32x4& y) {
    constexpr int N = sizeof(acc) / sizeof(acc[0]);
    const float xs[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[(4 * i + r) % N] = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[r], y[r], acc[(4 * i + r) % N], 0, 0, 0);
  };
  auto zero = [](auto& acc) {
    constexpr int N = sizeof(acc) / sizeof(acc[0]);
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  };
  auto total = [](auto& acc) {
    constexpr int N = sizeof(acc) / sizeof(acc[0]);
#pragma unroll
    for (int h = N / 2; h > 0; h /= 2)
#pragma unroll
      for (int i = 0; i < h; ++i) acc[i] += acc[i + h];
    return acc[0];
  };
  const int prep = wave >= L::PREP ? wave - L::PREP + L::EARLY : (wave < L::SCORES && wave >= L::SCORES - L::EARLY ? wave - (L::SCORES - L::EARLY) : -1);
  if (prep >= 0) {
    // ============================================================================================== preparing waves
    const int w = prep % NS, turn = prep / NS % 2, set = prep / (2 * NS);       // set: 0 the scores' operands, 1 the state's (or 0: both)
    if constexpr (L::CH) {
      // lane = channel.  Chunk c takes two steps of its wave: decays, then products and LDS.
      const int ch = 64 * w + lane, cc = min(ch, dk - 1);
      const bool in = ch < dk;
      const unsigned oq = cc * sizeof(TI), od = cc * 4;
      const char* db = (const char*)((const float*)a.aux1 + (size_t)row0 * a.aux1_stride + (size_t)head * dk);
      TI rq[C], rk[C];
      float rd[C], d[C];
      const float w0 = a.par1[(size_t)head * dk + cc], bonus = a.par2[(size_t)head * dk + cc];
      const float qs = in ? 1.f : 0.f;               // channels past dk: q = 0
      // the lane's offsets from a chunk's first row are kept, the row's address advances in scalar registers
      unsigned vq[C], vk[C], vd[C];
#pragma unroll
      for (int t = 0; t < C; ++t) {
        vq[t] = (unsigned)t * a.q_stride * (unsigned)sizeof(TI) + oq;
        vk[t] = (unsigned)t * a.k_stride * (unsigned)sizeof(TI) + oq;
        vd[t] = (unsigned)t * a.aux1_stride * 4u + od;
      }
      auto load_d = [&](int c) {
        const int first = min(c * C, n - 1);
        global_in p = (global_in)db + (size_t)first * a.aux1_stride * 4;
        asm volatile("" : "+s"(p));
        if (first + C <= n) {
#pragma unroll
          for (int t = 0; t < C; ++t) rd[t] = gload<float>(p + vd[t]);
        } else {
#pragma unroll
          for (int t = 0; t < C; ++t) rd[t] = gload<float>(p + ((unsigned)min(t, n - 1 - first) * a.aux1_stride * 4u + od));
        }
      };
      auto load_qk = [&](int c) {
        const int first = min(c * C, n - 1);
        global_in q = (global_in)(qb + (size_t)first * a.q_stride), k = (global_in)(kb + (size_t)first * a.k_stride);
        asm volatile("" : "+s"(q), "+s"(k));
        if (first + C <= n) {
#pragma unroll
          for (int t = 0; t < C; ++t) {
            rq[t] = gload<TI>(q + vq[t]);
            rk[t] = gload<TI>(k + vk[t]);
          }
        } else {
#pragma unroll
          for (int t = 0; t < C; ++t) {
            const unsigned r = (unsigned)min(t, n - 1 - first) * (unsigned)sizeof(TI);
            rq[t] = gload<TI>(q + (r * a.q_stride + oq));
            rk[t] = gload<TI>(k + (r * a.k_stride + oq));
          }
        }
      };
      auto decays = [&]() {
#pragma unroll
        for (int t = 0; t < C; ++t) d[t] = exp_neg_exp(rd[t] + w0);
      };
      auto prepare = [&](int c) {
        const int left = n - c * C;
        float* Q = sm + L::Q + (c % L::QB) * L::ROWS + ch;
        float* QT = sm + L::QT + (c & 1) * L::ROWS + ch;
        float* K = sm + L::K + (c & 1) * L::ROWS + ch;
        float* KT = sm + L::KT + ((c % L::KB) * DP + ch) * TR;
        float q[C], k[C];
#pragma unroll
        for (int t = 0; t < C; ++t) {
          q[t] = ldf<TI>(&rq[t]) * qs;
          k[t] = ldf<TI>(&rk[t]);
        }
        if (left < C) {                                      // rows past the portion: nothing read, nothing written, no decay
#pragma unroll
          for (int t = 0; t < C; ++t)
            if (t >= left) { q[t] = 0.f; k[t] = 0.f; d[t] = 1.f; }
        }
        float s[C];
        if (L::SETS == 1 || set == 1) {
          // suffix products: the state's update (their rounding errors carried along: they would stay in the state)
          float run = 1.f, low = 0.f;
#pragma unroll
          for (int t = C - 1; t >= 0; --t) {
            s[t] = k[t] * (run + low);
            const float next = run * d[t];
            low = fmaf(low, d[t], fmaf(run, d[t], -next));
            run = next;
          }
#pragma unroll
          for (int i = 0; i < 4; ++i) *reinterpret_cast<float4*>(KT + 4 * i) = make_float4(s[i], s[4 + i], s[8 + i], s[12 + i]);      // by place
          sm[L::DEC + (c % L::KB) * DP + ch] = run + low;
          // prefix products: the state's read-out, before the token's own decay
          float f = 1.f;
#pragma unroll
          for (int t = 0; t < C; ++t) {
            const float before = f;
            f *= d[t];
            Q[t * QR] = q[t] * before;
          }
        }
        if (L::SETS == 2 && set == 1) return;
        // the scores' scales, from the middle of the chunk out
        float lo = 1.f, hi = 1.f;
#pragma unroll
        for (int t = 7; t >= 0; --t) {                       // lo: decays of the tokens after t up to the middle
          const float own = lo * d[t];
          QT[t * QR] = q[t] * __builtin_amdgcn_rcpf(own);
          K[t * QR] = k[t] * lo;
          lo = own;
        }
#pragma unroll
        for (int t = 8; t < C; ++t) {                        // hi: decays from the middle on up to t
          const float before = hi;
          hi *= d[t];
          QT[t * QR] = q[t] * before;
          K[t * QR] = k[t] * __builtin_amdgcn_rcpf(hi);
        }
        float* R = sm + L::RAW + ((c & 1) * NS + w) * L::RAWN;
        // The scaled operands have to stay in the fp32 range.  Those divided are q of the tokens 1 to 7 and k of 8 to 14 (0 and 15 have no
        // partner in the chunk), those multiplied, and lost where they are small, k of 0 to 6 and q of 9 to 15.
        const float least = fminf(lo, hi);
        float top = 0.f;
#pragma unroll
        for (int t = 1; t < 8; ++t) top = larger3(top, q[t], k[t + 7]);
        bool raw = false;
        if (__builtin_expect(__any(!(least > 1e-8f && top < 1e30f)), 0)) {
          float low = 1.f;
#pragma unroll
          for (int t = 0; t < 7; ++t) low = fminf(low, fminf(q[t + 9] == 0.f ? 1.f : fabsf(q[t + 9]), k[t] == 0.f ? 1.f : fabsf(k[t])));
          raw = __any(!(least > SAFE && top < 1e38f * least && low * least > 1e-36f));
        }
        if (lane == 0) R[0] = raw ? 1.f : 0.f;
#pragma unroll
        for (int t = 0; t < C; ++t) s[t] = q[t] * bonus * k[t];
        const float bo = sum16(s, lane);
        if (lane < C) R[4 + lane] = bo;
        if (__builtin_expect(raw, 0)) {                      // scores of these 64 channels token by token
#pragma unroll 1
          for (int i = 0; i < C; ++i) {
            float ki = 0.f, run1 = 1.f;
#pragma unroll
            for (int t = 0; t < C; ++t) ki = t == i ? k[t] : ki;
#pragma unroll
            for (int t = 0; t < C; ++t) {
              const float before = run1;
              run1 = t > i ? run1 * d[t] : run1;
              s[t] = t >= i ? q[t] * ki * before : 0.f;
            }
            const float o = sum16(s, lane);
            if (lane < C) R[20 + i * C + lane] = o;
          }
        }
      };
      load_d(turn);
      load_qk(turn);
      barriers(turn);
      for (int c = turn; c < chunks; c += 2) {
        decays();
        load_d(c + 2);
        __syncthreads();
        prepare(c);
        load_qk(c + 2);
        __syncthreads();
      }
      barriers(LEAD - turn);
    } else {
      // lane = (token, quarter): sixteen channels of a token in four pieces
      const int t = lane >> 2, j = lane & 3;
      Raw4<TI> rq[2][4], rk[2][4];
      // the lane's offsets from a chunk's first row are kept, the row's address advances in scalar registers
      unsigned vx[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) vx[i] = (unsigned)min(64 * w + 16 * i + 4 * j, dk - 4) * (unsigned)sizeof(TI);
      const unsigned vq = (unsigned)t * a.q_stride * (unsigned)sizeof(TI), vk = (unsigned)t * a.k_stride * (unsigned)sizeof(TI);
      auto load = [&](int c, int st) {
        const int first = min(c * C, n - 1);
        global_in pq = (global_in)(qb + (size_t)first * a.q_stride), pk = (global_in)(kb + (size_t)first * a.k_stride);
        asm volatile("" : "+s"(pq), "+s"(pk));
        unsigned oq = vq, ok = vk;
        if (first + C > n) {
          const unsigned r = (unsigned)min(t, n - 1 - first) * (unsigned)sizeof(TI);
          oq = r * a.q_stride;
          ok = r * a.k_stride;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          rq[st][i] = gload<Raw4<TI>>(pq + (oq + vx[i]));
          rk[st][i] = gload<Raw4<TI>>(pk + (ok + vx[i]));
        }
      };
      float q[4][4], k[4][4];
      auto take = [&](int c, int st) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          widen(rq[st][i], q[i]);
          widen(rk[st][i], k[i]);
        }
        if (n - c * C < C || dk < DP) {                      // rows past the portion, channels past dk: zeros
          const bool ok = c * C + t < n;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              const bool in = ok && 64 * w + 16 * i + 4 * j + x < dk;
              q[i][x] = in ? q[i][x] : 0.f;
              k[i][x] = in ? k[i][x] : 0.f;
            }
        }
      };
      auto put = [&](int c) {
        float* Q = sm + L::Q + (c % L::QB) * L::ROWS + t * QR + 64 * w + 4 * j;
        float* K = sm + L::K + (c % L::KB) * L::ROWS + place(t) * QR + 64 * w + 4 * j;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          *reinterpret_cast<float4*>(Q + 16 * i) = make_float4(q[i][0], q[i][1], q[i][2], q[i][3]);
          *reinterpret_cast<float4*>(K + 16 * i) = make_float4(k[i][0], k[i][1], k[i][2], k[i][3]);
        }
        if constexpr (MODE == DELTA) {
          float sq = 0.f, sk = 0.f;
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              sq += q[i][x] * q[i][x];
              sk += k[i][x] * k[i][x];
            }
          sq += dpp_move<0xB1>(sq); sk += dpp_move<0xB1>(sk);
          sq += dpp_move<0x4E>(sq); sk += dpp_move<0x4E>(sk);
          float* N = sm + L::NRM + ((c & 3) * NS + w) * 32;
          if (j == 0) { N[t] = sk; N[16 + t] = sq; }
        }
      };
      if constexpr (L::TURNS) {
        load(turn, 0);
        barriers(turn);
        for (int c = turn; c < chunks; c += 2) {
          take(c, 0);
          load(c + 2, 0);
          __syncthreads();
          put(c);
          __syncthreads();
        }
        barriers(LEAD - turn);
      } else {
        load(0, 0);
        load(1, 1);
        for (int c = 0; c < chunks; c += 2) {
          take(c, 0);
          load(c + 2, 0);
          put(c);
          __syncthreads();
          take(c + 1, 1);
          load(c + 3, 1);
          put(c + 1);
          __syncthreads();
        }
        barriers(LEAD);
      }
    }
    return;
  }

  if (wave >= L::SCORES && wave < L::PREP) {
    // ============================================================================================== scores waves
    const int turn = wave - L::SCORES;
    f32x4 pa, ka;                                    // keys s = 4 g + r by queries (delta: also keys) t = n16
    float bon;
    // delta: 1 / |k_t|, dk^-1/2 / |q_t| and 1 / |k_s| of the tokens s (beside the products: the step after is the longer one)
    float nk, nq, ns[4];
    auto norms = [&](int c) {
      float sk = 0.f, sq = 0.f;
      float* N = sm + L::NRM + (c & 3) * NS * 32;
#pragma unroll
      for (int w = 0; w < NS; ++w) {
        sk += N[32 * w + n16];
        sq += N[32 * w + 16 + n16];
      }
      nk = 1.f / sqrtf(sk + 1e-6f);
      nq = qscale / sqrtf(sq + 1e-6f);
      __builtin_amdgcn_wave_barrier();
      if (g == 0) N[n16] = nk;
      __builtin_amdgcn_wave_barrier();
      const float4 x = ld4(N + 4 * g);
      ns[0] = x.x; ns[1] = x.y; ns[2] = x.z; ns[3] = x.w;
    };
    // Four channels are one product and the products are added as a tree (delta: two and two): this
    // error is all columns', and P is what the results of a fast decay consist of.
    auto products = [&](int c) {
      const float* Q = sm + (L::CH ? L::QT + (c & 1) * L::ROWS : L::Q + (c % L::QB) * L::ROWS) + n16 * QR + 4 * g;
      const float* K = sm + L::K + (L::CH ? (c & 1) * L::ROWS + n16 * QR : (c % L::KB) * L::ROWS + place(n16) * QR) + 4 * g;
      pa = ka = f32x4{0.f, 0.f, 0.f, 0.f};
      auto tiles = [&](int i0) {
        constexpr int N = 4, PER = MODE == DELTA ? 2 : 4;
        f32x4 ps[PER * N], ks[PER * N];
        zero(ps);
        zero(ks);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const float4 qf = ld4(Q + 16 * (i0 + i)), kf = ld4(K + 16 * (i0 + i));
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float qs[4] = {qf.x, qf.y, qf.z, qf.w}, kx[4] = {kf.x, kf.y, kf.z, kf.w};
            const int o = PER * i + r % PER;
            ps[o] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[r], qs[r], ps[o], 0, 0, 0);
            if constexpr (MODE == DELTA) ks[o] = __builtin_amdgcn_mfma_f32_16x16x4f32(kx[r], kx[r], ks[o], 0, 0, 0);
          }
        }
        pa += total(ps);
        if constexpr (MODE == DELTA) ka += total(ks);
      };
      if constexpr (L::CH) {
        bon = 0.f;
#pragma unroll
        for (int w = 0; w < NS; ++w) {
          const float* R = sm + L::RAW + ((c & 1) * NS + w) * L::RAWN;
          bon += R[4 + n16];
          if (R[0] != 0.f) {
#pragma unroll
            for (int r = 0; r < 4; ++r) pa[r] += R[20 + (4 * g + r) * C + n16];
          } else {
            tiles(4 * w);
          }
        }
      } else {
#pragma unroll
        for (int w = 0; w < NS; ++w) {
          tiles(4 * w);
          if constexpr (NT == 16) __builtin_amdgcn_sched_barrier(0);       // all tiles' products at once would not fit the registers
        }
      }
    };
    auto finish = [&](int c) {
      double* P = reinterpret_cast<double*>(sm + L::P) + (c % 3 * C + n16) * PR + g;      // s = 4 g + r at place 4 r + g
      double p[4];
      if constexpr (L::CH) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int s = 4 * g + r;
          p[r] = s < n16 ? pa[r] : (s == n16 ? bon : 0.f);
        }
      } else {
        const float* G = sm + L::GT + ((c >> 2) & 1) * 192 + 16 * (c & 3);
        const float* DM = sm + L::DM + (c & 3) * 272;
        const float4 wr = ld4(G + 64 + 4 * g), d4 = ld4(DM + 4 * lane);       // write factors of the tokens s
        const float D[4] = {d4.x, d4.y, d4.z, d4.w}, A = DM[256 + n16];
        float cf[4] = {wr.x, wr.y, wr.z, wr.w}, qs = 1.f, rk = 1.f;
        if constexpr (MODE == MLSTM) qs = qscale;
        if constexpr (MODE == DELTA) {
          qs = nq;
          rk = nk;
#pragma unroll
          for (int r = 0; r < 4; ++r) cf[r] = ns[r];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = 4 * g + r <= n16 ? (double)pa[r] * ((double)qs * cf[r]) * D[r] : 0.;
        float* S = sm + L::SC + (c & 3) * 96;
        if (g == 0) S[place(n16)] = A * qs;
        if (n16 == 15) {
#pragma unroll
          for (int r = 0; r < 4; ++r) S[16 + 4 * r + g] = D[r] * cf[r];
          if (g == 0) S[80] = A;
        }
        if constexpr (MODE == DELTA) {
          const float beta = G[128 + n16];
          if (g == 0) { S[32 + place(n16)] = beta; S[48 + place(n16)] = -beta * A * rk; }
          float* T = sm + L::T + (c & 1) * C * TR;
          float tt[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) tt[r] = 4 * g + r < n16 ? beta * rk * cf[r] * D[r] * ka[r] : 0.f;
          *reinterpret_cast<float4*>(T + n16 * TR + 4 * g) = make_float4(tt[0], tt[1], tt[2], tt[3]);
          __builtin_amdgcn_wave_barrier();
          // M: lane = (row n16, block g): m (I + T_gg) = row of the identity (own block) or - T (blocks below)
          const float4 row = ld4(T + n16 * TR + 4 * g);
          const float4 t1 = ld4(T + (4 * g + 1) * TR + 4 * g), t2 = ld4(T + (4 * g + 2) * TR + 4 * g), t3 = ld4(T + (4 * g + 3) * TR + 4 * g);
          const bool own = (n16 >> 2) == g, below = (n16 >> 2) > g;
          const int e = n16 & 3;
          const float e0 = own && e == 0 ? 1.f : 0.f, e1 = own && e == 1 ? 1.f : 0.f, e2 = own && e == 2 ? 1.f : 0.f, e3 = own && e == 3 ? 1.f : 0.f;
          const float m3 = below ? -row.w : e3;
          const float m2 = (below ? -row.z : e2) - m3 * t3.z;
          const float m1 = (below ? -row.y : e1) - m2 * t2.y - m3 * t3.y;
          const float m0 = (below ? -row.x : e0) - m1 * t1.x - m2 * t2.x - m3 * t3.x;
          float* M = sm + L::M + (c & 1) * C * TR + place(n16) * TR + g;      // rows and columns by place
          M[0] = m0 - e0; M[4] = m1 - e1; M[8] = m2 - e2; M[12] = m3 - e3;
        }
        if constexpr (MODE == MLSTM) {
          float rs = ((float)p[0] + (float)p[1]) + ((float)p[2] + (float)p[3]);
          rs += __shfl_xor(rs, 16, 64);
          rs += __shfl_xor(rs, 32, 64);
          if (g == 0) { S[32 + n16] = rs; S[48 + n16] = G[128 + n16]; S[64 + n16] = A * qs; }
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) P[4 * r] = p[r];
    };
    barriers(LEAD - 1 - L::W2 + turn);
    for (int c = turn; c < chunks; c += L::W2) {
      if constexpr (MODE == DELTA) norms(c);
      products(c);
      if constexpr (L::W2 == 2) __syncthreads();
      finish(c);
      __syncthreads();
    }
    barriers(1 + L::W2 - turn);
    return;
  }

  if constexpr (!L::CH) {
    if (wave == L::GATES) {
      // ============================================================================================ gates, 64 tokens (one per lane) in four steps
      float ga = 0.f, gb = 0.f;                      // raw gates of the next 64 tokens
      float p1 = 0.f, p2 = 0.f;
      if constexpr (MODE == DELTA || MODE == SSM) { p1 = -expf(a.par1[head]); p2 = a.par2[head]; }
      float m_run = 0.f, m_old = 0.f, m_new = 0.f, x = 0.f, z = 0.f;       // mlstm: running maximum, input gate, forget gate
      if constexpr (MODE == MLSTM) {
        if (stored) m_run = a.mx[(size_t)slot * H + head];
      }
      auto load_gates = [&](int b) {
        const size_t t = row0 + min(b * 64 + lane, n - 1);
        if constexpr (MODE == DELTA || MODE == MLSTM) {
          ga = ((const float*)a.aux1)[t * a.aux1_stride + head];
          gb = ((const float*)a.aux2)[t * a.aux2_stride + head];
        } else if constexpr (MODE == SSM) {
          const size_t at = t * a.aux1_stride + head;
          ga = a.aux_bf16 ? bf16_to_f32(((const uint16_t*)a.aux1)[at]) : ((const float*)a.aux1)[at];
        }
      };
      // phase 0: each token's own; mlstm 1 - 3: the running maximum over a third of the tokens (a serial chain of adds and maxima);
      // 3: to LDS
      auto gates = [&](int b, int phase) {
        if (phase == 0) {
          if constexpr (MODE == SSM) {
            x = softplus_f(ga + p2);
            z = expf(p1 * x);
          } else if constexpr (MODE == DELTA) {
            z = expf(p1 * softplus_f(gb + p2));
            x = 1.f / (1.f + expf(-ga));
          } else {
            // tokens past the portion leave the maximum as it is
            const bool ok = b * 64 + lane < n;
            x = ok ? a.cap * tanhf(ga / a.cap) : -__builtin_inff();
            z = ok ? logsigmoid_f(a.cap * tanhf(gb / a.cap)) : 0.f;
          }
          load_gates(b + 1);
        }
        if constexpr (MODE == MLSTM) {
          // every lane carries the maximum; each token's goes to LDS (the factors' place of the tokens' gates)
          float* G = sm + L::GT + (b & 1) * 192;
          auto run = [&](auto from, auto to) {
            if (from.value == 0) G[128] = m_run;
#pragma unroll
            for (int t = from.value; t < to.value; ++t) {
              const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, z), t));
              const float i = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, x), t));
              m_run = fmaxf(f + m_run, i);
              G[t] = m_run;
            }
          };
          if (phase == 1) run(std::integral_constant<int, 0>{}, std::integral_constant<int, 22>{});
          if (phase == 2) run(std::integral_constant<int, 22>{}, std::integral_constant<int, 43>{});
          if (phase == 3) {
            run(std::integral_constant<int, 43>{}, std::integral_constant<int, 64>{});
            __builtin_amdgcn_wave_barrier();
            m_new = G[lane];
            m_old = lane ? G[lane - 1] : G[128];
            __builtin_amdgcn_wave_barrier();
          }
        }
        if (phase == 3) {
          // decay | write factor | mlstm: exp(-maximum), delta: write strength; tokens past the portion: no decay, nothing written
          const bool ok = b * 64 + lane < n;
          float* G = sm + L::GT + (b & 1) * 192 + lane;
          G[0] = !ok ? 1.f : (MODE == MLSTM ? expf(z + m_old - m_new) : z);
          G[64] = !ok ? 0.f : (MODE == MLSTM ? expf(x - m_new) : x);
          G[128] = !ok ? 0.f : (MODE == MLSTM ? expf(-m_new) : x);
        }
      };
      // D[t = n16, s = 4 g + r] and A_t of a chunk: one running product down from t, with its rounding errors carried along (all
      // channels share these factors, so the errors would not average out over a read-out's sum)
      auto products = [&](int c) {
        const float* G = sm + L::GT + ((c >> 2) & 1) * 192 + 16 * (c & 3);
        float D[4], A = 1.f, low = 0.f;
        auto times = [&](float d) {
          const float next = A * d;
          low = fmaf(low, d, fmaf(A, d, -next));
          A = next;
        };
        auto product = [&]() { return A + low; };
#pragma unroll
        for (int i = 3; i > 0; --i) {                  // the tokens behind this lane's four, up to t
          const float4 d4 = ld4(G + 4 * i);
          const float dd[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
          for (int r = 3; r >= 0; --r) times(i > g && 4 * i + r <= n16 ? dd[r] : 1.f);
        }
        const float4 d4 = ld4(G + 4 * g);
        const float dd[4] = {d4.x, d4.y, d4.z, d4.w};
#pragma unroll
        for (int r = 3; r >= 0; --r) {
          D[r] = 4 * g + r <= n16 ? product() : 0.f;
          times(4 * g + r <= n16 ? dd[r] : 1.f);
        }
        A = product();                                 // lane group 0: of all tokens
        float* DM = sm + L::DM + (c & 3) * 272;
        *reinterpret_cast<float4*>(DM + 4 * lane) = make_float4(D[0], D[1], D[2], D[3]);
        if (g == 0) DM[256 + n16] = A;
      };
      load_gates(0);
      for (int k = 0; k < 4; ++k) gates(0, k);
      for (int i = 0; i < chunks + LEAD; ++i) {
        const int c = i - (LEAD - 1 - L::W2);        // as the scores waves count: while they use a batch, the next one is made
        const int b = (c >> 2) + 1;
        if (c >= 0 && b * 64 < n) gates(b, c & 3);
        // read a step later, by the second half of the scores (NT 16: in the next step, with the first)
        const int ready = L::W2 == 2 ? c : c + 1;
        if (ready >= 0 && ready < chunks) products(ready);
        __syncthreads();
      }
      if constexpr (MODE == MLSTM) {
        if (zb == 0 && lane == 0) (a.mx_new ? a.mx_new[(size_t)seq * H + head] : a.mx[(size_t)slot * H + head]) = m_run;
      }
      return;
    }
  }

  if constexpr (MODE == MLSTM) {
    if (wave == L::NORM) {
      // ============================================================================================ normaliser (lane = channel)
      float nrm[NS];
      const size_t nb = ((size_t)slot * H + head) * dk;
#pragma unroll
      for (int w = 0; w < NS; ++w) nrm[w] = (stored && 64 * w + lane < dk) ? a.norm[nb + 64 * w + lane] : 0.f;
      barriers(LEAD - 1);
      for (int c = 0; c < chunks; ++c) {
        const float* Q = sm + L::Q + (c % L::QB) * L::ROWS;
        const float* K = sm + L::K + (c % L::KB) * L::ROWS;
        float* S = sm + L::SC + (c & 3) * 96;
        float* N = sm + L::NRM;
#pragma unroll
        for (int w = 0; w < NS; ++w) N[64 * w + lane] = nrm[w];
        __builtin_amdgcn_wave_barrier();
        // normaliser . q_t: the scores' row sums and the chunk's starting normaliser; lane = (token n16, quarter of the channels)
        float dot = 0.f;
#pragma unroll
        for (int i = 0; i < NT; ++i) {
          const float4 nv = ld4(N + 16 * i + 4 * g), qv = ld4(Q + n16 * QR + 16 * i + 4 * g);
          dot += nv.x * qv.x + nv.y * qv.y + nv.z * qv.z + nv.w * qv.w;
        }
        dot += __shfl_xor(dot, 16, 64);
        dot += __shfl_xor(dot, 32, 64);
        const float nq = S[32 + n16] + dot * S[64 + n16];
        const float inv = 1.f / (fmaxf(fabsf(nq), S[48 + n16]) + 1e-6f);
        const float at = S[80];
        float f[C];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float4 f4 = ld4(S + 16 + 4 * i);
          f[place(4 * i)] = f4.x; f[place(4 * i + 1)] = f4.y; f[place(4 * i + 2)] = f4.z; f[place(4 * i + 3)] = f4.w;
        }
#pragma unroll
        for (int w = 0; w < NS; ++w) nrm[w] *= at;
#pragma unroll
        for (int t = 0; t < C; ++t)
#pragma unroll
          for (int w = 0; w < NS; ++w) nrm[w] += f[t] * K[place(t) * QR + 64 * w + lane];
        __builtin_amdgcn_wave_barrier();
        if (g == 0) S[32 + place(n16)] = inv;
        __syncthreads();
      }
      __syncthreads();
      if (zb == 0) {
        float* np = a.norm_new ? a.norm_new + ((size_t)seq * H + head) * dk : a.norm + nb;
#pragma unroll
        for (int w = 0; w < NS; ++w)
          if (64 * w + lane < dk) np[64 * w + lane] = nrm[w];
      }
      return;
    }
  }

  const bool outputs = wave >= L::OUT;
  // column block of the workgroup (two of four: those of the outputs beside other SIMDs than those of the state)
  const int cw = outputs ? wave - L::OUT - (COLS == 64 && blocks == 2 ? 2 : 0) : wave;
  if (COLS == 64 && (cw < 0 || cw >= blocks)) {
    barriers(chunks + LEAD);
    return;
  }
  const int col = (zb * blocks + cw) * 16 + n16, colc = min(col, dv - 1);
  const bool cok = col < dv;
  const TI* vb = (const TI*)a.v + (size_t)row0 * a.v_stride + (size_t)head * dv;
  auto tok = [&](int r) { return 4 * r + g; };
  TI rv[2][4];
  unsigned vv[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) vv[r] = (unsigned)(tok(r) * a.v_stride + colc) * (unsigned)sizeof(TI);
  // Flat in two places.  us with global loads and stores alone, and now: mlstm, fp32 rows, 128 channels, 70 rows 22.0, 21.2; 40 x 70 rows of 32 heads
  // 190, 182; 2007 rows 184, 186.  delta, fp32 rows, 64 channels, 2000 rows beside 7 149.3, 146; 20 x 40 + 300 rows of 32 heads 61.9, 60.9.
  typedef std::conditional_t<MODE == MLSTM, const char*, global_in> values_in;
  typedef std::conditional_t<MODE == DELTA, char*, global_out> outputs_to;
  auto load_v = [&](int c, int st) {
    const int first = min(c * C, n - 1);
    values_in p = (values_in)(vb + (size_t)first * a.v_stride);
    asm volatile("" : "+s"(p));
    if (first + C <= n) {
#pragma unroll
      for (int r = 0; r < 4; ++r) rv[st][r] = gload<TI>(p + vv[r]);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        rv[st][r] = gload<TI>(p + (unsigned)(min(tok(r), n - 1 - first) * a.v_stride + colc) * (unsigned)sizeof(TI));
    }
  };
  auto take_v = [&](int c, int st, float* u) {
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = ldf<TI>(&rv[st][r]);
    if ((c + 1) * C > n) {                           // rows past the portion
#pragma unroll
      for (int r = 0; r < 4; ++r) u[r] = c * C + tok(r) < n ? u[r] : 0.f;
    }
    load_v(c + 2, st);
  };
  load_v(0, 0);
  load_v(1, 1);

  if (!outputs) {
    // ============================================================================================== state waves
    // state rows (channels) 16 i + 4 g + r, column n16
    f32x4 S[NT];
    const size_t sbase = ((size_t)slot * H + head) * dk * dv, wbase = (((size_t)seq * gridDim.y + seg) * H + head) * dk * dv;
    const float* from = MODE == SSM && a.pass ? a.ws + wbase : a.state + sbase;
    float* to = MODE == SSM && a.pass == 1 ? a.ws + wbase : a.state + sbase;
    float all = 1.f;                                 // ssm, pass 1: decay of the segment
    auto sat = [&](int ch) { return MODE == SSM ? (size_t)colc * dk + ch : (size_t)ch * dv + colc; };
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ch = 16 * i + 4 * g + r;
        S[i][r] = (stored && ch < dk && cok) ? from[sat(ch)] : 0.f;
      }
    barriers(LEAD - 1);
    auto step = [&](int c, int st) {
      const float* K = sm + L::K + (c % L::KB) * L::ROWS;
      const float* KT = sm + L::KT + ((c % L::KB) * DP + n16) * TR + 4 * g;
      const float* DE = sm + L::DEC + (c % L::KB) * DP + 4 * g;
      const float* F = sm + L::SC + (c & 3) * 96;
      float u[4], x[4];
      take_v(c, st, u);
      float* ST = sm + L::ST + ((c & 1) * L::NC + cw) * DP * 16 + 4 * lane;
#pragma unroll
      for (int i = 0; i < NT; ++i) *reinterpret_cast<f32x4*>(ST + 256 * i) = S[i];
      const float at = L::CH ? 1.f : F[80];
      if constexpr (MODE == SSM) all *= at;
      if constexpr (MODE == DELTA) {
        // x = beta v - beta A S^T k / |k|, rows in the order of u's registers
        f32x4 xs[L::NA];
        zero(xs);
        const float* Kr = K + n16 * QR + 4 * g;
#pragma unroll
        for (int i = 0; i < NT; ++i) channels(xs, i, ld4(Kr + 16 * i), S[i]);
        const f32x4 kS = total(xs);
        f32x4 R;                                       // what is to be added to u: first what u lacks of 64 bits
        bool bad = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double x = (double)F[32 + 4 * g + r] * u[r] + (double)F[48 + 4 * g + r] * kS[r];
          u[r] = (float)x;
          R[r] = (float)(x - u[r]);
          bad |= !finite(u[r]);
        }
        if (__builtin_expect(!__any(bad), 1)) {
          // what the substitution adds is summed by itself: added to u product by product it would round at u's size sixteen times
          const float4 mf = ld4(sm + L::M + (c & 1) * C * TR + n16 * TR + 4 * g);
          R = __builtin_amdgcn_mfma_f32_16x16x4f32(mf.x, u[0] + R[0], R, 0, 0, 0);
          R = __builtin_amdgcn_mfma_f32_16x16x4f32(mf.y, u[1] + R[1], R, 0, 0, 0);
          R = __builtin_amdgcn_mfma_f32_16x16x4f32(mf.z, u[2] + R[2], R, 0, 0, 0);
          R = __builtin_amdgcn_mfma_f32_16x16x4f32(mf.w, u[3] + R[3], R, 0, 0, 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) u[r] += R[r];
        } else {
          const float* T = sm + L::T + (c & 1) * C * TR;
#pragma unroll
          for (int s = 0; s < C; ++s) {
            const float us = __shfl(u[s >> 2], (s & 3) * 16 + n16, 64);
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (tok(r) > s) u[r] -= T[tok(r) * TR + s] * us;
          }
        }
        *reinterpret_cast<float4*>(sm + L::U + ((c & 1) * L::NC + cw) * 256 + 4 * lane) = make_float4(u[0], u[1], u[2], u[3]);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) x[r] = L::CH ? u[r] : u[r] * F[16 + 4 * g + r];
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        float kt[4];
        // delta: the chunk's part by itself, so that the state is rounded once; where decays are short (mlstm, wkv) the state is the
        // smallest term and comes first
        f32x4 s = MODE == DELTA ? f32x4{0.f, 0.f, 0.f, 0.f} : S[i];
        if constexpr (L::CH) {
          const float4 k4 = ld4(KT + 16 * i * TR), de = ld4(DE + 16 * i);
          kt[0] = k4.x; kt[1] = k4.y; kt[2] = k4.z; kt[3] = k4.w;
          s[0] *= de.x; s[1] *= de.y; s[2] *= de.z; s[3] *= de.w;
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            kt[r] = K[(4 * g + r) * QR + 16 * i + n16];
            if (MODE != DELTA) s[r] *= at;
          }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[r], x[r], s, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = MODE == DELTA ? fmaf(at, S[i][r], s[r]) : s[r];
      }
      __syncthreads();
    };
    for (int c = 0; c < chunks; c += 2) {
      step(c, 0);
      step(c + 1, 1);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int ch = 16 * i + 4 * g + r;
        if (ch < dk && cok && (a.pass != 2 || last)) to[sat(ch)] = S[i][r];
      }
    if (MODE == SSM && a.pass == 1 && zb == 0 && wave == 0 && lane == 0) a.wsd[((size_t)seq * gridDim.y + seg) * H + head] = all;
    return;
  }

  // ================================================================================================ output waves
  if (MODE == SSM && a.pass == 1) {
    barriers(chunks + LEAD);
    return;
  }
  const float skip = MODE == SSM ? a.par3[head] : 0.f;
  float* yb = a.y + (size_t)row0 * H * dv + (size_t)head * dv;
  unsigned vy[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) vy[r] = (unsigned)(tok(r) * (H * dv) + colc) * 4u;
  barriers(LEAD);
  auto step = [&](int c, int st) {
    const int left = n - c * C;
    const float* Q = sm + L::Q + (c % L::QB) * L::ROWS + place(n16) * QR + 4 * g;
    const float* F = sm + L::SC + (c & 3) * 96 + 4 * g;
    const float* ST = sm + L::ST + ((c & 1) * L::NC + cw) * DP * 16 + 4 * lane;
    const double* P = reinterpret_cast<const double*>(sm + L::P) + c % 3 * C * PR;
    float u[4];
    if constexpr (MODE == DELTA) {
      const float4 u4 = ld4(sm + L::U + ((c & 1) * L::NC + cw) * 256 + 4 * lane);
      u[0] = u4.x; u[1] = u4.y; u[2] = u4.z; u[3] = u4.w;
    } else {
      take_v(c, st, u);
    }
    // P u in 64 bits (row m of these products comes out as u's token m): sixteen tokens' roundings are the result's otherwise
    const f64x2 p0 = *reinterpret_cast<const f64x2*>(P + n16 * PR + 4 * g), p1 = *reinterpret_cast<const f64x2*>(P + n16 * PR + 4 * g + 2);
    f64x4 o = {0., 0., 0., 0.};
    if (__builtin_expect(!__any(!finite(u[0]) || !finite(u[1]) || !finite(u[2]) || !finite(u[3])), 1)) {
      o = __builtin_amdgcn_mfma_f64_16x16x4f64(p0[0], u[0], o, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f64_16x16x4f64(p0[1], u[1], o, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f64_16x16x4f64(p1[0], u[2], o, 0, 0, 0);
      o = __builtin_amdgcn_mfma_f64_16x16x4f64(p1[1], u[3], o, 0, 0, 0);
    } else {
#pragma unroll
      for (int s = 0; s < C; ++s) {
        const float us = __shfl(u[s >> 2], (s & 3) * 16 + n16, 64);
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (tok(r) >= s) o[r] += P[tok(r) * PR + place(s)] * us;
      }
    }
    f32x4 os[L::NO];
    zero(os);
#pragma unroll
    for (int i = 0; i < NT; ++i) channels(os, i, ld4(Q + 16 * i), *reinterpret_cast<const f32x4*>(ST + 256 * i));
    const f32x4 qS = total(os);
    float out[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      out[r] = (float)(o[r] + (double)qS[r] * (L::CH ? 1.f : F[r]));
      if constexpr (MODE == MLSTM) out[r] *= F[32 + r];
      if constexpr (MODE == SSM) out[r] += skip * u[r];
    }
    outputs_to yc = (outputs_to)(yb + (size_t)c * C * H * dv);
    asm volatile("" : "+s"(yc));
    if (left >= C) {
      if (cok) {
#pragma unroll
        for (int r = 0; r < 4; ++r) gstore(yc + vy[r], out[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (cok && tok(r) < left) gstore(yc + vy[r], out[r]);
    }
    __syncthreads();
  };
  for (int c = 0; c < chunks; c += 2) {
    step(c, 0);
    step(c + 1, 1);
  }
}

// Between the passes of ssm in segments: per state element, walk a portion's segments in order; the workspace then holds every
// segment's incoming state.
__global__ __launch_bounds__(256) void ssm_segments_kernel(float* __restrict__ ws, const float* __restrict__ wsd, const float* __restrict__ state,
                                                           const int* __restrict__ positions, const int* __restrict__ seq_row0,
                                                           const int* __restrict__ seq_slots, int H, int per_head, int segs, int seg_rows,
                                                           int skip_rows) {
  const int seq = blockIdx.x, head = blockIdx.y, e = blockIdx.z * 256 + threadIdx.x;
  const int row0 = seq_row0[seq], n = seq_row0[seq + 1] - row0;
  if (e >= per_head || n <= skip_rows) return;
  float S = positions[row0] != 0 ? state[((size_t)seq_slots[seq] * H + head) * per_head + e] : 0.f;
  const int used = (n + seg_rows - 1) / seg_rows;
  for (int i = 0; i < used; ++i) {
    float* p = ws + (((size_t)seq * segs + i) * H + head) * per_head + e;
    const float own = i + 1 < used ? *p : 0.f;
    *p = S;
    if (i + 1 < used) S = wsd[((size_t)seq * segs + i) * H + head] * S + own;
  }
}

template <int MODE, typename TI, int NT, int COLS>
int launch_one(const ChunkArgs& a, dim3 grid, hipStream_t st) {
  using L = Lay<MODE, NT, COLS>;
  constexpr size_t lds = (size_t)L::END * 4;
  static_assert(lds <= 160 * 1024, "LDS");
  auto kernel = chunk_scan_kernel<MODE, TI, NT, COLS>;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
  }
  kernel<<<grid, 64 * L::WAVES, lds, st>>>(a);
  return 0;
}

template <int MODE, typename TI>
int launch_dims(const ChunkArgs& a, bool four, dim3 grid, hipStream_t st) {
  if (a.dk <= 64) {
    // not where its waves (thirteen, so 128 registers each) would spill: ssm, wkv, 1 prompt of 1000 and 5 decode rows, 64 heads, 219 us -> 268
    if constexpr (MODE == DELTA)
      if (four) return launch_one<MODE, TI, 4, 64>(a, grid, st);
    return launch_one<MODE, TI, 4, 32>(a, grid, st);
  }
  if (a.dk <= 128) return launch_one<MODE, TI, 8, 32>(a, grid, st);
  if constexpr (MODE != SSM) return -3;
  else return launch_one<MODE, TI, 16, 16>(a, grid, st);
}

template <int MODE>
int launch_mode(const ChunkArgs& a, int in_f32, bool four, dim3 grid, hipStream_t st) {
  return in_f32 ? launch_dims<MODE, float>(a, four, grid, st) : launch_dims<MODE, uint16_t>(a, four, grid, st);
}

}  // namespace

// Whether prompt portions of these shapes run here: key sizes of at most 128 (ssm: 256), and, but for wkv,
// rows of q and k that can be read four elements at a time.
extern "C" int dgi_chunk_scan_ok(int mode, int dk, const void* q, int q_stride, const void* k, int k_stride, int in_f32) {
  if (dk <= 0 || dk > (mode == SSM ? 256 : 128)) return 0;
  if (mode == WKV) return 1;
  const int piece = in_f32 ? 15 : 7;               // bytes of four elements, less one
  return dk % 4 == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && (((uintptr_t)q | (uintptr_t)k) & piece) == 0;
}

// mode as above (and light: par1 the decays; ssm: q = C, k = B, v = x, aux1 = dt_raw (aux_bf16), par1 a_log, par2 dt_bias, par3 d_skip).
// Needs dgi_chunk_scan_ok.  skip_rows: sequences of at most that many rows are left to another launch.  gla, light, mlstm with seg_rows: by chunk_segments.h, seg_rows
// and ws as dgi_chunk_segments_plan says, rows: of the step.  segs > 1 (ssm): portions are
// cut into segments of seg_rows rows (a multiple of 32, segs of them at least as long as the longest portion) that run side by side: each one's
// state from nothing, a short serial pass over those states, then the outputs from each segment's incoming state.  About
// twice the work, for steps whose heads leave most of the chip idle.  parts: ssm: dgi_ssm_parts_floats of workspace for chunk_parts.hip, delta:
// dgi_chunk_delta_floats for chunk_delta.hip, or null.
extern "C" int dgi_chunk_scan(float* y, int mode, const void* q, int q_stride, const void* k, int k_stride, const void* v,
                              int v_stride, int in_f32, const void* aux1, int aux1_stride, const void* aux2, int aux2_stride,
                              int aux_bf16, const float* par1, const float* par2, const float* par3, float cap, float* state,
                              float* norm, float* mx, float* norm_new, float* mx_new, const int* positions, const int* seq_row0,
                              const int* seq_slots, int n_seq, int H, int G, int dk, int dv, int skip_rows,
                              int segs, int seg_rows, float* ws, float* wsd, float* parts, int parts_chunks, int rows, hipStream_t st) {
  if (n_seq == 0) return 0;
  const int cols = dk <= 128 ? 32 : 16;            // value columns of a workgroup (or twice as many, see four_blocks)
  const bool beside = mode != SSM && seg_rows > 0;      // chunk_segments.h
  const long long nz = beside ? dgi_chunk_segments_groups(mode, dv) : (dv + cols - 1) / cols;
  if (!dgi_chunk_scan_ok(mode, dk, q, q_stride, k, k_stride, in_f32) || dv <= 0 || H <= 0 || G <= 0 || H % G) return -3;
  if (mode == MLSTM && nz > 1 && (!norm_new || !mx_new)) return -7;
  ChunkArgs a;
  a.y = y; a.q = q; a.k = k; a.v = v;
  a.q_stride = q_stride; a.k_stride = k_stride; a.v_stride = v_stride;
  a.aux1 = aux1; a.aux2 = aux2; a.aux1_stride = aux1_stride; a.aux2_stride = aux2_stride; a.aux_bf16 = aux_bf16;
  a.par1 = par1; a.par2 = par2; a.par3 = par3; a.cap = cap;
  a.state = state; a.norm = norm; a.mx = mx; a.norm_new = norm_new; a.mx_new = mx_new;
  a.positions = positions; a.seq_row0 = seq_row0; a.seq_slots = seq_slots;
  a.H = H; a.G = G; a.dk = dk; a.dv = dv; a.skip_rows = skip_rows;
  if (n_seq * nz * H > 0x3fffffff || segs > 65535 || (segs > 1 && (mode != SSM || !ws || !wsd || seg_rows <= 0))) return -3;
  a.n_seq = n_seq; a.seg_rows = seg_rows; a.ws = ws; a.wsd = wsd; a.parts = parts; a.parts_chunks = parts_chunks;
  if (beside) return dgi_chunk_segments(a, mode, in_f32, rows, ws, st);
  a.pass = segs > 1 ? 1 : 0;
  const dim3 grid((unsigned)(n_seq * nz * H), segs > 1 ? segs : 1);
  // more workgroups than compute units: possibly of four column blocks each
  const bool four = dv > 32 && n_seq <= MOST_SEQ && n_seq * nz * H > 256;
  const bool by_parts = dgi_chunk_parts_takes(mode, dk, H, G, in_f32);
  if (by_parts && segs > 1 && seg_rows % 32) return -3;
  if (a.pass) {
    int rc = by_parts ? dgi_chunk_parts(a, mode, in_f32, grid, st) : launch_dims<SSM, float>(a, false, grid, st);
    if (rc) return rc;
    ssm_segments_kernel<<<dim3(n_seq, H, (dk * dv + 255) / 256), 256, 0, st>>>(ws, wsd, state, positions, seq_row0, seq_slots, H, dk * dv, segs,
                                                                               seg_rows, skip_rows);
    a.pass = 2;
  }
  int rc = -2;
  if (by_parts) rc = dgi_chunk_parts(a, mode, in_f32, grid, st);
  else switch (mode) {
    case WKV: rc = launch_mode<WKV>(a, in_f32, four, grid, st); break;
    case DELTA: rc = parts ? dgi_chunk_delta(a, in_f32, grid, st) : launch_mode<DELTA>(a, in_f32, four, grid, st); break;
    case MLSTM: rc = in_f32 && dk > 64 ? launch_one<MLSTM, float, 8, 32>(a, grid, st) : -2; break;
    case SSM: rc = in_f32 ? launch_dims<SSM, float>(a, false, grid, st) : -2; break;
  }
  if (rc) return rc;
  DGI_CHECK_LAUNCH();
  return 0;
}
