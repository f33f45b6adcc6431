// dgi/csrc/mix/moe_group.hip — routing and experts of a step on the matrix cores (bf16), without a host round trip.
//
//   moe_router   router logits and the choice in one launch: z = h R^T with R in bf16 (products of bf16 numbers are exact
//                in fp32 and are summed in fp32), then sigmoid scores, the `top` largest (ties: lowest index), optionally
//                divided by their sum, times a factor.  A workgroup owns 16 tokens, its waves share K.
//   moe_plan     sorts the step's (token, route) pairs by expert: order[place] = pair, where[pair] = place and
//                seg[e] .. seg[e + 1] = the places of expert e; pairs of identity routes (e >= E) get no place.  One
//                workgroup per expert reads all routes, counts those of smaller experts (its first place) and lists its
//                own in pair order, so the sort is stable and needs no scan across workgroups.
//   moe_group    out[place][n] = A[row(place)] . B[e][n], n < N, for every place of every expert, with
//                  gate-up (GLU): B = gate_up [E, 2 ff, K], A = the step's hidden rows, row(place) = order[place] / top, and
//                                 out [places, ff] = act(s g, s u), s = pair_scale[order[place]] (or 1): the two projections
//                                 of an output sit in the same lane, so the activation is the product's epilogue;
//                  down:          B = down [E, N, K], A = the rows gate-up left, row(place) = place.
//
// Four kernels.  Few rows per expert (decode steps): bounded by the expert weights' bytes, so weights are read once, in whole
// 128-byte lines, straight to LDS.  Up to 64 places a tile: the workgroups share the weight rows out evenly and stream them with
// the tile's rows of A kept in registers; where those do not fit (or K is no multiple of 64), a workgroup owns 64 weight rows
// and both operands come through LDS stages.  Many rows: tiles of 128 places by 128 weight rows, K in steps of 64 through two
// LDS stages (32x32x16 products), or 256 by 256, loaded to LDS directly and multiplied by two groups of waves in turn (launch_group says which).
//
// The tile a workgroup owns is found from seg alone, so the grid is sized for the worst split of the places over the
// experts and a workgroup past the last tile leaves.  Weights are the A operand: a lane's result is four consecutive
// outputs of one place.  K must be a multiple of 8; N and the number of places are free.
#include <type_traits>

#include "../common.h"

using namespace dgi;

namespace {

constexpr int PLAN_NT = 1024;

// A workgroup per expert; a thread has `per` neighbouring pairs (a multiple of four), so that one scan over the workgroup gives every pair its
// place.  16 experts: 8192 pairs 4.3 us (a round and a scan for every 1024 pairs: 9.2), 2048 3.1 (4.2).
__global__ __launch_bounds__(PLAN_NT) void moe_plan_kernel(const int* __restrict__ idx, int P, int E, int* __restrict__ order,
                                                           int* __restrict__ where, int* __restrict__ seg) {
  __shared__ int red[2][PLAN_NT / 64];
  const int e = blockIdx.x, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int per = ((P - 1) / PLAN_NT + 4) & ~3;
  const int from = (int)min((long long)tid * per, (long long)P), to = min(from + per, P);
  const bool vec = ((uintptr_t)idx & 15) == 0;
  auto four = [&](int p, int (&r)[4]) {                // -1 past the thread's pairs
    if (vec && p + 4 <= to) {
      const int4 v = *reinterpret_cast<const int4*>(idx + p);
      r[0] = v.x; r[1] = v.y; r[2] = v.z; r[3] = v.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = p + i < to ? idx[p + i] : -1;
    }
  };
  int less = 0, mine = 0;
  for (int p = from; p < to; p += 4) {
    int r[4];
    four(p, r);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      less += (r[i] >= 0 && r[i] < e) ? 1 : 0;
      mine += r[i] == e ? 1 : 0;
    }
  }
  int upto = mine;                                     // inclusive over the lanes
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int v = __shfl_up(upto, o, 64);
    if (lane >= o) upto += v;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) less += __shfl_xor(less, o, 64);
  if (lane == 63) { red[0][w] = less; red[1][w] = upto; }
  __syncthreads();
  int at = upto - mine, all = 0;
  less = 0;
#pragma unroll
  for (int i = 0; i < PLAN_NT / 64; ++i) {
    const int c = red[1][i];
    less += red[0][i];
    at += i < w ? c : 0;
    all += c;
  }
  if (tid == 0) {
    seg[e] = less;
    if (e == E - 1) seg[E] = less + all;
  }
  at += less;                                          // the thread's first place
  if (mine == 0) return;
  for (int p = from; p < to; p += 4) {
    int r[4];
    four(p, r);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (r[i] == e) {
        order[at] = p + i;
        where[p + i] = at++;
      }
  }
}

// The m-tile `tile` of BM places: its expert and places [lo, hi); false past the last tile.  Uniform over the wave.
template <int BM, typename Seg>
__device__ __forceinline__ bool find_tile(const Seg& seg, int E, int tile, int& e, int& lo, int& hi) {
  const int lane = threadIdx.x & 63;
  int base = 0;                                        // tiles of the experts before this round's 64
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int ee = e0 + lane;
    const int s0 = ee < E ? seg(ee) : 0, s1 = ee < E ? seg(ee + 1) : 0;
    const int n = (s1 - s0 + BM - 1) / BM;
    int inc = n;                                       // inclusive prefix over the lanes
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if (lane >= o) inc += v;
    }
    const unsigned long long m = __ballot(base + inc > tile);
    if (m) {
      const int l = __ffsll(m) - 1;
      const int first = base + __shfl(inc - n, l, 64);
      e = e0 + l;
      lo = __shfl(s0, l, 64) + (tile - first) * BM;
      hi = min(__shfl(s1, l, 64), lo + BM);
      return true;
    }
    base += __shfl(inc, 63, 64);
  }
  return false;
}

// expert activation: kind 0 silu(g) * u; kind 1 the clamped sigmoid-GLU
__device__ __forceinline__ float glu_f(float g, float u, int kind, float limit, float alpha) {
  if (kind == 1) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.f + __expf(-alpha * g)) * (u + 1.f);
  }
  return g / (1.f + __expf(-g)) * u;
}

struct GroupArgs {
  const uint16_t* a;          // rows of K
  int a_stride;
  const uint16_t* b;          // [E, NB, K] (NB = N, or 2 N with the gate rows first)
  uint16_t* out;              // [places, N]
  const int* seg;
  const int* order;           // gate-up: place -> pair; down: nullptr (row = place)
  const float* pair_scale;    // gate-up: factor of g and u by pair, or nullptr
  int E, N, K, top, act;
  float limit, alpha;
  int mtiles;
  const int* idx;             // the pairs' experts where the kernel sorts them itself; to order, where and seg for the kernels that follow
  int pairs;
  int *order_out, *where_out, *seg_out;
};

__device__ __forceinline__ void load_lds16(const char* src, char* lds) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// the same for data that nothing reads again soon (nt): the chip's caches give it up first
__device__ __forceinline__ void load_lds16_once(const char* src, char* lds) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds, 16, 0, 2);
}

__device__ __forceinline__ void st_out4(uint16_t* p, const float* v, int n, bool vec) {
  if (vec && n == 4) {
    *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < n) p[i] = f32_to_bf16(v[i]);
  }
}

// ---- few rows per expert, rows of A that do not fit the registers: up to 16 MB places x 64 weight rows (GLU: 32 outputs, gate and
// up), a wave 16 of the weight rows, four stages of 64 of K.  16 experts, widths 4096 x 3584, top 4, 128 rows (64 places a tile): the
// whole feed-forward 270 us, on 128 x 128 tiles 302.
template <int MB, bool GLU>
__global__ __launch_bounds__(256) void moe_group_rows_kernel(GroupArgs g) {
  constexpr int D = 4;                                 // stages, of 64 of K each
  constexpr int CA = MB == 4 ? 2 : 1;                  // a wave's loads of rows of A per stage
  constexpr int STAGE = (4 + MB) * 2048;
  __shared__ __attribute__((aligned(16))) char lds[D * STAGE];       // [stage][weights 64 | rows 16 MB], rows of 128 bytes
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  int e, lo, hi;
  if (!find_tile<16 * MB>([&](int i) { return g.seg[i]; }, g.E, blockIdx.x % g.mtiles, e, lo, hi)) return;
  e = __builtin_amdgcn_readfirstlane(e);
  const int K = g.K;
  constexpr int NO = GLU ? 32 : 64;                    // outputs per workgroup
  const int n0 = (blockIdx.x / g.mtiles) * NO;
  // A load fills 8 LDS rows of 64 elements; piece c of LDS row r is piece c ^ (r & 7) of the row's 64 elements: reads of 8 rows spread
  // over all banks.  GLU: LDS row r holds the gate (r & 2: up) row of output 2 (r >> 2) + (r & 1), so both projections of an output
  // end up in one lane.
  const int row8 = lane >> 3, c8 = ((lane & 7) ^ row8) * 8;
  const char* B = reinterpret_cast<const char*>(g.b + (size_t)e * (GLU ? 2 : 1) * g.N * K);
  const char* bp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = 16 * w + 8 * i + row8;
    const int n = min(n0 + (GLU ? 2 * (r >> 2) + (r & 1) : r), g.N - 1) + (GLU && (r & 2) ? g.N : 0);
    bp[i] = B + (size_t)n * K * 2;
  }
  const char* ap[CA];
  int ai[CA];                                          // which 8 rows of A
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    ai[i] = (w + 4 * i) % (2 * MB);                    // MB 1: two waves load the same
    const int place = min(lo + 8 * ai[i] + row8, hi - 1);
    ap[i] = reinterpret_cast<const char*>(g.a + (size_t)(g.order ? g.order[place] / g.top : place) * g.a_stride);
  }
  // every weight tile starts at a stage of its own: workgroups in step with each other would read the same offset of rows that are
  // all the same power of two apart, from a few channels of the memory at a time
  const int steps = (K + 63) >> 6, first = blockIdx.x / g.mtiles % steps;
  auto stage = [&](int s) { return s + first < steps ? s + first : s + first - steps; };
  auto load = [&](int s) {
    char* st = lds + (s % D) * STAGE;
    const int k = min(64 * stage(s) + c8, K - 8) * 2;  // pieces past the row's end: its last one (zeros when they are used)
#pragma unroll
    for (int i = 0; i < 2; ++i) load_lds16_once(bp[i] + k, st + (2 * w + i) * 1024);
#pragma unroll
    for (int i = 0; i < CA; ++i) load_lds16(ap[i] + k, st + 8192 + ai[i] * 1024);
  };
  f32x4 acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int s, auto LEFT_) {
    constexpr int LEFT = decltype(LEFT_)::value;       // stages loaded after this one
    if constexpr (LEFT == 2) { if constexpr (CA == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); else asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); }
    else if constexpr (LEFT == 1) { if constexpr (CA == 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); else asm volatile("s_waitcnt vmcnt(3)" ::: "memory"); }
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (LEFT == 2 && s + 3 < steps) load(s + 3);       // into the stage that every wave has read before the barrier
    const char* st = lds + (s % D) * STAGE;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int at = lr * 128 + ((4 * h + lg) ^ (lr & 7)) * 16;
      u32x4 fb = *reinterpret_cast<const u32x4*>(st + w * 2048 + at), fa[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) fa[i] = *reinterpret_cast<const u32x4*>(st + 8192 + i * 2048 + at);
      if ((K & 63) && stage(s) == steps - 1) {
        const bool in = 64 * (steps - 1) + 32 * h + 8 * lg < K;
        const u32x4 zero = {0u, 0u, 0u, 0u};
        fb = in ? fb : zero;
#pragma unroll
        for (int i = 0; i < MB; ++i) fa[i] = in ? fa[i] : zero;
      }
#pragma unroll
      for (int i = 0; i < MB; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(fb), as_bf16x8(fa[i]), acc[i], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // read, before the barrier after which the stage is loaded again
  };
  load(0);
  if (steps > 1) load(1);
  if (steps > 2) load(2);
  int s = 0;
  for (; s + 2 < steps; ++s) step(s, std::integral_constant<int, 2>{});
  if (s + 1 < steps) step(s++, std::integral_constant<int, 1>{});
  step(s, std::integral_constant<int, 0>{});
  const bool vec = (g.N & 3) == 0 && ((uintptr_t)g.out & 7) == 0;
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int place = lo + 16 * i + lr;
    if (place >= hi) continue;
    uint16_t* row = g.out + (size_t)place * g.N;
    if constexpr (GLU) {
      const float ps = g.pair_scale ? g.pair_scale[g.order[place]] : 1.f;
      const int n = n0 + 8 * w + 2 * lg;
      const float a = glu_f(acc[i][0] * ps, acc[i][2] * ps, g.act, g.limit, g.alpha);
      const float b = glu_f(acc[i][1] * ps, acc[i][3] * ps, g.act, g.limit, g.alpha);
      if (vec) {
        if (n < g.N) *reinterpret_cast<uint32_t*>(row + n) = pack_bf16x2(a, b);
      } else {
        if (n < g.N) row[n] = f32_to_bf16(a);
        if (n + 1 < g.N) row[n + 1] = f32_to_bf16(b);
      }
    } else {
      const int n = n0 + 16 * w + 4 * lg;
      const float v[4] = {acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
      if (n < g.N) st_out4(row + n, v, min(4, g.N - n), vec);
    }
  }
}

// ---- few rows per expert: one workgroup per compute unit takes an equal run of the step's blocks (16 weight rows of one tile of places
// each) and streams them without a gap.  Its eight waves split K; a wave keeps its part of the tile's rows of A in registers (they
// come through the same ring of LDS stages first), so that all that moves is weights, and no wave waits for another but to add up
// the partial sums of a block.  A load takes 8 rows x 128 bytes: one compute unit reads 54 GB/s that way, but 37 with the products'
// own 16 rows x 64 bytes.  Weights are read as what nothing reads again soon (nt): 6.9 TB/s in all for reads alone, without it 6.3.
// Even shares: 64 weight rows a workgroup were 544 for 512 places.
//
// 16 experts, top 2, the whole feed-forward (16 to 20 us of it router, plan and combine), against weights straight to registers
// (64 rows a workgroup, K over its waves; 128 x 128 tiles from 4 or 12 places an expert on):
//   widths 2048 x 2048: 1 row 36 us -> 30, 8 rows 93 -> 62, 32 rows 110 -> 84 (6.0 TB/s in the products), 128 rows 130 -> 88 (a plan kernel before them)
//   widths 4096 x 3584: 1 row 70 -> 52, 8 rows 227 -> 165, 32 rows 285 -> 232 (6.5 TB/s)
constexpr int STREAM_WGS = 256;

// PLAN (gate-up of a step of at most PLAN_PAIRS pairs and PLAN_EXPERTS experts): every workgroup sorts the pairs itself, a pair per thread, where it
// would have read seg and order; the first one writes them for the kernels that follow.  A launch less: the whole feed-forward,
// 16 experts of 2048 x 2048, 1 row 31.0 us -> 28.7, 32 rows 86.0 -> 83.2.
//
// KS: stages of 64 of K per wave at the most.  K a multiple of 64.
constexpr int PLAN_PAIRS = 512, PLAN_EXPERTS = 64;

template <int MB, int KS, bool GLU, bool PLAN>
__global__ __launch_bounds__(512) void moe_group_stream_kernel(GroupArgs g) {
  constexpr int D = MB == 4 ? 5 : 6;                   // stages of 16 rows x 64 of K, 2 KB each, per wave
  // one array: with two, the compiler waits for all loads to LDS before every read of it
  constexpr int RED = 8 * D * 2048, TAB = RED + 2 * 8 * MB * 1024;
  __shared__ __attribute__((aligned(16))) char lds[TAB + (PLAN ? 4 * (PLAN_PAIRS + PLAN_EXPERTS + 1) : 0)];      // [wave][stage], partial sums [2][wave][MB][64][4], order and seg
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int K = g.K;
  constexpr int NO = GLU ? 8 : 16;                     // outputs of a block
  const int nblk = (g.N + NO - 1) / NO;
  int* const order_lds = reinterpret_cast<int*>(lds + TAB);
  int* const seg_lds = order_lds + PLAN_PAIRS;
  auto pair_of = [&](int place) { return PLAN ? order_lds[place] : g.order[place]; };
  if constexpr (PLAN) {
    // pairs of a wave's 64 threads by expert, then the experts' sums over the waves; a pair's place: those of lower experts, and of its own before it
    const int tid = threadIdx.x, r = tid < g.pairs ? g.idx[tid] : -1;
    const bool ok = r >= 0 && r < g.E;
    int* const cnt = reinterpret_cast<int*>(lds);      // [wave][expert]
    cnt[tid] = 0;
    unsigned long long same = __ballot(ok);
#pragma unroll
    for (int b = 0; b < 6; ++b) {
      const unsigned long long m = __ballot((r >> b) & 1);
      same &= (r >> b) & 1 ? m : ~m;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    __syncthreads();
    if (ok && rank == 0) cnt[w * 64 + r] = __popcll(same);
    __syncthreads();
    int all = 0, before = 0;                           // of expert `lane`, and of the waves before this one
#pragma unroll
    for (int ww = 0; ww < 8; ++ww) {
      const int c = cnt[ww * 64 + lane];
      all += c;
      before += ww < w ? c : 0;
    }
    int upto = all;                                    // inclusive over the experts
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(upto, o, 64);
      if (lane >= o) upto += v;
    }
    const int place = __shfl(upto - all + before, ok ? r : 0, 64) + rank;
    if (ok) order_lds[place] = tid;
    if (w == 0) {
      seg_lds[lane + 1] = upto;
      if (lane == 0) seg_lds[0] = 0;
    }
    if (blockIdx.x == 0) {
      if (ok) {
        g.order_out[place] = tid;
        g.where_out[tid] = place;
      }
      if (w == 0 && lane < g.E) g.seg_out[lane + 1] = upto;
      if (tid == 0) g.seg_out[0] = 0;
    }
    __syncthreads();                                   // the counts are read: the waves load over them
  }
  auto seg_of = [&](int e) { return PLAN ? seg_lds[e] : g.seg[e]; };
  // this workgroup's blocks
  int tiles = 0;
  for (int e0 = 0; e0 < g.E; e0 += 64) {
    const int ee = e0 + lane;
    tiles += ee < g.E ? (seg_of(ee + 1) - seg_of(ee) + 16 * MB - 1) / (16 * MB) : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) tiles += __shfl_xor(tiles, o, 64);
  const long long total = (long long)__builtin_amdgcn_readfirstlane(tiles) * nblk;
  int at = (int)(total * blockIdx.x / gridDim.x);
  const int end = (int)(total * (blockIdx.x + 1) / gridDim.x);
  // this wave's part of K: stages of 64
  const int stages = K >> 6, per = (stages + 7) >> 3;
  const int mine = max(0, min(per, stages - w * per));
  const int row8 = lane >> 3;
  const size_t koff = (size_t)w * per * 128 + (((lane & 7) ^ row8) << 4);
  char* const rg = lds + w * (D * 2048);
  float* const red = reinterpret_cast<float*>(lds + RED);
  auto sums = [&](int par, int ww, int i) { return reinterpret_cast<f32x4*>(red + ((par * 8 + ww) * MB + i) * 256 + 4 * lane); };
  const int rd0 = lr * 128 + ((lg ^ (lr & 7)) << 4), rd1 = lr * 128 + (((4 + lg) ^ (lr & 7)) << 4);
  int par = 0;
  while (at < end) {
    int e, lo, hi;
    find_tile<16 * MB>(seg_of, g.E, at / nblk, e, lo, hi);
    e = __builtin_amdgcn_readfirstlane(e);
    const int b0 = at % nblk, nb = min(nblk - b0, end - at);
    at += nb;
    const char* ap[MB][2];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int place = min(lo + 16 * i + 8 * j + row8, hi - 1);
        ap[i][j] = reinterpret_cast<const char*>(g.a + (size_t)(GLU ? pair_of(place) / g.top : place) * g.a_stride) + koff;
      }
    const char* B = reinterpret_cast<const char*>(g.b + (size_t)e * (GLU ? 2 : 1) * g.N * K) + koff;
    auto wrow = [&](int blk, int j) {                  // GLU: LDS row r holds the gate (r & 2: up) row of output 2 (r >> 2) + (r & 1)
      const int r = 8 * j + row8;
      const int n = min((b0 + blk) * NO + (GLU ? 2 * (r >> 2) + (r & 1) : r), g.N - 1) + (GLU && (r & 2) ? g.N : 0);
      return B + (size_t)n * K * 2;
    };
    // stages in order: the rows of A, then the blocks' weights
    const int all = (MB + nb) * mine;
    int issued = 0, l_ks = 0, l_blk = 0, l_slot = 0;
    const char *p0 = ap[0][0], *p1 = ap[0][1];
    auto load = [&]() {
      load_lds16_once(p0 + l_ks * 128, rg + l_slot * 2048);
      load_lds16_once(p1 + l_ks * 128, rg + l_slot * 2048 + 1024);
      ++issued;
      l_slot = l_slot + 1 == D ? 0 : l_slot + 1;
      if (++l_ks == mine) {
        l_ks = 0;
        ++l_blk;
        if (l_blk < MB) {
#pragma unroll
          for (int i = 1; i < MB; ++i)
            if (i == l_blk) { p0 = ap[i][0]; p1 = ap[i][1]; }
        } else {
          p0 = wrow(l_blk - MB, 0);
          p1 = wrow(l_blk - MB, 1);
        }
      }
    };
    for (int i = 0; i < D && i < all; ++i) load();
    int slot = 0;
    auto take = [&](u32x4& f0, u32x4& f1) {
      if (issued < all) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (D - 1)) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const char* st = rg + slot * 2048;
      f0 = *reinterpret_cast<const u32x4*>(st + rd0);
      f1 = *reinterpret_cast<const u32x4*>(st + rd1);
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f0), "+v"(f1)::"memory");      // read, before the stage is loaded again
      slot = slot + 1 == D ? 0 : slot + 1;
      if (issued < all) load();
    };
    u32x4 af[MB][KS][2];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        if (ks < mine) take(af[i][ks][0], af[i][ks][1]);
    for (int blk = 0; blk < nb; ++blk) {
      f32x4 acc[MB];
#pragma unroll
      for (int i = 0; i < MB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
        if (ks < mine) {
          u32x4 f0, f1;
          take(f0, f1);
#pragma unroll
          for (int i = 0; i < MB; ++i) {
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(f0), as_bf16x8(af[i][ks][0]), acc[i], 0, 0, 0);
            acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(f1), as_bf16x8(af[i][ks][1]), acc[i], 0, 0, 0);
          }
        }
#pragma unroll
      for (int i = 0; i < MB; ++i) *sums(par, w, i) = acc[i];
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        if (((blk * MB + i) & 7) != w) continue;       // uniform: one wave sums 16 places
        f32x4 t = *sums(par, 0, i);
#pragma unroll
        for (int ww = 1; ww < 8; ++ww) t += *sums(par, ww, i);
        const int place = lo + 16 * i + lr;
        if (place < hi) {
          uint16_t* row = g.out + (size_t)place * g.N;
          const bool vec = (g.N & 3) == 0 && ((uintptr_t)g.out & 7) == 0;
          if constexpr (GLU) {
            const float ps = g.pair_scale ? g.pair_scale[pair_of(place)] : 1.f;
            const int n = (b0 + blk) * NO + 2 * lg;
            const float x = glu_f(t[0] * ps, t[2] * ps, g.act, g.limit, g.alpha), y = glu_f(t[1] * ps, t[3] * ps, g.act, g.limit, g.alpha);
            if (vec) {
              if (n < g.N) *reinterpret_cast<uint32_t*>(row + n) = pack_bf16x2(x, y);
            } else {
              if (n < g.N) row[n] = f32_to_bf16(x);
              if (n + 1 < g.N) row[n + 1] = f32_to_bf16(y);
            }
          } else {
            const int n = (b0 + blk) * NO + 4 * lg;
            const float v[4] = {t[0], t[1], t[2], t[3]};
            if (n < g.N) st_out4(row + n, v, min(4, g.N - n), vec);
          }
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      par ^= 1;
    }
  }
}

// ---- many rows per expert: 128 places x 128 weight rows (GLU: 64 outputs, gate and up), 64 of K per LDS stage.
// LDS row of 64 elements = eight 16-byte chunks, chunk c of row r at c ^ (r & 7).
__device__ __forceinline__ int sw(int row, int c) { return row * 64 + ((c ^ (row & 7)) << 3); }

template <bool GLU>
__global__ __launch_bounds__(256, 2) void moe_group_tiles_kernel(GroupArgs g, int n_tiles) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[2][2][128 * 64];       // [stage][rows | weights]
  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int lr = lane & 31, hh = lane >> 5;
  // consecutive workgroups go to different XCDs: give every XCD a contiguous run of tiles, all m-tiles of a weight tile
  // in a row, so its L2 sees each weight tile once
  const int total = g.mtiles * n_tiles, chunk = (total + 7) / 8;
  const int id = (blockIdx.x & 7) * chunk + (blockIdx.x >> 3);
  if (id >= total) return;
  int e, lo, hi;
  if (!find_tile<128>([&](int i) { return g.seg[i]; }, g.E, id % g.mtiles, e, lo, hi)) return;
  constexpr int NO = GLU ? 64 : 128;
  const int n0 = (id / g.mtiles) * NO;
  const uint16_t* B = g.b + (size_t)e * (GLU ? 2 : 1) * g.N * g.K;
  // staging: thread -> chunk c of rows r0 + 32 i
  const int c = tid & 7, r0 = tid >> 3;
  const uint16_t *ap[4], *bp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + 32 * i;
    const int place = min(lo + r, hi - 1);
    ap[i] = g.a + (size_t)(g.order ? g.order[place] / g.top : place) * g.a_stride + c * 8;
    // GLU weight rows: wave column wn owns rows 64 wn .. of the stage: 32 gate rows, then the matching 32 up rows
    const int n = GLU ? n0 + 32 * (r >> 6) + (r & 31) : n0 + r;
    bp[i] = B + ((size_t)min(n, g.N - 1) + (GLU && (r & 32) ? g.N : 0)) * g.K + c * 8;
  }
  u32x4 ra[4], rb[4];
  const u32x4 zero = {0u, 0u, 0u, 0u};
  const int steps = (g.K + 63) >> 6;
  auto load = [&](int s) {
    const bool ok = s * 64 + c * 8 < g.K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ra[i] = ok ? *reinterpret_cast<const u32x4*>(ap[i] + s * 64) : zero;
      rb[i] = ok ? *reinterpret_cast<const u32x4*>(bp[i] + s * 64) : zero;
    }
  };
  auto store = [&](int st) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<u32x4*>(&lds[st][0][sw(r0 + 32 * i, c)]) = ra[i];
      *reinterpret_cast<u32x4*>(&lds[st][1][sw(r0 + 32 * i, c)]) = rb[i];
    }
  };
  const int wm = w >> 1, wn = w & 1;                   // 64 places x 64 weight rows per wave
  f32x16 acc[2][2];                                    // [places block][weights block]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  load(0);
  store(0);
  if (steps > 1) load(1);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const uint16_t* as = lds[s & 1][0];
    const uint16_t* bs = lds[s & 1][1];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      u32x4 fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[i] = *reinterpret_cast<const u32x4*>(as + sw(64 * wm + 32 * i + lr, 2 * k + hh));
        fb[i] = *reinterpret_cast<const u32x4*>(bs + sw(64 * wn + 32 * i + lr, 2 * k + hh));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_bf16x8(fb[j]), as_bf16x8(fa[i]), acc[i][j], 0, 0, 0);
    }
    if (s + 1 < steps) {
      store((s + 1) & 1);                              // the stage read in step s - 1: every wave is past that step's barrier
      if (s + 2 < steps) load(s + 2);
    }
    __syncthreads();
  }
  const bool vec = (g.N & 3) == 0 && ((uintptr_t)g.out & 7) == 0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int place = lo + 64 * wm + 32 * i + lr;
    if (place >= hi) continue;
    uint16_t* orow = g.out + (size_t)place * g.N;
    const float ps = GLU && g.pair_scale ? g.pair_scale[g.order[place]] : 1.f;
#pragma unroll
    for (int j = 0; j < (GLU ? 1 : 2); ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + (GLU ? 32 * wn : 64 * wn + 32 * j) + 8 * q + 4 * hh;
        if (n >= g.N) continue;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = GLU ? glu_f(acc[i][0][4 * q + r] * ps, acc[i][1][4 * q + r] * ps, g.act, g.limit, g.alpha) : acc[i][j][4 * q + r];
        st_out4(orow + n, v, min(4, g.N - n), vec);
      }
  }
}

// ---- very many rows per expert: up to 256 places x 256 weight rows (GLU: 128 outputs, gate and up), K in steps of 64
// through LDS, two stages of places and three of weights (all 160 KB), eight waves of 128 places x 64 weight rows.  The matrix cores
// have to be fed: loads go to LDS directly, and the two waves of a SIMD run one section apart (one reads its operands and issues
// loads while the other multiplies; every section ends at a barrier), so a SIMD's matrix core is never without work.
// What bounds experts of one tile of places is reading their weights (without its products gate-up of 222 places each took 147 us
// of 156, without the weights' loads 51): they are asked for one and a half steps ahead, half a step before, and marked as read once.
//
// An expert's n places are shared out in blocks of 64 over ceil(n / 256) tiles, and a tile of H blocks multiplies
// H blocks of 16 per wave and section, not 4: an expert of 520 places costs 3 x 3/4 tiles, not 3.
// Tiles are counted expert by expert, an expert's places fastest, and every XCD takes a contiguous run: the 32 tiles it
// works on at a time are a few tiles of places by about ten of weights of one or two experts, which meet in its L2
// (places of all experts first: each tile would read weights of its own).  Tiles left after an XCD's whole rounds of 32 are cut along their
// places where that gives its units more work: up to eight into four, up to sixteen into two (a tile takes about 0.32 + 0.17 H of a whole
// one's time, so more than sixteen gain nothing).
//
// 16 experts, K 4096, ff 3584, 512 places each: gate-up 796 us -> 406 (1184 TF/s), down 407 -> 187 (1288); 1024 places
// each 1342 and 1327 TF/s, 256 each 1028 (one tile of places: the weights come at 4.8 TB/s).  What is left is the last
// round of tiles: 520 places each are 5.25 rounds of 256 workgroups and take 513 us.  The whole feed-forward of 16 experts with two stages of
// weights, half a step ahead and nothing cut, and as it is: 2048 x 4096, 889 rows of top 4 320 us -> 279, 2000 490 -> 450; 2048 x 2048, top 2, 935 rows 147 ->
// 123, 1641 160 -> 137; 4096 x 3584, top 2, 2200 rows 582 -> 555, 4096 752 -> 752.
constexpr int WIDE = 256;
constexpr int W_TILE = WIDE * 64 * 2;                  // one operand of one stage, bytes
constexpr int W_AT = 2 * W_TILE;                       // the weights' stages behind the places'
constexpr int MORE = 24;                               // workgroups of an XCD for tiles that are cut

struct WideTile {
  int e, lo, hi, nt;                                   // expert, places [lo, hi), weight tile
  bool once;                                           // no other tile has these weights
};

// Tile blockIdx.x of the places' tiles times `ntn` weight tiles; false past the last.  Uniform over the workgroup.
__device__ __forceinline__ bool find_wide(const int* __restrict__ seg, int E, int ntn, WideTile& t) {
  const int lane = threadIdx.x & 63;
  int total = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int ee = e0 + lane;
    total += ee < E ? (seg[ee + 1] - seg[ee] + WIDE - 1) / WIDE : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) total += __shfl_xor(total, o, 64);
  total *= ntn;
  const int chunk = (total + 7) >> 3, first_id = (blockIdx.x & 7) * chunk, mine = min(chunk, total - first_id);
  if (mine <= 0) return false;
  const int left = mine & 31, most = left > 16 ? 1 : left > 8 ? 2 : 4;      // at most MORE workgroups more
  int at = blockIdx.x >> 3, parts = 1, part = 0;
  if (at >= mine - left) {
    const int k = at - (mine - left);
    parts = most;
    at = mine - left + k / most;
    part = k % most;
  }
  if (at >= mine) return false;
  const int id = first_id + at;
  int base = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int ee = e0 + lane;
    const int s0 = ee < E ? seg[ee] : 0, s1 = ee < E ? seg[ee + 1] : 0;
    const int n = (s1 - s0 + WIDE - 1) / WIDE;
    int inc = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(inc, o, 64);
      if (lane >= o) inc += v;
    }
    const unsigned long long m = __ballot((base + inc) * ntn > id);
    if (m) {
      const int l = __ffsll(m) - 1;
      const int tiles = __shfl(n, l, 64), first = base + __shfl(inc, l, 64) - tiles;
      const int a = __shfl(s0, l, 64), b = __shfl(s1, l, 64);
      const int blocks = (b - a + 63) >> 6, j = (id - first * ntn) % tiles;
      int lo = j * blocks / tiles, hi = (j + 1) * blocks / tiles;
      parts = min(parts, hi - lo);
      if (part >= parts) return false;
      t.once = tiles == 1 && parts == 1;
      const int own = hi - lo;
      hi = lo + (part + 1) * own / parts;
      lo += part * own / parts;
      t.e = e0 + l;
      t.nt = (id - first * ntn) / tiles;
      t.lo = a + 64 * lo;
      t.hi = min(b, a + 64 * hi);
      return true;
    }
    base += __shfl(inc, 63, 64);
  }
  return false;
}

// Two neighbouring blocks of 16 outputs (four of each per lane) as one 16-byte store: lane group g ends up with eight
// consecutive outputs, first block 0-7 (g 0), second 0-7 (g 1), first 8-15 (g 2), second 8-15 (g 3).
__device__ __forceinline__ void st_pair(uint16_t* row, int n0, int N, int g, const float (&a)[4], const float (&b)[4]) {
  const auto s0 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[0], a[1]), pack_bf16x2(b[0], b[1]), false, false);
  const auto s1 = __builtin_amdgcn_permlane16_swap(pack_bf16x2(a[2], a[3]), pack_bf16x2(b[2], b[3]), false, false);
  const int n = n0 + 16 * (g & 1) + 4 * (g & 2);
  if (n < N) *reinterpret_cast<uint4*>(row + n) = make_uint4(s0[0], s1[0], s0[1], s1[1]);   // N is a multiple of 8
}

// K a multiple of 128, N of 8, out at a 16-byte boundary; rows of A and the weights of an expert under 2 GiB each.
template <bool GLU>
__global__ __launch_bounds__(512) void moe_group_wide_kernel(GroupArgs g, int ntn) {
  __shared__ __attribute__((aligned(16))) char lds[5 * W_TILE];                // [stages][rows of 128 bytes]
  WideTile t;
  if (!find_wide(g.seg, g.E, ntn, t)) return;
  t.e = __builtin_amdgcn_readfirstlane(t.e);           // in scalar registers: bases and branches are
  t.nt = __builtin_amdgcn_readfirstlane(t.nt);
  t.lo = __builtin_amdgcn_readfirstlane(t.lo);
  t.hi = __builtin_amdgcn_readfirstlane(t.hi);
  t.once = __builtin_amdgcn_readfirstlane(t.once);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = w >> 2, wn = w & 3;
  const int H = (t.hi - t.lo + 63) >> 6;
  constexpr int NO = GLU ? 128 : 256;
  const int n0 = t.nt * NO;
  // Staging: slab i = 64 LDS rows.  Slabs 2 m, 2 m + 1 hold the first and second 16 H places of wave row m (rows past
  // 16 H repeat a place); slab i of the weights holds wave column i's rows (GLU: 32 gate rows, then the matching up rows).
  // Chunk c of LDS row r is chunk c ^ (r >> 1 & 7) of its 64 elements: reads of 16 rows spread over all banks.
  // Waves 0-3 load the weights, wave i slab i, eight rows a load; waves 4-7 the places, load j 16 rows of slab j / 2: loads land in
  // order, so each waits for its own kind only.
  const char* const src = wm ? reinterpret_cast<const char*>(g.a) : reinterpret_cast<const char*>(g.b + (size_t)t.e * (GLU ? 2 : 1) * g.N * g.K);
  unsigned off[8];
  if (wm) {
    int row[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) row[j] = min(t.lo + (j >> 1) * 16 * H + min(16 * wn + 8 * (j & 1) + (lane >> 3), 16 * H - 1), t.hi - 1);
    if (g.order) {                                     // all asked for before the first is divided
#pragma unroll
      for (int j = 0; j < 8; ++j) row[j] = g.order[row[j]];
#pragma unroll
      for (int j = 0; j < 8; ++j) row[j] = (int)((unsigned)row[j] / (unsigned)g.top);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) off[j] = (unsigned)row[j] * (unsigned)g.a_stride * 2u;
  } else {
    auto row = [&](int q) { return (unsigned)(min(n0 + (GLU ? 32 * wn + (q & 31) : 64 * wn + q), g.N - 1) + (GLU && q >= 32 ? g.N : 0)) * (unsigned)g.K * 2u; };
#pragma unroll
    for (int j = 0; j < 8; ++j) off[j] = row(8 * j + (lane >> 3));
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) off[j] += ((lane & 7) ^ ((4 * j + (lane >> 4)) & 7)) * 16;
  char* const la = lds + wn * 2048;
  char* const lb = lds + W_AT + wn * 8192;
  // the step's base stays in scalar registers, a lane keeps 32-bit offsets (64-bit addresses per lane spill)
  auto at = [&](int kt) {
    const char* p = src + (size_t)kt * 128;
    asm volatile("" : "+s"(p));
    return p;
  };
  auto ga = [&](int kt, int i, int st) {               // slab i of the places
    const char* p = at(kt);
#pragma unroll
    for (int u = 0; u < 2; ++u) load_lds16(p + off[2 * i + u], la + st * W_TILE + i * 8192 + u * 1024);
  };
  auto gb = [&](int kt, int st) {
    const char* p = at(kt);
    if (t.once) {
#pragma unroll
      for (int j = 0; j < 8; ++j) load_lds16_once(p + off[j], lb + st * W_TILE + j * 1024);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) load_lds16(p + off[j], lb + st * W_TILE + j * 1024);
    }
  };
  const int steps = g.K >> 6;                          // even

  const int lr = lane & 15, lg = lane >> 4, key = (lane >> 1) & 7;
  const int p0 = (lg ^ key) * 16, p1 = ((4 + lg) ^ key) * 16;
  const int abase = (wm * 128 + lr) * 128, bbase = W_AT + (wn * 64 + lr) * 128;
  f32x4 acc[2][4][4];                                  // [half][block of places][block of weights]
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto barrier = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // the K loop with HB blocks of 16 places per half.  A step is two sections per wave:
  //
  //   section  reads                        products             loads issued: weights      places
  //   0        first half, weights          first x weights      step + 2                   slabs 1, 3 of step + 1
  //   1        second half                  second x weights                                slabs 0, 2 of step + 2
  //
  // Places have landed a step after they were asked for, weights, which come from further away, a step and a half.  A slab is loaded
  // again two sections or more after its last read; what a wave waits for is visible to the others behind the barrier.
  // MODE 1, 2: the last step but one, the last.
  auto run = [&](auto HB_) {
    constexpr int HB = decltype(HB_)::value;
    bf16x8 fa[HB][2], fb[4][2];
    auto rows = [&](int st, int h) {
      const char* s = lds + st * W_TILE + abase + h * 8192;
#pragma unroll
      for (int i = 0; i < HB; ++i) {
        fa[i][0] = *reinterpret_cast<const bf16x8*>(s + i * 2048 + p0);
        fa[i][1] = *reinterpret_cast<const bf16x8*>(s + i * 2048 + p1);
      }
    };
    auto mma = [&](int h) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int i = 0; i < HB; ++i)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j][k], fa[i][k], acc[h][i][j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
    int wst = 0;                                       // the weights' stage of this step
    auto step = [&](int s, auto ST_, auto MODE_) {
      constexpr int ST = decltype(ST_)::value, MODE = decltype(MODE_)::value;
      if (wm) {
        if constexpr (MODE < 2) { ga(s + 1, 1, ST ^ 1); ga(s + 1, 3, ST ^ 1); }
      } else {
        if constexpr (MODE == 0) gb(s + 2, wst == 0 ? 2 : wst - 1);
      }
      const char* bs = lds + wst * W_TILE + bbase;
      wst = wst == 2 ? 0 : wst + 1;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        fb[j][0] = *reinterpret_cast<const bf16x8*>(bs + j * 2048 + p0);
        fb[j][1] = *reinterpret_cast<const bf16x8*>(bs + j * 2048 + p1);
      }
      rows(ST, 0);
      if (wm) {                                        // slabs 1, 3 of this step
        if constexpr (MODE < 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      barrier();
      mma(0);
      barrier();
      if (wm) {
        if constexpr (MODE == 0) { ga(s + 2, 0, ST); ga(s + 2, 2, ST); }
      }
      rows(ST, 1);
      // the weights of the next step, slabs 0, 2 of its places
      if constexpr (MODE == 0) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
      else if constexpr (MODE == 1) {
        if (wm) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      barrier();
      mma(1);
      barrier();
    };
    using Z = std::integral_constant<int, 0>;
    using O = std::integral_constant<int, 1>;
    using L = std::integral_constant<int, 2>;
    if (wm) {
      ga(0, 0, 0); ga(0, 2, 0); ga(0, 1, 0); ga(0, 3, 0); ga(1, 0, 1); ga(1, 2, 1);
    } else {
      gb(0, 0);
      gb(1, 1);
    }
    asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    barrier();
    if (wm == 1) barrier();                            // waves 4-7 run one section behind
    int s = 0;
    for (; s + 4 <= steps; s += 2) {
      step(s, Z{}, Z{});
      step(s + 1, O{}, Z{});
    }
    step(s, Z{}, O{});
    step(s + 1, O{}, L{});
    if (wm == 0) barrier();                            // the last barrier of waves 4-7
  };
  switch (H) {
    case 1: run(std::integral_constant<int, 1>{}); break;
    case 2: run(std::integral_constant<int, 2>{}); break;
    case 3: run(std::integral_constant<int, 3>{}); break;
    default: run(std::integral_constant<int, 4>{});
  }

#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int place = t.lo + (2 * wm + h) * 16 * H + 16 * i + lr;
      if (i >= H || place >= t.hi) continue;           // the four lanes of a place stay together
      uint16_t* row = g.out + (size_t)place * g.N;
      float x[4][4];
      if constexpr (GLU) {
        const float ps = g.pair_scale ? g.pair_scale[g.order[place]] : 1.f;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) x[j][r] = glu_f(acc[h][i][j][r] * ps, acc[h][i][j + 2][r] * ps, g.act, g.limit, g.alpha);
        st_pair(row, n0 + 32 * wn, g.N, lg, x[0], x[1]);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) x[j][r] = acc[h][i][j][r];
        st_pair(row, n0 + 64 * wn, g.N, lg, x[0], x[1]);
        st_pair(row, n0 + 64 * wn + 32, g.N, lg, x[2], x[3]);
      }
    }
}

template <int MB, int KS, bool GLU>
void launch_stream(const GroupArgs& g, hipStream_t s) {
  if constexpr (GLU)
    if (g.idx) {
      moe_group_stream_kernel<MB, KS, true, true><<<STREAM_WGS, 512, 0, s>>>(g);
      return;
    }
  moe_group_stream_kernel<MB, KS, GLU, false><<<STREAM_WGS, 512, 0, s>>>(g);
}

// a tile's rows of A fill half the registers of a compute unit at the most
bool streams(int bm, int K) { return bm <= 64 && K % 64 == 0 && bm * K <= 1 << 17; }

template <bool GLU>
int launch_group(GroupArgs g, int places, int rows_per_tile, hipStream_t s) {
  // worst split of the places over the experts: every non-empty expert may end in a partial tile
  const int nonempty = g.E < places ? g.E : places;
  int bm = rows_per_tile;
  if (bm == 128 || bm == WIDE) {
    // The wide tiles need 32-bit byte offsets into A and into an expert's weights, whole steps of 128 of K and 16-byte stores.  Where they can, they
    // are faster than tiles of 128 (128, 256: 16 experts of 2048 x 2048 mean 62 144 us, 117; 2048 x 4096 mean 75 256, 209; 4096 x 3584 mean 50 333, 293; 8 of
    // 4096 x 14336 mean 50 681, 614; 64 of 2048 x 1408 mean 61 292, 263; 128 of 2048 x 768 mean 81 393, 310; 16 of 1024 x 1024 mean 50 57, 52), but for small ones of
    // few steps (32 of 1024 x 512 mean 38 50, 52, mean 75 52, 51).  Up to 52 places an expert, which seldom are more than 64, streamed weights are faster
    // still (64, 256: 2048 x 2048 mean 50 101, 117, mean 62 141, 117; 2048 x 4096 mean 50 203, 213; 1024 x 2048 mean 50 44, 65; but 1024 x 1024 54, 52); of more than
    // sixteen experts one of them has more than 64 sooner, which costs those least whose weights are most of the work (mean 46, 51, 128 there, 64, 256: 32 of 1536 x 1024 92, 92, 78, 93, 97, 80; 32 of 1024 x 2048 119, 100, 106, 121, 120, 106; 32 of
    // 1536 x 1536 136, 117, 115, 137, 126, 118; 64 of 2048 x 1408 286, 233, 248, 289, 257, 253; but 32 of 2048 x 2048 226, 177, 210, 227, 182, 211).
    // The line is that of routes that are alike.  Where experts get very different numbers (the router's logits biased by normal values of spread 0.8) and the step
    // is one round of tiles of 128, small experts lose what alike ones gain (128, 256: 32 of 1024 x 512 mean 112 alike 56, 49, biased 55, 61; 16 of 1024 x 1024 mean 137
    // 57, 52, 57, 61; 8 of 1024 x 2048 mean 187 67, 61, 66, 73); from two rounds on both gain (16 of 1024 x 1024 mean 250 85, 65; 32 of 1536 x 1024 mean 112 135, 110).
    const long long a_bytes = 2ll * g.a_stride * (g.order ? (places + g.top - 1) / g.top : places);
    const long long b_bytes = 2ll * g.N * g.K * (GLU ? 2 : 1);
    if (g.K % 128 || g.N % 8 || ((uintptr_t)g.out & 15) || a_bytes >= 1ll << 31 || b_bytes >= 1ll << 31) bm = 128;
    else if (bm == 128 && places <= (g.E > 16 && (long long)g.N * g.K < 3 << 20 ? 48ll : 52ll) * g.E && (long long)g.N * g.K > 1 << 20 && streams(64, g.K)) bm = 64;
    else if ((long long)g.N * g.K > 1 << 19 || places > 64ll * g.E) bm = WIDE;
  }
  g.mtiles = places / bm + nonempty;
  const int no = (bm >= 128 ? bm : 64) / (GLU ? 2 : 1);
  const int ntn = (g.N + no - 1) / no;
  const long long blocks = (long long)g.mtiles * ntn;
  if (blocks > 0x3fffffff) return -4;
  const int padded = (int)((blocks + 7) / 8 * 8);
  if (bm == WIDE) {
    moe_group_wide_kernel<GLU><<<padded + 8 * MORE, 512, 0, s>>>(g, ntn);
  } else if (bm == 128) {
    moe_group_tiles_kernel<GLU><<<padded, 256, 0, s>>>(g, ntn);
  } else if (streams(bm, g.K)) {
    const int ks = (g.K / 64 + 7) / 8;                   // at most 16, 8, 4
    if (bm == 16) {
      if (ks <= 4) launch_stream<1, 4, GLU>(g, s);
      else if (ks <= 8) launch_stream<1, 8, GLU>(g, s);
      else launch_stream<1, 16, GLU>(g, s);
    } else if (bm == 32) {
      if (ks <= 4) launch_stream<2, 4, GLU>(g, s);
      else launch_stream<2, 8, GLU>(g, s);
    } else {
      launch_stream<4, 4, GLU>(g, s);
    }
  } else if (bm == 64) {
    moe_group_rows_kernel<4, GLU><<<(int)blocks, 256, 0, s>>>(g);
  } else if (bm == 32) {
    moe_group_rows_kernel<2, GLU><<<(int)blocks, 256, 0, s>>>(g);
  } else if (bm == 16) {
    moe_group_rows_kernel<1, GLU><<<(int)blocks, 256, 0, s>>>(g);
  } else {
    return -3;
  }
  return 0;
}

// EB blocks of 16 experts; RNW waves split K; logits meet in LDS, then wave w routes token w.  What bounds it is latency: a workgroup asks for all that a wave
// needs of 4096 channels at once, and the choice stays within the lanes' own data paths (us before, four steps
// at once and a choice by shuffles, and now: 16 experts, 1 row of 4096 6.9, 6.0; 8 of 2048 5.8, 4.8; 1097 of 4096, top 4 20.8, 12.0; 1500 of 2048 15.3, 8.0).
constexpr int RNW = 16;

// the largest of 64 lanes' values, in all of them: rows of 16 lanes turn, then four lanes are read
template <int ROWS>
__device__ __forceinline__ float largest(float v) {
  auto turned = [&](auto n) {
    const int i = __float_as_int(v);
    v = fmaxf(v, __int_as_float(__builtin_amdgcn_update_dpp(i, i, 0x120 + decltype(n)::value, 0xf, 0xf, false)));      // row_ror
  };
  turned(std::integral_constant<int, 8>{});
  turned(std::integral_constant<int, 4>{});
  turned(std::integral_constant<int, 2>{});
  turned(std::integral_constant<int, 1>{});
  float m = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
#pragma unroll
  for (int r = 1; r < ROWS; ++r) m = fmaxf(m, __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 16 * r)));
  return m;
}

template <int EB>
__global__ __launch_bounds__(64 * RNW) void moe_router_kernel(int* __restrict__ idx, float* __restrict__ wts,
                                                              const uint16_t* __restrict__ h, int h_stride,
                                                              const uint16_t* __restrict__ router, int T, int E, int K, int top,
                                                              int renorm, float wscale) {
  __shared__ __attribute__((aligned(16))) float part[RNW][EB][64][4];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int lr = lane & 15, lg = lane >> 4;
  const int t0 = blockIdx.x * 16;
  const uint16_t* hp = h + (size_t)min(t0 + lr, T - 1) * h_stride + 8 * lg;
  const uint16_t* rp[EB];
#pragma unroll
  for (int b = 0; b < EB; ++b) rp[b] = router + (size_t)min(16 * b + lr, E - 1) * K + 8 * lg;
  f32x4 acc[EB];
#pragma unroll
  for (int b = 0; b < EB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int steps = (K + 31) >> 5, per = (steps + RNW - 1) / RNW;
  const int s_hi = min(steps, (w + 1) * per);
  // U steps' operands at once; whole: none of them past the end
  auto take = [&](auto us, auto whole, int s) {
    constexpr int U = decltype(us)::value;
    u32x4 hf[U], rf[U][EB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const u32x4 zero = {0u, 0u, 0u, 0u};
      const int k = (s + u) * 32;
      const bool ok = decltype(whole)::value || (s + u < s_hi && k + 8 * lg < K);
      hf[u] = ok ? *reinterpret_cast<const u32x4*>(hp + k) : zero;
#pragma unroll
      for (int b = 0; b < EB; ++b) rf[u][b] = ok ? *reinterpret_cast<const u32x4*>(rp[b] + k) : zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int b = 0; b < EB; ++b)
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(rf[u][b]), as_bf16x8(hf[u]), acc[b], 0, 0, 0);
  };
  constexpr int U = EB == 1 ? 8 : EB == 2 ? 4 : 2;
  int s = w * per;
  if (K % 32 == 0) {
    for (; s + U <= s_hi; s += U) take(std::integral_constant<int, U>{}, std::true_type{}, s);
    if constexpr (U == 8)
      for (; s + 4 <= s_hi; s += 4) take(std::integral_constant<int, 4>{}, std::true_type{}, s);
  }
  for (; s < s_hi; s += 2) take(std::integral_constant<int, 2>{}, std::false_type{}, s);
#pragma unroll
  for (int b = 0; b < EB; ++b) *reinterpret_cast<f32x4*>(part[w][b][lane]) = acc[b];
  __syncthreads();
  // expert 16 b + 4 g + i of token j sits at part[.][b][16 g + j][i]; lane l of a wave takes expert l
  static_assert(RNW == 16, "one wave per token");
  const int j = w, t = t0 + j;
  if (t >= T) return;                                  // no barrier follows
  float z = -__builtin_inff();
  if (lane < E) {
    z = 0.f;
#pragma unroll
    for (int ww = 0; ww < RNW; ++ww) z += part[ww][lane >> 4][((lane >> 2) & 3) * 16 + j][lane & 3];
  }
  const float score = lane < E ? 1.f / (1.f + expf(-z)) : 0.f;
  // the largest score that is left; of equal ones, and where none is a number, the first lane's
  float c = lane < E && score == score ? score : -1.f, sum = 0.f;
  unsigned long long left = E < 64 ? (1ull << E) - 1 : ~0ull;
  int slot = -1;
  for (int k = 0; k < top; ++k) {
    const float best = largest<EB>(c);
    const int bi = __ffsll(__ballot(c == best) & left) - 1;
    left &= ~(1ull << bi);
    if (lane == bi) { slot = k; c = -2.f; }
    sum += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(score), bi));
  }
  if (slot >= 0) {
    idx[(size_t)t * top + slot] = lane;
    wts[(size_t)t * top + slot] = score * (renorm ? 1.f / (sum + 1e-20f) : 1.f) * wscale;
  }
}

}  // namespace

// h [T, K] bf16, router [E, K] bf16, E <= 64; K a multiple of 8
extern "C" int dgi_moe_router(int* idx, float* wts, const void* h, int h_stride, const void* router, int T, int E, int K, int top,
                              int renorm, float wscale, hipStream_t s) {
  if (T == 0) return 0;
  if (E < 1 || E > 64 || top < 1 || top > E || K < 8 || K % 8 || h_stride % 8 || (((uintptr_t)h | (uintptr_t)router) & 15)) return -2;
  const int grid = (T + 15) / 16;
#define DGI_RT(EB_)                                                                                                          \
  moe_router_kernel<EB_><<<grid, 64 * RNW, 0, s>>>(idx, wts, (const uint16_t*)h, h_stride, (const uint16_t*)router, T, E, K, top, \
                                                   renorm, wscale)
  if (E <= 16) DGI_RT(1);
  else if (E <= 32) DGI_RT(2);
  else if (E <= 48) DGI_RT(3);
  else DGI_RT(4);
#undef DGI_RT
  DGI_CHECK_LAUNCH();
  return 0;
}

extern "C" int dgi_moe_plan(const int* idx, int P, int E, int* order, int* where, int* seg, hipStream_t s) {
  if (E <= 0) return -2;
  moe_plan_kernel<<<E, PLAN_NT, 0, s>>>(idx, P, E, order, where, seg);
  DGI_CHECK_LAUNCH();
  return 0;
}

// glu: b [E, 2 N, K] and order / top (and pair_scale) map a place to its row of a; else b [E, N, K] and row = place.
// rows_per_tile: 16, 32, 64 (few rows per expert), 128 or 256.  places: the most places seg can hold.
extern "C" int dgi_moe_group(const void* a, int a_stride, const void* b, void* out, const int* seg, const int* order,
                             const float* pair_scale, int places, int E, int N, int K, int top, int glu, int act, float limit,
                             float alpha, int rows_per_tile, hipStream_t s) {
  if (places == 0 || N == 0) return 0;
  if (K <= 0 || K % 8 || a_stride % 8 || (((uintptr_t)a | (uintptr_t)b) & 15) || E <= 0 || (glu && (!order || top <= 0))) return -2;
  GroupArgs g{(const uint16_t*)a, a_stride, (const uint16_t*)b, (uint16_t*)out, seg, glu ? order : nullptr, pair_scale,
              E, N, K, top, act, limit, alpha, 0, nullptr, 0, nullptr, nullptr, nullptr};
  const int rc = glu ? launch_group<true>(g, places, rows_per_tile, s) : launch_group<false>(g, places, rows_per_tile, s);
  if (rc) return rc;
  DGI_CHECK_LAUNCH();
  return 0;
}

// moe_plan and the gate-up product: in one launch where the product's workgroups can sort the pairs themselves
extern "C" int dgi_moe_plan_group(const int* idx, int P, int* order, int* where, int* seg, const void* a, int a_stride, const void* b, void* out,
                                  const float* pair_scale, int E, int N, int K, int top, int act, float limit, float alpha, int rows_per_tile,
                                  hipStream_t s) {
  if (P == 0 || N == 0 || P > PLAN_PAIRS || E > PLAN_EXPERTS || !streams(rows_per_tile, K)) {
    const int rc = dgi_moe_plan(idx, P, E, order, where, seg, s);
    return rc ? rc : dgi_moe_group(a, a_stride, b, out, seg, order, pair_scale, P, E, N, K, top, 1, act, limit, alpha, rows_per_tile, s);
  }
  if (K <= 0 || a_stride % 8 || (((uintptr_t)a | (uintptr_t)b) & 15) || E <= 0 || top <= 0) return -2;
  if (rows_per_tile != 16 && rows_per_tile != 32 && rows_per_tile != 64) return -3;
  const GroupArgs g{(const uint16_t*)a, a_stride, (const uint16_t*)b, (uint16_t*)out, seg, order, pair_scale,
                    E, N, K, top, act, limit, alpha, 0, idx, P, order, where, seg};
  const int rc = launch_group<true>(g, P, rows_per_tile, s);
  if (rc) return rc;
  DGI_CHECK_LAUNCH();
  return 0;
}
