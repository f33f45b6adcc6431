// dgi/csrc/prefill_attention_kernel.h — the MFMA varlen flash-attention kernel template shared by
// prefill_attention.hip (plain causal / tree mask) and mix/masked_prefill.hip (block mask +
// output gate).  See prefill_attention.hip for the tiling; MASKED adds two things:
//   * a block ("chunk") mask: a query at position p sees keys [floor(p / mask) * mask, p]
//     (mask < 0: a sliding window, keys [max(0, p + mask + 1), p], i.e. the last -mask positions)
//     (mask > 0; blocks are counted from position 0 of the sequence, so the result does not
//     depend on where a prompt was cut).  K/V tiles wholly before the first block of the
//     workgroup's rows are never loaded, tiles before a wave's first block are skipped, and a
//     tile is "interior" (no per-element mask) only when it lies inside the block of the
//     wave's last row;
//   * an output gate: out *= sigmoid(gate) element by element, or one gate per head (gate_heads), in the
//     epilogue (fp32).
// With MASKED, softcap > 0 caps the scaled (and biased) score s at softcap * tanh(s / softcap), and sinks
// (one fp32 logit per head) adds exp(sink) to the softmax denominator in the epilogue.
// head_scale (one fp32 factor per head, any sign) multiplies the scaled score before the cap.
// HDV: value size where it differs from the key size HD.  PAD: the heads have dk <= HD and dv <= HDV dims (multiples of 8):
// fragments beyond them repeat a valid chunk, whose products are with a zero query chunk or are never stored.
// BIAS adds a learned distance bias to the scores before the mask: dist_bias[min(p - j, n_dist - 1)][head]
// (fp32, natural score units; the kernel works in raw q.k units, hence inv_scale = 1 / scale).
#pragma once
#include "common.h"

namespace dgi {
namespace prefill {


// Where the 16-byte chunk `ch` of an LDS row lies in it (and which chunk lies at `ch`), and its element offset.
// HD=128 (256-B rows): K chunk ^ (row & 15) — 16 consecutive rows at one chunk
// hit 16 distinct slots (ds_read_b128); V chunk ^ ((row & 3) << 2) for the
// transposed reads.  HD=64 (128-B rows, two rows per 64-bank line): row & 1
// already picks the bank half, so K XORs (row >> 1) & 7 and V shifts rows
// 2-3 of each 4-row block by 4 chunks.
template <int HD>
__device__ __forceinline__ int k_slot(int row, int ch) {
  return HD == 128 ? ch ^ (row & 15) : ch ^ ((row >> 1) & 7);
}
template <int HD>
__device__ __forceinline__ int v_slot(int row, int ch) {
  return HD == 128 ? ch ^ ((row & 3) << 2) : ch ^ (((row >> 1) & 1) << 2);
}
template <int HD>
__device__ __forceinline__ int k_off(int row, int ch) { return row * HD + (k_slot<HD>(row, ch) << 3); }
template <int HD>
__device__ __forceinline__ int v_off(int row, int ch) { return row * HD + (v_slot<HD>(row, ch) << 3); }

// One 16-byte chunk a lane from memory to LDS (`at` + 16 lane)
typedef __attribute__((address_space(3))) char* lds_ptr;
__device__ __forceinline__ void load_chunk(const char* src, lds_ptr at) {
  __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)at, 16, 0, 0);
}
// The same from `lane_at` bytes into the rows of a page; OFF bytes on on both sides.
template <int OFF>
__device__ __forceinline__ void load_chunk(__amdgpu_buffer_rsrc_t rows, int lane_at, lds_ptr at) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rows, (__attribute__((address_space(3))) void*)at, 16, lane_at, 0, OFF, 0);
}

template <int V> struct ic { static constexpr int value = V; };

template <int A, int B, class F>
__device__ __forceinline__ void each(F f) {
  if constexpr (A < B) {
    f(ic<A>{});
    each<A + 1, B>(f);
  }
}

constexpr int KT = 64;  // keys per tile

// 1 / (1 + e^-g) of a bf16 gate.  log2(e) in 16 bits times the gate is exact, and what both it and the quotient lack is put right at once.  Relative error over all bf16
// values up to 30, root mean square and largest, in 2^-24: 0.65, 2.0; expf and a division 0.66, 2.0; the hardware's exp of a rounded product and its reciprocal 2.5, 27.
// Infinities and NaN as expf and a division give them.
__device__ __forceinline__ float gate_factor(float g) {
  constexpr float HI = 1.44268798828125f, LO = 1.4426950408889634 - 1.44268798828125;
  const float x = g > 100.f ? 100.f : g;
  const float e = __builtin_amdgcn_exp2f(x * -HI), d = 1.f + e, r = __builtin_amdgcn_rcpf(d);
  const float rest = fmaf(-e * (x * (-LO * 0.6931471805599453f)), r, fmaf(-d, r, 1.f));      // what 1 - (1 + e^-g) r is
  return __builtin_amdgcn_div_fixupf(fmaf(rest, r, r), d, 1.f);
}

// NW waves x 32 query rows per workgroup (one K/V tile staging shared by all of them):
// NW = 4 -> 128-row tiles, 2 workgroups per CU; NW = 8 -> 256-row tiles, 1 per CU
// (same 2 waves per SIMD, half the K/V staging per query row).
//
// Two LDS stages: a tile goes from memory to one of them (no registers between) while the tile in the other is multiplied,
// one barrier per 64 keys.  One prompt of 8192 rows, 32 heads on 8 of 128 dims: 576 us -> 506 (1086 TF/s), 64 dims and 4096
// rows 107 -> 90, a tile 3830 cycles a SIMD against 4700, of which its products take 2048.  What the staging registers, the
// block ids' scalar loads, the addresses of each load and read and the copies around the mask cost went into it: 256
// registers with every operand waited for as it was read, now 214 with reads a product or more ahead, 185 -> 143 vector and
// 88 -> 50 scalar instructions a tile.  What is left: the clock falls to 1.85 GHz under it, a wave waits some 600 cycles a
// tile while the loads of all four are issued, and one wave's products and exponentials overlap the other's in part.
template <int HD, int NW, bool MASKED = false, bool BIAS = false, int HDV = HD, bool PAD = false>
__global__ __launch_bounds__(NW * 64, NW == 4 ? 2 : 1) void prefill_attn_kernel(
    const uint16_t* __restrict__ q, int q_stride, const uint16_t* __restrict__ k_cache,
    const uint16_t* __restrict__ v_cache, const int* __restrict__ block_tables, int bt_stride,
    const int* __restrict__ cu_seqlens_q, const int* __restrict__ context_lens,
    const int* __restrict__ tiles, uint16_t* __restrict__ out, int out_stride, int nh, int nkv,
    int bs_log2, float scale_log2, const unsigned long long* __restrict__ tree_mask, int tree_n,
    int mask = 0, const uint16_t* __restrict__ gate = nullptr, int gate_stride = 0,
    const float* __restrict__ dist_bias = nullptr, int n_dist = 0, float inv_scale = 0.f,
    float softcap = 0.f, const float* __restrict__ sinks = nullptr, const float* __restrict__ head_scale = nullptr,
    int dk_ = HD, int dv_ = HDV, int gate_heads = 0) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * KT * (HD + HDV)];
  const int dk = PAD ? dk_ : HD, dv = PAD ? dv_ : HDV;

  // Workgroup -> (tile, head): all heads of a tile before the next tile, so that in a list with the heaviest tiles first no
  // head's heavy tiles start when the others are nearly done, and neighbours take different key/value heads: XCD x (workgroup
  // x mod 8) works on the heads of key/value head x mod nkv, whose keys and values stay in its L2.  One prompt of 8192 rows,
  // 32 heads on 8, traced: head by head, the last head's heavy tiles ran almost alone, 969 us; so 739.
  const int hx = blockIdx.x % nh, tile = blockIdx.x / nh;
  const int b = tiles[2 * tile];
  const int t0 = tiles[2 * tile + 1];  // first query row (within seq) of this tile
  const int kvh = hx % nkv;
  const int head = kvh * (nh / nkv) + hx / nkv;
  // per-head score factor: folded into the scale; the softmax below takes maxima of raw scores, so a negative
  // factor flips the raw scores' sign (the query's; a distance bias never comes with factors), and a factor of zero stays above it (masked keys are -inf)
  bool flip = false;
  if (MASKED && head_scale) {
    scale_log2 *= head_scale[head];
    flip = scale_log2 < 0.f;
    scale_log2 = fmaxf(fabsf(scale_log2), 1e-30f);
  }
  const int q0 = cu_seqlens_q[b];
  const int qlen = cu_seqlens_q[b + 1] - q0;
  const int ctx = context_lens[b];
  const int pos_base = ctx - qlen;  // absolute position of query row 0
  const int bs = 1 << bs_log2;
  const int* bt = block_tables + (size_t)b * bt_stride;

  const int tid = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);      // in a scalar register: what depends on the wave alone is
  const int lane = tid & 63;
  const int lr = lane & 31;
  const int hh = lane >> 5;

  const int my_row = t0 + 32 * w + lr;  // query row within the sequence
  const bool row_valid = my_row < qlen;
  const int my_pos = pos_base + my_row;
  const int tree_first = qlen - tree_n;  // rows >= tree_first use the tree mask
  unsigned long long tmask = 0;
  const bool is_tree = tree_mask != nullptr && row_valid && my_row >= tree_first;
  if (is_tree) tmask = tree_mask[(size_t)b * 64 + (my_row - tree_first)];
  const int tree_key0 = pos_base + tree_first;  // key index of tree node 0

  constexpr int NS = HD / 16;   // k-steps of S^T = K Q^T
  constexpr int ND = HDV / 32;  // 32-dim blocks of O^T
  constexpr int CH = HD / 8, CHV = HDV / 8;    // 16-byte chunks per K / V row
  // Q fragments (B operand): lane holds Q[row lr][16 s + 8 hh + j]
  u32x4 qf[NS];
  {
    const uint16_t* qp = q + (size_t)(q0 + (row_valid ? my_row : 0)) * q_stride + head * dk;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      qf[s] = row_valid && (!PAD || 16 * s + 8 * hh < dk) ? *reinterpret_cast<const u32x4*>(qp + 16 * s + 8 * hh) : u32x4{0, 0, 0, 0};
    // Q lands before any K/V load is issued.  Without this wait the compiler's waitcnt pass
    // merges "Q pending" from the preheader into the loop header and, to reach the older Q
    // loads, emits vmcnt(0) before the first QK^T MFMA of EVERY tile — which also waits for
    // the next tile's loads issued a few instructions earlier: one full HBM round trip
    // per tile and no load/compute overlap at all.
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0), expcnt / lgkmcnt untouched (gfx9 encoding)
    if (MASKED && flip) {
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[s] ^= 0x80008000u;
    }
  }

  const int last_row = min(t0 + 32 * NW, qlen) - 1;
  const int kv_end = min(ctx, pos_base + last_row + 1);
  // block mask: first visible key of a position; the workgroup starts at the 64-key tile
  // holding the first block of its first row
  // (mask < 0: a sliding window of -mask positions instead, first key max(0, p + mask + 1))
  auto first_key = [&](int p) {
    if (!MASKED || mask == 0) return 0;
    return mask > 0 ? (p / mask) * mask : max(0, p + mask + 1);
  };
  const int kv_begin = MASKED ? (first_key(pos_base + t0) / KT) * KT : 0;
  const int my_first = first_key(my_pos);

  // what the softmax multiplies the scores that it gets by
  const float cap_log2 = MASKED && softcap > 0.f ? softcap * 1.4426950408889634f : 0.f;
  const float soft_scale = MASKED && softcap > 0.f ? 2.f * cap_log2 : scale_log2;
  float m_run = -1e30f, l_run = 0.f;
  f32x16 o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;

  const size_t head_stride = (size_t)bs * dk, v_head_stride = (size_t)bs * dv;
  // offset of chunk ch inside a key / value row
  auto kch = [&](int ch) { return PAD ? min(ch * 8, dk - 8) : ch * 8; };
  auto vch = [&](int ch) { return PAD ? min(ch * 8, dv - 8) : ch * 8; };
  // RW rows of a tile are staged by each wave, 1 KB (64 / CH rows) a load, one behind the other in LDS; in pages of at least RW tokens (the
  // engine's have 16) they lie in one page, one behind the other there too, so that its loads share one id and one address and
  // differ in their instruction's offset.  The swizzle is in which chunk of its row a lane loads.
  constexpr int RW = KT / NW;                                      // rows of a tile a wave stages
  constexpr int NP = RW * CH / 64, NPV = RW * CHV / 64;            // its loads of keys and of values
  static_assert(16 % RW == 0 && NP >= 1 && NPV >= 1, "a wave's rows lie in one page");
  const int row0 = w * RW;
  const bool whole_rows = bs >= RW;
  int k_at[NP], v_at[PAD ? NPV : 1];       // bytes from the wave's first row (whole rows: less the load's offset)
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int row = p * (64 / CH) + lane / CH;
    k_at[p] = 2 * (row * dk + kch(k_slot<HD>(row0 + row, lane % CH))) - (PAD ? 0 : 1024 * p);
  }
#pragma unroll
  for (int p = 0; p < (PAD ? NPV : 1); ++p) {
    const int row = p * (64 / CHV) + lane / CHV;
    v_at[p] = 2 * (row * dv + vch(v_slot<HDV>(row0 + row, lane % CHV))) - (PAD ? 0 : 1024 * p);
  }
  int none = 0;
  asm("" : "+v"(none));                   // a vector load: a scalar one's wait would be one for all reads of LDS
  // the page of the wave's rows of a tile, or of this lane's row of them where they have several
  auto read_id = [&](int kb0) __attribute__((always_inline)) {
    return whole_rows ? bt[(min(kb0 + row0, kv_end - 1) >> bs_log2) + none] : bt[min(kb0 + row0 + lane % RW, kv_end - 1) >> bs_log2];
  };
  auto full = [&](int kb0) __attribute__((always_inline)) { return whole_rows && kb0 + KT <= kv_end; };
  // rows of the page from a key on, and load l of the NP + NPV of a full tile
  __amdgpu_buffer_rsrc_t k_rows, v_rows;
  auto at_page = [&](int id, int key) __attribute__((always_inline)) {
    const size_t blk = (size_t)__builtin_amdgcn_readfirstlane(id) * nkv + kvh;
    k_rows = __builtin_amdgcn_make_buffer_rsrc((void*)(k_cache + blk * head_stride + (key & (bs - 1)) * dk), 0, RW * dk * 2, 0x00027000);
    v_rows = __builtin_amdgcn_make_buffer_rsrc((void*)(v_cache + blk * v_head_stride + (key & (bs - 1)) * dv), 0, RW * dv * 2, 0x00027000);
  };
  auto load = [&](auto l_, int stage) __attribute__((always_inline)) {
    constexpr int l = decltype(l_)::value, p = l < NP ? l : l - NP;
    const lds_ptr at = (lds_ptr)(lds + stage * KT * (HD + HDV) + (l < NP ? row0 * HD : KT * HD + row0 * HDV));
    if constexpr (PAD) load_chunk<0>(l < NP ? k_rows : v_rows, l < NP ? k_at[l < NP ? p : 0] : v_at[l < NP ? 0 : p], at + 1024 * p);
    else load_chunk<1024 * p>(l < NP ? k_rows : v_rows, l < NP ? k_at[p] : v_at[0], at);
  };
  // A tile that ends early, or whose rows have several pages: each lane finds its own, no row is after the last key.  The ids
  // are there by now: read here, each load would wait for its id and so for all loads before it (32 heads of 128, pages of
  // 32: 8192 rows 798 us, so 511; 3000 rows behind 5000 636, so 338; pages of 8: 816, 568 and 654, 355).
  auto load_part = [&](int kb0, int stage, int id) __attribute__((always_inline)) {
    const lds_ptr kl = (lds_ptr)(lds + stage * KT * (HD + HDV) + row0 * HD), vl = (lds_ptr)(lds + stage * KT * (HD + HDV) + KT * HD + row0 * HDV);
    const int first = min(kb0 + row0, kv_end - 1), last = kv_end - 1 - first;
    int part = lane;
    asm volatile("" : "+v"(part));      // computed here: kept from before the loop its addresses would cost registers
    if (whole_rows) {
      at_page(id, first);
#pragma unroll 1
      for (int p = 0; p < NP; ++p) {
        const int row = p * (64 / CH) + part / CH;
        load_chunk<0>(k_rows, 2 * (min(row, last) * dk + kch(k_slot<HD>(row0 + row, part % CH))), kl + p * 1024);
      }
#pragma unroll 1
      for (int p = 0; p < NPV; ++p) {
        const int row = p * (64 / CHV) + part / CHV;
        load_chunk<0>(v_rows, 2 * (min(row, last) * dv + vch(v_slot<HDV>(row0 + row, part % CHV))), vl + p * 1024);
      }
      return;
    }
    // rows of keys and of values of load p: the page and the row in it
    auto at = [&](int row) __attribute__((always_inline)) { return (size_t)__shfl(id, row, 64) * nkv + kvh; };
    auto in = [&](int row) __attribute__((always_inline)) { return min(kb0 + row0 + row, kv_end - 1) & (bs - 1); };
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const int row = p * (64 / CH) + part / CH;
      load_chunk((const char*)(k_cache + at(row) * head_stride + (size_t)in(row) * dk + kch(k_slot<HD>(row0 + row, part % CH))), kl + p * 1024);
    }
#pragma unroll
    for (int p = 0; p < NPV; ++p) {
      const int row = p * (64 / CHV) + part / CHV;
      load_chunk((const char*)(v_cache + at(row) * v_head_stride + (size_t)in(row) * dv + vch(v_slot<HDV>(row0 + row, part % CHV))), vl + p * 1024);
    }
  };
  int id = 0;
  if (kv_end > kv_begin) {
    id = read_id(kv_begin);
    if (full(kv_begin)) {
      at_page(id, kv_begin + row0);
      each<0, NP + NPV>([&](auto l) __attribute__((always_inline)) { load(l, 0); });
    } else load_part(kv_begin, 0, id);
    id = read_id(kv_begin + KT);
  }
  // LDS addresses of this lane's operands in stage 0: keys lr (the second 32 are 64 HD bytes on), dims 16 s + 8 hh ..; values
  // of dims 32 d .., keys 4 hh + tq (16 j + 8 more are 32 HDV j and 16 HDV bytes on)
  typedef __attribute__((address_space(3))) const char* lds_at;
  lds_at ka[NS], va[ND];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    ka[s] = (lds_at)(lds + k_off<HD>(lr, 2 * s + hh));
    asm("" : "+v"(ka[s]));
  }
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    const int col = 32 * d + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
    va[d] = (lds_at)(lds + KT * HD + v_off<HDV>(4 * hh + ((lane & 15) >> 2), col >> 3) + (col & 7));
    asm("" : "+v"(va[d]));
  }
  // last key this wave can see (causal); tiles beyond it are skipped
  const int wave_last_pos = pos_base + min(t0 + 32 * w + 31, qlen - 1);
  // keys <= wave_first_pos are visible to every row of the wave
  const int wave_first_pos = pos_base + t0 + 32 * w;
  const bool wave_tree = tree_mask != nullptr && (t0 + 32 * w + 31 >= tree_first);
  const bool wave_rows = t0 + 32 * w < qlen;
  const int wave_min_first = first_key(wave_first_pos);   // first block start among this wave's rows
  const int wave_max_first = first_key(wave_last_pos);    // last block start among them
  auto step = [&](int kb0, auto stage_) __attribute__((always_inline)) {
    constexpr int stage = decltype(stage_)::value, at = stage * KT * (HD + HDV) * 2;
    // this stage holds the tile once every wave's loads have landed; every wave has finished with the tile before, whose
    // stage the next tile goes to
    __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0)
    __syncthreads();
    const bool next = full(kb0 + KT);
    if (next) {
      at_page(id, kb0 + KT + row0);
      each<0, NP + NPV>([&](auto l) __attribute__((always_inline)) { load(l, 1 - stage); });
    } else if (kb0 + KT < kv_end) load_part(kb0 + KT, 1 - stage, id);
    id = read_id(kb0 + 2 * KT);
    if (kb0 > wave_last_pos || !wave_rows || (MASKED && kb0 + KT <= wave_min_first)) return;
    // ---- S^T = K Q^T for two 32-key blocks: the first block's operands are all under way before its products, the
    // second's come between them, the first values between the second's (left to itself the compiler waits out an LDS read
    // for every product or two, hence the fences).  The values' first read waits for the next tile's loads, too: the
    // compiler cannot tell the stages apart.  Read after the maxima instead 546 us for 538; all of them before the
    // exponentials, the loads among the products after them, 860 (64 more registers, they spill); the softmax in blocks of
    // 32 keys, each beside the other's products, 547 for 542.
    f32x16 sc[2];
    // operands of V^T: keys 32 (j >> 1) + 16 (j & 1) .. + 15 of the tile, dims 32 d ..
    auto read_v = [&](int j, int d) __attribute__((always_inline)) {
      const short4v lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(va[d] + (at + 32 * HDV * j)));
      const short4v hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(va[d] + (at + 32 * HDV * j + 16 * HDV)));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto read_k = [&](int kb, int s) __attribute__((always_inline)) {
      return *(const __attribute__((address_space(3))) bf16x8*)(ka[s] + (at + 64 * HD * kb));
    };
    typedef short short8v __attribute__((ext_vector_type(8)));
    short8v vf[2][ND];
    {
      bf16x8 kf[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) kf[s] = read_k(0, s);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[kb][r] = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s], as_bf16x8(qf[s]), sc[kb], 0, 0, 0);
          if (kb == 0) kf[s] = read_k(1, s);
          else {
#pragma unroll
            for (int f = s * 2 * ND / NS; f < (s + 1) * 2 * ND / NS; ++f) vf[f / ND][f % ND] = read_v(f / ND, f % ND);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if constexpr (BIAS) {
      // distance bias in raw score units (bias / scale): one table row per distance, the last row for
      // everything farther — a tile wholly beyond it for every row of the wave adds one constant
      if (wave_first_pos - (kb0 + KT - 1) >= n_dist - 1) {
        const float bl = dist_bias[(size_t)(n_dist - 1) * nh + head] * inv_scale;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) sc[kb][r] += bl;
      } else {
        const int keyb = kb0 + 4 * hh;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int d = my_pos - (keyb + 32 * kb + (r & 3) + 8 * (r >> 2));
            sc[kb][r] += dist_bias[(size_t)min(max(d, 0), n_dist - 1) * nh + head] * inv_scale;
          }
      }
    }
    if (MASKED && softcap > 0.f) {
      // soft cap of the scaled score: tanh(x) = 1 - 2 / (exp(2x) + 1) with the hardware exp2 / rcp.  What the softmax takes is -1 / (exp(2x) + 1) by
      // twice the cap (soft_scale): the capped scores less the cap, which it does not see (that step with a cap 192 us, so 160; a polynomial for
      // scores well below the cap took as long as exp and rcp: the multiplies and adds between them are what counts).
      const float to_arg = scale_log2 * 2.f / softcap;             // raw -> 2 x log2(e)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[kb][r] = __builtin_amdgcn_rcpf(-1.f - __builtin_amdgcn_exp2f(sc[kb][r] * to_arg));
    }
    // ---- online softmax; lane owns query lr, keys kb0 + 32kb + (r&3) + 8(r>>2) + 4hh.
    // Interior tiles (every key visible to every row of this wave, no tree rows) skip the mask.
    const bool interior = (kb0 + KT <= kv_end) && (kb0 + KT - 1 <= wave_first_pos) && !wave_tree &&
                          (!MASKED || kb0 >= wave_max_first);
    if (!interior) {
      // masked keys -> -inf in raw score units.  -inf, not a large finite value: a lane whose keys are all masked must get
      // max -inf (no rescale) and P = 2^(-inf) = 0, whatever the scale.  Bit i of `see`: this lane's row sees key key0 + i.
      const int key0 = kb0 + 4 * hh;
      const int lim = (row_valid ? min(my_pos, kv_end - 1) : -1) - key0;    // last visible key
      unsigned long long see = lim < 0 ? 0 : lim >= 63 ? ~0ull : (2ull << lim) - 1;
      if (MASKED) {
        const int from = my_first - key0;
        see = from <= 0 ? see : from > 63 ? 0 : see & (~0ull << from);
      }
      if (is_tree) {
        const int t = tree_key0 - key0;                                       // keys before t are seen, after it as the mask says
        see &= t >= 64 ? ~0ull : t >= 0 ? (tmask << t) | ((1ull << t) - 1) : t > -64 ? tmask >> -t : 0ull;
      }
      const unsigned see_lo = (unsigned)see, see_hi = (unsigned)(see >> 32);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[kb][r] = (kb ? see_hi : see_lo) >> ((r & 3) + 8 * (r >> 2)) & 1 ? sc[kb][r] : -__builtin_inff();
    }
    float mx = -1e30f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sc[kb][r]);
    mx *= soft_scale;
    // deferred max: rescale O / l only when the running max grows by > 2^8, so
    // most tiles skip the 64 O multiplies (P stays <= 256, safe in f32 / bf16) and the exchange with the half of the wave
    // that holds the query's other keys
    if (__any(mx > m_run + 8.f)) {
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float m_new = fmaxf(m_run, mx);
      const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int d = 0; d < ND; ++d) o[d] *= alpha;
      m_run = m_new;
    }
    // P = 2^(s * scale_log2 - m) (raw v_exp_f32: arguments <= 8, masked scores underflow to 0; four partial row sums instead
    // of one 32-long dependent add chain) and O^T += V^T P^T.  The second block's exponentials run between the first
    // block's products: each takes about as long as the other.  Values are read two groups of products ahead.
    float ps[4];
    u32x4 pf;
    auto weight = [&](int kb, int r) __attribute__((always_inline)) {
      sc[kb][r] = __builtin_amdgcn_exp2f(sc[kb][r] * soft_scale - m_run);
      ps[r & 3] = kb == 0 && r < 4 ? sc[kb][r] : ps[r & 3] + sc[kb][r];
    };
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      weight(0, r);
    }
    __builtin_amdgcn_sched_barrier(0);
    each<0, 4 * ND>([&](auto i_) __attribute__((always_inline)) {
      constexpr int i = decltype(i_)::value, j = i / ND, d = i % ND;
      if constexpr (d == 0) {
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) pf[jj] = pack_bf16x2(sc[j >> 1][8 * (j & 1) + 2 * jj], sc[j >> 1][8 * (j & 1) + 2 * jj + 1]);
      }
      o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vf[j & 1][d]), as_bf16x8(pf), o[d], 0, 0, 0);
      if constexpr (j < 2) {
        vf[j][d] = read_v(j + 2, d);
#pragma unroll
        for (int r = i * 8 / ND; r < (i + 1) * 8 / ND; ++r) weight(1, r);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    l_run += (ps[0] + ps[1]) + (ps[2] + ps[3]);      // this lane's keys; the halves of the wave meet after the loop
  };
  for (int kb0 = kv_begin; kb0 < kv_end; kb0 += 2 * KT) {
    step(kb0, ic<0>{});
    if (kb0 + KT < kv_end) step(kb0 + KT, ic<1>{});
  }
  // The gates of a row's elements are all asked for at once (64 heads of 128 dims, 7 prompts of 3637 rows in all behind 500 tokens each, blocks of 1024, us: one by one with expf and
  // a division 166, at once 155, so 144; without a gate 124).
  const bool gated = MASKED && gate && !gate_heads;
  uint2 gates[ND][4];
  if (gated) {
    const uint16_t* gp = gate + (size_t)(q0 + (row_valid ? my_row : 0)) * gate_stride + head * dv;
#pragma unroll
    for (int d = 0; d < ND; ++d)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int dim = 32 * d + 8 * rr + 4 * hh;
        gates[d][rr] = *reinterpret_cast<const uint2*>(gp + (PAD ? min(dim, dv - 4) : dim));
      }
  }
  l_run += __shfl_xor(l_run, 32, 64);

  if (!row_valid) return;
  // sink: denominator only (m_run lacks the cap)
  if (MASKED && sinks) l_run += __builtin_amdgcn_exp2f(sinks[head] * 1.4426950408889634f - (m_run + cap_log2));
  float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  if (MASKED && gate && gate_heads) inv *= 1.f / (1.f + expf(-bf16_to_f32(gate[(size_t)(q0 + my_row) * gate_stride + head])));
  uint16_t* op = out + (size_t)(q0 + my_row) * out_stride + head * dv;
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int dim = 32 * d + 8 * rr + 4 * hh;
      if (PAD && dim >= dv) continue;
      float ov[4] = {o[d][4 * rr] * inv, o[d][4 * rr + 1] * inv, o[d][4 * rr + 2] * inv, o[d][4 * rr + 3] * inv};
      if (gated) {
        const uint2 g = gates[d][rr];
        const float gf[4] = {__uint_as_float(g.x << 16), __uint_as_float(g.x & 0xffff0000u),
                             __uint_as_float(g.y << 16), __uint_as_float(g.y & 0xffff0000u)};
#pragma unroll
        for (int j = 0; j < 4; ++j) ov[j] *= gate_factor(gf[j]);
      }
      uint2 v;
      v.x = pack_bf16x2(ov[0], ov[1]);
      v.y = pack_bf16x2(ov[2], ov[3]);
      *reinterpret_cast<uint2*>(op + dim) = v;
    }
}



}  // namespace prefill
}  // namespace dgi
