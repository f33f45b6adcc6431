// dgi/csrc/mix/segments.h — long portions of a recurrence cut into segments that run side by side (chunk_segments.h).
//
// A step of few heads and long portions leaves most of the chip idle: a portion's chunks go one after the other.  So a first launch makes the state of every
// segment but a portion's last one, from nothing (the first segment's from what the portion starts from), and the product of its decays; a second launch,
// the outputs', starts each segment from the sum of the states before it, each times the decays since.  The last segment's place in the workspace holds
// what the portion starts from: its place among the states is written while others may still have to read it.  Every portion is cut by its own length;
// one that stays whole has no place.
#pragma once
#include "../common.h"

namespace {

constexpr int MOST_SEGMENTS = 16;    // of a portion: the last one sums the states of all others
constexpr int FIND_INTS = 48;        // of LDS that find_segment needs

// Segments of a portion of n rows, of `each` rows (a multiple of `chunk`), about seg_rows of them: at most n / seg_rows + 1, of all portions together
// rows / seg_rows + their number; of those that are cut (n >= 5 / 3 seg_rows) at most 6 / 5 n / seg_rows.
__device__ __forceinline__ int segments_of(int n, int seg_rows, int chunk, int& each) {
  const int k = max(1, min(MOST_SEGMENTS, (n + seg_rows / 3) / seg_rows));
  each = ((n + k - 1) / k + chunk - 1) / chunk * chunk;
  return (n + each - 1) / each;
}

struct Segment {
  int seq, seg, segs, each, place;   // place: in the workspace, if segs > 1
};
// Whether no portion gains from being cut: in segments the step takes some 1.3 times the chip's time for all of its rows (share of a row: workgroups of a
// portion over those the chip has at once) and a segment's, and starts twice, 7 us or 96 rows; whole the longest portion's.
__host__ __device__ inline bool whole(int longest, int rows, float share, int seg_rows) { return longest <= 1.3f * (rows * share + seg_rows) + 96; }

// The index-th segment of all: of a step's portions of more than skip_rows rows, one after the other.  False: there are fewer.  Up to 64 sequences every wave
// looks for itself, of more each a part (734 sequences by every wave: 5 us a workgroup); then it ends with a barrier, and what was in `lds` is lost.
__device__ __forceinline__ bool find_segment(const int* seq_row0, int n_seq, int skip_rows, int seg_rows, float share, int chunk, int index, int* lds, Segment& s) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const bool parts = n_seq > 64;
  const int step = parts ? blockDim.x : 64, own_i = parts ? threadIdx.x : lane;
  int longest = 0, rows = 0;
  auto rows_of = [&](int i) {
    const int at = min(i, n_seq - 1), n = seq_row0[at + 1] - seq_row0[at];
    return i < n_seq ? n : 0;
  };
  for (int first = 0; first < n_seq; first += step) {
    const int n = rows_of(first + own_i);
    longest = max(longest, n);
    rows += n > skip_rows ? n : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    longest = max(longest, __shfl_xor(longest, o, 64));
    rows += __shfl_xor(rows, o, 64);
  }
  if (parts) {
    if (lane == 0) { lds[wave] = longest; lds[16 + wave] = rows; }
    __syncthreads();
    rows = 0;
    for (int w = 0; w < waves; ++w) {
      longest = max(longest, lds[w]);
      rows += lds[16 + w];
    }
    __syncthreads();
  }
  if (whole(longest, rows, share, seg_rows)) seg_rows = 1 << 29;
  int before = 0, placed = 0;                          // segments and places of the sequences before
  for (int first = 0; first < n_seq; first += step) {
    const int n = rows_of(first + own_i);
    int each = 0;
    const int own = n > skip_rows ? segments_of(n, seg_rows, chunk, each) : 0, cut = own > 1 ? own : 0;
    int up = own, places = cut;                        // up to and with this lane's
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(up, o, 64), y = __shfl_up(places, o, 64);
      if (lane >= o) { up += x; places += y; }
    }
    int base = before, base_placed = placed;
    if (parts) {
      if (lane == 63) { lds[wave] = up; lds[16 + wave] = places; }
      __syncthreads();
      for (int w = 0; w < waves; ++w) {
        const int x = lds[w], y = lds[16 + w];
        if (w < wave) { base += x; base_placed += y; }
        before += x;
        placed += y;
      }
    } else {
      before += __builtin_amdgcn_readlane(up, 63);
      placed += __builtin_amdgcn_readlane(places, 63);
    }
    const bool mine = index >= base + up - own && index < base + up;
    s = {first + own_i, index - (base + up - own), own, each, base_placed + places - cut + index - (base + up - own)};
    if (parts) {
      if (mine) { lds[32] = s.seq; lds[33] = s.seg; lds[34] = s.segs; lds[35] = s.each; lds[36] = s.place; }
      __syncthreads();
      if (before > index) {
        s = {lds[32], lds[33], lds[34], lds[35], lds[36]};
        __syncthreads();
        return true;
      }
    } else if (before > index) {
      const int l = __ffsll(__ballot(mine)) - 1;
      s = {__builtin_amdgcn_readlane(s.seq, l), __builtin_amdgcn_readlane(s.seg, l), __builtin_amdgcn_readlane(s.segs, l),
           __builtin_amdgcn_readlane(s.each, l), __builtin_amdgcn_readlane(s.place, l)};
      return true;
    }
  }
  return false;
}

}  // namespace
