// dgi/csrc/mix/segments.h — long portions of a recurrence cut into segments that run side by side (chunk_segments.h).
//
// A step of few heads and long portions leaves most of the chip idle: a portion's chunks go one after the other.  So a first launch makes the state of every
// segment but a portion's last one, from nothing (the first segment's from what the portion starts from), and the product of its decays; a second launch,
// the outputs', starts each segment from the sum of the states before it, each times the decays since.  The last segment's place in the workspace holds
// what the portion starts from: its place among the states is written while others may still have to read it.  Every portion is cut by its own length.
#pragma once
#include "../common.h"

namespace {

// Segments of a portion of n rows, of `each` rows (a multiple of `chunk`), about seg_rows of them: at most n / seg_rows + 1, of all portions together
// rows / seg_rows + their number.
__device__ __forceinline__ int segments_of(int n, int seg_rows, int chunk, int& each) {
  const int k = max(1, (n + seg_rows / 3) / seg_rows);
  each = ((n + k - 1) / k + chunk - 1) / chunk * chunk;
  return (n + each - 1) / each;
}

struct Segment {
  int seq, seg, segs, each;
};
// Whether no portion gains from being cut: in segments the step takes some 1.6 times the chip's time for all of its rows (share of a row: workgroups of a
// portion over those the chip has at once), and a segment's; whole the longest portion's.
__host__ __device__ inline bool whole(int longest, int rows, float share, int seg_rows) { return longest <= 1.8f * (rows * share + seg_rows); }

// The index-th segment of all: of a step's portions of more than skip_rows rows, one after the other.  False: there are fewer.
__device__ __forceinline__ bool find_segment(const int* seq_row0, int n_seq, int skip_rows, int seg_rows, float share, int chunk, int index, Segment& s) {
  const int lane = threadIdx.x & 63;
  int before = 0, longest = 0, rows = 0;
  for (int first = 0; first < n_seq; first += 64) {
    const int i = min(first + lane, n_seq - 1), n = first + lane < n_seq ? seq_row0[i + 1] - seq_row0[i] : 0;
    longest = max(longest, n);
    rows += n > skip_rows ? n : 0;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    longest = max(longest, __shfl_xor(longest, o, 64));
    rows += __shfl_xor(rows, o, 64);
  }
  if (whole(longest, rows, share, seg_rows)) seg_rows = 1 << 29;
  for (int first = 0; first < n_seq; first += 64) {
    const int i = min(first + lane, n_seq - 1), n = seq_row0[i + 1] - seq_row0[i];
    int each = 0;
    const int own = first + lane < n_seq && n > skip_rows ? segments_of(n, seg_rows, chunk, each) : 0;
    int up = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int x = __shfl_up(up, o, 64);
      if (lane >= o) up += x;
    }
    const unsigned long long past = __ballot(before + up > index);
    if (past) {
      const int l = __ffsll(past) - 1;
      s.seq = first + l;
      s.segs = __builtin_amdgcn_readlane(own, l);
      s.each = __builtin_amdgcn_readlane(each, l);
      s.seg = index - (before + __builtin_amdgcn_readlane(up, l) - s.segs);
      return true;
    }
    before += __builtin_amdgcn_readlane(up, 63);
  }
  return false;
}

}  // namespace
