// dgi/csrc/mix/chunk_segments.hip — the plan of segments and the launches of chunk_segments.h.
#include <algorithm>
#include "chunk_split.h"
#include "segments.h"

constexpr int GLA = 3;
int dgi_segments_mlstm(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st);
int dgi_segments_light(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st);
int dgi_segments_gla(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st);

// blocks of 16 columns of a workgroup (the matrix memory's thirteen waves would have 128 registers each, and spill)
static int wide(int mode, int dv) { return dv <= 64 || mode == MLSTM ? 4 : 8; }
// workgroups of a head: the matrix memory's normaliser is staged if there are several
int dgi_chunk_segments_groups(int mode, int dv) { return (dv + 16 * wide(mode, dv) - 1) / (16 * wide(mode, dv)); }

static long state_floats(int mode, int dk, int dv) {
  return (dgi_chunk_segments_groups(mode, dv) * wide(mode, dv) + (mode == MLSTM ? 1 : 0)) * (dk <= 64 ? 4 : 8) * 256l;
}
static long decay_floats(int mode, int dk) { return mode == GLA ? dk : 4; }

// places in the workspace of all cut portions (segments_of): at most 1.2 times what the chip has at once, so 20 MB in all
static long long places(long rows, long each) { return 6ll * rows / (5 * each); }

// workgroups of a portion over those the chip has at once: a compute unit has two of eight waves, one of more
float dgi_chunk_segments_share(int mode, int dk, int dv, int H) {
  return (float)H * dgi_chunk_segments_groups(mode, dv) / (dk <= 64 && dv <= 64 && mode != MLSTM ? 512.f : 256.f);
}

// How a step of `rows` rows in n_seq portions goes: 0 not here but by the kernels of few tokens or of a pipeline for 16 or 32 columns (chunk_scan_decay.hip,
// chunk_parts.hip), else about how many rows a segment has; *floats of workspace (0: all portions whole).
//
// A workgroup here takes all columns of a head, so it repeats nothing, but goes 2.0 us a chunk of 32 tokens (mlstm 2.4) and 7 us before the first; the others
// repeat what columns share, but have it sooner.  So
// - many portions and heads go here (us there, here; 64 channels; heads, portions x rows: gla 64, 3 x 40 13.1, 10.9; 64, 16 x 70 83, 33; 64, 8 x 250 117, 39; 16, 16 x 20 12.3,
//   9.0, but 16, 8 x 20 7.6, 8.4; light 64, 3 x 70 17.4, 12.8; 64, 8 x 250 68, 40; but 16, 8 x 120 14.4, 16.8; mlstm fp32 64, 3 x 300 54, 39; 128 channels: gla 64, 8 x 70 130, 53;
//   16, 8 x 40 26, 20; light 64, 3 x 100 46, 30), but not few sequences of up to sixteen rows, which the others take in one launch (gla 16, 10 x 10 9.2, 12.6);
// - long portions of few heads go here in segments (gla 16, 1 x 2000 123, 31; 32, 2 x 500 41, 28; 64, 1 x 400 30, 24; light 16, 1 x 2000 96, 27; 64, 2 x 2048 125, 109; 128
//   channels 32, 2 x 750 78, 70; mlstm 32, 1 x 661 39, 25; 16, 1 x 2000 89, 33; but gla 16, 1 x 250 19, 21; light 16, 3 x 300 22, 22; 64, 2 x 549 39, 42; mlstm 16, 3 x 300 26, 26);
// - mlstm's nine waves fill a compute unit, so a chip nearly full of long portions is the pipeline's (32, 5 x 600 55, 60; bf16 64, 5 x 613 83, 98; fp32 64, 8 x 250 100,
//   77), and so are long portions beside decode rows (64, 8 of 3173 rows and 59 147, 195); more than 64 channels would spill.  Its token loop takes 0.5 us a token, so short
//   portions come here (64, 3 x 40 35, 12; 16, 8 x 20 20, 9; fp32 16, 8 x 40 14.6, 16.6; 64, 3 x 100 25, 16; 32, 4 x 117 19.9, 21.6).
// Where only the step's rows are known, 2.5 times a portion's least length may as well be one portion beside decode rows (64 channels of 64 or more workgroups: 4 times;
// light 32, 4 x 779 54, 58).  The launch of the states, in vain if the portions turn out to be alike, costs 2 to 3 us: many portions have to leave room for a long one,
// more than sixteen (decode rows, mostly) for a shorter one.
int dgi_chunk_segments_plan(int mode, int dk, int dv, int H, int n_seq, int rows, int in_f32, long long* floats) {
  *floats = 0;
  if ((mode != MLSTM && mode != LIGHT && mode != GLA) || dk > (mode == MLSTM ? 64 : 128) || n_seq > 32767) return 0;
  const long units = (long)n_seq * H * dgi_chunk_segments_groups(mode, dv), mean = rows / n_seq, over = rows - n_seq;
  const long least = mode == GLA ? 280 : units > 64 ? 800 : dk <= 64 ? 400 : 600;      // rows of a portion from which segments gain
  bool many = units >= (mode != MLSTM && dk > 64 ? 128 : 160);
  if (mode == GLA && units >= 128 && mean >= 48) many = true;
  if (mode != MLSTM && mean < 16 && n_seq <= 16) many = false;      // one launch takes them all
  bool here = many || mean >= least || over >= (units > 64 && mode != GLA ? 4 : 2.5) * least;
  if (mode == MLSTM) {
    if (mean < 64) here = mean >= (n_seq > 8 ? 24 : 16) && over < (units >= 160 ? 640 : 256);
    else here = (here && !(units >= 100 && (in_f32 ? units < 512 && mean >= 240 : mean >= 160 || n_seq > 16))) || (units >= 64 && mean < 80 && !in_f32);
  }
  if (!here) return 0;
  // segments that fill the chip once
  const float share = dgi_chunk_segments_share(mode, dk, dv, H);
  const long each = (std::max({96l, (long)(rows * share), std::min(128l, rows / 16l)}) + C - 1) / C * C;
  if (over < (!many ? 1 : n_seq > 16 ? 768 : 1000) || whole(over + 1, rows, share, each) || !places(rows, each)) return 1 << 29;
  *floats = places(rows, each) * H * (state_floats(mode, dk, dv) + decay_floats(mode, dk));
  return (int)each;
}

// a.seg_rows and ws as the plan says
int dgi_chunk_segments(ChunkArgs a, int mode, int in_f32, int rows, float* ws, hipStream_t st) {
  const int groups = dgi_chunk_segments_groups(mode, a.dv);
  const long most = ws ? rows / a.seg_rows + std::min(a.n_seq, rows / (a.skip_rows + 1)) : a.n_seq;
  a.blocks = groups * wide(mode, a.dv) + (mode == MLSTM ? 1 : 0);
  a.share = dgi_chunk_segments_share(mode, a.dk, a.dv, a.H);
  a.wsd = ws;
  a.ws = ws ? ws + places(rows, a.seg_rows) * a.H * decay_floats(mode, a.dk) : nullptr;
  if (most > 65535 || (long)a.H * groups > 0x3fffffff) return -3;
  const dim3 grid(a.H * groups, (unsigned)most);
  for (int only = ws ? 1 : 0; only >= 0; --only) {
    const int rc = mode == MLSTM ? dgi_segments_mlstm(a, in_f32, only, grid, st)
                   : mode == LIGHT ? dgi_segments_light(a, in_f32, only, grid, st) : dgi_segments_gla(a, in_f32, only, grid, st);
    if (rc) return rc;
    DGI_CHECK_LAUNCH();
  }
  return 0;
}
