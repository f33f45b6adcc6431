// dgi/csrc/mix/chunk_segments.hip — the plan of segments and the launches of chunk_segments.h.
#include <algorithm>
#include "chunk_split.h"
#include "segments.h"

constexpr int GLA = 3;
constexpr int APART_FROM = 8;        // as linear_scan.hip's
int dgi_segments_mlstm(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st);
int dgi_segments_light(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st);
int dgi_segments_gla(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st);

// blocks of 16 columns of a workgroup.  The matrix memory's thirteen waves would have 128 registers each, and spill.  gla's twelve, of more than 64 key channels, have 168
// and spill as well: the outputs' launch 78 registers of fp32 rows (52 bytes a lane), 10 of bf16 ones.
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

// How a step of `rows` rows in n_seq portions goes: 0 not here but by the kernels of few tokens or of a pipeline for 16 or 32 columns
// (chunk_scan_decay.hip, chunk_parts.hip, mlstm's token loop), else about how many rows a segment has; *floats of workspace (0: all portions whole).
//
// A workgroup here takes all columns of a head, so it repeats nothing, but goes 2.0 us a chunk of 32 tokens (mlstm 2.4) and 7 us before the first; the others
// repeat what columns share, but have it sooner.  Only the step's rows and portions are known, not who has the rows: the workgroups decide by the lengths how portions
// are cut, but a line here is where one long portion beside decode rows gains several times what portions that are alike lose ("but").
// us there, here; 64 channels and bf16 rows unless said; heads, portions x rows:
// - many portions and heads: gla 64, 3 x 40 13, 11; 64, 16 x 70 83, 33; 64, 8 x 250 117, 39; 16, 16 x 20 12.3, 9.0, but 16, 8 x 20 7.6, 8.4; light 64, 8 x 250 68, 40; 128
//   channels: gla 64, 8 x 70 130, 53; 16, 8 x 40 26, 20; light 64, 3 x 100 46, 30; not few sequences of up to sixteen rows (gla 16, 10 x 10 9.2, 12.6);
// - long portions of few heads, in segments: gla 16, 1 x 2000 123, 31; 32, 2 x 500 41, 28; light 16, 1 x 2000 96, 27; 64, 2 x 2048 125, 109; but gla 64, 1 x 300 23.2, 25.3; 128
//   channels, 300 rows 33, 42, so 400 there;
// - rows enough for one portion to be long: gla 16, 1 of 1521 among 5 95, 26; light 16, 1 of 1473 among 11 82, 47; but gla 16, 4 x 190 17, 23; fp32 4, 4 x 228 of 128
//   channels 28, 60, so from 1000 rows there; light 16, 8 x 500 38, 42;  of four and eight heads alike portions lose most, and long ones gain most: gla 8, 8 x 108 12, 20, but 1 of 850
//   among 10 55, 22; light of 128 channels 4, 10 x 270 34, 60, but 1 of 1554 among 30 164, 52;
// - mlstm's nine waves fill a compute unit, and its pipeline is the closer one: a nearly full chip of bf16 rows stays there (32, 5 x 600 55, 60; 64, 5 x 613 83, 98), as do long
//   portions beside decode rows of many heads (64, 8 of 3173 rows and 59 147, 195); more than 64 channels would spill.  Its token loop takes 0.5 us a token, so short portions come here
//   (64, 3 x 40 35, 12; 16, 8 x 20 20, 9), among nine sequences and more it has two launches to lose (16, 16 x 62 23, 15; fp32 64, 12 x 75 79, 45); full chips: 64, 3 x 100 25, 17; 32, 8 x 83
//   23, 15; fp32 64, 3 x 300 55, 45; 8 x 500 153, 128; long portions: 32, 1 x 661 39, 25; 16, 1 x 2000 89, 33; 32, 1 of 2000 among 17 107, 64; but 32, 3 x 459 35, 46;
//   fp32 rows of a third of the chip and more stay there (32, 3 x 535 48, 67), as do those beside more decode rows (32, 2 of 1547 and 92 114, 139).
// The launch of the states, in vain if no portion turns out to be worth cutting, costs 3 to 6 us; a long portion left whole 2 us for 32 rows of it, 4 of 128 channels.  Many portions
// and heads: it is launched where one may have more than 600 to 1000 rows, or, but for gla, whose kernel there is slower than whole portions here, more than it takes cut by 150 to 250 and by 10 a
// sequence: those lose most whole (there, whole, cut: light 32 heads of 128 channels, 1 of 665 rows and 9 74, 110, 61; 32, 1 of 801 and 5 43, 55, 29; mlstm 16, 1 of 597 and 6 37, 46, 28; 32, 1 of 900
// and 10 73, 91, 48), and where they are alike it is in vain, but no slower than there (light 64, 3 of 602 rows in all 30, 23, 29; 5 of 1043 47, 33, 39; gla 64 of 128 channels, 8 of 560 119, 44, 54, so
// whole).  Among more than 64 sequences it is launched where one may have more than 400 and more than
// the workgroups of those that turn out to be short cost: 2 us for as many as the chip has at once, in both launches (64 heads of 128 channels, 3747 rows of 203 sequences 772, cut 996; of
// 64, 4000 rows and 500 decode rows 635, 525; 2 of 2000 and 1000 744, 790).
int dgi_chunk_segments_plan(int mode, int dk, int dv, int H, int n_seq, int rows, int in_f32, long long* floats) {
  *floats = 0;
  if ((mode != MLSTM && mode != LIGHT && mode != GLA) || dk > (mode == MLSTM ? 64 : 128) || n_seq > 32767) return 0;
  const int groups = dgi_chunk_segments_groups(mode, dv);
  const long units = (long)n_seq * H * groups, mean = rows / n_seq, over = rows - n_seq;
  const float share = dgi_chunk_segments_share(mode, dk, dv, H), fill = rows * share;
  bool many, here;
  if (mode == MLSTM) {
    const bool f = in_f32;
    if (mean < 64 && over < (units >= 160 ? 640 : 256)) {      // the token loop's
      many = here = mean >= (n_seq > 2 * APART_FROM ? 24 : 16);
    } else if (n_seq > 2 * APART_FROM) {
      many = false;
      here = over >= (f ? 1000 : 1600) && H * groups <= (f && n_seq <= 32 ? 64 : 32) && n_seq <= 80 && fill < (f ? 700.f : 500.f);
    } else if (n_seq > APART_FROM) {
      many = here = mean >= 16 && (f || fill < 400.f);
    } else {
      many = f && mean >= 100 ? units >= 192 : units >= 96 && mean < 160;
      here = many || (units <= (f ? 64 : 100) && mean >= 400) || (units <= 64 && over >= 1000);
    }
  } else {
    const bool gla = mode == GLA, wide = dk > 64;
    const long least = gla ? (wide ? 400 : 280) : units > 64 ? 800 : wide ? 600 : 400;
    many = (units >= (wide ? 128 : 160) || (gla && units >= 128 && mean >= 48)) && (mean >= 16 || n_seq > 2 * APART_FROM);
    here = many || mean >= least || over >= (gla ? (wide ? 1000 : 700) : units > 64 ? 4 * least : 5 * least / 2);
  }
  if (!here) return 0;
  // segments that fill the chip once; of 128 rows at least where sixteen of them are no more than a portion
  const long each = (std::max({96l, (long)fill, std::min(128l, rows / 16l)}) + C - 1) / C * C;
  const float cut = 1.3f * (fill + each) + 96;         // as whole's
  const long least_cut = n_seq > 64 ? std::max(400l, (long)(80 * share * std::min(n_seq, rows / 17)))
                         : n_seq > 2 * APART_FROM ? 768 : n_seq > APART_FROM ? 1000 : mode == MLSTM ? 600 : dk > 64 ? 700 : 1000;
  const long gains = mode == GLA || n_seq > 64 ? least_cut : (long)cut + (mode == MLSTM ? 250 : dk > 64 ? 150 : 200) + 10 * n_seq;
  if ((many && over < std::min(least_cut, gains)) || whole(over + 1, rows, share, each) || !places(rows, each)) return 1 << 29;
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
