// dgi/csrc/mix/chunk_segments_gla.hip — chunk_segments.h for gated linear attention.
#include "chunk_segments.h"

int dgi_segments_gla(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st) { return launch_type<GLA>(a, in_f32, only, grid, st); }
