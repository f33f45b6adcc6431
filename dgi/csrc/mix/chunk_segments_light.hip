// dgi/csrc/mix/chunk_segments_light.hip — chunk_segments.h for lightning attention.
#include "chunk_segments.h"

int dgi_segments_light(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st) { return launch_type<LIGHT>(a, in_f32, only, grid, st); }
