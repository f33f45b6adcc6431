// dgi/csrc/mix/chunk_segments_mlstm.hip — chunk_segments.h for the matrix memory.
#include "chunk_segments.h"

int dgi_segments_mlstm(const ChunkArgs& a, int in_f32, bool only, dim3 grid, hipStream_t st) { return launch_type<MLSTM>(a, in_f32, only, grid, st); }
