// dgi/csrc/mix/chunk_args.h — what the kernels of prompt portions in chunks share (chunk_scan.hip, chunk_parts.hip, chunk_delta.hip).
#pragma once
#include "../common.h"

namespace {

constexpr int WKV = 0, DELTA = 1, MLSTM = 2, LIGHT = 4, SSM = 5;      // 3: gla, chunk_scan_decay.hip

using namespace dgi;

}  // namespace

struct ChunkArgs {
  float* y;                        // [T, H * dv]
  const void *q, *k, *v;           // rows with their own strides (elements); wkv: q the receptance; ssm: C, B, x
  int q_stride, k_stride, v_stride;
  const void *aux1, *aux2;         // per token: w_raw [T, H*dk] | b_raw | i_raw | - | dt_raw;  - | a_raw | f_raw | - | -
  int aux1_stride, aux2_stride, aux_bf16;
  const float *par1, *par2, *par3; // w0 | a_log | - | decay [H] | a_log;  u | dt_bias | - | - | dt_bias;  ssm: d_skip
  float *state, *norm, *mx;        // state [slots, H, dk, dv] (ssm: [slots, H, dv, dk])
  float *norm_new, *mx_new;        // mlstm with several workgroups per head: staged, as in linear_scan
  const int *positions, *seq_row0, *seq_slots;
  int H, G, dk, dv;
  int n_seq;
  int pass, seg_rows;              // ssm in segments: 0 whole portions, 1 and 2 the two passes
  float *ws, *wsd;                 // [n_seq, segments, H, dv, dk] states, [n_seq, segments, H] decays (chunk_segments.h: as said there)
  int skip_rows;                   // sequences of at most this many rows are not this launch's
  float cap;
  int blocks;                      // chunk_segments.h: of 16 columns, of a head in ws
  float share;                     // workgroups of a portion over those the chip has at once
  float* parts;                    // what a pass before keeps for the launch's chunks (parts_chunks of them): ssm chunk_parts.hip, delta chunk_delta.hip; or null
  int parts_chunks;
};

namespace {

template <typename T> __device__ __forceinline__ float ldf(const T* p);
template <> __device__ __forceinline__ float ldf<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ldf<uint16_t>(const uint16_t* p) { return bf16_to_f32(*p); }
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float silu(float x) { return x * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(x * -1.4426950408889634f)); }
__device__ __forceinline__ float logsigmoid_f(float x) { return fminf(x, 0.f) - log1pf(expf(-fabsf(x))); }
__device__ __forceinline__ bool finite(float x) { return fabsf(x) < __builtin_inff(); }

// Addresses that the compiler shall keep in scalar registers (an empty asm between) lose what it knew of them: loads and stores through them say that
// they are global ones.  As flat ones they would count as LDS accesses too, and every wait for LDS would wait for the memory.
typedef const __attribute__((address_space(1))) char* global_in;
typedef __attribute__((address_space(1))) char* global_out;
template <typename V> __device__ __forceinline__ V gload(global_in p) { return *reinterpret_cast<const __attribute__((address_space(1))) V*>(p); }
__device__ __forceinline__ void gstore(global_out p, float v) { *reinterpret_cast<__attribute__((address_space(1))) float*>(p) = v; }
// the same as flat accesses, where those measured faster (chunk_scan.hip)
template <typename V> __device__ __forceinline__ V gload(const char* p) { return *reinterpret_cast<const V*>(p); }
__device__ __forceinline__ void gstore(char* p, float v) { *reinterpret_cast<float*>(p) = v; }

// Rows of a chunk as a buffer: the first row's address and the rows' offsets are scalars, a lane's offset is kept; lane offsets beyond the bytes read
// zeros and write nothing (a row offset is not looked at, so it is added to the lane's where rows may be missing).
typedef __amdgpu_buffer_rsrc_t Rows;
__device__ __forceinline__ Rows rows_at(const void* p, unsigned bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00027000); }
template <typename V> __device__ __forceinline__ V row_load(Rows r, unsigned lane, unsigned row) {
  if constexpr (sizeof(V) == 2) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b16(r, lane, row, 0));
  else if constexpr (sizeof(V) == 4) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, lane, row, 0));
  else if constexpr (sizeof(V) == 8) return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, lane, row, 0));
  else return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, lane, row, 0));
}
__device__ __forceinline__ void row_store(Rows r, float v, unsigned lane, unsigned row) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, lane, row, 0);
}

// four consecutive elements as they lie in memory
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <typename T> struct Raw4Of;
template <> struct Raw4Of<float> { typedef f32x4 V; };
template <> struct Raw4Of<uint16_t> { typedef u32x2 V; };
template <typename T> using Raw4 = typename Raw4Of<T>::V;
__device__ __forceinline__ void widen(const f32x4& r, float* f) {
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = r[i];
}
__device__ __forceinline__ void widen(const u32x2& r, float* f) {
  f[0] = __uint_as_float(r[0] << 16); f[1] = __uint_as_float(r[0] & 0xffff0000u);
  f[2] = __uint_as_float(r[1] << 16); f[3] = __uint_as_float(r[1] & 0xffff0000u);
}

// the largest magnitude of values that are not NaN (fmaxf would first bring its operands into canonical form: three instructions)
__device__ __forceinline__ float larger3(float m, float a, float b) {
  asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(m) : "v"(a), "v"(b));
  return m;
}

}  // namespace

int dgi_chunk_segments_plan(int mode, int dk, int dv, int H, int n_seq, int rows, int in_f32, long long* floats);
int dgi_chunk_segments_groups(int mode, int dv);
float dgi_chunk_segments_share(int mode, int dk, int dv, int H);
int dgi_chunk_segments(ChunkArgs a, int mode, int in_f32, int rows, float* ws, hipStream_t st);
bool dgi_chunk_parts_takes(int mode, int dk, int H, int G, int in_f32);
int dgi_chunk_parts(const ChunkArgs& a, int mode, int in_f32, dim3 grid, hipStream_t st);
int dgi_chunk_delta(const ChunkArgs& a, int in_f32, dim3 grid, hipStream_t st);
