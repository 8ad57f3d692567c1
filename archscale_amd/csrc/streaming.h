// Device helpers shared by the kernels that stream over tensors: element access, ordered reductions, the norm of a matrix.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "elementwise.h"
#include "launch_rules.h"

namespace archscale {

static constexpr int EW_THREADS = 256;
static constexpr int EW_VEC = 8;                                   // elements per thread per trip
static constexpr int EW_TRIPS = MUON_CHUNK_ELEMS / (EW_THREADS * EW_VEC);
static_assert(EW_TRIPS * EW_THREADS * EW_VEC == MUON_CHUNK_ELEMS, "chunk must be a whole number of trips");

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint16_t f2bf(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
__device__ __forceinline__ float bf2f(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
// two at a time: one conversion for both instead of two and their merging (vocabulary matrices on the sphere 725 -> 717 us per
// step, 64 experts 1317 -> 1313)
__device__ __forceinline__ uint32_t f2bf_pair(float a, float b) {
  typedef float f32x2_ __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_ __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_){a, b}, bf16x2_));
}

// Most accesses stream: an element is touched once per launch and the tensors of a step are far larger than the caches, so
// 16-byte accesses carry the non-temporal hint (measured on a 2-read / 2-write stream of 1 GiB arrays: 5.87 TB/s with it,
// 5.57 TB/s without; a plain copy 6.29 against 5.72 TB/s).  Not the stores of what the next launch reads, the operand images and
// the update: where they fit the memory-side cache it serves them (steps of width 1024: EMA Muon 1210 -> 1192 us, MuonBall
// 1494 -> 1463; 3001 x 1023 188.5 -> 186), and where they do not nothing is lost (depth-16 set 22.15 ms either way).
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ u32x4 stream_load16(const void* p) { return __builtin_nontemporal_load((const u32x4*)p); }
__device__ __forceinline__ void stream_store16(void* p, u32x4 v) { __builtin_nontemporal_store(v, (u32x4*)p); }

// Runs of eight elements are read and written in 16-byte accesses wherever they start: the hardware takes global accesses of any alignment,
// and tensors of odd widths, or matrices inside one, rarely start at a multiple of 16 bytes.  A copy of 512 MiB so: 6.2 TB/s aligned, 5.9
// with the loads two bytes off, 5.7 the stores, 5.5 both; element by element 2.9.  A MuonH step of width 1001 in bfloat16 with 5003 x 1001
// under hyperball AdamW, per launch: momentum 156 / 87 us, norms 57 / 26, AdamW 132 / 33 and 44 / 17, results of the last product 114 / 73.
typedef u32x4 u32x4_any __attribute__((aligned(2)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));

template <int DT> struct Elem;  // DT_BF16 / DT_F32 access of 8 consecutive elements
template <> struct Elem<DT_BF16> {
  typedef uint16_t T;
  static __device__ __forceinline__ void load8(const void* p, long i, float (&v)[8]) {
    const u32x4 r = __builtin_nontemporal_load((const u32x4_any*)((const uint16_t*)p + i));
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) { v[2 * k] = bf2f(w[k] & 0xffff); v[2 * k + 1] = bf2f(w[k] >> 16); }
  }
  // the same through the caches, for lines that other accesses share
  static __device__ __forceinline__ void fetch8(const void* p, long i, float (&v)[8]) {
    const u32x4 r = *(const u32x4_any*)((const uint16_t*)p + i);
#pragma unroll
    for (int k = 0; k < 4; ++k) { v[2 * k] = bf2f(r[k] & 0xffff); v[2 * k + 1] = bf2f(r[k] >> 16); }
  }
  static __device__ __forceinline__ u32x4 pack8(const float (&v)[8]) {
    return u32x4{f2bf_pair(v[0], v[1]), f2bf_pair(v[2], v[3]), f2bf_pair(v[4], v[5]), f2bf_pair(v[6], v[7])};
  }
  static __device__ __forceinline__ void store8(void* p, long i, const float (&v)[8]) { __builtin_nontemporal_store(pack8(v), (u32x4_any*)((uint16_t*)p + i)); }
  static __device__ __forceinline__ void keep8(void* p, long i, const float (&v)[8]) { *(u32x4_any*)((uint16_t*)p + i) = pack8(v); }
  static __device__ __forceinline__ float load1(const void* p, long i) { return bf2f(((const uint16_t*)p)[i]); }
  static __device__ __forceinline__ void store1(void* p, long i, float v) { ((uint16_t*)p)[i] = f2bf(v); }
  static __device__ __forceinline__ float round(float v) { return bf2f(f2bf(v)); }
};
template <> struct Elem<DT_F32> {
  typedef float T;
  static __device__ __forceinline__ void load8(const void* p, long i, float (&v)[8]) {
    const f32x4 a = __builtin_nontemporal_load((const f32x4_any*)((const float*)p + i));
    const f32x4 b = __builtin_nontemporal_load((const f32x4_any*)((const float*)p + i + 4));
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  static __device__ __forceinline__ void fetch8(const void* p, long i, float (&v)[8]) {
    const f32x4 a = *(const f32x4_any*)((const float*)p + i), b = *(const f32x4_any*)((const float*)p + i + 4);
#pragma unroll
    for (int k = 0; k < 4; ++k) { v[k] = a[k]; v[4 + k] = b[k]; }
  }
  static __device__ __forceinline__ void store8(void* p, long i, const float (&v)[8]) {
    const f32x4 a = {v[0], v[1], v[2], v[3]}, b = {v[4], v[5], v[6], v[7]};
    __builtin_nontemporal_store(a, (f32x4_any*)((float*)p + i));
    __builtin_nontemporal_store(b, (f32x4_any*)((float*)p + i + 4));
  }
  static __device__ __forceinline__ void keep8(void* p, long i, const float (&v)[8]) {
    *(f32x4_any*)((float*)p + i) = f32x4{v[0], v[1], v[2], v[3]};
    *(f32x4_any*)((float*)p + i + 4) = f32x4{v[4], v[5], v[6], v[7]};
  }
  static __device__ __forceinline__ float load1(const void* p, long i) { return ((const float*)p)[i]; }
  static __device__ __forceinline__ void store1(void* p, long i, float v) { ((float*)p)[i] = v; }
  static __device__ __forceinline__ float round(float v) { return v; }
};

__device__ __forceinline__ bool aligned16(const void* p) { return (((uintptr_t)p) & 15) == 0; }

// ordered block reduction of up to 3 values; result valid in thread 0
template <int N>
__device__ __forceinline__ void block_reduce(float (&v)[N], float* smem /* N * 4 floats */) {
#pragma unroll
  for (int k = 0; k < N; ++k) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_down(v[k], off, 64);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) smem[k * 4 + w] = v[k];
  }
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int k = 0; k < N; ++k) v[k] = (smem[k * 4 + 0] + smem[k * 4 + 1]) + (smem[k * 4 + 2] + smem[k * 4 + 3]);
  }
}

// Sum of squares of a 256-thread block's share of a strided matrix: what thread `tid` adds up of the chunk (MUON_CHUNK_ELEMS
// consecutive elements in row-major order; 0 for a chunk past the end).  Whoever forms the norm of a matrix adds in this order.
// Dense matrices (dense_sumsq_ok) load a chunk whole before the first sum; the first elements of the matrix stand in past its
// end and are not counted; the elements after the last whole run join at the end.
__device__ __forceinline__ bool dense_sumsq_ok(int rows, int cols, int ld) { return sums_in_runs(rows, cols, ld, MUON_CHUNK_ELEMS); }
template <int DT>
__device__ __forceinline__ float thread_sumsq_dense(const char* base, long numel, int chunk, int tid, bool cast_first) {
  const long first = (long)chunk * MUON_CHUNK_ELEMS + (long)tid * EW_VEC, full = numel / EW_VEC * EW_VEC;
  float v[EW_TRIPS][EW_VEC], s = 0.f;
#pragma unroll
  for (int t = 0; t < EW_TRIPS; ++t) {
    const long i = first + (long)t * EW_THREADS * EW_VEC;
    Elem<DT>::load8(base, i < full ? i : 0, v[t]);
  }
#pragma unroll
  for (int t = 0; t < EW_TRIPS; ++t) {
    const bool in = first + (long)t * EW_THREADS * EW_VEC < full;
#pragma unroll
    for (int k = 0; k < EW_VEC; ++k) v[t][k] = in ? (DT == DT_F32 && cast_first ? bf2f(f2bf(v[t][k])) : v[t][k]) : 0.f;
    // (the second square is rounded before the first joins it)
#pragma unroll
    for (int k = 0; k < EW_VEC; ++k) {
      if (t == 0 && k < 2) s = k == 0 ? v[0][1] * v[0][1] : fmaf(v[0][0], v[0][0], s);
      else s = fmaf(v[t][k], v[t][k], s);
    }
  }
  if (full < numel && full / MUON_CHUNK_ELEMS == chunk && full / EW_VEC % EW_THREADS == tid) {
    for (long i = full; i < numel; ++i) {
      float x = Elem<DT>::load1(base, i);
      if (cast_first) x = bf2f(f2bf(x));
      s = fmaf(x, x, s);
    }
  }
  return s;
}
// (a dense matrix of one chunk that does not go in runs: nothing to divide, eight loads in flight.  Apart from the strided sums, which the kernel of
// small matrices holds three times: with it inside them 3 x (1083 x 33), which takes neither, 56.1 against 55.6 us, in fp32 53.6 / 52.9)
template <int DT>
__device__ __forceinline__ float thread_sumsq_one_chunk(const char* base, int numel, int tid, bool cast_first) {
  float s = 0.f;
#pragma unroll 8
  for (int i = tid; i < numel; i += EW_THREADS) {
    float x = Elem<DT>::load1(base, i);
    if (cast_first) x = bf2f(f2bf(x));
    s = fmaf(x, x, s);
  }
  return s;
}
template <int DT>
__device__ __forceinline__ float thread_sumsq_strided(const char* base, int rows, int cols, int ld, int chunk, int tid, bool cast_first) {
  const long numel = (long)rows * cols, begin = (long)chunk * MUON_CHUNK_ELEMS;
  const long end = begin + MUON_CHUNK_ELEMS < numel ? begin + MUON_CHUNK_ELEMS : numel;
  float s = 0.f;
  for (long i = begin + tid; i < end; i += EW_THREADS) {
    const long r = i / cols, cc = i - r * cols;
    float x = Elem<DT>::load1(base, r * ld + cc);
    if (cast_first) x = bf2f(f2bf(x));
    s = fmaf(x, x, s);
  }
  return s;
}

// normalisation factor of a matrix from its sum of squares; with pow2 it is split into a power of two (applied to the copy
// of the input, exactly) and a rest in [0.7, 1.5]
__device__ __forceinline__ float2 norm_factor(float sumsq, float eps, int eps_mode, bool pow2) {
  const float n = sqrtf(sumsq);
  const float sc = eps_mode == EPS_ADD ? 1.f / (n + eps) : 1.f / fmaxf(n, eps);
  if (!pow2) return make_float2(sc, 1.f);
  const bool ok = sc > 0.f && sc < 3.0e38f;
  const float p = ok ? exp2f(rintf(log2f(sc))) : sc;
  return make_float2(ok ? sc / p : 1.f, p);
}

}  // namespace archscale
