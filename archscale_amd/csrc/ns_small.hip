// The whole Newton-Schulz iteration of a small matrix in ONE block for gfx950: iterate, A and B stay in the LDS of one compute unit.
//
// As launches over tiles (ns_gemm.hip) a 128 x 384 matrix is a chain of 16 launches (and two of staging) of 3 us and 1.3 us between them, for a
// microsecond of matrix-core work each: what bounds it is the chain, not the work.  Here the chain is a sequence of barriers:
// 128 x 384 in 44 us (staging 7, A = X X^T 2.2, a product of two square matrices 1.4 to 1.8, X' 2.8; LDS reads are 1.3, 0.4 and
// 1.4 of those), 64 x 1024 in 42, 64 x 128 in 18, where a step is 0.8 us whatever it does.
// The products are those of the tile kernels, element by element: the same 16x16x32 MFMAs over k in the same order, the same
// epilogue arithmetic and the same rounding to storage, so a matrix has the same bits on either path.
//
// LDS: X^T (long side first, [np][mp]), then two mp x mp matrices: slot 0 holds A and, on the Gram side, T, A', P_N and Q in turn,
// slot 1 holds B (P_{N-1}).  A product keeps its result in registers until every wave has read its operands; X' = B X
// needs not even that, a wave owns whole rows of X^T and reads nothing of the others'.
// Rows are 16-byte chunks XOR-swizzled by the row so that both ways of reading are conflict-free: 16 rows at one chunk (K
// contiguous operand, 128-bit reads) and 8 rows k0 .. k0+3, k0+8 .. k0+11 at a pair of chunks (K-major operand, transpose reads).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>

#include "ns_small.h"
#include "streaming.h"

// the rounding points are those of ns_gemm.hip: no fused operations but the ones written out
#pragma clang fp contract(off)

namespace archscale {

namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));

constexpr int NT = 512, NW = NT / 64;
constexpr int LDS_BYTES = 160 * 1024;

template <bool HALF>
__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  if constexpr (HALF) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
template <bool HALF>
__device__ __forceinline__ float decode(uint32_t bits) {
  if constexpr (HALF) return (float)__builtin_bit_cast(_Float16, (uint16_t)bits);
  else return __builtin_bit_cast(float, bits << 16);
}
// two values, each rounded to float first (ns_gemm.hip: f16_bits)
template <bool HALF>
__device__ __forceinline__ uint32_t encode(float a, float b) {
  if constexpr (HALF) {
    asm("" : "+v"(a), "+v"(b));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
  } else {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
  }
}

// swizzle of row r: 16 chunks (256-byte rows) or 8 (128-byte rows, two of them to a pass over the banks)
template <int MF>
__device__ __forceinline__ int swz(int r) {
  if constexpr (MF == 8) return ((r & 3) << 2) | (((r >> 3) & 1) << 1) | ((r >> 2) & 1);
  else return (((r >> 1) & 1) << 2) | (((r >> 3) & 1) << 1) | ((r >> 2) & 1);
}

// MF: 16-row fragments along the short side (8: up to 128 rows, 4: up to 64)
template <int MF>
struct Small {
  static constexpr int ROW = MF * 32;          // bytes of a row of X^T and of the two square matrices
  static constexpr int KS = MF / 2;            // k-steps of 32 along the short side
  static constexpr int SQUARE = MF * 16 * ROW;
  // upper-triangle fragments of a symmetric product per wave.  MF = 8: the 4 x 4 blocks of 2 x 2 fragments, waves 0 to 5 one
  // off-diagonal block each, waves 6 and 7 two diagonal blocks (three fragments each); MF = 4: ten single fragments.
  static constexpr int NS = MF == 8 ? 6 : 2;

  int lane, l16, lg, wave;

  __device__ __forceinline__ Small() {
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    l16 = lane & 15;
    lg = lane >> 4;
  }
  static __device__ __forceinline__ int at(int row, int chunk) { return row * ROW + ((chunk ^ swz<MF>(row)) << 4); }

  // fragment f (16 rows) of a K-contiguous operand, k-step kk
  __device__ __forceinline__ u32x4 rows(const char* base, int f, int kk) const {
    return *(const u32x4*)(base + at(16 * f + l16, 4 * kk + lg));
  }
  // fragment f (16 columns) of a K-major operand, k-step kk: two transpose reads (ns_gemm.hip)
  __device__ __forceinline__ u32x4 cols(const char* base, int f, int kk) const {
    const int e = l16 >> 2, a = l16 & 3, k = 32 * kk + 8 * lg + e, chunk = 2 * f + (a >> 1);
    typedef __attribute__((address_space(3))) s16x4* lds_t;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(base + at(k, chunk) + (a & 1) * 8));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(base + at(k + 4, chunk) + (a & 1) * 8));
    const uint2 x = __builtin_bit_cast(uint2, lo), y = __builtin_bit_cast(uint2, hi);
    return u32x4{x.x, x.y, y.x, y.y};
  }

  // the off-diagonal block (2I, 2I + 1) x (2J, 2J + 1) of waves 0 to 5
  __device__ __forceinline__ void block_of(int& I, int& J) const {
    I = wave < 3 ? 0 : (wave < 5 ? 1 : 2);
    J = wave < 3 ? wave + 1 : (wave < 5 ? wave - 1 : 3);
  }
  // f(slot, row fragment, column fragment) for the fragments of this wave; `slot` is a compile-time constant
  template <class F>
  __device__ __forceinline__ void each(F&& f) const {
    if constexpr (MF == 8) {
      if (wave < 6) {
        int I, J;
        block_of(I, J);
        f(std::integral_constant<int, 0>{}, 2 * I, 2 * J);
        f(std::integral_constant<int, 1>{}, 2 * I, 2 * J + 1);
        f(std::integral_constant<int, 2>{}, 2 * I + 1, 2 * J);
        f(std::integral_constant<int, 3>{}, 2 * I + 1, 2 * J + 1);
      } else {
        const int D = 4 * (wave - 6);   // first fragment of the first of its two diagonal blocks
        f(std::integral_constant<int, 0>{}, D, D);
        f(std::integral_constant<int, 1>{}, D, D + 1);
        f(std::integral_constant<int, 2>{}, D + 1, D + 1);
        f(std::integral_constant<int, 3>{}, D + 2, D + 2);
        f(std::integral_constant<int, 4>{}, D + 2, D + 3);
        f(std::integral_constant<int, 5>{}, D + 3, D + 3);
      }
    } else {
      // (0,0) (0,1) (0,2) (0,3) (1,1) (1,2) (1,3) (2,2) | (2,3) (3,3)
      const int i = wave < 4 ? 0 : (wave < 7 ? 1 : 2), j = wave < 4 ? wave : (wave < 7 ? wave - 3 : 2);
      f(std::integral_constant<int, 0>{}, i, j);
      if (wave < 2) f(std::integral_constant<int, 1>{}, 2 + wave, 3);
    }
  }

  // step(kk, operands) for kk = 0 .. ksteps - 1 with operands = load(kk): the operands of two k-steps are read while the two before
  // them are multiplied (a k-step of MFMAs is shorter than the wait for an LDS read).  ksteps: a constant (KSTEPS), or a
  // multiple of four.
  template <int N, int KSTEPS, class L, class S>
  static __device__ __forceinline__ void pipelined(int ksteps, L&& load, S&& step) {
    struct Set { u32x4 x[2][N]; };
    auto load2 = [&](Set& s, int kk) __attribute__((always_inline)) { load(kk, s.x[0]); load(kk + 1, s.x[1]); };
    auto step2 = [&](Set& s) __attribute__((always_inline)) { step(s.x[0]); step(s.x[1]); };
    Set a, b;
    load2(a, 0);
    if constexpr (KSTEPS == 2) {
      step2(a);
    } else if constexpr (KSTEPS == 4) {
      load2(b, 2);
      step2(a);
      step2(b);
    } else {
      for (int kk = 0; kk < ksteps; kk += 4) {
        load2(b, kk + 2);
        step2(a);
        load2(a, kk + 4 < ksteps ? kk + 4 : kk);   // (the last trip reads what nobody uses)
        step2(b);
      }
    }
  }

  // acc <- upper-triangle fragments of P Q^T.  KMAJ: with k along the rows of X^T = P = Q (`ksteps` of them); SELF: P = Q
  template <bool HALF, bool KMAJ, bool SELF>
  __device__ __forceinline__ void product(const char* P, const char* Q, int ksteps, f32x4 (&acc)[NS]) const {
    constexpr int KC = KMAJ ? 0 : KS;
#pragma unroll
    for (int s = 0; s < NS; ++s) acc[s] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto p_of = [&](int f, int kk) __attribute__((always_inline)) { return KMAJ ? cols(P, f, kk) : rows(P, f, kk); };
    auto q_of = [&](int f, int kk) __attribute__((always_inline)) { return KMAJ ? cols(Q, f, kk) : rows(Q, f, kk); };
    if constexpr (MF == 8) {
      if (wave < 6) {
        int I, J;
        block_of(I, J);
        pipelined<4, KC>(ksteps,
            [&](int kk, u32x4 (&x)[4]) __attribute__((always_inline)) {
              x[0] = p_of(2 * I, kk); x[1] = p_of(2 * I + 1, kk); x[2] = q_of(2 * J, kk); x[3] = q_of(2 * J + 1, kk);
            },
            [&](const u32x4 (&x)[4]) __attribute__((always_inline)) {
              acc[0] = mfma<HALF>(x[0], x[2], acc[0]);
              acc[1] = mfma<HALF>(x[0], x[3], acc[1]);
              acc[2] = mfma<HALF>(x[1], x[2], acc[2]);
              acc[3] = mfma<HALF>(x[1], x[3], acc[3]);
            });
      } else {
        const int D = 4 * (wave - 6);
        constexpr int N = SELF ? 4 : 8;
        pipelined<N, KC>(ksteps,
            [&](int kk, u32x4 (&x)[N]) __attribute__((always_inline)) {
#pragma unroll
              for (int i = 0; i < 4; ++i) x[i] = p_of(D + i, kk);
              if constexpr (!SELF) {
#pragma unroll
                for (int i = 0; i < 4; ++i) x[4 + i] = q_of(D + i, kk);
              }
            },
            [&](const u32x4 (&x)[N]) __attribute__((always_inline)) {
              constexpr int o = SELF ? 0 : 4;
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                acc[3 * h] = mfma<HALF>(x[2 * h], x[o + 2 * h], acc[3 * h]);
                acc[3 * h + 1] = mfma<HALF>(x[2 * h], x[o + 2 * h + 1], acc[3 * h + 1]);
                acc[3 * h + 2] = mfma<HALF>(x[2 * h + 1], x[o + 2 * h + 1], acc[3 * h + 2]);
              }
            });
      }
    } else {
      each([&](auto s_, int fi, int fj) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value;
        pipelined<2, KC>(ksteps,
            [&](int kk, u32x4 (&x)[2]) __attribute__((always_inline)) { x[0] = p_of(fi, kk); x[1] = q_of(fj, kk); },
            [&](const u32x4 (&x)[2]) __attribute__((always_inline)) { acc[s] = mfma<HALF>(x[0], x[1], acc[s]); });
      });
    }
  }

  // Upper-triangle fragments and their mirror images into a square matrix.  `reflect`: the product of two different matrices,
  // whose diagonal fragments are symmetric only up to rounding: their upper half goes to both of its places.
  template <bool HALF, bool REFLECT>
  __device__ __forceinline__ void store(char* C, const f32x4 (&v)[NS]) const {
    each([&](auto s_, int fi, int fj) __attribute__((always_inline)) {
      constexpr int s = decltype(s_)::value;
      const int r = 16 * fi + 4 * lg, c = 16 * fj + l16;
      const uint32_t lo = encode<HALF>(v[s][0], v[s][1]), hi = encode<HALF>(v[s][2], v[s][3]);
      const uint16_t e[4] = {(uint16_t)lo, (uint16_t)(lo >> 16), (uint16_t)hi, (uint16_t)(hi >> 16)};
      // row c, columns r .. r + 3: eight bytes; rows r .. r + 3, column c: the row of `down` advances by one, which changes
      // its swizzle in bits of its own
      const int across = at(c, r >> 3) + (r & 7) * 2, down = at(r, c >> 3) + (c & 7) * 2;
      auto below = [&](int q) __attribute__((always_inline)) { return (uint16_t*)(C + (down ^ (q * ROW + (swz<MF>(q) << 4)))); };
      if (fi != fj || !REFLECT) *(uint2*)(C + across) = make_uint2(lo, hi);
      if (fi != fj) {
#pragma unroll
        for (int q = 0; q < 4; ++q) *below(q) = e[q];
      } else if constexpr (REFLECT) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (r + q <= c) {
            *(uint16_t*)(C + across + 2 * q) = e[q];
            *below(q) = e[q];
          }
      }
    });
  }

  // C = alpha X X^T
  template <bool HALF>
  __device__ __forceinline__ void gram(const char* X, char* C, int np, float alpha) const {
    f32x4 v[NS];
    product<HALF, true, true>(X, X, np / 32, v);
#pragma unroll
    for (int s = 0; s < NS; ++s) v[s] *= alpha;
    store<HALF, false>(C, v);
    __syncthreads();
  }
  // SELF: C = alpha P P + beta P (+ diag on the diagonal).  Otherwise C = alpha P Q, P and Q symmetric and commuting.  C may be
  // either of them.
  template <bool HALF, bool SELF>
  __device__ __forceinline__ void square(const char* P, const char* Q, char* C, float alpha, float beta, float diag) const {
    f32x4 v[NS];
    product<HALF, false, SELF>(P, Q, KS, v);
    if constexpr (SELF) {
      each([&](auto s_, int fi, int fj) __attribute__((always_inline)) {
        constexpr int s = decltype(s_)::value;
        const int r = 16 * fi + 4 * lg, c = 16 * fj + l16;
        const uint2 e = *(const uint2*)(P + at(c, r >> 3) + (r & 7) * 2);
        const float ev[4] = {decode<HALF>(e.x & 0xffff), decode<HALF>(e.x >> 16), decode<HALF>(e.y & 0xffff), decode<HALF>(e.y >> 16)};
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float x = fmaf(alpha, v[s][q], beta * ev[q]);
          if (fi == fj) x += (4 * lg + q == l16) ? diag : 0.f;
          v[s][q] = x;
        }
      });
    } else {
#pragma unroll
      for (int s = 0; s < NS; ++s) v[s] *= alpha;
    }
    if (C == P || C == Q) __syncthreads();
    store<HALF, !SELF>(C, v);
    __syncthreads();
  }
  // X <- (alpha X + B X) sc (alpha X only with `addend`), in place: the wave owns rows 16 f .. 16 f + 15 of X^T for f = wave,
  // wave + NW, ...; G of its fragments at a time share the reads of B.
  template <bool HALF, bool HALF_OUT, bool ADDEND, int G>
  __device__ __forceinline__ void advance_rows(char* X, const char* B, int f0, float alpha, float sc) const {
    u32x4 q[G][KS];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) q[g][kk] = rows(X, f0 + g * NW, kk);
#pragma unroll
    for (int i = 0; i < MF; ++i) {
      f32x4 v[G];
#pragma unroll
      for (int g = 0; g < G; ++g) v[g] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < KS; ++kk) {
        const u32x4 p = rows(B, i, kk);
#pragma unroll
        for (int g = 0; g < G; ++g) v[g] = mfma<HALF>(p, q[g][kk], v[g]);
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int r = 16 * i + 4 * lg, c = 16 * (f0 + g * NW) + l16;
        uint2* const to = (uint2*)(X + at(c, r >> 3) + (r & 7) * 2);
        float x[4];
        if constexpr (ADDEND) {
          const uint2 e = *to;
          const float ev[4] = {decode<HALF>(e.x & 0xffff), decode<HALF>(e.x >> 16), decode<HALF>(e.y & 0xffff), decode<HALF>(e.y >> 16)};
#pragma unroll
          for (int k = 0; k < 4; ++k) x[k] = fmaf(alpha, ev[k], v[g][k]) * sc;
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) x[k] = v[g][k] * sc;
        }
        *to = make_uint2(encode<HALF_OUT>(x[0], x[1]), encode<HALF_OUT>(x[2], x[3]));
      }
    }
  }
  template <bool HALF, bool HALF_OUT, bool ADDEND>
  __device__ __forceinline__ void advance(char* X, const char* B, int np, float alpha, float sc) const {
    constexpr int G = 3;
    const int nf = np / 16;
    int f = wave;
    for (; f + (G - 1) * NW < nf; f += G * NW) advance_rows<HALF, HALF_OUT, ADDEND, G>(X, B, f, alpha, sc);
    for (; f < nf; f += NW) advance_rows<HALF, HALF_OUT, ADDEND, 1>(X, B, f, alpha, sc);
    __syncthreads();
  }

  // ---- the operand into LDS, zero padded
  // staged: direct copies of 1 KiB, the swizzle in the source address
  __device__ __forceinline__ void copy_staged(char* X, const uint16_t* src, int ld, int np) const {
    typedef const __attribute__((address_space(1))) void* gptr_t;
    typedef __attribute__((address_space(3))) void* lptr_t;
    constexpr int CH = ROW / 16;
    for (int s = wave; s < np * ROW / 1024; s += NW) {
      const int i = s * 64 + lane, r = i / CH, c = (i % CH) ^ swz<MF>(r);
      __builtin_amdgcn_global_load_lds((gptr_t)(src + (size_t)r * ld + c * 8), (lptr_t)(X + s * 1024), 16, 0, 0);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
  // the caller's matrix: norm as stage_sumsq_kernel and stage_layout_kernel form it, copy as layout_tile makes it.  Returns what
  // is left to the first iteration's epilogues.
  template <int DT>
  __device__ __forceinline__ float stage(char* X, float* red, const SmallNsParams& sp, const SmallNsProblem& p, const char* base,
                                         int m, int n, int np) const {
    float s = 1.f, rest = 1.f;
    if (sp.normalize) {
      const int chunks = (int)(((long)m * n + MUON_CHUNK_ELEMS - 1) / MUON_CHUNK_ELEMS);
      // chunk j of this half of the block, `count` from `first` on (all their loads before the first sum)
      auto chunk_sums = [&](auto first_, auto count_) __attribute__((always_inline)) {
        constexpr int first = decltype(first_)::value, count = decltype(count_)::value;
        float v[count];
        if (dense_sumsq_ok(p.rows, p.cols, p.in_ld)) {
#pragma unroll
          for (int j = 0; j < count; ++j)
            v[j] = thread_sumsq_dense<DT>(base, (long)m * n, (wave >> 2) + 2 * (first + j), threadIdx.x & 255, sp.cast_first);
        } else if (first == 0 && p.in_ld == p.cols) {   // (one chunk: sums_in_runs)
#pragma unroll
          for (int j = 1; j < count; ++j) v[j] = 0.f;
          v[0] = wave >> 2 ? 0.f : thread_sumsq_one_chunk<DT>(base, m * n, threadIdx.x & 255, sp.cast_first);
        } else {
#pragma unroll
          for (int j = 0; j < count; ++j)
            v[j] = thread_sumsq_strided<DT>(base, p.rows, p.cols, p.in_ld, (wave >> 2) + 2 * (first + j), threadIdx.x & 255, sp.cast_first);
        }
#pragma unroll
        for (int j = 0; j < count; ++j) {
#pragma unroll
          for (int off = 32; off > 0; off >>= 1) v[j] += __shfl_down(v[j], off, 64);
          if (lane == 0) red[((wave >> 2) + 2 * (first + j)) * 4 + (wave & 3)] = v[j];
        }
      };
      chunk_sums(std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});   // up to 49152 elements
      if (MF == 4 && chunks > 6) chunk_sums(std::integral_constant<int, 3>{}, std::integral_constant<int, 2>{});   // up to 64 x 1152
      __syncthreads();
      float all = lane < chunks ? (red[lane * 4] + red[lane * 4 + 1]) + (red[lane * 4 + 2] + red[lane * 4 + 3]) : 0.f;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) all += __shfl_down(all, off, 64);
      const float2 f = norm_factor(__shfl(all, 0, 64), sp.eps, sp.eps_mode, sp.defer);
      s = sp.defer ? f.y : f.x;
      rest = sp.defer ? f.x : 1.f;
    }
    // whole runs of eight, or element by element (a branch per run would make every load wait for the one before)
    const bool vec = p.cols % 8 == 0;
    const float fs = __builtin_ldexpf(1.f, sp.half ? p.sx : 0);
    // eight elements of a row from column c on, and the eight as they go into the workspace
    auto fetch = [&](auto vec_, int r, int c, float (&v)[8]) __attribute__((always_inline)) {
      const bool in = r < p.rows && c < p.cols;
      if constexpr (decltype(vec_)::value) {
        Elem<DT>::load8(base, in ? (long)r * p.in_ld + c : 0, v);
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = in ? v[k] : 0.f;
      } else {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = (in && c + k < p.cols) ? Elem<DT>::load1(base, (long)r * p.in_ld + c + k) : 0.f;
      }
    };
    auto pack = [&](const float (&v)[8]) __attribute__((always_inline)) {
      u32x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const bool cast = DT == DT_F32 && sp.cast_first;
        const float x = cast ? bf2f(f2bf(v[2 * k])) : v[2 * k], y = cast ? bf2f(f2bf(v[2 * k + 1])) : v[2 * k + 1];
        o[k] = sp.half ? encode<true>(x * s * fs, y * s * fs) : encode<false>(x * s, y * s);
      }
      return o;
    };
    auto copy = [&](auto vec_) __attribute__((always_inline)) {
      constexpr int U = decltype(vec_)::value ? 6 : 1;   // runs in flight per lane
      float v[U][8];
      if (p.rows >= p.cols) {   // X^T is the matrix as it is
        constexpr int CH = ROW / 16;
        const int all = np * CH;
        for (int i0 = threadIdx.x; i0 < all; i0 += U * NT) {
#pragma unroll
          for (int u = 0; u < U; ++u) fetch(vec_, (i0 + u * NT) / CH, (i0 + u * NT) % CH * 8, v[u]);
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (i0 + u * NT < all) *(u32x4*)(X + at((i0 + u * NT) / CH, (i0 + u * NT) % CH)) = pack(v[u]);
        }
      } else {
        // a wave takes 16 rows of 32 columns: 64 bytes at a time in memory, 32 along a row of X^T
        const int all = MF * (np / 32);
        for (int i0 = wave; i0 < all; i0 += U * NW) {
#pragma unroll
          for (int u = 0; u < U; ++u) fetch(vec_, 16 * ((i0 + u * NW) % MF) + l16, 32 * ((i0 + u * NW) / MF) + 8 * lg, v[u]);
#pragma unroll
          for (int u = 0; u < U; ++u) {
            if (i0 + u * NW >= all) break;
            const int r = 16 * ((i0 + u * NW) % MF) + l16, c = 32 * ((i0 + u * NW) / MF) + 8 * lg;
            const u32x4 o = pack(v[u]);
#pragma unroll
            for (int k = 0; k < 8; ++k) *(uint16_t*)(X + at(c + k, r >> 3) + (r & 7) * 2) = (uint16_t)(o[k >> 1] >> ((k & 1) * 16));
          }
        }
      }
    };
    if (vec) copy(std::true_type{});
    else copy(std::false_type{});
    __syncthreads();
    return rest;
  }
};

template <int MF>
__global__ void __launch_bounds__(NT, 1) small_ns_kernel(const SmallNsParams sp) {
#if defined(__HIP_DEVICE_COMPILE__)
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  int g = 0;
  while (g + 1 < sp.n && (int)blockIdx.x >= sp.block_start[g + 1]) ++g;
  const SmallNsProblem p = sp.p[g];
  const int b = blockIdx.x - sp.block_start[g];
  const Small<MF> k;
  constexpr int ROW = Small<MF>::ROW, CH = ROW / 16;
  const int m = p.rows < p.cols ? p.rows : p.cols, n = p.rows < p.cols ? p.cols : p.rows;
  const int np = (n + 127) & ~127;
  char* const X = smem;
  char* const S0 = X + np * ROW;
  char* const S1 = S0 + Small<MF>::SQUARE;

  float deferred = 1.f;   // what the first iteration's epilogues multiply by
  if (p.in_dtype < 0) {
    k.copy_staged(X, (const uint16_t*)p.in + (size_t)b * p.in_stride, p.in_ld, np);
    if (p.scale) deferred = p.scale[b];
  } else if (p.in_dtype == DT_BF16) {
    deferred = k.template stage<DT_BF16>(X, (float*)S0, sp, p, (const char*)p.in + (size_t)b * p.in_stride * 2, m, n, np);
  } else {
    deferred = k.template stage<DT_F32>(X, (float*)S0, sp, p, (const char*)p.in + (size_t)b * p.in_stride * 4, m, n, np);
  }

  // The steps of the iteration (every kind of step stands in the code once: the chain walks it many times, and it has to stay
  // in the instruction cache).  Three steps to a plain iteration: A = X X^T, B, X' = a X + B X; seven to the last two iterations on
  // the Gram side: A1, P1, T = P1 A1, A2 = T P1, P2, Q = P2 P1, X' = Q X.  In half storage A carries 2^sa, everything else that is
  // square 2^sb and the iterate 2^sx; the caller's result carries nothing.
  const int plain = p.gram_tail ? sp.iters - 2 : sp.iters, steps = 3 * plain + (p.gram_tail ? 7 : 0);
  for (int step = 0; step < steps; ++step) {
    const int u = step - 3 * plain;
    const int it = u < 0 ? step / 3 : (u < 4 ? sp.iters - 2 : sp.iters - 1);
    const int kind = u < 0 ? step % 3 : (u == 0 ? 0 : (u == 6 ? 2 : 1));
    const SmallNsIteration c = sp.it[it];
    const int sai = c.half_in ? sp.sa : 0, sbi = c.half_in ? sp.sb : 0, sxi = c.half_in ? p.sx : 0;
    const float sc = it == 0 ? deferred : 1.f;
    if (kind == 0) {
      const float alpha = ldexpf(1.f, sai - 2 * sxi) * sc * sc;
      if (c.half_in) k.template gram<true>(X, S0, np, alpha);
      else k.template gram<false>(X, S0, np, alpha);
    } else if (kind == 1) {
      const bool pair = u == 2 || u == 3 || u == 5;
      const char* const P = u == 2 ? S1 : S0;
      const char* const Q = pair ? (u == 2 ? S0 : S1) : S0;
      char* const to = u <= 1 ? S1 : S0;
      const int shift = u == 2 ? -sai : (u == 3 ? sai - 2 * sbi : -sbi);
      const float alpha = pair ? ldexpf(1.f, shift) : ldexpf(c.c, sbi - 2 * sai);
      const float beta = ldexpf(c.b, sbi - sai), diag = c.fold ? ldexpf(c.a, sbi) : 0.f;
      if (pair) k.template square<true, false>(P, Q, to, alpha, 0.f, 0.f);   // (the Gram side is in half)
      else if (c.half_in) k.template square<true, true>(P, P, to, alpha, beta, diag);
      else k.template square<false, true>(P, P, to, alpha, beta, diag);
    } else {
      const float alpha = ldexpf(c.a, sbi), all = sc * ldexpf(1.f, (c.half_out ? p.sx : 0) - sbi - sxi);
      const char* const B = u < 0 ? S1 : S0;
      if (c.half_in) {
        if (c.half_out) c.fold ? k.template advance<true, true, false>(X, B, np, alpha, all) : k.template advance<true, true, true>(X, B, np, alpha, all);
        else c.fold ? k.template advance<true, false, false>(X, B, np, alpha, all) : k.template advance<true, false, true>(X, B, np, alpha, all);
      } else {
        if (c.half_out) c.fold ? k.template advance<false, true, false>(X, B, np, alpha, all) : k.template advance<false, true, true>(X, B, np, alpha, all);
        else c.fold ? k.template advance<false, false, false>(X, B, np, alpha, all) : k.template advance<false, false, true>(X, B, np, alpha, all);
      }
    }
  }

  // the result, out of LDS: rows of X^T as they are for a tall matrix, transpose reads for a wide one
  uint16_t* const out = p.out + (size_t)b * p.out_stride;
  auto put = [&](int row, int col, int cols, const u32x4& v) __attribute__((always_inline)) {
    uint16_t* to = out + (size_t)row * p.out_ld + col;
    if (col + 8 <= cols) {
      *(u32x4_any*)to = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < cols) to[e] = (uint16_t)(v[e >> 1] >> ((e & 1) * 16));
    }
  };
  if (p.rows >= p.cols) {
    for (int i = threadIdx.x; i < n * CH; i += NT) {
      const int r = i / CH, c = i % CH;
      if (c * 8 < m) put(r, c * 8, m, *(const u32x4*)(X + Small<MF>::at(r, c)));
    }
  } else {
    // fragment f of the short side, 32 columns from 32 kk on: lane l16 of a group has row 16 f + l16, eight columns
    for (int i = k.wave; i < MF * (np / 32); i += NW) {
      const int f = i % MF, kk = i / MF;
      const u32x4 v = k.cols(X, f, kk);
      const int row = 16 * f + k.l16, col = 32 * kk + 8 * k.lg;
      if (row < m && col < n) put(row, col, n, v);
    }
  }
#endif
}

template <int MF>
hipError_t launch(const SmallNsParams& p, int np, hipStream_t stream) {
  // (an attribute of the function on one device; a racing first call only repeats it)
  static std::atomic<bool> attr_set[64];
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const bool slot = dev >= 0 && dev < 64;
  if (!slot || !attr_set[dev].load(std::memory_order_acquire)) {
    e = hipFuncSetAttribute((const void*)small_ns_kernel<MF>, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
    if (e != hipSuccess) return e;
    if (slot) attr_set[dev].store(true, std::memory_order_release);
  }
  const int lds = np * Small<MF>::ROW + 2 * Small<MF>::SQUARE;
  if (lds > LDS_BYTES) return hipErrorInvalidValue;
  hipLaunchKernelGGL(small_ns_kernel<MF>, dim3(p.block_start[p.n]), dim3(NT), lds, stream, p);
  return hipGetLastError();
}

}  // namespace

bool small_ns_extents(int m, int n, int* mp, int* np) {
  if (m < 1 || m > 128 || n < m || n > 65536) return false;
  const int side = m <= 64 ? 64 : 128, rows = (n + 127) / 128 * 128;
  if (mp) *mp = side;
  if (np) *np = rows;
  return (long)(rows + 2 * side) * side * 2 <= LDS_BYTES;
}

hipError_t launch_small_ns(const SmallNsParams& p, hipStream_t stream) {
  if (p.n < 1 || p.n > SMALL_NS_MAX_PROBLEMS || p.iters < 1 || p.iters > SMALL_NS_MAX_ITERS || p.block_start[0] != 0) return hipErrorInvalidValue;
  int side = 0, rows = 0;
  for (int i = 0; i < p.n; ++i) {
    const SmallNsProblem& q = p.p[i];
    int mp, np;
    if (!small_ns_extents(q.rows < q.cols ? q.rows : q.cols, q.rows < q.cols ? q.cols : q.rows, &mp, &np)) return hipErrorInvalidValue;
    if ((side && mp != side) || !q.in || !q.out || p.block_start[i + 1] <= p.block_start[i] || (q.gram_tail && p.iters < 3)) return hipErrorInvalidValue;
    // a staged operand covers the kernel's extents in rows of whole chunks
    if (q.in_dtype < 0 && (q.in_ld < mp || q.in_ld % 8 || q.in_stride < (long)np * q.in_ld || q.in_stride % 8 || ((uintptr_t)q.in & 15))) return hipErrorInvalidValue;
    if (q.in_dtype >= 0 && q.in_ld < q.cols) return hipErrorInvalidValue;
    side = mp;
    rows = np > rows ? np : rows;
  }
  return side == 64 ? launch<4>(p, rows, stream) : launch<8>(p, rows, stream);
}

}  // namespace archscale
