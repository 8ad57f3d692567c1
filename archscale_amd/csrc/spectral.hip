// Spectral-norm estimate by power iteration and the MuonBall weight update for gfx950.
//
// The reference estimates the top singular value of every weight matrix W with `steps` rounds of
//   v <- normalize(W^T (W v)),  v0 = 1,   sigma = |W v|
// (emerging_optimizers/orthogonalized_optimizers/spectral_ball_utils.py:151-166): two matrix-vector
// products over W per round, 100 passes over all weights for the default 50 rounds.  Here the Gram
// matrix of the SHORT side, G = X X^T with X = W (rows <= cols) or W^T (rows > cols), is formed once on
// the matrix cores (the SYRK kernel of the Newton-Schulz iteration), and the rounds run on G:
//   rows >  cols:  G = W^T W,  x0 = 1,      x = G^steps x0,        sigma^2 = x^T G x / x^T x
//   rows <= cols:  G = W W^T,  x0 = W 1,    x = G^(steps-1) x0,    sigma^2 = |G x|^2 / x^T G x
// which is the same vector sequence ((W^T W)^k 1 = W^T (W W^T)^(k-1) W 1) at 1/2 .. 1/11 of the memory
// traffic per round.  The normalisation between two rounds only scales the vector, so all applications but the last
// (whose Rayleigh quotient is the result, and is taken with G itself) may be grouped: with G2 = G^2 and G4 = G2^2,
// formed once by the same SYRK kernel, 50 rounds are 12 passes over G4, one over G2 or G and the final one over G
// instead of 50 or 51 passes over G.  G carries a power-of-two factor (mean eigenvalue about 1) that keeps its powers
// in the bf16 range; the result is divided by it.  A rounding error in G2 / G4 perturbs the direction only, and the quotient is
// second-order in it.  Vectors stay in fp32 (the reference rounds them to bf16 every round); every application is ONE
// launch over all matrices of all shape classes; norms are ordered two-stage reductions.
//
// The weight update fuses decoupled weight decay, retraction to the spectral sphere and the step:
//   W <- f * decay * W - lr * ratio * Phi,   f from sigma(decay * W) = decay * sigma(W)
// (muon_ball.py:60-142, spectral_ball_utils.py:168-212, orthogonalized_optimizer.py:184-228).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "launch_rules.h"
#include "spectral.h"
#include "streaming.h"

namespace archscale {

namespace {

__device__ __forceinline__ float bf2f_(uint16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
__device__ __forceinline__ uint16_t f2bf_(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }

// sum over the wave, lanes i and i + 32, then 16, 8, 4, 2, 1 apart; in registers (by LDS permutes the six steps of a sum are six
// LDS latencies, a fifth of a round)
__device__ __forceinline__ float wave_sum(float v) {
  // (the two operands of a swap are two registers: one value in both, which the compiler must not know to be one)
  auto halves = [](auto swap, float x) {
    unsigned a = __builtin_bit_cast(unsigned, x), b = a;
    asm("" : "+v"(b));
    const auto r = swap(a, b);
    return __builtin_bit_cast(float, (unsigned)r[0]) + __builtin_bit_cast(float, (unsigned)r[1]);
  };
  v = halves([](unsigned a, unsigned b) { return __builtin_amdgcn_permlane32_swap(a, b, false, false); }, v);
  v = halves([](unsigned a, unsigned b) { return __builtin_amdgcn_permlane16_swap(a, b, false, false); }, v);
  auto from = [&](auto n_) {   // lane + n of the same 16 lanes
    constexpr int n = decltype(n_)::value;
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x100 | n, 0xf, 0xf, true));
  };
  v += from(std::integral_constant<int, 8>{});
  v += from(std::integral_constant<int, 4>{});
  v += from(std::integral_constant<int, 2>{});
  v += from(std::integral_constant<int, 1>{});
  return __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, v)));
}

// block -> (class, matrix, 16-row strip); per(class): blocks per matrix
template <class F>
__device__ __forceinline__ void locate(const SnParams& sp, int& g, int& b, int& s, F&& per) {
  // (all first blocks in one fetch instead of one after the other)
  const int blk = blockIdx.x;
  int first = 0;
  g = 0;
#pragma unroll
  for (int i = 1; i < SN_MAX_CLASSES; ++i) {
    const int at = sp.blk_start[i];
    if (i < sp.n && blk >= at) { g = i; first = at; }
  }
  const int local = blk - first;
  const int n = per(sp.c[g]);
  b = local / n;
  s = local - b * n;
}
// blocks per matrix of a launch over the strips, and of the first one
__host__ __device__ __forceinline__ int strips_of(const SnClass& c) { return c.nblk; }
__host__ __device__ __forceinline__ int init_blocks_of(const SnClass& c) { return c.own ? c.xparts : c.nblk; }

// Dot products of four rows of a row-major bf16 matrix (leading dimension ld, a multiple of 8) with an fp32 vector, over n_cols
// columns (a multiple of 8).  The first AHEAD runs of a lane can be fetched before anything else is known.
// (More of them make the waves of a launch ask for the same part of their rows at the same time: two against one, us per step, 15
// matrices of 1920 26.1 / 22.9, 16 of 2048 31.1 / 26.7, 8 of 2048 17.7 / 15.5; none ahead 24.2, 28.3, 15.8.  16 of 1024 5.5 / 5.3.)
constexpr int AHEAD = 1;   // 512 columns
struct Rows4 {
  uint4 r[AHEAD][4];
  float4 x[AHEAD][2];
};
__device__ __forceinline__ void rows4_fetch(Rows4& f, const uint16_t* __restrict__ row0, long ld, const float* __restrict__ x,
                                            int n_cols, int lane) {
#pragma unroll
  for (int t = 0; t < AHEAD; ++t) {
    const int j = t * 512 + lane * 8 < n_cols ? t * 512 + lane * 8 : 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) f.r[t][i] = *(const uint4*)(row0 + (size_t)i * ld + j);
    f.x[t][0] = *(const float4*)(x + j);
    f.x[t][1] = *(const float4*)(x + j + 4);
  }
}
__device__ __forceinline__ void rows4_add(const uint4 (&r)[4], const float4& a, const float4& c, float (&acc)[4]) {
  const float xv[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w[4] = {r[i].x, r[i].y, r[i].z, r[i].w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      acc[i] += bf2f_(w[k] & 0xffff) * xv[2 * k];
      acc[i] += bf2f_(w[k] >> 16) * xv[2 * k + 1];
    }
  }
}
__device__ __forceinline__ void rows4_finish(const Rows4& f, const uint16_t* __restrict__ row0, long ld, const float* __restrict__ x,
                                             int n_cols, int lane, float (&acc)[4]) {
  acc[0] = acc[1] = acc[2] = acc[3] = 0.f;
#pragma unroll
  for (int t = 0; t < AHEAD; ++t)
    if (t * 512 + lane * 8 < n_cols) rows4_add(f.r[t], f.x[t][0], f.x[t][1], acc);
  for (int j = AHEAD * 512 + lane * 8; j < n_cols; j += 512) {
    uint4 r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = *(const uint4*)(row0 + (size_t)i * ld + j);
    rows4_add(r, *(const float4*)(x + j), *(const float4*)(x + j + 4), acc);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = wave_sum(acc[i]);
}
// row sums of four rows and the sum of their squares (this lane's share)
__device__ __forceinline__ float rows4_sums(const uint16_t* __restrict__ row0, long ld, int n_cols, int lane, float (&acc)[4]) {
  acc[0] = acc[1] = acc[2] = acc[3] = 0.f;
  float sq = 0.f;
#pragma unroll 2
  for (int j = lane * 8; j < n_cols; j += 512) {
    uint4 r[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = *(const uint4*)(row0 + (size_t)i * ld + j);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t w[4] = {r[i].x, r[i].y, r[i].z, r[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float lo = bf2f_(w[k] & 0xffff), hi = bf2f_(w[k] >> 16);
        acc[i] += lo;
        acc[i] += hi;
        sq = fmaf(lo, lo, sq);
        sq = fmaf(hi, hi, sq);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i] = wave_sum(acc[i]);
  return sq;
}

// This lane's share of the sum of squares of `rows` x `cols` elements (cols a multiple of 8), by block `part` of `parts`.  The runs of
// all rows are dealt out as one sequence: every lane has work whatever the rows are, and eight loads in flight.
__device__ __forceinline__ float runs_sumsq(const uint16_t* __restrict__ X, int ld, int rows, int cols, int part, int parts) {
  constexpr int U = SUM_RUNS / 256;
  const int per_row = cols / 8, total = rows * per_row;
  const uint32_t inv = reciprocal(per_row);
  float sq = 0.f;
  for (int q0 = part * SUM_RUNS + threadIdx.x; q0 < total; q0 += parts * SUM_RUNS) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int at;
      const int row = divide(min(q0 + u * 256, total - 1), per_row, inv, at);
      v[u] = *(const uint4*)(X + (size_t)row * ld + at * 8);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = q0 + u * 256 < total;
      const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float lo = in ? bf2f_(w[k] & 0xffff) : 0.f, hi = in ? bf2f_(w[k] >> 16) : 0.f;
        sq = fmaf(lo, lo, sq);
        sq = fmaf(hi, hi, sq);
      }
    }
  }
  return sq;
}

// sums `n` (S, D) pairs in a fixed lane-strided order; result in all lanes
__device__ __forceinline__ void sum_pairs(const float* __restrict__ part, int n, int lane, float& S, float& D) {
  float s = 0.f, d = 0.f;
  for (int i = lane; i < n; i += 64) { s += part[2 * i]; d += part[2 * i + 1]; }
  S = wave_sum(s);
  D = wave_sum(d);
}

}  // namespace

// x0 = X 1 (row sums of the short-side-first operand) or 1;  z[0] <- x0, z[1] <- 0, part[0] <- (|x0|^2 per strip, 0); where X is
// the caller's, its sums of squares: one read of X, which the Gram product then finds in the caches.
// 16 matrices of 1024 x 2816: 16 us, where a copy of them with its sums took 35 and this pass came on top.  Tall matrices (x0 = 1)
// have as many blocks as they have data, not one per strip: us per spectral_norm call of 5 rounds, copied / one block per strip and one
// load per lane in flight / as here: 6144 x 128 67 / 91 / 55, 16384 x 128 96 / 181 / 72, 16 of 6144 x 128 84 / 111 / 62, 4096 x 1024
// 83 / 80 / 69, 2816 x 1024 76 / 67 / 63, 16 of them 155 / 124 / 125, 50304 x 512 474 / 482 / 363.
__global__ void __launch_bounds__(256)
sn_init_kernel(const SnParams sp) {
  __shared__ float red[8];
  int g, b, s;
  locate(sp, g, b, s, init_blocks_of);
  const SnClass c = sp.c[g];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r0 = s * SN_ROWS + wave * 4;
  const uint16_t* X = (const uint16_t*)c.X + (size_t)b * c.strideX;
  float v[4] = {1.f, 1.f, 1.f, 1.f}, sq = 0.f;
  if (!c.tall) {
    sq = rows4_sums(X + (size_t)r0 * c.ldx, c.ldx, c.L_p, lane, v);
  } else if (c.own) {
    sq = c.long_first ? runs_sumsq(X, c.ldx, c.L_p, c.d, s, c.xparts) : runs_sumsq(X, c.ldx, c.d, c.L_p, s, c.xparts);
  }
  if (c.own) sq = wave_sum(sq);
  float S = 0.f;
  if (s < c.nblk) {
    float* z0 = c.z + (size_t)b * c.d_p;
    float* z1 = c.z + ((size_t)c.batch + b) * c.d_p;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float val = (r0 + i < c.d) ? v[i] : 0.f;
      if (lane == 0) { z0[r0 + i] = val; z1[r0 + i] = 0.f; }
      S += val * val;
    }
  }
  if (lane == 0) { red[wave] = S; red[4 + wave] = sq; }
  __syncthreads();
  if (threadIdx.x == 0) {
    if (s < c.nblk) {
      float* p = c.part + ((size_t)b * c.nblk + s) * 2;
      p[0] = (red[0] + red[1]) + (red[2] + red[3]);
      p[1] = 0.f;
    }
    if (c.own) c.xpart[(size_t)b * c.xparts + s] = (red[4] + red[5]) + (red[6] + red[7]);
  }
}

// z[dst] <- M z[src] / max(|z[src]|, 1e-12);  part[dst] <- per strip (|z[dst]|^2,  z[src]^T z[dst] / |z[src]|)
// M = G, G2 or G4 (which = 0, 1, 2) and the source buffer are given per kind of class (wide, tall), whose sequences
// differ; which < 0: the classes of that kind sit this launch out.
// Latency bound (16 matrices of 1024: 32 MB that the caches hold): every load of the first 512 columns is on its way before the
// norm of z[src] is added up, and no sum goes through LDS: 5.3 us a launch, 6.2 before.
__global__ void __launch_bounds__(256)
sn_step_kernel(const SnParams sp, int src_wide, int which_wide, int src_tall, int which_tall) {
  __shared__ float red[8];
  int g, b, s;
  locate(sp, g, b, s, strips_of);
  const SnClass& c = sp.c[g];
  const int src = c.tall ? src_tall : src_wide, which = c.tall ? which_tall : which_wide;
  if (which < 0) return;
  const __bf16* M = which == 0 ? c.G : (which == 1 ? c.G2 : c.G4);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int dst = src ^ 1, d = c.d, d_p = c.d_p, nblk = c.nblk, batch = c.batch;
  const float* zin = c.z + ((size_t)src * batch + b) * d_p;
  float* zout = c.z + ((size_t)dst * batch + b) * d_p;
  float* const part = c.part;
  const float* pin = part + (((size_t)src * batch + b) * nblk) * 2;
  const int r0 = s * SN_ROWS + wave * 4;
  const uint16_t* row0 = (const uint16_t*)M + (size_t)b * d_p * d_p + (size_t)r0 * d_p;
  Rows4 ahead;
  rows4_fetch(ahead, row0, d_p, zin, d_p, lane);
  float own[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) own[i] = zin[r0 + i];
  float Sin, Din;
  sum_pairs(pin, nblk, lane, Sin, Din);
  const float inv = 1.f / fmaxf(sqrtf(Sin), 1e-12f);
  float acc[4];
  rows4_finish(ahead, row0, d_p, zin, d_p, lane, acc);
  float S = 0.f, D = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float out = (r0 + i < d) ? acc[i] * inv : 0.f;
    if (lane == 0) zout[r0 + i] = out;
    S += out * out;
    D += own[i] * inv * out;
  }
  if (lane == 0) { red[wave] = S; red[4 + wave] = D; }
  __syncthreads();
  if (threadIdx.x == 0) {
    float* p = part + (((size_t)dst * batch + b) * nblk + s) * 2;
    p[0] = (red[0] + red[1]) + (red[2] + red[3]);
    p[1] = (red[4] + red[5]) + (red[6] + red[7]);
  }
}

// sigma[blk] of a class from the partials of the last round, by one wave
__device__ __forceinline__ void sigma_of(const SnClass& c, int blk, int src, int lane) {
  float S, D;
  sum_pairs(c.part + (((size_t)src * c.batch + blk) * c.nblk) * 2, c.nblk, lane, S, D);
  const float s2 = c.tall ? D : (D > 0.f ? S / D : 0.f);
  const float xs = c.xscale[blk];   // G = xs^2 X X^T
  if (lane == 0) c.sigma[blk] = xs > 0.f ? sqrtf(fmaxf(s2, 0.f)) / xs : 0.f;
}
__global__ void __launch_bounds__(64)
sn_final_kernel(const SnParams sp, int src_wide, int src_tall) {
  // one wave per matrix: blocks are numbered class by class
  int blk = blockIdx.x, g = 0;
  while (g < sp.n && blk >= sp.c[g].batch) { blk -= sp.c[g].batch; ++g; }
  if (g >= sp.n) return;
  sigma_of(sp.c[g], blk, sp.c[g].tall ? src_tall : src_wide, threadIdx.x);
}

// xscale[b]: one wave per matrix, blocks numbered class by class; the tile sums are added in a fixed order
__global__ void __launch_bounds__(64)
sn_xscale_kernel(const SnParams sp) {
  int blk = blockIdx.x, g = 0;
  while (g < sp.n && blk >= sp.c[g].batch) { blk -= sp.c[g].batch; ++g; }
  if (g >= sp.n) return;
  const SnClass c = sp.c[g];
  const float* part = c.xpart + (size_t)blk * c.xparts;
  float t = 0.f;
  for (int i = threadIdx.x; i < c.xparts; i += 64) t += part[i];
  t = wave_sum(t);
  // a power of two: X and G are scaled exactly
  // (exponent clamped: xscale^2 multiplies an fp32 accumulator)
  if (threadIdx.x == 0)
    c.xscale[blk] = t > 0.f ? exp2f(fminf(fmaxf(rintf(0.5f * log2f((float)c.d / t)), -60.f), 60.f)) : 0.f;
}

int spectral_power_levels(int steps) {
  // G^4 pays from about a dozen applications on (two symmetric products against 3/4 of the passes), G^2 from half of that
  return steps >= 16 ? 2 : (steps >= 6 ? 1 : 0);
}

hipError_t launch_spectral_xscale(const SnParams& sp, hipStream_t stream) {
  if (sp.n < 1 || sp.n > SN_MAX_CLASSES) return hipErrorInvalidValue;
  int matrices = 0;
  for (int g = 0; g < sp.n; ++g) {
    if (sp.c[g].batch <= 0 || !sp.c[g].xscale || !sp.c[g].xpart || sp.c[g].xparts < 1) return hipErrorInvalidValue;
    matrices += sp.c[g].batch;
  }
  hipLaunchKernelGGL(sn_xscale_kernel, dim3(matrices), dim3(64), 0, stream, sp);
  return hipGetLastError();
}

// The vectors of a finished iteration of ONE class: short_out[b][0..d) = z_short[b] and long_out[b][0..L) = X_b^T z_prev[b]
// (X_b: d_p x L_p, zero padded).
// Bound by the one read of X (which the caches may still hold from the Gram product).  A block owns SNV_COLS = 64 columns
// (rows of 128 bytes: a whole cache line per eight lanes) and walks d / 32 rows per thread, its 32 row groups added in
// LDS in a fixed order.  One lane per eight columns walking all d rows is a chain of d dependent-in-order loads on too few
// waves: 16 matrices of 1024 x 2816 took 296 us that way and take 15 us
// now (6.1 TB/s).
constexpr int SNV_COLS = 64, SNV_GROUPS = 256 / (SNV_COLS / 8);
__global__ void __launch_bounds__(256)
sn_vectors_kernel(const uint16_t* __restrict__ X, long strideX, int ldx, const float* __restrict__ z_prev, const float* __restrict__ z_short,
                  float* __restrict__ short_out, float* __restrict__ long_out, int d, int d_p, int L, int L_p) {
  __shared__ float red[SNV_GROUPS][SNV_COLS + 4];   // (rows of 272 bytes: the row groups of a wave start on different banks)
  const int b = blockIdx.y;
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (short_out && t < d) short_out[(size_t)b * d + t] = z_short[(size_t)b * d_p + t];
  const int cg = threadIdx.x & (SNV_COLS / 8 - 1), rg = threadIdx.x / (SNV_COLS / 8);
  const long c0 = (long)blockIdx.x * SNV_COLS, j0 = c0 + cg * 8;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (j0 < L_p) {
    const uint16_t* col = X + (size_t)b * strideX + j0;
    const float* zp = z_prev + (size_t)b * d_p;
#pragma unroll 8
    for (int i = rg; i < d; i += SNV_GROUPS) {
      const uint4 r = *(const uint4*)(col + (size_t)i * ldx);
      const float zi = zp[i];
      const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        acc[2 * k] += bf2f_((uint16_t)(w[k] & 0xffff)) * zi;
        acc[2 * k + 1] += bf2f_((uint16_t)(w[k] >> 16)) * zi;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) red[rg][cg * 8 + k] = acc[k];
  __syncthreads();
  if (threadIdx.x < SNV_COLS && c0 + threadIdx.x < L) {
    float v = 0.f;
#pragma unroll
    for (int i = 0; i < SNV_GROUPS; ++i) v += red[i][threadIdx.x];
    long_out[(size_t)b * L + c0 + threadIdx.x] = v;
  }
}

// the same of matrices stored long side first, [L][d]: four rows per wave against the vector
__global__ void __launch_bounds__(256)
sn_vectors_rows_kernel(const uint16_t* __restrict__ X, long strideX, int ldx, const float* __restrict__ z_prev, const float* __restrict__ z_short,
                       float* __restrict__ short_out, float* __restrict__ long_out, int d, int d_p, int L) {
  const int b = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long t = (long)blockIdx.x * 256 + threadIdx.x;
  if (short_out && t < d) short_out[(size_t)b * d + t] = z_short[(size_t)b * d_p + t];
  const int r0 = (blockIdx.x * 4 + wave) * 4;
  if (r0 >= L) return;   // (L is a multiple of 4)
  const uint16_t* row0 = X + (size_t)b * strideX + (size_t)r0 * ldx;
  const float* zp = z_prev + (size_t)b * d_p;
  Rows4 ahead;
  rows4_fetch(ahead, row0, ldx, zp, d, lane);
  float acc[4];
  rows4_finish(ahead, row0, ldx, zp, d, lane, acc);
  if (lane == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) long_out[(size_t)b * L + r0 + i] = acc[i];
  }
}

const float* spectral_short_vectors(const SnClass& c, int src_final) {
  // wide matrices (G = W W^T): the short vector is the LAST iterate, G^steps W 1 (the reference's u); tall ones
  // (G = W^T W): the one before it, G^steps 1 (the reference's v)
  return c.z + (size_t)(c.tall ? src_final ^ 1 : src_final) * c.batch * c.d_p;
}

hipError_t launch_spectral_vectors(const SnClass& c, int L, int src_final, float* short_out, float* long_out,
                                   hipStream_t stream) {
  if (!long_out || c.batch <= 0 || c.batch > 65535 || c.d <= 0 || c.d > c.d_p || L <= 0 || L > c.L_p ||
      c.L_p % 8 || (src_final != 0 && src_final != 1))
    return hipErrorInvalidValue;
  const float* z_prev = c.z + (size_t)(src_final ^ 1) * c.batch * c.d_p;   // the long vector is X^T times the one before the last
  const float* z_short = spectral_short_vectors(c, src_final);
  if (c.long_first) {
    if (L % 4 || c.d % 8) return hipErrorInvalidValue;
    const unsigned blocks = (unsigned)std::max((L / 4 + 3) / 4, (c.d + 255) / 256);
    hipLaunchKernelGGL(sn_vectors_rows_kernel, dim3(blocks, c.batch), dim3(256), 0, stream, (const uint16_t*)c.X, c.strideX, c.ldx, z_prev,
                       z_short, short_out, long_out, c.d, c.d_p, L);
    return hipGetLastError();
  }
  const unsigned blocks = (unsigned)std::max(((long)c.L_p + SNV_COLS - 1) / SNV_COLS, ((long)c.d + 255) / 256);
  hipLaunchKernelGGL(sn_vectors_kernel, dim3(blocks, c.batch), dim3(256), 0, stream, (const uint16_t*)c.X, c.strideX, c.ldx, z_prev, z_short,
                     short_out, long_out, c.d, c.d_p, L, c.L_p);
  return hipGetLastError();
}

// one block per vector and one for sigma; the vectors are short, so the launch and its chain of loads are what it costs: 16 loads
// in flight per thread instead of one, and no launch of its own for sigma.  16 matrices of 1024 x 2816 with their vectors, 50
// rounds: 249.8 -> 243.4 us the whole call (as launches of the tensor library the unit vectors alone were 25)
__global__ void __launch_bounds__(256)
sn_units_kernel(const SnVectors a, const SnVectors o, const SnClass c, int src_final) {
  __shared__ float red[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (blockIdx.y == 2) {
    if (wave == 0) sigma_of(c, blockIdx.x, src_final, lane);
    return;
  }
  const SnVectors v = blockIdx.y ? o : a;
  const float* x = v.x + (size_t)blockIdx.x * v.stride;
  uint16_t* unit = v.unit + (size_t)blockIdx.x * v.len;
  constexpr int RUN = 16;
  float f[RUN], s = 0.f;
  auto fetch = [&](int i0) {
#pragma unroll
    for (int k = 0; k < RUN; ++k) f[k] = x[min(i0 + k * 256, v.len - 1)];
  };
  for (int i0 = threadIdx.x; i0 < v.len; i0 += RUN * 256) {
    fetch(i0);
#pragma unroll
    for (int k = 0; k < RUN; ++k) s = i0 + k * 256 < v.len ? fmaf(f[k], f[k], s) : s;
  }
  s = wave_sum(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  const float length = sqrtf((red[0] + red[1]) + (red[2] + red[3]));
  const float norm = length < 1e-12f ? 1e-12f : length;   // (a length that is not a number makes the whole vector so; fmaxf would hide it)
  for (int i0 = threadIdx.x; i0 < v.len; i0 += RUN * 256) {
    if (v.len > RUN * 256) fetch(i0);   // (else the run of the first loop)
#pragma unroll
    for (int k = 0; k < RUN; ++k)
      if (i0 + k * 256 < v.len) unit[i0 + k * 256] = f2bf_(f[k] / norm);
  }
}

hipError_t launch_spectral_units(const SnVectors& a, const SnVectors& b, const SnClass& c, int src_final, hipStream_t stream) {
  if (c.batch < 1 || !a.x || !b.x || !a.unit || !b.unit || a.len < 1 || b.len < 1 || a.stride < a.len || b.stride < b.len ||
      !c.part || !c.sigma || !c.xscale || (src_final != 0 && src_final != 1))
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(sn_units_kernel, dim3(c.batch, 3), dim3(256), 0, stream, a, b, c, src_final);
  return hipGetLastError();
}

namespace {
bool classes_ok(const SnParams& sp, int* matrices) {
  if (sp.n < 1 || sp.n > SN_MAX_CLASSES || sp.blk_start[sp.n] <= 0) return false;
  *matrices = 0;
  for (int g = 0; g < sp.n; ++g) {
    const SnClass& c = sp.c[g];
    if (c.batch <= 0 || c.d <= 0 || c.d_p % 128 || c.L_p % 8 || c.d > c.d_p || c.nblk * SN_ROWS != c.d_p || !c.xscale || c.ldx % 8) return false;
    // the caller's own matrices fill the extents that the kernels walk
    if (c.own && (c.d != c.d_p || (c.long_first && !c.tall))) return false;
    // (blocks of the first launch: one sum each, a wide matrix's over the rows of a strip)
    if (c.own && (c.xparts < c.nblk || (!c.tall && c.xparts != c.nblk))) return false;
    *matrices += c.batch;
  }
  return true;
}
}  // namespace

hipError_t launch_spectral_init(const SnParams& sp, hipStream_t stream) {
  int matrices;
  if (!classes_ok(sp, &matrices)) return hipErrorInvalidValue;
  SnParams ip = sp;
  for (int g = 0; g < ip.n; ++g) {
    const long end = ip.blk_start[g] + (long)ip.c[g].batch * init_blocks_of(ip.c[g]);
    if (end > 0x7ffffff0L) return hipErrorInvalidValue;
    ip.blk_start[g + 1] = (int)end;
  }
  hipLaunchKernelGGL(sn_init_kernel, dim3(ip.blk_start[ip.n]), dim3(256), 0, stream, ip);
  return hipGetLastError();
}

hipError_t launch_spectral_iterate(const SnParams& sp, int steps, hipStream_t stream, int* final_src, bool sigma) {
  int matrices;
  if (steps < 1 || !classes_ok(sp, &matrices)) return hipErrorInvalidValue;
  const int blocks = sp.blk_start[sp.n];
  bool have2 = true, have4 = true, any[2] = {false, false};
  for (int g = 0; g < sp.n; ++g) {
    have2 = have2 && sp.c[g].G2 != nullptr;
    have4 = have4 && sp.c[g].G4 != nullptr;
    any[sp.c[g].tall ? 1 : 0] = true;
  }
  // applications before the final one: `steps` for tall matrices (one more than for wide ones, see the file comment),
  // as many as possible with the highest power
  int seq[2][3];   // per kind: how many applications of G4, G2, G, in this order
  int len[2];
  for (int kind = 0; kind < 2; ++kind) {
    int n = kind ? steps : steps - 1;
    seq[kind][0] = have4 ? n / 4 : 0; n -= 4 * seq[kind][0];
    seq[kind][1] = have2 ? n / 2 : 0; n -= 2 * seq[kind][1];
    seq[kind][2] = n;
    len[kind] = any[kind] ? seq[kind][0] + seq[kind][1] + seq[kind][2] : 0;
  }
  auto which_at = [&](int kind, int i) {   // matrix of application i of a kind; -1 past its end
    if (i >= len[kind]) return -1;
    if (i < seq[kind][0]) return 2;
    if (i < seq[kind][0] + seq[kind][1]) return 1;
    return 0;
  };
  int src[2] = {0, 0};
  const int launches = len[0] > len[1] ? len[0] : len[1];
  for (int i = 0; i <= launches; ++i) {
    // the last launch is the final application of G for both kinds
    const int w0 = i == launches ? (any[0] ? 0 : -1) : which_at(0, i), w1 = i == launches ? (any[1] ? 0 : -1) : which_at(1, i);
    hipLaunchKernelGGL(sn_step_kernel, dim3(blocks), dim3(256), 0, stream, sp, src[0], w0, src[1], w1);
    if (w0 >= 0) src[0] ^= 1;
    if (w1 >= 0) src[1] ^= 1;
  }
  if (sigma) hipLaunchKernelGGL(sn_final_kernel, dim3(matrices), dim3(64), 0, stream, sp, src[0], src[1]);
  if (final_src) { final_src[0] = src[0]; final_src[1] = src[1]; }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// MuonBall weight update over a table of strided 2-D blocks
// ---------------------------------------------------------------------------
namespace {

__device__ __forceinline__ int find_item_(const int32_t* __restrict__ prefix, int n_items, int c) {
  int lo = 0, hi = n_items;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= c) lo = mid; else hi = mid;
  }
  return lo;
}

// Bound by memory.  Blocks whose rows follow one another (most: whole matrices and groups of their rows) are one row: runs of eight elements in
// 16-byte accesses past the caches, wherever they start, all loads of a chunk before the first store (they may alias as far as the
// compiler knows).  us for 268 million elements, bfloat16 / fp32: 250 / 486 at any width, 300 / 482 through the caches run by run, 417 / 535
// element by element; 17.8 million that are not in the caches 20 / 35, 24 / 38, 46 / 53.  (Repeated calls that find everything in
// the caches: 17.8 million 19.5 / 33.8, 17.2 / 27.5 through them; steps do not.)
template <int WD>
__device__ __forceinline__ void ball_dense(const muon_ball_item& it, long begin, long end, float fw, float fp) {
  float x[EW_TRIPS][8], u[EW_TRIPS][8];
#pragma unroll
  for (int t = 0; t < EW_TRIPS; ++t) {
    const long i = begin + ((long)t * EW_THREADS + threadIdx.x) * EW_VEC;
    if (i + EW_VEC <= end) {
      Elem<WD>::load8(it.w, i, x[t]);
      Elem<DT_BF16>::load8(it.phi, i, u[t]);
    } else {   // the last elements of a block
      for (long e = i; e < end; ++e)
        Elem<WD>::store1(it.w, e, fw * Elem<WD>::load1(it.w, e) - fp * Elem<DT_BF16>::load1(it.phi, e));
    }
  }
#pragma unroll
  for (int t = 0; t < EW_TRIPS; ++t) {
    const long i = begin + ((long)t * EW_THREADS + threadIdx.x) * EW_VEC;
    if (i + EW_VEC <= end) {
#pragma unroll
      for (int k = 0; k < 8; ++k) x[t][k] = fw * x[t][k] - fp * u[t][k];
      Elem<WD>::store8(it.w, i, x[t]);
    }
  }
}

// Blocks inside wider matrices, whose rows share lines with their neighbours: through the caches, runs of eight where rows are whole runs and
// one element per thread where a run would cross the end of a row.  us for 17.8 million elements, so / as dense blocks with the runs split
// at the ends of rows, bfloat16 and fp32: 24 columns in 32 32 / 34 and 53 / 74, 9 in 17 62 / 136 and 86 / 240, 1001 in 1009 46 / 46 and 58 / 54
// (30 / 45 and 37 / 52 where the caches hold everything).
template <int WD>
__device__ __forceinline__ void ball_strided(const muon_ball_item& it, long begin, long end, float fw, float fp) {
  if (it.cols % EW_VEC == 0) {
    for (long i = begin + (long)threadIdx.x * EW_VEC; i < end; i += EW_THREADS * EW_VEC) {
      const long r = i / it.cols, c = i - r * it.cols, w = r * it.ld_w + c;
      float x[8], u[8];
      Elem<DT_BF16>::fetch8(it.phi, r * it.ld_phi + c, u);
      Elem<WD>::fetch8(it.w, w, x);
#pragma unroll
      for (int k = 0; k < 8; ++k) x[k] = fw * x[k] - fp * u[k];
      Elem<WD>::keep8(it.w, w, x);
    }
  } else {
    for (long i = begin + threadIdx.x; i < end; i += EW_THREADS) {
      const long r = i / it.cols, c = i - r * it.cols;
      const float u = Elem<DT_BF16>::load1(it.phi, r * it.ld_phi + c);
      Elem<WD>::store1(it.w, r * it.ld_w + c, fw * Elem<WD>::load1(it.w, r * it.ld_w + c) - fp * u);
    }
  }
}

template <int WD>
__device__ __forceinline__ void ball_range(const muon_ball_item& it, long begin, long end, float fw, float fp) {
  if (it.ld_w == it.cols && it.ld_phi == it.cols) ball_dense<WD>(it, begin, end, fw, fp);
  else ball_strided<WD>(it, begin, end, fw, fp);
}

}  // namespace

__global__ void __launch_bounds__(256)
ball_apply_kernel(const muon_ball_item* __restrict__ items, const int32_t* __restrict__ prefix, int n_items, float lr,
                  float decay, int retract_mode, float retract_step, float* __restrict__ log_out) {
  const int chunk = blockIdx.x;
  const int ii = find_item_(prefix, n_items, chunk);
  const muon_ball_item it = items[ii];
  const long numel = (long)it.rows * it.cols;
  const long begin = (long)(chunk - prefix[ii]) * MUON_CHUNK_ELEMS;
  const long end = begin + MUON_CHUNK_ELEMS < numel ? begin + MUON_CHUNK_ELEMS : numel;
  // spectral norm of the decayed weights; retraction factor (spectral_ball_utils.py:168-212)
  const float sigma = it.sigma ? decay * *it.sigma : 0.f;
  float f, bias = 0.f;
  if (!it.sigma) {
    f = 1.f;   // a block that is not retracted
  } else if (retract_mode == MUON_RETRACT_HARD) {
    f = it.radius / (fmaxf(sigma, 0.f) + 1e-8f);
  } else {
    bias = sigma > it.radius ? -1.f : 1.f;
    f = 1.f + retract_step * bias;
  }
  if (log_out && chunk == prefix[ii] && threadIdx.x == 0) { log_out[2 * ii] = sigma; log_out[2 * ii + 1] = bias; }
  const float fw = f * decay, fp = lr * it.lr_ratio;
  if (it.w_dtype == MUON_DTYPE_BF16) ball_range<DT_BF16>(it, begin, end, fw, fp);
  else ball_range<DT_F32>(it, begin, end, fw, fp);
}

hipError_t launch_ball_apply(const muon_ball_item* items, const int32_t* prefix, int n_items, int total_chunks, float lr,
                             float decay, int retract_mode, float retract_step, float* log_out, hipStream_t stream) {
  if (total_chunks <= 0) return hipSuccess;
  hipLaunchKernelGGL(ball_apply_kernel, dim3(total_chunks), dim3(256), 0, stream, items, prefix, n_items, lr, decay,
                     retract_mode, retract_step, log_out);
  return hipGetLastError();
}

}  // namespace archscale
