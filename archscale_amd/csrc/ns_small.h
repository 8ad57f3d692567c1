// Internal interface between the one-block Newton-Schulz kernel and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace archscale {

// One problem (a batch of equal matrices) of a launch.  The matrices are either the caller's, as muon_ns_batched takes them, or
// operands that are staged already: X^T in bfloat16 (or scaled half), [batch][stride / ld][ld] with the long side first, zero
// padded at least to the kernel's extents (small_ns_extents).
struct SmallNsProblem {
  const void* in;
  long in_stride;
  const float* scale;   // staged: per matrix, or null: what the first iteration's epilogues multiply by (see GemmParams::scale)
  uint16_t* out;        // the caller's bfloat16 tensor
  long out_stride;
  int in_ld, out_ld;
  int rows, cols;
  int sx;               // half storage: the iterate is kept times 2^sx
  int8_t in_dtype;      // -1: staged
  uint8_t gram_tail;    // the last two iterations run on the Gram side
};

constexpr int SMALL_NS_MAX_PROBLEMS = 24, SMALL_NS_MAX_ITERS = 16;

struct SmallNsIteration {
  float a, b, c;
  uint8_t half_in, half_out, fold;   // storage of the operands / of the next iterate; a I goes into B
};

struct SmallNsParams {
  int n, iters;
  int sa, sb;                        // powers of two that A and B carry in half storage
  // matrices that are not staged: normalisation (see StageParams); `defer`: all but a power of two of it is left to the first
  // iteration; `half`: into scaled half
  float eps;
  int eps_mode;
  uint8_t normalize, cast_first, defer, half;
  int block_start[SMALL_NS_MAX_PROBLEMS + 1];   // one block per matrix
  SmallNsIteration it[SMALL_NS_MAX_ITERS];
  SmallNsProblem p[SMALL_NS_MAX_PROBLEMS];
};
static_assert(sizeof(SmallNsParams) <= 4096, "kernel arguments are limited to 4 KiB");

// Extents of the LDS image of an m x n matrix (m <= n) and whether it is taken at all: the iterate, A and B have to fit the
// 160 KiB of one compute unit.
bool small_ns_extents(int m, int n, int* mp, int* np);
hipError_t launch_small_ns(const SmallNsParams& p, hipStream_t stream);

}  // namespace archscale
