// Internal interface between the Newton-Schulz GEMM kernels and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "launch_rules.h"

namespace archscale {

constexpr int BK = 64;   // elements per k-tile

// MODE_SYRKT: as MODE_SYRK, but P = Q is given K-major ([K][M] row-major, ldp = leading dimension; P == Q required)
enum { MODE_SYRK = 0, MODE_SYRK2 = 1, MODE_BX = 2, MODE_SYRKT = 3 };

// who walks the parts of a reduction that is cut (GemmParams::ksplit): nobody has any, a block each, one block all of them
enum KCut { CUT_NONE = 0, CUT_BLOCKS, CUT_SEQUENCE };

// C[m][n] = sum_k P[m][k] * Q[n][k]; all leading dimensions / strides in elements.
struct GemmParams {
  // (what the start of a tile needs comes first and together)
  const __bf16* P;   // [batch][tilesM*BM][ldp]
  const __bf16* Q;   // [batch][tilesN*BN][ldq]
  long strideP, strideQ;
  int ldp, ldq;
  int K;             // reduction length, multiple of 64
  int tilesM, tilesN;
  int qt_first;          // quarter mode: first tile of this problem (in its own coarser enumeration) that is covered
  // a launch may cover only tiles [t_first, t_first + t_count) of every matrix of the problem (in the matrix's own
  // enumeration; t_count = 0: all of them), the flat tile index of the launch then counts t_count tiles per matrix
  int t_first;
  // filled in by the launch: tiles per matrix that it covers, reciprocals (floor((2^32 - 1) / d)) of that and of what a line
  // of the tile order holds, blocks of one part of a K-split
  int per_mat;
  uint32_t inv_per_mat, inv_line;
  int part_tiles;
  int t_count;
  int batch;
  const __bf16* P2;  // second pass over K for P (low half of a split B), or null
  const __bf16* E;   // epilogue addend, read as E[col][row..row+3]; MODE_BX: may be null (X' = B X, no addend)
  long strideE;
  int lde;
  __bf16* C;         // row-major output [row][col] (may be null in MODE_BX)
  __bf16* C2;        // low half of a split output (MODE_SYRK2 with split)
  long strideC;
  int ldc;
  __bf16* Ct;        // transposed output [col][row] (MODE_BX, may be null)
  long strideCt;
  int ldct;
  float alpha, beta;
  int out_shift;         // MODE_BX: the result is multiplied by 2^out_shift (0: as it is)
  float diag_add;        // MODE_SYRK2: added to the diagonal of the result (B + a I, so that B X needs no addend)
  const float* scale;    // per batch element, or null: SYRK / SYRKT multiply the product by scale^2, BX the result by scale
  int m_valid, n_valid;  // true extents for the bounds-checked final store
  // K-split (symmetric products of the 128x128 configuration only): `ksplit` > 1 blocks share every tile, block s of
  // them walks k-tiles [s KT / ksplit, (s + 1) KT / ksplit) and leaves its fp32 accumulators in sk_partial; the block
  // that finds itself last (sk_counter, one per tile, zero before the launch and zero again after it) adds the partial
  // results in the order s = 0, 1, ... and runs the epilogue.  The sums do not depend on which block came last.  With
  // CUT_SEQUENCE one block walks the parts one after the other and adds in that order: the same bits, no partial results in memory.
  int ksplit;
  float* sk_partial;     // [tiles of this problem in the launch][ksplit][128 * 128] fp32, accumulator layout
  int* sk_counter;       // [tiles of this problem in the launch]
};

// Several independent problems of one kind (same tile configuration, mode, split and final flags) in ONE
// launch: block b works on problem g with tile_start[g] <= b < tile_start[g+1] (a problem with a K-split owns
// ksplit blocks per tile: block tile_start[g] + s * tiles + t is part s of tile t).  Passed by value as a kernel
// argument (about 3 KiB).
constexpr int MAX_GROUPS = 16;
// Quarter mode (quarter = 1; 2: sixteenths): the blocks of the launch are the 4^quarter smaller tiles of each tile of a
// 2^quarter times coarser enumeration (tilesM, tilesN count the fine tiles; block 4q + s is quadrant s of coarse tile
// qt_first + q).  It lets a smaller configuration take over where the larger one would leave the chip idle.
struct GroupedGemmParams {
  int n_groups;
  int quarter;
  int backwards;                    // MODE_BX: the last tile of the last problem first (see BACKWARDS_BYTES)
  int total;                        // filled in by the launch: tile_start[n_groups] ...
  int tile_start[MAX_GROUPS + 1];   // ... and the places past n_groups, with the largest int
  GemmParams g[MAX_GROUPS];
};
static_assert(sizeof(GroupedGemmParams) <= 4096, "kernel arguments are limited to 4 KiB");

// number of block tiles of one problem
long ns_gemm_tiles(int mode, const GemmParams& p);

// Whether the tiles of a launch follow one another in a block (ns_gemm_stream_kernel): X' = B X in whole tiles of 256, nothing that needs the
// other kernel's bounds checks or unaligned stores, no rows of the caller's that lie STREAM_MAX_LD elements apart or more (its stores have one
// base per tile and signed 32-bit offsets of up to 510 bytes per element of that distance), and enough of them (stream_of_tiles).
constexpr int STREAM_MAX_LD = 1 << 22;
inline bool stream_takes(int tile, int mode, bool split, bool final_, const GroupedGemmParams& gp, int units) {
  if (tile != 256 || mode != MODE_BX || split || gp.quarter) return false;
  int longest = 0;
  for (int i = 0; i < gp.n_groups; ++i) {
    const GemmParams& g = gp.g[i];
    longest = g.K > longest ? g.K : longest;
    if (g.t_first || g.K < 4 * BK || g.ldp != g.ldq || (g.scale && !g.E)) return false;
    if (!final_) {
      if (!g.Ct || g.C) return false;
    } else {
      const bool rows = g.C != nullptr;
      const long stride = rows ? g.strideC : g.strideCt;
      if (g.E || rows == (g.Ct != nullptr) || g.m_valid != g.tilesM * 256 || g.n_valid != g.tilesN * 256) return false;
      const int ld = rows ? g.ldc : g.ldct;
      if (((uintptr_t)(rows ? g.C : g.Ct) & 15) || ld % 8 || ld >= STREAM_MAX_LD || (g.batch > 1 && stride % 8)) return false;
    }
  }
  return stream_of_tiles(units, gp.tile_start[gp.n_groups], longest);
}

// tile: side of the block tile, 256, 128, 64 or 32 (four waves each; 64 without the hi+lo pair, 32 for MODE_SYRKT alone)
// f16: 0 = the workspace matrices of the launch are bfloat16; 1 = IEEE half (see GemmParams::out_shift), not with split;
// 2 = bfloat16 operands, IEEE-half result (MODE_BX, not the final launch)
// units: compute units of the device
// cut: some problem of the launch has GemmParams::ksplit > 1 (symmetric modes, tile 128, no hi+lo pair)
hipError_t launch_ns_gemm_grouped(int tile, int mode, bool split, bool final_, const GroupedGemmParams& gp,
                                  hipStream_t stream, int units, int f16 = 0, KCut cut = CUT_NONE);
// bytes of GemmParams::sk_partial per tile of a K-split launch
constexpr long SK_TILE_BYTES = 128L * 128 * 4;

}  // namespace archscale
