// Newton-Schulz GEMMs for gfx950 (CDNA4): one MFMA kernel, three epilogues.
//
// The iteration  X <- aX + (bA + cA^2)X,  A = X X^T  keeps ONLY the transposed iterate X^T ([n_long][m]):
//   SYRKT  A  = X  * X^T         P = Q = X^T, a K-MAJOR operand ([k][m]); fragments by LDS transpose reads
//   SYRK2  B  = c*A*A + b*A      P = Q = A   (A symmetric, K-contiguous); optionally + a*I on the diagonal
//   BX     X' = a*X + B*X        P = B (symmetric), Q = X^T (K-contiguous); writes X'^T (and X' only for the caller);
//                                ADDEND = false: X' = B*X for a B that already carries a*I (no X tile in the epilogue)
// SYRK and SYRK2 compute upper-triangle tiles and mirror them.  SYRK (P = Q = X, K-contiguous) is the stand-alone
// symmetric rank-k product.  All modes share one main loop (replaces ns_line_1/ns_line_2 and the cuBLAS addmm of
// lit_gpt/optim/newton_schulz_triton.py:66-139, 181-266, 371-378 and the bf16 SYRK of
// emerging_optimizers/triton_kernels/syrk.py:104-185).
//
// Operands live in zero-padded workspace buffers whose extents are multiples of
// the tile sizes, so the main loop has no bounds checks; only the FINAL epilogue
// (which writes the caller's tensor) is bounds-checked.
//
// Data path: global -> LDS with direct 16-byte loads (no VGPR round trip) into two or
// more LDS stages, XOR-swizzled 16-byte chunks so the 128-bit MFMA operand reads are
// bank-conflict free; v_mfma_f32_16x16x32 (bf16 or half) with fp32 accumulation.  Four
// waves in a 2 x 2 arrangement, each with a quarter of the block tile.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <atomic>
#include <type_traits>
#include <utility>

#include "launch_rules.h"
#include "ns_gemm.h"

// The epilogue arithmetic is written out with explicit fmaf() and the compiler forms no fused operations of its own:
// the same element is computed by different code depending on the grid (tiles of 256, 128 or 64, straight or mirrored
// image), and all of them have to round in the same places for the result of a matrix not to
// depend on how the launch was cut into blocks.  Left to itself the compiler fuses a multiply-add with the conversion
// to half in one path and not in the other.
#pragma clang fp contract(off)

namespace archscale {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(2)));   // a result of the caller's, wherever it starts (16-byte stores of any alignment)

typedef const __attribute__((address_space(1))) void* gptr_t;
typedef __attribute__((address_space(3))) void* lptr_t;

static constexpr int ROW_BYTES = BK * 2;   // 8 chunks of 16 B

__device__ __forceinline__ uint16_t bf16_bits(float f) {
  __bf16 h = (__bf16)f;  // round to nearest even
  return __builtin_bit_cast(uint16_t, h);
}
__device__ __forceinline__ float bf16_to_f32(uint16_t b) {
  return __builtin_bit_cast(float, (uint32_t)b << 16);
}
// float -> half of a value that is ROUNDED TO FLOAT first: the empty asm keeps the compiler from merging the operation
// that produced `f` with the conversion (v_fma_mixlo_f16 rounds the exact multiply-add result once, a separate
// conversion rounds twice, and which of the two a code path got would otherwise depend on its shape)
__device__ __forceinline__ uint16_t f16_bits(float f) {
  asm("" : "+v"(f));
  return __builtin_bit_cast(uint16_t, (_Float16)f);
}
__device__ __forceinline__ float f16_to_f32(uint16_t b) { return (float)__builtin_bit_cast(_Float16, b); }
// two values at a time: one conversion instruction for both (converted one by one and put together afterwards they cost
// four instructions more per pair, and the 256 values of a lane are what the epilogue spends its time on)
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t bf16_pair(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}
__device__ __forceinline__ uint32_t f16_pair(float a, float b) {
  asm("" : "+v"(a), "+v"(b));   // (see f16_bits)
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, f16x2));
}

// LDS placement of the 16-byte chunk (row r, k-chunk c) of a [rows][64] bf16 tile.
// XOR with (r>>1)&7 makes any 16 consecutive rows at one k-chunk hit 16 distinct
// 16-byte bank groups (rows alternate between the two 128-byte halves of the 64 banks).
__device__ __forceinline__ int lds_chunk_off(int r, int c) { return r * ROW_BYTES + ((c ^ ((r >> 1) & 7)) << 4); }

// K-major tile in LDS: 64 k-rows of ROWS * 2 bytes.  The 16-byte chunk c of row k sits at chunk c ^ kmaj_swz<ROWS>(k), so
// that what the 32 lanes of a half-wave touch with one transpose read (eight k-rows: k0..k0+3 and k0+8..k0+11, 32 bytes
// each) covers all 64 banks.
template <int ROWS>
__device__ __forceinline__ int kmaj_swz(int k) {
  if constexpr (ROWS >= 128) return ((k & 3) << 2) | (((k >> 3) & 1) << 1);
  else if constexpr (ROWS == 64) return (((k >> 1) & 1) << 2) | (((k >> 3) & 1) << 1);
  else return ((k >> 3) & 1) << 1;
}

// consecutive tiles of a launch that go to one XCD (see the kernel); the grid is a multiple of eight runs
__host__ __device__ constexpr int xcd_run(int tiles) { return tiles < 256 ? (tiles + 7) / 8 : 32; }

// f(0), f(1), ... f(N - 1) with the index as a compile-time constant
template <class F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) { static_for_impl(f, std::make_integer_sequence<int, N>{}); }

// counted wait for this wave's vector-memory operations and for its LDS operations (N: how many of the former may still
// be in flight; vmcnt has six bits)
template <int N>
__device__ __forceinline__ void wait_copies() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

// What the start of a tile needs of its problem, and what its end needs.  The values are pinned to registers where they are
// fetched: left alone the compiler fetches each where it is used, and every fetch is a wait of its own.
struct TileArgs {
  const __bf16 *P, *Q;
  long strideP, strideQ;
  int ldp, ldq, K, tilesM, tilesN, qt_first, t_first, per_mat;
  uint32_t inv_per_mat, inv_line;
  int part_tiles;
};
struct LaunchHead { int n_groups, quarter, backwards, total, first[3]; };   // first tiles of problems 1 to 3
__device__ __forceinline__ TileArgs fetch_tile_args(const GemmParams& g) {
  return TileArgs{g.P, g.Q, g.strideP, g.strideQ, g.ldp, g.ldq, g.K, g.tilesM, g.tilesN, g.qt_first, g.t_first,
                  g.per_mat, g.inv_per_mat, g.inv_line, g.part_tiles};
}
#define ARCHSCALE_PIN_TILE_ARGS(a)                                                                                       \
  "+s"(a.P), "+s"(a.Q), "+s"(a.strideP), "+s"(a.strideQ), "+s"(a.ldp), "+s"(a.ldq), "+s"(a.K), "+s"(a.tilesM), "+s"(a.tilesN), \
      "+s"(a.qt_first), "+s"(a.t_first), "+s"(a.per_mat), "+s"(a.inv_per_mat), "+s"(a.inv_line), "+s"(a.part_tiles)
__device__ __forceinline__ void pin(TileArgs& a) { asm volatile("" : ARCHSCALE_PIN_TILE_ARGS(a)); }
__device__ __forceinline__ void pin(TileArgs& a, LaunchHead& h) {
  asm volatile("" : ARCHSCALE_PIN_TILE_ARGS(a), "+s"(h.n_groups), "+s"(h.quarter), "+s"(h.backwards), "+s"(h.total), "+s"(h.first[0]), "+s"(h.first[1]), "+s"(h.first[2]));
}
struct EndArgs {
  // (a pointer that comes out of an assembler statement would count as a generic one)
  const __attribute__((address_space(1))) __bf16* E;
  __attribute__((address_space(1))) __bf16 *C, *Ct;
  const __attribute__((address_space(1))) float* scale;
  long strideE, strideC, strideCt;
  int lde, ldc, ldct, out_shift, m_valid, n_valid;
  float alpha, beta, diag_add;
};
__device__ __forceinline__ EndArgs end_args(const GemmParams& g) {
  EndArgs a = {(const __attribute__((address_space(1))) __bf16*)g.E, (__attribute__((address_space(1))) __bf16*)g.C,
               (__attribute__((address_space(1))) __bf16*)g.Ct, (const __attribute__((address_space(1))) float*)g.scale,
               g.strideE, g.strideC, g.strideCt, g.lde, g.ldc, g.ldct, g.out_shift, g.m_valid, g.n_valid, g.alpha, g.beta, g.diag_add};
  asm volatile("" : "+s"(a.E), "+s"(a.C), "+s"(a.Ct), "+s"(a.scale), "+s"(a.strideE), "+s"(a.strideC), "+s"(a.strideCt), "+s"(a.lde),
                    "+s"(a.ldc), "+s"(a.ldct), "+s"(a.out_shift), "+s"(a.m_valid), "+s"(a.n_valid), "+s"(a.alpha), "+s"(a.beta), "+s"(a.diag_add));
  return a;
}
// acc += a * b on the matrix cores.  Inline assembly with the accumulator as a read-write operand: the builtin leaves the
// destination free, and over a software-pipelined loop the register allocator then rotates the accumulators with
// register moves between the MFMAs (measured: half the issue rate).  What the assembler statement hides from the compiler
// is kept by hand: an empty statement after the zero-initialisation keeps it away from the first MFMA, acc_settle() stands
// behind the last MFMA, and acc_touch() before every use of a result keeps that use behind acc_settle(), whose nops name no
// register (without it the compiler moved accumulator reads above the nops).  The epilogue touches one row of fragments at a
// time: all of them right after the nops cost one instantiation 64 spilled registers, one by one costs 2 to 5 % more
// instructions (waits inside each fragment).
template <bool HALF, bool AGPR>
__device__ __forceinline__ void mfma16(f32x4& acc, const u32x4& a, const u32x4& b) {
  if constexpr (AGPR) {
    if constexpr (HALF) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
  } else {
    if constexpr (HALF) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
  }
}
template <bool AGPR>
__device__ __forceinline__ void acc_touch(f32x4& acc) {
  if constexpr (AGPR) asm volatile("" : "+a"(acc));
  else asm volatile("" : "+v"(acc));
}
// 16-bit transpose read of four k-values of one column per lane; the result arrives later (see the kernel)
template <int OFF>
__device__ __forceinline__ void lds_tr_read(uint32_t addr, unsigned long long& raw) {
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(raw) : "v"(addr), "n"(OFF));
}
__device__ __forceinline__ void acc_settle() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// Tile t of a grid of dM x dN tiles that are all computed -> (ti, tj)
__device__ __forceinline__ void place_in_grid(int t, int dM, int dN, uint32_t inv_line, int& ti, int& tj) {
  if (dM > 8) {
    // A wide tile grid in blocks of 4 x 4 tiles, the blocks of one block row (4 row panels of P) one after the other:
    // the 32 tiles that an XCD works on at a time are two neighbouring blocks, 4 row panels of P and 8 of Q, 12 panels
    // per k-step.  Whole columns of dM tiles at a time would stream dM + 32 / dM panels (33 for dM = 32, 24 for 22).
    // The last block row and the last block of a row are as narrow as the grid leaves them (1 to 4 tiles).
    const int nbi = (dM + 3) >> 2, nbj = (dN + 3) >> 2;
    int r, bi = divide(t, 4 * dN, inv_line, r);
    if (bi >= nbi) { r += (bi - (nbi - 1)) * 4 * dN; bi = nbi - 1; }
    const int h = dM - 4 * bi < 4 ? dM - 4 * bi : 4;
    int bj = divide_1_to_4(r, h) >> 2;
    if (bj >= nbj) bj = nbj - 1;
    const int q = r - bj * 4 * h;
    const int qc = divide_1_to_4(q, h);
    ti = 4 * bi + (q - qc * h);
    tj = 4 * bj + qc;
  } else {
    tj = divide(t, dM, inv_line, ti);   // up to 8 row panels: whole columns, 8 x 4 tiles per XCD for dM = 8
  }
}

// F16 = 1: the workspace matrices (operands, addend, non-final outputs) are IEEE half instead of bfloat16 (the caller's
// tensors stay bfloat16); the host keeps them in range with power-of-two factors folded into alpha / beta / out_shift.
// F16 = 2: bfloat16 operands and addend, IEEE-half output (the step from a bfloat16 iteration to a half one).
// CUT: problems of the launch may carry a K-split (GemmParams::ksplit; symmetric products, 128x128 configuration).
// CUT_BLOCKS: the blocks that share a tile leave their fp32 accumulators in the workspace and the last one to arrive adds
// them up in the order of the parts and runs the epilogue.  CUT_SEQUENCE: one block walks all parts of its tile and adds up in the
// same order, in registers: the same bits for launches that fill the chip without the cut.
//
// One block is four waves (one per SIMD of a compute unit), wave (r, c) of the 2 x 2 arrangement computes rows
// r BT/2 .., columns c BT/2 .. of the BT x BT tile.  What bounds the 256 configuration is the LDS port and, at the power
// limit, the energy of operand movement: four waves of 128 x 128 read 128 KB of LDS per k-tile where eight waves of
// 128 x 64 read 192 KB, which with the 64 KB of copies is 2048 clk of LDS time per 2048 clk of matrix-core time.
// Measured on 16 x (2048 x 5632 x 2048), Gaussian operands: 1145 TFLOP/s with eight waves and 32x32x16 MFMAs, 1215 to 1240
// with four waves and 16x16x32 MFMAs, 1280 to 1300 with a third LDS stage for Q (zero operands, where power does not
// limit: 1320 / 1330 / 1525).  What a tile costs beside its k-tiles weighs little at this reduction of 2048 and at the power limit; where
// reductions are short X' = B X goes to ns_gemm_stream_kernel, whose copies run on into the next tile.
//
// LDS: SP stages of the P tile and SQ = SP + 1 of the Q tile.  The 256 configuration has room for 2 + 3: the
// operand that streams from memory (Q = X^T) gets two k-tiles of time to arrive, P, which the caches hold, gets one.
template <int BT, int SP, int SQ, int MODE, bool SPLIT, bool FINAL, bool ADDEND, int F16, int CUT>
__device__ __forceinline__ void ns_gemm_tile(const GroupedGemmParams& gp) {
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass does not know the buffer descriptor type)
  static_assert(BT == 256 || BT == 128 || BT == 64 || (BT == 32 && MODE == MODE_SYRKT && !SPLIT && CUT == CUT_NONE), "block tiles");
  constexpr bool SK = CUT == CUT_BLOCKS, SEQUENCE = CUT == CUT_SEQUENCE;
  static_assert(!(F16 && SPLIT), "the hi+lo pair is a bfloat16 device");
  static_assert(CUT == CUT_NONE || (BT == 128 && !SPLIT && !FINAL && MODE != MODE_BX), "the K-split serves symmetric products in the 128 configuration");
  static_assert(F16 != 2 || (MODE == MODE_BX && !FINAL), "only X' changes its storage type");
  constexpr bool IN16 = F16 == 1, OUT16 = F16 != 0;
  constexpr int NW = 4, NT = 256;
  constexpr int WT = BT / 2;            // side of a wave's sub-tile
  constexpr int FR = WT / 16;           // 16x16 fragments along a side of it
  constexpr bool AGPR = FR == 8;        // 256 accumulator registers per lane: they live in the accumulation half of the file
  constexpr int OPBYTES = BT * ROW_BYTES;   // one stage of one operand
  constexpr int NC = BT / 8 / NW;       // copies (1 KiB: 8 rows x 128 B) per wave, operand and k-tile
  static_assert(BT % (8 * NW) == 0, "tile rows must split over waves");
  static_assert(SP >= 2 && SQ == SP + 1, "stages");
  // MODE_SYRKT is MODE_SYRK with the operand given K-major: P = Q = X^T stored [K][M] (leading dimension ldp), so the
  // iteration needs no row-major copy of X at all; the MFMA fragments then come from LDS transpose reads
  constexpr bool KMAJ = (MODE == MODE_SYRKT);
  constexpr bool SYRK_PLAIN = (MODE == MODE_SYRK || MODE == MODE_SYRKT);   // alpha * product, no addend
  constexpr bool SYM = (SYRK_PLAIN || MODE == MODE_SYRK2);
  // SPLIT means "B is a hi+lo pair": SYRK2 WRITES the pair, BX READS it as a second pass over K
  constexpr bool KSPLIT = SPLIT && MODE == MODE_BX;
  // element codecs: workspace data is half or bfloat16; the final launch writes the caller's bfloat16
  auto dec = [](uint32_t bits) { return IN16 ? f16_to_f32((uint16_t)bits) : bf16_to_f32((uint16_t)bits); };
  auto enc = [](float f) { return (OUT16 && !FINAL) ? f16_bits(f) : bf16_bits(f); };
  auto pk4 = [&](float a, float b, float c, float d) {
    uint2 r;
    if constexpr (OUT16 && !FINAL) { r.x = f16_pair(a, b); r.y = f16_pair(c, d); }
    else { r.x = bf16_pair(a, b); r.y = bf16_pair(c, d); }
    return r;
  };

  extern __shared__ __attribute__((aligned(1024))) char smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;

  // ---- block -> (problem, matrix, tile).  Workgroups are dealt round-robin to the 8 XCDs; runs of 32
  // consecutive logical tiles (neighbouring tiles of one matrix: shared operand panels) are kept on ONE
  // XCD, i.e. in one L2, and successive runs go to successive XCDs so that long and short tiles of a
  // grouped launch spread evenly over the chip.  A launch of fewer than 8 * 32 tiles is dealt out in eight shorter runs:
  // runs of 32 would leave whole XCDs without work.
  // All of this is paid at the start of every tile, before its first copy: there is no division in it (the host sends
  // reciprocals), and it waits for the kernel arguments once - the first problem's come with the header, another
  // problem's take a second wait.  From the start of a tile to its first copy, with the accumulators cleared behind the copies
  // instead of before them: 1.1 to 2.2 -> 0.55 to 1.0 us (divisions and fields fetched where they are used before); the 64
  // expert matrices of 512 x 2048 and 2048 x 256 1375 -> 1320 us per step, one 512 x 2048 matrix 130 -> 123 us per call, both
  // together with the epilogue's paired conversions and running store addresses.
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  TileArgs p = fetch_tile_args(gp.g[0]);
  LaunchHead head = {gp.n_groups, gp.quarter, gp.backwards, gp.total, {gp.tile_start[1], gp.tile_start[2], gp.tile_start[3]}};
  pin(p, head);
  const int total = head.total, quarter = head.quarter;
  const int run = xcd_run(total);
  const int lap = total < 256 ? 0 : slot >> 5;   // (a launch of fewer than 256 tiles has `run` slots per XCD)
  int logical = (lap * 8 + xcd) * run + slot - lap * run;
  if (logical >= total) return;
  if (MODE == MODE_BX && head.backwards) logical = total - 1 - logical;
  int grp = 0, start = 0;
  auto from = [&](int i, int first) { if (logical >= first) { grp = i; start = first; } };   // (past every tile for i >= n_groups)
#pragma unroll
  for (int i = 1; i <= 3; ++i) from(i, head.first[i - 1]);
  if (head.n_groups > 4) {
#pragma unroll
    for (int i = 4; i < MAX_GROUPS; ++i) from(i, gp.tile_start[i]);
  }
  if (grp) {
    p = fetch_tile_args(gp.g[grp]);
    pin(p);
  }
  const GemmParams& g = gp.g[grp];
  int local = logical - start;
  int ks = 0;   // part of the K range this block walks
  if constexpr (SK) {
    while (local >= p.part_tiles) { local -= p.part_tiles; ++ks; }   // (up to `ksplit` parts)
  }
  const int sk_tile = local;   // this tile among the problem's tiles in the launch
  // grid the tile index is decoded in: the problem's own, or the coarser one whose tiles this launch quarters
  int quadrant = 0;
  const int dM = p.tilesM >> quarter, dN = p.tilesN >> quarter;
  if (quarter) {
    quadrant = local & ((1 << 2 * quarter) - 1);
    local = p.qt_first + (local >> 2 * quarter);
  }
  // the launch may cover only tiles [t_first, t_first + per_mat) of every matrix
  int t;
  const int b = divide(local, p.per_mat, p.inv_per_mat, t);
  t += p.t_first;
  int ti, tj;
  if (SYM && dM > 8) {
    // A large upper triangle in blocks of 4 x 4 tiles, block row by block row (a diagonal block holds the 10 tiles of
    // its own upper triangle): the 32 tiles that an XCD works on at a time are two neighbouring blocks, whose operand
    // panels are 4 + 8 row panels of the one matrix.  Row by row a run would be one row panel against 32 others.
    // The last block column is `last` (1 to 4) tiles wide, and the last diagonal block a triangle of that side.
    const int nb = (dM + 3) >> 2, last = dM - 4 * (nb - 1);
    int bi = 0, rowcount = 10 + (nb - 2) * 16 + 4 * last;
    while (bi < nb - 1 && t >= rowcount) { t -= rowcount; ++bi; rowcount -= 16; }
    const int side = bi == nb - 1 ? last : 4;
    if (t < side * (side + 1) / 2) {
      int i = 0, rowlen = side;                               // rows of the triangle hold side, side - 1, ... tiles
      while (t >= rowlen) { t -= rowlen; ++i; --rowlen; }
      ti = 4 * bi + i;
      tj = 4 * bi + i + t;
    } else {
      t -= 10;
      const int bj = bi + 1 + (t >> 4) < nb - 1 ? bi + 1 + (t >> 4) : nb - 1;
      const int w = t - 16 * (bj - bi - 1);                   // 0 .. 4 x (width of block bj) - 1
      ti = 4 * bi + (w & 3);
      tj = 4 * bj + (w >> 2);
    }
  } else if (SYM) {
    ti = 0;
    int rowlen = dM;
    while (t >= rowlen) { t -= rowlen; ++ti; --rowlen; }
    tj = ti + t;
  } else {
    place_in_grid(t, dM, dN, p.inv_line, ti, tj);
  }
  if (quarter) {
    ti = (ti << quarter) + (quadrant >> quarter);
    tj = (tj << quarter) + (quadrant & ((1 << quarter) - 1));
    if (SYM && ti > tj) return;   // lower part of a diagonal tile: its mirror image covers it
  }
  const int R0 = ti * BT, C0 = tj * BT;

  const char* Pb = KMAJ ? (const char*)(p.P + (size_t)b * p.strideP + R0)
                        : (const char*)(p.P + (size_t)b * p.strideP + (size_t)R0 * p.ldp);
  const char* Qb = KMAJ ? (const char*)(p.Q + (size_t)b * p.strideQ + C0)
                        : (const char*)(p.Q + (size_t)b * p.strideQ + (size_t)C0 * p.ldq);
  int KT = p.K / BK;
  if constexpr (SK) {
    // part ks of ksplit: k-tiles [ks KT / ksplit, (ks + 1) KT / ksplit), at least one (the host checks KT >= ksplit)
    const int kt0 = (int)((long)ks * KT / g.ksplit), kt1 = (int)((long)(ks + 1) * KT / g.ksplit);
    Pb += KMAJ ? (size_t)kt0 * BK * p.ldp * 2 : (size_t)kt0 * ROW_BYTES;
    Qb += KMAJ ? (size_t)kt0 * BK * p.ldq * 2 : (size_t)kt0 * ROW_BYTES;
    KT = kt1 - kt0;
  }
  const int KT_ALL = KSPLIT ? 2 * KT : KT;

  // ---- copies.  Buffer loads with a descriptor over the operand panel: the lane's place in the tile is a constant 32-bit
  // offset per copy, the k-tile a scalar one (the host keeps panels below 4 GiB), so a copy is one instruction and the
  // setting of M0.  The swizzle is folded into the SOURCE address of each lane, the LDS side is linear.
  uint32_t offP[NC], offQ[NC];
  auto lane_off = [&](int j, int ld) -> uint32_t {
    if constexpr (!KMAJ) {
      const int r = (wave * NC + j) * 8 + (lane >> 3);
      return (uint32_t)r * (uint32_t)ld * 2u + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    } else {
      constexpr int CPRK = BT / 8;   // chunks per k-row
      const int pidx = (wave * NC + j) * 64 + lane, k = pidx / CPRK, cpos = pidx % CPRK;
      return (uint32_t)k * (uint32_t)ld * 2u + (uint32_t)((cpos ^ kmaj_swz<BT>(k)) * 16);
    }
  };
#pragma unroll
  for (int j = 0; j < NC; ++j) {
    offP[j] = lane_off(j, p.ldp);
    offQ[j] = lane_off(j, p.ldq);
  }
  const uint32_t kstepP = KMAJ ? (uint32_t)BK * (uint32_t)p.ldp * 2u : (uint32_t)ROW_BYTES;
  const uint32_t kstepQ = KMAJ ? (uint32_t)BK * (uint32_t)p.ldq * 2u : (uint32_t)ROW_BYTES;
  const char* P2b = KSPLIT ? (const char*)(g.P2 + (size_t)b * p.strideP + (size_t)R0 * p.ldp) : Pb;
  // (the descriptors have to be seen to be uniform: each is a loop over the lanes otherwise)
  auto uniform = [](const char* q) {
    const uint64_t v = (uint64_t)q;
    return (void*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
  };
  void* const uP = uniform(Pb);
  void* const uQ = uniform(Qb);
  void* const uP2 = uniform(P2b);
  // What the copies of k-tile kt use.  Past the last k-tile the descriptor has no records: the load touches no memory, and
  // the main loop needs no tail without copies (three copies of its body cost registers where they meet).
  struct Source { __amdgpu_buffer_rsrc_t P, Q; uint32_t atP, atQ; };
  auto source = [&](int kt) __attribute__((always_inline)) {
    const int records = __builtin_amdgcn_readfirstlane(kt < KT_ALL ? -1 : 0);
    const int second = KSPLIT ? __builtin_amdgcn_readfirstlane(kt >= KT ? 1 : 0) : 0;
    const uint32_t k = (uint32_t)__builtin_amdgcn_readfirstlane(second ? kt - KT : kt);
    Source s = {__builtin_amdgcn_make_buffer_rsrc(second ? uP2 : uP, 0, records, 0x00027000),
                __builtin_amdgcn_make_buffer_rsrc(uQ, 0, records, 0x00027000), k * kstepP, k * kstepQ};
    return s;
  };
  // copy j of this wave of the P / Q tile into a stage (byte offset in LDS)
  auto copyP = [&](const Source& s, int stage, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.P, (lptr_t)(smem + stage + (wave * NC + j) * 1024), 16, (int)offP[j], (int)s.atP, 0, 0);
  };
  auto copyQ = [&](const Source& s, int stage, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.Q, (lptr_t)(smem + stage + (wave * NC + j) * 1024), 16, (int)offQ[j], (int)s.atQ, 0, 0);
  };
  constexpr int QBASE = SP * OPBYTES;   // the Q stages follow the P stages

  // first SP k-tiles, oldest first, on their way before anything else is set up (clearing 256 accumulators alone takes 1024 clk)
#pragma unroll
  for (int s = 0; s < SP; ++s) {
    const Source src = source(s);
#pragma unroll
    for (int j = 0; j < NC; ++j) copyQ(src, QBASE + s * OPBYTES, j);
#pragma unroll
    for (int j = 0; j < NC; ++j) copyP(src, s * OPBYTES, j);
  }
  __builtin_amdgcn_sched_barrier(0);

  f32x4 acc[FR][FR];
#pragma unroll
  for (int i = 0; i < FR; ++i)
#pragma unroll
    for (int j = 0; j < FR; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < FR; ++i)
#pragma unroll
    for (int j = 0; j < FR; ++j) acc_touch<AGPR>(acc[i][j]);
  const EndArgs out = end_args(g);   // (the wait for them falls into the one for the first copies)

  const int wr0 = (wave >> 1) * WT;     // wave origin inside the block tile
  const int wc0 = (wave & 1) * WT;
  // Diagonal tile of a symmetric product: wave (1, 0), whose sub-tile lies wholly BELOW the diagonal, computes nothing (it
  // only takes part in the copies and the barriers); its part of the tile is the mirror image of the sub-tile of wave
  // (0, 1), which writes it (a quarter of the tile's matrix-core work is saved).
  const bool diag = SYM && (ti == tj);
  const bool idle = diag && wave == 2;
  const bool above = diag && wave == 1;

  // ---- operand fragments.  A k-tile is two k-steps of 32.  Fragment f of a wave in k-step kk holds, in lane l16 + 16 lg, the
  // eight k-values 32 kk + 8 lg .. + 7 of row (column) 16 f + l16 of the wave's sub-tile: one 16-byte read.
  u32x4 af[2][FR], bq[2][FR];
  int rdP[2], rdQ[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    rdP[kk] = lds_chunk_off(wr0 + l16, 4 * kk + lg);
    rdQ[kk] = lds_chunk_off(wc0 + l16, 4 * kk + lg);
  }
  // K-major operands: a 16-lane group reads 4 k-rows x 16 columns with one LDS transpose read; lane s = 4e + a of the
  // group points at columns 4a..4a+3 of row k0 + e and receives, as lane 4a' + b', the 4 k-values of column 4a' + b'.
  // Two such reads (k0, k0 + 4) make the 8 k-values of a fragment; k0 = 32 kk + 8 lg.
  int trP[KMAJ ? FR : 1], trQ[KMAJ ? FR : 1];
  if constexpr (KMAJ) {
    const int e = l16 >> 2, a = l16 & 3, k = 8 * lg + e;   // kmaj_swz takes the same value for k + 4 and k + 32
#pragma unroll
    for (int f = 0; f < FR; ++f) {
      const int m = wr0 + f * 16 + 4 * a, n = wc0 + f * 16 + 4 * a;
      trP[f] = k * (BT * 2) + (((m >> 3) ^ kmaj_swz<BT>(k)) << 4) + ((m & 7) << 1);
      trQ[f] = k * (BT * 2) + (((n >> 3) ^ kmaj_swz<BT>(k)) << 4) + ((n & 7) << 1);
    }
  }
  // The transpose reads are inline assembly: the compiler makes the builtin wait for every outstanding global->LDS
  // copy (vmcnt(0)) before each read.  The compiler therefore does not know that their results arrive late.  The raw
  // results stay in variables of their own (afr / bqr, one 64-bit pair per read) that nothing touches until the explicit
  // s_waitcnt lgkmcnt(0) at the end of the k-step that reads them (the last read is a quarter of a k-step old by then); that
  // wait is followed by empty asm statements that take every raw result as a read-write operand, so each use (the
  // packing into an MFMA operand included) depends on a statement that comes after the wait, and none is in flight
  // where the loop closes.
  typedef unsigned long long u64;
  u64 afr[2][KMAJ ? FR : 1][2], bqr[2][KMAJ ? FR : 1][2];
  // LDS reads of a k-step into fragment set BUF: NRD of them (Q operand first: the first row of MFMAs needs all of it)
  constexpr int NRD = KMAJ ? 4 * FR : 2 * FR;
  auto fread = [&](auto buf_, int sP, int sQ, auto kk_, auto r_) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_)::value, kk = decltype(kk_)::value, r = decltype(r_)::value;
    if constexpr (!KMAJ) {
      if constexpr (r < FR) bq[buf][r] = *(const u32x4*)(smem + sQ + rdQ[kk] + r * 16 * ROW_BYTES);
      else af[buf][r - FR] = *(const u32x4*)(smem + sP + rdP[kk] + (r - FR) * 16 * ROW_BYTES);
    } else {
      constexpr int f = (r >> 1) % FR, h = r & 1, off = (32 * kk + 4 * h) * (BT * 2);
      if constexpr (r < 2 * FR) {
        const uint32_t addr = (uint32_t)(uintptr_t)(smem + sQ) + (uint32_t)trQ[f];
        lds_tr_read<off>(addr, bqr[buf][f][h]);
      } else {
        const uint32_t addr = (uint32_t)(uintptr_t)(smem + sP) + (uint32_t)trP[f];
        lds_tr_read<off>(addr, afr[buf][f][h]);
      }
    }
  };
  // K-major operands: wait for the transpose reads of fragment set BUF, then make fragments of them
  auto land = [&](auto buf_) __attribute__((always_inline)) {
    if constexpr (KMAJ) {
      constexpr int buf = decltype(buf_)::value;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
      for (int f = 0; f < FR; ++f) {
        asm volatile("" : "+v"(bqr[buf][f][0]), "+v"(bqr[buf][f][1]));
        asm volatile("" : "+v"(afr[buf][f][0]), "+v"(afr[buf][f][1]));
      }
#pragma unroll
      for (int f = 0; f < FR; ++f) {
        typedef u64 u64x2 __attribute__((ext_vector_type(2)));
        const u64x2 vb = {bqr[buf][f][0], bqr[buf][f][1]}, va = {afr[buf][f][0], afr[buf][f][1]};
        bq[buf][f] = __builtin_bit_cast(u32x4, vb);
        af[buf][f] = __builtin_bit_cast(u32x4, va);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- main loop.  The fragments of a k-step are read from LDS during the MFMAs of the k-step before it, and the copies
  // of later k-tiles are spread over the MFMAs too: every memory instruction is pinned behind an MFMA of its own
  // (sched_barrier fences).  Copies issued back to back hold the wave until the texture unit has accepted them (64 B per
  // clk and compute unit), and with one wave per SIMD nothing else runs meanwhile.
  // The barrier that publishes k-tile kt + 1 sits between the two k-steps of k-tile kt: by then every read of k-tile kt has
  // been issued and has returned (lgkmcnt(0)), so its stage is free for the copies that follow the barrier.
  constexpr int NMF = FR * FR;
  using Yes = std::true_type;
  using No = std::false_type;
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  // one k-step: MFMAs on fragment set CBUF (when ACTIVE), reads of k-step RKK of the stages at (rsP, rsQ) into the other
  // set, copies of P to stage dP (when CP) or of Q to stage dQ from src
  auto kstep = [&](auto active, auto cbuf_, int rsP, int rsQ, auto rkk_, auto cp, const Source& src, int dP, int dQ) __attribute__((always_inline)) {
    constexpr bool ACTIVE = decltype(active)::value, CP = decltype(cp)::value;
    constexpr int cbuf = decltype(cbuf_)::value;
    // reads within the first three quarters of the k-step, copies over all of it
    constexpr int RSPAN = NMF > 1 ? NMF * 3 / 4 : 1;
    static_for<NMF>([&](auto q_) __attribute__((always_inline)) {
      constexpr int q = decltype(q_)::value;
      if constexpr (ACTIVE) mfma16<IN16, AGPR>(acc[q / FR][q % FR], af[cbuf][q / FR], bq[cbuf][q % FR]);
      __builtin_amdgcn_sched_barrier(0);
      constexpr int c_lo = (q * NC + NMF - 1) / NMF, c_hi = ((q + 1) * NC + NMF - 1) / NMF;
      static_for<c_hi - c_lo>([&](auto d_) __attribute__((always_inline)) {
        constexpr int c = c_lo + decltype(d_)::value;
        if constexpr (CP) copyP(src, dP, c);
        else copyQ(src, dQ, c);
      });
      if constexpr (ACTIVE) {
        constexpr int r_lo = q < RSPAN ? (q * NRD + RSPAN - 1) / RSPAN : NRD, r_hi = q + 1 < RSPAN ? ((q + 1) * NRD + RSPAN - 1) / RSPAN : NRD;
        static_for<r_hi - r_lo>([&](auto d_) __attribute__((always_inline)) {
          fread(std::integral_constant<int, cbuf ^ 1>{}, rsP, rsQ, rkk_, std::integral_constant<int, r_lo + decltype(d_)::value>{});
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (ACTIVE) land(std::integral_constant<int, cbuf ^ 1>{});
  };
  auto nextP = [](int s) { return s + OPBYTES == SP * OPBYTES ? 0 : s + OPBYTES; };
  auto nextQ = [](int s) { return s + OPBYTES == QBASE + SQ * OPBYTES ? QBASE : s + OPBYTES; };
  // In k-tile kt: Q of k-tile kt + SP in the first k-step (its extra stage is the one of kt - 1, which is free), P of it after
  // the barrier.  In flight at the barrier, younger than what it publishes:
  constexpr int PAIR = 2 * NC;
  constexpr int INFLIGHT = (SP - 2) * PAIR + NC;
  f32x4 sum[SEQUENCE ? FR : 1][SEQUENCE ? FR : 1] = {};   // CUT_SEQUENCE: the parts that are done
  auto k_range = [&](auto active) __attribute__((always_inline)) {
    constexpr bool ACTIVE = decltype(active)::value;
    int sP = 0, sQ = QBASE;               // stages of k-tile kt
    if constexpr (BT == 32) {
      // A wave has one MFMA per k-step here, and what a k-step takes is the wait for its LDS reads: a whole k-tile at a time, the
      // reads of the next one behind the MFMAs of this one that used their registers (X X^T of 512 x 8192 188.6 -> 183.5 us a call;
      // tiles of 64, which the LDS port bounds, are 1 to 2 % slower so).
      auto reads = [&](auto kk_, int stP, int stQ) __attribute__((always_inline)) {
        if constexpr (ACTIVE) static_for<NRD>([&](auto r_) __attribute__((always_inline)) { fread(kk_, stP, stQ, kk_, r_); });
      };
      auto multiply = [&](auto kk_) __attribute__((always_inline)) {
        constexpr int kk = decltype(kk_)::value;
        if constexpr (ACTIVE) mfma16<IN16, AGPR>(acc[0][0], af[kk][0], bq[kk][0]);
        __builtin_amdgcn_sched_barrier(0);
      };
      auto arrive = [&]() __attribute__((always_inline)) {
        if constexpr (ACTIVE) { land(I0{}); land(I1{}); }
      };
      reads(I0{}, 0, QBASE);
      reads(I1{}, 0, QBASE);
      arrive();
      for (int kt = 0; kt < KT_ALL; ++kt) {
        const int nP = nextP(sP), nQ = nextQ(sQ), pQ = sQ == QBASE ? QBASE + (SQ - 1) * OPBYTES : sQ - OPBYTES;
        const Source src = source(kt + SP);
        wait_copies<(SP - 2) * PAIR>();   // k-tile kt + 1 has landed, and every wave has its fragments of kt
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        multiply(I0{});
        reads(I0{}, nP, nQ);
        multiply(I1{});
        reads(I1{}, nP, nQ);
        copyQ(src, pQ, 0);
        copyP(src, sP, 0);
        __builtin_amdgcn_sched_barrier(0);
        arrive();
        sP = nP;
        sQ = nQ;
      }
      return;
    }
    if constexpr (ACTIVE) {
      static_for<NRD>([&](auto r_) __attribute__((always_inline)) { fread(I0{}, 0, QBASE, I0{}, r_); });
      land(I0{});
    }
    int kt = 0;
    auto walk = [&](int end) __attribute__((always_inline)) {   // k-tiles kt .. end - 1
      for (; kt < end; ++kt) {
        const int nP = nextP(sP), nQ = nextQ(sQ);
        // the Q stage before this one in the ring is the one that k-tile kt + SP goes to
        const int pQ = sQ == QBASE ? QBASE + (SQ - 1) * OPBYTES : sQ - OPBYTES;
        const Source src = source(kt + SP);
        kstep(active, I0{}, sP, sQ, I1{}, No{}, src, 0, pQ);
        wait_copies<INFLIGHT>();
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        kstep(active, I1{}, nP, nQ, I0{}, Yes{}, src, sP, 0);
        sP = nP;
        sQ = nQ;
      }
    };
    if constexpr (!SEQUENCE) {
      walk(KT_ALL);
    } else {
      // part by part; a part's sum joins those before it, and the next part starts from zero
      for (int part = 1; part <= g.ksplit; ++part) {
        walk((int)((long)part * KT / g.ksplit));
        if constexpr (ACTIVE) {
          acc_settle();
#pragma unroll
          for (int i = 0; i < FR; ++i)
#pragma unroll
            for (int j = 0; j < FR; ++j) {
              acc_touch<AGPR>(acc[i][j]);
              sum[i][j] += acc[i][j];
              acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
              acc_touch<AGPR>(acc[i][j]);
            }
          acc_settle();   // (and these writes are away from the next MFMA)
        }
      }
    }
  };

  // (k-tile 0 has landed once only the copies of the younger ones are outstanding)
  wait_copies<(SP - 1) * PAIR>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (SYM) {
    if (idle) {   // the same copies and barriers as its block, nothing else
      k_range(No{});
      wait_copies<0>();
      if constexpr (SK) {
        if (g.ksplit > 1) {
          __syncthreads();
          __syncthreads();
          if (!*(volatile int*)smem) return;
        }
      }
      if constexpr (BT > 32) __syncthreads();   // (the one before the epilogue)
      return;
    }
  }
  k_range(Yes{});
  wait_copies<0>();   // (copies without records included: the epilogue reuses the stages)
  acc_settle();
  if constexpr (SEQUENCE) {
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
      for (int j = 0; j < FR; ++j) acc[i][j] = sum[i][j];
  }

  // ---- epilogue.  acc[i][j][e] of lane l is element
  //   r = wr0 + 16 i + 4 (l / 16) + e  (row in the tile),   c = wc0 + 16 j + l % 16  (column)
  // so a lane owns 4 consecutive rows of one column.  Every global access of the epilogue goes through
  // LDS (the operand stages are dead by now) so that it is a 16-byte, row-contiguous access:
  // scattered 8-byte / 2-byte global accesses straight from the accumulator layout flood L2 with
  // partial-line requests and cost a quarter of the kernel.
  if constexpr (SK) {
    if (g.ksplit > 1) {
      // Every part leaves its accumulators in the workspace (accumulator layout: one word per lane and accumulator
      // register, so every access of a wave is a run of 256 bytes), waits until they have arrived, and counts itself in.
      // The block that finds itself last adds ALL parts in the order 0, 1, ... (its own from memory like the others: the
      // sum of a tile is the same whichever block came last) and goes on to the epilogue; the others are done.  Nobody
      // waits for anybody.  The partial results travel as system-scope accesses (written through, read past the
      // caches): the eight L2 caches of the chip are not coherent with each other, and the alternative - a release /
      // acquire fence per block - writes back and invalidates a whole L2 each time (measured: the product twice as slow).
      int* sk_last = (int*)smem;   // the operand stages are dead after the barrier below
      float* part = g.sk_partial + (size_t)sk_tile * g.ksplit * (BT * BT);
      float* dst = part + (size_t)ks * (BT * BT);
#pragma unroll
      for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FR; ++j) {
          acc_touch<AGPR>(acc[i][j]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            __hip_atomic_store(dst + ((i * FR + j) * 4 + e) * NT + tid, acc[i][j][e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this lane's stores have been acknowledged
      __syncthreads();
      if (tid == 0) {
        const int old = __hip_atomic_fetch_add(g.sk_counter + sk_tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int last = old == g.ksplit - 1;
        if (last) __hip_atomic_store(g.sk_counter + sk_tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // for the next launch
        *sk_last = last;
      }
      __syncthreads();
      if (!*sk_last) return;
#pragma unroll
      for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FR; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int sidx = 0; sidx < g.ksplit; ++sidx) {
        const float* src = part + (size_t)sidx * (BT * BT);
#pragma unroll
        for (int i = 0; i < FR; ++i)
#pragma unroll
          for (int j = 0; j < FR; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[i][j][e] += __hip_atomic_load(src + ((i * FR + j) * 4 + e) * NT + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
  // optional per-matrix scale of the operand that was left out of it (deferred normalisation): the product of two
  // such operands carries sc^2, a product with one of them (and its addend) carries sc
  const float sc = out.scale ? out.scale[b] : 1.f;
  const float bx_sc = sc * __builtin_ldexpf(1.f, out.out_shift);   // MODE_BX: scale of the result (a power of two from the host)
  const float alpha = SYRK_PLAIN ? out.alpha * sc * sc : out.alpha, beta = out.beta;
  if constexpr (BT == 32) {
    // One fragment per wave, stored straight from the registers (a lane has four consecutive rows of one column).  On the
    // diagonal the fragment is its own mirror image.
    acc_touch<AGPR>(acc[0][0]);
    const uint2 bits = pk4(acc[0][0][0] * alpha, acc[0][0][1] * alpha, acc[0][0][2] * alpha, acc[0][0][3] * alpha);
    const int r = R0 + wr0 + 4 * lg, c = C0 + wc0 + l16;
    __bf16* const base = (__bf16*)out.C + (size_t)b * out.strideC;
    *(uint2*)(base + (size_t)c * out.ldc + r) = bits;
    if (!diag || above) {
      const uint16_t e[4] = {(uint16_t)bits.x, (uint16_t)(bits.x >> 16), (uint16_t)bits.y, (uint16_t)(bits.y >> 16)};
#pragma unroll
      for (int q = 0; q < 4; ++q) ((uint16_t*)base)[(size_t)(r + q) * out.ldc + c] = e[q];
    }
    return;
  }
  // A diagonal tile of a product of a matrix with ITSELF is symmetric bit for bit as it comes out of the matrix cores
  // (element (i,j) and element (j,i) are the same products summed in the same order over k), so it is stored like any
  // other tile, as one image.  A diagonal tile of P Q^T with two different (commuting, symmetric) matrices is symmetric
  // only up to rounding: it keeps its upper half and reflects it.
  const bool reflect = MODE == MODE_SYRK && diag && !(p.P == p.Q && p.strideP == p.strideQ && p.ldp == p.ldq);

  __syncthreads();  // every wave is done reading the operand stages
  // Wave-local: each wave stages its own WT x WT sub-tile in its own LDS region as the transposed image
  // W[c][r] (c = column in the sub-tile, r = row), so nothing below needs a block barrier:
  //   addend in:   16-byte direct copies of E[col][row..] rows into W, read back 8 bytes per lane
  //   W <- values: 8-byte LDS writes (a lane owns 4 consecutive r of one c), in place of the addend it has read
  //   transposed / mirrored image out: 16-byte reads of W rows -> 16-byte stores, up to 256 B contiguous per row
  //   row-major image out: LDS transpose reads (ds_read_b64_tr_b16: a lane receives 4 consecutive c of one
  //     r; two of them make 16 bytes) -> 16-byte stores, 64 B contiguous per row
  // The values are formed where they are packed, fragment by fragment: 256 accumulators updated in place would not fit
  // beside their copies in the register file.
  constexpr int WROW = WT * 2;                  // bytes per W row
  constexpr int RCH = WT / 8;                   // 16-byte chunks per W row
  constexpr int WBYTES = WT * WROW;
  constexpr int WSLABS = WBYTES / 1024;         // 64-chunk slabs of one region
  static_assert(NW * WBYTES <= (SP + SQ) * OPBYTES, "wave regions must fit in the operand stages");
  char* W = smem + wave * WBYTES;
  // chunk swizzle: the 8-byte accesses of 16 columns, and the four W rows of a transpose read, fall on different banks
  auto sw = [](int c) {
    if constexpr (RCH == 16) return ((c & 7) << 1) | ((c >> 3) & 1);
    else if constexpr (RCH == 8) return (((c >> 1) & 3) << 1) | ((c >> 3) & 1);
    else return (((c >> 2) & 1) << 1) | ((c >> 3) & 1);
  };
  constexpr int SLAB_ROWS = 64 / RCH;           // W rows of a slab; sw() repeats after SW_PERIOD slabs
  constexpr int SW_PERIOD = RCH == 16 ? 4 : (RCH == 8 ? 2 : 1);
  auto w_off = [&](int c, int r) { return c * WROW + (((r >> 3) ^ sw(c)) << 4) + ((r & 7) << 1); };
  const int wrow0 = R0 + wr0, wcol0 = C0 + wc0;  // global origin of this wave's sub-tile

  // MODE_BX without an addend (ADDEND = false): a*I was folded into B's diagonal by the product that made B
  constexpr bool has_e = !SYRK_PLAIN && (MODE != MODE_BX || ADDEND);
  const bool on_diag = diag && wr0 == wc0;       // the diagonal of the matrix runs through fragments (f, f) of this wave
  // PART 0: the values (high halves of a split pair); PART 1: the low halves, value - bf16(value)
  auto emit = [&](auto part_, __bf16* Cdst) __attribute__((always_inline)) {
    constexpr int PART = decltype(part_)::value;
    if constexpr (has_e) {
      if constexpr (PART == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the reads of the high half's image
      // as in the main loop: a descriptor, a constant offset per lane and a scalar one per slab
      void* const Eb = uniform((const char*)(out.E + (size_t)b * out.strideE + (size_t)wcol0 * out.lde + wrow0));
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(Eb, 0, -1, 0x00027000);
      uint32_t off[SW_PERIOD];
#pragma unroll
      for (int t = 0; t < SW_PERIOD; ++t)
        off[t] = (uint32_t)(lane / RCH) * (uint32_t)out.lde * 2u + (uint32_t)(((lane % RCH) ^ sw(t * SLAB_ROWS + lane / RCH)) * 16);
#pragma unroll
      for (int t = 0; t < WSLABS; ++t)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lptr_t)(W + t * 1024), 16, (int)off[t % SW_PERIOD], (int)(t * SLAB_ROWS * (uint32_t)out.lde * 2u), 0, 0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
#pragma unroll
    for (int i = 0; i < FR; ++i) {
#pragma unroll
      for (int j = 0; j < FR; ++j) acc_touch<AGPR>(acc[i][j]);
#pragma unroll
      for (int j = 0; j < FR; ++j) {
        const int c = j * 16 + l16, r = i * 16 + 4 * lg;
        float v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = acc[i][j][q];
        if constexpr (SYRK_PLAIN) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] *= alpha;
        } else if constexpr (has_e) {
          const uint2 e = *(const uint2*)(W + w_off(c, r));
          const float ev[4] = {dec(e.x & 0xffff), dec(e.x >> 16), dec(e.y & 0xffff), dec(e.y >> 16)};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if constexpr (MODE == MODE_SYRK2) v[q] = fmaf(alpha, v[q], beta * ev[q]);
            else v[q] = fmaf(alpha, ev[q], v[q]) * bx_sc;
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] *= bx_sc;
        }
        if constexpr (MODE == MODE_SYRK2) {   // B + a I
          if (i == j && on_diag) {
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] += (4 * lg + q == l16) ? out.diag_add : 0.f;
          }
        }
        if constexpr (PART == 1) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] -= bf16_to_f32(bf16_bits(v[q]));
        }
        if (MODE == MODE_SYRK && reflect && on_diag) {
          // upper half to both of its places
          if (i <= j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              if (i < j || r + q <= c) {
                const uint16_t bits = enc(v[q]);
                *(uint16_t*)(W + w_off(c, r + q)) = bits;
                *(uint16_t*)(W + w_off(r + q, c)) = bits;
              }
            }
          }
        } else {
          *(uint2*)(W + w_off(c, r)) = pk4(v[0], v[1], v[2], v[3]);
        }
        if ((j & 1) == 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    // transposed / mirrored image: rows of W
    __bf16* Tdst = SYM ? Cdst : (__bf16*)out.Ct;
    if (Tdst && (!diag || above)) {   // in a diagonal tile: only the image of the idle wave's part
      const long tbs = SYM ? out.strideC : out.strideCt;
      const int tld = SYM ? out.ldc : out.ldct;
      __bf16* base = Tdst + (size_t)b * tbs;
      const int row = lane / RCH, ch = lane % RCH;   // of a slab of SLAB_ROWS rows of W; W's rows are the tile's columns
      auto slab = [&](int t) { return *(const u32x4*)(W + t * 1024 + row * WROW + ((ch ^ sw(t * SLAB_ROWS + row)) << 4)); };
      using store_t = std::conditional_t<FINAL, u32x4_any, u32x4>;
      if (!FINAL || (wcol0 + WT <= out.n_valid && wrow0 + WT <= out.m_valid)) {
        char* to = (char*)(base + (size_t)(wcol0 + row) * tld + wrow0 + ch * 8);
        static_for<WSLABS>([&](auto t_) __attribute__((always_inline)) {
          constexpr int t = decltype(t_)::value;
          *(store_t*)(to + (long)(t * SLAB_ROWS * 2) * tld) = slab(t);
          if constexpr (t % 8 == 7) __builtin_amdgcn_sched_barrier(0);
        });
      } else {
#pragma unroll 4
        for (int t = 0; t < WSLABS; ++t) {
          const u32x4 val = slab(t);
          const int orow = wcol0 + t * SLAB_ROWS + row, ocol = wrow0 + ch * 8;
          if (orow < out.n_valid) {
            if (ocol + 7 < out.m_valid) {
              *(u32x4_any*)(base + (size_t)orow * tld + ocol) = val;
            } else {
              const uint32_t w[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
              for (int k = 0; k < 8; ++k)
                if (ocol + k < out.m_valid) ((uint16_t*)base)[(size_t)orow * tld + ocol + k] = (uint16_t)(w[k >> 1] >> ((k & 1) * 16));
            }
          }
        }
      }
    }
    // row-major image: transpose reads.  In a 16-lane group, source lane s points at W[c0 + s/4][r0 + 4*(s%4) ..+3];
    // lane L of the group then holds W[c0 .. c0+3][r0 + L].
    if (SYM || out.C) {
      __bf16* base = Cdst + (size_t)b * out.strideC;
      const int s = l16;
      // 16 rows, from row rb * 16 on, of the eight columns from cb * 32 + lg * 8 on
      auto rows16 = [&](int rb, int cb) {
        const int c0 = cb * 32 + lg * 8;
        const s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(W + w_off(c0 + (s >> 2), rb * 16 + 4 * (s & 3))));
        const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(W + w_off(c0 + 4 + (s >> 2), rb * 16 + 4 * (s & 3))));
        const uint2 lo = __builtin_bit_cast(uint2, lo4), hi = __builtin_bit_cast(uint2, hi4);
        return u32x4{lo.x, lo.y, hi.x, hi.y};
      };
      using store_t = std::conditional_t<FINAL, u32x4_any, u32x4>;
      if (!FINAL || (wcol0 + WT <= out.n_valid && wrow0 + WT <= out.m_valid)) {
        char* to = (char*)(base + (size_t)(wrow0 + s) * out.ldc + wcol0 + lg * 8);
        static_for<WT / 16>([&](auto rb_) __attribute__((always_inline)) {
          constexpr int rb = decltype(rb_)::value;
          static_for<WT / 32>([&](auto cb_) __attribute__((always_inline)) {
            constexpr int cb = decltype(cb_)::value;
            *(store_t*)(to + (long)(rb * 32) * out.ldc + cb * 64) = rows16(rb, cb);
          });
          if constexpr (rb % 2 == 1) __builtin_amdgcn_sched_barrier(0);
        });
      } else {
#pragma unroll 2
        for (int rb = 0; rb < WT / 16; ++rb)
#pragma unroll
          for (int cb = 0; cb < WT / 32; ++cb) {
            const u32x4 val = rows16(rb, cb);
            const int orow = wrow0 + rb * 16 + s, ocol = wcol0 + cb * 32 + lg * 8;
            if (orow < out.m_valid) {
              if (ocol + 7 < out.n_valid) {
                *(u32x4_any*)(base + (size_t)orow * out.ldc + ocol) = val;
              } else {
                const uint32_t w[4] = {val.x, val.y, val.z, val.w};
#pragma unroll
                for (int k = 0; k < 8; ++k)
                  if (ocol + k < out.n_valid) ((uint16_t*)base)[(size_t)orow * out.ldc + ocol + k] = (uint16_t)(w[k >> 1] >> ((k & 1) * 16));
              }
            }
          }
      }
    }
  };
  emit(I0{}, (__bf16*)out.C);
  if constexpr (SPLIT && MODE == MODE_SYRK2) emit(I1{}, g.C2);
#endif
}

// X' = B X in tiles of 256, a block's tiles one after the other: the k-tiles of all of them are ONE stream, the copies run on from the last
// k-tiles of a tile to the first ones of the next, which arrive during the epilogue, and the epilogue takes no LDS (the stages hold
// the next tile by then).  What bounds a lone tile of ns_gemm_tile at short reductions is its boundary - set-up, first copies, epilogue
// and hand-over are 20 of 40 thousand clocks at K = 512, with the matrix cores idle; here 5 are left, the epilogue's.  us per launch,
// tile by tile / as a stream: 64 x (512 x 2048) + 64 x (256 x 2048) 116 / 102 (with the addend 137 / 127, final 123 / 105; 4.4 TB/s of
// operands and results are what bounds it then), the EMA-Muon set of width 1024 (K = 1024, 688 tiles) 91 / 86.
// The arithmetic of an element is that of ns_gemm_tile (same sums, same epilogue roundings): the same bits.
//   epilogue  A lane has four consecutive rows of one column in every fragment.  Two fragments below one another make eight of them with
//             one exchange between neighbouring groups of 16 lanes (v_permlane16_swap): 16-byte stores, 64 bytes of each of 16 rows of
//             X'^T per instruction and 256 by four.  The addend comes the same way, all of it before the first store (loads return
//             in order behind stores): half of it during the last k-tile, half at the start of the epilogue, when the
//             fragments of the second k-step are dead.
//   final     A result wanted in rows (X', not X'^T) is the same computation with the operands' parts exchanged.
//   waits     The stores of a tile are younger than the copies of the next tile's first two k-tiles and older than the
//             rest: vector-memory operations complete in order, so the first wait of a tile leaves them outstanding.
__device__ __forceinline__ void* uniform_ptr(const void* q) {
  const uint64_t v = (uint64_t)q;
  return (void*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

template <bool FINAL, bool ADDEND, int F16>
__global__ void __launch_bounds__(256, 1) ns_gemm_stream_kernel(const GroupedGemmParams gp) {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(!(F16 == 2 && FINAL), "the final launch writes the caller's bfloat16");
  constexpr bool IN16 = F16 == 1, OUT16 = F16 != 0 && !FINAL;
  constexpr int BT = 256, WT = 128, FR = 8, NC = 8, SP = 2, SQ = 3, OPBYTES = BT * ROW_BYTES, QBASE = SP * OPBYTES;
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int wr0 = (wave >> 1) * WT, wc0 = (wave & 1) * WT;

  // this block's tiles: every gridDim-th, from the run of its XCD on
  const int total = gp.total, backwards = gp.backwards, step = (int)gridDim.x;
  int index = (int)(blockIdx.x & 7) * (step >> 3) + (int)(blockIdx.x >> 3);
  if (index >= total) return;

  struct Args {
    const __bf16 *P, *Q, *E;
    __bf16* Ct;
    const float* scale;
    long strideP, strideQ, strideE, strideCt;
    int ld, K, tilesM, tilesN, per_mat, lde, ldct, out_shift;
    uint32_t inv_per_mat, inv_line;
    float alpha;
  };
  int grp = -1;
  bool rows = false;   // of this problem X' is wanted, not X'^T
  Args a = {};
  struct End { char* to; const char* e; int ld, lde; float alpha, factor; };
  struct Place { const char *P, *Q; int KT; End end; };
  auto locate = [&](int i) __attribute__((always_inline)) {
    const int logical = backwards ? total - 1 - i : i;
    int now = 0;
#pragma unroll
    for (int k = 1; k < MAX_GROUPS; ++k) if (logical >= gp.tile_start[k]) now = k;   // (past every tile for k >= n_groups)
    if (now != grp) {
      const GemmParams& g = gp.g[now];
      rows = FINAL && g.C;
      a = Args{g.P, g.Q, g.E, rows ? g.C : g.Ct, g.scale, g.strideP, g.strideQ, g.strideE, rows ? g.strideC : g.strideCt, g.ldp, g.K, g.tilesM,
               g.tilesN, g.per_mat, g.lde, rows ? g.ldc : g.ldct, g.out_shift, g.inv_per_mat, g.inv_line, g.alpha};
      grp = now;
    }
    int t, ti, tj;
    const int b = divide(logical - gp.tile_start[now], a.per_mat, a.inv_per_mat, t);
    place_in_grid(t, a.tilesM, a.tilesN, a.inv_line, ti, tj);
    const int R0 = ti * BT, C0 = tj * BT;
    Place p;
    const char* const ofB = (const char*)(a.P + (size_t)b * a.strideP + (size_t)R0 * a.ld);
    const char* const ofX = (const char*)(a.Q + (size_t)b * a.strideQ + (size_t)C0 * a.ld);
    p.P = rows ? ofX : ofB;
    p.Q = rows ? ofB : ofX;
    p.KT = a.K / BK;
    p.end.to = (char*)(a.Ct + (size_t)b * a.strideCt + (rows ? (size_t)R0 * a.ldct + C0 : (size_t)C0 * a.ldct + R0));
    p.end.e = ADDEND ? (const char*)(a.E + (size_t)b * a.strideE + (size_t)C0 * a.lde + R0) : nullptr;
    p.end.ld = a.ldct;
    p.end.lde = a.lde;
    p.end.alpha = a.alpha;
    // (constant memory as far as this launch goes: a scalar load, where a vector one would wait for every copy in flight)
    p.end.factor = (ADDEND && a.scale ? ((const __attribute__((address_space(4))) float*)(uintptr_t)a.scale)[b] : 1.f) * __builtin_ldexpf(1.f, a.out_shift);
    return p;
  };

  Place next = locate(index);
  // ---- copies (see ns_gemm_tile): the state of what is copied next
  int off_ld = a.ld;
  uint32_t off[NC];
  auto lane_offsets = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int r = (wave * NC + j) * 8 + (lane >> 3);
      off[j] = (uint32_t)r * (uint32_t)off_ld * 2u + (uint32_t)(((lane & 7) ^ ((r >> 1) & 7)) * 16);
    }
  };
  lane_offsets();
  void *cP = uniform_ptr(next.P), *cQ = uniform_ptr(next.Q);
  int ck = 0, cKT = next.KT, records = -1;
  struct Source { __amdgpu_buffer_rsrc_t P, Q; uint32_t at; };
  auto source = [&]() __attribute__((always_inline)) {
    return Source{__builtin_amdgcn_make_buffer_rsrc(cP, 0, records, 0x00027000), __builtin_amdgcn_make_buffer_rsrc(cQ, 0, records, 0x00027000),
                  (uint32_t)ck * (uint32_t)ROW_BYTES};
  };
  auto copyP = [&](const Source& s, int stage, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.P, (lptr_t)(smem + stage + (wave * NC + j) * 1024), 16, (int)off[j], (int)s.at, 0, 0);
  };
  auto copyQ = [&](const Source& s, int stage, int j) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(s.Q, (lptr_t)(smem + stage + (wave * NC + j) * 1024), 16, (int)off[j], (int)s.at, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < SP; ++s) {
    const Source src = source();
#pragma unroll
    for (int j = 0; j < NC; ++j) copyQ(src, QBASE + s * OPBYTES, j);
#pragma unroll
    for (int j = 0; j < NC; ++j) copyP(src, s * OPBYTES, j);
    ++ck;
  }
  __builtin_amdgcn_sched_barrier(0);

  f32x4 acc[FR][FR];
#pragma unroll
  for (int i = 0; i < FR; ++i)
#pragma unroll
    for (int j = 0; j < FR; ++j) { acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f}; acc_touch<true>(acc[i][j]); }

  u32x4 af[2][FR], bq[2][FR];
  int rdP[2], rdQ[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    rdP[kk] = lds_chunk_off(wr0 + l16, 4 * kk + lg);
    rdQ[kk] = lds_chunk_off(wc0 + l16, 4 * kk + lg);
  }
  constexpr int NRD = 2 * FR, NMF = FR * FR, RSPAN = NMF * 3 / 4;
  auto fread = [&](auto buf_, int sP, int sQ, auto kk_, auto r_) __attribute__((always_inline)) {
    constexpr int buf = decltype(buf_)::value, kk = decltype(kk_)::value, r = decltype(r_)::value;
    if constexpr (r < FR) bq[buf][r] = *(const u32x4*)(smem + sQ + rdQ[kk] + r * 16 * ROW_BYTES);
    else af[buf][r - FR] = *(const u32x4*)(smem + sP + rdP[kk] + (r - FR) * 16 * ROW_BYTES);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  // one k-step, as in ns_gemm_tile; the first one copies Q, the second one P
  auto kstep = [&](auto cbuf_, int rsP, int rsQ, const Source& src, int dst) __attribute__((always_inline)) {
    constexpr int cbuf = decltype(cbuf_)::value;
    static_for<NMF>([&](auto q_) __attribute__((always_inline)) {
      constexpr int q = decltype(q_)::value;
      mfma16<IN16, true>(acc[q / FR][q % FR], af[cbuf][q / FR], bq[cbuf][q % FR]);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (q % (NMF / NC) == 0) {
        if constexpr (cbuf == 1) copyP(src, dst, q / (NMF / NC));
        else copyQ(src, dst, q / (NMF / NC));
      }
      constexpr int r_lo = q < RSPAN ? (q * NRD + RSPAN - 1) / RSPAN : NRD, r_hi = q + 1 < RSPAN ? ((q + 1) * NRD + RSPAN - 1) / RSPAN : NRD;
      static_for<r_hi - r_lo>([&](auto d_) __attribute__((always_inline)) {
        fread(std::integral_constant<int, cbuf ^ 1>{}, rsP, rsQ, std::integral_constant<int, cbuf ^ 1>{}, std::integral_constant<int, r_lo + decltype(d_)::value>{});
      });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto nextP = [](int s) { return s ? 0 : OPBYTES; };
  auto nextQ = [](int s) { return s == QBASE + (SQ - 1) * OPBYTES ? QBASE : s + OPBYTES; };

  wait_copies<2 * NC>();
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  static_for<NRD>([&](auto r_) __attribute__((always_inline)) { fread(I0{}, 0, QBASE, I0{}, r_); });
  int sP = 0, sQ = QBASE;
  constexpr int STORES = FR * FR / 2;   // of a wave and tile
  bool first = true;
  for (;;) {
    const End end = next.end;
    const int KT = next.KT;
    const int row = wc0 + l16, col = wr0 + 16 * (lg & 1) + 8 * (lg >> 1);   // of the tile in X'^T: this lane's first 16 bytes
    u32x4 add[ADDEND ? FR : 1][ADDEND ? FR / 2 : 1];
    auto fetch_addend = [&](auto j_) __attribute__((always_inline)) {
      constexpr int j = decltype(j_)::value;
      const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(end.e), 0, -1, 0x00027000);
#pragma unroll
      for (int i = 0; i < FR / 2; ++i)
        add[j][i] = __builtin_amdgcn_raw_buffer_load_b128(from, (row * end.lde + col) * 2 + i * 64, j * 32 * end.lde, 0);
    };
    for (int kt = 0; kt < KT; ++kt) {
      if (ck == cKT) {   // the next copies are those of the block's next tile, if it has one
        index += step;
        records = index < total ? -1 : 0;
        if (index < total) {
          next = locate(index);
          cP = uniform_ptr(next.P);
          cQ = uniform_ptr(next.Q);
          cKT = next.KT;
          if (a.ld != off_ld) { off_ld = a.ld; lane_offsets(); }
        }
        ck = 0;
      }
      if constexpr (ADDEND) {
        if (kt == KT - 1) static_for<FR / 2>([&](auto j_) __attribute__((always_inline)) { fetch_addend(j_); });
      }
      const Source src = source();
      ++ck;
      const int nP = nextP(sP), nQ = nextQ(sQ), pQ = sQ == QBASE ? QBASE + (SQ - 1) * OPBYTES : sQ - OPBYTES;
      kstep(I0{}, sP, sQ, src, pQ);
      // the stores of the tile before this one are younger than what the barrier publishes
      if (kt == 0 && !first) wait_copies<STORES + NC>();
      else wait_copies<NC>();
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      kstep(I1{}, nP, nQ, src, sP);
      sP = nP;
      sQ = nQ;
    }
    acc_settle();
    // ---- epilogue, straight from the registers
    {
      const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(end.to), 0, -1, 0x00027000);
      const int at = (row * end.ld + col) * 2;
      if constexpr (ADDEND) {   // (before the first store: loads return in order behind stores)
        static_for<FR / 2>([&](auto j_) __attribute__((always_inline)) { fetch_addend(std::integral_constant<int, FR / 2 + decltype(j_)::value>{}); });
        __builtin_amdgcn_sched_barrier(0);
      }
      static_for<FR>([&](auto j_) __attribute__((always_inline)) {
        constexpr int j = decltype(j_)::value;
#pragma unroll
        for (int i = 0; i < FR; ++i) acc_touch<true>(acc[i][j]);
        static_for<FR / 2>([&](auto p_) __attribute__((always_inline)) {
          constexpr int i = 2 * decltype(p_)::value;
          uint2 half[2], e[2];
          if constexpr (ADDEND) {   // (the exchange of the result, the other way round)
            const u32x4 w = add[j][i / 2];
            const auto x = __builtin_amdgcn_permlane16_swap(w[0], w[2], false, false);
            const auto y = __builtin_amdgcn_permlane16_swap(w[1], w[3], false, false);
            e[0] = make_uint2(x[0], y[0]);
            e[1] = make_uint2(x[1], y[1]);
          }
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = acc[i + h][j][q];
            if constexpr (ADDEND) {
              const uint32_t ew[2] = {e[h].x, e[h].y};
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const uint16_t bits = (uint16_t)(ew[q >> 1] >> (16 * (q & 1)));
                v[q] = fmaf(end.alpha, IN16 ? f16_to_f32(bits) : bf16_to_f32(bits), v[q]);
              }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] *= end.factor;
            if constexpr (OUT16) half[h] = make_uint2(f16_pair(v[0], v[1]), f16_pair(v[2], v[3]));
            else half[h] = make_uint2(bf16_pair(v[0], v[1]), bf16_pair(v[2], v[3]));
            acc[i + h][j] = f32x4{0.f, 0.f, 0.f, 0.f};
            acc_touch<true>(acc[i + h][j]);
          }
          const auto x = __builtin_amdgcn_permlane16_swap(half[0].x, half[1].x, false, false);
          const auto y = __builtin_amdgcn_permlane16_swap(half[0].y, half[1].y, false, false);
          __builtin_amdgcn_raw_buffer_store_b128((u32x4){x[0], y[0], x[1], y[1]}, to, at + i * 32, j * 32 * end.ld, 0);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      acc_settle();
    }
    first = false;
    if (records == 0) break;
  }
  wait_copies<0>();
#endif
}

// Configurations: block tile, LDS stages of P and Q, blocks that a compute unit holds.
//   256       all 160 KiB of LDS for one block
//   128       half of it for each of two blocks
//   128 deep  144 KiB for a block that has its compute unit to itself (a launch that gives no unit a second one): with two
//             stages and nothing else resident, a k-tile waits for its copies
//   64        launches that cannot occupy the chip with tiles of 128: latency bound, so as many stages as two blocks leave room for
//   32        X X^T of few tiles over a long reduction, which tiles of 64 walk at the rate of the LDS port of a few units
enum { CFG_256, CFG_128, CFG_128_DEEP, CFG_64, CFG_32 };
template <int CFG> struct Config;
template <> struct Config<CFG_256> { static constexpr int BT = 256, SP = 2, SQ = 3, BLOCKS = 1; };
template <> struct Config<CFG_128> { static constexpr int BT = 128, SP = 2, SQ = 3, BLOCKS = 2; };
template <> struct Config<CFG_128_DEEP> { static constexpr int BT = 128, SP = 4, SQ = 5, BLOCKS = 1; };
template <> struct Config<CFG_64> { static constexpr int BT = 64, SP = 4, SQ = 5, BLOCKS = 2; };
template <> struct Config<CFG_32> { static constexpr int BT = 32, SP = 4, SQ = 5, BLOCKS = 2; };

// The two configurations that fill the chip, by block tile and wave tile.
template <int BM, int BN, int WM, int WN, int MODE, bool SPLIT, bool FINAL, bool ADDEND, int F16, bool SK>
__global__ void __launch_bounds__(256, Config<BM == 256 ? CFG_256 : CFG_128>::BLOCKS)
ns_gemm_kernel(const GroupedGemmParams gp) {
  static_assert(BM == BN && WM == BM / 2 && WN == BN / 2 && (BM == 256 || BM == 128), "four waves of a quarter each");
  using C = Config<BM == 256 ? CFG_256 : CFG_128>;
  ns_gemm_tile<BM, C::SP, C::SQ, MODE, SPLIT, FINAL, ADDEND, F16, SK ? CUT_BLOCKS : CUT_NONE>(gp);
}

// The two configurations for launches that do not (deeper pipelines).
template <int CFG, int MODE, bool SPLIT, bool FINAL, bool ADDEND, int F16>
__global__ void __launch_bounds__(256, Config<CFG>::BLOCKS)
ns_gemm_deep_kernel(const GroupedGemmParams gp) {
  ns_gemm_tile<Config<CFG>::BT, Config<CFG>::SP, Config<CFG>::SQ, MODE, SPLIT, FINAL, ADDEND, F16, CUT_NONE>(gp);
}

// Tiles of 32 (X X^T only).
template <int MODE, int F16>
__global__ void __launch_bounds__(256, Config<CFG_32>::BLOCKS)
ns_gemm_fine_kernel(const GroupedGemmParams gp) {
  ns_gemm_tile<Config<CFG_32>::BT, Config<CFG_32>::SP, Config<CFG_32>::SQ, MODE, false, false, true, F16, CUT_NONE>(gp);
}

// Symmetric products whose reduction is cut, one block for all parts of a tile.
template <int CFG, int MODE>
__global__ void __launch_bounds__(256, Config<CFG>::BLOCKS)
ns_gemm_sequence_kernel(const GroupedGemmParams gp) {
  ns_gemm_tile<Config<CFG>::BT, Config<CFG>::SP, Config<CFG>::SQ, MODE, false, false, true, 0, CUT_SEQUENCE>(gp);
}

template <int CFG, int MODE, bool SPLIT, bool FINAL, bool ADDEND, int F16, int CUT>
static constexpr auto kernel_of() {
  constexpr int BT = Config<CFG>::BT;
  if constexpr (CUT == CUT_SEQUENCE) {
    return &ns_gemm_sequence_kernel<CFG, MODE>;
  } else if constexpr (CFG == CFG_32) {
    return &ns_gemm_fine_kernel<MODE, F16>;
  } else
  if constexpr (CFG == CFG_256 || CFG == CFG_128) {
    return &ns_gemm_kernel<BT, BT, BT / 2, BT / 2, MODE, SPLIT, FINAL, ADDEND, F16, CUT == CUT_BLOCKS>;
  } else {
    static_assert(CUT == CUT_NONE, "the K-split runs in the 128 configuration");
    return &ns_gemm_deep_kernel<CFG, MODE, SPLIT, FINAL, ADDEND, F16>;
  }
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------
long ns_gemm_tiles(int mode, const GemmParams& p) {
  const bool sym = (mode == MODE_SYRK || mode == MODE_SYRK2 || mode == MODE_SYRKT);
  return (long)p.batch * (sym ? (long)p.tilesM * (p.tilesM + 1) / 2 : (long)p.tilesM * p.tilesN);
}

// The dynamic-LDS limit of a kernel is an attribute of the function on ONE device: set once per device (and kernel, which has one of
// these; the call is idempotent, so two threads that race on the first launch only repeat it).
struct LdsLimit {
  std::atomic<bool> set[64] = {};
  hipError_t raise(const void* kern, int bytes) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    const bool slot = dev >= 0 && dev < 64;
    if (slot && set[dev].load(std::memory_order_acquire)) return hipSuccess;
    e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess && slot) set[dev].store(true, std::memory_order_release);
    return e;
  }
};

template <int CFG, int MODE, bool SPLIT, bool FINAL, bool ADDEND = true, int F16 = 0, int CUT = CUT_NONE>
static hipError_t launch_one(const GroupedGemmParams& gp, hipStream_t stream) {
  constexpr int NT = 256;
  constexpr int SMEM = (Config<CFG>::SP + Config<CFG>::SQ) * Config<CFG>::BT * ROW_BYTES;
  constexpr auto kern = kernel_of<CFG, MODE, SPLIT, FINAL, ADDEND, F16, CUT>();
  static LdsLimit limit;
  const hipError_t e = limit.raise((const void*)kern, SMEM);
  if (e != hipSuccess) return e;
  const long tiles = gp.total;
  if (tiles <= 0) return hipSuccess;
  const long unit = 8L * xcd_run((int)tiles);
  const long grid = (tiles + unit - 1) / unit * unit;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(NT), SMEM, stream, gp);
  return hipGetLastError();
}

template <int CFG, int F16>
static hipError_t launch_cfg(int mode, bool split, bool final_, const GroupedGemmParams& p, hipStream_t s) {
  if ((F16 || CFG == CFG_64) && split) return hipErrorInvalidValue;
  if constexpr (F16 == 2) {
    if (mode != MODE_BX || final_) return hipErrorInvalidValue;
    return p.g[0].E ? launch_one<CFG, MODE_BX, false, false, true, 2>(p, s)
                    : launch_one<CFG, MODE_BX, false, false, false, 2>(p, s);
  } else {
    switch (mode) {
      case MODE_SYRK:
        return launch_one<CFG, MODE_SYRK, false, false, true, F16>(p, s);
      case MODE_SYRKT:
        return launch_one<CFG, MODE_SYRKT, false, false, true, F16>(p, s);
      case MODE_SYRK2:
        if constexpr (!F16 && CFG != CFG_64) {
          if (split) return launch_one<CFG, MODE_SYRK2, true, false>(p, s);
        }
        return launch_one<CFG, MODE_SYRK2, false, false, true, F16>(p, s);
      case MODE_BX:
        if constexpr (!F16 && CFG != CFG_64) {
          if (split) {
            if (p.g[0].E)
              return final_ ? launch_one<CFG, MODE_BX, true, true>(p, s)
                            : launch_one<CFG, MODE_BX, true, false>(p, s);
            return final_ ? launch_one<CFG, MODE_BX, true, true, false>(p, s)
                          : launch_one<CFG, MODE_BX, true, false, false>(p, s);
          }
        }
        if (p.g[0].E)
          return final_ ? launch_one<CFG, MODE_BX, false, true, true, F16>(p, s)
                        : launch_one<CFG, MODE_BX, false, false, true, F16>(p, s);
        return final_ ? launch_one<CFG, MODE_BX, false, true, false, F16>(p, s)
                      : launch_one<CFG, MODE_BX, false, false, false, F16>(p, s);
    }
    return hipErrorInvalidValue;
  }
}

// the symmetric products of the 128x128 configuration with a K-split
template <int F16>
static hipError_t launch_ksplit(int mode, const GroupedGemmParams& p, hipStream_t s) {
  switch (mode) {
    case MODE_SYRK: return launch_one<CFG_128, MODE_SYRK, false, false, true, F16, CUT_BLOCKS>(p, s);
    case MODE_SYRKT: return launch_one<CFG_128, MODE_SYRKT, false, false, true, F16, CUT_BLOCKS>(p, s);
    case MODE_SYRK2: return launch_one<CFG_128, MODE_SYRK2, false, false, true, F16, CUT_BLOCKS>(p, s);
  }
  return hipErrorInvalidValue;
}

// the same with all parts of a tile in one block (bfloat16 operands in the caller's orientation: the products of muon_syrk)
template <int CFG>
static hipError_t launch_sequence(int mode, const GroupedGemmParams& p, hipStream_t s) {
  switch (mode) {
    case MODE_SYRK: return launch_one<CFG, MODE_SYRK, false, false, true, 0, CUT_SEQUENCE>(p, s);
    case MODE_SYRK2: return launch_one<CFG, MODE_SYRK2, false, false, true, 0, CUT_SEQUENCE>(p, s);
  }
  return hipErrorInvalidValue;
}

template <bool FINAL, bool ADDEND, int F16>
static hipError_t launch_stream_one(const GroupedGemmParams& gp, hipStream_t stream, int units) {
  constexpr int SMEM = (Config<CFG_256>::SP + Config<CFG_256>::SQ) * 256 * ROW_BYTES;
  constexpr auto kern = &ns_gemm_stream_kernel<FINAL, ADDEND, F16>;
  static LdsLimit limit;
  const hipError_t e = limit.raise((const void*)kern, SMEM);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)units), dim3(256), SMEM, stream, gp);
  return hipGetLastError();
}
static hipError_t launch_stream(const GroupedGemmParams& gp, bool final_, int f16, hipStream_t s, int units) {
  const bool addend = gp.g[0].E != nullptr;
  switch (f16) {
    case 0:
      if (final_) return launch_stream_one<true, false, 0>(gp, s, units);
      return addend ? launch_stream_one<false, true, 0>(gp, s, units) : launch_stream_one<false, false, 0>(gp, s, units);
    case 1:
      if (final_) return launch_stream_one<true, false, 1>(gp, s, units);
      return addend ? launch_stream_one<false, true, 1>(gp, s, units) : launch_stream_one<false, false, 1>(gp, s, units);
    case 2:
      if (final_) return hipErrorInvalidValue;
      return addend ? launch_stream_one<false, true, 2>(gp, s, units) : launch_stream_one<false, false, 2>(gp, s, units);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_ns_gemm_grouped(int tile, int mode, bool split, bool final_, const GroupedGemmParams& asked,
                                  hipStream_t stream, int units, int f16, KCut cut) {
  const bool ksplit = cut == CUT_BLOCKS;
  GroupedGemmParams gp = asked;
  if (gp.n_groups < 1 || gp.n_groups > MAX_GROUPS) return hipErrorInvalidValue;
  const bool sym = (mode == MODE_SYRK || mode == MODE_SYRK2 || mode == MODE_SYRKT);
  if (cut != CUT_NONE && (!sym || tile != 128 || split || final_ || f16 == 2)) return hipErrorInvalidValue;
  if (cut == CUT_SEQUENCE && (asked.quarter || f16)) return hipErrorInvalidValue;
  for (int i = 0; i < gp.n_groups; ++i) {
    GemmParams& g = gp.g[i];
    if (g.K % BK != 0 || g.K <= 0 || gp.tile_start[i + 1] < gp.tile_start[i]) return hipErrorInvalidValue;
    if (mode == MODE_SYRK2 && !g.E) return hipErrorInvalidValue;
    if (mode == MODE_BX && (g.E == nullptr) != (gp.g[0].E == nullptr)) return hipErrorInvalidValue;  // one kernel per launch
    long blocks = (long)gp.tile_start[i + 1] - gp.tile_start[i];
    if (cut == CUT_NONE) {
      if (g.ksplit > 1) return hipErrorInvalidValue;
    } else if (cut == CUT_SEQUENCE) {
      if (g.ksplit < 1 || g.ksplit > g.K / BK) return hipErrorInvalidValue;
    } else {
      // every part walks at least one k-tile; the parts of a tile find their partial results and their counter
      if (g.ksplit < 1 || g.ksplit > g.K / BK || blocks % g.ksplit) return hipErrorInvalidValue;
      if (g.ksplit > 1 && (!g.sk_partial || !g.sk_counter || ((uintptr_t)g.sk_partial & 15))) return hipErrorInvalidValue;
      blocks /= g.ksplit;
    }
    // every block must decode to a tile inside the problem
    if (g.t_first < 0 || g.t_count < 0 || (g.t_count == 0 && g.t_first != 0)) return hipErrorInvalidValue;
    if (!gp.quarter) {
      const long per = ns_gemm_tiles(mode, g) / g.batch;
      if (g.t_count ? (g.t_first + g.t_count > per || blocks > (long)g.batch * g.t_count) : blocks > ns_gemm_tiles(mode, g))
        return hipErrorInvalidValue;
    } else {
      const int side = 1 << gp.quarter;
      if (gp.quarter > 2 || (ksplit && gp.quarter != 1)) return hipErrorInvalidValue;
      if (g.tilesM % side || (!sym && g.tilesN % side) || g.qt_first < 0 || blocks % (side * side)) return hipErrorInvalidValue;
      const long cm = g.tilesM / side, cn = g.tilesN / side;
      const long per = sym ? cm * (cm + 1) / 2 : cm * cn;
      if (g.t_count && g.t_first + g.t_count > per) return hipErrorInvalidValue;
      const long coarse = (long)g.batch * (g.t_count ? g.t_count : per);
      if (g.qt_first + blocks / (side * side) > coarse) return hipErrorInvalidValue;
    }
  }
  // what the kernel would otherwise divide for at the start of every tile
  for (int i = 0; i < gp.n_groups; ++i) {
    GemmParams& g = gp.g[i];
    const int dM = g.tilesM >> gp.quarter, dN = g.tilesN >> gp.quarter;
    g.per_mat = g.t_count > 0 ? g.t_count : (sym ? dM * (dM + 1) / 2 : dM * dN);
    g.part_tiles = (gp.tile_start[i + 1] - gp.tile_start[i]) / (ksplit ? g.ksplit : 1);
    if (g.per_mat < 1 || (ksplit && g.part_tiles < 1)) return hipErrorInvalidValue;
    g.inv_per_mat = reciprocal(g.per_mat);
    g.inv_line = sym ? 0u : reciprocal(dM > 8 ? 4 * dN : dM);
  }
  gp.total = gp.tile_start[gp.n_groups];
  for (int i = gp.n_groups + 1; i <= MAX_GROUPS; ++i) gp.tile_start[i] = 0x7fffffff;
  if (ksplit) {
    if (f16 == 1) return launch_ksplit<1>(mode, gp, stream);
    return launch_ksplit<0>(mode, gp, stream);
  }
  int shortest = gp.g[0].K;
  for (int i = 1; i < gp.n_groups; ++i) shortest = gp.g[i].K < shortest ? gp.g[i].K : shortest;
  const bool deep = deep_pipeline(units, tile, gp.total, shortest);
  if (cut == CUT_SEQUENCE) return deep ? launch_sequence<CFG_128_DEEP>(mode, gp, stream) : launch_sequence<CFG_128>(mode, gp, stream);
  auto by_storage = [&](auto cfg_) -> hipError_t {
    constexpr int CFG = decltype(cfg_)::value;
    if (f16 == 1) return launch_cfg<CFG, 1>(mode, split, final_, gp, stream);
    if (f16 == 2) return launch_cfg<CFG, 2>(mode, split, final_, gp, stream);
    if (f16 == 0) return launch_cfg<CFG, 0>(mode, split, final_, gp, stream);
    return hipErrorInvalidValue;
  };
  if (stream_takes(tile, mode, split, final_, gp, units)) return launch_stream(gp, final_, f16, stream, units);
  if (tile == 256) return by_storage(std::integral_constant<int, CFG_256>{});
  if (tile == 128 && deep) return by_storage(std::integral_constant<int, CFG_128_DEEP>{});
  if (tile == 128) return by_storage(std::integral_constant<int, CFG_128>{});
  if (tile == 64) return by_storage(std::integral_constant<int, CFG_64>{});
  if (tile == 32 && mode == MODE_SYRKT && !split && !final_ && f16 != 2)
    return f16 ? launch_one<CFG_32, MODE_SYRKT, false, false, true, 1>(gp, stream) : launch_one<CFG_32, MODE_SYRKT, false, false, true, 0>(gp, stream);
  return hipErrorInvalidValue;
}

}  // namespace archscale
