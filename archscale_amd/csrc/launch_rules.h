// How the tiles of one product launch are cut for the chip: plain arithmetic (no HIP), so that it can be checked on the host for any
// number of compute units.  `units` is what the current device reports; the measured lines are those of 256 units (one MI355X)
// and are scaled with it.  What is chosen for a launch never changes a result: the sums of an element are the same in every
// configuration.  The one rule that cuts sums (product_parts) is asked about one matrix at RULE_UNITS, whatever the stack and the device.
#pragma once
#include <stdint.h>

namespace archscale {

// Division by multiplication, for the start of a tile (host and device): quotient and rest of x / d for 0 <= x < 2^31 and
// 0 < d < 2^31 with inv = reciprocal(d).  The estimate is at most one too small.
constexpr uint32_t reciprocal(int d) { return 0xffffffffu / (uint32_t)d; }
constexpr int divide(int x, int d, uint32_t inv, int& rest) {
  uint32_t q = (uint32_t)(((uint64_t)(uint32_t)x * inv) >> 32), r = (uint32_t)x - q * (uint32_t)d;
  if (r >= (uint32_t)d) { ++q; r -= (uint32_t)d; }
  rest = (int)r;
  return (int)q;
}
// x / d for d = 1 .. 4 and 0 <= x < 2^31
constexpr int divide_1_to_4(int x, int d) {
  const int third = (int)(((uint64_t)(uint32_t)x * 0xaaaaaaabu) >> 33);
  return d == 4 ? x >> 2 : (d == 3 ? third : (d == 2 ? x >> 1 : x));
}

// Tiles with numbers [0, whole) of a launch run as they are, the next `quarters` as four tiles of half the side each, the next
// `sixteenths` as sixteen of a quarter of it.
struct LaunchSplit { int whole, quarters, sixteenths; };

// Tiles of 256, more than one round (one tile per unit) of them: the full rounds run as they are, a last round of at most
// QUARTER_MAX_TAIL tiles is quartered.  A round of quadrants alone runs at about 0.6 of the rate of a full round of large tiles
// (it neither overlaps the stores of the round before nor shares operand panels as well), but it takes time only for the tiles
// that are there.  Per product: leftovers of 64 tiles (X X^T of 16 x 2048 x 5632) 379 -> 324 us, of 128 (X X^T of 32 x 2048 x
// 2048; X' = BX of 4096 x 14336) 274 -> 264 and 355 -> 333; of 160 (X X^T of the depth-16 set) 1173 us as it is, 1218
// quartered; of 176 (X' = BX of the EMA-Muon set of width 1024) 90 as it is, 93 quartered.
// Less than one round: as tiles of 256 the launch takes as long as its longest tile; quartered, the tiles spread over the
// chip, at the same 0.6 of the rate.  Quartered when the mean load of a unit is below QUARTER_LOAD of the longest tile.  At 0.59
// (208 tiles of 2816 and 1024 k-values, X X^T of that EMA-Muon set) a product takes 56 us quartered, 66 as it is; at 0.625
// (160 equal tiles, power iteration over 16 x 1024 x 2816) the call takes 259 against 250 us.
//
// Tiles of 128: quartered where two quadrants to a unit hold them all (one_round_of_quadrants).
// The same again one level down: 128 tiles of 256 are exactly one round of quadrants (two to a unit); up to SIXTEENTH_MAX tiles
// left beside whole rounds of either kind become sixteen tiles of 64 each, one block per unit at most.  The 136 triangle tiles of
// a short side of 4096: 97 -> 78 us per product; 4096 x 4096 1466 -> 1376 us, 4000 x 4100 (half storage) 1683 -> 1538, 4096 x
// 14336 3353 -> 3255; more than 16 tiles so: no further gain.
constexpr int RULE_UNITS = 256;   // the device of the figures
constexpr int QUARTER_MAX_TAIL = 128;
constexpr int SIXTEENTH_MAX = 16;
constexpr double QUARTER_LOAD = 0.6;

// Tiles of 128 whose quadrants find room in one round, two to a unit: quartered whatever their reductions.  us a call, as tiles of 128 / of 64:
// one 512 x 2048 matrix 203 / 133, 3001 x 1023 286 / 198, 1500 x 2000 (78 tiles) 268 / 241, 3 x (1000 x 2000) (108) 252 / 243, 1700 x 3000 (105)
// 368 / 340, 1900 x 1900 (120) 284 / 269, 12 x (500 x 4000) (120) 375 / 354, 6 x (700 x 1300) (126) 222 / 210, single products of 1024
// x 3072 (36) 22.4 / 13.1, 512 x 512 (10) 7.9 / 5.5, 1792 x 4096 (105) 27.9 / 25.2, 3 x (1000 x 960) 25.4 / 24.8.  With a second round they lose: 13 x (512 x 1000) (130) 198 / 212, 9 x (640 x 640) (135) 169 / 191,
// 5 x (896 x 1024) (140) 225 / 260, a product of 1826 x 960 (136) 28.0 / 28.9, 2048 x 2048 (136) 288 / 342.
inline bool one_round_of_quadrants(int units, int tile, bool pair, int total) { return tile == 128 && !pair && 2L * total <= units; }

// total: tiles of the launch; all, longest: k-values of all its tiles and of the longest one; pair: products of a hi+lo pair
// (there is no configuration of 64 for them)
inline LaunchSplit launch_split(int units, int tile, bool pair, int total, double all, double longest) {
  auto scaled = [&](int tiles) { return (int)((long)tiles * units / RULE_UNITS); };
  const LaunchSplit as_is = {total, 0, 0};
  if (one_round_of_quadrants(units, tile, pair, total)) return {0, total, 0};
  if (tile != 256) return as_is;
  const int full = total / units * units, tail = total - full;
  if (tail == 0 || (full > 0 ? tail > scaled(QUARTER_MAX_TAIL) : all > QUARTER_LOAD * units * longest)) return as_is;
  const int half = units / 2, few = scaled(SIXTEENTH_MAX);   // half: one round of quadrants
  if (!pair && full > 0 && tail <= few) return {full, 0, tail};
  if (!pair && tail > half && tail - half <= few) return {full, half, tail - half};
  return {full, tail, 0};
}

// Symmetric products in tiles of 256 that make less than a round and run as tiles of 128 of the same matrices instead (`smaller` of them), each
// matrix in the order of its own smaller tiles (the quadrants of launch_split hold an empty block per diagonal tile and end with a
// scattered last round).  These are
// - every launch that launch_split quarters as a whole, and those that it cuts into quarters and sixteenths if two smaller tiles to a
//   unit hold them: 14 x (1024 x 4096) 1106 / 981 us a call; not 4 x (2048 x 4096) (544 of them), 1140 / 1214.  Up to half a round, where
//   two quadrants to a unit hold it too, four neighbours share their rows of the operands and an empty one leaves its unit to the other, only
//   what is less than a third of a round with at most nine smaller tiles to eight units, most of them alone on theirs.  us of a stack of
//   single products as quadrants / so: 12 x (1024 x 2816) (120 large, 432 smaller tiles) 46.4 / 48.9, 9 x (1024 x 2816) (90, 324) 37.7 / 40.1,
//   128 x (256 x 1024) (128, 384) 18.1 / 20.0, 32 x (512 x 1024) (96, 320) 18.2 / 18.6, 17 x (768 x 2816) (102, 357) 38.5 / 40.0, 3 x (2048 x 2048)
//   (108, 408) 30.9 / 31.7, 14 x (768 x 1024) (84, 294) 18.2 / 18.4, 4 x (1521 x 416) (84, 312) 34.8 / 35.4, 96 x (256 x 1024) (96, 288) 17.7 / 18.1;
//   but 8 x (1024 x 2816) (80, 288) 37.3 / 35.7, 28 x (512 x 1024) (84, 280) 18.0 / 17.8, 2 x (2048 x 1024) (72, 272) 17.7 / 17.0, 25 x (512 x 2048)
//   (75, 250) 26.4 / 18.2;
// - launches up to a full round with reductions of up to HALVED_MAX_K: the results of a round of large tiles all leave at its end, 10 of 30 to
//   40 us with the matrix cores idle, while two smaller blocks to a unit store and multiply at the same time.  What decides is the
//   second round of smaller tiles, those beyond two to a unit (second_load: their k-values; HALVED_TILE_K more for what a tile costs
//   beside them).  As it is / so, us of a single product:
//   up to half of it, in tiles of the longest reduction: 60 x (512 x 768) (600 smaller tiles) 26.5 / 25.0, 36 x (768 x 768) (756) 27.7 / 26.9, 5 x (2048 x 768) (680) 27.6 / 26.2, 21 x
//     (1024 x 1024) (756) 31.9 / 30.5; more of it: 38 x (768 x 768) (798) 28.4 / 29.6, 6 x (2048 x 1024) (816) 33.5 / 36.2, 83 x (512 x 768) (830) 29.4 / 31.0;
//   beyond HALVED_LONG_K not where it is nearly empty: 16 x (1024 x 2816) (576), power iteration, 235 / 247 a call;
//   reductions of up to HALVED_SHORT_K whatever it holds: 83 x (512 x 256) (830) 20.2 / 18.3, 7 x (2048 x 256) (952) 22.2 / 19.7;
//   matrices of one tile a side (3 smaller tiles for one, not 3.3 and more) only where it holds next to nothing: 170 x (256 x 768) (510)
//     24.8 / 17.6, 180 (540) 24.9 / 24.6, but 190 (570) 25.1 / 26.3, 217 (651) 25.7 / 28.3; of 512 k-values 200 (600) 21.0 / 20.9, 210 (630) 21.2 / 21.6.
//   Whole steps: the EMA-Muon set of width 1024 (744) 1128 / 1090; 64 + 64 experts, whose short products are 640 tiles of 512 k-values and then 192 of
//   256 (320 in the second round) 1231 / 1220; a MuonH set of width 1001, whose products of the tail are 756 tiles of 1024 and then 42 of 256 (286),
//   37.7 / 43.6 us a product, 1713 / 1727 a step: with a HALVED_TILE_K of 52 to 256 it stays large and the experts do not.
// At longer reductions they lose: X X^T of 64 + 64 experts (K = 2048), 1214 / 1278 a step.
constexpr int HALVED_MAX_K = 1024, HALVED_LONG_K = 768, HALVED_ONE_K = 512, HALVED_SHORT_K = 256, HALVED_TILE_K = 160;
inline bool halved_tiles(int units, int tile, bool pair, int total, long smaller, double second_load, double longest, const LaunchSplit& cut) {
  if (tile != 256 || pair) return false;
  if (cut.whole == 0) return (2L * total > units || (3L * total < units && 8 * smaller <= 9L * units)) && (cut.sixteenths == 0 || smaller <= 2L * units);
  if (cut.whole != total || total > units || longest > HALVED_MAX_K) return false;
  const long second = smaller - 2L * units;   // tiles of the second round
  if (longest <= HALVED_SHORT_K) return true;
  if (5 * smaller < 16L * total) return 8 * second <= (longest <= HALVED_ONE_K ? 3L : 1L) * units;   // (mostly one tile a side)
  return second_load + (double)HALVED_TILE_K * second <= units * (longest + HALVED_TILE_K) && (longest <= HALVED_LONG_K || 3 * second >= units);
}

// Parts that the reduction of a single symmetric product (not of a Newton-Schulz call) is cut into, as tiles of 128 (`tiles` of one
// matrix) with at most one block to a unit.  The cut fixes the order of the sums, so callers ask for RULE_UNITS units and one
// matrix: a matrix has the same bits alone, in a stack and on any device.  Few tiles walk a long reduction on few units; a part costs 64 KiB of traffic each way and the call a
// launch that clears the counters, so a part has at least SPLIT_PART_KT k-tiles and there are three of them or none (five where there
// are only one or two tiles, which tiles of 64 walk faster: 100 x 4000 23.5 whole, 27.7 in three; 128 x 8192 25.6 / 23.2).
// us, whole / as split here: 512 x 4096 27.0 / 21.9, 512 x 16384 89 / 31, 1024 x 4096 27.9 / 22.4, 1024 x 8192 48.7 / 26.8, 1536 x
// 8192 50.1 / 34.6, 256 x 4096 26.2 / 24.2.  Not split: 512 x 2048 (16.5 whole, 18.8 in two), 2048 x 5632 (136 tiles: 37.7 whole, 41.3 in
// three with two blocks to a unit, which share the LDS port that bounds a lone one).
constexpr int SPLIT_PART_KT = 20, SPLIT_MIN_PARTS = 3, SPLIT_MAX_PARTS = 8;
inline int product_parts(int units, long tiles, int kt) {
  long parts = units / tiles;
  if (parts > kt / SPLIT_PART_KT) parts = kt / SPLIT_PART_KT;
  if (parts > SPLIT_MAX_PARTS) parts = SPLIT_MAX_PARTS;
  return parts < (tiles < 3 ? SPLIT_MIN_PARTS + 2 : SPLIT_MIN_PARTS) ? 1 : (int)parts;
}

// The same for a matrix whose extents call for tiles of `tile`.  Where that is 128, three tiles and more run whole as tiles of 64, which keep
// up with the parts until the reduction is SPLIT_MIN_KT_128 k-tiles long.  us, whole / cut: 384 x 4480 16.9 / 20.6, 640 x 3840 16.3 /
// 20.7, 896 x 4480 16.9 / 23.1, 1152 x 4480 17.5 / 24.2, 896 x 6400 22.0 / 23.8, 640 x 7680 25.2 / 25.7, 640 x 8192 26.6 / 25.2, 896 x
// 8192 26.6 / 25.2, 384 x 10240 31.9 / 25.9.
constexpr int SPLIT_MIN_KT_128 = 128;
inline int matrix_parts(int tile, long tiles, int kt) {
  return tile == 128 && tiles >= 3 && kt < SPLIT_MIN_KT_128 ? 1 : product_parts(RULE_UNITS, tiles, kt);
}

// Who walks the parts of a stack's tiles (`tiles` of all its matrices): a block each while the tiles alone would leave two thirds of
// the chip idle, one block all of them otherwise.  us, in sequence / by blocks: 60 tiles of 640 x 16384 (8 parts) 94 / 48, 72 of 1024 x
// 8192 (6) 51 / 38, 84 of 700 x 5800 (4) 61 / 60; 90 of 640 x 4096 (3) 29 / 31, 108 of 1000 x 4000 (3) 50 / 58, 120 of 256 x 8192
// (6) 54 / 61.  Large stacks pay for bits that do not depend on them: whole, in tiles of 256, 64 of 512 x 4096 take 97 us,
// in sequence 124; 256 of them 326 / 379, 64 of 1024 x 4096 275 / 325, 16 of them 89 / 88; extents that tiles of 128 serve
// anyway lose nothing (64 of 640 x 8192 267 / 268, 1000 of 128 x 8192 403 / 403).
inline bool parts_by_blocks(long tiles) { return tiles <= RULE_UNITS / SPLIT_MIN_PARTS; }

// X' = B X in tiles of 256 as a stream (ns_gemm_stream_kernel: one block per unit, its tiles one after the other) where units have two tiles
// or more (launch_split leaves a round and less or more than one and a half), for reductions of up to STREAM_MAX_K: what it saves
// is a constant per tile.  tile by tile / as a stream, us: the 64 + 64 expert matrices (K = 512 and 256) 1311 / 1250 a step, the EMA-Muon set
// of width 1024 1187 / 1163, the depth-16 set (K = 2048 and 512, at the power limit) 21980 / 21660; 4096 x 14336 (K = 4096) 3063 / 3106 a
// call.  The grid is a multiple of the eight XCDs.
constexpr int STREAM_MAX_K = 2048;
inline bool stream_of_tiles(int units, int total, int longest) {
  return units % 8 == 0 && total >= units + units / 2 && longest <= STREAM_MAX_K;
}

// X' = B X walks its problems and matrices backwards where the iterates of a call (bf16 bytes) are at most this: it then meets the
// matrices that X X^T has read last first, and the next X X^T the ones that it has written last, while the memory-side cache
// (256 MB for X, X' and the square matrices) still holds them.  Iterates of 90 MB: MuonBall step 1519 -> 1494 us, EMA Muon 1216 ->
// 1209; of 200 MB (64 experts), where neither order finds them, 1329 -> 1343; of 1.4 GB no difference.
constexpr long BACKWARDS_BYTES = 128L << 20;

// X X^T of so few tiles of 128 over a long reduction that even as tiles of 64 it leaves most of the chip idle: as tiles of 32, one
// block to a unit.  us per call, as tiles of 64 / of 32: 512 x 2048 119.5 / 108.3, 512 x 8192 215 / 183, 256 x 2048 104 / 90, 640 x
// 4096 (15 tiles) 167 / 147, 256 x 1024 88.6 / 82.5; beyond one block to a unit they lose: 700 x 3000 (21 tiles) 160 / 171, 1023 x 3001
// (36) 193 / 227.
constexpr int FINE_MAX_128 = 16, FINE_MIN_K = 1024;
inline bool fine_tiles(int units, int tile, int total, double longest) {
  return tile == 128 && (long)total * RULE_UNITS <= (long)FINE_MAX_128 * units && longest >= FINE_MIN_K;
}

// Tiles of 128 in the deep form where every block finds a unit of its own and the reductions are long: 3001 x 1023 302 -> 286 us,
// 1500 x 2000 290 -> 270, a symmetric product of 2048 x 5632 47 -> 41; filling four stages costs reductions of 640 and less
// 1 to 4 %.
inline bool deep_pipeline(int units, int tile, int blocks, int shortest_k) {
  return tile == 128 && blocks <= units && shortest_k >= 1024;
}

// Plain AdamW and Lion, by which of their arrays are in fp32 (weights, gradient, momentum, variance): in runs of eight elements, or one element
// per thread where the number of elements is no multiple of eight or an array is not 16-byte aligned and most accesses are fp32 (a run is
// then two accesses per lane that share lines with the neighbours').  us, in runs / element by element: all fp32, 34117 x 1641 twice, AdamW 638 /
// 614, Lion 453 / 426; 15916 x 1335 twice 245 / 235 and 174 / 170; 21.2 million elements, AdamW: state alone in fp32 99 / 91, all but the gradient
// 119 / 128, all but the weights 107 / 123, all in bfloat16 59 / 100; Lion: weights and momentum in fp32 80 / 63, gradient and momentum 67 / 62,
// momentum alone 59 / 73, all in bfloat16 40 / 74.
constexpr bool update_in_runs(bool adamw, bool w, bool g, bool m, bool v, bool whole_and_aligned) {
  return whole_and_aligned || !(adamw ? m && v && w == g : w + g + m >= 2);
}

// Whether the sum of squares of a matrix goes over its elements in runs of eight (thread_sumsq_dense): rows that follow one another, and whole
// runs or more than one chunk of `chunk` elements, whose blocks then load all they have at once.  An odd matrix of one chunk is over sooner one
// element per thread, whole small calls in bfloat16 / fp32, in runs / so: 8 x (67 x 33) 22.0 / 19.8 and 21.0 / 19.5 us, 16 x (101 x 51) 21.3 / 19.4 and
// 20.2 / 19.3, 3 x (61 x 95) 21.7 / 20.7 and 20.8 / 20.1; of two chunks and more 95 x 121 34.9 / 34.3 and 34.3 / 34.1 (before / in runs), 127 x 381 70.1 /
// 62.3 and 68.9 / 62.1.
constexpr bool sums_in_runs(int rows, int cols, int ld, int chunk) {
  const long n = (long)rows * cols;
  return ld == cols && (n % 8 == 0 || n > chunk);
}

// Blocks that sum the squares of one matrix of the power iteration that is read in place and needs no row sums (a tall one), each
// eight 16-byte runs per thread at a time: as many as the matrix has loads for, whatever its short side (`strips`, which the start
// vector is written by), up to two rounds of the chip, which keep the memory busy.
constexpr int SUM_RUNS = 2048, SUM_MAX_BLOCKS = 512;
inline int sum_blocks(long runs, int strips) {
  const long blocks = (runs + SUM_RUNS - 1) / SUM_RUNS;
  const int most = strips > SUM_MAX_BLOCKS ? strips : SUM_MAX_BLOCKS;
  return blocks < strips ? strips : (blocks > most ? most : (int)blocks);
}

}  // namespace archscale
