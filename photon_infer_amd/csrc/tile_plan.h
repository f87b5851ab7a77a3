// Which block tile a tile product takes (gemm_mfma.hip) and in how many pieces of k: plain host arithmetic, evaluated for
// every new number of tokens.  In continuous batching nearly every step has one: four products of a 1B layer are planned in
// 13 us here and in the calls that ask for it (135 in Python, where this rule stood first: steps of 154 to 524 tokens whose
// count changes each time 2,520 -> 2,445 us, as fast now as with a count seen before).
#pragma once

#include <cmath>

namespace tile_plan {

// A block tile: its code (0: 128 x 128, in the kernel that takes it the faster; 10 WI + WJ of the larger tiles), rows and columns, blocks that a unit
// holds at a time, and the microseconds of a block that has the chip nearly to itself and of one on a full chip, for k in
// units of 1,024.  Fitted on an MI355X to 402 products of 130 to 3,000 rows with twenty matrices of 832 x 2,048 to 28,672 x 4,096
// in every shape, weights cold, and to 301 of them in one to eight pieces with the norm that adds these: the shape it takes
// is 0.1 % slower than the fastest in the mean (10 % at worst, 1,293 x 3,072 x 3,072).  543 x 28,672 x 4,096: 336 tiles of
// 256 x 256 take two rounds of 256 units, 184 us; 225 of 192 x 384 one, 121 us.
struct Shape {
  int code, rows, cols, slots;
  double alone[3], full[2];
};
constexpr Shape SHAPES[] = {
    {0, 128, 128, 2, {1.0, 5.84, 0.66}, {4.95, 14.69}},
    {42, 256, 256, 1, {5.29, 15.8, 0.05}, {8.75, 19.82}},
    {33, 192, 384, 1, {6.33, 19.74, 0.41}, {9.56, 26.3}},
    {32, 192, 256, 1, {4.98, 13.26, 0.08}, {7.45, 17.28}},
    {23, 128, 384, 1, {5.81, 13.05, 1.03}, {5.25, 22.8}},
    {22, 128, 256, 1, {3.83, 9.42, 0.17}, {5.08, 13.23}},
};
// 128 x 128 in the larger tiles' kernel, one block of eight waves to a unit, for whole slabs of k: taken in the place of the
// 128 x 128 kernel where it is the faster one of the two (256 tiles of k = 8,192 82 us instead of 104; 512 of k = 256 15.5
// and of k = 2,048 50 us instead of 41, two of whose blocks a unit holds).
constexpr Shape RING_128 = {21, 128, 128, 1, {3.47, 6.48, 0.05}, {4.15, 8.63}};
constexpr int SLAB = 64;               // k per slab: the larger tiles take whole slabs only
constexpr int MAX_SPLITS = 8;
constexpr int MIN_K = 256;             // a piece keeps at least this much of k
// What the fit must promise at least before another shape or one more piece is taken.
constexpr double SHAPE_GAIN = 0.97, PIECES_GAIN = 0.945;
// Bytes per microsecond of pieces, or of the updated stream, on their way into the norm behind the product, and what every
// piece takes there besides (writing them is hidden in the times above).  Over the 301 products measured with the norm the
// choice is 0.9 % above the best in the mean: 300 x 2,048 x 8,192 takes 68 us in one piece, 28.2 in five and 29.5 in eight,
// 256 x 4,096 x 4,096 48, 25.7 in three and 28.5.  Rows of more than 4,096 columns go through the norm at a third of that
// rate (1,267 x 5,376 x 4,544: 104 us in one piece, 175 in two), through the rotation of q, k and v at the same (500 x 6,144 x
// 4,096 with the rotation 48.8 us in one float32 piece, 43.8 in two; 500 x 5,120 x 3,072 41.5, 34.1 in three).
constexpr double PIECES_READ = 5.8e6, WIDE_READ = PIECES_READ / 3, PIECE_US = 0.09;
constexpr int WIDE = 4096;

inline double shape_us(const Shape& s, int M, int N, int K, int splits, int units) {
  const int per_piece = (K + splits - 1) / splits;
  const double k = (per_piece + SLAB - 1) / SLAB * SLAB / 1024.0;
  const long tiles = ((long)M + s.rows - 1) / s.rows * (((long)N + s.cols - 1) / s.cols) * splits;
  const long slots = (long)s.slots * units, rounds = tiles / slots, rest = tiles % slots;
  const double top = s.full[0] + s.full[1] * k;
  double low = s.alone[0] + s.alone[1] * k + s.alone[2] * k * k;
  if (low > top) low = top;
  if (!rest) return rounds * top;
  // where a unit holds two blocks, the units that have two decide
  const double share = s.slots > 1 ? std::sqrt((double)rest / slots) : (double)rest / slots;
  return rounds * top + low + (top - low) * share;
}

inline bool ring_128_takes(int M, int N, int K, int splits, int units) {
  return K % SLAB == 0 && shape_us(RING_128, M, N, K, splits, units) < shape_us(SHAPES[0], M, N, K, splits, units);
}

struct Choice {
  int code;
  double us;
};
// The shape that takes the least time for the product in `splits` pieces, and that time.
inline Choice shape_for(int M, int N, int K, int splits, int units) {
  Choice best{0, shape_us(ring_128_takes(M, N, K, splits, units) ? RING_128 : SHAPES[0], M, N, K, splits, units)};
  if (K % SLAB) return best;
  for (const Shape& s : SHAPES) {
    if (s.code == 0) continue;
    const double us = shape_us(s, M, N, K, splits, units);
    if (us < best.us * (s.code == 42 ? 1.0 : SHAPE_GAIN)) best = Choice{s.code, us};
  }
  return best;
}

// In how many pieces a product is left whose reader adds them: as many as take the least time together with their way
// through memory, if they take at most `worth` of the time in one piece, and no more than `part_floats` floats hold.
// `norm`: the reader is a norm, whose rows may be wide.
inline int splits_for(int M, int N, int K, int units, long part_floats, double worth, bool norm) {
  const double read = norm && N > WIDE ? WIDE_READ : PIECES_READ;
  const double whole = shape_for(M, N, K, 1, units).us + 4.0 * M * N / read;      // the kernel adds into the stream
  int best = 1;
  double least = whole;
  for (int splits = 2; splits <= MAX_SPLITS; ++splits) {
    if (K / splits < MIN_K || (long)splits * M * N > part_floats) break;
    const double us = shape_for(M, N, K, splits, units).us + 4.0 * splits * M * N / read + PIECE_US * splits;
    if (us < PIECES_GAIN * least) { best = splits; least = us; }
  }
  return best > 1 && least > worth * whole ? 1 : best;
}

}  // namespace tile_plan
