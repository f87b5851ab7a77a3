// Which block tile a tile product takes (gemm_mfma.hip) and in how many pieces of k: plain host arithmetic, evaluated for
// every new number of tokens.  In continuous batching nearly every step has one: four products of a 1B layer are planned in
// 13 us here and in the calls that ask for it (135 in Python, where this rule stood first: steps of 154 to 524 tokens whose
// count changes each time 2,520 -> 2,445 us, as fast now as with a count seen before).
#pragma once

namespace tile_plan {

// A block tile: its code (0: the 128 x 128 kernel; 10 WI + WJ of the larger tiles), rows and columns, blocks that a unit
// holds at a time, and the microseconds of a block that has the chip nearly to itself and of one on a full chip, for k in
// units of 1,024.  Fitted to measurements on an MI355X of 129 to 2,627 rows with nine matrices of 2,048 x 2,048 to
// 28,672 x 4,096, whole and in two to four pieces.  543 x 28,672 x 4,096: 336 tiles of 256 x 256 take two rounds of 256
// units, 184 us; 225 of 192 x 384 one, 130 us.  2,048 x 4,384 x 2,048: 61 us on 128 x 128, 42 to 48.
struct Shape {
  int code, rows, cols, slots;
  double alone[3], full[2];
};
constexpr Shape SHAPES[] = {
    {0, 128, 128, 2, {6.0, 8.0, 0.35}, {6.0, 16.5}},
    {42, 256, 256, 1, {7.0, 15.0, 0.25}, {6.0, 26.0}},
    {33, 192, 384, 1, {8.0, 18.0, 0.3}, {7.0, 32.5}},
    {32, 192, 256, 1, {7.0, 12.5, 0.25}, {5.0, 23.5}},
    {23, 128, 384, 1, {7.0, 13.5, 0.3}, {5.0, 28.0}},
    {22, 128, 256, 1, {6.0, 10.0, 0.25}, {4.0, 20.5}},
};
constexpr int SLAB = 64;               // k per slab: the larger tiles take whole slabs only
constexpr int MAX_SPLITS = 8;
constexpr int MIN_K = 256;             // a piece keeps at least this much of k
// What the fit, which is good to some per cent, must promise at least before another shape or one more piece is taken.
constexpr double SHAPE_GAIN = 0.96, PIECES_GAIN = 0.96;
// Bytes per microsecond of pieces, or of the updated stream, on their way into the norm behind the product, and what every
// piece takes there besides (writing them is hidden in the times above).  Fitted to product and norm together, 176 sizes of 130
// to 2,627 rows in one to eight pieces, and to whole prompts, whose weights are cold: 300 x 2,048 x 2,048 takes
// 18.4 us in four pieces and 21.3 in eight, 256 x 4,096 x 4,096 24.3 and 28.7, 700 x 1,024 x 1,024 14.9 in two and 17.0 in four.
// Rows of more than 4,096 columns go through the norm at half that rate (1,267 x 5,376 x 4,544: 104 us in one piece, 175 in two).
constexpr double PIECES_READ = 4e6, WIDE_READ = 2e6, PIECE_US = 0.3;
constexpr int WIDE = 4096;

inline double shape_us(const Shape& s, int M, int N, int K, int splits, int units) {
  const int per_piece = (K + splits - 1) / splits;
  const double k = (per_piece + SLAB - 1) / SLAB * SLAB / 1024.0;
  const long tiles = ((long)M + s.rows - 1) / s.rows * (((long)N + s.cols - 1) / s.cols) * splits;
  const long slots = (long)s.slots * units, rounds = tiles / slots, rest = tiles % slots;
  const double top = s.full[0] + s.full[1] * k;
  double low = s.alone[0] + s.alone[1] * k + s.alone[2] * k * k;
  if (low > top) low = top;
  return rounds * top + (rest ? low + (top - low) * rest / slots : 0.0);
}

struct Choice {
  int code;
  double us;
};
// The shape that takes the least time for the product in `splits` pieces, and that time.
inline Choice shape_for(int M, int N, int K, int splits, int units) {
  Choice best{0, shape_us(SHAPES[0], M, N, K, splits, units)};
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
inline int splits_for(int M, int N, int K, int units, long part_floats, double worth) {
  const double read = N > WIDE ? WIDE_READ : PIECES_READ;
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
