// Partial stage tiles: the block of a tile of any width, and where its threads
// stand.  Plain arithmetic, for the launcher, the kernel and host code alike.
#pragma once

namespace solar {

// Threads of a stage block with tiles of width w: its points, and its halo
// cells (6 w above and below, filled up to a wave, and 6 tj beside).
constexpr int part_threads(int w, int tj) {
  const int points = (w * tj + 63) / 64 * 64, halo = ((6 * w + 63) / 64 * 64 + 6 * tj + 63) / 64 * 64;
  return points > halo ? points : halo;
}

// The column and row of the tile at which thread tid of a w x tj tile works,
// and whether that point is its own.  The block has surplus threads (tid / w of
// one reaches row 11 of 8 at w = 17): they work at the first point, so that
// every LDS cell they read is there, and own nothing.  (At the last row
// instead, a middle stage took 129 registers and three waves a SIMD for 127
// and four.)
struct PartPoint {
  int tx, ty;
  bool own;
};
constexpr PartPoint part_point(int tid, int w, int tj) {
  const bool own = tid < w * tj;
  const int t = own ? tid : 0;
  return {t % w, t / w, own};
}

// Width of a partial-tile panel's stage tiles: from 64 down to 33, the one
// that leaves the fewest lanes without a point, the widest of near equals (us
// per stage, 6x200^2x150: 40 wide 1177, 50 1432, 34 1608, 16x16 tiles 1240;
// 6x250^2x60: 63 wide 771, 50 856, 42 895).  Multiples of 8 where the rows
// are.  One shell makes too few blocks to fill the chip: there the narrowest
// of near equals, down to 26 (6x204^2: 30 wide 19.9, 51 22.8; 6x250^2: 32 wide
// 24.2, 63 26.2).
constexpr int part_width(int n, int nr) {
  const int narrow = nr == 1 ? 26 : 33;
  int best = 0;
  double least = 0.0;
  for (int t = (n + 63) / 64; t <= (n + narrow - 1) / narrow || t == (n + 63) / 64; ++t) {
    int w = (n + t - 1) / t;
    if (n % 8 == 0) w = (w + 7) / 8 * 8;
    const double lanes = (double)part_threads(w, 8) * t;
    if (least == 0.0 || lanes < (nr == 1 ? 1.03 : 0.97) * least) {
      least = lanes;
      best = w;
    }
  }
  return best;
}

}  // namespace solar
