// pair_range.hpp — a tile's share of the triangle pairs of two particles
// (host + device; the host build lets CPU tests walk the limits).
#pragma once
#include "exact_math.hpp"

namespace dh {

constexpr int kPairChunk = 256;  // triangle pairs a workgroup takes at a time

// `count` triangle pairs from (row, col) on, in row-major order.
struct PairRange {
  long long count;
  int row, col;
};

// Tile `tile` of `tiles` (at most 64) over the rows x cols pairs of two particles,
// in whole chunks of kPairChunk (the last one the remainder).  The number of
// pairs passes 32 bits from 65,536 triangles each; below, the three divisions
// are of 32 bits (64 bits took 1.3 us of the 147 of 363 pairs of 80 x 80).
DH_HD PairRange pair_range(int rows, int cols, int tiles, int tile) {
  const long long all = static_cast<long long>(rows) * cols;
  if (all <= 0xffffff00ll) {
    const unsigned n = static_cast<unsigned>(all), chunks = (n + kPairChunk - 1) / kPairChunk;
    const unsigned t = static_cast<unsigned>(tile), of = static_cast<unsigned>(tiles);
    const unsigned a = kPairChunk * (t * chunks / of), b = kPairChunk * ((t + 1) * chunks / of);
    const unsigned row = cols > 0 ? a / static_cast<unsigned>(cols) : 0u;
    return {static_cast<long long>((b < n ? b : n) - a), static_cast<int>(row),
            static_cast<int>(a - row * static_cast<unsigned>(cols))};
  }
  const long long chunks = (all + kPairChunk - 1) / kPairChunk;
  const long long a = kPairChunk * (tile * chunks / tiles);
  const long long b = kPairChunk * ((tile + 1) * chunks / tiles);
  const int row = static_cast<int>(a / cols);
  return {(b < all ? b : all) - a, row, static_cast<int>(a - static_cast<long long>(row) * cols)};
}

// The pairs t, t + kPairChunk, ... of a range: no product, and no quotient after
// the first (rows and columns below 2^31 - kPairChunk).
struct PairWalk {
  int iA, iB, rows, cols;  // the pair; kPairChunk as rows and columns
  DH_HD PairWalk(const PairRange& r, int n, int t) {
    const unsigned c = static_cast<unsigned>(r.col) + static_cast<unsigned>(t);
    const unsigned m = n > 0 ? static_cast<unsigned>(n) : 1u;
    iA = r.row + static_cast<int>(c / m);
    iB = static_cast<int>(c % m);
    rows = static_cast<int>(kPairChunk / m);
    cols = static_cast<int>(kPairChunk % m);
  }
  DH_HD void next(int n) {
    iA += rows;
    iB += cols;
    const bool wrap = iB >= n;
    iA += wrap ? 1 : 0;
    iB -= wrap ? n : 0;
  }
};

}  // namespace dh
