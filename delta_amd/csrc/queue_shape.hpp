// queue_shape.hpp — when the survivor queue is taken, and the places of its
// entries (detect.hip, learned.hip; the host build lets CPU tests check them).
#pragma once
#include "exact_math.hpp"

namespace dh {

// Items as detect_queue_min_items counts them: one for every 16 triangles of
// the mean particle.  The queue's launches and their chain of dependent loads
// cost some 40 us; without it each item is a workgroup's, which the larger
// particles make the costlier (captured steps with and without the queue: 36
// pairs of 80 triangles 92 and 83 us, 484 pairs 113 and 124, 2,500 pairs 134
// and 169, 33,000 pairs 235 and 612).  Never 2^30, the setting for no queue.
DH_HD long long queue_items(long long items, int ntri, int nparticles) {
  const long long per = nparticles > 0 ? static_cast<long long>(ntri) / nparticles / 16 : 0;
  const long long n = per > 1 ? items * per : items;
  return n < 1ll << 30 ? n : (1ll << 30) - 1;
}

// Parts of the pool, each with a counter of its own: a wave starts with the part
// of its workgroup's number and goes on to the next when that is used up.
constexpr int kPoolParts = 16;
// Counters this far apart (words), in lines of their own: next to one another,
// 4,096 waves that each took a block once made the 115 us of a lattice of 17,576
// spheres 326 us.
constexpr int kPoolStride = 64;

// The queue's segments: first one of rcap entries for every wave of the
// mid-phase, then the pool's blocks, numbered through the parts in turn, so
// that the blocks in use come first and lie evenly over the workgroups.
struct QueueShape {
  int rcap, regions;  // the waves' own
  int block, blocks;  // entries of a block, blocks of a part (one after another)

  DH_HD int segments() const { return regions + kPoolParts * blocks; }
  DH_HD long long entries() const {
    return static_cast<long long>(regions) * rcap +
           static_cast<long long>(kPoolParts) * blocks * block;
  }
  // the number of block b of a part
  DH_HD int pool_segment(int part, int b) const {
    return regions + kPoolParts * b + part;
  }
  // the place of segment r's first entry
  DH_HD long long place(int r) const {
    if (r < regions) return static_cast<long long>(r) * rcap;
    const int part = (r - regions) % kPoolParts, b = (r - regions) / kPoolParts;
    return static_cast<long long>(regions) * rcap +
           (static_cast<long long>(part) * blocks + b) * block;
  }
};

}  // namespace dh
